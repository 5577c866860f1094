"""get_kv through the HIP dequantiser (csrc/dequant.hip): the bits of the torch expressions it
replaces (kept for other dtypes), for every engine format, around a wave's 16 tokens, with static
(stride 0) and per-token scales, growth (capacity above the length) and a residual window."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _engines(n):
    import llm_kvcache_quantization_amd as K

    g = torch.Generator().manual_seed(1)
    s8 = 0.01 + 0.02 * torch.rand(1, 3, 8, generator=g)
    s4 = 0.1 + 0.4 * torch.rand(1, 3, 4, generator=g)
    return {
        "int8": lambda d: K.INT8KVCache(1, group_size=32, dtype=d),
        "int8_static": lambda d: K.INT8KVCache(1, group_size=16, dtype=d, static_k_scale=s8.half(),
                                               static_v_scale=s8),
        "int4": lambda d: K.INT4KVCache(1, group_size=16, dtype=d),
        "int4_static": lambda d: K.INT4KVCache(1, group_size=32, dtype=d, static_k_scale=s4, static_v_scale=s4),
        "int4_g128": lambda d: K.INT4KVCache(1, group_size=128, dtype=d),
        "kivi8": lambda d: K.KIVIStyleKVCache(1, quant_bits=8, dtype=d),
        "kivi4": lambda d: K.KIVIStyleKVCache(1, quant_bits=4, dtype=d, residual_length=3),
        **{f"alloc{a}{b}": (lambda d, p=(a, b): K.RoleAwareAllocatorKVCache(1, per_layer_bits=[p], dtype=d))
           for a, b in ((4, 8), (8, 4), (16, 4), (8, 16))},
        **{f"mixed{a}{b}": (lambda d, p=(a, b): K.MixedKVCache(1, k_group_size=64, k_bits=p[0], v_bits=p[1],
                                                                dtype=d))
           for a, b in ((8, 4), (4, 8), (4, 4), (8, 8), (16, 8), (4, 16))},
    }


@pytest.mark.parametrize("n", [1, 15, 16, 17, 331, 1100])
def test_get_kv_bits(n):
    g = torch.Generator(device="cuda").manual_seed(n)
    k, v = (torch.randn(2, 3, n + 4, 128, generator=g, device="cuda").half() * s for s in (3, 1))
    k[..., 7] *= 30
    k[0, 0, 0] = 0
    for name, make in _engines(n).items():
        got = []
        for dtype in (torch.float16, torch.float32):  # fp32: the torch expressions, not rounded yet
            c = make(dtype)
            c.append(0, k[:, :, :n], v[:, :, :n])
            for t in range(n, n + 4):
                c.append(0, k[:, :, t:t + 1], v[:, :, t:t + 1])
            got.append(c.get_kv(0))
        bits = c._bits[0] if hasattr(c, "_bits") else (0, 0)
        for a, b, w in zip(*got, bits):
            assert a.dtype == torch.float16 and a.shape == (2, 3, n + 4, 128), name
            assert w == 16 or a.is_contiguous(), name  # (a 16-bit side is a view of the cache)
            assert torch.equal(a, b.half()), name
