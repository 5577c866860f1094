"""The HIP per-channel range of a KIVI prompt (csrc/kivi_range.hip): bit-exact against the oracle's
quantize_asymmetric_per_channel (torch.quantile on the CPU), at the edges of the rows a thread holds
(2048 for 4 waves, 8192 for 16), for few and many (b, head) units, transposed and odd strides, ties
and subnormals; and the torch path's handling of NaN / Inf."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _k(B, H, S, seed):
    g = torch.Generator().manual_seed(seed)
    k = torch.randn(B, H, S, 128, generator=g).half()
    k[..., 5] *= 100
    k[..., 17] = torch.randint(-2, 3, k[..., 17].shape, generator=g).half()   # ties
    k[..., 31] *= 2.0 ** -20                                                    # subnormals
    k[..., 40] = 0.0
    k[..., 41] = -0.0
    k[..., 63] = -k[..., 63].abs()
    return k


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("pct", [100.0, 99.9, 97.3, 51.0])
@pytest.mark.parametrize("shape", [(1, 1, 1), (1, 2, 2), (2, 5, 37), (1, 2, 2048), (1, 1, 2049), (3, 3, 700),
                                   (1, 1, 8192), (1, 1, 8193), (1, 1, 17001)], ids=str)
def test_channel_range_bitexact(shape, pct, bits):
    from llm_kvcache_quantization_amd.cache import kivi_channel_params
    from oracle import quant as OQ

    k = _k(*shape, seed=shape[2])
    _, rs, rz = OQ.quantize_asymmetric_per_channel(k, bits, pct)
    s, z = kivi_channel_params(k.cuda(), bits, pct)
    assert torch.equal(s.cpu(), rs) and torch.equal(z.cpu(), rz)


@pytest.mark.parametrize("pct", [99.999999, 50.000001])
@pytest.mark.parametrize("n", [1, 2, 301, 9000])
def test_channel_range_rounded_levels(n, pct):
    """Percentiles whose fp32 levels are 1, or equal: the ranks are still torch.quantile's."""
    from llm_kvcache_quantization_amd.cache import kivi_channel_params
    from oracle import quant as OQ

    k = _k(1, 2, n, seed=n)
    _, rs, rz = OQ.quantize_asymmetric_per_channel(k, 4, pct)
    s, z = kivi_channel_params(k.cuda(), 4, pct)
    assert torch.equal(s.cpu(), rs) and torch.equal(z.cpu(), rz)


@pytest.mark.parametrize("pct", [100.0, 99.0])
def test_channel_range_many_units(pct):
    """More (b, head) units than one launch holds (2^18 x 16 work-groups of 1024 threads)."""
    from llm_kvcache_quantization_amd.cache import kivi_channel_params

    B, H, S = (1 << 15) + 3, 9, 2
    k = torch.randn(B, H, S, 128, generator=torch.Generator(device="cuda").manual_seed(3), device="cuda").half()
    s, z = kivi_channel_params(k, 8, pct)
    sel = [0, 7, 14563, 14564, 29127, B - 1]  # around the launches' boundaries at 2^17 and 2^18 units
    rs, rz = kivi_channel_params(k[sel].cpu(), 8, pct)
    assert torch.equal(s[sel].cpu(), rs) and torch.equal(z[sel].cpu(), rz)


@pytest.mark.parametrize("pct", [100.0, 99.9])
def test_channel_range_strides(pct):
    from llm_kvcache_quantization_amd.cache import kivi_channel_params

    k = _k(2, 3, 501, 1).cuda()
    ref = kivi_channel_params(k, 4, pct)
    t = k.transpose(1, 2).contiguous().transpose(1, 2)               # [B, S, H, D] storage
    odd = torch.zeros(2, 3, 501, 130, dtype=torch.float16, device="cuda")[..., 2:]
    odd.copy_(k)                                                     # rows aligned to 4 bytes only
    odd1 = torch.zeros(2, 3, 501, 131, dtype=torch.float16, device="cuda")[..., 1:129]
    odd1.copy_(k)                                                    # to 2 bytes: the torch path
    for x in (t, odd, odd1):
        for a, b in zip(kivi_channel_params(x, 4, pct), ref):
            assert torch.equal(a, b)


@pytest.mark.parametrize("pct", [100.0, 99.0])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), -float("inf")])
def test_channel_range_not_finite(bad, pct):
    """Without check_numerics: as torch's aminmax / sort and lerp, which keep a NaN range."""
    from llm_kvcache_quantization_amd.cache import kivi_channel_params

    k = _k(1, 2, 300, 2)
    k[0, 1, 7, 3] = k[0, 0, 250:, 9] = bad
    got = kivi_channel_params(k.cuda(), 8, pct)
    want = kivi_channel_params(k, 8, pct)
    for a, b in zip(got, want):
        assert torch.equal(a.cpu().nan_to_num(7e30, 8e30, -8e30), b.nan_to_num(7e30, 8e30, -8e30))


def test_prefill_rejects_nan_and_keeps_no_parameters():
    from llm_kvcache_quantization_amd import KIVIStyleKVCache

    cache = KIVIStyleKVCache(1, quant_bits=4)
    k = _k(1, 2, 40, 3).cuda()
    bad = k.clone()
    bad[0, 1, 20, 100] = float("nan")
    with pytest.raises(ValueError, match="quantize_asymmetric: input contains NaN or Inf"):
        cache.append(0, bad, k)
    assert cache.get_seq_len() == 0 and cache._k_scale[0] is None and not cache._k_scale_initialized[0]
    with pytest.raises(ValueError, match="V input contains NaN or Inf"):
        cache.append(0, k, bad)
    assert cache.get_seq_len() == 0
    cache.clear()
    cache.append(0, k, k)
    assert cache.get_seq_len() == 40


@pytest.mark.parametrize("side", ["k", "v"])
def test_rejected_prefill_then_another_prompt(side):
    """Without clear(): the next prompt is a prefill again, with parameters of its own, and checked."""
    from llm_kvcache_quantization_amd import KIVIStyleKVCache

    k = _k(1, 2, 40, 3).cuda()
    bad = k.clone()
    bad[0, 1, 20, 100] = float("inf")
    k2, v2 = _k(1, 2, 33, 4).cuda() * 0.25, _k(1, 2, 33, 5).cuda()
    cache, fresh = (KIVIStyleKVCache(1, quant_bits=4) for _ in range(2))
    for _ in range(2):  # the second rejection comes from the same check
        with pytest.raises(ValueError, match="NaN or Inf"):
            cache.append(0, *((bad, k) if side == "k" else (k, bad)))
        assert cache.get_seq_len() == 0
    cache.append(0, k2, v2)
    fresh.append(0, k2, v2)
    for a, b in zip(cache.get_kivi_tensors(0), fresh.get_kivi_tensors(0)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("shape", [(1, 1, 8193), (2, 32, 1024), (3, 5, 4370), (1, 2, 33000), (16, 9, 1100)], ids=str)
def test_split_range_equals_one_launch(shape):
    """Long prompts in two launches over splits of the tokens: the same bits as the single launch
    (no scratch), for dense, transposed and 4-byte aligned rows, with NaN and Inf."""
    import ctypes

    from llm_kvcache_quantization_amd import _capi as C

    L = C.lib()
    B, H, S = shape
    n = L.kvq_kivi_range_scratch_bytes(B, H, S, 0.0)
    assert n > 0 and L.kvq_kivi_range_scratch_bytes(B, H, S, 0.999) == 0
    k = _k(B, H, S, 3).cuda()
    k[0, 0, S - 1, 3], k[-1, -1, 0, 9], k[-1, 0, S // 2, 70] = float("nan"), float("inf"), -float("inf")
    t = k.transpose(1, 2).contiguous().transpose(1, 2)
    odd = torch.zeros(B, H, S, 130, dtype=torch.float16, device="cuda")[..., 2:]
    odd.copy_(k)
    for x in (k, t, odd):
        res = []
        for m in (n, 0):
            part = torch.full((n + 256,), 0xA5, dtype=torch.uint8, device="cuda")
            s, z = (torch.full((B, H, 128), -7.0, device="cuda") for _ in range(2))
            C.check(L.kvq_kivi_channel_range(x.data_ptr(), *x.stride()[:3], B, H, S, 8, 0.0, 0.0, s.data_ptr(),
                                             z.data_ptr(), part.data_ptr() if m else None, m,
                                             ctypes.c_void_p(C.stream_handle(x.device))))
            assert bool((part[n:] == 0xA5).all())
            res.append(torch.stack([s, z]).view(torch.int32))
        assert torch.equal(res[0], res[1])
