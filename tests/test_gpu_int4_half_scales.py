"""INT4_SYM K and V with per-token fp16 scales (decode_attn_int4's arguments) on the tiled kernel:
against the fp64 attention over the reference's dequantised values fp16(c * s), and against the row
kernel (the same tensors with code rows that are not dense), for every operand variant: groups of
16 / 32 / 64 / 128, staged V (dense 16-byte aligned scale rows) and gathered V (odd capacities,
padded scale rows), contexts around tile edges, ragged batches, one head and 10 heads per KV head.
Calls beyond the tiled kernel's limits keep the row kernel."""
import ctypes
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(B, Hkv, n_rep, S, gs, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    kc, vc = (torch.randint(-7, 8, (B, Hkv, S, 128), generator=g, device="cuda") for _ in range(2))
    ks, vs = (0.1 + 0.4 * torch.rand(B, Hkv, S, 128 // gs, generator=g, device="cuda") for _ in range(2))
    q = torch.randn(B, Hkv * n_rep, 128, generator=g, device="cuda").half()
    return q, kc, vc, ks.half(), vs.half()


def _pack(c):
    u = (c + 8).to(torch.uint8)
    return ((u[..., 0::2] << 4) | u[..., 1::2]).view(torch.int8)


def _ref(q, kc, vc, ks, vs, lens):
    B, Hkv, S, G = ks.shape
    out = []
    for b in range(B):
        n = lens[b]
        if n == 0:
            out.append(torch.zeros(q.shape[1], 128, dtype=torch.float64, device="cuda"))
            continue
        k, v = ((c[b, :, :n].half().view(Hkv, n, G, -1) * s[b, :, :n, :, None]).view(Hkv, n, 128).double()
                for c, s in ((kc, ks), (vc, vs)))
        p = torch.softmax(torch.matmul(q[b].double().view(Hkv, -1, 128), k.transpose(1, 2).contiguous())
                          / math.sqrt(128), -1)
        out.append(torch.matmul(p, v).reshape(-1, 128))
    return torch.stack(out)


@pytest.mark.parametrize("gs", [16, 32, 64, 128])
@pytest.mark.parametrize("shape", [(1, 2, 6, 1), (1, 1, 1, 31), (2, 4, 7, 33), (3, 2, 10, 257), (4, 4, 7, 1999),
                                   (2, 8, 5, 4096)], ids=str)
def test_half_scales(shape, gs):
    from llm_kvcache_quantization_amd import decode_attn_int4

    B, Hkv, n_rep, S = shape
    q, kc, vc, ks, vs = _inputs(B, Hkv, n_rep, S, gs, S + gs)
    kp, vp = _pack(kc), _pack(vc)
    wide = [torch.zeros(B, Hkv, S, 96, dtype=torch.int8, device="cuda")[..., :64] for _ in range(2)]
    for w, c in zip(wide, (kp, vp)):  # token rows 96 bytes apart: the row kernel
        w.copy_(c)
    pad = [torch.zeros(B, Hkv, S, 128 // gs + 2, dtype=torch.float16, device="cuda")[..., :128 // gs]
           for _ in range(2)]
    for w, c in zip(pad, (ks, vs)):  # padded scale rows: V gathered, not staged
        w.copy_(c)
    for lens in ([S] * B, [max(1, S * (b + 1) // B - b) for b in range(B)], [0] + [S] * (B - 1)):
        ctx = torch.tensor(lens, dtype=torch.int32, device="cuda")
        if max(lens) == 0:
            continue
        out = decode_attn_int4(q, kp, vp, ks, vs, ctx)
        ref = _ref(q, kc, vc, ks, vs, lens)
        # |v| <= 3.5: an fp16 output within an ulp (2^-10 of [1, 2), 2^-9 of [2, 4)) of the exact
        # value, the bound the other formats are held to
        assert (out.double() - ref).abs().max() <= 2e-3
        assert torch.equal(out, decode_attn_int4(q, kp, vp, *pad, ctx))
        row = decode_attn_int4(q, *wide, ks, vs, ctx)
        assert (row.double() - out.double()).abs().max() <= 2e-3


def _params(B, Hq, Hkv, cap, gs=32, sst=4):
    """Decode parameters over made-up addresses: planning only, nothing is launched."""
    from llm_kvcache_quantization_amd import _capi as C

    p = C.DecodeParams()
    p.k_format = p.v_format = C.KVQ_FMT_INT4_SYM
    for v in (p.k, p.v):
        v.codes, v.scale, v.scale_dtype = 1 << 20, 1 << 20, C.KVQ_DTYPE_F16
        v.stride_b, v.stride_h, v.stride_t = Hkv * cap * 64, cap * 64, 64
        v.scale_stride_b, v.scale_stride_h, v.scale_stride_t, v.scale_stride_g = Hkv * cap * sst, cap * sst, sst, 1
    p.context_lens = 1 << 20
    p.batch, p.q_heads, p.kv_heads, p.head_dim, p.group_size, p.capacity = B, Hq, Hkv, 128, gs, cap
    return C, p


def test_half_scales_limits():
    """Planning: a call whose row-kernel workspace fits the fixed scratch still fits it, and the
    planning calls take shapes that decode calls reject."""
    for B, Hq, Hkv, cap in ((1, 12, 2, 65536), (16, 40, 8, 65536), (64, 40, 8, 65536), (64, 28, 4, 4096),
                            (60, 16, 1, 100000), (2, 12, 2, 1 << 26)):
        C, p = _params(B, Hq, Hkv, cap)
        need = C.lib().kvq_decode_workspace_bytes(ctypes.byref(p))
        p.k.stride_t = p.v.stride_t = 96  # the row kernel
        row = C.lib().kvq_decode_workspace_bytes(ctypes.byref(p))
        assert need <= C.KVQ_NOALLOC_SCRATCH_BYTES or row > C.KVQ_NOALLOC_SCRATCH_BYTES, (B, Hq, Hkv, cap)
    for bad in ((0, 12, 2, 64), (1, 0, 2, 64), (1, 12, 0, 64)):
        C, p = _params(*bad)
        assert C.lib().kvq_decode_workspace_bytes(ctypes.byref(p)) >= 0
    # the fused append stays with the engines' fp32 scales
    C, p = _params(1, 12, 2, 64)
    a = C.AppendParams()
    assert C.lib().kvq_append_decode_attn(ctypes.byref(p), ctypes.byref(a), ctypes.byref(a), None) == \
        C.KVQ_ERR_UNSUPPORTED
