"""The one-token append's order statistics (csrc/append_row.h: group_top2, group_order_stats,
rescue_thr_rows) against torch.quantile, through the append kernel and the fused decode step.

A percentile whose ranks are the group's two largest (or, for a KIVI range, two smallest) values
takes one reduction; one further from the end walks or counts ranks.  Codes and scales must equal
the oracle's, whichever path a level takes and however the values tie."""
import math

import pytest
import torch

from oracle import quant as OQ

pytestmark = [pytest.mark.gpu, pytest.mark.filterwarnings("ignore:Static . scale overflow")]
DEV = "cuda:0"


def _k():
    import llm_kvcache_quantization_amd as K

    return K


def _rows(kind, B, H, S, g):
    x = torch.randn(B, H, S, 128, generator=g) * 2
    if kind == "ties":       # few magnitudes: the largest repeat within a group
        x = x.round().clamp(-2, 2)
    elif kind == "flat":     # one value per row
        x = x[..., :1].expand(B, H, S, 128).clone()
    elif kind == "edge":     # the extremes of fp16 beside zeros and subnormals
        x = x * 2.0 ** -18
        x[..., ::9] = 0.0
        x[..., 5], x[..., 64], x[..., 127] = 65504.0, -65504.0, 1.0
    return x.half()


def _both(mk, k, v, B, H, Hq, S0, fused=True):
    """The engine after S0 prompt tokens and one more: by append, and by the fused step."""
    out = []
    for step in (False, True)[:1 + fused]:
        c = mk()
        if S0:
            c.append(0, k[:, :, :S0].to(DEV), v[:, :, :S0].to(DEV))
        kn, vn = k[:, :, S0:].to(DEV), v[:, :, S0:].to(DEV)
        if step:
            c.append_decode_attn(0, torch.ones(B, Hq, 128, device=DEV).half(), kn, vn, 1 / math.sqrt(128))
        else:
            c.append(0, kn, vn)
        torch.cuda.synchronize()
        out.append(c)
    return out


@pytest.mark.parametrize("kind", ["normal", "ties", "flat", "edge"])
@pytest.mark.parametrize("gs", [8, 16, 32, 64, 128])
@pytest.mark.parametrize("bits,pct", [(8, 99.9), (4, 99.9), (8, 99.3), (4, 99.99999), (8, 97.0), (4, 60.0), (4, 0.5)])
def test_clipped_rows_equal_torch_quantile(bits, pct, gs, kind):
    K = _k()
    B, H, Hq = 2, 3, 6
    g = torch.Generator().manual_seed(int(pct * 10) + gs + bits)
    k, v = _rows(kind, B, H, 1, g), _rows(kind, B, H, 1, g)
    cls = K.INT8KVCache if bits == 8 else K.INT4KVCache
    ref = OQ.quantize_symmetric_int8 if bits == 8 else OQ.quantize_symmetric_int4
    mk = lambda: cls(1, device=DEV, group_size=gs, clip_percentile=pct)
    for c in _both(mk, k, v, B, H, Hq, 0, fused=gs > 8):  # (the decode kernel's groups start at 16)
        got = [t.cpu() for t in (c.get_int8_tensors(0) if bits == 8 else c.get_int4_tensors(0))]
        for x, codes, scale in ((k, got[0], got[2]), (v, got[1], got[3])):
            q, s = ref(x, pct, gs)
            assert torch.equal(scale.float().reshape(s.shape), s.float())
            assert torch.equal(codes, q if bits == 8 else OQ.pack_int4(q))


@pytest.mark.parametrize("kind", ["normal", "ties", "flat", "edge"])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("pct", [100.0, 99.9, 99.3, 96.0, 70.0])
def test_kivi_token_ranges_equal_torch_quantile(pct, bits, kind):
    K = _k()
    B, H, Hq, S0 = 2, 2, 4, 5
    g = torch.Generator().manual_seed(int(pct * 10) + bits)
    k = _rows("normal", B, H, S0 + 1, g)
    v = torch.cat([_rows("normal", B, H, S0, g), _rows(kind, B, H, 1, g)], dim=2)
    mk = lambda: K.KIVIStyleKVCache(1, device=DEV, quant_bits=bits, v_percentile=pct)
    for c in _both(mk, k, v, B, H, Hq, S0):
        got = [t.cpu() for t in c.get_kivi_tensors(0)]
        q, s, z = OQ.quantize_asymmetric_per_token(v[:, :, S0:], bits, pct)
        vc, vs, vz = got[1][:, :, S0:], got[4][..., S0:], got[5][..., S0:]
        assert torch.equal(vs.reshape(s.shape), s) and torch.equal(vz.reshape(z.shape), z)
        assert torch.equal(vc.view(torch.uint8), (q if bits == 8 else OQ.pack_int4(q)).view(torch.uint8))


@pytest.mark.parametrize("kind", ["normal", "ties", "flat", "edge"])
@pytest.mark.parametrize("gs", [16, 32, 64, 128])
@pytest.mark.parametrize("B,H,ratio", [(1, 1, 0.01), (1, 2, 0.01), (3, 5, 0.01), (8, 4, 0.01), (4, 8, 0.004),
                                       (2, 4, 0.1), (1, 1, 0.5)])
def test_rescue_threshold_equals_torch_quantile(B, H, ratio, gs, kind):
    K = _k()
    g = torch.Generator().manual_seed(B * 100 + H * 10 + gs)
    # K in dense rows, V in rows 130 values apart (not 16-byte aligned)
    k = _rows(kind, B, H, 1, g)
    v = _rows(kind, B, H, 1, g) * 0.5
    st = torch.rand(1, H, 128 // gs, generator=g) * 0.3 + 0.05
    mk = lambda: K.INT4KVCache(1, device=DEV, group_size=gs, static_k_scale=st, static_v_scale=st,
                               outlier_rescue_ratio=ratio)
    n = B * H * (128 // gs)
    fused = mk()._fused_step_ok(128, B, H)
    pad = torch.zeros(B, H, 1, 130, dtype=torch.float16, device=DEV)[..., :128]
    for i in range(2 if fused else 1):
        c = mk()
        kn, vn = k.to(DEV), pad.copy_(v.to(DEV))
        if i:
            c.append_decode_attn(0, torch.ones(B, 2 * H, 128, device=DEV).half(), kn, vn, 1 / math.sqrt(128))
        else:
            c.append(0, kn, vn)
        torch.cuda.synchronize()
        got = [t.cpu() for t in c.get_int4_tensors(0)]
        for x, codes, scale in ((k, got[0], got[2]), (v, got[1], got[3])):
            q, s = OQ.int4_cache_quantize(x, st[0], gs, outlier_rescue_ratio=ratio)
            assert torch.equal(scale.reshape(s.shape), s), (n, i)
            assert torch.equal(codes, OQ.pack_int4(q)), (n, i)
