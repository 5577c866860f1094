"""The prompt-sized append (csrc/append_bulk.hip) against the row kernel, bit for bit.

Both kernels append the same values: once from dense rows (which the tile kernel takes) and once
from rows 130 values apart (not 16-byte aligned, so the row kernel quantizes them); the library's
plan of each call says which kernel ran.  Codes, scales, zero-points, outlier values and status words
must be equal, also where the tile kernel hands tiles back: NaN / Inf rows, zero or infinite scales.
The row kernel itself is pinned to the oracle by the append tests of test_gpu_parity.py and
test_gpu_kivi_family.py: their appends of fewer than 8 tokens, and test_gpu_parity.py's unaligned
rows."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

D = 128


def _lib():
    from llm_kvcache_quantization_amd import _capi as C

    return C, C.lib()


def _side(C, fmt, gs, B, H, S, wpos, cap, x, policy, g, tile=False):
    """(AppendParams, tensors written) of one side."""
    p = C.AppendParams()
    p.format, p.x = fmt, x.data_ptr()
    p.x_stride_b, p.x_stride_h, p.x_stride_s = x.stride()[:3]
    p.batch, p.heads, p.seq_new, p.head_dim, p.group_size = B, H, S, D, gs
    i4 = fmt in (C.KVQ_FMT_INT4_SYM, C.KVQ_FMT_INT4_ASYM, C.KVQ_FMT_INT4_KIVI)
    cw = 64 if i4 else 128
    codes = torch.full((B, H, cap, cw), 0x5A, dtype=torch.uint8, device="cuda")
    p.codes, p.codes_stride_b, p.codes_stride_h, p.codes_stride_t = codes.data_ptr(), H * cap * cw, cap * cw, cw
    p.write_pos, p.capacity = wpos, cap
    p.codes_layout = C.KVQ_LAYOUT_TILE32 if tile else C.KVQ_LAYOUT_ROWS
    status = torch.zeros(2, dtype=torch.int32, device="cuda")
    p.status = status.data_ptr()
    out, keep = [codes, status], [x]

    def rnd(*shape):
        return torch.rand(*shape, generator=g, device="cuda")

    if fmt in (C.KVQ_FMT_INT4_KIVI, C.KVQ_FMT_INT8_KIVI):
        if policy.get("table"):
            s, z = 0.02 + 0.3 * rnd(B, H, D), rnd(B, H, D) - 0.5
            if policy.get("odd"):
                s[0, 0, 5], z[-1, -1, 9] = 0.0, float("inf")
            p.static_scale, p.static_zp, p.static_scale_dtype = s.data_ptr(), z.data_ptr(), C.KVQ_DTYPE_F32
            p.static_stride_b, p.static_stride_h, p.static_stride_g = s.stride()
            keep += [s, z]
        else:
            s, z = (torch.full((B, H, cap), 7.0, device="cuda") for _ in range(2))
            p.scale_out, p.zp_out, p.scale_out_dtype = s.data_ptr(), z.data_ptr(), C.KVQ_DTYPE_F32
            p.so_stride_b, p.so_stride_h, p.so_stride_t = s.stride()
            if "pct" in policy:
                p.dyn_quantile, p.dyn_quantile_lo = policy["pct"] / 100.0, (100.0 - policy["pct"]) / 100.0
            out += [s, z]
        return p, out, keep
    G = D // gs
    if policy.get("table"):
        f32 = fmt == C.KVQ_FMT_INT4_SYM or policy.get("f32", False)
        s = ((0.004 if fmt == C.KVQ_FMT_INT8_SYM else 0.15) * (0.5 + rnd(H, G))).to(
            torch.float32 if f32 else torch.float16)
        if policy.get("odd"):
            s[0, 0], s[-1, -1] = 0.0, float("inf")
        p.static_scale, p.static_scale_dtype = s.data_ptr(), C.KVQ_DTYPE_F32 if f32 else C.KVQ_DTYPE_F16
        p.static_stride_h, p.static_stride_g = s.stride()
        keep.append(s)
        if fmt == C.KVQ_FMT_INT4_ASYM:
            z = (rnd(H, G) - 0.5).half()
            p.static_zp = z.data_ptr()
            keep.append(z)
    p.adaptive, p.adaptive_margin = int("margin" in policy), policy.get("margin", 0.0)
    p.rescue_quantile = policy.get("rq", 0.0)
    p.mixed_rescue, p.rescue_all = int(policy.get("mixed", 0)), int(policy.get("all", 0))
    if "pct" in policy:
        p.dyn_quantile = policy["pct"] / 100.0
    if fmt != C.KVQ_FMT_INT4_ASYM and (not policy.get("table") or "margin" in policy or policy.get("mixed")
                                       or policy.get("all") or "rq" in policy):
        dt = torch.float16 if fmt == C.KVQ_FMT_INT8_SYM else torch.float32
        so = torch.full((B, H, cap, G), 7.0, dtype=dt, device="cuda")
        p.scale_out = so.data_ptr()
        p.scale_out_dtype = C.KVQ_DTYPE_F16 if dt == torch.float16 else C.KVQ_DTYPE_F32
        p.so_stride_b, p.so_stride_h, p.so_stride_t, p.so_stride_g = so.stride()
        out.append(so)
    nbytes = C.lib().kvq_append_scratch_bytes(ctypes.byref(p))
    if nbytes:
        sc = torch.full((nbytes,), 0xA5, dtype=torch.uint8, device="cuda")
        p.scratch, p.scratch_bytes = sc.data_ptr(), nbytes
        keep.append(sc)
    if policy.get("outliers"):
        oi = torch.stack([torch.randperm(D, generator=g, device="cuda")[:4] for _ in range(H)]).int()
        oo = torch.full((B, H, cap, 4), 7.0, dtype=torch.float16, device="cuda")
        p.n_outlier, p.outlier_idx, p.outlier_out = 4, oi.data_ptr(), oo.data_ptr()
        p.oo_stride_b, p.oo_stride_h, p.oo_stride_t = oo.stride()[:3]
        keep.append(oi)
        out.append(oo)
    return p, out, keep


I8, I4, A4, K4, K8 = 1, 2, 3, 4, 5
# (K side, V side): (format, group, policy, TILE32)
PAIRS = {
    "int8_p999": ((I8, 128, dict(pct=99.9)),) * 2,
    "int8_max_g32": ((I8, 32, {}),) * 2,
    "int8_table_g16": ((I8, 16, dict(table=1)), (I8, 16, dict(table=1, f32=True))),
    "int8_table_odd": ((I8, 32, dict(table=1, odd=1)),) * 2,
    "int8_adaptive": ((I8, 64, dict(table=1, margin=0.9)), (I8, 64, dict(table=1, f32=True, margin=1.2))),
    "int4_p999_g16": ((I4, 16, dict(pct=99.9)), (I4, 16, dict(pct=99.9))),
    "int4_p97": ((I4, 32, dict(pct=97.0)),) * 2,  # rank 30.07 of 31: within the two largest
    "int4_max_g8": ((I4, 8, {}),) * 2,
    "int4_table_mixed": ((I4, 32, dict(table=1, mixed=1)), (I4, 32, dict(table=1))),
    "int4_table_all": ((I4, 64, dict(table=1, all=1)), (I4, 64, dict(table=1, margin=0.8))),
    "int4_rescue_g16": ((I4, 16, dict(table=1, rq=0.99)), (I4, 16, dict(table=1, rq=0.4))),
    "int4_rescue_g8": ((I4, 8, dict(table=1, rq=0.999, margin=0.7)), (I4, 8, dict(table=1))),
    "int4_rescue_nan": ((I4, 32, dict(table=1, rq=0.5, odd=1)),) * 2,
    "asym_tile": ((A4, 32, dict(table=1, outliers=1)), (A4, 32, dict(table=1), True)),
    "asym_odd": ((A4, 32, dict(table=1, odd=1)), (A4, 32, dict(table=1, odd=1), True)),
    "k8_asym": ((I8, 32, dict(table=1)), (A4, 32, dict(table=1), True)),
    "kivi4": ((K4, 32, dict(table=1)), (K4, 32, {})),
    "kivi4_p999": ((K4, 32, dict(table=1)), (K4, 32, dict(pct=99.9))),
    "kivi8": ((K8, 32, dict(table=1)), (K8, 32, {})),
    "kivi8_odd": ((K8, 32, dict(table=1, odd=1)), (K8, 32, dict(pct=99.3))),
    "mixed": ((I8, 128, dict(pct=99.9)), (K4, 32, dict(pct=99.9))),
    "kivi48": ((K4, 32, dict(table=1)), (K8, 32, {})),
    "kivi84": ((K8, 32, dict(table=1)), (K4, 32, {})),
    "mixed48": ((K4, 32, dict(pct=99.9)), (I8, 32, dict(pct=99.9))),
}

# (batch, heads, tokens, write position): fewest tokens, a tile's edges, starts inside a tile, a
# size whose rescue threshold every work-group finds (1025 to 4096 scales), then 1032 and 2064
# 32-token tiles: 16 and 32 tokens a wave in every row format
SIZES = [(1, 2, 8, 0), (2, 3, 31, 5), (1, 1, 33, 31), (3, 2, 64, 32), (2, 4, 4099, 1), (2, 8, 4099, 1)]


def _plan(pk, pv):
    """(0 nothing / 1 row kernel / 2 tile kernel, tokens a wave, waves a work-group, work-groups)"""
    C, L = _lib()
    out = (ctypes.c_int32 * 4)()
    C.check(L.kvq_append_plan(*(None if p is None else ctypes.byref(p) for p in (pk, pv)), out))
    return tuple(out)


def _append(name, x, wpos, cap, sides=(0, 1)):
    """The tensors an append of x[side] (a list of 2) writes, and its plan; sides: those not NULL."""
    C, L = _lib()
    ps, wrote, keep = [None, None], [], []
    for side in sides:
        fmt, gs, policy = PAIRS[name][side][:3]
        B, H, S = x[side].shape[:3]
        g = torch.Generator(device="cuda").manual_seed(99 + side)
        p, o, kp = _side(C, fmt, gs, B, H, S, wpos, cap, x[side], policy, g, tile=len(PAIRS[name][side]) > 3)
        ps[side] = p
        wrote += o
        keep += kp
    plan = _plan(*ps)
    C.check(L.kvq_quant_append(*(None if p is None else ctypes.byref(p) for p in ps),
                               ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    return wrote, plan


def _apart(x, w):
    """x in rows w values apart."""
    out = torch.zeros(*x.shape[:3], w, dtype=torch.float16, device="cuda")[..., :D]
    return out.copy_(x)


def _same(a, b, what):
    for i, j in zip(a, b, strict=True):  # bits: NaN scales of NaN rows included
        assert torch.equal(i.contiguous().view(torch.uint8), j.contiguous().view(torch.uint8)), (what, i.dtype)


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("name", sorted(PAIRS))
def test_bulk_append_equals_row_kernel(name, size):
    C, L = _lib()
    B, H, S, wpos = size
    cap = -(-(wpos + S + 3) // 32) * 32
    x = []
    for side in range(2):
        g = torch.Generator(device="cuda").manual_seed(7 * S + side)
        v = torch.randn(B, H, S, D, generator=g, device="cuda").half()
        v[:, :, :, 3] *= 20
        v[0, 0, 0] = 0.0                     # an all-zero row
        v[0, 0, 1, :64] = v[0, 0, 1, 0]      # ties
        v[0, 0, 2, 7] = -0.0
        v[-1, -1, 3, 11] = 65504.0
        v[-1, -1, 4] *= 2.0 ** -20           # subnormals
        if "odd" in name:                    # the tables' odd groups meet ordinary rows too
            v[0, -1, 5, 100] = float("nan")
            v[-1, 0, 6, 2] = float("inf")
            v[-1, 0, 7, 90] = -float("inf")
        x.append(v)
    outs = []
    for route in range(2):
        ps, wrote, keep = [], [], []
        for side, spec in enumerate(PAIRS[name]):
            fmt, gs, policy = spec[:3]
            if route == 0:
                xs = x[side]
            else:
                xs = torch.zeros(B, H, S, 130, dtype=torch.float16, device="cuda")[..., :D]
                xs.copy_(x[side])
            g = torch.Generator(device="cuda").manual_seed(99 + side)
            p, o, kp = _side(C, fmt, gs, B, H, S, wpos, cap, xs, policy, g, tile=len(spec) > 3)
            ps.append(p)
            wrote += o
            keep += kp
        kernel, tok = _plan(*ps)[:2]
        if route == 0:
            t32 = B * H * -(-S // 32)
            tiled = any(len(spec) > 3 for spec in PAIRS[name])
            assert kernel == 2 and tok == (32 if tiled or t32 >= 2048 else 16 if t32 >= 512 else 8)
        else:
            assert kernel == 1
        C.check(L.kvq_quant_append(ctypes.byref(ps[0]), ctypes.byref(ps[1]),
                                   ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
        torch.cuda.synchronize()
        outs.append(wrote)
    for a, b in zip(*outs):
        # bits: NaN scales of NaN rows included
        assert torch.equal(a.contiguous().view(torch.uint8), b.contiguous().view(torch.uint8)), (name, a.dtype)


@pytest.mark.parametrize("name", ["int8_table_odd", "int4_rescue_nan", "asym_odd", "kivi8_odd"])
def test_tiles_after_a_waves_first(name):
    """More tiles than waves: those a wave takes second and third, some handed back."""
    B, H, S, wpos = 2, 8, 33000, 1
    cap = 33024
    x = []
    for side in range(2):
        v = torch.randn(B, H, S, D, generator=torch.Generator(device="cuda").manual_seed(side), device="cuda").half()
        v[-1, -1, -5, 100] = float("nan")  # the last tiles are some waves' third
        v[-1, -1, -70, 3] = float("inf")
        v[-1, 2, 40, 64] = -float("inf")   # a second one
        v[0, 1, 3, 9] = float("nan")       # a first one
        x.append(v)
    tile, plan = _append(name, x, wpos, cap)
    assert plan[:2] == (2, 32) and 2 * plan[2] * plan[3] < B * H * 1032
    row, plan = _append(name, [_apart(v, 130) for v in x], wpos, cap)
    assert plan[0] == 1
    _same(tile, row, name)


@pytest.mark.parametrize("side", [0, 1])
@pytest.mark.parametrize("name", ["int8_p999", "int8_table_g16", "int4_rescue_g16", "int4_p999_g16", "kivi4_p999",
                                  "kivi8", "kivi48", "mixed", "k8_asym", "asym_tile"])
@pytest.mark.parametrize("size", [(2, 3, 31, 5), (2, 4, 4099, 1)], ids=str)
def test_one_side(size, name, side):
    """K or V alone (a cache whose other side is 16-bit): the same bits as beside the other side."""
    B, H, S, wpos = size
    cap = -(-(wpos + S) // 32) * 32
    x = [torch.randn(B, H, S, D, generator=torch.Generator(device="cuda").manual_seed(s), device="cuda").half()
         for s in (5, 6)]
    both, _ = _append(name, x, wpos, cap)
    one, plan = _append(name, x, wpos, cap, sides=(side,))
    fmt = PAIRS[name][side][0]
    assert plan[0] == (1 if fmt == A4 else 2)
    _same(one, both[:len(one)] if side == 0 else both[-len(one):], name)


@pytest.mark.parametrize("name", ["int8_p999", "int4_rescue_g16", "asym_tile", "kivi8", "mixed"])
@pytest.mark.parametrize("size", [(2, 3, 131, 5), (2, 4, 4099, 1)], ids=str)
def test_strides(size, name):
    """Rows the tile kernel takes in other layouts: tokens outside the heads, padded rows."""
    B, H, S, wpos = size
    cap = -(-(wpos + S) // 32) * 32
    x = [torch.randn(B, H, S, D, generator=torch.Generator(device="cuda").manual_seed(s), device="cuda").half()
         for s in (5, 6)]
    ref, _ = _append(name, [_apart(v, 130) for v in x], wpos, cap)
    for layout in (lambda v: v.transpose(1, 2).contiguous().transpose(1, 2), lambda v: _apart(v, 136),
                   lambda v: v.permute(2, 0, 1, 3).contiguous().permute(1, 2, 0, 3)):
        got, plan = _append(name, [layout(v) for v in x], wpos, cap)
        assert plan[0] == 2
        _same(got, ref, name)
