"""Which kernel an append takes and how it is split (kvq_append_plan, host only), on the CPU."""
import ctypes

import pytest

I8, I4, A4, K4, K8, F16 = 1, 2, 3, 4, 5, 6
ROW, TILE = 1, 2


def _side(fmt, B=2, H=4, S=4096, gs=32, tile=False, table=None, status=True, **over):
    from llm_kvcache_quantization_amd import _capi as C

    if not C.LIB_PATH.exists():
        pytest.skip("libkvq.so not built (run __graft_entry__.build())")
    p = C.AppendParams()
    p.format, p.batch, p.heads, p.seq_new, p.head_dim, p.group_size = fmt, B, H, S, 128, gs
    p.x = p.codes = 1 << 20  # addresses only: nothing reads them
    p.x_stride_b, p.x_stride_h, p.x_stride_s = H * S * 128, S * 128, 128
    cw = {I8: 128, K8: 128, F16: 256}.get(fmt, 64)
    p.codes_stride_b, p.codes_stride_h, p.codes_stride_t = H * 65536 * cw, 65536 * cw, cw
    p.capacity, p.codes_layout = 65536, C.KVQ_LAYOUT_TILE32 if tile else C.KVQ_LAYOUT_ROWS
    if status:
        p.status = 1 << 20
    if fmt == A4 if table is None else table:
        p.static_scale = p.static_zp = 1 << 20
        p.static_scale_dtype = C.KVQ_DTYPE_F16 if fmt == A4 else C.KVQ_DTYPE_F32
        p.static_stride_b, p.static_stride_h, p.static_stride_g = H * 128, 128, 1
    elif fmt in (K4, K8):
        p.scale_out = p.zp_out = 1 << 20
        p.scale_out_dtype = C.KVQ_DTYPE_F32
    for name, value in over.items():
        setattr(p, name, value)
    return p


def _plan(k, v):
    from llm_kvcache_quantization_amd import _capi as C

    out = (ctypes.c_int32 * 4)()
    C.check(C.lib().kvq_append_plan(None if k is None else ctypes.byref(k), None if v is None else ctypes.byref(v), out))
    return tuple(out)


def test_format_pairs():
    taken = {(I8, I8), (I4, I4), (K4, K4), (K4, K8), (K8, K4), (K8, K8), (I8, K4), (K4, I8)}
    for fk in (I8, I4, A4, K4, K8, F16):
        for fv in (I8, I4, A4, K4, K8, F16):
            assert _plan(_side(fk), _side(fv))[0] == (TILE if (fk, fv) in taken else ROW), (fk, fv)
        assert _plan(_side(fk), _side(A4, tile=True))[0] == (TILE if fk in (I8, A4) else ROW)
        for one in ((_side(fk), None), (None, _side(fk))):
            assert _plan(*one)[0] == (ROW if fk in (A4, F16) else TILE)
    assert _plan(None, _side(A4, tile=True))[0] == ROW
    assert _plan(None, None) == _plan(_side(I8, S=0), _side(I8, S=0)) == (0, 0, 0, 0)


@pytest.mark.parametrize("over", [dict(S=7), dict(x=(1 << 20) + 8), dict(x_stride_s=132), dict(x_stride_h=4096 * 128 + 4),
                                  dict(codes=(1 << 20) + 2), dict(codes_stride_t=130), dict(dyn_quantile=0.9)],
                         ids=lambda o: next(iter(o)))
def test_row_kernel_keeps(over):
    """Few tokens, rows or codes that are not aligned, percentiles further from the end."""
    assert _plan(_side(I8), _side(I8))[0] == TILE
    assert _plan(_side(I8, **over), _side(I8, **{"S": over.get("S", 4096)}))[0] == ROW
    if "S" not in over:
        assert _plan(_side(I8), _side(I8, **over))[0] == ROW
    assert _plan(_side(I8, dyn_quantile=0.999), _side(I8, dyn_quantile=0.97))[0] == TILE  # rank 30.07 of 31


def test_kivi_tables():
    assert _plan(_side(K4, table=True), _side(K4))[0] == TILE
    for over in (dict(static_stride_g=2), dict(static_scale=(1 << 20) + 4), dict(static_stride_h=130)):
        assert _plan(_side(K4, table=True, **over), _side(K4))[0] == ROW


@pytest.mark.parametrize("S,tok", [(2016, 8), (2048, 16), (8160, 16), (8192, 32)])
def test_tokens_a_wave(S, tok):
    """16 tokens from 512 32-token tiles a side, 32 from 2048."""
    assert _plan(_side(I8, S=S), _side(I8, S=S))[:2] == (TILE, tok)
    assert _plan(_side(A4, S=S), _side(A4, S=S, tile=True))[:2] == (TILE, 32)


def test_grid_covers_the_tiles():
    """Every wave at most 64 tiles, and the waves at most 8192 while that holds."""
    for B, H, S in ((1, 1, 8), (2, 4, 4096), (8, 4, 32768), (64, 8, 40960), (128, 16, 65536)):
        kernel, tok, waves, groups = _plan(_side(I8, B, H, S), _side(I8, B, H, S))
        tiles = B * H * -(-S // tok)
        assert kernel == TILE and groups * waves * 64 >= tiles
        assert groups <= max(8192 // waves, -(-tiles // (64 * waves)))


def test_waves_a_work_group():
    """8 where a side counts clipped values and the tiles lie in the measured range, else 4."""
    for S, wide in ((2048, False), (4096, True), (32704, True), (32768, False)):  # 1024, 2048, 8176, 8192 tiles
        for k, v, counts in ((_side(I8, S=S, table=True), _side(I8, S=S, table=True), True),
                             (_side(I8, S=S), _side(I8, S=S, table=True), True),
                             (_side(K4, S=S, table=True), _side(K4, S=S), True),
                             (_side(I8, S=S, table=True), None, True),
                             (_side(I8, S=S, table=True, status=False), _side(I8, S=S, table=True, status=False), False),
                             (_side(I8, S=S), _side(I8, S=S), False), (_side(I8, S=S), _side(K4, S=S), False)):
            assert _plan(k, v)[2] == (8 if wide and counts else 4), S
    # a threshold found by every work-group: 8 waves at any size it applies to
    assert _plan(*(_side(I4, 1, 2, 60, table=True, rescue_quantile=0.99) for _ in range(2)))[2] == 8
