"""The format pairs kvq_dequant takes (csrc/dequant.hip), on the CPU: the entry checks them on the
host, and over no tokens it launches nothing."""
import ctypes

import pytest

I8, I4, A4, K4, K8, F16 = 1, 2, 3, 4, 5, 6
PAIRS = {(I8, I8), (I4, I4), (K4, K4), (K4, K8), (K8, K4), (K8, K8), (I8, K4), (K4, I8)}


def _call(fk, fv, tokens=0):
    from llm_kvcache_quantization_amd import _capi as C

    if not C.LIB_PATH.exists():
        pytest.skip("libkvq.so not built (run __graft_entry__.build())")
    args = []
    for f in (fk, fv):
        if f is None:
            args += [None, 0, 0, None]
            continue
        v = C.KvView()
        v.codes = v.scale = v.zero_point = 1 << 20  # addresses only: nothing reads them
        v.stride_b = v.stride_h = v.stride_t = 128
        v.scale_dtype = C.KVQ_DTYPE_F32
        args += [ctypes.byref(v), f, 32, 1 << 20]
    return C, C.lib().kvq_dequant(*args, 1, 1, tokens, None)


@pytest.mark.parametrize("fv", [None, I8, I4, K4, K8])
@pytest.mark.parametrize("fk", [None, I8, I4, K4, K8])
def test_pairs(fk, fv):
    C, rc = _call(fk, fv)
    pair = (fk or fv, fv or fk)
    assert rc == (C.KVQ_OK if pair in PAIRS or pair == (None, None) else C.KVQ_ERR_UNSUPPORTED)


def test_no_dequantiser():
    for f in (A4, F16):
        C, rc = _call(f, f)
        assert rc == C.KVQ_ERR_UNSUPPORTED
