"""The tile append's division (csrc/append_bulk.hip: recip, div_by) is the IEEE quotient: its codes
and scales equal the row kernel's because of that.  numpy's float32 division is the reference: reciprocals
by their bits, quotients by value (a zero's sign does not reach a code)."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _divide(x, s):
    from llm_kvcache_quantization_amd import _capi as C

    xd, sd = (torch.from_numpy(a).cuda() for a in (x, s))
    r, q = torch.empty_like(xd), torch.empty_like(xd)
    C.check(C.lib().kvq_append_division(xd.data_ptr(), sd.data_ptr(), r.data_ptr(), q.data_ptr(), x.size,
                                        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    return r.cpu().numpy(), q.cpu().numpy()


def _finite_halves():
    h = np.arange(65536, dtype=np.uint16).view(np.float16)
    return h[np.isfinite(h)].astype(np.float32)


@pytest.mark.parametrize("exponent", [-30, -17, -10, -1, 0, 1, 15, 29])
def test_reciprocal_of_every_significand(exponent):
    s = (np.arange(1 << 23, dtype=np.uint32) | np.uint32((127 + exponent) << 23)).view(np.float32)
    x = np.tile(_finite_halves(), (1 << 23) // 63488 + 1)[:1 << 23]
    r, q = _divide(x, s)
    assert np.array_equal(r.view(np.uint32), (np.float32(1) / s).view(np.uint32))
    assert np.array_equal(q, x / s)


@pytest.mark.parametrize("s", [7.0, 15.0, 127.0, 255.0, 1e-5, 1e-5 / 7, 2.0 ** -14, 2.0 ** -30, 2.0 ** 30, 65504.0])
def test_quotients_of_every_half(s):
    """The scales' own divisions (by 7, 15, 127, 255) and the range's ends."""
    x = _finite_halves()
    s = np.full_like(x, s)
    assert np.array_equal(_divide(x, s)[1], x / s)


def test_quotients_of_differences():
    """x - z of the asymmetric formats over random scales, and quotients next to a rounding boundary
    of the codes (n + 1/2) s."""
    g = np.random.default_rng(5)
    n = 1 << 24
    h = _finite_halves()
    x = g.choice(h, n) - (g.standard_normal(n) * 2.0 ** g.integers(-12, 12, n)).astype(np.float32)
    s = (g.uniform(1, 2, n) * 2.0 ** g.integers(-30, 30, n)).astype(np.float32)
    near = ((g.integers(-128, 128, n) + np.float32(0.5)) * s).astype(np.float32)
    near = (near.view(np.int32) + g.integers(-2, 3, n).astype(np.int32)).view(np.float32)
    for v in (x, near):
        assert np.array_equal(_divide(v, s)[1], v / s)
