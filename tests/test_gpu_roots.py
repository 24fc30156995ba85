"""sqrt_inv and div_by (one hardware reciprocal root, one coupled iteration,
one residual correction) against the correctly rounded root and quotient, over
the ranges the kernels call them with."""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "device", "_bin", "libroot_helpers.so")

# (smallest, largest) argument: drifts 1 + x'^2 + y'^2 of slopes below 1e9, -2 ln u
# of the normal pairs, squared radii of the field map off its axis
RANGES = {"drift": (1.0, 1e18), "normal": (2.0 ** -32, 46.0), "field": (2.0 ** -900, 1e4)}


def helpers(s, a):
    f = C.CDLL(LIB).root_helpers
    f.argtypes = [C.c_int64] + [C.c_void_p] * 6
    d = [torch.from_numpy(v).cuda() for v in (s, a)]
    out = [torch.empty_like(d[0]) for _ in range(3)]
    st = torch.cuda.current_stream().cuda_stream
    assert f(len(s), *[C.c_void_p(t.data_ptr()) for t in d + out], C.c_void_p(st)) == 0
    torch.cuda.synchronize()
    return [t.cpu().numpy() for t in out]


@pytest.mark.parametrize("name", RANGES)
@pytest.mark.parametrize("spread", ["log", "near_1", "squares"])
def test_roots_and_quotients_equal_the_rounded_ones(name, spread):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    n, (lo, hi) = 2_000_000, RANGES[name]
    rng = np.random.default_rng(7)
    s = np.exp(rng.uniform(np.log(lo), np.log(hi), n))
    if spread == "near_1":  # drifts of ordinary slopes
        s = 1.0 + rng.uniform(0.0, 0.2, n) ** 2 + rng.uniform(0.0, 0.2, n) ** 2
    elif spread == "squares":  # roots of 26 bits and their neighbours: the exact cases
        k = np.ldexp(np.floor(rng.uniform(2.0 ** 25, 2.0 ** 26, n)), -26)
        s = k * k * 4.0 ** np.floor(np.log2(s) / 2)
        s = np.where(rng.random(n) < 0.5, s, np.nextafter(s, rng.choice([0.0, np.inf], n)))
    s = np.clip(s, lo, np.nextafter(hi, 0.0))
    a = rng.standard_normal(n)
    root, inv, quot = helpers(s, a)
    # both results are within 2^-42 ulp of the exact value before the last
    # rounding, so 2e6 of them differ from the rounded one with probability
    # 1e-6; the samples are fixed
    exact = np.sqrt(s)
    np.testing.assert_array_equal(root, exact)
    np.testing.assert_array_equal(quot, a / exact)
    assert np.max(np.abs(inv * exact - 1.0)) < 2.0 ** -46  # 2^-47, and the product's rounding
