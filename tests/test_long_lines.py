"""Spatial lines that one FFT does not hold, beside lengths that do not fold.

P = 125 (windows of 100) splits into 5 x 25 only; lines above 65 fold also
where another dim (18, 19, 22, 23, 27, 29 values) has no two factors up to
16. Forward and adjoint against the FP64 oracle to 2e-6, as in
test_any_size; and the time of a launch: held by one thread as a plain sum,
a line of 125 took ten times the time of one of 120.
"""
import numpy as np
import pytest

from agdeblend_amd import lib as L
from tests.test_any_size import test_any_window_length_matches_fp64_oracle as check
from tests.test_gpu_parity import _kw, _spec_geometry

pytestmark = pytest.mark.gpu

# alone, strided and contiguous, both beside a codelet, a line and a folded
# dim; ragged windows of 100 and 101; other long lines beside 18 and 23
SIZES = [((100, 40), (100, 10)), ((250, 40), (100, 10)), ((100, 14, 40), (100, 14, 10)),
         ((14, 100, 40), (14, 100, 10)), ((100, 15, 40), (100, 15, 10)),
         ((18, 100, 40), (18, 100, 10)), ((100, 24, 40), (100, 24, 10)),
         ((2, 3, 100, 40), (2, 3, 100, 10)), ((151, 40), (100, 10)),
         ((96, 14, 40), (96, 14, 10)), ((18, 80, 40), (18, 80, 10)), ((56, 23, 40), (56, 23, 10)),
         ((2, 60, 14, 40), (2, 60, 14, 10)), ((104, 14, 40), (104, 14, 10)),
         ((14, 180, 40), (14, 180, 10))]


@pytest.mark.parametrize("shape,windows", SIZES, ids=["x".join(map(str, s + w)) for s, w in SIZES])
def test_long_lines_match_fp64_oracle(shape, windows):
    check(shape, windows)


def _spatial_us(n, w):
    kw = _kw(_spec_geometry((n, 512), (w, 128), 3))
    pm = L.Problem(**kw)
    try:
        pm.set_data([np.random.default_rng(1).standard_normal((n, 512)).astype(np.float32)])
        pm.run(1.0, 3)
        best = 1e9
        for _ in range(3):
            L.timing(True)
            pm.iterate(4, 0.0)
            L.timing(False)
            best = min(best, sum(L.timing_get(k)[0] for k in ("fwd_spatial", "adj_spatial")) / 4)
        return best * 1e3
    finally:
        pm.close()


@pytest.mark.parametrize("w,near", [(100, 96)])
def test_no_slow_length_among_its_neighbours(w, near):
    a, b = _spatial_us(40 * w, w), _spatial_us(40 * near, near)
    print("windows of %d: %.0f us, of %d: %.0f us" % (w, a, near, b), flush=True)
    assert a < 3.0 * b
