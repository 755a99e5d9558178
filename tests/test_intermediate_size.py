"""The device memory of a problem: the intermediates U and V hold the
windows' traces and no more, whatever their number.

A window of 2 traces must not be stored as a tile of 16 (that made a line in
windows of 2 x 64 take 2.7 times its memory). The bound counts the model,
U and V (one complex value per trace and frequency of a time window, 10 %
for alignment), the traces, three records and the data, and 48 MB for
tables. The numbers come with a deblend of such a line, whose odd widths
are compared with the FP64 oracle in test_any_size.
"""
import numpy as np
import pytest
import torch

from agdeblend_amd import lib as L
from tests.test_any_size import test_any_window_length_matches_fp64_oracle as check
from tests.test_gpu_parity import _kw, _spec_geometry

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,windows", [((2048, 1024), (2, 64)), ((2049, 1024), (3, 64)),
                                           ((2040, 1024), (17, 64))])
def test_memory_counts_the_traces(shape, windows):
    torch.zeros(1, device="cuda")
    L.Problem(**_kw(_spec_geometry((4, 64), (2, 64), 3))).close()  # the library is loaded
    before = torch.cuda.mem_get_info()[0]
    pm = L.Problem(**_kw(_spec_geometry(shape, windows, 3)))
    try:
        used = before - torch.cuda.mem_get_info()[0]
        model = inter = traces = 0
        for w in range(pm.n_windows):
            i = pm.window(w)
            model += i["ntw"] * i["Ft"] * i["S"]
            inter += i["ntw"] * i["Ft"] * i["ntr"]
            traces += i["ntr"] * i["nconv"]
        data = int(np.prod(shape))
        bound = 8 * model + 1.1 * 2 * 8 * inter + 4 * traces + 3 * 4 * pm.record_len + 4 * data
        print(shape, windows, "used %.1f MB, bound %.1f + 48" % (used / 1e6, bound / 1e6), flush=True)
        assert used <= bound + 48e6
    finally:
        pm.close()


# tiles of every width: odd and even last ones alone (1, 7, 9) and after
# whole ones (17, 31, 35); odd planes (Ft odd and ntr odd) under and over the
# cache-line rule, several patches' worth of windows in a row
@pytest.mark.parametrize("shape,windows", [
    ((1, 90), (1, 16)), ((25, 60), (7, 16)), ((28, 90), (9, 50)), ((45, 200), (17, 200)),
    ((63, 160), (31, 64)), ((71, 120), (35, 50)), ((9, 25, 60), (3, 5, 16)),
    ((8, 160), (8, 64)), ((24, 640), (8, 256)), ((9, 78), (9, 26))])
def test_tile_widths_match_fp64_oracle(shape, windows):
    check(shape, windows)
