"""What the interface says of a problem's time classes (CPU): the variant in
use, also where it cannot be set, and which classes have a choice.

Whole tiles of 16 traces and W_t of 64 to 512 have a specialised time kernel
beside any spatial size; only beside a specialised spatial size are its
factors, variant and runs the caller's. Generic: other W_t, partial tiles.
"""
import numpy as np
import pytest

from agdeblend_amd import lib as L
from tests.test_gpu_parity import _kw, _spec_geometry


def _problem(shape, windows):
    return L.Problem(host_only=True, **_kw(_spec_geometry(shape, windows, 3)))


@pytest.mark.parametrize("shape,windows,factors,variant", [
    ((64, 2048), (32, 256), (10, 16), 0), ((64, 2048), (32, 512), (20, 16), 1),  # to set
    ((96, 2048), (48, 256), (0, 0), 0), ((96, 2048), (48, 512), (0, 0), 1),      # fixed
    ((64, 2000), (32, 200), (0, 0), 0), ((68, 2048), (34, 512), (0, 0), 0)])     # generic
def test_factors_and_variant_in_use(shape, windows, factors, variant, monkeypatch):
    monkeypatch.setenv("AGD_TIME_TW", "2")
    pm = _problem(shape, windows)
    try:
        assert pm.time_factors() == [factors]
        assert pm.time_variants() == [variant]
        ntw = pm.window(0)["ntw"]
        runs = {b - a for _, _, a, b in pm.time_blocks().tolist()}
        if factors == (0, 0):
            assert runs == {ntw}
            with pytest.raises(ValueError):
                pm.set_time_variant(0, 0)
            with pytest.raises(ValueError):
                pm.set_time_factors(0, 10, 16)
        else:
            assert max(runs) == 2
            pm.set_time_variant(0, 1 - variant)
            assert pm.time_variants() == [1 - variant]
    finally:
        pm.close()


def test_one_time_length_beside_both_kinds_of_spatial_size():
    """Two volumes of one W_t, windows of 32 (specialised) and of 48 traces:
    two classes, one of them to set."""
    a, b = _spec_geometry((64, 2048), (32, 512), 3), _spec_geometry((96, 2048), (48, 512), 4)
    g = {k: a[k] + b[k] for k in a}
    g["volumes"] = [0, 1]
    g["channels"][1] = (g["channels"][1] + 1).astype(np.intc)
    pm = L.Problem(host_only=True, **_kw(g))
    try:
        assert sorted(pm.time_factors()) == [(0, 0), (20, 16)]
        assert pm.time_variants() == [1, 1]
    finally:
        pm.close()
