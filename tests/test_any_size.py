"""The run-time sized transforms (agd_general.hip): windows of any length.

A line of P padded values is held by one thread in registers: P up to 33,
49, 65, 97 and 129 by kernel instance, or folded into two short transforms (the windows below sit on both sides
of each edge, at lengths with a register codelet and at primes), longer ones
go to the LDS-resident kernels; the time transform takes Pt in two or three
register FFTs of up to 16 values, else in lines M1 M2, with M1 = 1 for a
prime Pt, and hands Pt = 313 to the LDS-resident kernels. Window traces that do not fill their last tile of 16, batches of
lines shared by several waves, one to four space dims, patches that a window
covers whole (odd lengths) or with windows of two lengths.

Forward and adjoint against the FP64 oracle to 2e-6, the suite's bound for
every operator (FP32 transforms: about 1e-7 times the square root of the
summed terms), and the adjoint test in FP64 to 1e-6.
"""
import zlib

import numpy as np
import pytest

from agdeblend_amd import lib as L
from tests.test_gpu_parity import (_kw, _mute_vec, _random_model, _spec_geometry,
                                   _to_oracle_layout, _to_product_layout)

pytestmark = pytest.mark.gpu

# (shape, windows): time last
SIZES = [
    ((2, 40), (2, 8)), ((3, 64), (3, 10)), ((5, 60), (5, 6)),
    ((13, 200), (13, 64)), ((14, 150), (14, 50)), ((26, 300), (26, 100)), ((27, 130), (27, 26)),
    ((39, 200), (39, 56)), ((40, 256), (40, 86)), ((51, 256), (51, 64)), ((53, 128), (52, 40)),
    ((77, 96), (77, 24)), ((79, 96), (78, 32)), ((103, 64), (103, 16)), ((104, 64), (104, 16)),
    ((33, 700), (32, 250)), ((100, 450), (32, 188)), ((20, 640), (18, 256)), ((61, 300), (24, 106)),
    ((9, 41, 120), (4, 16, 30)), ((17, 34, 160), (16, 33, 64)), ((23, 50, 128), (10, 24, 128)),
    ((45, 47, 66), (32, 34, 26)), ((3, 53, 64), (2, 53, 20)),
    ((5, 9, 14, 48), (4, 8, 10, 16)), ((4, 5, 6, 7, 40), (4, 4, 6, 6, 10)),
]


@pytest.mark.parametrize("shape,windows", SIZES, ids=["x".join(map(str, s + w)) for s, w in SIZES])
def test_any_window_length_matches_fp64_oracle(shape, windows):
    from oracle import oracle as O
    geo = _spec_geometry(shape, windows, zlib.crc32(repr((shape, windows)).encode()) % 1000)
    if len(shape) > 3:  # one shot time for every leading index: a bad trace would mute them all
        geo["trace_types"] = [np.zeros_like(t) for t in geo["trace_types"]]
    kw = _kw(geo)
    om = O.Model(double=True, **kw)
    pm = L.Problem(**kw)
    try:
        rng = np.random.default_rng(zlib.crc32(repr(shape).encode()))
        x = _random_model(om, rng)
        y = _mute_vec(om, rng.random(om.record_len) - 0.5)
        ref = om.forward(x)
        gref = om.adjoint_update(y, -1.0, om.zeros_model())
        got = pm.forward(_to_product_layout(om, x).astype(np.complex64)).astype(np.float64)
        gp = _to_oracle_layout(om, pm.adjoint(y.astype(np.float32)).astype(np.complex128))
        rel = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        rel_g = np.linalg.norm(gp - gref) / np.linalg.norm(gref)
        print(shape, windows, "forward %.2e adjoint %.2e" % (rel, rel_g), flush=True)
        assert rel <= 2e-6 and rel_g <= 2e-6
        lhs = float(np.dot(got, y))
        rhs = float(np.sum(x.real * gp.real + x.imag * gp.imag))
        assert abs(lhs - rhs) <= 1e-6 * np.linalg.norm(got) * np.linalg.norm(y)
    finally:
        pm.close()


# time transforms in register FFTs: two phases (15 x 16, 11 x 13), three (equal
# odd factors, a last factor with a power of two, the longest within the LDS
# limit), tiles of odd trace counts, several windows of a run
PHASES = [((19, 384), (18, 192)), ((7, 227), (6, 114)), ((22, 547), (22, 274)),
          ((21, 1024), (18, 512)), ((18, 1440), (18, 720)), ((35, 60), (34, 16))]


@pytest.mark.parametrize("shape,windows", PHASES, ids=[str(w[1]) for _, w in PHASES])
def test_time_phases_match_fp64_oracle(shape, windows):
    test_any_window_length_matches_fp64_oracle(shape, windows)


# spatial lines in two register FFTs: lengths 35, 64, 225 and 240, along a
# strided dim, along both, and beside a dim that one FFT holds
FOLDED = [((42, 64), (28, 20)), ((51, 80), (51, 20)), ((180, 40), (180, 10)), ((288, 40), (192, 10)),
          ((54, 18, 40), (36, 12, 10)), ((60, 48, 40), (40, 32, 10)), ((8, 64, 40), (8, 64, 10)),
          ((3, 4, 42, 40), (2, 4, 28, 10))]


@pytest.mark.parametrize("shape,windows", FOLDED, ids=["x".join(map(str, w)) for _, w in FOLDED])
def test_folded_lines_match_fp64_oracle(shape, windows):
    test_any_window_length_matches_fp64_oracle(shape, windows)


# the specialised time kernels (whole tiles of 16 traces, Wt 64 to 512) beside
# run-time sized spatial ones: folded, one FFT a line, 3-D, LDS-resident
MIXED = [((96, 192), (48, 64)), ((18, 18, 320), (12, 12, 128)), ((4, 12, 4, 256), (4, 8, 4, 256)),
         ((16, 768), (16, 512)), ((272, 160), (272, 64)), ((6, 12, 96), (4, 8, 64))]


@pytest.mark.parametrize("shape,windows", MIXED, ids=["x".join(map(str, w)) for _, w in MIXED])
def test_specialised_time_with_any_spatial_size(shape, windows):
    test_any_window_length_matches_fp64_oracle(shape, windows)


@pytest.mark.parametrize("nan", [False, True])
@pytest.mark.parametrize("shape,windows", [((61, 300), (24, 106)), ((17, 34, 160), (16, 33, 64))])
def test_fused_iterations_match_separate_transforms(shape, windows, nan, monkeypatch):
    """The update fused with the next forward, from a zero model that is
    never in memory, against a written zero model and the same transforms as
    two launches (AGD_NO_FUSE): the same operations, bit for bit; a NaN in
    the data reaches the same samples."""
    kw = _kw(_spec_geometry(shape, windows, 5))
    data = [np.random.default_rng(6).standard_normal(shape).astype(np.float32)]
    if nan:
        data[0][..., -1, 40] = np.nan
    outs = []
    for fused in (True, False):
        monkeypatch.delenv("AGD_NO_FUSE", raising=False)
        if not fused:
            monkeypatch.setenv("AGD_NO_FUSE", "1")
        pm = L.Problem(**kw)
        try:
            pm.set_data(data)
            pm.run(1.0, 2 if nan else 7)
            outs.append(pm.output()[0])
        finally:
            pm.close()
    assert np.array_equal(outs[0], outs[1], equal_nan=True)
    assert np.isnan(outs[0]).any() == nan


@pytest.mark.parametrize("n_its", [2, 7])
@pytest.mark.parametrize("shape,windows", [((61, 300), (24, 106)), ((17, 34, 160), (16, 33, 64)),
                                           ((64, 512), (32, 128)), ((16, 64, 512), (16, 32, 256))])
def test_zero_start_matches_a_zero_model(shape, windows, n_its):
    """The zero start keeps no model in memory before its first update; an
    initial model of zeros given by the caller is read: the same numbers,
    bit for bit."""
    kw = _kw(_spec_geometry(shape, windows, 5))
    data = [np.random.default_rng(6).standard_normal(shape).astype(np.float32)]
    pm = L.Problem(**kw)
    try:
        pm.set_data(data)
        pm.run(1.0, n_its)
        out = pm.output()[0]
        pm.set_data(data)
        pm.run(1.0, n_its, x0=np.zeros(pm.model_len, np.complex64))
        assert np.array_equal(out, pm.output()[0])
    finally:
        pm.close()
