"""Time blocks of one run of several time windows against runs split by the
launch.

A launch of few time blocks splits their runs over grid y, down to one time
window a block in the adjoint, so a problem of test size never shows a block
that goes on from one window to the next (the tile reused, the carry kept).
AGD_TIME_TW=0 keeps one run per block, as the launches of large volumes do.
Compared here, bit for bit (the same sums): both forms of every kernel, two
and three register-FFT phases, lines, whole and partial tiles, specialised
kernels in both variants; with a second patch of fewer
time windows in the same class, whose blocks get empty runs from a split.
The one-run form also meets the FP64 oracle, to the 2e-6 of test_any_size.
"""
import numpy as np
import pytest

from agdeblend_amd import lib as L
from tests.test_gpu_parity import (_kw, _mute_vec, _random_model, _spec_geometry,
                                   _to_oracle_layout, _to_product_layout)

pytestmark = pytest.mark.gpu

# (traces of the two patches, window of traces, time samples, window of time)
CASES = [((64, 32), 32, (2048, 512), 256),   # specialised
         ((64, 64), 32, (4096, 1024), 512),  # specialised, lean forward tile
         ((40, 23), 23, (1000, 300), 200),   # 10 x 5 x 5, a partial tile
         ((36, 18), 18, (1200, 384), 192),   # 15 x 16
         ((17, 17), 17, (684, 228), 114),    # 11 x 13
         ((45, 30), 15, (640, 160), 58),     # lines, prime 73
         ((20, 18), 18, (900, 200), 94)]     # lines 59 x 2


def _two_patches(ntr, w, nt, wt, seed):
    a = _spec_geometry((ntr[0], nt[0]), (w, wt), seed)
    b = _spec_geometry((ntr[1], nt[1]), (w, wt), seed + 1)
    g = {k: a[k] + b[k] for k in a}
    g["volumes"] = [0, 1]
    g["channels"][1] = g["channels"][1] + 1
    return _kw(g)


def _results(kw, runs, variant, monkeypatch, x, y, data):
    if runs is None:
        monkeypatch.delenv("AGD_TIME_TW", raising=False)
    else:
        monkeypatch.setenv("AGD_TIME_TW", runs)
    pm = L.Problem(**kw)
    try:
        for c, f in enumerate(pm.time_factors()):
            if f != (0, 0):
                pm.set_time_variant(c, variant)
        out = [pm.forward(x), pm.adjoint(y)]
        pm.set_data(data)
        pm.run(1.0, 5)
        out += pm.output()
        ntw = sorted({pm.window(i)["ntw"] for i in range(pm.n_windows)})
        return [np.array(o) for o in out], ntw
    finally:
        pm.close()


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("ntr,w,nt,wt", CASES, ids=["%dx%d" % (c[1], c[3]) for c in CASES])
def test_one_run_and_split_runs_agree(ntr, w, nt, wt, variant, monkeypatch):
    from oracle import oracle as O
    kw = _two_patches(ntr, w, nt, wt, 7 * w + wt)
    om = O.Model(double=True, **kw)
    rng = np.random.default_rng(wt)
    xo = _random_model(om, rng)
    y = _mute_vec(om, rng.random(om.record_len) - 0.5)
    x = _to_product_layout(om, xo).astype(np.complex64)
    data = [rng.standard_normal((n, t)).astype(np.float32) for n, t in zip(ntr, nt)]
    args = (variant, monkeypatch, x, y.astype(np.float32), data)
    one, ntw = _results(kw, "0", *args)
    split, _ = _results(kw, None, *args)
    assert len(ntw) == 2 and ntw[0] >= 2 and ntw[1] >= 2 * ntw[0]
    for a, b in zip(one, split):
        assert np.array_equal(a, b)
    ref, gref = om.forward(xo), om.adjoint_update(y, -1.0, om.zeros_model())
    got = one[0].astype(np.float64)
    gp = _to_oracle_layout(om, one[1].astype(np.complex128))
    assert np.linalg.norm(got - ref) <= 2e-6 * np.linalg.norm(ref)
    assert np.linalg.norm(gp - gref) <= 2e-6 * np.linalg.norm(gref)


def test_one_run_is_launched_as_one_run(monkeypatch):
    """30 blocks of 17 time windows: the one serial chain takes at least half
    as long again as the split ones (three times as measured)."""
    kw = _kw(_spec_geometry((64, 2304), (32, 256), 3))
    us = {}
    for runs in ("0", None):
        if runs is None:
            monkeypatch.delenv("AGD_TIME_TW", raising=False)
        else:
            monkeypatch.setenv("AGD_TIME_TW", runs)
        pm = L.Problem(**kw)
        try:
            y = np.ones(pm.record_len, np.float32)
            pm.adjoint(y)
            best = 1e9
            for _ in range(5):
                L.timing(True)
                pm.adjoint(y)
                L.timing(False)
                ms, n = L.timing_get("adj_time")
                best = min(best, ms / n)
            us[runs] = best * 1e3
        finally:
            pm.close()
    print("one run %.1f us, split %.1f us" % (us["0"], us[None]), flush=True)
    assert us["0"] > 1.5 * us[None]
