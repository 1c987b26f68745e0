"""GPU divergence screen (screen_div_error, src/module_io.f90:85-206) against
the oracle: mean |div|, the reference's signed running div_max and the
div_hist_max kept across calls; the per-substep screen of the step and its
NaN stop (src/module_navier_stokes.f90:344-350)."""
import numpy as np
import pytest

from hercules_amd import Channel, cases
from hercules_amd.channel import HerculesError
from tests.helpers import make_oracle
from tests.test_oracle_screen import random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cds,shape", [(1, (32, 32, 33)), (2, (32, 32, 33)), (2, (64, 16, 20)), (2, (16, 64, 9))])
def test_signed_screen_equals_oracle(cds, shape):
    nx, ny, nz = shape
    prm = cases.closed_channel(nx=nx, ny=ny, nz=nz, cds=cds)
    st = random_state(prm, 11 + nx + nz)
    o = make_oracle(prm, st)
    ch = Channel(prm)
    for k, v in st.items():
        ch.set_field(k, v)
    for scale, fin in ((1.0, 1), (0.7, 1), (3.0, 0)):
        for k in ("u", "v", "w"):
            ch.set_field(k, scale * st[k])
            o.set(k, scale * st[k])
        g = ch.screen_div_error_ref(fin)
        r = o.screen(fin)
        print("screen", cds, shape, fin, g, r)
        assert g[0] == pytest.approx(r[0], rel=1e-12)
        assert g[1] == pytest.approx(r[1], rel=1e-12)
        assert g[2] == pytest.approx(r[2], rel=1e-12)
    ch.close()


def test_substep_screen_records_and_hist():
    prm = cases.closed_channel(nx=32, ny=32, nz=33)
    st = cases.laminar_noise(prm, seed=5)
    ch = Channel(prm)
    for k, v in st.items():
        ch.set_field(k, v)
    ch.project()
    ch.init()
    ch.screen_substeps(True)
    ch.time_advancement_fd()
    recs = [ch.get_screen(s) for s in (1, 2, 3)]
    # the step's last record is the screen of the final fields
    again = ch.screen_div_error_ref(0)
    assert again[0] == recs[2][0] and again[1] == recs[2][1]
    # the history is the signed rule applied over the substeps
    hist = recs[0][2]
    assert abs(hist) >= abs(recs[0][1]) or hist == recs[0][1]
    for a, m, h in recs:
        assert np.isfinite(a) and abs(m) < 1e-9 and abs(h) < 1e-9
    u0 = ch.get_field("u")
    ch.screen_substeps(False)
    ch.close()
    # the screen does not change the step
    ch2 = Channel(prm)
    for k, v in st.items():
        ch2.set_field(k, v)
    ch2.project()
    ch2.init()
    ch2.time_advancement_fd()
    assert np.array_equal(ch2.get_field("u"), u0)
    ch2.close()


@pytest.mark.parametrize("entry", ["time_advancement_fd", "steps"])
def test_nan_stops_the_step(entry):
    prm = cases.closed_channel(nx=32, ny=32, nz=33)
    st = cases.laminar_noise(prm, seed=6)
    st["u"][4, 3, 2] = np.nan
    ch = Channel(prm)
    for k, v in st.items():
        ch.set_field(k, v)
    ch.init()
    ch.screen_substeps(True)
    with pytest.raises(HerculesError) as ei:
        if entry == "steps":
            ch.steps(3)
        else:
            ch.time_advancement_fd()
    assert ei.value.code == 4 and "NaN" in str(ei.value)
    if entry == "steps":
        assert ch.scalar("stps") == 1  # stopped after the first step
    ch.close()


def _planted(kind, shape, dz, rng):
    """w fields (nz, ny, nx) whose divergence in scan order is of one kind."""
    nz, ny, nx = shape
    n = nz * ny * nx
    d = rng.standard_normal(n)
    ramp = np.arange(1, n + 1) / n
    if kind == "rising":       # every point is a record
        d = ramp
    elif kind == "rising_alternate":
        d = ramp * np.where(np.arange(n) % 2, 1.0, -1.0)
    elif kind == "negative":
        d = -np.abs(d)
    elif kind == "zero":
        d = np.zeros(n)
    elif kind == "late_peak":  # long stretches that change nothing
        d = 1e-3 * d
        d[n // 3] = 5.0
        d[2 * n // 3] = -6.0
    w = np.cumsum(d.reshape(shape) * dz[:, None, None], axis=0)
    if kind == "infinite":
        w[nz // 2, ny // 2, nx // 2] = np.inf
    return w


@pytest.mark.parametrize("shape", [(9, 16, 16), (50, 16, 48), (65, 64, 64)])
@pytest.mark.parametrize("kind", ["random", "rising", "rising_alternate", "negative", "zero", "late_peak", "infinite"])
def test_scan_equals_the_point_by_point_rule(kind, shape):
    """div_max and div_hist_max bit for bit against the rule applied to one
    point after another (u = v = 0, so d = (w(k) - w(k-1)) / dz(k)), runs
    shorter and longer than the 2048 points of a unit, and more records than
    a unit keeps; div_avg to the rounding of a sum of positive terms."""
    nz, ny, nx = shape
    ch = Channel(cases.closed_channel(nx=nx, ny=ny, nz=nz))
    dz = ch.mesh()[1]
    rng = np.random.default_rng(nz)
    hist = 0.0
    import ctypes as C
    h2 = C.c_double(0.0)
    for fin in (1, 0, 1):
        w = _planted(kind, shape, dz, rng)
        ch.set_field("w", w)
        with np.errstate(invalid="ignore"):
            d = ((w - np.concatenate([np.zeros_like(w[:1]), w[:-1]], 0)) / dz[:, None, None]).reshape(-1)
        mx, hs = 0.0, hist
        for x in d.tolist():
            a = abs(x)
            if a > mx:
                mx = x
            if fin and a > hs:
                hs = x
        hist = hs
        got = ch.screen_div_error_ref(fin)
        assert got[1] == mx and got[2] == hist, (kind, fin, got, mx, hist)
        if np.isfinite(d).all():
            assert got[0] == pytest.approx(np.abs(d).mean(), rel=1e-12)
        a1, m1 = C.c_double(), C.c_double()
        assert ch.L.hc_screen_div_error_noalloc(ch.h, fin, C.byref(a1), C.byref(m1), C.byref(h2)) == 0
        assert m1.value == mx and h2.value == hist
    ch.close()
