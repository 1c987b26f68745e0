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


def _spectral_divergence(ch):
    """get_div_spec in numpy: Fourier derivatives without the Nyquist
    wavenumber, (w(k) - w(k-1)) / dz(k) in z."""
    p = ch.prm
    u, v, w = (ch.get_field(k).astype(np.float64) for k in ("u", "v", "w"))
    kx = 2 * np.pi / p.lx * np.arange(p.nx // 2 + 1)
    ky = 2 * np.pi / p.ly * np.fft.fftfreq(p.ny, 1.0 / p.ny)
    kx[-1] = ky[p.ny // 2] = 0.0
    dudx = np.fft.irfft(1j * kx * np.fft.rfft(u, axis=2), n=p.nx, axis=2)
    dvdy = np.fft.ifft(1j * ky[:, None] * np.fft.fft(v, axis=1), axis=1).real
    return dudx + dvdy + (w - np.concatenate([np.zeros_like(w[:1]), w[:-1]], 0)) / ch.mesh()[1][:, None, None]


@pytest.mark.parametrize("shape", [(16, 16, 3), (48, 16, 20), (64, 32, 33), (96, 96, 49)])
@pytest.mark.parametrize("precision", [0, 1])
def test_spectral_screen_is_the_plain_maximum(shape, precision):
    """cds = 3: |d| is stored (src/module_spectral.f90:931-946), so the states
    are plain maxima; sizes of less than a block, of a ragged last one and of
    several points per thread.  FP64 to the rounding of the transforms, FP32
    spectra to 2^-24 times their ten levels of butterflies."""
    nx, ny, nz = shape
    prm = cases.closed_channel(nx=nx, ny=ny, nz=nz, cds=3, issk=1, precision=precision)
    st = random_state(prm, 3 + nx)
    ch = Channel(prm)
    for k, v in st.items():
        ch.set_field(k, v)
    ch.init()
    st = {k: ch.get_field(k) for k in ("u", "v", "w")}
    d = np.abs(_spectral_divergence(ch))
    tol = 1e-5 if precision else 1e-12
    hist = 0.0
    for scale, fin in ((1.0, 1), (-0.5, 1), (4.0, 0), (2.0, 1)):
        for k, v in st.items():
            ch.set_field(k, scale * v)
        m = abs(scale) * d.max()
        hist = max(hist, m) if fin else hist
        got = ch.screen_div_error_ref(fin)
        assert got[0] == pytest.approx(abs(scale) * d.mean(), rel=tol)
        assert got[1] == pytest.approx(m, rel=tol) and got[2] == pytest.approx(hist, rel=tol)
    bad = st["v"].copy()
    bad[-1, -1, -1] = np.nan
    ch.set_field("v", bad)
    with pytest.raises(HerculesError) as ei:
        ch.screen_div_error_ref(1)
    assert ei.value.code == 4
    ch.close()


@pytest.mark.parametrize("cds", [1, 2])
def test_screen_of_fp32_fields_equals_fp64_fields_of_the_same_values(cds):
    """The mixed variant forms the divergence of its FP32 fields in FP64."""
    out = []
    for precision in (0, 1):
        prm = cases.closed_channel(nx=48, ny=32, nz=33, cds=cds, precision=precision)
        st = random_state(prm, 5)
        ch = Channel(prm)
        for k, v in st.items():
            ch.set_field(k, v.astype(np.float32).astype(np.float64))
        out.append([ch.screen_div_error_ref(f) for f in (1, 0)])
        ch.close()
    for a, b in zip(*out):
        assert a[0] == pytest.approx(b[0], rel=1e-12) and a[1:] == b[1:]


def test_units_of_several_batches_equal_units_of_one():
    """256x256x257: the allocation-free entry forms units of two batches, the
    other of one; a rising start (units with more records than are kept, walked
    point by point) and random signs after it."""
    import ctypes as C
    prm = cases.closed_channel(nx=256, ny=256, nz=257)
    ch = Channel(prm)
    rng = np.random.default_rng(1)
    d = rng.standard_normal(prm.nx * prm.ny * prm.nz)
    d[:20000] = np.arange(1, 20001) / 10000.0
    d[30000:40000] = -np.arange(1, 10001) / 3000.0
    dz = ch.mesh()[1]
    w = np.cumsum(d.reshape(prm.nz, prm.ny, prm.nx) * dz[:, None, None], axis=0)
    ch.set_field("w", w)
    h = C.c_double(0.0)
    for fin in (1, 0, 1):
        avg, mx, hist = ch.screen_div_error_ref(fin)
        a, m = C.c_double(), C.c_double()
        assert ch.L.hc_screen_div_error_noalloc(ch.h, fin, C.byref(a), C.byref(m), C.byref(h)) == 0
        assert m.value == mx and h.value == hist
        assert a.value == pytest.approx(avg, rel=1e-12)
    d = ((w - np.concatenate([np.zeros_like(w[:1]), w[:-1]], 0)) / dz[:, None, None]).reshape(-1)
    ref = 0.0
    for x in d.tolist():
        if abs(x) > ref:
            ref = x
    assert mx == ref
    ch.close()
