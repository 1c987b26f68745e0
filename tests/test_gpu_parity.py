"""HIP path vs the CPU oracle, through the C ABI (needs an MI355X)."""
import numpy as np
import pytest

from hercules_amd import Channel, cases
from tests.helpers import divergence, make_oracle, poisson_residual, rel_l2, small_case

pytestmark = pytest.mark.gpu


def _channel(prm, state):
    ch = Channel(prm)
    for k, v in state.items():
        ch.set_field(k, v)
    ch.init()
    return ch


SOLVE_SHAPES = [(16, 16, 17), (32, 32, 33), (64, 64, 65), (16, 16, 129), (16, 16, 193),
                (16, 16, 257), (256, 256, 9), (192, 192, 9), (32, 192, 65)]


@pytest.mark.parametrize("shape", SOLVE_SHAPES)
@pytest.mark.parametrize("eq", ["u", "v", "w", "p", "t"])
def test_poisson_solver_fft_matches_oracle(shape, eq):
    nx, ny, nz = shape
    prm = cases.closed_channel(nx=nx, ny=ny, nz=nz)
    rng = np.random.default_rng(3)
    src = rng.standard_normal((nz, ny, nx))
    if eq == "p":
        src -= src.mean(axis=(1, 2), keepdims=True)
    o = make_oracle(prm, {})
    ref = o.solve(eq, 8.0 / 15.0, src)
    with Channel(prm) as ch:
        got = ch.poisson_solver_fft(eq, 8.0 / 15.0, src)
    err = rel_l2(got, ref)
    print(f"poisson {eq} {shape}: rel L2 {err:.3e}")
    if eq == "p":
        # the Neumann Poisson problem on the zstretch=2 grid has a condition
        # number ~1e6-1e8 in its lowest modes: two backward-stable solvers
        # agree only to cond*eps; the residual is checked separately.
        assert err < 1e-9
        r_gpu = poisson_residual(prm, 8.0 / 15.0, got, src)
        r_orc = poisson_residual(prm, 8.0 / 15.0, ref, src)
        print(f"   residual gpu {r_gpu:.3e} oracle {r_orc:.3e}")
        assert r_gpu < 1e-14 and r_gpu < 10 * r_orc + 1e-15
    else:
        assert err < 1e-13


@pytest.mark.parametrize("shape", [(32, 32, 33), (16, 16, 129), (16, 32, 257), (64, 64, 9), (256, 256, 9),
                                   (192, 192, 9)])
def test_steps_shapes_match_oracle(shape):
    nx, ny, nz = shape
    prm, st = small_case("closed", nx=nx, ny=ny, nz=nz)
    o = make_oracle(prm, st)
    ch = _channel(prm, st)
    o.steps(2)
    ch.steps(2)
    for n in ["u", "v", "w", "p"]:
        err = rel_l2(ch.get_field(n), o.get(n))
        print(f"{shape} {n}: rel L2 {err:.3e}")
        assert err < 1e-10, (n, err)
    ch.close()


@pytest.mark.parametrize("shapes", [dict(rhs_xt=0), dict(rhs_xt=1), dict(rhs_xt=2, c2r_pts=512)])
def test_grid_stride_transforms_over_many_tiles_match_oracle(shapes):
    """256x256x25: the grid-stride x transforms run several trips per block
    (inverse x: 6400 tiles over 2048 blocks; the in-place R2C of the tiled
    right-hand side: 1600 tiles per field over 682 blocks), with the fused and
    the x-y tiled momentum right-hand side."""
    prm, st = small_case("closed", nx=256, ny=256, nz=25)
    o = make_oracle(prm, st)
    ch = _channel(prm, st)
    ch.set_tuning(**shapes)
    o.steps(2)
    ch.steps(2)
    for n in ["u", "v", "w", "p"]:
        err = rel_l2(ch.get_field(n), o.get(n))
        print(f"{shapes} {n}: rel L2 {err:.3e}")
        assert err < 1e-10, (n, err)
    ch.close()


@pytest.mark.parametrize("kind,kw", [
    ("closed", {}),
    ("closed", {"cds": 1}),
    ("closed", {"dp_opt": 2}),
    ("closed", {"u_mrf": 0.3}),
    ("closed", {"dp_opt": 3, "fc": 0.5, "ug": 1.0, "vg": 0.2}),
    ("closed", {"dts": 1}),
    ("open_t", {}),
    ("closed", {"isdamp": 1, "nzdamp": 8, "cdamp": 0.3}),
    ("open_t", {"isdamp": 1, "nzdamp": 10, "cdamp": 0.2}),
    ("closed", {"isdamp": 1, "nzdamp": 6, "cdamp": 1.0, "cds": 1, "dp_opt": 3, "fc": 0.5, "ug": 1.0}),
    # top temperature gradient instead of t = ttop (extension)
    ("open_t", {"tbc_top": 1, "dtdz_top": 0.5}),
    ("open_t", {"tbc_top": 1, "dtdz_top": -0.8, "cds": 1, "wall_rows": 1}),
    ("closed", {"isscalar": 1, "got": 0.05, "tbc_top": 1, "dtdz_top": -0.3}),
    ("open_t", {"tbc_top": 1, "dtdz_top": 0.5, "isdamp": 1, "nzdamp": 8, "cdamp": 0.2}),
    # sponge levels through x-y tiles with points clear of the x / y edges
    # (k_rhs_mom_xt<..., DAMP>) and the edge points through the accessor
    ("open_t", {"nx": 64, "ny": 64, "nz": 65, "isdamp": 1, "nzdamp": 12, "cdamp": 0.2}),
    ("closed", {"nx": 128, "ny": 32, "nz": 33, "isdamp": 1, "nzdamp": 8, "cdamp": 0.3, "dp_opt": 3, "fc": 0.5,
                "ug": 1.0, "vg": 0.2}),
])
def test_steps_match_oracle(kind, kw):
    prm, st = small_case(kind, **kw)
    o = make_oracle(prm, st)
    ch = _channel(prm, st)
    nsteps = 3
    o.steps(nsteps)
    ch.steps(nsteps)
    names = ["u", "v", "w", "p"] + (["t"] if prm.isscalar else [])
    for n in names:
        err = rel_l2(ch.get_field(n), o.get(n))
        print(f"{kind} {kw} {n}: rel L2 {err:.3e}")
        assert err < 1e-10, (n, err)
    ch.close()


def test_damping_of_a_passive_temperature_matches_oracle():
    """isscalar=0: rayleigh_damping still relaxes t in place every substep
    (src/module_navier_stokes.f90:258-264) while nothing else updates it."""
    prm, st = small_case("closed", isdamp=1, nzdamp=9, cdamp=0.4)
    st["t"] = np.random.default_rng(9).standard_normal(st["u"].shape)
    o = make_oracle(prm, st)
    ch = _channel(prm, st)
    o.steps(2)
    ch.steps(2)
    for n in ("u", "v", "w", "p", "t"):
        err = rel_l2(ch.get_field(n), o.get(n))
        print(f"damped, passive t: {n} rel L2 {err:.3e}")
        assert err < 1e-10, (n, err)
    ch.close()


@pytest.mark.parametrize("shape", [(32, 32, 33), (16, 16, 257), (64, 64, 65)])
def test_project_divergence_free_and_idempotent(shape):
    nx, ny, nz = shape
    prm, st = small_case("closed", nx=nx, ny=ny, nz=nz)
    with Channel(prm) as ch:
        for k in ("u", "v", "w"):
            ch.set_field(k, st[k])
        avg0, mx0 = ch.screen_div_error()
        ch.project()
        avg1, mx1 = ch.screen_div_error()
        once = [ch.get_field(k) for k in ("u", "v", "w")]
        ch.project()
        twice = [ch.get_field(k) for k in ("u", "v", "w")]
    d, terms = divergence(*once, prm)
    rel = np.abs(d).max() / terms.max()
    print(f"{shape}: max|div| {mx0:.3e} -> {mx1:.3e}; numpy max|div| {np.abs(d).max():.3e}, "
          f"relative to its terms {rel:.3e}")
    assert rel < 1e-12
    for a, b in zip(once, twice):
        assert rel_l2(b, a) < 1e-12


def test_config1_100_steps_match_oracle():
    """Neutral closed channel 64x64x65, laminar + 10% noise projected to zero
    divergence, RK3, dt=1e-3, 100 steps: fields, divergence, wall shear."""
    prm = cases.closed_channel(nx=64, ny=64, nz=65)
    st = cases.laminar_noise(prm, seed=1)
    ch = Channel(prm)
    for k, v in st.items():
        ch.set_field(k, v)
    ch.project()
    st = {k: ch.get_field(k) for k in ("u", "v", "w", "p", "t")}
    ch.init()
    o = make_oracle(prm, st)
    o.steps(100)
    ch.steps(100)
    for n in ("u", "v", "w", "p"):
        err = rel_l2(ch.get_field(n), o.get(n))
        print(f"config1 {n}: rel L2 {err:.3e}")
        assert err < 1e-10, (n, err)
    avg, mx = ch.screen_div_error()
    d, terms = divergence(ch.get_field("u"), ch.get_field("v"), ch.get_field("w"), prm)
    do, _ = divergence(o.get("u"), o.get("v"), o.get("w"), prm)
    print(f"config1 div avg {avg:.3e} max {mx:.3e} (oracle {np.abs(do).max():.3e}), "
          f"relative to its terms {np.abs(d).max() / terms.max():.3e}")
    assert np.abs(d).max() / terms.max() < 1e-13
    tw_g = cases.wall_shear(ch.get_field("u"), prm)
    tw_o = cases.wall_shear(o.get("u"), prm)
    print(f"wall shear gpu {tw_g} oracle {tw_o}")
    assert abs(tw_g[0] - tw_o[0]) <= 1e-10 * abs(tw_o[0])
    assert abs(tw_g[1] - tw_o[1]) <= 1e-10 * abs(tw_o[1])
    ch.close()


@pytest.mark.parametrize("kind,kw", [("closed", {"u_mrf": 0.25}), ("open_t", {})])
def test_wall_shear_entry(kind, kw):
    """hc_wall_shear against the closed form on the oracle's state after two
    steps: 2 nu (<u_1> + u_mrf) / dz_1 (no-slip ghost rule), top likewise for a
    closed channel and 0 under the free-slip top."""
    prm, st = small_case(kind, **kw)
    o = make_oracle(prm, st)
    ch = _channel(prm, st)
    o.steps(2)
    ch.steps(2)
    got = ch.wall_shear()
    want = cases.wall_shear(o.get("u"), prm)
    print(f"{kind}: wall shear gpu {got} oracle fields {want}")
    assert abs(got[0] - want[0]) <= 1e-10 * abs(want[0])
    if prm.ochannel == 0:
        assert abs(got[1] - want[1]) <= 1e-10 * abs(want[1])
    else:
        assert got[1] == 0.0
    ch.close()


@pytest.mark.parametrize("wall_rows", [0, 1])
def test_temperature_solve_with_top_gradient_matches_oracle(wall_rows):
    """poisson_solver_fft for t (tbnd) with the top gradient row and ghost."""
    prm = cases.stratified_open_channel(nx=32, ny=32, nz=65, tbc_top=1, dtdz_top=0.4, wall_rows=wall_rows)
    src = np.random.default_rng(9).standard_normal((prm.nz, prm.ny, prm.nx))
    ref = make_oracle(prm, {}).solve("t", 8.0 / 15.0, src)
    with Channel(prm) as ch:
        got = ch.poisson_solver_fft("t", 8.0 / 15.0, src)
    err = rel_l2(got, ref)
    print(f"t solve, top gradient, wall_rows {wall_rows}: rel L2 {err:.3e}")
    assert err < 1e-13


@pytest.mark.parametrize("shape,tile,kw", [
    ((96, 16, 3), 0, {}),                  # the fewest levels: a run's first level, interior and top
    ((32, 32, 13), 1, {"cds": 1}),         # one tile wide, forced on short rows
    ((128, 32, 50), 0, {"u_mrf": 0.3}),    # runs of unequal length, moving frame
    ((192, 48, 37), 4, {"dp_opt": 3, "fc": 0.5, "ug": 1.0, "vg": 0.2}),
    ((384, 16, 20), 0, {"cds": 1}),        # rows beyond 256
    ((512, 32, 26), 0, {"dp_opt": 2}),
    ((64, 64, 33), 3, {}),
])
def test_marching_tiles_match_oracle(shape, tile, kw):
    """k_rhs_mom_march at the edges of its tiles and runs of levels: 1e-10 as
    for every step here (agreement is round-off times the pressure solve's
    condition)."""
    nx, ny, nz = shape
    prm, st = small_case("closed", nx=nx, ny=ny, nz=nz, **{"dt": 5e-4, "wall_rows": 1, **kw})
    o = make_oracle(prm, st)
    ch = _channel(prm, st)
    ch.set_tuning(rhs_xt=tile)
    o.steps(2)
    ch.steps(2)
    for n in ["u", "v", "w", "p"]:
        err = rel_l2(ch.get_field(n), o.get(n))
        print(f"{shape} {tile} {kw} {n}: rel L2 {err:.3e}")
        assert err < 1e-10, (n, err)
    ch.close()


@pytest.mark.parametrize("nz,kw", [
    (3, {}), (64, {}), (65, {}), (127, {"isscalar": 1, "got": 0.05}), (129, {"cds": 1}), (320, {}), (321, {}),
    (448, {"dp_opt": 2}), (449, {}), (512, {}), (513, {}), (1024, {}),
])
def test_column_levels_match_oracle(nz, kw):
    """Column kernels at the ends of every number of levels per lane (2 to 16),
    of the block shapes (beyond 512 levels two columns) and of three and four
    LDS tiles.  u, v, w, t as for every step; p to round-off times the
    condition of the (0,0) Neumann system, 4/dz_min^2 over (pi/lz)^2."""
    prm, st = small_case("closed", nx=16, ny=16, nz=nz, wall_rows=1, dt=2e-4, **kw)
    o = make_oracle(prm, st)
    ch = _channel(prm, st)
    o.steps(1)
    ch.steps(1)
    kappa = 4.0 / ch.mesh()[1].min() ** 2 / (np.pi / prm.lz) ** 2
    for n in ["u", "v", "w", "p"] + (["t"] if prm.isscalar else []):
        err = rel_l2(ch.get_field(n), o.get(n))
        print(f"nz {nz} {kw} {n}: rel L2 {err:.3e}")
        assert err < max(1e-10, 10 * 2.3e-16 * kappa if n == "p" else 0.0), (n, err)
    ch.close()


def _kappa(ch):
    """condition of the (0,0) Neumann system: 4/dz_min^2 over (pi/lz)^2"""
    return 4.0 / ch.mesh()[1].min() ** 2 / (np.pi / ch.prm.lz) ** 2


# the first or last number of levels of every count per lane from 7 on
TALL = [321, 448, 449, 512, 513, 640, 641, 768, 769, 896, 897, 1024]


@pytest.mark.parametrize("nz", TALL)
@pytest.mark.parametrize("eq", ["u", "w", "p", "t"])
def test_tall_columns_solve_matches_oracle(nz, eq):
    """k_column_solve; tolerances as for the shapes above, p to round-off times
    the condition beyond that."""
    prm = cases.closed_channel(nx=16, ny=16, nz=nz, wall_rows=1)
    src = np.random.default_rng(nz).standard_normal((nz, 16, 16))
    if eq == "p":
        src -= src.mean(axis=(1, 2), keepdims=True)
    ref = make_oracle(prm, {}).solve(eq, 8.0 / 15.0, src)
    with Channel(prm) as ch:
        got = ch.poisson_solver_fft(eq, 8.0 / 15.0, src)
        kappa = _kappa(ch)
    err = rel_l2(got, ref)
    print(f"solve {eq} nz {nz}: rel L2 {err:.3e}")
    if eq == "p":
        assert err < max(1e-9, 10 * 2.3e-16 * kappa)
        assert poisson_residual(prm, 8.0 / 15.0, got, src) < 1e-14
    else:
        assert err < 1e-13


@pytest.mark.parametrize("nz", TALL)
def test_tall_columns_project(nz):
    """k_column_project: the divergence left is the pressure solve's residual,
    below 1e-14 of |L| |phi| + |div| as in the solves above, and the second
    projection removes no more than such a divergence holds (a field of
    divergence r differs from its projection by at most lz/pi |r|)."""
    prm, st = small_case("closed", nx=16, ny=16, nz=nz, wall_rows=1)
    d0, _ = divergence(st["u"], st["v"], st["w"], prm)
    with Channel(prm) as ch:
        for k in ("u", "v", "w"):
            ch.set_field(k, st[k])
        phi = ch.poisson_solver_fft("p", 1.0, d0)
        ch.project()
        once = [ch.get_field(k) for k in ("u", "v", "w")]
        ch.project()
        twice = [ch.get_field(k) for k in ("u", "v", "w")]
        lnorm = 4.0 / ch.mesh()[1].min() ** 2 + 6.0 * (prm.nx / prm.lx) ** 2 + 6.0 * (prm.ny / prm.ly) ** 2
    d = divergence(*once, prm)[0]
    scale = lnorm * np.abs(phi).max() + np.abs(d0).max()
    print(f"project nz {nz}: {np.abs(d).max() / scale:.3e}")
    assert np.abs(d).max() < 1e-14 * scale
    bound = prm.lz / np.pi * 1e-14 * scale
    assert bound < 1e-3 * max(np.abs(a).max() for a in once)  # the check has a meaning
    for a, b in zip(once, twice):
        assert np.abs(b - a).max() < bound


@pytest.mark.parametrize("nz", [513, 640, 641, 768, 769, 896, 897])
def test_tall_columns_steps_match_oracle(nz):
    """k_column_mom and k_column_t; p is left to the solves above (its error is
    the condition's, and three substeps add theirs)."""
    prm, st = small_case("open_t", nx=16, ny=16, nz=nz, wall_rows=1, dt=2e-4)
    o = make_oracle(prm, st)
    ch = _channel(prm, st)
    o.steps(1)
    ch.steps(1)
    for n in ["u", "v", "w", "t"]:
        err = rel_l2(ch.get_field(n), o.get(n))
        print(f"nz {nz} {n}: rel L2 {err:.3e}")
        assert err < 1e-10, (n, err)
    ch.close()


@pytest.mark.parametrize("shapes", [dict(), dict(rgroup=1), dict(rgroup=32)])
def test_whole_rows_over_many_tiles_match_oracle(shapes):
    """64x512x25: right-hand sides of whole rows fused with the x transform (the
    FP64 rows that do not march), 32 y tiles per level in every tile order."""
    prm, st = small_case("closed", nx=64, ny=512, nz=25)
    o = make_oracle(prm, st)
    ch = _channel(prm, st)
    ch.set_tuning(**shapes)
    o.steps(1)
    ch.steps(1)
    for n in ["u", "v", "w", "p"]:
        err = rel_l2(ch.get_field(n), o.get(n))
        print(f"{shapes} {n}: rel L2 {err:.3e}")
        assert err < 1e-10, (n, err)
    ch.close()
