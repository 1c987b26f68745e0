"""Transform lengths 48, 96 and 384 (2^a 3^b, beside the 16..512 powers of
two and 192): the x and y transforms, the right-hand-side tiles of those
widths (16 rows at nx = 48, 8 at 96, the one-pass kernel at 384) and the
column passes, against the oracle (whose DFT is pinned against numpy at
these lengths, tests/test_oracle_pins.py); needs an MI355X."""
import numpy as np
import pytest

from hercules_amd import Channel, cases
from tests.helpers import make_oracle, rel_l2, small_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(48, 96, 17), (96, 48, 33), (384, 16, 17), (16, 384, 17)])
@pytest.mark.parametrize("eq", ["u", "p"])
def test_poisson_solver_fft_new_lengths(shape, eq):
    nx, ny, nz = shape
    prm = cases.closed_channel(nx=nx, ny=ny, nz=nz)
    src = np.random.default_rng(4).standard_normal((nz, ny, nx))
    if eq == "p":
        src -= src.mean(axis=(1, 2), keepdims=True)
    ref = make_oracle(prm, {}).solve(eq, 8.0 / 15.0, src)
    with Channel(prm) as ch:
        got = ch.poisson_solver_fft(eq, 8.0 / 15.0, src)
    err = rel_l2(got, ref)
    print(shape, eq, f"{err:.2e}")
    assert err < (1e-9 if eq == "p" else 1e-13), err


@pytest.mark.parametrize("kind,shape,kw", [
    ("closed", (48, 48, 33), {}),
    ("closed", (96, 96, 33), {}),
    ("closed", (384, 32, 17), {}),
    ("closed", (48, 96, 17), {"cds": 1}),
    ("open_t", (96, 48, 33), {}),
    ("closed", (96, 48, 33), {"cds": 3, "issk": 1}),
    ("open_t", (48, 96, 17), {"cds": 3, "issk": 1}),
    ("closed", (384, 16, 17), {"cds": 3, "issk": 0}),
])
def test_steps_new_lengths_match_oracle(kind, shape, kw):
    nx, ny, nz = shape
    prm, st = small_case(kind, nx=nx, ny=ny, nz=nz, **kw)
    o = make_oracle(prm, st)
    ch = Channel(prm)
    for k, v in st.items():
        ch.set_field(k, v)
    ch.init()
    o.steps(2)
    ch.steps(2)
    names = ["u", "v", "w", "p"] + (["t"] if prm.isscalar else [])
    for n in names:
        err = rel_l2(ch.get_field(n), o.get(n))
        print(kind, shape, kw, n, f"{err:.2e}")
        assert err < 1e-10, (n, err)
    ch.close()


@pytest.mark.parametrize("shape,kw", [((96, 96, 33), {}), ((48, 96, 33), {"cds": 3, "issk": 1})])
def test_mixed_new_lengths_track_fp64(shape, kw):
    nx, ny, nz = shape
    prm, st = small_case("closed", nx=nx, ny=ny, nz=nz, **kw)
    out = {}
    for pr in (0, 1):
        ch = Channel(prm.replace(precision=pr))
        for k, v in st.items():
            ch.set_field(k, v)
        ch.project()
        ch.init()
        ch.steps(10)
        out[pr] = {n: ch.get_field(n) for n in ("u", "v", "w")}
        ch.close()
    for n in ("u", "v", "w"):
        err = rel_l2(out[1][n], out[0][n])
        print(shape, kw, n, f"{err:.2e}")
        assert err < (1e-5 if n == "u" else 1e-4), (n, err)


_REFUSED = """
import ctypes, sys
if len(sys.argv) > 2:
    ctypes.CDLL(sys.argv[2], mode=ctypes.RTLD_GLOBAL)
import numpy as np
from hercules_amd import Channel
from tests.helpers import small_case
out = {}
for nz in (257, 341, 342, 448, 449, 512):
    prm, st = small_case("open_t", nx=16, ny=16, nz=nz, wall_rows=1, dt=2e-4)
    ch = Channel(prm)
    for k, v in st.items():
        ch.set_field(k, v)
    ch.project()
    ch.init()
    assert ch.scalar("col_tiles") == (1 if len(sys.argv) > 2 else 4 if nz <= 320 else 1)
    ch.steps(1)
    for k in ("u", "v", "w", "p", "t"):
        out[f"{k}{nz}"] = ch.get_field(k)
    ch.close()
np.savez(sys.argv[1], **out)
"""


_RUNTIME = """
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>
typedef struct { unsigned x, y, z; } dim;
int hipFuncSetAttribute(const void *f, int a, int v) { return 1; }
int hipLaunchKernel(const void *f, dim g, dim b, void **args, size_t lds, void *st)
{
    static int (*next)(const void *, dim, dim, void **, size_t, void *);
    if (lds > 65536) return 1;
    if (!next) {
        void *h = dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_NOLOAD);
        next = (int (*)(const void *, dim, dim, void **, size_t, void *))dlsym(h, "hipLaunchKernel");
    }
    return next(f, g, b, args, lds, st);
}
"""


def test_column_kernels_within_the_default_lds(tmp_path):
    """Where the runtime refuses to raise the dynamic LDS of a kernel (here a
    stand-in does, and launches nothing that asks for more than 64 KB), the
    column kernels keep within that and return the same fields, up to 512
    levels."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    (tmp_path / "s.c").write_text(_RUNTIME)
    (tmp_path / "run.py").write_text(_REFUSED)
    stub = str(tmp_path / "s.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", stub, str(tmp_path / "s.c"), "-ldl"], check=True)
    got = []
    for args in ([str(tmp_path / "a.npz")], [str(tmp_path / "b.npz"), stub]):
        r = subprocess.run([sys.executable, str(tmp_path / "run.py"), *args], cwd=root, capture_output=True, text=True,
                           timeout=100, env={**os.environ, "PYTHONPATH": root})
        assert r.returncode == 0, r.stderr[-2000:]
        got.append(np.load(args[0]))
    for k in got[0].files:
        assert np.array_equal(got[0][k], got[1][k]), k
