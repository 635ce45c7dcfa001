"""Bounded rows of edge tiles only (one launch of the pass with x derivatives)
and split in edge and interior tiles (two), at the last size of the one form
and the first of the other, against the C oracle: 2 species (blocks of two
waves), 9 species and 16 species with every option (blocks of seven).
Tolerances are the suite's own bars: 1e-10 max-norm in FP64 (temperature
1e-12), 1e-5 in the mixed form, after one step."""
import numpy as np
import pytest

from conftest import assert_state_close

pytestmark = pytest.mark.gpu

H = 5.0e-3 / 127


def _case(kind, n):
    from sengapy import case as C
    length = tuple((m - 1) * H for m in n)
    if kind == "h2":
        return C.h2_nscbc(n=n, length=length, seed=n[2])
    if kind == "options":
        return C.ch4_16sp_nscbc(n=n, length=tuple(2 * v for v in length), seed=n[2])
    c = C.periodic_1step(n=n, length=4.0e-3, seed=n[2])   # the single-step flame, in a duct
    per = c.control.bc[2]
    c.control.bc = [(13, [1, 0, 0, 0], [5.0, 0.0, 0.0, 0.0]), (21, [0, 0, 0, 0], [1.0e5, 0.287, 1.0e-3, 0.0]),
                    per, per, per, per]
    c.control.urin = 5.0
    return c


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kind,n", [("onestep", (40, 24, 24)), ("onestep", (33, 32, 170)), ("onestep", (33, 32, 171)),
                                    ("h2", (33, 16, 170)), ("h2", (33, 16, 171)),
                                    ("options", (48, 11, 85)), ("options", (48, 11, 86))])
def test_edge_and_interior_tiles(kind, n, precision, oracle_built):
    from pyoracle import Oracle
    from sengapy.abi import Solver
    print("rows", kind, n, precision, flush=True)
    c = _case(kind, n)
    dt = 0.2 * c.dump.tstep
    o = Oracle(c)
    o.set_timestep(dt)
    o.set_state(c.dump.state, 0.0)
    o.step(1)
    ref, Tr, _, _ = o.get()
    assert np.isfinite(ref).all()
    s = Solver(c, precision=precision)
    s.set_timestep(dt)
    s.upload(c.dump.state, 0.0)
    s.step(1)
    run, T, _, _ = s.download()
    s.close()
    tol, tol_T = (1e-5, 1e-5) if precision else (1e-10, 1e-12)
    assert_state_close(f"{kind} {n} precision {precision}", run, T, ref, Tr, tol, tol_T)
