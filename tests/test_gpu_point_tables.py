"""The point kernels' coefficient tables, read a group ahead: waves whose points
all lie in one temperature interval (unburnt gas above the interval bound) and
waves that hold both, one or several interval bounds, and pair, row and species
counts that fill no whole group, for 9 and 16 species, against the C oracle
after one step at the suite's bars (1e-10 max-norm, temperature 1e-12; mixed
1e-5), on grids whose last block is partial."""
import numpy as np
import pytest

from conftest import assert_state_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kind", ["both", "upper", "uneven", "options"])
def test_point_tables(kind, precision, oracle_built):
    from pyoracle import Oracle
    from sengapy import case as C
    from sengapy.abi import Solver
    n = (24, 12, 13)
    length = tuple((m - 1) * 4.0e-5 for m in n)
    print("point tables", kind, precision, flush=True)
    if kind == "options":
        c = C.ch4_16sp_nscbc(n=n, length=tuple(2 * v for v in length), seed=7)
    else:
        c = C.h2_nscbc(n=n, length=length, seed=7, **({"Tu": 1150.0} if kind == "upper" else {}))
    if kind == "uneven":
        for s in (1, 3):
            c.tables.tinthi[0, s] = 950.0 + 20.0 * s
    out = []
    for r in (Solver(c, precision=precision), Oracle(c)):
        r.set_timestep(0.2 * c.dump.tstep)
        if isinstance(r, Solver):
            r.upload(c.dump.state, 0.0)
            r.step(1)
            out.append(r.download())
            r.close()
        else:
            r.set_state(c.dump.state, 0.0)
            r.step(1)
            out.append(r.get())
    (run, T, _, _), (ref, Tr, _, _) = out
    if kind == "upper":
        assert np.min(Tr) > 1000.0
    tol, tol_T = (1e-5, 1e-5) if precision else (1e-10, 1e-12)
    assert_state_close(f"{kind} precision {precision}", run, T, ref, Tr, tol, tol_T)
