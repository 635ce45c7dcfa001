"""The derivative passes at the edges of their 16 x 16 tiles: the smallest
grid, one point below, at and above a tile and two tiles, in every direction,
with all-edge and interior x tiles, against the C oracle.  Tolerances are the
suite's own bars: 1e-10 max-norm in FP64 (temperature 1e-12), 1e-5 in the
mixed form, after two steps."""
import numpy as np
import pytest

from conftest import assert_state_close

pytestmark = pytest.mark.gpu

H = 5.0e-3 / 127
SIZES = [(11, 11, 11), (16, 15, 17), (17, 32, 16), (31, 17, 33), (32, 16, 31), (33, 31, 12), (49, 33, 15)]


def _case(kind, n):
    from sengapy import case as C
    length = tuple((m - 1) * H for m in n)
    if kind == "duct":
        return C.h2_nscbc(n=n, length=length, seed=sum(n))
    if kind == "box":
        return C.h2_nscbc(n=n, length=length, seed=sum(n), periodic_x=True)
    return C.ch4_16sp_nscbc(n=n, length=tuple(2 * v for v in length), seed=sum(n), periodic_x=kind == "options_box")


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kind,sizes", [("duct", SIZES), ("box", SIZES), ("options", SIZES[:4]),
                                        ("options_box", SIZES[3:4])])
def test_pass_tiles_match_oracle(kind, sizes, precision, oracle_built):
    from pyoracle import Oracle
    from sengapy.abi import Solver
    for n in sizes:
        print("passes", kind, n, precision, flush=True)
        c = _case(kind, n)
        dt = 0.2 * c.dump.tstep
        s = Solver(c, precision=precision)
        s.set_timestep(dt)
        s.upload(c.dump.state, 0.0)
        s.step(2)
        run, T, _, _ = s.download()
        s.close()
        o = Oracle(c)
        o.set_timestep(dt)
        o.set_state(c.dump.state, 0.0)
        o.step(2)
        ref, Tr, _, _ = o.get()
        assert np.isfinite(run).all()
        tol, tol_T = (1e-5, 1e-5) if precision else (1e-10, 1e-12)
        assert_state_close(f"{kind} {n} precision {precision}", run, T, ref, Tr, tol, tol_T)
