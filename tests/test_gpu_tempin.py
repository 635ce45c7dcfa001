"""The initial temperature (TEMPIN) where the species share one interval bound
(sums formed once) and where they do not (formed for every evaluation), against
the C oracle: the suite's bars for the initial temperature (1e-9) and after a
step (1e-10 max-norm, temperature 1e-12; mixed 1e-5), on a grid whose last
block is partial."""
import numpy as np
import pytest

from conftest import assert_state_close, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("bounds", ["shared", "uneven"])
def test_initial_temperature(bounds, precision, oracle_built):
    from pyoracle import Oracle
    from sengapy import case as C
    from sengapy.abi import Solver
    n = (23, 12, 13)
    print("tempin", bounds, precision, flush=True)
    c = C.h2_nscbc(n=n, length=tuple((m - 1) * 4.0e-5 for m in n), seed=5)
    if bounds == "uneven":
        for s in (0, 4, 8):
            c.tables.tinthi[0, s] = 900.0 + 50.0 * s
    s = Solver(c, precision=precision)
    s.set_timestep(0.2 * c.dump.tstep)
    s.upload(c.dump.state, 0.0)
    o = Oracle(c)
    o.set_timestep(0.2 * c.dump.tstep)
    o.set_state(c.dump.state, 0.0)
    run, T0, _, _ = s.download()
    assert np.array_equal(run, c.dump.state)
    assert rel_err(T0, o.get()[1]) < (1e-6 if precision else 1e-9)
    s.step(1)
    o.step(1)
    run, T, _, _ = s.download()
    ref, Tr, _, _ = o.get()
    tol, tol_T = (1e-5, 1e-5) if precision else (1e-10, 1e-12)
    assert_state_close(f"{bounds} precision {precision}", run, T, ref, Tr, tol, tol_T)
    s.close()
