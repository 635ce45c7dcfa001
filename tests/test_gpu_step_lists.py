"""The table-driven step loop with lists longer than the packed record of a step
holds (4 reactants and products, 6 species) and at its lengths, forward and
reversible, against the C oracle after one step at the suite's bars (1e-10
max-norm, temperature 1e-12; mixed 1e-5)."""
import numpy as np
import pytest

from conftest import assert_state_close

pytestmark = pytest.mark.gpu


def _case(nr, nspec):
    from sengapy import case as C
    n = (24, 12, 13)
    c = C.h2_nscbc(n=n, length=tuple((m - 1) * 4.0e-5 for m in n), seed=11)
    m, t = c.mech, c.tables
    inert = len(m.species)   # nitrogen, the last species
    # two plain steps, made reversible, get nr reactants and products (padded
    # with nitrogen, whose concentration the pre-exponential factor makes up
    # for) and nspec species
    plain = [s for s in range(len(m.nsspec)) if not (m.mblist[s] or m.mllist[s] or m.mtlist[s] or m.mslist[s])]
    for s in plain[:2]:
        t.rparam[0][s] += 3.0 * (nr - len(m.nrspec[s]))
        m.nrspec[s] = (m.nrspec[s] + [inert] * 10)[:nr]
        m.npspec[s] = (m.npspec[s] + [inert] * 10)[:nr]
        for sp in range(1, len(m.species) + 1):
            if len(m.nsspec[s]) < nspec and sp not in m.nsspec[s]:
                m.nsspec[s].append(sp)
                m.diffmu[s].append(0.01 * (-1) ** sp)
                t.diffmw[s].append(m.diffmu[s][-1] * m.wmolar[sp - 1])
        m.mglist[s] = 1
    return c


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("nr,nspec", [(3, 5), (4, 6), (5, 7), (7, 9)])
def test_long_step_lists(nr, nspec, precision, oracle_built):
    from pyoracle import Oracle
    from sengapy.abi import Solver
    print("step lists", nr, nspec, precision, flush=True)
    c = _case(nr, nspec)
    s, o = Solver(c, precision=precision), Oracle(c)
    assert not s.mechanism_compiled()
    for r in (s, o):
        r.set_timestep(0.05 * c.dump.tstep)
    s.upload(c.dump.state, 0.0)
    o.set_state(c.dump.state, 0.0)
    s.step(1)
    o.step(1)
    run, T, _, _ = s.download()
    ref, Tr, _, _ = o.get()
    assert np.isfinite(ref).all()
    tol, tol_T = (1e-5, 1e-5) if precision else (1e-10, 1e-12)
    assert_state_close(f"lists {nr} {nspec} precision {precision}", run, T, ref, Tr, tol, tol_T)
    s.close()
