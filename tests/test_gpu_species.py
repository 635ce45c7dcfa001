"""More than nine species without the transport options, against the C oracle:
hydrogen-air whose nitrogen is split into 2 to 10 equal species (10 to 18 in
all), a mechanism read at run time.  13 and 17 species are the counts at which
the point kernels leave out fill-up rows of a step's lists (13 both in FP64,
one in the mixed form; 17 one in the mixed form).  Tolerances are the suite's
own bars: 1e-10 max-norm in FP64 (temperature 1e-12), 1e-5 in the mixed form,
after two steps."""
from types import SimpleNamespace

import numpy as np
import pytest

from conftest import assert_state_close

pytestmark = pytest.mark.gpu

N = (24, 12, 13)
PER_SPECIES = ("olewis", "wmolar", "ovwmol", "rgspec", "ntint", "ncpoly", "ncenth", "ncenpy", "tinthi", "amascp",
               "amasct", "amasch", "amolgb", "viscco", "condco")


def _split(ns):
    """(configuration, state, time step) with the last species in ns - 8 equal parts."""
    from sengapy import abi
    from sengapy import case as C
    c = C.h2_nscbc(n=N, length=tuple((m - 1) * 5.0e-3 / 127 for m in N), seed=ns)
    g = abi.config_from_case(c)
    last = g.nspec - 1
    for s in range(g.nspec, ns):
        for f in PER_SPECIES:
            getattr(g, f)[s] = getattr(g, f)[last]
        for b in range(abi.MAX_BODY):
            g.effy3b[b][s] = g.effy3b[b][last]
    of = [min(s, last) for s in range(ns)]
    for f in ("diffco", "wilko1", "wilko2"):
        a = np.ctypeslib.as_array(getattr(g, f))
        a[:ns, :ns] = a[np.ix_(of, of)].copy()
    parts = ns - last
    y = g.yrin[last] / parts
    for s in range(last, ns):
        g.yrin[s] = y
    g.nspec = ns
    q = np.concatenate([c.dump.state[:5 + last], np.repeat(c.dump.state[5 + last:] / parts, parts, axis=0)])
    return g, q, 0.1 * c.dump.tstep


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("ns", [10, 13, 16, 17, 18])
def test_species_counts_match_oracle(ns, precision, oracle_built, monkeypatch):
    import pyoracle
    from sengapy.abi import Solver
    print("species", ns, precision, flush=True)
    g, q, dt = _split(ns)
    case = SimpleNamespace(shape=N, nspec=ns)
    monkeypatch.setattr(pyoracle, "config_from_case", lambda _: g)
    o = pyoracle.Oracle(case)
    o.set_timestep(dt)
    o.set_state(q, 0.0)
    o.step(2)
    ref, Tr, _, _ = o.get()
    assert np.isfinite(ref).all()
    g.precision = precision
    s = Solver(case, cfg=g)
    assert not s.mechanism_compiled()
    s.set_timestep(dt)
    s.upload(q, 0.0)
    s.step(2)
    run, T, _, _ = s.download()
    s.close()
    tol, tol_T = (1e-5, 1e-5) if precision else (1e-10, 1e-12)
    assert_state_close(f"{ns} species precision {precision}", run, T, ref, Tr, tol, tol_T)
