"""sg_step lets each substage's register update (LINCOM) and inflow values
(BOUNDT) be formed by the next substage's point kernel; sg_substage does them
in the final kernel.  Both evaluate the same expressions on the same values,
so five substages and sg_end_step give bit for bit what sg_step gives: on
grids below and above the size where the cross-term kernel takes its larger
tiles, with inflow, periodic, with every transport option and radiation (which
read the whole stage register), with the mixed forms and with the adaptive
step's error register."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

H = 5.0e-3 / 127


def _case(kind, n):
    from sengapy import case as C
    length = tuple((m - 1) * H for m in n)
    if kind == "duct":
        return C.h2_nscbc(n=n, length=length, seed=3)
    if kind == "box":
        return C.h2_nscbc(n=n, length=length, seed=3, periodic_x=True)
    if kind == "cold":   # unburnt gas below the FP32 rate range
        return C.h2_nscbc(n=n, length=length, seed=3, Tu=180.0)
    return C.ch4_16sp_nscbc(n=n, length=tuple(2 * v for v in length), seed=3)


@pytest.mark.parametrize("kind,n,precision,adaptive", [
    ("duct", (21, 17, 15), 0, False), ("duct", (21, 17, 15), 0, True), ("duct", (21, 17, 15), 1, False),
    ("duct", (21, 17, 15), 2, False), ("box", (18, 25, 13), 0, False), ("box", (18, 25, 13), 1, True),
    ("cold", (24, 12, 12), 1, False), ("options", (24, 13, 12), 0, False), ("options", (24, 13, 12), 1, False),
    ("duct", (81, 83, 90), 0, False), ("box", (82, 81, 89), 1, False)])
def test_step_equals_substages(kind, n, precision, adaptive):
    from sengapy.abi import Solver
    print("step against substages", kind, n, precision, adaptive, flush=True)
    c = _case(kind, n)
    out = []
    for split in (False, True):
        s = Solver(c, precision=precision)
        s.set_timestep(0.1 * c.dump.tstep)
        if adaptive:
            s.set_adaptive(True)
        s.upload(c.dump.state, 0.0)
        if split:
            for _ in range(2):
                for r in range(1, 6):
                    s.substage(r)
                s.end_step()
        else:
            s.step(2)
        out.append(s.download() + (np.array(s.timestep()),))
        s.close()
    for name, a, b in zip(("registers", "temperature", "pressure", "rate", "time step"), *out):
        assert np.array_equal(a, b), f"{name}: {np.max(np.abs(a - b))}"
