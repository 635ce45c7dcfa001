"""A batch whose launches hold many more blocks than any member's own: every
member still equals its solo run bit for bit (needs the GPU)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(64, 48, 48), (48, 64, 40), (80, 40, 40), (64, 56, 32), (40, 48, 48)]   # 609 tiles of 16 x 8 x 8


@pytest.mark.parametrize("kind,precision", [("nscbc", 0), ("nscbc", 1), ("kernel", 0), ("kernel", 1)])
def test_large_batch_matches_alone(kind, precision):
    from sengapy import case as C
    from sengapy.abi import Batch, Solver
    specs = C.batch_specs(len(SHAPES), seed=7) if kind == "nscbc" else C.kernel_specs(len(SHAPES), seed=7)
    cases = []
    for s, n in zip(specs, SHAPES):
        s["n"] = n
        cases.append(C.make_case(s))
    print("large batch", kind, precision, SHAPES, flush=True)

    def solver(c):
        s = Solver(c, precision=precision)
        s.set_timestep(c.dump.tstep)
        s.upload(c.dump.state, 0.0)
        return s

    ref = []
    for c in cases:
        s = solver(c)
        s.step(1)
        ref.append(s.download()[:3])
        s.close()
    b = Batch()
    sol = [solver(c) for c in cases]
    for s in sol:
        b.add(s)
    b.step(1)
    b.sync()
    for q, s in enumerate(sol):
        for name, a, r in zip(("registers", "temperature", "pressure"), s.download()[:3], ref[q]):
            assert np.array_equal(a, r), f"member {q} {name} differ"
    b.close()
