"""External force of nodes with many load items: the device takes 32 items of a node at a time and adds them in input
order, so the counts around 32 and 64 are the edges.  Bitwise against the oracle, whose sums run in the same order with
the same FP64 operations (no contraction)."""
import numpy as np
import pytest

import mps_gpu as G
import oracle_ctypes as O
from meshgen import box, clamp_and_pull, perturb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tet", [False, True])
@pytest.mark.parametrize("n", [1, 31, 32, 33, 64, 65])
def test_item_counts(n, tet):
    m = perturb(box(4, 3, 3, tet=tet), 0.05, 9)
    rng = np.random.default_rng(n)
    node, other = m["n_nodes"] - 6, m["n_nodes"] - 1  # on the top face, inside and at a corner
    blocks = [("force", [node], rng.normal(size=(1, 3)), 0.0, 1.0) for _ in range(n // 2)]
    e = np.arange(m["n_elem"] - 6, m["n_elem"], dtype=np.int32)
    blocks.append(("traction_ramp", (0.3, -0.2, 1.0), 0.0, 2.0, e, np.full(e.size, 2, np.int32)))
    blocks += [("force", [node, other], rng.normal(size=(2, 3)), 0.1, 0.9) for _ in range(n - n // 2)]
    dd, dv = clamp_and_pull(m)
    op = O.OracleProblem(m, dir_dof=dd, dir_val=dv, n_steps=1, loads=blocks)
    with G.Solver(m, dir_dof=dd, dir_val=dv, n_steps=1) as s:
        s.set_loads(loads=blocks)
        for t in (0.05, 0.5, 1.5):
            assert np.array_equal(s.external_force(t), op.external_force(t)), t
