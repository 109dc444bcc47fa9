"""The coarsest level's direct solve: batched block inverses (whole components
below 2,048 dofs) and substructured components above, against a dense FP64
solve with the oracle's operator."""
import numpy as np
import pytest

from oracle import pyoracle as po
from tmr_amd import solver, workloads

pytestmark = pytest.mark.gpu

Q, K0 = 3.0, 1e-6

# elements per edge of independent cubes; dofs 3 (n + 1)^3
CASES = {
    "one block, padded": [1],              # 24 of 64 rows
    "exact block": [3],                    # 192 = 3 * 64 rows
    "ragged": [4],                         # 375 rows, 6 blocks, 9 padding rows
    "several sizes": [1, 2, 4, 3],         # matrices leave the batch at different steps
    "largest inverse": [7],                # 1,536
    "substructured": [8],                  # 2,187
    "mixed": [2, 9, 3, 8],                 # both kinds side by side
}


@pytest.mark.parametrize("name", list(CASES))
def test_coarse_solve_against_dense(name):
    edges = CASES[name]
    forests, rho = workloads.uneven_cube_batch(edges, nlevels=1, seed=4)
    prob = solver.Problem(forests, q=Q, k0=K0, bcs=[("fixed", 7)])
    prob.set_design(rho)
    orc = po.from_forest(forests[0], [("fixed", 7)])
    orc.assemble(rho ** Q + K0)
    n = prob.ndof
    b = np.random.default_rng(1).standard_normal(n)
    # FP64: the residual of a backward stable solve grows with the condition
    # number (below 1e5 here).  FP32 V-cycles read the factors rounded to
    # 2^-24; the error against the FP64 solve is that times the condition of
    # the parts.
    x64, _ = prob.mg_op("coarse", 0, b, opts=solver.default_opts(precision=0))
    r = np.linalg.norm(orc.matvec(x64) - b) / np.linalg.norm(b)
    x32, _ = prob.mg_op("coarse", 0, b, opts=solver.default_opts(precision=1))
    e = np.linalg.norm(x32 - x64) / np.linalg.norm(x64)
    print("%s: %d dofs, residual %.2e, FP32 against FP64 %.2e" % (name, n, r, e), flush=True)
    assert r < 1e-10
    assert e < 1e-5
    # several right-hand sides: the batched solve equals the single one
    f = prob.traction_load("load", [0.3, -0.2, -1.0])
    o = solver.default_opts(rtol=1e-12, precision=0)
    U = prob.solve_multi(np.stack([f, 2.0 * f, b]), opts=o)
    u = prob.solve(f, opts=o)
    assert np.array_equal(U[0], u) and prob.info.iters <= 2
