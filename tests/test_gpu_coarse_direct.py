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


# islands of material in void of k0 times the stiffness, next to floating, across
# the leaves of the substructured level and inside them: 675 dofs, one inverse of
# 11 blocks; 4,131 dofs, leaves and a separator
ISLANDS = {
    "across": (((0.6, 0.4, 0.4), (1.2, 0.6, 0.6), (1.6, 0.3, 0.5)), 0.26),
    "inside": (((0.3, 0.3, 0.3), (0.3, 0.8, 0.3), (1.5, 0.25, 0.8), (1.45, 0.8, 0.3)), 0.13),
}


@pytest.mark.parametrize("k0", [1e-6, 1e-9, 1e-12])
@pytest.mark.parametrize("where", list(ISLANDS))
@pytest.mark.parametrize("level", [2, 3])
def test_coarse_solve_with_floating_islands(level, where, k0):
    """The residual of a backward stable solve is a few roundings of |A| |x|,
    whatever the condition number (1 / k0 and more); a preconditioner that
    loses that is refused or useless there."""
    forests, _, _ = workloads.box(level=level, nlevels=1)
    pts, conn = forests[0].getPoints(), forests[0].getMeshConn()
    cen = pts[conn].mean(1)
    rho = np.full(len(conn), 1e-6)
    balls, half = ISLANDS[where]
    for c in balls:
        rho[(np.abs(cen - c) < half).all(1)] = 1.0
    prob = solver.Problem(forests, q=Q, k0=k0, bcs=[("fixed", 7)])
    prob.set_design(rho)
    opts = solver.default_opts(precision=0)
    prob.setup(opts)
    orc = po.from_forest(forests[0], [("fixed", 7)])
    orc.assemble(rho ** Q + k0)
    norm = 2.0  # largest eigenvalue of a unit cube's mesh of E = 1, about
    rng = np.random.default_rng(level)
    for k in range(4):
        b = rng.standard_normal(prob.ndof)
        for _ in range(k):  # right-hand sides of ever smoother solutions
            x = prob.mg_op("coarse", 0, prob.mg_op("coarse", 0, b, opts)[0], opts)[0]
            b = orc.matvec(x)
            b /= np.linalg.norm(b)
        x, _ = prob.mg_op("coarse", 0, b, opts)
        eta = (np.linalg.norm(orc.matvec(x) - b) /
               (norm * np.linalg.norm(x) + np.linalg.norm(b)))
        print("level %d, islands %s, k0 %.0e: right-hand side %d, backward error %.2e"
              % (level, where, k0, k, eta), flush=True)
        assert eta < 1e-15
