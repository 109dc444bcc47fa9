"""Owner tiles over their sizes and FP32 operator forms: the product against
the oracle's FP64 operator on forests with and without hanging nodes."""
import numpy as np
import pytest

from oracle import pyoracle as po
from tmr_amd import solver, workloads

pytestmark = pytest.mark.gpu

Q, K0 = 3.0, 1e-6


@pytest.fixture(scope="module")
def meshes():
    out = {}
    for name, (forests, rho, _) in (
            ("adaptive", workloads.adaptive(seed=5, base_level=2, max_level=4, nlevels=2)),
            ("cube", workloads.cube_l4(2))):
        orc = po.from_forest(forests[0], [("fixed", 7)])
        orc.assemble(rho ** Q + K0)
        prob = solver.Problem(forests, q=Q, k0=K0, bcs=[("fixed", 7)])
        prob.set_design(rho)
        x = np.random.default_rng(3).standard_normal(prob.ndof)
        out[name] = (prob, x, orc.matvec(x))
    return out


# 64: many small tiles; 100: ends inside a wave; 512: several rounds per
# thread; 800: tiles of 512 threads
@pytest.mark.parametrize("tile", [0, 64, 100, 512, 800])
@pytest.mark.parametrize("name", ["adaptive", "cube"])
def test_product_over_tile_sizes_and_forms(name, tile, meshes):
    prob, x, ref = meshes[name]
    if tile:
        prob.set_tiling(tile)
    print(name, tile, prob.tile_info(0), flush=True)
    # FP64 to rounding; plain FP32 sums of about 80 terms; three bf16 parts
    # keep 24 bits of each operand but drop products below 2^-16
    for form, precision, bound in ((0, 0, 1e-13), (0, 1, 1e-5), (1, 1, 1e-4), (2, 1, 1e-5)):
        prob.set_fp32_form(form)
        y = prob.apply(x, precision=precision)
        e = np.linalg.norm(y - ref) / np.linalg.norm(ref)
        print("  form %d precision %d: %.2e" % (form, precision, e), flush=True)
        assert e < bound
    prob.set_fp32_form(0)


@pytest.mark.parametrize("precision", [0, 1])
def test_product_in_place_and_overlapping_vectors(precision, meshes):
    """Device vectors are used in place; y on top of x, or overlapping it,
    gives the same values."""
    import torch
    prob, x, ref = meshes["adaptive"]
    n = prob.ndof
    buf = torch.zeros(2 * n, dtype=torch.float64, device="cuda")
    want = torch.from_numpy(prob.apply(x, precision=precision)).cuda()
    for a, b in ((0, n), (n, 0), (0, 0), (0, n // 2), (n // 2 + 1, 0)):
        buf.zero_()
        src, dst = buf[a:a + n], buf[b:b + n]
        src.copy_(torch.from_numpy(x))
        prob.apply(src, precision=precision, y=dst)
        assert torch.equal(dst, want), (a, b)
        if a + n <= b or b + n <= a:
            assert np.array_equal(src.cpu().numpy(), x)


@pytest.mark.parametrize("tile", [0, 200])
def test_failed_autotune_keeps_the_tiles(tile):
    """Candidates that do not fit in LDS (4096 owned nodes take 196 KB for x
    and the accumulators alone): the tiles, the operator form and the solution
    stay what they were."""
    from tmr_amd._lib import TmrxError
    forests, rho, _ = workloads.box(level=4, nlevels=3, seed=1)
    prob = solver.Problem(forests, q=Q, k0=K0, bcs=[("fixed", 7)])
    prob.set_design(rho)
    if tile:
        prob.set_tiling(tile)
    keep = [prob.tile_info(l) for l in range(3)], prob.tuning()
    f = prob.traction_load("load", [0.0, 0.2, -1.0])
    u = prob.solve(f)
    for call in (lambda: prob.autotune((4096, 4000)), lambda: prob.set_tiling(4096)):
        with pytest.raises(TmrxError, match="fit"):
            call()
        assert ([prob.tile_info(l) for l in range(3)], prob.tuning()) == keep
        assert np.array_equal(prob.solve(f), u)


def test_default_tiles_of_rows_of_single_element_blocks():
    """2.2M nodes numbered row by row: the 1,024-node tiles of large uniform
    levels do not fit in LDS there."""
    from tmr_amd import TMR
    f = TMR.createBoxForest(1100, 44, 44, (1100.0, 44.0, 44.0), face_names=workloads.FACES)
    f.createTrees(0)
    f.createNodes()
    prob = solver.Problem([f], q=Q, k0=K0, bcs=[("fixed", 7)])
    tiles, size = prob.tile_info(0)
    print("%d tiles of %d nodes" % (tiles, size), flush=True)
    assert size == 512
    rng = np.random.default_rng(6)
    prob.set_design(rng.uniform(0.1, 1.0, prob.nelem))
    x = rng.standard_normal(prob.ndof)
    y = prob.apply(x, precision=0)
    y32 = prob.apply(x, precision=1)
    prob.set_tiling(200)
    ref = prob.apply(x, precision=0)
    # sums of about 80 terms a row in another order; FP32 operands and sums
    assert np.linalg.norm(y - ref) < 1e-14 * np.linalg.norm(ref)
    assert np.linalg.norm(y32 - ref) < 1e-5 * np.linalg.norm(ref)
