"""Child process of test_host_alloc.py: drives the host code over the fake HIP
runtime (TMRX_LIB) and reports launches and copies that touch memory which is
not live."""
import ctypes as C
import sys

import numpy as np

from tmr_amd import _lib, solver, workloads

L = _lib.lib()


def violations():
    buf = C.create_string_buffer(2048)
    n = L.fake_bad(buf, 2048)
    return n, buf.value.decode()


def expect_clean(what):
    n, text = violations()
    assert n == 0, "%s: %d violations\n%s" % (what, n, text)


def quiet(fn, *args):
    """fn(*args); solutions mean nothing here, so that a solve may end above
    its tolerance."""
    try:
        fn(*args)
    except _lib.TmrxError as e:
        if "did not converge" not in str(e):
            raise


def mesh():
    return workloads.adaptive(seed=5, base_level=1, max_level=2, nlevels=2)


def solve(p, **kw):
    f = np.ones(p.ndof)
    quiet(p.solve, f, None, solver.default_opts(max_iters=3, **kw))


def matrix_filter(p):
    h = C.c_void_p()
    if not hasattr(p, "filt"):
        _lib.check(L.tmrx_filter_create(p.forests[0].ptr, 1, 0.1, 3, 0, C.byref(h)), "filter")
        p.filt = h
    x = np.ones(int(p.forests[0].getNodeRange()[1]) * 3)
    out = np.zeros_like(x)
    for nv in (1, 3):
        _lib.check(L.tmrx_filter_apply(p.filt, nv, C.c_void_p(x.ctypes.data),
                                       C.c_void_p(out.ctypes.data), 0), "apply")


def steps(nodes):
    """name -> call that reaches the allocations of one host path."""
    return {
        "solve": solve,
        "FP64 solve": lambda p: solve(p, precision=0),
        "three cases": lambda p: quiet(p.solve_multi, np.ones((3, p.ndof)), None,
                                       solver.default_opts(max_iters=3)),
        "degree": lambda p: solve(p, cheb_degree=4),
        "nodal design": lambda p: (p.set_design_nodal(np.full(nodes, 0.5)), solve(p)),
        "Galerkin": lambda p: (p.set_multigrid(use_galerkin=True), solve(p)),
        "SOR": lambda p: (p.set_multigrid(use_chebyshev_smoother=False), solve(p)),
        "matrix cores": lambda p: (p.set_fp32_form(1), solve(p)),
        "tiling": lambda p: (p.set_tiling(64), solve(p)),
        "autotune": lambda p: (p.autotune((64, 128), reps=1), solve(p)),
        "filter": matrix_filter,
    }


def use(p):
    """What a program does with a problem beside the call at hand."""
    for precision in (0, 1):
        p.apply(np.ones(p.ndof), precision=precision)
    p.setup()
    p.set_state(np.ones(p.ndof), np.ones(p.ndof))
    p.compliance()
    solve(p)


def allocation_failures(only):
    forests, rho, _ = mesh()
    nodes = int(forests[0].getNodeRange()[1])
    table = steps(nodes)
    count = {}

    def fresh(name):
        p = solver.Problem(forests, q=3.0, k0=1e-6, bcs=[("fixed", 7)])
        p.set_design(rho)
        if name not in ("solve", "FP64 solve"):
            solve(p)
        return p

    # what the kernels take when nothing fails
    L.fake_learn(1)
    for name, fn in table.items():
        p = fresh(name)
        a = L.fake_allocs()
        fn(p)
        count[name] = L.fake_allocs() - a
        fn(p)
        use(p)
        p.set_design(rho)
        use(p)
        solve(p, precision=0)
        expect_clean(name)
    L.fake_learn(0)
    for name in only or table:
        fn = table[name]
        failed = 0
        for k in range(1, count[name] + 1):
            p = fresh(name)
            L.fake_fail_in(k)
            try:
                fn(p)
            except _lib.TmrxError:
                failed += 1
            L.fake_fail_in(0)
            what = "%s, allocation %d of %d fails" % (name, k, count[name])
            expect_clean(what)
            # the problem is as usable as before the call, and the call
            # succeeds when it is made again
            use(p)
            expect_clean(what + ", problem used")
            fn(p)
            use(p)
            expect_clean(what + ", call repeated")
        print("%s: %d allocations, %d calls refused" % (name, count[name], failed), flush=True)
        assert failed > 0


def small_lds():
    """The default tiles get smaller until they fit."""
    forests, rho, _ = workloads.cube_l4(2)
    p = solver.Problem(forests, q=3.0, k0=1e-6, bcs=[("fixed", 7)])
    assert p.tile_info(0)[1] == 96
    L.fake_max_lds(9 * 1024)  # 96 nodes and their halo take 10,432 bytes, 64 take 8,320
    p = solver.Problem(forests, q=3.0, k0=1e-6, bcs=[("fixed", 7)])
    assert p.tile_info(0)[1] == 64
    p.set_design(rho)
    for precision in (0, 1):
        p.apply(np.ones(p.ndof), precision=precision)
    expect_clean("tiles in 9 KB")


if __name__ == "__main__":
    small_lds() if sys.argv[1:] == ["LDS"] else allocation_failures(sys.argv[1:])
