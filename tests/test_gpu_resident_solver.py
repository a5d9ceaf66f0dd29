"""Which systems the resident-grid PCG may take, and what becomes of the others."""

import ctypes as C
import dataclasses

import numpy as np
import pytest

import oracle as O
from higher_order_embedded_fem_amd import _lib, scenes

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def dev(x):
    return torch.as_tensor(np.ascontiguousarray(x), dtype=torch.float64, device="cuda")


def matrix(sc, stiff=1e-5):
    om = O.Model(sc)
    mu, lam = scenes.lame_from_young_poisson(sc.young, sc.poisson)
    rp, col = om.pattern()
    K = om.stiffness_add(mu, lam, np.zeros(sc.ndof), np.zeros(om.nnz))
    return rp, col, O.dirichlet_csr(rp, col, (0.0 + stiff * K) + 1.0 * om.mass(sc.density), sc.dirichlet_nodes)


def system(sc, seed):
    """The scene's matrix M + 1e-5 K on the device, a solution and its right-hand side."""
    rp, col, J = matrix(sc)
    x = np.random.default_rng(seed).standard_normal(sc.ndof)
    y = J * x[col]
    return dev(J), x, dev(np.add.reduceat(np.concatenate([y, [0.0]]), rp[:-1]))


def thinned(sc):
    """The scene without every other element that its nodes can spare: the same nodes, fewer couplings."""
    count = np.bincount(sc.connectivity.ravel(), minlength=sc.num_vertices)
    keep = np.ones(sc.num_elements, bool)
    for e in range(0, sc.num_elements, 2):
        if (count[sc.connectivity[e]] > 1).all():
            count[sc.connectivity[e]] -= 1
            keep[e] = False
    conn = np.ascontiguousarray(sc.connectivity[keep])
    off = np.arange(0, conn.size + 1, conn.shape[1], dtype=np.int64)
    return dataclasses.replace(sc, connectivity=conn, num_interior=len(conn), subdomain_offsets=off,
                               subdomain_nodes=conn.ravel().astype(np.int32),
                               untreated_nodes=np.zeros(0, np.int32))


# Both directions: rows shorter and longer than the preconditioner's model has them. The solve's residual of 1e-13
# times the mass-dominated matrix's condition (Jacobi-scaled at most about 1e4) bounds the error by 1e-9.
@pytest.mark.parametrize("cells,element", [(3, scenes.TET10), (9, scenes.TET4)])
@pytest.mark.parametrize("own_thinned", [False, True])
@pytest.mark.parametrize("entry", ["hoefem_pcg", "hoefem_pcg_noalloc"])
def test_preconditioner_of_another_model_on_the_same_nodes(cells, element, own_thinned, entry):
    from higher_order_embedded_fem_amd import fem

    full = scenes.cube_scene(cells, element)
    part = thinned(full)
    assert part.num_elements < 0.8 * full.num_elements
    own, other = (part, full) if own_thinned else (full, part)
    Jd, x_true, b = system(own, cells)
    gm, gother = fem.ElasticityModel(own), fem.ElasticityModel(other)
    pre = fem.SchwarzPreconditioner.from_scene(gother, other)
    pre.update(dev(matrix(other)[2]))
    solve = getattr(_lib.load(), entry)
    x, its = torch.zeros_like(b), C.c_int64()
    assert solve(gm.h, Jd.data_ptr(), pre.h, b.data_ptr(), x.data_ptr(), 1e-13, 20000, C.byref(its)) == 0
    assert np.linalg.norm(x.cpu().numpy() - x_true) <= 1e-9 * np.linalg.norm(x_true)


@pytest.mark.parametrize("entry", ["hoefem_pcg", "hoefem_pcg_noalloc"])
def test_preconditioner_of_another_size_is_refused(entry):
    from higher_order_embedded_fem_amd import fem

    small, large = scenes.cube_scene(2, scenes.TET10), scenes.cube_scene(3, scenes.TET10)
    Jd, _, b = system(large, 1)
    gm, gsmall = fem.ElasticityModel(large), fem.ElasticityModel(small)
    pre = fem.SchwarzPreconditioner.from_scene(gsmall, small)
    L = _lib.load()
    x, its = torch.zeros_like(b), C.c_int64()
    assert getattr(L, entry)(gm.h, Jd.data_ptr(), pre.h, b.data_ptr(), x.data_ptr(), 1e-8, 10, C.byref(its)) == 1
    assert b"nodes" in L.hoefem_last_error()


@pytest.mark.parametrize("schwarz", [False, True])
def test_sims_of_one_model_in_one_batch(schwarz):
    """Sims that share a model are in flight together: each ends where it ends alone, bit for bit."""
    from higher_order_embedded_fem_amd import fem

    sc = scenes.cube_scene(4, scenes.TET10)
    gm = fem.ElasticityModel(sc)
    sims = [fem.NewtonCgIntegrator(gm, sc, schwarz=schwarz, newton_tolerance_factor=1e-6, cg_max_iter=5000)
            for _ in range(4)]
    rng = np.random.default_rng(7)
    v0 = 0.2 * rng.standard_normal((len(sims), sc.ndof))
    v0.reshape(len(sims), -1, 3)[:, sc.dirichlet_nodes] = 0.0
    state = [(torch.zeros(sc.ndof, dtype=torch.float64, device="cuda"), dev(v)) for v in v0]
    alone = []
    for sim, (u, v) in zip(sims, state):
        ua, va = u.clone(), v.clone()
        for i in range(2):
            sim.step(i * sc.dt, sc.dt, ua, va)
        alone.append((ua, va))
    L, n = _lib.load(), len(sims)
    h = C.c_void_p()
    _lib.check(L.hoefem_batch_create((C.c_void_p * n)(*[s.h.value for s in sims]), n, C.byref(h)))
    us, vs = (C.c_void_p * n)(*[u.data_ptr() for u, _ in state]), (C.c_void_p * n)(*[v.data_ptr() for _, v in state])
    for _ in range(2):
        _lib.check(L.hoefem_batch_step(h, (C.c_double * n)(*[sc.dt] * n), us, vs, None, None, None))
    L.hoefem_batch_destroy(h)
    for (u, v), (ua, va) in zip(state, alone):
        assert torch.equal(u, ua) and torch.equal(v, va)


# With a poll limit of 0 every launch ends at once, unfinished, as one does whose work-groups cannot all become
# resident. Its solve is the two-kernel iteration's, bit for bit, and so are the 64 after it.
@pytest.mark.parametrize("schwarz", [True, False])
@pytest.mark.parametrize("entry", ["hoefem_pcg", "hoefem_pcg_noalloc"])
def test_launch_that_gives_up(entry, schwarz):
    from higher_order_embedded_fem_amd import fem

    sc = scenes.cube_scene(5, scenes.TET10)
    Jd, x_true, b = system(sc, 3)
    L = _lib.load()
    results = {}
    for way in ("kernels", "gives_up"):
        gm = fem.ElasticityModel(sc)
        pre = None
        if schwarz:
            pre = fem.SchwarzPreconditioner.from_scene(gm, sc)
            pre.update(Jd)

        def solve():
            x, its = torch.zeros_like(b), C.c_int64()
            assert getattr(L, entry)(gm.h, Jd.data_ptr(), pre.h if pre else None, b.data_ptr(), x.data_ptr(), 1e-13,
                                     20000, C.byref(its)) == 0
            assert np.linalg.norm(x.cpu().numpy() - x_true) <= 1e-9 * np.linalg.norm(x_true)
            return its.value, x

        gm.set_resident_solver(enable=way != "kernels", poll_limit=0)
        results[way] = solve()
        if way == "kernels":
            assert gm.resident_solver_stats() == (0, 0)
            continue
        assert results[way][0] == results["kernels"][0] and torch.equal(results[way][1], results["kernels"][1])
        assert gm.resident_solver_stats() == (0, 1)
        gm.set_resident_solver(poll_limit=-1)
        for _ in range(64):
            solve()
        assert gm.resident_solver_stats() == (0, 1)
        solve()
        assert gm.resident_solver_stats() == (1, 1)
        gm.set_resident_solver(poll_limit=0)  # the count starts again at the first failure after a good launch
        solve()
        gm.set_resident_solver(poll_limit=-1)
        for _ in range(65):
            solve()
        assert gm.resident_solver_stats() == (2, 2)


@pytest.mark.parametrize("precision", [0, 1])
def test_batch_launch_that_gives_up(precision):
    """Scenes whose launch gives up in the middle of a step, and those that rest after it, end where the two-kernel
    iteration takes them; a scene beside them keeps the resident grid."""
    from higher_order_embedded_fem_amd import batch

    scs = [scenes.cube_scene(c, scenes.TET10) for c in (3, 4, 5)]
    kw = dict(newton_tolerance_factor=1e-6, mixed_precision=precision, autotune=False)
    ref, st = batch.BatchedStepper(scs, **kw), batch.BatchedStepper(scs, **kw)
    for k in (0, 1):
        ref.models[k].set_resident_solver(enable=False)
        st.models[k].set_resident_solver(poll_limit=0)
    for _ in range(3):
        a, b = ref.step(), st.step()
        assert a["status"] == b["status"] == [0, 0, 0]
        assert [s["cg_iterations"] for s in a["stats"]] == [s["cg_iterations"] for s in b["stats"]]
    torch.cuda.synchronize()
    for k in range(3):
        assert torch.equal(ref.u[k], st.u[k]) and torch.equal(ref.v[k], st.v[k])
    for k in (0, 1):
        assert ref.models[k].resident_solver_stats() == (0, 0) and st.models[k].resident_solver_stats() == (0, 1)
    solves = st.models[2].resident_solver_stats()
    assert solves == ref.models[2].resident_solver_stats() and solves[0] >= 3 and solves[1] == 0


def two_jacobi_steps(rp, col, J, diag, b):
    """x after two iterations of Jacobi-preconditioned CG from zero, in FP64."""
    x, r = np.zeros_like(b), b.copy()
    z = r / diag
    p, ztr = z.copy(), z @ r
    for _ in range(2):
        ap = np.add.reduceat(np.append(J * p[col], 0.0), rp[:-1])
        alpha = ztr / (p @ ap)
        x += alpha * p
        r -= alpha * ap
        z = r / diag
        ztr, old = z @ r, ztr
        p = z + ztr / old * p
    return x


# The second iterate holds the rounding of one product of the FP32 operator. Both iterations round its operands alike;
# the resident grid rounds once per 3x3 block and row, the two kernels once per block and then along their lanes' sums.
@pytest.mark.parametrize("cells,element", [(5, scenes.TET10), (12, scenes.TET10), (15, scenes.TET10), (24, scenes.TET4)])
def test_fp32_products_are_no_less_accurate_than_the_two_kernels(cells, element):
    from higher_order_embedded_fem_amd import fem

    sc = scenes.cube_scene(cells, element)
    gm = fem.ElasticityModel(sc)
    sim = fem.NewtonCgIntegrator(gm, sc, schwarz=False, cg_tolerance=1e-15, cg_max_iter=2, mixed_precision=3)
    zero = torch.zeros(sc.ndof, dtype=torch.float64, device="cuda")
    sim.set_state(0.0, zero, zero)
    sim.init_solve_jacobian_combination(-sc.dt * sc.dt, None)
    b = np.random.default_rng(cells).standard_normal(sc.ndof)
    b.reshape(-1, 3)[sc.dirichlet_nodes] = 0.0
    error = {}
    for enable in (False, True):
        gm.set_resident_solver(enable=enable)
        sol = torch.zeros_like(zero)
        assert sim.solve_jacobian_combination(sol, dev(b)) == 2
        if not error:
            rp, col = gm.pattern()
            J = sim.jacobian().cpu().numpy()  # the FP32 values
            rows = np.repeat(np.arange(sc.ndof), np.diff(rp))
            exact = two_jacobi_steps(rp, col, J, J[rows == col], b)
        error[enable] = np.linalg.norm(sol.cpu().numpy() - exact) / np.linalg.norm(exact)
    assert gm.resident_solver_stats() == (1, 0)
    print(f"two kernels {error[False]:.2e}, resident grid {error[True]:.2e}")
    assert error[True] <= error[False] < 1e-6
