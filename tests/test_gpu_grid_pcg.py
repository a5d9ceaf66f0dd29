"""The resident-grid PCG (every solve of a system that fits it) on systems with known solutions, each test beside the
two-kernel iteration where both serve it.

Sizes at its edges: fewer nodes than work-groups, one block per thread, blocks in registers, in LDS and in
memory, rows of hundreds of blocks, several work-group counts; Schwarz and Jacobi; limits below, at and
above one launch's iterations (a solve then spans launches). Both sides solve to a relative residual of
1e-13 of the same matrix, whose Jacobi-scaled condition number is at most about 1e4 (mass-dominated
systems), so the solutions agree to 1e-13 * 1e4 = 1e-9.
"""

import numpy as np
import pytest

import oracle as O
from higher_order_embedded_fem_amd import scenes

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def system(sc, stiff):
    om = O.Model(sc)
    mu, lam = scenes.lame_from_young_poisson(sc.young, sc.poisson)
    rp, col = om.pattern()
    K = om.stiffness_add(mu, lam, np.zeros(sc.ndof), np.zeros(om.nnz))
    return rp, col, O.dirichlet_csr(rp, col, (0.0 + stiff * K) + 1.0 * om.mass(sc.density), sc.dirichlet_nodes)


def product(rp, col, A, x):
    y = A * x[col]
    return np.add.reduceat(np.concatenate([y, [0.0]]), rp[:-1])


CASES = [("cube", 1, scenes.TET4, "element"), ("cube", 1, scenes.TET10, "element"), ("cube", 2, scenes.TET10, "patches"),
         ("cube", 5, scenes.TET10, "element"), ("cube", 6, scenes.TET10, "patches"), ("cube", 8, scenes.TET10, "patches"),
         ("cube", 12, scenes.TET10, "element"), ("cube", 16, scenes.TET10, "element"), ("cube", 30, scenes.TET4, "element")]


@pytest.mark.parametrize("schwarz", [True, False])
@pytest.mark.parametrize("mesh,cells,element,subdomains", CASES)
def test_solution_matches_a_converged_residual(mesh, cells, element, subdomains, schwarz):
    from higher_order_embedded_fem_amd import fem

    sc = scenes.cube_scene(cells, element, schwarz=subdomains)
    rp, col, J = system(sc, 1e-5)
    gm = fem.ElasticityModel(sc)
    Jd = torch.as_tensor(J, device="cuda")
    pre = None
    if schwarz:
        pre = fem.SchwarzPreconditioner.from_scene(gm, sc)
        pre.update(Jd)
    rng = np.random.default_rng(cells)
    x_true = rng.standard_normal(sc.ndof)
    b = torch.as_tensor(product(rp, col, J, x_true), device="cuda")
    start = torch.as_tensor(rng.standard_normal(sc.ndof), device="cuda")
    x = start.clone()
    its, st = fem.conjugate_gradient(gm, Jd, b, x, pre, tol=1e-13, max_iter=20000)
    assert st == 0 and its > 0
    assert np.linalg.norm(x.cpu().numpy() - x_true) <= 1e-9 * np.linalg.norm(x_true)
    assert gm.resident_solver_stats() == (1, 0)
    again = start.clone()  # the same launches: the same bits
    assert fem.conjugate_gradient(gm, Jd, b, again, pre, tol=1e-13, max_iter=20000) == (its, 0)
    assert torch.equal(x, again)
    gm.set_resident_solver(False)
    x = start.clone()
    _, st = fem.conjugate_gradient(gm, Jd, b, x, pre, tol=1e-13, max_iter=20000)
    assert st == 0 and gm.resident_solver_stats() == (2, 0)
    assert np.linalg.norm(x.cpu().numpy() - x_true) <= 1e-9 * np.linalg.norm(x_true)


# (the two kernels' launches are batches of 8 iterations; 2300 is the resident grid's third launch)
@pytest.mark.parametrize("limit,resident", [(n, r) for r in (True, False) for n in (0, 1, 1023, 1024, 1025)] + [(2300, True)])
def test_iteration_limits_across_launches(limit, resident):
    """A solve whose tolerance is never met stops at its limit, whether or not the limit is a launch's end; limits
    past a launch continue the same iteration: the iterate at 1025 is one step from the one at 1024."""
    from higher_order_embedded_fem_amd import fem

    sc = scenes.cube_scene(3, scenes.TET10)
    _, _, J = system(sc, 1.0)
    gm = fem.ElasticityModel(sc)
    gm.set_resident_solver(resident)
    Jd = torch.as_tensor(J, device="cuda")
    pre = fem.SchwarzPreconditioner.from_scene(gm, sc)
    pre.update(Jd)
    b = torch.as_tensor(np.random.default_rng(4).standard_normal(sc.ndof), device="cuda")
    x = torch.zeros_like(b)
    its, st = fem.conjugate_gradient(gm, Jd, b, x, pre, tol=0.0, max_iter=limit)
    # with tolerance 0 the iteration goes on after x has converged; p.Ap can then underflow to 0, which ends the
    # solve as an indefinite operator (status 6) before the limit
    assert (its, st) == (limit, 5) or (limit == 2300 and st == 6 and its > 1025)
    assert gm.resident_solver_stats() == (int(resident), 0)
    assert bool(torch.isfinite(x).all())
    if limit == 0:
        assert not x.any()
        return
    r = b - gm.spmv(Jd, x)
    full = torch.zeros_like(b)
    fem.conjugate_gradient(gm, Jd, b, full, pre, tol=1e-13, max_iter=5000)
    rel = float((x - full).norm() / full.norm())
    assert rel < (1.0 if limit == 1 else 1e-9)
    assert float(r.norm()) < float(b.norm())


def test_fp32_operator_matches_the_fp64_step():
    """The FP32 operator inside the FP64 Newton loop (modes 1, 2, 3) reaches the FP64 step's solution, in either
    iteration: both Newton loops stop at 1e-11 of the representative force, and the cube's Jacobian is well conditioned."""
    from higher_order_embedded_fem_amd import fem

    sc = scenes.cube_scene(7, scenes.TET10)
    ref = None
    for mode, resident in ((0, True), (1, True), (2, True), (3, True), (0, False), (1, False), (2, False), (3, False)):
        gm = fem.ElasticityModel(sc)
        gm.set_resident_solver(resident)
        sim = fem.NewtonCgIntegrator(gm, sc, newton_tolerance_factor=1e-11, cg_tolerance=1e-7, cg_max_iter=5000,
                                     mixed_precision=mode)
        u = torch.zeros(sc.ndof, dtype=torch.float64, device="cuda")
        v = torch.zeros_like(u)
        sim.step(0.0, sc.dt, u, v)
        solves, failures = gm.resident_solver_stats()
        assert (solves > 0) == resident and failures == 0
        if ref is None:
            ref = u.clone()
        else:
            assert float((u - ref).norm() / ref.norm()) < 1e-8
