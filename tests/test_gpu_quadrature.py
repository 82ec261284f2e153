"""GPU parity of the quadrature switches of advection_solver.cc:110-116
(:440-445): use_gl_quad (operator and mass matrix with QGaussLobatto(k+1))
and use_gl_quad_mass (mass matrix only), against the CPU oracle at 1e-12
relative in FP64. The oracle's two switches are pinned in test_oracle.py
(summation-by-parts known answer, closed-form Gauss-Lobatto inverse mass,
and the remassed Gauss apply)."""
import numpy as np
import pytest
import torch

from advection_miniapp_amd import AdvectionOperation, \
    LowStorageRungeKuttaIntegrator
from advection_miniapp_amd import _lib as L
from helpers import Cfg, nodal_points, rel_diff

pytestmark = pytest.mark.gpu

TOL = 1e-12

CASES = {
    # tabulated geometry (perturbed cells, cellular speed)
    "3d_k3_pert_cellular": dict(dim=3, degree=3, refine=2, perturbation=0.1,
                                velocity_kind=1),
    # uniform geometry (axis-aligned cells, constant speed)
    "3d_k4_cart_const": dict(dim=3, degree=4, refine=2,
                             velocity=[1.0, 0.5, 0.25]),
    # inflow Dirichlet faces, skew-symmetric form
    "3d_k2_dirichlet_skew": dict(dim=3, degree=2, n_coarse=[2, 1, 1],
                                 refine=1, periodic=[0, 1, 0],
                                 velocity=[1.1, 0.15, -0.05],
                                 solution_kind=1, factor_skew=0.5),
    # 2D, time-dependent vortex on perturbed cells
    "2d_k5_pert_vortex": dict(dim=2, degree=5, refine=3, perturbation=0.1,
                              velocity_kind=2, time_factor=1,
                              final_time=8.0),
    "3d_k7_cart": dict(dim=3, degree=7, refine=1, velocity=[-1, 0.5, 0.25]),
    # SIPG on perturbed cells (a kernel of its own: with use_gl_quad_mass in
    # integrate form before the inverse mass), axis-aligned cells
    "3d_k3_sipg_pert": dict(dim=3, degree=3, n_coarse=[3, 5, 3], refine=0,
                            perturbation=0.15, velocity=[0.7, -0.4, 0.3],
                            operator_kind=1, viscosity=0.05,
                            penalty_factor=16.0),
    "3d_k4_sipg_pert_cellular": dict(dim=3, degree=4, refine=2,
                                     perturbation=0.1, velocity_kind=1,
                                     operator_kind=1, viscosity=0.05,
                                     penalty_factor=25.0),
    "2d_k5_sipg_pert_vortex": dict(dim=2, degree=5, refine=3,
                                   perturbation=0.1, velocity_kind=2,
                                   time_factor=1, final_time=8.0,
                                   operator_kind=1, viscosity=0.05,
                                   penalty_factor=36.0),
    "3d_k2_sipg_cart": dict(dim=3, degree=2, refine=2,
                            velocity=[0.7, -0.4, 0.3], operator_kind=1,
                            viscosity=0.05, penalty_factor=9.0),
}

SWITCHES = {"gl_quad": dict(use_gl_quad=1),
            "gl_quad_mass": dict(use_gl_quad_mass=1)}


def make(name, switch):
    kw = dict(CASES[name])
    kw.update(SWITCHES[switch])
    c = Cfg(**kw)
    return c, AdvectionOperation(c.dg()), c.oracle_handle()


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(t):
    return t.detach().cpu().numpy()


@pytest.mark.parametrize("switch", sorted(SWITCHES))
@pytest.mark.parametrize("name", sorted(CASES))
def test_apply_matches_oracle(gpu_lib, name, switch):
    c, op, o = make(name, switch)
    print(f"case {name} {switch}", flush=True)
    u = np.random.default_rng(11).standard_normal(o.n_dofs)
    for t in (0.0, 0.37):
        ref = o.apply(u, t)
        dst = op.initialize_dof_vector()
        op.apply(dev(u), dst, t)
        torch.cuda.synchronize()
        assert rel_diff(host(dst), ref) < TOL, (name, switch)
    # the switch changes the operator
    plain = Cfg(**CASES[name]).oracle_handle()
    assert rel_diff(plain.apply(u, 0.37), ref) > 1e-8


@pytest.mark.parametrize("switch", sorted(SWITCHES))
def test_inverse_mass_and_projection_match_oracle(gpu_lib, switch):
    c, op, o = make("3d_k3_pert_cellular", switch)
    v = np.random.default_rng(5).standard_normal(o.n_dofs)
    d = dev(v)
    op.apply_inverse_mass_matrix(d)
    torch.cuda.synchronize()
    assert rel_diff(host(d), o.inverse_mass(v)) < TOL
    c2 = Cfg(**dict(CASES["3d_k3_pert_cellular"], solution_kind=3,
                    solution_param=[0.5, 0.5, 0.5, 0.2],
                    **SWITCHES[switch]))
    op2 = AdvectionOperation(c2.dg())
    u = op2.initialize_dof_vector()
    op2.project_initial(u, 0.0)
    torch.cuda.synchronize()
    assert rel_diff(host(u), c2.oracle_handle().project(0.0)) < TOL


@pytest.mark.parametrize("switch", sorted(SWITCHES))
@pytest.mark.parametrize("name", ["3d_k3_pert_cellular",
                                  "3d_k2_dirichlet_skew", "3d_k3_sipg_pert",
                                  "2d_k5_sipg_pert_vortex"])
def test_perform_stage_matches_oracle(gpu_lib, name, switch):
    c, op, o = make(name, switch)
    rng = np.random.default_rng(3)
    ri, sol = rng.standard_normal((2, o.n_dofs))
    t, b, a = 0.2, 0.013, 0.021
    ki_o, sol_o, nri_o = np.zeros(o.n_dofs), sol.copy(), np.zeros(o.n_dofs)
    o.perform_stage(t, b, a, ri, ki_o, sol_o, nri_o)
    d_ri, d_sol = dev(ri), dev(sol)
    d_ki, d_nri = op.initialize_dof_vector(), op.initialize_dof_vector()
    op.perform_stage(t, b, a, d_ri, d_ki, d_sol, d_nri)
    assert rel_diff(host(d_sol), sol_o) < TOL
    assert rel_diff(host(d_nri), nri_o) < TOL
    # aliased registers (reference integrator's first stage)
    sol_o2, r_o2 = sol.copy(), np.zeros(o.n_dofs)
    o.perform_stage(t, b, a, sol_o2, r_o2, sol_o2, r_o2)
    d_sol2, d_r2 = dev(sol), op.initialize_dof_vector()
    op.perform_stage(t, b, a, d_sol2, d_r2, d_sol2, d_r2)
    assert rel_diff(host(d_sol2), sol_o2) < TOL
    assert rel_diff(host(d_r2), r_o2) < TOL


@pytest.mark.parametrize("switch", sorted(SWITCHES))
def test_lsrk_time_steps_match_oracle(gpu_lib, switch):
    kw = dict(dim=3, degree=3, n_coarse=[3, 3, 3], refine=1,
              lo=[-1, -1, -1], hi=[1, 1, 1], velocity=[0.3, -0.2, 0.9],
              solution_kind=1, **SWITCHES[switch])
    c = Cfg(**kw)
    op, o = AdvectionOperation(c.dg()), c.oracle_handle()
    u = o.project(0.0)
    r1, r2 = o.zeros(), o.zeros()
    d_u = dev(u)
    d_r1, d_r2 = op.initialize_dof_vector(), op.initialize_dof_vector()
    integ = LowStorageRungeKuttaIntegrator(1)
    t, dt = 0.0, 0.01
    for _ in range(3):
        o.lsrk_time_step(1, t, dt, u, r1, r2)
        integ.perform_time_step(op, t, dt, d_u, d_r1, d_r2)
        t += dt
    torch.cuda.synchronize()
    assert rel_diff(host(d_u), u) < TOL


def test_gl_quadrature_known_answer_polynomial(gpu_lib):
    """use_gl_quad on axis-aligned cells: M^-1(-L u) = -a.grad u at the
    nodes for u in Q_k (summation by parts; the oracle's pin of the same
    case)."""
    k, dim = 4, 3
    a = [0.7, -0.4, 0.3]
    c = Cfg(dim=dim, degree=k, refine=1, periodic=[0, 0, 0], velocity=a,
            solution_kind=4, solution_param=[k], lo=[-0.5, 0, 0.25],
            hi=[0.5, 1.5, 1.0], use_gl_quad=1)
    op = AdvectionOperation(c.dg())
    u = op.initialize_dof_vector()
    op.project_initial(u, 0.0)
    du = op.initialize_dof_vector()
    op.apply(u, du, 0.0)
    pts = nodal_points(op.cell_vertices(), k + 1, dim)
    s = 1 + sum((d + 1) * pts[..., d] for d in range(dim))
    exact = -k * s ** (k - 1) * sum((d + 1) * a[d] for d in range(dim))
    assert rel_diff(host(du), exact.ravel()) < 1e-11


@pytest.mark.parametrize("switch", sorted(SWITCHES))
def test_implicit_operators_reject_the_switches(gpu_lib, switch):
    """The implicit operators, their FDM and the IRK path are built for
    QGauss(k+1): they report DG_ERR_UNSUPPORTED instead of computing."""
    c = Cfg(dim=3, degree=2, refine=1, **SWITCHES[switch])
    op = AdvectionOperation(c.dg())
    src, dst = op.initialize_dof_vector(), op.initialize_dof_vector()
    op.set_time(0.0, 0.01)
    with pytest.raises(L.DgError) as e:
        op.vmult(dst, src)
    assert e.value.code == L.DG_ERR_UNSUPPORTED
