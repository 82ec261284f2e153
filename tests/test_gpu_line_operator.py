"""The operator kernel's line terms (cell and face terms on even and odd
parts, staged traces and normal derivatives) against the CPU oracle where
they can go wrong: every degree (odd and even numbers of points), ragged last
workgroups, boundary faces, several components, the speed per point."""
import numpy as np
import pytest

from helpers import Cfg, rel_diff

pytestmark = pytest.mark.gpu
# round-off of two orders of summation in double precision: the oracle's
# parity bar
TOL = 1e-12


def _coarse(dim, flat=False):
    # 77 (or 343) cells, without a factor 2, 3 or 5: the last workgroup is a
    # partial one at every degree (_ragged), and its first cell is not its
    # last. flat: in 3D one cell along z, its own neighbour on both sides
    # where z is periodic; else enough cells for inner, perturbed vertices
    return [7, 11, 1] if dim == 2 or flat else [7, 7, 7]


def _ragged(op):
    cells = op.tile_shape()["cells_per_workgroup"]
    assert cells > 1 and op.n_cells % cells != 0, (op.n_cells, cells)


def _apply(c, seed, t=0.1):
    import torch
    from advection_miniapp_amd import AdvectionOperation
    op, o = AdvectionOperation(c.dg()), c.oracle_handle()
    u = np.random.default_rng(seed).standard_normal(o.n_dofs)
    dst = op.initialize_dof_vector()
    op.apply(torch.as_tensor(u, device="cuda"), dst, t)
    _ragged(op)
    return dst.cpu().numpy(), o.apply(u, t)


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("degree", range(1, 8))
@pytest.mark.parametrize("speed", ["constant", "per point"])
def test_sipg_every_degree_on_ragged_meshes(dim, degree, speed):
    kind = 0 if speed == "constant" else (2 if dim == 2 else 1)
    c = Cfg(dim=dim, degree=degree, n_coarse=_coarse(dim, flat=True),
            refine=0, hi=[1.0, 1.0, 1.0], velocity_kind=kind,
            velocity=[0.7, -0.4, 0.3], operator_kind=1, viscosity=0.05,
            penalty_factor=(degree + 1) ** 2)
    got, ref = _apply(c, 10 * degree + dim)
    assert rel_diff(got, ref) < TOL


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("degree", range(1, 8))
@pytest.mark.parametrize("skew", [0.0, 0.5])
def test_advection_boundary_faces_on_ragged_meshes(dim, degree, skew):
    c = Cfg(dim=dim, degree=degree, n_coarse=_coarse(dim), refine=0,
            hi=[1.0, 1.0, 1.0], perturbation=0.1, periodic=[0, 1, 0],
            velocity_kind=2 if dim == 2 else 1, flux_alpha=0.5,
            factor_skew=skew, solution_kind=2,
            solution_param=[np.pi, 0.0])
    got, ref = _apply(c, 20 * degree + dim)
    assert rel_diff(got, ref) < TOL


@pytest.mark.parametrize("degree", [2, 3, 4, 7])
@pytest.mark.parametrize("fp32", [False, True])
def test_inverse_mass_rows_on_stretched_cells(degree, fp32):
    # the table row of 1/JxW on strongly deformed cells of unlike sides:
    # values at the points up to degree 2 and in FP32, coefficients of the
    # determinant above. FP32: the values' own rounding, at most 2 (k + 1)
    # sums of up to n terms in each direction
    import torch
    from advection_miniapp_amd import AdvectionOperation
    c = Cfg(dim=3, degree=degree, n_coarse=[3, 2, 1], refine=1,
            hi=[4.0, 1.0, 0.25], perturbation=0.3, velocity_kind=1,
            precision=int(fp32))
    op, o = AdvectionOperation(c.dg()), c.oracle_handle()
    u = np.random.default_rng(degree).standard_normal(o.n_dofs)
    u = u.astype(np.float32 if fp32 else np.float64).astype(np.float64)
    dst = op.initialize_dof_vector()
    op.apply(torch.as_tensor(u, device="cuda", dtype=dst.dtype), dst, 0.1)
    tol = 1.2e-7 * 6 * (degree + 1) ** 2 if fp32 else TOL
    assert rel_diff(dst.double().cpu().numpy(), o.apply(u, 0.1)) < tol


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("degree,stages", [(1, 3), (2, 3), (3, 2), (5, 2),
                                           (6, 3)])
def test_stage_operator_with_boundary_faces(dim, degree, stages):
    # boundary faces under the kernels with the most registers (2 and 3
    # stages: the 4-stage table has 7 digits, the oracle computes its own)
    import torch
    from advection_miniapp_amd import AdvectionOperation
    c = Cfg(dim=dim, degree=degree, n_coarse=_coarse(dim, flat=True),
            refine=0, perturbation=0.1, periodic=[1, 0, 0], factor_skew=0.5,
            velocity_kind=2, solution_kind=2, solution_param=[np.pi, 0.0],
            irk_stages=stages)
    op, o = AdvectionOperation(c.dg()), c.oracle_handle()
    Z = np.random.default_rng(degree).standard_normal(o.n_dofs * stages)
    op.set_time(0.2, 0.05)
    dst = op.initialize_dof_vector(blocks=stages)
    op.vmult_irk(dst, torch.as_tensor(Z, device="cuda"))
    _ragged(op)
    assert rel_diff(dst.cpu().numpy(), o.irk_vmult(Z, 0.2, 0.05)) < TOL


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("degree", range(1, 8))
@pytest.mark.parametrize("speed", ["constant", "tabulated"])
def test_sipg_on_perturbed_ragged_meshes(dim, degree, speed):
    # right-hand side, stage and implicit operator of the general-cell SIPG
    # kernel
    import torch
    from advection_miniapp_amd import AdvectionOperation
    kind = 0 if speed == "constant" else (2 if dim == 2 else 1)
    kw = dict(dim=dim, degree=degree, n_coarse=_coarse(dim), refine=0, seed=5,
              perturbation=0.15, velocity_kind=kind, viscosity=0.05,
              velocity=[0.7, -0.4, 0.3], operator_kind=1,
              penalty_factor=(degree + 1) ** 2)
    got, ref = _apply(Cfg(**kw), 30 * degree + dim)
    assert rel_diff(got, ref) < TOL
    c = Cfg(factor_skew=0.5, **kw)
    op, o = AdvectionOperation(c.dg()), c.oracle_handle()
    u = np.random.default_rng(degree).standard_normal(o.n_dofs)
    dst = op.initialize_dof_vector()
    op.set_time(0.2, 0.05)
    op.vmult(dst, torch.as_tensor(u, device="cuda"))
    assert rel_diff(dst.cpu().numpy(), o.vmult(u, 0.2, 0.05)) < TOL
    c = Cfg(**kw)
    op, o = AdvectionOperation(c.dg()), c.oracle_handle()
    sol = np.random.default_rng(degree + 50).standard_normal(o.n_dofs)
    ki, so, nx = np.zeros(o.n_dofs), sol.copy(), np.zeros(o.n_dofs)
    o.perform_stage(0.1, 0.01, 0.02, u, ki, so, nx)
    d_sol = torch.as_tensor(sol, device="cuda")
    d_nx = op.initialize_dof_vector()
    op.perform_stage(0.1, 0.01, 0.02, torch.as_tensor(u, device="cuda"),
                     op.initialize_dof_vector(), d_sol, d_nx)
    assert rel_diff(d_sol.cpu().numpy(), so) < TOL
    assert rel_diff(d_nx.cpu().numpy(), nx) < TOL
