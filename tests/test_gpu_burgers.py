"""GPU parity of the Burgers operator (over-integrated cell flux, Rusanov
faces) and its LSRK stages against the CPU oracle."""
import numpy as np
import pytest
import torch

from advection_miniapp_amd import AdvectionOperation, \
    LowStorageRungeKuttaIntegrator
from helpers import Cfg, rel_diff

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(t):
    return t.detach().cpu().numpy()


def burgers(dim, k, refine, **kw):
    return Cfg(dim=dim, degree=k, n_components=dim, operator_kind=2,
               refine=refine, lo=[-1, -1, -1], hi=[1, 1, 1],
               solution_kind=6, **kw)


@pytest.mark.parametrize("dim,k,pert", [(3, 3, 0.0), (3, 2, 0.1), (2, 4, 0.0),
                                        (2, 1, 0.15), (3, 4, 0.0),
                                        (3, 1, 0.0), (3, 5, 0.1), (3, 6, 0.0),
                                        (3, 7, 0.0), (3, 7, 0.1)])
def test_burgers_apply_matches_oracle(gpu_lib, dim, k, pert):
    c = burgers(dim, k, 1 if dim == 3 else 2, perturbation=pert)
    op, o = AdvectionOperation(c.dg()), c.oracle_handle()
    u = o.project(0.0) + 0.1 * np.random.default_rng(1).standard_normal(
        o.n_dofs * dim)
    dst = op.initialize_dof_vector()
    op.apply(dev(u), dst, 0.0)
    assert rel_diff(host(dst), o.burgers_apply(u)) < 1e-12


def test_burgers_projection_and_lsrk(gpu_lib):
    c = burgers(3, 3, 1)
    op, o = AdvectionOperation(c.dg()), c.oracle_handle()
    u = op.initialize_dof_vector()
    op.project_initial(u, 0.0)
    ref = o.project(0.0)
    assert rel_diff(host(u), ref) < 1e-13
    # two LSRK(5,4) steps; CPU side restated with the oracle's operator
    dt = 0.01
    integ = LowStorageRungeKuttaIntegrator(1)
    r1, r2 = op.initialize_dof_vector(), op.initialize_dof_vector()
    bi = [1153189308089. / 22510343858157., 1772645290293. / 4653164025191.,
          -1672844663538. / 4480602732383., 2114624349019. / 3568978502595.,
          5198255086312. / 14908931495163.]
    ai = [970286171893. / 4311952581923., 6584761158862. / 12103376702013.,
          2251764453980. / 15575788980749., 26877169314380. / 34165994151039.]
    sol = ref.copy()
    for _ in range(2):
        integ.perform_time_step(op, 0.0, dt, u, r1, r2)
        # reference recursion (advection_solver.cc:906-939)
        k = o.burgers_apply(sol)
        ri = sol + ai[0] * dt * k
        sol = sol + bi[0] * dt * k
        for s in range(1, 5):
            k = o.burgers_apply(ri)
            new_sol = sol + bi[s] * dt * k
            if s < 4:
                ri = sol + ai[s] * dt * k
            sol = new_sol
    assert rel_diff(host(u), sol) < 1e-12


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("k", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("pert", [0.0, 0.2])
def test_burgers_apply_and_stage_on_ragged_meshes(gpu_lib, dim, k, pert):
    # every kernel of the dispatch (2D point-wise: degree 1; lines: 2 to 4;
    # slabs: 1 and 5) on boxes of unlike sides whose cells fill no workgroup
    # evenly, right-hand side and fused stage, with a central-upwind blend
    if dim == 2 and k > 4:
        pytest.skip("2D is built for degrees 1..4")
    c = Cfg(dim=dim, degree=k, n_components=dim, operator_kind=2,
            n_coarse=[5, 3, 1], refine=0, lo=[-1, 0, 0], hi=[1, 2, 0.5],
            perturbation=pert, seed=3, flux_alpha=0.7, solution_kind=6)
    op, o = AdvectionOperation(c.dg()), c.oracle_handle()
    rng = np.random.default_rng(k + 10 * dim)
    u, sol = rng.standard_normal((2, o.n_dofs * dim))
    ref = o.burgers_apply(u)
    dst = op.initialize_dof_vector()
    op.apply(dev(u), dst, 0.0)
    assert rel_diff(host(dst), ref) < 1e-12
    d_sol, d_nri = dev(sol), op.initialize_dof_vector()
    op.perform_stage(0.1, 0.01, 0.02, dev(u), op.initialize_dof_vector(),
                     d_sol, d_nri)
    assert rel_diff(host(d_sol), sol + 0.01 * ref) < 1e-12
    assert rel_diff(host(d_nri), sol + 0.02 * ref) < 1e-12
