"""The one-launch step kernels, two cells per lane (both patterns) and one cell per lane (AB pattern), at the extents
where pairs, row ends and rules can go wrong, against the oracle bit for bit."""
import numpy as np
import pytest

from openaerolab_alpha_01_amd import solver
from openaerolab_alpha_01_amd.geometry import batch_grids, sphere_mask, uniform_grid
from test_gpu_parity import compare, fields, gpu_plan, oracle_run

pytestmark = pytest.mark.gpu

# x extents: one block, the outlet in the first cell of a block (lane 0, cell A), in its cell B, in the last
# cell but one (lane 7, cell A); y and z extents of one row or plane more or less than whole blocks
CASES = {
    "one_block": dict(n=(16, 16, 16), okw=dict(tau=0.53, u_inlet=0.05)),
    "outlet_lane0": dict(n=(33, 17, 15), solid=((30, 9, 8), 4.0), okw=dict(tau=0.53, u_inlet=0.05)),
    "outlet_b": dict(n=(34, 31, 33), solid=((18, 16, 16), 3.0),
                     okw=dict(tau=0.52, u_inlet=0.05, ymin_wall_bc=1, zwall_bc=2, inlet_turbulence=0.01)),
    "outlet_lane7": dict(n=(31, 18, 17), solid=((28, 4, 4), 3.5), okw=dict(tau=0.56, u_inlet=0.04, c_wale=0.2)),
    "tiny": dict(n=(3, 2, 1), okw=dict(tau=0.6, u_inlet=0.03)),
    "wraps": dict(n=(32, 16, 48), periodic=(True, True, True), solid=((15, 15, 31), 2.5),
                  okw=dict(tau=0.52, body_force=(1e-5, -2e-6, 3e-6), omega_3=0.9, omega_4=1.1, adaptive_omega4=0)),
    "channel": dict(n=(32, 32, 16), periodic=(True, False, True), solid=((1, 30, 8), 2.5),
                    okw=dict(tau=0.55, body_force=(1e-5, 0.0, 0.0), ymin_wall_bc=1, c_wale=0.2, omega_bulk=1.2)),
}


# (AB: so few blocks take the one-cell-per-lane form)
@pytest.mark.parametrize("stream", ["ab", "aa"])
@pytest.mark.parametrize("storage", ["f32", "f16s", "bf16s"])
@pytest.mark.parametrize("case", list(CASES))
def test_two_cells_per_lane(oracle, storage, case, stream):
    cfg = CASES[case]
    grid = uniform_grid(cfg["n"], periodic=cfg.get("periodic", (False, False, False)))
    if "solid" in cfg:
        grid.solid = sphere_mask(grid, *cfg["solid"])
    okw = cfg["okw"]
    rho, u = fields(grid, seed=23, u0=(okw.get("u_inlet", 0.0), 0, 0))
    steps = 4
    f_or, forces, _ = oracle_run(oracle, grid, storage, steps, okw, rho, u, force_steps=(3,) if "solid" in cfg else ())
    plan = gpu_plan(grid, storage, okw, stream)
    plan.init_equilibrium(rho, u)
    for t in range(steps):
        plan.level_step(0, t, force="solid" in cfg and t == 3)
    if "solid" in cfg:
        np.testing.assert_allclose(plan.force()[0], forces[0], rtol=1e-11, atol=1e-14)
    if stream == "ab":
        compare(oracle, plan, storage, f_or, grid)   # the cells beyond the extent too: never written
    else:
        # after an even number of steps the pull step's state in the stepped cells
        live = grid.inside() & ((grid.solid == 0) if "solid" in cfg else True)
        got = plan.download_f(dtype=np.float32 if storage == "f32" else np.float64)
        want = f_or if storage == "f32" else oracle.to_unshifted(storage, f_or)
        assert np.array_equal(got[..., live], want[..., live])
    plan.close()


@pytest.mark.parametrize("storage", ["f32", "f16s", "bf16s"])
@pytest.mark.parametrize("case", list(CASES))
def test_many_copies(oracle, storage, case):
    """Levels of more than 512 blocks take the two-cells-per-lane kernel in the AB pattern, smaller ones (the
    test above) the one-cell form: copies of a grid as the domains of one level, each the oracle's bits."""
    cfg = CASES[case]
    grid = uniform_grid(cfg["n"], periodic=cfg.get("periodic", (False, False, False)))
    if "solid" in cfg:
        grid.solid = sphere_mask(grid, *cfg["solid"])
    okw = cfg["okw"]
    rho, u = fields(grid, seed=31, u0=(okw.get("u_inlet", 0.0), 0, 0))
    f_or, _, _ = oracle_run(oracle, grid, storage, 2, okw, rho, u)
    copies = 512 // grid.n_blocks + 1
    big = batch_grids([grid] * copies)
    dom = {k: okw[k] for k in ("tau", "u_inlet", "body_force", "ymin_wall_bc", "zwall_bc") if k in okw}
    params = dict(omega_bulk=1.0, omega_3=1.0, omega_4=1.0, lambda_=1 / 6, adaptive_omega4=1, limiter=1, compressible=0,
                  c_wale=0.0, nu_sgs_background=0.0, inlet_turbulence=0.0)
    params.update({k: v for k, v in okw.items() if k not in dom})
    doms = [solver.Domain(extent=grid.n, periodic=grid.periodic, **dom) for _ in range(copies)]
    plan = solver.Plan(solver.Level(big, doms, block_domain=big.block_domain), storage=storage, stream="ab",
                       bb_mode="halfway", params=solver.StepParams(**params))
    plan.init_equilibrium(np.tile(rho, copies), np.tile(u, copies))
    for t in range(2):
        plan.level_step(0, t)
    got = plan.download_f(dtype=np.float32 if storage == "f32" else np.float64).reshape(27, copies, -1)
    want = f_or if storage == "f32" else oracle.to_unshifted(storage, f_or)
    assert all(np.array_equal(got[:, i], want) for i in range(copies))
    plan.close()


@pytest.mark.parametrize("limiter", [1, 2])
@pytest.mark.parametrize("case", list(CASES))
def test_one_cell_per_lane_fp64(oracle, case, limiter):
    """The FP64 kernel (AB pattern) on the same extents, without and with the positivity limiter's form."""
    cfg = CASES[case]
    grid = uniform_grid(cfg["n"], periodic=cfg.get("periodic", (False, False, False)))
    if "solid" in cfg:
        grid.solid = sphere_mask(grid, *cfg["solid"])
    okw = dict(cfg["okw"], limiter=limiter)
    rho, u = fields(grid, seed=29, u0=(okw.get("u_inlet", 0.0), 0, 0))
    force_steps = (2,) if "solid" in cfg else ()
    f_or, forces, _ = oracle_run(oracle, grid, "f64", 3, okw, rho, u, force_steps=force_steps)
    plan = gpu_plan(grid, "f64", okw)
    plan.init_equilibrium(rho, u)
    for t in range(3):
        plan.level_step(0, t, force=t in force_steps)
    if force_steps:
        np.testing.assert_allclose(plan.force()[0], forces[0], rtol=1e-11, atol=1e-14)
    compare(oracle, plan, "f64", f_or, grid)
    plan.close()
