"""Density and velocity downloads: chunks through the pinned slots and the worker threads, the last chunk
short, 16^3 and 8^3 blocks, every storage form and the AA pattern; bit for bit the moments of the downloaded
populations, summed in direction order."""
import numpy as np
import pytest

from openaerolab_alpha_01_amd import solver
from openaerolab_alpha_01_amd.geometry import lattice_d3q27, sphere_mask, uniform_grid

pytestmark = pytest.mark.gpu


def moments(plan):
    c, _, _, _, _ = lattice_d3q27()
    f = plan.download_f(dtype=np.float64)
    work = np.float64 if plan.storage == "f64" else np.float32
    w = np.array([(8, 2, 1, 1)[int(abs(v).sum())] for v in c], dtype=work) / np.array(
        [(27, 27, 54, 216)[int(abs(v).sum())] for v in c], dtype=work)
    dr = np.zeros(f.shape[1])
    j = np.zeros((3, f.shape[1]))
    for k in range(27):
        s = f[k] - float(w[k])
        dr += s
        for a in range(3):
            j[a] += s * c[k][a]
    return 1.0 + dr, j / (1.0 + dr)


@pytest.mark.parametrize("storage,stream,bs,n", [("f32", "ab", 16, (80, 72, 64)), ("f16s", "ab", 8, (80, 72, 64)),
                                                  ("bf16s", "ab", 8, (52, 44, 40)), ("f64", "ab", 16, (48, 32, 32)),
                                                  ("f32", "aa", 16, (64, 64, 48))])
def test_macro_chunks(storage, stream, bs, n):
    # 409600 and 368640 cells: seven and six chunks of 65536; one chunk; three whole ones
    grid = uniform_grid(n, bs=bs)
    grid.solid = sphere_mask(grid, (20, 18, 18), 6.0)
    rng = np.random.default_rng(5)
    plan = solver.uniform_plan(grid, 0.55, storage=storage, stream=stream, u_inlet=0.05,
                               params=solver.StepParams(c_wale=0.0, inlet_turbulence=0.0))
    plan.init_equilibrium(1.0 + rng.uniform(-1e-2, 1e-2, grid.n_cells), rng.uniform(-0.05, 0.05, (3, grid.n_cells)))
    plan.step(2, 0)
    for _ in range(2):      # the second call finds the slots in place
        rho, u = plan.macro()
        r, v = moments(plan)
        assert np.array_equal(rho, r) and np.array_equal(u, v)
        plan.step(2, 2)
    plan.close()
