"""The FP32 form's rounding error of one ternary timestep, against the FP64 form
from the same state."""
import numpy as np
import pytest

from lb3d_amd.gpu import LB3D_FP32_DEV, LB3D_FP64, Lattice

pytestmark = pytest.mark.gpu

# 2-norm of the error over the 2-norm of the result, of a form that sums the
# stencil with separate products and one rounding of the sum per neighbour
# (measured at 64x50x47, six states: dipoles 1.385e-7 to 1.391e-7, populations
# 1.932e-7 to 1.934e-7)
DIPOLES, POPULATIONS = 1.391e-7, 1.934e-7


@pytest.mark.parametrize("one_pass", [False, True])
def test_ternary_step_error(one_pass):
    dims = (64, 50, 47)
    nx, ny, nz = dims
    w = np.array([1 / 36] * 18 + [1 / 3])
    for seed in range(3):
        rng = np.random.default_rng(seed)
        N = np.zeros((nz + 2, ny + 2, nx + 2, 79))
        sites = N[1:-1, 1:-1, 1:-1]
        for c in range(3):
            dev = w * (0.01 * rng.uniform(-1, 1, (nz, ny, nx, 1)) + 0.002 * rng.uniform(-1, 1, (nz, ny, nx, 19)))
            sites[..., 24 * c:24 * c + 19] = w * 0.7 + dev.astype(np.float32)
        sites[..., 75:78] = (0.5 * rng.uniform(-1, 1, (nz, ny, nx, 3))).astype(np.float32)
        got = []
        for precision in (LB3D_FP64, LB3D_FP32_DEV):
            g = Lattice(*dims, ncomp=3, precision=precision, g_br=0.08, g_bs=-0.006, g_ss=-0.003)
            if one_pass and precision == LB3D_FP32_DEV:
                g.set_plan(3, 32, 8, 8)
            g.upload_sites(N)
            g.bc_init()
            g.time_loop(1)
            got.append((g.populations() - w[None, :, None, None, None] * 0.7,
                        g.download_sites()[1:-1, 1:-1, 1:-1, 75:78]))
        for what, k, most in (("populations", 0, POPULATIONS), ("dipoles", 1, DIPOLES)):
            err = np.linalg.norm(got[1][k] - got[0][k]) / np.linalg.norm(got[0][k])
            print(f"seed {seed} {what}: {err:.4e}", flush=True)
            assert err <= most, (seed, what)
