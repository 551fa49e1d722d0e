"""The direct solve in cosine modes (tb_spectral.hip) behind both Poisson
methods, at the sizes where its kernels can go wrong: axes at and around the
16-mode and 32-mode tile edges and the 64-column tiles, odd axes (a middle
row in the folded transform), the smallest axis, x lines at the edges of a
wave's points, the narrower column tiles of long axes, and axes past its
limits, where the mixed solve hands over to FP64 (fallback bit 1).

A random right-hand side of zero mean is solved from zero.  The solver stops
on its own residual, formed by the operator that is bit-identical to the
oracle's: the oracle's residual of the result is the tolerance up to its
summation order.  On grids that do not halve cleanly the FP64
preconditioner is the exact inverse, so CG ends within two iterations."""
import numpy as np
import pytest

from turbins_amd import Solver, abi, workload as W

pytestmark = pytest.mark.gpu

import oracle  # noqa: E402  (checker only)

RTOL = 1e-10
#        nx, ny, nz, lx, ly, lz, direct FP32 solve, exact FP64 preconditioner
CASES = [(64, 16, 32, 8.0, 1.0, 1.0, True, False),
         (65, 31, 17, 4.0, 1.0, 1.0, True, True),
         (63, 33, 15, 4.0, 1.0, 1.0, True, True),
         (4, 4, 5, 1.0, 1.0, 1.0, True, True),
         (5, 64, 66, 1.0, 1.0, 1.0, True, False),
         (129, 48, 34, 4.0, 1.0, 1.0, True, False),
         (257, 18, 9, 4.0, 1.0, 1.0, True, True),
         (513, 6, 7, 8.0, 1.0, 1.0, True, True),
         (1025, 5, 6, 16.0, 1.0, 1.0, True, True),
         (2048, 4, 5, 64.0, 1.0, 1.0, True, False),
         (20, 331, 6, 1.0, 8.0, 1.0, True, True),
         (12, 5, 651, 1.0, 1.0, 16.0, True, True),
         (6, 1201, 5, 1.0, 32.0, 1.0, True, True),
         (6, 1304, 5, 1.0, 32.0, 1.0, True, False),
         (4, 2560, 4, 1.0, 64.0, 1.0, False, False),
         (2064, 4, 4, 64.0, 1.0, 1.0, False, False)]


@pytest.mark.parametrize("nx,ny,nz,lx,ly,lz,direct32,exact64", CASES)
def test_poisson_at_tile_edges(nx, ny, nz, lx, ly, lz, direct32, exact64):
    print("spectral", nx, ny, nz, flush=True)
    c = W.case("lock64", nx=nx, ny=ny, nz=nz, lx=lx, ly=ly, lz=lz)
    cfg = W.config_for(c, pois_rtol=RTOL)
    g, o = Solver(cfg), oracle.Oracle(cfg)
    b = np.zeros((nz + 1, ny + 1, nx + 1))
    r = np.random.default_rng(nx * 7 + ny * 3 + nz).standard_normal((nz, ny, nx))
    b[:nz, :ny, :nx] = r - r.mean()
    for mode in (abi.POIS_MIXED_IR, abi.POIS_FP64_PCG):
        g.set_poisson_mode(mode, RTOL)
        g.upload("PHI", np.zeros(g.NT))
        g.upload("PRHS", b)
        st = g.poisson_solve()
        x = g.download("PHI")
        res = np.linalg.norm(b.ravel() - o.poisson_apply(x)) / np.linalg.norm(b)
        print("mode", mode, "its", st.iterations, "fallback", st.fallback, "res", st.res, "oracle", res, flush=True)
        assert st.converged and res <= RTOL * (1 + 1e-6)
        assert x.reshape(b.shape)[nz - 1, ny - 1, nx - 1] == 0.0     # the pinned corner
        if mode == abi.POIS_MIXED_IR:
            assert st.fallback == (0 if direct32 else 1)
        elif exact64:
            assert st.iterations <= 2
    g.close()
    o.close()
