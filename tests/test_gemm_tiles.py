"""The eigen-transform kernels' tiles (csrc/gemm.h, csrc/gemm_tile.h)."""
import pytest

import test_gpu_parity as par

BCT, SIGMA = (1, 1, 2, 2, 1, 2), -300.0


# the FP32 x transform's 16-deep quads: none, one, one and its least and largest
# overlap, two and the same, in front of 16 x 16 and of 32 x 32 tiles
@pytest.mark.gpu
@pytest.mark.parametrize("nx", [17, 18, 19, 33, 34, 35, 49])
@pytest.mark.parametrize("ny,nz", [(12, 14), (150, 122)])
def test_gpu_fp32_quads(nx, ny, nz):
    mf, torch = par._mf()
    shape = (nx, ny, nz)
    grids, sc, g, bcs, _ = par._make_problem(shape, BCT, SIGMA, 22)
    print("run fp32 quads %s" % (shape,), flush=True)
    got, rep = par._solve_gpu(mf, grids, BCT, g, bcs, SIGMA, mf.MF_MIXED, tol=1e-12)
    assert rep.residual <= 1e-12 and rep.iterations <= 4
    assert par._true_residual(sc, got, g, bcs, SIGMA) <= 2e-12
