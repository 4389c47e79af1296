"""The eigen-transform kernels' tiles (csrc/gemm.h, csrc/gemm_tile.h).

The solver's transforms are products on one of eight tiles, chosen by size; each
tile has its own remainder rows and columns, divide and scatter epilogues.  SHAPES
are solves whose x, y and z transforms together take every tile larger than
16 x 16 (which the small shapes of test_gpu_parity.py take), with remainders along
both sides of the tile; the first test asks the rule itself, on the CPU, so that a
change of it cannot drop a tile from the list.

GPU, with test_gpu_parity.py's bars (a wrong row or column is of order one): FP64
solves within 1e-12 of the FP64 oracle; FP32 inner solves by the refinement's
contract, checked by an 80-bit residual, and within 2e-11 of it.
"""
import os
import subprocess

import numpy as np
import pytest

import mf_oracle as o
import test_gpu_parity as par

SHAPES = [(57, 123, 70), (100, 122, 101), (142, 166, 69), (195, 192, 52),
          (69, 250, 121), (192, 134, 100), (100, 154, 166), (123, 92, 164)]
BCT, SIGMA = (1, 1, 2, 2, 1, 2), -300.0
CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "mflops3d-md_amd", "csrc")

ASK = r"""
#include "gemm_tile.h"
#include <cstdio>
int main() {
  int f32, M, N, K, batch;
  while (std::scanf("%d %d %d %d %d", &f32, &M, &N, &K, &batch) == 5) {
    const mf::GemmTile t = f32 ? mf::gemm_tile_x32(M, N, K, batch, 256) : mf::gemm_tile_of(M, N, K, batch, 256);
    std::printf("%d %d\n", t.mi, t.ni);
  }
}
"""


def _ask(tmp_path, problems):
    src, exe = tmp_path / "ask.cpp", tmp_path / "ask"
    src.write_text(ASK)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], input="\n".join("%d %d %d %d %d" % q for q in problems),
                       capture_output=True, text=True, check=True)
    return [tuple(int(v) for v in l.split()) for l in r.stdout.split("\n") if l]


def test_shapes_take_every_tile(tmp_path):
    problems = []
    for nx, ny, nz in SHAPES:
        n1, n2, n3 = nx - 2, ny - 2, nz - 2
        problems += [(0, n1, n2 * n3, n1, 1), (0, n1, n2, n2, n3), (0, n1 * n2, n3, n3, 1),
                     (1, n1, n2 * n3, n1, 1)]
    tiles = _ask(tmp_path, problems)
    large = {(a, b) for a in (1, 2, 3, 4) for b in (1, 2, 3, 4)} & {(4, 4), (4, 3), (3, 4), (3, 3),
                                                                   (4, 2), (2, 4), (2, 2)}
    for which, name in enumerate("xyz"):
        seen = set()
        for (f32, M, N, K, b), t in zip(problems[which::4], tiles[which::4]):
            assert M % (16 * t[0]) and N % (16 * t[1]), (name, M, N, t)
            seen.add(t)
        assert seen == large, (name, large - seen)
    assert set(tiles[3::4]) == {(1, 1), (2, 2)}
    assert {q[2] % 4 for q in problems if not q[0]} >= {0, 1, 2, 3}


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
def test_gpu_tiles(shape):
    mf, torch = par._mf()
    grids, sc, g, bcs, _ = par._make_problem(shape, BCT, SIGMA, 21)
    ref = np.full(shape, 7.0, order="F")
    o.solver_3d(sc, g, ref, *bcs, SIGMA)
    top = np.abs(ref).max()
    print("run tiles fp64 %s" % (shape,), flush=True)
    got, _ = par._solve_gpu(mf, grids, BCT, g, bcs, SIGMA, mf.MF_FP64)
    err = np.abs(got - ref).max() / top
    print("run tiles fp32 %s" % (shape,), flush=True)
    got, rep = par._solve_gpu(mf, grids, BCT, g, bcs, SIGMA, mf.MF_MIXED, tol=1e-12)
    err32 = np.abs(got - ref).max() / top
    res = par._true_residual(sc, got, g, bcs, SIGMA)
    print("  fp64 %.2e  fp32 %.2e  residual %.2e in %d solves" % (err, err32, res, rep.iterations),
          flush=True)
    assert err < 1e-12 and err32 < 2e-11
    assert rep.residual <= 1e-12 and res <= 2e-12


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
