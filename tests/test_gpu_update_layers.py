"""The staged MHD update runs its cells and face families as layers of the
grid up to 1,024 (mixed) or 2,048 (FP64) workgroups and in one layer above.
Either side of both lines against the fused kernels, bit for bit, on uniform
and on refined meshes (there a finer neighbour's faces are left out of the
sum and added after it)."""
import numpy as np
import pytest

import kratos_amd
from kratos_amd import problems

pytestmark = pytest.mark.gpu


def _workgroups(spec):
    n = [x + 1 for x in spec.n_cell_block]
    return -(-n[0] * n[1] * n[2] // 256) * spec.n_blocks


def _equal(spec, blocks, precision, tile):
    got = []
    for path, t in (("auto", tile), ("staged", (0, 0, 0))):
        ctx = kratos_amd.Context(spec, kratos_amd.Physics(mhd=True), precision, path=path, tile=t)
        ctx.upload_blocks(blocks)
        assert ctx.advance(3) == 3
        got.append((ctx.download_blocks(), ctx.time()))
        ctx.close()
    assert got[0][1] == got[1][1]
    for (u, f), (v, g) in zip(got[0][0], got[1][0]):
        assert np.array_equal(u, v) and np.array_equal(f, g)


@pytest.mark.parametrize("precision,k,layers", [("mixed", (8, 8, 4), True), ("mixed", (9, 8, 4), False),
                                                ("fp64", (8, 8, 8), True), ("fp64", (9, 8, 8), False)])
def test_uniform(gpu_lib, precision, k, layers):
    blk = (9, 9, 8)                                     # four workgroups a block
    spec = kratos_amd.MeshSpec(tuple(a * b for a, b in zip(k, blk)), blk)
    assert (_workgroups(spec) <= (2048 if precision == "fp64" else 1024)) == layers
    u, b, _ = problems.turbulence(spec.n_cell_global, seed=3)
    _equal(spec, spec.split(u, b), precision, (8, 8, 1))


@pytest.mark.parametrize("precision,blk,layers", [("mixed", (10, 8, 8), True), ("mixed", (14, 14, 14), False),
                                                  ("fp64", (10, 10, 10), True), ("fp64", (16, 16, 16), False)])
def test_refined(gpu_lib, precision, blk, layers):
    spec = kratos_amd.RefinedMeshSpec(tuple(4 * n for n in blk), blk, refine=[(1, (-0.25,) * 3, (0.25,) * 3)],
                                      x_min=(-0.5,) * 3, x_max=(0.5,) * 3)
    assert (_workgroups(spec) <= (2048 if precision == "fp64" else 1024)) == layers
    _equal(spec, problems.smooth_blocks(spec, seed=4, mhd=True), precision, (8, 8, 1))
