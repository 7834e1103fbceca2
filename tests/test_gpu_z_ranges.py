"""z ranges of the stage kernels: a launch with few tiles splits each block's
march into ranges; every cell and face must come out as the full march
gives it.  Block heights that the ranges do not divide, the smallest height
the fused kernels take, and meshes on both sides of the split."""
import numpy as np
import pytest

import kratos_amd
import oracle
from kratos_amd import problems

pytestmark = pytest.mark.gpu


def _run(spec, phys, u, b, precision, path, tile=(0, 0, 0), cycles=3):
    ctx = kratos_amd.Context(spec, phys, precision, path=path, tile=tile)
    ctx.upload(u, b)
    ctx.advance(cycles)
    out = ctx.download()
    ctx.close()
    return out


@pytest.mark.parametrize("nz", [4, 5, 7, 11])
@pytest.mark.parametrize("mhd", [True, False])
@pytest.mark.parametrize("sides", ["per", "out"])
def test_odd_heights_fp64(gpu_lib, nz, mhd, sides):
    spec = kratos_amd.MeshSpec((32, 16, 2 * nz), (16, 8, nz), bnd=(sides,) * 6)
    phys = kratos_amd.Physics(mhd=mhd)
    u, b, _ = problems.turbulence(spec.n_cell_global, seed=nz)
    if sides == "out":                      # a field that ends at the sides
        b = tuple(np.full_like(x, 0.3 + 0.1 * a) for a, x in enumerate(b))
        bcc = problems.cell_centred_b(*b)
        u[1] = problems.total_energy(u[0], 0.6 + 0 * u[0], u[2:] / u[0], bcc if mhd else None,
                                     phys.gamma)
    elif not mhd:
        u[1] -= 0.5 * sum(x * x for x in problems.cell_centred_b(*b))
    gu, gb = _run(spec, phys, u, b if mhd else None, "fp64", "fused")
    ref = oracle.OracleMesh(spec, phys)
    ref.upload(u, b if mhd else None)
    ref.advance(3)
    ou, ob = ref.download()
    assert np.array_equal(gu, ou)
    if mhd:
        assert all(np.array_equal(x, y) for x, y in zip(gb, ob))


@pytest.mark.parametrize("mhd", [True, False])
def test_mixed_few_blocks_equal_many(gpu_lib, mhd):
    """One 32x16x22 box alone (its few tiles split into ranges) and as 300
    members of an ensemble (its tiles fill the GPU): the same state bit for
    bit, every member."""
    spec = kratos_amd.MeshSpec((32, 16, 22), (32, 16, 22))
    phys = kratos_amd.Physics(mhd=mhd)
    u, b, _ = problems.turbulence(spec.n_cell_global, seed=3)
    if not mhd:
        b = None
    one = _run(spec, phys, u, b, "mixed", "fused", tile=(8, 8, 1))
    n = 300
    ctx = kratos_amd.Context(spec, phys, "mixed", path="fused", tile=(8, 8, 1), members=n)
    for m in range(n):
        ctx.upload(u, b, member=m)
    ctx.advance(3)
    for m in (0, 7, n - 1):
        gu, gb = ctx.download(member=m)
        assert np.array_equal(gu, one[0])
        if mhd:
            assert all(np.array_equal(x, y) for x, y in zip(gb, one[1]))
    ctx.close()
