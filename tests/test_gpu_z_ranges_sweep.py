"""z ranges of the mixed MHD kernel for physical sides and refined meshes
(k_sweep): launches whose few tiles are split into ranges and launches whose
many tiles are not must give the same cells and faces bit for bit."""
import numpy as np
import pytest

import kratos_amd
from kratos_amd import problems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nz", [4, 7, 21])
@pytest.mark.parametrize("tile", [(8, 8, 1), (16, 8, 1), (32, 8, 4)])
@pytest.mark.parametrize("sides", [("out",) * 6, ("per", "per", "ref", "out", "fre", "ref"),
                                   ("per",) * 4 + ("fixd", "out")])
def test_sides_one_box_equals_many(gpu_lib, nz, tile, sides):
    """A 32x16xnz box alone and as 300 members of an ensemble."""
    spec = kratos_amd.MeshSpec((32, 16, nz), (32, 16, nz), bnd=sides)
    fix_b = (0.3, 0.5, 0.2)
    phys = kratos_amd.Physics(mhd=True, fix_w=(0.9, 0.4, 0.1, 0.05, -0.1), fix_b=fix_b)
    u, b, _ = problems.turbulence(spec.n_cell_global, seed=nz)
    b = tuple(np.full_like(x, fix_b[a]) for a, x in enumerate(b))
    u[1] = problems.total_energy(u[0], 0.6 + 0 * u[0], u[2:] / u[0], problems.cell_centred_b(*b), phys.gamma)
    got = []
    for n in (1, 300):
        ctx = kratos_amd.Context(spec, phys, "mixed", path="fused", tile=tile, members=n)
        for m in range(n):
            ctx.upload(u, b, member=m)
        ctx.advance(3)
        assert ctx.stats()["sweep_kernel"] == 0 and ctx.stats()["sweep_tile"][:2] == tile[:2]
        got.append([ctx.download(member=m) for m in {0, n // 2, n - 1}])
        ctx.close()
    one = got[0][0]
    assert np.isfinite(one[0]).all()
    for gu, gb in got[1]:
        assert np.array_equal(gu, one[0])
        assert all(np.array_equal(x, y) for x, y in zip(gb, one[1]))


@pytest.mark.parametrize("nb", [8, 16])
def test_refined_mesh_equals_its_copies(gpu_lib, nb):
    """A two-level periodic mesh, and the mesh of 2^3 copies of it side by
    side: more tiles, fewer ranges, and every copy stays equal to the mesh
    alone."""
    phys = kratos_amd.Physics(mhd=True)

    def mesh(k):
        corners = [(x, y, z) for x in range(k) for y in range(k) for z in range(k)]
        return kratos_amd.RefinedMeshSpec(
            (4 * nb * k,) * 3, (nb,) * 3, x_min=(0.0,) * 3, x_max=(float(k),) * 3,
            refine=[(1, tuple(c + 0.375 for c in o), tuple(c + 0.625 for c in o)) for o in corners])

    spec, many = mesh(1), mesh(2)
    where = {leaf: i for i, leaf in enumerate(spec.leaves)}

    def source(i):
        lev, x, y, z = many.leaves[i]
        n = spec.nblk[0] << lev
        return where[(lev, x % n, y % n, z % n)]

    src = [source(i) for i in range(many.n_blocks)]
    assert many.n_blocks == 8 * spec.n_blocks
    blocks = problems.smooth_blocks(spec, seed=4)
    out = []
    for s, blk in ((spec, blocks), (many, [blocks[i] for i in src])):
        ctx = kratos_amd.Context(s, phys, "mixed")
        ctx.upload_blocks(blk)
        assert ctx.advance(3) == 3
        assert ctx.stats()["sweep_tile"][0] > 0
        out.append((ctx.download_blocks(), ctx.time()))
        ctx.close()
    assert out[0][1] == out[1][1]
    for i, (u, f) in enumerate(out[1][0]):
        assert np.array_equal(u, out[0][0][src[i]][0])
        assert np.array_equal(f, out[0][0][src[i]][1])
