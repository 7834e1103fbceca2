"""kr_stats.tune_ms reports every variant that the autotuner timed, whichever
kernel the mesh runs, and the variant kept is the one reported fastest."""
import numpy as np
import pytest

import kratos_amd
from kratos_amd import problems

pytestmark = pytest.mark.gpu

# kr_stats.tune_ms entry of a kept tile (x, y, threads, waves) where the
# header's table has one entry for it
ENTRY = {(8, 8, 192, 1): (5, 10), (16, 8, 256, 1): (4, 7, 13), (0, 0, 0, 0): (6,)}


@pytest.mark.parametrize("mhd", [True, False])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("blk,levels", [((8, 8, 8), 1), ((12, 12, 12), 1), ((20, 12, 10), 1), ((32, 32, 8), 1),
                                        ((8, 8, 8), 2), ((12, 12, 12), 2)])
def test_every_timed_variant_is_reported(gpu_lib, mhd, precision, blk, levels):
    phys = kratos_amd.Physics(mhd=mhd)
    if levels == 1:
        spec = kratos_amd.MeshSpec(tuple(2 * n for n in blk), blk)
        u, b, _ = problems.turbulence(spec.n_cell_global, seed=5)
        if not mhd:
            u[1] -= 0.5 * sum(x * x for x in problems.cell_centred_b(*b))
        blocks = spec.split(u, b if mhd else None)
    else:
        spec = kratos_amd.RefinedMeshSpec(tuple(4 * n for n in blk), blk, x_min=(-0.5,) * 3, x_max=(0.5,) * 3,
                                          refine=[(1, (-0.1,) * 3, (0.1,) * 3)])
        blocks = problems.smooth_blocks(spec, seed=2, mhd=mhd)
    ctx = kratos_amd.Context(spec, phys, precision)
    ctx.upload_blocks(blocks)
    ctx.step()
    st = ctx.stats()
    cand = st["tune_pending"] + 1
    while st["tune_pending"]:
        ctx.step()
        st = ctx.stats()
    ctx.close()
    ms = np.array(st["tune_ms"])
    timed = np.flatnonzero(ms)
    if cand == 1:                      # one variant fits: nothing to time
        assert timed.size <= 1
        return
    assert timed.size == cand, (cand, st["tune_ms"])
    best = timed[np.argmin(ms[timed])]
    kept = st["sweep_tile"]
    assert kept[0] > 0 or kept == (0, 0, 0, 0), kept      # zeros: the staged kernels
    if kept in ENTRY:
        assert best in ENTRY[kept], (kept, st["tune_ms"])


@pytest.mark.parametrize("path,n,tile,entries", [
    ("auto", 32, (8, 8, 0), [5, 14]), ("fused", 32, (8, 8, 0), [5, 14]), ("auto", 32, (16, 8, 0), [12, 13]),
    ("fused", 24, (0, 0, 0), [5, 14])])
def test_fp64_tile_times_both_thread_counts(gpu_lib, path, n, tile, entries):
    """Where an FP64 MHD mesh runs one tile, asked for by kr_config.tile or the
    only one that fits, both of its builds are timed."""
    spec = kratos_amd.MeshSpec((2 * n, 2 * n, n), (n, n, n))
    u, b, _ = problems.turbulence(spec.n_cell_global, seed=5)
    ctx = kratos_amd.Context(spec, kratos_amd.Physics(mhd=True), "fp64", path=path, tile=tile)
    ctx.upload(u, b)
    ctx.advance(4)
    st = ctx.stats()
    ctx.close()
    assert list(np.flatnonzero(st["tune_ms"])) == entries
    assert st["sweep_tile"][:2] == (tile[:2] if tile[0] else (8, 8))
