"""dt of a state with NaN in it.  The reduction keeps or drops a NaN by its
place; the place counts the same whether a launch of its own takes the dt or
the last workgroup of c2p does (meshes of up to 320 of them)."""
import numpy as np
import pytest

import kratos_amd

pytestmark = pytest.mark.gpu

FMAX = float(np.finfo(np.float32).max)


def _pmin(a, b):
    return np.where(a < b, a, b)


def _waves(v):
    """A workgroup's minimum: a butterfly in each wave of 64, then wave after wave."""
    v = np.array(v, float).reshape(-1, 64)
    for off in (32, 16, 8, 4, 2, 1):
        v = _pmin(v, v[:, np.arange(64) ^ off])
    m = v[0, 0]
    for x in v[1:, 0]:
        m = _pmin(m, x)
    return float(m)


@pytest.mark.parametrize("blocks", [(2, 2, 4), (5, 4, 1), (3, 7, 1)])
def test_nan_cells(gpu_lib, blocks):
    n = 16
    spec = kratos_amd.MeshSpec(tuple(n * b for b in blocks), (n, n, n))
    wgs = spec.n_blocks * 16                       # 256, 320: in c2p; 336: a launch
    rng = np.random.default_rng(wgs)
    base = np.zeros((n ** 3, 5))
    base[:, 0], base[:, 1] = 1.0, 1.5
    cases = [[]] + [[p] for p in (63, 127, 255, wgs - 1)] + [[63, wgs - 1], [127, 255]]
    cases += [sorted(rng.choice(wgs, 5, replace=False)) for _ in range(6)]
    ctx = kratos_amd.Context(spec, kratos_amd.Physics(mhd=False), "fp64")
    clean = None
    for parts in cases:
        blk = [base.copy() for _ in range(spec.n_blocks)]
        for p in parts:
            # the last thread of workgroup p: its NaN is what the workgroup reports
            blk[p // 16][(p % 16) * 256 + 255, 4] = np.nan
        ctx.upload_blocks([(u.reshape(-1), None) for u in blk])
        ctx.set_time(0.0, 0.0)
        dt = ctx.step()
        if clean is None:
            clean = dt
            assert 0 < clean < 1
            continue
        lanes = np.full(1024, FMAX)
        lanes[:wgs] = clean
        lanes[list(parts)] = np.nan
        want = _waves(lanes)
        seed = FMAX / 10                          # no dt seed given
        want = seed if np.isnan(want) else min(want, seed)
        assert dt == pytest.approx(want, rel=1e-12), (parts, dt, want)
    ctx.close()
