"""The staged FP64 flux kernels use the flux functions without repeated
divisions: bit for bit against the oracle inside and outside the range these
are exact for, on blocks whose sizes leave remainders."""
import numpy as np
import pytest

import kratos_amd
import oracle
from kratos_amd import problems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mhd", [True, False])
@pytest.mark.parametrize("N,blk", [((16, 16, 8), (16, 8, 8)), ((18, 9, 7), (9, 9, 7)), ((24, 18, 1), (12, 9, 1)),
                                   ((40, 1, 1), (20, 1, 1))])
@pytest.mark.parametrize("vel,bscale,cell", [
    ((1, 1, 1), 1.0, None), ((1, 1e-200, 0), 1e-160, None), ((0, 0, 0), 1e-170, None), ((8, 0.1, 0.1), 1.0, None),
    ((1, 1, 1), 1.0, (1, 1e150)), ((1, 1, 1), 1.0, (1, np.nan)), ((1, 1, 1), 1.0, (3, 1e-250))])
def test_staged_fp64(gpu_lib, mhd, N, blk, vel, bscale, cell):
    gamma = 5.0 / 3.0
    rng = np.random.default_rng(5)
    spec = kratos_amd.MeshSpec(N, blk)
    shape = tuple(reversed(N))
    v = [0.5 * rng.standard_normal(shape) * a for a in vel]
    r = 1 + 0.3 * rng.random(shape)
    # a face field without divergence: each component constant along its axis
    b = []
    for a in range(3):
        s = list(shape)
        s[2 - a] = 1
        f = 0.4 * rng.standard_normal(s) * bscale
        s[2 - a] = N[a] + 1
        b.append(np.ascontiguousarray(np.broadcast_to(f, s)))
    b = tuple(b)
    e = problems.total_energy(r, r / gamma, v, problems.cell_centred_b(*b) if mhd else None, gamma)
    u = np.stack([r, e] + [r * c for c in v])
    if cell:
        u[(cell[0],) + tuple(n // 2 for n in shape)] = cell[1]
    if not mhd:
        b = None
    phys = kratos_amd.Physics(mhd=mhd)
    ctx = kratos_amd.Context(spec, phys, "fp64", path="staged")
    ctx.upload(u, b)
    ctx.advance(1)
    gu, gb = ctx.download()
    ctx.close()
    ref = oracle.OracleMesh(spec, phys)
    ref.upload(u, b)
    ref.advance(1)
    ou, ob = ref.download()
    assert np.array_equal(gu, ou, equal_nan=True)
    if mhd:
        assert all(np.array_equal(x, y, equal_nan=True) for x, y in zip(gb, ob))
