"""FP64 HLLD on transverse velocities and fields down to the smallest
subnormals, bit for bit against the oracle.  With a strong field along x the
double-star velocity (m1 / q1 + m2 / q2) / (q1 + q2) is all there is of the
transverse momentum flux, so every bit of those quotients shows."""
import numpy as np
import pytest

import kratos_amd
import oracle
from kratos_amd import problems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path", ["fused", "staged"])
@pytest.mark.parametrize("scale", [1e-321, 3e-320, 1e-318, 1e-315, 1e-308, 1e-290, 1e-258])
def test_tiny_transverse_fp64(gpu_lib, scale, path):
    N, gamma = (128, 8, 4), 5.0 / 3.0
    rng = np.random.default_rng(13)
    spec = kratos_amd.MeshSpec(N, (64, 8, 4))
    phys = kratos_amd.Physics(mhd=True, gamma=gamma)
    shape = tuple(reversed(N))
    # a function of x, so that y and z stay tiny; a quantum of m / q is several
    # of rho (m / q)
    r = np.broadcast_to(30 + 3 * rng.random(N[0]), shape)
    v = [np.broadcast_to(s * rng.standard_normal(N[0]), shape) for s in (0.3, scale, scale)]
    b = []
    for a, f in enumerate((3.0, scale, 0.0)):
        s = list(shape)
        s[2 - a] += 1
        b.append(np.full(s, f))
    e = problems.total_energy(r, r / gamma, v, problems.cell_centred_b(*b), gamma)
    u = np.stack([r, e] + [r * c for c in v])
    ctx = kratos_amd.Context(spec, phys, "fp64", path=path)
    ctx.upload(u, tuple(b))
    ctx.advance(4)
    gu, gb = ctx.download()
    ctx.close()
    ref = oracle.OracleMesh(spec, phys)
    ref.upload(u, tuple(b))
    ref.advance(4)
    ou, ob = ref.download()
    assert 0 < np.abs(ou[3:]).max() < 1e3 * scale
    assert np.array_equal(gu, ou)
    assert all(np.array_equal(x, y) for x, y in zip(gb, ob))
