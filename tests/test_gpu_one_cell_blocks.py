"""Hydro blocks of one cell: no axis is active, so a cycle sweeps nothing
(geometry.cpp:46 counts the axes of more than one cell) and leaves the state
as it is, on every path that takes such blocks."""
import numpy as np
import pytest

import kratos_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("path", ["auto", "staged"])
@pytest.mark.parametrize("mesh", [(1, 1, 1), (4, 1, 1), (3, 4, 5)])
def test_state_stays(gpu_lib, mesh, path, precision):
    spec = kratos_amd.MeshSpec(mesh, (1, 1, 1))
    rng = np.random.default_rng(1)
    u = 1 + 0.1 * rng.random((5,) + mesh[::-1])
    u[1] += 10
    ctx = kratos_amd.Context(spec, kratos_amd.Physics(mhd=False), precision, path=path)
    ctx.upload(u, None)
    assert ctx.advance(3) == 3
    assert ctx.step() > 0
    assert np.array_equal(ctx.download()[0], u)
    ctx.close()
