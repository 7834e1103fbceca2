"""kr_upload / kr_download of blocks of every shape: what comes back is what
went up, cell-centred B is the face average, and ghost faces are zeros in
arrays that held something else, whatever part of them the library moves
(thin axes, blocks of one and of several chunks of its buffer)."""
import numpy as np
import pytest

import kratos_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mhd", [True, False])
@pytest.mark.parametrize("blk", [(2, 1, 1), (64, 1, 1), (4096, 1, 1), (60001, 1, 1), (2, 2, 1), (5, 3, 1), (64, 48, 1),
                                 (300, 301, 1), (4, 4, 4), (5, 7, 3), (24, 24, 24), (23, 23, 23), (32, 16, 64)])
def test_round_trip(gpu_lib, mhd, blk):
    spec = kratos_amd.MeshSpec((2 * blk[0],) + blk[1:], blk)
    n, nv = blk, 8 if mhd else 5
    faces = [x + (x > 1) for x in n]
    dims = tuple(f + 4 for f in faces)[::-1] + (3,)
    rng = np.random.default_rng(3)
    inner = tuple(slice(2, 2 + f) for f in faces[::-1])
    ctx = kratos_amd.Context(spec, kratos_amd.Physics(mhd=mhd), "fp64")
    sent = []
    for i in range(2):
        u = rng.random(n[::-1] + (nv,))
        f = rng.random(dims) if mhd else None        # also in the ghost layers
        assert ctx.lib.kr_upload(ctx.h, i, u.ctypes.data, f.ctypes.data if mhd else None) == 0
        sent.append((u, f))
    for bf in (True, False) if mhd else (False,):
        for i, (u, f) in enumerate(sent):
            gu, gf = np.full(u.shape, 9.0), np.full(dims, 9.0)
            assert ctx.lib.kr_download(ctx.h, i, gu.ctypes.data, gf.ctypes.data if bf else None) == 0
            want = u.copy()
            if mhd:
                g = f[inner]
                for a in range(3):
                    lo = g[tuple(slice(0, x) for x in n[::-1]) + (a,)]
                    hi = np.roll(g[..., a], -1, 2 - a) if n[a] > 1 else g[..., a]
                    want[..., 5 + a] = (lo + hi[tuple(slice(0, x) for x in n[::-1])]) / 2
            assert np.array_equal(gu, want)
            if bf:
                full = np.zeros(dims)
                full[inner] = f[inner]
                assert np.array_equal(gf, full)
    ctx.close()
