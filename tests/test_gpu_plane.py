"""The one-launch stage of 2-D and 1-D meshes (path auto) against the staged
kernels, bit for bit in both precision forms: blocks below, at and past its
tile, one and several tiles, every kind of side; and the dt that c2p's last
workgroup takes: stop rule, top-up and per-box dt of small meshes against
the oracle and against the boxes alone."""
import numpy as np
import pytest

import kratos_amd
import oracle
from kratos_amd import problems

pytestmark = pytest.mark.gpu

PER = ("per",) * 6


def _state(N, mhd, seed, sides):
    if sides == PER:
        u, b, _ = problems.turbulence(N, seed=seed)
        return u, b if mhd else None
    u, b = problems.blast(N, p0=0.3, p_in=5.0, r_in=0.2, b0=(0.3, 0.5, 0.2) if mhd else (0, 0, 0))
    return u, b if mhd else None


def _run(spec, phys, u, b, precision, path, cycles=6):
    ctx = kratos_amd.Context(spec, phys, precision, path=path)
    ctx.upload(u, b)
    ctx.advance(cycles)
    out = ctx.download(), ctx.time()
    ctx.close()
    return out


def _same(x, y):
    assert np.array_equal(x[0], y[0])
    if x[1] is not None:
        assert all(np.array_equal(p, q) for p, q in zip(x[1], y[1]))


@pytest.mark.parametrize("mhd", [True, False])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("N,blk", [((7, 3, 1), (7, 3, 1)), ((16, 8, 1), (8, 8, 1)), ((18, 34, 1), (9, 17, 1)),
                                   ((40, 2, 1), (20, 2, 1)), ((124, 1, 1), (124, 1, 1)),
                                   ((250, 1, 1), (125, 1, 1)), ((12, 1, 1), (4, 1, 1))])
@pytest.mark.parametrize("sides", [PER, ("out", "ref", "fre", "out", "per", "per"),
                                   ("fixd", "out", "ref", "fre", "per", "per"),
                                   ("per", "per", "out", "fixd", "per", "per")])
def test_equals_staged(gpu_lib, mhd, precision, N, blk, sides):
    if N[1] == 1:
        sides = sides[:2] + ("per",) * 4
    spec = kratos_amd.MeshSpec(N, blk, bnd=sides)
    phys = kratos_amd.Physics(mhd=mhd, fix_w=(0.9, 0.4, 0.1, 0.05, -0.1), fix_b=(0.3, 0.5, 0.2))
    u, b = _state(N, mhd, 3, sides)
    one, t1 = _run(spec, phys, u, b, precision, "auto")
    ref, t2 = _run(spec, phys, u, b, precision, "staged")
    assert t1 == t2
    _same(one, ref)


@pytest.mark.parametrize("mhd", [True, False])
@pytest.mark.parametrize("N,blk", [((24, 20, 1), (12, 10, 1)), ((16, 16, 8), (16, 8, 8))])
def test_stop_and_top_up_fp64(gpu_lib, mhd, N, blk):
    """A run to t_lim with the top-up, past its end and resumed from there."""
    spec = kratos_amd.MeshSpec(N, blk)
    phys = kratos_amd.Physics(mhd=mhd, t_lim=0.05, top_up=True)
    u, b = _state(N, mhd, 5, PER)
    ref = oracle.OracleMesh(spec, phys)
    ref.upload(u, b)
    done = ref.advance(1000)
    ctx = kratos_amd.Context(spec, phys, "fp64")
    ctx.upload(u, b)
    assert ctx.advance(1000) == done
    assert ctx.time()[0] == 0.05
    assert ctx.step() == 0.0 and ctx.advance(3) == 0
    _same(ctx.download(), ref.download())
    ctx.set_time(0.0, 0.0)
    assert ctx.advance(2) == 2
    ctx.close()


@pytest.mark.parametrize("N", [(24, 20, 1), (16, 8, 8)])
def test_small_ensemble_own_dt(gpu_lib, N):
    """Small boxes of one context, each with its own dt, against the same
    boxes alone; the groups' arrivals do not mix."""
    spec = kratos_amd.MeshSpec(N, N)
    phys = kratos_amd.Physics(mhd=True, t_lim=0.04, top_up=True)
    ics = [problems.turbulence(N, seed=s, beta_range=(0.1, 10.0))[:2] for s in range(7)]
    ctx = kratos_amd.Context(spec, phys, "fp64", members=len(ics))
    for m, (u, b) in enumerate(ics):
        ctx.upload(u, b, member=m)
    ctx.advance(1000)
    for m, (u, b) in enumerate(ics):
        one = kratos_amd.Context(spec, phys, "fp64")
        one.upload(u, b)
        n = one.advance(1000)
        assert ctx.time(member=m)[2] == n
        _same(ctx.download(member=m), one.download())
        one.close()
    ctx.close()
