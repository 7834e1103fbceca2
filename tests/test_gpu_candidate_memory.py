"""The array of cell-centred E that the staged kernels need where they are only
a candidate of the tuner: given back when they lose, and a mesh whose memory
ends at it runs the other candidates with the same state.  A program of its
own loads the library behind a hipMalloc / hipFree that watch one size."""
import json
import os
import shutil
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SHIM = r"""
#include <stddef.h>
static int (*real_malloc)(void **, size_t);
static int (*real_free)(void *);
static size_t watched;
static int refuse, asked;
static void *held;
void shim_set(void *m, void *f) {
    real_malloc = (int (*)(void **, size_t))m;
    real_free = (int (*)(void *))f;
}
void shim_watch(size_t n, int r) { watched = n; refuse = r; asked = 0; held = 0; }
int shim_asked(void) { return asked; }
int shim_held(void) { return held != 0; }
int hipMalloc(void **p, size_t n) {
    if (n != watched) return real_malloc(p, n);
    ++asked;
    if (refuse) return 2;                      /* hipErrorOutOfMemory */
    const int rc = real_malloc(p, n);
    if (rc == 0) held = *p;
    return rc;
}
int hipFree(void *p) {
    if (p && p == held) held = 0;
    return real_free(p);
}
"""
PROGRAM = r"""
import ctypes as C, json, sys
sys.path.insert(0, sys.argv[1])
hip = C.CDLL("libamdhip64.so")
shim = C.CDLL(sys.argv[2], mode=C.RTLD_GLOBAL)
shim.shim_set(C.cast(hip.hipMalloc, C.c_void_p), C.cast(hip.hipFree, C.c_void_p))
import numpy as np
import kratos_amd
from kratos_amd import problems
out = []
for blk, levels, precision in json.loads(sys.argv[3]):
    if levels == 1:
        spec = kratos_amd.MeshSpec(tuple(2 * n for n in blk), tuple(blk))
        blocks = spec.split(*problems.turbulence(spec.n_cell_global, seed=5)[:2])
    else:
        spec = kratos_amd.RefinedMeshSpec(tuple(4 * n for n in blk), tuple(blk), x_min=(-0.5,) * 3, x_max=(0.5,) * 3,
                                          refine=[(1, (-0.1,) * 3, (0.1,) * 3)])
        blocks = problems.smooth_blocks(spec, seed=2)
    size = spec.n_blocks * int(np.prod(blk)) * 3 * (4 if precision == "mixed" else 8)
    got, row = [], {}
    for refuse in (0, 1):
        shim.shim_watch(C.c_size_t(size), refuse)
        ctx = kratos_amd.Context(spec, kratos_amd.Physics(mhd=True), precision)
        ctx.upload_blocks(blocks)
        ctx.step()
        pending = [ctx.stats()["tune_pending"]]
        while pending[-1]:
            ctx.step()
            pending.append(ctx.stats()["tune_pending"])
        for _ in range(9 - len(pending)):
            ctx.step()
        got.append((ctx.download_blocks(), ctx.time()))
        tile = ctx.stats()["sweep_tile"]
        row["refused" if refuse else "given"] = {"asked": shim.shim_asked(), "held": shim.shim_held(),
                                                 "candidates": pending[0] + 1, "tile": tile}
        ctx.close()
        row["left"] = shim.shim_held()
    row["equal"] = got[0][1] == got[1][1] and all(
        np.array_equal(a, c) and np.array_equal(b, d) for (a, b), (c, d) in zip(got[0][0], got[1][0]))
    out.append(row)
print(json.dumps(out))
"""

CASES = [((16, 16, 16), 2, "fp64"), ((8, 8, 8), 2, "fp64"), ((20, 12, 10), 1, "fp64"), ((20, 12, 10), 1, "mixed"),
         ((9, 9, 6), 1, "mixed")]


def test_candidate_array_is_given_back(gpu_lib, tmp_path):
    if not shutil.which("gcc"):
        pytest.skip("no gcc")
    (tmp_path / "shim.c").write_text(SHIM)
    shim = str(tmp_path / "shim.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", str(tmp_path / "shim.c"), "-o", shim], check=True)
    run = subprocess.run([sys.executable, "-c", PROGRAM, ROOT, shim, json.dumps(CASES)], capture_output=True,
                         text=True, timeout=100)
    assert run.returncode == 0, run.stderr
    for case, row in zip(CASES, json.loads(run.stdout.splitlines()[-1])):
        print(case, row)
        given, refused = row["given"], row["refused"]
        assert given["asked"] == refused["asked"] == 1, (case, row)
        assert given["held"] == (given["tile"][0] == 0), (case, row)
        assert refused["tile"][0] > 0 and refused["candidates"] == given["candidates"] - 1, (case, row)
        assert row["left"] == 0 and row["equal"], (case, row)
