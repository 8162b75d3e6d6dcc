"""Dense grids that fit the device only without the build's densities by leaf (4 B per voxel
of temporaries) are built without them, to the same grid.  The build runs in a child process
whose device allocations fail beyond a budget (tight_hip.cpp, preloaded)."""
import os
import subprocess
import sys
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent

pytestmark = pytest.mark.gpu

BODY = """
import ctypes as C
import numpy as np
import renderer2_amd as r2

tight = C.CDLL(None)
for f in ("used", "peak"):
    getattr(tight, "tight_hip_" + f).restype = C.c_size_t
tight.tight_hip_set_budget.argtypes = [C.c_size_t]
ctx = r2.Context(0)
rng = np.random.default_rng(1)


def state(g, shape):
    nz, ny, nx = shape
    at = np.stack(np.meshgrid(np.arange(-1, nx + 1), np.arange(-1, ny + 1), np.arange(-1, nz + 1), indexing="ij"), -1)
    ranges, atlas, mips = g.download_bricks()
    info = g.info()
    return [ranges, atlas, *mips, g.lookup(at.reshape(-1, 3).astype(np.int32)), g.sample(np.random.default_rng(2).random((500, 3), np.float32)),
            *[np.asarray(info[k]) for k in sorted(info)]]


for shape, precision, cut in (((64, 64, 64), "fp32", 0.0), ((90, 70, 130), "packed", 0.6), ((90, 33, 41), "fp32", 0.9)):
    rec = rng.integers(0, 256, (*shape, 32), dtype=np.uint8)
    rec[..., 28:32] = 0
    rec[..., 29] = 0x3C
    dens = np.maximum(rng.random(shape, dtype=np.float32) - cut, 0).astype(np.float32)
    dens[:, :, shape[2] // 2:] = 0
    rec[..., :4] = dens[..., None].view(np.uint8)
    d = dict(records=rec, shape=shape, map_mat=(0.1, 0, 0, 0, 0.1, 0, 0, 0, 0.1), map_vec=(0, 0, 0), sigma_a=(0.1,) * 3,
             sigma_s=(0.9,) * 3, voxel_size_filtering=0.1, precision=precision)
    ctx.trim()
    start = tight.tight_hip_used()
    tight.tight_hip_reset_peak()
    g = ctx.upload_grid(d)
    peak = tight.tight_hip_peak()
    want = state(g, shape)
    g.free()
    ctx.trim()
    assert tight.tight_hip_used() == start
    by_leaf = int(np.prod([(n + 7) // 8 for n in shape])) * 512 * 4
    tight.tight_hip_set_budget(peak - by_leaf // 2)
    refused = tight.tight_hip_refused()
    g = ctx.upload_grid(d)
    assert tight.tight_hip_refused() > refused, "the budget was never reached"
    tight.tight_hip_set_budget((1 << 64) - 1)
    got = state(g, shape)
    assert all(a.tobytes() == b.tobytes() for a, b in zip(want, got)), shape
    g.free()
    # too little for either: the error is the device's memory, and nothing is lost
    ctx.trim()
    tight.tight_hip_set_budget(start + rec.nbytes)
    try:
        ctx.upload_grid(d)
        raise SystemExit("built in too little memory")
    except r2.R2Error as e:
        assert "R2_ERR_OOM" in str(e), e
    tight.tight_hip_set_budget((1 << 64) - 1)
    ctx.trim()
    assert tight.tight_hip_used() == start
    print(shape, precision, "built in", peak - by_leaf // 2 - start, "instead of", peak - start, "bytes", flush=True)
print("DONE")
"""


def test_dense_grids_build_without_densities_by_leaf(tmp_path):
    so = tmp_path / "libtight_hip.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I/opt/rocm/include", str(HERE / "tight_hip.cpp"),
                    "-o", str(so), "-ldl", "-L/opt/rocm/lib", "-Wl,-rpath,/opt/rocm/lib", "-Wl,--no-as-needed",
                    "-lamdhip64"], check=True)  # linked, so that the next definition after it is the runtime's
    preload = ":".join(x for x in (str(so), os.environ.get("LD_PRELOAD")) if x)
    env = dict(os.environ, LD_PRELOAD=preload, PYTHONPATH=os.pathsep.join([str(HERE.parent), str(HERE)]))
    r = subprocess.run([sys.executable, "-c", BODY], env=env, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "DONE" in r.stdout, r.stdout + r.stderr[-3000:]
    print(r.stdout)
