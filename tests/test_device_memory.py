"""The library's handling of device memory, on the CPU: the host code runs over a preloaded
stand-in for the HIP runtime (fake_hip.cpp) whose device memory has a budget and which refuses
launches beyond the runtime's limits.

* Blocks that a context keeps for its next grid are not lost to anything else: whatever
  allocation fails, of any entry point and any context of the device, gets them back first;
  they belong to the context's device.
* Host memory that runs out is an error code.
* Frames of every accepted shape can be post-processed."""
import os
import subprocess
import sys
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
PRELUDE = """
import ctypes as C
import numpy as np
import renderer2_amd as r2
from renderer2_amd import scenes

fake = C.CDLL(None)
fake.fake_hip_used.restype = C.c_size_t
fake.fake_hip_set_budget.argtypes = [C.c_int, C.c_size_t]


def sparse_grid(ctx, leaves=2):
    # kernels do nothing here: a grid given as leaves is the form that a build accepts
    d = dict(records=np.zeros((leaves, 512, 32), np.uint8), leaf_origins=np.arange(leaves)[:, None] * np.array([[8, 0, 0]], np.int32),
             shape=(8, 8, 8 * leaves), map_mat=(0.1, 0, 0, 0, 0.1, 0, 0, 0, 0.1), map_vec=(0, 0, 0), sigma_a=(0.1,) * 3,
             sigma_s=(0.9,) * 3, voxel_size_filtering=0.1)
    return ctx.upload_grid(d)


def fill_cache(ctx):
    # a grid of 256 MB is built and freed
    sparse_grid(ctx, 1000).free()


ctx = r2.Context(0)
grid, env = sparse_grid(ctx), ctx.upload_env(np.ones((8, 16, 3), np.float32))
cfg = dict(scenes.make_workload("c1", n=8)["render"], width=64, height=64, spp=1)
rng = np.random.default_rng(0)
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    so = tmp_path_factory.mktemp("fake") / "libfake_hip.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I/opt/rocm/include", str(HERE / "fake_hip.cpp"),
                    "-o", str(so)], check=True)
    return so


def run(fake, body):
    preload = ":".join(x for x in (str(fake), os.environ.get("LD_PRELOAD")) if x)
    env = dict(os.environ, LD_PRELOAD=preload, PYTHONPATH=os.pathsep.join([str(HERE.parent), str(HERE)]))
    r = subprocess.run([sys.executable, "-c", PRELUDE + body + "\nassert fake.fake_hip_bad_frees() == 0\nprint('DONE')"],
                       env=env, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "DONE" in r.stdout, r.stdout + r.stderr[-3000:]


CALLS = {
    "mesh": "ctx.upload_mesh(scenes.synth_mesh(24, 500))",
    "environment": "ctx.upload_env(np.ones((64, 128, 3), np.float32))",
    "scene table": "ctx.scene_intersect(cfg, [grid], [dict(grid=0)] * 6000, env, np.ones((4, 7), np.float32))",
    "paths": "ctx.render_paths(cfg, [grid], [dict(grid=0)], env, np.zeros(5000, np.int32), np.zeros(5000, np.int32))",
    "cells": "ctx.dda_cells(np.ones((500, 7), np.float32), 1.0, 0, 64)",
    "frame": "ctx.render(dict(cfg, width=640, height=480, spp=4), [grid], [dict(grid=0)], env)",
    "grid": "sparse_grid(ctx, 700)",
    "server": "ctx.server(hbm_budget_bytes=1 << 20).stop()",
    "another context": "r2.Context(0)",
    "another context's grid": "sparse_grid(other)",
    "another context's mesh": "other.upload_mesh(scenes.synth_mesh(24, 500))",
}


@pytest.mark.parametrize("call", CALLS)
def test_kept_blocks_come_back_when_an_allocation_fails(fake, call):
    run(fake, f"""
other = r2.Context(0)
fill_cache(ctx)
full = fake.fake_hip_used(0)
fake.fake_hip_set_budget(0, full)  # nothing fits any more but by giving blocks back
kept = {CALLS[call]}
""")


def test_trim_and_destroy_give_the_kept_blocks_back(fake):
    run(fake, """
before = fake.fake_hip_used(0)
fill_cache(ctx)
assert fake.fake_hip_used(0) > before + (1 << 24)
ctx.trim()
assert fake.fake_hip_used(0) <= before + 4096
other = r2.Context(0)
fill_cache(other)
other.close()
assert fake.fake_hip_used(0) <= before + 4096
""")


def test_blocks_of_lookups_belong_to_the_context_s_device(fake):
    # another device is the thread's current one when a context of device 0 answers
    run(fake, """
hip = C.CDLL(None)
for call in (lambda: grid.lookup(np.zeros((70000, 3), np.int32)), lambda: grid.sample(np.zeros((70000, 3), np.float32))):
    ctx.trim()
    before = fake.fake_hip_used(0)
    hip.hipSetDevice(1)
    call()
    assert fake.fake_hip_used(1) == 0
    assert fake.fake_hip_used(0) > before  # kept for the next call
    hip.hipSetDevice(0)
""")


# host memory that runs out inside the bookkeeping of blocks is an error code or nothing at
# all, never an exception through the C interface, and no device block is lost
@pytest.mark.parametrize("call", ["free", "sample", "lookup"])
def test_host_memory_running_out_ends_in_an_error_code(fake, call):
    run(fake, f"""
L = r2.capi.lib()
for k in range(4):
    ctx.trim()
    before = fake.fake_hip_used(0)
    g = sparse_grid(ctx, 40)
    pos, out = np.zeros((9, 3), np.float32), np.zeros((9, 17), np.float32)
    at, rec = np.zeros((9, 3), np.int32), np.zeros((9, 32), np.uint8)
    fake.fake_hip_fail_new(k)
    if "{call}" == "free":
        rc, g.h = L.r2_grid_free(ctx.h, g.h), None
    elif "{call}" == "sample":
        rc = L.r2_grid_sample(ctx.h, g.h, 9, pos.ctypes.data, out.ctypes.data)
    else:
        rc = L.r2_grid_lookup(ctx.h, g.h, 9, at.ctypes.data, rec.ctypes.data)
    fake.fake_hip_fail_new(-1)
    assert rc in (0, -3, -4), rc
    if g.h:
        g.free()
    ctx.trim()
    assert fake.fake_hip_used(0) == before, (k, fake.fake_hip_used(0), before)
""")


@pytest.mark.parametrize("w,h", [(1 << 28, 1), ((1 << 25) + 3, 7), (1, 1 << 28), (16384, 16384), (1, 1)])
def test_postprocess_launches_every_accepted_shape(fake, w, h):
    run(fake, f"""
L = r2.capi.lib()
p = C.create_string_buffer(64)  # kernels do nothing here: the frame is never read
rc = L.r2_postprocess(ctx.h, C.addressof(p), {w}, {h}, C.c_float(2.2), C.addressof(p), C.addressof(p), 1)
assert rc == 0, L.r2_last_error(ctx.h)
""")
