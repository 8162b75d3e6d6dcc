"""Frames keep their bits when the path program's control flow is rearranged.

The render kernels are compiled with fused multiply-adds.  In a sum of products the
compiler fuses by its own order of operands, which follows the blocks around the sum, so
moving code alone can turn the last bits of a direction, and with them single paths.  The
sums where that happened are written out; this test holds the frames of every kernel form
(one, a few and any number of instances, with and without surfaces, both record forms,
FP32 and compensated FP64 sums, DDA and tracking) to those recorded in
golden/frame_bits.npz, bit for bit, from r2_render and from the render server.

The recording was made with the library of commit 77486b4, whose kernels ran every scene of
more than one instance, and every scene with surfaces, in the general form:
    PYTHONPATH=.:oracle R2_LIB_PATH=<that librenderer2.so> python tests/test_gpu_frame_bits.py
"""
import functools
from pathlib import Path

import numpy as np
import pytest

from renderer2_amd import scenes

GOLDEN = Path(__file__).resolve().parent / "golden" / "frame_bits.npz"
SIDE = dict(width=32, height=24, spp=6)

pytestmark = pytest.mark.gpu


@functools.lru_cache(None)
def _base(name):
    if name == "one":
        return scenes.make_workload("c2", n=32, **SIDE)
    if name == "few":
        from test_gpu_instances import multi_instance_workload

        return multi_instance_workload(**SIDE)
    return scenes.forest_workload(40, ground=name == "forest on its ground", **SIDE)


def _one(packed=False, ground=False, **cfg):
    w = dict(_base("one"))
    if ground:
        w["render"] = dict(w["render"], cam_pos=(0.0, 0.7, 2.3), cam_look_at=(0.0, -0.15, 0.0))
    return _finish(w, packed, ground, -0.4, cfg)


def _few(packed=False, ground=False, **cfg):
    return _finish(dict(_base("few")), packed, ground, -0.6, cfg)


def _any(packed=False, ground=False, **cfg):
    w = dict(_base("forest on its ground" if ground else "forest"))
    return _finish(w, packed, False, 0.0, cfg)


def _finish(w, packed, ground, y, cfg):
    if packed:
        w["grids"] = [dict(g, precision="packed") for g in w["grids"]]
    if ground:
        ball = dict(shape="sphere", pos=(0.45, y + 0.25, 0.35), radius=0.25, diffuse=(0.6, 0.3, 0.1),
                    diffuse_roughness=0.5, specular=(0.9, 0.9, 0.9), alpha_x=0.2, alpha_y=0.35)
        cfg = dict(cfg, surfaces=[dict(scenes.GROUND, pos=(0.0, y, 0.0)), ball])
    w["render"] = dict(w["render"], **cfg)
    return w


FORMS = {f"{name}{'_ground' if g else ''}{'_packed' if p else ''}{'_fp64' if d else ''}":
         (lambda fn=fn, g=g, p=p, d=d: fn(packed=p, ground=g, fp64_accum=d))
         for name, fn in (("one", _one), ("few", _few), ("any", _any))
         for g, p, d in ((False, False, False), (True, False, False), (False, True, False), (False, False, True),
                         (True, True, False), (True, False, True))}
FORMS["one_tracking"] = lambda: _one(use_brick_grid=False)
FORMS["few_tracking"] = lambda: _few(use_brick_grid=False)


def _frame(ctx, w, server=False):
    grids, env = [ctx.upload_grid(g) for g in w["grids"]], ctx.upload_env(w["env"])
    if not server:
        return ctx.render(w["render"], grids, w["instances"], env)
    srv = ctx.server(max_inflight=2, slice_paths=1 << 13)
    try:
        return srv.wait(srv.submit(w["render"], grids, w["instances"], env))[0]
    finally:
        srv.stop()


@pytest.mark.parametrize("form", FORMS)
def test_frames_keep_their_bits(ctx, form):
    want = np.load(GOLDEN)[form]
    w = FORMS[form]()
    got = _frame(ctx, w)
    assert np.isfinite(want).all() and want.mean() > 0
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), \
        f"{form}: {np.mean(got != want):.4f} of the values differ, relative {np.linalg.norm(got - want) / np.linalg.norm(want):.1e}"
    assert np.array_equal(_frame(ctx, w, server=True).view(np.uint32), want.view(np.uint32)), f"{form}: server"


@pytest.mark.parametrize("form", FORMS)
def test_frames_are_the_sums_of_their_paths(ctx, form):
    """A frame of one sample per item is the sum of its paths in sample order.  The path
    probe, which the other tests compare with the oracle path by path, runs the counting
    kernels (one or any number of instances); the frame runs the form of its scene."""
    w = FORMS[form]()
    cfg = w["render"]
    grids, env = [ctx.upload_grid(g) for g in w["grids"]], ctx.upload_env(w["env"])
    n, spp = cfg["width"] * cfg["height"], cfg["spp"]
    pix = np.repeat(np.arange(n, dtype=np.int32), spp)
    smp = np.tile(np.arange(spp, dtype=np.int32), n)
    paths = ctx.render_paths(cfg, grids, w["instances"], env, pix, smp).reshape(n, spp, 3)
    acc = np.zeros((n, 3), np.float64 if cfg.get("fp64_accum") else np.float32)
    for s in range(spp):
        acc += paths[:, s]
    frame = ctx.render(cfg, grids, w["instances"], env).reshape(n, 3)
    assert np.array_equal(acc.astype(np.float32), frame), form


if __name__ == "__main__":
    import sys

    import renderer2_amd as r2

    c = r2.Context(0)
    np.savez_compressed(sys.argv[1] if len(sys.argv) > 1 else GOLDEN, **{k: _frame(c, f()) for k, f in FORMS.items()})
