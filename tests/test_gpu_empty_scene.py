"""A scene without instances, bound after one that filled the result buffers:
every ray of a launch larger than the static first fill (2,048 workgroups of
128 lanes on an MI355X, half of that in later bounces) must be answered as a
miss, by itself, in a batch beside other scenes, and in a frame that sees the
sky alone."""
import numpy as np
import pytest

from vitrum_amd import native
from vitrum_amd import workloads as W

pytestmark = pytest.mark.gpu

BOX = W.cornell_scene(2048)
NOTHING = dict(BOX, primitives=[])
N_RAYS = 700_001


def _rays():
    return np.resize(W.primary_rays(BOX["camera"], 64, 64, scene_radius=BOX["scene_radius"])[0], N_RAYS)


def _all_miss(hits):
    return (hits["inst"] == 0xFFFFFFFF).all() and (hits["prim"] == 0xFFFFFFFF).all() and np.isinf(hits["t"]).all()


@pytest.mark.parametrize("sided", [0, 1])
def test_every_ray_misses(engine, sided):
    rays = _rays()
    try:
        engine.set_hit_filter(sided)
        engine.set_scene(BOX)
        assert not _all_miss(engine.trace_closest(rays))
        engine.set_scene(NOTHING)
        assert _all_miss(engine.trace_closest(rays))
        engine.set_scene(BOX)
        assert engine.trace_any(rays).any()
        engine.set_scene(NOTHING)
        assert not engine.trace_any(rays).any()
    finally:
        engine.set_hit_filter(0)


def test_batch_beside_other_scenes(engine):
    engine.set_scene(BOX)
    rays = _rays()
    want = engine.trace_closest(rays)
    a, b = N_RAYS // 3, N_RAYS // 2
    for part in (want[:a], want[b:]):
        part[:] = (0xFFFFFFFF, 0xFFFFFFFF, np.inf, 0, 0)
    batch = native.Batch(engine)
    d_r, d_h = engine.alloc(rays.nbytes), engine.alloc(want.nbytes)
    try:
        for sc in (NOTHING, BOX, NOTHING):
            batch.add_scene(sc)
        engine.h2d(d_r, rays)
        engine.h2d(d_h, np.zeros_like(want))
        batch.trace_closest_device(d_r, np.array([0, a, b, N_RAYS], np.uint32), d_h)
        got = np.zeros_like(want)
        engine.d2h(got, d_h)
        for k in ("prim", "inst", "t", "u", "v"):
            assert np.array_equal(got[k].view(np.uint32), want[k].view(np.uint32)), k
    finally:
        batch.close()
        engine.free(d_r)
        engine.free(d_h)


def test_frame_of_the_sky_alone():
    eng = native.Engine(0)
    try:
        ivp = W.inv_view_proj(BOX["camera"], 1920, 1080)
        eng.set_scene(BOX)
        eng.render_frame(ivp, 1920, 1080, 0)
        eng.set_scene(dict(NOTHING, sky=[0.25, 0.5, 1.0]))
        eng.render_frame(ivp, 1920, 1080, 0)
        img = eng.capture(1920, 1080)[..., :3]
        assert (img == np.float32([0.25, 0.5, 1.0])).all()
    finally:
        eng.close()
