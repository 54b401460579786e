"""The device's light-tree descent over the nodes it prepares per scene:
trees of one leaf up to several levels, with boxes without extent (lights on
one point), spot cones beside all-round nodes and powers twelve decades
apart.  Every path must choose the light that the integrator's tree chooses;
the bounds are those of the mixed-emitter comparison (binary32 shading
against binary64, 1e-4 on 99.9% of the pixels)."""
import numpy as np
import pytest

from vitrum_amd import workloads as W

from render_cases import SEED, cpu_frames, floor_with_emitters

pytestmark = pytest.mark.gpu


def _lights(n):
    rng = np.random.default_rng(n)
    out = []
    for k in range(n):
        pos = [0.2, 1.5, -0.1] if k % 3 == 0 else [float(x) for x in rng.uniform([-3, 0.5, -3], [3, 3, 3])]
        e = {"kind": "point", "color": [1, 1, 1], "intensity": float(10.0 ** rng.uniform(-6, 6)), "position": pos}
        if k % 2:
            e = dict(e, kind="spot", direction=[0.2, -1.0, 0.1 * k], angle=0.7, penumbra=0.2)
        out.append(e)
    return out


@pytest.mark.parametrize("n", [1, 2, 3, 33])
def test_descent_picks_the_integrators_light(engine, n):
    sc = floor_with_emitters(_lights(n), view_deg=20.0, fov=1.2)
    res = 32
    engine.set_scene(sc)
    engine.reset()
    engine.render_frame(W.inv_view_proj(sc["camera"], res, res), res, res, 0, SEED, 3)
    gpu = engine.capture(res, res)[..., :3].astype(np.float64)
    cpu, csig = cpu_frames(sc, res, 1, engine.render_info()["ray_bias"], max_bounces=3)
    match = engine.capture_signatures(res, res) == csig[0]
    assert match.mean() >= 0.999, match.mean()
    ok = (np.abs(gpu - cpu[0]) <= 1e-4 * np.abs(cpu[0]) + 1e-7).all(axis=2) | ~match
    assert ok.mean() >= 0.999, ok.mean()
    assert gpu.max() > 0
