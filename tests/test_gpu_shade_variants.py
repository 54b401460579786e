"""The four builds of the shading kernel (sampler, with and without extension
lobes) at queue lengths around its workgroup of 256 entries: one path, less
than a wave, a few workgroups with a ragged last one.  Every kind of light is
in the scene.  Bounds as for the other frames against the binary64
integrator: 99.9% the same path decisions and of those 99.9% within 1e-4, so
at most 0.2% of the pixels may differ (none in the two small frames)."""
import numpy as np
import pytest

from vitrum_amd import native
from vitrum_amd import workloads as W

from render_cases import SEED, cpu_frames

pytestmark = pytest.mark.gpu


def _scene(lobes):
    sc = W.cornell_scene(2048)
    ext = dict(clearcoat=0.7, clearcoatRoughness=0.2, sheen=0.4, sheenRoughness=0.6, sheenColor=[0.9, 0.5, 0.4],
               anisotropy=0.5, roughness=0.4)
    prims = [dict(p, material=dict(p.get("material", {}), **(ext if lobes and i % 2 else {})))
             for i, p in enumerate(sc["primitives"])]
    lights = [{"kind": "directional", "color": [1, 1, 1], "intensity": 0.5, "direction": [0.3, -1, 0.2],
               "angularDiameter": 0.1},
              {"kind": "point", "color": [1, 0.5, 0.2], "intensity": 4, "position": [0.4, 1.5, 0]},
              {"kind": "spot", "color": [0.2, 0.5, 1], "intensity": 9, "position": [-0.4, 1.7, 0.2],
               "direction": [0, -1, 0], "angle": 0.8, "penumbra": 0.3},
              {"kind": "rect-area", "color": [1, 1, 1], "intensity": 2, "position": [0, 1.5, 0.4],
               "uAxis": [0.3, 0, 0], "vAxis": [0, 0, 0.3]},
              {"kind": "disc-area", "color": [1, 1, 0.5], "intensity": 3, "position": [0.3, 1.2, -0.4],
               "normal": [0, -1, 0], "radius": 0.2}]
    return dict(sc, primitives=prims, emitters=lights, sky=[0.05, 0.05, 0.06])


@pytest.fixture(scope="module", params=[0, 1], ids=["pcg", "sobol"])
def sampled(request):
    eng = native.Engine(0, sampling=request.param)
    yield eng, request.param
    eng.close()


@pytest.mark.parametrize("lobes", [False, True])
def test_every_build_matches_the_integrator(sampled, lobes):
    eng, sampling = sampled
    sc = _scene(lobes)
    eng.set_scene(sc)
    bias = eng.render_info()["ray_bias"]
    for res in (1, 7, 33):
        eng.reset()
        eng.render_frame(W.inv_view_proj(sc["camera"], res, res), res, res, 0, SEED, 6)
        gpu = eng.capture(res, res)[..., :3].astype(np.float64)
        cpu, csig = cpu_frames(sc, res, 1, bias, max_bounces=6, sampling=sampling)
        match = eng.capture_signatures(res, res) == csig[0]
        ok = match & (np.abs(gpu - cpu[0]) <= 1e-4 * np.abs(cpu[0]) + 1e-7).all(axis=2)
        assert (~ok).sum() <= int(res * res * 0.002), (res, (~match).sum(), (~ok).sum())
