"""The Node128 traversal kernel where its waves share work: launches of every
fill (one ray to several rays for each lane of the grid), so idle lanes walk
subtrees of busy lanes' rays, against the oracle, bit for bit -- closest hit
in each visiting order, any hit, and both with the path tracer's sided filter;
a scene of nearly coincident surfaces, whose near-ties a group has to walk
again alone; stacks deeper than LDS holds; and rays that are not finite.
"""
import numpy as np
import pytest

from oracle import oracle as O
from vitrum_amd import workloads as W

pytestmark = pytest.mark.gpu

FIELDS = ("prim", "inst", "t", "u", "v")


def _box():
    return W.cornell_scene(16384)


def _shells():
    """Three shells of one mesh, two of them 3e-7 apart, and a second
    instance coincident with the outer one."""
    v, i = W.octa_sphere(8, split=True)
    n = W._vertex_normals(v, i)
    v3 = np.concatenate([v, v * (1 + 3e-7), v * 0.9])
    i3 = np.concatenate([i, i + len(v), i + 2 * len(v)]).astype(np.uint32)
    cam = W.look_at_camera(eye=(0.0, 0.3, 2.5), target=(0.0, 0.0, 0.0), up=(0, 1, 0), vfov_deg=50.0)
    return {"primitives": [W._mesh(v3, np.concatenate([n, n, n]), i3, W.WHITE), W._mesh(v, n, i, W.RED)],
            "camera": cam, "scene_radius": 1.0}


@pytest.mark.parametrize("make", [_box, _shells])
def test_every_fill_matches_oracle(engine, make):
    sc = make()
    engine.set_scene(sc)
    pack = O.pack_scene([dict(p, material_id=i) for i, p in enumerate(sc["primitives"])])
    ps = O.PackedScene(pack)
    rays, st = W.primary_rays(sc["camera"], 256, 256, scene_radius=sc["scene_radius"])
    rays = np.concatenate([rays, W.bounce_rays(pack, rays, O.trace_closest(ps, rays), st, sc["scene_radius"])])
    rays = rays[np.random.default_rng(9).permutation(rays.size)]
    seg = rays.copy()  # any-hit rays of limited length
    seg["tmax"] = np.random.default_rng(10).uniform(0.05, 3.0, rays.size).astype(np.float32)
    flags = O.single_sided_flags(ps, [p["material"] for p in sc["primitives"]])
    want = {0: (O.trace_closest(ps, rays), O.trace_any(ps, seg)),
            1: (O.trace_closest_sided(ps, flags, rays), O.trace_occluded_sided(ps, flags, seg))}
    try:
        # one ray; a wave less and more than full; every wave one ray; a few
        # rays each; half of a full static fill (every wave helps from its
        # first step)
        for n in (1, 63, 64, 65, 4095, 16411, 70001, rays.size):
            for sided in (0, 1):
                engine.set_hit_filter(sided)
                for near in (0, 1, 2):
                    engine.set_trace_tuning(8, 16, near, 12)
                    got = engine.trace_closest(rays[:n])
                    for k in FIELDS:
                        assert np.array_equal(got[k].view(np.uint32), want[sided][0][k][:n].view(np.uint32)), (n, sided, near, k)
                assert np.array_equal(engine.trace_any(seg[:n]), want[sided][1][:n]), (n, sided)
    finally:
        engine.set_hit_filter(0)
        engine.set_trace_tuning(8, 16, 2, 12)


FILL = 256 * 8 * 128  # rays of one static fill: 8 workgroups of 128 on every CU of an MI355X


class _Device:
    """Traces through device buffers that hold no answer beforehand."""

    def __init__(self, engine, rays):
        self.e, self.n = engine, rays.size
        self.rays, self.out = engine.alloc(rays.nbytes), engine.alloc(rays.size * W.HIT_DTYPE.itemsize)
        engine.h2d(self.rays, rays)

    def close(self):
        self.e.free(self.rays)
        self.e.free(self.out)

    def _run(self, call, n, dtype):
        got = np.frombuffer(b"\x5a" * (n * np.dtype(dtype).itemsize), dtype).copy()
        self.e.h2d(self.out, got)
        call(self.rays, n, self.out)
        self.e.synchronize()
        self.e.d2h(got, self.out)
        return got

    def closest(self, n):
        return self._run(self.e.trace_closest_device, n, W.HIT_DTYPE)

    def any(self, n):
        return self._run(self.e.trace_any_device, n, np.uint32)


# Few triangles an instance and many: any-hit launches end in another order.
@pytest.mark.parametrize("make", [lambda: W.cornell_scene(2048), _box], ids=["small_meshes", "large_meshes"])
def test_past_the_static_fill_matches_oracle(engine, make):
    """More rays than the grid's lanes: waves fetch from the counter, without
    helpers until the supply ends, with a transposed end that is a part of the
    queue (first size) or its largest (second)."""
    sc = make()
    engine.set_scene(sc)
    pack = O.pack_scene([dict(p, material_id=i) for i, p in enumerate(sc["primitives"])])
    ps = O.PackedScene(pack)
    rays, st = W.primary_rays(sc["camera"], 128, 128, scene_radius=sc["scene_radius"])
    rays = np.concatenate([rays, W.bounce_rays(pack, rays, O.trace_closest(ps, rays), st, sc["scene_radius"])])
    rays = rays[np.random.default_rng(19).permutation(rays.size)]
    seg = rays.copy()
    seg["tmax"] = np.random.default_rng(20).uniform(0.05, 3.0, rays.size).astype(np.float32)
    flags = O.single_sided_flags(ps, [p["material"] for p in sc["primitives"]])
    sizes = (FILL + 4097, 3 * FILL + 777)
    want = {0: (O.trace_closest(ps, rays), O.trace_any(ps, seg)),
            1: (O.trace_closest_sided(ps, flags, rays), O.trace_occluded_sided(ps, flags, seg))}
    dev, dseg = _Device(engine, np.resize(rays, sizes[-1])), _Device(engine, np.resize(seg, sizes[-1]))
    try:
        for n in sizes:
            for sided in (0, 1):
                engine.set_hit_filter(sided)
                hits = np.resize(want[sided][0], n)
                for near in (0, 1, 2):
                    engine.set_trace_tuning(8, 16, near, 12)
                    got = dev.closest(n)
                    for k in FIELDS:
                        assert np.array_equal(got[k].view(np.uint32), hits[k].view(np.uint32)), (n, sided, near, k)
                assert np.array_equal(dseg.any(n), np.resize(want[sided][1], n)), (n, sided)
    finally:
        engine.set_hit_filter(0)
        engine.set_trace_tuning(8, 16, 2, 12)
        dev.close()
        dseg.close()


def _spine(near, far, ratio=1.5, seed=3):
    """Clusters of three triangles at distances ratio^k along +x, `near` of
    them in one mesh and each of the `far` others an instance: both trees are
    spines, and a ray from the origin goes down all of them with a sibling
    waiting at almost every level (86 entries at worst for 57 and 57)."""
    rng = np.random.default_rng(seed)
    n = near + far
    tri = rng.normal(size=(n, 3, 3, 3)) * [0.02, 0.04, 0.04]
    tri += rng.uniform(-0.25, 0.25, (n, 3, 1, 3)) * [0.2, 1.0, 1.0] + [1.0, 0.0, 0.0]
    tri *= (ratio ** np.arange(n))[:, None, None, None]

    def mesh(t):
        v = t.reshape(-1, 3)
        return W._mesh(v, np.tile([0, 1, 0], (len(v), 1)), np.arange(len(v), dtype=np.uint32).reshape(-1, 3), W.WHITE)

    return {"primitives": [mesh(tri[:near])] + [mesh(t) for t in tri[near:]], "scene_radius": float(ratio ** n)}


def test_deep_stacks_with_helpers(engine):
    """Stacks well past the 18 entries in LDS, whose bottom entries are given
    away and whose top is in the spill area."""
    sc = _spine(57, 57)
    engine.set_scene(sc)
    ps = O.PackedScene(O.pack_scene([dict(p, material_id=i) for i, p in enumerate(sc["primitives"])]))
    n, rng = 20000, np.random.default_rng(21)
    rays = np.zeros(n, W.RAY_DTYPE)
    d = np.concatenate([np.ones((n, 1)), rng.uniform(-0.22, 0.22, (n, 2))], 1)
    rays["d"] = W._unit_f32(d.astype(np.float32))
    rays["o"] = rng.uniform(-0.01, 0.01, (n, 3)).astype(np.float32)
    rays["tmin"], rays["tmax"] = 1e-4, W.TMAX_INFINITY
    ref, occ = O.trace_closest(ps, rays), O.trace_any(ps, rays)
    assert np.unique(ref["inst"]).size > 20 and 0.5 < occ.mean() < 0.9
    try:
        for near in (0, 1, 2):
            engine.set_trace_tuning(8, 16, near, 12)
            for count in (1, 100, 4097, n):
                got = engine.trace_closest(rays[:count])
                for k in FIELDS:
                    assert np.array_equal(got[k].view(np.uint32), ref[k][:count].view(np.uint32)), (near, count, k)
        for count in (1, 100, 4097, n):
            assert np.array_equal(engine.trace_any(rays[:count]), occ[:count]), count
    finally:
        engine.set_trace_tuning(8, 16, 2, 12)


def test_rays_that_are_not_finite(engine):
    """NaN, infinite, zero, denormal and huge components among usual rays:
    the records of the binary walk and of the oracle."""
    sc = W.cornell_scene(2048)
    engine.set_scene(sc)
    ps = O.PackedScene(O.pack_scene([dict(p, material_id=i) for i, p in enumerate(sc["primitives"])]))
    n, rng = 24000, np.random.default_rng(22)
    rays = np.zeros(n, W.RAY_DTYPE)
    rays["o"] = (np.array([0, 1, 0]) + rng.uniform(-0.9, 0.9, (n, 3))).astype(np.float32)
    rays["d"] = W._unit_f32(rng.normal(size=(n, 3)).astype(np.float32))
    rays["tmin"], rays["tmax"] = 1e-4, W.TMAX_INFINITY
    kind, axis = np.arange(n) % 24, np.arange(n) // 24 % 3
    odd = [("o", np.nan), ("o", np.inf), ("o", 3e38), ("d", np.nan), ("d", np.inf), ("d", -np.inf), ("d", 0.0), ("d", -0.0),
           ("d", 1e-45), ("d", 3e38), ("tmin", np.nan), ("tmin", np.inf), ("tmin", -1.0), ("tmax", np.nan),
           ("tmax", np.inf), ("tmax", 0.0)]
    for j, (field, value) in enumerate(odd):
        m = kind == j
        if rays[field].ndim == 2:
            rays[field][m, axis[m]] = value
        else:
            rays[field][m] = value
    m = (kind >= 6) & (kind <= 8)  # unit directions again, along an axis plane
    rays["d"][m] = np.where(np.abs(rays["d"][m]) <= 1e-45, rays["d"][m], W._unit_f32(rays["d"][m]))
    rays["d"][kind == 16] = 0.0
    rays["d"][kind == 17] *= np.float32(1e-30)
    rays["d"][kind == 18] *= np.float32(1e20)
    ref = O.trace_closest(ps, rays)
    try:
        for sided in (0, 1):
            engine.set_hit_filter(sided)
            for near in (0, 1, 2):
                engine.set_trace_tuning(8, 16, near, 12)
                got = {}
                for width in (2, 4):
                    engine.set_node_width(width)
                    got[width] = engine.trace_closest(rays), engine.trace_any(rays)
                for k in FIELDS:
                    assert np.array_equal(got[4][0][k].view(np.uint32), got[2][0][k].view(np.uint32)), (sided, near, k)
                    if not sided:
                        assert np.array_equal(got[4][0][k].view(np.uint32), ref[k].view(np.uint32)), (near, k)
                assert np.array_equal(got[4][1], got[2][1]), (sided, near)
    finally:
        engine.set_hit_filter(0)
        engine.set_node_width(4)
        engine.set_trace_tuning(8, 16, 2, 12)


def _grazing(n, seed):
    """A yawed box and rays that meet its faces at 1e-7 to 1e-2 rad, most near
    the edges and vertices of the grid: hits shared by two triangles and
    distances that the determinant hardly fixes."""
    rng = np.random.default_rng(seed)
    p, nn, i = W._merge([W._grid_quad(f[0], f[1], f[2], 20, 20, f[3])
                         for f in W._box_faces((-0.33, 0.6, -0.28), (0.56, 1.2, 0.56), 15.0)])
    sc = {"primitives": [W._mesh(p, nn, i, W.WHITE)], "scene_radius": 1.7}
    tri = p[i[rng.integers(0, len(i), n)]]
    b = rng.dirichlet([0.2, 0.2, 0.2], n)
    normal = np.cross(tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0])
    normal /= np.linalg.norm(normal, axis=1, keepdims=True)
    d = rng.normal(size=(n, 3))
    d -= normal * (d * normal).sum(1, keepdims=True)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    d -= normal * (10 ** rng.uniform(-7, -2, n))[:, None]
    rays = np.zeros(n, W.RAY_DTYPE)
    rays["d"] = W._unit_f32(d.astype(np.float32))
    rays["o"] = ((tri * b[:, :, None]).sum(1) - d * rng.uniform(0.01, 1.5, n)[:, None]).astype(np.float32)
    rays["tmin"], rays["tmax"] = 1e-4, W.TMAX_INFINITY
    return sc, rays


def test_grazing_hits_do_not_depend_on_the_group(engine):
    sc, rays = _grazing(40000, 4)
    engine.set_scene(sc)
    ps = O.PackedScene(O.pack_scene([dict(p, material_id=i) for i, p in enumerate(sc["primitives"])]))
    try:
        for near in (0, 1, 2):
            engine.set_trace_tuning(8, 16, near, 12)
            first = engine.trace_closest(rays)
            # 64 copies of a ray fill a wave and end together: no lane helps
            waves = FILL // 64
            for lo in range(0, 2 * waves, waves):
                alone = engine.trace_closest(np.repeat(rays[lo:lo + waves], 64))
                assert np.array_equal(np.repeat(first[lo:lo + waves], 64).view(np.uint8), alone.view(np.uint8)), near
            if near == 0:  # the reference's order is exact, ties included
                ref = O.trace_closest(ps, rays)
                for k in FIELDS:
                    assert np.array_equal(first[k].view(np.uint32), ref[k].view(np.uint32)), k
            for seed in range(3):  # other neighbours in the wave, other lanes to help
                order = np.random.default_rng(seed).permutation(rays.size)[: 40000 >> (2 * seed)]
                assert np.array_equal(engine.trace_closest(rays[order]).view(np.uint8),
                                      first[order].view(np.uint8)), (near, seed)
    finally:
        engine.set_trace_tuning(8, 16, 2, 12)


@pytest.mark.parametrize("extra", [-1, 0, 1, 63, 64, 65, 4097])
def test_every_ray_is_handed_out_once(engine, extra):
    """Queues around the ends of one fill of all waves (the order of the rays
    changes there) and past it, where the queue's end is transposed."""
    sc = W.cornell_scene(2048)
    engine.set_scene(sc)
    one = W.primary_rays(sc["camera"], 64, 64)[0]
    hits, occ = engine.trace_closest(one), engine.trace_any(one)
    for base in (FILL // 32, FILL):
        n = base + extra
        dev = _Device(engine, np.resize(one, n))
        try:
            assert np.array_equal(dev.closest(n).view(np.uint8), np.resize(hits, n).view(np.uint8)), n
            assert np.array_equal(dev.any(n), np.resize(occ, n)), n
        finally:
            dev.close()
