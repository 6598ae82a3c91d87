"""The wave-level traversal at its edges, against the oracle: queues of fewer
rays than a wave, of one wave and around multiples of 64 (claims of a queue),
clouds of one leaf, of a few leaves and of leaves with fewer than four
surfels, a top level too large for its copy in LDS, degenerate surfels (NaN
normals, whose tests accept a NaN distance), and entry buffers that waves
claim ahead of use and that overflow.

Hits, deposits and images are the same expressions in the same order on both
sides (bit-exact); gradients within 1e-4 of the largest (order of FP32
atomics), the repository's bars.
"""
import numpy as np
import pytest

from differentiablepointrendering_amd import scene

pytestmark = pytest.mark.gpu


def _pair(spec, settings):
    from differentiablepointrendering_amd.pale import Renderer
    from oracle.oracle import Oracle

    print(f"case: n={len(spec.points['position'])} meshes={len(spec.meshes)} settings={settings}", flush=True)
    return Renderer.from_spec(spec, settings), Oracle.from_spec(spec, settings)


def _check(gpu, orc, backward=True):
    a, b = gpu.render_forward()["camera1_raw"], orc.render_forward()["camera1_raw"]
    pa, pb = gpu.photons(), orc.photons()
    assert pa["count"] == pb["count"] and pa["attempted"] == pb["attempted"]
    for k in ("position", "power", "direction"):
        assert np.array_equal(pa[k], pb[k]), k
    assert np.array_equal(a, b, equal_nan=True)
    if backward:
        dl = (a[..., :3] / a[..., :3].size).astype(np.float32)
        g = gpu.render_backward({"camera1": dl})[0]["opacity"]
        want = orc.render_backward({"camera1": dl})
        assert np.allclose(g, want, rtol=1e-4, atol=1e-4 * (float(np.abs(want).max()) or 1.0))


@pytest.mark.parametrize("photons", [1, 63, 64, 65, 127, 129, 1000])
@pytest.mark.parametrize("size", [(1, 1), (9, 7), (65, 1)])
def test_queue_sizes(photons, size):
    spec = scene.config_scene(0, n=700, width=size[0], height=size[1])
    gpu, orc = _pair(spec, dict(photons=photons, gather_passes=2, adjoint_passes=2))
    _check(gpu, orc)


@pytest.mark.parametrize("n", [1, 3, 4, 5, 11, 13, 50])
def test_leaf_sizes(n):
    pts = scene.uniform_surfels(n, seed=3, scale_lo=0.3, scale_hi=0.6)[0]
    spec = scene.SceneSpec([scene.light_quad()], [scene.default_camera(40, 24)], pts,
                           dict(photons=3000, bounces=4, forward_passes=2, gather_passes=3, adjoint_bounces=4,
                                adjoint_passes=2, seed=5, gather_radius=0.2, spp_decorrelate=1))
    gpu, orc = _pair(spec, {})
    _check(gpu, orc)


@pytest.mark.parametrize("meshes", [7, 8, 20])
def test_top_level_beside_its_lds_copy(meshes):
    spec = scene.config_scene(0, n=300, width=40, height=32)
    for i in range(meshes - 1):
        a = 2.0 * np.pi * i / (meshes - 1)
        spec.meshes.append(scene.quad_mesh(f"q{i}", (1.2 * np.cos(a), -1.1 + 0.02 * i, 1.2 * np.sin(a)),
                                           scene.FACING_UP, 0.25, (0.6, 0.5, 0.4)))
    gpu, orc = _pair(spec, dict(photons=4000, gather_passes=2, adjoint_passes=2))
    _check(gpu, orc)


def test_degenerate_surfels_accept_nan_distances():
    pts = scene.uniform_surfels(40, seed=4, scale_lo=0.2, scale_hi=0.4)[0]
    pts["tangent_v"][[3, 17, 18]] = pts["tangent_u"][[3, 17, 18]]  # no plane: normalize(0)
    spec = scene.SceneSpec([scene.light_quad()], [scene.default_camera(24, 24)], pts, {})
    gpu, orc = _pair(spec, dict(photons=100))
    rng = np.random.default_rng(1)
    o = rng.uniform(-1.5, 1.5, size=(3000, 3)).astype(np.float32)
    d = rng.normal(size=(3000, 3)).astype(np.float32)
    a, b = gpu.trace_rays(o, d), orc.trace(o, d)
    for k in ("instance", "primitive"):
        assert np.array_equal(a[k], b[k]), k
    # The same through the wave traversal: one-layer photon map over the cloud.
    gpu, orc = _pair(spec, dict(photons=2000, bounces=1, forward_passes=1, gather_passes=1))
    gpu.build_photon_map()
    orc.build_photon_map()
    pa, pb = gpu.photons(), orc.photons()
    assert pa["count"] == pb["count"]
    assert np.array_equal(pa["position"], pb["position"], equal_nan=True)


@pytest.mark.parametrize("budget", [8, 9, 16, 60])
def test_entry_claims_and_their_holes(budget):
    pts = scene.uniform_surfels(30_000, seed=6, scale_lo=0.03, scale_hi=0.08)[0]  # about 20 layers per pixel
    spec = scene.SceneSpec([scene.light_quad()], [scene.default_camera(150, 90)], pts,
                           dict(photons=5000, bounces=3, forward_passes=1, gather_passes=3, adjoint_passes=1,
                                gather_radius=0.05, spp_decorrelate=1))
    from differentiablepointrendering_amd.pale import Renderer

    print(f"case: entries per pixel {budget}", flush=True)
    want = Renderer.from_spec(spec, dict(gather_entry_budget=1)).render_forward()["camera1_raw"]  # claims nothing ahead
    r = Renderer.from_spec(spec, dict(gather_entry_budget=budget))
    got = r.render_forward()["camera1_raw"]
    rounds = r.stats()["camera_rounds"]
    assert np.array_equal(got, want)
    assert rounds > 1 if budget < 10 else rounds >= 1


@pytest.mark.parametrize("radius", [0.004, 0.02, 0.11, 0.7])
@pytest.mark.parametrize("offset", [0.0, 37.0])
def test_gather_rows_against_all_photons(radius, offset):
    """The row bounds of the gather skip no accepted photon: irradiance at
    points around the photons, at cell faces, at distance r of a photon and
    outside the grid equals the oracle's walk over the reference's whole box,
    also far from the origin, where the coordinates' rounding is a larger part
    of a cell."""
    pts = scene.uniform_surfels(2000, seed=8, scale_lo=0.05, scale_hi=0.1)[0]
    pts["position"] = (pts["position"] + np.float32(offset)).astype(np.float32)
    light = scene.light_quad()
    light.object_to_world[:3, 3] += offset
    light.world_to_object = np.linalg.inv(light.object_to_world.astype(np.float64)).astype(np.float32)
    spec = scene.SceneSpec([light], [scene.default_camera(8, 8)], pts, {})
    gpu, orc = _pair(spec, dict(photons=4000 if radius > 0.5 else 20_000, bounces=3, forward_passes=1,
                                gather_radius=radius))
    gpu.build_photon_map()
    orc.build_photon_map()
    p = gpu.photons()["position"]
    rng = np.random.default_rng(2)
    near = p[rng.integers(0, len(p), 3000)]
    d = rng.normal(size=(3000, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    on = near + radius * d * rng.choice([0.3, 0.999999, 1.0, 1.000001, 1.4], size=(3000, 1))
    cell = 0.5 * radius
    lo = p.min(axis=0)
    faces = lo + np.round((near - lo) / cell) * cell
    out = near + 4.0 * (near - p.mean(axis=0))
    q = np.concatenate([near, on, faces, out]).astype(np.float32)
    n = rng.normal(size=q.shape)
    n = (n / np.linalg.norm(n, axis=1, keepdims=True)).astype(np.float32)
    assert np.array_equal(gpu.gather_irradiance(q, n), orc.gather(q, n))


@pytest.mark.parametrize("n", [6, 9, 17, 33, 37, 70, 515, 4099, 70_001])
def test_quad_nodes_over_tree_shapes(n):
    """Trees whose levels pair up in every way (odd and even depths, leaves
    beside subtrees) and both builds: closest hits, ties by leaf order, and the
    photon map through the two-level steps equal the oracle's binary walk."""
    pts = scene.uniform_surfels(n, seed=n, scale_lo=0.02 if n > 4000 else 0.1, scale_hi=0.05 if n > 4000 else 0.3)[0]
    # coincident surfels: exact ties in distance go to the leaf visited first
    for k in pts:
        pts[k][1::5] = pts[k][0::5][:len(pts[k][1::5])]
    spec = scene.SceneSpec([scene.light_quad()], [scene.default_camera(32, 24)], pts,
                           dict(photons=3000, bounces=3, forward_passes=1, gather_passes=2, adjoint_bounces=3,
                                adjoint_passes=1, gather_radius=0.1, spp_decorrelate=1))
    gpu, orc = _pair(spec, {})
    rng = np.random.default_rng(3)
    o = rng.uniform(-1.2, 1.2, size=(4000, 3)).astype(np.float32)
    d = rng.normal(size=(4000, 3)).astype(np.float32)
    d[::7, 0] = 0.0  # axis-parallel rays
    d[::11, 1:] = 0.0
    d = (d / np.maximum(np.linalg.norm(d, axis=1, keepdims=True), 1e-6)).astype(np.float32)
    a, b = gpu.trace_rays(o, d), orc.trace(o, d)
    for k in ("instance", "primitive", "t", "position"):
        assert np.array_equal(a[k], b[k]), k
    _check(gpu, orc)


@pytest.mark.parametrize("photons", [1, 1023, 1024, 1025, 65 * 1024 - 1, 70 * 1024 + 3])
@pytest.mark.parametrize("capacity", [0, 900])
def test_queue_compaction_tiles(photons, capacity):
    """Survivors, deposits and gradient events keep queue order across the
    tiles of the compaction: one tile, a tile's edge, more tiles than one look
    back window, queues that run empty before the last bounce, and a photon map
    that fills in the middle of a tile (the reservoir's draws follow)."""
    pts = scene.uniform_surfels(3000, seed=2, scale_lo=0.03, scale_hi=0.1)[0]
    spec = scene.SceneSpec([scene.light_quad()], [scene.default_camera(300, 230)], pts,
                           dict(photons=photons, bounces=12, forward_passes=2, gather_passes=1, adjoint_bounces=9,
                                adjoint_passes=2, seed=3, gather_radius=0.05, spp_decorrelate=1,
                                photon_map_capacity=capacity))
    gpu, orc = _pair(spec, {})
    _check(gpu, orc, backward=photons == 70 * 1024 + 3)


def test_queue_beyond_the_grid():
    """More rays and pixels than the device holds lanes (8 waves on each of
    1024 SIMDs at most): after the units that the waves start with come those
    claimed region by region, the last ones ragged."""
    spec = scene.config_scene(0, n=500, width=1031, height=691)
    gpu, orc = _pair(spec, dict(photons=700_001, bounces=2, gather_passes=1, adjoint_passes=1, adjoint_bounces=2,
                                gather_radius=0.02))
    _check(gpu, orc)


@pytest.mark.parametrize("size", [(1, 1), (127, 129), (128, 128), (29, 565), (257, 255)])
@pytest.mark.parametrize("radius", [0.3, 0.0118, 0.004])
def test_scans_and_sort_buckets(size, radius):
    """Scans of pixels and cells at the edges of a tile (16384 items, the last
    vector of four cut off at every place), and sorts by whole cells (0.3) and
    by runs of cells where the grid has more cells than the entries have places
    (up to 125M against 65,536)."""
    pts = scene.uniform_surfels(1500, seed=6, scale_lo=0.04, scale_hi=0.1)[0]
    spec = scene.SceneSpec([scene.light_quad()], [scene.default_camera(*size)], pts,
                           dict(photons=5000, bounces=3, forward_passes=1, gather_passes=1, adjoint_bounces=3,
                                adjoint_passes=1, gather_radius=radius, spp_decorrelate=1))
    gpu, orc = _pair(spec, {})
    _check(gpu, orc)


@pytest.mark.parametrize("full", [0, 1])
def test_default_adjoint_batches(full):
    """The default batch of several samples of a large view (16 x 640x512 rays,
    an event pool of fewer bounces than the samples have) gives the gradients
    of one sample per batch: sums in another order, 1e-4 of the largest."""
    from differentiablepointrendering_amd.pale import Renderer

    pts = scene.uniform_surfels(3000, seed=4, scale_lo=0.05, scale_hi=0.15)[0]
    spec = scene.SceneSpec([scene.light_quad()], [scene.default_camera(64, 64)], pts,
                           dict(photons=20_000, bounces=3, forward_passes=1, gather_passes=1, adjoint_bounces=20,
                                adjoint_passes=1, gather_radius=0.05, full_gradients=full, adjoint_decorrelate=1))
    print(f"case: full={full}", flush=True)
    r = Renderer.from_spec(spec, {})
    r.render_forward()
    cam = scene.default_camera(640, 512)
    rng = np.random.default_rng(1)
    dl = rng.normal(size=(512, 640, 3)).astype(np.float32)
    grads = []
    for slots in (0, 640 * 512):
        r.set_batch_tuning(slots_per_batch=slots)
        grads.append(r.render_view_backward(cam, 16, dl))
    for k in grads[0]:
        a, b = grads[0][k], grads[1][k]
        assert np.allclose(a, b, rtol=1e-4, atol=1e-4 * (float(np.abs(b).max()) or 1.0)), k
