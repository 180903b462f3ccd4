"""Pool chunking: a film does not depend on the pool size, so every chunk
shape (one slot, less and more than a wave, several rows, the four-wave NEE
phase of large pools) must give the same bits; shadow-queue forms (one to
eight, sixteen and thirty-two light samples a vertex take different stripe
counts, more take the ungrouped queue) and odd image sizes (partial 8-row
strips) follow the oracle."""
import numpy as np
import pytest

from hierarchy_cases import instanced_scene
from raytracer import abi, native, scenes

pytestmark = pytest.mark.gpu


def _scene(W, H, samples):
    """A corner lit by area lights with `samples` shadow samples in all
    (squares of 1 and 4 a light).  Area lights are sampled without
    trigonometry: a sphere light's limb samples flip with the last bit of
    cosf, which differs between the device and the C library."""
    b = scenes.SceneBuilder()
    white = b.lambertian((0.7, 0.7, 0.7))
    shiny = b.disney((0.6, 0.3, 0.2), roughness=0.3)
    b.quad((-3, 0, -3), (0, 0, 6), (6, 0, 0), white)
    b.quad((-3, 0, -3), (6, 0, 0), (0, 6, 0), white)
    b.sphere((-0.6, 0.6, 0.0), 0.6, shiny)
    b.sphere((0.7, 0.4, 0.5), 0.4, white)
    left, k = samples, 0
    while left > 0:
        ss = 4 if left >= 4 else 1
        ang = 0.7 * k
        b.area_light((2.0 * np.cos(ang), 3.0 + 0.1 * k, 2.0 * np.sin(ang)), (0.3, 0.0, 0.0), (0.0, 0.0, 0.3),
                     intensity=12.0, shadow_samples=ss)
        left, k = left - ss, k + 1
    return b.build(scenes.make_camera((0.0, 1.5, 5.0), (0.0, 0.7, 0.0), 45.0, W / H))


def _film(sc, W, H, spp, pool, aovs=True):
    return native.Renderer(sc, spp, 4, paths_in_flight=pool).render(W, H, capture_aovs=aovs).buffers


PLANES = ("beauty", "beauty_a", "beauty_b", "albedo_a", "albedo_b", "normal_a", "normal_b", "depth_a", "depth_b")


@pytest.mark.parametrize("samples", [1, 8, 9, 17, 32, 40])
def test_pool_sizes_and_queue_forms(gpu_ctx, oracle, samples):
    W, H, spp = 37, 19, 3
    desc = _scene(W, H, samples)
    sc = native.Scene(gpu_ctx, desc)
    try:
        ref = _film(sc, W, H, spp, 0)
        for pool in (1 if samples == 1 else 61, 64, 65, 257, 1000):
            got = _film(sc, W, H, spp, pool)
            for k in PLANES:
                assert np.array_equal(getattr(ref, k), getattr(got, k)), (samples, pool, k)
        st = abi.settings_defaults(W, H, spp, 4)
        o = oracle.OracleScene(desc).render(st)["beauty"]
    finally:
        sc.close()
    err = np.abs(ref.beauty - o) / np.maximum(np.abs(o), 1e-2)
    print(f"{samples} samples a vertex: {np.mean(err < 1e-3):.4f} of the values within 1e-3, max {err.max():.2e}", flush=True)
    assert np.mean(err < 1e-3) > 0.99


@pytest.mark.parametrize("size", [(1, 1), (3, 200), (200, 3), (65, 8), (64, 9)])
def test_image_shapes(gpu_ctx, oracle, size):
    W, H = size
    desc = _scene(W, H, 2)
    sc = native.Scene(gpu_ctx, desc)
    try:
        ref = _film(sc, W, H, 5, 0)
    finally:
        sc.close()
    o = oracle.OracleScene(desc).render(abi.settings_defaults(W, H, 5, 4))["beauty"]
    err = np.abs(ref.beauty - o) / np.maximum(np.abs(o), 1e-2)
    assert np.mean(err < 1e-3) > 0.99, (size, err.max())


def test_wide_nee_pool(gpu_ctx):
    # 5.2 M samples: the default pool runs the NEE phase four waves wide
    W = H = 1024
    sc = native.Scene(gpu_ctx, _scene(W, H, 2))
    try:
        a = _film(sc, W, H, 5, 0, aovs=False)
        b = _film(sc, W, H, 5, 1 << 20, aovs=False)
    finally:
        sc.close()
    for k in ("beauty", "beauty_a", "beauty_b"):
        assert np.array_equal(getattr(a, k), getattr(b, k)), k


@pytest.mark.parametrize("aovs", [False, True])
def test_large_pool_shadow_runs(gpu_ctx, aovs):
    # 8.9 M samples of five light samples: the default pool's shadow waves work
    # through runs of the queue and refill their lanes; a 1 M pool's keep a ray
    # a lane
    W, H = 1920, 929
    desc = scenes.displaced_icosphere_scene(W, H, subdiv=4, sphere_lights=4)
    sc = native.Scene(gpu_ctx, desc)
    try:
        a = _film(sc, W, H, 5, 0, aovs=aovs)
        b = _film(sc, W, H, 5, 1 << 20, aovs=aovs)
    finally:
        sc.close()
    assert a.beauty.mean() > 0
    for k in ("beauty", "beauty_a", "beauty_b"):
        assert np.array_equal(getattr(a, k), getattr(b, k)), k


@pytest.mark.parametrize("name", ["cornell", "icosphere", "boxes"])
def test_lds_stack_renders_the_same(gpu_ctx, name):
    # the depth classes of the traversal stack (24, 32 and 64 entries)
    desc = {"cornell": lambda: scenes.cornell(64, 48),
            "icosphere": lambda: scenes.displaced_icosphere_scene(64, 48, subdiv=6),
            "boxes": lambda: scenes.batch_scene(60000, 64, 48, 5, 2)}[name]()
    sc = native.Scene(gpu_ctx, desc)
    try:
        a = _film(sc, 64, 48, 4, 0)
        gpu_ctx.tune(traversal_stack=2)
        b = _film(sc, 64, 48, 4, 0)
    finally:
        gpu_ctx.tune(traversal_stack=1)
        sc.close()
    for k in PLANES:
        assert np.array_equal(getattr(a, k), getattr(b, k)), (name, k)


@pytest.mark.parametrize("kind", ["flat", "instances", "batch"])
def test_closest_hits_of_small_and_large_pools(gpu_ctx, kind):
    # 525,312 samples: closest hits by four-wave workgroups; the 64 k pool's
    # by one-wave workgroups
    W, H, spp = 1024, 513, 1
    desc = instanced_scene(W, H) if kind == "instances" else _scene(W, H, 2)
    sc = native.Scene(gpu_ctx, desc)
    try:
        if kind == "batch":
            r = native.Renderer(sc, spp, 4)
            a, b = (native.render_batch([(r, W, H), (r, W, H)], pool_paths=n)[0][1].buffers for n in (0, 1 << 16))
        else:
            a, b = (_film(sc, W, H, spp, n, aovs=False) for n in (0, 1 << 16))
    finally:
        sc.close()
    assert a.beauty.mean() > 0
    for k in ("beauty", "beauty_a", "beauty_b"):
        assert np.array_equal(getattr(a, k), getattr(b, k)), k


@pytest.mark.parametrize("sampler", ["sobol", "prng"])
@pytest.mark.parametrize("W,H,spp,pools", [(65, 47, 5, (64, 1000, 0)), (1100, 1000, 4, (1 << 20, 0))])
def test_caustic_films_of_any_pool(gpu_ctx, sampler, W, H, spp, pools):
    # gather requests go through a queue with a stripe per XCD, filled by
    # one-wave chunks and in pools of 4 M slots (Sobol) by four-wave ones
    sc = native.Scene(gpu_ctx, scenes.caustics_scene(W, H, water_cells=20))
    try:
        films = [native.Renderer(sc, spp, 4, paths_in_flight=n, sampler=sampler, enable_caustics=True, caustic_photons=20000,
                                 caustic_gather_radius=0.05).render(W, H).buffers for n in pools]
    finally:
        sc.close()
    assert films[0].beauty.mean() > 0
    for f in films[1:]:
        assert np.array_equal(films[0].beauty, f.beauty)


def _mixed(W, H, samples):
    """_scene's corner with nested meshes among the tree's leaves, and an
    infinite plane at the top level beside the tree."""
    b = scenes.SceneBuilder()
    white = b.lambertian((0.7, 0.7, 0.7))
    shiny = b.disney((0.6, 0.3, 0.2), roughness=0.3)
    b.plane((0.0, 0.0, 0.0), (0.0, 1.0, 0.0), white)
    b.quad((-3, 0, -3), (6, 0, 0), (0, 6, 0), white)
    v, f = scenes.icosphere(3)
    for k in range(5):
        at = np.array([-1.6 + 0.8 * k, 0.45, 0.3 * (k % 2)])
        if k % 2 == 0:
            b.mesh(0.4 * v + at, f, shiny)
        else:
            b.sphere(at, 0.35, white)
    for k in range(samples):
        ang = 0.7 * k
        b.area_light((2.0 * np.cos(ang), 3.0 + 0.1 * k, 2.0 * np.sin(ang)), (0.3, 0.0, 0.0), (0.0, 0.0, 0.3),
                     intensity=12.0, shadow_samples=1)
    return b.build(scenes.make_camera((0.0, 1.5, 5.0), (0.0, 0.7, 0.0), 45.0, W / H))


@pytest.mark.parametrize("scene,samples", [("corner", 9), ("corner", 17), ("corner", 40), ("mixed", 5), ("mixed", 7)])
def test_large_pool_shadow_runs_of_queue_forms(gpu_ctx, scene, samples):
    # 8.4 M samples of at least 5 light samples: runs with refilled lanes, of 8,
    # 4 and 2 stripes and of the ungrouped queue, and of rays that leave the
    # tree for top-level entries and nested ones
    W, H = 1024, 512
    sc = native.Scene(gpu_ctx, (_scene if scene == "corner" else _mixed)(W, H, samples))
    try:
        a, b = (native.Renderer(sc, 16, 2, paths_in_flight=n).render(W, H).buffers for n in (0, 1 << 20))
    finally:
        sc.close()
    assert a.beauty.mean() > 0
    for k in ("beauty", "beauty_a", "beauty_b"):
        assert np.array_equal(getattr(a, k), getattr(b, k)), k


def test_wide_nee_pool_with_picked_lights(gpu_ctx):
    W, H = 1024, 512
    sc = native.Scene(gpu_ctx, _scene(W, H, 9))
    try:
        a, b = (native.Renderer(sc, 8, 4, light_sampling_strategy="power", paths_in_flight=n).render(W, H).buffers
                for n in (0, 1 << 20))
    finally:
        sc.close()
    assert a.beauty.mean() > 0
    for k in ("beauty", "beauty_a", "beauty_b"):
        assert np.array_equal(getattr(a, k), getattr(b, k)), k


def test_large_batch_pool(gpu_ctx):
    # 8.4 M samples of two scenes in one window: runs with refilled lanes
    W, H = 1024, 512
    scs = [native.Scene(gpu_ctx, _scene(W, H, 2)), native.Scene(gpu_ctx, _mixed(W, H, 6))]
    try:
        items = [(native.Renderer(sc, 8, 2), W, H) for sc in scs]
        a, b = (native.render_batch(items, pool_paths=n)[0] for n in (0, 1 << 20))
        for x, y in zip(a, b):
            assert x.buffers.beauty.mean() > 0
            assert np.array_equal(x.buffers.beauty, y.buffers.beauty)
    finally:
        for sc in scs:
            sc.close()
