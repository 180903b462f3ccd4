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
    # 8.9 M samples: the default pool's shadow waves work through runs of the
    # queue and refill their lanes; a 1 M pool's keep a ray a lane
    W, H = 1920, 929
    desc = scenes.displaced_icosphere_scene(W, H, subdiv=4, sphere_lights=2)
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
