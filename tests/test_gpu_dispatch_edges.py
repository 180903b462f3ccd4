"""Sizes at which kernels change form: ray queries on both sides of the
stack-placement threshold, gather points at the faces of the photons'
bounding box (the k-nearest search visits only its cells), and films at the
edges of the denoiser's tiles (16- and 64-column runs, 16 x 16 regression
centres) and on both sides of its rows-a-thread line.  All bit-exact."""
import numpy as np
import pytest

from helpers import random_rays, random_triangles
from hierarchy_cases import instanced_scene
from raytracer import denoise, native, scenes
from test_gpu_caustics import _settings, _small_caustics
from test_gpu_denoise import _check, _film

pytestmark = pytest.mark.gpu

QUERY_LDS = 1 << 17   # rays up to which the query kernels keep their stacks in LDS


@pytest.mark.parametrize("scene", ["mixed", "instances"])
def test_query_stack_placements_agree(gpu_ctx, scene):
    desc = random_triangles(3000, 5) if scene == "mixed" else instanced_scene()
    rays = random_rays(QUERY_LDS + 65, 11, spread=6.0)
    segs = np.concatenate([rays, np.full((len(rays), 1), 1e-4, np.float32), np.full((len(rays), 1), 4.0, np.float32)], 1)
    sc = native.Scene(gpu_ctx, desc)
    try:
        big = sc.trace_rays(rays)
        occ = sc.occluded(segs)
        for lo, hi in ((0, 1), (0, QUERY_LDS), (QUERY_LDS, QUERY_LDS + 65)):
            for a, b in zip(big, sc.trace_rays(rays[lo:hi])):
                assert np.array_equal(a[lo:hi].view(np.uint32), b.view(np.uint32)), (lo, hi)
            assert np.array_equal(occ[lo:hi], sc.occluded(segs[lo:hi]))
    finally:
        sc.close()
    assert 0.02 < (big[0] >= 0).mean() < 0.98


@pytest.mark.parametrize("radius", [0.05, 0.2])
def test_gather_at_the_photon_bounds(gpu_ctx, oracle, radius):
    sc = native.Scene(gpu_ctx, _small_caustics())
    st = _settings(64, 48, 1, 8, 50000, radius)
    m = sc.photon_map(st)
    lo, hi = m["pos"].min(0), m["pos"].max(0)
    rng = np.random.default_rng(2)
    pts = rng.uniform(lo, hi, (6000, 3))
    for axis in range(3):
        s = slice(2000 * axis, 2000 * axis + 2000)
        face = np.where(rng.random(2000) < 0.5, lo[axis], hi[axis])
        pts[s, axis] = face + rng.choice([-3.0, -1.0, -0.5, 0.0, 0.25, 1.0, 2.0, 50.0], 2000) * radius
    pts = np.concatenate([pts, m["pos"][:500], [[1e9, 0, 0], [-1e9, 0, 0], [0, 3e38, 0]]]).astype(np.float32)
    cnt, rad, idx = sc.photon_gather(st, pts)
    h = oracle.PhotonMap.from_positions(m["pos"], float(m["grid"][3]))
    near = len(pts) - 3           # the oracle's cell loop overflows at the far points
    ocnt, orad, oidx = h.gather(pts[:near], 40, radius)
    assert np.array_equal(cnt[:near], ocnt) and np.array_equal(rad[:near].view(np.int32), orad.view(np.int32))
    assert np.array_equal(idx[:near], oidx)
    assert (cnt[near:] == 0).all() and (cnt[:near] > 0).any() and (cnt[:near] == 0).any()


@pytest.mark.parametrize("W,H", [(1, 1), (15, 5), (65, 66), (129, 34)])
@pytest.mark.parametrize("kind", ["nlm", "nfor"])
def test_denoise_tile_edges(gpu_ctx, oracle, W, H, kind):
    buf = _film(gpu_ctx, scenes.cornell(W, H), W, H, 4)
    got = denoise.denoise(buf, denoise.DenoiserOptions(kind, "high"), gpu_ctx)
    _check(got, oracle.denoise(buf, kind, "high"), f"{kind} {W}x{H}")


@pytest.mark.parametrize("W,H", [(297, 295), (513, 513)])
def test_nlm_rows_a_thread(gpu_ctx, oracle, W, H):
    # from 524,288 pixels times filterings (six in the prefilter, two in the
    # main filter) a thread sums two rows: the prefilter only, then both
    buf = _film(gpu_ctx, scenes.cornell(W, H), W, H, 2)
    got = denoise.denoise(buf, denoise.DenoiserOptions("nlm", "fast"), gpu_ctx)
    _check(got, oracle.denoise(buf, "nlm", "fast"), f"nlm {W}x{H}")


@pytest.mark.parametrize("W,H", [(2, 9000), (2, 16420)])
def test_nfor_offset_slices(gpu_ctx, oracle, W, H):
    # 282 and 514 tiles of centres: the offsets in three slices, and in one
    # (small films, as above, take up to 45)
    buf = _film(gpu_ctx, scenes.cornell(W, H), W, H, 2)
    got = denoise.denoise(buf, denoise.DenoiserOptions("nfor", "high"), gpu_ctx)
    _check(got, oracle.denoise(buf, "nfor", "high"), f"nfor {W}x{H}")


@pytest.mark.parametrize("caustics", [False, True])
def test_stage_times(gpu_ctx, caustics):
    # the shadow stage's time starts behind the gather where there is one
    sc = native.Scene(gpu_ctx, _small_caustics())
    try:
        st = native.Renderer(sc, 4, 8, enable_caustics=caustics, caustic_photons=20000 if caustics else 0).render(64, 48).stats
    finally:
        sc.close()
    assert min(st.trace_ms, st.shade_ms, st.shadow_ms) > 0
    assert st.trace_ms + st.shade_ms + st.shadow_ms < st.device_ms
