"""Device memory: what the library holds beyond a call's needs, and what it gives
back when an allocation would fail."""
import numpy as np
import pytest

import scenes
from conftest import print_case
from hipmem import FullCard, free_bytes

pytestmark = pytest.mark.gpu
GIB = 1 << 30


def test_surface_renders_keep_a_pool_of_2_23_slots():
    """A render of 2^25 paths of a scene without a volume: the path pool (240 B
    a slot) stays at 2^23 slots; samples take 12 B each."""
    from narvalengine_amd import Context
    print_case("pool of a surface render")
    ctx = Context(0)
    g = ctx.upload(scenes.small_surface(subdiv=2))
    f = ctx.film(1024, 1024)
    ctx.synchronize()
    before = free_bytes()
    ctx.render(g, scenes.BOX_CAMERA, f, spp=32, max_bounces=2, seed=3)
    used = before - free_bytes()
    assert f.read().any()
    assert used < (1 << 23) * 260 + (1 << 25) * 12 + (64 << 20), used / GIB
    ctx.close()


def test_quads_make_room_for_other_allocations(ctx):
    """The quad copies of the grids (four times the bricks) are a convenience: an
    allocation that they leave no room for gets it, and the scenes then read the
    bricks, with the same films."""
    print_case("quads and a full card")
    from narvalengine_amd import Batch
    from narvalengine_amd.abi import NE_BATCH_PERSISTENT, NE_BATCH_WAVEFRONT
    rng = np.random.default_rng(4)
    s = scenes.small_volume(res=8, maj_res=4)
    s.set_volume(rng.random((192, 192, 192), np.float32), 12.0, (0.95,) * 3, (0.05,) * 3, 0.7, maj_res=4)
    g = [ctx.upload(s) for _ in range(24)]
    size = g[0].info()["device_bytes"]
    small = ctx.film(40, 30)

    def frame():
        small.clear()
        ctx.render(g[5], scenes.VOLUME_CAMERA, small, spp=4, max_bounces=8, seed=3)
        return small.read()

    job = dict(scene=g[7], camera=scenes.VOLUME_CAMERA, width=40, height=30, spp=4, max_bounces=8, seed=3, job=0)
    batch = Batch(ctx, [job])

    def batches():
        out = []
        for executor in (NE_BATCH_PERSISTENT, NE_BATCH_WAVEFRONT):
            batch.run((8, 8, 4, executor))
            out.append(batch.read(0))
        return out

    want, want_batches = frame(), batches()
    assert want.any()
    # all but 1 GiB taken by others, then a film of 2 GiB: 2.7 GiB are in quads
    fill = FullCard(leave=GIB)
    try:
        big = ctx.film(32768, 2731)
    finally:
        fill.free()
    assert g[5].info()["device_bytes"] < size // 3
    np.testing.assert_array_equal(frame(), want)
    np.testing.assert_array_equal(batches(), want_batches)
    big.close()
    batch.close()
    # an upload after that has its quads again
    h = ctx.upload(s)
    assert h.info()["device_bytes"] == size
    for x in g:
        x.close()
    h.close()


def test_a_homogeneous_medium_has_no_quads(ctx):
    """Its density is not read: the 1^3 grid's bricks (two of 128 B in z, one of
    slack), a majorant and its pair."""
    from narvalengine_amd.scene import Scene
    print_case("homogeneous medium")
    s = Scene()
    s.set_homogeneous_volume(3.0, (0.9,) * 3, (0.1,) * 3, 0.6)
    s.set_sun((1, -1, 0.3))
    g = ctx.upload(s)
    assert g.info()["device_bytes"] == 3 * 128 + 4 + 8
    g.close()


def test_scene_info_does_not_wait_for_a_render(ctx):
    """A scene's info is read while another thread holds the context in a batch of
    a quarter of a second."""
    import threading
    import time
    from narvalengine_amd import Batch
    from narvalengine_amd.abi import NE_BATCH_WAVEFRONT
    print_case("info beside a batch")
    g = ctx.upload(scenes.small_surface(subdiv=3))
    job = dict(scene=g, camera=scenes.BOX_CAMERA, width=1024, height=1024, spp=64, max_bounces=8, seed=3, job=0)
    batch = Batch(ctx, [dict(job, job=j) for j in range(4)])
    batch.run((8, 8, 4, NE_BATCH_WAVEFRONT))
    took = []

    def run():
        t = time.perf_counter()
        batch.run((8, 8, 4, NE_BATCH_WAVEFRONT))
        took.append(time.perf_counter() - t)

    th = threading.Thread(target=run)
    th.start()
    time.sleep(0.02)
    t = time.perf_counter()
    assert g.info()["device_bytes"] > 0
    waited, alive = time.perf_counter() - t, th.is_alive()
    th.join()
    assert alive and waited < 0.25 * took[0], (waited, took)
    batch.close()


def test_long_surface_renders_fit_in_a_smaller_pool(ctx):
    """2^27 paths of a BVH of 2^16 nodes take a pool of 2^24 slots (3.6 GB), or half
    of it where the card has no more room: the same film."""
    from narvalengine_amd import Context
    print_case("long surface render on a full card")
    s = scenes.small_surface(subdiv=7)
    films, used = [], []
    for room in (0, 2304 << 20):  # (beside the first render's pool of 2^20 slots)
        c = Context(0)
        g = c.upload(s)
        assert g.info()["bvh_nodes"] >= 1 << 16
        f = c.film(1024, 1024)
        c.render(g, scenes.BOX_CAMERA, f, spp=1, max_bounces=1, seed=3, fixed_film=True)
        f.clear()
        c.synchronize()
        before = free_bytes()
        fill = FullCard(leave=room) if room else None
        try:
            c.render(g, scenes.BOX_CAMERA, f, spp=128, max_bounces=1, seed=3, fixed_film=True)
        finally:
            if fill:
                fill.free()
        used.append(before - free_bytes())
        films.append(f.read())
        c.close()
    assert films[0].any()
    np.testing.assert_array_equal(films[0], films[1])
    assert used[0] > 1.5 * used[1], used
