"""Copies between the device and the caller's arrays through the context's pinned
staging: sizes below, at and above its chunks (2 MiB) and the direct path's limit
(512 KiB of rays and radiance)."""
import numpy as np
import pytest

import scenes
from conftest import print_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from narvalengine_amd import Context
    return Context(0)


@pytest.mark.parametrize("n", [1, 4, 14563, 14564, 30000])
def test_li_is_the_same_through_either_path(ctx, n):
    """36 bytes a ray: 14563 rays are the most that the kernel reads in place.
    A ray's estimate depends on its place in the call alone."""
    print_case(f"li of {n} rays")
    g = ctx.upload(scenes.small_volume(res=16, maj_res=4))
    rng = np.random.default_rng(3)
    o = rng.uniform(-1.5, 1.5, (60000, 3))
    d = rng.uniform(-0.4, 0.4, (60000, 3)) - o
    rays = np.concatenate([o, d / np.linalg.norm(d, axis=1, keepdims=True)], 1).astype(np.float32)
    whole = ctx.li(g, rays, 8, seed=5)  # above the limit
    assert whole.any()
    np.testing.assert_array_equal(ctx.li(g, rays[:n], 8, seed=5), whole[:n])


@pytest.mark.parametrize("log2_table", [10, 14, 15])
def test_parameters_come_back_as_they_were_set(ctx, log2_table):
    """Tables of 128 KiB, one chunk and two."""
    from narvalengine_amd import Guide
    print_case(f"guide parameters, log2_table {log2_table}")
    g = Guide(ctx, log2_table=log2_table, batch=16)
    rng = np.random.default_rng(log2_table)
    table, mlp = rng.normal(size=g.table_floats).astype(np.float32), rng.normal(size=g.mlp_floats).astype(np.float32)
    g.set_params(table, mlp)
    t, m = g.params()
    np.testing.assert_array_equal(t, table)
    np.testing.assert_array_equal(m, mlp)


@pytest.mark.parametrize("w,h", [(431, 211), (640, 409)])
def test_films_and_tiles_come_back_whole(ctx, w, h):
    """A film of a chunk and a remainder, and of three chunks: the same pixels
    as one of its tiles, read by itself into the caller's frame."""
    from narvalengine_amd.engine import OfflineEngine, SceneSettings
    print_case(f"film {w} x {h}")
    eng = OfflineEngine(scenes.VOLUME_CAMERA, SceneSettings((w, h), 1, 4), scenes.small_volume(res=16, maj_res=4),
                        ctx=ctx, seed=9)
    f = ctx.film(w, h)
    ctx.render(eng.gscene, scenes.VOLUME_CAMERA, f, spp=1, max_bounces=4, seed=9)
    frame, sums = f.tonemap(1), f.read()
    assert frame.any() and ((frame > 0) == (sums > 0)).all()
    tw, th = w // 40, h // 10
    index = 4 * 40 + 19
    eng.renderTile(scenes.VOLUME_CAMERA, index)
    y, x = (index // 40) * th, (index % 40) * tw
    assert frame[y:y + th, x:x + tw].any()
    np.testing.assert_array_equal(eng.pixels[y:y + th, x:x + tw], frame[y:y + th, x:x + tw])
    eng.pixels[y:y + th, x:x + tw] = 0
    assert not eng.pixels.any()


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf, -1e-38])
def test_a_bad_voxel_is_refused_wherever_it_lies(ctx, value):
    """17 x 17 x 15 voxels: a block of 4096 that are looked over together and a
    remainder; first and last of each."""
    from narvalengine_amd import NarvalError
    print_case(f"voxel {value}")
    for at in (0, 4095, 4096, 17 * 17 * 15 - 1):
        grid = np.full((15, 17, 17), -0.0, np.float32)
        grid.reshape(-1)[::3] = np.finfo(np.float32).max
        s = scenes.small_volume(res=8, maj_res=2)
        s.set_volume(grid, 1e-6, (0.95,) * 3, (0.05,) * 3, 0.7, maj_res=2)
        ctx.upload(s).close()
        grid.reshape(-1)[at] = value
        s.set_volume(grid, 1e-6, (0.95,) * 3, (0.05,) * 3, 0.7, maj_res=2)
        with pytest.raises(NarvalError, match="finite"):
            ctx.upload(s)


def test_a_tile_of_more_than_a_chunk_comes_back_whole(ctx):
    """A tile of 440 x 420 pixels, 2.2 MB in rows of 5,280 bytes: 397 rows in the
    first chunk, 23 in the second; nothing beside the tile is written."""
    from narvalengine_amd.engine import OfflineEngine, SceneSettings
    print_case("large tile")
    w, h, tw, th = 17600, 4200, 440, 420
    eng = OfflineEngine(scenes.VOLUME_CAMERA, SceneSettings((w, h), 1, 2), scenes.small_volume(res=16, maj_res=4),
                        ctx=ctx, seed=9)
    index = 4 * 40 + 19
    y, x = (index // 40) * th, (index % 40) * tw
    eng.renderTile(scenes.VOLUME_CAMERA, index)
    f = ctx.film(w, h)
    ctx.render(eng.gscene, scenes.VOLUME_CAMERA, f, spp=1, max_bounces=2, seed=9, rect=(x, y, x + tw, y + th))
    want = f.tonemap(1)
    f.close()
    assert want[y:y + th, x:x + tw].any()
    np.testing.assert_array_equal(eng.pixels[y - 1:y + th + 1, x - 1:x + tw + 1], want[y - 1:y + th + 1, x - 1:x + tw + 1])
    assert not eng.pixels[:y].any() and not eng.pixels[y + th:].any()


@pytest.mark.parametrize("n", [6553, 6554, 13107, 13108, 26214, 26215, 39322])
def test_reads_come_back_whole_at_their_chunks_edges(ctx, n):
    """160 B a query: below and above 1 MiB (one chunk or two halves), 2 MiB,
    4 MiB (two chunks and a remainder) and 6 MiB; a query's mixture does not
    depend on its place in the call."""
    from narvalengine_amd import Guide
    print_case(f"eval of {n} queries")
    g = Guide(ctx, log2_table=10, batch=16, seed=3)
    q = np.random.default_rng(7).uniform(0, 1, (n, 6)).astype(np.float32)
    whole = g.eval(q)
    parts = np.concatenate([g.eval(q[k:k + 1600]) for k in range(0, n, 1600)])
    assert whole.any()
    np.testing.assert_array_equal(whole, parts)
    g.close()
