"""Launch shapes of the one-path-per-thread kernels: Li with its rays spread over
more or fewer waves, FP64 renders held to 1, 2 or 3 waves per SIMD.  The shape
changes no path, so results are equal bit for bit."""
import numpy as np
import pytest

import scenes
from conftest import print_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from narvalengine_amd import Context
    return Context(0)


def _scene(which):
    if which == "surface":
        return scenes.small_surface(subdiv=2), scenes.BOX_CAMERA
    if which == "mixed":
        return scenes.env_map_scene(), scenes.VOLUME_CAMERA
    return scenes.small_volume(res=24, maj_res=4), scenes.VOLUME_CAMERA


@pytest.mark.parametrize("which", ["volume", "surface", "mixed"])
def test_li_does_not_depend_on_the_spread(ctx, which):
    """A ray's estimate depends on its place in the call alone: 1, 2 and 3 rays a
    wave, ragged last waves, and (200,000 rays) whole waves."""
    print_case(f"li spread {which}")
    s, cam = _scene(which)
    g = ctx.upload(s)
    rng = np.random.default_rng(3)
    o = rng.uniform(-0.9, 0.9, (200000, 3)) + [0.0, 1.0 if which == "surface" else 0.0, 0.0]
    d = rng.normal(size=(200000, 3))
    rays = np.concatenate([o, d / np.linalg.norm(d, axis=1, keepdims=True)], 1).astype(np.float32)
    whole = ctx.li(g, rays, 5, seed=5)
    assert whole.any()
    for n in (2, 63, 2047, 2048, 4095, 4096, 6145):
        np.testing.assert_array_equal(ctx.li(g, rays[:n], 5, seed=5), whole[:n], err_msg=str(n))


@pytest.mark.parametrize("which", ["volume", "surface", "mixed"])
@pytest.mark.parametrize("w,h,spp", [(256, 511, 1), (512, 257, 1), (505, 521, 1), (1024, 1024, 1), (1031, 1024, 2)])
def test_fp64_render_does_not_depend_on_the_occupancy(ctx, which, w, h, spp):
    """Blocks of 64 threads take the unbounded kernel at any size; 2048,
    4096 and 16,384 waves of 8 x 8 pixels are where blocks of 128 change theirs."""
    print_case(f"fp64 {which} {w}x{h}x{spp}")
    from narvalengine_amd.abi import NE_FP64
    s, cam = _scene(which)
    g = ctx.upload(s)
    films = []
    for block in (64, 128):
        f = ctx.film(w, h)
        ctx.render(g, cam, f, spp=spp, max_bounces=4, seed=3, precision=NE_FP64, block_size=block)
        films.append(f.read())
    assert films[0].any()
    np.testing.assert_array_equal(films[0], films[1])
