"""The BVH stages' units of 64 rays (narvalengine_amd/csrc/wavefront.hip): any
number of paths against a unit, a chunk of 256 slots, the pool and the resident
blocks; shadow rays with surfaces, with surfaces and a volume (occlusion, then
packed tracking) and with neither.  The wavefront traces the megakernel's paths:
equal counts, and films that differ by the fixed-point rounding of a path's
final light sample alone."""
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
    from narvalengine_amd import configs
    from narvalengine_amd.scene import Scene
    if which == "surface":
        return scenes.small_surface(subdiv=2), scenes.BOX_CAMERA
    if which == "mixed":
        s = scenes.env_map_scene()  # a volume over a floor, under a map and the sun
        s.add_rectangle(s.add_emitter((4.0, 4.0, 4.0)), position=(0, 0.9, 0), rotation=(-90, 0, 0), scale=(0.5, 0.5, 1))
        s.add_point_light((0.7, 0.1, -0.6), s.add_emitter((0.8, 0.8, 0.6)))
        return s, scenes.VOLUME_CAMERA
    if which == "mixed_mesh":  # a BVH of many nodes
        s = scenes.small_surface(subdiv=2)
        s.set_volume(configs.fbm_grid(16, 0), 12.0, (0.95,) * 3, (0.05,) * 3, 0.7, maj_res=4)
        return s, scenes.BOX_CAMERA
    s = Scene()
    s.add_point_light((0.3, 0.35, -0.2), s.add_emitter((3.0, 2.5, 2.0)))
    return s, scenes.VOLUME_CAMERA


# width, height, spp, pool slots (0: the default)
SIZES = [(1, 1, 1, 0), (63, 1, 1, 0), (64, 1, 1, 0), (65, 1, 1, 256), (255, 1, 1, 0), (257, 1, 1, 0),
         (45, 37, 5, 1000), (320, 200, 12, 0)]


# (with nothing to hit, the wavefront has no stage that counts extension rays)
EVENTS = {"surface": ("paths", "ext_rays", "shadow_rays"), "neither": ("paths", "shadow_rays"),
          "mixed": ("paths", "ext_rays", "shadow_rays", "density_lookups", "majorant_cells")}
EVENTS["mixed_mesh"] = EVENTS["mixed"]


@pytest.mark.parametrize("which", ["surface", "mixed", "mixed_mesh", "neither"])
@pytest.mark.parametrize("order", ["plain", "sort", "spatial"])
def test_units_trace_the_megakernels_paths(ctx, which, order):
    print_case(f"units {which} {order}")
    from narvalengine_amd.abi import NE_MODE_MEGAKERNEL, NE_MODE_WAVEFRONT
    s, cam = _scene(which)
    g = ctx.upload(s)
    kw = {} if order == "plain" else {order: True}
    for w, h, spp, pool in SIZES:
        films, counts = [], []
        for mode, pool_size, extra in ((NE_MODE_MEGAKERNEL, 0, {}), (NE_MODE_WAVEFRONT, pool, kw)):
            f = ctx.film(w, h)
            ctx.render(g, cam, f, spp=spp, max_bounces=6, seed=11, mode=mode, pool_size=pool_size, **extra)
            films.append(f.read())
            ctx.render(g, cam, ctx.film(w, h), spp=spp, max_bounces=6, seed=11, mode=mode, pool_size=pool_size,
                       count=True, **extra)
            counts.append({k: ctx.counters()[k] for k in EVENTS[which]})
        np.testing.assert_allclose(films[1], films[0], rtol=1e-6, atol=spp * 2.0 ** -30, err_msg=f"{w}x{h}x{spp}")
        assert counts[0] == counts[1], (w, h, spp, counts)


@pytest.mark.parametrize("which", ["surface", "mixed", "mixed_mesh"])
@pytest.mark.parametrize("bounces", [0, 1, 5, 6, 7, 8, 13, 14, 15, 16])
@pytest.mark.parametrize("pool", [0, 1024])
def test_the_last_shadow_rays_are_delivered(ctx, which, bounces, pool):
    """The loop looks every 8 iterations whether paths are left; the last vertices'
    shadow rays are traced with the next segments, or after the loop: max_bounces
    around the iterations where it ends, all paths issued at once (1045 in a pool
    of their own) and in a pool that is refilled (4180 in 1024 slots)."""
    print_case(f"last shadow rays {which}, {bounces} bounces, pool {pool}")
    from narvalengine_amd.abi import NE_MODE_MEGAKERNEL, NE_MODE_WAVEFRONT
    s, cam = _scene(which)
    g = ctx.upload(s)
    spp = 4 if pool else 1
    films = []
    for mode, pool_size in ((NE_MODE_MEGAKERNEL, 0), (NE_MODE_WAVEFRONT, pool)):
        f = ctx.film(55, 19)
        ctx.render(g, cam, f, spp=spp, max_bounces=bounces, seed=11, mode=mode, pool_size=pool_size)
        films.append(f.read())
    np.testing.assert_allclose(films[1], films[0], rtol=1e-6, atol=spp * 2.0 ** -30)
