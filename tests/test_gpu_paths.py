"""The persistent volume path kernel (mode AUTO on scenes without surfaces)
against the staged wavefront (NE_MODE_WAVEFRONT): the same paths, draws and
arithmetic, so the films are equal bit for bit, whatever the number of paths
against the block's 256 slots, the id batches and the resident blocks."""
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
    if which == "cloud":
        return scenes.small_cloud()
    if which == "one_majorant":
        return configs.volume_scene(configs.fbm_grid(40, 3))
    if which == "homogeneous":
        s = Scene()
        s.set_homogeneous_volume(3.0, (0.9,) * 3, (0.1,) * 3, 0.6, rotation=(20, 35, 0), scale=(0.8, 0.5, 0.6))
        s.set_sun((1, -1, 0.3))
        return s
    if which == "point_light":
        s = scenes.small_volume(res=32, maj_res=4, env=False)
        s.add_point_light((0.3, 0.35, -0.2), s.add_emitter((3.0, 2.5, 2.0)))
        return s
    if which == "env_map":
        s = scenes.env_map_scene()
        s.rect, s.rect_mat = [], []
        return s
    return scenes.small_volume(res=32, maj_res=4)


# width, height, spp, bounces, rect: one path; fewer paths than a wave; the
# block's 256 slots less and plus one; strips beside the 8x8 tiles; more
# paths than all resident blocks hold (refills from the id counter); no
# scattering vertex; long paths
SIZES = [(1, 1, 1, 3, None), (7, 5, 1, 16, None), (17, 15, 1, 16, None), (257, 1, 1, 16, None),
         (45, 37, 8, 64, (3, 5, 42, 36)), (320, 200, 12, 8, None), (64, 64, 4, 0, None), (31, 33, 16, 128, None)]


@pytest.mark.parametrize("which", ["volume", "cloud", "one_majorant", "homogeneous", "point_light", "env_map"])
@pytest.mark.parametrize("form", ["slots", "fixed_film", "wide", "guided"])
def test_persistent_paths_equal_the_staged_wavefront(ctx, which, form):
    print_case(f"persistent paths {which} {form}")
    from narvalengine_amd.abi import NE_MODE_AUTO, NE_MODE_WAVEFRONT
    from narvalengine_amd.runtime import Guide
    kw = {"fixed_film": {"fixed_film": True}, "wide": {"wide": True}}.get(form, {})
    if form == "guided":
        kw = {"guide": Guide(ctx, log2_table=12, cache_res=8, guided_vertices=3, guide_prob=0.5)}
    g = ctx.upload(_scene(which))
    lit = False
    for w, h, spp, bounces, rect in SIZES:
        films = []
        for mode in (NE_MODE_WAVEFRONT, NE_MODE_AUTO):
            f = ctx.film(w, h)
            ctx.render(g, scenes.VOLUME_CAMERA, f, spp=spp, max_bounces=bounces, seed=7, rect=rect, mode=mode, **kw)
            films.append(f.read())
        np.testing.assert_array_equal(films[0], films[1], err_msg=f"{w}x{h}x{spp}, {bounces} bounces")
        lit = lit or films[0].any()
    assert lit


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("side", [-0.5, 0.5])
@pytest.mark.parametrize("toward", [-1.0, 1.0])
def test_rays_in_a_face_of_the_volume(ctx, axis, side, toward):
    """Camera rays that run in a face's plane, parallel to another axis: a
    direction component of 0 or -0 there has an infinite reciprocal of that
    sign, and with the origin on the face that sign decides the box test.  A
    field of view of 1e-9 degrees makes every ray the axis itself."""
    print_case(f"rays in a face: axis {axis}, side {side}, toward {toward}")
    from narvalengine_amd import configs
    from narvalengine_amd.abi import NE_MODE_AUTO, NE_MODE_MEGAKERNEL, NE_MODE_WAVEFRONT
    from narvalengine_amd.scene import Camera
    along = (axis + 1) % 3
    pos, target, up = [0.1, 0.1, 0.1], [0.1, 0.1, 0.1], [0.0, 0.0, 0.0]
    pos[axis] = target[axis] = side
    pos[along], target[along] = -2.0 * toward, 0.0
    up[axis] = 1.0
    cam = Camera(position=tuple(pos), look_at=tuple(target), up=tuple(up), vfov=1e-9, aspect=1.0)
    g = ctx.upload(configs.volume_scene(np.ones((8, 8, 8), np.float32), maj_res=2))
    films = []
    for mode in (NE_MODE_MEGAKERNEL, NE_MODE_WAVEFRONT, NE_MODE_AUTO):
        f = ctx.film(16, 16)
        ctx.render(g, cam, f, spp=16, max_bounces=8, seed=5, mode=mode)
        films.append(f.read())
    np.testing.assert_array_equal(films[1], films[2])
    np.testing.assert_allclose(films[2], films[0], rtol=1e-6, atol=16 * 2.0 ** -30)


# how a render is run, and whether a guide is sampled
RUNS = {"persistent": {}, "fixed_film": {"fixed_film": True}, "staged": {"mode": 2}, "small_pool": {"mode": 2, "pool_size": 1000},
        "sort": {"mode": 2, "sort": True}, "spatial": {"mode": 2, "spatial": True}, "count": {"count": True},
        "guided": {"guide": True}, "guided_staged": {"guide": True, "mode": 2},
        "guided_sort": {"guide": True, "mode": 2, "sort": True}, "training": {"guide": True, "train": True}}


@pytest.mark.parametrize("which", ["volume", "cloud", "point_light", "surfaces"])
@pytest.mark.parametrize("run", list(RUNS))
def test_the_grids_forms_give_the_same_film(ctx, which, run):
    """Quads, bricks by 32-bit offsets (what grids of 645^3 to 1024^3 take, and
    any grid whose quads found no room) and by 64-bit offsets hold the same
    voxels: equal films and event counts in every kernel that reads them."""
    print_case(f"grid forms {which} {run}")
    from narvalengine_amd.runtime import Guide
    kw = dict(RUNS[run])
    if kw.get("guide"):  # rates of 0: a training render leaves the guide as it is
        kw["guide"] = Guide(ctx, log2_table=12, cache_res=8, guided_vertices=3, guide_prob=0.5, batch=4096,
                            lr_table=0.0, lr_mlp=0.0)
    g = ctx.upload(scenes.env_map_scene() if which == "surfaces" else _scene(which))
    for w, h, spp, bounces in [(45, 37, 8, 24), (7, 5, 1, 16)]:
        out = []
        for form in ({}, {"brick": True}, {"wide": True}):
            f = ctx.film(w, h)
            ctx.render(g, scenes.VOLUME_CAMERA, f, spp=spp, max_bounces=bounces, seed=41, **kw, **form)
            out.append((f.read(), ctx.counters() if run == "count" else None))
        assert out[0][0].any()
        for o in out[1:]:
            np.testing.assert_array_equal(out[0][0], o[0], err_msg=f"{w}x{h}")
            assert out[0][1] == o[1]
