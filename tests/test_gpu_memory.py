"""Device memory: what the library holds beyond a call's needs, and what it gives
back when an allocation would fail."""
import pytest

import scenes
from conftest import print_case
from hipmem import free_bytes

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
