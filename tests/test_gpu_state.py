"""State transfers: an uploaded state comes back bit for bit, at the edges of the transfer's body
tiles (64 bodies a workgroup, 16,384 a transfer)."""
import numpy as np
import pytest

from cannon_physics_amd import _abi as A
from cannon_physics_amd.objects import Body, Sphere
from cannon_physics_amd.world import Context, World

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 129, 16384, 16385])
def test_uploaded_state_comes_back(n):
    rng = np.random.default_rng(n)
    w, ball = World(), Sphere(0.5)
    for _ in range(n):
        w.addBody(Body(mass=1, shape=ball))
    for precision in (A.PRECISION_F32, A.PRECISION_F64):
        ctx = Context(precision=precision)
        wid = ctx.create_world(w.recipe())
        arr, k = ctx.download(wid)
        s = np.ctypeslib.as_array(arr)
        for name in s.dtype.names:
            if s[name].dtype.kind == "f":
                s[name] = rng.normal(size=s[name].shape)
        s["aabb_needs_update"] = rng.integers(0, 2, n)
        s["sleep_state"] = rng.integers(0, 3, n)
        want = s.copy()
        ctx.upload(wid, arr, k)
        got = np.ctypeslib.as_array(ctx.download(wid)[0])
        assert np.array_equal(got.view(np.uint8), want.view(np.uint8))
        ctx.close()
