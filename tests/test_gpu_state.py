"""The state read-out of the VBD, XPBD and rigid-body contexts: every value of every object, whatever its size, in
particle order. Positions and velocities are set first (32-bit in the particle solvers), so the expected values are
exact."""
import numpy as np
import pytest

from gpu_common import gpu_context
from spg_amd import native, scenes

pytestmark = pytest.mark.gpu

PART = 32768  # particles gathered by one launch (positions and velocities), and ten of these go out at once
BODIES = 8192  # rigid bodies gathered by one launch


def _free(n, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((n, 3))
    return {"x": x, "v": rng.standard_normal((n, 3)), "m": np.ones(n), "w": np.ones(n), "energies": []}


def _f32(a):
    return a.astype(np.float32).astype(np.float64)


# the edges of one and of several launches, and more than the staging memory holds at once
@pytest.mark.parametrize("sizes", [[1], [85], [86], [PART - 1], [PART + 1], [5 * PART, 3, 2 * PART + 7], [400_001]])
def test_particle_states_read_back(sizes):
    objs = [_free(n, k) for k, n in enumerate(sizes)]
    for ctx in (native.VbdContext(objs), native.XpbdContext(objs)):
        for k in reversed(range(len(objs))):
            x, v = ctx.state(k)
            assert np.array_equal(x, _f32(objs[k]["x"])) and np.array_equal(v, _f32(objs[k]["v"]))


def test_one_field_alone():
    """Either array may be null (include/spg_vbd.h): the other is read as before."""
    s = scenes.cloth(20, young=1e4)
    ctx = gpu_context(s)
    ctx.step(s.dt, 1, 2, s.gravity)
    x, v = ctx.state()
    for which in (0, 1):
        out = np.full((s.n, 3), np.nan)
        p = native._d(out)
        ctx._check(ctx._L.spg_vbd_get_state(ctx.h, 0, *((p, None) if which == 0 else (None, p))))
        assert np.array_equal(out, (x, v)[which])
    ctx._check(ctx._L.spg_vbd_get_state(ctx.h, 0, None, None))


@pytest.mark.parametrize("sizes", [[1], [BODIES], [BODIES + 1, 5, 700], [90_001]])
def test_rigid_states_read_back(sizes):
    rng = np.random.default_rng(3)
    groups = [{"x": rng.standard_normal((n, 3)), "theta": 0.5 * rng.standard_normal((n, 3)),
               "v": rng.standard_normal((n, 3)), "omega": rng.standard_normal((n, 3)), "m": np.ones(n),
               "inertia": np.tile(np.eye(3), (n, 1, 1)), "energies": []} for n in sizes]
    ctx = native.RigidContext(groups)
    for k, g in enumerate(groups):
        for got, want in zip(ctx.state(k), (g["x"], g["theta"], g["v"], g["omega"])):
            assert np.array_equal(got, want)
