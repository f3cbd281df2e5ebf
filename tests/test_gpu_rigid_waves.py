"""The wavefronts that share a group of 64 bodies in a colour (one, four or five, by the bodies of the colour): copies of a
small scene side by side in one group, with counts around a wavefront and around both lines of the rule, each end where the
scene alone ends. Both sides are FP64 and differ by the order of at most 40 summands per block (1e-14 relative), times the
condition of a body's block (below 1e2 here) over 60 solves: below 1e-10."""
import numpy as np
import pytest

from spg_amd import native, scenes

pytestmark = pytest.mark.gpu


def _copies(s, k):
    energies = [(kind, (st[None] + s.nb * np.arange(k)[:, None, None]).reshape(-1, st.shape[1]).astype(np.int32),
                 np.tile(p, (k, 1))) for kind, st, p in s.energies]
    return scenes.RigidScene(x=np.tile(s.x, (k, 1)), theta=np.tile(s.theta, (k, 1)), m=np.tile(s.m, k),
                             inertia=np.tile(s.inertia, (k, 1, 1)), iterations=s.iterations, energies=energies)


def _star(rays=13):
    """A box joined to others by springs and squared springs in turn, three to a ray: one row of 39 entries."""
    rng = np.random.default_rng(6)
    x = np.vstack([np.zeros((1, 3)), 3 * rng.standard_normal((rays, 3))])
    pairs = np.column_stack([np.zeros(rays, np.int32), np.arange(1, rays + 1, dtype=np.int32)])
    joint = lambda: np.column_stack([0.5 * rng.standard_normal((rays, 6)), np.full(rays, 2.0), np.full(rays, 50.0)])
    return scenes.RigidScene(x=x, theta=0.2 * rng.standard_normal((rays + 1, 3)), m=np.ones(rays + 1),
                             inertia=np.tile(scenes.box_inertia(1.0, 1.0, 0.8, 0.6), (rays + 1, 1, 1)), iterations=10,
                             energies=[("rb_spring", pairs, joint()), ("rb_spring_squared", pairs[:, ::-1].copy(), 0.1 * joint()),
                                       ("rb_alignment", pairs, np.full((rays, 1), 5.0))])


@pytest.mark.parametrize("build,counts", [(lambda: scenes.rb_lattice(2), (31, 32, 33, 8192, 8193, 16384, 16385)),
                                          (_star, (63, 65, 1261))], ids=["lattice", "star"])
def test_copies_end_where_one_scene_ends(build, counts):
    s = build()
    one = native.RigidContext([s])
    for _ in range(3):
        one.step(s.dt, 2, s.iterations, s.gravity)
    expected = one.state()
    for k in counts:
        many = native.RigidContext([_copies(s, k)])
        assert many.colors()[1] == one.colors()[1]
        for _ in range(3):
            many.step(s.dt, 2, s.iterations, s.gravity)
        for got, want in zip(many.state(), expected):
            got = got.reshape(k, -1)
            assert np.abs(got - want.ravel()).max() <= 1e-10 * max(np.abs(want).max(), 1.0)
        assert many.stats()["skipped_blocks"] == 0


def test_bytes_of_a_sweep():
    """What a sweep has to move, from the element counts: a body's pose read and written and the rest of its state read (the
    rotation vectors are formed at the substep's end), per entry its 8 bytes, the parameters and the other body's pose."""
    s = scenes.rb_lattice(6)
    n = {kind: len(st) for kind, st, _ in s.energies}
    want = s.nb * (96 + 16 + 8 + 24 + 24 + 72 + 72 + 96) + 2 * n["rb_spring"] * (8 + 64 + 96) + n["rb_anchor"] * (8 + 56)
    want += 2 * n["rb_alignment"] * (8 + 8 + 96)
    assert native.RigidContext([s]).stats()["solve_bytes"] == want
