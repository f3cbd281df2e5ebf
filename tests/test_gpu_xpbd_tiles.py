"""XPBD steps over tiles of particles (group_runs 1) against one launch per stencil group (group_runs 0): bitwise the same
state and the same number of FP64 solves, for every energy type, both stencil orders and the sizes at which tiles and
batches change."""
import numpy as np
import pytest

from spg_amd import native, scenes

pytestmark = pytest.mark.gpu


def _cloth(n, **kw):
    return scenes.cloth(n, young=1e4, pin="top_row", noise=3e-3 / n, **kw)


def _springs(n, seed=0):
    rng = np.random.default_rng(seed)
    x = rng.uniform(size=(n, 3))
    pairs = np.unique(np.sort(rng.integers(0, n, (3 * n, 2)), axis=1), axis=0).astype(np.int32)
    pairs = pairs[pairs[:, 0] != pairs[:, 1]]
    length = np.linalg.norm(x[pairs[:, 0]] - x[pairs[:, 1]], axis=1) * 0.9
    return scenes.Scene(x=x, x0=x, m=np.full(n, 0.01),
                        energies=[("spring", pairs, np.column_stack([length, np.full(len(length), 50.0)])),
                                  ("anchor", np.array([[0]], np.int32), np.array([[*x[0], 1e4]]))])


SCENES = {
    "cloth 3": lambda: [_cloth(3)],
    "cloth 16": lambda: [_cloth(16)],
    "cloth 33": lambda: [_cloth(33)],
    "cloth 97": lambda: [_cloth(97)],
    "baraff-witkin cloth": lambda: [_cloth(40, membrane="membrane_bw", bending_kind="bending_bw",
                                           edge_springs="spring_continuum", edge_k=5.0)],
    "choi cloth": lambda: [_cloth(21, membrane="membrane_choi", bending_kind="bending_quadratic",
                                  edge_springs="spring_squared_continuum", edge_k=5.0)],
    "cube 2": lambda: [scenes.cube(2)],
    "cube 11": lambda: [scenes.cube(11)],
    "stiff cube": lambda: [scenes.cube(5, young=1e7, stretch_y=1.0, side=0.1)],  # 2 cm tetrahedra: solved in FP64
    "stvk cube": lambda: [scenes.cube(5, material="stvk_tet")],
    "ssnh cube": lambda: [scenes.cube(5, material="ssnh")],
    "springs": lambda: [_springs(300)],
    "springs anywhere": lambda: [_springs(6000)],  # most of a tile's particles lie in others
    "objects": lambda: [_cloth(20), scenes.cube(4), _springs(50), _cloth(35),
                        scenes.Scene(x=np.ones((1, 3)), x0=np.ones((1, 3)), m=np.ones(1))],
}


def _run(objs, parallel, runs, nsub):
    ctx = native.XpbdContext(objs, parallel_gauss_seidel=parallel)
    ctx.set_launch(group_runs=runs)
    ctx.save_state()
    out = []
    for k in range(3):  # the captured step replayed, with the program's own work between
        ctx.step(scenes.DT, nsub, scenes.GRAVITY)
        out += [a for o in range(len(objs)) for a in ctx.state(o)]
        if k == 1:
            ctx.restore_state()
    return out, ctx.stats()["fp64_solves"]


@pytest.mark.parametrize("parallel", [True, False])
@pytest.mark.parametrize("name", list(SCENES))
def test_tiles_bitwise_equal_single_launches(name, parallel):
    objs = [s.xpbd_object() for s in SCENES[name]()]
    if not parallel and sum(len(o["x"]) for o in objs) > 3000:
        objs = objs[:1] if len(objs) > 1 else pytest.skip("thousands of levels")
    for nsub in (1, 2, 5):
        a, fa = _run(objs, parallel, 0, nsub)
        b, fb = _run(objs, parallel, 1, nsub)
        assert all(np.array_equal(p, q) for p, q in zip(a, b)), (name, nsub)
        assert fa == fb, (name, nsub)
    if name == "stiff cube":
        assert fa > 0


@pytest.mark.parametrize("nsub", [1, 2, 3, 4, 5, 6, 7])
def test_substep_counts(nsub):
    """The position buffers change roles every substep: with one batch to a substep, a step of 1, 4, 7 ... substeps ends
    with its start in the buffer that receives the new positions, whose velocities need it."""
    ctx = {}
    for runs in (0, 1):
        ctx[runs] = native.XpbdContext([_cloth(24).xpbd_object()])
        ctx[runs].set_launch(group_runs=runs)
        for _ in range(2):
            ctx[runs].step(scenes.DT, nsub, scenes.GRAVITY)
    (x0, v0), (x1, v1) = ctx[0].state(), ctx[1].state()
    assert np.array_equal(x0, x1) and np.array_equal(v0, v1)
    assert np.abs(v1).max() > 0.1  # gravity over two frames: 0.33 m/s where the cloth falls freely


@pytest.mark.parametrize("parallel", [True, False])
@pytest.mark.parametrize("name", list(SCENES))
def test_scenes_are_stepped_over_tiles(name, parallel):
    """The scenes above do take tiles with group_runs 1, and none with group_runs 0."""
    objs = [s.xpbd_object() for s in SCENES[name]()]
    if not parallel and sum(len(o["x"]) for o in objs) > 3000:
        objs = objs[:1] if len(objs) > 1 else pytest.skip("thousands of levels")
    ctx = native.XpbdContext(objs, parallel_gauss_seidel=parallel)
    plan, stencils = ctx.substep_plan(), sum(len(st) for o in objs for _, st, _ in o["energies"])
    assert plan["tiled_launches"] > 0 and plan["tiles"] >= plan["tiled_launches"]
    assert plan["launches"] <= ctx.num_launches() and plan["tile_bytes"] > 0
    if plan["launches"] == plan["tiled_launches"]:  # everything over tiles: each stencil at least once
        assert plan["tile_projections"] >= stencils
        assert plan["tile_particles"] >= sum(len(o["x"]) for o in objs) * plan["tiled_launches"]
    ctx.set_launch(group_runs=0)
    assert ctx.substep_plan() == dict(launches=ctx.num_launches(), tiled_launches=0, tiles=0, tile_particles=0,
                                      tile_projections=0, tile_bytes=0)


@pytest.mark.parametrize("parallel", [True, False])
@pytest.mark.parametrize("name", ["cloth 97", "baraff-witkin cloth", "cube 11", "stiff cube", "objects"])
def test_runs_of_small_groups_bitwise_equal_single_launches(name, parallel):
    """Timed steps with group_runs 1 take the small groups in runs of one workgroup (the launches of num_launches), not
    tiles: the same state as one launch per group."""
    objs = [s.xpbd_object() for s in SCENES[name]()]
    if not parallel:
        objs = objs[:1]
    out = []
    for runs in (0, 1):
        ctx = native.XpbdContext(objs, parallel_gauss_seidel=parallel)
        ctx.set_launch(group_runs=runs)
        ctx.set_timing(True)
        ctx.step(scenes.DT, 3, scenes.GRAVITY)
        st = ctx.stats()
        assert st["projection_launches"] == 3 * ctx.num_launches()
        assert ("small_group_runs" in st["per_type"]) == (runs == 1)
        out.append([a for o in range(len(objs)) for a in ctx.state(o)] + [st["fp64_solves"]])
    assert all(np.array_equal(p, q) for p, q in zip(*out))
