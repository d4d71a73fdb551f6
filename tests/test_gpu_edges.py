"""The device kernels at the edges of their tiles and of the rules that choose between them, bit for
bit against the oracle: body counts around a wave, a workgroup and the segments of the sweeps, rows
beyond what the level schedule keeps in LDS, few bodies and many, hulls and polygons around a wave's
workspace, more ray candidates and event keys than one round takes."""
import numpy as np
import pytest

import oracle_lib as O
from cannon_physics_amd import _abi as A
from cannon_physics_amd import scenes
from cannon_physics_amd.objects import Body, Box, NaiveBroadphase, SAPBroadphase, Sphere
from cannon_physics_amd.world import Context, World, state_to_numpy

pytestmark = pytest.mark.gpu
DT = 1 / 60
_ctx = {}


def ctx(mode):
    if mode not in _ctx:
        _ctx[mode] = Context(device=0, precision=A.PRECISION_F64 if mode == "f64" else A.PRECISION_F32)
    return _ctx[mode]


def bits(a):
    return np.ascontiguousarray(a).view(np.uint8)


def create(c, rec):
    """the world, with room for the contacts of overlapping heaps"""
    wid = c.create_world(rec)
    c.set_capacity(wid, max_pairs=1 << 15, max_contacts=1 << 15, max_rows=1 << 17)
    return wid


def same(c, wid, ow):
    g, o = state_to_numpy(*c.download(wid)), ow.state()
    return all(np.array_equal(bits(g[k]), bits(o[k])) for k in g)


def heap(bodies, side, sap=False, seed=1):
    """`bodies` bodies with the plane, boxes and spheres overlapping in a cube of `side`."""
    rng = np.random.default_rng(seed)
    w = World(gravity=(0, -9.82, 0), broadphase=SAPBroadphase() if sap else NaiveBroadphase())
    w.addBody(scenes.ground_plane())
    for i in range(bodies - 1):
        w.addBody(Body(mass=1.0, position=rng.uniform(0.3, 0.3 + side, 3).tolist(),
                       quaternion=scenes.shoemake_quaternion(rng),
                       shape=Box((0.3, 0.3, 0.3)) if i % 4 else Sphere(0.3)))
    return w


def check_steps(world, mode, steps=3):
    """`steps` steps, then one captured: pairs, rows, multipliers, state."""
    rec = world.recipe()
    c, ow = ctx(mode), O.OracleWorld(rec, mode)
    wid = create(c, rec)
    try:
        c.step([wid], DT, steps)
        ow.step(DT, steps)
        assert same(c, wid, ow)
        pi, pj, rows, it = c.step_capture(wid, DT, pair_cap=1 << 17, row_cap=1 << 17)
        ow.step(DT, 1)
        opi, opj = ow.pairs()
        assert np.array_equal(pi, opi) and np.array_equal(pj, opj)
        orow = ow.rows()
        for k in rows:
            assert np.array_equal(bits(rows[k]), bits(orow[k])), k
        assert it == ow.iterations() and same(c, wid, ow)
        return len(orow["kind"])
    finally:
        c.destroy_world(wid)


@pytest.mark.parametrize("mode", ["f32", "f64"])
@pytest.mark.parametrize("sap", [False, True])
@pytest.mark.parametrize("bodies", [1, 2, 63, 64, 65, 66, 127, 128, 129, 255, 256, 257, 511, 512, 513])
def test_body_counts(bodies, sap, mode):
    check_steps(heap(bodies, 1.2 * bodies ** (1 / 3), sap), mode)


# rows over the LDS schedule of a wave's world (1024) and of a workgroup's (6144); bodies that share
# mask entries (over 1024), and the sweeps' four waves and eight (4096 bodies)
@pytest.mark.parametrize("mode,bodies,side,rows", [("f32", 128, 2.0, 1025), ("f64", 128, 2.0, 1025), ("f32", 512, 5.0, 6145),
                                                   ("f64", 512, 5.0, 6145), ("f32", 1025, 7.0, 6145), ("f64", 1025, 9.0, 1),
                                                   ("f32", 4095, 18.0, 1), ("f32", 4097, 18.0, 1)])
def test_many_rows(mode, bodies, side, rows):
    assert check_steps(heap(bodies, side, sap=bodies > 600), mode, 2) >= rows


# a chain's rows are one chain of runs: longer than the rounds of relaxation, and than 64 runs
@pytest.mark.parametrize("mode", ["f32", "f64"])
@pytest.mark.parametrize("length", [2, 12, 13, 64, 65, 130])
def test_long_chains(length, mode):
    rec = scenes.c4_chain_world(17, length=length, joints=["p2p"]).recipe()
    c, ow = ctx(mode), O.OracleWorld(rec, mode)
    wid = create(c, rec)
    try:
        c.step([wid], 1 / 120, 10)
        ow.step(1 / 120, 10)
        assert same(c, wid, ow)
    finally:
        c.destroy_world(wid)


# one list over all segments of the sweeps; and enough bodies (over 4096) that hull pairs take a
# thread each where the same world alone gives them a wave each
@pytest.mark.parametrize("mode", ["f32", "f64"])
def test_mixed_lists_and_few_or_many_bodies(mode):
    sizes = [1100, 700, 513, 512, 300, 129, 128, 40, 9, 2]
    worlds = [heap(n, 1.3 * n ** (1 / 3), seed=n) for n in sizes] + [scenes.prism_world(9), scenes.c5_terrain_world(4, n=40)]
    recs = [w.recipe() for w in worlds]
    c = ctx(mode)
    ows = [O.OracleWorld(r, mode) for r in recs]
    for o in ows:
        o.step(DT, 4)
    for extra in (0, 4):
        wids = [create(c, r) for r in recs]
        more = [create(c, recs[0]) for _ in range(extra)]
        try:
            c.step(wids + more, DT, 4)
            assert all(same(c, wid, ow) for wid, ow in zip(wids, ows))
        finally:
            for wid in wids + more:
                c.destroy_world(wid)


# faces of 16, 17 and 32 vertices (32 and 34 vertices a hull: a wave's workspace holds 32; 32: the
# largest face) against boxes and each other
@pytest.mark.parametrize("mode", ["f32", "f64"])
@pytest.mark.parametrize("segments", [3, 4, 5, 8, 16, 17, 32])
def test_prism_faces(segments, mode):
    check_steps(scenes.prism_world(9, segments=segments), mode, 20)


@pytest.mark.parametrize("mode", ["f32", "f64"])
def test_terrain_hulls(mode):
    check_steps(scenes.c5_terrain_world(8, n=60), mode, 60)


# the sphere-box resolver's early return: spheres at, just inside and just outside a box' faces,
# edges and corners
@pytest.mark.parametrize("mode", ["f32", "f64"])
def test_spheres_about_a_box(mode):
    w = World(gravity=(0, 0, 0), broadphase=NaiveBroadphase())
    w.addBody(Body(mass=0, shape=Box((0.5, 0.5, 0.5)), position=(0, 0, 0)))
    r = 0.25
    for d in [(1, 0, 0), (0, 1, 0), (0, 0, -1), (1, 1, 0), (0, 1, -1), (1, 1, 1), (-1, 1, -1)]:
        u = np.array(d) / np.linalg.norm(d)
        for gap in (-1e-3, -1e-7, 0.0, 1e-7, 1e-3):
            w.addBody(Body(mass=1.0, shape=Sphere(r), position=(0.5 * np.array(d) + (r + gap) * u).tolist()))
    check_steps(w, mode, 1)


@pytest.mark.parametrize("mode", ["f32", "f64"])
@pytest.mark.parametrize("sap", [False, True])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 130])
def test_rays_through_many_candidates(n, sap, mode):
    w = World(gravity=(0, 0, 0), broadphase=SAPBroadphase() if sap else NaiveBroadphase())
    order = np.random.default_rng(n).permutation(n)
    for i in order:
        w.addBody(Body(mass=1.0, position=(1.5 * float(i), 0.1 * float(i % 3), 0.0),
                       shape=Sphere(0.5) if i % 2 else Box((0.4, 0.4, 0.4))))
    rec = w.recipe()
    c, ow = ctx(mode), O.OracleWorld(rec, mode)
    wid = create(c, rec)
    try:
        rays = []
        for k in range(9):
            ray = A.Ray()
            ray.from_[:] = [-2.0, 0.05 * k, 0.01 * k] if k % 2 else [1.5 * n + 2.0, 0.05 * k, 0.0]
            ray.to[:] = [1.5 * n + 2.0, 0.05 * k, 0.0] if k % 2 else [-2.0, 0.1, 0.0]
            ray.mode = [A.RAY_CLOSEST, A.RAY_ANY, A.RAY_ALL][k % 3]
            ray.skip_backfaces, ray.check_collision_response = k // 5, 1
            ray.collision_filter_group = ray.collision_filter_mask = -1
            rays.append(ray)
        g, o = c.raycast(wid, rays), ow.raycast(rays)
        assert len(g) == len(o) > 0
        for k in g.dtype.names:
            assert np.array_equal(bits(g[k]), bits(o[k])), k
    finally:
        c.destroy_world(wid)


# events of fewer and of more touching pairs than are sorted in LDS (2048)
@pytest.mark.parametrize("mode", ["f32", "f64"])
@pytest.mark.parametrize("bodies,side,pairs", [(64, 2.0, 100), (512, 4.0, 2049)])
def test_events_of_many_pairs(bodies, side, pairs, mode):
    rec = heap(bodies, side).recipe()
    c, ow = ctx(mode), O.OracleWorld(rec, mode)
    wid = create(c, rec)
    try:
        c.set_events(wid, capacity=1 << 17)
        ow.set_events(True)
        raised = 0
        for _ in range(4):
            c.step([wid], DT, 1)
            ow.step(DT, 1)
            g, o = c.events(wid), ow.events()
            assert len(g) == len(o)
            for k in g.dtype.names:
                assert np.array_equal(bits(g[k]), bits(o[k])), k
            raised = max(raised, len(o))
        assert raised >= pairs
    finally:
        c.destroy_world(wid)


# the Solver slot with an equation of a body with itself among the scene's own
@pytest.mark.parametrize("mode", ["f32", "f64"])
@pytest.mark.parametrize("bodies", [12, 100, 300])
def test_solver_slot_with_a_self_equation(bodies, mode):
    rec = heap(bodies, 1.2 * bodies ** (1 / 3)).recipe()
    c, ow = ctx(mode), O.OracleWorld(rec, mode)
    wid = create(c, rec)
    try:
        arr, n = c.download(wid)
        ow.set_state_raw(arr)
        pi, pj = c.broadphase(wid)
        ow.broadphase()
        eqs, k, nf, nc = c.narrowphase(wid, pi, pj, DT)
        assert ow.narrowphase(pi, pj, DT)[1] == k > 0
        ids = np.ctypeslib.as_array(eqs)[:k]
        ids["body_j"][k // 2] = ids["body_i"][k // 2]
        it, mult = c.solve(wid, eqs, k, DT)
        oit, omult = ow.solve(eqs, k, DT)
        assert it == oit and np.array_equal(bits(mult), bits(omult)) and same(c, wid, ow)
    finally:
        c.destroy_world(wid)
