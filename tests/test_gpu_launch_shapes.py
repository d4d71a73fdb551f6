"""Launches that a world alone does not reach: the sweeps of worlds over 512 bodies in a launch of
their own, at every workgroup size; a large world whose sweep has more steps than its table in LDS
holds; the slots beyond a few thousand bodies.  Bit for bit against the oracle."""
import numpy as np
import pytest

import oracle_lib as O
from cannon_physics_amd import _abi as A
from cannon_physics_amd import scenes
from cannon_physics_amd.objects import Body, Box, SAPBroadphase, Sphere
from cannon_physics_amd.world import Context, World, state_to_numpy

pytestmark = pytest.mark.gpu
DT = 1 / 60
PREC = {"f32": A.PRECISION_F32, "f64": A.PRECISION_F64}


def bits(a):
    return np.ascontiguousarray(a).view(np.uint8)


def same(c, wid, ow):
    g, o = state_to_numpy(*c.download(wid)), ow.state()
    return all(np.array_equal(bits(g[k]), bits(o[k])) for k in g)


def heap(bodies, side):
    """`bodies` bodies with the plane, boxes and spheres overlapping in a cube of `side`."""
    rng = np.random.default_rng(bodies)
    w = World(gravity=(0, -9.82, 0), broadphase=SAPBroadphase())
    w.addBody(scenes.ground_plane())
    for i in range(bodies - 1):
        w.addBody(Body(mass=1.0, position=rng.uniform(0.3, 0.3 + side, 3).tolist(),
                       quaternion=scenes.shoemake_quaternion(rng),
                       shape=Box((0.3, 0.3, 0.3)) if i % 4 else Sphere(0.3)))
    return w.recipe()


def create(c, rec):
    wid = c.create_world(rec)
    c.set_capacity(wid, max_pairs=1 << 15, max_contacts=1 << 15, max_rows=1 << 17)
    return wid


# Over 256 workgroups in all the worlds of 513 to 4096 bodies are not taken into the small worlds'
# launch (graphs on: one stream, so one list of all the worlds, captured at the second call)
@pytest.mark.parametrize("mode", ["f32", "f64"])
def test_worlds_over_512_bodies_among_hundreds(mode):
    sizes = [3000, 600, 513]
    recs = [heap(n, 0.9 * n ** (1 / 3)) for n in sizes]
    small = heap(129, 1.2 * 129 ** (1 / 3))
    ows = [O.OracleWorld(r, mode) for r in recs + [small]]
    for o in ows:
        o.step(DT, 6)
    c = Context(device=0, precision=PREC[mode])
    try:
        c.set_graphs(True)
        for solve, levels in [(64, 256), (128, 128), (256, 64), ("auto", None)]:
            print(f"[shapes] {mode} solve {solve} levels {levels}", flush=True)
            big, few = [create(c, r) for r in recs], [c.create_world(small) for _ in range(256)]
            if solve == "auto":
                c.autotune()
            else:
                c.set_tuning(solve_block=solve, levels_block=levels)
            for _ in range(2):
                c.step(few[:128] + big + few[128:], DT, 3)
            assert all(same(c, w, o) for w, o in zip(big + few[::85], ows + ows[3:] * 3))
            for w in big + few:
                c.destroy_world(w)
    finally:
        c.close()


# a chain of 4200 links: over 4096 bodies (velocities in memory) and three levels a joint, more steps
# than the table in LDS holds
@pytest.mark.parametrize("mode", ["f32", "f64"])
def test_large_world_with_more_steps_than_the_table_holds(mode):
    w = scenes.c4_chain_world(43, length=4200, joints=["p2p"])
    assert len(w.bodies) > 4096
    rec = w.recipe()
    ow = O.OracleWorld(rec, mode)
    ow.step(1 / 120, 2)
    rows = ow.rows()
    assert np.sum(rows["kind"] == A.ROW_CONTACT) >= 3 * 4199
    c = Context(device=0, precision=PREC[mode])
    try:
        for solve in (64, 128, 256):
            print(f"[shapes] chain {mode} solve {solve}", flush=True)
            wid = c.create_world(rec)
            c.set_tuning(solve_block=solve)
            c.step([wid], 1 / 120, 2)
            assert same(c, wid, ow)
            c.destroy_world(wid)
    finally:
        c.close()


# the slots: hull pairs a thread each (over 4096 bodies) and a wave each; an equation of a body with
# itself in a world of one workgroup's sweep and in one of a launch of its own
@pytest.mark.parametrize("mode", ["f32", "f64"])
@pytest.mark.parametrize("bodies,side", [(600, 9.0), (4097, 18.0)])
def test_slots_of_large_worlds(bodies, side, mode):
    rec = heap(bodies, side)
    c, ow = Context(device=0, precision=PREC[mode]), O.OracleWorld(rec, mode)
    try:
        wid = create(c, rec)
        ow.set_state_raw(c.download(wid)[0])
        pi, pj = c.broadphase(wid)
        oi, oj = ow.broadphase()
        assert np.array_equal(pi, oi) and np.array_equal(pj, oj)
        eqs, k, nf, nc = c.narrowphase(wid, pi, pj, DT)
        oeqs, ok, onf, onc = ow.narrowphase(pi, pj, DT)
        assert (k, nf, nc) == (ok, onf, onc) and k > 0
        ids = np.ctypeslib.as_array(eqs)[:k]
        assert np.array_equal(bits(ids), bits(np.ctypeslib.as_array(oeqs)[:k]))
        ids["body_j"][k // 2] = ids["body_i"][k // 2]
        it, mult = c.solve(wid, eqs, k, DT)
        oit, omult = ow.solve(eqs, k, DT)
        assert it == oit and np.array_equal(bits(mult), bits(omult)) and same(c, wid, ow)
    finally:
        c.close()


# the autotuner leaves the sweeps' size alone where no sweep of the list depends on it
@pytest.mark.parametrize("bodies", [40, 600])
def test_autotune_of_lists_without_sized_sweeps(bodies):
    c = Context(device=0)
    try:
        ids = [create(c, heap(bodies, 0.9 * bodies ** (1 / 3))) for _ in range(3)]
        for solve in (64, 128, 256):
            c.set_tuning(solve_block=solve, levels_block=128)
            c.autotune()
            c.step(ids, DT, 2)
            assert c.tuning()["solve_block"] == solve
    finally:
        c.close()
