"""Captured steps after a world of the list gave its id to another: a replay must run with the new
world's segment and LDS, so the step is captured anew.  Bit for bit against a context without graphs."""
import numpy as np
import pytest

from cannon_physics_amd import _abi as A
from cannon_physics_amd import scenes
from cannon_physics_amd.objects import Body, Box, Sphere
from cannon_physics_amd.world import Context, World, state_to_numpy

pytestmark = pytest.mark.gpu
DT = 1 / 60


def heap(bodies):
    """`bodies` bodies with the plane, boxes and spheres overlapping in a cube."""
    rng = np.random.default_rng(bodies)
    side = 1.2 * bodies ** (1 / 3)
    w = World(gravity=(0, -9.82, 0))
    w.addBody(scenes.ground_plane())
    for i in range(bodies - 1):
        w.addBody(Body(mass=1.0, position=rng.uniform(0.3, 0.3 + side, 3).tolist(),
                       quaternion=scenes.shoemake_quaternion(rng),
                       shape=Box((0.3, 0.3, 0.3)) if i % 4 else Sphere(0.3)))
    return w.recipe()


def same(a, b):
    return all(np.array_equal(np.ascontiguousarray(a[k]).view(np.uint8), np.ascontiguousarray(b[k]).view(np.uint8)) for k in a)


# the world that goes and the one that gets its id: within a segment of the sweeps (a wave, a
# workgroup), and from one to another, up and down; the largest of the list stays
@pytest.mark.parametrize("mode", ["f32", "f64"])
@pytest.mark.parametrize("sizes,new", [((400, 100), 120), ((600, 200), 500), ((300, 100), 250), ((300, 250), 60),
                                       ((700, 60, 20), 50), ((1100, 600), 100), ((1100, 100), 600)])
def test_replay_after_an_id_changed_hands(sizes, new, mode):
    prec = A.PRECISION_F64 if mode == "f64" else A.PRECISION_F32
    old, recs = heap(sizes[-1]), [heap(n) for n in sizes[:-1]]
    fresh = heap(new)
    ctxs = [Context(device=0, precision=prec) for _ in range(2)]
    try:
        out = []
        for c, graphs in zip(ctxs, (True, False)):
            def create(rec):
                w = c.create_world(rec)
                c.set_capacity(w, max_pairs=1 << 15, max_contacts=1 << 15, max_rows=1 << 17)
                return w
            c.set_graphs(graphs)
            many = [create(recs[0]) for _ in range(4)]   # a queue that no later list outgrows
            c.step(many, DT, 1)
            for w in many:
                c.destroy_world(w)
            ids = [create(r) for r in recs + [old]]
            for _ in range(3):   # captured at the second call
                c.step(ids, DT, 3)
            c.destroy_world(ids[-1])
            assert create(fresh) == ids[-1]
            for _ in range(2):
                c.step(ids, DT, 3)
            out.append([state_to_numpy(*c.download(w)) for w in ids])
        for a, b in zip(*out):
            assert same(a, b)
    finally:
        for c in ctxs:
            c.close()


# serving gives a finished request's id to the next one admitted
def test_served_requests_with_graphs():
    worlds = [scenes.c3_world(60 + n, n=n, kind="pile") for n in (600, 300, 120, 100, 250, 60, 130, 40)]
    recs, sizes = [w.recipe() for w in worlds], [len(w.bodies) for w in worlds]
    out = []
    for graphs in (True, False):
        c = Context(device=0)
        try:
            c.set_graphs(graphs)
            done = []

            def serve(t, n):
                while c.serve_status(t)["state"] < A.REQ_DONE:
                    c.serve_tick(4)
                assert c.serve_status(t)["state"] == A.REQ_DONE
                done.append(state_to_numpy(c.serve_result(t, n), n))
            serve(c.serve_submit(recs[0], DT, 4), sizes[0])
            stays = c.serve_submit(recs[1], DT, 12 * len(recs))
            for rec, n in zip(recs[2:], sizes[2:]):
                serve(c.serve_submit(rec, DT, 12), n)
            serve(stays, sizes[1])
            out.append(done)
        finally:
            c.close()
    for a, b in zip(*out):
        assert same(a, b)
