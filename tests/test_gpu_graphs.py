"""Graph replay on every plan: long runs, with the program's own launches, other
calls and new states between the replays, against the same steps launched one
by one (the staged surface, which replays nothing)."""
import numpy as np
import pytest

from lb3d_amd.gpu import LB3D_BC_LEES_EDWARDS, LB3D_FP32_DEV, LB3D_FP64, Batch, Lattice

pytestmark = pytest.mark.gpu

LE = dict(boundary=LB3D_BC_LEES_EDWARDS, shear_u=0.03)
TERN = dict(ncomp=3, g_br=0.08, g_bs=-0.006, g_ss=-0.003)
DIMS = (10, 6, 7)


def rock_records(g):
    """The lattice's records with a wall along y and a stray rock site."""
    N = g.download_sites()
    N[:, 0:2, :, -1] = 1.0
    N[3, 4, 5, -1] = 1.0
    return N


@pytest.mark.parametrize("precision", [LB3D_FP64, LB3D_FP32_DEV])
@pytest.mark.parametrize("name,kw,plan", [
    ("two-pass", dict(ncomp=2, g_br=0.09), (0,)),
    ("one-pass", dict(ncomp=2, g_br=0.09), (2, 32, 4, 3)),
    ("walls", dict(ncomp=2, g_br=0.06, g_wr=0.02, g_wb=-0.02), (0,)),
    ("Lees-Edwards two-pass", dict(LE, ncomp=2, g_br=0.09), (0,)),
    ("Lees-Edwards one-pass", dict(LE, ncomp=2, g_br=0.09), (2, 32, 4, 3)),
    ("ternary", TERN, (0,)),
    ("ternary one-pass", TERN, (3, 32, 4, 3)),
])
def test_replayed_steps_are_the_launched_ones(name, kw, plan, precision):
    g, ref = (Lattice(*DIMS, precision=precision, **kw) for _ in range(2))

    def state(seed, sites=None):
        for L in (g, ref):
            if sites is None:
                L.init_noise(seed, amp=(0.01, 0.01, 0.01))
                if name == "walls":
                    L.upload_sites(rock_records(L))
            else:
                L.upload_sites(sites)
            L.bc_init()

    def advance(n):
        g.time_loop(n)
        for _ in range(n):
            ref.time_step()

    def same(what):
        assert g.nt == ref.nt
        assert np.array_equal(g.populations(), ref.populations()), what
        assert np.array_equal(g.download_sites(), ref.download_sites()), what

    for L in (g, ref):
        L.set_plan(*plan)
    state(3)
    advance(2048)           # a graph from the first step of a fresh lattice
    same("one long call")
    sites = ref.download_sites()
    for n in (49, 1, 96, 203):  # odd counts: replays begin at either parity
        advance(n)
        same(f"{n} more")
    for L in (g, ref):      # launches of the program's own between replays
        L.time_step()
    advance(51)
    same("after a staged step")
    if "Lees" in name:
        assert np.array_equal(g.le_halo(), ref.le_halo())
    g.profile_steps(3)
    for _ in range(3):
        ref.time_step()
    advance(97)
    same("after profiled steps")
    g.autotune(1)
    g.set_plan(*plan)       # drops the graph; the state is the same
    advance(5)
    same("after the tuner")
    for n in (1025, 99):    # a graph once 1024 steps have been run on the plan
        g.time_loop(n // 2), g.time_loop(n - n // 2)
        for _ in range(n):
            ref.time_step()
    same("after 1024 steps in parts")
    state(4)                # a new state under a captured graph
    advance(99)
    same("after init_noise")
    state(0, sites)
    advance(98)
    same("after an upload")
    assert np.isfinite(g.populations()).all()


@pytest.mark.parametrize("plan,ncomp", [("groups", 2), ("groups", 3), ("sequential", 2), ("sequential", 3),
                                        ("persistent", 2), ("persistent", 3), ("collide-moments", 3)])
def test_replayed_batch_steps_are_the_launched_ones(plan, ncomp):
    """The batch's plans: groups of lattices, lattice by lattice, collide-moments
    (whose graph carries the moments from step to step)."""
    dims = [(8, 6, 6), (6, 10, 7), (12, 5, 9)]

    def replan(b):          # (sets the plan anew, which drops a graph)
        if plan == "groups":
            b.set_groups(2 * ncomp * 19 * 4 * 300)
        elif plan == "sequential":
            b.set_plan(1)
        elif plan == "collide-moments":
            b.set_collide_moments(6, 3, 4)
        else:
            b.set_groups(0)

    a, ref = (Batch(dims, ncomp=ncomp, precision=LB3D_FP32_DEV) for _ in range(2))
    for b in (a, ref):
        for k in range(3):
            b.init_noise(k, 5 + k, amp=(0.01, 0.01, 0.01))
        replan(b)

    def advance(*counts):
        for n in counts:
            a.time_loop(n)
            for _ in range(n):
                ref.time_loop(1)
                if ref.nt % 500 == 0:
                    replan(ref)
        assert a.nt == ref.nt
        for k in range(3):
            assert np.array_equal(a.populations(k), ref.populations(k)), (counts, k)

    advance(2049)           # one long call
    advance(1, 50, 101)
    for b in (a, ref):
        b.profile_steps(2)
    advance(97)
    a.init_noise(1, 9, amp=(0.02, 0.01, 0.01))
    ref.init_noise(1, 9, amp=(0.02, 0.01, 0.01))
    for b in (a, ref):
        assert b.nt == 0
    advance(99)
    replan(a)
    advance(700, 500, 75)   # a graph once 1024 steps have been run on the plan
