"""The moments of the last advection (the rho and da of download_sites, the
forces of arrows) on every plan: the one-pass plans keep none and rebuild them
on demand, whatever was called in between and at whatever stage of a step."""
import numpy as np
import pytest

from lb3d_amd.gpu import LB3D_BC_LEES_EDWARDS, LB3D_FP32_DEV, LB3D_FP64, LB3DError, Lattice

pytestmark = pytest.mark.gpu

LE = dict(ncomp=2, g_br=0.09, boundary=LB3D_BC_LEES_EDWARDS, shear_u=0.07)
FORMS = [(dict(ncomp=2, g_br=0.09), (2, 32, 4, 4)), (LE, (2, 32, 4, 4)), (LE, (3, 32, 8, 3)),
         (dict(ncomp=3, g_br=0.08, g_bs=-0.006, g_ss=-0.003), (3, 32, 4, 4))]


def lattice(dims, plan, steps, **kw):
    """A lattice after whole steps; plan None: untuned, 0: the two-pass plan."""
    g = Lattice(*dims, **kw)
    if plan is not None:
        g.set_plan(*plan) if plan else g.set_plan(0)
    g.init_noise(7, amp=(0.2, 0.2, 0.1))
    g.bc_init()
    g.time_loop(steps)
    return g


def inner(N):
    return N[1:-1, 1:-1, 1:-1]


@pytest.mark.parametrize("precision,dims,plan", [
    (LB3D_FP64, (20, 9, 12), (2, 32, 4, 4)),
    (LB3D_FP32_DEV, (20, 9, 12), (1, 32, 4, 12)),
    (LB3D_FP64, (64, 84, 96), None),
])
@pytest.mark.parametrize("steps", [4, 5])
def test_building_the_next_halo_planes_keeps_the_last_moments(precision, dims, plan, steps):
    """le_halo() and bc_apply(6) build the halo planes of the new state; the
    moments at x = 0 and nx-1 are still those of the planes the last step
    streamed through."""
    kw = dict(LE, precision=precision)
    for call in ("le_halo", "bc_apply"):
        got = []
        for p in (0, plan):
            g = lattice(dims, p, steps, **kw)
            halo = g.le_halo() if call == "le_halo" else g.bc_apply(6, steps + 1)
            got.append((halo, inner(g.download_sites()), g.arrows() if call == "le_halo" else None))
        (h0, n0, a0), (h1, n1, a1) = got
        assert np.array_equal(n0, n1), f"{call}: rho differs by {np.abs(n0 - n1).max()}"
        if call == "le_halo":
            assert np.array_equal(h0, h1) and np.array_equal(a0, a1)


@pytest.mark.parametrize("kw,plan", FORMS)
@pytest.mark.parametrize("precision", [LB3D_FP64, LB3D_FP32_DEV])
def test_records_at_every_stage_do_not_depend_on_the_plan(kw, plan, precision):
    """Records taken after each call of the staged surface, with the one-pass
    and the two-pass plan, and the populations after the step."""
    kw = dict(kw, precision=precision)
    dims = (20, 9, 12)
    got = []
    for p in (0, plan):
        g = lattice(dims, p, 3, **kw)
        recs = []
        for call in (lambda: None, lambda: g.bc_apply(6, 4), g.advection, lambda: g.bc_apply(8, 4), g.collision):
            call()
            recs.append(inner(g.download_sites()))
        got.append(recs + [g.populations()])
    for stage, (a, b) in enumerate(zip(*got)):
        assert np.array_equal(a, b), f"stage {stage}: {np.abs(a - b).max()}"


@pytest.mark.parametrize("kw,plan", FORMS)
def test_records_within_a_step_leave_the_step_alone(kw, plan):
    """One-pass steps, then a staged two-pass step: records taken after its
    advection, and an upload that is refused there, do not replace the moments
    that its collision reads."""
    kw = dict(kw, precision=LB3D_FP64)
    dims = (20, 9, 12)
    ref = lattice(dims, 0, 4, **kw)
    want = ref.populations()
    for what in ("download", "refused upload"):
        g = lattice(dims, plan, 3, **kw)
        rec = g.download_sites() if what == "refused upload" else None
        g = lattice(dims, plan, 3, **kw)
        g.set_plan(0)
        g.bc_apply(6, 4)
        g.advection()
        if what == "download":
            g.download_sites()
        elif kw["ncomp"] == 3 or "boundary" in kw:
            rec[..., -1] = 1.0
            with pytest.raises(LB3DError):
                g.upload_sites(rec)
        g.bc_apply(8, 4)
        g.collision()
        assert np.array_equal(g.populations(), want), f"{what}: {np.abs(g.populations() - want).max()}"


@pytest.mark.parametrize("kw,plan", FORMS)
@pytest.mark.parametrize("precision", [LB3D_FP64, LB3D_FP32_DEV])
@pytest.mark.parametrize("first", [False, True])
def test_plan_changes_within_a_step(kw, plan, precision, first):
    """set_plan between any two calls of a staged step, in either direction and
    back again, on the first step of a state too: populations and records are
    those of the two-pass plan."""
    kw = dict(kw, precision=precision)
    dims = (20, 9, 12)
    steps = 0 if first else 3
    ref = lattice(dims, 0, steps + 2, **kw)
    want, want_rec = ref.populations(), ref.download_sites()
    for switch in range(4):
        for plans in ((plan, 0), (0, plan), (plan, 0, plan), (0, plan, 0)):
            g = lattice(dims, plans[0], steps, **kw)
            calls = [lambda: g.bc_apply(6), g.advection, lambda: g.bc_apply(8), g.collision]
            for k, call in enumerate(calls):
                if k == switch:
                    for p in plans[1:]:
                        g.set_plan(*p) if p else g.set_plan(0)
                call()
            g.time_step()
            got = g.populations()
            assert np.array_equal(got, want), f"{plans} before call {switch}: {np.abs(got - want).max()}"
            assert np.array_equal(g.download_sites(), want_rec), f"{plans} before call {switch}: records"
