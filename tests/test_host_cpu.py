"""The library's host code (device bookkeeping, transfers, graphs, plans) on the
CPU, against a stand-in for the HIP runtime (fakehip/fakehip.c)."""
import ctypes
import os
import random
import subprocess
import timeit

import pytest

from lb3d_amd import gpu
from tests import fakehip

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def so(tmp_path_factory):
    return fakehip.compile_fake(tmp_path_factory.mktemp("fakehip"))


def test_read_backs_and_uploads_run_on_the_contexts_device(so):
    """Uploads and read-backs of a lattice of device 1 while device 0 is
    current: buffers, events and kernels are those of device 1, and device 0 is
    current again afterwards."""
    fakehip.run(so, """
        fake.hipSetDevice(1)
        made = [Lattice(12, 10, 8, ncomp=c, precision=p) for c in (2, 3) for p in (0, 1)]
        batch = Batch([(8, 6, 6), (6, 6, 6)], ncomp=3)
        fake.hipSetDevice(0)
        home = Lattice(12, 10, 8, ncomp=2)
        for g in [home] + made:
            g.upload_sites(np.zeros((10, 12, 14, g.site_doubles)))
            g.populations(), g.density(), g.momentum(), g.download_sites()
        batch.populations(1)
        d = ctypes.c_int(-1)
        fake.hipGetDevice(ctypes.byref(d))
        assert d.value == 0
        assert len(log()) > 10
    """)


@pytest.mark.parametrize("dims,halo,ncomp", [((300, 300, 2), 1, 2), ((400, 120, 1), 3, 3)])
def test_transfer_buffers_do_not_grow_with_the_plane(so, dims, halo, ncomp):
    """A z plane of records larger than a piece: the pinned and device buffers
    of an upload stay those of a piece."""
    fakehip.run(so, f"""
        dims, h, ncomp = {dims}, {halo}, {ncomp}
        g = Lattice(*dims, ncomp=ncomp)
        knob("fake_largest_device").value = 0
        g.upload_sites(np.zeros((dims[2] + 2 * h, dims[1] + 2 * h, dims[0] + 2 * h, g.site_doubles)), halo_extent=h)
        g.download_sites(h)
        assert sum("put_sites" in l for l in log()) > 1
        for k in ("fake_largest_pinned", "fake_largest_device"):
            assert 0 < knob(k).value <= 8 << 20, (k, knob(k).value)
    """)


def test_transfers_without_pinned_memory(so):
    """Where nothing can be pinned the transfers go through pageable memory, and
    through pinned memory again once it can be had."""
    fakehip.run(so, """
        g = Lattice(70, 60, 40, ncomp=2)          # 51 MB of populations
        batch = Batch([(8, 6, 6), (6, 6, 6)], ncomp=3)
        knob("fake_device_fill").value = 1
        other = Lattice(70, 60, 40, ncomp=2)
        want = np.arange(2 * 19 * 40 * 60 * 70, dtype=float).reshape(2, 19, 40, 60, 70)
        fail = knob("fake_fail_pinned", ctypes.c_int)
        for fail.value in (1, 2, 0):
            assert np.array_equal(other.populations(), want)
            g.density(), g.momentum(), batch.populations(0)
            g.upload_sites(g.download_sites())
            assert (knob("fake_live_pinned").value > 0) == (fail.value == 0)
    """)


@pytest.mark.parametrize("limit", [3 << 20, 100 << 10, 65536])
def test_transfers_on_a_full_device(so, limit):
    """Conversion pieces shrink to the device memory that is left, and FP64
    populations, which need none, come without any."""
    fakehip.run(so, f"""
        lattices = [Lattice(70, 60, 40, ncomp=2, precision=p) for p in (0, 1)]
        knob("fake_device_limit").value = {limit}
        for g in lattices:
            g.populations(), g.density(), g.momentum()
            g.upload_sites(g.download_sites())
        assert sum("get_density" in l for l in log()) >= 2 * (8 * 2 * 40 * 60 * 70) // {limit}
        del lattices[1:]
        knob("fake_device_limit").value = 0
        lattices[0].populations()
    """)


def test_copy_threads_copy_and_rest(tmp_path):
    """The helper threads of large transfers copy every byte and nothing else,
    and take no processor time while the caller waits for the device."""
    exe = str(tmp_path / "copycrew")
    subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", "-I", os.path.join(HERE, "..", "lb3d_amd", "csrc"),
                    os.path.join(HERE, "copycrew.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert float(r.stdout) < 0.05  # 0.3 s per helper if they spin


STEPS_DONE = """
    def steps(kernels):
        \"\"\"Whole steps in the log, of so many kernels each, and the graphs replayed.\"\"\"
        plain = graphs = replayed = 0
        for l in log():
            plain += l.startswith("launch")
            if l.startswith("graph"):
                graphs += 1
                replayed += int(l.split()[1])
        assert (plain + replayed) % kernels == 0
        return (plain + replayed) // kernels, graphs
"""


def test_one_long_call_replays_a_graph(so):
    """A fresh lattice that is asked for a long run in one call replays a graph
    in that call where launches count (small lattices), runs as many steps as it
    was asked for, and captures nothing for a short call."""
    fakehip.run(so, STEPS_DONE + """
    def fresh(n, **kw):
        g = Lattice(n, n, n, **kw)
        g.init_noise(1); g.bc_init(); log()
        return g
    for n, call, replays in ((16, 2047, False), (16, 2048, True), (16, 100001, True), (48, 5000, False)):
        g = fresh(n, ncomp=2)
        g.time_loop(call)
        done, graphs = steps(2)
        assert done == call and graphs == (call // 24 if replays else 0), (n, call, done, graphs)
    g = fresh(16, ncomp=2)
    g.time_loop_timed(4001)
    assert steps(2)[0] == 4001
    g.time_loop(51)             # the graph is there: shorter calls replay it too
    assert steps(2) == (51, 2)
    g = fresh(64, ncomp=2)
    g.time_loop(1024)
    assert steps(2) == (1024, 0)
    g.time_loop(100)            # a run that has shown to be long, of any size
    assert steps(2) == (100, 4)
    b = Batch([(16, 16, 16), (8, 8, 8)], ncomp=3)
    b.init_noise(0, 1), b.init_noise(1, 2), log()
    b.time_loop(3000)
    done, graphs = steps(3)
    assert done == 3000 and graphs > 0
    """)


def test_graphs_hold_at_least_48_kernels(so):
    """A captured graph holds an even number of steps of at least 48 kernels in
    all, and not two steps more than that takes, on every plan."""
    fakehip.run(so, """
    LE = dict(boundary=LB3D_BC_LEES_EDWARDS, shear_u=0.02)
    forms = [(dict(ncomp=2), None, 2), (dict(ncomp=2), (1, 32, 4, 4), 1), (LE, None, 4), (LE, (2, 32, 4, 4), 3),
             (dict(ncomp=3, precision=LB3D_FP32_DEV), None, 2),       # dipoles and collision in one launch
             (dict(ncomp=3), None, 3), (dict(ncomp=3), (3, 32, 4, 4), 1)]
    for kw, plan, kernels in forms:
        g = Lattice(8, 8, 8, **kw)
        if plan:
            g.set_plan(*plan)
        g.init_noise(1)
        g.time_loop(1)
        log()
        g.time_loop(1)
        assert len(log()) == kernels, (kw, plan)
        g.time_loop(1024)
        g.time_loop(200)
        sizes = {int(l.split()[1]) for l in log() if l.startswith("graph")}
        assert len(sizes) == 1
        size = sizes.pop()
        assert 48 <= size < 48 + 2 * kernels and size % (2 * kernels) == 0, (kw, plan, size)
    """)


class Plan(ctypes.Structure):
    """lb3d::Plan of csrc/lb3d_solver.h."""
    _fields_ = [("fused", ctypes.c_bool), ("tx", ctypes.c_int), ("ty", ctypes.c_int), ("lz", ctypes.c_int),
                ("stage", ctypes.c_int), ("xg", ctypes.c_uint32)]


def default_plan(p):
    f = getattr(gpu.lib(), "_ZN4lb3d12default_planERK11lb3d_params")
    f.restype, f.argtypes = Plan, [ctypes.POINTER(gpu.Params)]
    return f(ctypes.byref(p))


def searched_plan(nx, ny, nz, fp64, le):
    """The tile and z-chunk that cost least, over every number of tiles and chunks."""
    def up(a, b):
        return (a + b - 1) // b
    T, best = 512, None
    for kx in range(1, nx + 1):
        tx = up(nx, kx)
        if tx < (48 if le and not fp64 else 16) and kx > 1:
            break
        ty = min(T // tx, ny, 1040 // (tx + 2) - 2)
        if ty < 1:
            continue
        ky = up(ny, ty)
        ty = up(ny, ky)
        if tx * ty <= T // 2:
            continue
        halo = 2.0 * (tx + 2) + 2.0 * ty
        cost = float(kx) * ky * (T + 0.2 * halo if fp64 or le else T) * (1.04 + 6.0 / tx if kx > 1 else 1.0)
        if best is None or cost < best[0]:
            best = (cost, tx, ty)
    if best is None:
        return None
    _, tx, ty = best
    tiles = up(nx, tx) * up(ny, ty)
    lz = min((up(tiles * up(nz, lz), 256) * (lz + 2), -lz) for lz in {up(nz, kz) for kz in range(1, nz + 1)})[1]
    return tx, ty, -lz


def test_untuned_plan_is_the_cheapest_of_all():
    rng = random.Random(5)
    dims = [(2, 1, 300000), (300000, 2, 1), (1, 1, 1), (513, 900, 3), (512, 512, 4), (256, 64, 64), (90, 100, 77)]
    dims += [tuple(int(2 ** rng.uniform(1, 11)) for _ in range(3)) for _ in range(200)]
    fused = 0
    for nx, ny, nz in dims:
        nx = max(nx, 2)
        if not 400000 <= nx * ny * nz <= 100000000:
            continue
        for fp64, le, line in ((1, 0, 400000), (0, 0, 600000), (1, 1, 500000), (0, 1, 1000000)):
            if nx * ny * nz < line:
                continue
            q = default_plan(gpu.make_params(nx, ny, nz, precision=0 if fp64 else 1, boundary=le))
            want = searched_plan(nx, ny, nz, fp64, le)
            assert ((q.tx, q.ty, q.lz) if q.fused else None) == want, (nx, ny, nz, fp64, le)
            fused += q.fused
    assert fused > 100


def test_untuned_plan_is_found_at_once():
    """lb3d_gpu_step_noalloc looks for it in every call, on a lattice of any shape."""
    for dims in ((270, 1, 400000), (50000000, 1, 1), (3, 30000000, 1), (40, 9, 300000), (640, 7, 24999)):
        p = gpu.make_params(*dims)
        default_plan(p)
        t = min(timeit.repeat(lambda: default_plan(p), number=1, repeat=5))
        assert t < 5e-4, (dims, t)


@pytest.mark.parametrize("dims,kw,kernel", [
    ((90, 100, 77), "ncomp=2, precision=1", "k_fused2"), ((16, 12, 10), "ncomp=2", "k_moments"),
    ((128, 96, 90), "ncomp=2, precision=1, boundary=1", "k_fused2"), ((16, 12, 10), "ncomp=3", "k_moments"),
])
def test_tuner_keeps_the_untuned_plan_unless_another_is_faster(so, dims, kw, kernel):
    """Where every plan takes the same time, as on the stand-in, the tuner leaves
    the untuned plan, and state, parity and offset; without memory for a copy of
    the state it goes by the trials."""
    fakehip.run(so, f"""
        g = Lattice(*{dims}, {kw})
        g.init_noise(1)
        g.time_loop(3)
        log()
        rep = g.autotune(2).strip().splitlines()
        assert rep[-1].startswith("chosen: ") and any(l.startswith("steps: ") for l in rep)
        log()
        g.time_loop(1)
        assert any({kernel!r} in l for l in log()), rep[-1]
        assert g.nt == 4
        knob("fake_device_limit").value = 1 << 10
        assert not any(l.startswith("steps: ") for l in g.autotune(2).splitlines())
        g.time_loop(1)
    """)


FORCES_FIRST, PULLS_FIRST, NON_TEMPORAL = range(3)
LE = dict(boundary=gpu.LB3D_BC_LEES_EDWARDS, shear_u=0.02)
ZH = dict(inv_fluid=12)


def test_order_of_the_collides_loads(so):
    """Whether the two-pass collide pulls before its forces, by component count,
    precision, equilibrium form, boundary and size."""
    cases = []
    for precision in (gpu.LB3D_FP64, gpu.LB3D_FP32_DEV):
        fp64 = precision == gpu.LB3D_FP64
        for bdist in range(7):
            for ncomp, kw in ((2, {}), (2, ZH), (2, LE), (3, {}), (3, ZH)):
                for n in (24, 41, 48, 56, 72):
                    if kw is LE and bdist != 2:
                        first = fp64 or n < 72
                    elif bdist == 2:
                        first = ncomp == 2 or fp64
                    elif bdist == 1:
                        first = fp64
                    else:
                        first = fp64 and bdist == 0 and (n < 56 if ncomp == 2 else n < 48)
                    cases.append((n, dict(kw, ncomp=ncomp, bdist=bdist, precision=precision),
                                  PULLS_FIRST if first else FORCES_FIRST))
            cases.append((124, dict(ncomp=2, bdist=bdist, precision=precision), NON_TEMPORAL))
    fakehip.run(so, f"""
        for n, kw, mode in {cases}:
            g = Lattice(n, n, n, **kw)
            g.set_plan(0)
            log()
            g.time_loop(1)
            name = [l.split()[1] for l in log() if "collide" in l]
            # ..., Rock, Zou-He, mode, then the arguments
            assert len(name) == 1 and name[0].split("EvNS")[0].endswith(f"Li{{mode}}EE"), (n, kw, name)
            g.close()
    """)


def test_a_pending_error_of_the_caller_does_not_fail_transfers(so):
    """An error that an earlier call of the program left behind in the runtime
    is not the transfer's."""
    fakehip.run(so, """
        for precision in (0, 1):
            g = Lattice(12, 10, 8, ncomp=2, precision=precision)
            batch = Batch([(8, 6, 6)], ncomp=2, precision=precision)
            for call in (g.populations, g.density, g.momentum, g.download_sites, lambda: batch.populations(0),
                         lambda: g.upload_sites(np.zeros((10, 12, 14, 49)))):
                assert fake.hipSetDevice(7) != 0
                call()
    """)


@pytest.mark.parametrize("copy", [1, 2])
def test_failed_upload_leaves_the_step_alone(so, copy):
    """An upload that fails on its first or its last copy: before anything was
    written the moments of the last advection are still there; after it a
    two-pass step under way gets its moments again."""
    fakehip.run(so, f"""
        N = np.zeros((10, 12, 14, 49))
        fail = knob("fake_fail_copy", ctypes.c_int)
        for plan, calls in (((0,), 2), ((2, 32, 4, 4), 2), ((2, 32, 4, 4), 0)):
            g = Lattice(12, 10, 8, ncomp=2)
            g.set_plan(*plan)
            g.init_noise(1)
            g.time_loop(1)
            if calls:
                g.bc_apply(6, 2), g.advection()
            log()
            fail.value = {copy}
            try:
                g.upload_sites(N)
            except LB3DError as e:
                assert e.code == 2
            else:
                raise AssertionError("no error")
            names = "".join(log())
            assert ("put_sites" in names) == ({copy} == 2)
            again = {copy} == 2 and plan == (0,)
            assert ("k_moments" in names) == again, (plan, calls, names)
            g.download_sites()
            rebuilt = {copy} == 1 and plan != (0,)
            assert any("k_moments" in l for l in log()) == rebuilt, (plan, calls)
            if calls:
                g.bc_apply(8, 2), g.collision()
    """)
