"""Observables read back from the device: the Lees-Edwards x-halo planes, the
momentum field and the momentum transfer through x-planes (the reference's
shear stress, code/lb3d_io_stress.F90:38-173), against the oracle on the same
state."""
import numpy as np
import pytest

from lb3d_amd.gpu import LB3D_BC_LEES_EDWARDS, LB3D_FP32_DEV, LB3D_FP64, LB3DError, Lattice
from tests.test_gpu_parity import pair

pytestmark = pytest.mark.gpu

CX = np.array([1, -1, 0, 0, 0, 0, 1, 1, 1, 1, -1, -1, -1, -1, 0, 0, 0, 0, 0])
CY = np.array([0, 0, 1, -1, 0, 0, 1, -1, 0, 0, 1, -1, 0, 0, 1, 1, -1, -1, 0])
CZ = np.array([0, 0, 0, 0, 1, -1, 0, 0, 1, -1, 0, 0, 1, -1, 1, -1, 1, -1, 0])
G = np.array([2] * 6 + [1] * 13, dtype=float)


def oracle_halo(o):
    """x = 0 and x = nx+1 planes of the oracle's whole_N, shape (2, 2, 19, nz, ny)."""
    o.halo_refresh()
    N = o.N
    out = np.empty((2, 2, 19, o.nz, o.ny))
    for f, x in ((0, 0), (1, o.nx + 1)):
        for c in (0, 1):
            out[f, c] = N[1:-1, 1:-1, x, 24 * c:24 * c + 19].transpose(2, 0, 1)
    return out


@pytest.mark.parametrize("shear_u", [0.04, -0.3])
def test_le_halo_and_stress_match_oracle(shear_u):
    """Positive and negative offsets (lelo < 0 takes the other interpolation
    pair, and -0.3 drives the negativity clamp)."""
    o, g = pair(16, 12, 20, ncomp=2, g_br=0.09, boundary=LB3D_BC_LEES_EDWARDS, shear_u=shear_u,
                amp=(0.3, 0.3, 0.0) if shear_u < 0 else (0.01, 0.01, 0.0))
    o.run(7)
    g.time_loop(7)
    assert g.le_state()[1] == o.le_state()[1]
    want = oracle_halo(o)
    got = g.le_halo()
    d = np.abs(got - want).max()
    print(f"shear_u {shear_u}: max |halo diff| {d:.3e}")
    assert d <= 1e-12
    for planes in ((1, 16), (4, 9)):
        s_o = o.stress(*planes)
        s_g = g.shear_stress(*planes)
        np.testing.assert_allclose(s_g, s_o, rtol=1e-10, atol=1e-14)


def test_stress_periodic_matches_oracle_and_halo_needs_le():
    o, g = pair(12, 10, 8, ncomp=2, g_br=0.09)
    o.run(5)
    g.time_loop(5)
    o.halo_refresh()
    np.testing.assert_allclose(g.shear_stress(), o.stress(), rtol=1e-10, atol=1e-14)
    with pytest.raises(LB3DError):
        g.le_halo()


@pytest.mark.parametrize("ncomp", [2, 3])
def test_momentum_field(ncomp):
    """P_c = sum_i g_i n_c,i c_i of the device populations (FP64 form) and of
    the oracle's populations after the same steps."""
    o, g = pair(10, 9, 7, ncomp=ncomp, amp=(0.02, 0.02, 0.01))
    o.run(4)
    g.time_loop(4)
    P = g.momentum()
    n = o.populations()  # (C, 19, nz, ny, nx)
    want = np.stack([np.einsum("i,izyx->zyx", G * cv, n[c]) for c in range(ncomp)
                     for cv in (CX, CY, CZ)]).reshape(P.shape)
    np.testing.assert_allclose(P, want, rtol=0, atol=1e-13)


def test_fp32_le_halo_close_to_fp64():
    kw = dict(ncomp=2, g_br=0.08, boundary=LB3D_BC_LEES_EDWARDS, shear_u=0.05)
    _, g64 = pair(16, 16, 24, precision=LB3D_FP64, **kw)
    _, g32 = pair(16, 16, 24, precision=LB3D_FP32_DEV, **kw)
    g64.time_loop(20)
    g32.time_loop(20)
    h64, h32 = g64.le_halo(), g32.le_halo()
    rel = np.abs(h32 - h64).max() / np.abs(h64).max()
    print(f"FP32 vs FP64 halo planes: {rel:.3e}")
    assert rel < 1e-5
    s64, s32 = g64.shear_stress(), g32.shear_stress()
    print(f"mean shear stress FP64 {s64[2]:.6e} FP32 {s32[2]:.6e}")
    assert abs(s32[2] - s64[2]) <= 1e-3 * abs(s64[2]) + 1e-8


@pytest.mark.parametrize("ncomp", [2, 3])
def test_full_sanity_matches_oracle(ncomp):
    o, g = pair(11, 9, 7, ncomp=ncomp, amp=(0.02, 0.02, 0.01))
    o.run(6)
    g.time_loop(6)
    want, got = o.sanity_full(), g.sanity()
    for k in ("fluid_sites", "nan_sites", "negative_sites", "fast_sites"):
        assert got[k] == want[k], k
    np.testing.assert_allclose(got["mass"], want["mass"], rtol=1e-13)
    np.testing.assert_allclose(got["momentum"], want["momentum"], rtol=1e-9, atol=1e-13)
    np.testing.assert_allclose(got["vel_sum"], want["vel_sum"], rtol=1e-9, atol=1e-13)
    np.testing.assert_allclose(got["max_vel"], want["max_vel"], rtol=1e-12)
    np.testing.assert_array_equal(got["max_pos"], want["max_pos"])


@pytest.mark.parametrize("precision", [LB3D_FP64, LB3D_FP32_DEV])
def test_full_sanity_ties_keep_the_last_site(precision):
    """A uniform state: every site has the same velocity, and the maximum is
    reported at the last site of the reference's loop, (nx, ny, nz)."""
    g = Lattice(12, 10, 6, ncomp=2, precision=precision)
    g.init_noise(1, amp=(0.0, 0.0, 0.0), dipoles=False)
    s = g.sanity()
    assert s["fluid_sites"] == 720 and s["fast_sites"] == 0
    assert (s["max_pos"][:2] == [12, 10, 6]).all()
    assert (s["max_pos"][2] == 0).all()


@pytest.mark.parametrize("precision", [LB3D_FP64, LB3D_FP32_DEV])
@pytest.mark.parametrize("ncomp,dims,halo", [
    (2, (5, 3, 2), 1),          # fewer records than a block holds
    (3, (7, 9, 5), 3),          # a halo wider than one site
    (2, (2, 1, 1), 4),          # a halo wider than the lattice
    (2, (131, 130, 129), 1),    # several pieces of densities and of records
    (3, (57, 61, 66), 1),
    (2, (151, 150, 3), 1),      # one z plane of records larger than a piece
])
def test_device_conversions_equal_the_host_sums_bitwise(precision, ncomp, dims, halo):
    """Uploads, downloads, densities and momenta are converted on the device in
    the order of a host conversion: bitwise the numpy values."""
    nx, ny, nz = dims
    sd = 79 if ncomp == 3 else 49
    r = np.random.default_rng(7)
    N = np.full((nz + 2 * halo, ny + 2 * halo, nx + 2 * halo, sd), np.nan)  # the halo is not read
    I = N[halo:-halo, halo:-halo, halo:-halo]
    I[...] = 0.0
    for c in range(ncomp):
        I[..., 24 * c:24 * c + 19] = r.random((nz, ny, nx, 19)) / 20
    if ncomp == 3:
        I[..., 75:78] = r.random((nz, ny, nx, 3)) - 0.5
    w = np.array([1.0 / 36.0] * 18 + [1.0 / 3.0]) * 0.7
    g = Lattice(nx, ny, nz, ncomp=ncomp, precision=precision)
    for _ in range(2):  # the second upload lands in the other buffer
        g.upload_sites(N, halo_extent=halo, nt0=3)
    assert g.nt == 3
    want = np.stack([np.moveaxis(I[..., 24 * c:24 * c + 19], -1, 0) for c in range(ncomp)])
    if precision == LB3D_FP32_DEV:
        ww = w[None, :, None, None, None]
        want = ww + (want - ww).astype(np.float32).astype(np.float64)
    pops = g.populations()
    assert np.array_equal(pops, want)
    rho = np.zeros((ncomp, nz, ny, nx))
    mom = np.zeros((ncomp, 3, nz, ny, nx))
    for i in range(19):
        rho = rho + pops[:, i] * G[i]
        for a, cv in enumerate((CX, CY, CZ)):
            if cv[i]:
                mom[:, a] = mom[:, a] + (pops[:, i] * G[i]) * float(cv[i])
    assert np.array_equal(g.density(), rho)
    assert np.array_equal(g.momentum(), mom)
    J = np.zeros((nz, ny, nx, sd))
    for c in range(ncomp):
        J[..., 24 * c:24 * c + 19] = np.moveaxis(pops[c], 0, -1)
        J[..., 24 * c + 19] = rho[c]
        J[..., 24 * c + 20:24 * c + 23] = np.moveaxis(mom[c], 0, -1)
    if ncomp == 3:
        db = I[..., 75:78]
        J[..., 75:78] = db if precision == LB3D_FP64 else db.astype(np.float32)
    pad = ((halo, halo),) * 3 + ((0, 0),)
    assert np.array_equal(g.download_sites(halo_extent=halo), np.pad(J, pad, mode="wrap"))


def test_refused_rock_sites_leave_the_state():
    """Records with rock sites are refused on a ternary lattice; state, step
    counter and the moments of the last advection stay."""
    g = Lattice(6, 5, 4, ncomp=3)
    g.init_noise(1, amp=(0.01, 0.01, 0.01))
    g.set_plan(3, 32, 4, 4)  # one-pass: the moments are rebuilt when asked for
    g.time_loop(2)
    before = g.download_sites()
    g2 = Lattice(6, 5, 4, ncomp=3)
    g2.init_noise(1, amp=(0.01, 0.01, 0.01))
    g2.set_plan(3, 32, 4, 4)
    g2.time_loop(2)
    bad = before.copy()
    bad[2, 2, 2, 78] = 1.0
    with pytest.raises(LB3DError):
        g2.upload_sites(bad)
    assert g2.nt == 2
    assert np.array_equal(g2.download_sites(), before)
    g.time_loop(1)
    g2.time_loop(1)
    assert np.array_equal(g.populations(), g2.populations())


def test_transfers_of_several_threads_do_not_mix():
    """Transfer buffers are shared by all contexts, one set per transfer: two
    threads reading back and uploading their own lattices at the same time
    see their own data."""
    import threading
    lats = [Lattice(60, 61, 62, ncomp=2), Lattice(33, 70, 41, ncomp=3, precision=LB3D_FP32_DEV)]
    for k, g in enumerate(lats):
        g.init_noise(k, amp=(0.02, 0.01, 0.01))
    want = [(g.populations(), g.download_sites(), g.density()) for g in lats]
    bad = []

    def work(g, w):
        for _ in range(6):
            g.upload_sites(w[1])
            got = (g.populations(), g.download_sites(), g.density())
            if not all(np.array_equal(a, b) for a, b in zip(got, w)):
                bad.append(g)

    ts = [threading.Thread(target=work, args=a) for a in zip(lats, want)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


@pytest.mark.parametrize("precision", [LB3D_FP64, LB3D_FP32_DEV])
@pytest.mark.parametrize("dims,halo,ncomp", [((150, 149, 3), 1, 2), ((211, 97, 2), 3, 3), ((31, 5, 3000), 2, 2),
                                              ((40000, 1, 1), 1, 2)])
def test_uploads_in_several_pieces(precision, dims, halo, ncomp):
    """Records that cross to the device in pieces, which end anywhere in a row
    or its halo: populations, dipoles and rock sites as uploaded, whatever the
    halo records hold."""
    rng = np.random.default_rng(11)
    g = Lattice(*dims, ncomp=ncomp, precision=precision)
    nx, ny, nz = dims
    N = np.full((nz + 2 * halo, ny + 2 * halo, nx + 2 * halo, g.site_doubles), np.nan)
    sites = N[halo:-halo, halo:-halo, halo:-halo]
    sites[...] = rng.random(sites.shape)
    sites[..., -1] = rng.random((nz, ny, nx)) < 0.3 if ncomp == 2 else 0.0
    g.upload_sites(N, halo_extent=halo)
    want = np.stack([np.moveaxis(sites[..., 24 * c:24 * c + 19], -1, 0) for c in range(ncomp)])
    tol = 0.0 if precision == LB3D_FP64 else 2.0**-24  # the deviations are below 1
    assert np.abs(g.populations() - want).max() <= tol
    got = g.download_sites(halo)
    assert np.isfinite(got).all()
    got = got[halo:-halo, halo:-halo, halo:-halo]
    if ncomp == 3:
        assert np.abs(got[..., 75:78] - sites[..., 75:78]).max() <= tol
    assert np.array_equal(got[..., -1], sites[..., -1])


@pytest.mark.parametrize("dims", [(73, 42, 9), (5519, 5, 1)])
def test_fp32_populations_on_either_side_of_the_host_conversion(dims):
    """FP32 populations of up to 2^20 values are converted by the host, more by
    the device: w_i rho0 plus the stored deviation in 64 bits, bit for bit."""
    nx, ny, nz = dims
    w = np.array([1.0 / 36.0] * 18 + [1.0 / 3.0])
    rng = np.random.default_rng(3)
    g = Lattice(*dims, ncomp=2, precision=LB3D_FP32_DEV, rho0=(0.7, 0.6, 0.7))
    N = np.zeros((nz + 2, ny + 2, nx + 2, 49))
    want = []
    for c, rho0 in ((0, 0.7), (1, 0.6)):
        v = w * rho0 * rng.uniform(0.8, 1.2, (nz, ny, nx, 19))
        N[1:-1, 1:-1, 1:-1, 24 * c:24 * c + 19] = v
        base = w * rho0
        want.append(np.moveaxis(base + (v - base).astype(np.float32).astype(np.float64), -1, 0))
    g.upload_sites(N)
    assert (38 * nx * ny * nz <= 1 << 20) == (dims == (73, 42, 9))
    assert np.array_equal(g.populations(), np.stack(want))
