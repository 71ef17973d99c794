// lb3d_gpu.hip -- the C ABI of include/lb3d_gpu.h: contexts, device memory,
// the reference's stage sequence, HIP-graph replay, diagnostics and the
// conversion between the reference's AoS lattice and the device layout.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <utility>
#include <string>
#include <vector>

#include "lb3d_kernels.h"
#include "lb3d_readback.h"
#include "lb3d_solver.h"

using namespace lb3d;

namespace {

thread_local std::string g_err;

int fail(int code, const std::string &msg)
{
    g_err = msg;
    return code;
}

#define HIP_TRY(expr)                                                                     \
    do {                                                                                  \
        hipError_t e_ = (expr);                                                           \
        if (e_ != hipSuccess) {                                                           \
            (void)hipGetLastError(); /* reported here, not by the next call */            \
            return fail(LB3D_EHIP, std::string(#expr) + ": " + hipGetErrorString(e_));   \
        }                                                                                 \
    } while (0)

enum StageState { IDLE = 0, AFTER_BC6 = 1, AFTER_ADV = 2, AFTER_BC8 = 3 };

// The moments of the last advection: none since the state was set; in the aux
// field; or, after the one-pass plans, which keep none, to be rebuilt from the
// populations that it streamed: f[1-cur] once the step is complete, f[cur]
// between advection and collision.
enum MomentState { MOMENTS_NONE = 0, MOMENTS_KEPT, MOMENTS_PREV, MOMENTS_CUR };

// HIP events that are destroyed when the scope ends, also on an early error return
struct Events {
    std::vector<hipEvent_t> e;
    explicit Events(size_t n) : e(n, nullptr) {}
    Events(const Events &) = delete;
    Events &operator=(const Events &) = delete;
    ~Events()
    {
        for (hipEvent_t x : e)
            if (x) (void)hipEventDestroy(x);
    }
    hipError_t create()
    {
        for (hipEvent_t &x : e) {
            hipError_t r = hipEventCreate(&x);
            if (r != hipSuccess) return r;
        }
        return hipSuccess;
    }
    hipEvent_t &operator[](size_t i) { return e[i]; }
};

const char *const KNAMES[] = {"le_faces_pc", "moments",
                              "le_faces_aux",  "dipole",      "collide", "fused",
                              "dipole_collide"};
enum { K_LE6 = 0, K_MOM, K_LE8, K_DIP, K_COL, K_FUS, K_DC, K_COUNT };

const char *const STAGE_NAMES[3] = {"regs", "lds", "reload"};

// Tile shapes that lb3d_gpu_set_plan takes.
static bool listed_shape(int ncomp, int tx, int ty)
{
    if (ncomp == 2 && tx == 16) return false;  // 16 x 16 is a shape of the ternary kernel only
    for (auto &sh : FUSED_SHAPES)
        if (sh[0] == tx && sh[1] == ty) return true;
    return false;
}


}  // namespace

struct lb3d_ctx {
    lb3d_params p{};
    Launcher *L = nullptr;
    DevBufs b;
    hipStream_t stream = nullptr;
    int device = 0;  // that the context was made on
    int nt = 0;
    int state = IDLE;
    bool le = false;
    MomentState moments = MOMENTS_NONE;
    LEState host_le{};
    hipGraphExec_t graph = nullptr;
    int graph_len = 0;     // steps of the captured graph
    int64_t plan_steps = 0;  // steps run on the current plan (see replay_graph)
    double *d_partials = nullptr;
    uint8_t *rock_dev = nullptr;  // rock mask (lattices with walls)
    size_t f_bytes = 0, aux_bytes = 0, db_bytes = 0;
    size_t aux_elems = 0;  // elements of the aux field
    Plan plan;
    Plan displaced;  // fused: the one-pass plan that walls have taken the place of
    bool tuned = false;
    // ternary dipole fields, tied to the population parity: a step reads
    // dbk[cur] (the field of the state) and writes dbk[1-cur] (the relaxed
    // field), so a captured two-step graph finds the live field where it
    // expects it whatever the host did before
    void *dbk[2] = {nullptr, nullptr};
    // Lees-Edwards halo planes of the populations f[0] and f[1]: those that the
    // last step streamed through stay what they were while the planes of the
    // new state are built (rebuild_aux may still need them)
    void *facek[2] = {nullptr, nullptr};
    // Lees-Edwards: the edge columns b.edge_pc hold f[cur]'s (written by the
    // last kernel of a step, else gathered before the next halo-plane pass)
    bool edges_ok = false;
};

// The halo-plane kernels read the compact edge columns, which every step
// writes.
static void ensure_edges(lb3d_ctx *c)
{
    if (c->le && !c->edges_ok) {
        c->L->le_gather_edges(c->b, c->stream);
        c->edges_ok = true;
    }
}

// Points b.db / b.db_alt / b.face_pc at the fields of the current parity.
static void set_cur(lb3d_ctx *c, int cur)
{
    c->b.cur = cur;
    c->b.db = c->dbk[cur];
    c->b.db_alt = c->dbk[1 - cur];
    c->b.face_pc = c->facek[cur];
}

static void flip(lb3d_ctx *c) { set_cur(c, 1 - c->b.cur); }

static void drop_graph(lb3d_ctx *c)
{
    c->plan_steps = 0;
    if (c->graph) {
        (void)hipGraphExecDestroy(c->graph);
        c->graph = nullptr;
    }
}

static int check_params(const lb3d_params *p)
{
    if (!p) return fail(LB3D_EINVAL, "params is NULL");
    if (p->nx < 2 || p->ny < 1 || p->nz < 1)
        return fail(LB3D_EINVAL, "lattice extent must be nx>=2, ny>=1, nz>=1");
    if (p->ncomp != 2 && p->ncomp != 3) return fail(LB3D_EINVAL, "ncomp must be 2 or 3");
    if (p->bdist < 0 || p->bdist > 6)
        return fail(LB3D_EINVAL, "bdist must be 0-6 (code/lb3d_bdist.F90; 7 computes nothing there)");
    if (p->precision != LB3D_FP64 && p->precision != LB3D_FP32_DEV)
        return fail(LB3D_EINVAL, "precision must be LB3D_FP64 or LB3D_FP32_DEV");
    if (p->boundary != LB3D_BC_PERIODIC && p->boundary != LB3D_BC_LEES_EDWARDS)
        return fail(LB3D_EINVAL, "boundary must be periodic or Lees-Edwards");
    if (p->boundary == LB3D_BC_LEES_EDWARDS && p->ncomp == 3)
        // code/lb3d_compatibility.F90:105-108
        return fail(LB3D_EINVAL, "Lees-Edwards boundaries are not supported with surfactant");
    for (int c = 0; c < p->ncomp; c++)
        if (!(p->tau[c] > 0.0) || !(p->amass[c] > 0.0))
            return fail(LB3D_EINVAL, "tau and amass must be positive");
    if (p->ncomp == 3 && !(p->tau_d > 0.0)) return fail(LB3D_EINVAL, "tau_d must be positive");
    if (p->inv_fluid != 0 && p->inv_fluid != 12)
        return fail(LB3D_EINVAL, "inv_fluid must be 0 (no invasion) or 12 (the Zou-He flux boundary)");
    if (p->inv_fluid == 12 && p->boundary == LB3D_BC_LEES_EDWARDS)
        return fail(LB3D_EINVAL, "the Zou-He boundary needs a periodic lattice");
    if (p->inv_fluid == 12 && (p->inv_type < -1 || p->inv_type > 1))
        return fail(LB3D_EINVAL, "inv_type must be -1, 0 or 1 (code/lb3d_invasion.F90:2136-2140)");
    double sites = (double)p->nx * (double)p->ny * (double)p->nz;
    if (sites * 19.0 * p->ncomp >= 4294967296.0)
        return fail(LB3D_EINVAL, "lattice too large for 32-bit population indexing");
    return LB3D_OK;
}

namespace lb3d {
namespace {
std::mutex g_io_mu;
HostIO *g_io[IO_KEPT] = {};
int g_io_users = 0;
}  // namespace

HostIO *io_lend()
{
    int dev = -1;
    (void)hipGetDevice(&dev);
    {
        std::lock_guard<std::mutex> lock(g_io_mu);
        for (HostIO *&q : g_io)
            if (q && q->device == dev) {
                HostIO *io = q;
                q = nullptr;
                return io;
            }
    }
    HostIO *io = new HostIO();
    io->device = dev;
    return io;
}

void io_give_back(HostIO *io)
{
    if (!io->pageable) {
        std::lock_guard<std::mutex> lock(g_io_mu);
        if (g_io_users > 0)
            for (HostIO *&q : g_io)
                if (!q) {
                    q = io;
                    return;
                }
    }
    io->release();
    delete io;
}

void io_users(int change)
{
    HostIO *gone[IO_KEPT] = {};
    {
        std::lock_guard<std::mutex> lock(g_io_mu);
        g_io_users += change;
        if (g_io_users == 0)
            for (size_t k = 0; k < IO_KEPT; k++) std::swap(gone[k], g_io[k]);
    }
    for (HostIO *io : gone)
        if (io) {
            io->release();
            delete io;
        }
}

// The one-pass kernel (binary, bdist 2) with a tile fitted to the
// lattice, or the two-pass kernels.
//
// Which: the one-pass kernel moves 60% of the two-pass plan's bytes, but every
// z-chunk computes 2 planes of psi more than it collides and its planes are a
// serial chain, so it needs enough planes for all CUs.  Measured per step,
// two-pass against one-pass with the tile below (us):
//   FP32  64^3 24 / 26, 80^3 41 / 41, 90x100x77 51 / 47, 96^3 70 / 58,
//         112^3 135 / 103, 128^3 202 / 142, 200^3 757 / 554, 256^3 1592 / 1088;
//   FP64  61x47x53 31 / 35, 64^3 44 / 45, 77x91x69 87 / 80, 90x100x77 141 / 130,
//         128^3 386 / 300, 256^3 3170 / 2390.
// So the lines lie at 0.6 and 0.4 million sites.  Lees-Edwards, whose one-pass
// plan streams the edge columns once more for the post-advection halo planes:
//   FP32  96^3 91 / 93, 256x64x64 109 / 102, 96x100x110 127 / 118, 128x128x64
//         112 / 108, 128x128x80 138 / 133, 89x135x140 216 / 193, 128^3 224 / 191,
//         160^3 424 / 389, 192^3 690 / 599 (the two passes' figures are up to 9%
//         lower or higher from one allocation of the lattice to the next);
//   FP64  140x41x93 126 / 122, 60x84x111 134 / 128, 96^3 187 / 181, 256x64x64
//         223 / 194, 128^3 421 / 358, 160^3 840 / 775:
// 1 and 0.5 million sites.
//
// Tile: 512 threads (one work-group fills a CU's registers), the shape that
// leaves the fewest threads idle over the whole plane.  A tile narrower than
// the row pays for its x halo, the more the narrower it is (FP32, against the
// time of the whole-row tile with as many tiles: 128 columns +10-18%, 100
// +16%, 75 +4%, 64 +7%, 45 +11%, 42 +15%, 32 +25%, 30 +36%; 96^3: 96x5 58 us,
// 32x16 65, 90x100x77: 90x5 47 us, 30x17 58).  FP64 planes do not fit the L2
// with their halos, so there the halo sites count too (256^3: 64x8 2.39 ms,
// 128x4 2.49, 256x2 2.62; 200^3: 100x5 1.24 ms, 50x10 1.31); and with
// Lees-Edwards (256x64x64 FP32: 64x8 95 us, 128x4 103, 256x2 106; not below
// 48 columns there: 134x90x104 in 34x15 took 1.17 of the two-pass step).
//
// z-chunk: the work-groups run in rounds of 256 (one per CU), each lz + 2
// planes long; the fewest planes in a row win (200^3 FP32: 240 work-groups of
// 67 planes 555 us, 480 of 34 614).
//
// XCD chunks of the two-pass plan: one run of tiles per XCD while the
// populations fit the memory-side cache (90x100x77 ternary FP32 132 us, in
// chunks of 8 136, plain order 143); beyond it the eight runs open eight times
// as many DRAM pages as chunks of 8 tiles do (80x96x88 ternary FP64 256 / 237
// us, 192^3 ternary FP32 1249 / 1199, 160^3 FP64 794 / 753).
Plan two_pass_plan(const lb3d_params &p)
{
    Plan q;
    const uint64_t sites = (uint64_t)p.nx * (uint64_t)p.ny * (uint64_t)p.nz;
    if (19u * (uint64_t)p.ncomp * sites * (p.precision == LB3D_FP64 ? 8u : 4u) > MALL_BYTES) q.xg = 8;
    return q;
}

// The search visits each tile width and each chunk length once and ends where
// nothing shorter can cost less (lb3d_gpu_step_noalloc does it in every call: some us
// at most, 2 ms for a column of 400,000 planes when every number of chunks was tried).
Plan default_plan(const lb3d_params &p)
{
    Plan q = two_pass_plan(p);
    const bool fp64 = p.precision == LB3D_FP64;
    const int64_t sites = (int64_t)p.nx * p.ny * p.nz;
    const bool le = p.boundary == LB3D_BC_LEES_EDWARDS;
    if (p.ncomp != 2 || p.bdist != 2 || p.inv_fluid != 0 || !(le || p.boundary == LB3D_BC_PERIODIC)) return q;
    if (sites < (le ? (fp64 ? 500000 : 1000000) : (fp64 ? 400000 : 600000))) return q;
    const int T = 512, CUS = 256;
    double best = 0.0;
    // (the smallest number of tiles of each width: more of them cost more)
    for (int kx = (p.nx + T - 1) / T, tx; ; kx = (p.nx + tx - 2) / (tx - 1)) {
        tx = (p.nx + kx - 1) / kx;
        if (tx < (le && !fp64 ? 48 : 16) && kx > 1) break;
        int ty = T / tx < p.ny ? T / tx : p.ny;
        if (ty > fused2_sites(T) / (tx + 2) - 2) ty = fused2_sites(T) / (tx + 2) - 2;
        if (ty < 1) continue;
        const int ky = (p.ny + ty - 1) / ty;
        ty = (p.ny + ky - 1) / ky;
        // more than 256 sites, or the kernel would be that of a smaller work-group
        if (tx * ty <= T / 2) continue;
        const double nh = 2.0 * (tx + 2) + 2.0 * ty;
        const double cost = (double)kx * ky * (fp64 || le ? T + 0.2 * nh : T) * (kx > 1 ? 1.04 + 6.0 / tx : 1.0);
        if (best == 0.0 || cost < best) {
            best = cost;
            q.tx = tx;
            q.ty = ty;
            q.fused = true;
        }
    }
    if (!q.fused) return q;
    const int64_t tiles = (int64_t)((p.nx + q.tx - 1) / q.tx) * ((p.ny + q.ty - 1) / q.ty);
    const int64_t least = (tiles * p.nz + CUS - 1) / CUS;  // planes in a row without those computed twice
    int64_t planes = 0;
    for (int kz = 1, lz; ; kz = (p.nz + lz - 2) / (lz - 1)) {
        lz = (p.nz + kz - 1) / kz;
        const int64_t rounds = (tiles * ((p.nz + lz - 1) / lz) + CUS - 1) / CUS, c = rounds * (lz + 2);
        if (!planes || c < planes) {
            planes = c;
            q.lz = lz;
        }
        // shorter chunks take as many rounds at least
        if (lz == 1 || least + 2 * rounds >= planes) break;
    }
    q.stage = 0;
    q.xg = 32;
    return q;
}

void reduce_sanity(const double *h, unsigned nb, int ncomp, int nx, int ny, int nz, lb3d_sanity *out)
{
    std::memset(out, 0, sizeof *out);
    double acc[SAN_MAX] = {0};
    double mx[9], key[9];
    for (int k = 0; k < 9; k++) mx[k] = key[k] = -1.0;
    for (unsigned b = 0; b < nb; b++) {
        const double *p = h + (size_t)b * NSAN;
        for (int k = 0; k < SAN_MAX; k++) acc[k] = acc[k] + p[k];
        for (int k = 0; k < 9; k++) {
            double m = p[SAN_MAX + k], q = p[SAN_KEY + k];
            if (m > mx[k] || (m == mx[k] && q > key[k])) {
                mx[k] = m;
                key[k] = q;
            }
        }
    }
    for (int k = 0; k < 3; k++) {
        out->mass[k] = k < ncomp ? acc[k] : 0.0;
        out->momentum[k] = acc[3 + k];
    }
    out->nan_sites = (int64_t)llround(acc[6]);
    out->negative_sites = (int64_t)llround(acc[7]);
    out->fast_sites = (int64_t)llround(acc[8]);
    out->fluid_sites = (int64_t)llround(acc[SAN_FLUID]);
    for (int c = 0; c < 3; c++)
        for (int a = 0; a < 3; a++) {
            int k = 3 * c + a;
            out->vel_sum[c][a] = c < ncomp ? acc[SAN_VSUM + k] : 0.0;
            if (c < ncomp && key[k] >= 0.0) {
                long long q = llround(key[k]);
                out->max_vel[c][a] = mx[k];
                out->max_pos[c][a][0] = (int32_t)(q / ((long long)ny * nz)) + 1;
                out->max_pos[c][a][1] = (int32_t)((q / nz) % ny) + 1;
                out->max_pos[c][a][2] = (int32_t)(q % nz) + 1;
            }
        }
    (void)nx;
}

int set_error(int code, const char *msg) { return fail(code, msg); }
void clear_error() { g_err.clear(); }
double rho0_of(const lb3d_params &p, int k) { return p.rho0[k] > 0.0 ? p.rho0[k] : 0.7; }

int aos_to_device_layout(const lb3d_params &p, const double *N, int h, int sd,
                         std::vector<unsigned char> &f_bytes, std::vector<unsigned char> &db_bytes)
{
    const int C = p.ncomp;
    if (sd != (C == 3 ? 79 : 49)) return fail(LB3D_EINVAL, "site_doubles must be 79 (ternary) or 49 (binary)");
    if (h < 1) return fail(LB3D_EINVAL, "halo_extent must be >= 1");
    const int nx = p.nx, ny = p.ny, nz = p.nz;
    const size_t ns = (size_t)nx * ny * nz;
    const size_t lx = nx + 2 * h, ly = ny + 2 * h;
    const int rock_off = C == 3 ? 78 : 48;
    const bool dev = p.precision == LB3D_FP32_DEV;
    const size_t rs = dev ? 4 : 8;
    f_bytes.assign((size_t)C * 19 * ns * rs, 0);
    db_bytes.assign(C == 3 ? 3 * ns * rs : 0, 0);
    float *ff = (float *)f_bytes.data();
    double *fd = (double *)f_bytes.data();
    float *dbf = (float *)db_bytes.data();
    double *dbd = (double *)db_bytes.data();
    for (int z = 0; z < nz; z++)
        for (int y = 0; y < ny; y++)
            for (int x = 0; x < nx; x++) {
                const double *S = N + ((size_t)(x + h) + lx * ((size_t)(y + h) + ly * (size_t)(z + h))) * sd;
                size_t s = (size_t)x + (size_t)nx * ((size_t)y + (size_t)ny * z);
                if (S[rock_off] != 0.0)
                    return fail(LB3D_EINVAL, "rock sites are not supported here (rock_state must be 0)");
                for (int k = 0; k < C; k++)
                    for (int i = 0; i < 19; i++) {
                        double v = S[24 * k + i];
                        size_t q = ((size_t)k * 19 + i) * ns + s;
                        if (dev)
                            ff[q] = (float)(v - (i < 18 ? 1.0 / 36.0 : 1.0 / 3.0) * rho0_of(p, k));
                        else
                            fd[q] = v;
                    }
                if (C == 3)
                    for (int k = 0; k < 3; k++) {
                        if (dev)
                            dbf[k * ns + s] = (float)S[75 + k];
                        else
                            dbd[k * ns + s] = S[75 + k];
                    }
            }
    return LB3D_OK;
}

}  // namespace lb3d

extern "C" {

int lb3d_gpu_abi_version(void) { return LB3D_ABI_VERSION; }

const char *lb3d_gpu_last_error(void) { return g_err.c_str(); }

int lb3d_gpu_create(const lb3d_params *p, lb3d_ctx **out)
{
    g_err.clear();
    if (!out) return fail(LB3D_EINVAL, "out is NULL");
    *out = nullptr;
    int rc = check_params(p);
    if (rc) return rc;
    lb3d_ctx *c = new lb3d_ctx();
    io_users(1);
    (void)hipGetDevice(&c->device);
    c->p = *p;
    c->le = p->boundary == LB3D_BC_LEES_EDWARDS;
    c->L = p->precision == LB3D_FP64 ? make_launcher_fp64(*p) : make_launcher_fp32(*p);
    size_t rs = c->L->real_bytes();
    size_t ns = (size_t)p->nx * p->ny * p->nz;
    c->aux_elems = aux_elems(p->ncomp, ns);
    c->f_bytes = (size_t)p->ncomp * 19 * ns * rs;
    c->aux_bytes = c->aux_elems * rs;
    c->db_bytes = p->ncomp == 3 ? 3 * ns * rs : 0;
    size_t plane = (size_t)p->ny * p->nz;
    auto cleanup = [&](int code, const std::string &m) {
        lb3d_gpu_destroy(c);
        return fail(code, m);
    };
    hipError_t e;
    if ((e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking)) != hipSuccess)
        return cleanup(LB3D_EHIP, std::string("hipStreamCreate: ") + hipGetErrorString(e));
    for (int k = 0; k < 2; k++)
        if ((e = hipMalloc(&c->b.f[k], c->f_bytes)) != hipSuccess)
            return cleanup(LB3D_ENOMEM, std::string("hipMalloc populations: ") + hipGetErrorString(e));
    if ((e = hipMalloc(&c->b.aux, c->aux_bytes)) != hipSuccess)
        return cleanup(LB3D_ENOMEM, std::string("hipMalloc aux: ") + hipGetErrorString(e));
    if (c->db_bytes && ((e = hipMalloc(&c->dbk[0], c->db_bytes)) != hipSuccess ||
                        (e = hipMalloc(&c->dbk[1], c->db_bytes)) != hipSuccess))
        return cleanup(LB3D_ENOMEM, std::string("hipMalloc db: ") + hipGetErrorString(e));
    if (c->le) {
        const size_t edges = EDGE_SITES * plane * rs;
        if ((e = hipMalloc(&c->b.edge_pc, edges)) != hipSuccess || (e = hipMalloc(&c->b.edge_adv, edges)) != hipSuccess)
            return cleanup(LB3D_ENOMEM, std::string("hipMalloc LE edge columns: ") + hipGetErrorString(e));
        const size_t faces = 2 * 2 * 19 * plane * rs, step = (faces + 255) / 256 * 256;
        if ((e = hipMalloc(&c->facek[0], step + faces)) != hipSuccess ||
            (e = hipMalloc(&c->b.face_aux, 2 * 4 * plane * rs)) != hipSuccess)
            return cleanup(LB3D_ENOMEM, std::string("hipMalloc LE planes: ") + hipGetErrorString(e));
        c->facek[1] = (char *)c->facek[0] + step;
    }
    set_cur(c, 0);
    if ((e = hipMalloc((void **)&c->b.le, sizeof(LEState))) != hipSuccess ||
        (e = hipMalloc((void **)&c->d_partials, (size_t)c->L->diag_blocks() * NSAN * sizeof(double))) !=
            hipSuccess)
        return cleanup(LB3D_ENOMEM, std::string("hipMalloc: ") + hipGetErrorString(e));
    // lb3d_gpu_autotune picks the measured best
    c->plan = default_plan(*p);
    if (c->plan.fused && !c->L->fused_supported(c->plan.tx, c->plan.ty, c->plan.stage)) c->plan = two_pass_plan(*p);
    c->L->xg = c->plan.xg;
    c->host_le.shear_u = p->shear_u;
    c->host_le.shear_tmp = p->shear_u;
    c->host_le.shear_sum = p->shear_sum;
    c->host_le.shear_omega = p->shear_omega;
    *out = c;
    return LB3D_OK;
}

int lb3d_gpu_destroy(lb3d_ctx *c)
{
    if (!c) return LB3D_OK;
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    drop_graph(c);
    for (int k = 0; k < 2; k++)
        if (c->b.f[k]) (void)hipFree(c->b.f[k]);
    if (c->b.aux) (void)hipFree(c->b.aux);
    for (int k = 0; k < 2; k++)
        if (c->dbk[k]) (void)hipFree(c->dbk[k]);
    if (c->b.edge_pc) (void)hipFree(c->b.edge_pc);
    if (c->b.edge_adv) (void)hipFree(c->b.edge_adv);
    if (c->facek[0]) (void)hipFree(c->facek[0]);  // (one allocation)
    if (c->b.face_aux) (void)hipFree(c->b.face_aux);
    if (c->b.le) (void)hipFree(c->b.le);
    if (c->d_partials) (void)hipFree(c->d_partials);
    if (c->rock_dev) (void)hipFree(c->rock_dev);
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c->L;
    delete c;
    io_users(-1);
    return LB3D_OK;
}

static int push_le(lb3d_ctx *c)
{
    HIP_TRY(hipMemcpyAsync(c->b.le, &c->host_le, sizeof(LEState), hipMemcpyHostToDevice, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    return LB3D_OK;
}

static int pull_le(lb3d_ctx *c)
{
    HIP_TRY(hipMemcpyAsync(&c->host_le, c->b.le, sizeof(LEState), hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    return LB3D_OK;
}

static bool is_dev(const lb3d_ctx *c) { return c->p.precision == LB3D_FP32_DEV; }
static double rho0_of(const lb3d_ctx *c, int k) { return lb3d::rho0_of(c->p, k); }
static double w_of(int i) { return i < 18 ? 1.0 / 36.0 : 1.0 / 3.0; }

// Walls on (the mask is in rock_dev) or off.  With walls only the two-pass
// plan exists, so a one-pass plan falls back to it, and is back once the walls
// are gone unless another plan has been set since.
static void set_walls(lb3d_ctx *c, bool on)
{
    // a captured graph holds the kernels of the old wall state (the mask
    // itself is read from the same buffer by every replay)
    if (on != (c->b.rock != nullptr)) drop_graph(c);
    c->L->walls = on;
    c->b.rock = on ? c->rock_dev : nullptr;
    if (on && c->plan.fused) {
        c->displaced = c->plan;
        c->plan = two_pass_plan(c->p);
    } else if (!on && c->displaced.fused) {
        c->plan = c->displaced;
        c->displaced = Plan();
    }
    c->L->xg = c->plan.xg;
}

// Site records.
static RecLayout rec_layout(const lb3d_params &p, int h, int sd)
{
    RecLayout L;
    L.nx = p.nx;
    L.ny = p.ny;
    L.nz = p.nz;
    L.h = h;
    L.sd = sd;
    L.C = p.ncomp;
    L.ns = (uint32_t)p.nx * (uint32_t)p.ny * (uint32_t)p.nz;
    L.rock_r = p.rock_colour_r;
    L.rock_b = p.rock_colour_b;
    return L;
}
static int rebuild_aux(lb3d_ctx *c);

int lb3d_gpu_upload_sites(lb3d_ctx *c, const double *N, int32_t h, int32_t sd, int32_t nt0)
{
    g_err.clear();
    if (!c || !N) return fail(LB3D_EINVAL, "NULL argument");
    const OnDevice on(c->device);
    const lb3d_params &p = c->p;
    if (sd != (p.ncomp == 3 ? 79 : 49)) return fail(LB3D_EINVAL, "site_doubles must be 79 (ternary) or 49 (binary)");
    if (h < 1) return fail(LB3D_EINVAL, "halo_extent must be >= 1");
    const bool walls_ok = p.ncomp == 2 && !c->le && p.inv_fluid != 12;
    // The records are converted into the buffers that do not hold the state,
    // which becomes current only once the rock sites are known to be
    // supported.  (Where they are not, what those buffers hold, the input of
    // the last step, may still be asked for: its moments are kept first.)
    int rc = LB3D_OK;
    if (!walls_ok && (rc = rebuild_aux(c))) return rc;
    const RecLayout L = rec_layout(p, h, sd);
    // the mask goes to the aux field, which holds nothing after an upload, and
    // from there to its own memory if there are rock sites
    uint8_t *mask = walls_ok ? (uint8_t *)c->b.aux : nullptr;
    // where the upload fails after that, the moments of the last advection are
    // gone, and a two-pass step under way gets its own again
    struct Lost {
        lb3d_ctx *c;
        bool armed = false;
        ~Lost()
        {
            if (!armed) return;
            const bool under_way = !c->plan.fused && (c->state == AFTER_ADV || c->state == AFTER_BC8);
            if (under_way) c->L->moments(c->b, c->stream);
            c->moments = under_way && c->moments != MOMENTS_NONE ? MOMENTS_KEPT : MOMENTS_NONE;
        }
    } lost{c};
    IoLoan io;
    const PopBase pb = pop_base(p);
    const int to = 1 - c->b.cur;
    // the records of the z planes that hold sites
    const size_t plane = (size_t)(p.nx + 2 * h) * (size_t)(p.ny + 2 * h), skip = (size_t)h * plane;
    const size_t rec = (size_t)sd * 8, lds = (size_t)REC_SITES * rec;  // bytes of a record and of a block of them
    HIP_TRY(io->counter());
    HIP_TRY(hipMemsetAsync(io->count, 0, sizeof(uint32_t), c->stream));
    HIP_TRY(io->up(c->stream, N + skip * sd, (size_t)p.nz * plane * rec, lds, [&](size_t at, size_t len, void *buf) {
        const uint32_t n = (uint32_t)(len / rec), nb = (n + REC_SITES - 1) / REC_SITES;
        lost.armed = walls_ok;
        auto go = [&](auto r) {
            using R = decltype(r);
            k_put_sites<R><<<nb, 256, lds, c->stream>>>((const double *)buf, L, pb, (uint32_t)(skip + at / rec), n,
                                                        (R *)c->b.f[to], (R *)c->dbk[to], mask, io->count);
        };
        is_dev(c) ? go(float()) : go(double());
    }));
    uint32_t nrock = 0;
    const hipError_t counted = hipMemcpyAsync(io->pin[0], io->count, sizeof nrock, hipMemcpyDeviceToHost, c->stream);
    HIP_TRY(hipStreamSynchronize(c->stream));  // (the loan ends with its buffers at rest)
    HIP_TRY(counted);
    std::memcpy(&nrock, io->pin[0], sizeof nrock);
    if (nrock && !walls_ok) {
        if (p.ncomp != 2 || c->le)
            return fail(LB3D_EINVAL, "rock sites (walls) are supported on periodic binary lattices");
        return fail(LB3D_EINVAL, "rock sites (walls) and the Zou-He boundary are not supported together");
    }
    if (nrock) {
        if (!c->rock_dev) HIP_TRY(hipMalloc((void **)&c->rock_dev, L.ns));
        HIP_TRY(hipMemcpyAsync(c->rock_dev, mask, L.ns, hipMemcpyDeviceToDevice, c->stream));
    }
    lost.armed = false;
    set_walls(c, nrock != 0);
    set_cur(c, to);
    c->nt = nt0;
    c->host_le.nt = nt0;
    c->state = IDLE;
    c->moments = MOMENTS_NONE;
    c->edges_ok = false;
    return LB3D_OK;
}

int lb3d_gpu_init_noise(lb3d_ctx *c, uint64_t seed, const double rho_mean[3], const double amp[3],
                        int32_t dipoles)
{
    g_err.clear();
    if (!c || !rho_mean || !amp) return fail(LB3D_EINVAL, "NULL argument");
    set_walls(c, false);
    set_cur(c, 0);
    c->L->init_noise(c->b, seed, rho_mean, amp, dipoles, c->stream);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(c->stream));
    c->nt = 0;
    c->host_le.nt = 0;
    c->state = IDLE;
    c->moments = MOMENTS_NONE;
    c->edges_ok = false;
    return LB3D_OK;
}

int lb3d_gpu_get_populations(lb3d_ctx *c, double *out)
{
    g_err.clear();
    if (!c || !out) return fail(LB3D_EINVAL, "NULL argument");
    const OnDevice on(c->device);
    const void *f = c->b.f[c->b.cur];
    HIP_TRY(is_dev(c) ? fetch_populations<float>(c->stream, c->p, f, out)
                      : fetch_populations<double>(c->stream, c->p, f, out));
    return LB3D_OK;
}

// The one-pass plans keep no moments: rebuild those of the last advection
// from the populations that it streamed, with the dipole field that its step
// read and the Lees-Edwards halo planes of that step.
static int rebuild_aux(lb3d_ctx *c)
{
    if (c->moments != MOMENTS_PREV && c->moments != MOMENTS_CUR) return LB3D_OK;
    DevBufs src = c->b;
    if (c->moments == MOMENTS_PREV) {
        src.cur = 1 - c->b.cur;
        src.db = c->b.db_alt;
        src.face_pc = c->facek[src.cur];
    }
    c->L->moments(src, c->stream);
    HIP_TRY(hipGetLastError());
    c->moments = MOMENTS_KEPT;
    return LB3D_OK;
}

int lb3d_gpu_download_sites(lb3d_ctx *c, double *N, int32_t h, int32_t sd)
{
    g_err.clear();
    if (!c || !N) return fail(LB3D_EINVAL, "NULL argument");
    const OnDevice on(c->device);
    const int C = c->p.ncomp;
    if (sd != (C == 3 ? 79 : 49)) return fail(LB3D_EINVAL, "site_doubles must be 79 (ternary) or 49 (binary)");
    if (h < 1) return fail(LB3D_EINVAL, "halo_extent must be >= 1");
    if (int rc = rebuild_aux(c)) return rc;
    const RecLayout L = rec_layout(c->p, h, sd);
    const PopBase pb = pop_base(c->p);
    const size_t recs = (size_t)(c->p.nx + 2 * h) * (size_t)(c->p.ny + 2 * h) * (size_t)(c->p.nz + 2 * h);
    const size_t rec = (size_t)sd * 8, lds = (size_t)REC_SITES * rec;  // bytes of a record and of a block of them
    IoLoan io;
    HIP_TRY(io->down(c->stream, N, recs * rec, lds, true, [&](size_t at, size_t len, void *buf) -> const void * {
        const uint32_t n = (uint32_t)(len / rec), nb = (n + REC_SITES - 1) / REC_SITES;
        auto go = [&](auto r) {
            using R = decltype(r);
            k_get_sites<R><<<nb, 256, lds, c->stream>>>(
                (const R *)c->b.f[c->b.cur], c->moments == MOMENTS_KEPT ? (const R *)c->b.aux : nullptr, (const R *)c->b.db,
                c->b.rock, pb, rho0_of(c, 0), rho0_of(c, 1), rho0_of(c, 2), L, (uint32_t)(at / rec), n, (double *)buf);
        };
        is_dev(c) ? go(float()) : go(double());
        return buf;
    }));
    return LB3D_OK;
}

int lb3d_gpu_bc_init(lb3d_ctx *c)
{
    g_err.clear();
    if (!c) return fail(LB3D_EINVAL, "NULL context");
    if (c->le) {
        // code/lb3d_bc.F90:58-78 then le_neighbours (code/lb3d_bc_leesedwards.F90:86-140)
        LEState &L = c->host_le;
        L.shear_u = ((double)c->p.nx / ((double)c->p.nx - 1.0)) * c->p.shear_u;
        L.shear_tmp = L.shear_u;
        L.shear_sum = c->p.shear_sum;
        L.shear_omega = c->p.shear_omega;
        if (c->p.restore) L.shear_sum = L.shear_sum - L.shear_u;
        L.shear_sum = L.shear_sum + L.shear_u;
        long t = (long)(2.0 * L.shear_sum);
        L.lelo = (int)(t % (long)c->p.nz);
        double lf = 2.0 * L.shear_sum;
        L.lefrac = std::fabs(lf - std::trunc(lf));
        L.nt = c->nt;
        return push_le(c);
    }
    return LB3D_OK;
}

int lb3d_gpu_force_apply(lb3d_ctx *c, int32_t stage)
{
    g_err.clear();
    if (!c) return fail(LB3D_EINVAL, "NULL context");
    // lbe_force_apply: the constant and Kolmogorov forces are outside this path
    if (stage != 6 && stage != 8 && stage != 10) return fail(LB3D_EINVAL, "force_apply stage must be 6, 8 or 10");
    return LB3D_OK;
}

static void launch_le_neighbours(lb3d_ctx *c, int nt_set)
{
    k_le_neighbours<<<1, 64, 0, c->stream>>>(c->b.le, c->p.nz, nt_set);
}

int lb3d_gpu_bc_apply(lb3d_ctx *c, int32_t stage, int32_t nt)
{
    g_err.clear();
    if (!c) return fail(LB3D_EINVAL, "NULL context");
    if (stage == 6) {
        if (c->state != IDLE) return fail(LB3D_ESTATE, "bc_apply(6) must follow a collision or init");
        if (c->le) {
            ensure_edges(c);
            launch_le_neighbours(c, nt);
            c->L->le_faces(c->b, false, false, c->stream);
            HIP_TRY(hipGetLastError());
        }
        c->nt = nt;
        c->state = AFTER_BC6;
    } else if (stage == 8) {
        if (c->state != AFTER_ADV) return fail(LB3D_ESTATE, "bc_apply(8) must follow advection");
        if (c->le) {
            ensure_edges(c);  // (set_plan may have come between, for whose plan they are gathered anew)
            c->L->le_faces(c->b, true, c->plan.fused, c->stream);
            HIP_TRY(hipGetLastError());
        }
        c->state = AFTER_BC8;
    } else if (stage == 10) {
        if (c->state != IDLE) return fail(LB3D_ESTATE, "bc_apply(10) must follow a collision");
    } else {
        return fail(LB3D_EINVAL, "bc_apply stage must be 6, 8 or 10");
    }
    return LB3D_OK;
}

int lb3d_gpu_advection(lb3d_ctx *c)
{
    g_err.clear();
    if (!c) return fail(LB3D_EINVAL, "NULL context");
    if (c->state != AFTER_BC6) return fail(LB3D_ESTATE, "advection must follow bc_apply(6)");
    // the one-pass plan streams inside the collision kernel
    if (!c->plan.fused) {
        c->L->moments(c->b, c->stream);
        HIP_TRY(hipGetLastError());
    }
    if (c->moments != MOMENTS_NONE) c->moments = c->plan.fused ? MOMENTS_CUR : MOMENTS_KEPT;
    c->state = AFTER_ADV;
    return LB3D_OK;
}

// The collision of the current plan: f[cur] -> f[1-cur]; the ternary dipole
// relaxation reads the state's field db and writes db_alt (both plans).
// Plans are validated when they are set (lb3d_gpu_set_plan, autotune,
// create); a launcher that still rejects one returns LB3D_EINVAL.
static int launch_collision(lb3d_ctx *c)
{
    if (c->plan.fused) {
        if (!c->L->fused(c->b, c->plan.tx, c->plan.ty, c->plan.lz, c->plan.stage, c->stream))
            return fail(LB3D_EINVAL, "the one-pass plan has no kernel for this lattice");
    } else if (!c->L->dipole_collide(c->b, c->stream)) {
        c->L->dipole(c->b, c->stream);
        c->L->collide(c->b, c->stream);
    }
    return LB3D_OK;
}

static void mark_stepped(lb3d_ctx *c)
{
    c->moments = c->plan.fused ? MOMENTS_PREV : MOMENTS_KEPT;
}

int lb3d_gpu_collision(lb3d_ctx *c)
{
    g_err.clear();
    if (!c) return fail(LB3D_EINVAL, "NULL context");
    if (c->state != AFTER_BC8) return fail(LB3D_ESTATE, "collision must follow bc_apply(8)");
    int rc = launch_collision(c);
    if (rc) return rc;
    HIP_TRY(hipGetLastError());
    flip(c);
    c->edges_ok = true;
    c->state = IDLE;
    mark_stepped(c);
    return LB3D_OK;
}

// One whole timestep on the stream (graph-capturable: kernels only).
static int enqueue_step(lb3d_ctx *c)
{
    // Lees-Edwards: the halo-plane kernels compute the step's offset state from
    // the stored one and the step's last kernel stores it (no launch of
    // k_le_neighbours); the edge columns are valid (ensure_edges before the
    // steps are enqueued).
    if (c->le) c->L->le_faces(c->b, false, false, c->stream, -1);
    if (!c->plan.fused) c->L->moments(c->b, c->stream);
    if (c->le) {
        c->L->le_faces(c->b, true, c->plan.fused, c->stream, -1);
        c->L->set_le_commit(-1);
    }
    int rc = launch_collision(c);
    c->L->set_le_commit(LE_STATE_AS_IS);
    if (rc) return rc;
    flip(c);
    return LB3D_OK;
}

static int ensure_graph(lb3d_ctx *c)
{
    if (c->graph) return LB3D_OK;
    // an even number of steps starting from cur = 0 (A -> B -> ... -> A)
    const int kernels = c->plan.fused ? (c->le ? 3 : 1) : (c->le ? 4 : (c->L->small() ? 2 : c->p.ncomp));
    const int len = graph_steps(kernels);
    int saved = c->b.cur;
    set_cur(c, 0);
    hipGraph_t g = nullptr;
    HIP_TRY(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
    int rc = LB3D_OK;
    for (int q = 0; q < len && rc == LB3D_OK; q++) rc = enqueue_step(c);
    hipError_t e = hipStreamEndCapture(c->stream, &g);
    set_cur(c, saved);
    if (rc) {
        if (g) (void)hipGraphDestroy(g);
        return rc;
    }
    if (e != hipSuccess) return fail(LB3D_EHIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
    e = hipGraphInstantiate(&c->graph, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (e != hipSuccess) {
        c->graph = nullptr;
        return fail(LB3D_EHIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
    }
    c->graph_len = len;
    return LB3D_OK;
}

static bool replays(const lb3d_ctx *c, int32_t nsteps)
{
    return c->graph || replay_graph(c->plan_steps, nsteps, (uint64_t)c->p.nx * c->p.ny * c->p.nz);
}

static int sync_le_counter(lb3d_ctx *c)
{
    if (!c->le) return LB3D_OK;
    // the device step counter follows the host's nt
    int rc = pull_le(c);
    if (rc) return rc;
    if (c->host_le.nt != c->nt) {
        c->host_le.nt = c->nt;
        if ((rc = push_le(c))) return rc;
    }
    return LB3D_OK;
}

int lb3d_gpu_run_steps(lb3d_ctx *c, int32_t nsteps)
{
    g_err.clear();
    if (!c) return fail(LB3D_EINVAL, "NULL context");
    if (nsteps < 0) return fail(LB3D_EINVAL, "nsteps must be >= 0");
    if (c->state != IDLE) return fail(LB3D_ESTATE, "run_steps needs a completed timestep");
    if (nsteps == 0) return LB3D_OK;
    int rc = sync_le_counter(c);
    if (rc) return rc;
    ensure_edges(c);
    int left = nsteps;
    if (replays(c, nsteps)) {
        if ((rc = ensure_graph(c))) return rc;
        if (c->b.cur == 1) {
            if ((rc = enqueue_step(c))) return rc;
            left--;
        }
        for (; left >= c->graph_len; left -= c->graph_len) HIP_TRY(hipGraphLaunch(c->graph, c->stream));
    }
    for (; left > 0; left--)
        if ((rc = enqueue_step(c))) return rc;
    c->plan_steps += nsteps;
    HIP_TRY(hipGetLastError());
    c->edges_ok = true;
    c->nt += nsteps;
    mark_stepped(c);
    return LB3D_OK;
}

int lb3d_gpu_run_steps_timed(lb3d_ctx *c, int32_t nsteps, double *ms)
{
    g_err.clear();
    if (!c || !ms) return fail(LB3D_EINVAL, "NULL argument");
    if (c->state != IDLE) return fail(LB3D_ESTATE, "run_steps needs a completed timestep");
    int rc = sync_le_counter(c);
    if (rc) return rc;
    if (replays(c, nsteps) && (rc = ensure_graph(c))) return rc;
    Events ev(2);
    HIP_TRY(ev.create());
    hipEvent_t e0 = ev[0], e1 = ev[1];
    HIP_TRY(hipEventRecord(e0, c->stream));
    rc = lb3d_gpu_run_steps(c, nsteps);
    if (rc == LB3D_OK) {
        HIP_TRY(hipEventRecord(e1, c->stream));
        HIP_TRY(hipEventSynchronize(e1));
        float t = 0.f;
        HIP_TRY(hipEventElapsedTime(&t, e0, e1));
        *ms = t;
    }
    return rc;
}

// A copy of a context's state (populations, dipoles, Lees-Edwards offset) for
// the length of a scope in which the lattice is stepped; put back at its end.
class SavedState {
  public:
    explicit SavedState(lb3d_ctx *c) : c_(c), cur_(c->b.cur) {}
    SavedState(const SavedState &) = delete;
    SavedState &operator=(const SavedState &) = delete;
    ~SavedState()
    {
        if (!mem_) return;
        (void)restore();
        (void)hipStreamSynchronize(c_->stream);
        (void)hipFree(mem_);
    }
    // no memory for it: hipErrorOutOfMemory, and nothing is done
    hipError_t save()
    {
        hipError_t e = hipMalloc(&mem_, c_->f_bytes + c_->db_bytes);
        if (e != hipSuccess) {
            mem_ = nullptr;
            (void)hipGetLastError();
            return hipErrorOutOfMemory;
        }
        e = copy(mem_, c_->b.f[cur_], c_->f_bytes);
        if (e == hipSuccess && c_->db_bytes) e = copy((char *)mem_ + c_->f_bytes, c_->dbk[cur_], c_->db_bytes);
        if (e == hipSuccess && c_->le) {
            if ((e = hipMemcpyAsync(&le_, c_->b.le, sizeof le_, hipMemcpyDeviceToHost, c_->stream)) == hipSuccess)
                e = hipStreamSynchronize(c_->stream);
        }
        if (e != hipSuccess) {
            (void)hipStreamSynchronize(c_->stream);
            (void)hipFree(mem_);
            mem_ = nullptr;
        }
        return e;
    }
    hipError_t restore()
    {
        set_cur(c_, cur_);
        c_->edges_ok = false;
        hipError_t e = copy(c_->b.f[cur_], mem_, c_->f_bytes);
        if (e == hipSuccess && c_->db_bytes) e = copy(c_->dbk[cur_], (char *)mem_ + c_->f_bytes, c_->db_bytes);
        if (e == hipSuccess && c_->le) {
            if ((e = hipMemcpyAsync(c_->b.le, &le_, sizeof le_, hipMemcpyHostToDevice, c_->stream)) == hipSuccess)
                e = hipStreamSynchronize(c_->stream);
        }
        return e;
    }

  private:
    hipError_t copy(void *d, const void *s, size_t n)
    {
        return hipMemcpyAsync(d, s, n, hipMemcpyDeviceToDevice, c_->stream);
    }
    lb3d_ctx *c_;
    int cur_;
    void *mem_ = nullptr;
    LEState le_{};
};

// Autotuner: times each candidate plan on the context's own lattice.  Trial
// steps read f[cur] and write f[1-cur] without swapping, so the state is
// unchanged (the LE scalars are not advanced).  They reread one state, which
// flatters the two-pass plan where the populations are about as large as the
// memory-side cache (Lees-Edwards FP32 256x64x64: trials of 102 us, steps of
// 109).  So the best plans of either kind and the untuned one are then timed
// over real steps, on a copy of the state, and the untuned plan stays unless
// another is faster there.
int lb3d_gpu_autotune(lb3d_ctx *c, int32_t trial_steps, char *report, int32_t report_len)
{
    g_err.clear();
    if (!c) return fail(LB3D_EINVAL, "NULL context");
    if (c->state != IDLE) return fail(LB3D_ESTATE, "autotune needs a completed timestep");
    if (trial_steps < 1) trial_steps = 1;
    std::vector<Plan> cands;
    cands.push_back(two_pass_plan(c->p));
    // the untuned plan's tile, which is fitted to the lattice
    const Plan fit = c->L->walls ? two_pass_plan(c->p) : default_plan(c->p);
    if (fit.fused)
        for (int lz : {fit.lz, (fit.lz + 1) / 2}) {
            Plan q = fit;
            q.lz = lz;
            if (c->L->fused_supported(q.tx, q.ty, q.stage) && (cands.size() < 2 || lz != fit.lz)) cands.push_back(q);
        }
    auto name = [&](const Plan &q) {
        return !q.fused ? "two-pass" : (listed_shape(c->p.ncomp, q.tx, q.ty) ? "fused" : "fitted");
    };
    if (c->p.ncomp == 3) {
        const int lzs[] = {8, 16, 32, 64};
        for (int k = 0; k < N_FUSED_SHAPES; k++)
            for (int lz : lzs) {
                if (!c->L->fused_supported(FUSED_SHAPES[k][0], FUSED_SHAPES[k][1], 2)) continue;
                if (lz > c->p.nz && lz != 8) continue;
                Plan q;
                q.fused = true;
                q.tx = FUSED_SHAPES[k][0];
                q.ty = FUSED_SHAPES[k][1];
                q.lz = lz < c->p.nz ? lz : c->p.nz;
                q.stage = 2;
                q.xg = 0;
                cands.push_back(q);
            }
    }
    if (c->p.ncomp == 2) {
        const int lzs[] = {16, 32, 64, 128, 256};
        for (int k = 0; k < N_FUSED_SHAPES; k++)
            for (int st = 0; st < 3; st++)
                for (int lz : lzs) {
                    if (!listed_shape(2, FUSED_SHAPES[k][0], FUSED_SHAPES[k][1])) continue;
                    if (!c->L->fused_supported(FUSED_SHAPES[k][0], FUSED_SHAPES[k][1], st)) continue;
                    if (lz > c->p.nz && lz != 16) continue;
                    Plan q;
                    q.fused = true;
                    q.tx = FUSED_SHAPES[k][0];
                    q.ty = FUSED_SHAPES[k][1];
                    q.lz = lz < c->p.nz ? lz : c->p.nz;
                    q.stage = st;
                    q.xg = 0;
                    cands.push_back(q);
                }
    }
    // the trials write f[1-cur] and the ternary dipole field db_alt, never
    // the state (f[cur], db); the guard puts back the plan if a trial fails
    struct Guard {
        lb3d_ctx *c;
        Plan saved;
        bool restore = true;
        ~Guard()
        {
            if (restore) {
                c->plan = saved;
                c->L->xg = saved.xg;
            }
        }
    } g{c, c->plan};
    // f[1-cur] and db_alt no longer hold the last step's input, so the
    // moments of the last advection cannot be rebuilt from them afterwards;
    // the edge columns are gathered for the trials and are stale after them
    c->moments = MOMENTS_NONE;
    if (c->le) {
        c->L->le_gather_edges(c->b, c->stream);
        c->edges_ok = false;
    }
    Events ev(2);
    HIP_TRY(ev.create());
    hipEvent_t e0 = ev[0], e1 = ev[1];
    double best = 1e300;
    Plan bestp = g.saved;
    std::string rep;
    auto line = [&](const char *before, const Plan &q, double ms) {
        char buf[112];
        std::snprintf(buf, sizeof buf, "%s%s %dx%d lz=%d %s xg=%u %.4f ms\n", before, name(q), q.fused ? q.tx : 0,
                      q.fused ? q.ty : 0, q.fused ? q.lz : 0, q.fused ? STAGE_NAMES[q.stage] : "-", q.xg, ms);
        rep += buf;
    };
    double best_of[2] = {1e300, 1e300};  // two-pass, one-pass
    Plan plan_of[2];
    auto time_plan = [&](const Plan &q, double &per) -> int {
        c->plan = q;
        c->L->xg = q.xg;
        auto trial = [&]() {
            // (the edge columns are those of the state, gathered before the
            // trials; a trial's collision overwrites them with values of the
            // trial, which are not the state's)
            if (c->le) c->L->le_faces(c->b, false, false, c->stream);
            if (!q.fused) c->L->moments(c->b, c->stream);
            if (c->le) c->L->le_faces(c->b, true, q.fused, c->stream);
            return launch_collision(c);
        };
        if (int rc = trial()) return rc;  // warm-up
        HIP_TRY(hipEventRecord(e0, c->stream));
        for (int t = 0; t < trial_steps; t++)
            if (int rc = trial()) return rc;
        HIP_TRY(hipEventRecord(e1, c->stream));
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipEventSynchronize(e1));
        float ms = 0.f;
        HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
        per = ms / trial_steps;
        line("", q, per);
        if (per < best_of[q.fused]) {
            best_of[q.fused] = per;
            plan_of[q.fused] = q;
        }
        if (per < best) {
            best = per;
            bestp = q;
        }
        return LB3D_OK;
    };
    double per = 0.0;
    for (const Plan &q : cands)
        if (int rc = time_plan(q, per)) return rc;
    // then the XCD chunking of the best plan
    const Plan top = bestp;
    for (uint32_t xg : {1u, 2u, 4u, 8u, 16u, 32u, 64u, 0u}) {
        if (xg == top.xg) continue;
        Plan q = top;
        q.xg = xg;
        if (int rc = time_plan(q, per)) return rc;
    }
    // the finalists, the untuned plan first
    const Plan untuned = fit.fused && !c->L->fused_supported(fit.tx, fit.ty, fit.stage) ? two_pass_plan(c->p) : fit;
    std::vector<Plan> finals{untuned};
    for (int k = 0; k < 2; k++)
        if (best_of[k] < 1e300 && !same_plan(plan_of[k], untuned)) finals.push_back(plan_of[k]);
    SavedState state(c);
    hipError_t e = finals.size() > 1 ? state.save() : hipErrorOutOfMemory;
    if (e != hipSuccess && e != hipErrorOutOfMemory)
        return fail(LB3D_EHIP, std::string("autotune: ") + hipGetErrorString(e));
    if (e == hipSuccess) {
        // 2 ms of them, between 10 and 400
        const int steps = (int)std::min(400.0, std::max(10.0, 2.0 / std::max(best, 1e-3)));
        std::vector<double> took(finals.size(), 1e300);
        for (int round = 0; round < 2; round++)
            for (size_t k = 0; k < finals.size(); k++) {
                c->plan = finals[k];
                c->L->xg = finals[k].xg;
                HIP_TRY(state.restore());
                ensure_edges(c);
                for (int t = 0; t < 2 + steps; t++) {
                    if (t == 2) HIP_TRY(hipEventRecord(e0, c->stream));
                    if (int rc = enqueue_step(c)) return rc;
                }
                HIP_TRY(hipEventRecord(e1, c->stream));
                HIP_TRY(hipGetLastError());
                HIP_TRY(hipEventSynchronize(e1));
                float t = 0.f;
                HIP_TRY(hipEventElapsedTime(&t, e0, e1));
                if (t / steps < took[k]) took[k] = t / steps;
            }
        size_t pick = 0;
        for (size_t k = 0; k < finals.size(); k++) {
            line("steps: ", finals[k], took[k]);
            if (k && took[k] < 0.99 * took[0] && (!pick || took[k] < took[pick])) pick = k;
        }
        bestp = finals[pick];
        best = took[pick];
    }
    g.restore = false;
    c->plan = bestp;
    c->displaced = Plan();
    c->L->xg = bestp.xg;
    c->tuned = true;
    drop_graph(c);
    line("chosen: ", bestp, best);
    if (report && report_len > 0) {
        std::strncpy(report, rep.c_str(), (size_t)report_len - 1);
        report[report_len - 1] = 0;
    }
    return LB3D_OK;
}

int lb3d_gpu_set_plan(lb3d_ctx *c, int32_t fused, int32_t tx, int32_t ty, int32_t lz, int32_t xcd_group)
{
    g_err.clear();
    if (!c) return fail(LB3D_EINVAL, "NULL context");
    if (xcd_group < 0) return fail(LB3D_EINVAL, "xcd_group must be >= 0");
    Plan q;
    q.xg = (uint32_t)xcd_group;
    q.fused = fused != 0;
    // fused = 1: LDS stage, 2: registers, 3: pulled again by the collide
    if (fused < 0 || fused > 3) return fail(LB3D_EINVAL, "fused must be 0..3");
    q.stage = fused == 1 ? 1 : (fused == 2 ? 0 : 2);
    if (q.fused) {
        if (c->p.ncomp == 2 && c->p.bdist != 2)
            return fail(LB3D_EINVAL, "the binary one-pass kernel needs bdist 2");
        if (c->p.ncomp == 3 && (fused != 3 || c->le))
            return fail(LB3D_EINVAL, "the ternary one-pass kernel is fused = 3 on periodic lattices");
        bool ok = listed_shape(c->p.ncomp, tx, ty) && c->L->fused_supported(tx, ty, q.stage);
        if (!ok || lz < 1) return fail(LB3D_EINVAL, "no such tile shape");
        q.tx = tx;
        q.ty = ty;
        q.lz = lz < c->p.nz ? lz : c->p.nz;
    }
    // A step under way goes on with the new plan.  The one-pass plans stream
    // in their collision; the two-pass collision, and the Lees-Edwards planes
    // before it, read what the moments pass of the advection has written.
    if (c->plan.fused && !q.fused && (c->state == AFTER_ADV || c->state == AFTER_BC8)) {
        c->L->moments(c->b, c->stream);
        HIP_TRY(hipGetLastError());
        if (c->moments != MOMENTS_NONE) c->moments = MOMENTS_KEPT;
    }
    c->plan = q;
    c->displaced = Plan();
    c->L->xg = q.xg;
    c->edges_ok = false;
    drop_graph(c);
    return LB3D_OK;
}

int lb3d_gpu_synchronize(lb3d_ctx *c)
{
    g_err.clear();
    if (!c) return fail(LB3D_EINVAL, "NULL context");
    HIP_TRY(hipStreamSynchronize(c->stream));
    return LB3D_OK;
}

int lb3d_gpu_get_density(lb3d_ctx *c, double *out)
{
    g_err.clear();
    if (!c || !out) return fail(LB3D_EINVAL, "NULL argument");
    const OnDevice on(c->device);
    const uint32_t ns = (uint32_t)c->p.nx * (uint32_t)c->p.ny * (uint32_t)c->p.nz;
    const PopBase pb = pop_base(c->p);
    const void *f = c->b.f[c->b.cur];
    HIP_TRY(fetch_f64(c->stream, out, (uint64_t)c->p.ncomp * ns, [&](uint32_t q, uint32_t m, double *o) {
        if (is_dev(c))
            k_get_density<float><<<(m + 255) / 256, 256, 0, c->stream>>>((const float *)f, pb, ns, q, m, o);
        else
            k_get_density<double><<<(m + 255) / 256, 256, 0, c->stream>>>((const double *)f, pb, ns, q, m, o);
    }));
    return LB3D_OK;
}

int lb3d_gpu_get_momentum(lb3d_ctx *c, double *out)
{
    g_err.clear();
    if (!c || !out) return fail(LB3D_EINVAL, "NULL argument");
    const OnDevice on(c->device);
    const uint32_t ns = (uint32_t)c->p.nx * (uint32_t)c->p.ny * (uint32_t)c->p.nz;
    const PopBase pb = pop_base(c->p);
    const void *f = c->b.f[c->b.cur];
    HIP_TRY(fetch_f64(c->stream, out, (uint64_t)c->p.ncomp * 3u * ns, [&](uint32_t q, uint32_t m, double *o) {
        if (is_dev(c))
            k_get_momentum<float><<<(m + 255) / 256, 256, 0, c->stream>>>((const float *)f, pb, ns, q, m, o);
        else
            k_get_momentum<double><<<(m + 255) / 256, 256, 0, c->stream>>>((const double *)f, pb, ns, q, m, o);
    }));
    return LB3D_OK;
}

// The reference's arr observable (dump_arrows, code/lb3d_io_dump_data.F90:
// 1308-1460): per site the momentum of every component less half its
// Shan-Chen force times its density, weighted by amass, over the
// amass-weighted density (max with 10.e-9 in single precision, as the
// reference's real() and single literal give), less half the body-force
// acceleration inside its box.  The forces come from the device (the
// collide's own force code, from the moments of the last advection and the
// dipole field); the sums are FP64 in the reference's order.
int lb3d_gpu_get_arrows(lb3d_ctx *c, double *out)
{
    g_err.clear();
    if (!c || !out) return fail(LB3D_EINVAL, "NULL argument");
    if (c->state != IDLE) return fail(LB3D_ESTATE, "get_arrows needs a completed timestep");
    int rc = rebuild_aux(c);
    if (rc) return rc;
    if (c->moments != MOMENTS_KEPT)
        return fail(LB3D_ESTATE, "get_arrows needs the moments of an advection: run a timestep first");
    const int C = c->p.ncomp, nx = c->p.nx, ny = c->p.ny, nz = c->p.nz;
    const size_t ns = (size_t)nx * ny * nz, rs = c->L->real_bytes();
    std::vector<double> pops((size_t)C * 19 * ns), F((size_t)C * 3 * ns);
    if ((rc = lb3d_gpu_get_populations(c, pops.data()))) return rc;
    {
        // a temporary device buffer of the force field (not a hot path)
        void *d = nullptr;
        HIP_TRY(hipMalloc(&d, F.size() * rs));
        c->L->forces(c->b, d, c->stream);
        std::vector<unsigned char> h(F.size() * rs);
        hipError_t e = hipGetLastError();
        if (e == hipSuccess) e = hipMemcpyAsync(h.data(), d, h.size(), hipMemcpyDeviceToHost, c->stream);
        if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
        (void)hipFree(d);
        if (e != hipSuccess) return fail(LB3D_EHIP, std::string("forces: ") + hipGetErrorString(e));
        for (size_t q = 0; q < F.size(); q++)
            F[q] = rs == 8 ? ((const double *)h.data())[q] : (double)((const float *)h.data())[q];
    }
    std::vector<uint8_t> rock;
    if (c->b.rock) {
        rock.resize(ns);
        HIP_TRY(hipMemcpyAsync(rock.data(), c->b.rock, ns, hipMemcpyDeviceToHost, c->stream));
        HIP_TRY(hipStreamSynchronize(c->stream));
    }
    const lb3d_params &p = c->p;
    const bool body = p.g_accn[0] != 0.0 || p.g_accn[1] != 0.0 || p.g_accn[2] != 0.0;
    const int ext[3] = {nx, ny, nz};
    int bmax[3];
    for (int k = 0; k < 3; k++) bmax[k] = p.g_accn_max[k] == 0 ? ext[k] : p.g_accn_max[k];
    const int *cv[3] = {host::CX, host::CY, host::CZ};
    for (int z = 0; z < nz; z++)
        for (int y = 0; y < ny; y++)
            for (int x = 0; x < nx; x++) {
                const size_t s = (size_t)x + (size_t)nx * ((size_t)y + (size_t)ny * z);
                const bool fluid = rock.empty() || !rock[s];
                double rho[3] = {0, 0, 0}, mom[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
                for (int k = 0; k < C; k++)
                    for (int i = 0; i < 19; i++) {
                        const double v = pops[((size_t)k * 19 + i) * ns + s] * (double)host::GD[i];
                        rho[k] = rho[k] + v;
                        for (int a = 0; a < 3; a++) mom[k][a] = mom[k][a] + v * (double)cv[a][i];
                    }
                double den = rho[0] * p.amass[0];
                for (int k = 1; k < C; k++) den = den + rho[k] * p.amass[k];
                const float denf = (float)den;
                const double dd = (double)(denf > 10.e-9f ? denf : 10.e-9f);
                const bool inbox = body && fluid && z + 1 >= p.g_accn_min[2] && z + 1 <= bmax[2] &&
                                   x + 1 >= p.g_accn_min[0] && x + 1 <= bmax[0] && y + 1 >= p.g_accn_min[1] &&
                                   y + 1 <= bmax[1];
                for (int a = 0; a < 3; a++) {
                    double v = 0.0;
                    for (int k = 0; k < C; k++) {
                        const double fa = fluid ? F[((size_t)k * 3 + a) * ns + s] : 0.0;
                        const double A = mom[k][a] * p.amass[k];
                        const double B = ((fa / 2.0) * rho[k]) * p.amass[k];
                        v = k == 0 ? A - B : (v + A) - B;
                    }
                    v = v / dd;
                    if (inbox) v = v - p.g_accn[a] / 2.0;
                    out[3 * s + a] = v;
                }
            }
    return LB3D_OK;
}

int lb3d_gpu_le_halo(lb3d_ctx *c, double *out)
{
    g_err.clear();
    if (!c || !out) return fail(LB3D_EINVAL, "NULL argument");
    if (!c->le) return fail(LB3D_EINVAL, "not a Lees-Edwards lattice");
    if (c->state != IDLE) return fail(LB3D_ESTATE, "le_halo needs a completed timestep");
    int rc = sync_le_counter(c);
    if (rc) return rc;
    // the stage-6 x-halo planes of the current populations and offset
    ensure_edges(c);
    c->L->le_faces(c->b, false, false, c->stream);
    HIP_TRY(hipGetLastError());
    const size_t plane = (size_t)c->p.ny * c->p.nz;
    const size_t n = 2 * 2 * 19 * plane;
    const size_t rs = c->L->real_bytes();
    if (is_dev(c)) {
        std::vector<float> h(n);
        HIP_TRY(hipMemcpyAsync(h.data(), c->b.face_pc, n * rs, hipMemcpyDeviceToHost, c->stream));
        HIP_TRY(hipStreamSynchronize(c->stream));
        for (size_t f = 0; f < 2; f++)
            for (int k = 0; k < 2; k++)
                for (int i = 0; i < 19; i++) {
                    size_t o = ((f * 2 + k) * 19 + i) * plane;
                    double base = w_of(i) * rho0_of(c, k);
                    for (size_t t = 0; t < plane; t++) out[o + t] = base + (double)h[o + t];
                }
    } else {
        HIP_TRY(hipMemcpyAsync(out, c->b.face_pc, n * rs, hipMemcpyDeviceToHost, c->stream));
        HIP_TRY(hipStreamSynchronize(c->stream));
    }
    return LB3D_OK;
}

int lb3d_gpu_get_nt(lb3d_ctx *c, int32_t *nt)
{
    if (!c || !nt) return fail(LB3D_EINVAL, "NULL argument");
    *nt = c->nt;
    return LB3D_OK;
}

int lb3d_gpu_diagnostics(lb3d_ctx *c, double mass[3], double momentum[3], int64_t counts[3])
{
    g_err.clear();
    if (!c || !mass || !momentum || !counts) return fail(LB3D_EINVAL, "NULL argument");
    unsigned nb = c->L->diag_blocks();
    c->L->diagnostics(c->b, c->d_partials, c->stream);
    HIP_TRY(hipGetLastError());
    std::vector<double> h((size_t)nb * NDIAG);
    HIP_TRY(hipMemcpyAsync(h.data(), c->d_partials, h.size() * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    double acc[NDIAG] = {0};
    for (unsigned b = 0; b < nb; b++)
        for (int k = 0; k < NDIAG; k++) acc[k] = acc[k] + h[(size_t)b * NDIAG + k];
    for (int k = 0; k < 3; k++) {
        mass[k] = k < c->p.ncomp ? acc[k] : 0.0;
        momentum[k] = acc[3 + k];
        counts[k] = (int64_t)llround(acc[6 + k]);
    }
    return LB3D_OK;
}


int lb3d_gpu_sanity(lb3d_ctx *c, lb3d_sanity *out)
{
    g_err.clear();
    if (!c || !out) return fail(LB3D_EINVAL, "NULL argument");
    unsigned nb = c->L->diag_blocks();
    c->L->sanity(c->b, c->d_partials, c->stream);
    HIP_TRY(hipGetLastError());
    std::vector<double> h((size_t)nb * NSAN);
    HIP_TRY(hipMemcpyAsync(h.data(), c->d_partials, h.size() * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    reduce_sanity(h.data(), nb, c->p.ncomp, c->p.nx, c->p.ny, c->p.nz, out);
    return LB3D_OK;
}

int lb3d_gpu_le_state(lb3d_ctx *c, double *shear_sum, int32_t *lelo, double *lefrac, double *shear_u)
{
    g_err.clear();
    if (!c || !shear_sum || !lelo || !lefrac || !shear_u) return fail(LB3D_EINVAL, "NULL argument");
    if (c->le) {
        int rc = pull_le(c);
        if (rc) return rc;
    }
    *shear_sum = c->host_le.shear_sum;
    *lelo = c->host_le.lelo;
    *lefrac = c->host_le.lefrac;
    *shear_u = c->host_le.shear_u;
    return LB3D_OK;
}

}  // extern "C"

// ---------------------------------------------------------------------------
// lb3d_gpu_step_noalloc: one timestep over caller-owned device buffers that
// allocates nothing.  The moments field of the two-pass step (the scratch
// of lb3d_gpu_run_steps' kernels) lives in a file-scope device array of
// LB3D_NOALLOC_SCRATCH_BYTES, which every GPU the library runs on holds
// until the process ends.  In host code `scratch` names a host-side stand-in;
// its device address is looked up once per device and used instead.
static __device__ __align__(256) unsigned char scratch[LB3D_NOALLOC_SCRATCH_BYTES];

namespace {
constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
void *g_scratch[MAX_DEVICES] = {};

// The device address of `scratch` on the current device.
int scratch_on_device(void **out)
{
    int dev = -1;
    HIP_TRY(hipGetDevice(&dev));
    if (dev < 0 || dev >= MAX_DEVICES) return fail(LB3D_EINVAL, "device index beyond 64");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[dev]) {
        void *ptr = nullptr;
        hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr)
            return fail(LB3D_EHIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        g_scratch[dev] = ptr;
    }
    *out = g_scratch[dev];
    return LB3D_OK;
}
}  // namespace

extern "C" int lb3d_gpu_step_noalloc(const lb3d_params *p, const void *f_in, void *f_out, const void *db_in,
                                     void *db_out, void *stream)
{
    g_err.clear();
    int rc = check_params(p);
    if (rc) return rc;
    if (!f_in || !f_out || f_in == f_out) return fail(LB3D_EINVAL, "f_in and f_out must be distinct device buffers");
    if (p->boundary != LB3D_BC_PERIODIC)
        return fail(LB3D_EINVAL, "lb3d_gpu_step_noalloc runs periodic lattices (Lees-Edwards needs face planes)");
    if (p->ncomp == 3 && (!db_in || !db_out || db_in == db_out))
        return fail(LB3D_EINVAL, "ternary lattices need distinct db_in and db_out device buffers");
    const uint64_t ns = (uint64_t)p->nx * p->ny * p->nz;
    const size_t rs = p->precision == LB3D_FP64 ? 8 : 4;
    const uint64_t need = aux_elems(p->ncomp, ns) * rs;
    if (need > LB3D_NOALLOC_SCRATCH_BYTES) {
        char m[200];
        std::snprintf(m, sizeof m,
                      "lattice needs %llu bytes of scratch, lb3d_gpu_step_noalloc has %llu: use lb3d_gpu_create "
                      "and lb3d_gpu_run_steps",
                      (unsigned long long)need, (unsigned long long)LB3D_NOALLOC_SCRATCH_BYTES);
        return fail(LB3D_EINVAL, m);
    }
    void *aux = nullptr;
    if ((rc = scratch_on_device(&aux))) return rc;
    DevBufs b;
    b.f[0] = const_cast<void *>(f_in);
    b.f[1] = f_out;
    b.cur = 0;
    b.aux = aux;  // written in full by the moments pass before anything reads it
    b.db = const_cast<void *>(db_in);
    b.db_alt = db_out;
    hipStream_t s = (hipStream_t)stream;
    if (p->precision == LB3D_FP64)
        step_buffers_fp64(*p, b, s);
    else
        step_buffers_fp32(*p, b, s);
    HIP_TRY(hipGetLastError());
    return LB3D_OK;
}

extern "C" {

int lb3d_gpu_profile_steps(lb3d_ctx *c, int32_t nsteps, int32_t max_kernels, const char **names, double *ms,
                           int32_t *nkernels, double *ms_per_step)
{
    g_err.clear();
    if (!c || !names || !ms || !nkernels || !ms_per_step) return fail(LB3D_EINVAL, "NULL argument");
    if (nsteps < 1 || max_kernels < K_COUNT) return fail(LB3D_EINVAL, "nsteps >= 1 and room for 6 kernels needed");
    if (c->state != IDLE) return fail(LB3D_ESTATE, "profile_steps needs a completed timestep");
    int rc0 = sync_le_counter(c);
    if (rc0) return rc0;
    Events ev((size_t)nsteps * K_COUNT * 2 + 2);
    std::vector<int> used((size_t)nsteps * K_COUNT, 0);
    HIP_TRY(ev.create());
    hipEvent_t t0 = ev[ev.e.size() - 2], t1 = ev[ev.e.size() - 1];
    auto rec = [&](int step, int k, bool start) {
        return hipEventRecord(ev[((size_t)step * K_COUNT + k) * 2 + (start ? 0 : 1)], c->stream);
    };
    HIP_TRY(hipEventRecord(t0, c->stream));
    for (int st = 0; st < nsteps; st++) {
        auto mark = [&](int k) { used[(size_t)st * K_COUNT + k] = 1; };
        if (c->le) {  // as enqueue_step
            HIP_TRY(rec(st, K_LE6, true));
            ensure_edges(c);
            c->L->le_faces(c->b, false, false, c->stream, -1);
            HIP_TRY(rec(st, K_LE6, false));
            mark(K_LE6);
        }
        if (!c->plan.fused) {
            HIP_TRY(rec(st, K_MOM, true));
            c->L->moments(c->b, c->stream);
            HIP_TRY(rec(st, K_MOM, false));
            mark(K_MOM);
        }
        if (c->le) {
            HIP_TRY(rec(st, K_LE8, true));
            c->L->le_faces(c->b, true, c->plan.fused, c->stream, -1);
            HIP_TRY(rec(st, K_LE8, false));
            mark(K_LE8);
        }
        if (c->le) c->L->set_le_commit(-1);
        if (c->plan.fused) {
            HIP_TRY(rec(st, K_FUS, true));
            if (!c->L->fused(c->b, c->plan.tx, c->plan.ty, c->plan.lz, c->plan.stage, c->stream))
                return fail(LB3D_EINVAL, "the one-pass plan has no kernel for this lattice");
            HIP_TRY(rec(st, K_FUS, false));
            mark(K_FUS);
        } else if (c->L->small()) {
            HIP_TRY(rec(st, K_DC, true));
            c->L->dipole_collide(c->b, c->stream);
            HIP_TRY(rec(st, K_DC, false));
            mark(K_DC);
        } else {
            if (c->p.ncomp == 3) {
                HIP_TRY(rec(st, K_DIP, true));
                c->L->dipole(c->b, c->stream);
                HIP_TRY(rec(st, K_DIP, false));
                mark(K_DIP);
            }
            HIP_TRY(rec(st, K_COL, true));
            c->L->collide(c->b, c->stream);
            HIP_TRY(rec(st, K_COL, false));
            mark(K_COL);
        }
        c->L->set_le_commit(LE_STATE_AS_IS);
        flip(c);
        c->edges_ok = true;
    }
    HIP_TRY(hipEventRecord(t1, c->stream));
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(c->stream));
    double tot[K_COUNT] = {0};
    int cnt[K_COUNT] = {0};
    for (int st = 0; st < nsteps; st++)
        for (int k = 0; k < K_COUNT; k++)
            if (used[(size_t)st * K_COUNT + k]) {
                float m = 0.f;
                HIP_TRY(hipEventElapsedTime(&m, ev[((size_t)st * K_COUNT + k) * 2], ev[((size_t)st * K_COUNT + k) * 2 + 1]));
                tot[k] += m;
                cnt[k]++;
            }
    float all = 0.f;
    HIP_TRY(hipEventElapsedTime(&all, t0, t1));
    int nk = 0;
    for (int k = 0; k < K_COUNT; k++)
        if (cnt[k]) {
            names[nk] = KNAMES[k];
            ms[nk] = tot[k] / cnt[k];
            nk++;
        }
    *nkernels = nk;
    *ms_per_step = all / nsteps;
    c->nt += nsteps;
    mark_stepped(c);
    return LB3D_OK;
}

}  // extern "C"
