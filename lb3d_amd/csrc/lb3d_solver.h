// lb3d_solver.h -- host-side interface between the C ABI (lb3d_gpu.hip) and
// the precision-specific kernel launchers (lb3d_fp64.hip, lb3d_fp32.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "../../include/lb3d_gpu.h"
#include "lb3d_lattice.h"

namespace lb3d {

// Device buffers of one lattice.  f[cur] holds the post-collision populations
// of step nt; collide writes f[1-cur].
struct DevBufs {
    void *f[2] = {nullptr, nullptr};
    // ternary: db is the dipole field of the state (read by the moments and
    // the one-pass kernel), db_alt receives the relaxed field of the step
    // (written by the dipole pass or the one-pass kernel, read by the collide);
    // a single lattice alternates the two with the population parity, the
    // batch relaxes one field in place (db_alt == db)
    void *aux = nullptr, *db = nullptr, *face_pc = nullptr, *face_aux = nullptr;
    void *db_alt = nullptr;
    // Lees-Edwards edge columns (x = nx-1 and x = 0) in a compact layout: the
    // post-collision populations (edge_pc) and the streamed ones (edge_adv)
    void *edge_pc = nullptr, *edge_adv = nullptr;
    const uint8_t *rock = nullptr;  // 1 at rock sites, or nullptr for a lattice without walls
    LEState *le = nullptr;
    int cur = 0;
};

// How a timestep is executed: the two-pass sequence (moments, [dipole],
// collide) or the one-pass z-march kernel with a tile shape (tx, ty) and a
// z-chunk lz.
struct Plan {
    bool fused = false;
    int tx = 64, ty = 4, lz = 0;
    int stage = 1;      // plane k's populations: 0 registers, 1 LDS, 2 pulled again
    uint32_t xg = 0;    // tiles per XCD chunk (xcd_tile): 1 plain order, 0 one run per XCD
};
inline bool same_plan(const Plan &a, const Plan &b)
{
    if (a.fused != b.fused || a.xg != b.xg) return false;
    return !a.fused || (a.tx == b.tx && a.ty == b.ty && a.lz == b.lz && a.stage == b.stage);
}
// The plan of a lattice that nobody has tuned, and its two-pass plan.
Plan default_plan(const lb3d_params &p);
Plan two_pass_plan(const lb3d_params &p);

// Steps of a captured graph, and when one is captured.  Measured per step
// (us), plain launches against graphs of 2, 16 and 64 steps: 16^3 binary FP64
// 10.0 against 12.3, 9.6, 9.3; 32^3 binary FP64 11.6 / 13.5, 10.8, 10.5; 32^3
// ternary FP32 15.4 / 17.0, 14.6, 14.3; 128^3 ternary 359 / 363, 359, 358: a
// graph launch costs about 4 us more than a kernel launch, a kernel inside it
// about 0.4 us less, and capturing one 0.4-0.7 ms plus 10 us per kernel.  So
// a graph holds an even number of steps of at least GRAPH_KERNELS kernels, and
// is captured once GRAPH_AFTER steps on one plan have shown a long run, or where
// one call of twice as many steps says so beforehand, if the kernels are about
// as short as a launch.  That call, plain and with the capture (us a step):
// 2,048 steps of 16^3 binary FP32 7.7 / 6.5, FP64 7.7 / 7.5, 32^3 FP64 9.46 /
// 9.49, 16^3 ternary FP64 17.1 / 16.2, 32^3 FP32 14.6 / 14.1, 32^3 Lees-Edwards
// 20.6 / 20.2; 48^3 binary FP32 10.9 / 11.3, FP64 17.9 / 18.2.
constexpr int GRAPH_KERNELS = 48;
constexpr int64_t GRAPH_AFTER = 1024;
constexpr uint64_t GRAPH_SITES = 40000;
inline bool replay_graph(int64_t steps_before, int64_t steps, uint64_t sites)
{
    return steps_before >= GRAPH_AFTER || (steps >= 2 * GRAPH_AFTER && sites <= GRAPH_SITES);
}
inline int graph_steps(int kernels_per_step)
{
    const int k = (GRAPH_KERNELS + 2 * kernels_per_step - 1) / (2 * kernels_per_step);
    return 2 * (k < 1 ? 1 : k);
}

// One precision's kernels for one parameter set.
class Launcher {
  public:
    virtual ~Launcher() {}
    // chunk of consecutive tiles per XCD in the stepping kernels (xcd_tile);
    // 0 is one run of tiles per XCD
    uint32_t xg = 0;
    bool walls = false;  // the lattice has rock sites (the one-pass plans are then unavailable)
    virtual void moments(const DevBufs &b, hipStream_t s) = 0;
    // dipole and collide in one launch, for lattices of few sites (small());
    // false: not done
    virtual bool small() const = 0;
    virtual bool dipole_collide(const DevBufs &b, hipStream_t s) = 0;
    virtual void dipole(const DevBufs &b, hipStream_t s) = 0;
    virtual void collide(const DevBufs &b, hipStream_t s) = 0;  // f[cur] -> f[1-cur]
    // Lees-Edwards x-halo planes, pre- (post = false) or post-advection, from
    // the edge columns b.edge_pc (written by the step's last kernel or
    // le_gather_edges); post-advection from the streamed ones b.edge_adv that
    // the moments pass has written, or (stream) by streaming b.edge_pc
    // adv: LE_STATE_AS_IS, or the halo-plane kernels compute the step's state
    // from the stored one (le_advance with nt_set = adv) and the next collide
    // stores it (set_le_commit)
    virtual void le_faces(const DevBufs &b, bool post, bool stream, hipStream_t s, int adv = LE_STATE_AS_IS) = 0;
    virtual void set_le_commit(int adv) = 0;
    // b.edge_pc from the populations f[cur]
    virtual void le_gather_edges(const DevBufs &b, hipStream_t s) = 0;
    // the Shan-Chen force field from b.aux and b.db into out[(c*3 + k)*ns + s]
    // (working type R), periodic in x
    virtual void forces(const DevBufs &b, void *out, hipStream_t s) = 0;
    // the whole binary step in one kernel (f[cur] -> f[1-cur]); false if the
    // tile shape has no instantiation or the form is not binary
    // stage: where plane k's populations wait for the collide: 0 registers,
    // 1 LDS (both pulled one plane ahead), 2 pulled again by the collide
    virtual bool fused(const DevBufs &b, int tx, int ty, int lz, int stage, hipStream_t s) = 0;
    virtual bool fused_supported(int tx, int ty, int stage) = 0;
    virtual void init_noise(const DevBufs &b, uint64_t seed, const double rho_mean[3],
                            const double amp[3], int dipoles, hipStream_t s) = 0;
    // per-block FP64 partial sums for the sanity reductions (NDIAG per block)
    virtual void diagnostics(const DevBufs &b, double *partials, hipStream_t s) = 0;
    // per-block partials of the full sanity check (NSAN per block)
    virtual void sanity(const DevBufs &b, double *partials, hipStream_t s) = 0;
    virtual unsigned diag_blocks() const = 0;
    virtual size_t real_bytes() const = 0;
};

// Tile shapes (TX, TY) that a plan can be set to: k_fused3 has an instance of
// each that fits, k_fused2 takes its tile at run time.
constexpr int FUSED_SHAPES[][2] = {{64, 4}, {32, 8}, {64, 8}, {32, 16}, {128, 4}, {32, 4}, {16, 16},
                                   {128, 2}, {256, 2}};
constexpr int N_FUSED_SHAPES = sizeof(FUSED_SHAPES) / sizeof(FUSED_SHAPES[0]);

constexpr int NDIAG = 9;  // mass[3], momentum[3], nan sites, negative sites, fast sites
// full sanity partials: NDIAG values, fluid sites, velocity sums [3][3], then
// per (species, axis) the largest |velocity| and its loop-order key
constexpr int SAN_FLUID = 9, SAN_VSUM = 10, SAN_MAX = 19, SAN_KEY = 28, NSAN = 37;
// fill *out from nb blocks of k_sanity partials (host)
void reduce_sanity(const double *partials, unsigned nb, int ncomp, int nx, int ny, int nz, lb3d_sanity *out);
constexpr unsigned BLOCK = 256;

// Batched ensemble kernels of one precision.  The lattice table (BatchLat<R>
// per lattice) and the work list live in device memory.
class BatchLauncher {
  public:
    virtual ~BatchLauncher() {}
    uint32_t xg = 0;  // chunk of consecutive work items per XCD (xcd_tile)
    virtual size_t lat_bytes() const = 0;   // sizeof(BatchLat<R>)
    virtual void set_bdist_mask(int mask) = 0;
    // bytes of one copy of the batch's populations (chooses the collide's store form)
    virtual void set_pop_bytes(uint64_t bytes) = 0;
    // host image of the lattice table entry k
    virtual void fill_lat(void *dst, const lb3d_params &p, uint64_t f_off, uint64_t aux_off,
                          uint64_t db_off) const = 0;
    // phase ph (0 moments, 1 dipole, 2 collide) over nitems work items;
    // packed: the ternary moments and dipole phases use the packed layout of
    // the moments field (one psi_r, psi_b, psi_s, rho_s 4-vector per site),
    // else the planes; the ternary collide phase always reads the packed one
    virtual void phase(int ph, const void *lat, const void *items, uint32_t nitems, unsigned nwg,
                       const void *f, void *fout, void *aux, void *db, int ncomp, hipStream_t s,
                       bool packed) = 0;
    // the collide-moments plan (FP32 ternary only): k_batch_cm over nitems
    // tiles (uint4 items) with work-groups of threads = 256 or 512, and k_batch_edge_moments over nitems runs of 256
    // edge sites (uint2 items into the site list)
    virtual bool cm_supported(int ncomp) const = 0;
    virtual void cm_collide(const void *lat, const void *items, uint32_t nitems, unsigned nwg, int threads,
                            const void *f, void *fout, const void *aux_in, void *aux_out, const void *db,
                            hipStream_t s) = 0;
    virtual void edge_moments(const void *lat, const void *items, uint32_t nitems, unsigned nwg, const void *sites,
                              const void *f, const void *db, void *aux, hipStream_t s) = 0;
};

Launcher *make_launcher_fp64(const lb3d_params &p);
// one timestep of the default plan over caller-provided buffers (no allocation)
void step_buffers_fp64(const lb3d_params &p, const DevBufs &b, hipStream_t s);
void step_buffers_fp32(const lb3d_params &p, const DevBufs &b, hipStream_t s);
Launcher *make_launcher_fp32(const lb3d_params &p);
BatchLauncher *make_batch_launcher_fp64();
BatchLauncher *make_batch_launcher_fp32();

// Error state of the C ABI (thread-local message, returns code).
int set_error(int code, const char *msg);
void clear_error();
// Host conversion of the reference's AoS lattice (lbe_site records) into the
// device layout of one lattice: populations (FP64, or FP32 deviations from
// w_i*rho0) and the ternary dipole field; rock sites are refused.  Returns 0 or an LB3D_E* code.
int aos_to_device_layout(const lb3d_params &p, const double *whole_N, int halo, int site_doubles,
                         std::vector<unsigned char> &f_bytes, std::vector<unsigned char> &db_bytes);
double rho0_of(const lb3d_params &p, int c);

// Parameters in the kernels' working type.
template <typename R>
Phys<R> make_phys(const lb3d_params &p);

}  // namespace lb3d
