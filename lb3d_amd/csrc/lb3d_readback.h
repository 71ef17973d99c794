// lb3d_readback.h -- the state in the host's formats: observables in FP64 and
// the reference's site records (lbe_site), converted on the device.  The
// sums keep the host order of the reference (directions ascending, FP64), so
// the values are those of a conversion on the host bit for bit; include only
// from units compiled with -ffp-contract=off.
//
// What bounds them: PCIe (57 GB/s pinned) and the pages of the caller's memory.
// Before, the populations crossed PCIe plane by plane and one host thread
// converted and summed them (256^3 binary FP32 density: 345 ms); converted on
// the device and copied straight to pageable memory the result took 41 ms
// (11 GB/s to fresh pages).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>

#include "lb3d_copycrew.h"
#include "lb3d_kernels.h"
#include "lb3d_solver.h"

namespace lb3d {

// w_i * rho0 per component as the host computes it (FP32 deviations; unused in FP64)
struct PopBase {
    double move[3], rest[3];
};
inline PopBase pop_base(const lb3d_params &p)
{
    PopBase b;
    for (int c = 0; c < 3; c++) {
        b.move[c] = (1.0 / 36.0) * rho0_of(p, c);
        b.rest[c] = (1.0 / 3.0) * rho0_of(p, c);
    }
    return b;
}

// population (c, i) of a site in FP64 from its stored value
template <typename R>
__device__ __forceinline__ double pop_f64(R v, const PopBase &b, uint32_t c, uint32_t i)
{
    if constexpr (sizeof(R) == 8)
        return v;
    else
        return (i < 18u ? b.move[c] : b.rest[c]) + (double)v;
}

// Elements [q0, q0 + n) of the populations, f[(c*19 + i)*ns + s], in FP64.
template <typename R>
__global__ __launch_bounds__(256) void k_get_populations(const R *__restrict__ f, PopBase b, uint32_t ns,
                                                         uint32_t q0, uint32_t n, double *__restrict__ out)
{
    const uint32_t t = blockIdx.x * 256u + threadIdx.x;
    if (t >= n) return;
    const uint32_t ci = (q0 + t) / ns;
    out[t] = pop_f64<R>(f[q0 + t], b, ci / 19u, ci % 19u);
}

// Elements [q0, q0 + n) of the densities, rho[c*ns + s].
template <typename R>
__global__ __launch_bounds__(256) void k_get_density(const R *__restrict__ f, PopBase b, uint32_t ns, uint32_t q0,
                                                     uint32_t n, double *__restrict__ out)
{
    const uint32_t t = blockIdx.x * 256u + threadIdx.x;
    if (t >= n) return;
    const uint32_t c = (q0 + t) / ns, s = (q0 + t) - c * ns;
    double rho = 0.0;
#pragma unroll
    for (uint32_t i = 0; i < 19u; i++)
        rho = rho + pop_f64<R>(f[(c * 19u + i) * ns + s], b, c, i) * (double)GD[i];
    out[t] = rho;
}

// Elements [q0, q0 + n) of the momenta, P[(c*3 + a)*ns + s].
template <typename R>
__global__ __launch_bounds__(256) void k_get_momentum(const R *__restrict__ f, PopBase b, uint32_t ns, uint32_t q0,
                                                      uint32_t n, double *__restrict__ out)
{
    const uint32_t t = blockIdx.x * 256u + threadIdx.x;
    if (t >= n) return;
    const uint32_t ca = (q0 + t) / ns, s = (q0 + t) - ca * ns, c = ca / 3u, a = ca - 3u * c;
    double p = 0.0;
#pragma unroll
    for (uint32_t i = 0; i < 18u; i++) {
        const int cv = a == 0 ? CX[i] : (a == 1 ? CY[i] : CZ[i]);
        if (cv != 0) p = p + (pop_f64<R>(f[(c * 19u + i) * ns + s], b, c, i) * (double)GD[i]) * (double)cv;
    }
    out[t] = p;
}

// One lattice's site records: whole_N with halo h, extent lx x ly x lz, sd
// doubles per record (code/lb3d_lattice.F90:35-83).  A block of 256 threads
// holds 64 consecutive records in LDS, so that both the record side and the
// plane side are read and written in whole lines.
constexpr int REC_SITES = 64;
struct RecLayout {
    int nx, ny, nz, h, sd, C;
    uint32_t ns;
    double rock_r, rock_b;  // colours of rock sites (download)
};

// Records [r0, r0 + n) of the lattice (z slowest, halo included) to out.
// aux: the moments of the last advection, or nullptr (rho is then that of the
// populations and da zero); the halo holds the periodic images.
template <typename R>
__global__ __launch_bounds__(256) void k_get_sites(const R *__restrict__ f, const R *__restrict__ aux,
                                                   const R *__restrict__ db, const uint8_t *__restrict__ rock,
                                                   PopBase b, double r00, double r01, double r02, RecLayout L,
                                                   uint32_t r0, uint32_t n, double *__restrict__ out)
{
    extern __shared__ double rec[];  // REC_SITES records of sd doubles
    const int j = (int)(threadIdx.x % REC_SITES), g = (int)(threadIdx.x / REC_SITES);
    const uint32_t first = blockIdx.x * REC_SITES;
    const uint32_t m = n - first < (uint32_t)REC_SITES ? n - first : (uint32_t)REC_SITES;
    const uint32_t lx = (uint32_t)(L.nx + 2 * L.h), ly = (uint32_t)(L.ny + 2 * L.h);
    uint32_t s = 0;
    if ((uint32_t)j < m) {
        const uint32_t r = r0 + first + (uint32_t)j;
        const uint32_t t = r / lx, z = t / ly, y = t - z * ly, x = r - t * lx;
        // periodic image: (v - h) mod n with v - h >= -h
        const uint32_t wx = (x + (uint32_t)L.h * (uint32_t)(L.nx - 1)) % (uint32_t)L.nx;
        const uint32_t wy = (y + (uint32_t)L.h * (uint32_t)(L.ny - 1)) % (uint32_t)L.ny;
        const uint32_t wz = (z + (uint32_t)L.h * (uint32_t)(L.nz - 1)) % (uint32_t)L.nz;
        s = wx + (uint32_t)L.nx * (wy + (uint32_t)L.ny * wz);
        for (int p = g; p < 19 * L.C; p += 4)
            rec[j * L.sd + 24 * (p / 19) + p % 19] =
                pop_f64<R>(f[(uint32_t)p * L.ns + s], b, (uint32_t)p / 19u, (uint32_t)p % 19u);
    }
    __syncthreads();
    if ((uint32_t)j < m && g < L.C) {
        double *S = rec + j * L.sd + 24 * g;
        double rho = 0.0, m0 = 0.0, m1 = 0.0, m2 = 0.0;
#pragma unroll
        for (int i = 0; i < 19; i++) {
            const double ng = S[i] * (double)GD[i];
            rho = rho + ng;
            m0 = m0 + ng * (double)CX[i];
            m1 = m1 + ng * (double)CY[i];
            m2 = m2 + ng * (double)CZ[i];
        }
        if (aux) {
            const double r = (double)aux[(uint32_t)(L.C + g) * L.ns + s];
            rho = sizeof(R) == 4 ? (g == 0 ? r00 : (g == 1 ? r01 : r02)) + r : r;
        }
        S[19] = rho;
        S[20] = m0;
        S[21] = m1;
        S[22] = m2;
        S[23] = 0.0;
    } else if ((uint32_t)j < m && g == 3) {
        double *S = rec + j * L.sd;
        if (L.C == 3)
            for (int a = 0; a < 3; a++) {
                S[72 + a] = aux ? (double)aux[aux3_vec_off(L.ns) + (uint64_t)4 * s + 1 + a] : 0.0;
                S[75 + a] = (double)db[(uint32_t)a * L.ns + s];
            }
        S[L.sd - 1] = rock && rock[s] ? 1.0 : 0.0;
    }
    __syncthreads();
    if (rock && (uint32_t)j < m && g == 0 && rock[s]) {
        if (L.rock_r > 0) rec[j * L.sd + 23] = L.rock_r;
        if (L.rock_b > 0) rec[j * L.sd + 24 + 23] = L.rock_b;
    }
    __syncthreads();
    for (uint32_t q = threadIdx.x; q < m * (uint32_t)L.sd; q += 256u)
        out[(size_t)first * (uint32_t)L.sd + q] = rec[q];
}

// Records [r0, r0 + n) of the lattice (z slowest, halo included), which in
// starts with: populations, dipoles and the rock mask (mask may be nullptr) of
// those that are interior sites; *nrock counts the rock sites.
template <typename R>
__global__ __launch_bounds__(256) void k_put_sites(const double *__restrict__ in, RecLayout L, PopBase b, uint32_t r0,
                                                   uint32_t n, R *__restrict__ f, R *__restrict__ db,
                                                   uint8_t *__restrict__ mask, uint32_t *__restrict__ nrock)
{
    extern __shared__ double rec[];
    const int j = (int)(threadIdx.x % REC_SITES), g = (int)(threadIdx.x / REC_SITES);
    const uint32_t first = blockIdx.x * REC_SITES;
    const uint32_t m = n - first < (uint32_t)REC_SITES ? n - first : (uint32_t)REC_SITES;
    for (uint32_t q = threadIdx.x; q < m * (uint32_t)L.sd; q += 256u)
        rec[q] = in[(size_t)first * (uint32_t)L.sd + q];
    __syncthreads();
    if ((uint32_t)j >= m) return;
    const uint32_t r = r0 + first + (uint32_t)j, h = (uint32_t)L.h;
    const uint32_t lx = (uint32_t)L.nx + 2u * h, ly = (uint32_t)L.ny + 2u * h;
    // (a halo coordinate below 0 is a large unsigned one)
    const uint32_t t = r / lx, x = r - t * lx - h, y = t % ly - h, z = t / ly - h;
    if (x >= (uint32_t)L.nx || y >= (uint32_t)L.ny || z >= (uint32_t)L.nz) return;
    const uint32_t s = x + (uint32_t)L.nx * (y + (uint32_t)L.ny * z);
    const double *S = rec + j * L.sd;
    for (int p = g; p < 19 * L.C; p += 4) {
        const int c = p / 19, i = p % 19;
        const double v = S[24 * c + i];
        f[(uint32_t)p * L.ns + s] = sizeof(R) == 8 ? R(v) : R(v - (i < 18 ? b.move[c] : b.rest[c]));
    }
    if (g == 0 && L.C == 3)
        for (int a = 0; a < 3; a++) db[(uint32_t)a * L.ns + s] = R(S[75 + a]);
    if (g == 1) {
        const bool rk = S[L.sd - 1] != 0.0;
        if (mask) mask[s] = rk ? 1 : 0;
        if (rk) atomicAdd(nrock, 1u);
    }
}

// Transfers in pieces through two pinned buffers: while one piece crosses
// PCIe, the one before it is copied to (or from) the caller's memory.  The
// buffers grow to what is asked of them, at most IO_PIECE bytes each.  Where
// no memory can be pinned they are pageable, and where the device has no room
// for a piece the pieces are smaller: slower, but nothing that copies straight
// to the caller's pages could do is refused.
constexpr size_t IO_PIECE = 8u << 20;
struct HostIO {
    int device = -1;
    void *pin[2] = {nullptr, nullptr}, *dev[2] = {nullptr, nullptr};
    hipEvent_t ev[2] = {nullptr, nullptr};
    uint32_t *count = nullptr;  // device counter of an upload's rock sites
    size_t host_cap = 0, dev_cap = 0;
    bool pageable = false;
    static size_t round_up(size_t n) { return (n + 65535) & ~(size_t)65535; }
    hipError_t counter()
    {
        return count ? hipSuccess : hipMalloc((void **)&count, sizeof(uint32_t));
    }
    // Host buffers of n bytes.
    hipError_t host_room(size_t n)
    {
        if (n <= host_cap) return hipSuccess;
        free_host();
        n = round_up(n);
        for (void *&q : pin)
            if (!pageable && hipHostMalloc(&q, n, hipHostMallocPortable) != hipSuccess) {
                q = nullptr;
                (void)hipGetLastError();
                pageable = true;
            }
        if (pageable) {
            if (pin[0]) (void)hipHostFree(pin[0]);
            for (void *&q : pin) q = std::malloc(n);
            if (!pin[0] || !pin[1]) {
                free_host();
                return hipErrorOutOfMemory;
            }
        }
        host_cap = n;
        return hipSuccess;
    }
    // Device buffers of n bytes, or as many as can be had, at least `least`.
    hipError_t dev_room(size_t n, size_t least)
    {
        if (n <= dev_cap) return hipSuccess;
        free_dev();
        for (n = round_up(n);; n = round_up(n / 2)) {
            hipError_t e = hipMalloc(&dev[0], n);
            if (e != hipSuccess) dev[0] = nullptr;
            if (e == hipSuccess && (e = hipMalloc(&dev[1], n)) != hipSuccess) dev[1] = nullptr;
            if (e == hipSuccess) break;
            (void)hipGetLastError();
            free_dev();
            if (n <= round_up(least)) return e;
        }
        dev_cap = n;
        return hipSuccess;
    }
    // The bytes of a piece, whole units, for a transfer of total; room: the
    // pieces need device memory of their own.
    hipError_t prepare(size_t total, size_t unit, bool room, size_t *piece)
    {
        size_t n = unit < IO_PIECE ? IO_PIECE / unit * unit : unit;
        const size_t want = total < n ? total : n;
        hipError_t e = hipSuccess;
        for (int j = 0; j < 2 && e == hipSuccess; j++)
            if (!ev[j]) e = hipEventCreateWithFlags(&ev[j], hipEventDisableTiming);
        if (e == hipSuccess && room) e = dev_room(want, total < unit ? total : unit);
        if (room && dev_cap < want) n = dev_cap < unit ? unit : dev_cap / unit * unit;
        if (e == hipSuccess) e = host_room(total < n ? total : n);
        *piece = n;
        return e;
    }
    void free_host()
    {
        for (void *&q : pin) {
            if (q) pageable ? std::free(q) : (void)hipHostFree(q);
            q = nullptr;
        }
        pageable = false;
        host_cap = 0;
    }
    void free_dev()
    {
        for (void *&q : dev) {
            if (q) (void)hipFree(q);
            q = nullptr;
        }
        dev_cap = 0;
    }
    void release()
    {
        free_host();
        free_dev();
        for (hipEvent_t &x : ev) {
            if (x) (void)hipEventDestroy(x);
            x = nullptr;
        }
        if (count) (void)hipFree(count);
        count = nullptr;
    }
    // dst[0..total) bytes in pieces: go(off, n, buf) returns the device memory
    // that holds bytes [off, off + n), having launched what fills it (buf, with
    // room: memory for a piece).  Pieces are whole units.
    template <typename Go>
    hipError_t down(hipStream_t st, void *dst, size_t total, size_t unit, bool room, Go go)
    {
        size_t piece = 0;
        hipError_t e = prepare(total, unit, room, &piece);
        if (e != hipSuccess) return e;
        CopyCrew crew(total);
        const size_t n = (total + piece - 1) / piece;
        auto len = [&](size_t k) { return total - k * piece < piece ? total - k * piece : piece; };
        auto start = [&](size_t k) {
            (void)hipGetLastError();  // (an error that an earlier call left is not go's)
            const void *src = go(k * piece, len(k), dev[k & 1]);
            hipError_t r = hipGetLastError();
            if (r == hipSuccess) r = hipMemcpyAsync(pin[k & 1], src, len(k), hipMemcpyDeviceToHost, st);
            return r == hipSuccess && n > 1 ? hipEventRecord(ev[k & 1], st) : r;
        };
        for (size_t k = 0; k < 2 && k < n && e == hipSuccess; k++) e = start(k);
        for (size_t k = 0; k < n && e == hipSuccess; k++) {
            // (a single piece: the wait for the stream is 5 us shorter than an event's)
            e = n > 1 ? hipEventSynchronize(ev[k & 1]) : hipStreamSynchronize(st);
            if (e == hipSuccess) crew.copy((char *)dst + k * piece, pin[k & 1], len(k));
            if (e == hipSuccess && k + 2 < n) e = start(k + 2);
        }
        if (e != hipSuccess) (void)hipStreamSynchronize(st);
        return e;
    }
    // src[0..total) bytes in pieces to the device: go(off, n, buf) launches
    // what reads piece [off, off + n) from buf.  All work is queued on st when
    // this returns, and src has been read.
    template <typename Go>
    hipError_t up(hipStream_t st, const void *src, size_t total, size_t unit, Go go)
    {
        size_t piece = 0;
        hipError_t e = prepare(total, unit, true, &piece);
        if (e != hipSuccess) return e;
        CopyCrew crew(total);
        size_t k = 0;
        for (size_t off = 0; off < total && e == hipSuccess; off += piece, k++) {
            const size_t n = total - off < piece ? total - off : piece;
            if (k >= 2) e = hipEventSynchronize(ev[k & 1]);  // piece k - 2 has left its pinned buffer
            if (e != hipSuccess) break;
            crew.copy(pin[k & 1], (const char *)src + off, n);
            e = hipMemcpyAsync(dev[k & 1], pin[k & 1], n, hipMemcpyHostToDevice, st);
            if (e == hipSuccess) e = hipEventRecord(ev[k & 1], st);
            if (e != hipSuccess) break;
            (void)hipGetLastError();
            go(off, n, dev[k & 1]);
            e = hipGetLastError();
        }
        if (e != hipSuccess) (void)hipStreamSynchronize(st);
        return e;
    }
};

// Makes a context's device current for the length of a call.  Copies on a
// stream run whatever device is current; the events, buffers and kernels of a
// transfer have to be those of the stream's device.
class OnDevice {
  public:
    explicit OnDevice(int device)
    {
        if (hipGetDevice(&was_) == hipSuccess && was_ != device) moved_ = hipSetDevice(device) == hipSuccess;
    }
    OnDevice(const OnDevice &) = delete;
    OnDevice &operator=(const OnDevice &) = delete;
    ~OnDevice()
    {
        if (moved_) (void)hipSetDevice(was_);
    }

  private:
    int was_ = -1;
    bool moved_ = false;
};

// Transfer buffers are lent for one call and shared by all contexts (pinning
// them takes about 4 ms, more than a small lattice's whole run between two
// dumps): IoLoan takes a set of the current device from a pool, or a new one,
// and gives it back.  The pool keeps at most IO_KEPT sets, of at most 2 IO_PIECE
// bytes pinned and as many on the device each (64 MiB and 64 MiB in all), and
// frees them when the last context goes (io_users counts contexts); sets of
// pageable memory it does not keep.  Loans of several threads are different
// sets.  The borrower's work on the set is complete when the loan ends.
constexpr size_t IO_KEPT = 4;
HostIO *io_lend();
void io_give_back(HostIO *io);
void io_users(int change);
struct IoLoan {
    HostIO *io = io_lend();
    IoLoan() = default;
    IoLoan(const IoLoan &) = delete;
    IoLoan &operator=(const IoLoan &) = delete;
    ~IoLoan() { io_give_back(io); }
    HostIO *operator->() const { return io; }
    HostIO &operator*() const { return *io; }
};

// dst[0..n) in FP64: go(q0, m, out) launches the kernel that fills out with
// elements [q0, q0 + m).
template <typename Go>
hipError_t fetch_f64(hipStream_t st, double *dst, uint64_t n, Go go)
{
    IoLoan io;
    return io->down(st, dst, n * sizeof(double), 65536, true, [&](size_t off, size_t len, void *buf) -> const void * {
        go((uint32_t)(off / sizeof(double)), (uint32_t)(len / sizeof(double)), (double *)buf);
        return buf;
    });
}

// The populations of one lattice in FP64.
constexpr uint64_t SMALL_POPS = 1u << 20;
template <typename R>
hipError_t fetch_populations(hipStream_t st, const lb3d_params &p, const void *f, double *out)
{
    const uint32_t ns = (uint32_t)p.nx * (uint32_t)p.ny * (uint32_t)p.nz;
    const uint64_t n = (uint64_t)p.ncomp * 19u * ns;
    if constexpr (sizeof(R) == 8) {  // as stored
        IoLoan io;
        return io->down(st, out, n * 8, 65536, false,
                       [&](size_t off, size_t, void *) -> const void * { return (const char *)f + off; });
    } else {
        const PopBase b = pop_base(p);
        // Few values: converted by the host, straight from pinned memory to the
        // caller's; half as many bytes cross the bus and none is copied twice
        // (16^3 binary 83 -> 43 us, 20^3 139 -> 71, 28^3 354 -> 172).
        if (n <= SMALL_POPS) {
            IoLoan io;
            size_t piece = 0;
            hipError_t e = io->prepare(n * 4, 65536, false, &piece);
            if (e == hipSuccess) e = hipMemcpyAsync(io->pin[0], f, n * 4, hipMemcpyDeviceToHost, st);
            if (e == hipSuccess) e = hipStreamSynchronize(st);
            if (e != hipSuccess) {
                (void)hipStreamSynchronize(st);
                return e;
            }
            const float *v = (const float *)io->pin[0];
            for (int ci = 0; ci < 19 * p.ncomp; ci++, v += ns, out += ns) {
                const double base = ci % 19 < 18 ? b.move[ci / 19] : b.rest[ci / 19];
                for (uint32_t s = 0; s < ns; s++) out[s] = base + (double)v[s];
            }
            return hipSuccess;
        }
        return fetch_f64(st, out, n, [&](uint32_t q, uint32_t m, double *o) {
            k_get_populations<R><<<(m + 255) / 256, 256, 0, st>>>((const R *)f, b, ns, q, m, o);
        });
    }
}

}  // namespace lb3d
