// lb3d_readback.h -- the state in the host's formats: observables in FP64 and
// the reference's site records (lbe_site), converted on the device.  The
// sums keep the host order of the reference (directions ascending, FP64), so
// the values are those of a conversion on the host bit for bit; include only
// from units compiled with -ffp-contract=off.
//
// What bounds them: the transfer over PCIe (pageable 11-31 GB/s).  Before, the
// populations crossed it plane by plane and one host thread converted and
// summed them (256^3 binary FP32 density 345 ms, of which 25 ms is the
// transfer of the result).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>

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

// Interior sites [s0, s0 + n) from records of the z planes that in starts
// with (plane z0 of the halo'd lattice): populations, dipoles and the rock
// mask (mask may be nullptr); *nrock counts the rock sites.
template <typename R>
__global__ __launch_bounds__(256) void k_put_sites(const double *__restrict__ in, uint32_t z0, RecLayout L,
                                                   PopBase b, uint32_t s0, uint32_t n, R *__restrict__ f,
                                                   R *__restrict__ db, uint8_t *__restrict__ mask,
                                                   uint32_t *__restrict__ nrock)
{
    extern __shared__ double rec[];
    __shared__ size_t off[REC_SITES];  // first double of each record
    const int j = (int)(threadIdx.x % REC_SITES), g = (int)(threadIdx.x / REC_SITES);
    const uint32_t first = blockIdx.x * REC_SITES;
    const uint32_t m = n - first < (uint32_t)REC_SITES ? n - first : (uint32_t)REC_SITES;
    const uint32_t s = s0 + first + (uint32_t)j;
    if (g == 0 && (uint32_t)j < m) {
        const uint32_t t = s / (uint32_t)L.nx, x = s - t * (uint32_t)L.nx;
        const uint32_t z = t / (uint32_t)L.ny, y = t - z * (uint32_t)L.ny;
        const size_t lx = (size_t)(L.nx + 2 * L.h), ly = (size_t)(L.ny + 2 * L.h);
        off[j] = ((x + L.h) + lx * ((y + L.h) + ly * (size_t)(z + L.h - z0))) * (size_t)L.sd;
    }
    __syncthreads();
    for (uint32_t q = threadIdx.x; q < m * (uint32_t)L.sd; q += 256u) {
        const uint32_t r = q / (uint32_t)L.sd;
        rec[q] = in[off[r] + (q - r * (uint32_t)L.sd)];
    }
    __syncthreads();
    if ((uint32_t)j >= m) return;
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

// A device buffer that grows to what is asked of it and is kept.
struct DevScratch {
    void *p = nullptr;
    size_t bytes = 0;
    hipError_t ensure(size_t n)
    {
        if (n <= bytes) return hipSuccess;
        release();
        hipError_t e = hipMalloc(&p, n);
        if (e == hipSuccess) bytes = n;
        return e;
    }
    void release()
    {
        if (p) (void)hipFree(p);
        p = nullptr;
        bytes = 0;
    }
};

// dst[0..n) in FP64 through the scratch buffer, in pieces of at most
// FETCH_ELEMS: go(q0, m, out) launches the kernel that fills out with
// elements [q0, q0 + m).
constexpr uint64_t FETCH_ELEMS = 4u << 20;
template <typename Go>
hipError_t fetch_f64(DevScratch &sc, hipStream_t st, double *dst, uint64_t n, Go go)
{
    const uint64_t cap = n < FETCH_ELEMS ? n : FETCH_ELEMS;
    hipError_t e = sc.ensure(cap * sizeof(double));
    for (uint64_t q = 0; q < n && e == hipSuccess; q += cap) {
        const uint64_t m = n - q < cap ? n - q : cap;
        go((uint32_t)q, (uint32_t)m, (double *)sc.p);
        e = hipGetLastError();
        if (e == hipSuccess) e = hipMemcpyAsync(dst + q, sc.p, m * sizeof(double), hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipStreamSynchronize(st);
    }
    return e;
}

// The populations of one lattice in FP64.
template <typename R>
hipError_t fetch_populations(DevScratch &sc, hipStream_t st, const lb3d_params &p, const void *f, double *out)
{
    const uint32_t ns = (uint32_t)p.nx * (uint32_t)p.ny * (uint32_t)p.nz;
    const uint64_t n = (uint64_t)p.ncomp * 19u * ns;
    if constexpr (sizeof(R) == 8) {  // as stored
        hipError_t e = hipMemcpyAsync(out, f, n * 8, hipMemcpyDeviceToHost, st);
        return e == hipSuccess ? hipStreamSynchronize(st) : e;
    } else {
        const PopBase b = pop_base(p);
        return fetch_f64(sc, st, out, n, [&](uint32_t q, uint32_t m, double *o) {
            k_get_populations<R><<<(m + 255) / 256, 256, 0, st>>>((const R *)f, b, ns, q, m, o);
        });
    }
}

}  // namespace lb3d
