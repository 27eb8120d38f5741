// direct_sum.hip -- the exact pair sum of the scalar potential on gfx950.
//
// phi_i = (dV/dx) * sum_{j != i} rho_j / |r_i - r_j|_u   with distances in units
// of dx (r_u = (dxi, dyi*ay, dzi*az)), the computation of the reference's
// calc_potential_exact (fmm_calc.cu:412-461) and calc_potential_exact_kernel
// (potential_calc.cu:18-116).
//
// Three forms (direct_form): direct_small_kernel on a 1/r table in LDS for
// small grids, FP64 transforms (direct_fft.hip) for larger ones, and the pair
// loop over source chunks for grids that fit neither (very long or many layers).
//
// The pair loop: a 2D grid of (target block of 256) x (source chunk).  A block
// stages its chunk through LDS in tiles of 256 sources as float4 (x, y, z,
// rho) built from the linear index once per tile; every lane then walks the
// tile with LDS broadcast reads (one ds_read_b128 per source per wave).  Each
// lane accumulates a tile in FP32 and folds the tile sum into an FP64
// accumulator, so summation error grows with the tile, not with N.  Chunk
// partials go to an FP64 scratch [nchunk][n] and a second kernel adds them in
// fixed order (bitwise reproducible run to run).  The self pair is excluded by
// r^2 > 0.  1/r is the hardware reciprocal square root (v_rsq_f32): r^2 of
// two distinct cells is at least min(1, ay^2, az^2) in cell units, never
// denormal, so the denormal scaling of rsqrtf is not needed.
#include <mutex>
#include <type_traits>

#include "div_by.hpp"
#include "mms_internal.hpp"

namespace mms {
namespace {

constexpr int TB = 256;    // targets per block (one per lane)
constexpr int TILE = 256;  // sources per LDS tile

// Reference-order direct sum: padding entries of the 1 / r table (reads pass a
// row's end by at most 6), and the cells between which the table form is taken.
constexpr long kRefPad = 8, kRefTableMin = 4096, kRefTableMax = 1L << 24;

// Scratch of the entry point that allocates nothing
// (mms_potential_exact_noalloc), per GPU, held until the process ends: chunk
// partial sums (16 MiB for its largest grids) or the transforms' tables and
// work arrays (at most 32 bytes a cell each while no side is padded more
// than four times; 124.2 MiB, on 1025 x 136 x 15, is the most that any grid
// of 2,097,152 cells takes).
constexpr long kScratchCells = 2L * 1024 * 1024;
constexpr size_t kScratchBytes = 128u << 20;
static __device__ __align__(256) double scratch[kScratchBytes / sizeof(double)];

__global__ __launch_bounds__(TB) void direct_partial_kernel(const float *__restrict__ rho, double *__restrict__ part,
                                                            int xd, int yd, int zd, float ay, float az,
                                                            long n, long chunk) {
    __shared__ float4 src[TILE];
    const long t = (long)blockIdx.x * TB + threadIdx.x;
    const long c0 = (long)blockIdx.y * chunk;
    long c1 = c0 + chunk;
    if (c1 > n) c1 = n;
    const long plane = (long)xd * yd;
    float tx = 0.f, ty = 0.f, tz = 0.f;
    if (t < n) {
        tx = (float)(t % xd);
        ty = (float)((t / xd) % yd) * ay;
        tz = (float)(t / plane) * az;
    }
    double acc = 0.0;
    for (long base = c0; base < c1; base += TILE) {
        const long j = base + threadIdx.x;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (j < c1) {
            v.x = (float)(j % xd);
            v.y = (float)((j / xd) % yd) * ay;
            v.z = (float)(j / plane) * az;
            v.w = rho[j];
        }
        __syncthreads();
        src[threadIdx.x] = v;
        __syncthreads();
        const int cnt = (int)((c1 - base) < TILE ? (c1 - base) : TILE);
        float s = 0.f;
#pragma unroll 8
        for (int k = 0; k < cnt; k++) {
            const float4 q = src[k];
            const float ddx = tx - q.x, ddy = ty - q.y, ddz = tz - q.z;
            const float r2 = ddx * ddx + ddy * ddy + ddz * ddz;
            const float inv = (r2 > 0.f) ? __builtin_amdgcn_rsqf(r2) : 0.f;  // r2 >= min(1, ay^2, az^2): never denormal
            s = fmaf(q.w, inv, s);
        }
        acc += (double)s;
    }
    if (t < n) part[(long)blockIdx.y * n + t] = acc;
}

__global__ __launch_bounds__(256) void direct_reduce_kernel(const double *__restrict__ part, float *__restrict__ phi,
                                                            long n, int nchunk, double scale) {
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    double s = 0.0;
    for (int c = 0; c < nchunk; c++) s += part[(long)c * n + t];
    phi[t] = (float)(s * scale);
}

// Small grids: the 1/r table G[|dz|][|dy|][|dx|] (FP64 rounded once, G[0] = 0
// excludes the cell itself) and every charge in LDS.  A thread sums four
// consecutive x targets: their seven table entries of four sources slide
// along the row, so four LDS words and one 16-byte charge read serve 16
// products (the batch's table kernel reads a word per product).  A workgroup
// takes kSmallGroups such groups and splits the source rows (in pieces of
// kSmallRun) over 64 slices, so that a 32 x 32 x 3 film has 96 workgroups of
// eight waves; FP32 over a piece, FP64 across pieces and slices.  With FROM_M
// every workgroup forms all charges itself (div M, vector_functions.cpp:8-28)
// and a separate charge launch falls away.  A third of the kernel's 10 us is a
// launch and its first loads, the rest instructions: buffer loads whose range
// check stands for the stencil's edge branches and divisions by known
// divisors took 6 of 58.5 us off a step of the 32 x 32 x 3 film, half the groups a workgroup 4
// (40 x 36 x 4: 84 -> 72 -> 62 us; 4 groups a workgroup 76, 4-cell batches
// against 8 62 against 64).  Charge, pair loop and reduction as three launches
// an evaluation took 128 us; error against 64 bits 6e-7 -> 2.8e-7.
constexpr int kSmallGroups = 8, kSmallSlices = 64, kSmallRun = 128, kSmallBatch = 4;
constexpr int kSmallThreads = kSmallGroups * kSmallSlices;
// e / d for 0 <= e < 2^21 with inv = 1 / d: (e + 1/2) / d is at least 1 / 2d
// away from an integer, the rounding at most e 2^-22 / d
__device__ __forceinline__ int small_div(int e, float inv) { return (int)(((float)e + 0.5f) * inv); }
struct SmallShape {
    int xq, ts;      // row lengths in LDS: charges (4 mod 8: rows on different banks), table (odd)
    int rows, nseg;
};
__host__ __device__ inline SmallShape small_shape(int xd, int yd, int zd) {
    SmallShape h;
    const int r4 = (xd + 3) & ~3;
    h.xq = (r4 & 7) ? r4 : r4 + 4;
    h.ts = xd | 1;
    h.rows = yd * zd;
    h.nseg = (r4 + kSmallRun - 1) / kSmallRun;
    return h;
}
// the table's LDS floats: reads pass a row's end by at most 3 entries
__host__ __device__ inline int small_table_floats(const SmallShape &h) { return (h.rows * h.ts + 7) & ~3; }
size_t small_lds(const Grid &g) {
    const SmallShape h = small_shape(g.xd, g.yd, g.zd);
    const size_t q = (size_t)h.rows * h.xq, red = 2 * 4 * kSmallGroups * kSmallSlices;
    return sizeof(float) * ((size_t)small_table_floats(h) + (q > red ? q : red));
}

__global__ __launch_bounds__(256) void small_table_kernel(float *__restrict__ tab, int xd, int yd, int zd, double ay,
                                                          double az) {
    const SmallShape h = small_shape(xd, yd, zd);
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= small_table_floats(h)) return;
    const int r = e / h.ts, x = e - r * h.ts, z = r / yd, y = r - z * yd;
    const double ry = y * ay, rz = z * az, r2 = (double)x * x + ry * ry + rz * rz;
    tab[e] = (r < h.rows && r2 > 0.0) ? (float)(1.0 / sqrt(r2)) : 0.0f;
}

template <bool FROM_M>
__global__ __launch_bounds__(kSmallThreads) void direct_small_kernel(const float *__restrict__ src,
                                                                     float *__restrict__ rho_out,
                                                                     float *__restrict__ phi,
                                                                     const float *__restrict__ gtab, int xd, int yd,
                                                                     int zd, float dx, float dy, float dz,
                                                                     double scale) {
    extern __shared__ __attribute__((aligned(16))) float slds[];
    const SmallShape h = small_shape(xd, yd, zd);
    const int tf = small_table_floats(h), n = xd * h.rows, nq = h.rows * h.xq, plane = xd * yd;
    float *tab = slds, *q = slds + tf;
    const float ixq = 1.0f / (float)h.xq, iyd = 1.0f / (float)yd;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(src), (short)0, (FROM_M ? 12 : 4) * n, 0x00020000);
    const float rdx = 1.0f / dx, rdy = 1.0f / dy, rdz = 1.0f / dz;
    auto ld = [&](int off) { return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0)); };
    for (int e0 = threadIdx.x, k0 = 0; e0 < nq; e0 += kSmallThreads * kSmallBatch, k0 += kSmallBatch) {
        constexpr int NV = FROM_M ? 6 : 1;
        float v[kSmallBatch][NV];
#pragma unroll
        for (int k = 0; k < kSmallBatch; k++) {
            const int e = e0 + k * kSmallThreads, r = small_div(e, ixq), x = e - r * h.xq, c = r * xd + x;
            const bool ok = e < nq && x < xd;
            if constexpr (FROM_M) {
                const int z = small_div(r, iyd), y = r - z * yd;
                // buffer loads: zeros past the planes' end, no branches
                v[k][0] = ld(ok && x != xd - 1 ? 4 * (c + 1) : 12 * n);
                v[k][1] = ld(ok && x != 0 ? 4 * (c - 1) : 12 * n);
                v[k][2] = ld(ok && y != yd - 1 ? 4 * (n + c + xd) : 12 * n);
                v[k][3] = ld(ok && y != 0 ? 4 * (n + c - xd) : 12 * n);
                v[k][4] = ld(ok && z != zd - 1 ? 4 * (2 * n + c + plane) : 12 * n);
                v[k][5] = ld(ok && z != 0 ? 4 * (2 * n + c - plane) : 12 * n);
            } else {
                v[k][0] = ld(ok ? 4 * c : 4 * n);
            }
        }
        if (k0 == 0)  // the table, while the first charges' loads are in flight
            for (int e = threadIdx.x; e < tf / 4; e += kSmallThreads)
                reinterpret_cast<float4 *>(tab)[e] = reinterpret_cast<const float4 *>(gtab)[e];
#pragma unroll
        for (int k = 0; k < kSmallBatch; k++) {
            const int e = e0 + k * kSmallThreads;
            float c = v[k][0];
            if constexpr (FROM_M) c = (div_by(v[k][0] - v[k][1], dx, rdx) + div_by(v[k][2] - v[k][3], dy, rdy) + div_by(v[k][4] - v[k][5], dz, rdz)) * 0.5f;
            if (e < nq) {
                q[e] = c;
                if constexpr (FROM_M) {  // one workgroup writes each charge
                    const int r = small_div(e, ixq), x = e - r * h.xq;
                    if (x < xd && (k0 + k) % gridDim.x == blockIdx.x) rho_out[r * xd + x] = c;
                }
            }
        }
    }
    __syncthreads();
    const int ngx = (xd + 3) >> 2, ngroup = ngx * h.rows;
    const float ingx = 1.0f / (float)ngx, inseg = 1.0f / (float)h.nseg;
    const int gi = threadIdx.x % kSmallGroups, sl = threadIdx.x / kSmallGroups;
    const int grp = blockIdx.x * kSmallGroups + gi;
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    if (grp < ngroup) {
        const int rt = small_div(grp, ingx), xt = 4 * (grp - rt * ngx), zt = small_div(rt, iyd), yt = rt - zt * yd;
        for (int it = sl; it < h.rows * h.nseg; it += kSmallSlices) {
            const int rs = small_div(it, inseg), xs0 = (it - rs * h.nseg) * kSmallRun, zs = small_div(rs, iyd);
            const int ys = rs - zs * yd, xs1 = xs0 + kSmallRun < xd ? xs0 + kSmallRun : xd;
            const float *g = tab + (abs(zt - zs) * yd + abs(yt - ys)) * h.ts;
            const float4 *qr = reinterpret_cast<const float4 *>(q + rs * h.xq);
            // w0 .. w6 = G[|xt - xs - 3|] .. G[|xt - xs + 3|]: entries of the sources xs .. xs + 3
            float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
            int d = xt - xs0;
            float w4 = g[abs(d + 1)], w5 = g[abs(d + 2)], w6 = g[abs(d + 3)];
#pragma unroll 4
            for (int xs = xs0; xs < xs1; xs += 4, d -= 4) {
                const float4 c = qr[xs >> 2];
                const float w0 = g[abs(d - 3)], w1 = g[abs(d - 2)], w2 = g[abs(d - 1)], w3 = g[abs(d)];
                s0 = fmaf(c.x, w3, s0); s1 = fmaf(c.x, w4, s1); s2 = fmaf(c.x, w5, s2); s3 = fmaf(c.x, w6, s3);
                s0 = fmaf(c.y, w2, s0); s1 = fmaf(c.y, w3, s1); s2 = fmaf(c.y, w4, s2); s3 = fmaf(c.y, w5, s3);
                s0 = fmaf(c.z, w1, s0); s1 = fmaf(c.z, w2, s1); s2 = fmaf(c.z, w3, s2); s3 = fmaf(c.z, w4, s3);
                s0 = fmaf(c.w, w0, s0); s1 = fmaf(c.w, w1, s1); s2 = fmaf(c.w, w2, s2); s3 = fmaf(c.w, w3, s3);
                w4 = w0; w5 = w1; w6 = w2;
            }
            acc[0] += (double)s0; acc[1] += (double)s1; acc[2] += (double)s2; acc[3] += (double)s3;
        }
    }
    __syncthreads();  // the charges' LDS becomes the slices' sums [slice][target]
    double *red = reinterpret_cast<double *>(q);
#pragma unroll
    for (int i = 0; i < 4; i++) red[sl * 4 * kSmallGroups + 4 * gi + i] = acc[i];
    __syncthreads();
    // four slices a thread, kRed threads a target
    constexpr int kRed = kSmallSlices / 4;
    static_assert(kRed * 4 * kSmallGroups == kSmallThreads, "one thread per four slices of a target");
    const int o = threadIdx.x / kRed, p = threadIdx.x % kRed;
    double v = 0.0;
#pragma unroll
    for (int k = 0; k < 4; k++) v += red[(4 * p + k) * 4 * kSmallGroups + o];
#pragma unroll
    for (int m = 1; m < kRed; m <<= 1) v += __shfl_xor(v, m);
    const int go = blockIdx.x * kSmallGroups + (o >> 2);
    if (p == 0 && go < ngroup) {
        const int r = small_div(go, ingx), x = 4 * (go - r * ngx) + (o & 3);
        if (x < xd) phi[r * xd + x] = (float)(v * scale);
    }
}

// FP64 probe oracle on the device: a 2D grid of (block of 256 probes) x
// (source chunk); sources are staged through LDS as (x, y, z, rho) once per
// tile and every pair is evaluated in FP64.  Chunk partials [nchunk][np] are
// added in fixed order by probes_f64_reduce_kernel.
__global__ __launch_bounds__(256) void probes_f64_kernel(const float *__restrict__ rho, const int64_t *__restrict__ probes,
                                                         double *__restrict__ part, int np, int xd, int yd, int zd,
                                                         double dx, double dy, double dz, long chunk) {
    __shared__ double4 src[TILE];
    const long n = (long)xd * yd * zd, plane = (long)xd * yd;
    const int p = blockIdx.x * 256 + threadIdx.x;
    double tx = 0.0, ty = 0.0, tz = 0.0;
    if (p < np) {
        const long i = probes[p];
        tx = (double)(i % xd) * dx;
        ty = (double)((i / xd) % yd) * dy;
        tz = (double)(i / plane) * dz;
    }
    const long c0 = (long)blockIdx.y * chunk;
    const long c1 = (c0 + chunk < n) ? c0 + chunk : n;
    double acc = 0.0;
    for (long base = c0; base < c1; base += TILE) {
        const long j = base + threadIdx.x;
        double4 v = make_double4(0.0, 0.0, 0.0, 0.0);
        if (j < c1) {
            v.x = (double)(j % xd) * dx;
            v.y = (double)((j / xd) % yd) * dy;
            v.z = (double)(j / plane) * dz;
            v.w = (double)rho[j];
        }
        __syncthreads();
        src[threadIdx.x] = v;
        __syncthreads();
        const int cnt = (int)((c1 - base) < TILE ? (c1 - base) : TILE);
        for (int k = 0; k < cnt; k++) {
            const double4 q = src[k];
            const double rx = tx - q.x, ry = ty - q.y, rz = tz - q.z;
            const double r2 = rx * rx + ry * ry + rz * rz;
            if (r2 > 0.0) acc += q.w / sqrt(r2);
        }
    }
    if (p < np) part[(long)blockIdx.y * np + p] = acc;
}

__global__ __launch_bounds__(256) void probes_f64_reduce_kernel(const double *__restrict__ part, double *__restrict__ out,
                                                                int np, int nchunk, double dv) {
    const int p = blockIdx.x * 256 + threadIdx.x;
    if (p >= np) return;
    double s = 0.0;
    for (int c = 0; c < nchunk; c++) s += part[(long)c * np + p];
    out[p] = s * dv;
}

// Batched small films: block b takes work item items[b] = (film, target block)
// and sums every source of its film (LDS tiles, FP32 per tile, FP64 across
// tiles), writing phi directly.
__global__ __launch_bounds__(TB) void direct_batch_kernel(const float *__restrict__ rho, float *__restrict__ phi,
                                                          const int2 *__restrict__ items,
                                                          const BatchFilm *__restrict__ films, float ay, float az,
                                                          double scale) {
    __shared__ float4 src[TILE];
    const int2 it = items[blockIdx.x];
    const BatchFilm f = films[it.x];
    const int xd = f.xd, yd = f.yd;
    const long plane = (long)xd * yd, n = plane * f.zd;
    rho += f.off;
    phi += f.off;
    const long t = (long)it.y * TB + threadIdx.x;
    float tx = 0.f, ty = 0.f, tz = 0.f;
    if (t < n) {
        tx = (float)(t % xd);
        ty = (float)((t / xd) % yd) * ay;
        tz = (float)(t / plane) * az;
    }
    double acc = 0.0;
    for (long base = 0; base < n; base += TILE) {
        const long j = base + threadIdx.x;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (j < n) {
            v.x = (float)(j % xd);
            v.y = (float)((j / xd) % yd) * ay;
            v.z = (float)(j / plane) * az;
            v.w = rho[j];
        }
        __syncthreads();
        src[threadIdx.x] = v;
        __syncthreads();
        const int cnt = (int)((n - base) < TILE ? (n - base) : TILE);
        float s = 0.f;
#pragma unroll 8
        for (int k = 0; k < cnt; k++) {
            const float4 q = src[k];
            const float ddx = tx - q.x, ddy = ty - q.y, ddz = tz - q.z;
            const float r2 = ddx * ddx + ddy * ddy + ddz * ddz;
            const float inv = (r2 > 0.f) ? __builtin_amdgcn_rsqf(r2) : 0.f;  // r2 >= min(1, ay^2, az^2): never denormal
            s = fmaf(q.w, inv, s);
        }
        acc += (double)s;
    }
    if (t < n) phi[t] = (float)(acc * scale);
}

// Batched small films on a 1/r table.  On the grid, 1/r depends only on the
// absolute cell offsets, so the film's table G[|dz|][|dy|][|dx|] (xd*yd*zd
// floats, built on the host in FP64 and rounded once; G[0] = 0 excludes the
// cell itself) and its charges (rows padded to a multiple of 4 with zeros)
// sit in LDS.  Per pair: one absolute difference plus row base (the table
// byte offset, v_sad_u32), one LDS read, one FMA; FP32 over a source row (at
// most 256 sources, four interleaved chains), FP64 across rows.  Two threads
// per target (the even and the odd source rows of every layer), added at the end.  The
// padded sources read table entries past the row (or past the table, into
// its zeroed padding and the charges), all finite, times a zero charge.
constexpr int TT = 2 * TB;  // threads of the table kernel
__global__ __launch_bounds__(TT) void direct_table_kernel(const float *__restrict__ rho, float *__restrict__ phi,
                                                          const float *__restrict__ gtab,
                                                          const int2 *__restrict__ items,
                                                          const BatchFilm *__restrict__ films, double scale) {
    extern __shared__ __attribute__((aligned(16))) float dlds[];
    __shared__ double half1[TB];
    const int2 it = items[blockIdx.x];
    const BatchFilm f = films[it.x];
    const int xd = f.xd, yd = f.yd, zd = f.zd, xdp = (xd + 3) & ~3;
    const int plane = xd * yd, n = plane * zd, n4 = (n + 3) & ~3;
    float *tab = dlds;       // [zd][yd][xd]
    float *q = dlds + n4;    // [zd][yd][xdp]
    rho += f.off;
    phi += f.off;
    gtab += f.off;
    for (int e = threadIdx.x; e < n4; e += TT) tab[e] = e < n ? gtab[e] : 0.0f;  // padding read by padded sources
    for (int e = threadIdx.x; e < zd * yd * xdp; e += TT) {
        const int xs = e % xdp, r = e / xdp;
        q[e] = xs < xd ? rho[(long)r * xd + xs] : 0.0f;
    }
    __syncthreads();
    const int h = threadIdx.x / TB, t = it.y * TB + (threadIdx.x % TB);
    double acc = 0.0;
    if (t < n) {
        const int xt = t % xd, yt = (t / xd) % yd, zt = t / plane;
        const char *tb = reinterpret_cast<const char *>(tab);
        const unsigned x4t = 4u * (unsigned)xt;
        const int ng = xdp >> 2;  // float4 groups of a row
        for (int zs = 0; zs < zd; zs++) {
            const unsigned bz = 4u * (unsigned)((zt > zs ? zt - zs : zs - zt) * plane);
            for (int ys = h; ys < yd; ys += 2) {
                // byte offset of the table row; a source's entry is |4 xt - 4 xs| further
                const unsigned rb = __umul24((unsigned)(yt > ys ? yt - ys : ys - yt), 4u * (unsigned)xd) + bz;
                const float4 *qr = reinterpret_cast<const float4 *>(q + (zs * yd + ys) * xdp);
                for (int g0 = 0; g0 < ng; g0 += 64) {  // FP32 over at most 256 sources
                    const int g1 = (g0 + 64 < ng) ? g0 + 64 : ng;
                    float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;  // one chain per column mod 4
                    for (int g = g0; g < g1; g++) {
                        const float4 c = qr[g];
                        const unsigned x4s = 16u * (unsigned)g;
                        s0 = fmaf(c.x, *reinterpret_cast<const float *>(tb + (max(x4t, x4s) - min(x4t, x4s) + rb)), s0);
                        s1 = fmaf(c.y, *reinterpret_cast<const float *>(tb + (max(x4t, x4s + 4) - min(x4t, x4s + 4) + rb)), s1);
                        s2 = fmaf(c.z, *reinterpret_cast<const float *>(tb + (max(x4t, x4s + 8) - min(x4t, x4s + 8) + rb)), s2);
                        s3 = fmaf(c.w, *reinterpret_cast<const float *>(tb + (max(x4t, x4s + 12) - min(x4t, x4s + 12) + rb)), s3);
                    }
                    acc += (double)((s0 + s1) + (s2 + s3));
                }
            }
        }
    }
    if (h == 1) half1[threadIdx.x - TB] = acc;
    __syncthreads();
    if (h == 0 && t < n) phi[t] = (float)((acc + half1[threadIdx.x]) * scale);
}

// The summation order and float arithmetic of the reference's CUDA kernel
// calc_potential_exact_kernel (potential_calc.cu:18-116), for callers that
// want its results bit for bit:
//   - 1024 partial sums per target: partial t adds the sources
//     [t * tstride, (t + 1) * tstride), tstride = ceilf(N / 1024.f), in
//     index order, each term (charge_i * dV) / sqrtf(Rx^2 + Ry^2 + Rz^2)
//     with R = ((x - x_) dx, (y - y_) dy, (z - z_) dz), dV = dx dy dz, the
//     self term skipped (potential_calc.cu:57-75);
//   - the partials added by the halving tree s[t] += s[t + h], h = 512 .. 1
//     (potential_calc.cu:82-111).
// Every operation is rounded on its own (no fused multiply-add), with
// IEEE division and square root.  A workgroup is the reference's 1024
// virtual threads applied to RT targets at once: each source is loaded and
// its coordinates decoded once for the RT targets, and the RT reduction
// trees run together in LDS.
//
// Two kernels.  direct_refgpu_kernel divides as the reference does.
// refgpu_pairs_kernel (with refgpu_prepare_kernel before it) forms the same
// bits faster:
//   - r depends on the absolute offsets only, so 1 / r is read from a table of
//     doubles (r itself by the reference's operations);
//   - the quotient q / r of two floats rounded to 24 bits is the double
//     product q (1/r) rounded to 24 bits: the product is within 2^-52 of the
//     quotient, and no quotient of 24-bit numbers is nearer than 2^-49 to a
//     midpoint of floats (b m, the divisor times a 25-bit midpoint, is an
//     integer multiple of the dividend's unit and never equal to it) as long
//     as the result is a normal float;
//   - lanes are targets (four neighbours in x each) and the sources
//     wave-uniform, so four table entries serve 16 pairs; the 1024 partials of a target are
//     taken in bit-reversed order, which the halving tree turns into a stack
//     of sums, the waves of a workgroup holding the subtrees of equal t mod 4
//     within the workgroup's t mod C (refgpu_join_kernel adds the C subtrees).
// refgpu_prepare_kernel notes a source whose quotients may be denormal or not
// finite; the dividing kernel then takes the call.  A 100 x 75 x 3 potential on host arrays:
// 677 -> 140 us, 128 x 128 x 3 2.99 -> 0.39 ms; below kRefTableMin cells the three extra launches cost
// more than they give (32 x 32 x 3: 51 us without, 64 with).
constexpr int RT = 8;

__global__ __launch_bounds__(1024) void direct_refgpu_kernel(const float *__restrict__ rho, float *__restrict__ phi,
                                                             int xd, int yd, int n, float dx, float dy, float dz,
                                                             int tstride, const int *__restrict__ need) {
#pragma clang fp contract(off)
    if (need && *need == 0) return;  // the table form has taken this call
    __shared__ float sdata[RT][1024];
    const int t = threadIdx.x;
    const int plane = xd * yd;
    for (int b0 = blockIdx.x * RT; b0 < n; b0 += gridDim.x * RT) {
        int tx[RT], ty[RT], tz[RT];
#pragma unroll
        for (int k = 0; k < RT; k++) {
            const int bi = (b0 + k < n) ? b0 + k : 0;
            tx[k] = bi % xd;
            ty[k] = ((bi - tx[k]) / xd) % yd;
            tz[k] = (bi - tx[k] - ty[k] * xd) / plane;
        }
        float pot[RT];
#pragma unroll
        for (int k = 0; k < RT; k++) pot[k] = 0.0f;
        const int ti1 = t * tstride;
        if (ti1 < n) {
            const float dV = dx * dy * dz;
            const int i1 = (ti1 + tstride < n) ? ti1 + tstride : n;
            for (int i = ti1; i < i1; i++) {
                const float q = rho[i] * dV;
                const int x_ = i % xd;
                const int y_ = ((i - x_) / xd) % yd;
                const int z_ = (i - x_ - y_ * xd) / plane;
#pragma unroll
                for (int k = 0; k < RT; k++) {
                    if (b0 + k == i) continue;
                    const float Rx = (float)(tx[k] - x_) * dx, Ry = (float)(ty[k] - y_) * dy, Rz = (float)(tz[k] - z_) * dz;
                    const float r = sqrtf(Rx * Rx + Ry * Ry + Rz * Rz);
                    pot[k] += q / r;
                }
            }
        }
#pragma unroll
        for (int k = 0; k < RT; k++) sdata[k][t] = pot[k];
        __syncthreads();
        for (int h = 512; h > 0; h >>= 1) {
            if (t < h) {
#pragma unroll
                for (int k = 0; k < RT; k++) sdata[k][t] += sdata[k][t + h];
            }
            __syncthreads();
        }
        if (t < RT && b0 + t < n) phi[b0 + t] = sdata[t][0];
        __syncthreads();
    }
}

// 1 / r of every absolute offset, r by the reference's float operations; 0 at
// the cell itself (its term is skipped) and in the padding past the last row.
__global__ __launch_bounds__(256) void refgpu_table_kernel(double *__restrict__ tab, int xd, int yd, long n, float dx,
                                                           float dy, float dz) {
#pragma clang fp contract(off)
    const long e = blockIdx.x * 256L + threadIdx.x;
    if (e >= n + kRefPad) return;
    const int x = (int)(e % xd);
    const long r = e / xd;
    const int y = (int)(r % yd), z = (int)(r / yd);
    const float Rx = (float)x * dx, Ry = (float)y * dy, Rz = (float)z * dz;
    const float d = sqrtf(Rx * Rx + Ry * Ry + Rz * Rz);
    tab[e] = (e > 0 && e < n) ? 1.0 / (double)d : 0.0;
}

// q = rho dV in float, as a double; *need = 1 if a non-zero |q| is below qmin
// (a quotient might be denormal) or not finite.  *need is 0 before.
__global__ __launch_bounds__(256) void refgpu_prepare_kernel(const float *__restrict__ rho, double *__restrict__ qd,
                                                             int *__restrict__ need, int n, float dV, float qmin) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float q = rho[i] * dV;
    qd[i] = (double)q;
    const float a = fabsf(q);
    if (!(a <= 3.402823466e38f) || (a < qmin && q != 0.0f)) *need = 1;
}

__global__ void refgpu_clear_kernel(int *need) { *need = 0; }

// Targets of this wave: groups of four x neighbours, group 64 blockIdx.x + lane.
// Wave w of workgroup (., c) sums the partials t = j + S m, j = c + C w,
// S = 4 C, m = 0 .. 1024 / S - 1, for its targets.
template <int C>
__global__ __launch_bounds__(256) void refgpu_pairs_kernel(const double *__restrict__ qd, const double *__restrict__ tab,
                                                           float *__restrict__ part,
                                                           const int *__restrict__ need, int xd, int yd, int zd, int n,
                                                           int tstride) {
#pragma clang fp contract(off)
    if (*need != 0) return;
    constexpr int S = 4 * C, M = 1024 / S, D = __builtin_ctz(M);
    __shared__ float4 sub[4][64];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), j = blockIdx.y + C * w;
    const int ngx = (xd + 3) >> 2, ngroup = ngx * yd * zd;
    const int grp = blockIdx.x * 64 + lane < ngroup ? blockIdx.x * 64 + lane : ngroup - 1;
    const int rt = grp / ngx, xt = 4 * (grp - rt * ngx), zt = rt / yd, yt = rt - zt * yd;
    float st[D][4], acc[4];
    for (int i = 0; i < M; i++) {
        const int m = (int)(__builtin_bitreverse32((unsigned)i) >> (32 - D)), t = j + S * m;
        float p0 = 0.0f, p1 = 0.0f, p2 = 0.0f, p3 = 0.0f;
        const long lo = (long)t * tstride;
        if (lo < n) {
            int s = (int)lo;
            const int end = n - s < tstride ? n : s + tstride;
            int r = s / xd, xs = s - r * xd, zs = r / yd, ys = r - zs * yd;
            while (s < end) {  // the pieces of the chunk in one row of sources
                const int len = xd - xs < end - s ? xd - xs : end - s;
                const double *g = tab + ((long)abs(zt - zs) * yd + abs(yt - ys)) * xd;
                int d = xt - xs;
                double w4 = g[abs(d + 1)], w5 = g[abs(d + 2)], w6 = g[abs(d + 3)];
                for (int k = 0; k < len; k += 4, d -= 4) {
                    // sources past the piece add 0
                    const double q0 = qd[s + k], q1 = k + 1 < len ? qd[s + k + 1] : 0.0;
                    const double q2 = k + 2 < len ? qd[s + k + 2] : 0.0, q3 = k + 3 < len ? qd[s + k + 3] : 0.0;
                    const double w0 = g[abs(d - 3)], w1 = g[abs(d - 2)], w2 = g[abs(d - 1)], w3 = g[abs(d)];
                    p0 += (float)(q0 * w3); p1 += (float)(q0 * w4); p2 += (float)(q0 * w5); p3 += (float)(q0 * w6);
                    p0 += (float)(q1 * w2); p1 += (float)(q1 * w3); p2 += (float)(q1 * w4); p3 += (float)(q1 * w5);
                    p0 += (float)(q2 * w1); p1 += (float)(q2 * w2); p2 += (float)(q2 * w3); p3 += (float)(q2 * w4);
                    p0 += (float)(q3 * w0); p1 += (float)(q3 * w1); p2 += (float)(q3 * w2); p3 += (float)(q3 * w3);
                    w4 = w0; w5 = w1; w6 = w2;
                }
                s += len;
                xs = 0;
                if (++ys == yd) { ys = 0; zs++; }
            }
        }
        // s[t] += s[t + h]: merge equal subtrees, as a binary counter carries
        acc[0] = p0; acc[1] = p1; acc[2] = p2; acc[3] = p3;
#pragma unroll
        for (int l = 0; l < D; l++) {
            if ((i & ((1 << l) - 1)) == (1 << l) - 1) {  // the carry reaches level l
                if (i & (1 << l)) {
#pragma unroll
                    for (int k = 0; k < 4; k++) acc[k] = st[l][k] + acc[k];
                } else {
#pragma unroll
                    for (int k = 0; k < 4; k++) st[l][k] = acc[k];
                }
            }
        }
    }
    sub[w][lane] = make_float4(acc[0], acc[1], acc[2], acc[3]);
    for (int h = 2; h > 0; h >>= 1) {
        __syncthreads();
        if (w < h) {
            const float4 a = sub[w][lane], b = sub[w + h][lane];
            sub[w][lane] = make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
        }
    }
    if (w == 0 && blockIdx.x * 64 + lane < ngroup) {
        const float4 v = sub[0][lane];
        float *dst = part + (long)blockIdx.y * n + (long)rt * xd + xt;
        dst[0] = v.x;
        if (xt + 1 < xd) dst[1] = v.y;
        if (xt + 2 < xd) dst[2] = v.z;
        if (xt + 3 < xd) dst[3] = v.w;
    }
}

// the last levels of the tree: partials c = 0 .. C - 1
template <int C>
__global__ __launch_bounds__(256) void refgpu_join_kernel(const float *__restrict__ part, float *__restrict__ phi,
                                                          const int *__restrict__ need, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n || *need != 0) return;
    float v[C];
#pragma unroll
    for (int c = 0; c < C; c++) v[c] = part[(long)c * n + i];
#pragma unroll
    for (int h = C / 2; h > 0; h >>= 1)
#pragma unroll
        for (int c = 0; c < h; c++) v[c] += v[c + h];
    phi[i] = v[0];
}

}  // namespace

static int refgpu_groups(const Grid &g) { return (int)(((long)((g.xd + 3) / 4) * g.yd * g.zd + 63) / 64); }

// The table form needs r finite and well inside the float range, and quotients
// that are normal floats (checked charge by charge against qmin = 2^-125 rmax).
// Films one cell wide fill a quarter of its groups of four x neighbours and
// stay with the division (1 x 5000 x 1: 144 us by the table, 96 by the
// division; 2 x 2100 x 1: 67 and 78).
int RefgpuPlan::init(const Grid &g) {
    release();
    const long n = g.n();
    const double ext = (double)g.xd * g.dx + (double)g.yd * g.dy + (double)g.zd * g.dz;
    const float small = fminf(g.dx, fminf(g.dy, g.dz));
    if (g.xd == 1 || n < kRefTableMin || n > kRefTableMax || small < 1e-15f || ext > 1e15) return 0;  // direct_refgpu_kernel alone
    qmin = (float)(ext * 2.3509887e-38);
    split = refgpu_groups(g) < 1024 ? 16 : 4;  // workgroups a target group: enough to fill the chip
    if (hipMalloc(&tab, sizeof(double) * (n + kRefPad)) != hipSuccess ||
        hipMalloc(&qd, sizeof(double) * n + sizeof(float) * split * n + 256) != hipSuccess) {
        (void)hipGetLastError();
        release();
        return 0;  // no memory for it: direct_refgpu_kernel alone
    }
    part = reinterpret_cast<float *>(qd + n);
    need = reinterpret_cast<int *>(part + split * n);
    hipLaunchKernelGGL(refgpu_table_kernel, dim3((unsigned)((n + kRefPad + 255) / 256)), dim3(256), 0, nullptr, tab, g.xd,
                       g.yd, n, g.dx, g.dy, g.dz);
    MMS_HIP(hipGetLastError());
    MMS_HIP(hipStreamSynchronize(nullptr));
    return 0;
}

void RefgpuPlan::release() {
    if (tab) (void)hipFree(tab);
    if (qd) (void)hipFree(qd);
    tab = qd = nullptr;
    part = nullptr;
    need = nullptr;
}

int direct_refgpu_potential(const Grid &g, const RefgpuPlan &plan, const float *rho, float *phi, hipStream_t s,
                            Profiler *prof) {
    KTimer kt(prof, K_DIRECT);
    const long n = g.n();
    MMS_CHECK(n < (1L << 30), "reference-order direct sum: grid too large");
    // tstride as the reference computes it: ceilf(N / (float)blockDim.x)
    const int tstride = (int)ceilf((float)n / 1024.0f);
    if (plan.tab) {
        const int wb = refgpu_groups(g);
        const float dV = g.dx * g.dy * g.dz;
        hipLaunchKernelGGL(refgpu_clear_kernel, dim3(1), dim3(1), 0, s, plan.need);
        hipLaunchKernelGGL(refgpu_prepare_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, rho, plan.qd,
                           plan.need, (int)n, dV, plan.qmin);
        MMS_HIP(hipGetLastError());
        auto pairs = [&](auto c) {
            constexpr int C = decltype(c)::value;
            hipLaunchKernelGGL(refgpu_pairs_kernel<C>, dim3(wb, C), dim3(256), 0, s, plan.qd, plan.tab, plan.part,
                               plan.need, g.xd, g.yd, g.zd, (int)n, tstride);
            hipLaunchKernelGGL(refgpu_join_kernel<C>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, plan.part, phi,
                               plan.need, (int)n);
        };
        if (plan.split == 16) pairs(std::integral_constant<int, 16>());
        else pairs(std::integral_constant<int, 4>());
        MMS_HIP(hipGetLastError());
    }
    // after the table form a few workgroups, which find nothing to do but in the rare case
    const long nb = (n + RT - 1) / RT;
    hipLaunchKernelGGL(direct_refgpu_kernel, dim3((unsigned)(plan.tab && nb > 512 ? 512 : nb)), dim3(1024), 0, s, rho, phi, g.xd,
                       g.yd, (int)n, g.dx, g.dy, g.dz, tstride, plan.need);
    MMS_HIP(hipGetLastError());
    return 0;
}

int direct_batch_potential(const float *rho, float *phi, const int2 *items, int nitems, const BatchFilm *films,
                           float ay, float az, double scale, const float *tab, size_t tab_lds, hipStream_t s,
                           Profiler *prof) {
    KTimer kt(prof, K_DIRECT);
    if (nitems <= 0) return 0;
    if (tab) {
        MMS_CHECK(tab_lds <= kDirectTableLds, "direct sum: film table exceeds LDS");
        static bool attr = false;
        if (!attr) {
            MMS_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&direct_table_kernel),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)kDirectTableLds));
            attr = true;
        }
        hipLaunchKernelGGL(direct_table_kernel, dim3(nitems), dim3(TT), tab_lds, s, rho, phi, tab, items, films, scale);
    } else {
        hipLaunchKernelGGL(direct_batch_kernel, dim3(nitems), dim3(TB), 0, s, rho, phi, items, films, ay, az, scale);
    }
    MMS_HIP(hipGetLastError());
    return 0;
}

size_t direct_table_lds(int xd, int yd, int zd) {
    const long n = (long)xd * yd * zd;
    return sizeof(float) * (size_t)(((n + 3) & ~3L) + (long)zd * yd * ((xd + 3) & ~3));
}

// Source chunks of the direct sum for n cells: aim for >= 1024 blocks in
// total (4 per CU) without chunks below one tile.
static void direct_chunks(long n, int split, long *chunk, int *nchunk) {
    const long tblocks = (n + TB - 1) / TB;
    long want = (1024L * split + tblocks - 1) / tblocks;
    long maxchunks = (n + TILE - 1) / TILE;
    if (want > maxchunks) want = maxchunks;
    if (want < 1) want = 1;
    long c = (n + want - 1) / want;
    c = ((c + TILE - 1) / TILE) * TILE;
    *chunk = c;
    *nchunk = (int)((n + c - 1) / c);
}

// Which form serves a grid.  One RK4 step of a film (four evaluations and
// stage kernels, step graph), table / transforms: 48x48x3 67 / 69 us, 55x55x2
// 68 / 74, 64x64x2 72 / 72, 55x50x3 100 / 73, 64x64x3 157 / 71; 40x36x4 takes the
// table 62.  Up to 6,000 cells the table, and only while its workgroups fit the
// chip at once (256 of 8 groups): narrow films fill their groups of four
// poorly (5x1100x1 157 / 106).  The pair loop (37 ms a step on 161x117x3, where
// the transforms take 0.09) keeps the grids that fit neither.
constexpr long kTableCells = 6000;
constexpr size_t kSmallLds = 80 * 1024;
DirectForm direct_form(const Grid &g) {
    const long n = g.n();
    const bool table = n <= 16384 && small_lds(g) <= kSmallLds, fft = direct_fft_fits(g);
    const long groups = (long)((g.xd + 3) / 4) * g.yd * g.zd;
    if (table && ((n <= kTableCells && groups <= 256 * kSmallGroups) || !fft)) return kDirectTable;
    return fft ? kDirectFft : kDirectChunks;
}

static int small_table(const Grid &g, float *tab, hipStream_t s) {
    const int tf = small_table_floats(small_shape(g.xd, g.yd, g.zd));
    hipLaunchKernelGGL(small_table_kernel, dim3((tf + 255) / 256), dim3(256), 0, s, tab, g.xd, g.yd, g.zd,
                       (double)g.dy / (double)g.dx, (double)g.dz / (double)g.dx);
    MMS_HIP(hipGetLastError());
    return 0;
}

// m not null: the charges are formed from m and left in rho
static int small_potential(const Grid &g, const float *tab, const float *m, float *rho, const float *rho_in, float *phi,
                           hipStream_t s) {
    const int groups = ((g.xd + 3) / 4) * g.yd * g.zd;
    const dim3 grid((groups + kSmallGroups - 1) / kSmallGroups);
    const size_t lds = small_lds(g);
    const double scale = (double)g.dy * (double)g.dz;
    // the attribute is set on every call (a host-side table write) rather than remembered per device
    if (m) {
        MMS_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&direct_small_kernel<true>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)kSmallLds));
        hipLaunchKernelGGL(direct_small_kernel<true>, grid, dim3(kSmallThreads), lds, s, m, rho, phi, tab, g.xd, g.yd, g.zd, g.dx,
                           g.dy, g.dz, scale);
    } else {
        MMS_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&direct_small_kernel<false>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)kSmallLds));
        hipLaunchKernelGGL(direct_small_kernel<false>, grid, dim3(kSmallThreads), lds, s, rho_in, nullptr, phi, tab, g.xd, g.yd,
                           g.zd, g.dx, g.dy, g.dz, scale);
    }
    MMS_HIP(hipGetLastError());
    return 0;
}

int DirectPlan::init(const Grid &g, int split_) {
    release();
    split = (split_ == 2 || split_ == 4) ? split_ : 1;
    const long n = g.n();
    form = direct_form(g);
    if (form == kDirectTable) {
        MMS_HIP(hipMalloc(&table, sizeof(float) * small_table_floats(small_shape(g.xd, g.yd, g.zd))));
        if (small_table(g, static_cast<float *>(table), nullptr)) return 1;
        MMS_HIP(hipStreamSynchronize(nullptr));
    } else if (form == kDirectFft) {
        // tables and work arrays of up to 64 bytes a cell; where they cannot be
        // had the pair loop serves the grid, with 8 bytes a cell at least
        if (hipMalloc(&table, direct_fft_table_bytes(g)) != hipSuccess ||
            hipMalloc(&work, direct_fft_work_bytes(g)) != hipSuccess) {
            (void)hipGetLastError();
            release();
            form = kDirectChunks;
        } else {
            if (direct_fft_tables(g, table, nullptr)) return 1;
            MMS_HIP(hipStreamSynchronize(nullptr));
        }
    }
    if (form == kDirectChunks) {
        direct_chunks(n, split, &chunk, &nchunk);
        MMS_HIP(hipMalloc(&work, sizeof(double) * (size_t)n * nchunk));
    }
    return 0;
}

void DirectPlan::release() {
    if (table) (void)hipFree(table);
    if (work) (void)hipFree(work);
    table = work = nullptr;
    nchunk = 0;
}

// the two kernels of the direct sum with the chunk partials in `part`
static int direct_launch(const Grid &g, long chunk, int nchunk, double *part, const float *rho, float *phi,
                         hipStream_t s, Profiler *prof) {
    const long n = g.n();
    {
        KTimer kt(prof, K_DIRECT);
        dim3 grid((unsigned)((n + TB - 1) / TB), (unsigned)nchunk);
        hipLaunchKernelGGL(direct_partial_kernel, grid, dim3(TB), 0, s, rho, part, g.xd, g.yd, g.zd, g.ay, g.az, n,
                           chunk);
        MMS_HIP(hipGetLastError());
    }
    {
        KTimer kt(prof, K_DIRECT_REDUCE);
        const double scale = (double)(g.dx * g.dy * g.dz) / (double)g.dx;
        hipLaunchKernelGGL(direct_reduce_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, part, phi, n,
                           nchunk, scale);
        MMS_HIP(hipGetLastError());
    }
    return 0;
}

int direct_potential(const Grid &g, DirectPlan &plan, const float *rho, float *phi, hipStream_t s,
                     Profiler *prof) {
    MMS_CHECK(plan.table != nullptr || plan.work != nullptr, "direct solver plan not initialised");
    if (plan.form == kDirectChunks)
        return direct_launch(g, plan.chunk, plan.nchunk, static_cast<double *>(plan.work), rho, phi, s, prof);
    KTimer kt(prof, K_DIRECT);
    if (plan.form == kDirectTable)
        return small_potential(g, static_cast<const float *>(plan.table), nullptr, nullptr, rho, phi, s);
    return direct_fft_potential(g, plan.table, plan.work, nullptr, const_cast<float *>(rho), phi, s);
}

int direct_potential_of(const Grid &g, DirectPlan &plan, const float *m, float *rho, float *phi, hipStream_t s,
                        Profiler *prof) {
    MMS_CHECK(plan.table != nullptr || plan.work != nullptr, "direct solver plan not initialised");
    // the other forms' charges are read with 32-bit byte offsets and divide by div_by
    const bool own = 12 * g.n() < (1L << 31) && div_by_ok(g.dx) && div_by_ok(g.dy) && div_by_ok(g.dz);
    if (plan.form == kDirectChunks || !own) {
        if (launch_div(g, m, rho, s, prof)) return 1;
        return direct_potential(g, plan, rho, phi, s, prof);
    }
    KTimer kt(prof, K_DIRECT);
    if (plan.form == kDirectTable)
        return small_potential(g, static_cast<const float *>(plan.table), m, rho, nullptr, phi, s);
    return direct_fft_potential(g, plan.table, plan.work, m, rho, phi, s);
}

// Device address of this GPU's `scratch`, looked up once per device with
// that device current (the host-side name of a __device__ array is not a
// device address).
static int scratch_ptr(double **out) {
    static std::mutex mu;
    static double *ptr[64] = {nullptr};
    int dev = 0;
    MMS_HIP(hipGetDevice(&dev));
    MMS_CHECK(dev >= 0 && dev < 64, "device index out of range");
    std::lock_guard<std::mutex> lk(mu);
    if (!ptr[dev]) {
        void *p = nullptr;
        MMS_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        MMS_CHECK(p != nullptr, "no device address for the direct-sum scratch");
        ptr[dev] = static_cast<double *>(p);
    }
    *out = ptr[dev];
    return 0;
}

int direct_probes_f64(const Grid &g, const float *rho, const int64_t *probes, int np, double *out,
                      hipStream_t s, Profiler *prof) {
    if (np <= 0) return 0;
    const long n = g.n();
    const int nbp = (np + 255) / 256;
    int nchunk = 2048 / nbp;
    if (nchunk < 1) nchunk = 1;
    if (nchunk > 64) nchunk = 64;
    long chunk = (n + nchunk - 1) / nchunk;
    chunk = ((chunk + TILE - 1) / TILE) * TILE;
    nchunk = (int)((n + chunk - 1) / chunk);
    double *part = nullptr;
    MMS_HIP(hipMalloc(&part, sizeof(double) * (size_t)nchunk * np));
    int st = 0;
    {
        KTimer kt(prof, K_PROBES);
        hipLaunchKernelGGL(probes_f64_kernel, dim3(nbp, nchunk), dim3(256), 0, s, rho, probes, part, np, g.xd, g.yd,
                           g.zd, (double)g.dx, (double)g.dy, (double)g.dz, chunk);
        if (hipGetLastError() != hipSuccess) st = 1;
        if (!st) {
            hipLaunchKernelGGL(probes_f64_reduce_kernel, dim3(nbp), dim3(256), 0, s, part, out, np, nchunk,
                               (double)g.dx * (double)g.dy * (double)g.dz);
            if (hipGetLastError() != hipSuccess) st = 1;
        }
    }
    if (hipStreamSynchronize(s) != hipSuccess) st = 1;
    (void)hipFree(part);
    MMS_CHECK(st == 0, "probe kernel launch failed");
    return 0;
}

}  // namespace mms

// Direct-sum potential from device arrays without any allocation: tables,
// work arrays or chunk partial sums live in the file-scope `scratch` array of
// each GPU; the form, kernels and chunking are those of calc_potential_exact,
// so the results are the same bit for bit.  Calls that overlap on one GPU
// share `scratch` and race.  Every value is written before it is read, so
// nothing has to be cleared between calls.
extern "C" int mms_potential_exact_noalloc(const float *charge_dev, float *potential_dev, int xdim, int ydim,
                                           int zdim, float dx, float dy, float dz, void *stream) {
    using namespace mms;
    MMS_CHECK(charge_dev && potential_dev, "null device array");
    MMS_CHECK(xdim > 0 && ydim > 0 && zdim > 0, "grid dimensions must be positive");
    MMS_CHECK(dx > 0 && dy > 0 && dz > 0, "cell sizes must be positive");
    Grid g;
    g.xd = xdim; g.yd = ydim; g.zd = zdim;
    g.dx = dx; g.dy = dy; g.dz = dz;
    g.ay = dy / dx; g.az = dz / dx;
    const long n = g.n();
    if (n > kScratchCells) {
        set_error("mms_potential_exact_noalloc: grid of " + std::to_string(n) + " cells exceeds the scratch (at most " +
                  std::to_string(kScratchCells) + " cells)");
        return 1;
    }
    double *mem = nullptr;
    if (scratch_ptr(&mem)) return 1;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const DirectForm form = direct_form(g);
    if (form == kDirectTable) {
        float *tab = reinterpret_cast<float *>(mem);
        if (small_table(g, tab, s)) return 1;
        return small_potential(g, tab, nullptr, nullptr, charge_dev, potential_dev, s);
    }
    if (form == kDirectFft) {
        const size_t tb = direct_fft_table_bytes(g);
        MMS_CHECK(tb + direct_fft_work_bytes(g) <= kScratchBytes, "mms_potential_exact_noalloc: scratch too small");
        void *work = reinterpret_cast<char *>(mem) + tb;
        return direct_fft_potential_once(g, mem, work, charge_dev, potential_dev, s);
    }
    long chunk = 0;
    int nchunk = 0;
    direct_chunks(n, 1, &chunk, &nchunk);
    MMS_CHECK(sizeof(double) * (size_t)(n * nchunk) <= kScratchBytes, "mms_potential_exact_noalloc: scratch too small");
    return direct_launch(g, chunk, nchunk, mem, charge_dev, potential_dev, s, nullptr);
}
