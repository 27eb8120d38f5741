// direct_fft.hip -- the exact pair potential of large regular grids on gfx950
// by FP64 transforms.
//
//   phi_i = (dV/dx) sum_{j != i} rho_j / |r_i - r_j|_u
//
// is a convolution on the grid (fmm_calc.cu:412-461 sums it pair by pair), so
// the sum over the N^2 pairs is one zero-padded 2D transform per layer, a
// zd x zd real product per frequency and the transform back.  Everything
// between the FP32 charges and the FP32 potential is FP64: the error (about
// 1e-15 of the largest potential) is far below the pair loop's FP32 sums.
//
// Three launches (Stockham FFTs in LDS, eight elements a thread, radix 8 with
// one radix-2 or -4 pass; W[z][kx][y] is stored transposed so that every pass
// reads and writes runs of consecutive y):
//   fft_rows     charges (or div M formed in place of the charge kernel) ->
//                x transforms, two real rows per complex transform;
//   fft_columns  one kx per workgroup: y transforms of every layer, product
//                with the kernel's spectrum, inverse y transforms, in place;
//   fft_back     inverse x transforms, two real rows each, FP32 potential.
// A call that keeps no tables forms them in the first two (fft_rows_tables,
// fft_columns<.., true>): three more launches before them took 12 of 26 us on
// 33 x 32 x 6 (now 15; the pair loop 23) and 9 of 37 on 1300 x 5 x 1, where
// the padded length is 40 times the film (now 28; 23).
// Measured against the pair loop (FP32 rsqrt pairs, 3.8e12 a second): the
// 256 x 256 x 3 potential on host arrays 9.46 -> 0.11 ms, an RK4 step of a
// 161 x 117 x 3 film 3.67 -> 0.086 ms (fft_rows 6.8 us with div M, fft_columns
// 6.4 us, fft_back 4.6 us an evaluation: launch and load latency at this
// size, so all that a thread loads, twiddles and kernel spectrum too, is
// requested before the first barrier and none behind a branch; one after the
// other where needed they took 8.9, 7.0 and 5.4 us, a step 106);
// relative error against 64 bits 5.8e-7 -> 2.5e-8.
// A charge that is not finite would spread through the transforms; fft_rows
// notes it and fft_back then sums that call pair by pair.
#include "div_by.hpp"
#include "mms_internal.hpp"

namespace mms {
namespace {

typedef double2 cd;

constexpr int kTw = 4096;  // entries of the twiddle table, the longest transform

// Several kernels run the same transform, and their results must not depend on
// which one: no multiply-adds but the written ones.
#pragma clang fp contract(off)

__device__ __forceinline__ cd cmul(cd a, cd b) {
    return make_double2(fma(-a.y, b.y, a.x * b.x), fma(a.x, b.y, a.y * b.x));
}
__device__ __forceinline__ cd cadd(cd a, cd b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ cd csub(cd a, cd b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ cd cfma(double h, cd a, cd b) { return make_double2(fma(h, a.x, b.x), fma(h, a.y, b.y)); }
__device__ __forceinline__ cd mul_mi(cd a) { return make_double2(a.y, -a.x); }  // -i a

// LDS slot of element i: one free slot in nine keeps the strided stores of
// the passes on different banks
__device__ __forceinline__ int slot(int i) { return i + (i >> 3); }
constexpr int slots(int n) { return n + (n >> 3); }

__device__ __forceinline__ void dft4(cd &a, cd &b, cd &c, cd &d) {
    const cd s = cadd(a, c), u = csub(a, c), v = cadd(b, d), w = mul_mi(csub(b, d));
    a = cadd(s, v); b = cadd(u, w); c = csub(s, v); d = csub(u, w);
}

template <int R>
__device__ __forceinline__ void dft(cd (&v)[R]) {
    if constexpr (R == 2) {
        const cd a = v[0];
        v[0] = cadd(a, v[1]);
        v[1] = csub(a, v[1]);
    } else if constexpr (R == 4) {
        dft4(v[0], v[1], v[2], v[3]);
    } else {
        const double h = 0.70710678118654752440;  // sqrt(1/2)
        dft4(v[0], v[2], v[4], v[6]);
        dft4(v[1], v[3], v[5], v[7]);
        // w_8 v = h t1, w_8^2 v = t2, w_8^3 v = h t3
        const cd t1 = make_double2(v[3].x + v[3].y, v[3].y - v[3].x), t2 = mul_mi(v[5]);
        const cd t3 = make_double2(v[7].y - v[7].x, -(v[7].x + v[7].y));
        const cd e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6], o0 = v[1];
        v[0] = cadd(e0, o0); v[4] = csub(e0, o0);
        v[1] = cfma(h, t1, e1); v[5] = cfma(-h, t1, e1);
        v[2] = cadd(e2, t2); v[6] = csub(e2, t2);
        v[3] = cfma(h, t3, e3); v[7] = cfma(-h, t3, e3);
    }
}

// One Stockham pass of radix R after sub-transforms of length NS; thread t of
// the transform's N / 8, w its twiddle (radix 8; the passes before have none).
template <int N, int R, int NS>
__device__ __forceinline__ void fft_pass(cd *buf, int t, cd w) {
    static_assert(NS == 1 || R == 8, "one twiddle a thread");
    constexpr int Q = 8 / R;
    cd v[Q][R];
#pragma unroll
    for (int b = 0; b < Q; b++) {
#pragma unroll
        for (int k = 0; k < R; k++) v[b][k] = buf[slot(t + b * (N / 8) + k * (N / R))];
        if constexpr (NS > 1) {
            const cd w1 = w;
            v[b][1] = cmul(v[b][1], w1);
            if constexpr (R > 2) {
                const cd w2 = cmul(w1, w1), w3 = cmul(w2, w1);
                v[b][2] = cmul(v[b][2], w2);
                v[b][3] = cmul(v[b][3], w3);
                if constexpr (R > 4) {
                    const cd w4 = cmul(w2, w2);
                    v[b][4] = cmul(v[b][4], w4);
                    v[b][5] = cmul(v[b][5], cmul(w4, w1));
                    v[b][6] = cmul(v[b][6], cmul(w3, w3));
                    v[b][7] = cmul(v[b][7], cmul(w4, w3));
                }
            }
        }
        dft<R>(v[b]);
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < Q; b++) {
        const int j = t + b * (N / 8), jm = j & (NS - 1), base = (j - jm) * R + jm;
#pragma unroll
        for (int k = 0; k < R; k++) buf[slot(base + k * NS)] = v[b][k];
    }
    __syncthreads();
}

// First radix of a transform (its other passes are radix 8) and its twiddles, loaded
// with the kernels' other first loads: in the passes each would be waited
// for between two barriers.
template <int N>
constexpr int first_radix() { return __builtin_ctz(N) % 3 == 1 ? 2 : (__builtin_ctz(N) % 3 == 2 ? 4 : 8); }
// FORM: formed instead, by the expression that fills the table.
struct Twiddles { cd w[4]; };
__device__ __forceinline__ cd twiddle(int i) {
    double s, c;
    sincospi(-2.0 * (double)i / (double)kTw, &s, &c);
    return make_double2(c, s);
}
template <int N, bool FORM = false>
__device__ __forceinline__ Twiddles fft_twiddles(int t, const cd *__restrict__ tw) {
    Twiddles r;
#pragma unroll
    for (int p = 0, ns = first_radix<N>(); p < 4; p++, ns *= 8) {
        const int i = (t & (ns - 1)) * (kTw / (ns * 8));
        r.w[p] = ns < N ? (FORM ? twiddle(i) : tw[i]) : make_double2(0.0, 0.0);
    }
    return r;
}
template <int N, int NS, int P>
__device__ __forceinline__ void fft_rest(cd *buf, int t, const Twiddles &tw) {
    if constexpr (NS < N) {
        fft_pass<N, 8, NS>(buf, t, tw.w[P]);
        fft_rest<N, NS * 8, P + 1>(buf, t, tw);
    }
}

// Forward transform of buf[slot(0 .. N-1)], N a power of two >= 64; called
// by every thread of the workgroup (the inverse: re and im swapped before
// and after).
template <int N>
__device__ __forceinline__ void fft(cd *buf, int t, const Twiddles &tw) {
    constexpr int R = first_radix<N>();
    fft_pass<N, R, 1>(buf, t, make_double2(1.0, 0.0));
    fft_rest<N, R, 0>(buf, t, tw);
}

// transforms per workgroup of the row kernels: at least a wave of threads
// and, up to 2048 points, at least four consecutive rows (64-byte runs of W)
template <int N>
constexpr int row_batch() { return N >= 4096 ? 1 : (N >= 256 ? 2 : 512 / N); }

struct FftArgs {
    const float *rho;  // charges (fft_back's pair sum too)
    float *rho_out;    // charges formed from m (fft_rows<N, true>)
    const float *m;    // FP32 SoA magnetisation
    float *phi;
    cd *w;             // [zd][nxh][yd]
    double *ghat;      // [zd][nxh][ny / 2 + 1]; before its y transforms [zd][nxh][|dy|]
    const cd *tw;
    int *flags;        // [workgroups of fft_rows], then the combined flag
    int nflags;
    int xd, yd, zd, nxh, ny;
    float dx, dy, dz, ay, az;
    double scale;
    double ayd, azd, gscale;  // of the kernel's spectrum
};

// workgroups of a layer's rows of charges
template <int N>
__device__ __forceinline__ int row_groups(int yd) { return (yd + 2 * row_batch<N>() - 1) / (2 * row_batch<N>()); }

// rows 2 B bx .. of layer z
template <int N, bool FROM_M, bool FORM>
__device__ __forceinline__ void rows_of(const FftArgs A, cd *lds, int bx, int z) {
    constexpr int B = row_batch<N>(), T = N / 8;
    const int f = threadIdx.x / T, t = threadIdx.x % T;
    const int y0 = bx * 2 * B, ya = y0 + 2 * f;
    const long plane = (long)A.xd * A.yd, n = plane * A.zd;
    const long row = (long)z * plane + (long)ya * A.xd;
    const Twiddles tw = fft_twiddles<N, FORM>(t, A.tw);
    bool bad = false;
    // the rows' upper half is padding (xd <= N / 2).  Every load of a thread is
    // issued before one is used: none sits behind a branch
    float q[8][2];
    if constexpr (FROM_M) {
        // div M by the charge kernel's expression (vector_functions.cpp:8-28);
        // buffer loads return 0 past the three planes
        const int end = 12 * (int)n;
        const __amdgpu_buffer_rsrc_t rm = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(A.m), (short)0, end, 0x00020000);
        auto ld = [&](bool ok, int i) { return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rm, ok ? 4 * i : end, 0, 0)); };
        const float rdx = 1.0f / A.dx, rdy = 1.0f / A.dy, rdz = 1.0f / A.dz;
        float v[4][2][6];
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int x = t + k * T, y = ya + h, c = (int)row + h * A.xd + x;
                const bool ok = x < A.xd && y < A.yd;
                v[k][h][0] = ld(ok && x != A.xd - 1, c + 1);
                v[k][h][1] = ld(ok && x != 0, c - 1);
                v[k][h][2] = ld(ok && y != A.yd - 1, (int)n + c + A.xd);
                v[k][h][3] = ld(ok && y != 0, (int)n + c - A.xd);
                v[k][h][4] = ld(ok && z != A.zd - 1, 2 * (int)n + c + (int)plane);
                v[k][h][5] = ld(ok && z != 0, 2 * (int)n + c - (int)plane);
            }
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const float(&u)[6] = v[k][h];
                q[k][h] = (div_by(u[0] - u[1], A.dx, rdx) + div_by(u[2] - u[3], A.dy, rdy) + div_by(u[4] - u[5], A.dz, rdz)) * 0.5f;
            }
    } else {
        float v[4][2];
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int h = 0; h < 2; h++) {  // past the film: its last cell, then 0
                const long c = row + (long)h * A.xd + t + k * T;
                v[k][h] = A.rho[c < n ? c : n - 1];
            }
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int h = 0; h < 2; h++) q[k][h] = (t + k * T < A.xd && ya + h < A.yd) ? v[k][h] : 0.0f;
    }
#pragma unroll
    for (int k = 4; k < 8; k++) q[k][0] = q[k][1] = 0.0f;
    cd *buf = lds + f * slots(N);
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const int x = t + k * T;
        if constexpr (FROM_M) {
            if (x < A.xd && ya < A.yd) A.rho_out[row + x] = q[k][0];
            if (x < A.xd && ya + 1 < A.yd) A.rho_out[row + A.xd + x] = q[k][1];
        }
        bad |= !(fabsf(q[k][0]) <= 3.402823466e38f) || !(fabsf(q[k][1]) <= 3.402823466e38f);
        buf[slot(x)] = make_double2((double)q[k][0], (double)q[k][1]);
    }
    const int any = __syncthreads_or(bad ? 1 : 0);
    if (threadIdx.x == 0) A.flags[z * row_groups<N>(A.yd) + bx] = any;
    fft<N>(buf, t, tw);
    // spectra of the two real rows of each transform: with Z = FFT(a + i b),
    // A[k] = (Z[k] + conj Z[N-k]) / 2, B[k] = (Z[k] - conj Z[N-k]) / 2i
    for (int i = threadIdx.x; i < 2 * B * (N / 2 + 1); i += B * T) {
        const int r = i % (2 * B), k = i / (2 * B), y = y0 + r;
        if (y >= A.yd) continue;
        const cd *zb = lds + (r >> 1) * slots(N);
        const cd u = zb[slot(k)], v = zb[slot((N - k) & (N - 1))];
        const cd s = (r & 1) ? make_double2(0.5 * (u.y + v.y), 0.5 * (v.x - u.x))
                             : make_double2(0.5 * (u.x + v.x), 0.5 * (u.y - v.y));
        A.w[((long)z * A.nxh + k) * A.yd + y] = s;
    }
}

template <int N, bool FROM_M>
__global__ __launch_bounds__(row_batch<N>() * N / 8) void fft_rows(FftArgs A) {
    __shared__ cd lds[row_batch<N>() * slots(N)];
    rows_of<N, FROM_M, false>(A, lds, blockIdx.x, blockIdx.y);
}

// The tables' first launch: x transforms of the rows |dy| = 0 .. ny/2 of 1/r
// (real and even in both axes) into ghat[dz][kx][|dy|] and the twiddles, by
// workgroups nbx .. of each layer; the first nbx transform the charges' rows, where a
// call forms its tables anew (nbx 0: a plan's tables).
template <int N>
__global__ __launch_bounds__(row_batch<N>() * N / 8) void fft_rows_tables(FftArgs A, cd *tw, int nbx) {
    constexpr int B = row_batch<N>(), T = N / 8;
    __shared__ cd lds[B * slots(N)];
    if ((int)blockIdx.x < nbx) {
        rows_of<N, false, true>(A, lds, blockIdx.x, blockIdx.y);
        return;
    }
    const int f = threadIdx.x / T, t = threadIdx.x % T, z = blockIdx.y, bk = blockIdx.x - nbx, nyh = A.ny / 2 + 1;
    const int y = bk * B + f;
    cd *buf = lds + f * slots(N);
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const int x = t + k * T;
        const double rx = (double)(x <= N / 2 ? x : N - x), ry = y * A.ayd, rz = z * A.azd;
        const double r2 = rx * rx + ry * ry + rz * rz;
        buf[slot(x)] = make_double2(r2 > 0.0 ? 1.0 / sqrt(r2) : 0.0, 0.0);
    }
    const int nk = gridDim.x - nbx;
    for (int i = ((int)blockIdx.y * nk + bk) * B * T + threadIdx.x; i < kTw; i += nk * gridDim.y * B * T) tw[i] = twiddle(i);
    __syncthreads();
    fft<N>(buf, t, fft_twiddles<N, true>(t, nullptr));
    for (int i = threadIdx.x; i < B * (N / 2 + 1); i += B * T) {
        const int r = i % B, k = i / B;
        if (bk * B + r < nyh) A.ghat[((long)z * A.nxh + k) * nyh + bk * B + r] = lds[r * slots(N) + slot(k)].x;
    }
}

// The tables' second launch: y transforms of the mirrored columns of
// ghat, in place and scaled; one column of N elements by its N / 8 threads.
template <int N>
__device__ __forceinline__ void kernel_column(double *col, cd *buf, int t, const Twiddles &tw, double scale) {
    constexpr int T = N / 8;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const int y = t + k * T;
        buf[slot(y)] = make_double2(col[y <= N / 2 ? y : N - y], 0.0);
    }
    __syncthreads();
    fft<N>(buf, t, tw);
    for (int k = t; k <= N / 2; k += T) col[k] = buf[slot(k)].x * scale;
}
template <int N>
__global__ __launch_bounds__(N / 8) void fft_kernel_columns(FftArgs A) {
    __shared__ cd buf[slots(N)];
    kernel_column<N>(A.ghat + ((long)blockIdx.y * A.nxh + blockIdx.x) * (N / 2 + 1), buf, threadIdx.x,
                     fft_twiddles<N>(threadIdx.x, A.tw), A.gscale);
}

// the layers' product at one (kx, ky): out[z] = sum_z' ghat[|z - z'|] in[z'];
// re and im are stored swapped (the inverse transform follows)
template <int ZD, int N>
__device__ __forceinline__ void layer_product(cd *lds, const double (&g)[ZD]) {
    cd in[ZD];
#pragma unroll
    for (int z = 0; z < ZD; z++) in[z] = lds[z * slots(N)];
#pragma unroll
    for (int z = 0; z < ZD; z++) {
        double re = 0.0, im = 0.0;
#pragma unroll
        for (int s = 0; s < ZD; s++) {
            re = fma(g[z > s ? z - s : s - z], in[s].x, re);
            im = fma(g[z > s ? z - s : s - z], in[s].y, im);
        }
        lds[z * slots(N)] = make_double2(im, re);
    }
}
// ... of zd layers, at most ZM, whose spectrum is read from memory, all of it
// at once: a load a product, each waited for, took most of the kernel (a step of a
// 20 x 20 x 16 film 145 us, so 74; 128 x 64 x 16 176 / 94; 500 x 64 x 7 161 /
// 122).  Layers past the last add 0.
template <int ZM, int N>
__device__ __forceinline__ void layers_product(cd *lds, const double *gh, long gstride, int zd) {
    cd in[ZM];
    double g[ZM];
#pragma unroll
    for (int z = 0; z < ZM; z++) {
        g[z] = gh[min(z, zd - 1) * gstride];
        in[z] = z < zd ? lds[z * slots(N)] : make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int z = 0; z < ZM; z++) {
        double re = 0.0, im = 0.0;
#pragma unroll
        for (int s = 0; s < ZM; s++) {
            re = fma(g[z > s ? z - s : s - z], in[s].x, re);
            im = fma(g[z > s ? z - s : s - z], in[s].y, im);
        }
        if (z < zd) lds[z * slots(N)] = make_double2(im, re);
    }
}

// TAB: ghat holds the kernel's rows; their columns are transformed here first
template <int N, int ZD, bool TAB>
__global__ __launch_bounds__(ZD ? ZD * N / 8 : (16 * N / 8 < 1024 ? 16 * N / 8 : 1024)) void fft_columns(FftArgs A) {
    extern __shared__ __attribute__((aligned(16))) char fft_lds[];
    cd *lds = reinterpret_cast<cd *>(fft_lds);
    constexpr int T = N / 8;
    const int z = threadIdx.x / T, t = threadIdx.x % T, kx = blockIdx.x;
    cd *col = A.w + ((long)z * A.nxh + kx) * A.yd;
    cd *buf = lds + z * slots(N);
    const Twiddles tw = fft_twiddles<N>(t, A.tw);
    if constexpr (TAB) {
        kernel_column<N>(A.ghat + ((long)z * A.nxh + kx) * (N / 2 + 1), buf, t, tw, A.gscale);
        __syncthreads();  // the layers' spectra are read below, buf is written again
    }
    // the column's upper half is padding (yd <= N / 2); past yd its last entry, then 0
    cd v[4];
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = col[min(t + k * T, A.yd - 1)];
    const long gs = (long)A.nxh * (N / 2 + 1);
    // this thread's kernel spectrum, in flight during the first transform
    constexpr int NI = ZD ? (8 + ZD - 1) / ZD : 1;
    double g[NI][ZD ? ZD : 1];
    auto spectrum = [&](int ky) -> const double * { return A.ghat + (long)kx * (N / 2 + 1) + (ky <= N / 2 ? ky : N - ky); };
    if constexpr (ZD != 0) {
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const double *gh = spectrum(min((int)threadIdx.x + i * ZD * T, N - 1));
#pragma unroll
            for (int s = 0; s < ZD; s++) g[i][s] = gh[s * gs];
        }
    }
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const int y = t + k * T;
        buf[slot(y)] = k < 4 && y < A.yd ? v[k & 3] : make_double2(0.0, 0.0);
    }
    if (kx == 0) {  // one flag for fft_back
        int any = 0;
        for (int i = threadIdx.x; i < A.nflags; i += blockDim.x) any |= A.flags[i];
        any = __syncthreads_or(any);
        if (threadIdx.x == 0) A.flags[A.nflags] = any;
    }
    __syncthreads();
    fft<N>(buf, t, tw);
    if constexpr (ZD != 0) {
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const int ky = threadIdx.x + i * ZD * T;
            if (ky < N) layer_product<ZD, N>(lds + slot(ky), g[i]);
        }
    } else {
        for (int ky = threadIdx.x; ky < N; ky += blockDim.x) {
            if (A.zd <= 8) layers_product<8, N>(lds + slot(ky), spectrum(ky), gs, A.zd);
            else layers_product<16, N>(lds + slot(ky), spectrum(ky), gs, A.zd);
        }
    }
    __syncthreads();
    fft<N>(buf, t, tw);
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int y = t + k * T;
        if (y < A.yd) {
            const cd v = buf[slot(y)];
            col[y] = make_double2(v.y, v.x);
        }
    }
}

// the pair sum of one target (charges that are not finite): as the pair
// kernels form it, FP32 over 256 sources, FP64 across
__device__ double pair_sum(const FftArgs &A, int xt, int yt, int zt) {
    const long n = (long)A.xd * A.yd * A.zd;
    double acc = 0.0;
    int xs = 0, ys = 0, zs = 0;
    for (long base = 0; base < n; base += 256) {
        const long end = base + 256 < n ? base + 256 : n;
        float s = 0.0f;
        for (long j = base; j < end; j++) {
            const float rx = (float)(xt - xs), ry = (float)(yt - ys) * A.ay, rz = (float)(zt - zs) * A.az;
            const float r2 = rx * rx + ry * ry + rz * rz;
            s = fmaf(A.rho[j], r2 > 0.f ? __builtin_amdgcn_rsqf(r2) : 0.f, s);
            if (++xs == A.xd) { xs = 0; if (++ys == A.yd) { ys = 0; zs++; } }
        }
        acc += (double)s;
    }
    return acc * A.scale;
}

template <int N>
__global__ __launch_bounds__(row_batch<N>() * N / 8) void fft_back(FftArgs A) {
    constexpr int B = row_batch<N>(), T = N / 8;
    __shared__ cd lds[B * slots(N)];
    const int f = threadIdx.x / T, t = threadIdx.x % T;
    const int z = blockIdx.y, y0 = blockIdx.x * 2 * B, ya = y0 + 2 * f;
    const long row = ((long)z * A.yd + ya) * A.xd;
    const Twiddles tw = fft_twiddles<N>(t, A.tw);
    // the rows' spectra, four k a thread and k = N / 2 by the first ones; past yd the last row's, then 0
    auto load = [&](int i, cd &u, cd &v) {
        const int y = y0 + 2 * (i % B);
        const cd *p = A.w + ((long)z * A.nxh + i / B) * A.yd;
        u = p[min(y, A.yd - 1)];
        v = p[min(y + 1, A.yd - 1)];
    };
    cd u[4], v[4];
#pragma unroll
    for (int q = 0; q < 4; q++) load(threadIdx.x + q * B * T, u[q], v[q]);
    if (A.flags[A.nflags]) {
        for (int h = 0; h < 2; h++)
            for (int x = t; x < A.xd; x += T)
                if (ya + h < A.yd) A.phi[row + (long)h * A.xd + x] = (float)pair_sum(A, x, ya + h, z);
        return;
    }
    auto put = [&](int i, cd u, cd v) {
        const int r = i % B, k = i / B, y = y0 + 2 * r;
        if (y >= A.yd) u = make_double2(0.0, 0.0);
        if (y + 1 >= A.yd) v = make_double2(0.0, 0.0);
        cd *zb = lds + r * slots(N);
        // Z[k] = U + i V, Z[N-k] = conj(U) + i conj(V), re and im swapped
        zb[slot(k)] = make_double2(u.y + v.x, u.x - v.y);
        if (k > 0 && k < N / 2) zb[slot(N - k)] = make_double2(v.x - u.y, u.x + v.y);
    };
#pragma unroll
    for (int q = 0; q < 4; q++) put(threadIdx.x + q * B * T, u[q], v[q]);
    if (threadIdx.x < B) {
        cd ul, vl;
        load(threadIdx.x + 4 * B * T, ul, vl);
        put(threadIdx.x + 4 * B * T, ul, vl);
    }
    __syncthreads();
    cd *buf = lds + f * slots(N);
    fft<N>(buf, t, tw);
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int x = t + k * T;
        if (x < A.xd) {
            const cd v = buf[slot(x)];
            if (ya < A.yd) A.phi[row + x] = (float)v.y;
            if (ya + 1 < A.yd) A.phi[row + A.xd + x] = (float)v.x;
        }
    }
}

int fft_len(int d) {
    int n = 64;
    while (n < 2 * d - 1) n <<= 1;
    return n;
}

#define MMS_FFT_SIZES(X, n, ...)                                                    \
    switch (n) {                                                                    \
    case 64: X(64, __VA_ARGS__); break;                                            \
    case 128: X(128, __VA_ARGS__); break;                                          \
    case 256: X(256, __VA_ARGS__); break;                                          \
    case 512: X(512, __VA_ARGS__); break;                                          \
    case 1024: X(1024, __VA_ARGS__); break;                                        \
    case 2048: X(2048, __VA_ARGS__); break;                                        \
    case 4096: X(4096, __VA_ARGS__); break;                                        \
    default: set_error("direct sum: transform length"); return 1;                  \
    }

template <int N>
int launch_rows(const FftArgs &A, bool from_m, hipStream_t s) {
    constexpr int B = row_batch<N>();
    dim3 grid((A.yd + 2 * B - 1) / (2 * B), A.zd);
    if (from_m)
        hipLaunchKernelGGL((fft_rows<N, true>), grid, dim3(B * N / 8), 0, s, A);
    else
        hipLaunchKernelGGL((fft_rows<N, false>), grid, dim3(B * N / 8), 0, s, A);
    MMS_HIP(hipGetLastError());
    return 0;
}

// the tables, with the charges' rows if the call has any
template <int N>
int launch_rows_tables(const FftArgs &A, cd *tw, bool charges, hipStream_t s) {
    constexpr int B = row_batch<N>();
    const int nbx = charges ? (A.yd + 2 * B - 1) / (2 * B) : 0;
    hipLaunchKernelGGL((fft_rows_tables<N>), dim3(nbx + (A.ny / 2 + B) / B, A.zd), dim3(B * N / 8), 0, s, A, tw, nbx);
    MMS_HIP(hipGetLastError());
    return 0;
}

template <int N, int ZD, bool TAB>
int launch_columns_z(const FftArgs &A, hipStream_t s) {
    if constexpr (ZD * N <= 8192) {
        // The limit is the kernel's, not this call's: callers of other depths
        // share it.  Set on every call (a host-side table write) rather than
        // remembered per device.
        constexpr int layers = ZD ? ZD : (8192 / N < 16 ? 8192 / N : 16);
        const size_t lds = sizeof(cd) * (size_t)A.zd * slots(N);
        MMS_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&fft_columns<N, ZD, TAB>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)(sizeof(cd) * layers * slots(N))));
        hipLaunchKernelGGL((fft_columns<N, ZD, TAB>), dim3(A.nxh), dim3(A.zd * (N / 8)), lds, s, A);
        MMS_HIP(hipGetLastError());
        return 0;
    } else {
        set_error("direct sum: transforms exceed LDS");
        return 1;
    }
}

template <int N, bool TAB>
int launch_columns(const FftArgs &A, hipStream_t s) {
    switch (A.zd) {
    case 1: return launch_columns_z<N, 1, TAB>(A, s);
    case 2: return launch_columns_z<N, 2, TAB>(A, s);
    case 3: return launch_columns_z<N, 3, TAB>(A, s);
    case 4: return launch_columns_z<N, 4, TAB>(A, s);
    default: return launch_columns_z<N, 0, TAB>(A, s);
    }
}

template <int N>
int launch_back(const FftArgs &A, hipStream_t s) {
    constexpr int B = row_batch<N>();
    dim3 grid((A.yd + 2 * B - 1) / (2 * B), A.zd);
    hipLaunchKernelGGL((fft_back<N>), grid, dim3(B * N / 8), 0, s, A);
    MMS_HIP(hipGetLastError());
    return 0;
}

int row_blocks(int nx, const Grid &g) {
    const int b = nx >= 4096 ? 1 : (nx >= 256 ? 2 : 512 / nx);
    return ((g.yd + 2 * b - 1) / (2 * b)) * g.zd;
}

}  // namespace

bool direct_fft_fits(const Grid &g) {
    // transforms of at most 4096 points, layers of one kx together in LDS
    // (16 bytes x zd x 9/8 ny <= 147 KB)
    return g.xd <= 2048 && g.yd <= 2048 && g.zd <= 16 && (long)g.zd * fft_len(g.yd) <= 8192;
}

// bytes of the tables (kept by a plan) and of the work arrays; both 256-byte multiples
size_t direct_fft_table_bytes(const Grid &g) {
    const size_t nxh = fft_len(g.xd) / 2 + 1, nyh = fft_len(g.yd) / 2 + 1;
    return (sizeof(cd) * kTw + sizeof(double) * g.zd * nxh * nyh + 255) & ~(size_t)255;
}
size_t direct_fft_work_bytes(const Grid &g) {
    const int nx = fft_len(g.xd);
    return (sizeof(cd) * g.zd * (nx / 2 + 1) * g.yd + sizeof(int) * (row_blocks(nx, g) + 1) + 255) & ~(size_t)255;
}

static FftArgs fft_args(const Grid &g, void *table, void *work) {
    const int nx = fft_len(g.xd), ny = fft_len(g.yd);
    FftArgs A{};
    A.tw = static_cast<const cd *>(table);
    A.ghat = reinterpret_cast<double *>(static_cast<cd *>(table) + kTw);
    A.w = static_cast<cd *>(work);
    A.xd = g.xd; A.yd = g.yd; A.zd = g.zd; A.nxh = nx / 2 + 1; A.ny = ny;
    A.flags = reinterpret_cast<int *>(A.w + (size_t)g.zd * A.nxh * g.yd);
    A.nflags = row_blocks(nx, g);
    A.dx = g.dx; A.dy = g.dy; A.dz = g.dz; A.ay = g.ay; A.az = g.az;
    A.scale = (double)g.dy * (double)g.dz;
    A.ayd = (double)g.dy / (double)g.dx;
    A.azd = (double)g.dz / (double)g.dx;
    A.gscale = A.scale / ((double)nx * (double)ny);
    return A;
}

int direct_fft_tables(const Grid &g, void *table, hipStream_t s) {
    const FftArgs A = fft_args(g, table, nullptr);
    cd *tw = static_cast<cd *>(table);
#define X(N, ...) \
    if (launch_rows_tables<N>(A, tw, false, s)) return 1
    MMS_FFT_SIZES(X, 2 * (A.nxh - 1), 0)
#undef X
#define X(N, ...) hipLaunchKernelGGL((fft_kernel_columns<N>), dim3(A.nxh, A.zd), dim3(N / 8), 0, s, A)
    MMS_FFT_SIZES(X, A.ny, 0)
#undef X
    MMS_HIP(hipGetLastError());
    return 0;
}

static int fft_back_of(const FftArgs &A, hipStream_t s) {
#define X(N, ...) \
    if (launch_back<N>(A, s)) return 1
    MMS_FFT_SIZES(X, 2 * (A.nxh - 1), 0)
#undef X
    return 0;
}

int direct_fft_potential(const Grid &g, const void *table, void *work, const float *m, float *rho, float *phi,
                         hipStream_t s) {
    FftArgs A = fft_args(g, const_cast<void *>(table), work);
    A.rho = rho; A.rho_out = rho; A.m = m; A.phi = phi;
#define X(N, ...) \
    if (launch_rows<N>(A, m != nullptr, s)) return 1
    MMS_FFT_SIZES(X, 2 * (A.nxh - 1), 0)
#undef X
#define X(N, ...) \
    if (launch_columns<N, false>(A, s)) return 1
    MMS_FFT_SIZES(X, A.ny, 0)
#undef X
    return fft_back_of(A, s);
}

int direct_fft_potential_once(const Grid &g, void *table, void *work, const float *rho, float *phi, hipStream_t s) {
    FftArgs A = fft_args(g, table, work);
    A.rho = rho; A.phi = phi;
    cd *tw = static_cast<cd *>(table);
#define X(N, ...) \
    if (launch_rows_tables<N>(A, tw, true, s)) return 1
    MMS_FFT_SIZES(X, 2 * (A.nxh - 1), 0)
#undef X
#define X(N, ...) \
    if (launch_columns<N, true>(A, s)) return 1
    MMS_FFT_SIZES(X, A.ny, 0)
#undef X
    return fft_back_of(A, s);
}

}  // namespace mms
