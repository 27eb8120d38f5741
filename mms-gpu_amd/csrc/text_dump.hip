// text_dump.hip -- the time loop's vector dump (helper_functions.cpp:107-123:
// "%g %g %g \n" a cell in z, x, y order) formatted on the GPU.
//
// The dump of every accepted step is the most expensive part of the loop on
// the host: three numbers a cell through printf take 2 us a cell, 25 times
// the step itself on a 64 x 64 x 3 film.  Here a thread splits the three
// numbers of its line into digits and lengths (text_format.hpp, glibc's bytes), the
// workgroup scans the lengths, writes its 256 lines packed into LDS and
// copies them out; the host appends the workgroups' pieces to the file while
// the next step runs.  time_marching of a 64 x 64 x 3 film to 3e-14 s (about 27
// accepted steps): 91 -> 11 ms a call, with one wait for the device a step
// instead of five.
#include "mms_internal.hpp"
#include "text_format.hpp"

namespace mms {
namespace {

static __device__ const Pow10 kPow10[] = {MMS_POW10_ROWS};

constexpr int kLineMax = 3 * 12 + 4;  // "-1.17549e-38 " three times, and the newline
constexpr int kBlockLines = 256, kBlockBytes = kBlockLines * kLineMax;

__global__ __launch_bounds__(kBlockLines) void text_kernel(const float *__restrict__ m, long line0, long n, int xd,
                                                           int yd, char *__restrict__ out, int *__restrict__ len) {
    __shared__ __attribute__((aligned(16))) char text[kBlockBytes];
    __shared__ int wsum[kBlockLines / 64];
    const long i = line0 + (long)blockIdx.x * kBlockLines + threadIdx.x;
    GNum g[3];
    int l = 0;
    if (i < n) {
        const int y = (int)(i % yd);
        const long r = i / yd, z = r / xd, c = (z * yd + y) * (long)xd + r % xd;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            g[k] = g_split(m[(long)k * n + c], kPow10);
            l += g_length(g[k]) + 1;
        }
        l++;
    }
    // exclusive scan of the line lengths over the workgroup
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int s = l;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int v = __shfl_up(s, d);
        if (lane >= d) s += v;
    }
    if (lane == 63) wsum[w] = s;
    __syncthreads();
    int base = s - l, total = 0;
#pragma unroll
    for (int k = 0; k < kBlockLines / 64; k++) {
        if (k < w) base += wsum[k];
        total += wsum[k];
    }
    if (i < n) {
        char *o = text + base;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            g_write(g[k], o);
            o += g_length(g[k]);
            *o++ = ' ';
        }
        *o = '\n';
    }
    __syncthreads();
    int4 *dst = reinterpret_cast<int4 *>(out + (long)blockIdx.x * kBlockBytes);
    for (int e = threadIdx.x; e < (total + 15) / 16; e += kBlockLines) dst[e] = reinterpret_cast<const int4 *>(text)[e];
    if (threadIdx.x == 0) len[blockIdx.x] = total;
}

}  // namespace

int TextDump::init(const Grid &g_) {
    release();
    g = g_;
    blocks = (g.n() + kBlockLines - 1) / kBlockLines;
    cap = blocks < 256 ? blocks : 256;
    const size_t bytes = (size_t)cap * kBlockBytes + sizeof(int) * cap;
    MMS_HIP(hipMalloc(&dev, bytes));
    if (host.alloc(bytes)) return 1;
    MMS_HIP(hipEventCreateWithFlags(&copied, hipEventDisableTiming));
    return 0;
}

void TextDump::release() {
    if (dev) (void)hipFree(dev);
    host.release();
    if (copied) (void)hipEventDestroy(copied);
    dev = nullptr;
    copied = nullptr;
    blocks = cap = 0;
}

// formats blocks first .. first + cap - 1 of the state m and copies the text to the host
int TextDump::enqueue(const float *m, long first, hipStream_t s) {
    const long nb = blocks - first < cap ? blocks - first : cap;
    int *len = reinterpret_cast<int *>(dev + (size_t)cap * kBlockBytes);
    hipLaunchKernelGGL(text_kernel, dim3((unsigned)nb), dim3(kBlockLines), 0, s, m, first * kBlockLines, g.n(), g.xd, g.yd,
                       dev, len);
    MMS_HIP(hipGetLastError());
    MMS_HIP(hipMemcpyAsync(host.p, dev, (size_t)cap * kBlockBytes + sizeof(int) * nb, hipMemcpyDeviceToHost, s));
    MMS_HIP(hipEventRecord(copied, s));
    return 0;
}

// waits for the blocks enqueued last and appends them to the file
int TextDump::write(FILE *fh, long first) const {
    MMS_HIP(hipEventSynchronize(copied));
    const long nb = blocks - first < cap ? blocks - first : cap;
    const int *len = reinterpret_cast<const int *>(host.p + (size_t)cap * kBlockBytes);
    for (long b = 0; b < nb; b++) fwrite(host.p + b * kBlockBytes, 1, len[b], fh);
    return 0;
}

}  // namespace mms
