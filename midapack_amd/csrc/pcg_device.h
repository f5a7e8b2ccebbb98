// pcg_device.h -- device-side helpers shared by the PCG kernels (pcg.hip)
// and the two-level preconditioner (twolvl.hip): per-segment scalar slots,
// stop flags, workgroup reductions in a fixed order and the map-domain
// workgroup -> (segment, pixel) mapping.
#pragma once
#include "mgpu_internal.h"

namespace mgpu {

// scalar slots of one segment in d_scal (segment r at r * S_NSCAL)
enum {
    S_G2PIX = 0,
    S_RES,
    S_RES0,
    S_TOL2,
    S_RO,
    S_GAMMA,
    S_COEFF,
    S_POLAK,
    S_G2PIXP,   // g2pix of the iteration before (fused sums: the two slots alternate)
    S_K,        // iteration counter (as double)
    S_TOL,
    S_STOPK,    // stop_after (0 = off)
    S_MAXK,
    S_TRUE_R2,  // ||b - A x||^2 of the returned x (mixed precision)
    S_TRUE_B2,  // ||b||^2
    S_PEND,     // mixed precision: 1 while an FP32-updated residual of this segment
                // met the stop test (or, with adaptive refreshes, drifted far enough
                // from its last FP64 value) and awaits its FP64 refresh
    S_RREF,     // adaptive refreshes: ||g||^2 of the last FP64 residual
    S_KREF,     // adaptive refreshes: iteration of the last FP64 residual
    S_NSCAL = 18
};

// Adaptive refreshes (MGPU_REFRESH_ADAPTIVE): a segment asks for an FP64
// residual once its FP32-updated ||g||^2 has fallen below kAdaptDrop times the
// last FP64 one (the norm by 10x), or kAdaptGap iterations after it.  The
// recurrence's drift grows with the largest residual since the last
// replacement, so replacing it at every decade keeps the drift a small
// fraction of the current residual (reliable updates, Sleijpen and van der
// Vorst 1996).
constexpr double kAdaptDrop = 1e-2;
constexpr double kAdaptGap = 64.0;

// device flags: [0] every segment stopped, [1] segment 0 converged, [2] largest
// iteration count reached, [3] number of stopped segments, [4] never set,
// [5] number of segments whose FP32-updated residual met the stop test
// (mixed precision: S_PEND set; the first iteration of the next block
// refreshes their residual in FP64 and tests it), [6] FP64 residual refreshes
// performed
enum { F_STOP = 0, F_CONV0, F_KMAX, F_NDONE, F_NEVER = 4, F_NPEND = 5, F_NREF = 6, F_NFLAGS = 8 };

// iteration kinds of k_scalars / k_refresh: FP64 solve; mixed precision without
// a refresh; every live segment refreshed in FP64 (every refresh_every
// iterations); only the segments with S_PEND set refreshed
enum { IT_FP64 = 0, IT_MIXED = 1, IT_REFRESH_ALL = 2, IT_REFRESH_PENDING = 3 };

constexpr int kMB = kMapWG;  // map-domain workgroup size (pixels)

__device__ __forceinline__ bool stopped(const int *flag) { return *(volatile const int *) flag != 0; }

__device__ __forceinline__ double block_sum(double v, double *red) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0)
        for (int i = 0; i < (int) (blockDim.x >> 6); i++) s += red[i];
    return s;
}

// three block_sums at once, with their bits (red: 3 * blockDim.x / 64 doubles)
__device__ __forceinline__ void block_sum3(double &a, double &b, double &c, double *red) {
    const int W = (int) (blockDim.x >> 6), w = (int) (threadIdx.x >> 6);
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_xor(a, o);
        b += __shfl_xor(b, o);
        c += __shfl_xor(c, o);
    }
    __syncthreads();
    if ((threadIdx.x & 63) == 0) {
        red[w] = a;
        red[W + w] = b;
        red[2 * W + w] = c;
    }
    __syncthreads();
    a = b = c = 0.0;
    if (threadIdx.x == 0)
        for (int i = 0; i < W; i++) {
            a += red[i];
            b += red[W + i];
            c += red[2 * W + i];
        }
}

// threads of the scalar reductions (one workgroup per segment)
constexpr int kRB = 1024;

// fixed-order reduction of nparts partials by one workgroup of kRB threads
// (red: kRB / 64 doubles of LDS); every thread returns the sum
__device__ __forceinline__ double reduce_parts(const double *__restrict__ p, int nparts, double *red) {
    double s = 0.0;
    for (int i = threadIdx.x; i < nparts; i += kRB) s += p[i];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    __syncthreads();  // a previous call may still read red
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    double t = 0.0;
    for (int w = 0; w < kRB / 64; w++) t += red[w];
    return t;
}

// Largest number of partials of a segment that the map kernels sum themselves
// (`fused` of pcg_run): every workgroup then reads them all, four loads a thread and
// set, which costs about 1 us against 4.3-7.3 us and a launch for a reduction
// kernel.  A segment of 1024 workgroups is a map of 262144 pixels; with the
// 4096 of a 1024^2 map the reads (32 KB a set and workgroup) would add more
// than the kernel's own traffic.
constexpr int kFusedParts = 1024;

// reduce_parts for NS sets of nparts <= kFusedParts partials (set k at p + k
// stride) by a workgroup of kMB threads, in reduce_parts' order and so with its
// bits: thread t holds the values of its threads t, t + kMB, ...  red: NS * kRB
// / 64 doubles of LDS; every thread gets the sums.
template <int NS>
__device__ __forceinline__ void reduce_parts_wg(const double *__restrict__ p, int64_t stride, int nparts, double *red,
                                                double (&out)[NS]) {
    constexpr int J = kRB / kMB, W = kRB / 64;
    const int w0 = __builtin_amdgcn_readfirstlane((int) threadIdx.x & ~63);  // the wave's first thread
    double v[NS][J];
#pragma unroll
    for (int k = 0; k < NS; k++)
#pragma unroll
        for (int j = 0; j < J; j++) {
            const int i = (int) threadIdx.x + j * kMB;
            v[k][j] = i < nparts ? p[k * stride + i] : 0.0;
        }
#pragma unroll
    for (int k = 0; k < NS; k++)
#pragma unroll
        for (int j = 0; j < J; j++) {
            double s = 0.0 + v[k][j];
            if (w0 + j * kMB < nparts)  // a wave without partials has the sum +0.0
                for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
            if ((threadIdx.x & 63) == 0) red[k * W + (threadIdx.x >> 6) + j * (kMB / 64)] = s;
        }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NS; k++) {
        double t = 0.0;
#pragma unroll
        for (int w = 0; w < W; w++) t += red[k * W + w];
        out[k] = t;
    }
}

// pixel handled by this thread of a map-domain workgroup, its segment and the segment end
struct SegPix {
    int r, q, qend;
};
__device__ __forceinline__ SegPix seg_pixel(const int *__restrict__ wg_seg, const int *__restrict__ wg_q0,
                                            const int *__restrict__ seg_q) {
    SegPix p;
    p.r = wg_seg[blockIdx.x];
    p.q = wg_q0[blockIdx.x] + (int) threadIdx.x;
    p.qend = seg_q[p.r + 1];
    return p;
}

}  // namespace mgpu
