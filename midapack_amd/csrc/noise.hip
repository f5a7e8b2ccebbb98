// noise.hip -- the noise-model builder on the device: per Toeplitz block, the
// first row of the banded inverse noise covariance from a noise timestream.
//
// Reference: compute_invtt / noise2invtt (TOAST_interface/utils.py:435-601).
// For a block of n samples:
//   1. periodogram: Welch with one segment of n samples (nperseg = n, utils.py
//      527), Hann window (periodic), linear detrend, one-sided density scaling;
//   2. fit of the log-PSD model a + log10(1 + ((f + fmin)/fknee)^alpha) to
//      log10 psd[1:] (utils.py:530-538: p0 = (-7, -1, 0.1, 1e-6), bounds
//      a in [-20, 0], alpha in [-10, 0], fknee in [0, 20], fmin in [0, 1]);
//   3. psdm1 = 10^-a / (1 + ((f + fmin)/fknee)^alpha) on rfftfreq(n);
//   4. inv_tt = irfft(psdm1, n); result = window[:lambda] * inv_tt[:lambda],
//      window = ifftshift(chebwin(2 lambda, 150 dB)) (or the general Gaussian
//      of utils.py:569-573).
// The reference fits with scipy's trust-region-reflective least squares; here
// a bounded Levenberg-Marquardt runs on the device, one workgroup for a short block
// and 16 for a step of a long one.
// Both minimise the same objective; results agree to the fit tolerance.
//
// FFTs: batched Stockham passes in HBM, four radix-2 stages a launch in
// registers (k_fft_step), for power-of-two n; other n use Bluestein's chirp-z
// transform on the next power of two >= 2n - 1.  The forward transform of the
// periodogram and the inverse transform of psdm1 (real and even, so its
// inverse DFT is its forward DFT divided by n) share the same machinery.
//
// Sums over a block's samples or frequencies (the line fit of the detrending,
// the window's power, the normal equations of the fit) are 256 chains, chain c
// adding the terms c, c + 256, ... in order, then a fixed tree over the chains.
// chain_sums computes the terms of 16 chains by 1024 threads and adds them up in
// that order from LDS, so one block's sum runs on 16 CUs at once with the bits
// of one workgroup of 256 threads.
#include "mgpu_internal.h"

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>

namespace mgpu {

namespace {

// LR radix-2 Stockham passes over `batch` transforms of length M = 2^logm in one
// launch: sub-transform size ns -> ns 2^LR; sign -1 forward, +1 inverse (no
// scaling).  A thread holds the 2^LR points x[j + t M / 2^LR]; the passes' pairs
// and twiddles are those of one pass at a time.  REAL: the input is the real
// sequence xr + xoff[b].  Bound by HBM and the sincospi of the twiddles (15 for
// 16 points): 64 transforms of 2^17 points, 17 passes of 38 us -> 5 launches of
// 37-76 us.
template <int LR, bool REAL>
__global__ __launch_bounds__(256) void k_fft_step(const double2 *__restrict__ in, const double *__restrict__ xr,
                                                  const int64_t *__restrict__ xoff, double2 *__restrict__ out,
                                                  int logm, int ns, int sign, int batch) {
    constexpr int R = 1 << LR;
    const int64_t M = (int64_t) 1 << logm, per = M >> LR;
    const int64_t gid = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= per * batch) return;
    const int64_t b = gid / per, j = gid % per;
    double2 v[R];
    if constexpr (REAL) {
        const double *x = xr + xoff[b];
#pragma unroll
        for (int t = 0; t < R; t++) v[t] = make_double2(x[j + t * per], 0.0);
    } else {
        const double2 *x = in + b * M;
#pragma unroll
        for (int t = 0; t < R; t++) v[t] = x[j + t * per];
    }
    const int64_t r = j & (ns - 1);
    // before stage s, v[t (1 << s) + u] is the point of offset u ns inside a
    // group of ns 2^s points, t the group's place among the 2^(LR-s) it holds
#pragma unroll
    for (int st = 0; st < LR; st++) {
        double2 o[R];
        const double nsd = (double) ((int64_t) ns << st);
#pragma unroll
        for (int u = 0; u < (1 << st); u++) {
            double s, c;
            sincospi((double) sign * (double) (r + (int64_t) u * ns) / nsd, &s, &c);
#pragma unroll
            for (int t = 0; t < (R >> (st + 1)); t++) {
                const double2 v0 = v[(t << st) + u], w = v[((t + (R >> (st + 1))) << st) + u];
                const double2 v1 = make_double2(w.x * c - w.y * s, w.x * s + w.y * c);
                o[(t << (st + 1)) + u] = make_double2(v0.x + v1.x, v0.y + v1.y);
                o[(t << (st + 1)) + u + (1 << st)] = make_double2(v0.x - v1.x, v0.y - v1.y);
            }
        }
#pragma unroll
        for (int t = 0; t < R; t++) v[t] = o[t];
    }
    double2 *y = out + b * M + (j - r) * R + r;
#pragma unroll
    for (int t = 0; t < R; t++) y[(int64_t) t * ns] = v[t];
}

// exp(sign * pi * i * j^2 / n), with j^2 reduced mod 2n exactly
__device__ __forceinline__ double2 chirp(int64_t j, int64_t n, int sign) {
    const int64_t e = (j * j) % (2 * n);
    double s, c;
    sincospi((double) sign * (double) e / (double) n, &s, &c);
    return make_double2(c, s);
}

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// Bluestein, step 1: A_t = x_t w_t (t < n), 0 beyond; B = conj chirp, wrapped
__global__ void k_blue_prep(const double *__restrict__ x, const int64_t *__restrict__ xoff,
                            const int *__restrict__ nlen, int logm, int batch, double2 *__restrict__ A,
                            double2 *__restrict__ B) {
    const int64_t M = (int64_t) 1 << logm;
    const int64_t gid = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= M * batch) return;
    const int64_t b = gid / M, t = gid % M;
    const int64_t n = nlen[b];
    A[gid] = t < n ? cmul(make_double2(x[xoff[b] + t], 0.0), chirp(t, n, -1)) : make_double2(0.0, 0.0);
    double2 v = make_double2(0.0, 0.0);
    if (t < n)
        v = chirp(t, n, +1);
    else if (t > M - n)
        v = chirp(M - t, n, +1);
    B[gid] = v;
}

__global__ void k_pointwise(double2 *__restrict__ A, const double2 *__restrict__ B, int64_t total) {
    const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i < total) A[i] = cmul(A[i], B[i]);
}

// Bluestein, last step: X_k = w_k conv_k / M for k < nout
__global__ void k_blue_post(const double2 *__restrict__ C, const int *__restrict__ nlen, int logm, int batch,
                            int64_t nout_max, double2 *__restrict__ X) {
    const int64_t M = (int64_t) 1 << logm;
    const int64_t gid = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= nout_max * batch) return;
    const int64_t b = gid / nout_max, k = gid % nout_max;
    const int64_t n = nlen[b];
    if (k >= n) return;
    const double2 v = cmul(C[b * M + k], chirp(k, n, -1));
    X[b * nout_max + k] = make_double2(v.x / (double) M, v.y / (double) M);
}

// forward DFTs of `batch` real sequences of lengths nlen[b] (all with the same
// transform size M = 2^logm: n = M for powers of two, else the Bluestein size),
// with the work buffers of one group of blocks
struct Dft {
    Problem &pb;
    int logm, batch;
    bool pow2;
    int64_t nout_max;
    double2 *a = nullptr, *b = nullptr, *c = nullptr;  // c: the chirp's spectrum (Bluestein)
    double2 *X = nullptr;                              // [batch * stride] the transform
    int64_t stride = 0;

    Dft(Problem &p, int logm_, int batch_, bool pow2_, int64_t nout)
        : pb(p), logm(logm_), batch(batch_), pow2(pow2_), nout_max(nout) {}
    ~Dft() {
        for (double2 *p : {a, b, c})
            if (p) pb.arena.release(p);
    }
    int alloc() {
        const size_t total = ((size_t) 1 << logm) * batch;
        MGPU_RET(pb.arena.alloc(&a, total));
        MGPU_RET(pb.arena.alloc(&b, total));
        if (!pow2) MGPU_RET(pb.arena.alloc(&c, total));
        return MGPU_OK;
    }
    // transform of src (or of the real sequences xr + xoff[b]) through tmp: src holds the result
    int fft(double2 *&src, double2 *&tmp, int sign, const double *xr, const int64_t *xoff) {
        const int64_t M = (int64_t) 1 << logm;
        for (int done = 0; done < logm;) {
            const int lr = std::min(4, logm - done), ns = 1 << done;
            const unsigned g = grid_for((M >> lr) * batch, 256);
            hipStream_t s = pb.stream;
#define MGPU_FFT(LR)                                                                                    \
    case LR:                                                                                            \
        if (xr && done == 0)                                                                            \
            k_fft_step<LR, true><<<g, 256, 0, s>>>(src, xr, xoff, tmp, logm, ns, sign, batch);          \
        else                                                                                            \
            k_fft_step<LR, false><<<g, 256, 0, s>>>(src, nullptr, nullptr, tmp, logm, ns, sign, batch); \
        break
            switch (lr) {
                MGPU_FFT(1);
                MGPU_FFT(2);
                MGPU_FFT(3);
                MGPU_FFT(4);
            }
#undef MGPU_FFT
            MGPU_LAUNCHED();
            std::swap(src, tmp);
            done += lr;
        }
        return MGPU_OK;
    }
    // X[b * stride + k] = DFT_k for k < min(n, nout_max)
    int run(const double *d_x, const int64_t *d_xoff, const int *d_nlen, double2 *d_out) {
        hipStream_t s = pb.stream;
        const int64_t M = (int64_t) 1 << logm, total = M * batch;
        if (pow2) {
            MGPU_RET(fft(a, b, -1, d_x, d_xoff));
            X = a;
            stride = M;
            return MGPU_OK;
        }
        k_blue_prep<<<grid_for(total, 256), 256, 0, s>>>(d_x, d_xoff, d_nlen, logm, batch, a, c);
        MGPU_LAUNCHED();
        MGPU_RET(fft(a, b, -1, nullptr, nullptr));
        MGPU_RET(fft(c, b, -1, nullptr, nullptr));
        k_pointwise<<<grid_for(total, 256), 256, 0, s>>>(a, c, total);
        MGPU_LAUNCHED();
        MGPU_RET(fft(a, b, +1, nullptr, nullptr));
        k_blue_post<<<grid_for(nout_max * batch, 256), 256, 0, s>>>(a, d_nlen, logm, batch, nout_max, d_out);
        MGPU_LAUNCHED();
        X = d_out;
        stride = nout_max;
        return MGPU_OK;
    }
};

constexpr int kChains = 256;                       // chains of a sum
constexpr int kChainCols = 16;                     // chains of a workgroup
constexpr int kChainRows = 64;                     // terms of a chain computed at once
constexpr int kChainWG = kChainCols * kChainRows;  // threads
constexpr int kChainGroups = kChains / kChainCols;

// sums over terms 0 .. count-1: chain c of `group` (c = 16 group + lane) adds its
// terms c, c + 256, ... in order.  term(i, v) gives the NV values of term i, and
// sum s of the NS adds v[ia(s)] * v[ib(s)] (ib < 0: v[ia(s)] itself).  out[s *
// kChains + c].  The terms of 64 rows go to LDS, are added by the first NS * 16
// threads while all compute the next 64 (two buffers, one barrier a turn).
template <int NV, int NS, typename Term, typename Pair>
__device__ __forceinline__ void chain_sums(int64_t count, int group, Term term, Pair pair, double *__restrict__ out) {
    static_assert(NS * kChainCols <= kChainWG, "one thread per chain and sum");
    __shared__ double buf[2][kChainRows][NV][kChainCols];
    const int t = threadIdx.x, col = t % kChainCols, row = t / kChainCols;
    const int s = t / kChainCols;  // sum of a summing thread (its chain is col)
    int ia = 0, ib = -1;
    if (s < NS) pair(s, ia, ib);
    double acc = 0.0;
    const int64_t c = (int64_t) group * kChainCols + col;
    const int64_t rows = (count + kChains - 1) / kChains;
    for (int64_t r0 = 0, turn = 0; r0 < rows; r0 += kChainRows, turn++) {
        double(*bf)[NV][kChainCols] = buf[turn & 1];
        const int64_t i = (r0 + row) * kChains + c;
        if (i < count) {
            double v[NV];
            term(i, v);
#pragma unroll
            for (int k = 0; k < NV; k++) bf[row][k][col] = v[k];
        }
        __syncthreads();
        if (s < NS) {
            const int64_t left = (count - c + kChains - 1) / kChains - r0;  // terms of the chain from row r0 on
            const int m = (int) (left < kChainRows ? left : kChainRows);
#pragma unroll 8
            for (int q = 0; q < m; q++) {
                const double x = bf[q][ia][col];
                acc += ib < 0 ? x : x * bf[q][ib][col];
            }
        }
    }
    if (s < NS) out[s * kChains + c] = acc;
}

// the tree over 256 chains that a workgroup of 256 threads would run (halves
// added pairwise), by one wave: every lane gets the sum
__device__ __forceinline__ double chain_tree(const double *__restrict__ v) {
    const int l = threadIdx.x & 63;
    double a = (v[l] + v[l + 128]) + (v[l + 64] + v[l + 192]);
    for (int o = 32; o > 0; o >>= 1) a += __shfl_down(a, o);
    return __shfl(a, 0);
}

// sums of x and t x over a block (the least-squares line): parts[b][2][256]
__global__ __launch_bounds__(kChainWG) void k_line_sums(const double *__restrict__ noise,
                                                        const int64_t *__restrict__ start,
                                                        const int *__restrict__ nlen, const int *__restrict__ blocks,
                                                        double *__restrict__ parts) {
    const int bi = blockIdx.x / kChainGroups, g = blockIdx.x % kChainGroups;
    const double *x = noise + start[blocks[bi]];
    chain_sums<2, 2>(
            nlen[bi], g,
            [&](int64_t t, double *v) {
                v[0] = x[t];
                v[1] = (double) t * x[t];
            },
            [](int s, int &ia, int &ib) { ia = s; }, parts + (int64_t) bi * 2 * kChains);
}

// detrended, Hann-windowed segment: xw[t] = w_t (x_t - (c0 + c1 t)), the line
// fitted by least squares (scipy.signal.detrend type 'linear'), and the chains of
// sum w^2: wparts[b][256]
__global__ __launch_bounds__(kChainWG) void k_detrend_window(const double *__restrict__ noise,
                                                             const int64_t *__restrict__ start,
                                                             const int *__restrict__ nlen,
                                                             const int *__restrict__ blocks,
                                                             const int64_t *__restrict__ xoff,
                                                             const double *__restrict__ parts,
                                                             double *__restrict__ xw, double *__restrict__ wparts) {
    const int bi = blockIdx.x / kChainGroups, g = blockIdx.x % kChainGroups;
    const int64_t n = nlen[bi];
    const double *x = noise + start[blocks[bi]];
    double *__restrict__ o = xw + xoff[bi];
    const double sx = chain_tree(parts + (int64_t) bi * 2 * kChains);
    const double stx = chain_tree(parts + ((int64_t) bi * 2 + 1) * kChains);
    const double dn = (double) n;
    const double st = dn * (dn - 1.0) / 2.0, stt = (dn - 1.0) * dn * (2.0 * dn - 1.0) / 6.0;
    const double det = dn * stt - st * st;
    const double c1 = (dn * stx - st * sx) / det, c0 = (sx - c1 * st) / dn;
    chain_sums<1, 1>(
            n, g,
            [&](int64_t t, double *v) {
                double sn, cs;
                sincospi(2.0 * (double) t / dn, &sn, &cs);
                const double w = 0.5 - 0.5 * cs;  // periodic Hann
                o[t] = w * (x[t] - (c0 + c1 * (double) t));
                v[0] = w * w;
            },
            [](int, int &ia, int &) { ia = 0; }, wparts + (int64_t) bi * kChains);
}

__global__ __launch_bounds__(64) void k_chain_tree(const double *__restrict__ parts, double *__restrict__ out) {
    const double v = chain_tree(parts + (int64_t) blockIdx.x * kChains);
    if (threadIdx.x == 0) out[blockIdx.x] = v;
}

// log10 of the one-sided density periodogram, k = 1 .. n/2
// (y of block blocks[b] at yoff[blocks[b]])
__global__ void k_logpsd(const double2 *__restrict__ X, int64_t stride, const int *__restrict__ nlen, int64_t nmax,
                         int batch, const double *__restrict__ wsum2, double fsamp, const int *__restrict__ blocks,
                         const int64_t *__restrict__ yoff, double *__restrict__ y) {
    const int64_t gid = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t half = nmax / 2 + 1;
    if (gid >= half * batch) return;
    const int64_t b = gid / half, k = gid % half;
    const int64_t n = nlen[b];
    if (k > n / 2) return;
    const double2 v = X[b * stride + k];
    double p = (v.x * v.x + v.y * v.y) / (fsamp * wsum2[b]);
    const bool nyq = (n % 2 == 0) && k == n / 2;
    if (k > 0 && !nyq) p *= 2.0;
    y[yoff[blocks[b]] + k] = log10(p);
}

// model pieces at frequency f: h = log10(1 + g), g = u^alpha, u = (f + fmin) / fknee
struct Model {
    double h, dh_alpha, dh_fknee, dh_fmin;
};
__device__ __forceinline__ Model model_at(double f, double alpha, double fknee, double fmin) {
    const double u = (f + fmin) / fknee;
    const double lu = log(u);
    const double g = exp(alpha * lu);
    const double k = g / ((1.0 + g) * 2.302585092994045684);  // g / ((1 + g) ln 10)
    Model m;
    m.h = log10(1.0 + g);
    m.dh_alpha = k * lu;
    m.dh_fknee = -k * alpha / fknee;
    m.dh_fmin = k * alpha / (f + fmin);
    return m;
}

constexpr int kFitIter = 400;

// Bounded Levenberg-Marquardt fit of a + log10(1 + ((f+fmin)/fknee)^alpha) to
// y[1..n/2], every block of the noise model at once.  One evaluation of the
// model at a block's trial point q gives its cost and, if q is accepted, the
// normal equations of the next step: k_fit_eval sums both (16 workgroups a
// block), k_fit_step decides and takes the step.  Bound by the logarithms and
// exponentials (VALU): on 64 blocks of 2^17 samples one workgroup a block, with
// two model passes an iteration, took 18.4 ms; 64 evaluations of 28 us and
// decisions of 6 us take 2.2 ms.  Short blocks are fitted by a workgroup each
// (k_fit_block, see kBlockRows).
struct FitState {
    double p[4], q[4];   // best point, trial point (a, alpha, fknee, fmin)
    double A[13];        // normal equations at p: J^T J (0..9), J^T r (10..12: its last three)
    double jr0;          // J^T r, first entry
    double cost, mu;
    int it, tiny, done, first;
};

constexpr int kFitSums = 14;  // 13 products of J and r (below) and the cost

// products of the values (r, dh_alpha, dh_fknee, dh_fmin), J = (1, dh...):
// J_i J_j for i <= j without 1 * 1, then J_i r, then r r
__device__ __forceinline__ void fit_pair(int s, int &ia, int &ib) {
    const int a[kFitSums] = {1, 2, 3, 1, 1, 1, 2, 2, 3, 0, 1, 2, 3, 0};
    const int b[kFitSums] = {-1, -1, -1, 1, 2, 3, 2, 3, 3, -1, 0, 0, 0, 0};
    ia = a[s];
    ib = b[s];
}

__global__ void k_fit_init(FitState *__restrict__ st, int nb) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nb) return;
    FitState &F = st[b];
    const double p0[4] = {-7.0, -1.0, 0.1, 1e-6};
    for (int i = 0; i < 4; i++) F.p[i] = F.q[i] = p0[i];
    F.mu = 1e-3;
    F.it = F.tiny = F.done = 0;
    F.first = 1;
}

// (r, dh_alpha, dh_fknee, dh_fmin) of frequency i + 1 at the trial point
__device__ __forceinline__ void fit_term(int64_t i, double n, double fsamp, const double (&q)[4],
                                         const double *__restrict__ yb, double *v) {
    const double f = (double) (i + 1) * fsamp / n;
    const Model md = model_at(f, q[1], q[2], q[3]);
    v[0] = q[0] + md.h - yb[i];
    v[1] = md.dh_alpha;
    v[2] = md.dh_fknee;
    v[3] = md.dh_fmin;
}

__global__ __launch_bounds__(kChainWG) void k_fit_eval(const double *__restrict__ y, const int64_t *__restrict__ yoff,
                                                       const int *__restrict__ nlen, double fsamp,
                                                       const int *__restrict__ list,
                                                       const FitState *__restrict__ st, double *__restrict__ parts) {
    const int k = blockIdx.x / kChainGroups, g = blockIdx.x % kChainGroups, b = list[k];
    if (st[b].done) return;
    const int64_t n = nlen[b], K = n / 2;
    const double *yb = y + yoff[b] + 1;
    const double q[4] = {st[b].q[0], st[b].q[1], st[b].q[2], st[b].q[3]};
    chain_sums<4, kFitSums>(
            K, g, [&](int64_t i, double *v) { fit_term(i, (double) n, fsamp, q, yb, v); }, fit_pair,
            parts + (int64_t) k * kFitSums * kChains);
}

// The sums of an evaluation at q, by one thread: accept or reject, then the next
// trial point or F.done
__device__ __forceinline__ void fit_decide(FitState &F, const double *sums, int n) {
    const double lo[4] = {-20.0, -10.0, 1e-12, 0.0}, hi[4] = {0.0, 0.0, 20.0, 1.0};
    const double cq = sums[13];
    bool accept = false, stop = false;
    if (F.first) {
        F.first = 0;
        accept = true;
        F.cost = cq;
    } else {
        if (cq < F.cost) {
            const double rel = (F.cost - cq) / fmax(F.cost, 1e-300);
            for (int i = 0; i < 4; i++) F.p[i] = F.q[i];
            accept = true;
            F.cost = cq;
            F.mu = fmax(F.mu * 0.3, 1e-12);
            stop = rel < 1e-15 || F.tiny;
        } else {
            F.mu *= 10.0;
            stop = F.mu > 1e12 || F.tiny;
        }
        stop = stop || ++F.it >= kFitIter;
    }
    if (stop) {
        F.done = 1;
        return;
    }
    if (accept) {
        F.A[0] = (double) (n / 2);  // the sum of 1 * 1
        for (int e = 0; e < 9; e++) F.A[1 + e] = sums[e];
        F.jr0 = sums[9];
        for (int e = 0; e < 3; e++) F.A[10 + e] = sums[10 + e];
    }
    // damped step (J^T J + mu diag) d = -J^T r, projected on the bounds
    const double mu = F.mu;
    double p[4];
    for (int i = 0; i < 4; i++) p[i] = F.p[i];
    double A[4][4], g[4];
    int e = 0;
    for (int i = 0; i < 4; i++)
        for (int j = i; j < 4; j++) {
            A[i][j] = F.A[e];
            A[j][i] = F.A[e];
            e++;
        }
    g[0] = -F.jr0;
    for (int i = 1; i < 4; i++) g[i] = -F.A[9 + i];
    for (int i = 0; i < 4; i++) A[i][i] += mu * (A[i][i] > 0.0 ? A[i][i] : 1.0);
    // active set: a parameter on a bound whose descent direction points
    // outside stays fixed (its row and column leave the system)
    for (int i = 0; i < 4; i++) {
        const bool act = (p[i] <= lo[i] && g[i] < 0.0) || (p[i] >= hi[i] && g[i] > 0.0);
        if (act) {
            for (int j = 0; j < 4; j++) {
                A[i][j] = 0.0;
                A[j][i] = 0.0;
            }
            A[i][i] = 1.0;
            g[i] = 0.0;
        }
    }
    // Gaussian elimination with partial pivoting (4x4)
    for (int c = 0; c < 4; c++) {
        int pr = c;
        for (int r = c + 1; r < 4; r++)
            if (fabs(A[r][c]) > fabs(A[pr][c])) pr = r;
        for (int j = 0; j < 4; j++) {
            const double t = A[c][j];
            A[c][j] = A[pr][j];
            A[pr][j] = t;
        }
        const double tg = g[c];
        g[c] = g[pr];
        g[pr] = tg;
        for (int r = c + 1; r < 4; r++) {
            const double fct = A[c][c] != 0.0 ? A[r][c] / A[c][c] : 0.0;
            for (int j = c; j < 4; j++) A[r][j] -= fct * A[c][j];
            g[r] -= fct * g[c];
        }
    }
    double d[4];
    for (int r = 3; r >= 0; r--) {
        double v = g[r];
        for (int j = r + 1; j < 4; j++) v -= A[r][j] * d[j];
        d[r] = A[r][r] != 0.0 ? v / A[r][r] : 0.0;
    }
    double dn = 0.0, pn = 0.0;
    for (int i = 0; i < 4; i++) {
        const double q = fmin(fmax(p[i] + d[i], lo[i]), hi[i]);
        F.q[i] = q;
        dn += (q - p[i]) * (q - p[i]);
        pn += p[i] * p[i];
    }
    F.tiny = sqrt(dn) <= 1e-14 * (sqrt(pn) + 1e-14) ? 1 : 0;
}

// one workgroup per listed block: the chains' trees and the decision; *left counts
// the blocks that go on
__global__ __launch_bounds__(64 * kFitSums) void k_fit_step(const double *__restrict__ parts,
                                                            const int *__restrict__ nlen,
                                                            const int *__restrict__ list, FitState *__restrict__ st,
                                                            int *__restrict__ left) {
    __shared__ double sums[kFitSums];
    const int b = list[blockIdx.x];
    FitState &F = st[b];
    if (F.done) return;  // written by this block's thread 0 of an earlier launch only
    const int wv = threadIdx.x >> 6;
    const double v = chain_tree(parts + ((int64_t) blockIdx.x * kFitSums + wv) * kChains);
    if ((threadIdx.x & 63) == 0) sums[wv] = v;
    __syncthreads();
    if (threadIdx.x != 0) return;
    fit_decide(F, sums, nlen[b]);
    if (F.done) atomicSub(left, 1);
}

// The whole fit of a listed block by one workgroup, a thread a chain: the terms,
// their order and so the bits are those of k_fit_eval and k_fit_step.
__global__ __launch_bounds__(kChains) void k_fit_block(const double *__restrict__ y, const int64_t *__restrict__ yoff,
                                                       const int *__restrict__ nlen, double fsamp,
                                                       const int *__restrict__ list, FitState *__restrict__ st) {
    __shared__ double chain[kFitSums][kChains];
    __shared__ double sums[kFitSums];
    __shared__ FitState F;
    const int b = list[blockIdx.x], t = threadIdx.x, n = nlen[b], K = n / 2;
    const double *__restrict__ yb = y + yoff[b] + 1;
    if (t == 0) F = st[b];
    __syncthreads();
    while (!F.done) {  // kFitIter + 1 evaluations at most
        const double q[4] = {F.q[0], F.q[1], F.q[2], F.q[3]};
        double acc[kFitSums];
#pragma unroll
        for (int s = 0; s < kFitSums; s++) acc[s] = 0.0;
        for (int i = t; i < K; i += kChains) {
            double v[4];
            fit_term(i, (double) n, fsamp, q, yb, v);
#pragma unroll
            for (int s = 0; s < kFitSums; s++) {
                int ia, ib;
                fit_pair(s, ia, ib);
                acc[s] += ib < 0 ? v[ia] : v[ia] * v[ib];
            }
        }
#pragma unroll
        for (int s = 0; s < kFitSums; s++) chain[s][t] = acc[s];
        __syncthreads();
        for (int s = t >> 6; s < kFitSums; s += kChains / 64) {
            const double v = chain_tree(chain[s]);
            if ((t & 63) == 0) sums[s] = v;
        }
        __syncthreads();
        if (t == 0) fit_decide(F, sums, n);
        __syncthreads();
    }
    if (t == 0) st[b] = F;
}

// psdm1 of the fitted model on rfftfreq(n), extended to the full even sequence
// of length n (each value computed once and written to both its places)
__global__ void k_psdm1_even(const FitState *__restrict__ st, const int *__restrict__ blocks,
                             const int *__restrict__ nlen, int64_t nmax, int batch, double fsamp,
                             double *__restrict__ out) {
    const int64_t gid = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t half = nmax / 2 + 1;
    if (gid >= half * batch) return;
    const int64_t b = gid / half, k = gid % half;
    const int64_t n = nlen[b];
    if (k > n / 2) return;
    const double *p = st[blocks[b]].p;
    const double f = (double) k * fsamp / (double) n;
    const double u = (f + p[3]) / p[2];
    const double v = pow(10.0, -p[0]) / (1.0 + pow(u, p[1]));
    out[b * nmax + k] = v;
    if (k > 0 && n - k > n / 2) out[b * nmax + n - k] = v;
}

// invtt row: window[j] * Re(DFT(psdm1_even))[j] / n for j < lambda
__global__ void k_invtt_rows(const double2 *__restrict__ X, int64_t stride, const int *__restrict__ nlen,
                             const int *__restrict__ blocks, int batch, int lambda,
                             const double *__restrict__ window, double *__restrict__ invtt) {
    const int64_t gid = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= (int64_t) lambda * batch) return;
    const int64_t b = gid / lambda, j = gid % lambda;
    invtt[(int64_t) blocks[b] * lambda + j] = window[j] * (X[b * stride + j].x / (double) nlen[b]);
}

}  // namespace

// Symmetric Dolph-Chebyshev window of M points, attenuation at dB, by its
// frequency-domain definition: W_k = T_{M-1}(beta cos(pi k / M)) with
// beta = cosh(acosh(10^(at/20)) / (M-1)); the window is the real DFT of W
// (with a half-sample phase for even M), mirrored and normalised to a unit
// maximum.  Direct DFT over a cosine table: set-up work, cached per lambda.
static std::vector<double> chebwin_sym(int M, double at) {
    const double order = M - 1.0;
    const double beta = std::cosh(std::acosh(std::pow(10.0, std::fabs(at) / 20.0)) / order);
    std::vector<double> pr((size_t) M), pi((size_t) M), ct((size_t) M), st((size_t) M);
    for (int k = 0; k < M; k++) {
        ct[k] = std::cos(2.0 * M_PI * k / M);
        st[k] = std::sin(2.0 * M_PI * k / M);
    }
    for (int k = 0; k < M; k++) {
        const double x = beta * std::cos(M_PI * k / M);
        double v;
        if (x > 1.0)
            v = std::cosh(order * std::acosh(x));
        else if (x < -1.0)
            v = (2.0 * (M % 2) - 1.0) * std::cosh(order * std::acosh(-x));
        else
            v = std::cos(order * std::acos(x));
        if (M % 2) {
            pr[k] = v;
            pi[k] = 0.0;
        } else {
            pr[k] = v * std::cos(M_PI * k / M);
            pi[k] = v * std::sin(M_PI * k / M);
        }
    }
    const int n = M % 2 ? (M + 1) / 2 : M / 2 + 1;
    std::vector<double> w((size_t) n);
    for (int t = 0; t < n; t++) {  // real part of the forward DFT at t
        double acc = 0.0;
        for (int k = 0; k < M; k++) {
            const size_t e = (size_t) (((int64_t) k * t) % M);
            acc += pr[k] * ct[e] + pi[k] * st[e];
        }
        w[t] = acc;
    }
    std::vector<double> full;
    full.reserve((size_t) M);
    for (int t = n - 1; t >= 1; t--) full.push_back(w[t]);
    for (int t = (M % 2 ? 0 : 1); t < n; t++) full.push_back(w[t]);
    double mx = 0.0;
    for (double v : full) mx = std::max(mx, v);
    for (double &v : full) v /= mx;
    return full;
}

// window[:lambda] of ifftshift(get_window(kind, 2 lambda)) (utils.py:562-577):
// the DFT-even ("fftbins") window of 2 lambda points is the symmetric window of
// 2 lambda + 1 points without its last point
static const std::vector<double> &apod_window(int lambda, int kind) {
    static std::mutex mu;
    static std::map<std::pair<int, int>, std::vector<double>> cache;
    std::lock_guard<std::mutex> g(mu);
    auto it = cache.find({lambda, kind});
    if (it != cache.end()) return it->second;
    const int N = 2 * lambda;
    std::vector<double> full;
    if (kind == MGPU_APOD_CHEBWIN) {
        full = chebwin_sym(N + 1, 150.0);
    } else {  // general Gaussian, p = 1, sigma = lambda / 3 (q_apo = 3)
        const double sigma = lambda / 3.0, c = lambda;  // centre of N + 1 points
        full.resize((size_t) N + 1);
        for (int t = 0; t <= N; t++) full[t] = std::exp(-0.5 * ((t - c) / sigma) * ((t - c) / sigma));
    }
    std::vector<double> w((size_t) lambda);
    for (int j = 0; j < lambda; j++) w[j] = full[(size_t) ((j + lambda) % N)];
    return cache[{lambda, kind}] = w;
}

// Longest chains of a block that one workgroup fits (n <= 8193).  It runs through
// them at about 0.5 us a term where k_fit_eval and k_fit_step cost two launches a step,
// for every block until the last one is done: 4096 blocks of 300 samples 71.6 ms with
// them and 6.0 with k_fit_block, 256 of 4096 samples 6.0 and 2.9, one of 8192 0.54 and
// 0.47; with 32 terms (16384 samples) it loses unless the blocks fill the chip (one
// block 0.51 and 0.71, 256 blocks 5.66 and 5.56), with 256 always (64 blocks 6.0 and 15.6).
static constexpr int kBlockRows = 16;

int noise_invtt(Problem &pb, const double *d_noise, int nb, const int *block_sizes, int lambda, double fsamp,
                int window_kind, double *d_invtt, double *h_params) {
    hipStream_t s = pb.stream;
    MGPU_ARG(nb > 0 && lambda >= 1 && fsamp > 0.0, "nb=%d lambda=%d fsamp=%g", nb, lambda, fsamp);
    std::vector<int64_t> start((size_t) nb + 1, 0);
    for (int b = 0; b < nb; b++) {
        MGPU_ARG(block_sizes[b] >= 4, "block %d has %d samples", b, block_sizes[b]);
        MGPU_ARG(lambda <= block_sizes[b] / 2, "Bandwidth cannot be larger than timestream (utils.py:561): "
                                               "lambda=%d, block %d has %d samples", lambda, b, block_sizes[b]);
        start[b + 1] = start[b] + block_sizes[b];
    }
    MGPU_ARG(window_kind == MGPU_APOD_CHEBWIN || window_kind == MGPU_APOD_GAUSSIAN, "unknown window %d",
             window_kind);
    const std::vector<double> &win = apod_window(lambda, window_kind);
    // every block's log periodogram, transform group by group; one fit of all of
    // them; then the rows, group by group again
    std::vector<int64_t> yoff((size_t) nb + 1, 0);
    for (int b = 0; b < nb; b++) yoff[b + 1] = yoff[b] + block_sizes[b] / 2 + 1;
    double *d_win, *d_y, *d_parts;
    int64_t *d_start, *d_yoff;
    int *d_len, *d_left, *d_list;
    FitState *d_fit;
    MGPU_RET(pb.arena.alloc(&d_win, (size_t) lambda));
    MGPU_RET(pb.arena.alloc(&d_start, (size_t) nb + 1));
    MGPU_RET(pb.arena.alloc(&d_yoff, (size_t) nb + 1));
    MGPU_RET(pb.arena.alloc(&d_len, (size_t) nb));
    MGPU_RET(pb.arena.alloc(&d_left, 1));
    MGPU_RET(pb.arena.alloc(&d_y, (size_t) yoff[nb]));
    MGPU_RET(pb.arena.alloc(&d_fit, (size_t) nb));
    // the blocks that a workgroup each fits, then the others
    std::vector<int> list((size_t) nb);
    for (int b = 0; b < nb; b++) list[b] = b;
    const auto split = std::stable_partition(list.begin(), list.end(),
                                             [&](int b) { return block_sizes[b] / 2 <= kBlockRows * kChains; });
    const int nshort = (int) (split - list.begin()), nlong = nb - nshort;
    const int fit_run = std::min(nlong, 1 << 14);  // blocks evaluated by one launch (28 KB of chains each)
    MGPU_RET(pb.arena.alloc(&d_list, (size_t) nb));
    MGPU_RET(pb.arena.alloc(&d_parts, (size_t) std::max(fit_run, 1) * kFitSums * kChains));
    MGPU_HIP(hipMemcpyAsync(d_list, list.data(), sizeof(int) * nb, hipMemcpyHostToDevice, s));
    MGPU_HIP(hipMemcpyAsync(d_win, win.data(), sizeof(double) * lambda, hipMemcpyHostToDevice, s));
    MGPU_HIP(hipMemcpyAsync(d_start, start.data(), sizeof(int64_t) * (nb + 1), hipMemcpyHostToDevice, s));
    MGPU_HIP(hipMemcpyAsync(d_yoff, yoff.data(), sizeof(int64_t) * (nb + 1), hipMemcpyHostToDevice, s));
    MGPU_HIP(hipMemcpyAsync(d_len, block_sizes, sizeof(int) * nb, hipMemcpyHostToDevice, s));
    // group blocks by transform size (power of two n, or the Bluestein size)
    std::map<std::pair<int, int>, std::vector<int>> groups;  // (logm, pow2) -> blocks
    for (int b = 0; b < nb; b++) {
        const int64_t n = block_sizes[b];
        const bool p2 = (n & (n - 1)) == 0;
        int logm = 0;
        while (((int64_t) 1 << logm) < (p2 ? n : 2 * n - 1)) logm++;
        groups[{logm, p2 ? 1 : 0}].push_back(b);
    }
    for (int pass = 0; pass < 2; pass++) {
        if (pass == 1) {
            k_fit_init<<<grid_for(nb, 256), 256, 0, s>>>(d_fit, nb);
            MGPU_LAUNCHED();
            if (nshort > 0) {
                k_fit_block<<<nshort, kChains, 0, s>>>(d_y, d_yoff, d_len, fsamp, d_list, d_fit);
                MGPU_LAUNCHED();
            }
            int left = nlong;
            MGPU_HIP(hipMemcpyAsync(d_left, &left, sizeof(int), hipMemcpyHostToDevice, s));
            // an evaluation and a decision a step, kFitIter of them after the first at
            // most; the host looks every kFitPoll steps whether a block is left
            constexpr int kFitPoll = 8;
            for (int it = 0; it <= kFitIter && left > 0; it++) {
                for (int b0 = nshort; b0 < nb; b0 += fit_run) {
                    const unsigned n = (unsigned) std::min(fit_run, nb - b0);
                    k_fit_eval<<<n * kChainGroups, kChainWG, 0, s>>>(d_y, d_yoff, d_len, fsamp, d_list + b0, d_fit,
                                                                     d_parts);
                    MGPU_LAUNCHED();
                    k_fit_step<<<n, 64 * kFitSums, 0, s>>>(d_parts, d_len, d_list + b0, d_fit, d_left);
                    MGPU_LAUNCHED();
                }
                if (it % kFitPoll == kFitPoll - 1) {
                    MGPU_HIP(hipMemcpyAsync(&left, d_left, sizeof(int), hipMemcpyDeviceToHost, s));
                    MGPU_HIP(hipStreamSynchronize(s));
                }
            }
            if (h_params) {
                std::vector<FitState> hf((size_t) nb);
                MGPU_HIP(hipMemcpyAsync(hf.data(), d_fit, sizeof(FitState) * nb, hipMemcpyDeviceToHost, s));
                MGPU_HIP(hipStreamSynchronize(s));
                for (int b = 0; b < nb; b++)
                    for (int k = 0; k < 4; k++) h_params[4 * (int64_t) b + k] = hf[b].p[k];
            }
        }
        for (auto &kv : groups) {
            const int logm = kv.first.first;
            const bool p2 = kv.first.second != 0;
            const std::vector<int> &bl = kv.second;
            // batches bounded to ~2 GiB of complex work per buffer
            const int64_t M = (int64_t) 1 << logm;
            const int per = (int) std::min<int64_t>(1 << 17, std::max<int64_t>(1, ((int64_t) 1 << 27) / M));
            for (size_t g0 = 0; g0 < bl.size(); g0 += (size_t) per) {
                const int batch = (int) std::min<size_t>((size_t) per, bl.size() - g0);
                std::vector<int> blk(bl.begin() + g0, bl.begin() + g0 + batch), nlen((size_t) batch);
                std::vector<int64_t> xoff((size_t) batch);
                int64_t nmax = 0, tot = 0;
                for (int i = 0; i < batch; i++) {
                    nlen[i] = block_sizes[blk[i]];
                    nmax = std::max<int64_t>(nmax, nlen[i]);
                }
                for (int i = 0; i < batch; i++) {
                    xoff[i] = tot;
                    tot += nmax;
                }
                int *d_blk, *d_nlen;
                int64_t *d_xoff;
                double *d_xw, *d_w2 = nullptr, *d_ps = nullptr;
                double2 *d_X = nullptr;
                Dft dft(pb, logm, batch, p2, nmax);
                MGPU_RET(dft.alloc());
                MGPU_RET(pb.arena.alloc(&d_blk, (size_t) batch));
                MGPU_RET(pb.arena.alloc(&d_nlen, (size_t) batch));
                MGPU_RET(pb.arena.alloc(&d_xoff, (size_t) batch));
                MGPU_RET(pb.arena.alloc(&d_xw, (size_t) tot));
                if (pass == 0) {
                    MGPU_RET(pb.arena.alloc(&d_w2, (size_t) batch));
                    MGPU_RET(pb.arena.alloc(&d_ps, (size_t) 3 * kChains * batch));
                }
                if (!p2) MGPU_RET(pb.arena.alloc(&d_X, (size_t) tot));
                MGPU_HIP(hipMemcpyAsync(d_blk, blk.data(), sizeof(int) * batch, hipMemcpyHostToDevice, s));
                MGPU_HIP(hipMemcpyAsync(d_nlen, nlen.data(), sizeof(int) * batch, hipMemcpyHostToDevice, s));
                MGPU_HIP(hipMemcpyAsync(d_xoff, xoff.data(), sizeof(int64_t) * batch, hipMemcpyHostToDevice, s));
                const unsigned gc = (unsigned) batch * kChainGroups, gh = grid_for((nmax / 2 + 1) * batch, 256);
                if (pass == 0) {
                    double *wparts = d_ps + (size_t) 2 * kChains * batch;
                    k_line_sums<<<gc, kChainWG, 0, s>>>(d_noise, d_start, d_nlen, d_blk, d_ps);
                    MGPU_LAUNCHED();
                    k_detrend_window<<<gc, kChainWG, 0, s>>>(d_noise, d_start, d_nlen, d_blk, d_xoff, d_ps, d_xw,
                                                             wparts);
                    MGPU_LAUNCHED();
                    k_chain_tree<<<batch, 64, 0, s>>>(wparts, d_w2);
                    MGPU_LAUNCHED();
                    MGPU_RET(dft.run(d_xw, d_xoff, d_nlen, d_X));
                    k_logpsd<<<gh, 256, 0, s>>>(dft.X, dft.stride, d_nlen, nmax, batch, d_w2, fsamp, d_blk, d_yoff,
                                                d_y);
                } else {
                    k_psdm1_even<<<gh, 256, 0, s>>>(d_fit, d_blk, d_nlen, nmax, batch, fsamp, d_xw);
                    MGPU_LAUNCHED();
                    MGPU_RET(dft.run(d_xw, d_xoff, d_nlen, d_X));
                    k_invtt_rows<<<grid_for((int64_t) lambda * batch, 256), 256, 0, s>>>(
                            dft.X, dft.stride, d_nlen, d_blk, batch, lambda, d_win, d_invtt);
                }
                MGPU_LAUNCHED();
                MGPU_HIP(hipStreamSynchronize(s));  // before the work buffers go back to the block cache
                for (void *p : {(void *) d_blk, (void *) d_nlen, (void *) d_xoff, (void *) d_xw, (void *) d_w2,
                                (void *) d_ps, (void *) d_X})
                    if (p) pb.arena.release(p);
            }
        }
    }
    for (void *p : {(void *) d_win, (void *) d_start, (void *) d_yoff, (void *) d_len, (void *) d_left, (void *) d_y,
                    (void *) d_fit, (void *) d_parts, (void *) d_list})
        pb.arena.release(p);
    return MGPU_OK;
}

}  // namespace mgpu
