// omx_ir.hip -- FP64 kernels of the iterative refinement: the on-the-fly
// residual GEMV (A regenerated from the LCG), infinity norms, vector ops and
// the blocked triangular solves with the FP32 LU factors.
#include <float.h>

#include <mutex>

#include "omx_common.hpp"

// Partial sums of omx_otf_gemv_f64_noalloc: the device memory that entry
// point uses in place of a caller's workspace.  64 MiB covers every order n
// (the residual GEMV's largest need is two column segments at n = 4194048,
// 67104768 bytes).  Each GPU the library runs on holds its own copy from
// module load until the process ends.  Host code never passes this name to a
// kernel (on the host it is only a stand-in for the symbol): it passes the
// device address hipGetSymbolAddress returns for the current device.
constexpr size_t kNoAllocScratchBytes = (size_t)64 << 20;
static __device__ __align__(256) double scratch[kNoAllocScratchBytes / sizeof(double)];

namespace {

constexpr int kGemvRows = 256;     // rows per workgroup (one per thread)
constexpr int kGemvTargetWG = 16384;
constexpr int kGemvMaxSeg = 64;

// Number of column segments of the residual GEMV for order n: enough
// workgroups to fill the 256 CUs several times, each segment >= 64 columns
// (the jump to a segment's first column costs about as much as 30 columns'
// steps).  At n = 1024 segments of 256 columns left 15 of 16 SIMDs without a
// wave, and the columns of the diagonal, a load and a step at a time,
// took longer than all others: 22.4 us, 10.6 now; 5120 29.0 -> 20, 10240 48 -> 39.
// mincols = 256: the fewer segments of a call with a smaller workspace.
int gemv_segments(int64_t n, int64_t mincols = 64) {
    const int64_t nrb = omx_cdiv(n, kGemvRows);
    int64_t s = omx_cdiv(kGemvTargetWG, nrb);
    if (s > kGemvMaxSeg) s = kGemvMaxSeg;
    const int64_t smax = omx_cdiv(n, mincols);
    if (s > smax) s = smax;
    if (s < 1) s = 1;
    return (int)s;
}

// The generator's state with its top bit flipped, t = s + 2^63 mod 2^64, steps
// by the same map as s (its multiplier is odd).  2^-64 double(int64(s)) from it
// (the factor keeps the sums within the range that the entries' have):
// 2^-64 times 2^52 + lo and 2^84 + 2^32 hi are t's halves under constant high
// words, and 2^-64 ((2^84 + 2^32 hi) - (2^84 + 2^63 + 2^52)) is exact, so the
// last addition rounds the exact integer once, as the conversion does.
__device__ __forceinline__ double otf_int(uint64_t t) {
    const double lo = __builtin_bit_cast(double, 0x3F30000000000000ull | (uint32_t)t);
    const double hi = __builtin_bit_cast(double, 0x4130000000000000ull | (t >> 32));
    return (hi - 0x1.00000801p20) + lo;  // 2^20 + 2^-1 + 2^-12
}

// acc += 2^-64 int64(s_ij) x_j for the columns j of [j0, j1), in column order, the
// row's state t stepping by the map jn per column (t leaves as the state of
// column j1).  The entries' common factor is applied to the sum, and the
// conversion above takes two additions in place of two conversions, which run
// at half the rate, and an FMA.  Four columns per trip with a 32-bit trip
// count: the loop test is scalar, the state copies amortised.
// n = 40960, with the copy and the norm of a refinement step: 468 us with
// converted and scaled entries, 379 now (and a rounding less per entry).
// kDiag: column j0 + skip (the row's diagonal, where it is one of these) is
// left out.
template <bool kDiag>
__device__ __forceinline__ void otf_columns(uint64_t &t, double &acc, omx_map jn, const double *__restrict__ x,
                                            int64_t j0, int64_t j1, int skip = -1) {
    const double *__restrict__ xp = x + j0;
    const int cnt = (int)(j1 - j0);
    auto add = [&](int c, uint64_t tc, double xc) {
        const double sum = __builtin_fma(otf_int(tc), xc, acc);
        acc = kDiag && c == skip ? acc : sum;
    };
    int c = 0;
    for (; c + 4 <= cnt; c += 4) {
        const uint64_t t1 = omx_apply(jn, t);
        const uint64_t t2 = omx_apply(jn, t1);
        const uint64_t t3 = omx_apply(jn, t2);
        const double x0 = xp[c], x1 = xp[c + 1], x2 = xp[c + 2], x3 = xp[c + 3];
        add(c, t, x0);
        add(c + 1, t1, x1);
        add(c + 2, t2, x2);
        add(c + 3, t3, x3);
        t = omx_apply(jn, t3);
    }
    for (; c < cnt; ++c) {
        add(c, t, xp[c]);
        t = omx_apply(jn, t);
    }
}

// Row i of the workgroup's 256-row block, columns [c0, c1): walk along the
// row with the map a^n (one affine step per column).  The diagonal column
// takes diag[i] instead of the LCG value (otf_gemv_diag_d,
// panel_gemv.hpp:13-47).  part[seg*n + i] = the segment's FP64 sum, or, with
// a single segment, y_i += alpha * sum directly.
__global__ void __launch_bounds__(kGemvRows)
k_otf_gemv(int64_t n, uint64_t x00, omx_map jn, const double *__restrict__ diag,
           const double *__restrict__ x, int64_t seglen, double *__restrict__ part,
           double *__restrict__ y, double alpha) {
    const int64_t i = (int64_t)blockIdx.x * kGemvRows + threadIdx.x;
    const int64_t seg = blockIdx.y;
    const int64_t c0 = seg * seglen;
    int64_t c1 = c0 + seglen;
    if (c1 > n) c1 = n;
    if (i >= n) return;
    uint64_t t = omx_apply(omx_jump((uint64_t)i + (uint64_t)n * (uint64_t)c0), x00) ^ (1ull << 63);
    double acc = 0.0;
    // diagonal columns of this row block
    const int64_t d0 = (int64_t)blockIdx.x * kGemvRows;
    const int64_t d1 = d0 + kGemvRows;
    // c0 <= lo <= hi <= c1
    const int64_t lo = c0 > d0 ? c0 : (d0 < c1 ? d0 : c1);
    const int64_t hi = c1 < d1 ? (c1 > lo ? c1 : lo) : (d1 > lo ? d1 : lo);
    otf_columns<false>(t, acc, jn, x, c0, lo);
    otf_columns<true>(t, acc, jn, x, lo, hi, (int)(i - lo));
    otf_columns<false>(t, acc, jn, x, hi, c1);
    acc *= 0x1.fffffffffffffp-1;  // the rest of RandStat's scale (omx_lcg_value)
    if (i >= lo && i < hi) acc = __builtin_fma(diag[i], x[i], acc);
    if (part)
        part[seg * n + i] = acc;
    else
        y[i] = y[i] + alpha * acc;
}

__global__ void k_gemv_reduce(int64_t n, int nseg, const double *__restrict__ part,
                              double *__restrict__ y, double alpha) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    // eight loads in flight: one after the other 64 segments took 12 us
    double s = part[i];
    int q = 1;
    for (; q + 8 <= nseg; q += 8) {
        double v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = part[(int64_t)(q + e) * n + i];
#pragma unroll
        for (int e = 0; e < 8; ++e) s += v[e];
    }
    for (; q < nseg; ++q) s += part[(int64_t)q * n + i];
    y[i] = y[i] + alpha * s;
}

__global__ void __launch_bounds__(1024)
k_norm_inf(int64_t n, const double *__restrict__ x, double *__restrict__ out) {
    __shared__ double sh[1024];
    double m = 0.0;
    for (int64_t i = threadIdx.x; i < n; i += 1024) m = fmax(m, fabs(x[i]));
    sh[threadIdx.x] = m;
    __syncthreads();
    for (int w = 512; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) sh[threadIdx.x] = fmax(sh[threadIdx.x], sh[threadIdx.x + w]);
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = sh[0];
}

__global__ void k_copy(int64_t n, const double *__restrict__ x, double *__restrict__ y) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        y[i] = x[i];
}

__global__ void k_div(int64_t n, const double *__restrict__ b, const double *__restrict__ d,
                      double *__restrict__ x) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        x[i] = b[i] / d[i];
}

__global__ void k_axpy(int64_t n, double alpha, const double *__restrict__ x,
                       double *__restrict__ y) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        y[i] = y[i] + alpha * x[i];
}

// ---------------------------------------------------------------------------
// Triangular solves with the FP32 factors, FP64 vector and arithmetic,
// without a workspace (or too small, or unaligned): one launch per 256 columns.
//
// The matrix is walked in blocks of kTB = 256 rows/columns.  One launch per
// block column J (solved values x_J final in x), workgroups of 1024
// threads (16 waves):
//   workgroup 0   rows of the next diagonal block D: r_D -= M(D, J) x_J, then
//                 D is solved in LDS: four sub-blocks of 64, each a 64-step
//                 lane-to-lane chain in one wave, while twelve more waves
//                 fold each solved sub-block into the later sub-blocks' rows;
//   workgroup w   the remaining rows beyond D, 256 per workgroup:
//                 r -= M(rows, J) x_J.
// A wave takes 16 of the 256 columns: its sixteen 16-byte loads per lane
// are in flight together, so a workgroup's 256 KB of the factor arrive in
// one round trip and the launch is bound by HBM rather than by the latency
// of one workgroup's reads.  Summation order per row and block column: each
// wave sums its 16 columns in order, the 16 partial sums are added in wave
// order, the total is subtracted from r.  Every FP32 factor entry is read
// once (2 n^2 bytes per triangle).
// ---------------------------------------------------------------------------
constexpr int kTB = 256;
constexpr int kSB = 64;
constexpr int kTW = 16;         // waves per workgroup
constexpr int kTT = 64 * kTW;   // threads per workgroup
constexpr int kTC = kTB / kTW;  // columns per wave

typedef float f32x4 __attribute__((ext_vector_type(4)));

struct TrsvShared {
    double xv[kTB];          // x_J
    double xs[kTB];          // r_D, then x_D
    double part[kTW][kTB];   // per-wave partial sums of rows_dot
    double pp[4][4][kSB];    // diagonal block: [sub-block][column chunk][row] sums
};

// Lane l's value of v in every lane (l uniform): two readlanes.
__device__ __forceinline__ double bcast_lane(double v, int l) {
    const uint64_t u = __builtin_bit_cast(uint64_t, v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, l);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(u >> 32), l);
    return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// sum over the block's ncols <= 256 columns from c0 of M(row, c) x_c for
// the 256 rows from r0 (rows >= rmax ignored); sh.xv holds x of the
// columns.  Wave w takes columns [16 w, 16 w + 16), lane l rows 4l .. 4l+3
// (one 16-byte load per column when kVec).  Returns the row's total in
// thread t = row - r0 for t < 256 (0 elsewhere).
template <bool kVec>
__device__ __forceinline__ double rows_dot(const float *__restrict__ A, int64_t lda, int64_t r0, int64_t rmax,
                                           int64_t c0, int ncols, TrsvShared &sh) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int cb = wave * kTC;
    const int ce = min(ncols, cb + kTC);
    const int64_t row = r0 + 4 * lane;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    if (kVec && row + 3 < rmax) {
        const float *p = A + row + (c0 + cb) * lda;
        if (ce - cb == kTC) {
            f32x4 v[kTC];
#pragma unroll
            for (int u = 0; u < kTC; ++u) v[u] = *reinterpret_cast<const f32x4 *>(p + (int64_t)u * lda);
#pragma unroll
            for (int u = 0; u < kTC; ++u) {
                const double xc = sh.xv[cb + u];
                s0 = __builtin_fma((double)v[u].x, xc, s0);
                s1 = __builtin_fma((double)v[u].y, xc, s1);
                s2 = __builtin_fma((double)v[u].z, xc, s2);
                s3 = __builtin_fma((double)v[u].w, xc, s3);
            }
        } else {
            for (int c = cb; c < ce; ++c) {
                const f32x4 v = *reinterpret_cast<const f32x4 *>(p + (int64_t)(c - cb) * lda);
                const double xc = sh.xv[c];
                s0 = __builtin_fma((double)v.x, xc, s0);
                s1 = __builtin_fma((double)v.y, xc, s1);
                s2 = __builtin_fma((double)v.z, xc, s2);
                s3 = __builtin_fma((double)v.w, xc, s3);
            }
        }
    } else {
        for (int c = cb; c < ce; ++c) {
            const float *q = A + row + (c0 + c) * lda;
            const double xc = sh.xv[c];
            if (row < rmax) s0 = __builtin_fma((double)q[0], xc, s0);
            if (row + 1 < rmax) s1 = __builtin_fma((double)q[1], xc, s1);
            if (row + 2 < rmax) s2 = __builtin_fma((double)q[2], xc, s2);
            if (row + 3 < rmax) s3 = __builtin_fma((double)q[3], xc, s3);
        }
    }
    sh.part[wave][4 * lane] = s0;
    sh.part[wave][4 * lane + 1] = s1;
    sh.part[wave][4 * lane + 2] = s2;
    sh.part[wave][4 * lane + 3] = s3;
    __syncthreads();
    double t = 0.0;
    if (tid < kTB) {
        t = sh.part[0][tid];
#pragma unroll
        for (int w = 1; w < kTW; ++w) t += sh.part[w][tid];
    }
    __syncthreads();
    return t;
}

// x_D <- T_DD^-1 r_D for the diagonal block at d0 of order dim (<= 256),
// unit lower (kUpper false, sub-blocks first to last) or upper non-unit
// (kUpper, last to first); r_D in sh.xs.  Roles:
//   waves 0-3    wave s runs sub-block s's 64-step chain at stage s (lane l:
//                row 64 s + l, its 64 entries of the diagonal sub-block in
//                registers, x_c read from lane c);
//   waves 4-15   wave 4 + 4 j + c accumulates, for the rows of target
//                sub-block t (lower t = j + 1, upper t = j), the products
//                with columns [16 c, 16 c + 16) of every sub-block solved
//                before t, each right after that sub-block's stage, and
//                hands its sum to t's chain, which subtracts the four chunk
//                sums (in chunk order) before it starts.
// All factor entries are loaded at the start, with row and column indices
// clamped into the block so every load is unconditional; entries outside
// the block meet x = 0 or are masked.  The upper chain divides by u_ii as
// q0 = r y, q = q0 + (r - u q0) y with y = RN(1/u): the correctly rounded
// quotient (Markstein's correction with a correctly rounded reciprocal).
template <bool kUpper>
__device__ __forceinline__ void diag_solve(const float *__restrict__ A, int64_t lda, int64_t d0, int dim,
                                           TrsvShared &sh) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nsb = (dim + kSB - 1) / kSB;
    const float *D = A + d0 + d0 * lda;
    const bool chain = wave < 4;
    const int t = chain ? wave : (kUpper ? (wave - 4) / 4 : 1 + (wave - 4) / 4);
    const int c = (wave - 4) & 3;
    const int i = kSB * t + lane;
    const float *Drow = D + min(i, dim - 1);
    float w[kSB];
    float ud = 1.0f;
    if (t < nsb) {
        if (chain) {
#pragma unroll
            for (int q = 0; q < kSB; ++q) w[q] = Drow[(int64_t)min(kSB * t + q, dim - 1) * lda];
            if (kUpper) ud = Drow[(int64_t)min(i, dim - 1) * lda];
            // lower: multipliers outside the triangle or past the block are
            // zeroed now, so that the chain's dependent steps carry no
            // selects (in the upper solve this spills; it selects in the
            // chain)
            if (!kUpper) {
#pragma unroll
                for (int q = 0; q < kSB; ++q) w[q] = (lane > q && i < dim) ? w[q] : 0.0f;
            }
        } else {
            // source sub-block s at slot s (lower, s < t) or s - 1 (upper, s > t)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const int s = kUpper ? k + 1 : k;
                if (kUpper ? (s > t && s < nsb) : s < t) {
#pragma unroll
                    for (int u = 0; u < kTC; ++u)
                        w[kTC * k + u] = Drow[(int64_t)min(kSB * s + kTC * c + u, dim - 1) * lda];
                }
            }
        }
    }
    double acc = 0.0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int st = kUpper ? 3 - k : k;
        if (st >= nsb) continue;
        if (chain && st == t) {
            const int c0 = kSB * st;
            const bool fed = kUpper ? st < nsb - 1 : st > 0;
            double v = (i < dim) ? sh.xs[i] : 0.0;
            if (fed) v -= ((sh.pp[st][0][lane] + sh.pp[st][1][lane]) + sh.pp[st][2][lane]) + sh.pp[st][3][lane];
            if (kUpper) {
                // the multipliers outside the triangle or past the block are
                // zeroed in place first (so the chain's steps carry no
                // selects; masking them with the loads spills here)
#pragma unroll
                for (int q = 0; q < kSB; ++q) {
                    float wq = (lane < q && c0 + q < dim) ? w[q] : 0.0f;
                    asm volatile("" : "+v"(wq));
                    w[q] = wq;
                }
                const double u = (i < dim) ? (double)ud : 1.0;
                const double y = 1.0 / u;
                auto quot = [&](double r) {
                    const double q0 = r * y;
                    return __builtin_fma(__builtin_fma(-u, q0, r), y, q0);
                };
                // step q: every lane forms its quotient, lane q's is x_q;
                // rows above subtract x_q u(i, q).  Lane q's own v is
                // untouched from then on, so its final quotient equals x_q.
#pragma unroll
                for (int q = kSB - 1; q >= 0; --q) v = __builtin_fma(-bcast_lane(quot(v), q), (double)w[q], v);
                v = quot(v);
            } else {
#pragma unroll
                for (int q = 0; q < kSB; ++q) {
                    // converted in place (hoisting all 64 conversions would
                    // take 128 registers)
                    float wq = w[q];
                    asm volatile("" : "+v"(wq));
                    v = __builtin_fma(-bcast_lane(v, q), (double)wq, v);
                }
            }
            if (i < dim) sh.xs[i] = v;
        }
        __syncthreads();
        if (!chain && t < nsb && (kUpper ? st > t : st < t)) {
            const int slot = kUpper ? st - 1 : st;
            const int cb = kSB * st + kTC * c;
            // four entries at a time: the scheduler must not convert all 16
            // up front (that would spill in the upper solve)
#pragma unroll
            for (int u = 0; u < kTC; ++u) {
                acc = __builtin_fma((double)w[kTC * slot + u], sh.xs[cb + u], acc);
                if ((u & 3) == 3) __builtin_amdgcn_sched_barrier(0);
            }
            if (st == (kUpper ? t + 1 : t - 1)) sh.pp[t][c][lane] = acc;
        }
        __syncthreads();
    }
}

// One block column of the forward solve.  j0 = first column of the solved
// block J (j0 < 0: nothing solved yet, only the first diagonal block).
template <bool kVec>
__global__ void __launch_bounds__(kTT)
k_trsv_lower_step(int64_t n, int64_t j0, const float *__restrict__ A, int64_t lda, double *__restrict__ x) {
    __shared__ TrsvShared sh;
    const int tid = threadIdx.x;
    const int64_t jb = j0 < 0 ? 0 : j0;
    const int ncols = j0 < 0 ? 0 : (int)min((int64_t)kTB, n - j0);
    const int64_t d0 = j0 < 0 ? 0 : j0 + kTB;
    if (ncols > 0 && tid < kTB) sh.xv[tid] = tid < ncols ? x[jb + tid] : 0.0;
    __syncthreads();
    if (blockIdx.x == 0) {
        const int dim = (int)min((int64_t)kTB, n - d0);
        const double t = ncols > 0 ? rows_dot<kVec>(A, lda, d0, d0 + dim, jb, ncols, sh) : 0.0;
        if (tid < kTB) sh.xs[tid] = (tid < dim) ? x[d0 + tid] - t : 0.0;
        __syncthreads();
        diag_solve<false>(A, lda, d0, dim, sh);
        if (tid < dim) x[d0 + tid] = sh.xs[tid];
        return;
    }
    const int64_t r0 = d0 + (int64_t)blockIdx.x * kTB;
    const double t = rows_dot<kVec>(A, lda, r0, n, jb, ncols, sh);
    if (tid < kTB && r0 + tid < n) x[r0 + tid] -= t;
}

// One block column of the backward solve: J = [j0, j0 + ncols) solved
// (j0 >= n: nothing solved yet, only the last diagonal block, which may be
// shorter than kTB); D = the block before J; rows [0, d0) updated.
template <bool kVec>
__global__ void __launch_bounds__(kTT)
k_trsv_upper_step(int64_t n, int64_t j0, const float *__restrict__ A, int64_t lda, double *__restrict__ x) {
    __shared__ TrsvShared sh;
    const int tid = threadIdx.x;
    const int64_t last0 = ((n - 1) / kTB) * kTB;  // first row of the last block
    const bool none = j0 >= n;
    const int ncols = none ? 0 : (int)min((int64_t)kTB, n - j0);
    const int64_t d0 = none ? last0 : j0 - kTB;
    const int dim = (int)min((int64_t)kTB, n - d0);
    if (ncols > 0 && tid < kTB) sh.xv[tid] = tid < ncols ? x[j0 + tid] : 0.0;
    __syncthreads();
    if (blockIdx.x == 0) {
        const double t = ncols > 0 ? rows_dot<kVec>(A, lda, d0, d0 + dim, j0, ncols, sh) : 0.0;
        if (tid < kTB) sh.xs[tid] = (tid < dim) ? x[d0 + tid] - t : 0.0;
        __syncthreads();
        diag_solve<true>(A, lda, d0, dim, sh);
        if (tid < dim) x[d0 + tid] = sh.xs[tid];
        return;
    }
    const int64_t r0 = (int64_t)(blockIdx.x - 1) * kTB;
    const double t = rows_dot<kVec>(A, lda, r0, d0, j0, ncols, sh);
    if (tid < kTB && r0 + tid < d0) x[r0 + tid] -= t;
}

// ---------------------------------------------------------------------------
// The same solves in one launch, with a workspace: rows in blocks of 256,
// workgroup by workgroup (a ticket each, in solution order: a workgroup only
// waits for blocks whose tickets were taken before its own, so whatever is
// resident, the first unfinished block never waits).  For its block row I a
// workgroup
//   1. keeps its diagonal block in LDS and registers, none of which needs x;
//   2. adds up M(I, J) x_J in registers for J in solution order as the x_J
//      appear; the next 256 x 256 tile of M is loaded while it waits;
//   3. solves x_I by substitution, 16 rows a phase, a wave each: the rows'
//      triangle in the lanes (tri16_solve), then their products with the later
//      waves' rows; and publishes it.
// Published values are their own flags: xs starts as kUnset, a NaN that no
// result is published as; readers poll it with device-scope loads.
// The launch per 256 columns it replaces took 14 (lower) and 18 us (upper)
// however few rows were left: launch, 256 KB through one CU, and 256
// dependent steps.  A block now takes 7 us from x_J to x_I: hand-over between
// XCDs 0.5, the last tile 0.5, sums 1.0, 16 phases of 0.3 (16 FMAs 0.1, the
// way to the next wave through LDS and the sums of its lanes 0.2).  Products
// with FP64 inverses of the 64 x 64 diagonal sub-blocks in place of the
// substitution took 5 to 6 us, but are not backward stable: with factors of a
// randsvd system of condition 1e6 a row was off by 3e-12 of its terms' sum,
// which substitution keeps at 3e-16 (per-block launches 4e-16), and with one
// pivot of 1e-12 by 1e-5.  Where the matrix is large the tiles' traffic bounds
// it (figures at trsv_launch).
// ---------------------------------------------------------------------------
constexpr uint64_t kUnset = 0x7FF4A5A5D00D5EEDull;  // a signalling NaN: arithmetic quiets it
constexpr int kOffSub = kSB * kSB;                  // entries of a sub-block between the diagonal ones
constexpr int kT16 = 20;                            // row stride of a staged 16 x 16 triangle

struct __align__(16) TrsvFused {
    double xd[kTB];                // x_I (first: its reads have no address to form)
    double rd[kTB];                // r_I less what is known
    double xv[2][kTB];             // x_J, alternating
    double part[kTW][kTB];         // per-wave sums of step 2
    float t16[kTW][16][kT16];      // the 16 x 16 triangles on the diagonal, negated: [block][row][column]
    float off[6][kOffSub];         // sub-blocks (t, s) at slot off_slot: [c 64 + (r ^ 16 (c % 4))]
    int ticket;
};

// slot of the sub-block in block row t, block column s (s < t lower, s > t upper)
__device__ __forceinline__ int off_slot(int t, int s) {
    const int hi = t > s ? t : s, lo = t > s ? s : t;
    return hi * (hi - 1) / 2 + lo;
}

__global__ void __launch_bounds__(256) k_trsv_reset(int64_t n, uint64_t *__restrict__ xs, int *__restrict__ ticket) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) xs[i] = kUnset;
    if (blockIdx.x == 0 && threadIdx.x == 0) *ticket = 0;
}

// v summed over the lanes l, l ^ 16, l ^ 32, l ^ 48, in every one of them:
// row (16 lanes) and half swaps in the VALU (a shuffle goes through LDS)
__device__ __forceinline__ double sum_groups(double v) {
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    uint64_t u = __builtin_bit_cast(uint64_t, v);
    u32x2 lo = __builtin_amdgcn_permlane16_swap((unsigned)u, (unsigned)u, false, false);
    u32x2 hi = __builtin_amdgcn_permlane16_swap((unsigned)(u >> 32), (unsigned)(u >> 32), false, false);
    v = __builtin_bit_cast(double, (uint64_t)hi[0] << 32 | lo[0]) + __builtin_bit_cast(double, (uint64_t)hi[1] << 32 | lo[1]);
    u = __builtin_bit_cast(uint64_t, v);
    lo = __builtin_amdgcn_permlane32_swap((unsigned)u, (unsigned)u, false, false);
    hi = __builtin_amdgcn_permlane32_swap((unsigned)(u >> 32), (unsigned)(u >> 32), false, false);
    return __builtin_bit_cast(double, (uint64_t)hi[0] << 32 | lo[0]) +
           __builtin_bit_cast(double, (uint64_t)hi[1] << 32 | lo[1]);
}

// v += x m with x of lane q of the lane's row of 16: one FMA, whose DPP form
// reads x across the row (after two wait states if x was just written)
#define OMX_ROW_FMA(v, x, m, q) "s_nop 1\n\tv_fmac_f64_dpp " v ", " x ", " m " row_newbcast:" q " row_mask:0xf bank_mask:0xf\n\t"

// Substitution with a 16 x 16 unit triangle: lane i of each row of 16 lanes
// holds entry i of the right-hand side v and the negated row i of the triangle,
// zero on and outside its diagonal: entries solved before stay as they are.
// (One asm block: between two the compiler puts a wait state more.)
template <bool kUpper>
__device__ __forceinline__ double tri16_solve(double v, const double (&nt)[16]) {
    if (kUpper)
        asm(OMX_ROW_FMA("%0", "%0", "%1", "15") OMX_ROW_FMA("%0", "%0", "%2", "14") OMX_ROW_FMA("%0", "%0", "%3", "13")
            OMX_ROW_FMA("%0", "%0", "%4", "12") OMX_ROW_FMA("%0", "%0", "%5", "11") OMX_ROW_FMA("%0", "%0", "%6", "10")
            OMX_ROW_FMA("%0", "%0", "%7", "9") OMX_ROW_FMA("%0", "%0", "%8", "8") OMX_ROW_FMA("%0", "%0", "%9", "7")
            OMX_ROW_FMA("%0", "%0", "%10", "6") OMX_ROW_FMA("%0", "%0", "%11", "5") OMX_ROW_FMA("%0", "%0", "%12", "4")
            OMX_ROW_FMA("%0", "%0", "%13", "3") OMX_ROW_FMA("%0", "%0", "%14", "2") OMX_ROW_FMA("%0", "%0", "%15", "1")
            : "+&v"(v)
            : "v"(nt[15]), "v"(nt[14]), "v"(nt[13]), "v"(nt[12]), "v"(nt[11]), "v"(nt[10]), "v"(nt[9]), "v"(nt[8]),
              "v"(nt[7]), "v"(nt[6]), "v"(nt[5]), "v"(nt[4]), "v"(nt[3]), "v"(nt[2]), "v"(nt[1]));
    else
        asm(OMX_ROW_FMA("%0", "%0", "%1", "0") OMX_ROW_FMA("%0", "%0", "%2", "1") OMX_ROW_FMA("%0", "%0", "%3", "2")
            OMX_ROW_FMA("%0", "%0", "%4", "3") OMX_ROW_FMA("%0", "%0", "%5", "4") OMX_ROW_FMA("%0", "%0", "%6", "5")
            OMX_ROW_FMA("%0", "%0", "%7", "6") OMX_ROW_FMA("%0", "%0", "%8", "7") OMX_ROW_FMA("%0", "%0", "%9", "8")
            OMX_ROW_FMA("%0", "%0", "%10", "9") OMX_ROW_FMA("%0", "%0", "%11", "10") OMX_ROW_FMA("%0", "%0", "%12", "11")
            OMX_ROW_FMA("%0", "%0", "%13", "12") OMX_ROW_FMA("%0", "%0", "%14", "13") OMX_ROW_FMA("%0", "%0", "%15", "14")
            : "+&v"(v)
            : "v"(nt[0]), "v"(nt[1]), "v"(nt[2]), "v"(nt[3]), "v"(nt[4]), "v"(nt[5]), "v"(nt[6]), "v"(nt[7]),
              "v"(nt[8]), "v"(nt[9]), "v"(nt[10]), "v"(nt[11]), "v"(nt[12]), "v"(nt[13]), "v"(nt[14]));
    return v;
}

// The same where an entry is infinite or NaN, which times a zero multiplier is
// no 0: solved entries are left by selection.  nt: the lane's negated row of
// the triangle in LDS, not scaled; u: its diagonal (lower: 1).
template <bool kUpper>
__device__ __forceinline__ double tri16_select(double v, int i16, const float *nt, double u) {
#pragma unroll 1
    for (int q = 0; q < 16; ++q) {
        const int c = kUpper ? 15 - q : q;
        const double d = __builtin_fma(__shfl(kUpper ? v / u : v, c, 16), (double)nt[c], v);
        v = (kUpper ? i16 < c : i16 > c) ? d : v;
    }
    return kUpper ? v / u : v;
}

// Barrier that orders LDS accesses only: __syncthreads() would also wait for
// the tile loads in flight and, after a publication, for its way to memory
// (1.5 us a stage).
__device__ __forceinline__ void lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <bool kUpper>
__global__ void __launch_bounds__(kTT)
k_trsv_fused(int64_t n, const float *__restrict__ A, int64_t lda, double *__restrict__ x, uint64_t *xs, int *ticket) {
    __shared__ TrsvFused sh;
    const int64_t nb = omx_cdiv(n, kTB);
    for (;;) {
        // (opaque: a hundred addresses derived from it, computed once before
        // the loop, would live through it in scratch memory)
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int lane = tid & 63, i16 = lane & 15, g = lane >> 4;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        lds_sync();
        if (tid == 0) sh.ticket = atomicAdd(ticket, 1);
        lds_sync();
        const int64_t t = sh.ticket;
        if (t >= nb) return;
        const int64_t I = kUpper ? nb - 1 - t : t;
        const int64_t d0 = I * kTB;
        const int dim = (int)min((int64_t)kTB, n - d0);
        const float *D = A + d0 + d0 * lda;
        // ---- 1. the diagonal block: this wave's rows 16 wave .. + 15, lane
        // (i16, g) row i16.  Their triangle goes to LDS; sub[c][b]: columns
        // 4 b + g of the 16 x 16 block left (right) of it that is solved c-th
        // in the 64 x 64 sub-block.  Rows and columns past the matrix: the
        // identity ----
        const int k4 = wave >> 2, rb = wave & 3, row = 16 * wave + i16;
        float sub[3][4], ud = 1.0f;
        {
            const float *Drow = D + min(row, dim - 1);
            auto entry = [&](int c, bool in) {
                const float e = Drow[(int64_t)min(c, dim - 1) * lda];
                return in && row < dim && c < dim ? e : 0.0f;
            };
            f32x4 t;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                t[j] = -entry(16 * wave + 4 * g + j, kUpper ? 4 * g + j > i16 : 4 * g + j < i16);
            *reinterpret_cast<f32x4 *>(&sh.t16[wave][i16][4 * g]) = t;
            if (kUpper && row < dim) ud = Drow[(int64_t)row * lda];
#pragma unroll
            for (int c = 0; c < 3; ++c)
#pragma unroll
                for (int b = 0; b < 4; ++b) sub[c][b] = entry(kSB * k4 + 16 * (kUpper ? 3 - c : c) + 4 * b + g, true);
        }
#pragma unroll
        for (int q = 0; q < 6; ++q) {
            const int hi = q < 1 ? 1 : (q < 3 ? 2 : 3), lo = q - hi * (hi - 1) / 2;
            const int rt = kSB * (kUpper ? lo : hi), ct = kSB * (kUpper ? hi : lo);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int c = wave + 16 * e;
                const bool in = rt + lane < dim && ct + c < dim;
                const float v = D[min(rt + lane, dim - 1) + (int64_t)min(ct + c, dim - 1) * lda];
                sh.off[q][c * kSB + (lane ^ ((c & 3) << 4))] = in ? v : 0.0f;
            }
        }
        const double r_in = tid < dim ? x[d0 + tid] : 0.0;
        // ---- 2. the block row's products ----
        // The tiles' sums are added with what each addition rounds off (two-sum)
        // kept in LDS, so that the error is no larger than when every block
        // column was taken off the rows by itself: as one sum of n / 16 terms a
        // wave, solutions of systems of condition 1e4 were 1.4 to 3 times as
        // far off.
        double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
        double *part = &sh.part[wave][4 * lane];
        part[0] = part[1] = part[2] = part[3] = 0.0;
        auto add = [](double &s, double &e, double t) {
            const double d = s + t, b = d - s, r = (s - (d - b)) + (t - b);
            e += fabs(r) < __builtin_inf() ? r : 0.0;  // (an infinite sum stays one)
            s = d;
        };
        // (rows past the matrix, in the lower solve's last block, read within
        // the column's padding, and not the last column's; their sums are not
        // used.  The upper solve's first block, whose tile holds the last
        // column, is read within the matrix and not used)
        const float *rows = A + min(d0 + 4 * lane, (kUpper ? n - 4 : n - 1) & ~(int64_t)3);
        f32x4 v[kTC];
        auto load_tile = [&](int64_t J) {
            const int64_t c0 = J * kTB + kTC * wave;
            const float *p = rows + min(c0, n - 1) * lda;
            const int64_t cmax = n - 1 - c0;  // (columns past the matrix: the last one, times x = 0)
            if (cmax >= kTC - 1) {
#pragma unroll
                for (int u = 0; u < kTC; ++u) v[u] = *reinterpret_cast<const f32x4 *>(p + u * lda);
            } else {
#pragma unroll
                for (int u = 0; u < kTC; ++u)
                    v[u] = *reinterpret_cast<const f32x4 *>(p + max(min((int64_t)u, cmax), (int64_t)0) * lda);
            }
        };
        load_tile(kUpper ? nb - 1 : 0);  // (the first block has no use for it)
        for (int64_t b = 0; b < t; ++b) {
            const int64_t J = kUpper ? nb - 1 - b : b;
            double *xv = sh.xv[b & 1];
            if (tid < kTB) {
                uint64_t w = 0;
                if (J * kTB + tid < n) {
                    const uint64_t *src = xs + J * kTB + tid;
                    w = __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    while (w == kUnset) {
                        // the further off, the less often
                        if (t - b > 2) __builtin_amdgcn_s_sleep(24);
                        else if (t - b > 1) __builtin_amdgcn_s_sleep(6);
                        w = __hip_atomic_load(src, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
                }
                xv[tid] = __builtin_bit_cast(double, w);
            }
            lds_sync();
            const int64_t Jn = kUpper ? J - 1 : J + 1;
            const bool more = b + 1 < t;
            // (each tile summed by itself)
            double t0 = 0.0, t1 = 0.0, t2 = 0.0, t3 = 0.0;
#pragma unroll
            for (int u = 0; u < kTC; ++u) {
                const double xc = xv[kTC * wave + u];
                t0 = __builtin_fma((double)v[u].x, xc, t0);
                t1 = __builtin_fma((double)v[u].y, xc, t1);
                t2 = __builtin_fma((double)v[u].z, xc, t2);
                t3 = __builtin_fma((double)v[u].w, xc, t3);
                if ((u & 3) == 3) {
                    // (four columns' factors at a time in registers)
                    asm volatile("" : "+v"(t0), "+v"(t1), "+v"(t2), "+v"(t3)::"memory");
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            add(s0, part[0], t0);
            add(s1, part[1], t1);
            add(s2, part[2], t2);
            add(s3, part[3], t3);
            if (more) load_tile(Jn);
        }
        part[0] += s0;
        part[1] += s1;
        part[2] += s2;
        part[3] += s3;
        lds_sync();
        if (tid < kTB) {
            double q[kTW];
#pragma unroll
            for (int w = 0; w < kTW; ++w) q[w] = sh.part[w][tid];
            __builtin_amdgcn_sched_barrier(0);  // (all reads in flight)
#pragma unroll
            for (int w = 1; w < kTW; ++w) q[0] += q[w];
            sh.rd[tid] = tid < dim ? r_in - q[0] : 0.0;
        }
        lds_sync();
        // ---- 3. x_I: phase p solves 16 rows by substitution in their wave
        // and takes them off the rows of the later waves (whose sums wait) ----
        // The upper solve's rows are scaled by their diagonals beforehand (the
        // right-hand side divided, as diag_solve's quotient), so that its
        // chain is one FMA an entry too.
        const double r_own = sh.rd[row], u = (double)ud, y = kUpper ? 1.0 / u : 1.0;
        double nt[16], acc = 0.0;  // acc: this lane's share of what its row loses to solved rows
#pragma unroll
        for (int j = 0; j < 16; j += 4) {
            const f32x4 t = *reinterpret_cast<const f32x4 *>(&sh.t16[wave][i16][j]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                nt[j + e] = kUpper ? (double)t[e] * y : (double)t[e];
                asm volatile("" : "+v"(nt[j + e]));  // (converted now, not in the chain)
            }
        }
        const int own = kUpper ? 15 - wave : wave;  // this wave's phase
        // phase p: the products with the rows it solves, of which o are this
        // lane's four entries
        auto wait = [&](int p, const float (&o)[4]) {
            double m[4], xc[4];
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                m[b] = (double)o[b];
                asm volatile("" : "+v"(m[b]));
            }
            const double *xd = sh.xd + 16 * (kUpper ? 15 - p : p) + g;
            lds_sync();
            if (p == own - 1) __builtin_amdgcn_s_setprio(3);
#pragma unroll
            for (int b = 0; b < 4; ++b) xc[b] = xd[4 * b];
            acc += __builtin_fma(m[1], xc[1], m[0] * xc[0]) + __builtin_fma(m[3], xc[3], m[2] * xc[2]);
        };
#pragma unroll 1
        for (int p = 0; p < (own & ~3); ++p) {  // other sub-blocks
            const int wp = kUpper ? 15 - p : p;
            const float *src = sh.off[off_slot(k4, wp >> 2)] + (16 * (wp & 3) + g) * kSB + ((16 * rb + i16) ^ (g << 4));
            const float o[4] = {src[0], src[4 * kSB], src[8 * kSB], src[12 * kSB]};
            wait(p, o);
        }
#pragma unroll
        for (int c = 0; c < 3; ++c)  // its own
            if (c < (own & 3)) wait((own & ~3) + c, sub[c]);
        {
            const double r = r_own - sum_groups(acc), q0 = r * y;
            double v = tri16_solve<kUpper>(kUpper ? __builtin_fma(__builtin_fma(-u, q0, r), y, q0) : r, nt);
            if (__builtin_expect(!__all(fabs(v) < __builtin_inf()), 0))
                v = tri16_select<kUpper>(r, i16, sh.t16[wave][i16], u);
            if (g == 0) sh.xd[row] = v;
            lds_sync();
            __builtin_amdgcn_s_setprio(0);
            if (g == 0 && row < dim) {
                uint64_t w = __builtin_bit_cast(uint64_t, v);
                if (w == kUnset) w |= 1ull << 51;  // (quiet)
                __hip_atomic_store(xs + d0 + row, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                x[d0 + row] = v;
            }
        }
        for (int p = own + 1; p < 16; ++p) lds_sync();
    }
}

int grid_for(int64_t n, int threads) {
    int64_t g = omx_cdiv(n, threads);
    if (g > 65536) g = 65536;
    if (g < 1) g = 1;
    return (int)g;
}

// bytes of nseg column segments' partial sums
size_t segment_bytes(int64_t n, int nseg) {
    return nseg > 1 ? (size_t)nseg * (size_t)n * sizeof(double) : 0;
}

// The residual GEMV's launches; work holds segment_bytes(n, nseg).
int otf_gemv_launch(int64_t n, int nseg, uint64_t seed, const double *diag, double alpha, const double *x, double *y,
                    void *work, hipStream_t st) {
    const int64_t seglen = omx_cdiv(n, nseg);
    const int64_t nrb = omx_cdiv(n, kGemvRows);
    double *part = nseg > 1 ? static_cast<double *>(work) : nullptr;
    hipLaunchKernelGGL(k_otf_gemv, dim3((unsigned)nrb, (unsigned)nseg), dim3(kGemvRows), 0, st, n,
                       omx_lcg_init(seed), omx_jump((uint64_t)n), diag, x, seglen, part, y, alpha);
    OMX_LAUNCH_CHECK();
    if (nseg > 1) {
        hipLaunchKernelGGL(k_gemv_reduce, dim3((unsigned)omx_cdiv(n, 256)), dim3(256), 0, st, n,
                           nseg, part, y, alpha);
        OMX_LAUNCH_CHECK();
    }
    return OMX_OK;
}

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double *g_scratch_dev[kMaxDevices] = {};

// Device address of `scratch` on the current device, looked up once per
// device (hipGetSymbolAddress with that device current) and kept.
int noalloc_scratch(double **out) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return OMX_ERR_HIP;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_dev[dev]) {
        void *p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return OMX_ERR_HIP;
        g_scratch_dev[dev] = static_cast<double *>(p);
    }
    *out = g_scratch_dev[dev];
    return OMX_OK;
}

}  // namespace

extern "C" {

size_t omx_otf_gemv_workspace_bytes(int64_t n) {
    return n > 0 ? segment_bytes(n, gemv_segments(n)) : 0;
}

int omx_otf_gemv_f64(int64_t n, uint64_t seed, const double *diag, double alpha,
                     const double *x, double *y, void *work, size_t work_bytes,
                     void *stream) {
    if (n <= 0 || !diag || !x || !y) return OMX_ERR_ARG;
    const size_t have = work ? work_bytes : 0;
    int nseg = gemv_segments(n);
    if (have < segment_bytes(n, nseg)) nseg = gemv_segments(n, 256);
    if (have < segment_bytes(n, nseg)) return OMX_ERR_WORKSPACE;
    return otf_gemv_launch(n, nseg, seed, diag, alpha, x, y, work, omx_stream(stream));
}

int omx_otf_gemv_f64_noalloc(int64_t n, uint64_t seed, const double *diag, double alpha, const double *x,
                             double *y, void *stream) {
    if (n <= 0 || !diag || !x || !y) return OMX_ERR_ARG;
    if (omx_otf_gemv_workspace_bytes(n) > kNoAllocScratchBytes) return OMX_ERR_WORKSPACE;
    double *part = nullptr;
    const int rc = noalloc_scratch(&part);
    if (rc) return rc;
    return otf_gemv_launch(n, gemv_segments(n), seed, diag, alpha, x, y, part, omx_stream(stream));
}

int omx_norm_inf_f64(int64_t n, const double *x, double *result, void *stream) {
    if (n <= 0 || !x || !result) return OMX_ERR_ARG;
    hipLaunchKernelGGL(k_norm_inf, dim3(1), dim3(1024), 0, omx_stream(stream), n, x, result);
    OMX_LAUNCH_CHECK();
    return OMX_OK;
}

int omx_copy_f64(int64_t n, const double *x, double *y, void *stream) {
    if (n <= 0 || !x || !y) return OMX_ERR_ARG;
    hipLaunchKernelGGL(k_copy, dim3(grid_for(n, 256)), dim3(256), 0, omx_stream(stream), n, x, y);
    OMX_LAUNCH_CHECK();
    return OMX_OK;
}

int omx_div_f64(int64_t n, const double *b, const double *d, double *x, void *stream) {
    if (n <= 0 || !b || !d || !x) return OMX_ERR_ARG;
    hipLaunchKernelGGL(k_div, dim3(grid_for(n, 256)), dim3(256), 0, omx_stream(stream), n, b, d, x);
    OMX_LAUNCH_CHECK();
    return OMX_OK;
}

int omx_axpy_f64(int64_t n, double alpha, const double *x, double *y, void *stream) {
    if (n <= 0 || !x || !y) return OMX_ERR_ARG;
    hipLaunchKernelGGL(k_axpy, dim3(grid_for(n, 256)), dim3(256), 0, omx_stream(stream), n, alpha,
                       x, y);
    OMX_LAUNCH_CHECK();
    return OMX_OK;
}

size_t omx_trsv_workspace_bytes(int64_t n) {
    if (n <= 0) return 0;
    return ((size_t)omx_cdiv(n, kTB) * kTB + 32) * sizeof(double);
}

static int trsv_args(int64_t n, int64_t b, const float *A, int64_t lda, double *x) {
    if (n <= 0 || b <= 0 || n % b || lda < n || !A || !x) return OMX_ERR_ARG;
    return OMX_OK;
}

static bool trsv_vec(const float *A, int64_t lda) {
    return (reinterpret_cast<uintptr_t>(A) & 15) == 0 && (lda & 3) == 0;
}

// The solve in one launch when the caller gives the workspace; OMX_OK and
// *done = true if it was queued.  From three blocks on: with two the launch
// and the diagonal block's staging cost what they save.  us, a launch per block
// -> one launch, lower | upper:
//   n =   768    30 ->   29 |   43 ->   29    n =  61440   3674 ->  1908 |  4807 ->  1940
//   n =  1024    40 ->   35 |   59 ->   36    n = 122880   8501 ->  5661 | 10737 ->  5697
//   n = 10240   461 ->  282 |  652 ->  295    n = 204800  18568 -> 14521 | 21010 -> 14584
// (5.8 TB/s of factor entries at n = 204800: the tiles' traffic).
static int trsv_launch(bool upper, int64_t n, const float *A, int64_t lda, double *x, void *work, size_t work_bytes,
                       hipStream_t st, bool *done) {
    *done = false;
    const int64_t nb = omx_cdiv(n, kTB);
    if (nb < 3 || !trsv_vec(A, lda) || !work || work_bytes < omx_trsv_workspace_bytes(n) ||
        (reinterpret_cast<uintptr_t>(work) & 7))
        return OMX_OK;
    uint64_t *xs = static_cast<uint64_t *>(work);
    int *ticket = reinterpret_cast<int *>(xs + nb * kTB);
    hipLaunchKernelGGL(k_trsv_reset, dim3(grid_for(nb * kTB, 256)), dim3(256), 0, st, nb * kTB, xs, ticket);
    OMX_LAUNCH_CHECK();
    const dim3 grid((unsigned)(nb < 256 ? nb : 256));  // one workgroup per CU
    if (upper)
        hipLaunchKernelGGL(k_trsv_fused<true>, grid, dim3(kTT), 0, st, n, A, lda, x, xs, ticket);
    else
        hipLaunchKernelGGL(k_trsv_fused<false>, grid, dim3(kTT), 0, st, n, A, lda, x, xs, ticket);
    OMX_LAUNCH_CHECK();
    *done = true;
    return OMX_OK;
}

int omx_trsv_lower_unit_f32f64(int64_t n, int64_t b, const float *A, int64_t lda, double *x,
                               void *work, size_t work_bytes, void *stream) {
    int rc = trsv_args(n, b, A, lda, x);
    if (rc) return rc;
    hipStream_t st = omx_stream(stream);
    bool done;
    rc = trsv_launch(false, n, A, lda, x, work, work_bytes, st, &done);
    if (rc || done) return rc;
    const bool vec = trsv_vec(A, lda);
    for (int64_t j0 = -kTB; j0 + kTB < n; j0 += kTB) {
        const int64_t d0 = j0 + kTB;
        const int64_t beyond = n - d0 - kTB;
        const unsigned grid = 1u + (unsigned)(beyond > 0 && j0 >= 0 ? omx_cdiv(beyond, kTB) : 0);
        if (vec)
            hipLaunchKernelGGL(k_trsv_lower_step<true>, dim3(grid), dim3(kTT), 0, st, n, j0, A, lda, x);
        else
            hipLaunchKernelGGL(k_trsv_lower_step<false>, dim3(grid), dim3(kTT), 0, st, n, j0, A, lda, x);
        OMX_LAUNCH_CHECK();
    }
    return OMX_OK;
}

int omx_trsv_upper_f32f64(int64_t n, int64_t b, const float *A, int64_t lda, double *x,
                          void *work, size_t work_bytes, void *stream) {
    int rc = trsv_args(n, b, A, lda, x);
    if (rc) return rc;
    hipStream_t st = omx_stream(stream);
    bool done;
    rc = trsv_launch(true, n, A, lda, x, work, work_bytes, st, &done);
    if (rc || done) return rc;
    const bool vec = trsv_vec(A, lda);
    const int64_t last0 = ((n - 1) / kTB) * kTB;
    // j0 = n: the last block alone; then J = each block from the last down
    for (int64_t j0 = n; j0 > 0; j0 = (j0 == n) ? last0 : j0 - kTB) {
        const int64_t d0 = (j0 == n) ? last0 : j0 - kTB;
        if (d0 < 0) break;
        const unsigned grid = 1u + (unsigned)(j0 < n ? omx_cdiv(d0, kTB) : 0);
        if (vec)
            hipLaunchKernelGGL(k_trsv_upper_step<true>, dim3(grid), dim3(kTT), 0, st, n, j0, A, lda, x);
        else
            hipLaunchKernelGGL(k_trsv_upper_step<false>, dim3(grid), dim3(kTT), 0, st, n, j0, A, lda, x);
        OMX_LAUNCH_CHECK();
    }
    return OMX_OK;
}

double omx_harness(double normr, double norma, double normx, double normb, int64_t n) {
    return normr / (norma * normx + normb) * 1.0 / ((double)n * DBL_EPSILON / 2);
}

}  // extern "C"
