// omx_dense.hip -- FP32 dense kernels on the LU critical path: the no-pivot
// LU of the b x b diagonal block (panel_trf), the triangular solves with its
// factors (panel_trsm and the -alt inverses), and the FP32 GEMM that updates
// inside them.
//
// All are blocked by 64: a 64-wide diagonal piece is handled by one small
// kernel (rows or columns in parallel, the 64 x 64 triangle staged in LDS),
// the rest of the update is an FP32 GEMM.  Pivots are applied as
// multiplication by the reciprocal, as sgetrf_nopiv_naive does
// (sgetrf_nopiv.cpp:27-61) and as reference BLAS strsm does for a non-unit
// diagonal.
#include <algorithm>
#include <utility>
#include <vector>

#include "omx_common.hpp"

namespace {

constexpr int kNB = 64;
#define RC(x)                  \
    do {                       \
        const int rc_ = (x);   \
        if (rc_) return rc_;   \
    } while (0)

// The triangular solves (omx_trsm_f32) go in blocks of kOB: a block is solved
// in one launch (RLNU: 64 columns at a time) and updates everything beyond it
// in one product of depth kOB, so the large products read and write their C a
// quarter as often as with 64.
constexpr int64_t kOB = 256;

// ---------------------------------------------------------------------------
// FP32 GEMM, C = beta*C + alpha * A * B (all column-major, no transposes).
// 64 x 64 tile per workgroup of 256 threads, 4 x 4 results per thread,
// k advanced 16 at a time through LDS.  k must be a multiple of 16.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
k_sgemm_nn(int64_t M, int64_t N, int64_t K, float alpha, const float *__restrict__ A, int64_t lda,
           const float *__restrict__ B, int64_t ldb, float beta, float *__restrict__ C, int64_t ldc,
           int64_t sA, int64_t sB, int64_t sC) {
    __shared__ float As[16][64 + 4];
    __shared__ float Bs[16][64 + 4];
    // batch blockIdx.z: operands sA / sB / sC floats further on
    A += (int64_t)blockIdx.z * sA;
    B += (int64_t)blockIdx.z * sB;
    C += (int64_t)blockIdx.z * sC;
    const int tid = threadIdx.x;
    const int tx = tid & 15, ty = tid >> 4;
    const int64_t i0 = (int64_t)blockIdx.x * 64, j0 = (int64_t)blockIdx.y * 64;
    float acc[4][4] = {};
    for (int64_t k0 = 0; k0 < K; k0 += 16) {
        // A tile: 64 rows x 16 columns; thread -> (row = tid % 64, 4 columns)
        {
            const int r = tid & 63, c4 = (tid >> 6) * 4;
            const int64_t gi = i0 + r;
#pragma unroll
            for (int c = 0; c < 4; ++c) As[c4 + c][r] = (gi < M) ? A[gi + (k0 + c4 + c) * lda] : 0.0f;
        }
        // B tile: 16 rows x 64 columns; thread -> (column = tid / 4, 4 rows)
        {
            const int cc = tid >> 2, r4 = (tid & 3) * 4;
            const int64_t gj = j0 + cc;
#pragma unroll
            for (int r = 0; r < 4; ++r) Bs[r4 + r][cc] = (gj < N) ? B[(k0 + r4 + r) + gj * ldb] : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < 16; ++kk) {
            float a[4], b[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                a[q] = As[kk][tx + 16 * q];
                b[q] = Bs[kk][ty + 16 * q];
            }
#pragma unroll
            for (int p = 0; p < 4; ++p)
#pragma unroll
                for (int q = 0; q < 4; ++q) acc[p][q] = __builtin_fmaf(a[p], b[q], acc[p][q]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const int64_t gi = i0 + tx + 16 * p;
        if (gi >= M) continue;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int64_t gj = j0 + ty + 16 * q;
            if (gj >= N) continue;
            float *c = C + gi + gj * ldc;
            *c = (beta == 0.0f) ? alpha * acc[p][q] : beta * *c + alpha * acc[p][q];
        }
    }
}

// ---------------------------------------------------------------------------
// The same product on the matrix cores (v_mfma_f32_32x32x2_f32), for the
// large updates: a kT x kT tile (64, or 128: sgemm_mfma) per workgroup of four
// waves (a kT/2 square quadrant each, made of 32 x 32 MFMA blocks), k in groups
// of up to 64, staged through LDS kQ of each half at a time, the next stage's
// global loads in flight during the current stage's MFMAs.  The MFMA's first
// operand takes B (lane l: column l % 32), the second A (lane l: row l % 32),
// so every accumulator register of lane l belongs to row l % 32 of its block
// and a half-wave's C access is 32 consecutive rows of one column (one
// 128-byte line).  In a group of kc columns, lanes 0-31 carry k in [0, kc/2)
// and lanes 32-63 k in [kc/2, kc); the MFMA adds the two halves.  Needs A and
// B 16-byte aligned with lda and ldb multiples of 4, and k % 16 == 0 (so kc
// is a multiple of 16).
//
// Bound by the MFMAs where k is deep and by C's traffic where it is not; what
// stood between was the time from a stage's loads to the next's.  A product
// of whole groups of 64 and whole float4s of rows therefore steps pointers
// and has no bounds in its loop: with the clamps the compiler put waits
// between a stage's own loads, and four waves alone on their CU paid for
// every address instruction.  Its last stage stands outside the loop, so that
// C's old values (kT = 128: those of half its blocks, all spill)
// are on their way during that stage's MFMAs.  A 128-tile's stages hold half a
// group, so that three workgroups fit a CU instead of two.  Measured (bounds
// in the loop, no XCD order -> now), C -= A B: 30000 x 2304 x 256 456 -> 379 us,
// 2048 x 2048 x 512 47.5 -> 41.7, 30000 x 256 x 256 54.4 -> 46, 512 x 512 x 512
// 17.6 -> 13.5, 60000 x 2304 x 64 289 -> 270, 4096 x 4096 x 8192 2200 -> 2060,
// 61440 x 61440 x 2560 161 -> 141 ms (137 TFLOP/s), 20480 x 20480 x 10240 68.8 ->
// 61.7.
// ---------------------------------------------------------------------------
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// The MFMA kernel takes products with at least this many C entries per
// launch (2^18 = 512 x 512; smaller ones are latency-bound and the 64 x 64
// VALU tiles spread them over more CUs) when its alignment conditions hold.
#ifndef OMX_SGEMM_MFMA_MIN
#define OMX_SGEMM_MFMA_MIN (int64_t{1} << 18)
#endif

__host__ __device__ __forceinline__ bool mfma_size(int64_t m, int64_t n, int64_t batch) {
    return m * n * batch >= OMX_SGEMM_MFMA_MIN;
}

constexpr int kMG = 64;         // k per group

template <int kT>
__device__ __forceinline__ void sgemm_tile(int64_t M, int64_t N, int64_t K, float alpha,
                                           const float *__restrict__ A, int64_t lda, const float *__restrict__ B,
                                           int64_t ldb, float beta, float *__restrict__ C, int64_t ldc,
                                           int64_t ti, int64_t tj, int64_t k0 = 0) {
    constexpr int kB = kT / 64;              // MFMA blocks per quadrant side
    constexpr int kQ = kT == 64 ? 32 : 16;   // a stage's k in each half of a group
    constexpr int kS = kT * kQ / 512;        // float4 loads per thread per operand and stage
    constexpr int kAK = 1024 / kT;           // stage columns between a thread's A loads
    constexpr int kBJ = 512 / kQ;            // columns between a thread's B loads
    constexpr int kBLd = 2 * kQ + 4;         // row stride of Bs: conflict-free 16-byte reads
    __shared__ float As[2 * kQ][kT];         // As[q][i], As[kQ + q][i] = A(i0 + i, p0 + q), A(i0 + i, p1 + q)
    __shared__ float Bs[kT][kBLd];           // Bs[j][q], Bs[j][kQ + q] = B(p0 + q, j0 + j), B(p1 + q, j0 + j)
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l32 = lane & 31, h = lane >> 5;
    const int64_t i0 = ti * kT, j0 = tj * kT;
    const int wi = (wave & 1) * (kT / 2), wj = (wave >> 1) * (kT / 2);
    // global -> LDS: A rows ar .. ar+3 at stage columns ak + kAK s; B column
    // bj + kBJ s, stage rows bk .. bk+3 of half bh.  Rows (columns) past M
    // (N) are clamped: their products land only in results that are not
    // stored.
    const int ar = 4 * (tid % (kT / 4)), ak = tid / (kT / 4);
    const int bk = 4 * (tid % (kQ / 4)), bh = tid / (kQ / 4) & 1, bj = tid / (kQ / 2);
    const int64_t arow = i0 + ar;
    const float *Bcol[kS];
#pragma unroll
    for (int s = 0; s < kS; ++s) Bcol[s] = B + min(j0 + bj + kBJ * s, N - 1) * ldb;
    f32x4 ra[kS], rb[kS];
    f32x16 acc[kB][kB];
#pragma unroll
    for (int a = 0; a < kB; ++a)
#pragma unroll
        for (int b = 0; b < kB; ++b)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[a][b][v] = 0.0f;
    // the products of a stage's first hc columns of each half
    auto products = [&](int hc) {
        for (int s = 0; s < hc; s += 4) {
            f32x4 y[kB];
#pragma unroll
            for (int b = 0; b < kB; ++b) y[b] = *reinterpret_cast<const f32x4 *>(&Bs[wj + 32 * b + l32][kQ * h + s]);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                float x[kB];
#pragma unroll
                for (int a = 0; a < kB; ++a) x[a] = As[kQ * h + s + u][wi + 32 * a + l32];
#pragma unroll
                for (int a = 0; a < kB; ++a)
#pragma unroll
                    for (int b = 0; b < kB; ++b)
                        acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(y[b][u], x[a], acc[a][b], 0, 0, 0);
            }
        }
    };
    // acc[a][b][v] and cv[a][b][v]: row i0 + wi + 32 a + l32, column
    // jb + 32 b + 8 (v / 4) + v % 4.  C's columns are walked by one pointer,
    // opaque to the compiler (which otherwise forms all 64 addresses first
    // and spills), and a column past N repeats the one before it.
    float cv[kB][kB][16];
    const int64_t jb = j0 + wj + 4 * h;
    const int ncols = (int)max(min(N - jb, (int64_t)kT), (int64_t)0);
    auto load_c = [&](int a0, int a1) {
        if (beta == 0.0f) return;
#pragma unroll
        for (int a = a0; a < a1; ++a) {
            const float *c = C + min(i0 + wi + 32 * a + l32, M - 1) + min(jb, N - 1) * ldc;
#pragma unroll
            for (int b = 0; b < kB; ++b)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    cv[a][b][v] = *c;
                    const int step = v % 4 < 3 ? 1 : 5;
                    c += 32 * b + 8 * (v >> 2) + (v & 3) + step < ncols ? step * ldc : 0;
                    asm volatile("" : "+v"(c));
                }
        }
    };
    if (K - k0 >= kMG && (K - k0) % kMG == 0 && (M % 4 == 0 || i0 + kT <= M)) {
        // whole groups and whole float4s: pointers that step, no bounds
        const float *Ap = A + min(arow, M - 4) + (k0 + ak) * lda;
#pragma unroll
        for (int s = 0; s < kS; ++s) Bcol[s] += k0 + bk + kMG / 2 * bh;
        int64_t left = (K - k0) / (2 * kQ);
        int t = 0;
        auto load = [&] {
#pragma unroll
            for (int s = 0; s < kS; ++s)
                ra[s] = *reinterpret_cast<const f32x4 *>(
                    Ap + (kAK * s < kQ ? kAK * s : kMG / 2 + kAK * s - kQ) * lda);
#pragma unroll
            for (int s = 0; s < kS; ++s) rb[s] = *reinterpret_cast<const f32x4 *>(Bcol[s]);
            t += kQ;
            const int step = t < kMG / 2 ? kQ : kMG / 2 + kQ;
            if (t == kMG / 2) t = 0;
            Ap += step * lda;
#pragma unroll
            for (int s = 0; s < kS; ++s) Bcol[s] += step;
        };
        auto put = [&] {
#pragma unroll
            for (int s = 0; s < kS; ++s) *reinterpret_cast<f32x4 *>(&As[ak + kAK * s][ar]) = ra[s];
#pragma unroll
            for (int s = 0; s < kS; ++s) *reinterpret_cast<f32x4 *>(&Bs[bj + kBJ * s][kQ * bh + bk]) = rb[s];
        };
        load();
        for (; left > 1; --left) {
            put();
            __syncthreads();
            load();
            products(kQ);
            __syncthreads();
        }
        put();
        __syncthreads();
        load_c(0, 1);   // its latency passes behind the last stage's products
        products(kQ);
    } else {
        int half = (int)min(K - k0, (int64_t)kMG) >> 1, t = 0;
        int hh = min(half, kQ);
        // columns p0 .. p0 + hh and p1 .. p1 + hh into ra / rb.  Every load
        // is unconditional: what lies past hh reads the last column (rows)
        // before it instead and is not stored to LDS.
        auto load = [&](int64_t p0, int64_t p1) {
#pragma unroll
            for (int s = 0; s < kS; ++s) {
                const int q = min((ak + kAK * s) % kQ, hh - 1);
                const float *p = A + ((kAK * s < kQ ? p0 : p1) + q) * lda;
                ra[s] = arow + 3 < M ? *reinterpret_cast<const f32x4 *>(p + arow)
                                     : f32x4{p[min(arow, M - 1)], p[min(arow + 1, M - 1)], p[min(arow + 2, M - 1)],
                                             p[min(arow + 3, M - 1)]};
            }
            const int64_t kb4 = (bh ? p1 : p0) + min(bk, hh - 4);
#pragma unroll
            for (int s = 0; s < kS; ++s) rb[s] = *reinterpret_cast<const f32x4 *>(Bcol[s] + kb4);
        };
        load(k0, k0 + half);
        for (;;) {
#pragma unroll
            for (int s = 0; s < kS; ++s)
                if ((ak + kAK * s) % kQ < hh) *reinterpret_cast<f32x4 *>(&As[ak + kAK * s][ar]) = ra[s];
            if (bk < hh) {
#pragma unroll
                for (int s = 0; s < kS; ++s) *reinterpret_cast<f32x4 *>(&Bs[bj + kBJ * s][kQ * bh + bk]) = rb[s];
            }
            __syncthreads();
            const int hc = hh;
            t += kQ;
            if (t >= half) {
                k0 += 2 * half;
                half = (int)min(K - k0, (int64_t)kMG) >> 1;
                t = 0;
            }
            hh = min(half - t, kQ);
            if (hh > 0) load(k0 + t, k0 + half + t);
            products(hc);
            if (hh <= 0) break;
            __syncthreads();
        }
        load_c(0, 1);
    }
#pragma unroll
    for (int a = 0; a < kB; ++a) {
        if (a > 0) load_c(a, a + 1);
        const int64_t i = i0 + wi + 32 * a + l32;
        if (i >= M) continue;
        float *c = C + i + jb * ldc;
#pragma unroll
        for (int b = 0; b < kB; ++b)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const float r = beta == 0.0f ? alpha * acc[a][b][v] : beta * cv[a][b][v] + alpha * acc[a][b][v];
                if (32 * b + 8 * (v >> 2) + (v & 3) < ncols) *c = r;
                c += (v % 4 < 3 ? 1 : 5) * ldc;
                asm volatile("" : "+v"(c));
            }
    }
}

template <int kT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kT == 64 ? 4 : 3)))
k_sgemm_mfma(int64_t M, int64_t N, int64_t K, float alpha, const float *__restrict__ A, int64_t lda,
             const float *__restrict__ B, int64_t ldb, float beta, float *__restrict__ C, int64_t ldc,
             int64_t sA, int64_t sB, int64_t sC) {
    const int64_t z = blockIdx.z;
    // Workgroup l runs on XCD l % 8: each XCD takes a contiguous eighth of the
    // tiles, and these in strips of eight rows of tiles, so that the tiles an
    // XCD has at a time share their operands in its L2
    const unsigned gx = gridDim.x, gy = gridDim.y, l = blockIdx.x + gx * blockIdx.y;
    const unsigned xcd = l & 7, t = xcd * (gx * gy >> 3) + min(xcd, gx * gy & 7) + (l >> 3);
    const unsigned strip = t / (8 * gy), r = t - strip * 8 * gy, rows = min(8u, gx - 8 * strip);
    sgemm_tile<kT>(M, N, K, alpha, A + z * sA, lda, B + z * sB, ldb, beta, C + z * sC, ldc,
                   8 * strip + r % rows, r / rows);
}

// Two independent batches of products C_p = alpha A_p B_p in one launch
// (blockIdx.z below batch: the first): the merges of the two triangular
// inverses, which would otherwise wait for each other's launches.  tri: one
// factor is triangular and the tile's k range ends or begins with it (the
// products left out are exact zeros): 1 B upper (k below the tile's last
// column), 2 B lower (from its first column), 3 A upper (from its first row),
// 4 A lower (below its last row).
struct SgemmTwin {
    int64_t M, N, K, lda, ldb, ldc, sA, sB, sC;
    int tri;
    const float *A, *B;
    float *C;
};

__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4)))
k_sgemm_twin(SgemmTwin g0, SgemmTwin g1, float alpha, int batch) {
    const bool second = (int)blockIdx.z >= batch;
    const SgemmTwin g = second ? g1 : g0;
    const int64_t z = second ? blockIdx.z - batch : blockIdx.z;
    constexpr int kT = 64;
    const int64_t i0 = (int64_t)blockIdx.x * kT, j0 = (int64_t)blockIdx.y * kT;
    if (i0 >= g.M || j0 >= g.N) return;
    const int64_t k0 = g.tri == 2 ? j0 : (g.tri == 3 ? i0 : 0);
    const int64_t k1 = g.tri == 1 ? j0 + kT : (g.tri == 4 ? i0 + kT : g.K);
    sgemm_tile<kT>(g.M, g.N, k1 < g.K ? k1 : g.K, alpha, g.A + z * g.sA, g.lda, g.B + z * g.sB, g.ldb, 0.0f,
                          g.C + z * g.sC, g.ldc, blockIdx.x, blockIdx.y, k0);
}

__device__ __forceinline__ float lane_bcast(float v, int l) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}

// The 64 x 64 triangle T (column-major, leading dimension ldt) into LDS:
// t[r][c] = T(r, c).
__device__ __forceinline__ void load_tri64(const float *__restrict__ T, int64_t ldt, float (*t)[kNB + 1]) {
    for (int e = threadIdx.x; e < kNB * kNB; e += blockDim.x) t[e & 63][e >> 6] = T[(e & 63) + (int64_t)(e >> 6) * ldt];
    __syncthreads();
}

// value of v in quad lane o (o compile-time) for every lane of the quad
template <int o>
__device__ __forceinline__ float quad_bcast(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), o | (o << 2) | (o << 4) | (o << 6),
                                                              0xF, 0xF, false));
}

// rd[j] = 1 / t[j][j] (the diagonal's reciprocals, shared by the workgroup)
__device__ __forceinline__ void diag_recip64(const float (*t)[kNB + 1], float *rd) {
    if (threadIdx.x < kNB) rd[threadIdx.x] = 1.0f / t[threadIdx.x][threadIdx.x];
    __syncthreads();
}

// Solves of 64 entries a line with a 64 x 64 triangle t in LDS: rows
// x <- x U^-1 (kUp; RUNN, x_j = (b_j - sum_{l<j} x_l u_lj) rd_j) or columns
// y <- L^-1 y (LLNU, unit L).  The calling wave owns 16 lines of xs (its
// rows; nothing else reads or writes them), xs[line][entry].  Entries go in
// four blocks of 16: inside a block a quad of lanes has a line, lane q the
// entries q, q + 4, q + 8, q + 12 (step j: the owner, lane j % 4, finalises
// entry j, the quad reads it with a DPP broadcast, later entries take one
// fused multiply-add each); then the block's product with the triangle is
// taken off the later blocks on the matrix cores (v_mfma_f32_16x16x4_f32:
// lane = line, registers = entries).  The FP32 MFMAs add their products one
// by one, each rounded as a fused multiply-add, so every entry still gets its
// terms in the order l = 0, 1, ... with one rounding each, as in
// column-by-column substitution.  The code is a loop over the blocks on
// purpose: 64 unrolled steps are 16 KB of instructions that every launch
// fetches anew, which took longer than the steps.
constexpr int kXS = kNB + 4;  // row stride of xs: conflict-free operand reads, 16-byte aligned rows
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Step j of a block.  kUp: x holds b_j - sum until the end, where its owner
// scales it as every lane does here.
template <int j, bool kUp>
__device__ __forceinline__ void tri16_step(float (&x)[4], int q, const float (&e)[16][4], const float (&r)[16]) {
    constexpr int o = j & 3, s = j >> 2;
    const float xj = quad_bcast<o>(kUp ? x[s] * r[j] : x[s]);
    if (o < 3) {
        const float later = __builtin_fmaf(-xj, e[j][s], x[s]);
        x[s] = q > o ? later : x[s];
    }
#pragma unroll
    for (int t = s + 1; t < 4; ++t) x[t] = __builtin_fmaf(-xj, e[j][t], x[t]);
}

template <bool kUp, int... J>
__device__ __forceinline__ void tri16_steps(float (&x)[4], int q, const float (&e)[16][4], const float (&r)[16],
                                            std::integer_sequence<int, J...>) {
    (tri16_step<J, kUp>(x, q, e, r), ...);
}

template <bool kUp, int kLd>
__device__ __forceinline__ void tri_solve64(float (*xs)[kLd], const float (*t)[kNB + 1], const float *rd) {
    const int lane = threadIdx.x & 63, q = lane & 3;
    const int i16 = lane & 15, g = lane >> 4;
#pragma unroll 1
    for (int c0 = 0; c0 < kNB; c0 += 16) {
        float x[4], e[16][4], r[16], a[3][4];
        float *line = xs[lane >> 2] + c0 + q;
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = line[4 * u];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            if (kUp) r[j] = rd[c0 + j];
#pragma unroll
            for (int u = j >> 2; u < 4; ++u)
                e[j][u] = kUp ? t[c0 + j][c0 + q + 4 * u] : t[c0 + q + 4 * u][c0 + j];
        }
        // the triangle's operands of the later blocks' products (past the
        // last block: read from within the triangle, not used)
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            const int cb = (c0 + 16 * (b + 1)) & (kNB - 1);
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                const int k = c0 + 4 * kk + g;
                a[b][kk] = kUp ? t[k][cb + i16] : t[cb + i16][k];
            }
        }
        tri16_steps<kUp>(x, q, e, r, std::make_integer_sequence<int, 16>{});
        if (kUp) {
#pragma unroll
            for (int u = 0; u < 4; ++u) x[u] *= rd[c0 + q + 4 * u];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) line[4 * u] = x[u];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        // the solved block's operand: line i16, entry c0 + 4 kk + g
        float xk[4];
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) xk[kk] = -xs[i16][c0 + 4 * kk + g];
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            const int cb = c0 + 16 * (b + 1);
            if (cb < kNB) {
                f32x4 *dst = reinterpret_cast<f32x4 *>(&xs[i16][cb + 4 * g]);
                f32x4 acc = *dst;
#pragma unroll
                for (int kk = 0; kk < 4; ++kk)
                    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[b][kk], xk[kk], acc, 0, 0, 0);
                *dst = acc;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
}

// 64 rows per workgroup of 256 threads, 16 per wave: X(i, :) <- X(i, :) U^-1.
// Rows past m are read as row m - 1 and not stored.
__global__ void __launch_bounds__(256)
k_trsm_rows_runn64(int64_t m, const float *__restrict__ U, int64_t ldu, float *__restrict__ X,
                   int64_t ldx) {
    __shared__ float u[kNB][kNB + 1];
    __shared__ __align__(16) float xs[kNB][kXS];
    __shared__ float rd[kNB];
    // element (row, column): lanes along the rows, 16 columns a wave
    const int r = threadIdx.x & 63, c0 = 16 * (threadIdx.x >> 6);
    const int64_t i = (int64_t)blockIdx.x * 64 + r;
    float *row = X + (i < m ? i : m - 1) + (int64_t)c0 * ldx;
    float v[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) v[c] = row[c * ldx];
    load_tri64(U, ldu, u);
#pragma unroll
    for (int c = 0; c < 16; ++c) xs[r][c0 + c] = v[c];
    diag_recip64(u, rd);
    tri_solve64<true, kXS>(xs + c0, u, rd);
    __syncthreads();
    if (i < m) {
#pragma unroll
        for (int c = 0; c < 16; ++c) row[c * ldx] = xs[r][c0 + c];
    }
}

// ---------------------------------------------------------------------------
// One 64-column step j of the blocked LU in one launch, the rank-64 update
// of the step before (p = j - 64) included.  At its start the column block
// L_p = A(j.., p) and the row block U_p = A(p, j..) are final and everything
// at and beyond (j, j) still lacks their product.  Workgroups of 512 threads:
//   [0, np)        128 rows of the column block j each: the 64 x 64 diagonal
//                  block D = A_jj - L_p U_p is formed and factored by every
//                  one of them for itself (into LDS; all get the same
//                  factors), the rows receive their update and are solved
//                  with D's U;
//   [np, 2 np)     128 columns of the row block j likewise, with D's unit L;
//   1 more (j > 0) D_p, factored once more as in the step before, is written
//                  (in its own step other workgroups, which need not all run
//                  at the same time, still read the original);
//   the rest       the 128 x 64 tiles beyond row and column block j: the
//                  update alone.
// The last step's workgroup 0, with nothing below or right of D, writes its
// own D.  What bounds a step is the chain of one such workgroup (launch,
// loads, 64 pivots, 64 solve steps), not its operations: with the update in a
// launch of its own and D factored by one wave a step took 34 us at n = 2560
// and 36 us at n = 256 (idle GPU), now 20.5 and 15.5 us, with the same
// factors bit for bit; beside the LU's trailing product, where every
// launch waits for CUs, half the launches wait.
//
// D is factored by eight waves, wave w holding columns 8 w .. 8 w + 7 with
// lane i = row i: wave s factors its 8 columns (row k read from lane k with
// v_readlane; multipliers x reciprocal pivot, as sgetrf_nopiv_naive) and
// hands each over through LDS; the waves beyond apply it meanwhile.  A wave's
// part of the tile's update (32 x 32, 32 MFMAs) follows its own columns.
//
// Operands: L_p straight from global memory (a lane's row, 32 consecutive
// rows per half-wave: the MFMA's second operand), U_p, contiguous along k,
// through LDS (the first).  n is a multiple of 64; rows and columns past n of
// a last, half-empty 128-tile are clamped and not stored.
// ---------------------------------------------------------------------------
constexpr int kGT = 512;           // threads
constexpr int kUS = kXS;           // row stride of the staged U_p: conflict-free 16-byte reads

struct __align__(16) GetrfShared {
    float su[kNB][kUS];       // U_p, columns of block j (or of the trailing tile): su[c][k]
    float sx[2 * kNB][kUS];   // U_p, the 128 columns of a row-block workgroup; then the tile to solve
    float d[kNB][kNB + 1];    // D
    float rd[kNB];            // reciprocal pivots
    int prog;                 // columns of D factored so far
};

// Columns [0, 32 kN) of U (64 rows, leading dimension ld), 16 bytes per thread
// of 32 columns each, into registers; columns at or past cmax are read as
// column cmax - 1.  put_u: to su[c][k].
template <bool kVec, int kN>
__device__ __forceinline__ void get_u(const float *__restrict__ U, int64_t ld, int64_t cmax, f32x4 (&v)[kN]) {
    const int k = 4 * (threadIdx.x & 15), c = threadIdx.x >> 4;
#pragma unroll
    for (int i = 0; i < kN; ++i) {
        const float *g = U + min((int64_t)(c + 32 * i), cmax - 1) * ld + k;
        v[i] = kVec ? *reinterpret_cast<const f32x4 *>(g) : f32x4{g[0], g[1], g[2], g[3]};
    }
}

// The update's 64 products of an entry are summed in the order of the products
// that the library would launch for it: k_sgemm_mfma (0, 32, 1, 33, ...: a
// lane of half h takes k = 32 h + s in its s-th MFMA) or, for small or
// unaligned blocks, k_sgemm_nn (0, 1, 2, ..: k = 2 s + h; seq).  su holds
// k in that order: lane half h reads positions 32 h .. 32 h + 31.
template <int kN>
__device__ __forceinline__ void put_u(const f32x4 (&v)[kN], float (*su)[kUS], bool seq) {
    const int k = 4 * (threadIdx.x & 15), c = threadIdx.x >> 4;
    typedef float f32x2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int i = 0; i < kN; ++i) {
        float *d = su[c + 32 * i];
        if (seq) {
            *reinterpret_cast<f32x2 *>(d + k / 2) = f32x2{v[i].x, v[i].z};
            *reinterpret_cast<f32x2 *>(d + 32 + k / 2) = f32x2{v[i].y, v[i].w};
        } else {
            *reinterpret_cast<f32x4 *>(d + k) = v[i];
        }
    }
}

typedef float f32x32 __attribute__((ext_vector_type(32)));

// a lane's row of L_p (pointer to it at column 0): 32 of the 64 columns, by
// half-wave and order (put_u)
__device__ __forceinline__ void load_l(const float *__restrict__ row, int64_t ld, int h, bool seq, f32x32 &l) {
    const float *g = row + (seq ? h : 32 * h) * ld;
    const int64_t step = seq ? 2 * ld : ld;
#pragma unroll
    for (int s = 0; s < 32; ++s) l[s] = g[s * step];
}

// four of the 32 products of a wave's 32 x 32 block: acc[v] is row lane % 32,
// column 8 (v / 4) + 4 (lane / 32) + v % 4; su is the lane's column of U_p
// from k = 32 (lane / 32) on
__device__ __forceinline__ void mfma4(const f32x32 &l, const float *su, int g, f32x16 &acc) {
    const f32x4 y = *reinterpret_cast<const f32x4 *>(su + 4 * g);
#pragma unroll
    for (int u = 0; u < 4; ++u) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(y[u], l[4 * g + u], acc, 0, 0, 0);
}

__device__ __forceinline__ void mfma32(const f32x32 &l, const float *su, f32x16 &acc) {
#pragma unroll
    for (int g = 0; g < 8; ++g) mfma4(l, su, g, acc);
}

// LDS hand-over between the waves; outstanding global loads stay in flight
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// LDS accesses that other waves of the workgroup watch: relaxed atomics, which
// stay in program order (volatile ones wait for their completion each time)
template <class T>
__device__ __forceinline__ T lds_get(const T *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
template <class T>
__device__ __forceinline__ void lds_put(T *p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// 1 / u: the hardware reciprocal (1 ulp) and one Newton step, 3 dependent
// instructions in the pivots' chain where the division has 11.  For pivots
// that pivot_ok admits; the others take the division (kDiv).
template <bool kDiv>
__device__ __forceinline__ float pivot_recip(float u) {
    if (kDiv) return 1.0f / u;
    const float y = __builtin_amdgcn_rcpf(u);
    return __builtin_fmaf(__builtin_fmaf(-u, y, 1.0f), y, y);
}

// neither u nor 1 / u subnormal, zero, infinite or NaN
__device__ __forceinline__ bool pivot_ok(float u) {
    const int ex = (__builtin_bit_cast(int, u) >> 23) & 255;
    return ex >= 4 && ex <= 250;
}

// r -= m u in the rows below the pivot.  The others have m = 0 (up to the sign
// of a zero this leaves r as it is), but where a pivot was not pivot_ok (kDiv)
// m can be 0 times an infinite reciprocal and u what an earlier such pivot
// left: finished rows of U are selected there.
template <bool kDiv>
__device__ __forceinline__ void lu_update(float &r, float m, float u, bool below) {
    const float d = __builtin_fmaf(-m, u, r);
    r = kDiv && !below ? r : d;
}

// Factorisation of sh.d (see above) by the calling wave's share.  Columns
// are handed over one by one: the wave that factors writes column g of the
// factors to sh.d, then sh.prog = g + 1 (LDS operations of a wave complete in
// order); a wave that waits for it reads both at once, the next column's while
// it applies the current one.  What it costs is instructions: a wave issues
// one in about six cycles, dependent or not.  A loop over the stages:
// unrolled, they are 30 KB of instructions to fetch in every launch.
template <bool kDiv>
__device__ __forceinline__ void lu_stages(float (&r)[8], int lane, int wave, GetrfShared &sh) {
    float *col = &sh.d[lane][0];
#pragma unroll 1
    for (int s = 0; s < wave; ++s) {
        int f = lds_get(&sh.prog);
        float mg = lds_get(&col[8 * s]);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int g = 8 * s + k;
            while (f <= g) {
                if (s + 1 < wave) __builtin_amdgcn_s_sleep(2);
                f = lds_get(&sh.prog);
                mg = lds_get(&col[g]);
            }
            const float m = lane > g ? mg : 0.0f;
            if (k < 7) {
                f = lds_get(&sh.prog);
                mg = lds_get(&col[g + 1]);
            }
            float u[8];  // the pivot row, read together: a read just before its use waits
#pragma unroll
            for (int c = 0; c < 8; ++c) u[c] = lane_bcast(r[c], g);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int c = 0; c < 8; ++c) lu_update<kDiv>(r[c], m, u[c], lane > g);
        }
    }
    const int g0 = 8 * wave, ln = lane - g0;
    int pv = g0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const float inv = pivot_recip<kDiv>(lane_bcast(r[k], g0 + k));
        // rows at or above the pivot take multiplier 0: fma(-0, u, r) leaves
        // r as it is (up to the sign of a zero)
        const float m = (ln > k ? r[k] : 0.0f) * inv;
        r[k] = ln > k ? m : r[k];
        lds_put(&col[g0 + k], r[k]);
        asm volatile("v_add_u32 %0, 1, %0" : "+v"(pv));
        lds_put(&sh.prog, pv);  // (every lane the same value: no branch)
        float u[8];
#pragma unroll
        for (int c = k + 1; c < 8; ++c) u[c] = lane_bcast(r[c], g0 + k);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int c = k + 1; c < 8; ++c) lu_update<kDiv>(r[c], m, u[c], ln > k);
    }
}

// A: the order-n block; j: first column of the step; np: 128-row workgroups
// of the column block (= those of the row block).  The first step (no update:
// kUpd false) sets info, the later ones lower it.
template <bool kUpd, bool kVec>
__global__ void __launch_bounds__(kGT) __attribute__((amdgpu_waves_per_eu(4)))
k_getrf_step64(int64_t n, int64_t j, int np, float *__restrict__ A, int64_t lda, int *__restrict__ info) {
    __shared__ GetrfShared sh;
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int bid = blockIdx.x;
    const int nch = np > 0 ? 2 * np : 1;  // workgroups that solve (the last step: that factors)
    const bool trail = kUpd && bid > nch;
    const bool writer = kUpd && bid == nch;
    const bool cols = !trail && !writer && bid >= np && np > 0;
    const bool solve = !trail && !writer && np > 0;
    // the step whose D this workgroup factors, and whose update it applies
    const int64_t jj = writer ? j - kNB : j;
    const bool upd = kUpd && jj > 0;
    const bool seq = !kVec || !mfma_size(n - jj, n - jj, 1);
    const float *Lp = A + (jj - kNB) * lda;         // column block p: row i at Lp + i
    const float *Up = A + (jj - kNB);               // row block p: column c at Up + c lda
    // the tile: rows from i0, columns from c0; the wave's 32 x 32 block of it
    int64_t i0 = j + kNB, c0 = j;
    int wr = 32 * (wave & 3), wc = 32 * (wave >> 2);
    if (trail) {
        const int t = bid - nch - 1;
        i0 = j + kNB + (int64_t)(t % np) * 128;
        c0 = j + kNB + (int64_t)(t / np) * kNB;
    } else if (cols) {
        i0 = j;
        c0 = j + kNB + (int64_t)(bid - np) * 128;
        wr = 32 * (wave & 1);
        wc = 32 * (wave >> 1);
    } else if (solve) {
        i0 = j + kNB + (int64_t)bid * 128;
    }
    f32x16 acc;
    f32x32 l;
    float cv[16];
    const int64_t row = min(i0 + wr + l32, n - 1);  // the lane's row of the tile
    if (trail) {
        f32x4 u2[2];
        get_u<kVec>(Up + c0 * lda, lda, kNB, u2);
        load_l(Lp + row, lda, h, seq, l);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            acc[v] = 0.0f;
            cv[v] = A[row + (c0 + wc + 8 * (v >> 2) + 4 * h + (v & 3)) * lda];
        }
        put_u(u2, sh.su, seq);
        lds_barrier();
        mfma32(l, &sh.su[wc + l32][32 * h], acc);
        if (i0 + wr + l32 < n) {
#pragma unroll
            for (int v = 0; v < 16; ++v)
                A[row + (c0 + wc + 8 * (v >> 2) + 4 * h + (v & 3)) * lda] = cv[v] - acc[v];
        }
        return;
    }
    // (a trailing tile may share the CU; the chain goes first)
    __builtin_amdgcn_s_setprio(3);
    // D - L_p U_p into LDS, a 32 x 32 quadrant by each of waves 0-3; all
    // loads first, the products' operands before the rest
    const int dr = 32 * (wave & 1), dc = 32 * ((wave >> 1) & 1);
    f32x4 u2[2], u4[4];
    if (upd) {
        get_u<kVec>(Up + jj * lda, lda, kNB, u2);
        if (wave < 4) load_l(Lp + jj + dr + l32, lda, h, seq, l);
        if (cols) get_u<kVec>(Up + c0 * lda, lda, n - c0, u4);
    }
    if (wave < 4) {
        const float *dp = A + jj + dr + l32;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            acc[v] = 0.0f;
            cv[v] = dp[(jj + dc + 8 * (v >> 2) + 4 * h + (v & 3)) * lda];
        }
    }
    if (tid == 0) sh.prog = 0;
    if (upd) {
        put_u(u2, sh.su, seq);
        if (cols) put_u(u4, sh.sx, seq);
    }
    lds_barrier();
    if (wave < 4) {
        if (upd) mfma32(l, &sh.su[dc + l32][32 * h], acc);
#pragma unroll
        for (int v = 0; v < 16; ++v) sh.d[dr + l32][dc + 8 * (v >> 2) + 4 * h + (v & 3)] = cv[v] - acc[v];
    }
    if (solve) {
        // the tile's operands, in flight during the factorisation
        if (upd) load_l(Lp + row, lda, h, seq, l);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            acc[v] = 0.0f;
            cv[v] = A[row + min(c0 + wc + 8 * (v >> 2) + 4 * h + (v & 3), n - 1) * lda];
        }
    }
    lds_barrier();
    float r[8], r0[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) r[k] = r0[k] = sh.d[lane][8 * wave + k];
    lu_stages<false>(r, lane, wave, sh);
    // the tile's update, after the wave's own stage
    if (kUpd && solve) mfma32(l, cols ? &sh.sx[wc + l32][32 * h] : &sh.su[wc + l32][32 * h], acc);
    lds_barrier();
    float piv = sh.d[lane][lane];
    if (__builtin_expect(!__all(pivot_ok(piv)), 0)) {
        // (every wave sees the same pivots) once more, with divisions
        lds_barrier();
        if (tid == 0) sh.prog = 0;
#pragma unroll
        for (int k = 0; k < 8; ++k) r[k] = r0[k];
        lds_barrier();
        lu_stages<true>(r, lane, wave, sh);
        lds_barrier();
        piv = sh.d[lane][lane];
    }
    if (wave == 0) sh.rd[lane] = 1.0f / piv;
    if (bid == 0 && wave == 0 && info) {
        const uint64_t zero = __ballot(piv == 0.0f);
        const int b = zero ? (int)jj + (int)__builtin_ctzll(zero) + 1 : 0x7fffffff;
        if (lane == 0) {
            if (!kUpd)
                *info = b;  // the first step sets it
            else if (zero)
                atomicMin(info, b);
        }
    }
    if (!solve) {
        // the previous step's D, or the last one's own
#pragma unroll
        for (int k = 0; k < 8; ++k) A[jj + lane + (jj + 8 * wave + k) * lda] = r[k];
        return;
    }
    // the tile into LDS, a line to solve per row of sx; 16 lines a wave
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const int rr = wr + l32, cc = wc + 8 * (v >> 2) + 4 * h + (v & 3);
        sh.sx[cols ? cc : rr][cols ? rr : cc] = cv[v] - acc[v];
    }
    lds_barrier();
    if (cols)
        tri_solve64<false, kXS>(sh.sx + 16 * wave, sh.d, nullptr);
    else
        tri_solve64<true, kXS>(sh.sx + 16 * wave, sh.d, sh.rd);
    lds_barrier();
    // lanes along the matrix rows (of a row-block tile: the wave's own lines)
    if (cols) {
#pragma unroll
        for (int c = 0; c < 16; ++c) {
            const int64_t col = c0 + 16 * wave + c;
            if (col < n) A[j + lane + col * lda] = sh.sx[16 * wave + c][lane];
        }
    } else {
        const int e = tid & 127, cq = 16 * (tid >> 7);
        if (i0 + e < n) {
#pragma unroll
            for (int c = 0; c < 16; ++c) A[i0 + e + (j + cq + c) * lda] = sh.sx[e][cq + c];
        }
    }
}

// Rows: X(i, :) <- X(i, :) * L^-1 for a 64 x 64 unit lower L (RLNU),
// columns from the last to the first.
__global__ void __launch_bounds__(256)
k_trsm_rows_rlnu64(int64_t m, const float *__restrict__ L, int64_t ldl, float *__restrict__ X,
                   int64_t ldx) {
    __shared__ float l[kNB][kNB + 1];
    load_tri64(L, ldl, l);
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= m) return;
    float x[kNB];
#pragma unroll
    for (int j = 0; j < kNB; ++j) x[j] = X[i + j * ldx];
#pragma unroll
    for (int j = kNB - 1; j >= 0; --j) {
        float v = x[j];
#pragma unroll
        for (int q = j + 1; q < kNB; ++q) v -= l[q][j] * x[q];
        x[j] = v;
    }
#pragma unroll
    for (int j = 0; j < kNB; ++j) X[i + j * ldx] = x[j];
}

// One block of kOB columns (RUNN, kUp) or rows (LLNU) of the triangular solves
// in one launch: a workgroup of 256 threads takes 64 lines (rows of X, columns
// of Y) of w = 64, 128, 192 or 256 entries.  64 entries at a time are read,
// lose their products with the lines' solved entries (each block of 64 summed
// by itself and subtracted, in the order of the product that a launch of its
// own would run: trsm_block_y), are solved (tri_solve64) and written; the
// solved entries stay in LDS.  As launches of 64 entries each (solve, then a
// depth-64 product over the rest of the block) the lines went to memory and
// back four times: 110 us a block for 30000 lines of 256.  Bound by the chain
// of four solves and their operands' latency, so what counts is how many
// workgroups a CU holds: two, with 70 KB of LDS each - the triangle lies in
// the piece's buffer that is free (the next one's, or the first's, whose
// products are then done), and the factor's blocks between go from memory to
// the registers of the lanes that multiply them.  RUNN blocks of 256 x 30000
// lines 61 -> 44 us, 58880 115 -> 80 (LLNU 55 -> 40, 106 -> 74) against the form
// with one workgroup a CU (100 KB); 16384 lines and below, where no CU has two,
// 32 (28).
constexpr int kXT = kNB + 4;
struct __align__(16) TrsmShared {
    float xs[kOB / kNB][kNB][kXT];  // the lines, a piece each: xs[piece][line][entry]
    float rd[kNB];
};

// a lane's factor entries for solved entries [64 i, +64) and its entry c of
// [64 j, +64): y[g][s] is U(64 i + k, 64 j + c) (kUp) or L(64 j + c, 64 i + k)
// with k = 32 h + 4 g + s, or 8 g + 2 s + h (seq: sums in the order of k)
template <bool kUp, bool kVec>
__device__ __forceinline__ void trsm_block_y(const float *__restrict__ T, int64_t ldt, int i, int j, int c, int h,
                                             bool seq, f32x4 (&y)[8]) {
    if constexpr (kUp) {
        const float *p = T + i * kNB + (int64_t)(j * kNB + c) * ldt;
        if (kVec) {  // always the first form: trsm_block_order makes the second of it
#pragma unroll
            for (int g = 0; g < 8; ++g) y[g] = *reinterpret_cast<const f32x4 *>(p + 32 * h + 4 * g);
        } else {
#pragma unroll
            for (int g = 0; g < 8; ++g)
#pragma unroll
                for (int s = 0; s < 4; ++s) y[g][s] = p[8 * g + 2 * s + h];
        }
    } else {
        const float *p = T + j * kNB + c + (int64_t)(i * kNB + (seq ? h : 32 * h)) * ldt;
        const int64_t step = (seq ? 2 : 1) * ldt;
#pragma unroll
        for (int g = 0; g < 8; ++g)
#pragma unroll
            for (int s = 0; s < 4; ++s) y[g][s] = p[(4 * g + s) * step];
    }
}

// y's k = 32 h + 4 g + s to k = 8 g + 2 s + h: of an even and the following odd
// k the two halves of the wave trade places (at the use, not at the load,
// where it would wait for it)
__device__ __forceinline__ void trsm_block_order(f32x4 (&y)[8]) {
    f32x4 o[8];
#pragma unroll
    for (int p = 0; p < 16; ++p) {
        // (through scalars: __builtin_bit_cast of a vector's element takes its first)
        const float a = y[p / 2][2 * p % 4], b = y[p / 2][2 * p % 4 + 1];
        const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b),
                                                        false, false);
        const unsigned lo = r[0], hi = r[1];
        o[p / 4][p % 4] = __builtin_bit_cast(float, lo);
        o[p / 4 + 4][p % 4] = __builtin_bit_cast(float, hi);
    }
#pragma unroll
    for (int g = 0; g < 8; ++g) y[g] = o[g];
}

template <bool kUp, bool kVec>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
k_trsm_block(int64_t lines, int w, const float *__restrict__ T, int64_t ldt, float *__restrict__ X, int64_t ldx) {
    __shared__ TrsmShared sh;
    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t e0 = (int64_t)blockIdx.x * kNB;
    const int nb = w / kNB;
    // 32 lines x 32 entries a wave
    const int wl = 32 * (wave & 1), wc = 32 * (wave >> 1);
    // the update's order of sums: that of the product over the rest of the
    // block that followed solved piece i
    auto in_order = [&](int i) {
        const int64_t inner = w - kNB * (i + 1);
        return !kVec || !mfma_size(kUp ? lines : inner, kUp ? inner : lines, 1);
    };
    // a thread's 16 values of a 64 x 64 piece: memory rows along the lanes;
    // lines past the end are read as the last one and not stored
    const int64_t le = min(e0 + lane, lines - 1) - e0;
    auto addr = [&](int j, int q) -> float * {
        return kUp ? X + e0 + le + (int64_t)(kNB * j + 16 * wave + q) * ldx
                   : X + kNB * j + lane + min(e0 + 16 * wave + q, lines - 1) * ldx;
    };
    float v[16];
    f32x4 y[8];
#pragma unroll
    for (int q = 0; q < 16; ++q) v[q] = *addr(0, q);
#pragma unroll 1
    for (int j = 0; j < nb; ++j) {
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int line = kUp ? lane : 16 * wave + q, c = kUp ? 16 * wave + q : lane;
            sh.xs[j][line][c] = v[q];
        }
        const float *tj = T + (kNB * j + lane) + (int64_t)(kNB * j + 16 * wave) * ldt;
        float d[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) d[q] = tj[(int64_t)q * ldt];
        if (j + 1 < nb) {  // the next piece, in flight during this one
#pragma unroll
            for (int q = 0; q < 16; ++q) v[q] = *addr(j + 1, q);
        }
        if (j > 0) lds_barrier();
#pragma unroll 1
        for (int i = 0; i < j; ++i) {
            const bool seq = in_order(i);
            const float *x = &sh.xs[i][wl + l32][seq ? h : 32 * h];
            f32x4 yn[8];
            if (i + 1 < j) trsm_block_y<kUp, kVec>(T, ldt, i + 1, j, wc + l32, h, in_order(i + 1), yn);
            if (kUp && kVec && seq) trsm_block_order(y);
            f32x16 acc;
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
#pragma unroll
            for (int g = 0; g < 8; ++g) {
                f32x4 xv;
                if (seq)
                    xv = f32x4{x[8 * g], x[8 * g + 2], x[8 * g + 4], x[8 * g + 6]};
                else
                    xv = *reinterpret_cast<const f32x4 *>(x + 4 * g);
#pragma unroll
                for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(y[g][s], xv[s], acc, 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                f32x4 *o = reinterpret_cast<f32x4 *>(&sh.xs[j][wl + l32][wc + 8 * r + 4 * h]);
                f32x4 n = *o;
#pragma unroll
                for (int s = 0; s < 4; ++s) n[s] -= acc[4 * r + s];
                *o = n;
            }
#pragma unroll
            for (int g = 0; g < 8; ++g) y[g] = yn[g];
        }
        // the triangle over the next piece's buffer, or the first's: neither
        // is read by now (the last solve is past a barrier, and so, below, are
        // the products)
        if (j > 0) lds_barrier();
        float (*t)[kNB + 1] = reinterpret_cast<float (*)[kNB + 1]>(&sh.xs[(j + 1) % (kOB / kNB)][0][0]);
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            t[lane][16 * wave + q] = d[q];
            if (kUp && lane == 16 * wave + q) sh.rd[lane] = 1.0f / d[q];
        }
        // (the next piece's first factor block, in flight during the solve)
        if (j + 1 < nb) trsm_block_y<kUp, kVec>(T, ldt, 0, j + 1, wc + l32, h, in_order(0), y);
        lds_barrier();
        tri_solve64<kUp, kXT>(&sh.xs[j][16 * wave], t, sh.rd);
        lds_barrier();
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int line = kUp ? lane : 16 * wave + q, c = kUp ? 16 * wave + q : lane;
            if (e0 + line < lines) *addr(j, q) = sh.xs[j][line][c];
        }
    }
}

// Inverses of the 64 x 64 diagonal blocks of the factored block D (L unit
// lower, U upper in one array): workgroup w < nblk writes U_ww^-1 into Xu
// (row r of it = e_r U_ww^-1, a row solve of the identity), workgroup nblk + w
// writes L_ww^-1 into Xl (column c = L_ww^-1 e_c).  The next 8 nblk workgroups
// clear what neither these nor the merges write, eight columns each: Xu below
// and Xl above the columns' diagonal block (a launch of its own took 5 us).
__global__ void __launch_bounds__(256)
k_tri_inv64(int nblk, const float *__restrict__ D, int64_t ldd, float *__restrict__ Xu, float *__restrict__ Xl,
            int64_t ldx) {
    __shared__ float t[kNB][kNB + 1];
    __shared__ __align__(16) float xs[kNB][kXS];
    __shared__ float rd[kNB];
    const int role = (int)blockIdx.x / nblk;
    if (role >= 2) {
        const int64_t n = (int64_t)nblk * kNB, c0 = (int64_t)((int)blockIdx.x - 2 * nblk) * 8;
        const int64_t o = c0 / kNB * kNB;
        for (int64_t c = c0; c < c0 + 8; ++c) {
            float *u = Xu + c * ldx, *l = Xl + c * ldx;
            for (int64_t i = o + kNB + threadIdx.x; i < n; i += 256) u[i] = 0.0f;
            for (int64_t i = threadIdx.x; i < o; i += 256) l[i] = 0.0f;
        }
        return;
    }
    const int64_t o = (int64_t)((int)blockIdx.x % nblk) * kNB;
    const bool up = role == 0;
    const int lane = threadIdx.x & 63, w0 = 16 * (threadIdx.x >> 6);
#pragma unroll
    for (int c = 0; c < 16; ++c) xs[w0 + c][lane] = w0 + c == lane ? 1.0f : 0.0f;
    load_tri64(D + o + o * ldd, ldd, t);
    if (up) {
        diag_recip64(t, rd);
        tri_solve64<true, kXS>(xs + w0, t, rd);
        __syncthreads();
#pragma unroll
        for (int c = 0; c < 16; ++c) Xu[o + lane + (o + w0 + c) * ldx] = xs[lane][w0 + c];
    } else {
        tri_solve64<false, kXS>(xs + w0, t, nullptr);
#pragma unroll
        for (int c = 0; c < 16; ++c) Xl[o + lane + (o + w0 + c) * ldx] = xs[w0 + c][lane];
    }
}

// One level of merges of the two inverses, ranges of up to kMergeMax rows:
//   U: X12 = -X1 (U12 X2)      L: X21 = -X2 (L21 X1)
// A workgroup of 512 threads takes 64 columns of one pair's X12 or X21: the
// inner product W stays in LDS between the two (as separate products a level
// took four launches of 14-25 us each; this one takes 23 us on average over
// the ranges of 64, 128 and 256 rows at n = 2560; beyond, the few workgroups
// a level has would run longer than two launches of more, k_sgemm_twin:
// 48 us each where the four took 100).  The triangles' zero blocks of
// 64 are skipped: their products are exact zeros.  Eight waves, 32 x 32 of
// a 128-row panel each, operands as in k_getrf_step64 (left operand's rows
// from global memory, right operand's columns, contiguous along k, from LDS)
// and sums in the order of the products this replaces (put_u).
constexpr int64_t kMergeMax = 256;

struct __align__(16) MergeShared {
    float su[kNB][kUS];                // a 64 x 64 block of the right operand: su[c][k]
    float sw[kNB][kMergeMax + 4];      // W: sw[c][k], each 64 of k in put_u's order
};

template <bool kVec>
__global__ void __launch_bounds__(kGT)
k_tri_merge(int64_t s1, int64_t s2, int64_t a0, const float *__restrict__ D, int64_t ldd, float *__restrict__ Xu,
            float *__restrict__ Xl, int64_t ldx, int seq_) {
    __shared__ MergeShared sh;
    const bool seq = seq_ != 0;
    const int nu = (int)(s2 / kNB), nl = (int)(s1 / kNB);  // strips of a pair's X12 and X21
    const int p = (int)blockIdx.x / (nu + nl), t = (int)blockIdx.x % (nu + nl);
    const bool up = t < nu;
    const int strip = up ? t : t - nu;
    a0 += p * (s1 + s2);
    const int64_t a1 = a0 + s1;
    float *X = up ? Xu : Xl;
    const int64_t ra = up ? a0 : a1, ca = up ? a1 : a0;  // the result's place
    const int64_t m = up ? s1 : s2;                      // its rows
    const int nk = (int)((up ? s2 : s1) / kNB);          // blocks of the inner product's k
    const float *P = X + ra + ra * ldx, *Q = D + ra + ca * ldd;
    const float *R = X + ca + (ca + (int64_t)strip * kNB) * ldx;  // the right operand's columns
    float *out = X + ra + (ca + (int64_t)strip * kNB) * ldx;
    const int lane = threadIdx.x & 63, l32 = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wc = 32 * (wave >> 2);
    f32x32 l;
    f32x16 acc;
    // W = Q R: R is triangular with its blocks on the diagonal
    const int k0 = up ? 0 : strip, k1 = up ? strip + 1 : nk;
    for (int64_t r0 = 0; r0 < m; r0 += 128) {
        const int64_t row = r0 + 32 * (wave & 3);
        const bool act = row < m;
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
#pragma unroll 1
        for (int k = k0; k < k1; ++k) {
            f32x4 u2[2];
            get_u<kVec>(R + (int64_t)k * kNB, ldx, kNB, u2);
            if (act) load_l(Q + row + l32 + (int64_t)k * kNB * ldd, ldd, h, seq, l);
            lds_barrier();  // (the block before is read)
            put_u(u2, sh.su, seq);
            lds_barrier();
            if (act) mfma32(l, &sh.su[wc + l32][32 * h], acc);
        }
        if (act) {
            // row index as the k of the second product
            const int kk = (int)((row + l32) & 63);
            const int pos = (int)((row + l32) & ~63) + (seq ? (kk & 1) * 32 + (kk >> 1) : kk);
#pragma unroll
            for (int v = 0; v < 16; ++v) sh.sw[wc + 8 * (v >> 2) + 4 * h + (v & 3)][pos] = acc[v];
        }
    }
    lds_barrier();
    // result = -P W
    for (int64_t r0 = 0; r0 < m; r0 += 128) {
        const int64_t row = r0 + 32 * (wave & 3);
        if (row >= m) break;
        const int rb = (int)(row / kNB), nb = (int)(m / kNB);
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
#pragma unroll 1
        for (int k = up ? rb : 0; k < (up ? nb : rb + 1); ++k) {
            load_l(P + row + l32 + (int64_t)k * kNB * ldx, ldx, h, seq, l);
            mfma32(l, &sh.sw[wc + l32][kNB * k + 32 * h], acc);
        }
#pragma unroll
        for (int v = 0; v < 16; ++v) out[row + l32 + (int64_t)(wc + 8 * (v >> 2) + 4 * h + (v & 3)) * ldx] = -acc[v];
    }
}

__global__ void k_identity(int64_t n, float *__restrict__ A, int64_t lda) {
    const int64_t j = blockIdx.y;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        A[i + j * lda] = (i == j) ? 1.0f : 0.0f;
}

__global__ void k_copy_block(int64_t m, const float *__restrict__ A, int64_t lda, float *__restrict__ B,
                             int64_t ldb) {
    const int64_t j = blockIdx.y;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (int64_t)gridDim.x * blockDim.x)
        B[i + j * ldb] = A[i + j * lda];
}

bool use_mfma(int64_t m, int64_t n, int64_t k, int64_t batch, const float *A, int64_t lda, const float *B,
              int64_t ldb) {
    const bool aligned = (reinterpret_cast<uintptr_t>(A) & 15) == 0 && (reinterpret_cast<uintptr_t>(B) & 15) == 0 &&
                         (lda & 3) == 0 && (ldb & 3) == 0 && k >= 16 && k % 16 == 0;
    return aligned && mfma_size(m, n, batch);
}

int sgemm_mfma(int64_t m, int64_t n, int64_t k, float alpha, const float *A, int64_t lda, int64_t sA, const float *B,
               int64_t ldb, int64_t sB, float beta, float *C, int64_t ldc, int64_t sC, int64_t batch, hipStream_t st) {
    // 128-tiles halve the operands' traffic, which counts where k is deep and
    // the matrix large (61440 x 61440 x 2560: 141 ms, 64-tiles 155); otherwise
    // four workgroups a CU of 64-tiles hide one another's loads and C as well
    // or better (30000 x 2304 x 256: 383 and 393 us; 7680 x 7680 x 512: both
    // 528), and few tiles leave CUs idle
    const bool big = k >= 512 && omx_cdiv(m, 128) * omx_cdiv(n, 128) * batch >= 1024;
    const int t = big ? 128 : 64;
    const dim3 grid((unsigned)omx_cdiv(m, t), (unsigned)omx_cdiv(n, t), (unsigned)batch);
    if (big)
        hipLaunchKernelGGL(k_sgemm_mfma<128>, grid, dim3(256), 0, st, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, sA,
                           sB, sC);
    else
        hipLaunchKernelGGL(k_sgemm_mfma<64>, grid, dim3(256), 0, st, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, sA,
                           sB, sC);
    OMX_LAUNCH_CHECK();
    return OMX_OK;
}

// msel: the row count the kernel is chosen for (default m).  A caller that
// skips rows known to be zero passes the full count, so that the rows it
// does compute round exactly as in the full product.
int sgemm(int64_t m, int64_t n, int64_t k, float alpha, const float *A, int64_t lda, const float *B,
          int64_t ldb, float beta, float *C, int64_t ldc, hipStream_t st, int64_t msel = -1) {
    if (m <= 0 || n <= 0) return OMX_OK;
    if (use_mfma(msel < 0 ? m : msel, n, k, 1, A, lda, B, ldb)) {
        return sgemm_mfma(m, n, k, alpha, A, lda, 0, B, ldb, 0, beta, C, ldc, 0, 1, st);
    }
    dim3 grid((unsigned)omx_cdiv(m, 64), (unsigned)omx_cdiv(n, 64));
    if (grid.y > 65535) return OMX_ERR_ARG;
    hipLaunchKernelGGL(k_sgemm_nn, grid, dim3(256), 0, st, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc,
                       (int64_t)0, (int64_t)0, (int64_t)0);
    OMX_LAUNCH_CHECK();
    return OMX_OK;
}

// batch products C_p = beta C_p + alpha A_p B_p, X_p = X + p * sX
int sgemm_batched(int64_t m, int64_t n, int64_t k, float alpha, const float *A, int64_t lda, int64_t sA,
                  const float *B, int64_t ldb, int64_t sB, float beta, float *C, int64_t ldc, int64_t sC,
                  int64_t batch, hipStream_t st) {
    if (m <= 0 || n <= 0 || batch <= 0) return OMX_OK;
    dim3 grid((unsigned)omx_cdiv(m, 64), (unsigned)omx_cdiv(n, 64), (unsigned)batch);
    if (grid.y > 65535 || batch > 65535 || k % 16) return OMX_ERR_ARG;
    if (use_mfma(m, n, k, batch, A, lda, B, ldb) && (sA & 3) == 0 && (sB & 3) == 0) {
        return sgemm_mfma(m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, batch, st);
    }
    hipLaunchKernelGGL(k_sgemm_nn, grid, dim3(256), 0, st, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, sA, sB,
                       sC);
    OMX_LAUNCH_CHECK();
    return OMX_OK;
}

// two batches of batch products each (k_sgemm_twin)
int sgemm_twin(const SgemmTwin &g0, const SgemmTwin &g1, float alpha, int64_t batch, hipStream_t st) {
    const int64_t m = std::max(g0.M, g1.M), n = std::max(g0.N, g1.N);
    const dim3 grid((unsigned)omx_cdiv(m, 64), (unsigned)omx_cdiv(n, 64), (unsigned)(2 * batch));
    hipLaunchKernelGGL(k_sgemm_twin, grid, dim3(256), 0, st, g0, g1, alpha, (int)batch);
    OMX_LAUNCH_CHECK();
    return OMX_OK;
}

// one block of the triangular solves (k_trsm_block); the order of its sums
// goes by the operands' alignment as in the products it replaces
template <bool kUp>
int trsm_block(int64_t lines, int64_t w, const float *T, int64_t ldt, float *X, int64_t ldx, hipStream_t st) {
    const bool vec = ((reinterpret_cast<uintptr_t>(T) | reinterpret_cast<uintptr_t>(X)) & 15) == 0 && (ldt & 3) == 0 &&
                     (ldx & 3) == 0;
    const dim3 grid((unsigned)omx_cdiv(lines, kNB));
    if (omx_cdiv(lines, kNB) >= ((int64_t)1 << 31)) return OMX_ERR_ARG;
    if (vec)
        hipLaunchKernelGGL((k_trsm_block<kUp, true>), grid, dim3(256), 0, st, lines, (int)w, T, ldt, X, ldx);
    else
        hipLaunchKernelGGL((k_trsm_block<kUp, false>), grid, dim3(256), 0, st, lines, (int)w, T, ldt, X, ldx);
    OMX_LAUNCH_CHECK();
    return OMX_OK;
}

// sgemm with n split into chunks of at most 65535*64 columns
int sgemm_big(int64_t m, int64_t n, int64_t k, float alpha, const float *A, int64_t lda, const float *B,
              int64_t ldb, float beta, float *C, int64_t ldc, hipStream_t st, int64_t msel = -1) {
    const int64_t nmax = (int64_t)65535 * 64;
    for (int64_t j = 0; j < n; j += nmax) {
        const int64_t nn = (n - j < nmax) ? n - j : nmax;
        int rc = sgemm(m, nn, k, alpha, A, lda, B + j * ldb, ldb, beta, C + j * ldc, ldc, st, msel);
        if (rc) return rc;
    }
    return OMX_OK;
}

}  // namespace

extern "C" {

int omx_sgemm_f32(int64_t m, int64_t n, int64_t k, float alpha, const float *A, int64_t lda,
                  const float *B, int64_t ldb, float beta, float *C, int64_t ldc, void *stream) {
    if (m < 0 || n < 0 || k <= 0 || k % 16 || !A || !B || !C || lda < m || ldb < k || ldc < m)
        return OMX_ERR_ARG;
    return sgemm_big(m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, omx_stream(stream));
}

int omx_getrf_nopiv_f32(int64_t n, float *A, int64_t lda, int *info, void *stream) {
    if (n <= 0 || n % kNB || !A || lda < n) return OMX_ERR_ARG;
    hipStream_t st = omx_stream(stream);
    const bool vec = (reinterpret_cast<uintptr_t>(A) & 15) == 0 && (lda & 3) == 0;
    for (int64_t j = 0; j < n; j += kNB) {
        const int64_t rest = n - j - kNB;
        const int64_t np = omx_cdiv(rest, 128);
        int64_t grid = np > 0 ? 2 * np : 1;
        if (j > 0) grid += 1 + np * (rest / kNB);  // the previous D's writer, the trailing tiles
        if (grid >= ((int64_t)1 << 31)) return OMX_ERR_ARG;
        if (j == 0)  // no update yet: nothing is staged
            hipLaunchKernelGGL((k_getrf_step64<false, false>), dim3((unsigned)grid), dim3(kGT), 0, st, n, j, (int)np,
                               A, lda, info);
        else if (vec)
            hipLaunchKernelGGL((k_getrf_step64<true, true>), dim3((unsigned)grid), dim3(kGT), 0, st, n, j, (int)np, A,
                               lda, info);
        else
            hipLaunchKernelGGL((k_getrf_step64<true, false>), dim3((unsigned)grid), dim3(kGT), 0, st, n, j, (int)np, A,
                               lda, info);
        OMX_LAUNCH_CHECK();
    }
    return OMX_OK;
}

int omx_trsm_f32(int variant, int64_t m, int64_t n, const float *T, int64_t ldt, float *B, int64_t ldb,
                 void *stream) {
    if (m < 0 || n < 0 || !T || !B || ldb < m) return OMX_ERR_ARG;
    if (m == 0 || n == 0) return OMX_OK;
    hipStream_t st = omx_stream(stream);
    if (variant == OMX_TRSM_RUNN || variant == OMX_TRSM_RLNU) {
        // B (m x n) times the inverse of an n x n triangle, n % 64 == 0
        if (n % kNB || ldt < n) return OMX_ERR_ARG;
        const unsigned g = (unsigned)omx_cdiv(m, 256);
        if (variant == OMX_TRSM_RUNN) {
            for (int64_t J0 = 0; J0 < n; J0 += kOB) {
                const int64_t w = std::min(kOB, n - J0);
                RC(trsm_block<true>(m, w, T + J0 + J0 * ldt, ldt, B + J0 * ldb, ldb, st));
                const int64_t rest = n - J0 - w;
                if (rest > 0) RC(sgemm_big(m, rest, w, -1.0f, B + J0 * ldb, ldb, T + J0 + (J0 + w) * ldt, ldt, 1.0f,
                                           B + (J0 + w) * ldb, ldb, st));
            }
        } else {
            for (int64_t J1 = n; J1 > 0; J1 -= kOB) {
                const int64_t J0 = std::max<int64_t>(0, J1 - kOB);
                for (int64_t j = J1 - kNB; j >= J0; j -= kNB) {
                    hipLaunchKernelGGL(k_trsm_rows_rlnu64, dim3(g), dim3(256), 0, st, m, T + j + j * ldt, ldt,
                                       B + j * ldb, ldb);
                    OMX_LAUNCH_CHECK();
                    if (j > J0) RC(sgemm_big(m, j - J0, kNB, -1.0f, B + j * ldb, ldb, T + j + J0 * ldt, ldt, 1.0f,
                                             B + J0 * ldb, ldb, st));
                }
                if (J0 > 0) RC(sgemm_big(m, J0, J1 - J0, -1.0f, B + J0 * ldb, ldb, T + J0, ldt, 1.0f, B, ldb, st));
            }
        }
        return OMX_OK;
    }
    if (variant == OMX_TRSM_LLNU) {
        // inverse of an m x m unit lower triangle times B (m x n), m % 64 == 0
        if (m % kNB || ldt < m) return OMX_ERR_ARG;
        for (int64_t I0 = 0; I0 < m; I0 += kOB) {
            const int64_t w = std::min(kOB, m - I0);
            RC(trsm_block<false>(n, w, T + I0 + I0 * ldt, ldt, B + I0, ldb, st));
            const int64_t rest = m - I0 - w;
            if (rest > 0) RC(sgemm_big(rest, n, w, -1.0f, T + (I0 + w) + I0 * ldt, ldt, B + I0, ldb, 1.0f,
                                       B + I0 + w, ldb, st));
        }
        return OMX_OK;
    }
    return OMX_ERR_ARG;
}

int omx_trtri_lu_f32(int64_t n, const float *D, int64_t ldd, float *Xu, float *Xl, int64_t ldx, float *work,
                     void *stream) {
    if (n <= 0 || n % kNB || n > 65535 || !D || !Xu || !Xl || !work || ldd < n || ldx < n) return OMX_ERR_ARG;
    hipStream_t st = omx_stream(stream);
    const int nblk = (int)(n / kNB);
    hipLaunchKernelGGL(k_tri_inv64, dim3((unsigned)(10 * nblk)), dim3(256), 0, st, nblk, D, ldd, Xu, Xl, ldx);
    OMX_LAUNCH_CHECK();
    // Merge adjacent ranges of diagonal blocks level by level: ranges of s0
    // blocks pair up (the last, odd one waits for a later level).  For the
    // pair [R1 | R2] with inverses X1, X2 on the diagonal:
    //   U: X12 = -X1 (U12 X2)      L: X21 = -X2 (L21 X1)
    // with the inner product in LDS (k_tri_merge) or in work (n x n, leading
    // dimension n, at the position of the block it becomes).  Pairs of equal
    // sizes run batched.
    const bool vec = ((reinterpret_cast<uintptr_t>(D) | reinterpret_cast<uintptr_t>(Xu) |
                       reinterpret_cast<uintptr_t>(Xl) | reinterpret_cast<uintptr_t>(work)) & 15) == 0 &&
                     (ldd & 3) == 0 && (ldx & 3) == 0;
    std::vector<int64_t> sz(nblk, kNB);  // range sizes in rows, in order
    while (sz.size() > 1) {
        std::vector<int64_t> next;
        int64_t pos = 0;
        size_t i = 0;
        while (i + 1 < sz.size()) {
            // a batch: consecutive pairs with the same (s1, s2)
            const int64_t s1 = sz[i], s2 = sz[i + 1];
            int64_t cnt = 0;
            while (i + 1 < sz.size() && sz[i] == s1 && sz[i + 1] == s2) {
                ++cnt;
                i += 2;
            }
            const int64_t stride = s1 + s2;  // along the diagonal, per pair
            const int64_t a0 = pos, a1 = pos + s1;
            for (int64_t c = 0; c < cnt; ++c) next.push_back(stride);
            pos += cnt * stride;
            if (std::max(s1, s2) <= kMergeMax) {
                const dim3 grid((unsigned)(cnt * (stride / kNB)));
                const int seq = vec && mfma_size(s1, s2, cnt) ? 0 : 1;
                if (vec)
                    hipLaunchKernelGGL(k_tri_merge<true>, grid, dim3(kGT), 0, st, s1, s2, a0, D, ldd, Xu, Xl, ldx, seq);
                else
                    hipLaunchKernelGGL(k_tri_merge<false>, grid, dim3(kGT), 0, st, s1, s2, a0, D, ldd, Xu, Xl, ldx,
                                       seq);
                OMX_LAUNCH_CHECK();
                continue;
            }
            const int64_t dstep = stride * (ldd + 1), xstep = stride * (ldx + 1), wstep = stride * (n + 1);
            if (vec && 2 * cnt <= 65535) {
                // both sides' inner products, then both results, on the matrix
                // cores however few the tiles: the 512 + 256 of n = 768 took
                // 190 us as four products of 64 x 64 VALU tiles, now 35
                const SgemmTwin wu{s1, s2, s2, ldd, ldx, n, dstep, xstep, wstep, 1, D + a0 + a1 * ldd,
                                   Xu + a1 + a1 * ldx, work + a0 + a1 * n};
                const SgemmTwin wl{s2, s1, s1, ldd, ldx, n, dstep, xstep, wstep, 2, D + a1 + a0 * ldd,
                                   Xl + a0 + a0 * ldx, work + a1 + a0 * n};
                const SgemmTwin xu{s1, s2, s1, ldx, n, ldx, xstep, wstep, xstep, 3, Xu + a0 + a0 * ldx,
                                   work + a0 + a1 * n, Xu + a0 + a1 * ldx};
                const SgemmTwin xl{s2, s1, s2, ldx, n, ldx, xstep, wstep, xstep, 4, Xl + a1 + a1 * ldx,
                                   work + a1 + a0 * n, Xl + a1 + a0 * ldx};
                RC(sgemm_twin(wu, wl, 1.0f, cnt, st));
                RC(sgemm_twin(xu, xl, -1.0f, cnt, st));
                continue;
            }
            int rc;
            // U: work(a0.., a1..) = U12 X2;  Xu(a0.., a1..) = -X1 work
            rc = sgemm_batched(s1, s2, s2, 1.0f, D + a0 + a1 * ldd, ldd, stride * (ldd + 1), Xu + a1 + a1 * ldx, ldx,
                               stride * (ldx + 1), 0.0f, work + a0 + a1 * n, n, stride * (n + 1), cnt, st);
            if (rc) return rc;
            rc = sgemm_batched(s1, s2, s1, -1.0f, Xu + a0 + a0 * ldx, ldx, stride * (ldx + 1), work + a0 + a1 * n, n,
                               stride * (n + 1), 0.0f, Xu + a0 + a1 * ldx, ldx, stride * (ldx + 1), cnt, st);
            if (rc) return rc;
            // L: work(a1.., a0..) = L21 X1;  Xl(a1.., a0..) = -X2 work
            rc = sgemm_batched(s2, s1, s1, 1.0f, D + a1 + a0 * ldd, ldd, stride * (ldd + 1), Xl + a0 + a0 * ldx, ldx,
                               stride * (ldx + 1), 0.0f, work + a1 + a0 * n, n, stride * (n + 1), cnt, st);
            if (rc) return rc;
            rc = sgemm_batched(s2, s1, s2, -1.0f, Xl + a1 + a1 * ldx, ldx, stride * (ldx + 1), work + a1 + a0 * n, n,
                               stride * (n + 1), 0.0f, Xl + a1 + a0 * ldx, ldx, stride * (ldx + 1), cnt, st);
            if (rc) return rc;
        }
        if (i < sz.size()) next.push_back(sz[i]);
        sz.swap(next);
    }
    return OMX_OK;
}

int omx_trsm_identity_f32(int variant, int64_t n, const float *T, int64_t ldt, float *X, int64_t ldx,
                          void *stream) {
    if (n <= 0 || n % kNB || n > 65535 || !T || !X || ldt < n || ldx < n) return OMX_ERR_ARG;
    if (variant != OMX_TRSM_RUNN && variant != OMX_TRSM_RLNU) return OMX_ERR_ARG;
    hipStream_t st = omx_stream(stream);
    hipLaunchKernelGGL(k_identity, dim3((unsigned)omx_cdiv(n, 256), (unsigned)n), dim3(256), 0, st, n, X, ldx);
    OMX_LAUNCH_CHECK();
    // the blocking of omx_trsm_f32, the products restricted to the rows
    // that can be nonzero, the kernels chosen for all n rows: the results are
    // those of omx_trsm_f32 on the identity
    if (variant == OMX_TRSM_RUNN) {
        // block column j of I * U^-1 is zero below row j + 63
        for (int64_t J0 = 0; J0 < n; J0 += kOB) {
            const int64_t w = std::min(kOB, n - J0);
            for (int64_t j = J0; j < J0 + w; j += kNB) {
                const int64_t rows = j + kNB;
                hipLaunchKernelGGL(k_trsm_rows_runn64, dim3((unsigned)omx_cdiv(rows, 64)), dim3(256), 0, st, rows,
                                   T + j + j * ldt, ldt, X + j * ldx, ldx);
                OMX_LAUNCH_CHECK();
                const int64_t inner = J0 + w - j - kNB;
                if (inner > 0) RC(sgemm_big(rows, inner, kNB, -1.0f, X + j * ldx, ldx, T + j + (j + kNB) * ldt, ldt,
                                            1.0f, X + (j + kNB) * ldx, ldx, st, n));
            }
            const int64_t rest = n - J0 - w;
            if (rest > 0) RC(sgemm_big(J0 + w, rest, w, -1.0f, X + J0 * ldx, ldx, T + J0 + (J0 + w) * ldt, ldt, 1.0f,
                                       X + (J0 + w) * ldx, ldx, st, n));
        }
        return OMX_OK;
    }
    // block column j of I * L^-1 is zero above row j
    for (int64_t J1 = n; J1 > 0; J1 -= kOB) {
        const int64_t J0 = std::max<int64_t>(0, J1 - kOB);
        for (int64_t j = J1 - kNB; j >= J0; j -= kNB) {
            const int64_t rows = n - j;
            hipLaunchKernelGGL(k_trsm_rows_rlnu64, dim3((unsigned)omx_cdiv(rows, 256)), dim3(256), 0, st, rows,
                               T + j + j * ldt, ldt, X + j + j * ldx, ldx);
            OMX_LAUNCH_CHECK();
            if (j > J0) RC(sgemm_big(rows, j - J0, kNB, -1.0f, X + j + j * ldx, ldx, T + j + J0 * ldt, ldt, 1.0f,
                                     X + j + J0 * ldx, ldx, st, n));
        }
        if (J0 > 0) RC(sgemm_big(n - J0, J0, J1 - J0, -1.0f, X + J0 + J0 * ldx, ldx, T + J0, ldt, 1.0f, X + J0, ldx,
                                 st, n));
    }
    return OMX_OK;
}

int omx_identity_f32(int64_t n, float *A, int64_t lda, void *stream) {
    if (n <= 0 || !A || lda < n || n > 65535) return OMX_ERR_ARG;
    hipLaunchKernelGGL(k_identity, dim3((unsigned)omx_cdiv(n, 256), (unsigned)n), dim3(256), 0,
                       omx_stream(stream), n, A, lda);
    OMX_LAUNCH_CHECK();
    return OMX_OK;
}

int omx_copy_block_f32(int64_t m, int64_t n, const float *A, int64_t lda, float *B, int64_t ldb,
                       void *stream) {
    if (m < 0 || n < 0 || n > 65535 || !A || !B || lda < m || ldb < m) return OMX_ERR_ARG;
    if (m == 0 || n == 0) return OMX_OK;
    hipLaunchKernelGGL(k_copy_block, dim3((unsigned)omx_cdiv(m, 256), (unsigned)n), dim3(256), 0,
                       omx_stream(stream), m, A, lda, B, ldb);
    OMX_LAUNCH_CHECK();
    return OMX_OK;
}

}  // extern "C"
