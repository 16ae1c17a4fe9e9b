// omx_mlp.hip -- the learned per-step precision scheduler: an MLP
// 16-64-64-3 (FP32, ReLU) with forward, backward and Adam kernels, and the
// feature kernel that turns a panel step's statistics into its 16 inputs.
// No reference counterpart (the reference always uses FP16).
//
// Parameters are one flat FP32 array (OMX_MLP_NPARAMS):
//   W1[16][64] | b1[64] | W2[64][64] | b2[64] | W3[64][3] | b3[3]
// with W[i][j] the weight from input i to unit j.  Outputs z0, z1 are the
// logits of FP16 / FP8 for the step's Schur update; z2 is the FP8 tile-scale
// headroom in bits (rounded and clamped to 0..3).
//
// Contraction is off in this file: each sum is the same sequence of FP32
// roundings (bias first, inputs in order) as the CPU oracle, so the forward
// pass is bit-identical to it.
#include <algorithm>
#include <cmath>

#include "omx_common.hpp"

#pragma clang fp contract(off)

namespace {

constexpr int kIn = 16, kH = 64, kOut = 3;
constexpr int kW1 = 0;
constexpr int kB1 = kW1 + kIn * kH;
constexpr int kW2 = kB1 + kH;
constexpr int kB2 = kW2 + kH * kH;
constexpr int kW3 = kB2 + kH;
constexpr int kB3 = kW3 + kH * kOut;
constexpr int kNP = kB3 + kOut;
static_assert(kNP == OMX_MLP_NPARAMS, "parameter count");
constexpr int kD = kOut + 2 * kH;  // per-sample backward deltas: dz, d2, d1

__device__ __forceinline__ void load_params(float *p, const float *__restrict__ params) {
    for (int i = threadIdx.x; i < kNP; i += blockDim.x) p[i] = params[i];
    __syncthreads();
}

// 16 samples per workgroup: a wave takes four, a lane one hidden unit, so the
// 64 x 64 layer is 64 steps of one weight read and four independent sums
// (each in the oracle's order: bias, then inputs ascending) instead of a
// thread walking all 64 units of a sample by itself.  Bound by launch,
// parameter load and those sums' latency: 2658 samples 47 -> 7 us, a single
// sample (one step of the LU's policy) 52 -> 7 us.
constexpr int kFS = 16;        // samples per workgroup
constexpr int kFW = kFS / 4;   // per wave

__global__ void __launch_bounds__(256)
k_mlp_forward(int64_t batch, const float *__restrict__ params, const float *__restrict__ X, float *__restrict__ H1,
              float *__restrict__ H2, float *__restrict__ Z) {
    __shared__ float p[kNP];
    __shared__ __align__(16) float xs[4][kIn][kFW];  // [wave][input][sample]
    __shared__ __align__(16) float hs[4][kH][kFW];   // hidden layer of the wave's samples
    const int wave = threadIdx.x >> 6, j = threadIdx.x & 63;
    const int64_t s0 = (int64_t)blockIdx.x * kFS + wave * kFW;
    {
        const int64_t s = s0 + (j >> 4);
        xs[wave][j & 15][j >> 4] = s < batch ? X[s * kIn + (j & 15)] : 0.0f;
    }
    load_params(p, params);
    float a[kFW];
#pragma unroll
    for (int u = 0; u < kFW; ++u) a[u] = p[kB1 + j];
#pragma unroll
    for (int i = 0; i < kIn; ++i) {
        const float w = p[kW1 + i * kH + j];
#pragma unroll
        for (int u = 0; u < kFW; ++u) a[u] += xs[wave][i][u] * w;
    }
#pragma unroll
    for (int u = 0; u < kFW; ++u) {
        const float h = a[u] > 0.0f ? a[u] : 0.0f;
        hs[wave][j][u] = h;
        if (s0 + u < batch) H1[(s0 + u) * kH + j] = h;
        a[u] = p[kB2 + j];
    }
    __syncthreads();
#pragma unroll 16
    for (int i = 0; i < kH; ++i) {
        const float w = p[kW2 + i * kH + j];
#pragma unroll
        for (int u = 0; u < kFW; ++u) a[u] += hs[wave][i][u] * w;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kFW; ++u) {
        const float h = a[u] > 0.0f ? a[u] : 0.0f;
        hs[wave][j][u] = h;
        if (s0 + u < batch) H2[(s0 + u) * kH + j] = h;
    }
    __syncthreads();
    // z_o = b3_o + sum_i h2_i W3[i][o], a lane per (sample, output)
    if (j < kFW * kOut) {
        const int u = j / kOut, o = j % kOut;
        float z = p[kB3 + o];
#pragma unroll 16
        for (int i = 0; i < kH; ++i) z += hs[wave][i][u] * p[kW3 + i * kOut + o];
        if (s0 + u < batch) Z[(s0 + u) * kOut + o] = z;
    }
}

// Backward of a chunk of samples in one workgroup of 1024 threads, 16
// samples at a time through LDS: per sample the deltas dz (3), d2 = dL/d
// (pre-activation 2), d1 (64 each) of the mean loss, then their products with
// the layer inputs added, sample by sample, to the gradient entries that the
// threads hold in registers (thread t: the 4 entries of W2 row t / 16 from
// column 4 (t % 16), one entry of W1, and one of W3 or the biases).  A batch
// of one chunk is finished here; otherwise the chunk's sums go to part and
// k_mlp_grad_reduce adds them in chunk order.  The chunks are as many as the
// workspace holds (one per 41 samples, kMaxChunks at most).  With a thread
// per parameter walking the whole batch, a thread per sample for the deltas
// and one thread for the loss, 2658 samples took 874 us (grad 679, loss 137,
// deltas 58); bound now by LDS reads and the latency of the 64-step d1 sums.
constexpr int kBS = 16;          // samples per pass
constexpr int kBT = 1024;        // threads
constexpr int kMaxChunks = 256;

// bytes of a chunk's partial sums: the gradient and the loss (FP64)
constexpr size_t kChunkBytes = ((size_t)kNP * sizeof(float) + sizeof(double) + 15) / 8 * 8;
static_assert(kChunkBytes <= 41 * (kD * sizeof(float) + sizeof(double)), "one chunk per 41 samples");

__global__ void __launch_bounds__(kBT)
k_mlp_backward(int64_t batch, int64_t chunk, const float *__restrict__ params, const float *__restrict__ X,
               const float *__restrict__ H1, const float *__restrict__ H2, const float *__restrict__ Z,
               const int32_t *__restrict__ y, const float *__restrict__ t, const float *__restrict__ m,
               float *__restrict__ grad, float *__restrict__ loss, float *__restrict__ part,
               double *__restrict__ lpart) {
    __shared__ float xs[kBS][kIn], h1[kBS][kH], h2[kBS][kH], dz[kBS][kOut], d1[kBS][kH];
    __shared__ __align__(16) float d2[kBS][kH];
    __shared__ double ls[kBS];
    const int tid = threadIdx.x, lane = tid & 63;
    const int sl = tid >> 6;  // this thread's sample of a pass, in the per-sample phases
    const int64_t b0 = (int64_t)blockIdx.x * chunk;
    const int64_t b1 = b0 + chunk < batch ? b0 + chunk : batch;
    const float inv = 1.0f / (float)batch;
    // row `lane` of W2 and of W3
    float w2[kH], w3[kOut];
#pragma unroll
    for (int j = 0; j < kH; ++j) w2[j] = params[kW2 + lane * kH + j];
#pragma unroll
    for (int j = 0; j < kOut; ++j) w3[j] = params[kW3 + lane * kOut + j];
    const int gi = tid >> 4, gj = (tid & 15) * 4;  // W2 entries (gi, gj .. gj + 3)
    float g2[4] = {}, g1 = 0.0f, g3 = 0.0f;
    double lsum = 0.0;
    for (int64_t s0 = b0; s0 < b1; s0 += kBS) {
        const int cnt = (int)(b1 - s0 < kBS ? b1 - s0 : kBS);
        const int64_t s = s0 + sl;
        const bool in = sl < cnt;
        if (in) {
            h1[sl][lane] = H1[s * kH + lane];
            h2[sl][lane] = H2[s * kH + lane];
            if (lane < kIn) xs[sl][lane] = X[s * kIn + lane];
            // the sample's three deltas, the same in every lane
            const float z0 = Z[s * kOut], z1 = Z[s * kOut + 1], z2 = Z[s * kOut + 2];
            const float mx = z0 > z1 ? z0 : z1;
            const float e0 = expf(z0 - mx), e1 = expf(z1 - mx);
            const float p0 = e0 / (e0 + e1), p1 = e1 / (e0 + e1);
            const int ys = y[s];
            const float ms = m[s], diff = z2 - t[s];
            const float q0 = (p0 - (ys ? 0.0f : 1.0f)) * inv;
            const float q1 = (p1 - (ys ? 1.0f : 0.0f)) * inv;
            const float q2 = ms * diff * inv;
            if (lane == 0) {
                dz[sl][0] = q0;
                dz[sl][1] = q1;
                dz[sl][2] = q2;
                const float lse = mx + logf(e0 + e1);
                ls[sl] = (double)(lse - (ys ? z1 : z0)) + 0.5 * (double)(ms * diff * diff);
            }
            float a = 0.0f;
            a += w3[0] * q0;
            a += w3[1] * q1;
            a += w3[2] * q2;
            d2[sl][lane] = h2[sl][lane] > 0.0f ? a : 0.0f;
        }
        __syncthreads();
        if (in) {
            float a = 0.0f;
#pragma unroll
            for (int j = 0; j < kH; ++j) a += w2[j] * d2[sl][j];
            d1[sl][lane] = h1[sl][lane] > 0.0f ? a : 0.0f;
        }
        __syncthreads();
        for (int q = 0; q < cnt; ++q) {
            const float h = h1[q][gi];
#pragma unroll
            for (int e = 0; e < 4; ++e) g2[e] += h * d2[q][gj + e];
            g1 += xs[q][sl] * d1[q][lane];
        }
        if (tid < kH * kOut) {
            for (int q = 0; q < cnt; ++q) g3 += h2[q][tid / kOut] * dz[q][tid % kOut];
        } else if (tid < kH * kOut + kH) {
            for (int q = 0; q < cnt; ++q) g3 += d2[q][tid - kH * kOut];
        } else if (tid < kH * kOut + 2 * kH) {
            for (int q = 0; q < cnt; ++q) g3 += d1[q][tid - kH * kOut - kH];
        } else if (tid < kH * kOut + 2 * kH + kOut) {
            for (int q = 0; q < cnt; ++q) g3 += dz[q][tid - kH * kOut - 2 * kH];
        } else if (tid == kBT - 1) {
            for (int q = 0; q < cnt; ++q) lsum += ls[q];
        }
        __syncthreads();
    }
    float *out = part ? part + (int64_t)blockIdx.x * kNP : grad;
#pragma unroll
    for (int e = 0; e < 4; ++e) out[kW2 + gi * kH + gj + e] = g2[e];
    out[kW1 + sl * kH + lane] = g1;
    if (tid < kH * kOut) out[kW3 + tid] = g3;
    else if (tid < kH * kOut + kH) out[kB2 + tid - kH * kOut] = g3;
    else if (tid < kH * kOut + 2 * kH) out[kB1 + tid - kH * kOut - kH] = g3;
    else if (tid < kH * kOut + 2 * kH + kOut) out[kB3 + tid - kH * kOut - 2 * kH] = g3;
    else if (tid == kBT - 1) {
        if (part) lpart[blockIdx.x] = lsum;
        else *loss = (float)(lsum / (double)batch);
    }
}

// grad = the chunks' sums in chunk order, a thread per parameter; the loss
// likewise in the last workgroup's last thread.
__global__ void __launch_bounds__(64)
k_mlp_grad_reduce(int64_t batch, int nchunk, const float *__restrict__ part, const double *__restrict__ lpart,
                  float *__restrict__ grad, float *__restrict__ loss) {
    const int q = blockIdx.x * 64 + threadIdx.x;
    if (q < kNP) {
        float g = 0.0f;
#pragma unroll 16
        for (int c = 0; c < nchunk; ++c) g += part[(int64_t)c * kNP + q];
        grad[q] = g;
    } else if (q == (int)gridDim.x * 64 - 1) {
        double a = 0.0;
#pragma unroll 16
        for (int c = 0; c < nchunk; ++c) a += lpart[c];
        *loss = (float)(a / (double)batch);
    }
}

__global__ void k_mlp_adam(int64_t np, float *__restrict__ params, const float *__restrict__ grad,
                           float *__restrict__ mom, float *__restrict__ vel, float lr, float b1, float b2, float eps,
                           float c1, float c2) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= np) return;
    const float g = grad[q];
    const float mq = b1 * mom[q] + (1.0f - b1) * g;
    const float vq = b2 * vel[q] + (1.0f - b2) * g * g;
    mom[q] = mq;
    vel[q] = vq;
    params[q] -= lr * (mq / c1) / (sqrtf(vq / c2) + eps);
}

__global__ void k_mlp_sgd(int64_t np, float *__restrict__ params, const float *__restrict__ grad,
                          float *__restrict__ vel, float lr, float mu) {
    const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= np) return;
    float g = grad[q];
    if (vel) {
        g = mu * vel[q] + g;
        vel[q] = g;
    }
    params[q] -= lr * g;
}

// Statistics of log2 of the non-zero tile maxima of a panel: max, min,
// mean, standard deviation (thread-strided partial sums, then a fixed-order
// tree in LDS).
struct LogStats {
    float mx, mn, mean, sd;
};

__device__ LogStats log_stats(int64_t cnt, const float *__restrict__ v, float *red) {
    const int t = threadIdx.x;
    float mx = -1e30f, mn = 1e30f, s1 = 0.0f, s2 = 0.0f, c = 0.0f;
    for (int64_t i = t; i < cnt; i += blockDim.x) {
        const float a = v[i];
        if (a > 0.0f && a < __builtin_inff()) {
            const float l = log2f(a);
            mx = fmaxf(mx, l);
            mn = fminf(mn, l);
            s1 += l;
            s2 += l * l;
            c += 1.0f;
        }
    }
    red[t] = mx;
    red[256 + t] = mn;
    red[512 + t] = s1;
    red[768 + t] = s2;
    red[1024 + t] = c;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (t < w) {
            red[t] = fmaxf(red[t], red[t + w]);
            red[256 + t] = fminf(red[256 + t], red[256 + t + w]);
            red[512 + t] += red[512 + t + w];
            red[768 + t] += red[768 + t + w];
            red[1024 + t] += red[1024 + t + w];
        }
        __syncthreads();
    }
    LogStats r;
    const float n = red[1024];
    if (n > 0.0f) {
        r.mx = red[0];
        r.mn = red[256];
        r.mean = red[512] / n;
        r.sd = sqrtf(fmaxf(red[768] / n - r.mean * r.mean, 0.0f));
    } else {
        r.mx = r.mn = r.mean = -64.0f;
        r.sd = 0.0f;
    }
    __syncthreads();
    return r;
}

__device__ __forceinline__ float clip8(float v) {
    if (!(v == v)) return 0.0f;
    return fminf(fmaxf(v, -8.0f), 8.0f);
}

// The 16 inputs of one panel step (one workgroup of 256 threads).
__global__ void __launch_bounds__(256)
k_sched_features(int64_t nl, const float *__restrict__ lmax, int64_t nr, const float *__restrict__ rmax,
                 const float *__restrict__ Akk, int64_t lda, int64_t b, int64_t step, int64_t nb, int64_t n,
                 int prev, float *__restrict__ out) {
    __shared__ float red[5 * 256];
    const LogStats L = log_stats(nl, lmax, red);
    const LogStats R = log_stats(nr, rmax, red);
    // |u_ii| of the factored diagonal block
    const int t = threadIdx.x;
    float mx = -1e30f, mn = 1e30f;
    for (int64_t i = t; i < b; i += blockDim.x) {
        const float u = fabsf(Akk[i + i * lda]);
        const float l = (u > 0.0f && u < __builtin_inff()) ? log2f(u) : -64.0f;
        mx = fmaxf(mx, l);
        mn = fminf(mn, l);
    }
    red[t] = mx;
    red[256 + t] = mn;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (t < w) {
            red[t] = fmaxf(red[t], red[t + w]);
            red[256 + t] = fminf(red[256 + t], red[256 + t + w]);
        }
        __syncthreads();
    }
    if (t != 0) return;
    const float umx = red[0], umn = red[256];
    const int64_t rest = n - (step + 1) * b;
    float f[16];
    f[0] = L.mx / 16.0f;
    f[1] = L.mn / 16.0f;
    f[2] = L.mean / 16.0f;
    f[3] = L.sd / 8.0f;
    f[4] = R.mx / 16.0f;
    f[5] = R.mn / 16.0f;
    f[6] = R.mean / 16.0f;
    f[7] = R.sd / 8.0f;
    f[8] = umx / 16.0f;
    f[9] = umn / 16.0f;
    f[10] = (umx - umn) / 16.0f;
    f[11] = (float)step / (float)nb;
    f[12] = log2f((float)(rest > 0 ? rest : 1) / (float)n) / 8.0f;
    f[13] = (L.mx - umx) / 16.0f;
    f[14] = (R.mx - umx) / 16.0f;
    f[15] = (float)prev;
#pragma unroll
    for (int i = 0; i < 16; ++i) out[i] = clip8(f[i]);
}

}  // namespace

extern "C" {

int omx_mlp_forward_f32(int64_t batch, const float *params, const float *X, float *H1, float *H2, float *Z,
                        void *stream) {
    if (batch <= 0 || !params || !X || !H1 || !H2 || !Z) return OMX_ERR_ARG;
    hipLaunchKernelGGL(k_mlp_forward, dim3((unsigned)omx_cdiv(batch, kFS)), dim3(256), 0, omx_stream(stream),
                       batch, params, X, H1, H2, Z);
    OMX_LAUNCH_CHECK();
    return OMX_OK;
}

size_t omx_mlp_backward_workspace_bytes(int64_t batch) {
    if (batch <= 0) return 0;
    return (size_t)batch * (kD * sizeof(float) + sizeof(double));
}

int omx_mlp_backward_f32(int64_t batch, const float *params, const float *X, const float *H1, const float *H2,
                         const float *Z, const int32_t *y, const float *t, const float *m, float *grad, float *loss,
                         void *work, size_t work_bytes, void *stream) {
    if (batch <= 0 || !params || !X || !H1 || !H2 || !Z || !y || !t || !m || !grad || !loss) return OMX_ERR_ARG;
    if (!work || work_bytes < omx_mlp_backward_workspace_bytes(batch)) return OMX_ERR_WORKSPACE;
    hipStream_t st = omx_stream(stream);
    // chunks: as many as their partial sums fit the workspace, multiples of
    // 41 samples or so each; one chunk writes the results itself
    const int64_t most = std::min<int64_t>(kMaxChunks, (int64_t)(omx_mlp_backward_workspace_bytes(batch) / kChunkBytes));
    int64_t nchunk = std::max<int64_t>(1, most);
    const int64_t chunk = omx_cdiv(batch, nchunk);
    nchunk = omx_cdiv(batch, chunk);
    double *lpart = static_cast<double *>(work);
    float *part = nchunk > 1 ? reinterpret_cast<float *>(lpart + nchunk) : nullptr;
    hipLaunchKernelGGL(k_mlp_backward, dim3((unsigned)nchunk), dim3(kBT), 0, st, batch, chunk, params, X, H1, H2, Z, y,
                       t, m, grad, loss, part, lpart);
    OMX_LAUNCH_CHECK();
    if (nchunk > 1) {
        // kNP is not a multiple of 64: the last thread is free for the loss
        static_assert(kNP % 64 != 0, "a spare thread in the last workgroup");
        hipLaunchKernelGGL(k_mlp_grad_reduce, dim3((unsigned)omx_cdiv(kNP, 64)), dim3(64), 0, st, batch, (int)nchunk,
                           part, lpart, grad, loss);
        OMX_LAUNCH_CHECK();
    }
    return OMX_OK;
}

int omx_mlp_adam_f32(int64_t nparams, float *params, const float *grad, float *mom, float *vel, float lr,
                     float beta1, float beta2, float eps, int step, void *stream) {
    if (nparams <= 0 || !params || !grad || !mom || !vel || step < 1 || !(lr > 0) || !(beta1 >= 0) ||
        !(beta1 < 1) || !(beta2 >= 0) || !(beta2 < 1) || !(eps > 0))
        return OMX_ERR_ARG;
    const float c1 = 1.0f - powf(beta1, (float)step), c2 = 1.0f - powf(beta2, (float)step);
    hipLaunchKernelGGL(k_mlp_adam, dim3((unsigned)omx_cdiv(nparams, 256)), dim3(256), 0, omx_stream(stream),
                       nparams, params, grad, mom, vel, lr, beta1, beta2, eps, c1, c2);
    OMX_LAUNCH_CHECK();
    return OMX_OK;
}

int omx_mlp_sgd_f32(int64_t nparams, float *params, const float *grad, float *vel, float lr, float momentum,
                    void *stream) {
    if (nparams <= 0 || !params || !grad || !(lr > 0) || !(momentum >= 0) || !(momentum < 1) ||
        (momentum > 0 && !vel))
        return OMX_ERR_ARG;
    hipLaunchKernelGGL(k_mlp_sgd, dim3((unsigned)omx_cdiv(nparams, 256)), dim3(256), 0, omx_stream(stream),
                       nparams, params, grad, momentum > 0 ? vel : nullptr, lr, momentum);
    OMX_LAUNCH_CHECK();
    return OMX_OK;
}

int omx_sched_features_f32(int64_t ntiles_l, const float *lmax, int64_t ntiles_r, const float *rmax,
                           const float *Akk, int64_t lda, int64_t b, int64_t step, int64_t nb, int64_t n, int prev,
                           float *features, void *stream) {
    if (ntiles_l < 0 || ntiles_r < 0 || (ntiles_l > 0 && !lmax) || (ntiles_r > 0 && !rmax) || !Akk || b <= 0 ||
        lda < b || step < 0 || nb <= 0 || n <= 0 || !features)
        return OMX_ERR_ARG;
    hipLaunchKernelGGL(k_sched_features, dim3(1), dim3(256), 0, omx_stream(stream), ntiles_l, lmax, ntiles_r, rmax,
                       Akk, lda, b, step, nb, n, prev, features);
    OMX_LAUNCH_CHECK();
    return OMX_OK;
}

}  // extern "C"
