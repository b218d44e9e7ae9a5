// The two ends of a PPO update that belong to the policy, forward and gradient in one pass each.
//
// Written in torch ops the log-probability and entropy of given actions were 9 launches forward and as many back, the HL-Gauss
// critic loss 15 and 12: ~0.5 ms of host time per update for a few MB of traffic, a fifth of what an update of 1500 envs took.
#include "bsrl_common.h"

namespace {

// one thread per (env, head): d logits of glp * logp(action) + gent * entropy, with logp = log_softmax,
// d logp(a) / d x_k = [k = a] - p_k and d H / d x_k = -p_k (logp_k + H)
__global__ __launch_bounds__(256) void heads_logp_bwd_kernel(const float* __restrict__ logits, const int64_t* __restrict__ action,
                                                             const float* __restrict__ glp, const float* __restrict__ gent,
                                                             float* __restrict__ dlogits, int64_t rows, int n_heads, int K) {
    constexpr int KMAX = 8;
    const int64_t row = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (row >= rows) return;
    const int64_t env = row / n_heads;
    const float* x = logits + row * K;
    float v[KMAX], m = -INFINITY, s = 0.f, ent = 0.f;
#pragma unroll
    for (int k = 0; k < KMAX; ++k) { v[k] = k < K ? x[k] : -INFINITY; m = fmaxf(m, v[k]); }
#pragma unroll
    for (int k = 0; k < KMAX; ++k) s += k < K ? expf(v[k] - m) : 0.f;
    const float ls = logf(s), gl = glp ? glp[env] : 0.f, ge = gent ? gent[env] : 0.f;
#pragma unroll
    for (int k = 0; k < KMAX; ++k) if (k < K) { v[k] = (v[k] - m) - ls; ent -= expf(v[k]) * v[k]; }
    const int64_t act = action[row];
    const float hit = act < 0 || act >= K ? NAN : 1.f;       // an action outside its head has no log-probability
#pragma unroll
    for (int k = 0; k < KMAX; ++k)
        if (k < K) {
            const float p = expf(v[k]);
            dlogits[row * K + k] = gl * ((k == act ? 1.f : hit - 1.f) - p) - ge * p * (v[k] + ent);
        }
}

// one wave per row: target = the mass of N(v, sigma^2) in each bin (v clamped into the support, renormalised), loss = its
// cross-entropy with softmax(logits), dlogits = softmax(logits) - target
template <int PER>
__global__ __launch_bounds__(256) void hl_loss_kernel(const float* __restrict__ logits, const float* __restrict__ v_tgt,
                                                      const float* __restrict__ centers, float inv_s, float* __restrict__ loss,
                                                      float* __restrict__ dlogits, int64_t rows, int n) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const float c0 = centers[0], half = 0.5f * (centers[1] - c0);
    const float vt = v_tgt[row];                             // a NaN return stays NaN (fmin / fmax would drop it): loss and gradient show it
    const float v = vt != vt ? vt : fminf(fmaxf(vt, c0 - half), centers[n - 1] + half);
    const float* x = logits + row * n;
    float l[PER], p[PER], m = -INFINITY, tot = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int k = lane + 64 * i;
        l[i] = -INFINITY; p[i] = 0.f;
        if (k < n) {
            l[i] = x[k];
            const float hi = centers[k] + half, lo = k == 0 ? c0 - half : centers[k - 1] + half;      // edges of the bin
            p[i] = 0.5f * (1.0f + erff((hi - v) * inv_s)) - 0.5f * (1.0f + erff((lo - v) * inv_s));
        }
        m = fmaxf(m, l[i]); tot += p[i];
    }
    m = group_max<64>(m);
    tot = group_sum<64>(tot);
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i) s += lane + 64 * i < n ? expf(l[i] - m) : 0.f;
    s = group_sum<64>(s);
    const float ls = logf(s);
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int k = lane + 64 * i;
        if (k < n) {
            const float t = p[i] / tot, lp = (l[i] - m) - ls;
            acc -= t * lp;
            dlogits[row * n + k] = expf(lp) - t;
        }
    }
    acc = group_sum<64>(acc);
    if (lane == 0) loss[row] = acc;
}

}  // namespace

extern "C" int bsrl_heads_logp_bwd(const float* logits, const int64_t* action, const float* glp, const float* gent, float* dlogits,
                                   int64_t B, int64_t n_heads, int64_t K, bsrl_stream stream) {
    if (!logits || !action || !dlogits) BSRL_FAIL(BSRL_EINVAL, "bsrl_heads_logp_bwd: null pointer");
    if (B < 0 || n_heads < 1 || n_heads > 32 || K < 1 || K > 8) BSRL_FAIL(BSRL_EINVAL, "bsrl_heads_logp_bwd: need B >= 0, 1 <= n_heads <= 32, 1 <= K <= 8");
    if (B == 0) return BSRL_OK;
    const int64_t rows = B * n_heads;
    hipLaunchKernelGGL(heads_logp_bwd_kernel, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, static_cast<hipStream_t>(stream), logits, action, glp, gent,
                       dlogits, rows, (int)n_heads, (int)K);
    BSRL_CHECK_LAUNCH("bsrl_heads_logp_bwd");
    return BSRL_OK;
}

extern "C" int bsrl_hl_loss(const float* logits, const float* v_tgt, const float* centers, float sigma, float* loss, float* dlogits,
                            int64_t B, int64_t n, bsrl_stream stream) {
    if (!logits || !v_tgt || !centers || !loss || !dlogits) BSRL_FAIL(BSRL_EINVAL, "bsrl_hl_loss: null pointer");
    if (B < 0 || n < 2 || !(sigma > 0.f)) BSRL_FAIL(BSRL_EINVAL, "bsrl_hl_loss: need B >= 0, n >= 2 and sigma > 0");
    if (n > 512) return BSRL_UNSUPPORTED;
    if (B == 0) return BSRL_OK;
    const float inv_s = (float)(1.0 / ((double)sigma * 1.41421356237309504880));
    const dim3 grid((unsigned)((B + 3) / 4)), block(256);
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (n <= 128) hipLaunchKernelGGL(hl_loss_kernel<2>, grid, block, 0, st, logits, v_tgt, centers, inv_s, loss, dlogits, B, (int)n);
    else hipLaunchKernelGGL(hl_loss_kernel<8>, grid, block, 0, st, logits, v_tgt, centers, inv_s, loss, dlogits, B, (int)n);
    BSRL_CHECK_LAUNCH("bsrl_hl_loss");
    return BSRL_OK;
}
