// What follows NotePolicy's block stack - trunk, action heads, the critic's projections, the value MLP - for batches of up to 32
// envs per CU (READOUT_MOST in note_forward.hip), as two launches around the critic's attention pool instead of seventeen.
//
// Every one of those Linears is a few 100 KB of weights against B rows: 4 - 5.5 us a launch whatever B is, 70 us of a one-env
// forward's 177 and most of its host time.  Here a workgroup takes up to 16 envs - the columns of one MFMA tile - through a chain
// of Linears and LayerNorms with the activations in LDS as operand pieces; its sixteen waves deal the output tiles of a step
// between them and stream the weight rows from L2 into registers, eight 1 KB fragments ahead, across the steps' barriers.
// The actor's and the critic's chains run in workgroups of their own.  Bound: the weight stream of a CU (1.4 MB for the actor's
// chain at the recipe's widths: 22 us, 28 B/clk; 46 us from row-major weights, of whose lines a fragment takes half).  Arithmetic is the Linear and LayerNorm kernels': k ascending from zero, then the bias, the
// activation, the residual; the LayerNorm lane layout of ln_kernel.  Same bits.
// Whole forward, one env: recipe shape 180 -> 157 us, default shape 103 -> 65; 2048 envs: 463 -> 429, 175 -> 143.
#include "ln_io.h"
#include "note_readout.h"

namespace {

constexpr int NW = READOUT_WAVES, PF = 8;        // waves; weight fragments in flight per wave

template <typename DT, int LPR, int NCH>
__device__ __forceinline__ void ln_row(const uint4* in, uint4* out, u16* gout, const float* w, const float* bias, int env, int lane, int d) {
    typedef LnIO<DT> io;
    // ln_kernel's row: LPR lanes, NCH 16-byte chunks each
    if (lane >= LPR) return;
    float v[NCH][8], s = 0.f;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const int e0 = (c * LPR + lane) * 8;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[c][j] = 0.f;
        if (e0 < d) io::cvt(in[(e0 >> 3) * 16 + env], v[c]);
#pragma unroll
        for (int j = 0; j < 8; ++j) s += v[c][j];
    }
    const float inv_d = 1.0f / (float)d;
    const float mean = keep_f32(group_sum<LPR>(s) * inv_d);
    float q = 0.f;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const int e0 = (c * LPR + lane) * 8;
        if (e0 < d) {
#pragma unroll
            for (int j = 0; j < 8; ++j) v[c][j] -= mean;
            // ln_kernel's code: the first two squares as fma(t0, t0, t1 t1), the rest added in order
            if (c == 0) q = fmaf(v[0][0], v[0][0], keep_f32(v[0][1] * v[0][1]));
#pragma unroll
            for (int j = c == 0 ? 2 : 0; j < 8; ++j) q = fmaf(v[c][j], v[c][j], q);
        }
    }
    const float rstd = 1.0f / sqrtf(fmaf(group_sum<LPR>(q), inv_d, 1e-5f));
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const int e0 = (c * LPR + lane) * 8;
        if (e0 < d) {
            float o[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) o[j] = fmaf(keep_f32(v[c][j] * rstd), w[e0 + j], bias[e0 + j]);
            io::store(out, ((e0 >> 3) * 16 + env) * 8, o);
            if (gout) io::store(gout, e0, o);
        }
    }
}

template <typename DT>
__global__ __launch_bounds__(NW * 64) void note_readout_kernel(ReadoutArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint4 lds[];
    const ReadoutProg& p = a.prog[blockIdx.y];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
    const int64_t env0 = (int64_t)blockIdx.x * a.per;
    const int ne = (int)(a.B - env0 < a.per ? a.B - env0 : a.per);
    uint4 buf[PF];
    // A wave's fragments of a step are one contiguous stream.  Each slot of the loop below issues one load, with no branch around
    // it, so that the wait for a fragment leaves the younger ones in flight; the last round of a step loads the first of the
    // next Linear, the one before it may run past the wave's stream.
    auto stream = [&](int i) __attribute__((always_inline)) {
        while (i < p.n && p.step[i].kind != READOUT_LINEAR) ++i;
        if (i == p.n) return reinterpret_cast<const uint4*>(p.step[0].kind == READOUT_LINEAR ? p.step[0].w : p.step[1].w);     // read, not used
        const int nt = (p.step[i].M + 15) / 16, before = wave * (nt / NW) + (wave < nt % NW ? wave : nt % NW);
        return reinterpret_cast<const uint4*>(p.step[i].w) + (int64_t)before * (p.step[i].K / 32) * 64;
    };
    const uint4* next = stream(0);
#pragma unroll
    for (int j = 0; j < PF; ++j) buf[j] = next[j * 64 + lane];
    next += PF * 64;
    float* const ldsf = reinterpret_cast<float*>(lds);
    for (int i = 0; i < p.n; ++i) {          // biases, LayerNorm scales and shifts, bin centres
        const ReadoutStep& s = p.step[i];
        const int n = s.kind == READOUT_LINEAR ? s.M : s.K;
        for (int k = tid; k < n; k += NW * 64) {
            ldsf[s.vec + k] = s.bias ? s.bias[k] : 0.f;
            if (s.kind == READOUT_LN) ldsf[s.vec + n + k] = s.bias2[k];
        }
    }
    for (int i = 0; i < p.n_in; ++i) {
        const int pieces = p.in[i].K / 8;
        for (int k = tid; k < ne * pieces; k += NW * 64) {
            const int e = k / pieces, c = k - e * pieces;
            lds[p.in[i].at + c * 16 + e] = *reinterpret_cast<const uint4*>(p.in[i].src + (env0 + e) * p.in[i].ld + c * 8);
        }
    }
    __syncthreads();
    for (int i = 0; i < p.n; ++i) {
        const ReadoutStep& s = p.step[i];
        const uint4* in = lds + s.in;
        if (s.kind == READOUT_LINEAR) {
            const int nk = s.K / 32, total = ((s.M + 15) / 16 - wave + NW - 1) / NW * nk;
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
            int tile = wave, kc = 0, rk = 0, f0 = 0;
            do {
                if (f0 + PF >= total) next = stream(i + 1);
                uint4 b[PF];
#pragma unroll
                for (int j = 0; j < PF; j += 2) {
                    b[j] = in[(rk * 4 + g) * 16 + r16]; b[j + 1] = in[(rk * 4 + 4 + g) * 16 + r16];
                    rk = rk + 2 == nk ? 0 : rk + 2;
                }
#pragma unroll
                for (int j = 0; j < PF; ++j) {
                    acc = DT::mfma32(__builtin_bit_cast(s16x8, buf[j]), __builtin_bit_cast(s16x8, b[j]), acc);      // past the last tile: not used
                    buf[j] = next[j * 64 + lane];
                    if (j % 2 == 0 || (kc += 2) < nk || f0 + j >= total) continue;
                    // a tile is done: lane holds outputs col .. col + 3 of env r16
                    const int col = 16 * tile + 4 * g, at = ((col >> 3) * 16 + r16) * 2 + ((col >> 2) & 1);      // 8-byte half piece
                    float o[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        o[e] = acc[e] + ldsf[s.vec + col + e];               // room for whole tiles
                        if (!s.f32) o[e] = s.relu ? apply_act16<BSRL_ACT_RELU>(o[e]) : apply_act16<BSRL_ACT_NONE>(o[e]);
                        o[e] = keep_f32(o[e]);
                    }
                    if (s.res >= 0 && col < s.M) {
                        const uint2 r = reinterpret_cast<const uint2*>(lds + s.res)[at];
                        o[0] += DT::to_f((u16)(r.x & 0xffff)); o[1] += DT::to_f((u16)(r.x >> 16));
                        o[2] += DT::to_f((u16)(r.y & 0xffff)); o[3] += DT::to_f((u16)(r.y >> 16));
                    }
                    if (s.f32) {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (col + e < s.M) {
                                if (s.out >= 0) ldsf[s.out * 4 + r16 * ((s.M + 3) & ~3) + col + e] = o[e];
                                else if (r16 < ne) static_cast<float*>(s.gout)[(env0 + r16) * s.gld + col + e] = o[e];
                            }
                    } else if (col < s.M) {
                        uint2 ov;
                        ov.x = DT::pack2(o[0], o[1]); ov.y = DT::pack2(o[2], o[3]);
                        if (s.out >= 0) reinterpret_cast<uint2*>(lds + s.out)[at] = ov;
                        if (s.gout && r16 < ne) *reinterpret_cast<uint2*>(static_cast<u16*>(s.gout) + (env0 + r16) * s.gld + col) = ov;
                    }
                    acc = (f32x4){0.f, 0.f, 0.f, 0.f};
                    kc = 0; tile += NW;
                }
                next += PF * 64;
                f0 += PF;
            } while (f0 < total);
        } else if (s.kind == READOUT_LN) {
            if (wave < ne) {
                u16* go = s.gout ? static_cast<u16*>(s.gout) + (env0 + wave) * s.gld : nullptr;
                uint4* out = lds + s.out;
                if (s.K <= 128) ln_row<DT, 16, 1>(in, out, go, ldsf + s.vec, ldsf + s.vec + s.K, wave, lane, s.K);
                else if (s.K <= 256 && s.K % 128 == 0) ln_row<DT, 16, 2>(in, out, go, ldsf + s.vec, ldsf + s.vec + s.K, wave, lane, s.K);
                else if (s.K <= 256) ln_row<DT, 32, 1>(in, out, go, ldsf + s.vec, ldsf + s.vec + s.K, wave, lane, s.K);
                else ln_row<DT, 16, 3>(in, out, go, ldsf + s.vec, ldsf + s.vec + s.K, wave, lane, s.K);
            }
        } else if (wave < ne) {              // softmax(logits) . centers, as softmax_expect_kernel
            const float* lr = reinterpret_cast<const float*>(in) + wave * ((s.K + 3) & ~3);
            float m = -INFINITY;
            for (int k = lane; k < s.K; k += 64) m = fmaxf(m, lr[k]);
            m = group_max<64>(m);
            float se = 0.f, sc = 0.f;
            for (int k = lane; k < s.K; k += 64) {
                const float e = expf(lr[k] - m);
                se += e; sc = fmaf(e, ldsf[s.vec + k], sc);
            }
            se = group_sum<64>(se); sc = group_sum<64>(sc);
            if (lane == 0) static_cast<float*>(s.gout)[env0 + wave] = sc / se;
        }
        __syncthreads();
    }
}

template <typename DT>
int launch(const ReadoutArgs& a, int n_prog, size_t bytes, hipStream_t st) {
    auto kern = note_readout_kernel<DT>;
    static const bool ready = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) == hipSuccess;
    if (!ready) { (void)hipGetLastError(); return BSRL_UNSUPPORTED; }
    hipLaunchKernelGGL(kern, dim3((unsigned)((a.B + a.per - 1) / a.per), (unsigned)n_prog), dim3(NW * 64), bytes, st, a);
    BSRL_CHECK_LAUNCH("bsrl_note_readout");
    return BSRL_OK;
}

struct FragArgs { ReadoutMat m[READOUT_MATS]; int first[READOUT_MATS]; int n; };

__global__ __launch_bounds__(256) void note_readout_frags_kernel(FragArgs a) {
    int j = 0;
    while (j + 1 < a.n && (int)blockIdx.x >= a.first[j + 1]) ++j;
    const ReadoutMat& m = a.m[j];
    const int nk = m.K / 32, nt = (m.M + 15) / 16, lane = threadIdx.x & 63, f = (blockIdx.x - a.first[j]) * 4 + (threadIdx.x >> 6);
    if (f >= nt * nk) return;
    const int tile = f / nk, k = f - tile * nk, wave = tile % NW, row = 16 * tile + (lane & 15);
    const int before = wave * (nt / NW) + (wave < nt % NW ? wave : nt % NW);
    uint4 v = make_uint4(0, 0, 0, 0);
    if (row < m.M) v = *reinterpret_cast<const uint4*>(m.src + (int64_t)row * m.K + 32 * k + 8 * (lane >> 4));
    reinterpret_cast<uint4*>(m.dst)[((int64_t)(before + tile / NW) * nk + k) * 64 + lane] = v;
}

}  // namespace

int bsrl_note_readout_frags(const ReadoutMat* m, int n, hipStream_t st) {
    FragArgs a = {};
    a.n = n;
    int wgs = 0;
    for (int i = 0; i < n; ++i) {
        a.m[i] = m[i]; a.first[i] = wgs;
        wgs += ((m[i].M + 15) / 16 * (m[i].K / 32) + 3) / 4;
    }
    hipLaunchKernelGGL(note_readout_frags_kernel, dim3((unsigned)wgs), dim3(256), 0, st, a);
    BSRL_CHECK_LAUNCH("bsrl_note_readout_frags");
    return BSRL_OK;
}

size_t bsrl_note_readout_lds(ReadoutArgs& a, int n_prog, size_t bytes) {
    size_t most = bytes;
    for (int i = 0; i < n_prog; ++i) {
        size_t at = bytes / 4;
        for (int j = 0; j < a.prog[i].n; ++j) {
            ReadoutStep& s = a.prog[i].step[j];
            s.vec = (int)at;
            at += s.kind == READOUT_LINEAR ? (s.M + 15) / 16 * 16 : s.kind == READOUT_LN ? 2 * s.K : s.K;
        }
        if (at * 4 > most) most = at * 4;
    }
    return most;
}

int bsrl_note_readout(ReadoutArgs a, int n_prog, size_t lds_bytes, int dtype, hipStream_t st) {
    // an env per workgroup while the CUs last: the 16 columns of a tile cost what one does
    const int64_t wgs = (int64_t)bsrl_cus() / n_prog;
    a.per = (int)((a.B + wgs - 1) / wgs);
    if (a.per > 16) a.per = 16;
    return dtype == BSRL_F16 ? launch<F16>(a, n_prog, lds_bytes, st) : launch<BF16>(a, n_prog, lds_bytes, st);
}
