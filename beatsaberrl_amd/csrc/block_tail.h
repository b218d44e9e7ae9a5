// A transformer block from the attention output on, as ONE kernel on plain rows (d = 192 / 256 / 384):
//   x1 = x + att Wo^T + bo,  h2 = LN(x1; ln2),  xo = x1 + act(h2 W0^T + b0) W2^T + b2,  ho = LN(xo; ln),  qo = ho Wn^T + bn
// (output projection + residual, LayerNorm, FFN + residual, the next block's LayerNorm and its packed projection; the last
// two are optional).  x1, h2 and the hidden never leave the registers.  The LEAD form is the last phase alone: qo = LN(x) Wn^T
// + bn for the first block.  Rounding points are those of the separate launches: x1, h2, the hidden, xo, ho, qo rounded once
// each, LayerNorm statistics on the rounded row, fp32 accumulation.
//
// Rows are whatever the caller packs: with `extra` the row count is rows + *extra, read from device memory, so that a batch
// whose tokens were compacted on the device (padding tokens dropped) needs no host round trip; the launch is sized for the
// bound the host knows and workgroups past the end leave at once.
//
// Mapping.  A wave owns RT 16-row MFMA tiles and carries their fp32 accumulator (RT d/4 registers) and operand fragments
// (RT d/8) in registers; a workgroup is 4 waves, one per SIMD with the whole register file (512), one workgroup per CU.
// Every weight fragment read from LDS feeds RT MFMAs: 2 / 3 / 4 at d = 384 / 256 / 192 fill the register file, and the 128 B/clk
// of LDS serve 4 waves x 1 KB per RT x 16 cycles (128 B/clk at RT = 2, 64 at RT = 4).  Weights stream L2 -> LDS in stages of
// d/16 fragments through the direct-to-LDS ring (block_stage.h), entered in pairs; fragment reads run three ahead of the
// MFMAs through four rotating register quads, across stage boundaries too.
// The fragments of an up-projection stage alternate between its two column tiles, so that 2 RT independent MFMAs lie between
// two that meet in one accumulator.
// Feature order ("wide"): the weight rows of an accumulator-tile PAIR are ordered so that a lane's four features of tile 2p
// and its four of tile 2p + 1 are EIGHT CONSECUTIVE features, 32 p + 8 g + 0..7 (A row m of tile i is feature
// 32 (i / 2) + 8 (m / 4) + 4 (i % 2) + m % 4): rows come in and leave in 16-byte pieces, and both an input row's and a
// LayerNorm output's operand fragment hold their k values in natural order.
// The residual stream between blocks is 16-bit, or fp32 (XI32: x comes in as fp32, XO32: xo leaves as fp32; then x1 is not
// rounded either and both LayerNorms see the unrounded rows) where the caller's other route keeps it in fp32 registers.
// Small row counts take half the row tiles per wave: twice the workgroups, each with half the MFMAs per stage.
#pragma once
#include "block_stage.h"

namespace {

struct TailArgs {
    const void* frags; const float* vec;         // stages: d/32 projection | 2 F/32 FFN | nq next;  b0 (F) | b2 (d) | bo (d) | bn (32 nq)
    const void* x; const u16* att; void* xo; u16* ho; u16* qo;
    const float* ln2_w; const float* ln2_b; float eps2;
    const float* ln_w; const float* ln_b; float eps;
    int64_t rows, ho_rows; const int32_t* extra;
    int F, nq, total_stages;
};

template <int D> struct TailGeo {
    // row tiles per wave: accumulator, operand fragments, two chunks of hidden values on their way and the fragment
    // registers fill the 512 registers at 2 / 3 / 4 tiles (four tiles at d = 256 left no room for the second chunk)
    static constexpr int RT = D == 384 ? 2 : D == 256 ? 3 : 4;
    static constexpr int SLOTS = D == 384 ? 5 : D == 256 ? 8 : 10;       // ring slots of d/16 KB
};
template <int D, int XS = 0> struct TailRing : StageRing<Geo<D>::SF, TailGeo<D>::SLOTS + XS, 4> {};

template <typename DT, int D, int RT, int ACT, bool LN, int XS, bool LEAD, bool XI32, bool XO32>
__global__ __launch_bounds__(256, 1) void block_tail_kernel(TailArgs a) {
    typedef Geo<D> G;
    typedef TailRing<D, XS> R;
    static_assert(!LEAD || LN, "the lead form ends in the LayerNorm and its projection");
    constexpr int NW = 4, NT = G::NT, KC = G::KC, SF = G::SF, NBUF = 4, RH = XI32 ? 1 : RT % 2 == 0 ? 2 : RT < 3 ? RT : 3;
    constexpr bool F32S = XI32 || XO32;
    static_assert(SF % NBUF == 0 && KC % 2 == 0 && RT % RH == 0, "rotating fragment registers; stage parities; loads in row-tile pairs");
    const int64_t rows = a.rows + (a.extra ? (int64_t)*a.extra : 0);
    const int64_t ntiles = (rows + NW * RT * 16 - 1) / (NW * RT * 16);
    if ((int64_t)blockIdx.x >= ntiles) return;
    extern __shared__ float4 tvl4[];          // b0 (F) | b2 | ln_w | ln_b | bo | ln2_w | ln2_b (d each) | bn (32 nq), then the ring (1 KB aligned)
    float* vlds = reinterpret_cast<float*>(tvl4);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int nvec = a.F + 6 * D + 32 * a.nq;
    const uint4* ring = reinterpret_cast<const uint4*>(tvl4) + ((nvec / 4 + 63) & ~63);
    const float* B1 = vlds; const float* B2 = vlds + a.F; const float* LNG = B2 + D; const float* LNB = LNG + D;
    const float* BO = LNB + D; const float* LN2G = BO + D; const float* LN2B = LN2G + D; const float* BN = LN2B + D;
    auto foff = [&](int nt) __attribute__((always_inline)) { return 32 * (nt >> 1) + 8 * g + 4 * (nt & 1); };

    // the lane for an address that is needed once a tile: computed where it is used, not kept across the tile (kept, addresses and row
    // conditions were 26 spilled registers at d = 256 and 12 at d = 384, each reload behind the stores in flight: four blocks at
    // d = 256, 541k rows, 4.55 -> 4.35 ms, six at d = 384, 1.2M rows, 31.3 -> 31.1)
    auto lane_here = [&] __attribute__((always_inline)) { int l = lane; asm volatile("" : "+v"(l)); return l; };
    R pipe;
    {   // SLOTS - 2 stages in flight (the host checks that the image is longer), then the vectors
        pipe.start(ring, a.frags, a.total_stages, wave, lane);
        for (int i = tid; i < a.F + D; i += NW * 64) vlds[i] = a.vec[i];
        for (int i = tid; i < D; i += NW * 64) {
            if (LN) { vlds[a.F + D + i] = a.ln_w[i]; vlds[a.F + 2 * D + i] = a.ln_b[i]; }
            vlds[a.F + 3 * D + i] = a.vec[a.F + D + i];
            if (!LEAD) { vlds[a.F + 4 * D + i] = a.ln2_w[i]; vlds[a.F + 5 * D + i] = a.ln2_b[i]; }
        }
        for (int i = tid; i < 32 * a.nq; i += NW * 64) vlds[a.F + 6 * D + i] = a.vec[a.F + 2 * D + i];
        blk_barrier();
    }
    const int nch = a.F / 32;

    for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        // a wave's rows from a scalar base, so that a lane's share of an address is one 32-bit offset
        const int64_t row0 = (tile * NW + wave) * (RT * 16), base0 = row0 < rows ? row0 : rows - 1;
        const int left = rows - row0 > RT * 16 ? RT * 16 : rows > row0 ? (int)(rows - row0) : 0, last = left > 0 ? left - 1 : 0;
        f32x4 x[RT][NT];
        BFrag8 hf[RT][KC];
        // The tile's loads: two row tiles of x and every operand row at once (the compiler counts its own loads, not the
        // ring's transfers, which only make its waits stricter), the other pairs of x behind the first pair's conversion
        if constexpr (!LEAD)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const int l = lane_here(), row = 16 * rt + (l & 15) < last ? 16 * rt + (l & 15) : last;
            const u16* hr = a.att + base0 * D + (uint32_t)(row * D + 8 * (l >> 4));
#pragma unroll
            for (int c = 0; c < KC; ++c) hf[rt][c].u = *reinterpret_cast<const uint4*>(hr + 32 * c);
        }
#pragma unroll
        for (int half = 0; half < RT / RH; ++half) {
            uint4 rx[RH][XI32 ? NT : NT / 2];
#pragma unroll
            for (int rr = 0; rr < RH; ++rr) {
                const int l = lane_here(), rl = 16 * (half * RH + rr) + (l & 15), row = rl < last ? rl : last;
                if constexpr (XI32) {
                    const float* xr = static_cast<const float*>(a.x) + base0 * D + (uint32_t)(row * D + 8 * (l >> 4));
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) rx[rr][nt] = *reinterpret_cast<const uint4*>(xr + 32 * (nt >> 1) + 4 * (nt & 1));
                } else {
                    const u16* xr = static_cast<const u16*>(a.x) + base0 * D + (uint32_t)(row * D + 8 * (l >> 4));
#pragma unroll
                    for (int p = 0; p < NT / 2; ++p) rx[rr][p] = *reinterpret_cast<const uint4*>(xr + 32 * p);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int rr = 0; rr < RH; ++rr)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    f32x4& xx = x[half * RH + rr][nt];
                    float4 b = make_float4(0.f, 0.f, 0.f, 0.f);
                    if constexpr (!LEAD) b = *reinterpret_cast<const float4*>(BO + foff(nt));
                    if constexpr (XI32) {
                        const f32x4 r = __builtin_bit_cast(f32x4, rx[rr][nt]);
                        xx[0] = r[0] + b.x; xx[1] = r[1] + b.y; xx[2] = r[2] + b.z; xx[3] = r[3] + b.w;
                    } else {
                    const uint32_t lo = (nt & 1) ? rx[rr][nt >> 1].z : rx[rr][nt >> 1].x, hi = (nt & 1) ? rx[rr][nt >> 1].w : rx[rr][nt >> 1].y;
                    xx[0] = DT::to_f((u16)(lo & 0xffff)) + b.x; xx[1] = DT::to_f((u16)(lo >> 16)) + b.y;
                    xx[2] = DT::to_f((u16)(hi & 0xffff)) + b.z; xx[3] = DT::to_f((u16)(hi >> 16)) + b.w;
                    }
                    asm("" : "+a"(xx));        // the accumulator lives in accumulation registers from here on
                    if ((nt & 3) == 3) __builtin_amdgcn_sched_barrier(0);
                }
        }
        s16x8 wr[NBUF];
        // one stage: before the MFMAs of fragment i are issued, fragment i + NBUF - 1 is requested (behind the next stage's
        // admission when it opens a stage).  next: 0 = nothing follows in this tile, 1 = an odd stage (entered without a
        // barrier), 2 = an even one (the pair admission, which reuses the slot of the stage being left: every wave's reads of
        // it must have returned before the barrier).  mm(i, rt, fragment): one MFMA; fill(slot): the vector work that goes
        // behind it, slot = i RT + rt.  The order is pinned: an MFMA occupies the matrix pipe for 16 cycles and its wave for
        // four, so two or three vector instructions behind each one are free, and the same instructions in a block of their
        // own cost their full issue time (measured on one wave per SIMD: 18 cycles per MFMA alone, 19.5 with two FMAs behind
        // it, 28 with four; an FMA alone 5.5, exp2 11.5).  At d = 256: 1.25 -> 1.18 ms on 541k rows; a stage of the FFN then takes
        // 0.63 us (ReLU), i.e. the matrix rate that a large product sustains on this card (1.25 PFLOP/s): what is left of the
        // kernel's distance to it are the loads, LayerNorms and stores between the stages
        auto stage = [&](int next, auto&& mm, auto&& fill) __attribute__((always_inline)) {
            static_for<0, SF>([&](auto i_) __attribute__((always_inline)) {
                constexpr int i = decltype(i_)::value, n = i + NBUF - 1;
                if constexpr (n < SF) wr[n % NBUF] = pipe.frag(n, lane);
                else if (next) {
                    if constexpr (n == SF) {
                        if (next == 2) { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); pipe.template admit<0>(); }
                        else pipe.template admit<1>();
                    }
                    wr[n % NBUF] = pipe.frag(n - SF, lane);
                }
                __builtin_amdgcn_sched_barrier(0);
                static_for<0, RT>([&](auto rt_) __attribute__((always_inline)) {
                    constexpr int rt = decltype(rt_)::value;
                    mm(i_, rt_, wr[i % NBUF]);
                    __builtin_amdgcn_sched_barrier(0);
                    fill(std::integral_constant<int, i * RT + rt>{});
                    __builtin_amdgcn_sched_barrier(0);
                });
            });
        };
        auto idle = [](auto) __attribute__((always_inline)) {};
        typedef f32x4 Acc[2][RT];                            // [column tile of the stage][row tile]
        Acc acc0, acc1;
        f32x4 bias[2];
        // wide: the stage's 32 columns in the paired order (a lane's four of tile 0 and four of tile 1 adjacent)
        auto load_bias = [&](const float* from, int ch, bool wide) __attribute__((always_inline)) {
#pragma unroll
            for (int ntl = 0; ntl < 2; ++ntl) bias[ntl] = *reinterpret_cast<const f32x4*>(from + 32 * ch + (wide ? 8 * g + 4 * ntl : 16 * ntl + 4 * g));
        };
        // an up-projection stage's MFMA; the first one of an accumulator takes the bias as its addend
        auto up_into = [&](Acc& acc) __attribute__((always_inline)) {
            return [&](auto i_, auto rt_, const s16x8& wf) __attribute__((always_inline)) {
                constexpr int ntl = decltype(i_)::value % 2, c = decltype(i_)::value / 2, rt = decltype(rt_)::value;
                acc[ntl][rt] = DT::mfma32(wf, hf[rt][c].v, c == 0 ? bias[ntl] : acc[ntl][rt]);
            };
        };
        pipe.template admit<0>();
#pragma unroll
        for (int f = 0; f < NBUF - 1; ++f) wr[f] = pipe.frag(f, lane);
        if constexpr (!LEAD) {
            // KC projection stages (KC is even, so W1(0) is an even stage): stage c adds Wo[:, 32 c .. 32 c + 31] times the
            // attention output's chunk c into every feature tile
            static_for<0, KC>([&](auto c_) __attribute__((always_inline)) {
                constexpr int c = decltype(c_)::value;
                stage((c & 1) ? 2 : 1, [&](auto i_, auto rt_, const s16x8& wo) __attribute__((always_inline)) {
                    constexpr int i = decltype(i_)::value, rt = decltype(rt_)::value;
                    x[rt][i] = DT::mfma32(wo, hf[rt][c].v, x[rt][i]);
                }, idle);
            });
            // W1(0) is admitted and its first fragments requested.  x1 rounded as the stream stores it, LayerNorm on the
            // rounded row, h2 rounded into the operand fragments, and the FFN's accumulator x1 + b2
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                float s1 = 0.f, q1 = 0.f;
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    f32x4 r = x[rt][nt];
                    if constexpr (!F32S) {
                        const uint32_t lo = bpack2<DT>(r[0], r[1]), hi = bpack2<DT>(r[2], r[3]);
                        r[0] = DT::to_f((u16)(lo & 0xffff)); r[1] = DT::to_f((u16)(lo >> 16));
                        r[2] = DT::to_f((u16)(hi & 0xffff)); r[3] = DT::to_f((u16)(hi >> 16));
                    }
#pragma unroll
                    for (int i = 0; i < 4; ++i) { s1 += r[i]; q1 = fmaf(r[i], r[i], q1); }
                    if constexpr (!F32S) { asm("" : "+a"(r)); x[rt][nt] = r; }
                    if ((nt & 3) == 3) __builtin_amdgcn_sched_barrier(0);      // keeps the accumulator's trips through the vector registers short
                }
                rows_reduce2(s1, q1, OpAdd());
                const float mean = s1 * (1.0f / D);
                const float rstd = rsqrtf(fmaxf(fmaf(-mean, mean, q1 * (1.0f / D)), 0.f) + a.eps2);
                const float shift = -mean * rstd;
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    const float4 gm = *reinterpret_cast<const float4*>(LN2G + foff(nt));
                    const float4 bt = *reinterpret_cast<const float4*>(LN2B + foff(nt));
                    const float4 b2 = *reinterpret_cast<const float4*>(B2 + foff(nt));
                    f32x4 r = x[rt][nt];
                    uint2 v;
                    v.x = bpack2<DT>(fmaf(fmaf(r[0], rstd, shift), gm.x, bt.x), fmaf(fmaf(r[1], rstd, shift), gm.y, bt.y));
                    v.y = bpack2<DT>(fmaf(fmaf(r[2], rstd, shift), gm.z, bt.z), fmaf(fmaf(r[3], rstd, shift), gm.w, bt.w));
                    hf[rt][nt >> 1].h[nt & 1] = v;
                    r[0] += b2.x; r[1] += b2.y; r[2] += b2.z; r[3] += b2.w;
                    asm("" : "+a"(r));
                    x[rt][nt] = r;
                    if ((nt & 1) == 1) __builtin_amdgcn_sched_barrier(0);      // (the scheduler would hoist every vector read above the first use)
                }
            }
            // The hidden chunks: stage parities W1(0) even, then {W1(ch + 1) odd, W2(ch) even} ..., W2(last) odd.  The activation
            // of chunk ch runs behind the MFMAs of W2(ch - 1) and W1(ch + 1) - two values at a time, one step of their chain
            // per slot -, so two chunks' accumulators and hidden fragments alternate
            typedef BFrag8 Hid[RT];
            Hid hid0, hid1;
            constexpr int STEPS = ACT == BSRL_ACT_GELU ? 10 : 2, TOT = 4 * RT * STEPS, NH = TOT / 2;
            float av[2], aw[2], ax[2];                      // the pair's chain
            auto act_step = [&](auto k_, Acc& acc, Hid& hid) __attribute__((always_inline)) {
                constexpr int k = decltype(k_)::value, pair = k / STEPS, step = k % STEPS;
                constexpr int ntl = (pair >> 1) & 1, rt = pair >> 2, e = 2 * (pair & 1);
                f32x4& a4 = acc[ntl][rt];
                if constexpr (ACT == BSRL_ACT_GELU) {       // apply_act16, one operation at a time
                    constexpr float L2E = 1.44269504088896340736f;
                    constexpr float C0 = -1.59501576f * L2E, C1 = -7.40113019e-02f * L2E, C2 = 7.03035067e-04f * L2E;
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        if constexpr (step == 0) av[u] = __builtin_amdgcn_fmed3f(a4[e + u], -9.0f, 9.0f);
                        if constexpr (step == 1) ax[u] = av[u] * av[u];
                        if constexpr (step == 2) aw[u] = fmaf(C2, ax[u], C1);
                        if constexpr (step == 3) aw[u] = fmaf(aw[u], ax[u], C0);
                        if constexpr (step == 4) aw[u] = av[u] * aw[u];
                        if constexpr (step == 5) aw[u] = __builtin_amdgcn_exp2f(aw[u]);
                        if constexpr (step == 6) aw[u] = aw[u] + 1.0f;
                        if constexpr (step == 7) aw[u] = __builtin_amdgcn_rcpf(aw[u]);
                        if constexpr (step == 8) aw[u] = keep_f32(a4[e + u] * aw[u]);
                    }
                } else if constexpr (step == 0) { aw[0] = relu1(a4[e]); aw[1] = relu1(a4[e + 1]); }
                if constexpr (step == STEPS - 1) hid[rt].w[ntl * 2 + (pair & 1)] = bpack2<DT>(aw[0], aw[1]);
            };
            // the steps [LO, HI) dealt over the NS slots of a stage
            auto act_slots = [&](auto lo_, auto hi_, Acc& acc, Hid& hid) __attribute__((always_inline)) {
                return [&](auto s_) __attribute__((always_inline)) {
                    constexpr int lo = decltype(lo_)::value, n = decltype(hi_)::value - lo, NS = SF * RT, s = decltype(s_)::value;
                    static_for<lo + s * n / NS, lo + (s + 1) * n / NS>([&](auto k_) __attribute__((always_inline)) { act_step(k_, acc, hid); });
                };
            };
            typedef std::integral_constant<int, 0> K0; typedef std::integral_constant<int, NH> KH; typedef std::integral_constant<int, TOT> KT;
            auto down = [&](Hid& hid) __attribute__((always_inline)) {
                return [&](auto i_, auto rt_, const s16x8& w2) __attribute__((always_inline)) {
                    constexpr int i = decltype(i_)::value, rt = decltype(rt_)::value;      // feature tile i
                    x[rt][i] = DT::mfma32(w2, hid[rt].v, x[rt][i]);
                };
            };
            load_bias(B1, 0, false);
            stage(1, up_into(acc0), idle);
            load_bias(B1, 1, false);
            static_for<0, NH>([&](auto k_) __attribute__((always_inline)) { act_step(k_, acc0, hid0); });
            auto half = [&](int ch, Acc& ca, Hid& ha, Acc& na, Hid& hb) __attribute__((always_inline)) {
                stage(2, up_into(na), act_slots(KH{}, KT{}, ca, ha));             // W1(ch + 1); W2(ch) is an even stage
                if (ch + 2 < nch) load_bias(B1, ch + 2, false);
                stage(1, down(ha), act_slots(K0{}, KH{}, na, hb));                // W2(ch); an odd stage follows
            };
            // two chunks a round: they alternate by name, nothing moves (with one chunk a round, whose accumulators and hidden then took
            // the other's place, 12 RT moves stood between two chunks: 4 blocks at d = 256, 541k rows, 4.91 -> 4.58 ms; at d = 384 1 %)
            int ch = 0;
            for (; ch + 2 < nch; ch += 2) { half(ch, acc0, hid0, acc1, hid1); half(ch + 1, acc1, hid1, acc0, hid0); }
            if (ch + 1 < nch) {
                half(ch, acc0, hid0, acc1, hid1);
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) { acc0[0][rt] = acc1[0][rt]; acc0[1][rt] = acc1[1][rt]; hid0[rt] = hid1[rt]; }
            }
            static_for<NH, TOT>([&](auto k_) __attribute__((always_inline)) { act_step(k_, acc0, hid0); });
            stage(a.nq > 0 ? 2 : 0, down(hid0), idle);                            // W2(last) ends the tile or is followed by an even stage
        }
        // round, store, LayerNorm on the rounded row, its output as operand fragments
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const int l = lane_here(), row = 16 * rt + (l & 15);
            const uint32_t at = (uint32_t)((l & 15) * D + 8 * (l >> 4));
            const int64_t first = (row0 + 16 * rt) * D;
            float s = 0.f, q = 0.f;
            uint2 vprev = make_uint2(0, 0);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                f32x4 r = x[rt][nt];
                if constexpr (XO32) {
                    if (row < left) *reinterpret_cast<f32x4*>(static_cast<float*>(a.xo) + first + at + 32 * (nt >> 1) + 4 * (nt & 1)) = r;
                } else {
                    uint2 v;
                    v.x = bpack2<DT>(r[0], r[1]); v.y = bpack2<DT>(r[2], r[3]);
                    if constexpr (!LEAD) {
                        if (nt & 1) { if (row < left) *reinterpret_cast<uint4*>(static_cast<u16*>(a.xo) + first + at + 32 * (nt >> 1)) = make_uint4(vprev.x, vprev.y, v.x, v.y); }
                        else vprev = v;
                    }
                    r[0] = DT::to_f((u16)(v.x & 0xffff)); r[1] = DT::to_f((u16)(v.x >> 16));
                    r[2] = DT::to_f((u16)(v.y & 0xffff)); r[3] = DT::to_f((u16)(v.y >> 16));
                }
                if constexpr (LN) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) { s += r[i]; q = fmaf(r[i], r[i], q); }
                    x[rt][nt] = r;
                }
            }
            if constexpr (LN) {
                rows_reduce2(s, q, OpAdd());
                // one pass: var = E[x^2] - mean^2 clamped at 0
                const float mean = s * (1.0f / D);
                const float rstd = rsqrtf(fmaxf(fmaf(-mean, mean, q * (1.0f / D)), 0.f) + a.eps);
                const float shift = -mean * rstd;
                const bool keep = a.ho && row < left && row0 + row < a.ho_rows;
                uint2 hprev = make_uint2(0, 0);
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    const float4 gm = *reinterpret_cast<const float4*>(LNG + foff(nt));
                    const float4 bt = *reinterpret_cast<const float4*>(LNB + foff(nt));
                    uint2 v;
                    v.x = bpack2<DT>(fmaf(fmaf(x[rt][nt][0], rstd, shift), gm.x, bt.x), fmaf(fmaf(x[rt][nt][1], rstd, shift), gm.y, bt.y));
                    v.y = bpack2<DT>(fmaf(fmaf(x[rt][nt][2], rstd, shift), gm.z, bt.z), fmaf(fmaf(x[rt][nt][3], rstd, shift), gm.w, bt.w));
                    if (nt & 1) { if (keep) *reinterpret_cast<uint4*>(a.ho + first + at + 32 * (nt >> 1)) = make_uint4(hprev.x, hprev.y, v.x, v.y); }
                    else hprev = v;
                    hf[rt][nt >> 1].h[nt & 1] = v;
                }
            }
        }
        if (LN && a.nq > 0) {
            // qo = ho Wn^T + bn: nq stages of 32 columns in the up-projection's form (the first is admitted and its first
            // fragments are in flight).  A stage's columns are packed and stored behind the MFMAs of the next one, whose
            // successor's bias is read behind them too (together: d = 256 as above 4.58 -> 4.55 ms, six at d = 384 31.65 -> 31.28; the q|k|v launch of the first
            // block is bound by its MFMAs, loads and LayerNorm: without its stores 16 % faster, without the weight stream 16 %)
            const int ldq = 32 * a.nq;
            const int ql = lane_here();
            const uint32_t qat = (uint32_t)((ql & 15) * ldq + 8 * (ql >> 4));
            uint4 qv;
            auto q_step = [&](auto k_, int sq, Acc& acc) __attribute__((always_inline)) {      // three steps per row tile
                constexpr int rt = decltype(k_)::value / 3, step = decltype(k_)::value % 3;
                // the stage's columns in the paired order: 16 bytes per lane
                if constexpr (step == 0) { qv.x = bpack2<DT>(acc[0][rt][0], acc[0][rt][1]); qv.y = bpack2<DT>(acc[0][rt][2], acc[0][rt][3]); }
                if constexpr (step == 1) { qv.z = bpack2<DT>(acc[1][rt][0], acc[1][rt][1]); qv.w = bpack2<DT>(acc[1][rt][2], acc[1][rt][3]); }
                if constexpr (step == 2) { if (16 * rt + (ql & 15) < left) *reinterpret_cast<uint4*>(a.qo + (row0 + 16 * rt) * ldq + 32 * sq + qat) = qv; }
            };
            auto q_slots = [&](int sq, Acc& acc) __attribute__((always_inline)) {
                return [&, sq](auto s_) __attribute__((always_inline)) {
                    constexpr int n = 3 * RT, NS = SF * RT, s = decltype(s_)::value;
                    if constexpr (s == 4 * RT) load_bias(BN, sq + 2 < a.nq ? sq + 2 : 0, true);       // (the first 2 RT MFMAs took this stage's)
                    if constexpr (s >= NS / 4) static_for<(s - NS / 4) * n / (NS - NS / 4), (s + 1 - NS / 4) * n / (NS - NS / 4)>([&](auto k_) __attribute__((always_inline)) { q_step(k_, sq, acc); });
                };
            };
            load_bias(BN, 0, true);
            stage(1, up_into(acc0), idle);
            load_bias(BN, 1, true);
            for (int sq = 0; sq + 2 < a.nq; sq += 2) {       // nq is even: an even stage, then an odd one
                stage(2, up_into(acc1), q_slots(sq, acc0));
                stage(1, up_into(acc0), q_slots(sq + 1, acc1));
            }
            stage(0, up_into(acc1), q_slots(a.nq - 2, acc0));
            static_for<0, 3 * RT>([&](auto k_) __attribute__((always_inline)) { q_step(k_, a.nq - 1, acc1); });
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // no transfer into LDS may outlive the workgroup
    blk_barrier();
}

bool tail_width_ok(int64_t d, int dtype) { return (d == 192 || d == 256 || d == 384) && (dtype == BSRL_F16 || dtype == BSRL_BF16); }
int64_t tail_slots(int64_t d) { return d == 384 ? TailGeo<384>::SLOTS : d == 256 ? TailGeo<256>::SLOTS : TailGeo<192>::SLOTS; }
int64_t tail_stages(int64_t d, int64_t F, int64_t n_next) { return (F ? d / 32 + 2 * (F / 32) : 0) + n_next / 32; }
int64_t tail_frag_bytes(int64_t d, int64_t F, int64_t n_next) { return tail_stages(d, F, n_next) * (d / 16) * 1024; }
size_t tail_dyn_bytes(int64_t d, int64_t F, int64_t n_next, int64_t slots) {
    return (size_t)(((F + 6 * d + n_next) / 4 + 63) & ~(int64_t)63) * 16 + (size_t)(slots * (d / 16) * 1024);
}
// F = 0: the lead form
bool tail_shape_ok(int64_t d, int64_t F, int64_t n_next, int dtype) {
    if (!tail_width_ok(d, dtype) || n_next < 0 || n_next % 64 != 0 || n_next > 3 * d) return false;
    if (F == 0 ? n_next == 0 : (F < 64 || F % 32 != 0 || F > 16384)) return false;
    // the ring's first fill must end inside the image, and vectors and ring fit a workgroup's LDS
    return tail_stages(d, F, n_next) >= tail_slots(d) && tail_dyn_bytes(d, F, n_next, tail_slots(d)) + 1024 <= (size_t)LDS_BUDGET;
}

// bound: the most rows there can be (the row count itself when the device adds none)
template <typename DT, int D, int RT, int ACT, bool LN, int XS, bool LEAD, bool XI32 = false, bool XO32 = false>
int tail_launch_xs(const TailArgs& a, int64_t bound, int cus, hipStream_t st) {
    const size_t dyn = tail_dyn_bytes(D, a.F, 32 * a.nq, TailRing<D, XS>::SLOTS);
    if (dyn + 1024 > (size_t)LDS_BUDGET || a.total_stages < TailRing<D, XS>::SLOTS) return BSRL_UNSUPPORTED;
    const int64_t ntiles = (bound + 64 * RT - 1) / (64 * RT);
    auto kern = block_tail_kernel<DT, D, RT, ACT, LN, XS, LEAD, XI32, XO32>;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)dyn) != hipSuccess)
        return BSRL_UNSUPPORTED;
    hipLaunchKernelGGL(kern, dim3((unsigned)(ntiles < cus ? ntiles : cus)), dim3(256), dyn, st, a);
    return BSRL_OK;
}
template <typename DT, int D, int ACT, bool LN, bool LEAD, bool XI32 = false, bool XO32 = false>
int tail_launch(const TailArgs& a, int64_t bound, int cus, hipStream_t st) {
    constexpr int RT = TailGeo<D>::RT, RS = (RT + 1) / 2;
    // up to a round of half-sized tiles: half the row tiles per wave, twice the workgroups
    if (bound <= (int64_t)cus * 64 * RS) return tail_launch_xs<DT, D, RS, ACT, LN, 0, LEAD, XI32, XO32>(a, bound, cus, st);
    if constexpr (D == 384) {      // a sixth slot of 24 KB where the vectors leave room for it
        const int rc = tail_launch_xs<DT, D, RT, ACT, LN, 1, LEAD, XI32, XO32>(a, bound, cus, st);
        if (rc != BSRL_UNSUPPORTED) return rc;
    }
    return tail_launch_xs<DT, D, RT, ACT, LN, 0, LEAD, XI32, XO32>(a, bound, cus, st);
}
template <typename DT, int D, int ACT>
int tail_act(const TailArgs& a, int64_t bound, bool xi32, bool xo32, int cus, hipStream_t st) {
    if constexpr (D == 256) {      // the fp32 stream: into it, along it, out of it (the last block has no LayerNorm behind)
        if (xo32) return !a.ln_w ? (int)BSRL_UNSUPPORTED : xi32 ? tail_launch<DT, D, ACT, true, false, true, true>(a, bound, cus, st)
                                                                : tail_launch<DT, D, ACT, true, false, false, true>(a, bound, cus, st);
        if (xi32) return a.ln_w ? (int)BSRL_UNSUPPORTED : tail_launch<DT, D, ACT, false, false, true, false>(a, bound, cus, st);
    } else if (xi32 || xo32) return BSRL_UNSUPPORTED;
    return a.ln_w ? tail_launch<DT, D, ACT, true, false>(a, bound, cus, st) : tail_launch<DT, D, ACT, false, false>(a, bound, cus, st);
}
template <typename DT, int D>
int tail_go(const TailArgs& a, int64_t bound, int act, bool xi32, bool xo32, int cus, hipStream_t st) {
    if (a.F == 0) return xi32 || xo32 ? (int)BSRL_UNSUPPORTED : tail_launch<DT, D, BSRL_ACT_RELU, true, true>(a, bound, cus, st);
    return act == BSRL_ACT_RELU ? tail_act<DT, D, BSRL_ACT_RELU>(a, bound, xi32, xo32, cus, st) : tail_act<DT, D, BSRL_ACT_GELU>(a, bound, xi32, xo32, cus, st);
}

}  // namespace

// one per width and type (block_tail_192_f16.hip, ...: they compile side by side): the launch for an activation
#define TAIL_GO(D, T) int bsrl_tail_go_##D##_##T(const void* args, int64_t bound, int act, bool xi32, bool xo32, int cus, hipStream_t st)
TAIL_GO(192, F16); TAIL_GO(256, F16); TAIL_GO(384, F16); TAIL_GO(192, BF16); TAIL_GO(256, BF16); TAIL_GO(384, BF16);
#define TAIL_INSTANCE(D, T) TAIL_GO(D, T) { return tail_go<T, D>(*static_cast<const TailArgs*>(args), bound, act, xi32, xo32, cus, st); }
