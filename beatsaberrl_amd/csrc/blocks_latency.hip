// The block stack for few envs (blocks_fused.hip: same weight image, same bits): ONE ENV PER WORKGROUP, its features dealt over
// the waves.
//
// With an env per wave (or wave pair) a single env runs at the latency of one wave's MFMA chains and LDS reads per weight stage:
// 206 us for six blocks at d = 192, 55 us for three at d = 128, whatever the chip.  Here a workgroup is NT = d / 16 waves and wave
// w owns feature tile w: the weight fragments that produce its features are read by no other wave, so they go from L2 straight
// into its registers, a group of KC fragments in use and two (d = 128: three) in flight.  What the waves share - the residual stream (fp32),
// LayerNorm's output, q | k | v, attention's output, the hidden - crosses LDS as MFMA operand fragments, seven barriers per
// block.  Bound: the weight stream of a CU, 0.88 MB per block at d = 192 at the ~40 B/clk that it reaches (10 of 11 us per block;
// six blocks do not fit an XCD's L2), and the barriers and LayerNorms between.
// Per-row arithmetic and its order are those of blocks_kernel: an accumulator starts at its bias or at the residual and takes the
// k chunks in ascending order; LayerNorm's sums and softmax's reductions run in the same lane layout.
// Six blocks at d = 192, 1 .. 256 envs: 206 - 216 -> 68 - 76 us (79 - 84 while the key mask and row addresses were spilled); three at
// d = 128: 55 - 59 -> 18 - 22 us.
#include "block_stage.h"
#include "blocks_latency.h"

namespace {

template <typename DT, int D, int DH, int ACT>
__global__ __launch_bounds__(D * 4) void blocks_latency_kernel(BlocksLatencyArgs a) {
    typedef Geo<D> G;
    constexpr int NT = G::NT, KC = G::KC, SF = G::SF, H = D / DH, TPH = DH / 16, NTHR = 64 * NT;
    constexpr int M = 4, NG = 4 + 2 * M, NBUF = D == 128 ? 4 : 3;        // groups of an FFN half and of a block per wave; buffers: register budget
    static_assert(SF == NT && 2 * H <= NT && NG % NBUF == 0 && NT % 4 == 0, "a stage is a row of tiles; an attention unit per wave");
    extern __shared__ float4 lds4[];
    const int tid = threadIdx.x, lane_ = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane_ & 15, g = lane_ >> 4;
    constexpr int F = M * D, nch = F / 32, nv4 = G::lv_size(F) / 4, lfr = G::layer_stages(F) * SF;
    f32x4* xs = reinterpret_cast<f32x4*>(lds4);                          // [row tile][feature tile][lane]
    uint4* hfr = reinterpret_cast<uint4*>(xs + 2 * NT * 64);             // [row tile][k chunk][lane]: LayerNorm output
    uint4* un = hfr + 2 * KC * 64;                                       // q | k | v | attention output, then the hidden
    uint2* qkv = reinterpret_cast<uint2*>(un);                           // [(part H + head) 2 + row tile][feature tile of the head][lane]
    uint4* ofr = un + 3 * NT * 64;                                       // [row tile][k chunk][lane]
    uint4* hid = un;                                                     // [row tile][chunk][lane]
    const int un_u4 = 3 * NT * 64 + 2 * KC * 64 > 2 * nch * 64 ? 3 * NT * 64 + 2 * KC * 64 : 2 * nch * 64;
    float4* vb = reinterpret_cast<float4*>(un + un_u4);                  // fp32 vectors of two blocks
    float* km = reinterpret_cast<float*>(vb + 2 * nv4);                  // the env's 32 slots
    const float scale_l2e = (DH == 32 ? 0.17677669529663688110f : 0.14433756729740644113f) * 1.44269504088896340736f;

    // group gi of a block: KC fragments in the order of their use (0 .. 2: q | k | v tiles w, w + NT, w + 2 NT; 3: output
    // projection; 4 .. 3 + M: W1 tiles; then W2, KC hidden chunks each); byte offsets in 32 bits (an image is a few MB)
    auto load = [&](uint4 (&f)[KC], int l, auto gi_) __attribute__((always_inline)) {
        constexpr int gi = decltype(gi_)::value;
        const char* img = reinterpret_cast<const char*>(a.frags);
        int at = 0;                                                       // first fragment
        if constexpr (gi < 3) { const int j = w + NT * gi; at = (j >> 1) * SF + (j & 1) * G::KB; }
        else if constexpr (gi == 3) at = 3 * NT * KC + (w >> 1) * SF + (w & 1) * G::KB;
        else if constexpr (gi < 4 + M) {
            const int ft = w + NT * (gi - 4), ch = ft >> 1;
            at = 4 * NT * KC + (ch == 0 ? 0 : 2 * ch - 1) * SF + (ft & 1) * G::KB;
        } else at = 4 * NT * KC + (2 * KC * (gi - 4 - M) + 2) * SF + w;
        uint32_t off = (uint32_t)(l * lfr + at) * 1024u;                  // scalar and opaque: kept out of the registers across blocks
        asm volatile("" : "+s"(off));
        const uint32_t l16 = lane_ * 16;
#pragma unroll
        for (int c = 0; c < KC; ++c) {
            // k chunks inside a two-tile stage; W2 stages alternate with W1's, but the last follows the one before it directly
            const int step = gi < 4 + M ? (c / G::KB) * G::FB + c % G::KB : (gi + 1 == NG && c + 1 == KC ? 2 * c - 1 : 2 * c) * SF;
            f[c] = *reinterpret_cast<const uint4*>(img + (off + step * 1024u) + l16);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto frag = [](const uint4& u) __attribute__((always_inline)) { return __builtin_bit_cast(s16x8, u); };

    int vp = 0;              // buffer of the current block's vectors
    uint4 buf[NBUF][KC];
    static_for<0, NBUF>([&](auto i) __attribute__((always_inline)) { load(buf[decltype(i)::value], 0, i); });
    for (int i = tid; i < nv4; i += NTHR) vb[i] = reinterpret_cast<const float4*>(a.vec)[i];
    for (int64_t env = blockIdx.x; env < a.B; env += gridDim.x) {
        // additive key bias * log2(e) of every slot, -inf past T: read where attention wants it (kept in registers it was spilled, and
        // its reload waited behind the weights in flight)
        if (tid < 32) km[tid] = tid < a.T ? DT::to_f(a.key_bias[env * a.T + tid]) * 1.44269504088896340736f : -INFINITY;
        f32x4 x[2];              // this wave's feature tile of the residual stream, both row tiles
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            const int row = 16 * rt + r16;
            const bool ok = row < a.T;
            const uint2 v = *reinterpret_cast<const uint2*>(a.x_in + (env * a.T + (ok ? row : 0)) * D + 16 * w + 4 * g);
            x[rt] = (f32x4){ok ? DT::to_f((u16)(v.x & 0xffff)) : 0.f, ok ? DT::to_f((u16)(v.x >> 16)) : 0.f,
                            ok ? DT::to_f((u16)(v.y & 0xffff)) : 0.f, ok ? DT::to_f((u16)(v.y >> 16)) : 0.f};
        }
        auto put_x = [&](int tiles) __attribute__((always_inline)) {
            xs[w * 64 + lane_] = x[0];
            if (tiles == 2) xs[(NT + w) * 64 + lane_] = x[1];
        };
        auto store_rows = [&](int rt, u16* dst, int rows_per_env, int nrows_valid) __attribute__((always_inline)) {
            int l = lane_;                                                // opaque: as in layer()
            asm volatile("" : "+v"(l));
            const int row = 16 * rt + (l & 15), g = l >> 4;
            if (row < nrows_valid) {
                uint2 v;
                v.x = bpack2<DT>(x[rt][0], x[rt][1]); v.y = bpack2<DT>(x[rt][2], x[rt][3]);
                *reinterpret_cast<uint2*>(dst + (env * rows_per_env + row) * D + 16 * w + 4 * g) = v;
            }
        };
        put_x(2);
        blk_barrier();

        auto layer = [&](int l, auto pruned_) __attribute__((always_inline)) {
            constexpr bool pruned = decltype(pruned_)::value;
            constexpr int QT = pruned ? 1 : 2;
            // opaque per block: addresses derived from the lane stay inside it instead of living in registers across blocks
            int lane = lane_;
            asm volatile("" : "+v"(lane));
            const int g = lane >> 4;
            const float* lv = reinterpret_cast<const float*>(vb + vp * nv4);
            const int ln = l + 1 == a.n_layers ? 0 : l + 1;               // the block whose first groups follow (the next env's)
            float4 vnext[2] = {make_float4(0.f, 0.f, 0.f, 0.f), make_float4(0.f, 0.f, 0.f, 0.f)};
#pragma unroll
            for (int u = 0; u < 2; ++u)
                if (tid + u * NTHR < nv4) vnext[u] = reinterpret_cast<const float4*>(a.vec)[ln * nv4 + tid + u * NTHR];
            if (pruned && a.x_res) { store_rows(0, a.x_res, a.T, a.T); store_rows(1, a.x_res, a.T, a.T); }

            // LayerNorm: four waves per row tile form its statistics (one pass, var = E[x^2] - mean^2 clamped at 0) and normalise
            // a quarter of the features each; with one wave per tile it was 3000 clk, twice in a block's 31000
            auto norm = [&](int tiles, const float* gptr, const float* bptr) __attribute__((always_inline)) {
                if (w < 4 * tiles) {
                    const int rt = w >> 2, q4 = w & 3;
                    const f32x4* row = xs + rt * NT * 64 + lane;
                    float s = 0.f, q = 0.f;
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) {
                        const f32x4 v = row[nt * 64];
#pragma unroll
                        for (int i = 0; i < 4; ++i) { s += v[i]; q = fmaf(v[i], v[i], q); }
                    }
                    f32x4 v[NT / 4]; float4 gm[NT / 4], bt[NT / 4];
#pragma unroll
                    for (int k = 0; k < NT / 4; ++k) {
                        const int nt = q4 * (NT / 4) + k;
                        v[k] = row[nt * 64];
                        gm[k] = *reinterpret_cast<const float4*>(gptr + 16 * nt + 4 * g);
                        bt[k] = *reinterpret_cast<const float4*>(bptr + 16 * nt + 4 * g);
                    }
                    rows_reduce2(s, q, OpAdd());
                    const float mean = s * (1.0f / D);
                    const float rstd = rsqrtf(fmaxf(fmaf(-mean, mean, q * (1.0f / D)), 0.f) + 1e-5f);
                    const float shift = -mean * rstd;
#pragma unroll
                    for (int k = 0; k < NT / 4; ++k) {
                        const int nt = q4 * (NT / 4) + k;
                        const float y0 = fmaf(fmaf(v[k][0], rstd, shift), gm[k].x, bt[k].x);
                        const float y1 = fmaf(fmaf(v[k][1], rstd, shift), gm[k].y, bt[k].y);
                        const float y2 = fmaf(fmaf(v[k][2], rstd, shift), gm[k].z, bt[k].z);
                        const float y3 = fmaf(fmaf(v[k][3], rstd, shift), gm[k].w, bt[k].w);
                        reinterpret_cast<uint2*>(hfr)[((rt * KC + (nt >> 1)) * 64 + lane) * 2 + (nt & 1)] = make_uint2(bpack2<DT>(y0, y1), bpack2<DT>(y2, y3));
                    }
                }
                blk_barrier();
            };
            // the other operand of a group: KC fragments of `tiles` row tiles out of LDS in one burst (left to itself the compiler
            // reads one, waits, multiplies: 12 LDS latencies per group)
            s16x8 act[2][KC];
            auto get = [&](const uint4* p, int pitch, int tiles) __attribute__((always_inline)) {
#pragma unroll
                for (int c = 0; c < KC; ++c)
#pragma unroll
                    for (int rt = 0; rt < 2; ++rt) if (rt < tiles) act[rt][c] = frag(p[(rt * pitch + c) * 64 + lane]);
                __builtin_amdgcn_sched_barrier(0);
            };
            // group gi's buffer has had its last use: the group NBUF behind it takes its place
            auto next = [&](auto gi_) __attribute__((always_inline)) {
                constexpr int gi = decltype(gi_)::value + NBUF;
                load(buf[gi % NBUF], gi < NG ? l : ln, std::integral_constant<int, gi % NG>{});
            };
            auto bias4 = [&](const float* p) __attribute__((always_inline)) {
                const float4 b = *reinterpret_cast<const float4*>(p + 4 * g);
                return (f32x4){b.x, b.y, b.z, b.w};
            };

            norm(2, lv + G::LN1G, lv + G::LN1B);
            get(hfr, KC, 2);
            // ---- q | k | v: head-major tiles [q | k | v] of TPH tiles each, tile w + NT t ----
            auto project = [&](const uint4 (&f)[KC], int t_) __attribute__((always_inline)) {
                const int j = w + NT * t_, hd = j / (3 * TPH), r = j % (3 * TPH), part = r / TPH, t = r % TPH;       // uniform over the wave
                f32x4 acc[2];
                if (part < 2) {
                    acc[0] = bias4(lv + (part == 0 ? G::BQ : G::BK) + DH * hd + 16 * t); acc[1] = acc[0];
#pragma unroll
                    for (int c = 0; c < KC; ++c)
#pragma unroll
                        for (int rt = 0; rt < 2; ++rt) acc[rt] = DT::mfma32(frag(f[c]), act[rt][c], acc[rt]);
                } else {                                                   // V^T: operand roles swapped
                    acc[0] = acc[1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int c = 0; c < KC; ++c)
#pragma unroll
                        for (int rt = 0; rt < 2; ++rt) acc[rt] = DT::mfma32(act[rt][c], frag(f[c]), acc[rt]);
                }
#pragma unroll
                for (int rt = 0; rt < 2; ++rt)
                    qkv[(((part * H + hd) * 2 + rt) * TPH + t) * 64 + lane] = make_uint2(bpack2<DT>(acc[rt][0], acc[rt][1]), bpack2<DT>(acc[rt][2], acc[rt][3]));
            };
            static_for<0, 3>([&](auto i) __attribute__((always_inline)) { project(buf[decltype(i)::value % NBUF], decltype(i)::value); next(i); });
            blk_barrier();
            // ---- attention: wave w is (head w / 2, query tile w % 2) ----
            if (w < 2 * H && (w & 1) < QT) {
                const int hd = w >> 1, qt = w & 1;
                auto part = [&](int p, int rt, int t) __attribute__((always_inline)) { return qkv[(((p * H + hd) * 2 + rt) * TPH + t) * 64 + lane]; };
                f32x4 sc[2];
                BFrag8 qf;
                BFrag4 q2;
                qf.h[0] = part(0, qt, 0); qf.h[1] = part(0, qt, 1);
                if (TPH == 3) q2.h = part(0, qt, TPH - 1);
#pragma unroll
                for (int kt = 0; kt < 2; ++kt) {
                    BFrag8 kf;
                    kf.h[0] = part(1, kt, 0); kf.h[1] = part(1, kt, 1);
                    sc[kt] = DT::mfma32(kf.v, qf.v, (f32x4){0.f, 0.f, 0.f, 0.f});
                    if (TPH == 3) {             // features 32..47 into their own accumulator, as in the other kernels
                        BFrag4 k2;
                        k2.h = part(1, kt, TPH - 1);
                        const f32x4 s2 = DT::mfma16(k2.v, q2.v, (f32x4){0.f, 0.f, 0.f, 0.f});
#pragma unroll
                        for (int i = 0; i < 4; ++i) sc[kt][i] += s2[i];
                    }
                }
                float sv[2][4], mx = -INFINITY, sum = 0.f;
                f32x4 kmask[2];
#pragma unroll
                for (int kt = 0; kt < 2; ++kt) kmask[kt] = *reinterpret_cast<const f32x4*>(km + 16 * kt + 4 * g);
#pragma unroll
                for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) { sv[kt][i] = fmaf(sc[kt][i], scale_l2e, kmask[kt][i]); mx = fmaxf(mx, sv[kt][i]); }
                mx = fmaxf(mx, __shfl_xor(mx, 16, WAVE)); mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE));
#pragma unroll
                for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) { sv[kt][i] = __builtin_amdgcn_exp2f(sv[kt][i] - mx); sum += sv[kt][i]; }
                sum += __shfl_xor(sum, 16, WAVE); sum += __shfl_xor(sum, 32, WAVE);
                const float inv = __builtin_amdgcn_rcpf(sum);
                BFrag8 pf;
#pragma unroll
                for (int kt = 0; kt < 2; ++kt) {
                    pf.w[2 * kt] = bpack2<DT>(sv[kt][0] * inv, sv[kt][1] * inv);
                    pf.w[2 * kt + 1] = bpack2<DT>(sv[kt][2] * inv, sv[kt][3] * inv);
                }
#pragma unroll
                for (int t = 0; t < TPH; ++t) {
                    BFrag8 vf;
                    vf.h[0] = part(2, 0, t); vf.h[1] = part(2, 1, t);
                    const f32x4 o = DT::mfma32(vf.v, pf.v, bias4(lv + G::BV + DH * hd + 16 * t));
                    const int nt = hd * TPH + t;
                    reinterpret_cast<uint2*>(ofr)[((qt * KC + (nt >> 1)) * 64 + lane) * 2 + (nt & 1)] = make_uint2(bpack2<DT>(o[0], o[1]), bpack2<DT>(o[2], o[3]));
                }
            }
            blk_barrier();
            // ---- output projection onto the residual ----
            {
                get(ofr, KC, QT);
                const f32x4 b = bias4(lv + G::BOUT + 16 * w);
#pragma unroll
                for (int rt = 0; rt < QT; ++rt) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[rt][i] += b[i];
                }
#pragma unroll
                for (int c = 0; c < KC; ++c)
#pragma unroll
                    for (int rt = 0; rt < QT; ++rt) x[rt] = DT::mfma32(frag(buf[3 % NBUF][c]), act[rt][c], x[rt]);
                next(std::integral_constant<int, 3>{});
                put_x(QT);
#pragma unroll
                for (int u = 0; u < 2; ++u)                                // the next block's vectors: their buffer was last read a block ago
                    if (tid + u * NTHR < nv4) vb[(vp ^ 1) * nv4 + tid + u * NTHR] = vnext[u];
            }
            blk_barrier();
            // ---- LayerNorm + FFN ----
            norm(QT, lv + G::LN2G, lv + G::LN2B);
            get(hfr, KC, QT);
            {
                const f32x4 b = bias4(lv + G::b2(F) + 16 * w);
#pragma unroll
                for (int rt = 0; rt < QT; ++rt) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[rt][i] += b[i];
                }
            }
            auto up = [&](const uint4 (&f)[KC], int i_) __attribute__((always_inline)) {
                const int ft = w + NT * i_;
                f32x4 acc[2];
                acc[0] = bias4(lv + G::B1 + 16 * ft); acc[1] = acc[0];
#pragma unroll
                for (int c = 0; c < KC; ++c)
#pragma unroll
                    for (int rt = 0; rt < QT; ++rt) acc[rt] = DT::mfma32(frag(f[c]), act[rt][c], acc[rt]);
#pragma unroll
                for (int rt = 0; rt < QT; ++rt)
                    reinterpret_cast<uint2*>(hid)[((rt * nch + (ft >> 1)) * 64 + lane) * 2 + (ft & 1)] =
                        make_uint2(bpack2<DT>(apply_act16<ACT>(acc[rt][0]), apply_act16<ACT>(acc[rt][1])),
                                   bpack2<DT>(apply_act16<ACT>(acc[rt][2]), apply_act16<ACT>(acc[rt][3])));
            };
            static_for<0, M>([&](auto i) __attribute__((always_inline)) {
                constexpr int gi = 4 + decltype(i)::value;
                up(buf[gi % NBUF], decltype(i)::value);
                next(std::integral_constant<int, gi>{});
            });
            blk_barrier();
            auto down = [&](const uint4 (&f)[KC], int i_) __attribute__((always_inline)) {
                get(hid + KC * i_ * 64, nch, QT);
#pragma unroll
                for (int c = 0; c < KC; ++c)
#pragma unroll
                    for (int rt = 0; rt < QT; ++rt) x[rt] = DT::mfma32(frag(f[c]), act[rt][c], x[rt]);
            };
            static_for<0, M>([&](auto i) __attribute__((always_inline)) {
                constexpr int gi = 4 + M + decltype(i)::value;
                down(buf[gi % NBUF], decltype(i)::value);
                next(std::integral_constant<int, gi>{});
            });
            if (l + 1 < a.n_layers) { put_x(2); blk_barrier(); }
            vp ^= 1;
        };
        const int n_full = a.n_queries > 0 ? a.n_layers - 1 : a.n_layers;
        for (int l = 0; l < n_full; ++l) layer(l, std::false_type{});
        if (a.n_queries > 0) {
            layer(a.n_layers - 1, std::true_type{});
            store_rows(0, a.x_out, a.n_queries, a.n_queries);
        } else { store_rows(0, a.x_out, a.T, a.T); store_rows(1, a.x_out, a.T, a.T); }
    }
}

template <int D> size_t latency_bytes() {
    constexpr int NT = Geo<D>::NT, KC = Geo<D>::KC, F = 4 * D;
    const size_t qkvo = (size_t)(3 * NT + 2 * KC) * 64, hid = (size_t)2 * (F / 32) * 64;
    return ((size_t)2 * NT * 64 + 2 * KC * 64 + (qkvo > hid ? qkvo : hid)) * 16 + (size_t)2 * Geo<D>::lv_size(F) * 4 + 128;
}
template <typename DT, int D, int DH, int ACT>
bool go(const BlocksLatencyArgs& a, int cus, hipStream_t st) {
    if (a.F != 4 * D) return false;
    const size_t dyn = latency_bytes<D>();
    auto kern = blocks_latency_kernel<DT, D, DH, ACT>;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)dyn) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)(a.B < cus ? a.B : cus)), dim3(64 * Geo<D>::NT), dyn, st, a);
    return true;
}
template <typename DT>
bool by_shape(const BlocksLatencyArgs& a, int d, int act, int cus, hipStream_t st) {
    if (d == 128) return act == BSRL_ACT_RELU ? go<DT, 128, 32, BSRL_ACT_RELU>(a, cus, st) : go<DT, 128, 32, BSRL_ACT_GELU>(a, cus, st);
    if (d == 192) return act == BSRL_ACT_RELU ? go<DT, 192, 48, BSRL_ACT_RELU>(a, cus, st) : go<DT, 192, 48, BSRL_ACT_GELU>(a, cus, st);
    return false;
}

}  // namespace

bool bsrl_blocks_latency(const BlocksLatencyArgs& a, int d, int act, int dtype, int cus, hipStream_t st) {
    return dtype == BSRL_F16 ? by_shape<F16>(a, d, act, cus, st) : by_shape<BF16>(a, d, act, cus, st);
}
