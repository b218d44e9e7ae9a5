// The block stack (blocks_fused.hip: same weight image, same bits) over the ATTENDABLE tokens of TWO ENVS PER WAVE.
//
// A masked token has weight zero in every softmax (its score would have to lead by thousands): no output depends on its row.  With one
// env per wave (blocks_env_kernel) the two 16-row tiles of an env hold 29 tokens of which, notes being there six times in ten, 19 are
// attendable; here the attendable tokens of two envs share THREE tiles.  A workgroup is four waves, one per SIMD in 512 registers, so that
// every weight fragment read from LDS feeds three MFMAs, reads run three fragments ahead of them across the stages, and the FFN's vector
// work is dealt behind them (block_tail.h has the measurements).  The final block, whose queries all sit in the first tile, has code of
// its own.  What bounds it: vector instructions beside the MFMAs, 2.7 for each (both envs' scores for a mixed query tile, LayerNorm out of
// accumulation registers); MFMAs are busy for 0.4 of the time, the weight stream is not felt.
// Whole forward, recipe shape (d = 192, six blocks, F = 768), f16, us, one env per wave / two: 1250 envs 398 / 379, 2048 441 / 400,
// 4096 800 / 704, 8192 1598 / 1374, 16384 2986 / 2565; up to 4 envs per CU, where one env per wave leaves half of the waves away,
// 328 / 379.  At d = 128 the share of vector work is larger and two lose: 16384 envs, bf16, 828 / 928.
// Rows of a wave: lead tokens of A, lead tokens of B, A's attendable notes, B's; queries of the final block are then the first tile's.
// Everything row-wise does not care.  Attention does: its sums over keys run over the SLOTS of the full stream (a dropped token's is
// zero), which keeps their order and with it the bits.  A wave scatters K and V^T of the head that it has projected from its rows
// into the slots of their env, in LDS, and reads them back as fragments; a query tile that holds rows of both envs takes the scores
// against both and selects by lane - as it does the products with V, where a zero probability would not keep out an infinity.
// Envs are paired by rank, the i-th longest of 64 with the i-th shortest; two that do not fit 48 rows go alone.  Where that leaves too many
// alone, which only the device knows, this kernel steps aside for blocks_env_kernel or the other way round: both are launched, both ask
// blocks_pairs_pay.
#include "block_stage.h"
#include "blocks_pair.h"

namespace {

constexpr int RT = 3, ROWS = 16 * RT, CHUNK = BLOCKS_PAIR_CHUNK;

// ---- pairs: one wave per 64 envs ----------------------------------------------------------------------------------
// entry {a, b, notes of a, notes of b}; b = -1: a alone; a = -1: none.  A chunk's entries fill its first tiles[chunk] groups of four.
template <typename DT>
__global__ __launch_bounds__(64) void blocks_pairs_kernel(const u16* __restrict__ key_bias, int4* __restrict__ pairs, int* __restrict__ tiles, int64_t B, int T, int lead) {
    __shared__ int ord[CHUNK];
    const int lane = threadIdx.x;
    const int64_t first = (int64_t)blockIdx.x * CHUNK, env = first + lane;
    const int envs = B - first < CHUNK ? (int)(B - first) : CHUNK;
    uint32_t mask = 0;
    if (lane < envs)
        for (int t = lead; t < T; ++t) mask |= (DT::to_f(key_bias[env * T + t]) < -0.5f * BSRL_MASK_BIAS ? 0u : 1u) << (t - lead);
    const int n = lane < envs ? __popc(mask) : 32;   // rank by notes, lanes past the end last
    int rank = 0;
#pragma unroll
    for (int j = 0; j < CHUNK; ++j) {
        const int nj = __builtin_amdgcn_readlane(n, j);
        rank += nj < n || (nj == n && j < lane) ? 1 : 0;
    }
    ord[rank] = lane;
    __syncthreads();
    const int half = (envs + 1) / 2, i = lane < half ? lane : 0;               // a wave's shuffles need every lane
    const int la = ord[envs - 1 - i], lb = ord[i];                            // the odd one out meets itself
    const int ma = __shfl((int)mask, la, WAVE), mb = __shfl((int)mask, lb, WAVE);
    const bool two = lane < half && la != lb, apart = two && 2 * lead + __popc(ma) + __popc(mb) > ROWS;
    const uint64_t splits = __ballot(apart);
    const int used = half + __popcll(splits), at = lane + __popcll(splits & ((1ull << lane) - 1));
    int4* const out = pairs + (int64_t)blockIdx.x * CHUNK;
    if (lane < half) {
        out[at] = two && !apart ? make_int4((int)(first + la), (int)(first + lb), ma, mb) : make_int4((int)(first + la), -1, ma, 0);
        if (apart) out[at + 1] = make_int4((int)(first + lb), -1, mb, 0);
    }
    const int ntiles = (used + 3) / 4;
    if (lane >= used && lane < 4 * ntiles) out[lane] = make_int4(-1, -1, 0, 0);
    if (lane == 0) tiles[blockIdx.x] = ntiles;
}

// two rounded relus in a word: v_cvt_pk, then the sign clears its half
template <typename DT> __device__ __forceinline__ uint32_t relu2(float a, float b) { return bpack2<DT>(relu1(a), relu1(b)); }
template <> __device__ __forceinline__ uint32_t relu2<F16>(float a, float b) {
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    const f16x2 z = {(_Float16)0.f, (_Float16)0.f};
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(f16x2, bpack2<F16>(a, b)), z));
}
template <int D> struct PairRing : StageRing<Geo<D>::SF, D == 128 ? 10 : 7, 4> {};
template <int D, int DH> struct PairGeo {
    static constexpr int KB = 32 * DH * 2, VB = DH * 64, ENV = KB + VB, WAVE_B = 2 * ENV;            // a head's K, V^T of an env, a wave's
    static constexpr int vec_bytes(int F) { return (Geo<D>::lv_size(F) * 4 + 1023) & ~1023; }
    static constexpr size_t lds(int F) { return 2 * vec_bytes(F) + 4 * WAVE_B + (size_t)PairRing<D>::SLOTS * PairRing<D>::STAGE_BYTES; }
};

template <typename DT, int D, int DH>
__global__ __launch_bounds__(256, 1) void blocks_pair_kernel(BlocksPairArgs a) {
    typedef Geo<D> G;
    typedef PairRing<D> R;
    typedef PairGeo<D, DH> P;
    constexpr int NT = G::NT, KC = G::KC, SF = G::SF, H = D / DH, TPH = DH / 16, NBUF = 4;
    static_assert(H * DH == D, "whole heads");
    extern __shared__ float4 lds4[];                 // ring | K / V^T of the four waves | vectors of two blocks
    char* const lds = reinterpret_cast<char*>(lds4);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
    const int T = a.T, lead = a.lead, nl = a.n_layers, vecb = P::vec_bytes(a.F), lvn = G::lv_size(a.F);
    const float scale_l2e = (DH == 32 ? 0.17677669529663688110f : 0.14433756729740644113f) * 1.44269504088896340736f;
    constexpr int RING_B = R::SLOTS * R::STAGE_BYTES;
    char* const kv = lds + RING_B + wave * P::WAVE_B;
    char* const vbuf = lds + RING_B + 4 * P::WAVE_B;
    const int ntiles = blocks_pair_tiles(a.plan, lane);
    if (!blocks_pairs_pay(a.plan, ntiles)) return;

    R pipe;
    int vp = 0;                                      // buffer of the current block's vectors
    pipe.start(reinterpret_cast<const uint4*>(lds4), a.frags, a.total_stages, wave, lane);
    for (int i = tid; i < lvn / 4; i += 256) reinterpret_cast<float4*>(vbuf)[i] = reinterpret_cast<const float4*>(a.vec)[i];
    blk_barrier();
    // block l's vectors on their way into the other buffer: called behind a barrier that every wave reaches with its last read of it done
    // (the first stage's admission); they have landed when a few stages more have been admitted
    auto fetch_vectors = [&](int l) __attribute__((always_inline)) {
        const uint32_t dst = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)(vbuf + (vp ^ 1) * vecb);
        for (int p = wave; p * 1024 < lvn * 4; p += 4)
            if (p * 1024 + lane * 16 < lvn * 4) env_ring_load((uint32_t)(p * 1024 + lane * 16), a.vec + (int64_t)l * lvn, dst + p * 1024);
    };

    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        // the chunk that holds the tile: 64 chunks a step
        int before = 0, c0 = 0, upto;
        uint64_t past;
        for (;; c0 += WAVE) {
            const int n = c0 + lane < a.plan.chunks ? a.plan.tiles[c0 + lane] : 0;
            upto = n;
#pragma unroll
            for (int o = 1; o < WAVE; o *= 2) {
                const int v = __shfl_up(upto, o, WAVE);
                if (lane >= o) upto += v;
            }
            past = __ballot(before + upto > tile);
            if (past || c0 + WAVE >= a.plan.chunks) break;
            before += __builtin_amdgcn_readlane(upto, WAVE - 1);
        }
        const int at = __builtin_ctzll(past);        // (not empty: tile < ntiles)
        if (at > 0) before += __builtin_amdgcn_readlane(upto, at - 1);
        const int4 pair = a.pairs[(int64_t)(c0 + at) * CHUNK + (tile - before) * 4 + wave];
        const int ea = __builtin_amdgcn_readfirstlane(pair.x), eb = __builtin_amdgcn_readfirstlane(pair.y);
        const uint32_t ma = __builtin_amdgcn_readfirstlane(pair.z), mb = __builtin_amdgcn_readfirstlane(pair.w);
        if (ea < 0) {                                // no env: this wave only moves its share of the weight stream
            for (int l = 0; l < nl; ++l) {
                for (int s = 0; s < a.total_stages / nl; s += 2) {
                    pipe.template admit<0>();
                    if (s == 0) fetch_vectors(l + 1 == nl ? 0 : l + 1);
                    pipe.template admit<1>();
                }
                vp ^= 1;
            }
            continue;
        }
        const bool two = eb >= 0;
        const int na = __popc(ma);
        // rows -> (env, token): a byte per row, 32 env + token, token 31 where there is none (a slot that no softmax looks at)
        uint8_t* const code = reinterpret_cast<uint8_t*>(kv);
        {
            const int half = lane >> 5, t = lane & 31;                       // lanes 0 .. 23 A's notes, 32 .. 55 B's
            const uint32_t m = half ? mb : ma;
            if (lane < ROWS) code[lane] = (uint8_t)(lane < lead ? lane : two && lane < 2 * lead ? 32 + lane - lead : 31);
            asm volatile("" ::: "memory");
            if (m >> t & 1) code[2 * lead + (half ? na : 0) + __popc(m & ((1u << t) - 1u))] = (uint8_t)(32 * half + lead + t);
            asm volatile("" ::: "memory");
        }
        bool isb[RT];                                // of this lane's row of every tile
        int tok[RT], kat[RT];                        // its token, its K row's place
        uint32_t vat[RT][2];                         // places of rows 4 g + 0..3 in V^T, two to a register
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            const int c = code[16 * rt + r16];
            const uint32_t c4 = *reinterpret_cast<const uint32_t*>(code + 16 * rt + 4 * g);
            isb[rt] = c & 32; tok[rt] = c & 31;
            kat[rt] = (isb[rt] ? P::ENV : 0) + tok[rt] * (DH * 2) + 8 * g;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int t = c4 >> (8 * i) & 31;
                const uint32_t at = (c4 >> (8 * i) & 32 ? P::ENV : 0) + P::KB + r16 * 64 + ((((t >> 2) ^ (((r16 >> 2) & 1) << 2)) << 3)) + (t & 3) * 2;
                if (i & 1) vat[rt][i >> 1] |= at << 16; else vat[rt][i >> 1] = at;
            }
        }
        asm volatile("" ::: "memory");
        const int64_t base_a = (int64_t)ea * T, base_b = (int64_t)(two ? eb : ea) * T;
        f32x4 x[RT][NT];
        float km[2][2][4];                           // [env][key tile]: additive key bias * log2(e) per slot; -inf past T
        {
            // the loads of a pass at once, waited for once, with the wait the compiler can see
            uint2 raw[RT][NT];
            u16 kraw[2][2][4];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const u16* xr = a.x_in + ((isb[rt] ? base_b : base_a) + (tok[rt] < T ? tok[rt] : 0)) * D;
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) raw[rt][nt] = *reinterpret_cast<const uint2*>(xr + 16 * nt + 4 * g);
            }
#pragma unroll
            for (int e = 0; e < 2; ++e)
#pragma unroll
                for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int key = 16 * kt + 4 * g + i;
                        kraw[e][kt][i] = a.key_bias[(e ? base_b : base_a) + (key < T ? key : 0)];
                    }
            // slots of dropped tokens: zeros for the whole pass
#pragma unroll
            for (int i = 0; i < P::WAVE_B / 1024; ++i) reinterpret_cast<uint4*>(kv)[i * 64 + lane] = make_uint4(0, 0, 0, 0);
            asm volatile("" ::: "memory");           // (stores and loads of other types follow: the order is the wave's program order)
            __builtin_amdgcn_s_waitcnt(0x0F70);
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    const uint32_t lo = tok[rt] < T ? raw[rt][nt].x : 0u, hi = tok[rt] < T ? raw[rt][nt].y : 0u;
                    f32x4& xx = x[rt][nt];
                    xx[0] = DT::to_f((u16)(lo & 0xffff)); xx[1] = DT::to_f((u16)(lo >> 16));
                    xx[2] = DT::to_f((u16)(hi & 0xffff)); xx[3] = DT::to_f((u16)(hi >> 16));
                    asm("" : "+a"(xx));              // the stream lives in accumulation registers
                }
#pragma unroll
            for (int e = 0; e < 2; ++e)
#pragma unroll
                for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) km[e][kt][i] = 16 * kt + 4 * g + i < T ? DT::to_f(kraw[e][kt][i]) * 1.44269504088896340736f : -INFINITY;
        }

        // one stage: fragment i + 3 is requested before fragment i's MFMAs.  next: 0 = nothing follows, 1 = an odd stage, 2 = an even one (a
        // scalar); mm(i, fragment, fill): its MFMAs; fill(k): the vector work behind the k-th (block_tail.h)
        s16x8 wr[NBUF];
        auto stage = [&](auto next, auto&& mm, auto&& fill) __attribute__((always_inline)) {
            static_for<0, SF>([&](auto i_) __attribute__((always_inline)) {
                constexpr int i = decltype(i_)::value, n = i + NBUF - 1;
                if constexpr (n < SF) wr[n % NBUF] = pipe.frag(n, lane);
                else if (next != 0) {
                    if constexpr (n == SF) {
                        if (next == 2) { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); pipe.template admit<0>(); }
                        else if (next == 1) pipe.template admit<1>();
                    }
                    wr[n % NBUF] = pipe.frag(n - SF, lane);              // (behind the last stage: read, not used)
                }
                __builtin_amdgcn_sched_barrier(0);
                mm(i_, wr[i % NBUF], fill);
                __builtin_amdgcn_sched_barrier(0);
            });
        };
        static_assert(SF % NBUF == 0, "rotating fragment registers");
        auto idle = [](auto) __attribute__((always_inline)) {};

        typedef std::integral_constant<int, 1> S1; typedef std::integral_constant<int, 2> S2;
        typedef BFrag8 Frags[RT][KC];                // LayerNorm's output
        typedef std::integral_constant<int, 1> Q1; typedef std::integral_constant<int, RT> QA;
        // LayerNorm of the first row tiles -> operand fragments; the bias of what is added to the stream next goes in on the way
        auto norm = [&](Frags& hf, auto tiles_, auto added_, const float* gptr, const float* bptr, const float* bias) __attribute__((always_inline)) {
            static_for<0, decltype(tiles_)::value>([&](auto rt_) __attribute__((always_inline)) {
                constexpr int rt = decltype(rt_)::value;
                float s = 0.f, q = 0.f;
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    const f32x4 r = x[rt][nt];
#pragma unroll
                    for (int i = 0; i < 4; ++i) { s += r[i]; q = fmaf(r[i], r[i], q); }
                    if ((nt & 3) == 3) __builtin_amdgcn_sched_barrier(0);
                }
                rows_reduce2(s, q, OpAdd());
                const float mean = s * (1.0f / D);
                const float rstd = rsqrtf(fmaxf(fmaf(-mean, mean, q * (1.0f / D)), 0.f) + 1e-5f);
                const float shift = -mean * rstd;
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    const float4 gm = *reinterpret_cast<const float4*>(gptr + 16 * nt + 4 * g);
                    const float4 bt = *reinterpret_cast<const float4*>(bptr + 16 * nt + 4 * g);
                    f32x4 r = x[rt][nt];
                    hf[rt][nt >> 1].w[(nt & 1) * 2] = bpack2<DT>(fmaf(fmaf(r[0], rstd, shift), gm.x, bt.x), fmaf(fmaf(r[1], rstd, shift), gm.y, bt.y));
                    hf[rt][nt >> 1].w[(nt & 1) * 2 + 1] = bpack2<DT>(fmaf(fmaf(r[2], rstd, shift), gm.z, bt.z), fmaf(fmaf(r[3], rstd, shift), gm.w, bt.w));
                    if constexpr (rt < decltype(added_)::value) {
                        const float4 b = *reinterpret_cast<const float4*>(bias + 16 * nt + 4 * g);
                        r[0] += b.x; r[1] += b.y; r[2] += b.z; r[3] += b.w;
                        asm("" : "+a"(r));
                        x[rt][nt] = r;
                    }
                    if ((nt & 1) == 1) __builtin_amdgcn_sched_barrier(0);
                }
            });
        };
        // the attention sub-block: two heads at a time
        constexpr int HP = H / 2, PST = 3 * TPH, PCH = TPH;      // pairs of heads; stages and chunks of attention's output per pair
        auto attention_block = [&](const Frags& hf, const float* lv, auto qt_) __attribute__((always_inline)) {
            constexpr int QT = decltype(qt_)::value;
            uint2 q[2][QT][TPH];                     // Q fragments [head of the pair][row tile][feature tile]
            BFrag8 on[QT][PCH], of[QT][KC];          // the pair's output, all heads'
            // attention of the pair's head hd over the slots of both envs
            auto attention = [&](auto hd_, const float* bv_) __attribute__((always_inline)) {
                constexpr int hd = decltype(hd_)::value;
                BFrag8 kf[2][2]; BFrag4 k2[2][2];
#pragma unroll
                for (int e = 0; e < 2; ++e)
#pragma unroll
                    for (int kt = 0; kt < 2; ++kt) {
                        const char* p = kv + e * P::ENV + (16 * kt + r16) * (DH * 2) + 8 * g;
                        kf[e][kt].h[0] = *reinterpret_cast<const uint2*>(p); kf[e][kt].h[1] = *reinterpret_cast<const uint2*>(p + 32);
                        if (TPH == 3) k2[e][kt].h = *reinterpret_cast<const uint2*>(p + 64);
                    }
                BFrag8 vf[2][TPH];
#pragma unroll
                for (int e = 0; e < 2; ++e)
#pragma unroll
                    for (int t = 0; t < TPH; ++t) {
                        const char* p = kv + e * P::ENV + P::KB + (16 * t + r16) * 64;
                        const int sw = ((r16 >> 2) & 1) << 2;
                        vf[e][t].h[0] = *reinterpret_cast<const uint2*>(p + ((g ^ sw) << 3)); vf[e][t].h[1] = *reinterpret_cast<const uint2*>(p + (((4 + g) ^ sw) << 3));
                    }
                float sv[QT][2][4], m[QT + 1], sum[QT + 1];
#pragma unroll
                for (int qt = 0; qt < QT; ++qt) {
                    BFrag8 qf; BFrag4 q2;
                    qf.h[0] = q[hd][qt][0]; qf.h[1] = q[hd][qt][1];
                    if (TPH == 3) q2.h = q[hd][qt][TPH - 1];
                    m[qt] = -INFINITY;
#pragma unroll
                    for (int kt = 0; kt < 2; ++kt) {
                        f32x4 sc[2];
#pragma unroll
                        for (int e = 0; e < 2; ++e) {
                            sc[e] = DT::mfma32(kf[e][kt].v, qf.v, (f32x4){0.f, 0.f, 0.f, 0.f});
                            if (TPH == 3) {          // features 32..47 into their own accumulator, as in the other kernels
                                const f32x4 s2 = DT::mfma16(k2[e][kt].v, q2.v, (f32x4){0.f, 0.f, 0.f, 0.f});
#pragma unroll
                                for (int i = 0; i < 4; ++i) sc[e][i] += s2[i];
                            }
                        }
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            sv[qt][kt][i] = fmaf(isb[qt] ? sc[1][i] : sc[0][i], scale_l2e, isb[qt] ? km[1][kt][i] : km[0][kt][i]);
                            m[qt] = fmaxf(m[qt], sv[qt][kt][i]);
                        }
                    }
                }
                m[QT] = m[QT - 1];
#pragma unroll
                for (int p = 0; p < QT; p += 2) rows_reduce2(m[p], m[p + 1], OpMax());
#pragma unroll
                for (int qt = 0; qt < QT; ++qt) {
                    sum[qt] = 0.f;
#pragma unroll
                    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                        for (int i = 0; i < 4; ++i) { sv[qt][kt][i] = __builtin_amdgcn_exp2f(sv[qt][kt][i] - m[qt]); sum[qt] += sv[qt][kt][i]; }
                }
                sum[QT] = sum[QT - 1];
#pragma unroll
                for (int p = 0; p < QT; p += 2) rows_reduce2(sum[p], sum[p + 1], OpAdd());
                float4 bv[TPH];
#pragma unroll
                for (int t = 0; t < TPH; ++t) bv[t] = *reinterpret_cast<const float4*>(bv_ + DH * hd + 16 * t + 4 * g);
#pragma unroll
                for (int qt = 0; qt < QT; ++qt) {
                    const float inv = __builtin_amdgcn_rcpf(sum[qt]);
                    BFrag8 pf;
#pragma unroll
                    for (int kt = 0; kt < 2; ++kt) {
                        pf.w[2 * kt] = bpack2<DT>(sv[qt][kt][0] * inv, sv[qt][kt][1] * inv);
                        pf.w[2 * kt + 1] = bpack2<DT>(sv[qt][kt][2] * inv, sv[qt][kt][3] * inv);
                    }
#pragma unroll
                    for (int t = 0; t < TPH; ++t) {
                        const f32x4 b4 = {bv[t].x, bv[t].y, bv[t].z, bv[t].w};
                        const f32x4 oa = DT::mfma32(vf[0][t].v, pf.v, b4), ob = DT::mfma32(vf[1][t].v, pf.v, b4);
                        f32x4 o;
#pragma unroll
                        for (int i = 0; i < 4; ++i) o[i] = isb[qt] ? ob[i] : oa[i];
                        constexpr int nt0 = hd * TPH;
                        on[qt][(nt0 + t) >> 1].w[((nt0 + t) & 1) * 2] = bpack2<DT>(o[0], o[1]);
                        on[qt][(nt0 + t) >> 1].w[((nt0 + t) & 1) * 2 + 1] = bpack2<DT>(o[2], o[3]);
                    }
                }
            };
            // ---- packed q|k|v projection, head-major; a head's attention behind the stage that completes it ----
            static_for<0, HP>([&](auto hp_) __attribute__((always_inline)) {
                constexpr int hp = decltype(hp_)::value;
                f32x4 acc[2][RT];
                const float* lb = lv + 2 * DH * hp;
                constexpr int par = hp * PST;            // (nine stages a pair at d = 192: the second one's parities are the other way round)
                static_for<0, PST>([&](auto st_) __attribute__((always_inline)) {
                    constexpr int st = decltype(st_)::value;
                    f32x4 bias[2];
#pragma unroll
                    for (int ntl = 0; ntl < 2; ++ntl) {
                        const int j = 2 * st + ntl, hd = j / (3 * TPH), r = j % (3 * TPH), part = r / TPH, t = r % TPH;
                        bias[ntl] = (f32x4){0.f, 0.f, 0.f, 0.f};
                        if (part < 2) bias[ntl] = *reinterpret_cast<const f32x4*>(lb + (part == 0 ? G::BQ : G::BK) + DH * hd + 16 * t + 4 * g);
                    }
                    stage(std::integral_constant<int, (par + st) & 1 ? 2 : 1>(), [&](auto i_, const s16x8& w, auto&&) __attribute__((always_inline)) {
                        constexpr int i = decltype(i_)::value, burst = i / G::FB, ntl = i % G::FB / G::KB, c = burst * G::KB + i % G::KB;
                        constexpr int part = (2 * st + ntl) % (3 * TPH) / TPH;
                        static_for<0, part == 0 ? QT : RT>([&](auto rt_) __attribute__((always_inline)) {
                            constexpr int rt = decltype(rt_)::value;
                            if constexpr (part < 2) acc[ntl][rt] = DT::mfma32(w, hf[rt][c].v, c == 0 ? bias[ntl] : acc[ntl][rt]);
                            else acc[ntl][rt] = DT::mfma32(hf[rt][c].v, w, c == 0 ? bias[ntl] : acc[ntl][rt]);       // V^T: operand roles swapped
                        });
                    }, idle);
                    static_for<0, 2>([&](auto ntl_) __attribute__((always_inline)) {
                        constexpr int ntl = decltype(ntl_)::value, j = 2 * st + ntl, hd = j / (3 * TPH), r = j % (3 * TPH), part = r / TPH, t = r % TPH;
#pragma unroll
                        for (int rt = 0; rt < (part == 0 ? QT : RT); ++rt) {
                            const uint2 pk = make_uint2(bpack2<DT>(acc[ntl][rt][0], acc[ntl][rt][1]), bpack2<DT>(acc[ntl][rt][2], acc[ntl][rt][3]));
                            if constexpr (part == 0) q[hd][rt][t] = pk;
                            else if constexpr (part == 1) *reinterpret_cast<uint2*>(kv + kat[rt] + 32 * t) = pk;
                            else {
                                *reinterpret_cast<u16*>(kv + (vat[rt][0] & 0xffff) + 1024 * t) = (u16)(pk.x & 0xffff);
                                *reinterpret_cast<u16*>(kv + (vat[rt][0] >> 16) + 1024 * t) = (u16)(pk.x >> 16);
                                *reinterpret_cast<u16*>(kv + (vat[rt][1] & 0xffff) + 1024 * t) = (u16)(pk.y & 0xffff);
                                *reinterpret_cast<u16*>(kv + (vat[rt][1] >> 16) + 1024 * t) = (u16)(pk.y >> 16);
                            }
                        }
                        if constexpr (r == 3 * TPH - 1) {
                            asm volatile("" ::: "memory");
                            attention(std::integral_constant<int, hd>(), lb + G::BV);
                            asm volatile("" ::: "memory");
                        }
                    });
                });
#pragma unroll
                for (int rt = 0; rt < QT; ++rt)
#pragma unroll
                    for (int c = 0; c < PCH; ++c) { of[rt][c] = of[rt][KC - PCH + c]; of[rt][KC - PCH + c] = on[rt][c]; }
            });
            static_assert(HP == 2 && KC == 2 * PCH, "two pairs of heads: the first one's output moves down as the second one's comes in");
            // ---- output projection onto the residual ----
            static_for<0, NT / 2>([&](auto st_) __attribute__((always_inline)) {
                constexpr int st = decltype(st_)::value;
                stage(std::integral_constant<int, (st & 1) ? 2 : 1>(), [&](auto i_, const s16x8& w, auto&&) __attribute__((always_inline)) {
                    constexpr int i = decltype(i_)::value, burst = i / G::FB, ntl = i % G::FB / G::KB, c = burst * G::KB + i % G::KB;
                    static_for<0, QT>([&](auto rt_) __attribute__((always_inline)) {
                        constexpr int rt = decltype(rt_)::value;
                        x[rt][2 * st + ntl] = DT::mfma32(w, of[rt][c].v, x[rt][2 * st + ntl]);
                    });
                }, idle);
            });
        };
        // FFN on the first QT row tiles: W1(0) even, then {W1(ch + 1) odd, W2(ch) even} ..., W2(last) odd; a chunk's activation behind
        // the MFMAs of the stages between (block_tail.h)
        auto ffn = [&](auto qt_, const Frags& hf, const float* lv) __attribute__((always_inline)) {
            constexpr int QT = decltype(qt_)::value;
            const int nch = a.F / 32;
            typedef f32x4 Acc[2][QT];
            typedef BFrag8 Hid[QT];
            Acc acc0, acc1;
            Hid hid0, hid1;
            f32x4 bias[2];
            auto load_bias = [&](int ch) __attribute__((always_inline)) {
#pragma unroll
                for (int ntl = 0; ntl < 2; ++ntl) bias[ntl] = *reinterpret_cast<const f32x4*>(lv + G::B1 + 32 * ch + 16 * ntl + 4 * g);
            };
            auto up = [&](Acc& ac) __attribute__((always_inline)) {
                return [&](auto i_, const s16x8& w, auto&& fill) __attribute__((always_inline)) {
                    constexpr int i = decltype(i_)::value, burst = i / G::FB, ntl = i % G::FB / G::KB, c = burst * G::KB + i % G::KB;
                    static_for<0, QT>([&](auto rt_) __attribute__((always_inline)) {
                        constexpr int rt = decltype(rt_)::value;
                        ac[ntl][rt] = DT::mfma32(w, hf[rt][c].v, c == 0 ? bias[ntl] : ac[ntl][rt]);
                        __builtin_amdgcn_sched_barrier(0);
                        fill(std::integral_constant<int, i * QT + rt>());
                        __builtin_amdgcn_sched_barrier(0);
                    });
                };
            };
            auto down = [&](Hid& hid) __attribute__((always_inline)) {
                return [&](auto i_, const s16x8& w, auto&& fill) __attribute__((always_inline)) {
                    constexpr int i = decltype(i_)::value;             // feature tile
                    static_for<0, QT>([&](auto rt_) __attribute__((always_inline)) {
                        constexpr int rt = decltype(rt_)::value;
                        x[rt][i] = DT::mfma32(w, hid[rt].v, x[rt][i]);
                        __builtin_amdgcn_sched_barrier(0);
                        fill(std::integral_constant<int, i * QT + rt>());
                        __builtin_amdgcn_sched_barrier(0);
                    });
                };
            };
            // a step: two values rounded and activated (the rounding does not see the sign: relu behind it is relu in front of it)
            constexpr int TOT = 4 * QT, NH = TOT / 2, NS = SF * QT;
            auto act_step = [&](auto k_, Acc& ac, Hid& hid) __attribute__((always_inline)) {
                constexpr int k = decltype(k_)::value, ntl = (k >> 1) & 1, rt = k >> 2, e = 2 * (k & 1);
                hid[rt].w[ntl * 2 + (k & 1)] = relu2<DT>(ac[ntl][rt][e], ac[ntl][rt][e + 1]);
            };
            auto act_slots = [&](auto lo_, auto hi_, Acc& ac, Hid& hid) __attribute__((always_inline)) {
                return [&](auto s_) __attribute__((always_inline)) {
                    constexpr int lo = decltype(lo_)::value, n = decltype(hi_)::value - lo, s = decltype(s_)::value;
                    static_for<lo + s * n / NS, lo + (s + 1) * n / NS>([&](auto k_) __attribute__((always_inline)) { act_step(k_, ac, hid); });
                };
            };
            typedef std::integral_constant<int, 0> K0; typedef std::integral_constant<int, NH> KH; typedef std::integral_constant<int, TOT> KT;
            // chunk ch's accumulators and hidden alternate with chunk ch + 1's: two chunks per round, nothing moves
            auto half = [&](int ch, Acc& ca, Hid& ha, Acc& na, Hid& hb) __attribute__((always_inline)) {
                stage(S2(), up(na), act_slots(KH(), KT(), ca, ha));        // W1(ch + 1); the second half of chunk ch's activation
                load_bias(ch + 2 < nch ? ch + 2 : 0);
                stage(S1(), down(ha), act_slots(K0(), KH(), na, hb));      // W2(ch); the first half of chunk ch + 1's
            };
            load_bias(0);
            stage(S1(), up(acc0), idle);
            load_bias(1);
            static_for<0, NH>([&](auto k_) __attribute__((always_inline)) { act_step(k_, acc0, hid0); });
            for (int ch = 0; ch + 2 < nch; ch += 2) { half(ch, acc0, hid0, acc1, hid1); half(ch + 1, acc1, hid1, acc0, hid0); }
            half(nch - 2, acc0, hid0, acc1, hid1);
            static_for<NH, TOT>([&](auto k_) __attribute__((always_inline)) { act_step(k_, acc1, hid1); });
            stage(std::integral_constant<int, QT == RT ? 2 : 0>(), down(hid1), idle);       // the final block's is the end of the pass
        };
        // the stream entering the final block: the rows, zeros for the dropped tokens
        auto store_stream = [&] __attribute__((always_inline)) {
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
                if (tok[rt] < T) {
                    u16* o = a.x_res + ((isb[rt] ? base_b : base_a) + tok[rt]) * D;
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) {
                        const f32x4 r = x[rt][nt];
                        *reinterpret_cast<uint2*>(o + 16 * nt + 4 * g) = make_uint2(bpack2<DT>(r[0], r[1]), bpack2<DT>(r[2], r[3]));
                    }
                }
            for (int e = 0; e < (two ? 2 : 1); ++e) {
                uint32_t out = ~(e ? mb : ma) & ((1u << (T - lead)) - 1u);
                while (out) {
                    const int t = lead + __builtin_ctz(out);
                    out &= out - 1;
                    u16* o = a.x_res + ((e ? base_b : base_a) + t) * D;
                    if (lane < D / 4) *reinterpret_cast<uint2*>(o + 4 * lane) = make_uint2(0, 0);
                }
            }
        };
        pipe.template admit<0>();
#pragma unroll
        for (int f = 0; f < NBUF - 1; ++f) wr[f] = pipe.frag(f, lane);
        auto layer = [&](int l, auto qt_) __attribute__((always_inline)) {        // the final block's queries, output projection and FFN are the first tile's
            const float* lv = reinterpret_cast<const float*>(vbuf + vp * vecb);
            fetch_vectors(l + 1 == nl ? 0 : l + 1);
            if (decltype(qt_)::value < RT && a.x_res) store_stream();
            {
                Frags hf;
                norm(hf, QA(), qt_, lv + G::LN1G, lv + G::LN1B, lv + G::BOUT);
                attention_block(hf, lv, qt_);
            }
            Frags hf;
            norm(hf, qt_, qt_, lv + G::LN2G, lv + G::LN2B, lv + G::b2(a.F));
            ffn(qt_, hf, lv);
            vp ^= 1;
        };
        for (int l = 0; l + 1 < nl; ++l) layer(l, QA());
        layer(nl - 1, Q1());
        if (tok[0] < lead) {                         // the first 2 lead rows
            u16* o = a.x_out + ((int64_t)(isb[0] ? eb : ea) * lead + tok[0]) * D;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const f32x4 r = x[0][nt];
                *reinterpret_cast<uint2*>(o + 16 * nt + 4 * g) = make_uint2(bpack2<DT>(r[0], r[1]), bpack2<DT>(r[2], r[3]));
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // no transfer into LDS may outlive the workgroup
    blk_barrier();
}

template <typename DT, int D, int DH>
int go(const BlocksPairArgs& a, hipStream_t st) {
    const size_t dyn = PairGeo<D, DH>::lds(a.F);
    if (dyn > (size_t)LDS_BUDGET || a.F % 64 != 0 || a.total_stages < PairRing<D>::SLOTS) return BSRL_UNSUPPORTED;
    auto kern = blocks_pair_kernel<DT, D, DH>;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)dyn) != hipSuccess) {
        (void)hipGetLastError();
        return BSRL_UNSUPPORTED;
    }
    hipLaunchKernelGGL(blocks_pairs_kernel<DT>, dim3((unsigned)a.plan.chunks), dim3(WAVE), 0, st, a.key_bias, a.pairs, a.plan.tiles, a.plan.B, a.T, a.lead);
    hipLaunchKernelGGL(kern, dim3((unsigned)a.plan.cus), dim3(256), dyn, st, a);
    BSRL_CHECK_LAUNCH("bsrl_blocks_pair");
    return BSRL_OK;
}

}  // namespace

int bsrl_blocks_pair(const BlocksPairArgs& a, int d, int dtype, hipStream_t st) {
    if (d != 192 || a.lead < 1 || a.lead > 5 || a.T <= a.lead || a.T - a.lead > 24 || a.n_layers < 1) return BSRL_UNSUPPORTED;
    if (a.plan.B <= 4 * (int64_t)a.plan.cus || a.plan.B > 0x7fffffffLL / 2) return BSRL_UNSUPPORTED;
    return dtype == BSRL_F16 ? go<F16, 192, 48>(a, st) : go<BF16, 192, 48>(a, st);
}
