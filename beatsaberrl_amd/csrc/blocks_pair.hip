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
// 4096 800 / 704, 8192 1598 / 1374, 16384 2986 / 2565 (the rollout since the ring's loads are spread over the stages: 2618 -> 2550); up to 4 envs per CU, where one env per wave leaves half of the waves away,
// 328 / 379.  Narrower FFNs gain less and lose at F = d (blocks_pair.h).  At d = 128 the share of vector work is larger and two lost:
// 16384 envs, bf16, 828 / 928.
// Rows of a wave: lead tokens of A, lead tokens of B, A's attendable notes, B's; queries of the final block are then the first tile's.
// Everything row-wise does not care.  Attention does: its sums over keys run over the SLOTS of the full stream (a dropped token's is
// zero), which keeps their order and with it the bits.  A wave scatters K and V^T of the head that it has projected from its rows
// into the slots of their env, in LDS, and reads them back as fragments; a query tile that holds rows of both envs takes the scores
// against both and selects by lane - as it does the products with V, where a zero probability would not keep out an infinity.
// Envs are paired by rank, the i-th longest of 64 with the i-th shortest; two that do not fit 48 rows go alone.  Where that leaves too many
// alone, which only the device knows, this kernel steps aside for blocks_env_kernel or the other way round: both are launched, both ask
// blocks_pairs_pay.
// SAVE: the update's forward is this kernel too (note_train.h).  It leaves what the backward reads of a block, 4.6 KB a row, as it goes:
// 8.1 GB for 16384 envs at the recipe's shape, where the update's own forward had seven launches per block, each an HBM stream (4.8 ms beside
// the 2.4 of this kernel without SAVE).  3.65 - 3.9 ms in one launch, by the card, and its stream is not rounded between blocks.  2.9 of them are the arithmetic
// with every store taken out (LDS transposes, packing, addresses); the rest is the stores, which lie scattered over 40 000 rows at a time.
// Precision against 64 bits, error of this update over that of the one that computes its own stream, recipe shape, 36 draws of 2049 - 16384
// envs, both types: bin logits 0.87 (0.89 at most), all gradients 0.95 (a draw: 0.73 - 1.08; which units a rounding switches decides it).
// What the backward takes of a LayerNorm are the statistics of the fp32 row, in one pass: E[x^2] - mean^2 costs about (mean / deviation)^2 2^-24
// of the variance, the row's own rounding to 16 bits (mean / deviation) 2^-12 and more of a value.  Two passes over the stored row instead
// gave gradients equally far off (5.65e-3 for 5.63e-3, 6.735e-3 for 6.727e-3).
#include "block_stage.h"
#include "blocks_pair.h"

namespace {

constexpr int D = 192, DH = 48, RT = 3, ROWS = 16 * RT, CHUNK = BLOCKS_PAIR_CHUNK;

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
// what follows a stage: an even stage, with the stores that its admission does not wait for, an odd one, or nothing
template <int YOUNGER, int MORE = YOUNGER> struct Even { static constexpr bool follows = true, even = true; static constexpr int Y = YOUNGER, Z = MORE; };
struct Odd { static constexpr bool follows = true, even = false; };
struct Last { static constexpr bool follows = false; };
struct PairRing : StageRing<Geo<D>::SF, 7, 4> {};
struct PairGeo {
    static constexpr int KB = 32 * DH * 2, VB = DH * 64, ENV = KB + VB, WAVE_B = 2 * ENV;            // a head's K, V^T of an env, a wave's
    static constexpr int vec_bytes(int F) { return (Geo<D>::lv_size(F) * 4 + 1023) & ~1023; }
    static constexpr int PLACES = ROWS + 64;                                                         // SAVE: stream rows of a wave's rows and key slots
    static constexpr size_t lds(int F, bool save) { return 2 * vec_bytes(F) + 4 * WAVE_B + (size_t)PairRing::SLOTS * PairRing::STAGE_BYTES + (save ? 4 * PLACES * 4 : 0); }
};

// ---- SAVE: a block's operands, as the update's backward reads them --------------------------------------------------
// Rows go to their places in the update's compacted stream (note_train.hip) through buffer stores: a row without a token goes to row
// `rows`, past every buffer's end, which drops it without a branch.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
struct SaveBuf {
    __amdgpu_buffer_rsrc_t r;
    __device__ __forceinline__ SaveBuf(void* p, uint32_t bytes) : r(__builtin_amdgcn_make_buffer_rsrc(p, 0, (int)bytes, 0x27000)) {}
    // the quads of two feature tiles a, b (lane: 4 features of its row in each) as one 16-byte piece per lane: rows of lanes change
    // places so that a lane has eight features in a row, lanes of odd rows tile b's
    __device__ __forceinline__ void pair(uint32_t at, int soff, uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1) const {
        // (row_swap16 twice, behind one wait)
        asm("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3" : "+v"(a0), "+v"(b0), "+v"(a1), "+v"(b1));
        __builtin_amdgcn_raw_buffer_store_b128((u32x4){a0, a1, b0, b1}, r, (int)at, soff, 0);
    }
    __device__ __forceinline__ void quad(uint32_t at, int soff, uint32_t a0, uint32_t a1) const {
        __builtin_amdgcn_raw_buffer_store_b64((u32x2){a0, a1}, r, (int)at, soff, 0);
    }
    __device__ __forceinline__ void line(uint32_t at, int soff, const uint4& v) const {
        __builtin_amdgcn_raw_buffer_store_b128((u32x4){v.x, v.y, v.z, v.w}, r, (int)at, soff, 0);
    }
    __device__ __forceinline__ void one(uint32_t at, float v) const { __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, (int)at, 0, 0); }
};
// rows are fewer than 2^24 (bsrl_blocks_pair_saves); the row behind the last is past the buffer's end
__device__ __forceinline__ uint32_t save_at(uint32_t row, uint32_t pitch, uint32_t lane_part) { return __umul24(row, pitch) + lane_part; }

template <typename DT, bool SAVE>
__global__ __launch_bounds__(256, 1) void blocks_pair_kernel(BlocksPairArgs a, BlocksSave save) {
    typedef Geo<D> G;
    typedef PairRing R;
    typedef PairGeo P;
    constexpr int NT = G::NT, KC = G::KC, SF = G::SF, H = D / DH, TPH = DH / 16, NBUF = 4, LINES = D / 64;
    static_assert(H * DH == D && TPH == 3, "whole heads, of 32 features and 16");
    extern __shared__ float4 lds4[];                 // ring | K / V^T of the four waves | vectors of two blocks
    char* const lds = reinterpret_cast<char*>(lds4);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
    const int T = a.T, lead = a.lead, nl = a.n_layers, vecb = P::vec_bytes(a.F), lvn = G::lv_size(a.F);
    const float scale_l2e = 0.14433756729740644113f * 1.44269504088896340736f;        // log2(e) / sqrt(48)
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
                    pipe.template admit<0, 0, 0, true>();
                    pipe.template load_due_all<0>();
                    if (s == 0) fetch_vectors(l + 1 == nl ? 0 : l + 1);
                    pipe.template admit<1>();
                    pipe.template load_due_all<1>();
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
        // SAVE: stream rows of the wave's rows and of both envs' key slots, in LDS: eight registers more were spilled ones
        uint32_t* const place = reinterpret_cast<uint32_t*>(vbuf + 2 * vecb) + wave * P::PLACES;
        const uint32_t lp16 = (g & 1) * 32 + (g >> 1) * 16;                   // SaveBuf::pair's lane order
        if constexpr (SAVE) {
            const uint32_t first = (uint32_t)(a.plan.B * lead), oa = first + save.noff[ea], ob = first + save.noff[two ? eb : ea];
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
                const uint32_t own = isb[rt] ? (uint32_t)eb : (uint32_t)ea, note = (isb[rt] ? ob - na : oa) + 16 * rt + r16 - 2 * lead;
                place[16 * rt + r16] = tok[rt] >= T ? save.rows : tok[rt] < lead ? own * lead + tok[rt] : note;
            }
#pragma unroll
            for (int e = 0; e < 2; ++e)
#pragma unroll
                for (int kt = 0; kt < 2; ++kt) {
                    const int s = 16 * kt + r16, bit = s < lead ? 0 : s - lead;
                    const uint32_t m = e ? mb : ma, below = __popc(m & ((1u << bit) - 1u));
                    place[ROWS + 32 * e + s] = e && !two ? save.rows : s < lead ? (uint32_t)(e ? eb : ea) * lead + s : m >> bit & 1 ? (e ? ob : oa) + below : save.rows;
                }
            asm volatile("" ::: "memory");
        }
        auto clear_slots = [&] __attribute__((always_inline)) {            // slots of dropped tokens hold zeros
#pragma unroll
            for (int i = 0; i < P::WAVE_B / 1024; ++i) reinterpret_cast<uint4*>(kv)[i * 64 + lane] = make_uint4(0, 0, 0, 0);
            asm volatile("" ::: "memory");           // (stores and loads of other types follow: the order is the wave's program order)
        };
        // a row of the wave; in the final block, whose queries are lead tokens, theirs only
        auto row_at = [&](int row, bool final) __attribute__((always_inline)) {
            uint32_t r = place[row];
            asm("" : "+v"(r));                       // (a choice of values, not of addresses)
            return final && row >= 2 * lead ? save.rows : r;
        };
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
            if (!SAVE) clear_slots();                // (for the whole pass)
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

        // SAVE: what a wave stores, dealt behind the MFMAs of the stages of a block (0 .. 17 q|k|v, 18 .. 23 output projection, then the FFN's): the
        // rows that a LayerNorm reads where it reads them (LN), its output in the stages behind it, a head's q in the one behind it, its
        // k and v behind its attention, attention's output, the hidden in W2's.  Stores retire in order with the ring's loads, and the
        // admission of stage s, in stage s - 1, waits for loads issued up to fragment 6 of stage s - 4: it need not wait for the stores of the
        // two stages since, nor for a LayerNorm's between them.  None of them is conditional.
        constexpr auto stored = [](int s, int tiles) {
            constexpr int Q = 2, KV = 16;
            const int t = s < 2 ? RT : tiles, first = (LINES * t + 2) / 2 - 2, all = 2 * LINES * t;           // (Rows' steps of the first stage of two; the first two of them store nothing)
            return s == 0 || s == 19 ? 2 * (first > 0 ? first : 0) : s == 1 || s == 20 ? all - 2 * (first > 0 ? first : 0) : s == 24 ? all
                 : s == 2 || s == 7 || s == 11 || s == 16 ? Q * tiles : s == 5 || s == 9 || s == 14 || s == 18 ? KV : 0;
        };
        constexpr auto younger = [stored](int s, int tiles) {
            constexpr int LN = 2 + 2 * LINES;
            int n = s == 2 ? RT * LN : s == 26 ? tiles * LN : 0;
            for (int i = s - 3; i <= s - 2; ++i) n += i < 0 ? 0 : stored(i, tiles);
            return n;
        };
        // slot i's share of n steps over a stage of `slots`
        auto deal = [&](auto i_, auto slots_, auto n_, auto&& step) __attribute__((always_inline)) {
            constexpr int n = decltype(n_)::value, i = decltype(i_)::value, slots = decltype(slots_)::value;
            if constexpr (SAVE) static_for<i * n / slots, (i + 1) * n / slots>(step);
        };
        // Rows leave as whole 128-byte lines: a row tile's 64 columns go through LDS (the wave's K / V^T, whenever no head lies there), from where
        // eight lanes take a row's line.  In the accumulators' order a lane's 16 bytes have 48 others of the line three lane rows away, and
        // the vector cache passes on a request per 64 bytes at the rate of one per 128: 2.4 TB/s chip-wide whatever else goes on, 4.7 with whole lines.
        constexpr int LP = 144;                      // row pitch in LDS
        uint4 line[2];
        uint32_t lrow[2];
        auto line_put = [&](int rt, int at, const uint2& q) __attribute__((always_inline)) { *reinterpret_cast<uint2*>(kv + (16 * rt + r16) * LP + at + 8 * g) = q; };
        auto line_get = [&](int rt, bool final) __attribute__((always_inline)) {
            asm volatile("" ::: "memory");           // (what was put, in another type, by other lanes of the wave)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                line[h] = *reinterpret_cast<const uint4*>(kv + (16 * rt + 8 * h + (lane >> 3)) * LP + (lane & 7) * 16);
                lrow[h] = row_at(16 * rt + 8 * h + (lane >> 3), final);
            }
            asm volatile("" ::: "memory");
        };
        auto line_store = [&](u16* to, uint32_t pitch, int soff) __attribute__((always_inline)) {
#pragma unroll
            for (int h = 0; h < 2; ++h) SaveBuf(to, save.rows * pitch).line(save_at(lrow[h], pitch, (lane & 7) * 16), soff, line[h]);
        };
        // step k of rows of 16-bit fragments: (line, row tile) k into LDS, k - 1 out of it, k - 2 to its place
        auto save_rows = [&](auto k_, auto tiles_, u16* to, const auto& f, bool final) __attribute__((always_inline)) {
            constexpr int k = decltype(k_)::value, tiles = decltype(tiles_)::value, n = LINES * tiles;
            if constexpr (k >= 2) line_store(to, 2 * D, 128 * ((k - 2) / tiles));
            if constexpr (k >= 1 && k - 1 < n) line_get((k - 1) % tiles, final);
            if constexpr (k < n) {
                constexpr int rt = k % tiles, c = 2 * (k / tiles);
                line_put(rt, 0, f[rt][c].h[0]); line_put(rt, 32, f[rt][c].h[1]); line_put(rt, 64, f[rt][c + 1].h[0]); line_put(rt, 96, f[rt][c + 1].h[1]);
            }
        };
        // one stage: fragment i + 3 is requested before fragment i's MFMAs.  next: what follows
        // (Even, Odd, Last); mm(i, fragment, fill): its MFMAs; fill(k): the vector work behind the k-th (block_tail.h)
        s16x8 wr[NBUF];
        auto stage = [&](auto next, auto&& mm, auto&& fill, bool more = false) __attribute__((always_inline)) {
            static_for<0, SF>([&](auto i_) __attribute__((always_inline)) {
                constexpr int i = decltype(i_)::value, n = i + NBUF - 1;
                if constexpr (n < SF) wr[n % NBUF] = pipe.frag(n, lane);
                else if constexpr (decltype(next)::follows) {
                    if constexpr (n == SF) {
                        if constexpr (decltype(next)::even) {
                            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                            pipe.template admit<0, SAVE ? decltype(next)::Y : 0, SAVE ? decltype(next)::Z : 0, true>(more);
                        } else pipe.template admit<1>();
                    }
                    wr[n % NBUF] = pipe.frag(n - SF, lane);              // (behind the last stage: read, not used)
                }
                __builtin_amdgcn_sched_barrier(0);
                mm(i_, wr[i % NBUF], fill);
                // its share of the ring's loads, all before the admission above (fragment SF - NBUF + 1)
                if constexpr (i % 3 == 0 && i / 3 < R::FPW) pipe.template load_due<std::is_same<decltype(next), Odd>::value ? 0 : 1, i / 3>();
                __builtin_amdgcn_sched_barrier(0);
            });
        };
        static_assert(SF % NBUF == 0 && 3 * (R::FPW - 1) < SF - NBUF + 1, "rotating fragment registers; loads ahead of the admission");
        auto idle = [](auto) __attribute__((always_inline)) {};

        typedef BFrag8 Frags[RT][KC];                // LayerNorm's output
        typedef std::integral_constant<int, 1> Q1; typedef std::integral_constant<int, RT> QA;
        // LayerNorm of the first row tiles -> operand fragments; the bias of what is added to the stream next goes in on the way
        // SAVE: its input rows, means and 1 / deviations to their places
        auto norm = [&](Frags& hf, auto tiles_, auto added_, const float* gptr, const float* bptr, const float* bias, u16* sx, float* sm, float* sr,
                        bool final) __attribute__((always_inline)) {
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
                if constexpr (SAVE) {
                    const uint32_t row = row_at(16 * rt + r16, final), at = save_at(g == 0 ? row : save.rows, 4, 0);
                    SaveBuf(sm, save.rows * 4).one(at, mean); SaveBuf(sr, save.rows * 4).one(at, rstd);
                }
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    const float4 gm = *reinterpret_cast<const float4*>(gptr + 16 * nt + 4 * g);
                    const float4 bt = *reinterpret_cast<const float4*>(bptr + 16 * nt + 4 * g);
                    f32x4 r = x[rt][nt];
                    hf[rt][nt >> 1].w[(nt & 1) * 2] = bpack2<DT>(fmaf(fmaf(r[0], rstd, shift), gm.x, bt.x), fmaf(fmaf(r[1], rstd, shift), gm.y, bt.y));
                    hf[rt][nt >> 1].w[(nt & 1) * 2 + 1] = bpack2<DT>(fmaf(fmaf(r[2], rstd, shift), gm.z, bt.z), fmaf(fmaf(r[3], rstd, shift), gm.w, bt.w));
                    if constexpr (SAVE) {
                        line_put(rt, 32 * (nt & 3), make_uint2(bpack2<DT>(r[0], r[1]), bpack2<DT>(r[2], r[3])));
                        if ((nt & 3) == 2 && nt > 4) line_store(sx, 2 * D, 32 * (nt - 6));
                        if ((nt & 3) == 3) line_get(rt, final);
                        if (nt == NT - 1) line_store(sx, 2 * D, 32 * (nt - 3));
                    }
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
        auto attention_block = [&](const Frags& hf, const float* lv, auto qt_, const BlocksSaveLayer& sl) __attribute__((always_inline)) {
            constexpr int QT = decltype(qt_)::value;
            constexpr bool final = QT < RT;
            uint2 q[2][QT][TPH];                     // Q fragments [head of the pair][row tile][feature tile]
            BFrag8 on[QT][PCH], of[QT][KC];          // the pair's output, all heads'
            // SAVE: k and v of the head that lies in LDS, by key slots; v without its bias, a constant per query that the softmax's gradient cancels.
            // Steps: 0 reads the first tile of slots, then k and v of tile i by turns, v's with the reads of the next
            uint32_t kvrow = 0;
            uint2 kq[TPH], vq[TPH];
            auto head_rows = [&](u16* p, int i, uint32_t rows) __attribute__((always_inline)) {
                return SaveBuf(p + (int64_t)i * rows * DH, rows * 2 * DH);
            };
            auto save_kv = [&](auto s_, auto head_) __attribute__((always_inline)) {
                constexpr int s = decltype(s_)::value, head = decltype(head_)::value, next = s / 2;
                if constexpr (s > 0) {
                    const SaveBuf b = head_rows(sl.qkv, (final ? 0 : H) + (s % 2 ? 0 : H) + head, save.rows);
                    const uint2* t = s % 2 ? kq : vq;
                    b.pair(save_at(kvrow, 2 * DH, lp16), 0, t[0].x, t[0].y, t[1].x, t[1].y);
                    b.quad(save_at(kvrow, 2 * DH, 8 * g) + 64, 0, t[2].x, t[2].y);
                }
                if constexpr (s % 2 == 0 && next < 4) {
                    constexpr int e = next / 2, kt = next % 2;
                    typedef short s16x4t __attribute__((ext_vector_type(4)));
                    typedef __attribute__((address_space(3))) s16x4t* lptr;
                    kvrow = place[ROWS + 32 * e + 16 * kt + r16];
#pragma unroll
                    for (int t = 0; t < TPH; ++t) {
                        kq[t] = *reinterpret_cast<const uint2*>(kv + e * P::ENV + (16 * kt + r16) * (DH * 2) + 8 * g + 32 * t);
                        // (a 16-lane group presents features 16 t + 4 g + 0..3 over the tile's 16 slots, a lane receives its slot's)
                        vq[t] = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                            (lptr)(kv + e * P::ENV + P::KB + (16 * t + 4 * g + (r16 >> 2)) * 64 + (((4 * kt + (r16 & 3)) ^ ((g & 1) << 2)) << 3))));
                    }
                }
            };
            auto save_q = [&](auto k_, auto head_) __attribute__((always_inline)) {          // step k: row tile k - 1, and the next one's rows
                constexpr int head = decltype(head_)::value, k = decltype(k_)::value;
                if constexpr (k > 0) {
                    const uint2* t = q[head & 1][k - 1];
                    const SaveBuf b = head_rows(sl.q, head, final ? (uint32_t)(a.plan.B * lead) : save.rows);
                    b.pair(save_at(kvrow, 2 * DH, lp16), 0, t[0].x, t[0].y, t[1].x, t[1].y);
                    b.quad(save_at(kvrow, 2 * DH, 8 * g) + 64, 0, t[2].x, t[2].y);
                }
                if constexpr (k < QT) kvrow = row_at(16 * k + r16, final);
            };
            // what is stored behind fragment i of stage s of the block (`stored`)
            auto save_behind = [&](auto s_, auto i_) __attribute__((always_inline)) {
                constexpr int s = decltype(s_)::value, i = decltype(i_)::value;
                typedef std::integral_constant<int, SF> Slots;
                typedef std::integral_constant<int, 2 * SF> Slots2;
                if constexpr (s < 2)
                    deal(std::integral_constant<int, SF * s + i>(), Slots2(), std::integral_constant<int, LINES * RT + 2>(),
                         [&](auto k_) __attribute__((always_inline)) { save_rows(k_, QA(), sl.h, hf, false); });
                else if constexpr (s == 2 || s == 7 || s == 11 || s == 16)
                    deal(i_, Slots(), std::integral_constant<int, QT + 1>(), [&](auto k_) __attribute__((always_inline)) { save_q(k_, std::integral_constant<int, s / 5>()); });
                else if constexpr (s == 5 || s == 9 || s == 14 || s == 18)
                    deal(i_, Slots(), std::integral_constant<int, 9>(), [&](auto k_) __attribute__((always_inline)) { save_kv(k_, std::integral_constant<int, (s - 4) / 4>()); });
                else if constexpr (s == 19 || s == 20)
                    deal(std::integral_constant<int, SF * (s - 19) + i>(), Slots2(), std::integral_constant<int, LINES * QT + 2>(),
                         [&](auto k_) __attribute__((always_inline)) { save_rows(k_, qt_, sl.att, of, final); });
            };
            // attention of the pair's head hd over the slots of both envs
            auto attention = [&](auto hp_, auto hd_, const float* bv_) __attribute__((always_inline)) {
                constexpr int hd = decltype(hd_)::value, head = 2 * decltype(hp_)::value + hd;
                BFrag8 kf[2][2]; BFrag4 k2[2][2];
#pragma unroll
                for (int e = 0; e < 2; ++e)
#pragma unroll
                    for (int kt = 0; kt < 2; ++kt) {
                        const char* p = kv + e * P::ENV + (16 * kt + r16) * (DH * 2) + 8 * g;
                        kf[e][kt].h[0] = *reinterpret_cast<const uint2*>(p); kf[e][kt].h[1] = *reinterpret_cast<const uint2*>(p + 32);
                        k2[e][kt].h = *reinterpret_cast<const uint2*>(p + 64);
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
                    q2.h = q[hd][qt][TPH - 1];
                    m[qt] = -INFINITY;
#pragma unroll
                    for (int kt = 0; kt < 2; ++kt) {
                        f32x4 sc[2];
#pragma unroll
                        for (int e = 0; e < 2; ++e) {
                            sc[e] = DT::mfma32(kf[e][kt].v, qf.v, (f32x4){0.f, 0.f, 0.f, 0.f});
                            // features 32..47 into their own accumulator, as in the other kernels
                            const f32x4 s2 = DT::mfma16(k2[e][kt].v, q2.v, (f32x4){0.f, 0.f, 0.f, 0.f});
#pragma unroll
                            for (int i = 0; i < 4; ++i) sc[e][i] += s2[i];
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
                constexpr int par = hp * PST;            // (nine stages a pair: the second one's parities are the other way round)
                static_for<0, PST>([&](auto st_) __attribute__((always_inline)) {
                    constexpr int st = decltype(st_)::value;
                    f32x4 bias[2];
#pragma unroll
                    for (int ntl = 0; ntl < 2; ++ntl) {
                        const int j = 2 * st + ntl, hd = j / (3 * TPH), r = j % (3 * TPH), part = r / TPH, t = r % TPH;
                        bias[ntl] = (f32x4){0.f, 0.f, 0.f, 0.f};
                        if (part < 2) bias[ntl] = *reinterpret_cast<const f32x4*>(lb + (part == 0 ? G::BQ : G::BK) + DH * hd + 16 * t + 4 * g);
                    }
                    constexpr int s = par + st;
                    stage(std::conditional_t<s % 2 == 1, Even<younger(s + 1, QT)>, Odd>(), [&](auto i_, const s16x8& w, auto&&) __attribute__((always_inline)) {
                        constexpr int i = decltype(i_)::value, burst = i / G::FB, ntl = i % G::FB / G::KB, c = burst * G::KB + i % G::KB;
                        constexpr int part = (2 * st + ntl) % (3 * TPH) / TPH;
                        static_for<0, part == 0 ? QT : RT>([&](auto rt_) __attribute__((always_inline)) {
                            constexpr int rt = decltype(rt_)::value;
                            if constexpr (part < 2) acc[ntl][rt] = DT::mfma32(w, hf[rt][c].v, c == 0 ? bias[ntl] : acc[ntl][rt]);
                            else acc[ntl][rt] = DT::mfma32(hf[rt][c].v, w, c == 0 ? bias[ntl] : acc[ntl][rt]);       // V^T: operand roles swapped
                        });
                        if constexpr (SAVE) { __builtin_amdgcn_sched_barrier(0); save_behind(std::integral_constant<int, s>(), i_); }
                    }, idle);
                    if constexpr (SAVE && s == 1) {          // the block's first K: lines have been where dropped tokens' zeros belong
                        asm volatile("" ::: "memory");
                        clear_slots();
                    }
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
                            attention(hp_, std::integral_constant<int, hd>(), lb + G::BV);
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
                constexpr int s = HP * PST + st;
                stage(std::conditional_t<s % 2 == 1, Even<younger(s + 1, QT)>, Odd>(), [&](auto i_, const s16x8& w, auto&&) __attribute__((always_inline)) {
                    constexpr int i = decltype(i_)::value, burst = i / G::FB, ntl = i % G::FB / G::KB, c = burst * G::KB + i % G::KB;
                    static_for<0, QT>([&](auto rt_) __attribute__((always_inline)) {
                        constexpr int rt = decltype(rt_)::value;
                        x[rt][2 * st + ntl] = DT::mfma32(w, of[rt][c].v, x[rt][2 * st + ntl]);
                    });
                    if constexpr (SAVE) { __builtin_amdgcn_sched_barrier(0); save_behind(std::integral_constant<int, s>(), i_); }
                }, idle);
            });
        };
        // FFN on the first QT row tiles: W1(0) even, then {W1(ch + 1) odd, W2(ch) even} ..., W2(last) odd; a chunk's activation behind
        // the MFMAs of the stages between (block_tail.h)
        auto ffn = [&](auto qt_, const Frags& hf, const float* lv, u16* sh2, u16* sh) __attribute__((always_inline)) {
            constexpr int QT = decltype(qt_)::value;
            // chunks 2 i and 2 i + 1 make a line: the odd one's stage stores both
            auto save_hidden = [&](auto s_, auto odd_, int ch, const BFrag8 (&hid)[QT]) __attribute__((always_inline)) {
                constexpr int odd = decltype(odd_)::value;
                deal(s_, std::integral_constant<int, SF * QT>(), std::integral_constant<int, odd ? 2 * QT + 1 : QT>(), [&](auto k_) __attribute__((always_inline)) {
                    constexpr int k = decltype(k_)::value;
                    if constexpr (k < QT) { line_put(k, 64 * odd, hid[k].h[0]); line_put(k, 64 * odd + 32, hid[k].h[1]); }
                    else {
                        if constexpr (k > QT) line_store(sh, 2 * a.F, 64 * (ch - 1));
                        if constexpr (k < 2 * QT) line_get(k - QT, QT < RT);
                    }
                });
            };
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
            typedef std::integral_constant<int, 0> K0; typedef std::integral_constant<int, 1> K1; typedef std::integral_constant<int, NH> KH; typedef std::integral_constant<int, TOT> KT;
            // chunk ch's accumulators and hidden alternate with chunk ch + 1's: two chunks per round, nothing moves
            // (an admission among them has the stores of one odd chunk behind it: of stage s - 2, or of s - 4 behind its loads; the second
            // one has as many of h2's)
            static_assert(SF * QT * (QT + 2) / (2 * QT + 1) >= 7 * QT, "the hidden's stores behind fragment 6");
            auto half = [&](auto odd_, int ch, Acc& ca, Hid& ha, Acc& na, Hid& hb) __attribute__((always_inline)) {
                stage(Even<2 * QT, younger(26, QT)>(), up(na), act_slots(KH(), KT(), ca, ha), ch == 0);        // W1(ch + 1); the second half of chunk ch's activation
                load_bias(ch + 2 < nch ? ch + 2 : 0);
                const auto act = act_slots(K0(), KH(), na, hb);
                stage(Odd(), down(ha), [&](auto s_) __attribute__((always_inline)) { act(s_); save_hidden(s_, odd_, ch, ha); });      // W2(ch); the first half of chunk ch + 1's
            };
            load_bias(0);
            stage(Odd(), up(acc0), [&](auto s_) __attribute__((always_inline)) {
                deal(s_, std::integral_constant<int, SF * QT>(), std::integral_constant<int, LINES * QT + 2>(), [&](auto k_) __attribute__((always_inline)) {
                    save_rows(k_, qt_, sh2, hf, QT < RT);
                });
            });
            load_bias(1);
            static_for<0, NH>([&](auto k_) __attribute__((always_inline)) { act_step(k_, acc0, hid0); });
            for (int ch = 0; ch + 2 < nch; ch += 2) { half(K0(), ch, acc0, hid0, acc1, hid1); half(K1(), ch + 1, acc1, hid1, acc0, hid0); }
            half(K0(), nch - 2, acc0, hid0, acc1, hid1);
            static_for<NH, TOT>([&](auto k_) __attribute__((always_inline)) { act_step(k_, acc1, hid1); });
            stage(std::conditional_t<QT == RT, Even<2 * QT>, Last>(), down(hid1), [&](auto s_) __attribute__((always_inline)) { save_hidden(s_, K1(), nch - 1, hid1); });       // the final block's is the end of the pass
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
        pipe.template admit<0, 0, 0, true>();
#pragma unroll
        for (int f = 0; f < NBUF - 1; ++f) wr[f] = pipe.frag(f, lane);
        auto layer = [&](int l, auto qt_) __attribute__((always_inline)) {        // the final block's queries, output projection and FFN are the first tile's
            const float* lv = reinterpret_cast<const float*>(vbuf + vp * vecb);
            fetch_vectors(l + 1 == nl ? 0 : l + 1);
            if (decltype(qt_)::value < RT && a.x_res) store_stream();
            const BlocksSaveLayer& sl = save.blk[SAVE ? l : 0];
            {
                Frags hf;
                norm(hf, QA(), qt_, lv + G::LN1G, lv + G::LN1B, lv + G::BOUT, sl.x, sl.mean1, sl.rstd1, false);
                attention_block(hf, lv, qt_, sl);
            }
            Frags hf;
            norm(hf, qt_, qt_, lv + G::LN2G, lv + G::LN2B, lv + G::b2(a.F), sl.xm, sl.mean2, sl.rstd2, decltype(qt_)::value < RT);
            ffn(qt_, hf, lv, sl.h2, sl.hid);
            vp ^= 1;
        };
        for (int l = 0; l + 1 < nl; ++l) layer(l, QA());
        layer(nl - 1, Q1());
        if (tok[0] < lead) {                         // the first 2 lead rows
            const int64_t at = ((int64_t)(isb[0] ? eb : ea) * lead + tok[0]) * D + 4 * g;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const f32x4 r = x[0][nt];
                const uint2 q = make_uint2(bpack2<DT>(r[0], r[1]), bpack2<DT>(r[2], r[3]));
                *reinterpret_cast<uint2*>(a.x_out + at + 16 * nt) = q;
                if constexpr (SAVE) *reinterpret_cast<uint2*>(save.lead + at + 16 * nt) = q;
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // no transfer into LDS may outlive the workgroup
    blk_barrier();
}

template <typename DT, bool SAVE>
int go(const BlocksPairArgs& a, const BlocksSave& save, hipStream_t st) {
    const size_t dyn = PairGeo::lds(a.F, SAVE);
    if (dyn > (size_t)LDS_BUDGET || a.F % 64 != 0 || a.total_stages < PairRing::SLOTS) return BSRL_UNSUPPORTED;
    auto kern = blocks_pair_kernel<DT, SAVE>;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)dyn) != hipSuccess) {
        (void)hipGetLastError();
        return BSRL_UNSUPPORTED;
    }
    hipLaunchKernelGGL(blocks_pairs_kernel<DT>, dim3((unsigned)a.plan.chunks), dim3(WAVE), 0, st, a.key_bias, a.pairs, a.plan.tiles, a.plan.B, a.T, a.lead);
    hipLaunchKernelGGL(kern, dim3((unsigned)a.plan.cus), dim3(256), dyn, st, a, save);
    BSRL_CHECK_LAUNCH("bsrl_blocks_pair");
    return BSRL_OK;
}

}  // namespace

int bsrl_blocks_pair(const BlocksPairArgs& a, int d, int dtype, hipStream_t st) {
    if (d != D || a.lead < 1 || a.lead > 5 || a.T <= a.lead || a.T - a.lead > 24 || a.n_layers < 1) return BSRL_UNSUPPORTED;
    if (a.plan.B <= 4 * (int64_t)a.plan.cus || a.plan.B > 0x7fffffffLL / 2) return BSRL_UNSUPPORTED;
    if (!blocks_pairs_pay(a.plan, (a.plan.B + 7) / 8)) return BSRL_UNSUPPORTED;      // not even with every env in a pair
    return dtype == BSRL_F16 ? go<F16, false>(a, {}, st) : go<BF16, false>(a, {}, st);
}

bool bsrl_blocks_pair_saves(int64_t B, int d, int heads, int F, int T, int cus) {
    // Up to 8 envs per CU the update computes its own stream, whose bits are the op-by-op update's.  That line is one of bits: the saving
    // stack is the faster on both sides of it.  Update at the recipe's shape, f16, ms, own stream / this: 512 envs 1.88 / 1.84, 1025 2.60 / 2.10,
    // 2048 3.34 / 2.72, 2049 3.75 / 3.11, 4096 5.36 / 4.37, 16384 18.0 / 14.5; every note there, which leaves an env to a wave, 2049 4.42 / 3.87,
    // 16384 23.9 / 20.8; F = d, where the rollout takes the other kernel, 2049 3.00 / 2.50, with every note 3.41 / 3.07; one block 1.59 / 1.55.
    return d == D && heads == D / DH && F % 64 == 0 && PairGeo::lds(F, true) <= (size_t)LDS_BUDGET && B > 8 * (int64_t)cus &&
           B * T * 2 * (F > 3 * D ? F : 3 * D) < 0x7fffffffLL;           // (offsets past the end, 32 bits, are still past it)
}

int bsrl_blocks_pair_save(const BlocksPairArgs& a, const BlocksSave& save, int dtype, hipStream_t st) {
    if (a.lead < 1 || a.lead > 5 || a.T <= a.lead || a.T - a.lead > 24 || a.n_layers < 1 || a.n_layers > BSRL_MAX_LAYERS) return BSRL_UNSUPPORTED;
    BlocksPairArgs every = a;
    every.plan.env_ns = 0;                           // no other kernel runs the envs that this one would leave
    return dtype == BSRL_F16 ? go<F16, true>(every, save, st) : go<BF16, true>(every, save, st);
}
