// Pieces shared by the kernels that stream a weight image through LDS in stages of MFMA fragments: fragment geometry,
// the direct-to-LDS stage ring, packing helpers (blocks_fused.hip, ffn_rows.hip, block_tail.hip).
#pragma once
#include "bsrl_common.h"
#include <type_traits>

namespace {

template <typename DT> __device__ __forceinline__ uint32_t bpack2(float a, float b) {
    return DT::pack2(a, b);
}
template <> __device__ __forceinline__ uint32_t bpack2<F16>(float a, float b) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    f32x2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2));
}
template <> __device__ __forceinline__ uint32_t bpack2<BF16>(float a, float b) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    f32x2 v = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
union BFrag8 { s16x8 v; uint32_t w[4]; uint2 h[2]; uint4 u; };
union BFrag4 { s16x4 v; uint32_t w[2]; uint2 h; };

__device__ __forceinline__ void blk_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// compile-time loop: the body sees its index as a constant (the loop unroller gives up on the
// larger bodies, and register arrays indexed by the loop variable would then live in scratch)
template <int I, int N, typename Fn> __device__ __forceinline__ void static_for(Fn&& fn) {   // fn: an always_inline lambda
    if constexpr (I < N) { fn(std::integral_constant<int, I>{}); static_for<I + 1, N>(fn); }
}

template <int D> struct Geo {
    static constexpr int NT = D / 16, KC = D / 32, SF = 2 * KC;          // feature tiles, k chunks, fragments per stage
    // a stage is consumed in NB bursts of FB fragments (KB k chunks of both feature tiles): one burst of LDS
    // reads, then its MFMAs; bursts are sized to keep the fragment registers at 16-24 VGPRs
    static constexpr int NB = SF > 12 ? 4 : 2, FB = SF / NB, KB = KC / NB;
    static constexpr int STAGE_U2 = SF * 128;                             // uint2 per stage
    static constexpr int U2PT = STAGE_U2 / 512;                           // uint2 per thread per stage (2 or 3)
    __host__ __device__ static constexpr int layer_stages(int F) { return 3 * NT / 2 + NT / 2 + 2 * (F / 32); }
    // per-block fp32 vector region (floats)
    static constexpr int LN1G = 0, LN1B = D, BQ = 2 * D, BK = 3 * D, BV = 4 * D, BOUT = 5 * D, LN2G = 6 * D, LN2B = 7 * D, B1 = 8 * D;
    __host__ __device__ static constexpr int b2(int F) { return 8 * D + F; }
    __host__ __device__ static constexpr int lv_size(int F) { return 9 * D + F; }
};

__device__ __forceinline__ int bperm_k(int c, int gg, int j) { return 32 * c + 4 * gg + (j & 3) + (j >> 2) * 16; }
constexpr int LDS_BUDGET = 160 * 1024;

// m0 (the LDS base of the transfer) is written without telling the compiler, which rejects reserved registers in a
// clobber list: nothing else in the kernel uses it.  No "memory" clobber: what orders these asynchronous LDS writes
// against the fragment reads is the vmcnt wait + barrier of the stage admission.  The instruction's immediate offset
// moves BOTH addresses of a transfer, the global one and the LDS one: a wave's second fragment of a stage is the one
// right after its first and costs no further scalar work.
__device__ __forceinline__ void env_ring_load(uint32_t voff, const void* sbase, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "s"(lds_addr));
}
__device__ __forceinline__ void env_ring_load2(uint32_t voff, const void* sbase, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\tglobal_load_lds_dwordx4 %0, %1 offset:1024"
                 ::"v"(voff), "s"(sbase), "s"(lds_addr));
}
__device__ __forceinline__ void env_ring_load3(uint32_t voff, const void* sbase, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\tglobal_load_lds_dwordx4 %0, %1 offset:1024\n\t"
                 "global_load_lds_dwordx4 %0, %1 offset:2048" ::"v"(voff), "s"(sbase), "s"(lds_addr));
}

__device__ __forceinline__ void env_ring_load4(uint32_t voff, const void* sbase, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\tglobal_load_lds_dwordx4 %0, %1 offset:1024\n\t"
                 "global_load_lds_dwordx4 %0, %1 offset:2048\n\tglobal_load_lds_dwordx4 %0, %1 offset:3072" ::"v"(voff), "s"(sbase), "s"(lds_addr));
}

// The weight-stage ring of the one-wave-per-env kernels: stages of SF 1 KB fragments go global -> LDS directly, SLOTS
// stage slots deep.  Stages are entered in PAIRS (every block has an even number of them): one wait + barrier admits
// two stages and refills the two slots behind them, so all but those four slots may be in flight (AHEAD).  A loading
// wave moves FPW ADJACENT fragments of every stage (eight waves: SF = 8 one each; 12: six waves two each; 16: two each;
// four waves: 8: two each; 12: three each; 16: four each; 24: six each); image and ring are addressed by running byte offsets, no
// multiplies in the loop.
template <int SF_, int SLOTS_, int NW_ = 8> struct StageRing {
    static constexpr int NW = NW_, SF = SF_, SLOTS = SLOTS_, AHEAD = SLOTS - 4;
    static constexpr int FPW = (SF + NW - 1) / NW <= 1 ? 1 : SF % 2 == 0 && SF / 2 <= NW ? 2 : SF % 3 == 0 && SF / 3 <= NW ? 3 : SF % 4 == 0 && SF / 4 <= NW ? 4 : 6;
    static constexpr int NLW = SF / FPW;               // FPW = 6: two transfers of three (the immediate offset ends at 4095)
    static constexpr uint32_t STAGE_BYTES = SF * 1024;
    static_assert(SLOTS >= 5 && FPW * NLW == SF && NLW <= NW && FPW * (AHEAD + 2) < 64, "fragment split; vmcnt is 6 bits");
    const uint4* ring;             // slot 0
    const char* wsrc;              // this wave's fragments of stage 0
    uint32_t wdst;                 // ... and their place in slot 0 (LDS byte address)
    uint32_t voff;                 // lane * 16
    uint32_t src_off, src_end;     // next stage to load, image length (bytes)
    uint32_t cur, prev;            // slot of the current stage and of the one before it (bytes from slot 0)
    uint32_t due_slot[2], due_src[2];          // admit<.., SPREAD>: what the even and the odd stage of the pair have to load
    bool loader;

    __device__ __forceinline__ void issue(uint32_t slot_off) {
        if (NLW == NW || loader) {
            if constexpr (FPW == 6) {
                env_ring_load3(voff, wsrc + src_off, wdst + slot_off);
                env_ring_load3(voff, wsrc + src_off + 3072, wdst + slot_off + 3072);
            } else if constexpr (FPW == 4) env_ring_load4(voff, wsrc + src_off, wdst + slot_off);
            else if constexpr (FPW == 3) env_ring_load3(voff, wsrc + src_off, wdst + slot_off);
            else if constexpr (FPW == 2) env_ring_load2(voff, wsrc + src_off, wdst + slot_off);
            else env_ring_load(voff, wsrc + src_off, wdst + slot_off);
        }
        src_off = src_off + STAGE_BYTES == src_end ? 0 : src_off + STAGE_BYTES;
    }
    // SLOTS - 2 stages in flight (the host checks that the image is longer)
    __device__ __forceinline__ void start(const uint4* ring_, const void* img, int total_stages, int wave, int lane) {
        ring = ring_;
        wsrc = reinterpret_cast<const char*>(img) + wave * (FPW * 1024);
        wdst = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)const_cast<uint4*>(ring_) + wave * (FPW * 1024);
        voff = lane * 16;
        loader = wave < NLW;
        src_off = 0;
        src_end = (uint32_t)total_stages * STAGE_BYTES;
        cur = (SLOTS - 1) * STAGE_BYTES;
        prev = (SLOTS - 2) * STAGE_BYTES;
#pragma unroll
        for (int i = 0; i < SLOTS - 2; ++i) issue(i * STAGE_BYTES);
    }
    // transfer K (of FPW) of the stage that admit<.., SPREAD> left to the even (0) or odd stage of its pair
    template <int PARITY, int K> __device__ __forceinline__ void load_due() {
        static_assert(1024 * K < 4096, "the immediate offset ends at 4095");
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 offset:%3"
                     ::"v"(voff), "s"(wsrc + due_src[PARITY]), "s"(wdst + due_slot[PARITY]), "n"(1024 * K));
    }
    template <int PARITY> __device__ __forceinline__ void load_due_all() {
        static_for<0, FPW>([&](auto k) __attribute__((always_inline)) { load_due<PARITY, decltype(k)::value>(); });
    }
    // entry of the next stage (PARITY = its index in its block, mod 2): on return it is readable in slot `cur`.  YOUNGER: other memory
    // instructions that this wave has certainly issued since the loads that are waited for, which need not be waited for then; where `more`
    // holds, MORE of them.  SPREAD: the two stages behind are not requested here, where every wave's transfers meet in the 64 B/clk of the path
    // into LDS and hold the waves up (350 - 600 clk per pair at four waves and 12 KB stages), but one by one by the pair's own stages
    // (load_due; all of them before the next pair's admission).  blocks_pair.hip, 16384 envs: 2540 -> 2427 us; block_tail.h, where LDS reads
    // take 80 - 100 % of what the LDS gives, the same to 1 % slower, and stays as it was
    template <int PARITY, int YOUNGER = 0, int MORE = YOUNGER, bool SPREAD = false> __device__ __forceinline__ void admit(bool more = false) {
        const uint32_t older = prev;
        prev = cur;
        cur = cur + STAGE_BYTES == SLOTS * STAGE_BYTES ? 0 : cur + STAGE_BYTES;
        if constexpr (PARITY == 0) {
            // this wave's loads of this stage and the next have landed once at most the AHEAD younger stages' are
            // outstanding (loads retire in order; any other load or store in flight, or a wave that loads nothing,
            // only makes the wait stricter) ...
            static_assert(FPW * AHEAD + YOUNGER < 64 && FPW * AHEAD + MORE < 64, "vmcnt is 6 bits");
            // (the choice inside one statement: as a branch that the compiler sees it splits the stage, and its registers with it)
            if constexpr (MORE > YOUNGER)
                asm volatile("s_cmp_eq_u32 %0, 0\n\ts_cbranch_scc1 less%=\n\ts_waitcnt vmcnt(%2)\n\ts_branch done%=\nless%=:\n\ts_waitcnt vmcnt(%1)\ndone%=:"
                             ::"s"(__builtin_amdgcn_readfirstlane((int)more)), "n"(FPW * AHEAD + YOUNGER), "n"(FPW * AHEAD + MORE) : "memory", "scc");
            else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(FPW * AHEAD + YOUNGER) : "memory");
            blk_barrier();             // ... and every wave's have; every wave is done reading the two stages before this one
            if constexpr (SPREAD) {
                static_assert(NLW == NW, "every wave loads");
                due_slot[0] = older; due_slot[1] = prev;
#pragma unroll
                for (int i = 0; i < 2; ++i) { due_src[i] = src_off; src_off = src_off + STAGE_BYTES == src_end ? 0 : src_off + STAGE_BYTES; }
            } else {
                issue(older);
                issue(prev);
            }
        }
    }
    // fragment i of the current stage, this lane's 16 bytes
    __device__ __forceinline__ s16x8 frag(int i, int lane) const {
        return __builtin_bit_cast(s16x8, ring[(cur >> 4) + i * 64 + lane]);
    }
};
}  // namespace
