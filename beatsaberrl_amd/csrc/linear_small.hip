// y = act(x W^T + b) (+ residual) for problems that are latency, not throughput: up to a few thousand rows, where 128 x 128
// tiles leave most of the chip without a workgroup and a wave's chain of dependent loads is the kernel's time.
//
// A wave owns RT x CT MFMA tiles (16 rows x 16 columns each), a workgroup 4 waves; tiles shrink with the problem until the
// grid covers the chip (the host picks them).  Operand fragments come straight from global memory, PF k-chunks in flight: at
// K <= 32 PF every load of the wave is issued before its first MFMA, so the kernel is two memory round trips (operands,
// residual) and a launch.  16-bit: v_mfma_f32_16x16x32; fp32: four v_mfma_f32_16x16x4 per 16-byte fragment (k 4 g + j in the
// j-th one: both operands in the same order, fp32 products and sums throughout).
// Same arithmetic contract as the other linear kernels in 16 bit: fp32 accumulation in ascending chunks of 32 k, the same
// epilogue; a row's bits do not depend on the tile.
#include "linear_args.h"

namespace {

template <typename DT> struct Mma {
    static constexpr int KF = 32;                 // k per 16-byte fragment over the four lane groups
    static __device__ __forceinline__ f32x4 go(const s16x8& w, const s16x8& x, f32x4 c) { return DT::mfma32(w, x, c); }
    static __device__ __forceinline__ float ld(const void* p, int64_t i) { return DT::to_f(static_cast<const u16*>(p)[i]); }
    template <int ACT> static __device__ __forceinline__ float act(float v, bool f32) { return f32 ? apply_act<ACT>(v) : apply_act16<ACT>(v); }
};
template <> struct Mma<F32IO> {
    static constexpr int KF = 16;
    static __device__ __forceinline__ f32x4 go(const s16x8& w, const s16x8& x, f32x4 c) {
        const f32x4 a = __builtin_bit_cast(f32x4, w), b = __builtin_bit_cast(f32x4, x);
#pragma unroll
        for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], c, 0, 0, 0);
        return c;
    }
    static __device__ __forceinline__ float ld(const void* p, int64_t i) { return static_cast<const float*>(p)[i]; }
    template <int ACT> static __device__ __forceinline__ float act(float v, bool) { return apply_act<ACT>(v); }
};
template <typename DT> constexpr int elem_bytes() { return 2; }
template <> constexpr int elem_bytes<F32IO>() { return 4; }

// acc[column tile][row tile] of the wave tile at (row0, col0) -> y.  RF: the residual is fp32 (ACT_NONE alone; as a run-time switch
// it cost every other instance 1 % of a 16-bit small batch's forward)
template <typename DT, int ACT, bool RF, int RT, int CT>
__device__ __forceinline__ void small_epilogue(const LinArgs& a, int64_t rows, int64_t row0, int col0, int r16, int g, const f32x4 (&acc)[CT][RT]) {
    constexpr int ES = elem_bytes<DT>();
    // lane holds columns col .. col + 3 of its rows
    const bool f32out = ES == 4 || a.out_f32;
#pragma unroll
    for (int i = 0; i < CT; ++i) {
        const int col = col0 + i * 16 + g * 4;
        if (col >= a.M) continue;
        float bv[4] = {0.f, 0.f, 0.f, 0.f};
        if (a.bias) {
#pragma unroll
            for (int e = 0; e < 4; ++e) if (col + e < a.M) bv[e] = a.bias[col + e];
        }
#pragma unroll
        for (int j = 0; j < RT; ++j) {
            const int64_t row = row0 + j * 16 + r16;
            if (row >= rows) continue;
            float o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = keep_f32(Mma<DT>::template act<ACT>(acc[i][j][e] + bv[e], f32out));
            if (a.vec_ok) {               // M % 4 == 0, aligned rows, no split: 8- / 16-byte pieces
                if (a.res) {
                    if (ES == 4 || RF) {
                        const float4 r = *reinterpret_cast<const float4*>(static_cast<const float*>(a.res) + row * a.ldr + col);
                        o[0] += r.x; o[1] += r.y; o[2] += r.z; o[3] += r.w;
                    } else {
                        const uint2 r = *reinterpret_cast<const uint2*>(static_cast<const u16*>(a.res) + row * a.ldr + col);
                        const u16 h[4] = {(u16)(r.x & 0xffff), (u16)(r.x >> 16), (u16)(r.y & 0xffff), (u16)(r.y >> 16)};
#pragma unroll
                        for (int e = 0; e < 4; ++e) o[e] += Mma<DT>::ld(h, e);
                    }
                }
                if (a.gate) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) if (!(Mma<DT>::ld(a.gate, row * a.ldgate + col + e) > 0.f)) o[e] = 0.f;
                }
                if (f32out) *reinterpret_cast<float4*>(static_cast<float*>(a.y) + lin_yoff(a, row) + col) = make_float4(o[0], o[1], o[2], o[3]);
                else if constexpr (ES == 2) {
                    uint2 ov;
                    ov.x = DT::pack2(o[0], o[1]); ov.y = DT::pack2(o[2], o[3]);
                    *reinterpret_cast<uint2*>(static_cast<u16*>(a.y) + lin_yoff(a, row) + col) = ov;
                }
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int c = col + e;
                    if (c >= a.M) break;
                    float v = o[e];
                    if (a.res) v += RF ? static_cast<const float*>(a.res)[row * a.ldr + c] : Mma<DT>::ld(a.res, row * a.ldr + c);
                    if (a.gate && !(Mma<DT>::ld(a.gate, row * a.ldgate + c) > 0.f)) v = 0.f;
                    const bool second = a.y2 && c >= a.split;
                    void* dst = second ? a.y2 : a.y;
                    const int64_t off = second ? row * a.ldy2 + (c - a.split) : lin_yoff(a, row) + c;
                    if (f32out) static_cast<float*>(dst)[off] = v;
                    else if constexpr (ES == 2) static_cast<u16*>(dst)[off] = DT::from_f(v);
                }
            }
        }
    }
}

// WR wave rows x 4 / WR wave columns per workgroup
template <typename DT, int ACT, bool RF, int RT, int CT, int WR, int PF>
__global__ __launch_bounds__(256) void linear_small_kernel(LinArgs a, int ncb) {
    constexpr int ES = elem_bytes<DT>(), WC = 4 / WR, KF = Mma<DT>::KF, KL = KF / 4;       // KL: k per lane and fragment
    const int64_t rows = lin_rows(a);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int rb = blockIdx.x / ncb, cb = blockIdx.x - rb * ncb;
    const int64_t row0 = (int64_t)(rb * WR + wave / WC) * (RT * 16);
    const int col0 = (cb * WC + wave % WC) * (CT * 16);
    if (row0 >= rows || col0 >= a.M) return;
    const char* xp[RT]; const char* wp[CT];
#pragma unroll
    for (int t = 0; t < RT; ++t) {      // clamp instead of branching: rows and columns past the end are never stored
        int64_t r = row0 + 16 * t + r16; r = r < rows ? r : rows - 1;
        xp[t] = static_cast<const char*>(a.x) + (r * a.ldx + g * KL) * ES;
    }
#pragma unroll
    for (int t = 0; t < CT; ++t) {
        int c = col0 + 16 * t + r16; c = c < a.M ? c : a.M - 1;
        wp[t] = static_cast<const char*>(a.w) + ((int64_t)c * a.K + g * KL) * ES;
    }
    const int nk = (a.K + KF - 1) / KF;
    auto load = [&](const char* p, int kc) __attribute__((always_inline)) {
        s16x8 r = {0, 0, 0, 0, 0, 0, 0, 0};
        if (kc * KF + g * KL < a.K) r = *reinterpret_cast<const s16x8*>(p + kc * (KF * ES));      // K is a whole number of lane pieces
        return r;
    };
    f32x4 acc[CT][RT];
#pragma unroll
    for (int i = 0; i < CT; ++i)
#pragma unroll
        for (int j = 0; j < RT; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    s16x8 xf[PF][RT], wf[PF][CT];
#pragma unroll
    for (int s = 0; s < PF; ++s) {
#pragma unroll
        for (int t = 0; t < RT; ++t) xf[s][t] = load(xp[t], s);
#pragma unroll
        for (int t = 0; t < CT; ++t) wf[s][t] = load(wp[t], s);
    }
    for (int k0 = 0; k0 < nk; k0 += PF) {
#pragma unroll
        for (int s = 0; s < PF; ++s) {
            if (k0 + s < nk) {
#pragma unroll
                for (int i = 0; i < CT; ++i)
#pragma unroll
                    for (int j = 0; j < RT; ++j) acc[i][j] = Mma<DT>::go(wf[s][i], xf[s][j], acc[i][j]);
                if (k0 + s + PF < nk) {
#pragma unroll
                    for (int t = 0; t < RT; ++t) xf[s][t] = load(xp[t], k0 + s + PF);
#pragma unroll
                    for (int t = 0; t < CT; ++t) wf[s][t] = load(wp[t], k0 + s + PF);
                }
            }
        }
    }
    small_epilogue<DT, ACT, RF, RT, CT>(a, rows, row0, col0, r16, g, acc);
}

// The same tiles with the operands shared through LDS, for K a whole number of 128-byte pieces and enough rows that the
// direct kernel's redundant fragment loads are its time (16 bit, 2048 rows, 1536 -> 384: 226 MB through L1 for 7.9 MB of operands:
// 35 us against 14 here; 1024 rows, 960 -> 384 16 against 6.0; 97 rows, 384 -> 1536 5.5 against 4.0; fp32, 4096 rows, 128 -> 512
// 17 against 13, 128 -> 384 13 against 9).
// A workgroup is 2 x 2 waves of RT x CT tiles; each 1 KB operand block (8 rows x 128 B) goes global -> LDS by one wave
// instruction, NS - 1 stages of 128 bytes of k ahead, one barrier per stage (the layout and its swizzle: linear_ring.hip).
__device__ __forceinline__ void lds_block_load(uint32_t voff, const void* sbase, uint32_t lds_addr) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "s"(lds_addr));
}
template <typename DT, int ACT, bool RF, int RT, int CT, int NS>
__global__ __launch_bounds__(256, 2) void linear_lds_kernel(LinArgs a, int ncb) {
    constexpr int XB = 4 * RT, WB = 4 * CT, NB = XB + WB, NL = NB / 4;           // 1 KB blocks per stage, loads per wave
    constexpr int ES = elem_bytes<DT>();
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    extern __shared__ __attribute__((aligned(16))) u32x4 lds[];
    const int64_t rows = lin_rows(a);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, g = lane >> 4, wr = wave & 1, wc = wave >> 1;
    const int rb = blockIdx.x / ncb, cb = blockIdx.x - rb * ncb;
    const int64_t row0 = (int64_t)rb * (32 * RT);
    const int col0 = cb * (32 * CT);
    if (row0 >= rows) return;                       // uniform over the workgroup
    // this wave's blocks: block i holds rows (or weight rows) 8 i .. 8 i + 7 of the tile, lane -> (row lane / 8, k piece swizzled)
    const int lrow = lane >> 3, piece = (lane & 7) ^ lrow;
    uint32_t voff[NL]; const char* base[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        const int blk = wave * NL + i;
        if (blk < XB) {
            int64_t r = row0 + 8 * blk + lrow; r = r < rows ? r : rows - 1;
            voff[i] = (uint32_t)((r - row0) * a.ldx * ES + piece * 16);
            base[i] = static_cast<const char*>(a.x) + row0 * a.ldx * ES;
        } else {
            int c = col0 + 8 * (blk - XB) + lrow; c = c < a.M ? c : a.M - 1;
            voff[i] = (uint32_t)((c - col0) * a.K * ES + piece * 16);
            base[i] = static_cast<const char*>(a.w) + (int64_t)col0 * a.K * ES;
        }
    }
    const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char*)lds + wave * (NL * 1024);
    const int nsteps = a.K * ES / 128;
    auto issue = [&](int step) __attribute__((always_inline)) {
        const uint32_t sb = lds0 + (step % NS) * (NB * 1024);
#pragma unroll
        for (int i = 0; i < NL; ++i) lds_block_load(voff[i], base[i] + (int64_t)step * 128, sb + i * 1024);
    };
    f32x4 acc[CT][RT];
#pragma unroll
    for (int i = 0; i < CT; ++i)
#pragma unroll
        for (int j = 0; j < RT; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < NS - 1; ++s) if (s < nsteps) issue(s);
    auto rd = [&](int t, int c) __attribute__((always_inline)) { return (2 * t + (r16 >> 3)) * 64 + (r16 & 7) * 8 + ((4 * c + g) ^ (r16 & 7)); };
    for (int s = 0; s < nsteps; ++s) {
        // this wave's loads of step s have landed when only the younger steps' are outstanding; the barrier says so of the
        // others and that slot (s - 1) % NS is no longer read
        if (s + NS - 2 < nsteps) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NL * (NS - 2)) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (s + NS - 1 < nsteps) issue(s + NS - 1);
        const u32x4* st = lds + (s % NS) * (NB * 64);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            s16x8 xf[RT], wf[CT];
#pragma unroll
            for (int j = 0; j < RT; ++j) xf[j] = __builtin_bit_cast(s16x8, st[rd(wr * RT + j, c)]);
#pragma unroll
            for (int i = 0; i < CT; ++i) wf[i] = __builtin_bit_cast(s16x8, st[XB * 64 + rd(wc * CT + i, c)]);
#pragma unroll
            for (int i = 0; i < CT; ++i)
#pragma unroll
                for (int j = 0; j < RT; ++j) acc[i][j] = Mma<DT>::go(wf[i], xf[j], acc[i][j]);
        }
    }
    small_epilogue<DT, ACT, RF, RT, CT>(a, rows, row0 + wr * (16 * RT), col0 + wc * (16 * CT), r16, g, acc);
}
template <typename DT, int ACT, bool RF, int RT, int CT, int NS>
bool go_lds(const LinArgs& a, hipStream_t st) {
    constexpr int BYTES = NS * 4 * (RT + CT) * 1024;
    auto kern = linear_lds_kernel<DT, ACT, RF, RT, CT, NS>;
    static const bool ready = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, BYTES) == hipSuccess;
    if (!ready) { (void)hipGetLastError(); return false; }
    const int ncb = (a.M + 32 * CT - 1) / (32 * CT);
    hipLaunchKernelGGL(kern, dim3((unsigned)(((a.rows + 32 * RT - 1) / (32 * RT)) * ncb)), dim3(256), BYTES, st, a, ncb);
    return true;
}

template <typename DT, int ACT, bool RF, int RT, int CT, int WR, int PF>
void go(const LinArgs& a, hipStream_t st) {
    const int ncb = (a.M + CT * 16 * (4 / WR) - 1) / (CT * 16 * (4 / WR));
    const int64_t nrb = (a.rows + RT * 16 * WR - 1) / (RT * 16 * WR);
    hipLaunchKernelGGL((linear_small_kernel<DT, ACT, RF, RT, CT, WR, PF>), dim3((unsigned)(nrb * ncb)), dim3(256), 0, st, a, ncb);
}

template <typename DT, int ACT, bool RF = false>
void pick(const LinArgs& a, hipStream_t st) {
    const int64_t cus = bsrl_cus(), wg64 = ((a.rows + 63) / 64) * ((a.M + 63) / 64);
    if (a.K * elem_bytes<DT>() % 128 == 0 && a.rows > 16 && a.ldx <= (1 << 22) && a.K <= (1 << 22)) {
        // 32 x 32 tiles until 64 x 64 ones cover the chip, 64 x 128 once three of those per CU would queue
        if (wg64 >= 3 * cus ? go_lds<DT, ACT, RF, 2, 4, 3>(a, st) : wg64 >= cus ? go_lds<DT, ACT, RF, 2, 2, 4>(a, st)
                                                                                 : go_lds<DT, ACT, RF, 1, 1, 8>(a, st)) return;
    }
    // the largest tile that still gives every CU a workgroup: 64 x 64, 32 x 64, 32 x 32; one row tile: 16 x 64
    if (a.rows <= 16) go<DT, ACT, RF, 1, 1, 1, 12>(a, st);
    else if (wg64 >= cus) go<DT, ACT, RF, 2, 2, 2, 6>(a, st);
    else if (2 * wg64 >= cus) go<DT, ACT, RF, 1, 2, 2, 8>(a, st);
    else go<DT, ACT, RF, 1, 1, 2, 12>(a, st);
}
template <typename DT>
void by_act(const LinArgs& a, int act, hipStream_t st) {
    if (act == BSRL_ACT_RELU) pick<DT, BSRL_ACT_RELU>(a, st);
    else if (act == BSRL_ACT_GELU) pick<DT, BSRL_ACT_GELU>(a, st);
    else if constexpr (elem_bytes<DT>() == 2) { if (a.res_f32) pick<DT, BSRL_ACT_NONE, true>(a, st); else pick<DT, BSRL_ACT_NONE>(a, st); }
    else pick<DT, BSRL_ACT_NONE>(a, st);
}

}  // namespace

bool bsrl_linear_small(const LinArgs& a_, int act, int dtype, hipStream_t st) {
    const int es = dtype == BSRL_F32 ? 4 : 2, per = 16 / es;           // elements per 16-byte lane piece
    LinArgs a = a_;
    if (a.res_f32 && act != BSRL_ACT_NONE) return false;
    if (a.K % per != 0 || a.ldx % per != 0 || !bsrl_aligned(a.x, 16) || !bsrl_aligned(a.w, 16)) return false;
    if (((a.rows + 31) / 32) * (int64_t)((a.M + 31) / 32) > 0x3fffffff) return false;
    const int osz = a.out_f32 ? 4 : es;
    a.vec_ok = !a.y2 && a.M % 4 == 0 && a.ldy % 4 == 0 && a.y_gstride % 4 == 0 && bsrl_aligned(a.y, 4 * osz) &&
               (!a.res || (a.ldr % 4 == 0 && bsrl_aligned(a.res, a.res_f32 ? 16 : 4 * es))) && (!a.gate || (a.ldgate % 4 == 0 && bsrl_aligned(a.gate, 4 * es)));
    if (dtype == BSRL_F32) by_act<F32IO>(a, act, st);
    else if (dtype == BSRL_F16) by_act<F16>(a, act, st);
    else by_act<BF16>(a, act, st);
    return true;
}
