// Affine codes as the quantised caches of the reference form them (quant_dyn_kv_cache.rs:118-192; kv_quant.rs:105-236): shared by
// the stores' own kernels and the attention launch that takes a step's new token.  The codes are the same in every file that
// includes this, whether it is compiled with contraction or without: __fadd_rn and its like are plain operators here, so the
// functions turn contraction off themselves.
#pragma once
#include <hip/hip_fp16.h>
#include "common.h"

namespace trocm {
namespace {

// A value on its way into fminf / fmaxf: a signalling NaN is quieted first.  v_min_f32 / v_max_f32 answer NaN for a
// signalling one, and the next operation of the chain, which ignores that NaN, has then lost what came before it;
// f32::min / f32::max skip every NaN alike.
__device__ __forceinline__ float quiet(float x) { return __builtin_canonicalizef(x); }

// Exchanges between lanes on the vector ALU (DPP modifiers and the lane-swap instructions) instead of through the LDS
// crossbar (`__shfl_xor` = ds_bpermute_b32: the per-token ingest spent 14 of its 101 us on eight of those per lane).
template <int CTRL>
__device__ __forceinline__ float dpp_move(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, false));
}
// x of lane (l ^ M) for M = 8, 16, 32 combined with this lane's by OP (min or max): exact partners.
template <int M, typename Op>
__device__ __forceinline__ float xor_combine(float x, Op op) {
    static_assert(M == 8 || M == 16 || M == 32, "lane distances 8, 16, 32");
    if constexpr (M == 8) {
        return op(x, dpp_move<0x128>(x));                       // row_ror:8 within a row of 16 lanes
    } else {   // rows 2k and 2k + 1 (halves of the wave) trade places between the two results: one of them is this lane's own
        unsigned a = __builtin_bit_cast(unsigned, x), b = a;
        asm("" : "+v"(b));   // two registers: the instruction swaps in place, and both results are read
        const auto sw = M == 16 ? __builtin_amdgcn_permlane16_swap(a, b, false, false) : __builtin_amdgcn_permlane32_swap(a, b, false, false);
        unsigned s0 = sw[0], s1 = sw[1];
        asm("" : "+v"(s0), "+v"(s1));   // (this compiler folds op(sw[0], sw[1]) to sw[0] when both operands were one value: the minimum was lost)
        return op(__builtin_bit_cast(float, s0), __builtin_bit_cast(float, s1));
    }
}
// Minimum and maximum over aligned groups of N lanes (8, 16, 32, 64), left in every lane of the group.  (Any order of
// exchanges gives the same bits: both are exact.)  Quads, halves of a row and rows by DPP, then pairs of rows, then the
// two halves of the wave.
template <int N>
__device__ __forceinline__ void group_min_max(float &lo, float &hi) {
    static_assert(N == 8 || N == 16 || N == 32 || N == 64, "groups of 8, 16, 32 or 64 lanes");
    auto mn = [](float a, float b) { return fminf(a, b); };
    auto mx = [](float a, float b) { return fmaxf(a, b); };
    lo = fminf(lo, dpp_move<0xB1>(lo)), hi = fmaxf(hi, dpp_move<0xB1>(hi));       // quad_perm [1,0,3,2]
    lo = fminf(lo, dpp_move<0x4E>(lo)), hi = fmaxf(hi, dpp_move<0x4E>(hi));       // quad_perm [2,3,0,1]
    lo = fminf(lo, dpp_move<0x141>(lo)), hi = fmaxf(hi, dpp_move<0x141>(hi));     // row_half_mirror: the other quad of 8 lanes
    if constexpr (N >= 16) lo = fminf(lo, dpp_move<0x140>(lo)), hi = fmaxf(hi, dpp_move<0x140>(hi));   // row_mirror: the other half of the row
    if constexpr (N >= 32) lo = xor_combine<16>(lo, mn), hi = xor_combine<16>(hi, mx);
    if constexpr (N >= 64) lo = xor_combine<32>(lo, mn), hi = xor_combine<32>(hi, mx);
}

// f32::round(): half away from zero, as trunc(x + copysign(0.49999997, x)) (the float below 0.5; the sum rounds to
// nearest even, so an exact half ties up to the integer and anything less stays below it; exact for every float,
// checked exhaustively on the host for the exponents where it matters; inf and NaN pass through).
__device__ __forceinline__ float round_half_away(float x) {
#pragma clang fp contract(off)
    return truncf(__fadd_rn(x, __builtin_copysignf(0.49999997f, x)));
}

// ((x - lo) / scale).round().clamp(0.0, lv) as u8   (quant_dyn_kv_cache.rs:128, :190; kv_quant.rs:110, :219)
__device__ __forceinline__ uint32_t affine_code(float x, float lo, float scale, float lv) {
#pragma clang fp contract(off)
    float q = round_half_away(__fdiv_rn(__fsub_rn(x, lo), scale));
    if (!(q == q)) return 0;            // clamp keeps NaN, the cast turns it into 0
    q = q < 0.0f ? 0.0f : (q > lv ? lv : q);
    return (uint32_t)q;
}
__device__ __forceinline__ float affine_scale(float lo, float hi, float lv) {   // :127, :186
#pragma clang fp contract(off)
    return hi > lo ? __fdiv_rn(__fsub_rn(hi, lo), lv) : 1.0f;
}

}  // namespace
}  // namespace trocm
