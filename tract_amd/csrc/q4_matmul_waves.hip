// Q4_0 weights x more than a few f16 activation rows on the matrix cores, k shared among the waves of a workgroup: gfx950.
//
//   out[b, i, j] = sum_k act[b, i, k] * dequant(W[b / ratio, j, k]),   f16 activations and results
//
// The matrix-matrix arm of GgmlGemm (cuda/src/kernels/matmul/mod.rs:605-610) where q4_matmul.hip is not the right one: products
// of so few tiles that its workgroups leave compute units idle, and planes whose k is no multiple of its 64-feature chunks.
//
// Arithmetic: a code - 8 is one f16 number, so every product is exact.  A quantisation block (32 features, one
// v_mfma_f32_16x16x32_f16) is summed from zero in f32, its f16 scale multiplies the block's sum, and the blocks are added in
// f32, as the matrix-vector kernels do (q4_matmul.hip rounds every dequantised weight to f16 first; error against f64 2.6e-4
// there, 2.07e-4 here, all but the last rounding).
//
// A workgroup of 8 waves owns 16 MS (activation rows) x 16 NI (weight rows) of the result.  Its waves share k, not the
// tile: wave w takes units (4 blocks, a record of tiled weights) w, w + 8, ..  Both operands then go from memory straight
// into the registers that feed the instruction, without LDS and without a barrier; the eight sums are added through LDS at
// the end.  A launch is bound by a wave's own chain (first loads, one load latency per unit, the sums) while there is no
// more than a workgroup per compute unit, and by the conversions (11 operations per 8 codes, one per result and block) and
// the activations' way through the L2 beyond that, where q4_matmul.hip, which shares both in LDS, is the better one.
// Measured (us, before | now): 476 rows of 1000 x 2080 (planes, in groups of 8 rows) 444.6 | 15.4, 64 rows 51.2 | 7.5, 9 rows
// 10.3 | 7.2; tiles, q4_matmul.hip: 64 rows of 1024 x 4096 12.3 | 7.8, 128 rows 12.9 | 8.8; q4_tiled.hip: 9 rows of
// 4096 x 14336 18.4 | 13.6, 16 rows 23.1 | 18.3.
#include <hip/hip_runtime.h>
#include <string.h>
#include <type_traits>
#include "common.h"

namespace trocm {
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kW = 8;          // waves per workgroup
constexpr int kTile = 1152;    // bytes of a record of tiled weights (q4_tiled.hip)

struct MatMulWaves {
    const uint8_t *codes;     // planes: [w_batch, n, k/2]; tiles: [w_batch, n / 16, k / 128] records
    const uint16_t *scales;   // planes: [w_batch, n, k/32]
    const _Float16 *act;      // [act_batch, m, k]
    _Float16 *out;            // [act_batch, m, n]
    int n, k, m, ratio;       // ratio = act_batch / w_batch
};

__device__ __forceinline__ uint32_t perm(uint32_t hi, uint32_t lo, uint32_t sel) { return __builtin_amdgcn_perm(hi, lo, sel); }
__device__ __forceinline__ float f16_to_f32(uint32_t h) { return (float)__builtin_bit_cast(_Float16, (uint16_t)h); }

// Eight codes (elements e and 16 + e of a block in the nibbles of byte e) -> code - 8 as f16: 1024 + code (the code under the
// exponent byte 0x64) minus 1032 is exact.
__device__ __forceinline__ u32x4 codes_f16(uint32_t word) {
    const half2_t off = {(_Float16)1032.0f, (_Float16)1032.0f};
    u32x4 o;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const uint32_t c = h ? (word >> 4) & 0x0F0F0F0Fu : word & 0x0F0F0F0Fu;
        o[2 * h] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, perm(0x64646464u, c, 0x04010400u)) - off);
        o[2 * h + 1] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, perm(0x64646464u, c, 0x04030402u)) - off);
    }
    return o;
}
// DB: blocks of activations on their way (4, 2 where four have no registers)
template <int MS, int NI, int DB, bool TILED>
__global__ __launch_bounds__(64 * kW, 2) void q4_0_matmul_waves_kernel(MatMulWaves p) {
    constexpr int RW = 16 * NI + 4;   // floats per row of a wave's sums in LDS (4 rows apart: 16 banks)
    constexpr int PER_WAVE = 16 * MS * RW;
    constexpr int COPIES = PER_WAVE * kW * 4 <= 72 * 1024 ? kW : kW / 2;   // the waves' sums that LDS holds at once
    __shared__ __attribute__((aligned(16))) float lds[COPIES * PER_WAVE];

    const int tid = threadIdx.x, lane = tid & 63, row = lane & 15, grp = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n0 = blockIdx.x * 16 * NI, m0 = blockIdx.y * 16 * MS, b = blockIdx.z, wb = b / p.ratio;
    const int nb = p.k / 32, units = (nb + 3) / 4;

    // Lane (row, grp) contracts the block's features 4 grp .. + 3 and 16 + 4 grp .. + 3, the order of the records.  It loads
    // features 8 c .. 8 c + 7 with c = 0, 2, 1, 3 for grp 0 .. 3, whose halves two swaps between neighbouring groups put in
    // their places: one load takes 64 contiguous bytes of 16 rows.
    // Buffers: activation rows past m, and planes' blocks past the end of the matrix, read as zeros (the range check sees
    // the vector offset only); weight rows past n repeat the last ones, their results are not stored.
    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<_Float16 *>(p.act + (int64_t)b * p.m * p.k), 0, (uint32_t)((int64_t)p.m * p.k * 2), 0x00020000);
    const int64_t w_bytes = TILED ? (int64_t)(p.n / 16) * units * kTile : (int64_t)p.n * (p.k / 2);
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(p.codes + wb * w_bytes), 0, (uint32_t)w_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t s_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t *>(TILED ? nullptr : p.scales + (int64_t)wb * p.n * nb), 0, TILED ? 0u : (uint32_t)((int64_t)p.n * nb * 2), 0x00020000);
    uint32_t a_off[MS], w_off[NI], s_off[NI];
#pragma unroll
    for (int i = 0; i < MS; i++)
        a_off[i] = (uint32_t)(m0 + 16 * i + row) * (uint32_t)p.k * 2u + 16u * (((grp & 1) << 1) | (grp >> 1));
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int j = min(n0 + 16 * i + row, p.n - 1);
        if constexpr (TILED) {
            w_off[i] = (uint32_t)(j >> 4) * (uint32_t)units * kTile + 16u * (j & 15) + 256u * grp;
            s_off[i] = (uint32_t)(j >> 4) * (uint32_t)units * kTile + 1024 + 8u * (j & 15);
        } else {
            w_off[i] = (uint32_t)j * (uint32_t)(p.k / 2) + 4u * grp;
            s_off[i] = (uint32_t)j * (uint32_t)nb * 2u;
        }
    }

    struct Weights { uint32_t c[NI][4], s[NI][2]; };   // a unit: a word per block, the scales of its blocks
    struct Act { u32x4 x[MS]; };                       // a block
    auto load_w = [&](Weights &d, int u) {
#pragma unroll
        for (int i = 0; i < NI; i++) {
            if constexpr (TILED) {
                const u32x4 c = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, w_off[i], u * kTile, 0));
#pragma unroll
                for (int j = 0; j < 4; j++) d.c[i][j] = c[j];
                const u32x2 s = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(w_rsrc, s_off[i], u * kTile, 0));
                d.s[i][0] = s.x, d.s[i][1] = s.y;
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) d.c[i][j] = __builtin_amdgcn_raw_buffer_load_b32(w_rsrc, w_off[i] + 64u * u + 16 * j, 0, 0);
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const uint32_t lo = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(s_rsrc, s_off[i] + 8u * u + 4 * j, 0, 0);
                    const uint32_t hi = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(s_rsrc, s_off[i] + 8u * u + 4 * j + 2, 0, 0);
                    d.s[i][j] = lo | (hi << 16);
                }
            }
        }
    };
    auto load_a = [&](Act &d, int blk) {
#pragma unroll
        for (int i = 0; i < MS; i++) d.x[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, a_off[i], blk * 64, 0));
    };
    auto wave_block = [&](int u, int j) { return 4 * (u + (j >> 2) * kW) + (j & 3); };   // block j of this wave from unit u on

    f32x4 acc[MS][NI];
#pragma unroll
    for (int i = 0; i < MS; i++)
#pragma unroll
        for (int j = 0; j < NI; j++) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    // result register r of a lane: activation row 16 i + 4 grp + r of the workgroup's, weight row 16 j + row
    Weights wt, wt_next;
    Act ring[DB];
    int u = w;
    if (u < units) {
        load_w(wt_next, u);
#pragma unroll
        for (int j = 0; j < DB; j++)
            load_a(ring[j], min(wave_block(u, j), nb - 1));
    }
    for (; u < units; u += kW) {
        wt = wt_next;
        load_w(wt_next, min(u + kW, units - 1));
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int blk = 4 * u + j;
            if (!TILED && blk >= nb) break;
            __builtin_amdgcn_sched_barrier(0);   // (a block's fragments live only as long as the block)
            u32x4 a[MS];
            const Act &cur = ring[j % DB];
#pragma unroll
            for (int i = 0; i < MS; i++)
#pragma unroll
                for (int h = 0; h < 2; h++) {   // the odd groups' lower halves change places with the even groups' upper ones
                    const u32x2 s = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(cur.x[i][h], cur.x[i][2 + h], false, false));
                    a[i][h] = s.x, a[i][2 + h] = s.y;
                }
            load_a(ring[j % DB], min(wave_block(u, j + DB), nb - 1));   // (past this wave's last block: the last one again, unused)
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int jj = 0; jj < NI; jj++) {
                const half8_t cf = __builtin_bit_cast(half8_t, codes_f16(wt.c[jj][j]));
                const float d = f16_to_f32(wt.s[jj][j >> 1] >> (16 * (j & 1)));
                f32x4 sum[MS];
#pragma unroll
                for (int i = 0; i < MS; i++)
                    sum[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, a[i]), cf, f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
                for (int i = 0; i < MS; i++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[i][jj][r] = fmaf(sum[i][r], d, acc[i][jj][r]);
            }
        }
    }
    // ---- the eight sums, rows of RW floats in LDS, added in the order of the waves -------------------------------------
    auto write = [&](int at) {
#pragma unroll
        for (int i = 0; i < MS; i++)
#pragma unroll
            for (int j = 0; j < NI; j++)
#pragma unroll
                for (int r = 0; r < 4; r++) lds[at * PER_WAVE + (16 * i + 4 * grp + r) * RW + 16 * j + row] = acc[i][j][r];
    };
    if constexpr (COPIES < kW) {
        if (w >= COPIES) write(w - COPIES);
        __syncthreads();
        if (w < COPIES) {
#pragma unroll
            for (int i = 0; i < MS; i++)
#pragma unroll
                for (int j = 0; j < NI; j++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[i][j][r] += lds[w * PER_WAVE + (16 * i + 4 * grp + r) * RW + 16 * j + row];
            write(w);   // (read and written by the same thread)
        }
    } else {
        write(w);
    }
    __syncthreads();
    const int64_t out0 = (int64_t)b * p.m * p.n;
    const bool whole = p.n % 4 == 0;   // (then four consecutive results are all inside or all outside, and aligned)
    for (int e = tid; e < 16 * MS * 4 * NI; e += 64 * kW) {
        const int r = e / (4 * NI), c = e % (4 * NI) * 4, mi = m0 + r, ni = n0 + c;
        f32x4 sum = *reinterpret_cast<const f32x4 *>(&lds[r * RW + c]);
#pragma unroll
        for (int q = 1; q < COPIES; q++) sum += *reinterpret_cast<const f32x4 *>(&lds[q * PER_WAVE + r * RW + c]);
        if (mi >= p.m || ni >= p.n) continue;
        const int64_t at = out0 + (int64_t)mi * p.n + ni;
        _Float16 *o = p.out + at;
        const half4_t h = {(_Float16)sum[0], (_Float16)sum[1], (_Float16)sum[2], (_Float16)sum[3]};
        if (whole) *reinterpret_cast<half4_t *>(o) = h;
        else
            for (int x = 0; x < 4 && ni + x < p.n; x++) o[x] = h[x];
    }
}

struct Shape { int ms, ni; float tiled, first, later; };
// us of a round of workgroups, one per compute unit: tiles at 4096 features when there are several rounds; planes at 2080 features, the first
// and later ones.  16 x 64 is for tiles where it saves a second round.  32 x 16, 48 x 32 and 64 x 32 are for planes, whose codes come in words of 4 bytes, so that a weight row costs more there:
// 100 rows of 1000 x 2080 10.9 (16 x 32) -> 9.3 (32 x 16), 300 19.7 (32 x 64) -> 14.5 (48 x 32), 500 19.9 -> 15.4 (64 x 32).  32 x 64 is still
// the best where the others need one more round (150 rows of 3000 x 3104 25.8, 64 x 64 30.3).  144 products with planes, 9 to 500 rows, 250
// to 8200 weight rows, 544 to 14368 features: 0.93 of the time without these three, none longer.
constexpr float kNever = 1e9f;
constexpr Shape kShapes[] = {{1, 1, 5.0f, 7.3f, 6.0f},    {1, 2, 6.0f, 10.6f, 8.5f},    {2, 2, 10.0f, 12.4f, 10.5f},  {2, 4, 13.0f, 22.7f, 16.5f},
                             {4, 4, 20.0f, 23.0f, 20.0f}, {2, 1, kNever, 9.2f, 6.7f},   {3, 2, kNever, 14.5f, 12.5f}, {4, 2, kNever, 15.2f, 14.0f},
                             {1, 4, 9.0f, kNever, kNever}};
int64_t workgroups(const Shape &c, int64_t n, int64_t m, int64_t act_batch) {
    return (n + 16 * c.ni - 1) / (16 * c.ni) * ((m + 16 * c.ms - 1) / (16 * c.ms)) * act_batch;
}

}  // namespace

// Whether a product has so few tiles that this kernel's smallest shapes need no more than a workgroup per compute unit (us,
// q4_matmul.hip | here; inside the line: 128 rows of 1024 x 4096 12.9 | 8.8, 32 of 4096 x 4096 9.3 | 8.7; outside: 64 of
// 4096 x 4096 13.1 | 12.9, 200 of 1024 x 4096 13.2 | 13.1, 32 of 14336 x 4096 14.1 | 15.0).
// Tiles, up to 16 rows: also those of 16 x 64 (us, q4_tiled.hip | here: 9 rows of 14336 x 4096 10.8 | 10.1, 16 rows 11.7 | 10.8, of 9216 x 5120
// 21.2 | 11.5, of 14336 x 8192 22.9 | 18.6; 8 rows of 12288 x 4096 11.3 | 9.7, 10240 x 4096 11.2 | 9.2, 14336 x 4096 10.4 | 10.2, x 8192
// 16.7 | 17.2).
bool q4_0_matmul_waves_fits(int64_t n, int64_t m, int64_t act_batch, bool tiled) {
    const int64_t cus = num_compute_units();
    return workgroups(kShapes[1], n, m, act_batch) <= cus || (tiled && m <= 16 && workgroups(kShapes[8], n, m, act_batch) <= (m > 8 ? cus : 3 * cus / 4));
}

// 2 = not taken: operands beyond 32-bit offsets, misaligned ones.
int launch_q4_0_matmul_waves(const void *codes, const void *scales, int64_t w_batch, int64_t n, int64_t k, const void *act, int64_t act_batch,
                             int64_t m, void *out, hipStream_t s, int tiled) {
    if (m < 1 || n < 1 || k % 32 || (tiled && (n % 16 || k % 128))) return 2;
    if ((uintptr_t)codes % 16 || (uintptr_t)act % 16 || (uintptr_t)out % 8 || act_batch > 65535) return 2;
    if (n >= (1ll << 30) || m >= (1ll << 30) || k >= (1ll << 30)) return 2;
    if ((m + 64) * k >= (1ll << 30) || n * (k / 32) >= (1ll << 32) / 18 - 4096) return 2;
    MatMulWaves p;
    p.codes = (const uint8_t *)codes, p.scales = (const uint16_t *)scales;
    p.act = (const _Float16 *)act, p.out = (_Float16 *)out;
    p.n = (int)n, p.k = (int)k, p.m = (int)m, p.ratio = (int)(act_batch / w_batch);
    // The shape that takes the least time (1000 x 2080: 64 rows 16 x 16 7.9 us, 16 x 32 11.2; 200 rows 32 x 32 13.1, 16 x 32 19.7).  Below
    // 1024 features, where some waves have no unit (before | here: 9 rows of 4096 x 512 4.9 | 4.4, 128 rows 4.6 | 4.5, 16 rows of 320 x 992
    // 8.3 | 5.0).
    int best = 0;
    float best_us = 0.0f;
    for (int c = 0; c < 9; c++) {
        const Shape &x = kShapes[c];
        const float rounds = (float)((workgroups(x, n, m, act_batch) + num_compute_units() - 1) / num_compute_units());
        const float us = tiled ? rounds * x.tiled : x.first + (rounds - 1.0f) * x.later;
        if (c == 0 || us < best_us) best = c, best_us = us;
    }
    auto go = [&](auto ms, auto ni) -> int {
        constexpr int MS = decltype(ms)::value, NI = decltype(ni)::value, DB = MS < 4 ? 4 : 2;
        const dim3 grid((unsigned)((n + 16 * NI - 1) / (16 * NI)), (unsigned)((m + 16 * MS - 1) / (16 * MS)), (unsigned)act_batch);
        if (grid.y > 65535) return 2;
        constexpr bool TILES = !(NI == 1 && MS == 2) && !(NI == 2 && MS > 2), PLANES = !(MS == 1 && NI == 4);   // (the other's never chosen)
        if constexpr (TILES)
            if (tiled) hipLaunchKernelGGL((q4_0_matmul_waves_kernel<MS, NI, DB, true>), grid, dim3(64 * kW), 0, s, p);
        if constexpr (PLANES)
            if (!tiled) hipLaunchKernelGGL((q4_0_matmul_waves_kernel<MS, NI, DB, false>), grid, dim3(64 * kW), 0, s, p);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return fail("q4_0_matmul (shared k) launch failed: %s", hipGetErrorString(e));
        return 0;
    };
    typedef std::integral_constant<int, 1> I1;
    typedef std::integral_constant<int, 2> I2;
    typedef std::integral_constant<int, 3> I3;
    typedef std::integral_constant<int, 4> I4;
    switch (best) {
        case 0: return go(I1(), I1());
        case 1: return go(I1(), I2());
        case 2: return go(I2(), I2());
        case 3: return go(I2(), I4());
        case 4: return go(I4(), I4());
        case 5: return go(I2(), I1());
        case 6: return go(I3(), I2());
        case 7: return go(I4(), I2());
        default: return go(I1(), I4());
    }
}

}  // namespace trocm
