// Q4_0 weights x more than a few f32 activation rows on the matrix cores: gfx950.
//
//   out[b, i, j] = sum_k act[b, i, k] * dequant(W[b / ratio, j, k]),   f32 activations and results
//
// The f32 side of the matrix-matrix arm of GgmlGemm (cuda/src/kernels/matmul/mod.rs:605-610).  Arithmetic: an activation is
// the sum of three bf16 numbers of 8 significant bits (x = b1 + b2 + b3 by truncation and exact remainders; exact from 2^-110
// on, below that within 2^-133), a code - 8 is one bf16 number, so every product of v_mfma_f32_*_bf16 is exact and its sums are
// f32.  A quantisation block (32 features) is summed from zero, smallest part first, its f16 scale multiplies the block's sum,
// and the blocks are added in f32.  Blocks with values that have no such three parts (`kBig` and more, infinities) are done in
// f32; planes' blocks also where a lane's values are so small that 2^-133 counts among them (tiled weights are split the same way
// by the kernel for few rows, q4_tiled.hip; the test costs 2 % of 150 rows of 4096 x 4096).
//
// A workgroup of 8 waves owns SUB MS (activation rows) x SUB NI (weight rows) of the result.  Its waves share k, not the
// tile: wave w takes units (4 blocks, a record of tiled weights) w, w + 8, ..  Both operands then go from memory straight
// into the registers that feed the instruction, without LDS and without a barrier; the eight sums are added through LDS at
// the end.  Eight short sums are also more exact than one long one (error against f64, 150 rows of 4096 features: 9.5e-8;
// in groups of 8 rows on the matrix-vector kernel 1.02e-7).
//
// What bounds it is the vector work around the instructions: per block, 6 operations per activation for the split, 2.1 per
// code to make it bf16, one per result for the scale, against three passes of the matrix cores.  Wider tiles share the
// split, which is what `launch_q4_0_matmul_f32` weighs against idle compute units.  Measured (us; before, in groups of
// 8 rows on q4_tiled.hip or q4_matvec.hip): 150 rows of 4096 x 4096 234.6 -> 26.4; 500 of 14336 x 4096 990.9 -> 216 (272
// TFLOP/s; the f32 matrix instruction's peak is 157); 200 of 4096 x 14336 856 -> 92; 9 of 4096 x 4096 18.6 -> 8.2 (launch,
// first loads and the final sum: about 5); 40 of 1000 x 2080, planes, 54.7 -> 7.9.
#include <hip/hip_runtime.h>
#include <string.h>
#include <type_traits>
#include <algorithm>
#include "common.h"

namespace trocm {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kW = 8;          // waves per workgroup
constexpr int kTile = 1152;    // bytes of a record of tiled weights (q4_tiled.hip)
constexpr float kBig = 0x1p118f;     // from here on a block's unscaled sum could overflow
constexpr float kSmall = 0x1p-100f;  // from here on what the split loses, 2^-133, is less than 2^-32 of the largest value

struct MatMulF32 {
    const uint8_t *codes;     // planes: [w_batch, n, k/2]; tiles: [w_batch, n / 16, k / 128] records
    const uint16_t *scales;   // planes: [w_batch, n, k/32]
    const float *act;         // [act_batch, m, k]
    float *out;               // [act_batch, m, n]
    int n, k, m, ratio;       // ratio = act_batch / w_batch
};

template <int SUB> struct AccOf;
template <> struct AccOf<16> { typedef f32x4 type; };
template <> struct AccOf<32> { typedef f32x16 type; };

__device__ __forceinline__ uint32_t perm(uint32_t hi, uint32_t lo, uint32_t sel) { return __builtin_amdgcn_perm(hi, lo, sel); }
__device__ __forceinline__ uint32_t bits(float x) { return __builtin_bit_cast(uint32_t, x); }
__device__ __forceinline__ float f16_to_f32(uint32_t h) { return (float)__builtin_bit_cast(_Float16, (uint16_t)h); }

template <int SUB>
__device__ __forceinline__ typename AccOf<SUB>::type mfma(bf16x8_t a, bf16x8_t b, typename AccOf<SUB>::type c) {
    if constexpr (SUB == 32) return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// two floats -> the bf16 pair of their upper halves; what truncation leaves
__device__ __forceinline__ uint32_t upper2(float x0, float x1) { return perm(bits(x1), bits(x0), 0x07060302u); }
__device__ __forceinline__ float rest(float x) { return x - __builtin_bit_cast(float, bits(x) & 0xFFFF0000u); }

// Eight codes (elements e and 16 + e of a block in the nibbles of byte e) -> code - 8 as bf16: 1024 + code as f16 (the code
// under the exponent byte 0x64) minus 1032 is exact, a number of three significant bits is its f16's upper byte read as
// e5m2, and that converts in pairs.  17 operations for eight codes; through f32 (byte to float, minus 8, upper halves) 23.
__device__ __forceinline__ bf16x8_t codes_bf16(uint32_t word) {
    const half2_t off = {(_Float16)1032.0f, (_Float16)1032.0f};
    u32x4 o;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const uint32_t c = h ? (word >> 4) & 0x0F0F0F0Fu : word & 0x0F0F0F0Fu;
        const uint32_t lo = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, perm(0x64646464u, c, 0x04010400u)) - off);
        const uint32_t hi = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, perm(0x64646464u, c, 0x04030402u)) - off);
        const uint32_t e5m2 = perm(hi, lo, 0x07050301u);
        o[2 * h] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(e5m2, 1.0f, false));
        o[2 * h + 1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(e5m2, 1.0f, true));
    }
    return __builtin_bit_cast(bf16x8_t, o);
}

template <int SUB, int MS, int NI, bool TILED>
__global__ __launch_bounds__(64 * kW, 2) void q4_0_matmul_f32_kernel(MatMulF32 p) {
    typedef typename AccOf<SUB>::type acc_t;
    constexpr int R = SUB == 32 ? 16 : 4;        // results per lane and subtile
    constexpr int KST = SUB == 32 ? 2 : 1;       // instructions per block
    constexpr int PER_WAVE = MS * NI * R * 64;   // results of a wave
    constexpr int COPIES = PER_WAVE * kW * 4 <= 65536 ? kW : kW / 2;   // the waves' sums that LDS holds at once
    __shared__ __attribute__((aligned(16))) float lds[COPIES * PER_WAVE];

    const int tid = threadIdx.x, lane = tid & 63, row = lane % SUB, grp = lane / SUB;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n0 = blockIdx.x * SUB * NI, m0 = blockIdx.y * SUB * MS, b = blockIdx.z, wb = b / p.ratio;
    const int nb = p.k / 32, units = (nb + 3) / 4;
    // slot g of a block: its features 4 g .. 4 g + 3 and 16 + 4 g .. 16 + 4 g + 3.  Instruction st of a block contracts slots
    // 2 st + grp (SUB 32) or all four (SUB 16).
    auto slot = [&](int st) { return SUB == 32 ? 2 * st + grp : grp; };

    // Buffers: activation rows past m, and planes' blocks past the end of the matrix, read as zeros (the range check sees
    // the vector offset only); weight rows past n repeat the last ones, their results are not stored.
    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(p.act + (int64_t)b * p.m * p.k), 0, (uint32_t)((int64_t)p.m * p.k * 4), 0x00020000);
    const int64_t w_bytes = TILED ? (int64_t)(p.n / 16) * units * kTile : (int64_t)p.n * (p.k / 2);
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(p.codes + wb * w_bytes), 0, (uint32_t)w_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t s_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t *>(TILED ? nullptr : p.scales + (int64_t)wb * p.n * nb), 0, TILED ? 0u : (uint32_t)((int64_t)p.n * nb * 2), 0x00020000);
    uint32_t a_off[MS], w_off[NI], s_off[NI];
#pragma unroll
    for (int i = 0; i < MS; i++) a_off[i] = (uint32_t)(m0 + SUB * i + row) * (uint32_t)p.k * 4u + 16u * slot(0);
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int j = min(n0 + SUB * i + row, p.n - 1);
        if constexpr (TILED) {
            w_off[i] = (uint32_t)(j >> 4) * (uint32_t)units * kTile + 16u * (j & 15) + 256u * slot(0);
            s_off[i] = (uint32_t)(j >> 4) * (uint32_t)units * kTile + 1024 + 8u * (j & 15);
        } else {
            w_off[i] = (uint32_t)j * (uint32_t)(p.k / 2) + 4u * slot(0);
            s_off[i] = (uint32_t)j * (uint32_t)nb * 2u;
        }
    }

    struct Weights { uint32_t c[NI][KST][4]; uint32_t s[NI][2]; };   // a unit: words per (instruction, block), scales of its blocks
    struct Act { f32x4 x[MS][KST][2]; };                             // a block: features 4 g .., 16 + 4 g ..
    auto load_w = [&](Weights &d, int u) {
#pragma unroll
        for (int i = 0; i < NI; i++) {
            if constexpr (TILED) {
#pragma unroll
                for (int st = 0; st < KST; st++) {
                    const u32x4 c = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, w_off[i] + 512 * st, u * kTile, 0));
#pragma unroll
                    for (int j = 0; j < 4; j++) d.c[i][st][j] = c[j];
                }
                const u32x2 s = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(w_rsrc, s_off[i], u * kTile, 0));
                d.s[i][0] = s.x, d.s[i][1] = s.y;
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++)
#pragma unroll
                    for (int st = 0; st < KST; st++) d.c[i][st][j] = __builtin_amdgcn_raw_buffer_load_b32(w_rsrc, w_off[i] + 64u * u + 16 * j + 8 * st, 0, 0);
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
        for (int i = 0; i < MS; i++)
#pragma unroll
            for (int st = 0; st < KST; st++)
#pragma unroll
                for (int h = 0; h < 2; h++)
                    d.x[i][st][h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, a_off[i] + 32 * st + 64 * h, blk * 128, 0));
    };

    acc_t acc[MS][NI];
#pragma unroll
    for (int i = 0; i < MS; i++)
#pragma unroll
        for (int j = 0; j < NI; j++)
#pragma unroll
            for (int r = 0; r < R; r++) acc[i][j][r] = 0.0f;

    // result register r of a lane: activation row SUB i + out_row(r) of the workgroup's, weight row SUB j + lane % SUB
    auto out_row = [&](int r) { return SUB == 32 ? 8 * (r / 4) + 4 * grp + r % 4 : 4 * grp + r; };

    // Whether a block is one of those, by the largest magnitude among a lane's 8 values of each of its activation rows.
    auto needs_f32 = [](const float (&big)[MS]) {
        bool any = false;
#pragma unroll
        for (int i = 0; i < MS; i++) any = any || big[i] >= kBig || (!TILED && big[i] < kSmall && big[i] > 0.0f);
        return __any(any);
    };
    // Products with the dequantised weights, one after the other.
    auto slow_block = [&](int blk) {
        const float *act = p.act + (int64_t)b * p.m * p.k + blk * 32;
#pragma unroll 1
        for (int ij = 0; ij < MS * NI; ij++) {
            const int i = ij / NI, jj = ij % NI, j = min(n0 + SUB * jj + row, p.n - 1);
            acc_t sum;
#pragma unroll
            for (int r = 0; r < R; r++) sum[r] = 0.0f;
#pragma unroll 1
            for (int e = 0; e < 32; e++) {
                const int byte = e & 15;
                uint32_t c, d;
                if constexpr (TILED) {
                    const uint8_t *rec = p.codes + wb * w_bytes + ((int64_t)(j >> 4) * units + (blk >> 2)) * kTile;
                    c = rec[256 * (byte >> 2) + 16 * (j & 15) + 4 * (blk & 3) + (byte & 3)];
                    d = reinterpret_cast<const uint16_t *>(rec + 1024)[4 * (j & 15) + (blk & 3)];
                } else {
                    c = p.codes[wb * w_bytes + (int64_t)j * (p.k / 2) + blk * 16 + byte];
                    d = p.scales[((int64_t)wb * p.n + j) * nb + blk];
                }
                const float wt = ((float)(e < 16 ? c & 15 : c >> 4) - 8.0f) * f16_to_f32(d);
#pragma unroll
                for (int r = 0; r < R; r++)
                    sum[r] = fmaf(act[(int64_t)min(m0 + SUB * i + out_row(r), p.m - 1) * p.k + e], wt, sum[r]);
            }
#pragma unroll
            for (int x = 0; x < MS; x++)
#pragma unroll
                for (int y = 0; y < NI; y++)
                    if (x * NI + y == ij) acc[x][y] += sum;
        }
    };

    Weights wt, wt_next;
    Act cur, nxt;
    bool skipped = false;
    int u = w;
    if (u < units) load_w(wt_next, u), load_a(nxt, 4 * u);
    for (; u < units; u += kW) {
        wt = wt_next;
        if (u + kW < units) load_w(wt_next, u + kW);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int blk = 4 * u + j;
            if (!TILED && blk >= nb) break;
            cur = nxt;
            {   // the next block of this wave (a load of a block past the end is never used)
                const int next = j < 3 ? blk + 1 : 4 * (u + kW);
                if (next < nb) load_a(nxt, next);
            }
            __builtin_amdgcn_sched_barrier(0);   // (a block's fragments live only as long as the block)
            bf16x8_t part[3][MS][KST];   // the smallest first
            float big[MS];
#pragma unroll
            for (int i = 0; i < MS; i++) big[i] = 0.0f;
#pragma unroll
            for (int i = 0; i < MS; i++)
#pragma unroll
                for (int st = 0; st < KST; st++) {
                    u32x4 b1, b2, b3;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float x0 = cur.x[i][st][e >> 1][2 * (e & 1)], x1 = cur.x[i][st][e >> 1][2 * (e & 1) + 1];
                        big[i] = fmaxf(fmaxf(fabsf(x0), fabsf(x1)), big[i]);
                        const float r0 = rest(x0), r1 = rest(x1);
                        b1[e] = upper2(x0, x1), b2[e] = upper2(r0, r1), b3[e] = upper2(rest(r0), rest(r1));
                    }
                    part[0][i][st] = __builtin_bit_cast(bf16x8_t, b3);
                    part[1][i][st] = __builtin_bit_cast(bf16x8_t, b2);
                    part[2][i][st] = __builtin_bit_cast(bf16x8_t, b1);
                }
            if (needs_f32(big)) {   // after the loop
                skipped = true;
                continue;
            }
#pragma unroll
            for (int jj = 0; jj < NI; jj++) {
                bf16x8_t cf[KST];
#pragma unroll
                for (int st = 0; st < KST; st++) cf[st] = codes_bf16(wt.c[jj][st][j]);
                const float d = f16_to_f32(wt.s[jj][j >> 1] >> (16 * (j & 1)));
                acc_t sum[MS];
#pragma unroll
                for (int i = 0; i < MS; i++)
#pragma unroll
                    for (int r = 0; r < R; r++) sum[i][r] = 0.0f;
#pragma unroll
                for (int q = 0; q < 3; q++)
#pragma unroll
                    for (int st = 0; st < KST; st++)
#pragma unroll
                        for (int i = 0; i < MS; i++) sum[i] = mfma<SUB>(part[q][i][st], cf[st], sum[i]);
#pragma unroll
                for (int i = 0; i < MS; i++)
#pragma unroll
                    for (int r = 0; r < R; r++) acc[i][jj][r] = fmaf(sum[i][r], d, acc[i][jj][r]);
            }
        }
    }

    if (skipped) {
        for (u = w; u < units; u += kW)
            for (int blk = 4 * u; blk < min(4 * u + 4, nb); blk++) {
                float big[MS];
                load_a(cur, blk);
#pragma unroll
                for (int i = 0; i < MS; i++) big[i] = 0.0f;
#pragma unroll
                for (int i = 0; i < MS; i++)
#pragma unroll
                    for (int st = 0; st < KST; st++)
#pragma unroll
                        for (int e = 0; e < 8; e++) big[i] = fmaxf(big[i], fabsf(cur.x[i][st][e >> 2][e & 3]));
                if (needs_f32(big)) slow_block(blk);
            }
    }

    // ---- the eight sums, [wave][subtile][register][lane] in LDS, added in the order of the waves ---------------------
    auto write = [&](int at) {
#pragma unroll
        for (int i = 0; i < MS; i++)
#pragma unroll
            for (int j = 0; j < NI; j++)
#pragma unroll
                for (int r = 0; r < R; r++) lds[at * PER_WAVE + ((i * NI + j) * R + r) * 64 + lane] = acc[i][j][r];
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
                    for (int r = 0; r < R; r++) acc[i][j][r] += lds[w * PER_WAVE + ((i * NI + j) * R + r) * 64 + lane];
            write(w);   // (read and written by the same thread)
        }
    } else {
        write(w);
    }
    __syncthreads();
    float *out = p.out + (int64_t)b * p.m * p.n;
    for (int e = tid; e < PER_WAVE; e += 64 * kW) {
        float sum = lds[e];
#pragma unroll
        for (int c = 1; c < COPIES; c++) sum += lds[c * PER_WAVE + e];
        // (an element's lane is its thread's: 64 divides the workgroup)
        const int r = (e >> 6) % R, j = (e >> 6) / R % NI, i = (e >> 6) / (R * NI);
        const int mi = m0 + SUB * i + out_row(r), ni = n0 + SUB * j + row;
        if (mi < p.m && ni < p.n) out[(int64_t)mi * p.n + ni] = sum;
    }
}

}  // namespace

// 2 = not taken (rows in groups on the matrix-vector kernels): operands beyond 32-bit offsets, misaligned ones.
int launch_q4_0_matmul_f32(const void *codes, const void *scales, int64_t w_batch, int64_t n, int64_t k, const void *act,
                           int64_t act_batch, int64_t m, void *out, hipStream_t s, int tiled) {
    if (m < 1 || n < 1 || k % 32 || (tiled && (n % 16 || k % 128))) return 2;
    if ((uintptr_t)codes % 16 || (uintptr_t)act % 16 || (uintptr_t)out % 4 || act_batch > 65535) return 2;
    if (n >= (1ll << 30) || m >= (1ll << 30) || k >= (1ll << 30)) return 2;
    if ((m + 64) * k >= (1ll << 30) || n * (k / 32) >= (1ll << 32) / 18 - 4096) return 2;
    MatMulF32 p;
    p.codes = (const uint8_t *)codes, p.scales = (const uint16_t *)scales;
    p.act = (const float *)act, p.out = (float *)out;
    p.n = (int)n, p.k = (int)k, p.m = (int)m, p.ratio = (int)(act_batch / w_batch);

    const int64_t cus = num_compute_units();
    auto launch = [&](auto sub, auto ms, auto ni) -> int {
        constexpr int SUB = decltype(sub)::value, MS = decltype(ms)::value, NI = decltype(ni)::value;
        constexpr bool TILES = !(SUB == 32 && (MS == 2 || NI == 1)), PLANES = SUB == 16 ? NI <= 2 : NI <= 3;   // (the other's never chosen)
        auto grid_of = [&](const MatMulF32 &part, int64_t batches) {
            const dim3 grid((unsigned)((n + SUB * NI - 1) / (SUB * NI)), (unsigned)((part.m + SUB * MS - 1) / (SUB * MS)), (unsigned)batches);
            if constexpr (TILES)
                if (tiled) hipLaunchKernelGGL((q4_0_matmul_f32_kernel<SUB, MS, NI, true>), grid, dim3(64 * kW), 0, s, part);
            if constexpr (PLANES)
                if (!tiled) hipLaunchKernelGGL((q4_0_matmul_f32_kernel<SUB, MS, NI, false>), grid, dim3(64 * kW), 0, s, part);
        };
        const int64_t most = 65535ll * SUB * MS;   // rows that a grid has tiles for
        if (m <= most) grid_of(p, act_batch);
        for (int64_t b = 0; m > most && b < act_batch; b++)
            for (int64_t row = 0; row < m; row += most) {
                MatMulF32 part = p;
                part.codes += b / p.ratio * (tiled ? n / 16 * (k / 128) * kTile : n * (k / 2));
                if (!tiled) part.scales += b / p.ratio * n * (k / 32);
                part.act += (b * m + row) * k, part.out += (b * m + row) * n;
                part.m = (int)std::min(most, m - row), part.ratio = 1;
                grid_of(part, 1);
            }
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return fail("q4_0_matmul (f32) launch failed: %s", hipGetErrorString(e));
        return 0;
    };
    std::integral_constant<int, 1> one;
    std::integral_constant<int, 2> two;
    std::integral_constant<int, 3> three;
    std::integral_constant<int, 4> four;
    std::integral_constant<int, 16> sub16;
    std::integral_constant<int, 32> sub32;
    // The shape that takes the least time: rounds of workgroups, one per compute unit, the first and the later ones as measured (us, straight
    // lines in the units of the busiest wave), tiles with 1024, 4096 and 14336 features, planes at 12 matrices of 512 to 14336 and 8 to 500
    // rows.  Against squares of 32 and 64 and oblongs of 16 x 16, 16 x 32 and 32 x 64 by one number each: tiles, 150 rows of 4096 x 4096 36.7
    // -> 26.4 (32 x 96; 32 x 128 29.2), 40 17.8 -> 14.1 (16 x 64), 512 74.5 -> 62.3 (32 x 128), 16 of 14336 x 4096 20.0 -> 15.0, 500 252
    // -> 216.  Squares share more of the split of the activations, oblongs of the same size have half the registers for it: 64 x 64 is
    // 250 there.  The codes of planes come in words of 4 bytes, so that a weight row costs more and squares stay the better ones (us, as
    // for tiles | as here: 40 rows of 4090 x 4096 39.3 | 27.1 (32 x 32), 500 127 | 111 (64 x 64), 200 of 1000 x 2080 16.2 | 13.1); 0.984 of
    // the time by one number each over those 144 products, none longer, and 0.96 over 539 of up to 50000 x 4128 and 2000 rows (at most
    // 1.07, but for 8 and 16 rows of 16390 x 2080, one tile more than two rounds, 1.18 and 1.10).  Below 1024 features, where some waves have no unit, a launch takes its
    // 4 to 5 us and is still the faster side (groups of 8 rows | here: 7 rows of 4096 x 32 7.1 | 4.1, of 4096 x 512 5.4 | 4.2; 40 rows of
    // 16384 x 128 23.7 | 7.7, of 1000 x 96 24.7 | 4.5).
    struct Times { float first, first_k, later, later_k; };
    constexpr float kNever = 1e9f;
    struct Shape { int sub, ms, ni; Times tiles, planes; };
    const Shape shapes[] = {{16, 1, 1, {1.3f, 1.75f, 0.4f, 1.75f}, {1.24f, 2.92f, -0.74f, 2.57f}}, {16, 1, 2, {1.4f, 2.27f, 0.2f, 1.93f}, {0.89f, 4.37f, -1.35f, 3.75f}},
                            {16, 1, 3, {2.6f, 2.45f, 0.25f, 2.17f}, {kNever}},                     {16, 1, 4, {2.3f, 2.93f, 0.3f, 2.45f}, {kNever}},
                            {32, 1, 1, {kNever}, {0.78f, 5.04f, -1.76f, 5.06f}},                   {32, 1, 2, {2.6f, 4.08f, 1.9f, 4.1f}, {0.68f, 7.33f, -0.06f, 7.24f}},
                            {32, 1, 3, {3.6f, 5.05f, 3.0f, 5.45f}, {0.92f, 9.86f, 1.87f, 9.37f}},  {32, 1, 4, {4.3f, 6.1f, 4.2f, 6.4f}, {kNever}},
                            {32, 2, 2, {kNever}, {1.64f, 10.62f, 2.59f, 10.0f}}};
    const int64_t units = (k + 127) / 128, last = k / 32 - 4 * (units - 1);   // blocks of the last unit, which is a wave's last if no other one has as many
    const float per_wave = std::max(0.5f, (float)((units - 1) / 8 * 4 + ((units - 1) % 8 ? 4 : last)) / 4.0f);   // (the lines end there)
    int best = 0;
    float best_us = 0.0f;
    for (int c = 0; c < 9; c++) {
        const Shape &x = shapes[c];
        const Times &t = tiled ? x.tiles : x.planes;
        const int64_t bm = x.sub * x.ms, bn = x.sub * x.ni, rounds = ((n + bn - 1) / bn * ((m + bm - 1) / bm) * act_batch + cus - 1) / cus;
        const float us = t.first + t.first_k * per_wave + (t.later + t.later_k * per_wave) * (float)(rounds - 1);
        if (c == 0 || us < best_us) best = c, best_us = us;
    }
    switch (best) {
        case 0: return launch(sub16, one, one);
        case 1: return launch(sub16, one, two);
        case 2: return launch(sub16, one, three);
        case 3: return launch(sub16, one, four);
        case 4: return launch(sub32, one, one);
        case 5: return launch(sub32, one, two);
        case 6: return launch(sub32, one, three);
        case 7: return launch(sub32, one, four);
        default: return launch(sub32, two, two);
    }
}

}  // namespace trocm
