// Attention of many f32 query rows on the matrix cores (prompts, chunks of one, a few proposed tokens): gfx950.
//
// The f32 counterpart of sdpa_prefill_pp.hip: q, K and V stay f32, both products run on v_mfma_f32_32x32x2_f32 (f32
// operands, f32 accumulation), probabilities are never narrowed.
//
// The query rows of a kv head are its G heads times q_len queries, row r = query r / G of head r % G, so that 32
// consecutive rows see almost the same keys whatever G is.  A workgroup of 4 waves owns 32 such rows and one range of key
// tiles; its waves take the range's 32-key tiles in turn (wave w: w, w + 4, ..), each with a running maximum and sum of its
// own, and are merged through LDS at the end.  Dividing the keys and not the rows is what fills the chip: 1000 rows of
// 32 heads are 1000 workgroups of at most 8 tiles per wave, the longest of which start first; 128-row workgroups would be
// 256 of 1 .. 32 tiles.  Ranges (`nsplit` > 1, partial results in the workspace, a merge launch) are for launches that have
// fewer than two workgroups per compute unit.
//
//   S^T[key, row] = K . q^T   A = K: lane (key = lane % 32, half = lane / 32) holds features 8 j + 4 half .. + 3 of its key,
//                             B = q from LDS, the same features (the order inside the contraction is free)
//   O^T[d, row]   = V^T . P^T  register r of S^T is key 8 (r / 4) + 4 half + r % 4: exactly the B operand of a step
//                             that contracts keys (8 q + e, 8 q + 4 + e), so P needs no transposition; A = V of those two
//                             keys, lane % 32 = feature T d' + t of subtile t (T = D / 32): one load of T floats per key
//
// K and V go from memory straight into those registers: V rows in whole 512-byte lines, K in 32-byte pieces of 32 rows
// whose lines the next three loads use up.  A tile is 8192 matrix cycles (D = 128) against 32 KB of loads, so neither path
// is near its rate, and without LDS copies there is no barrier in the loop.  The next tile's K is requested when this
// tile's is used up, V before the scores: each has a phase of 4096 cycles to arrive.  K / V of a kv head stay in one XCD's L2:
// workgroup ids run over kv heads first.
//
// Bound by the f32 matrix rate (152 TFLOP/s reached by a large product) and, with up to 32 rows, mostly by the chain of a short
// launch.  The generic kernel, a wave per query with scalar fused multiply-adds, took 9040 us for 1000 queries of 32 heads.
//
// More than 32 rows (sdpa_prefill_f32x2_kernel): every f32 is a power of two times the sum of two f16 numbers, and a product is three
// of v_mfma_f32_32x32x16_f16 (upper by upper, upper by lower, lower by upper; f32 accumulation): three times the f32 instruction's
// rate, 23 of the 24 bits of every operand, and fewer roundings in the sums.  Error against f64, 1000 causal queries of 32 heads
// over 8, 2.7e-7, 771 over 451 past tokens 3.9e-7 (the f32 instruction: 3.3e-7, 4.7e-7).
//  * Two row tiles of 32 per workgroup and two key sets of two waves: a set's waves share the 32-key tiles that its 128 threads turn
//    into pairs on the way into LDS (K by rows, V transposed into the order in which P comes out of the scores).
//  * Scales, powers of two: q's per row, K's and V's from the first two tiles of the range, with room for 16 to 32 (K) and 8 to 16 (V)
//    times their largest value in what comes later.  A pair is exact to 2^-23 of its number, or to 2^-25 in the scaled unit where
//    that is more.  What this leaves of K changes a score by at most |q| sqrt(D) scale 2^-25 / k_up, which has to be below 2^-21 (a
//    few 2^-24 as a rule), and no feature of V may be 2^13 weaker than the strongest in those tiles.  Otherwise the workgroup runs
//    the f32 code (attend_tile) and nothing else.
//  * What shows only later is seen in the sums, and the workgroup starts again with the f32 code: values beyond the room, infinities
//    and NaN (sums that are no numbers), and V that has become too weak for its unit (a row, or a feature over all the rows, that is
//    small against what the pairs leave).
//  * What bounds it is the issue of instructions: per tile and wave 48 matrix and about 550 vector instructions.  1000 queries of 32
//    heads over 8: matrix units busy 23 % of the kernel's cycles and vector units 44, which do not overlap, and the longest row tiles
//    run on alone (2000 queries: 33 and 64).  Loads have no condition around them, or the waits for one tile's V would be waits for
//    the next tile's K (71.6 -> 58.2 us).
// us of a call with its append, on the f32 instruction | as pairs | refused: 1000 queries of 32 heads over 8 (D = 128) 102.6 | 54.4 | 103;
// 771 over 451 tokens 130.9 | 63.7 | 152; 10 queries of 4 x 64 heads over 8, 3629 tokens, 96.5 | 65.0 | 114; 2 x 251 queries 28.1 | 24.9 |
// 41 (refused tiles cost more where few workgroups of 64 rows take the place of twice as many of 32; 135, 197, 141 and 49 while
// the pairs' loop ran before them).  What only the sums show: 138, 199, 112 and 51.
// From 4 tiles on (2 x 70 queries of 32 heads over 32, 3 tiles: 15.3 | 17.5; 2 x 116 of 40 over 8 20.0 | 18.0); ranges of keys (us
// without | with): 49 queries, 32 over 8, 396 tokens 29.7 | 21.5, but 2 x 251, a workgroup per compute unit, 25.0 | 33.7.
#include <hip/hip_runtime.h>
#include <limits.h>
#include <string.h>
#include <algorithm>
#include "decode_common.h"

namespace trocm {
namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kRows = 32, kMaxSplits = 64;
// least result, in V's scaled unit: the sum of a row's magnitudes, and the strongest row of a feature.  What the pairs leave, 2^-25 of
// that unit at most for each number, is then below 2^-22 of a row's norm and 2^-21 of a feature, as much as f32 sums leave.  (A mean of
// n keys of normal V is about 2^10 / sqrt(n) in that unit: only rows that weigh ten thousands of keys all alike, or features a
// thousand times weaker than the strongest, fall below these by chance.)
constexpr float kLeastOfRow = 16.0f, kLeastOfFeature = 0.0625f;

struct PrefillF32 {
    const float *q, *k, *v;
    float *out;
    float *part_o;    // [nsplit][n_wg][32][D], not normalised
    float *part_ml;   // [nsplit][n_wg][64]: maxima, then sums
    int64_t kv_stride_b, kv_stride_h;   // elements
    uint32_t kv_row_bytes;              // bytes between token rows
    int Hq, Hkv, Sq, Sk, G;
    int n_bh, n_rt, nsplit;             // batch * kv_heads, 32-row tiles per kv head
    int n_rt2, paired;                  // sdpa_prefill_f32x2_kernel: 64-row tiles per kv head; whether the short ones run beside the long ones
    int causal;
    float scale;
    // Fused append (dense token rows): the tokens from `past` on are read from the call's own dense rows, [B, Hkv, Sq, D], and copied to
    // the cache by this launch.  NULL: all Sk = `past` are in the cache, n_new is 0.
    const float *k_new, *v_new;
    int past, n_new;
};


template <int T> struct VecOf;
template <> struct VecOf<2> { typedef f32x2 type; };
template <> struct VecOf<4> { typedef f32x4 type; };

__device__ __forceinline__ f32x4 buffer_f32x4(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
template <int T>
__device__ __forceinline__ typename VecOf<T>::type buffer_vec(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    if constexpr (T == 4) return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
    else return __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}
// all ones if x is finite, else 0.  (Arithmetic: as a condition for each of 32 numbers it takes more scalar registers than there are.)
__device__ __forceinline__ uint32_t finite_mask(float x) {
    return (uint32_t)((int)((__builtin_bit_cast(uint32_t, x) & 0x7f800000u) - 0x7f800000u) >> 31);
}
__device__ __forceinline__ float masked(float x, uint32_t mask) { return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x) & mask); }

// Tiles of 32 keys: those of the cache, the last of them with fewer rows, then those of the call's rows.  NEW: the launch has such rows (what
// picks between the two costs calls over a cache alone 1.4 % on average and 4 % of the shortest).
template <bool NEW>
struct KeyTiles {
    int past, old;   // tokens and tiles in the cache
    __device__ __forceinline__ int first_key(int kt) const { return !NEW || kt < old ? 32 * kt : past + 32 * (kt - old); }
    __device__ __forceinline__ int end(int kt) const { return NEW && kt < old ? min(32 * kt + 32, past) : INT_MAX; }   // keys from here on are not its own
    __device__ __forceinline__ int count(int n_vis) const { return !NEW || n_vis <= past ? (n_vis + 31) / 32 : old + (n_vis - past + 31) / 32; }
};
// The rows of one kv head of K or V: rows after the last one of a buffer read as zeros.
template <bool NEW>
struct Rows {
    const float *head, *head_new;
    int past, n_new;
    uint32_t row_bytes;
    __device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(int kt) const {
        const bool old = !NEW || 32 * kt < past;
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(old ? head : head_new), 0, (uint32_t)(old ? past : n_new) * row_bytes, 0x00020000);
    }
    __device__ __forceinline__ uint32_t off(int kt, int row) const { return (uint32_t)(32 * (!NEW || 32 * kt < past ? kt : kt - (past + 31) / 32) + row) * row_bytes; }   // row of tile kt
};
template <bool NEW>
__device__ __forceinline__ Rows<NEW> rows_of(const PrefillF32 &p, const float *cache, const float *call, int b, int kvh, int D) {
    return Rows<NEW>{cache + b * p.kv_stride_b + kvh * p.kv_stride_h, call + ((int64_t)b * p.Hkv + kvh) * p.Sq * D, p.past, p.n_new, p.kv_row_bytes};
}

// the weight exp(m - ref) of a partial result whose maximum is m; nothing seen: m = -inf, weight 0 whatever ref is
__device__ __forceinline__ float ref_of(float m) { return m == -INFINITY ? 0.0f : m; }

// LDS of a workgroup: q, then the waves' outputs; their maxima and sums
template <int D>
struct TileLds {
    float rows[kWaves * kRows * (D + 4)];
    float m[kWaves][kRows], l[kWaves][kRows];
};

// Row tile rt of a (batch, kv head) over the key tiles kt_first .. kt_last - 1 that it sees, by one workgroup.
template <int D, bool NEW>
__device__ __forceinline__ void attend_tile(const PrefillF32 &p, TileLds<D> &shared, int bh, int rt, int split, int kt_first, int kt_last) {
    constexpr int T = D / 32, KJ = D / 8, ROW = D + 4;   // (ROW: 16 rows of a 128-bit LDS pass in 16 distinct bank groups)
    typedef typename VecOf<T>::type vec;
    float *lds = shared.rows;
    auto &lds_m = shared.m;
    auto &lds_l = shared.l;

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hb = lane >> 5;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int b = bh / p.Hkv, kvh = bh % p.Hkv;
    const int n_rows = p.Sq * p.G, r0 = rt * kRows;
    auto q_row = [&](int r) {   // offset of row r's query (and output) in elements
        const int i = r / p.G, g = r - i * p.G;
        return (((int64_t)b * p.Hq + kvh * p.G + g) * p.Sq + i) * D;
    };
    // keys [0, limit) are visible to a row; the tile as a whole sees n_vis
    auto limit_of = [&](int r) { return p.causal ? min(r, n_rows - 1) / p.G + (p.Sk - p.Sq) + 1 : p.Sk; };
    const int limit = limit_of(r0 + l32), limit_first = limit_of(r0), n_vis = limit_of(r0 + kRows - 1);
    const KeyTiles<NEW> keys{p.past, (p.past + 31) / 32};
    const int kt_end = min(keys.count(n_vis), kt_last);

    // rows past the last key read as zeros: the buffer ends with that row
    const Rows<NEW> k_rows = rows_of<NEW>(p, p.k, p.k_new, b, kvh, D), v_rows = rows_of<NEW>(p, p.v, p.v_new, b, kvh, D);

    f32x4 kreg[KJ];
    vec vreg[16];
    auto load_k = [&](int kt) {
        const __amdgpu_buffer_rsrc_t rsrc = k_rows.rsrc(kt);
        const uint32_t off = k_rows.off(kt, l32) + 16 * hb;
#pragma unroll
        for (int j = 0; j < KJ; j++) kreg[j] = buffer_f32x4(rsrc, off + 32 * j);
    };
    auto load_v = [&](int kt) {
        const __amdgpu_buffer_rsrc_t rsrc = v_rows.rsrc(kt);
        const uint32_t off = v_rows.off(kt, 4 * hb) + 4 * T * l32;
#pragma unroll
        for (int i = 0; i < 16; i++) vreg[i] = buffer_vec<T>(rsrc, off + (uint32_t)(8 * (i / 4) + i % 4) * p.kv_row_bytes);
    };

    int kt = kt_first + w;
    if (kt < kt_end) load_k(kt);
#pragma unroll
    for (int j = 0; j < kRows * D / 4 / kThreads; j++) {
        const int f = j * kThreads + tid, r = f / (D / 4), c = f % (D / 4);
        *reinterpret_cast<f32x4 *>(&lds[r * ROW + 4 * c]) = *reinterpret_cast<const f32x4 *>(p.q + q_row(min(r0 + r, n_rows - 1)) + 4 * c);
    }
    __syncthreads();

    f32x16 o[T];
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[t][r] = 0.0f;
    float m_run = -INFINITY, l_run = 0.0f;   // the maximum of the row; the sum over this lane's half of the keys

    const float *q_frag = &lds[l32 * ROW + 4 * hb];
    for (; kt < kt_end; kt += kWaves) {
        load_v(kt);
        __builtin_amdgcn_sched_barrier(0);   // (requested before the scores, not after)
        f32x16 s;
#pragma unroll
        for (int r = 0; r < 16; r++) s[r] = 0.0f;
#pragma unroll
        for (int j = 0; j < KJ; j++) {
            const f32x4 qf = *reinterpret_cast<const f32x4 *>(q_frag + 8 * j);
#pragma unroll
            for (int e = 0; e < 4; e++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kreg[j][e], qf[e], s, 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (kt + kWaves < kt_end) load_k(kt + kWaves);
        __builtin_amdgcn_sched_barrier(0);

        const int key0 = keys.first_key(kt), own = min(limit, keys.end(kt));
        const bool edge = key0 + 32 > min(limit_first, keys.end(kt));   // some row does not see all of the tile
#pragma unroll
        for (int r = 0; r < 16; r++) s[r] *= p.scale;
        if (edge) {
#pragma unroll
            for (int r = 0; r < 16; r++)
                if (key0 + 8 * (r / 4) + 4 * hb + r % 4 >= own) s[r] = -INFINITY;
        }
        float mx = s[0];
#pragma unroll
        for (int r = 1; r < 16; r++) mx = fmaxf(mx, s[r]);
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float m_new = fmaxf(m_run, mx), ref = ref_of(m_new);
        if (__any(m_new != m_run)) {
            const float alpha = expf(m_run - ref);
            l_run *= alpha;
#pragma unroll
            for (int t = 0; t < T; t++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[t][r] *= alpha;
            m_run = m_new;
        }
#pragma unroll
        for (int r = 0; r < 16; r++) {
            s[r] = expf(s[r] - ref);
            l_run += s[r];
        }

        // A key that a row does not see must not reach its sum, and 0 times an infinity or a NaN of V would: in a tile
        // with such keys the products take V's finite values only, and the others are added to the rows that do see them.
        if (edge) {
            float probe = 0.0f;   // NaN once one is not finite (one register; a condition per element takes 86 scalar ones too many)
#pragma unroll
            for (int i = 0; i < 16; i++)
#pragma unroll
                for (int t = 0; t < T; t++) probe = fmaf(vreg[i][t], 0.0f, probe);
            if (__any(probe != 0.0f)) {
#pragma unroll 1
                for (int kk = 0; kk < 32; kk++) {
                    // p of (row = lane % 32, key kk): register 4 (kk / 8) + kk % 4 of the half (kk / 4) % 2
                    float pk = 0.0f;
#pragma unroll
                    for (int r = 0; r < 16; r++)
                        if (r == 4 * (kk >> 3) + (kk & 3)) pk = s[r];
                    pk = __shfl(pk, l32 + 32 * ((kk >> 2) & 1), 64);
                    const uint32_t seen = key0 + kk < own ? ~0u : 0u;
                    const __amdgpu_buffer_rsrc_t rsrc = v_rows.rsrc(kt);
                    const uint32_t off = v_rows.off(kt, kk);
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const vec x = buffer_vec<T>(rsrc, off + 4 * T * (8 * (r / 4) + 4 * hb + r % 4));
#pragma unroll
                        for (int t = 0; t < T; t++)
                            o[t][r] = fmaf(pk, masked(x[t], seen & ~finite_mask(x[t])), o[t][r]);
                    }
                }
#pragma unroll
                for (int i = 0; i < 16; i++)
#pragma unroll
                    for (int t = 0; t < T; t++) vreg[i][t] = masked(vreg[i][t], finite_mask(vreg[i][t]));
            }
        }
#pragma unroll
        for (int i = 0; i < 16; i++)
#pragma unroll
            for (int t = 0; t < T; t++) o[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(vreg[i][t], s[i], o[t], 0, 0, 0);
    }

    // ---- the waves' results: out = sum_w e^(m_w - M) O_w / sum_w e^(m_w - M) l_w -------------------------------
    // (the thread's number taken anew: what the tail makes of it would otherwise be kept through the loop, in scratch memory)
    int tid_end = tid;
    asm("" : "+v"(tid_end));
    const int l_end = tid_end & 31, h_end = (tid_end >> 5) & 1;
    l_run += __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(((tid_end & 63) ^ 32) * 4, __builtin_bit_cast(int, l_run)));
    if (h_end == 0) lds_m[w][l_end] = m_run, lds_l[w][l_end] = l_run;
    __syncthreads();   // (and every wave is done with q)
    float m_all = lds_m[0][l_end];
#pragma unroll
    for (int i = 1; i < kWaves; i++) m_all = fmaxf(m_all, lds_m[i][l_end]);
    const float wgt = expf(m_run - ref_of(m_all));
    float *mine = &lds[w * kRows * ROW + l_end * ROW];
#pragma unroll
    for (int r = 0; r < 16; r++) {
        vec x;
#pragma unroll
        for (int t = 0; t < T; t++) x[t] = o[t][r] * wgt;
        *reinterpret_cast<vec *>(mine + T * (8 * (r / 4) + 4 * h_end + r % 4)) = x;
    }
    __syncthreads();
    const int64_t wb = (int64_t)bh * p.n_rt + rt, n_wb = (int64_t)p.n_bh * p.n_rt;
#pragma unroll
    for (int j = 0; j < kRows * D / 4 / kThreads; j++) {
        const int f = j * kThreads + tid_end, r = f / (D / 4), c = f % (D / 4);
        f32x4 sum = *reinterpret_cast<const f32x4 *>(&lds[r * ROW + 4 * c]);
        float mm = lds_m[0][r];
#pragma unroll
        for (int i = 1; i < kWaves; i++) {
            sum += *reinterpret_cast<const f32x4 *>(&lds[i * kRows * ROW + r * ROW + 4 * c]);
            mm = fmaxf(mm, lds_m[i][r]);
        }
        float l = 0.0f;
#pragma unroll
        for (int i = 0; i < kWaves; i++) l += lds_l[i][r] * expf(lds_m[i][r] - ref_of(mm));
        if (p.nsplit > 1) {
            *reinterpret_cast<f32x4 *>(p.part_o + (((int64_t)split * n_wb + wb) * kRows + r) * D + 4 * c) = sum;
            if (c == 0) {
                float *ml = p.part_ml + ((int64_t)split * n_wb + wb) * 64;
                ml[r] = mm, ml[32 + r] = l;
            }
        } else if (r0 + r < n_rows) {
#pragma unroll
            for (int e = 0; e < 4; e++) sum[e] = l > 0.0f ? sum[e] / l : 0.0f;
            *reinterpret_cast<f32x4 *>(p.out + q_row(r0 + r) + 4 * c) = sum;
        }
    }
}

template <int D, bool NEW>
__global__ __launch_bounds__(kThreads, 2) void sdpa_prefill_f32_kernel(PrefillF32 p) {
    __shared__ __attribute__((aligned(16))) TileLds<D> shared;
    const int bh = blockIdx.x % p.n_bh, rest = blockIdx.x / p.n_bh;
    const int split = rest % p.nsplit, rt = p.n_rt - 1 - rest / p.nsplit;
    const int last = min(rt * kRows + kRows, p.Sq * p.G) - 1, n_vis = p.causal ? last / p.G + (p.Sk - p.Sq) + 1 : p.Sk;
    const int per_split = (KeyTiles<NEW>{p.past, (p.past + 31) / 32}.count(n_vis) + p.nsplit - 1) / p.nsplit;
    // The append: this workgroup's share of its kv head's rows (contiguous in both places; ahead of the attention, through which the
    // addresses would be kept in more scalar registers than there are).  With an append launch | now: 69 rows of 32 heads
    // over 8 14.3 | 12.2 us, 10 of 14 over 2 behind 348 18.8 | 16.4.
    if constexpr (NEW) {
        const int64_t from = (int64_t)bh * p.Sq * D, to = (bh / p.Hkv) * p.kv_stride_b + (bh % p.Hkv) * p.kv_stride_h + (int64_t)p.past * D;
        for (int i = rest * kThreads + threadIdx.x; i < p.Sq * (D / 4); i += p.n_rt * p.nsplit * kThreads) {
            reinterpret_cast<f32x4 *>(const_cast<float *>(p.k) + to)[i] = reinterpret_cast<const f32x4 *>(p.k_new + from)[i];
            reinterpret_cast<f32x4 *>(const_cast<float *>(p.v) + to)[i] = reinterpret_cast<const f32x4 *>(p.v_new + from)[i];
        }
    }
    attend_tile<D, NEW>(p, shared, bh, rt, split, split * per_split, (split + 1) * per_split);
}

// ---- more than 32 rows: every f32 as a pair of f16 ---------------------------------------------------------------------
__device__ __forceinline__ int exp_field(float x) { return (int)(__builtin_bit_cast(uint32_t, x) >> 23) & 255; }
__device__ __forceinline__ float pow2_field(int e) { return __builtin_bit_cast(float, (uint32_t)min(max(e, 0), 254) << 23); }
// exponent field of the scale that puts `largest` in 2^top .. 2^(top + 1) (at most 2^55, so that products of two scales and their
// inverses are normal numbers)
__device__ __forceinline__ int up_field(float largest, int top) { return min(254 + top - exp_field(largest), 127 + 55); }
typedef float f32x2_t __attribute__((ext_vector_type(2)));
// x times a power of two as the sum of two f16 numbers, each rounded once: 23 of its 24 bits.  (Six operations for a pair, all at
// the full rate: the instructions that multiply, add and round to f16 in one, five for a pair, take two cycles for one.)
__device__ __forceinline__ void split_pair(float x0, float x1, float scale, uint32_t &hi, uint32_t &lo) {
    const half2_t h = __builtin_convertvector(f32x2_t{x0 * scale, x1 * scale}, half2_t);
    const float h0 = (float)h.x, h1 = (float)h.y;
    hi = __builtin_bit_cast(uint32_t, h);
    lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{fmaf(x0, scale, -h0), fmaf(x1, scale, -h1)}, half2_t));
}
struct Split8 { half8_t hi, lo; };
template <typename F>
__device__ __forceinline__ Split8 split8(F x, float scale) {   // x(0) .. x(7)
    u32x4 h, l;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        uint32_t a, c;
        split_pair(x(2 * i), x(2 * i + 1), scale, a, c);
        h[i] = a, l[i] = c;
    }
    return Split8{__builtin_bit_cast(half8_t, h), __builtin_bit_cast(half8_t, l)};
}
__device__ __forceinline__ f32x16 mfma3(const Split8 &a, const Split8 &b, f32x16 c) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.lo, b.hi, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.hi, b.lo, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a.hi, b.hi, c, 0, 0, 0);
}
template <int D>
struct PairLds {
    _Float16 k[2][2][kRows * (D + 8)];          // [key set][upper, lower]: 32 keys of D features
    _Float16 vt[2][2][D / 32][32 * 40];         // [key set][upper, lower][subtile][feature]: 32 keys in the order of P's registers
};

template <int D, bool NEW>
__global__ __launch_bounds__(kThreads, 2) void sdpa_prefill_f32x2_kernel(PrefillF32 p) {
    constexpr int T = D / 32, C4 = D / 4, NG = 8 * C4 / 128, KROW = D + 8, ROW = D + 4;
    typedef typename VecOf<T>::type vec;
    __shared__ __attribute__((aligned(16))) union { PairLds<D> pair; TileLds<D> tile; float rows[2 * kRows * ROW]; } lds;
    __shared__ float lds_m[kWaves][kRows], lds_l[kWaves][kRows], lds_big[4][kWaves];
    __shared__ float lds_least[2 * kRows];   // by row: what a feature has to reach
    __shared__ int lds_odd;
    __shared__ uint64_t lds_strong[kWaves];

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hb = lane >> 5;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), rg = w & 1, ks = w >> 1;
    const int bh = blockIdx.x % p.n_bh, rest = blockIdx.x / p.n_bh, at = rest / p.nsplit, split = rest % p.nsplit;
    const int half = (p.n_rt2 + 1) / 2, rt2 = p.paired && at >= half ? at - half : p.n_rt2 - 1 - at;
    const int b = bh / p.Hkv, kvh = bh % p.Hkv;
    const int n_rows = p.Sq * p.G, r0 = rt2 * 2 * kRows;
    auto q_row = [&](int r) {
        const int i = r / p.G, g = r - i * p.G;
        return (((int64_t)b * p.Hq + kvh * p.G + g) * p.Sq + i) * D;
    };
    auto limit_of = [&](int r) { return p.causal ? min(r, n_rows - 1) / p.G + (p.Sk - p.Sq) + 1 : p.Sk; };
    const int limit = limit_of(r0 + kRows * rg + l32), limit_first = limit_of(r0), n_vis = limit_of(r0 + 2 * kRows - 1);
    const KeyTiles<NEW> keys{p.past, (p.past + 31) / 32};
    const int tiles = keys.count(n_vis), per_split = (tiles + p.nsplit - 1) / p.nsplit;
    const int kt_first = split * per_split, kt_last = min(tiles, kt_first + per_split);

    const Rows<NEW> k_rows = rows_of<NEW>(p, p.k, p.k_new, b, kvh, D), v_rows = rows_of<NEW>(p, p.v, p.v_new, b, kvh, D);
    // a key set's 128 threads: features 4 c4 .. + 3 of the keys 4 (g0 + 4 i) .. + 3
    const int st = tid & 127, c4 = st % C4, g0 = st / C4;
    f32x4 kpre[NG][4], vpre[NG][4];
    auto load_rows = [&](f32x4 (&dst)[NG][4], const Rows<NEW> &rows, int kt) {
        const __amdgpu_buffer_rsrc_t rsrc = rows.rsrc(kt);
        const uint32_t off = rows.off(kt, 4 * g0) + 16 * c4;
#pragma unroll
        for (int i = 0; i < NG; i++)
#pragma unroll
            for (int j = 0; j < 4; j++) dst[i][j] = buffer_f32x4(rsrc, off + (uint32_t)(16 * i + j) * p.kv_row_bytes);
    };
    int kt = kt_first + ks;
    load_rows(kpre, k_rows, min(kt, tiles)), load_rows(vpre, v_rows, min(kt, tiles));   // (past the last tile: zeros)

    // The append.  A workgroup copies its share of its kv head's rows (contiguous in both places), the first two 16-byte pieces of
    // each tensor per thread beside the loads above and of q, the others after the loop; nobody waits for another's copy, the new rows
    // of K and V are read from the call's input.  1000 queries of 32 heads over 8, with an append launch | now: 57.3 | 51.8 us; 900 of 32 over
    // 32 59.1 | 51.5; behind a cache 2 x 3 rows of 40 heads over 2579 tokens, 64 features, 19.5 | 17.8, 373 of 32 heads over 224 49.2 | 46.7.
    const f32x4 *src_k = nullptr, *src_v = nullptr;
    f32x4 *dst_k = nullptr, *dst_v = nullptr;
    int piece = 0, pieces = 0;   // this thread's next one, and how many there are
    const int hop = p.n_rt2 * p.nsplit * kThreads;
    if constexpr (NEW) {
        src_k = reinterpret_cast<const f32x4 *>(k_rows.head_new), src_v = reinterpret_cast<const f32x4 *>(v_rows.head_new);
        dst_k = reinterpret_cast<f32x4 *>(const_cast<float *>(k_rows.head) + (int64_t)p.past * D), dst_v = reinterpret_cast<f32x4 *>(const_cast<float *>(v_rows.head) + (int64_t)p.past * D);
        piece = rest * kThreads + tid, pieces = p.Sq * C4;
    }
    f32x4 ck[2], cv[2];
#pragma unroll
    for (int j = 0; j < 2; j++)
        if (NEW && piece + j * hop < pieces) ck[j] = src_k[piece + j * hop], cv[j] = src_v[piece + j * hop];

    // Scales, powers of two: q's per row, K's and V's from the first tiles of the range.
    Split8 q[D / 16];
    float c;   // what makes scores of the sums
    int k_field, v_field;
    bool odd;
    {
        auto largest = [](const f32x4 (&x)[NG][4]) {
            float big = 0.0f;
#pragma unroll
            for (int i = 0; i < NG; i++)
#pragma unroll
                for (int j = 0; j < 4; j++)
#pragma unroll
                    for (int e = 0; e < 4; e++) big = fmaxf(big, fabsf(x[i][j][e]));
            return wave_max(big);
        };
        const float *row = p.q + q_row(min(r0 + kRows * rg + l32, n_rows - 1)) + 8 * hb;
        f32x4 x[D / 8];
        float big = 0.0f;
#pragma unroll
        for (int j = 0; j < D / 8; j++) {
            x[j] = *reinterpret_cast<const f32x4 *>(row + 16 * (j / 2) + 4 * (j % 2));
#pragma unroll
            for (int e = 0; e < 4; e++) big = fmaxf(big, fabsf(x[j][e]));
        }
        big = fmaxf(big, __shfl_xor(big, 32, 64));
        const int q_field = up_field(big, 13);
#pragma unroll
        for (int j = 0; j < D / 16; j++) q[j] = split8([&](int i) { return x[2 * j + i / 4][i % 4]; }, pow2_field(q_field));
        float square = 0.0f;   // of the scaled row, which is neither too large nor too small for it
#pragma unroll
        for (int j = 0; j < D / 16; j++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const half2_t h = __builtin_bit_cast(half2_t, __builtin_bit_cast(u32x4, q[j].hi)[i]);
                square = __builtin_amdgcn_fdot2(h, h, square, false);
            }
        square += __shfl_xor(square, 32, 64);
        const float q_norm = wave_max(sqrtf(square) * pow2_field(254 - q_field)), k_big = kt < kt_last ? largest(kpre) : 0.0f, v_big = kt < kt_last ? largest(vpre) : 0.0f;
        auto weak = [](float x, int field) { return x > 0.0f && x * pow2_field(field) < 1.0f; };   // (below 2^-55)
        const bool weak_q = __any(weak(big, q_field));
        float v_weak = 0.0f;   // 1 / the largest of eight keys of the weakest feature that has one
        if (keys.first_key(kt) + 32 <= min(p.Sk, keys.end(kt)) && kt < kt_last) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float m = 0.0f;
#pragma unroll
                for (int i = 0; i < NG; i++)
#pragma unroll
                    for (int j = 0; j < 4; j++) m = fmaxf(m, fabsf(vpre[i][j][e]));
                v_weak = fmaxf(v_weak, m > 0.0f ? __builtin_amdgcn_rcpf(m) : 0.0f);
            }
            v_weak = wave_max(v_weak);
        }
#pragma unroll
        for (int j = 0; j < 2; j++)
            if (NEW && piece + j * hop < pieces) dst_k[piece + j * hop] = ck[j], dst_v[piece + j * hop] = cv[j];
        if (lane == 0) lds_big[0][w] = weak_q ? INFINITY : q_norm, lds_big[1][w] = k_big, lds_big[2][w] = v_big, lds_big[3][w] = v_weak;
        if (tid == 0) lds_odd = 0;
        __syncthreads();
        auto of_all = [&](int i) { return fmaxf(fmaxf(lds_big[i][0], lds_big[i][1]), fmaxf(lds_big[i][2], lds_big[i][3])); };
        k_field = up_field(of_all(1), 11), v_field = up_field(of_all(2), 12);
        c = p.scale * pow2_field(254 - q_field) * pow2_field(254 - k_field);
        odd = !(of_all(0) * p.scale * (sqrtf(D) * 0x1p-25f) * pow2_field(254 - k_field) < 0x1p-21f) || weak(of_all(1), k_field);
        odd = odd || (kt_first < kt_last && of_all(2) == 0.0f);   // (nothing that says what V's unit should be)
        // features of V that are 2^13 times weaker than the strongest: their lower numbers would lose bits
        odd = odd || of_all(3) * 0.5f > pow2_field(v_field);
    }

    f32x16 o[T];
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) o[t][r] = 0.0f;
    float m_run = -INFINITY, l_run = 0.0f;   // l and P are counted in 2^-14
    const float k_up = pow2_field(k_field), v_up = pow2_field(v_field);
    const int steps = odd ? 0 : (kt_last - kt_first + 1) / 2;
    for (int it = 0; it < steps; it++, kt += 2) {
        const int key0 = keys.first_key(kt);
        const bool live = kt < kt_last, edge = key0 + 32 > min(limit_first, keys.end(kt));   // edge: some row does not see all of the tile
        if (live) {
#pragma unroll
            for (int i = 0; i < NG; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    uint32_t h0, l0, h1, l1;
                    split_pair(kpre[i][j][0], kpre[i][j][1], k_up, h0, l0), split_pair(kpre[i][j][2], kpre[i][j][3], k_up, h1, l1);
                    const int dst = (4 * (g0 + 4 * i) + j) * KROW + 4 * c4;
                    *reinterpret_cast<u32x2 *>(&lds.pair.k[ks][0][dst]) = u32x2{h0, h1};
                    *reinterpret_cast<u32x2 *>(&lds.pair.k[ks][1][dst]) = u32x2{l0, l1};
                }
        }
        // (always, a tile again at the end: with a condition around them the wait for V below would be one for these too)
        load_rows(kpre, k_rows, min(kt + 2, kt_last));
        __syncthreads();   // K is in LDS; every wave is done with the last V
        f32x16 s;
        if (live) {
#pragma unroll
            for (int r = 0; r < 16; r++) s[r] = 0.0f;
#pragma unroll
            for (int j = 0; j < D / 16; j++) {
                Split8 kf;
                kf.hi = *reinterpret_cast<const half8_t *>(&lds.pair.k[ks][0][l32 * KROW + 16 * j + 8 * hb]);
                kf.lo = *reinterpret_cast<const half8_t *>(&lds.pair.k[ks][1][l32 * KROW + 16 * j + 8 * hb]);
                s = mfma3(kf, q[j], s);
            }
#pragma unroll
            for (int i = 0; i < NG; i++) {
                const int g = g0 + 4 * i, pos = 16 * (g / 4) + 8 * (g % 2) + 4 * (g % 4 / 2);
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    uint32_t h0, l0, h1, l1;
                    split_pair(vpre[i][0][e], vpre[i][1][e], v_up, h0, l0), split_pair(vpre[i][2][e], vpre[i][3][e], v_up, h1, l1);
                    const int f = 4 * c4 + e, dst = f / T * 40 + pos;
                    *reinterpret_cast<u32x2 *>(&lds.pair.vt[ks][0][f % T][dst]) = u32x2{h0, h1};
                    *reinterpret_cast<u32x2 *>(&lds.pair.vt[ks][1][f % T][dst]) = u32x2{l0, l1};
                }
            }
        }
        load_rows(vpre, v_rows, min(kt + 2, kt_last));
        __syncthreads();   // V is in LDS; every wave is done with K
        if (!live) continue;

        if (edge) {
#pragma unroll
            for (int r = 0; r < 16; r++)
                if (key0 + 8 * (r / 4) + 4 * hb + r % 4 >= min(limit, keys.end(kt))) s[r] = -INFINITY;
        }
        float mx = s[0];
#pragma unroll
        for (int r = 1; r < 16; r++) mx = fmaxf(mx, s[r]);
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64)) * c;
        const float m_new = fmaxf(m_run, mx), ref = ref_of(m_new);
        if (__any(m_new != m_run)) {
            const float alpha = expf(m_run - ref);
            l_run *= alpha;
#pragma unroll
            for (int t = 0; t < T; t++)
#pragma unroll
                for (int r = 0; r < 16; r++) o[t][r] *= alpha;
            m_run = m_new;
        }
#pragma unroll
        for (int r = 0; r < 16; r++) {   // 2^14 e^(s c - ref)
            s[r] = fast_exp2(fmaf(fmaf(s[r], c, -ref), 1.4426950408889634f, 14.0f));
            l_run += s[r];
        }
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const Split8 pf = split8([&](int i) { return s[8 * u + i]; }, 1.0f);
#pragma unroll
            for (int t = 0; t < T; t++) {
                Split8 vf;
                vf.hi = *reinterpret_cast<const half8_t *>(&lds.pair.vt[ks][0][t][l32 * 40 + 16 * u + 8 * hb]);
                vf.lo = *reinterpret_cast<const half8_t *>(&lds.pair.vt[ks][1][t][l32 * 40 + 16 * u + 8 * hb]);
                o[t] = mfma3(vf, pf, o[t]);
            }
        }
    }
    for (piece += 2 * hop; NEW && piece < pieces; piece += 4 * hop) {   // what is left of the append
        f32x4 rk[4], rv[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int i = min(piece + j * hop, pieces - 1);
            rk[j] = src_k[i], rv[j] = src_v[i];
        }
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (piece + j * hop < pieces) dst_k[piece + j * hop] = rk[j], dst_v[piece + j * hop] = rv[j];
    }
    // ---- the two key sets' results ---------------------------------------------------------------------------------
    l_run += __shfl_xor(l_run, 32, 64);
    if (hb == 0) lds_m[w][l32] = m_run, lds_l[w][l32] = l_run * 0x1p-14f;
    __syncthreads();   // (and every wave is done with V)
    const float m_other = lds_m[w ^ 2][l32], ref_all = ref_of(fmaxf(m_run, m_other)), v_down = pow2_field(254 - v_field);
    const float f_run = expf(m_run - ref_all), wgt = f_run * (v_down * 0x1p-14f);   // o is counted in 1 / (2^14 v_up)
    float *mine = &lds.rows[(kRows * rg + l32) * ROW];
#pragma unroll
    for (int set = 1; set >= 0; set--) {
        if (ks == set) {
            const float l_all = l_run * 0x1p-14f * f_run + lds_l[w ^ 2][l32] * expf(m_other - ref_all), unit = l_all * v_down;
            float sum = l_all;   // of the row's magnitudes: no number if one is none
#pragma unroll
            for (int r = 0; r < 16; r++) {
                vec *dst = reinterpret_cast<vec *>(mine + T * (8 * (r / 4) + 4 * hb + r % 4));
                vec x;
#pragma unroll
                for (int t = 0; t < T; t++) x[t] = o[t][r] * wgt;
                if (set == 0) {
                    x += *dst;
                    if (r == 0) sum *= 0.0f;
#pragma unroll
                    for (int t = 0; t < T; t++) sum += fabsf(x[t]);
                }
                *dst = x;
            }
            if (set == 0) {
                sum += __shfl_xor(sum, 32, 64);
                if (!(sum >= unit * kLeastOfRow) || sum == INFINITY) lds_odd = 1;
                if (hb == 0) lds_least[kRows * rg + l32] = l_all > 0.0f ? unit * kLeastOfFeature : INFINITY;
            }
        }
        __syncthreads();
    }
    odd = odd || lds_odd != 0;
    // A thread per feature and part of the rows: four of them, which is enough for all but a few tiles, then all.
    constexpr int N = 2 * kRows * D / kThreads;
    const int feature = tid % D, first = tid / D * N;
    for (int n = 4; !odd && kt_first < kt_last; n = N) {
        float most = -INFINITY;
#pragma unroll 4
        for (int r = 0; r < n; r++) most = fmaxf(most, fabsf(lds.rows[(first + r) * ROW + feature]) - lds_least[first + r]);
        const uint64_t strong = __ballot(most >= 0.0f);
        if (lane == 0) lds_strong[w] = strong;
        __syncthreads();
        const bool all = D == 128 ? ((lds_strong[0] | lds_strong[2]) & (lds_strong[1] | lds_strong[3])) == ~0ull
                                  : (lds_strong[0] | lds_strong[1] | lds_strong[2] | lds_strong[3]) == ~0ull;
        if (all) break;
        odd = n == N;
        __syncthreads();
    }
    if (odd) {   // for this row tile everything (again), in f32
        for (int i = 0; i < 2 && r0 + kRows * i < n_rows; i++) {
            __syncthreads();
            attend_tile<D, NEW>(p, lds.tile, bh, 2 * rt2 + i, split, kt_first, kt_last);
        }
        return;
    }
    const int64_t wb0 = (int64_t)bh * p.n_rt + 2 * rt2, n_wb = (int64_t)p.n_bh * p.n_rt;
#pragma unroll 4
    for (int j = 0; j < 2 * kRows * C4 / kThreads; j++) {
        const int f = j * kThreads + tid, r = f / C4, cc = f % C4, r32 = r % kRows, wr = r / kRows;   // waves wr and wr + 2 had the row
        if (r0 + kRows * wr >= n_rows) continue;
        f32x4 sum = *reinterpret_cast<const f32x4 *>(&lds.rows[r * ROW + 4 * cc]);
        const float m0 = lds_m[wr][r32], m1 = lds_m[wr + 2][r32], mm = fmaxf(m0, m1), ref = ref_of(mm);
        const float l = lds_l[wr][r32] * expf(m0 - ref) + lds_l[wr + 2][r32] * expf(m1 - ref);
        if (p.nsplit > 1) {
            const int64_t rec = split * n_wb + wb0 + wr;
            *reinterpret_cast<f32x4 *>(p.part_o + (rec * kRows + r32) * D + 4 * cc) = sum;
            if (cc == 0) p.part_ml[rec * 64 + r32] = mm, p.part_ml[rec * 64 + 32 + r32] = l;
        } else if (r0 + r < n_rows) {
#pragma unroll
            for (int e = 0; e < 4; e++) sum[e] = l > 0.0f ? sum[e] / l : 0.0f;
            *reinterpret_cast<f32x4 *>(p.out + q_row(r0 + r) + 4 * cc) = sum;
        }
    }
}

// The ranges of keys of a row tile: a thread per four features of a row.
template <int D>
__global__ __launch_bounds__(kThreads) void sdpa_prefill_f32_merge_kernel(PrefillF32 p) {
    const int64_t f = (int64_t)blockIdx.x * kThreads + threadIdx.x, n_wb = (int64_t)p.n_bh * p.n_rt, wb = f / (kRows * D / 4);
    const int r = (int)(f / (D / 4) % kRows), c = (int)(f % (D / 4));
    const int bh = (int)(wb / p.n_rt), rt = (int)(wb % p.n_rt), b = bh / p.Hkv, kvh = bh % p.Hkv, row = rt * kRows + r;
    if (row >= p.Sq * p.G) return;
    const float *ml = p.part_ml + wb * 64 + r, *po = p.part_o + (wb * kRows + r) * D + 4 * c;
    const int64_t ml_step = n_wb * 64, po_step = n_wb * kRows * D;
    float mm = -INFINITY, l = 0.0f;
    f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int s0 = 0; s0 < p.nsplit; s0 += 8) {   // eight ranges in flight at a time
        float m8[8], l8[8], top = mm;
        f32x4 o8[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int s = min(s0 + i, p.nsplit - 1);
            m8[i] = ml[s * ml_step], l8[i] = ml[s * ml_step + 32];
            o8[i] = *reinterpret_cast<const f32x4 *>(po + s * po_step);
        }
#pragma unroll
        for (int i = 0; i < 8; i++) top = fmaxf(top, m8[i]);
        const float ref = ref_of(top), keep = expf(mm - ref);
        sum *= keep, l *= keep, mm = top;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const bool there = s0 + i < p.nsplit;   // (the weight 0 alone would make a NaN of an infinity)
            const float wgt = there ? expf(m8[i] - ref) : 0.0f;
            l += wgt * l8[i];
#pragma unroll
            for (int e = 0; e < 4; e++) sum[e] += wgt * (there ? o8[i][e] : 0.0f);
        }
    }
    const int i = row / p.G, g = row - i * p.G;
#pragma unroll
    for (int e = 0; e < 4; e++) sum[e] = l > 0.0f ? sum[e] / l : 0.0f;
    *reinterpret_cast<f32x4 *>(p.out + (((int64_t)b * p.Hq + kvh * p.G + g) * p.Sq + i) * D + 4 * c) = sum;
}

template <int D, bool NEW>
int launch(const PrefillF32 &p, hipStream_t s) {
    if (p.n_rt2) hipLaunchKernelGGL((sdpa_prefill_f32x2_kernel<D, NEW>), dim3((unsigned)(p.n_bh * p.n_rt2 * p.nsplit)), dim3(kThreads), 0, s, p);
    else hipLaunchKernelGGL((sdpa_prefill_f32_kernel<D, NEW>), dim3((unsigned)(p.n_bh * p.n_rt * p.nsplit)), dim3(kThreads), 0, s, p);
    if (p.nsplit > 1)
        hipLaunchKernelGGL((sdpa_prefill_f32_merge_kernel<D>), dim3((unsigned)((int64_t)p.n_bh * p.n_rt * (kRows * D / 4 / kThreads))), dim3(kThreads), 0, s, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail("sdpa_prefill_f32 launch failed: %s", hipGetErrorString(e));
    return 0;
}

}  // namespace

// Ranges of keys for sdpa_prefill_f32x2_kernel: the number with the least expected time, in us.  1.5 (D = 64: 1.0) for each pair of
// tiles of the longest range, or of a compute unit's half of all tiles if that is more; where more than one workgroup shares a compute
// unit up to 1.9 times that again, and a quarter where not all are resident; 2.5 + 0.12 a range for the merge, and 0.85 for every
// 1024 blocks of 32 x 128 outputs and range.  55 drawn prompts, each timed at 1 .. 32 ranges: 1.2 % above the best of them on
// average; ranges of 4 or 16 tiles, as many as two workgroups per compute unit allow, were 2.9 % above (2 x 14 heads x 7 queries
// behind 401: 20.8 -> 18.7 us; 14 x 143 behind 1750: 30.2 -> 27.9; 3 x 32 x 79 behind 276: 30.9 -> 26.5).
static int64_t choose_pair_splits(const PrefillF32 &p, int D, int64_t tiles, int64_t n_wg, int64_t cus) {
    int64_t all = tiles * n_wg;
    if (p.causal) {
        all = 0;
        for (int rt = 0; rt < p.n_rt2; rt++) all += ((std::min(2 * kRows * (rt + 1), p.Sq * p.G) - 1) / p.G + p.Sk - p.Sq + 1 + 31) / 32;
        all *= p.n_bh;
    }
    const float pair = D == 64 ? 1.0f : 1.5f, busy = (float)all / (float)(4 * cus);
    int64_t best = 1;
    float best_time = 0.0f;
    for (int64_t n = 1; n <= kMaxSplits && (n == 1 || 2 * n <= tiles); n++) {
        const float per_unit = (float)(n_wg * n) / (float)cus, range = (float)(((tiles + n - 1) / n + 1) / 2);
        float time = range > busy ? range : busy;
        if (per_unit > 1.0f) time += 1.9f * range * std::min(1.0f, per_unit - 1.0f);
        if (per_unit > 2.0f) time += 0.25f * range * std::min(1.0f, per_unit / 2.0f - 1.0f);
        time *= pair;
        if (n > 1) time += 2.5f + 0.12f * n + 0.85f / 1024 / 128 * (float)((int64_t)p.n_bh * p.n_rt * D * n);
        if (n == 1 || time < best_time) best = n, best_time = time;
    }
    return best;
}

// 2 = not taken (the generic kernel runs): masks, other types and head sizes, rows that see no key, unaligned rows, a kv
// head of 4 GB or more.
int launch_sdpa_prefill_f32(const SdpaArgs &a, hipStream_t s) {
    if (a.q_dtype != TROCM_F32 || a.kv_fmt != TROCM_F32 || a.mask) return 2;
    if (a.D != 128 && a.D != 64) return 2;
    if (a.Sq < 2 || a.Sk < 1 || a.Hq % a.Hkv) return 2;
    if (a.causal && a.Sk < a.Sq) return 2;
    if (a.kv_stride_t < a.D || a.kv_stride_b % 4 || a.kv_stride_h % 4 || a.kv_stride_t % 4) return 2;
    if ((uintptr_t)a.q % 16 || (uintptr_t)a.k % 16 || (uintptr_t)a.v % 16 || (uintptr_t)a.out % 16) return 2;
    const int64_t G = a.Hq / a.Hkv;
    if (a.Sk >= (1ll << 30) || a.Sq >= (1ll << 30) || a.Sq * G >= (1ll << 30) || a.B * a.Hkv >= (1ll << 30)) return 2;
    if ((a.Sk + 96) * a.kv_stride_t >= (1ll << 30)) return 2;   // byte offsets of the rows a tile addresses are 32-bit

    PrefillF32 p;
    memset(&p, 0, sizeof(p));
    p.q = (const float *)a.q, p.k = (const float *)a.k, p.v = (const float *)a.v, p.out = (float *)a.out;
    p.kv_stride_b = a.kv_stride_b, p.kv_stride_h = a.kv_stride_h;
    p.kv_row_bytes = (uint32_t)(a.kv_stride_t * 4);
    p.Hq = (int)a.Hq, p.Hkv = (int)a.Hkv, p.Sq = (int)a.Sq, p.Sk = (int)a.Sk, p.G = (int)G;
    p.n_bh = (int)(a.B * a.Hkv), p.n_rt = (int)((a.Sq * G + kRows - 1) / kRows);
    p.causal = a.causal, p.scale = a.scale;

    // Pairs of f16 from 33 rows and 5 tiles on; 4 where half the compute units have a workgroup (3 x 32 heads x 117 queries 20.6 -> 18.2
    // us; but 14 x 107, whose four tiles go to a workgroup's four waves at once on the f32 instruction, 14.0, not 16.8).
    const int64_t tiles = (a.Sk + 31) / 32, cus = num_compute_units(), want = 2 * cus, n_rt2 = (a.Sq * G + 2 * kRows - 1) / (2 * kRows);
    const bool pairs = p.n_rt > 1 && (tiles >= 5 || (tiles == 4 && 2 * p.n_bh * n_rt2 > cus)) && a.scale >= 0x1p-16f && a.scale <= 0x1p16f;
    if (pairs) p.n_rt2 = (int)n_rt2;
    p.past = (int)a.Sk;
    if (a.k_new) {   // the last Sq tokens, stored to the cache by this launch
        if (a.kv_stride_t != a.D || a.Sk < a.Sq || !a.v_new) return 2;
        if ((uintptr_t)a.k_new % 16 || (uintptr_t)a.v_new % 16 || a.Sq > (1 << 20) || (int64_t)p.n_rt * kMaxSplits >= (1 << 18)) return 2;
        p.k_new = (const float *)a.k_new, p.v_new = (const float *)a.v_new;
        p.past = (int)(a.Sk - a.Sq), p.n_new = (int)a.Sq;
    }
    // (as the launch counts them: the call's rows begin a tile of their own)
    const int64_t cut_tiles = (p.past + 31) / 32 + (p.n_new + 31) / 32;
    const int64_t n_wb = (int64_t)p.n_bh * p.n_rt, n_wg = pairs ? (int64_t)p.n_bh * p.n_rt2 : n_wb;
    int64_t ns;
    if (pairs) {
        ns = n_wg < want ? choose_pair_splits(p, (int)a.D, cut_tiles, n_wg, cus) : 1;
    } else {
        // Ranges of four tiles, one for each wave, where all of them are at work at once or there are few; otherwise the next longer ones.
        // (A call with its append, us, ranges of five | of four: 2 x 32 heads over 8, 2 queries behind 618 tokens 19.7 | 15.2, 1 x 5 behind
        // 1910 21.4 | 17.0, 4 x 32 over 32, 6 behind 395 27.1 | 24.0; of four, more than a workgroup per unit, | of five: 3 x 64 over 8, 4 behind
        // 1405 24.8 | 22.8; a merge for two ranges | none: 6 x 4 over 184 tokens of 64 features 10.9 | 10.3.)
        auto ranges_of = [&](int64_t t) {
            const int64_t most = n_wg < want ? (want + n_wg - 1) / n_wg : 1, fours = t < 8 ? 1 : (t + 3) / 4;
            const int64_t n = std::min(most, n_wg * fours <= cus || (fours <= 4 && n_wg * fours <= want) ? fours : t / 4), longest = (t + n - 1) / n;
            return (t + longest - 1) / longest;   // (none of them empty)
        };
        ns = ranges_of(cut_tiles);
        // An append launch instead where one tile more costs more than that launch, by the rounds that four waves take a range's tiles in (us;
        // `alone` on a compute unit or two of them sharing it, the last of five tiles in a round of its own, and `phase` where some wait for
        // others to end).  Fitted to 40 calls of 5 queries of 16 to 192 kv heads over 8 to 24 whole tiles, each with an append launch and
        // without: 0.6 us (64 features) and 1.6 off, and the slower side in two of the 40 (1.012, 1.046 of the faster).  Append launch | in here, us: 32
        // heads over 32, 10 queries behind 100 tokens 13.3 | 15.8, 3 x 32 over 32, 5 behind 244 18.1 | 20.4, 2 x 32, 5 behind 500 18.9 | 20.7, 16 x 32, 4
        // behind 760 84.1 | 86.4; kept: 3 x 32, 5 behind 756 35.3 | 28.3, 4 x 32, 5 behind 372 25.5 | 23.2, 14 over 2, 20 behind 90 13.7 | 11.7.
        struct Rounds { float alone, shared, fifth, phase, range, append; };
        const Rounds c = a.D == 64 ? Rounds{2.6f, 5.2f, 2.6f, 1.3f, 0.1f, 2.3f} : Rounds{5.2f, 12.8f, 8.0f, 2.5f, 0.2f, 3.1f};
        auto expected = [&](int64_t t) {
            const int64_t n = ranges_of(t), longest = (t + n - 1) / n, rounds = (longest + 3) / 4, wgs = n_wg * n, full = wgs / (2 * cus), rest = wgs - 2 * cus * full;
            const float alone = c.alone * (float)rounds, shared = c.shared * (float)rounds - (longest > 4 && longest % 4 == 1 ? c.fifth : 0.0f);
            return (float)full * shared + (rest > cus ? shared : rest > 0 ? alone : 0.0f) + c.phase * (float)(full + (rest > 0)) + c.range * (float)n;
        };
        if (cut_tiles > tiles && expected(cut_tiles) > expected(tiles) + c.append) return 2;
    }
    ns = ns < kMaxSplits ? ns : kMaxSplits;
    p.paired = pairs && a.causal && n_wg <= want;
    const size_t per_split = (size_t)n_wb * (kRows * a.D + 64) * sizeof(float);
    const size_t avail = a.workspace && a.workspace_bytes > kWsCounterBytes + 256 ? a.workspace_bytes - kWsCounterBytes - 256 : 0;
    if (ns > 1 && (size_t)ns * per_split > avail) ns = (int64_t)(avail / per_split);
    p.nsplit = ns > 1 ? (int)ns : 1;
    if (p.nsplit > 1) {
        char *base = (char *)a.workspace + kWsCounterBytes;
        base += (256 - ((uintptr_t)base & 255)) & 255;
        p.part_o = (float *)base;
        p.part_ml = p.part_o + (size_t)p.nsplit * n_wb * kRows * a.D;
    }
    if (n_wb * p.nsplit >= (1ll << 31) || n_wb * (kRows * a.D / 4 / kThreads) >= (1ll << 31)) return 2;
    if (a.k_new) return a.D == 128 ? launch<128, true>(p, s) : launch<64, true>(p, s);
    return a.D == 128 ? launch<128, false>(p, s) : launch<64, false>(p, s);
}

}  // namespace trocm
