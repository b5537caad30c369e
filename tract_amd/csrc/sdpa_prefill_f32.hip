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
// Bound by the f32 matrix rate: 1000 causal queries of 32 heads over 8 kv heads (D = 128) are 8.2 GFLOP, 54 us at the 152
// TFLOP/s that a large f32 matrix product reaches; a call with its append takes 102.5 us (105.2 while 28 bytes per lane were
// in scratch memory; the diagonal tiles are computed whole, and the last workgroups leave compute units idle).  The generic
// kernel, a wave per query with scalar fused multiply-adds and every key row read once per query, took 9040 us.  Error
// against f64 over the same call 3.3e-7 (generic: 3.8e-7).
#include <hip/hip_runtime.h>
#include <string.h>
#include "common.h"

namespace trocm {
namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kRows = 32, kWaves = 4, kThreads = 64 * kWaves, kMaxSplits = 16;

struct PrefillF32 {
    const float *q, *k, *v;
    float *out;
    float *part_o;    // [nsplit][n_wg][32][D], not normalised
    float *part_ml;   // [nsplit][n_wg][64]: maxima, then sums
    int64_t kv_stride_b, kv_stride_h;   // elements
    uint32_t kv_row_bytes, kv_bytes;    // bytes between token rows; bytes of one kv head's rows, from the first to the last
    int Hq, Hkv, Sq, Sk, G;
    int n_bh, n_rt, nsplit;             // batch * kv_heads, row tiles per kv head
    int causal;
    float scale;
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
__device__ __forceinline__ bool finite(float x) { return __builtin_isfinite(x); }

// the weight exp(m - ref) of a partial result whose maximum is m; nothing seen: m = -inf, weight 0 whatever ref is
__device__ __forceinline__ float ref_of(float m) { return m == -INFINITY ? 0.0f : m; }

template <int D>
__global__ __launch_bounds__(kThreads, 2) void sdpa_prefill_f32_kernel(PrefillF32 p) {
    constexpr int T = D / 32, KJ = D / 8, ROW = D + 4;   // (ROW: 16 rows of a 128-bit LDS pass in 16 distinct bank groups)
    typedef typename VecOf<T>::type vec;
    __shared__ __attribute__((aligned(16))) float lds[kWaves * kRows * ROW];   // q; then the waves' outputs
    __shared__ float lds_m[kWaves][kRows], lds_l[kWaves][kRows];

    const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hb = lane >> 5;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int bh = blockIdx.x % p.n_bh, rest = blockIdx.x / p.n_bh;
    const int split = rest % p.nsplit, rt = p.n_rt - 1 - rest / p.nsplit;
    const int b = bh / p.Hkv, kvh = bh % p.Hkv;
    const int n_rows = p.Sq * p.G, r0 = rt * kRows;
    auto q_row = [&](int r) {   // offset of row r's query (and output) in elements
        const int i = r / p.G, g = r - i * p.G;
        return (((int64_t)b * p.Hq + kvh * p.G + g) * p.Sq + i) * D;
    };
    // keys [0, limit) are visible to a row; the tile as a whole sees n_vis
    auto limit_of = [&](int r) { return p.causal ? min(r, n_rows - 1) / p.G + (p.Sk - p.Sq) + 1 : p.Sk; };
    const int limit = limit_of(r0 + l32), limit_first = limit_of(r0), n_vis = limit_of(r0 + kRows - 1);
    const int tiles = (n_vis + 31) / 32, per_split = (tiles + p.nsplit - 1) / p.nsplit;
    const int kt_end = min(tiles, (split + 1) * per_split);

    // rows past the last key read as zeros: the buffer ends with that row
    const float *k_head = p.k + b * p.kv_stride_b + kvh * p.kv_stride_h, *v_head = p.v + b * p.kv_stride_b + kvh * p.kv_stride_h;
    const __amdgpu_buffer_rsrc_t k_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(k_head), 0, p.kv_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t v_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(v_head), 0, p.kv_bytes, 0x00020000);

    f32x4 kreg[KJ];
    vec vreg[16];
    auto load_k = [&](int kt) {
        const uint32_t off = (uint32_t)(32 * kt + l32) * p.kv_row_bytes + 16 * hb;
#pragma unroll
        for (int j = 0; j < KJ; j++) kreg[j] = buffer_f32x4(k_rsrc, off + 32 * j);
    };
    auto load_v = [&](int kt) {
        const uint32_t off = (uint32_t)(32 * kt + 4 * hb) * p.kv_row_bytes + 4 * T * l32;
#pragma unroll
        for (int i = 0; i < 16; i++) vreg[i] = buffer_vec<T>(v_rsrc, off + (uint32_t)(8 * (i / 4) + i % 4) * p.kv_row_bytes);
    };

    int kt = split * per_split + w;
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

        const bool edge = 32 * kt + 32 > limit_first;   // some row does not see all of the tile
#pragma unroll
        for (int r = 0; r < 16; r++) s[r] *= p.scale;
        if (edge) {
#pragma unroll
            for (int r = 0; r < 16; r++)
                if (32 * kt + 8 * (r / 4) + 4 * hb + r % 4 >= limit) s[r] = -INFINITY;
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
                    const bool seen = 32 * kt + kk < limit;
                    const uint32_t off = (uint32_t)(32 * kt + kk) * p.kv_row_bytes;
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const vec x = buffer_vec<T>(v_rsrc, off + 4 * T * (8 * (r / 4) + 4 * hb + r % 4));
#pragma unroll
                        for (int t = 0; t < T; t++)
                            o[t][r] = fmaf(pk, seen && !finite(x[t]) ? x[t] : 0.0f, o[t][r]);
                    }
                }
#pragma unroll
                for (int i = 0; i < 16; i++)
#pragma unroll
                    for (int t = 0; t < T; t++) vreg[i][t] = finite(vreg[i][t]) ? vreg[i][t] : 0.0f;
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

// The ranges of keys of one row tile per workgroup.
template <int D>
__global__ __launch_bounds__(kThreads) void sdpa_prefill_f32_merge_kernel(PrefillF32 p) {
    const int tid = threadIdx.x;
    const int64_t wb = blockIdx.x, n_wb = (int64_t)p.n_bh * p.n_rt;
    const int bh = (int)(wb / p.n_rt), rt = (int)(wb % p.n_rt), b = bh / p.Hkv, kvh = bh % p.Hkv;
    for (int f = tid; f < kRows * D / 4; f += kThreads) {
        const int r = f / (D / 4), c = f % (D / 4), row = rt * kRows + r;
        if (row >= p.Sq * p.G) continue;
        float mm = -INFINITY;
        for (int s = 0; s < p.nsplit; s++) mm = fmaxf(mm, p.part_ml[(s * n_wb + wb) * 64 + r]);
        const float ref = ref_of(mm);
        float l = 0.0f;
        f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int s = 0; s < p.nsplit; s++) {
            const float *ml = p.part_ml + (s * n_wb + wb) * 64;
            const float wgt = expf(ml[r] - ref);
            l += wgt * ml[32 + r];
            sum += wgt * *reinterpret_cast<const f32x4 *>(p.part_o + ((s * n_wb + wb) * kRows + r) * D + 4 * c);
        }
        const int i = row / p.G, g = row - i * p.G;
#pragma unroll
        for (int e = 0; e < 4; e++) sum[e] = l > 0.0f ? sum[e] / l : 0.0f;
        *reinterpret_cast<f32x4 *>(p.out + (((int64_t)b * p.Hq + kvh * p.G + g) * p.Sq + i) * D + 4 * c) = sum;
    }
}

template <int D>
int launch(const PrefillF32 &p, hipStream_t s) {
    const int64_t n_wb = (int64_t)p.n_bh * p.n_rt;
    hipLaunchKernelGGL((sdpa_prefill_f32_kernel<D>), dim3((unsigned)(n_wb * p.nsplit)), dim3(kThreads), 0, s, p);
    if (p.nsplit > 1) hipLaunchKernelGGL((sdpa_prefill_f32_merge_kernel<D>), dim3((unsigned)n_wb), dim3(kThreads), 0, s, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail("sdpa_prefill_f32 launch failed: %s", hipGetErrorString(e));
    return 0;
}

}  // namespace

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
    if ((a.Sk + 32) * a.kv_stride_t >= (1ll << 30)) return 2;   // byte offsets of the rows a tile addresses are 32-bit

    PrefillF32 p;
    memset(&p, 0, sizeof(p));
    p.q = (const float *)a.q, p.k = (const float *)a.k, p.v = (const float *)a.v, p.out = (float *)a.out;
    p.kv_stride_b = a.kv_stride_b, p.kv_stride_h = a.kv_stride_h;
    p.kv_row_bytes = (uint32_t)(a.kv_stride_t * 4), p.kv_bytes = (uint32_t)(((a.Sk - 1) * a.kv_stride_t + a.D) * 4);
    p.Hq = (int)a.Hq, p.Hkv = (int)a.Hkv, p.Sq = (int)a.Sq, p.Sk = (int)a.Sk, p.G = (int)G;
    p.n_bh = (int)(a.B * a.Hkv), p.n_rt = (int)((a.Sq * G + kRows - 1) / kRows);
    p.causal = a.causal, p.scale = a.scale;

    // Two workgroups fit a compute unit.  Fewer than that: ranges of keys, each of at least a tile per wave.
    const int64_t n_wb = (int64_t)p.n_bh * p.n_rt, want = 2 * (int64_t)num_compute_units(), tiles = (a.Sk + 31) / 32;
    int64_t ns = n_wb < want ? (want + n_wb - 1) / n_wb : 1;
    ns = ns < tiles / kWaves ? ns : tiles / kWaves;
    ns = ns < kMaxSplits ? ns : kMaxSplits;
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
    if (n_wb * p.nsplit >= (1ll << 31)) return 2;
    return a.D == 128 ? launch<128>(p, s) : launch<64>(p, s);
}

}  // namespace trocm
