// Attention of one f32 query token per sequence, 3 to 16 query heads per kv head, over plain f32 rows: gfx950.
//
// The query heads of a kv head are the 16 columns of v_mfma_f32_16x16x4_f32 tiles (f32 operands, f32
// accumulation), so that a K or V element that has arrived feeds all of them with one instruction:
//
//   S^T[key, head] = K . q^T    A = K: lane (key = lane % 16, g = lane / 16) holds features 16 j + 4 g .. + 3 of its key,
//                               B = q, the same features (the order inside the contraction is free)
//   O^T[d, head]   = V^T . P^T  register r of S^T is key 4 g + r: exactly the B operand of the step that contracts the keys
//                               4 g + r of all g, so P needs no transposition; A = V of those keys, lane % 16 = a run of
//                               D / 16 features
//
// K and V go from memory straight into those registers, the next tile's K requested when this tile's is used up, the next
// V after the products with this one.  A tile of 16 keys is 2048 matrix cycles against 16 KB (D = 128): 32 bytes per cycle and
// compute unit, where HBM gives 11.  Waves take the tiles of a workgroup's range in turn and are merged through LDS; several
// ranges (`nsplit`) are merged by the workgroup that arrives last.
//
// Bound by HBM where the launch is long (13 x 10082 tokens, 64 heads over 8: 216 us for 1.07 GB, 5.0 TB/s), by the chain of a
// short launch else (1 x 160 tokens 8.8).  The vector kernel (sdpa_decode.hip) parks K in LDS, reads it back once per query head
// and multiplies on the vector ALU, 16 multiply-adds per lane and 16 bytes of K at 8 heads: 326 us and 21.4 (with two launches
// that rotated q and k); more than 8 heads per kv head ran on the generic kernel (32 over 2, 4000 tokens 4220 us, 16.0 now).
// Forms that were slower than the vector kernel and are not here: one head per kv head from the same registers, and sixteen
// waves of one workgroup with a tile each for short contexts (250 tokens, 32 heads over 8: 12.2 us; four waves and a merge 7.9).
#include <hip/hip_runtime.h>
#include "decode_common.h"

namespace trocm {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kMaxSplitsF32 = 32;

struct DecodeF32 {
    const float *q, *k, *v, *k_new, *v_new;   // k_new, v_new: dense [B, Hkv, D], the token new_pos (NULL: none)
    float *out;
    float *part_o;    // [nsplit][B * Hkv][G][D], not normalised
    float *part_ml;   // [nsplit][B * Hkv][G][2]: maximum (log2 units), sum
    int *counters;
    const float *rope_cos, *rope_sin;   // != NULL: q and k_new are rotated on the way in
    int64_t rope_stride_b;
    int64_t kv_stride_b, kv_stride_h;   // elements
    uint32_t kv_row_bytes, kv_bytes;    // bytes between token rows; bytes of one kv head's rows, from the first to the last
    int Hq, Hkv, T, G, new_pos, nsplit;
    float scale_log2;
};

__device__ __forceinline__ float ref_of(float m) { return m == -INFINITY ? 0.0f : m; }
// ApplyRope's element: every product and the sum rounded by itself
__device__ __forceinline__ f32x4 rotated(f32x4 x, f32x4 partner, f32x4 c, f32x4 s, bool upper) {
#pragma clang fp contract(off)
    f32x4 y;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const float xe = x[e], pe = partner[e], ce = c[e], se = s[e];
        y[e] = xe * ce + (upper ? pe : -pe) * se;
    }
    return y;
}
__device__ __forceinline__ f32x4 load_x4(const float *p) { return *reinterpret_cast<const f32x4 *>(p); }

template <int D>
__global__ __launch_bounds__(kThreads, 2) void sdpa_decode_f32_kernel(DecodeF32 p) {
    constexpr int KJ = D / 16, T4 = D / 64, C4 = D / 4, R = 16, ROW = D + 4;
    // q, then the waves' outputs (a wave's rows G apart: only real heads are combined)
    __shared__ __attribute__((aligned(16))) float lds[kWaves * R * ROW];
    __shared__ __attribute__((aligned(16))) float lds_new[2 * D];
    __shared__ float lds_m[kWaves][R], lds_l[kWaves][R];

    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int split = blockIdx.x, kvh = blockIdx.y, b = blockIdx.z, bh = b * p.Hkv + kvh;
    const int tiles = (p.T + 15) / 16, step = kWaves * p.nsplit;

    const float *k_head = p.k + b * p.kv_stride_b + kvh * p.kv_stride_h, *v_head = p.v + b * p.kv_stride_b + kvh * p.kv_stride_h;
    // rows past the last token read as zeros: the buffer ends with that row
    const __amdgpu_buffer_rsrc_t k_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(k_head), 0, p.kv_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t v_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(v_head), 0, p.kv_bytes, 0x00020000);
    constexpr int kNt = 2;   // non-temporal: K and V are read once
    f32x4 kreg[KJ], vreg[4][T4];
    auto load_k = [&](int tile) {
        const uint32_t off = (uint32_t)(16 * tile + l16) * p.kv_row_bytes + 16 * g;
#pragma unroll
        for (int j = 0; j < KJ; j++) kreg[j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(k_rsrc, off + 64 * j, 0, kNt));
    };
    auto load_v = [&](int tile) {
        const uint32_t off = (uint32_t)(16 * tile + 4 * g) * p.kv_row_bytes + 16 * T4 * l16;
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int t = 0; t < T4; t++)
                vreg[r][t] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(v_rsrc, off + r * p.kv_row_bytes + 16 * t, 0, kNt));
    };

    int tile = split * kWaves + w;
    if (tile < tiles) load_k(tile), load_v(tile);

    const float *cos_row = p.rope_cos + b * p.rope_stride_b, *sin_row = p.rope_sin + b * p.rope_stride_b;
    const int64_t q_row0 = ((int64_t)b * p.Hq + (int64_t)kvh * p.G) * D;
    // a chunk of four features of a row, rotated where the call says so
    auto chunk = [&](const float *row, int c) {
        f32x4 x = load_x4(row + 4 * c);
        if (p.rope_cos) x = rotated(x, load_x4(row + 4 * (c ^ (C4 / 2))), load_x4(cos_row + 4 * c), load_x4(sin_row + 4 * c), c >= C4 / 2);
        return x;
    };
    for (int i = tid; i < R * C4; i += kThreads) {
        const int r = i / C4, c = i % C4;
        *reinterpret_cast<f32x4 *>(&lds[r * ROW + 4 * c]) = chunk(p.q + q_row0 + (int64_t)min(r, p.G - 1) * D, c);
    }
    if (p.k_new && tid < 2 * C4) {
        const int c = tid % C4;
        const int64_t new_row = (int64_t)bh * D;
        const f32x4 x = tid < C4 ? chunk(p.k_new + new_row, c) : load_x4(p.v_new + new_row + 4 * c);
        *reinterpret_cast<f32x4 *>(&lds_new[(tid < C4 ? 0 : D) + 4 * c]) = x;
        if (split == 0) {
            char *dst = reinterpret_cast<char *>(const_cast<float *>(tid < C4 ? k_head : v_head)) + (int64_t)p.new_pos * p.kv_row_bytes;
            *reinterpret_cast<f32x4 *>(dst + 16 * c) = x;
        }
    }
    __syncthreads();

    // element r of o[t]: feature (D / 16) (4 g + r) + t of head l16.  D = 64: two sums of half the keys each, 9 to 17 % closer to 64 bits than one
    constexpr int NO = D == 64 ? 2 : 1;
    f32x4 o_part[NO][4 * T4];
    f32x4 (&o)[4 * T4] = o_part[0];
#pragma unroll
    for (int n = 0; n < NO; n++)
#pragma unroll
        for (int t = 0; t < 4 * T4; t++) o_part[n][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    float m_run = -INFINITY, l_run = 0.0f;   // of head l16 (the sum: over this lane's keys only)

    const float *q_frag = &lds[l16 * ROW + 4 * g];
    for (; tile < tiles; tile += step) {
        const bool has_new = p.new_pos >= 16 * tile && p.new_pos < 16 * tile + 16;   // the row comes from the step's input
        if (has_new) {
#pragma unroll
            for (int j = 0; j < KJ; j++) {
                const f32x4 x = load_x4(&lds_new[16 * j + 4 * g]);
                if (16 * tile + l16 == p.new_pos) kreg[j] = x;
            }
        }
        const bool more = tile + step < tiles;
        f32x4 part[4];   // (four sums of a quarter of the features each: a third less rounding than in one)
#pragma unroll
        for (int e = 0; e < 4; e++) part[e] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < KJ; j++) {
            const f32x4 qf = load_x4(q_frag + 16 * j);
#pragma unroll
            for (int e = 0; e < 4; e++) part[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(kreg[j][e], qf[e], part[e], 0, 0, 0);
        }
        f32x4 s = (part[0] + part[1]) + (part[2] + part[3]);
        __builtin_amdgcn_sched_barrier(0);
        if (more) load_k(tile + step);
        __builtin_amdgcn_sched_barrier(0);
        f32x4 scaled = s * p.scale_log2;
        const bool edge = 16 * tile + 16 > p.T;
        if (edge) {
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (16 * tile + 4 * g + r >= p.T) scaled[r] = -INFINITY;
        }
        float mx = fmaxf(fmaxf(scaled[0], scaled[1]), fmaxf(scaled[2], scaled[3]));
        if (__any(mx > m_run)) {   // (rarely after the first tiles)
            mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            const float m_new = fmaxf(m_run, mx), alpha = fast_exp2(m_run - ref_of(m_new));
            l_run *= alpha;
#pragma unroll
            for (int n = 0; n < NO; n++)
#pragma unroll
                for (int t = 0; t < 4 * T4; t++) o_part[n][t] *= alpha;
            m_run = m_new;
        }
        const float ref = ref_of(m_run);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            s[r] = fast_exp2(scaled_from(s[r], p.scale_log2, scaled[r], ref));
            if (edge && 16 * tile + 4 * g + r >= p.T) s[r] = 0.0f;
            l_run += s[r];
        }
        if (has_new) {
#pragma unroll
            for (int t = 0; t < T4; t++) {
                const f32x4 x = load_x4(&lds_new[D + 4 * T4 * l16 + 4 * t]);
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (16 * tile + 4 * g + r == p.new_pos) vreg[r][t] = x;
            }
        }
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int t = 0; t < 4 * T4; t++) o_part[r % NO][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(vreg[r][t / 4][t % 4], s[r], o_part[r % NO][t], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (more) load_v(tile + step);
    }

    if constexpr (NO == 2) {
#pragma unroll
        for (int t = 0; t < 4 * T4; t++) o[t] += o_part[1][t];
    }

    // ---- the waves' results: out = sum_w 2^(m_w - M) O_w / sum_w 2^(m_w - M) l_w ---------------------------------
    l_run += __shfl_xor(l_run, 16, 64);
    l_run += __shfl_xor(l_run, 32, 64);
    if (g == 0) lds_m[w][l16] = m_run, lds_l[w][l16] = l_run;
    __syncthreads();   // (and every wave is done with q)
    const int G = p.G;
    if (l16 < G) {   // element r of o[t] is feature (D / 16) (4 g + r) + t: four consecutive t make a 16-byte piece
        float *mine = &lds[(w * G + l16) * ROW];
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int t = 0; t < T4; t++)
                *reinterpret_cast<f32x4 *>(mine + 4 * T4 * (4 * g + r) + 4 * t) = f32x4{o[4 * t][r], o[4 * t + 1][r], o[4 * t + 2][r], o[4 * t + 3][r]};
    }
    __syncthreads();
    const int64_t n_bh = (int64_t)gridDim.z * p.Hkv, rec = (split * n_bh + bh) * G;
    float *out = p.out + q_row0;
    for (int i = tid; i < G * C4; i += kThreads) {
        const int r = i / C4, c = i % C4;
        float mm = lds_m[0][r];
#pragma unroll
        for (int j = 1; j < kWaves; j++) mm = fmaxf(mm, lds_m[j][r]);
        const float ref = ref_of(mm);
        f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
        float l = 0.0f;
#pragma unroll
        for (int j = 0; j < kWaves; j++) {
            const float f = fast_exp2(lds_m[j][r] - ref);
            sum += f * load_x4(&lds[(j * G + r) * ROW + 4 * c]);
            l += f * lds_l[j][r];
        }
        if (p.nsplit == 1) {
#pragma unroll
            for (int e = 0; e < 4; e++) sum[e] = l > 0.0f ? sum[e] / l : 0.0f;
            *reinterpret_cast<f32x4 *>(out + r * D + 4 * c) = sum;
        } else {   // write-through stores: visible to every compute unit when they complete
            const float s0 = sum[0], s1 = sum[1], s2 = sum[2], s3 = sum[3];
            uint64_t *po = reinterpret_cast<uint64_t *>(p.part_o + (rec + r) * D + 4 * c);
            auto pair = [](float lo, float hi) { return (uint64_t)__builtin_bit_cast(uint32_t, lo) | (uint64_t)__builtin_bit_cast(uint32_t, hi) << 32; };
            __hip_atomic_store(po, pair(s0, s1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(po + 1, pair(s2, s3), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (c == 0)
                __hip_atomic_store(reinterpret_cast<uint64_t *>(p.part_ml + (rec + r) * 2), pair(mm, l), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if (p.nsplit == 1) return;

    // ---- the last workgroup of this sequence-head to arrive merges the ranges ------------------------------------
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this thread's partial stores have completed
    __syncthreads();                                     // ... and so have the whole workgroup's
    __shared__ int s_last;
    if (tid == 0) {
        const int arrived = __hip_atomic_fetch_add(p.counters + bh, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = arrived == p.nsplit - 1;
        if (s_last) __hip_atomic_store(p.counters + bh, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!s_last) return;
    auto aload = [](const float *a) { return __hip_atomic_load(reinterpret_cast<const uint64_t *>(a), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    auto lo_of = [](uint64_t x) { return __builtin_bit_cast(float, (uint32_t)x); };
    auto hi_of = [](uint64_t x) { return __builtin_bit_cast(float, (uint32_t)(x >> 32)); };
    __shared__ float lds_wt[R][kMaxSplitsF32];
    for (int i = tid; i < G * kMaxSplitsF32; i += kThreads) {   // thread (head, range): whole groups of 32 lanes share a head
        const int r = i / kMaxSplitsF32, sp = i % kMaxSplitsF32;
        const uint64_t ml = aload(p.part_ml + ((min(sp, p.nsplit - 1) * n_bh + bh) * G + r) * 2);
        const float m = lo_of(ml);
        float mm = m;
#pragma unroll
        for (int d = 1; d < 32; d <<= 1) mm = fmaxf(mm, __shfl_xor(mm, d, 64));
        const float f = sp < p.nsplit ? fast_exp2(m - ref_of(mm)) : 0.0f;
        float ll = hi_of(ml) * f;
#pragma unroll
        for (int d = 1; d < 32; d <<= 1) ll += __shfl_xor(ll, d, 64);
        lds_wt[r][sp] = ll > 0.0f ? f / ll : 0.0f;
    }
    __syncthreads();
    for (int i = tid; i < G * C4; i += kThreads) {
        const int r = i / C4, c = i % C4;
        f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
        const float *po = p.part_o + ((int64_t)bh * G + r) * D + 4 * c;
        const int64_t po_step = n_bh * G * D;
        for (int s0 = 0; s0 < p.nsplit; s0 += 8) {
            uint64_t x[8][2];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const float *a = po + min(s0 + u, p.nsplit - 1) * po_step;
                x[u][0] = aload(a), x[u][1] = aload(a + 2);
            }
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const bool there = s0 + u < p.nsplit;   // (the weight 0 alone would make a NaN of an infinity)
                const float f = there ? lds_wt[r][s0 + u] : 0.0f;
                if (!there) x[u][0] = x[u][1] = 0;
                sum[0] = fmaf(f, lo_of(x[u][0]), sum[0]), sum[1] = fmaf(f, hi_of(x[u][0]), sum[1]);
                sum[2] = fmaf(f, lo_of(x[u][1]), sum[2]), sum[3] = fmaf(f, hi_of(x[u][1]), sum[3]);
            }
        }
        *reinterpret_cast<f32x4 *>(out + r * D + 4 * c) = sum;
    }
}

template <int D>
int launch(const DecodeF32 &p, int B, hipStream_t s) {
    hipLaunchKernelGGL((sdpa_decode_f32_kernel<D>), dim3((unsigned)p.nsplit, (unsigned)p.Hkv, (unsigned)B), dim3(kThreads), 0, s, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail("sdpa_decode_f32 launch failed: %s", hipGetErrorString(e));
    return 0;
}

}  // namespace

// Where it is faster than the vector kernel (us of a step, there | here): 128 features from 3 heads per kv head on (24 over 8,
// 6 x 3500 tokens 44.7 | 39.0, 1 x 250 10.6 | 8.0; two heads, 32 over 16, 1 x 700 8.5 | 10.0, 6 x 3500 93 | 96), 64 features
// from 5 on (14 over 2, 1 x 250 9.6 | 6.3; four, 32 over 8, 24 x 600 14.2 | 16.2).  Up to 32 ranges per sequence-head are merged here: one
// or two of them over more than 8192 tokens each take the vector kernel's many ranges and its merge launch (8 heads over one,
// 30000 tokens 32.4 | 41.8).
// 2 = not taken: masks, other types and head sizes, more than 16 heads per kv head, unaligned rows, a kv head of 4 GB or more;
// an output that lies over rows which other workgroups still read (the caller then stores the token and rotates first).
int launch_sdpa_decode_f32(const SdpaArgs &a, hipStream_t s) {
    if (a.Sq != 1 || a.q_dtype != TROCM_F32 || a.kv_fmt != TROCM_F32 || a.mask) return 2;
    if (a.D != 128 && a.D != 64) return 2;
    if (a.Sk < 1 || a.Hq % a.Hkv || a.Hq / a.Hkv > 16 || a.Hq / a.Hkv < (a.D == 128 ? 3 : 5)) return 2;
    if (a.kv_stride_t < a.D || a.kv_stride_b % 4 || a.kv_stride_h % 4 || a.kv_stride_t % 4) return 2;
    if ((uintptr_t)a.q % 16 || (uintptr_t)a.k % 16 || (uintptr_t)a.v % 16 || (uintptr_t)a.out % 16) return 2;
    if (a.Sk >= (1ll << 30) || (a.Sk + 16) * a.kv_stride_t >= (1ll << 30)) return 2;   // byte offsets of the rows a tile addresses are 32-bit
    const int64_t BH = a.B * a.Hkv;
    if (a.B > 65535 || a.Hkv > 65535) return 2;
    const size_t q_bytes = (size_t)a.B * a.Hq * a.D * 4, new_bytes = (size_t)BH * a.D * 4;
    if (a.k_new) {
        if (!a.v_new || (uintptr_t)a.k_new % 16 || (uintptr_t)a.v_new % 16) return 2;
        if (ranges_meet(a.out, q_bytes, a.k_new, new_bytes) || ranges_meet(a.out, q_bytes, a.v_new, new_bytes)) return 2;
    }
    if (a.rope_cos) {
        const size_t rope_bytes = (size_t)((a.B - 1) * a.rope_stride_b + a.D) * 4;
        if (!a.rope_sin || (uintptr_t)a.rope_cos % 16 || (uintptr_t)a.rope_sin % 16 || a.rope_stride_b % 4) return 2;
        if (ranges_meet(a.out, q_bytes, a.rope_cos, rope_bytes) || ranges_meet(a.out, q_bytes, a.rope_sin, rope_bytes)) return 2;
    }
    if (a.out != a.q && ranges_meet(a.out, q_bytes, a.q, q_bytes)) return 2;

    DecodeF32 p;
    memset(&p, 0, sizeof(p));
    p.q = (const float *)a.q, p.k = (const float *)a.k, p.v = (const float *)a.v, p.out = (float *)a.out;
    p.k_new = (const float *)a.k_new, p.v_new = (const float *)a.v_new;
    p.new_pos = !a.k_new ? -1 : a.new_pos >= 0 ? (int)a.new_pos : (int)a.Sk - 1;
    p.rope_cos = (const float *)a.rope_cos, p.rope_sin = (const float *)a.rope_sin, p.rope_stride_b = a.rope_stride_b;
    p.kv_stride_b = a.kv_stride_b, p.kv_stride_h = a.kv_stride_h;
    p.kv_row_bytes = (uint32_t)(a.kv_stride_t * 4), p.kv_bytes = (uint32_t)(((a.Sk - 1) * a.kv_stride_t + a.D) * 4);
    p.Hq = (int)a.Hq, p.Hkv = (int)a.Hkv, p.T = (int)a.Sk, p.G = (int)(a.Hq / a.Hkv);
    p.scale_log2 = a.scale * 1.4426950408889634f;

    const int64_t tiles = (a.Sk + 15) / 16;
    if (p.G <= 8 && tiles > 512 * BH) return 2;
    int64_t ns = BH > (int64_t)(kWsCounterBytes / sizeof(int)) ? 1 : choose_step_splits(BH, p.G, (int)tiles, a.D == 128 ? kCrowdWide : kCrowdNarrow);
    if (ns > kMaxSplitsF32) ns = kMaxSplitsF32;
    const int64_t per_split = BH * p.G * (a.D + 2) * (int64_t)sizeof(float);
    const int64_t avail = a.workspace && a.workspace_bytes > kWsCounterBytes ? (int64_t)(a.workspace_bytes - kWsCounterBytes) : 0;
    if (ns > 1 && ns * per_split > avail) ns = avail / per_split;
    if (ns < 1) ns = 1;
    p.nsplit = (int)ns;
    if (ns > 1) {
        p.counters = (int *)a.workspace;
        p.part_o = (float *)((char *)a.workspace + kWsCounterBytes);
        p.part_ml = p.part_o + ns * BH * p.G * a.D;
    }
    return a.D == 128 ? launch<128>(p, (int)a.B, s) : launch<64>(p, (int)a.B, s);
}

}  // namespace trocm
