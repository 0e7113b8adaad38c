// Attention on device: RoPE, head transpose, the KV-cache copy and the
// attention kernel of a LlamaTransformer layer.
//
//   apply_rope      models/src/transformer.rs:514-562 (Interleaved / SplitHalf)
//   transpose_heads models/src/transformer.rs:598-611
//   compute_attention models/src/transformer.rs:301-374:
//     kv_h = h * n_head_kv / n_head                                (:318)
//     score_j = (q . K[j]) * (1 / sqrt(head_dim))                  (:311,327-335)
//     score_j = -inf for j >= start_pos + i + 1                    (:337-342)
//     p = softmax(score); out[i, h, :] = sum_j p_j V[j, :]        (:344-356)
//
// Layouts (the reference's): q is [n_head, q_len, head_dim] (apply_rope's
// output); the cache holds, per layer and kv head, positions x head_dim
// contiguous (KVCache, models/src/context.rs:245-340), here preallocated to
// max_size positions; out is [q_len, n_head, head_dim].
//
// The attention kernel streams K and V rows from HBM once per kv head for all
// the query heads that share it (GQA), split over the positions so that
// enough workgroups run: a row of head_dim floats is read by head_dim / 8
// lanes (two float4 each), every lane keeps its own online-softmax state
// (running max, sum, and its 8 output dims) for each query head, and the
// states are merged in LDS and then across splits.  Exponentials are base 2
// on scores pre-scaled by log2(e) (v_exp_f32), so the weights agree with the
// reference's expf to a few ulp, not bit for bit; sums run in a different
// order from the reference's sequential ones.
#include "common.hpp"
#include "launch.hpp"
#include "mfma_common.hpp"
#include "q8k_block.hpp"

#include <atomic>
#include <cstdlib>

namespace barq {

// ---- RoPE / transpose ----------------------------------------------------------
// One thread per (position, head, pair).  out[h * out_head_stride + p * hd + ...]
// so that the rotated rows can go straight into a cache.
template <int LAYOUT>
__global__ __launch_bounds__(256)
void rope_kernel(const float* __restrict__ x, float* __restrict__ out, int seq, int heads, int hd, long long start_pos,
                 float freq_scale, const float* __restrict__ inv_freq, size_t out_head_stride) {
    const int half = hd / 2;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)seq * heads * half) return;
    const int i = (int)(t % half);
    const size_t ph = t / half;
    const int h = (int)(ph % heads), p = (int)(ph / heads);
    // (abs_pos as f32 * rope_freq_scale) * rope_inv_freq[i]
    const float angle = ((float)(start_pos + p) * freq_scale) * inv_freq[i];
    float sn, cs;
    sincosf(angle, &sn, &cs);
    const float* src = x + ((size_t)p * heads + h) * hd;
    float* dst = out + (size_t)h * out_head_stride + (size_t)p * hd;
    const int i0 = LAYOUT == ROPE_INTERLEAVED ? 2 * i : i;
    const int i1 = LAYOUT == ROPE_INTERLEAVED ? 2 * i + 1 : i + half;
    const float x0 = src[i0], x1 = src[i1];
    dst[i0] = x0 * cs - x1 * sn;
    dst[i1] = x0 * sn + x1 * cs;
}

__global__ __launch_bounds__(256)
void transpose_heads_kernel(const float* __restrict__ x, float* __restrict__ out, int seq, int heads, int hd,
                            size_t out_head_stride) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)seq * heads * hd) return;
    const int d = (int)(t % hd);
    const size_t ph = t / hd;
    const int h = (int)(ph % heads), p = (int)(ph / heads);
    out[(size_t)h * out_head_stride + (size_t)p * hd + d] = x[t];
}

// RoPE of q, RoPE of k into the cache and the copy of v into the cache in
// one launch (apply_rope twice and transpose_heads, transformer.rs:222-245
// and 514-611): slot s of a position is query head s (s < n_q), kv head
// s - n_q of k, or of v; one thread per pair of dims.  The angles and the
// rotation are rope_kernel's, so the results are the same bits.
template <int LAYOUT>
__global__ __launch_bounds__(256)
void rope_qkv_kernel(const float* __restrict__ qx, const float* __restrict__ kx, const float* __restrict__ vx,
                     float* __restrict__ q_out, float* __restrict__ k_out, float* __restrict__ v_out, int seq, int n_q,
                     int n_kv, int hd, long long start_pos, float freq_scale, const float* __restrict__ inv_freq,
                     size_t cache_head_stride) {
    const int half = hd / 2, slots = n_q + 2 * n_kv;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)seq * slots * half) return;
    const int i = (int)(t % half);
    const size_t ps = t / half;
    const int sl = (int)(ps % slots), p = (int)(ps / slots);
    if (sl >= n_q + n_kv) {   // v: transpose_heads into the cache
        const int h = sl - n_q - n_kv;
        const float* src = vx + ((size_t)p * n_kv + h) * hd;
        float* dst = v_out + (size_t)h * cache_head_stride + (size_t)p * hd;
        dst[2 * i] = src[2 * i];
        dst[2 * i + 1] = src[2 * i + 1];
        return;
    }
    const bool is_q = sl < n_q;
    const int h = is_q ? sl : sl - n_q, heads = is_q ? n_q : n_kv;
    const float angle = ((float)(start_pos + p) * freq_scale) * inv_freq[i];
    float sn, cs;
    sincosf(angle, &sn, &cs);
    const float* src = (is_q ? qx : kx) + ((size_t)p * heads + h) * hd;
    float* dst = is_q ? q_out + ((size_t)h * seq + p) * hd : k_out + (size_t)h * cache_head_stride + (size_t)p * hd;
    const int i0 = LAYOUT == ROPE_INTERLEAVED ? 2 * i : i;
    const int i1 = LAYOUT == ROPE_INTERLEAVED ? 2 * i + 1 : i + half;
    const float x0 = src[i0], x1 = src[i1];
    dst[i0] = x0 * cs - x1 * sn;
    dst[i1] = x0 * sn + x1 * cs;
}

hipError_t rope_qkv_launch(int layout, const float* qx, const float* kx, const float* vx, float* q_out, float* k_out,
                           float* v_out, size_t seq, size_t n_q, size_t n_kv, size_t hd, size_t start_pos,
                           float freq_scale, const float* inv_freq, size_t cache_head_stride, hipStream_t s) {
    const size_t n = seq * (n_q + 2 * n_kv) * (hd / 2);
    if (n == 0) return hipSuccess;
    const unsigned grid = (unsigned)((n + 255) / 256);
    if (layout == ROPE_INTERLEAVED)
        hipLaunchKernelGGL(rope_qkv_kernel<ROPE_INTERLEAVED>, dim3(grid), dim3(256), 0, s, qx, kx, vx, q_out, k_out,
                           v_out, (int)seq, (int)n_q, (int)n_kv, (int)hd, (long long)start_pos, freq_scale, inv_freq,
                           cache_head_stride);
    else
        hipLaunchKernelGGL(rope_qkv_kernel<ROPE_SPLIT_HALF>, dim3(grid), dim3(256), 0, s, qx, kx, vx, q_out, k_out,
                           v_out, (int)seq, (int)n_q, (int)n_kv, (int)hd, (long long)start_pos, freq_scale, inv_freq,
                           cache_head_stride);
    return hipGetLastError();
}

hipError_t rope_launch(int layout, const float* x, float* out, size_t seq, size_t heads, size_t hd, size_t start_pos,
                       float freq_scale, const float* inv_freq, size_t out_head_stride, hipStream_t s) {
    const size_t n = seq * heads * (hd / 2);
    if (n == 0) return hipSuccess;
    const unsigned grid = (unsigned)((n + 255) / 256);
    if (layout == ROPE_INTERLEAVED)
        hipLaunchKernelGGL(rope_kernel<ROPE_INTERLEAVED>, dim3(grid), dim3(256), 0, s, x, out, (int)seq, (int)heads,
                           (int)hd, (long long)start_pos, freq_scale, inv_freq, out_head_stride);
    else
        hipLaunchKernelGGL(rope_kernel<ROPE_SPLIT_HALF>, dim3(grid), dim3(256), 0, s, x, out, (int)seq, (int)heads,
                           (int)hd, (long long)start_pos, freq_scale, inv_freq, out_head_stride);
    return hipGetLastError();
}

hipError_t transpose_heads_launch(const float* x, float* out, size_t seq, size_t heads, size_t hd,
                                  size_t out_head_stride, hipStream_t s) {
    const size_t n = seq * heads * hd;
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(transpose_heads_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, x, out, (int)seq,
                       (int)heads, (int)hd, out_head_stride);
    return hipGetLastError();
}

// ---- attention -----------------------------------------------------------------
constexpr int ATT_THREADS = 256;
constexpr float LOG2E = 1.44269504088896340736f;

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// K/V rows are streamed once per call: loaded with the non-temporal hint
// (measured in one run: 55.1 -> 49.5 us at 32K positions, 14.1 -> 13.5 us at 4K),
// through a buffer descriptor over `bytes` bytes from `base`: reads at or past
// the limit return zeros and touch no memory.  Cache policy 2 is the
// non-temporal bit.
typedef float f32x4n __attribute__((ext_vector_type(4)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t kv_rows(const float* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ float4 kv_ld(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    const f32x4n v = __builtin_bit_cast(f32x4n, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 2));
    return make_float4(v.x, v.y, v.z, v.w);
}

// Partial state of one (query row, head, split): running max m (log2 units),
// sum l, then HD output sums.  Stored as HD + 2 floats.
//
// Grid: x = split, y = head group (kv head for G > 1; query head for G == 1),
// z = query row i.  The workgroup covers positions [split * chunk, ...) of
// the visible prefix [0, min(kv_len, start_pos + i + 1)).
template <int HD, int G>
__global__ __launch_bounds__(ATT_THREADS)
void attn_kernel(const float* __restrict__ q, const float* __restrict__ kc, const float* __restrict__ vc,
                 size_t layer_off, size_t head_stride, int n_head, int n_head_kv, int q_len, int kv_len,
                 long long start_pos, int chunk, float score_scale, float* __restrict__ part, float* __restrict__ out) {
    constexpr int LPR = HD / 8;              // lanes per K/V row
    constexpr int R = ATT_THREADS / LPR;     // rows per pass
    static_assert(LPR == 8 || LPR == 16 || LPR == 32, "head_dim 64, 128 or 256");
    __shared__ float red_o[R][G][HD];
    __shared__ float red_ml[R][G][2];
    __shared__ float red_ms[G][2];

    const int t = threadIdx.x, c = t % LPR, r = t / LPR;
    const int split = blockIdx.x, grp = blockIdx.y, i = blockIdx.z, n_split = gridDim.x;
    const int hk = G > 1 ? grp : (int)((long long)grp * n_head_kv / n_head);
    const long long vis = start_pos + i + 1;
    const int valid = (int)(vis < kv_len ? vis : kv_len);
    const int j0 = split * chunk, j1 = min(valid, j0 + chunk);

    // query rows of the group's heads (pre-scaled: score * log2e is the exponent)
    float qv[G][8];
    #pragma unroll
    for (int g = 0; g < G; g++) {
        const int h = G > 1 ? grp * G + g : grp;
        const float4* qp = reinterpret_cast<const float4*>(q + ((size_t)h * q_len + i) * HD);
        const float4 a = qp[c], b = qp[c + LPR];
        qv[g][0] = a.x; qv[g][1] = a.y; qv[g][2] = a.z; qv[g][3] = a.w;
        qv[g][4] = b.x; qv[g][5] = b.y; qv[g][6] = b.z; qv[g][7] = b.w;
    }
    float m[G], l[G], o[G][8];
    #pragma unroll
    for (int g = 0; g < G; g++) {
        m[g] = -INFINITY;
        l[g] = 0.0f;
        #pragma unroll
        for (int d = 0; d < 8; d++) o[g][d] = 0.0f;
    }

    // lane c of a row holds dims 4c..4c+3 and 4(c+LPR)..: each load
    // instruction reads whole contiguous half-rows
    const float* kh = kc + layer_off + (size_t)hk * head_stride;
    const float* vh = vc + layer_off + (size_t)hk * head_stride;
    // P passes of R rows form a block; the next block's rows are loaded
    // while this block's are scored, so every lane keeps K/V loads in
    // flight.  The softmax state moves once per block: all P scores first,
    // then one rescale of the running sums by the block's new maximum.
    constexpr int P = G <= 4 ? 2 : 1;
    struct Rows {
        float4 k[P][2], v[P][2];
    };
    // Rows are read through buffer descriptors limited to [j0, j1): a row
    // past the range reads as zeros without a memory access (its score is
    // masked and its weight is 0), so a block's loads need no condition.
    const __amdgpu_buffer_rsrc_t kr = kv_rows(kh + (size_t)j0 * HD, (uint32_t)(j1 - j0) * (HD * 4));
    const __amdgpu_buffer_rsrc_t vr = kv_rows(vh + (size_t)j0 * HD, (uint32_t)(j1 - j0) * (HD * 4));
    auto load = [&](Rows& b, int blk) {
        #pragma unroll
        for (int p = 0; p < P; p++) {
            const uint32_t off = (uint32_t)(blk - j0 + p * R + r) * (HD * 4) + (uint32_t)c * 16;
            b.k[p][0] = kv_ld(kr, off); b.k[p][1] = kv_ld(kr, off + LPR * 16);
            b.v[p][0] = kv_ld(vr, off); b.v[p][1] = kv_ld(vr, off + LPR * 16);
        }
    };
    auto block = [&](const Rows& b, int blk) {
        #pragma unroll
        for (int g = 0; g < G; g++) {
            float sc[P];
            float bm = -INFINITY;
            #pragma unroll
            for (int p = 0; p < P; p++) {
                const float4 k0 = b.k[p][0], k1 = b.k[p][1];
                float dot = qv[g][0] * k0.x;
                dot = __builtin_fmaf(qv[g][1], k0.y, dot);
                dot = __builtin_fmaf(qv[g][2], k0.z, dot);
                dot = __builtin_fmaf(qv[g][3], k0.w, dot);
                dot = __builtin_fmaf(qv[g][4], k1.x, dot);
                dot = __builtin_fmaf(qv[g][5], k1.y, dot);
                dot = __builtin_fmaf(qv[g][6], k1.z, dot);
                dot = __builtin_fmaf(qv[g][7], k1.w, dot);
                dot = group_sum<LPR>(dot);
                // (q . k) / sqrt(hd) * log2(e); rows past the range do not count
                sc[p] = blk + p * R + r < j1 ? dot * score_scale : -INFINITY;
                bm = fmaxf(bm, sc[p]);
            }
            // No branch on a block without live rows: a branch around the
            // V products lets the compiler's wait insertion assume the V
            // loads may still be in flight at the next block's loads into
            // the same registers, and it waits for every load there.  With
            // no live row so far (mn = -inf) the reference point 0 gives
            // corr = e = 0; with no live row in the block but some before,
            // corr = exp2(0) = 1 and e = 0, leaving the state as it was.
            const float mn = fmaxf(m[g], bm);
            const float ref = mn == -INFINITY ? 0.0f : mn;
            const float corr = fast_exp2(m[g] - ref);  // 0 while m is -inf
            m[g] = mn;
            l[g] *= corr;
            #pragma unroll
            for (int d = 0; d < 8; d++) o[g][d] *= corr;
            #pragma unroll
            for (int p = 0; p < P; p++) {
                const float e = fast_exp2(sc[p] - ref);  // 0 for rows past the range
                const float4 v0 = b.v[p][0], v1 = b.v[p][1];
                l[g] += e;
                o[g][0] = __builtin_fmaf(e, v0.x, o[g][0]);
                o[g][1] = __builtin_fmaf(e, v0.y, o[g][1]);
                o[g][2] = __builtin_fmaf(e, v0.z, o[g][2]);
                o[g][3] = __builtin_fmaf(e, v0.w, o[g][3]);
                o[g][4] = __builtin_fmaf(e, v1.x, o[g][4]);
                o[g][5] = __builtin_fmaf(e, v1.y, o[g][5]);
                o[g][6] = __builtin_fmaf(e, v1.z, o[g][6]);
                o[g][7] = __builtin_fmaf(e, v1.w, o[g][7]);
            }
        }
    };
    if (j0 < j1) {
        // NB row buffers used in turn (no register copies between blocks),
        // each refilled NB blocks ahead as soon as it has been scored.  The
        // loads carry no condition (past the range they read zeros), so
        // every block waits for its own loads only: with a conditional
        // issue the compiler's wait counts cover both paths, and each block
        // would also wait for the loads issued after it.
        // Scheduling barriers keep the loads where they are written (the
        // scheduler otherwise gathers all loads after the blocks).
        constexpr int NB = 2;
        Rows rows[NB];
        #pragma unroll
        for (int q = 0; q < NB; q++) {
            load(rows[q], j0 + q * R * P);
            __builtin_amdgcn_sched_barrier(0);
        }
        for (int blk = j0; blk < j1; blk += NB * R * P) {
            #pragma unroll
            for (int q = 0; q < NB; q++) {
                __builtin_amdgcn_sched_barrier(0);
                block(rows[q], blk + q * R * P);
                __builtin_amdgcn_sched_barrier(0);
                load(rows[q], blk + (q + NB) * R * P);
            }
        }
    }

    // merge the R row states of the workgroup
    #pragma unroll
    for (int g = 0; g < G; g++) {
        #pragma unroll
        for (int d = 0; d < 4; d++) {
            red_o[r][g][4 * c + d] = o[g][d];
            red_o[r][g][4 * (c + LPR) + d] = o[g][4 + d];
        }
        if (c == 0) {
            red_ml[r][g][0] = m[g];
            red_ml[r][g][1] = l[g];
        }
    }
    __syncthreads();
    // each row state's weight exp2(m_rr - M) once per (row, head), in place
    // of its max (then the same sums in the same order for every dim): one
    // thread per (head, row state), each head's R states an aligned group of
    // lanes (G * R <= ATT_THREADS)
    static_assert(G * R <= ATT_THREADS && R <= 32, "one thread per row state");
    if (t < G * R) {
        const int g = t / R, rr = t % R;
        const float mr = red_ml[rr][g][0];
        const float M = group_max<R>(mr);
        const float w = M == -INFINITY ? 0.0f : fast_exp2(mr - M);
        const float L = group_sum<R>(red_ml[rr][g][1] * w);
        red_ml[rr][g][0] = w;
        if (rr == 0) {
            red_ms[g][0] = M;
            red_ms[g][1] = L;
        }
    }
    __syncthreads();
    for (int e = t; e < G * HD; e += ATT_THREADS) {
        const int g = e / HD, d = e % HD;
        const float M = red_ms[g][0], L = red_ms[g][1];
        float O = 0.0f;
        if (M != -INFINITY) {
            #pragma unroll
            for (int rr = 0; rr < R; rr++) O = __builtin_fmaf(red_o[rr][g][d], red_ml[rr][g][0], O);
        }
        const int h = G > 1 ? grp * G + g : grp;
        if (n_split == 1) {
            out[((size_t)i * n_head + h) * HD + d] = O / L;
        } else {
            float* pp = part + (((size_t)i * n_head + h) * n_split + split) * (HD + 2);
            pp[2 + d] = O;
            if (d == 0) {
                pp[0] = M;
                pp[1] = L;
            }
        }
    }
}

constexpr int ATT_MAX_SPLIT = 1024;

// One output head: out value of dim t (t < HD) from the n_split partial
// states at pp, by NT threads t = 0 .. NT - 1 (all of them call it: it
// synchronises the workgroup).  The split maxima and weights are spread over
// the threads; the output sums run over SUB = 1024 / HD subsets of the splits
// (split s in subset s % SUB, in increasing order), then are added in LDS in
// subset order.  With NT < 1024 each thread runs 1024 / NT subsets one after
// another, so the sums and their order do not depend on NT: the Q8_K merge
// (heads side by side) quantizes exactly the f32 merge's values.
template <int HD>
struct CombineLds {
    float w[ATT_MAX_SPLIT];
    float red[1024 / HD][HD];
    float wred[2][1024 / 64];
};

template <int HD, int NT>
__device__ __forceinline__ float attn_combine_head(const float* __restrict__ pp, int n_split, CombineLds<HD>& sm,
                                                   int t) {
    constexpr int NWV = NT / 64, SUB = 1024 / HD, K = 1024 / NT, STEP = NT / HD, PRE = 8;
    static_assert(NT % HD == 0 && 1024 % NT == 0, "threads per head");
    const int lane = t & 63, wave = t >> 6;
    const int sub = t / HD, d = t % HD;   // subsets sub + STEP j, j < K
    // every load of the first PRE rounds is issued before any reduction
    float ov[K][PRE];
    #pragma unroll
    for (int j = 0; j < K; j++)
        #pragma unroll
        for (int u = 0; u < PRE; u++) {
            const int s = sub + STEP * j + SUB * u;
            ov[j][u] = s < n_split ? pp[(size_t)s * (HD + 2) + 2 + d] : 0.0f;
        }
    // the maximum and sum of the splits t + NT j (j < K), loaded with the
    // output sums above (n_split <= ATT_MAX_SPLIT = 1024, so these are all of
    // this thread's splits): no load waits once the reductions start
    static_assert(ATT_MAX_SPLIT <= 1024, "one split per virtual lane");
    float Msj[K], Lsj[K];
    #pragma unroll
    for (int j = 0; j < K; j++) {
        const int s = t + NT * j;
        Msj[j] = s < n_split ? pp[(size_t)s * (HD + 2)] : -INFINITY;
        Lsj[j] = s < n_split ? pp[(size_t)s * (HD + 2) + 1] : 0.0f;
    }
    float M = Msj[0];
    #pragma unroll
    for (int j = 1; j < K; j++) M = fmaxf(M, Msj[j]);
    M = wave_max_all(M);
    if (lane == 0) sm.wred[0][wave] = M;
    __syncthreads();
    M = sm.wred[0][0];
    #pragma unroll
    for (int u = 1; u < NWV; u++) M = fmaxf(M, sm.wred[0][u]);
    // The denominator in the 1024-thread merge's order whatever NT is: thread
    // t plays the 1024 lanes t + NT j (j < K), each holding its one split; a
    // reduction per 64 of those lanes (a real wave holds 64 consecutive ones);
    // then the 16 wave partials in lane order.  So the Q8_K merge's rows are
    // the f32 merge's to the bit.
    float Lj[K];
    #pragma unroll
    for (int j = 0; j < K; j++) {
        const int s = t + NT * j;
        float L = 0.0f;
        if (s < n_split) {
            const float ws = Msj[j] == -INFINITY ? 0.0f : fast_exp2(Msj[j] - M);
            sm.w[s] = ws;
            L = Lsj[j] * ws;
        }
        L = wave_sum_all(L);
        Lj[j] = L;
    }
    if (lane == 0) {
        #pragma unroll
        for (int j = 0; j < K; j++) sm.wred[1][NWV * j + wave] = Lj[j];
    }
    __syncthreads();
    float L = sm.wred[1][0];
    #pragma unroll
    for (int u = 1; u < 1024 / 64; u++) L += sm.wred[1][u];
    #pragma unroll
    for (int j = 0; j < K; j++) {
        const int sj = sub + STEP * j;
        float O = 0.0f;
        #pragma unroll
        for (int u = 0; u < PRE; u++) {
            const int s = sj + SUB * u;
            if (s < n_split) O = __builtin_fmaf(ov[j][u], sm.w[s], O);
        }
        for (int s = sj + SUB * PRE; s < n_split; s += SUB) O = __builtin_fmaf(pp[(size_t)s * (HD + 2) + 2 + d], sm.w[s], O);
        sm.red[sj][d] = O;
    }
    __syncthreads();
    float acc = 0.0f;
    if (t < HD) {
        acc = sm.red[0][t];
        #pragma unroll
        for (int u = 1; u < SUB; u++) acc += sm.red[u][t];
        acc = acc / L;
    }
    return acc;
}

// out[i, h, :] from the n_split partial states of (i, h): one workgroup of
// 1024 threads per (h, i).
template <int HD>
__global__ __launch_bounds__(1024)
void attn_combine_kernel(const float* __restrict__ part, int n_split, int n_head, float* __restrict__ out) {
    __shared__ CombineLds<HD> sm;
    const int h = blockIdx.x, i = blockIdx.y, t = threadIdx.x;
    const float v = attn_combine_head<HD, 1024>(part + ((size_t)i * n_head + h) * n_split * (HD + 2), n_split, sm, t);
    if (t < HD) out[((size_t)i * n_head + h) * HD + t] = v;
}

// The same merge with the output row written as Q8_K blocks (the o
// projection's activation): workgroup (b, i) merges the 256 / HD heads of
// block b of row i side by side (1024 / (256 / HD) threads each), then one
// wave quantizes the block (q8_k_block: the bytes quantize_q8_k_kernel
// writes for the same values).
template <int HD>
__global__ __launch_bounds__(1024)
void attn_combine_q8k_kernel(const float* __restrict__ part, int n_split, int n_head, uint8_t* __restrict__ out) {
    constexpr int NH = 256 / HD, NT = 1024 / NH;
    __shared__ CombineLds<HD> sm[NH];
    __shared__ __align__(16) float vals[256];
    const int b = blockIdx.x, i = blockIdx.y, t = threadIdx.x;
    const int hh = t / NT, tg = t % NT, h = b * NH + hh;
    const float v = attn_combine_head<HD, NT>(part + ((size_t)i * n_head + h) * n_split * (HD + 2), n_split, sm[hh], tg);
    if (tg < HD) vals[hh * HD + tg] = v;
    __syncthreads();
    if (t < 64) {
        const float4 v4 = reinterpret_cast<const float4*>(vals)[t];
        const float vv[4] = {v4.x, v4.y, v4.z, v4.w};
        q8_k_block(vv, t, out + ((size_t)i * (n_head * HD / 256) + b) * Q8_K_BYTES);
    }
}

bool attention_supported(size_t head_dim) { return head_dim == 64 || head_dim == 128 || head_dim == 256; }

int cu_count_attn() {
    static std::atomic<int> n[64] = {};   // per device; racing callers store the same value
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    int v = n[dev].load(std::memory_order_relaxed);
    if (!v) {
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) v = 256;
        n[dev].store(v, std::memory_order_relaxed);
    }
    return v;
}

size_t attention_workspace(size_t n_head, size_t head_dim, size_t q_len, size_t kv_len, size_t n_head_kv) {
    if (attn_prompt_path(n_head, n_head_kv, head_dim, q_len, kv_len)) return attn_prompt_workspace(n_head, n_head_kv, head_dim, q_len, kv_len);
    int ns = 0, chunk = 0;
    attention_plan(n_head, n_head_kv, q_len, kv_len, &ns, &chunk);
    return ns > 1 ? (size_t)ns * n_head * q_len * (head_dim + 2) * sizeof(float) : 0;
}


// Splits: at most about three workgroups per four CUs in all, whole
// multiples of 64 positions each.  A CU that runs two workgroups while
// others run one finishes last, so the launch keeps to one per CU; fewer,
// longer workgroups keep more loads in flight each.  Measured on MI355X
// (Llama-3-8B heads, us per call, targets 192 / 256 / 320 / 512 workgroups):
// 4096 positions 10.96 / 11.09 / 11.08 / 11.73, 4097 11.03 / 11.00 / 13.30 /
// 13.27, 8192 15.62 / 15.88 / 15.92 / 16.04, 16384 25.13 / 25.39 / 31.01 /
// 25.68; the decode layer about 51.5 / 51.6 / 53.9 / 53.9.
void attention_plan(size_t n_head, size_t n_head_kv, size_t q_len, size_t kv_len, int* n_split, int* chunk) {
    const size_t g = (n_head_kv && n_head % n_head_kv == 0) ? n_head / n_head_kv : 1;
    const size_t groups = (g == 1 || g > 8 || (g & (g - 1))) ? n_head : n_head_kv;
    const size_t wg = groups * (q_len ? q_len : 1);
    const int wg_override = tuning_env(TUNE_ATTN_WG);   // workgroup-count target (tuning)
    const size_t cus = (size_t)cu_count_attn();
    const size_t target = wg_override > 0 ? (size_t)wg_override : (cus * 3 / 4 > 0 ? cus * 3 / 4 : 1);
    size_t ns = (target + wg - 1) / wg;
    size_t max_ns = (kv_len + 63) / 64;
    if (max_ns > (size_t)ATT_MAX_SPLIT) max_ns = ATT_MAX_SPLIT;
    if (ns > max_ns) ns = max_ns;
    // at most 2^20 positions per split: the split kernel addresses its rows
    // with 32-bit byte offsets (under 1 GiB at head_dim 256)
    const size_t min_ns = (kv_len + ((size_t)1 << 20) - 1) >> 20;
    if (ns < min_ns) ns = min_ns;
    if (ns < 1) ns = 1;
    size_t ch = (kv_len + ns - 1) / ns;
    ch = (ch + 63) / 64 * 64;
    ns = (kv_len + ch - 1) / ch;
    if (ns < 1) ns = 1;
    *n_split = (int)ns;
    *chunk = (int)ch;
}

// Whether attention_launch writes a.out_q8 itself (the split path's merge
// emits Q8_K rows); otherwise it writes f32 rows to a.out and the caller
// quantizes them.
bool attention_q8_direct(const AttnArgs& a) {
    if ((a.n_head * a.head_dim) % 256 != 0) return false;
    if (attn_prompt_path(a.n_head, a.n_head_kv, a.head_dim, a.q_len, a.kv_len)) return attn_prompt_q8_direct(a);
    int ns = 0, chunk = 0;
    attention_plan(a.n_head, a.n_head_kv, a.q_len, a.kv_len, &ns, &chunk);
    return ns > 1;
}

template <int HD, int G>
static hipError_t attn_launch_t(const AttnArgs& a, int ns, int chunk, int groups, hipStream_t s) {
    const float scale = (1.0f / sqrtf((float)HD)) * LOG2E;
    hipLaunchKernelGGL((attn_kernel<HD, G>), dim3(ns, groups, (unsigned)a.q_len), dim3(ATT_THREADS), 0, s, a.q, a.k,
                       a.v, a.layer_off, a.head_stride, (int)a.n_head, (int)a.n_head_kv, (int)a.q_len, (int)a.kv_len,
                       (long long)a.start_pos, chunk, scale, a.part, a.out);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || ns == 1) return e;
    if (a.out_q8 && attention_q8_direct(a))
        hipLaunchKernelGGL(attn_combine_q8k_kernel<HD>, dim3((unsigned)(a.n_head * HD / 256), (unsigned)a.q_len),
                           dim3(1024), 0, s, a.part, ns, (int)a.n_head, a.out_q8);
    else
        hipLaunchKernelGGL(attn_combine_kernel<HD>, dim3((unsigned)a.n_head, (unsigned)a.q_len), dim3(1024), 0, s,
                           a.part, ns, (int)a.n_head, a.out);
    return hipGetLastError();
}

template <int HD>
static hipError_t attn_launch_hd(const AttnArgs& a, hipStream_t s) {
    int ns = 0, chunk = 0;
    attention_plan(a.n_head, a.n_head_kv, a.q_len, a.kv_len, &ns, &chunk);
    const size_t g = (a.n_head_kv && a.n_head % a.n_head_kv == 0) ? a.n_head / a.n_head_kv : 1;
    switch (g) {
    case 2: return attn_launch_t<HD, 2>(a, ns, chunk, (int)a.n_head_kv, s);
    case 4: return attn_launch_t<HD, 4>(a, ns, chunk, (int)a.n_head_kv, s);
    case 8: return attn_launch_t<HD, 8>(a, ns, chunk, (int)a.n_head_kv, s);
    default: return attn_launch_t<HD, 1>(a, ns, chunk, (int)a.n_head, s);
    }
}

hipError_t attention_launch(const AttnArgs& a, hipStream_t s) {
    if (a.q_len == 0 || a.n_head == 0) return hipSuccess;
    if (attn_prompt_path(a.n_head, a.n_head_kv, a.head_dim, a.q_len, a.kv_len)) return attn_prompt_launch(a, s);
    switch (a.head_dim) {
    case 64: return attn_launch_hd<64>(a, s);
    case 128: return attn_launch_hd<128>(a, s);
    case 256: return attn_launch_hd<256>(a, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace barq
