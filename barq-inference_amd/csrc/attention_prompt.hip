// Attention of prompt chunks (many query rows) on the matrix cores; see
// attention.hip for the reference's functions, the layouts and the decode
// kernel.
//
// A workgroup of four waves takes a tile of 128 query rows that share one kv
// head and walks the positions they see in blocks of 32.  The rows of a kv
// head's group are flattened as query * G + head (G query heads share the kv
// head), so a tile holds whole groups of heads for any G and its rows see
// nearly the same positions; a wave owns 32 of them:
//   S^T[kv, row] = K[kv, :] . Q[row, :]    A = K rows, B = Q^T
//   online softmax per column: a lane holds 16 positions of its row, the
//   other 16 sit in lane c ^ 32
//   O^T[d, row] += V[kv, d] P[row, kv]     A = V^T, B = P^T straight from
//                                          S^T's registers
//
// What bounds it.  v_mfma_f32_32x32x2_f32 has a sixteenth of the f16 matrix
// rate (157 TFLOP/s against 2.5 PFLOP/s), and a kernel on it ran at 105
// TFLOP/s.  Here every f32 operand x is scaled by a power of two and split
// into two f16 values, each rounded to nearest: x = hi + lo + e with |e| <=
// 2^-23 |x| (2^-24.5 root mean square; three quarters of all mantissas split
// exactly), and a product takes three f16 MFMAs (hi hi, hi lo, lo hi; lo lo is
// at most 2^-22 of it, 2^-24.6 root mean square) with f32 sums, 5.3 times the
// f32 rate.  Scales keep the split away from f16's limits:
//   K: per position, the row's largest |k| into [2^14, 2^15); the inverse
//      multiplies the scores
//   Q: per query row, the same
//   P: per query row and block, the largest p just below 2^15
//   V: per output dim, the largest |v| so far into [2^14, 2^15); the scale
//      only ever shrinks, and O's dim is multiplied by the ratio when it does
// f16 steps end at 2^-24.  K's and Q's elements below 2^-15 of the largest
// they share a scale with therefore lose bits: up to 2^-39 of the row's
// largest each, and of their score in log2 units about 2^-41 |k||q| (root mean
// square over 128 normal dims, |k| and |q| the rows' largest).  Below |k||q| =
// 2^18 that is 2^-23, what f32 rounds a score of 4 to; a tile with larger ones
// (or with |k| from 2^74 on, whose scores could overflow before |q| is taken
// into account) is computed again by ap_rows_f32, on f32 MFMAs without scales.
// Weights and values spread further (a first position that takes nearly all
// the weight; a large value that a row does not see), and what they lose is
// not small against the result when the large ones add little to it.  lo of P
// and V is held times 2^12, so that its steps end at 2^-36: weights down to
// 2^-27 of their block's largest (19 nats) and values down to 2^-26 of their
// dim's keep all bits.  Weights further down lose one per halving (in that
// block alone); a tile with values below 2^-31 of their dim's scale (at 2^-31
// they are off by 2^-20 at most), or with a scale that shrinks by more than
// that, goes to ap_rows_f32 too, and so does one whose sums are not finite
// (infinities and NaN turn into NaN here).
//
// Data movement: a block's K and V rows are loaded into registers one block
// ahead of the conversion, converted by all four waves and stored as f16 in
// one of two LDS stages; one barrier per block.  V is loaded with lanes along
// the dims, so its transpose is a matter of which register goes where.
// Two workgroups share a CU.
//
// Measured on MI355X, us per call with the merge (the f32-MFMA kernel for 128
// dims, the decode kernel for 64, before this one): Llama-3-8B heads, 2048 /
// 1024 / 512 / 256 tokens 206 / 73 / 40 / 26 against 337 / 135 / 54 / 30;
// 200 rows after 800 with heads of 64 dims 26 against 55.  (With lo as it is,
// one scale per row for P and no look at V's spread: 190 / 68 / 37 / 24 / 25.
// P V on f32 MFMAs: 317 / 100 / 48 / 27 / 28.)  Error against 64 bits (relative
// 2-norm, the same calls) 1.5e-7 to 1.9e-7 against 2.0e-7 to 3.9e-7.  At 2048
// tokens the matrix unit is 23 % busy and vector issue 31 % (524 vector
// instructions besides the 48 MFMAs per wave and block): a wave's scores,
// weights and output follow one another, and two waves share a SIMD.
#include "attention_prompt_plan.hpp"
#include "common.hpp"
#include "launch.hpp"
#include "mfma_common.hpp"
#include "q8k_block.hpp"

#include <cmath>

namespace barq {

typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4n __attribute__((ext_vector_type(4)));

constexpr float LOG2E = 1.44269504088896340736f;

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// The merge of a row's pieces: one wave per 256 output values (256 / HD heads
// of row i; fewer in a last wave), four values per lane; Q8, whose rows are
// whole blocks, writes the values' Q8_K block (q8_k_block) instead of them.  One pass over
// the pieces, each rescaling what was summed before it, so a row waits for
// memory once per two pieces and not twice per piece.
template <int HD, bool Q8>
__global__ __launch_bounds__(256)
void attn_combine_few_kernel(const float* __restrict__ part, int stride, int chunk, int n_head, int G, int q_len,
                             int kv_len, long long start_pos, float* __restrict__ out, uint8_t* __restrict__ out_q8) {
    const int nblk = (n_head * HD + 255) / 256;
    const int b = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), i = blockIdx.y;
    if (b >= nblk) return;
    const int l = threadIdx.x & 63;
    const int h = b * (256 / HD) + 4 * l / HD, d = 4 * l % HD;
    if (!Q8 && h >= n_head) return;
    // the pieces of the row's tile (attn_prompt_kernel's list)
    const int tile = (i * G + h % G) / AP_ROWS;
    const int n_split = (ap_tile_blocks(tile, G, q_len, kv_len, start_pos) + chunk - 1) / chunk;
    if (!Q8 && n_split == 1) return;   // stored by the kernel itself
    const float* pp = part + ((size_t)i * n_head + h) * stride * (HD + 2);
    float M = -INFINITY, L = 0.0f, O[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    #pragma unroll 2
    for (int sp = 0; sp < n_split; sp++, pp += HD + 2) {
        const float2 ml = *reinterpret_cast<const float2*>(pp);   // 8-byte aligned rows
        const float2 o0 = *reinterpret_cast<const float2*>(pp + 2 + d), o1 = *reinterpret_cast<const float2*>(pp + 4 + d);
        const float mn = fmaxf(M, ml.x);
        // a piece that saw no position is (-inf, 0, 0)
        const float c = M == -INFINITY ? 0.0f : fast_exp2(M - mn), w = ml.x == -INFINITY ? 0.0f : fast_exp2(ml.x - mn);
        M = mn;
        L = __builtin_fmaf(ml.y, w, L * c);
        O[0] = __builtin_fmaf(o0.x, w, O[0] * c);
        O[1] = __builtin_fmaf(o0.y, w, O[1] * c);
        O[2] = __builtin_fmaf(o1.x, w, O[2] * c);
        O[3] = __builtin_fmaf(o1.y, w, O[3] * c);
    }
    const float vv[4] = {O[0] / L, O[1] / L, O[2] / L, O[3] / L};
    if constexpr (!Q8)
        *reinterpret_cast<float4*>(out + ((size_t)i * n_head + h) * HD + d) = make_float4(vv[0], vv[1], vv[2], vv[3]);
    else
        q8_k_block(vv, l, out_q8 + ((size_t)i * nblk + b) * Q8_K_BYTES);
}

// ---- the kernel ---------------------------------------------------------------

struct ApArgs {
    const float* q;       // [n_head, q_len, HD]
    const float* k;       // the layer's rows of kv head 0
    const float* v;
    size_t head_stride;   // floats between kv heads
    int n_head, n_head_kv, G, groups;   // groups of G heads that share a kv head
    int q_len, kv_len;
    long long start_pos;
    float scale;          // log2(e) / sqrt(HD)
    float* out;           // [q_len, n_head, HD]
    float* part;          // partial states (chunk > 0)
    int chunk, stride;
    int all_parts;        // tiles of one piece store their state too (the merge quantizes)
};

// LDS: two stages of a block's split K and V, the V dims' largest values and
// rescale factors of two blocks, the dims' final inverse scales.  The f32
// kernel's two stages share the space.
template <int HD>
struct ApLds {
    static constexpr int KRS = 2 * HD + 16;   // bytes of a K row (hi or lo): fragment reads of 16 rows on distinct banks
    static constexpr int KLO = 32 * KRS;
    static constexpr int V = 2 * KLO;
    static constexpr int VRS = 144;           // bytes of a V^T row: 32 positions hi, 32 lo, pad (distinct banks likewise)
    static constexpr int KF = V + HD * VRS;   // per position: the inverse of its scale
    static constexpr int STAGE = KF + 128;
    static constexpr int NB = HD / 32;        // O's accumulators
    static constexpr int NT = 64 * AP_NW;
    static constexpr int TPR = NT / 32;       // threads that share a K row
    static constexpr int PARTS = NT / HD;     // threads that share a dim
    static constexpr int PP = 32 / PARTS;     // positions each of them takes
    static constexpr int VMAX = 2 * STAGE;    // [2][PARTS][HD]
    static constexpr int VR = VMAX + 2 * PARTS * HD * 4;   // [2][HD]
    static constexpr int GROW = VR + 2 * HD * 4;           // [2]: the last block of that parity with a rescale
    static constexpr int QM = GROW + 16;      // [AP_NW]: the waves' largest |q|
    static constexpr int VS = QM + 16;        // [HD]
    static constexpr int F32_RS = 4 * HD + 16, F32_PIECES = HD / 4 + 1, F32_BLK = 32 * F32_RS;
    static constexpr int TOTAL = VS + 4 * HD;
    static_assert(4 * F32_BLK <= TOTAL, "the f32 stages fit");
    static_assert(8 / AP_NW * TOTAL <= 163840, "eight waves per CU");
    static_assert(AP_NW == 4, "four waves' largest |q|");
    static_assert(PP >= 4 && HD % (4 * TPR) == 0, "whole float4 loads and position groups");
};

// The tile's place: group, rows, the lane's row.
struct ApRow {
    int h, i;        // query head and row of the lane
    bool ok;
    int vis;         // positions the lane's row sees
    int vis_first;   // ... the wave's first row
    int vis_last;    // ... the wave's last row (0: the wave has no rows)
};

__device__ __forceinline__ int ap_vis(const ApArgs& a, int i) {
    const long long v = a.start_pos + i + 1;
    return (int)(v < a.kv_len ? v : a.kv_len);
}

__device__ __forceinline__ ApRow ap_row(const ApArgs& a, int grp, int tile, int wave, int c) {
    const int rows = a.q_len * a.G, r0 = tile * AP_ROWS + 32 * wave;
    ApRow r;
    const int row = r0 + c < rows ? r0 + c : rows - 1;
    r.ok = r0 + c < rows;
    r.i = row / a.G;
    r.h = grp * a.G + (row - r.i * a.G);
    r.vis = ap_vis(a, r.i);
    const int first = r0 < rows ? r0 : rows - 1, last = r0 + 31 < rows ? r0 + 31 : rows - 1;
    r.vis_first = __builtin_amdgcn_readfirstlane(ap_vis(a, first / a.G));
    r.vis_last = r0 < rows ? __builtin_amdgcn_readfirstlane(ap_vis(a, last / a.G)) : 0;
    return r;
}

// Results of a lane: output dims through dim(r, t), unnormalised sums o, the
// row's sum and reference maximum.
template <int HD>
__device__ __forceinline__ void ap_store4(const ApArgs& a, const ApRow& r, int piece, int d, float4 o, float lsum) {
    if (piece >= 0) {
        float* p = a.part + (((size_t)r.i * a.n_head + r.h) * a.stride + piece) * (HD + 2) + 2 + d;   // 8-byte aligned
        *reinterpret_cast<float2*>(p) = make_float2(o.x, o.y);
        *reinterpret_cast<float2*>(p + 2) = make_float2(o.z, o.w);
    } else {
        *reinterpret_cast<float4*>(a.out + ((size_t)r.i * a.n_head + r.h) * HD + d) =
            make_float4(o.x / lsum, o.y / lsum, o.z / lsum, o.w / lsum);
    }
}

template <int HD>
__device__ __forceinline__ void ap_store_ml(const ApArgs& a, const ApRow& r, int piece, float m, float lsum) {
    float* p = a.part + (((size_t)r.i * a.n_head + r.h) * a.stride + piece) * (HD + 2);
    p[0] = m;
    p[1] = lsum;
}

// ---- f32 MFMAs: tiles with values that are not finite ----------------------------
// v_mfma_f32_32x32x2_f32 on K and V rows copied to LDS as they are.  The dims
// of a lane: HD / 32 consecutive ones per register (output row i of block b
// stands for dim (HD / 32) i + b, so one read per lane feeds every block).
template <int HD>
__device__ __forceinline__ void ap_f32_issue(uint32_t stage, i32x4v kr, i32x4v vr, uint32_t soff, int wave, int l) {
    using L = ApLds<HD>;
    constexpr int INSTR = (32 * L::F32_PIECES + 63) / 64;
    #pragma unroll
    for (int q = 0; q < (2 * INSTR + AP_NW - 1) / AP_NW; q++) {
        const int idx = q * AP_NW + wave;
        if (idx < 2 * INSTR) {
            const int kvsel = idx >= INSTR, ii = idx - kvsel * INSTR;
            const int p = ii * 64 + l, row = p / L::F32_PIECES, piece = p - row * L::F32_PIECES;
            if (p < 32 * L::F32_PIECES) {
                const uint32_t voff = (uint32_t)row * (4u * HD) + 16u * (uint32_t)(piece < HD / 4 ? piece : 0);
                lds_load16_at(kvsel ? vr : kr, stage + kvsel * L::F32_BLK + 1024 * ii, voff, soff);
            }
        }
    }
}

template <int HD>
__device__ __forceinline__ void ap_rows_f32(const uint8_t* lds, uint32_t lds0, const ApArgs& a, int grp, int tile, int piece, int b_lo, int b_hi) {
    using L = ApLds<HD>;
    constexpr int NB = HD / 32;
    typedef float fvec __attribute__((ext_vector_type(NB)));
    const int l = threadIdx.x & 63, c = l & 31, g = l >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const ApRow row = ap_row(a, grp, tile, wave, c);
    const int hk = (int)((long long)(grp * a.G) * a.n_head_kv / a.n_head);
    const i32x4v kr = make_rsrc4(a.k + (size_t)hk * a.head_stride, (uint32_t)a.kv_len * (4u * HD));
    const i32x4v vr = make_rsrc4(a.v + (size_t)hk * a.head_stride, (uint32_t)a.kv_len * (4u * HD));
    ap_f32_issue<HD>(lds0, kr, vr, (uint32_t)b_lo * (128u * HD), wave, l);
    float qv[HD / 2];
    const float4* qp = reinterpret_cast<const float4*>(a.q + ((size_t)row.h * a.q_len + row.i) * HD + HD / 2 * g);
    #pragma unroll
    for (int u = 0; u < HD / 8; u++) {
        const float4 t = qp[u];
        qv[4 * u] = t.x; qv[4 * u + 1] = t.y; qv[4 * u + 2] = t.z; qv[4 * u + 3] = t.w;
    }
    f32x16 o[NB] = {};
    float m = -INFINITY, lsum = 0.0f;
    for (int b = b_lo; b < b_hi; b++) {
        const int j0 = 32 * b;
        wait_vmcnt<0>();
        asm volatile("" ::: "memory");
        __syncthreads();   // block b is in its stage; every wave is done with the other one
        if (b + 1 < b_hi)
            ap_f32_issue<HD>(lds0 + ((b + 1 - b_lo) & 1) * 2 * L::F32_BLK, kr, vr, (uint32_t)(b + 1) * (128u * HD), wave, l);
        const uint8_t* ks = lds + ((b - b_lo) & 1) * 2 * L::F32_BLK;
        const uint8_t* vs = ks + L::F32_BLK;
        f32x16 sa = {}, sb = {};
        #pragma unroll
        for (int u = 0; u < HD / 8; u++) {
            const float4 kk = *reinterpret_cast<const float4*>(ks + c * L::F32_RS + 2 * HD * g + 16 * u);
            sa = __builtin_amdgcn_mfma_f32_32x32x2f32(kk.x, qv[4 * u], sa, 0, 0, 0);
            sb = __builtin_amdgcn_mfma_f32_32x32x2f32(kk.y, qv[4 * u + 1], sb, 0, 0, 0);
            sa = __builtin_amdgcn_mfma_f32_32x32x2f32(kk.z, qv[4 * u + 2], sa, 0, 0, 0);
            sb = __builtin_amdgcn_mfma_f32_32x32x2f32(kk.w, qv[4 * u + 3], sb, 0, 0, 0);
        }
        float sc[16];
        float bm = -INFINITY;
        #pragma unroll
        for (int r = 0; r < 16; r++) {
            const int kv = j0 + 8 * (r >> 2) + 4 * g + (r & 3);
            sc[r] = kv < row.vis ? (sa[r] + sb[r]) * a.scale : -INFINITY;
            bm = fmaxf(bm, sc[r]);
        }
        {
            auto hb = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(int, bm), __builtin_bit_cast(int, bm), false, false);
            bm = fmaxf(__builtin_bit_cast(float, (int)hb[0]), __builtin_bit_cast(float, (int)hb[1]));
        }
        // a piece can hold blocks a row sees none of: exponents then use 0 as
        // the reference, so they are 0 and the state stays (-inf, 0, 0)
        const float mn = fmaxf(m, bm);
        const float mref = mn == -INFINITY ? 0.0f : mn;
        const float corr = fast_exp2(m - mref);   // 0 while m is -inf
        m = mn;
        float p[16];
        float rs = 0.0f;
        #pragma unroll
        for (int r = 0; r < 16; r++) {
            p[r] = fast_exp2(sc[r] - mref);   // 0 for masked positions
            rs += p[r];
        }
        rs = swap32_add(rs, rs);   // + the other half-wave's
        lsum = lsum * corr + rs;
        #pragma unroll
        for (int t = 0; t < NB; t++) o[t] *= corr;
        bool inf_or_nan = false;
        #pragma unroll
        for (int st = 0; st < 16; st++) {
            const int kv = 8 * (st >> 2) + 4 * g + (st & 3);
            const fvec vv = *reinterpret_cast<const fvec*>(vs + kv * L::F32_RS + 4 * NB * c);
            #pragma unroll
            for (int t = 0; t < NB; t++) {
                const bool finite = __builtin_fabsf(vv[t]) < INFINITY;
                inf_or_nan |= !finite;
                o[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(finite ? vv[t] : 0.0f, p[st], o[t], 0, 0, 0);
            }
        }
        // Infinities and NaN in V only go to the rows that see their position
        // (in a product 0 * inf would be NaN for the others).
        if (__any(inf_or_nan)) {
            #pragma unroll 1
            for (int st = 0; st < 16; st++) {
                float ps = p[0];
                #pragma unroll
                for (int u = 1; u < 16; u++) ps = st == u ? p[u] : ps;
                const auto pp = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(int, ps), __builtin_bit_cast(int, ps), false, false);
                #pragma unroll
                for (int h = 0; h < 2; h++) {   // the positions of the two half-waves
                    const int kv = 8 * (st >> 2) + 4 * h + (st & 3);
                    const float ph = __builtin_bit_cast(float, (int)pp[h]);
                    const bool seen = j0 + kv < row.vis;
                    #pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const fvec vv = *reinterpret_cast<const fvec*>(vs + kv * L::F32_RS + 4 * NB * (8 * (r >> 2) + 4 * g + (r & 3)));
                        #pragma unroll
                        for (int t = 0; t < NB; t++)
                            if (seen && !(__builtin_fabsf(vv[t]) < INFINITY)) o[t][r] = __builtin_fmaf(ph, vv[t], o[t][r]);
                    }
                }
            }
        }
    }
    if (!row.ok) return;
    if (piece >= 0 && g == 0) ap_store_ml<HD>(a, row, piece, m, lsum);
    #pragma unroll
    for (int r = 0; r < 16; r += 4 / NB) {
        // registers r .. of the NB blocks: four consecutive dims
        const int i = 8 * (r >> 2) + 4 * g + (r & 3);
        float4 v;
        if constexpr (NB == 4) v = make_float4(o[0][r], o[1][r], o[2][r], o[3][r]);
        else v = make_float4(o[0][r], o[1][r], o[0][r + 1], o[1][r + 1]);
        ap_store4<HD>(a, row, piece, NB * i, v, lsum);
    }
}

// ---- split f16 ----------------------------------------------------------------------

// x0, x1 -> packed f16 (hi) and packed f16 of what hi leaves (lo): one packed
// conversion and two v_fma_mix{lo,hi}_f16.  The empty asm keeps the compiler
// from converting every value a second time, and minus_one (-1 in a register
// it knows nothing of) from turning the fma into a conversion and a
// subtraction.
__device__ __forceinline__ float ap_minus_one() {
    float v = -1.0f;
    asm("" : "+s"(v));
    return v;
}
__device__ __forceinline__ void ap_split(float x0, float x1, float minus_one, uint32_t& hi, uint32_t& lo) {
    asm("" : "+v"(x0), "+v"(x1));
    const h2v hv = {(_Float16)x0, (_Float16)x1};
    hi = __builtin_bit_cast(uint32_t, hv);
    asm("" : "+v"(hi));
    const h2v h = __builtin_bit_cast(h2v, hi);
    const float r0 = __builtin_fmaf((float)h[0], minus_one, x0), r1 = __builtin_fmaf((float)h[1], minus_one, x1);
    const h2v r = {(_Float16)r0, (_Float16)r1};
    lo = __builtin_bit_cast(uint32_t, r);
}

// x0, x1, given times 2^12 -> packed f16 (hi) and 2^12 times what hi leaves
// (lo; at most 2^15 for |x| up to 2^15): lo's smallest step is then 2^-36 of
// x's unit instead of 2^-24.  Two
// v_fma_mix{lo,hi}_f16 per value.
struct ApExt {
    float down, neg;   // 2^-12 and -2^12 in registers that the compiler knows nothing of
};
__device__ __forceinline__ ApExt ap_ext() {
    ApExt e{0x1p-12f, -0x1p12f};
    asm("" : "+s"(e.down), "+s"(e.neg));
    return e;
}
__device__ __forceinline__ void ap_split_ext(float x0, float x1, const ApExt& e, uint32_t& hi, uint32_t& lo) {
    const h2v h = {(_Float16)__builtin_fmaf(x0, e.down, 0.0f), (_Float16)__builtin_fmaf(x1, e.down, 0.0f)};
    hi = __builtin_bit_cast(uint32_t, h);
    asm("" : "+v"(hi));
    const h2v g = __builtin_bit_cast(h2v, hi);
    const h2v r = {(_Float16)__builtin_fmaf((float)g[0], e.neg, x0), (_Float16)__builtin_fmaf((float)g[1], e.neg, x1)};
    lo = __builtin_bit_cast(uint32_t, r);
}

// The biased exponent of |x| (at least 15, so that the scales below are normal
// f32 values; 255 for infinities) and the powers of two that take such an x
// into [2^P, 2^(P + 1)) and back.
__device__ __forceinline__ uint32_t ap_exp(float ax) {
    const uint32_t e = __builtin_bit_cast(uint32_t, ax) >> 23;
    return e > 15u ? e : 15u;
}
template <int P>
__device__ __forceinline__ float ap_scale(uint32_t e) { return __builtin_bit_cast(float, (254u + P - e) << 23); }
template <int P>
__device__ __forceinline__ float ap_unscale(uint32_t e) { return __builtin_bit_cast(float, (e - P) << 23); }

constexpr int AP_KQ = 14, AP_V = 14;
constexpr int AP_P = 2;               // the largest p before its scale: its exponents are then near 0, where f32 is finest
constexpr uint32_t AP_SCORE = 18;     // log2 of the |k||q| from which scores are left to the f32 kernel
constexpr uint32_t AP_SPREAD = 31;    // octaves below a dim's largest |v| that the split takes

template <int HD>
struct ApRegs {
    using L = ApLds<HD>;
    static constexpr int NK = HD / (4 * L::TPR);
    f32x4n k[NK];     // row t / TPR, dims 4 (t % TPR) + 4 TPR i
    float v[L::PP];   // dim t % HD, positions PP * (t / HD) + j
};

template <int HD>
__device__ __forceinline__ void ap_load(ApRegs<HD>& r, __amdgpu_buffer_rsrc_t kr, __amdgpu_buffer_rsrc_t vr, int b, int t) {
    using L = ApLds<HD>;
    const uint32_t soff = (uint32_t)b * (128u * HD);
    const uint32_t ko = (uint32_t)(t / L::TPR) * (4u * HD) + 16u * (uint32_t)(t % L::TPR);
    const uint32_t vo = (uint32_t)(t / HD) * (L::PP * 4u * HD) + 4u * (uint32_t)(t % HD);
    #pragma unroll
    for (int i = 0; i < ApRegs<HD>::NK; i++)
        r.k[i] = __builtin_bit_cast(f32x4n, __builtin_amdgcn_raw_buffer_load_b128(kr, ko + 16u * L::TPR * i, soff, 0));
    #pragma unroll
    for (int j = 0; j < L::PP; j++)
        r.v[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(vr, vo + 4u * HD * j, soff, 0));
}

// this thread's largest |v| of the loaded block, for the threads of its dim
template <int HD>
__device__ __forceinline__ void ap_vmax(uint8_t* lds, const ApRegs<HD>& r, int par, int t) {
    using L = ApLds<HD>;
    float m = 0.0f;
    #pragma unroll
    for (int j = 0; j < L::PP; j++) m = fmaxf(m, __builtin_fabsf(r.v[j]));
    reinterpret_cast<float*>(lds + L::VMAX)[L::NT * par + t] = m;
}

// The loaded block n as f16 hi and lo into its stage.  ve: the exponent state
// of the thread's dim (0: nothing but zeros so far).  ke_max: the largest
// exponent of its K rows.  bad: set when its values spread further than the
// split can hold.
template <int HD>
__device__ __forceinline__ void ap_convert(uint8_t* lds, const ApRegs<HD>& r, int n, int t, uint32_t& ve, uint32_t& ke_max, bool& bad) {
    using L = ApLds<HD>;
    uint8_t* st = lds + (n & 1) * L::STAGE;
    const float mo = ap_minus_one();
    const int d = t % HD, part = t / HD;
    float mx = 0.0f;   // V: one scale per dim
    {
        const float* vm = reinterpret_cast<const float*>(lds + L::VMAX) + L::NT * (n & 1) + d;
        #pragma unroll
        for (int p = 0; p < L::PARTS; p++) mx = fmaxf(mx, vm[p * HD]);
    }
    // K: one scale per row, found by its threads
    float km = 0.0f;
    #pragma unroll
    for (int i = 0; i < ApRegs<HD>::NK; i++)
        #pragma unroll
        for (int j = 0; j < 4; j++) km = fmaxf(km, __builtin_fabsf(r.k[i][j]));
    const uint32_t ke = ap_exp(group_max<L::TPR>(km));
    ke_max = ke > ke_max ? ke : ke_max;
    const float ks = ap_scale<AP_KQ>(ke);
    uint8_t* krow = st + (t / L::TPR) * L::KRS + 8 * (t % L::TPR);
    #pragma unroll
    for (int i = 0; i < ApRegs<HD>::NK; i++) {
        uint2 h, lo;
        ap_split(r.k[i][0] * ks, r.k[i][1] * ks, mo, h.x, lo.x);
        ap_split(r.k[i][2] * ks, r.k[i][3] * ks, mo, h.y, lo.y);
        *reinterpret_cast<uint2*>(krow + 8 * L::TPR * i) = h;
        *reinterpret_cast<uint2*>(krow + L::KLO + 8 * L::TPR * i) = lo;
    }
    if (t % L::TPR == 0) reinterpret_cast<float*>(st + L::KF)[t / L::TPR] = ap_unscale<AP_KQ>(ke);
    uint32_t e = __builtin_bit_cast(uint32_t, mx) >> 23;
    e = mx > 0.0f ? (e > 30u ? e : 30u) : 0u;
    float ratio = 1.0f;
    if (e > ve) {
        // (nothing to rescale while O's dim is zero)
        if (ve) {
            ratio = ve + 126u > e ? __builtin_bit_cast(float, (127u + ve - e) << 23) : 0.0f;
            reinterpret_cast<int*>(lds + L::GROW)[n & 1] = n;
            bad |= e > ve + AP_SPREAD;
        }
        ve = e;
    }
    // The smallest of the thread's values that are not zero (2 |bits| - 1 orders
    // them with zero last).  Dims below 2^-87 are left to the f32 kernel too.
    // Standard normal values come that far apart once in 10^9.
    uint32_t um = 0xFFFFFFFFu;
    #pragma unroll
    for (int j = 0; j < L::PP; j++) {
        const uint32_t u = (__builtin_bit_cast(uint32_t, r.v[j]) << 1) - 1u;
        um = u < um ? u : um;
    }
    bad |= um < (ve < 40u ? 0xFFFFFFFFu : (ve - AP_SPREAD) << 24);
    const uint32_t vu = ve ? ve : 30u;
    if (part == 0) {
        reinterpret_cast<float*>(lds + L::VR)[HD * (n & 1) + d] = ratio;
        reinterpret_cast<float*>(lds + L::VS)[d] = ap_unscale<AP_V>(vu);
    }
    const float vs = ap_scale<AP_V + 12>(vu);
    const ApExt ex = ap_ext();
    uint32_t hi[L::PP / 2], lo[L::PP / 2];
    #pragma unroll
    for (int j = 0; j < L::PP / 2; j++) ap_split_ext(r.v[2 * j] * vs, r.v[2 * j + 1] * vs, ex, hi[j], lo[j]);
    // Positions 4 u .. 4 u + 3 of a row are 8 bytes at 32 s + 16 g + 8 w with
    // u = 4 s + 2 w + g: the 16 bytes (s, g) are those whose probabilities
    // lane half g holds for step s.
    uint8_t* vrow = st + L::V + d * L::VRS;
    if constexpr (L::PP == 16) {
        vrow += 32 * part;
        *reinterpret_cast<uint4*>(vrow) = make_uint4(hi[0], hi[1], hi[4], hi[5]);
        *reinterpret_cast<uint4*>(vrow + 16) = make_uint4(hi[2], hi[3], hi[6], hi[7]);
        *reinterpret_cast<uint4*>(vrow + 64) = make_uint4(lo[0], lo[1], lo[4], lo[5]);
        *reinterpret_cast<uint4*>(vrow + 80) = make_uint4(lo[2], lo[3], lo[6], lo[7]);
    } else {
        #pragma unroll
        for (int i = 0; i < L::PP / 4; i++) {
            const int u = L::PP / 4 * part + i, at = 32 * (u >> 2) + 16 * (u & 1) + 8 * ((u >> 1) & 1);
            *reinterpret_cast<uint2*>(vrow + at) = make_uint2(hi[2 * i], hi[2 * i + 1]);
            *reinterpret_cast<uint2*>(vrow + 64 + at) = make_uint2(lo[2 * i], lo[2 * i + 1]);
        }
    }
}

// O into the scales of block n (rarely; a wave that skips the block needs it
// too, since the final scales are the last block's).
template <int HD>
__device__ __forceinline__ void ap_rescale(const uint8_t* lds, int n, int grown, int g, f32x16 (&o)[ApLds<HD>::NB]) {
    using L = ApLds<HD>;
    if (grown == n) {
        #pragma unroll
        for (int t = 0; t < L::NB; t++)
            #pragma unroll
            for (int q = 0; q < 4; q++) {
                const float4 f = *reinterpret_cast<const float4*>(lds + L::VR + 4 * (HD * (n & 1) + 32 * t + 8 * q + 4 * g));
                o[t][4 * q] *= f.x; o[t][4 * q + 1] *= f.y; o[t][4 * q + 2] *= f.z; o[t][4 * q + 3] *= f.w;
            }
    }
}

// One block from its stage: scores, softmax, O.
template <int HD>
__device__ __forceinline__ void ap_compute(const uint8_t* lds, int n, int j0, const h8v (&qh)[HD / 16],
                                           const h8v (&ql)[HD / 16], float qf, int c, int g, const ApRow& row, float& m,
                                           float& lsum, f32x16 (&o)[ApLds<HD>::NB]) {
    using L = ApLds<HD>;
    const uint8_t* st = lds + (n & 1) * L::STAGE;
    const uint8_t* kp = st + c * L::KRS + 16 * g;
    // the small products first: one accumulator, and the large ones round last
    f32x16 sa = {};
    #pragma unroll
    for (int s = 0; s < HD / 16; s++) {
        const h8v kh = *reinterpret_cast<const h8v*>(kp + 32 * s);
        const h8v kl = *reinterpret_cast<const h8v*>(kp + L::KLO + 32 * s);
        sa = __builtin_amdgcn_mfma_f32_32x32x16_f16(kl, qh[s], sa, 0, 0, 0);
        sa = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, ql[s], sa, 0, 0, 0);
    }
    #pragma unroll
    for (int s = 0; s < HD / 16; s++) {
        const h8v kh = *reinterpret_cast<const h8v*>(kp + 32 * s);
        sa = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, qh[s], sa, 0, 0, 0);
    }
    // sc * qf are the scores in log2 units (qf > 0)
    float sc[16];
    float bm = -INFINITY;
    #pragma unroll
    for (int q = 0; q < 4; q++) {
        const float4 kf = *reinterpret_cast<const float4*>(st + L::KF + 4 * (8 * q + 4 * g));
        sc[4 * q] = sa[4 * q] * kf.x;
        sc[4 * q + 1] = sa[4 * q + 1] * kf.y;
        sc[4 * q + 2] = sa[4 * q + 2] * kf.z;
        sc[4 * q + 3] = sa[4 * q + 3] * kf.w;
    }
    if (j0 + 32 > row.vis_first) {   // some row of the wave does not see the whole block
        #pragma unroll
        for (int r = 0; r < 16; r++) sc[r] = j0 + 8 * (r >> 2) + 4 * g + (r & 3) < row.vis ? sc[r] : -INFINITY;
    }
    #pragma unroll
    for (int r = 0; r < 16; r++) bm = fmaxf(bm, sc[r]);
    {
        auto hb = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(int, bm), __builtin_bit_cast(int, bm), false, false);
        bm = fmaxf(__builtin_bit_cast(float, (int)hb[0]), __builtin_bit_cast(float, (int)hb[1])) * qf;
    }
    // o and lsum are relative to m, the largest score when m was last moved, up to
    // a multiple of 2^-14; it moves when the maximum has grown by 2^32.  A
    // block's p are relative to m plus a whole number (exact, and so is the
    // factor between the two), at most 2^AP_P.  A row's largest weight is then
    // 2^AP_P itself while m is its score.
    if (__any(bm > m + 32.0f)) {
        const float mn = fmaxf(m, __builtin_ceilf(bm * 0x1p14f) * 0x1p-14f);
        const float corr = m == -INFINITY ? 0.0f : fast_exp2(m - mn);
        m = mn;
        lsum *= corr;
        #pragma unroll
        for (int t = 0; t < L::NB; t++) o[t] *= corr;
    }
    const bool none = bm == -INFINITY;   // a row that sees no position of the block
    const float k = none ? 0.0f : __builtin_ceilf(bm - m) - (float)AP_P;
    const float pref = none ? 0.0f : m + k, step = none ? 0.0f : fast_exp2(k);
    const float inv = step * (1.0f / (float)(1 << (15 - AP_P)));
    const ApExt ex = ap_ext();
    float rs[8];
    uint32_t ph[8], pl[8];
    #pragma unroll
    for (int r = 0; r < 8; r++) {
        const float p0 = fast_exp2(__builtin_fmaf(sc[2 * r], qf, -pref)), p1 = fast_exp2(__builtin_fmaf(sc[2 * r + 1], qf, -pref));
        rs[r] = p0 + p1;
        ap_split_ext(p0 * (float)(1 << (27 - AP_P)), p1 * (float)(1 << (27 - AP_P)), ex, ph[r], pl[r]);
    }
    // (as a tree: a chain of sixteen rounds more)
    const float rsum = ((rs[0] + rs[1]) + (rs[2] + rs[3])) + ((rs[4] + rs[5]) + (rs[6] + rs[7]));
    lsum = __builtin_fmaf(swap32_add(rsum, rsum), step, lsum);   // + the other half-wave's positions
    const uint8_t* vp = st + L::V + c * L::VRS + 16 * g;
    h8v bh[2], bl[2];
    #pragma unroll
    for (int s = 0; s < 2; s++) {
        bh[s] = __builtin_bit_cast(h8v, u32x4v{ph[4 * s], ph[4 * s + 1], ph[4 * s + 2], ph[4 * s + 3]});
        bl[s] = __builtin_bit_cast(h8v, u32x4v{pl[4 * s], pl[4 * s + 1], pl[4 * s + 2], pl[4 * s + 3]});
    }
    // A block's products start from zero and are added to O once: the matrix
    // unit's f32 sums do not round to nearest, and over many blocks of one
    // accumulator that adds up.
    constexpr int U = HD == 64 ? 2 : 1;   // accumulators at a time (128 dims: two would not fit the registers)
    #pragma unroll
    for (int t = 0; t < L::NB; t += U) {
        f32x16 d[U] = {};
        h8v vh[U][2];
        #pragma unroll
        for (int s = 0; s < 2; s++)
            #pragma unroll
            for (int u = 0; u < U; u++) {
                const h8v vl = *reinterpret_cast<const h8v*>(vp + 32 * (t + u) * L::VRS + 64 + 32 * s);
                vh[u][s] = *reinterpret_cast<const h8v*>(vp + 32 * (t + u) * L::VRS + 32 * s);
                d[u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vl, bh[s], d[u], 0, 0, 0);
                d[u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh[u][s], bl[s], d[u], 0, 0, 0);
            }
        #pragma unroll
        for (int u = 0; u < U; u++) {
            d[u] *= 0x1p-12f;
            #pragma unroll
            for (int s = 0; s < 2; s++) d[u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh[u][s], bh[s], d[u], 0, 0, 0);
        }
        #pragma unroll
        for (int u = 0; u < U; u++)
            #pragma unroll
            for (int r = 0; r < 16; r++) o[t + u][r] = __builtin_fmaf(d[u][r], inv, o[t + u][r]);
    }
}

// One tile, or with chunk > 0 (and more blocks than that) piece `piece` of it: position blocks [piece,
// piece + 1) * chunk, whose partial state (reference maximum in log2 units,
// sum, unnormalised output) goes to the merge kernel.
template <int HD>
__device__ __forceinline__ void ap_tile(uint8_t* lds, uint32_t lds0, const ApArgs& a, int grp, int tile, int piece) {
    using L = ApLds<HD>;
    const int t = threadIdx.x, l = t & 63, c = l & 31, g = l >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int blocks = ap_tile_blocks(tile, a.G, a.q_len, a.kv_len, a.start_pos);
    const int b_lo = a.chunk > 0 ? piece * a.chunk : 0;
    const int b_hi = a.chunk > 0 && b_lo + a.chunk < blocks ? b_lo + a.chunk : blocks;
    if (b_lo >= b_hi) return;   // (not in the launch's list)
    if (a.chunk == 0 || (blocks <= a.chunk && !a.all_parts)) piece = -1;   // the rows' results, no partial state
    const ApRow row = ap_row(a, grp, tile, wave, c);
    const int hk = (int)((long long)(grp * a.G) * a.n_head_kv / a.n_head);   // the same for the group's heads
    const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(a.k + (size_t)hk * a.head_stride), (short)0, (int)((uint32_t)a.kv_len * (4u * HD)), 0x00020000);
    const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(a.v + (size_t)hk * a.head_stride), (short)0, (int)((uint32_t)a.kv_len * (4u * HD)), 0x00020000);
    ApRegs<HD> reg;
    uint32_t ve = 0, ke_max = 0;
    bool bad = false;
    ap_load<HD>(reg, kr, vr, b_lo, t);

    // the lane's query row: dims 16 s + 8 g .. + 7 of every step s
    h8v qh[HD / 16], ql[HD / 16];
    float qf;
    {
        const float4* qp = reinterpret_cast<const float4*>(a.q + ((size_t)row.h * a.q_len + row.i) * HD + 8 * g);
        float4 qv[HD / 8];
        float qm = 0.0f;
        #pragma unroll
        for (int s = 0; s < HD / 16; s++) {
            qv[2 * s] = qp[4 * s];
            qv[2 * s + 1] = qp[4 * s + 1];
        }
        #pragma unroll
        for (int s = 0; s < HD / 8; s++)
            qm = fmaxf(fmaxf(fmaxf(qm, __builtin_fabsf(qv[s].x)), fmaxf(__builtin_fabsf(qv[s].y), __builtin_fabsf(qv[s].z))),
                       __builtin_fabsf(qv[s].w));
        auto hb = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(int, qm), __builtin_bit_cast(int, qm), false, false);
        qm = fmaxf(__builtin_bit_cast(float, (int)hb[0]), __builtin_bit_cast(float, (int)hb[1]));
        const uint32_t qe = ap_exp(qm);
        qm = group_max<32>(qm);
        if (l == 0) reinterpret_cast<float*>(lds + L::QM)[wave] = qm;
        const float qs = ap_scale<AP_KQ>(qe), mo = ap_minus_one();
        qf = ap_unscale<AP_KQ>(qe) * a.scale;
        #pragma unroll
        for (int s = 0; s < HD / 16; s++) {
            uint32_t h[4], lo[4];
            ap_split(qv[2 * s].x * qs, qv[2 * s].y * qs, mo, h[0], lo[0]);
            ap_split(qv[2 * s].z * qs, qv[2 * s].w * qs, mo, h[1], lo[1]);
            ap_split(qv[2 * s + 1].x * qs, qv[2 * s + 1].y * qs, mo, h[2], lo[2]);
            ap_split(qv[2 * s + 1].z * qs, qv[2 * s + 1].w * qs, mo, h[3], lo[3]);
            qh[s] = __builtin_bit_cast(h8v, u32x4v{h[0], h[1], h[2], h[3]});
            ql[s] = __builtin_bit_cast(h8v, u32x4v{lo[0], lo[1], lo[2], lo[3]});
        }
    }
    const int nb = b_hi - b_lo;
    if (t < 2) reinterpret_cast<int*>(lds + L::GROW)[t] = -1;
    ap_vmax<HD>(lds, reg, 0, t);
    __syncthreads();
    ap_convert<HD>(lds, reg, 0, t, ve, ke_max, bad);
    if (nb > 1) {
        ap_load<HD>(reg, kr, vr, b_lo + 1, t);
        ap_vmax<HD>(lds, reg, 1, t);
    }
    f32x16 o[L::NB] = {};
    float m = -INFINITY, lsum = 0.0f;
    for (int n = 0; n < nb; n++) {
        // block n is in its stage, block n + 1's V maxima are there, and
        // every wave is done with the other stage
        __syncthreads();
        const int grown = reinterpret_cast<const int*>(lds + L::GROW)[n & 1];
        if (n + 1 < nb) ap_convert<HD>(lds, reg, n + 1, t, ve, ke_max, bad);
        if (n + 2 < nb) ap_load<HD>(reg, kr, vr, b_lo + n + 2, t);
        const int j0 = 32 * (b_lo + n);
        ap_rescale<HD>(lds, n, __builtin_amdgcn_readfirstlane(grown), g, o);
        if (j0 < row.vis_last) ap_compute<HD>(lds, n, j0, qh, ql, qf, c, g, row, m, lsum, o);
        if (n + 2 < nb) ap_vmax<HD>(lds, reg, n & 1, t);
    }
    // values too far apart, sums that are not finite: the whole tile again in
    // f32 (0 * x is 0 or NaN)
    const float* qw = reinterpret_cast<const float*>(lds + L::QM);
    const uint32_t qe = ap_exp(fmaxf(fmaxf(qw[0], qw[1]), fmaxf(qw[2], qw[3])));
    bad |= ke_max + qe >= 2u * 127u + AP_SCORE || ke_max > 200u;
    float z = lsum * 0.0f;
    #pragma unroll
    for (int u = 0; u < HD / 32; u++)
        #pragma unroll
        for (int r = 0; r < 16; r++) z = __builtin_fmaf(o[u][r], 0.0f, z);
    if (__syncthreads_or(bad || (row.ok && z != 0.0f))) {
        ap_rows_f32<HD>(lds, lds0, a, grp, tile, piece, b_lo, b_hi);
        return;
    }
    if (!row.ok) return;
    // the sum into [1, 2) and O with it, so that O times V's scale stays in
    // f32's range wherever its results do (m can lag by 2^32)
    const uint32_t le = lsum > 0.0f ? __builtin_bit_cast(uint32_t, lsum) >> 23 : 127u;
    const float dn = __builtin_bit_cast(float, (254u - le) << 23);
    lsum *= dn;
    if (piece >= 0 && g == 0) ap_store_ml<HD>(a, row, piece, m + (float)((int)le - 127), lsum);
    #pragma unroll
    for (int u = 0; u < HD / 32; u++)
        #pragma unroll
        for (int q = 0; q < 4; q++) {
            const int d = 32 * u + 8 * q + 4 * g;
            const float4 f = *reinterpret_cast<const float4*>(lds + L::VS + 4 * d);
            ap_store4<HD>(a, row, piece, d,
                          make_float4(o[u][4 * q] * dn * f.x, o[u][4 * q + 1] * dn * f.y, o[u][4 * q + 2] * dn * f.z,
                                      o[u][4 * q + 3] * dn * f.w), lsum);
        }
}

// Causal prompts leave a tile with more position blocks the later it comes.
// Workgroup x takes entry x / groups of group x % groups of the list that
// runs from the longest tile down (a free CU takes the longest piece left;
// with eight kv heads each XCD keeps to one head's K and V): whole tiles, or
// with chunk > 0 each tile's pieces of chunk blocks.
template <int HD>
__global__ __launch_bounds__(64 * AP_NW, 2)
void attn_prompt_kernel(ApArgs a) {
    __shared__ __align__(16) uint8_t lds[ApLds<HD>::TOTAL];
    const int grp = blockIdx.x % a.groups;
    int tile = (a.q_len * a.G + AP_ROWS - 1) / AP_ROWS - 1, piece = blockIdx.x / a.groups;
    if (a.chunk > 0) {
        for (; tile >= 0; tile--) {
            const int pieces = (ap_tile_blocks(tile, a.G, a.q_len, a.kv_len, a.start_pos) + a.chunk - 1) / a.chunk;
            if (piece < pieces) break;
            piece -= pieces;
        }
    } else {
        tile -= piece;
        piece = 0;
    }
    if (tile < 0) return;   // past the list (the grid is its length)
    ap_tile<HD>(lds, lds_addr(lds), a, grp, tile, piece);
}

// ---- launch ------------------------------------------------------------------

// The plan of the last shape and device this thread asked for: the choice of
// the kernel, the workspace query and the launch ask in turn.
static ApPlan attn_prompt_plan(size_t n_head, size_t n_head_kv, size_t head_dim, size_t q_len, size_t kv_len) {
    struct Entry {
        size_t key[5];
        int dev;
        ApPlan plan;
        bool valid;
    };
    thread_local Entry last = {{0, 0, 0, 0, 0}, -1, ApPlan{}, false};
    const int ovr = tuning_env(TUNE_ATTN_MFMA_SPLIT);   // pieces of the longest tile (tuning)
    if (ovr > 0) return ap_plan(n_head, n_head_kv, head_dim, q_len, kv_len, (size_t)cu_count_attn(), ovr);
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess) dev = -1;
    if (last.valid && last.dev == dev && last.key[0] == n_head && last.key[1] == n_head_kv && last.key[2] == head_dim &&
        last.key[3] == q_len && last.key[4] == kv_len)
        return last.plan;
    const ApPlan p = ap_plan(n_head, n_head_kv, head_dim, q_len, kv_len, (size_t)cu_count_attn(), 0);
    last = Entry{{n_head, n_head_kv, head_dim, q_len, kv_len}, dev, p, true};
    return p;
}

bool attn_prompt_path(size_t n_head, size_t n_head_kv, size_t head_dim, size_t q_len, size_t kv_len) {
    const int min_q = tuning_env(TUNE_ATTN_MFMA_MIN_Q);
    if (!ap_supported(head_dim, kv_len) || q_len < (min_q > 0 ? (size_t)min_q : 2)) return false;
    if (min_q > 0) return true;
    return ap_path(n_head, n_head_kv, head_dim, q_len, kv_len, attn_prompt_plan(n_head, n_head_kv, head_dim, q_len, kv_len));
}

size_t attn_prompt_workspace(size_t n_head, size_t n_head_kv, size_t head_dim, size_t q_len, size_t kv_len) {
    const ApPlan p = attn_prompt_plan(n_head, n_head_kv, head_dim, q_len, kv_len);
    return p.chunk > 0 ? (size_t)p.stride * n_head * q_len * (head_dim + 2) * sizeof(float) : 0;
}

bool attn_prompt_q8_direct(const AttnArgs& a) {
    return attn_prompt_plan(a.n_head, a.n_head_kv, a.head_dim, a.q_len, a.kv_len).chunk > 0;
}

template <int HD>
static hipError_t attn_prompt_launch_t(const AttnArgs& a, hipStream_t s) {
    const ApPlan p = attn_prompt_plan(a.n_head, a.n_head_kv, HD, a.q_len, a.kv_len);
    ApArgs k{};
    k.q = a.q;
    k.k = a.k + a.layer_off;
    k.v = a.v + a.layer_off;
    k.head_stride = a.head_stride;
    k.n_head = (int)a.n_head;
    k.n_head_kv = (int)a.n_head_kv;
    k.G = p.G;
    k.groups = p.groups;
    k.q_len = (int)a.q_len;
    k.kv_len = (int)a.kv_len;
    k.start_pos = (long long)a.start_pos;
    k.scale = (1.0f / sqrtf((float)HD)) * LOG2E;
    k.out = a.out;
    k.part = a.part;
    k.chunk = p.chunk;
    k.stride = p.stride;
    k.all_parts = a.out_q8 != nullptr;
    unsigned n = (unsigned)p.tiles;
    if (p.chunk > 0) {   // the pieces of every tile at the actual start position
        n = 0;
        for (int t = 0; t < p.tiles; t++)
            n += (unsigned)((ap_tile_blocks(t, p.G, k.q_len, k.kv_len, k.start_pos) + p.chunk - 1) / p.chunk);
    }
    hipLaunchKernelGGL(attn_prompt_kernel<HD>, dim3(n * (unsigned)p.groups), dim3(64 * AP_NW), 0, s, k);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || p.chunk == 0) return e;
    const dim3 cg((unsigned)(((a.n_head * HD + 255) / 256 + 3) / 4), (unsigned)a.q_len);
    if (a.out_q8)
        hipLaunchKernelGGL((attn_combine_few_kernel<HD, true>), cg, dim3(256), 0, s, a.part, p.stride, p.chunk,
                           (int)a.n_head, p.G, (int)a.q_len, (int)a.kv_len, (long long)a.start_pos, a.out, a.out_q8);
    else
        hipLaunchKernelGGL((attn_combine_few_kernel<HD, false>), cg, dim3(256), 0, s, a.part, p.stride, p.chunk,
                           (int)a.n_head, p.G, (int)a.q_len, (int)a.kv_len, (long long)a.start_pos, a.out, a.out_q8);
    return hipGetLastError();
}

hipError_t attn_prompt_launch(const AttnArgs& a, hipStream_t s) {
    return a.head_dim == 64 ? attn_prompt_launch_t<64>(a, s) : attn_prompt_launch_t<128>(a, s);
}

}  // namespace barq
