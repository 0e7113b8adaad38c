// Prompt attention on the host: which calls take the kernel of
// attention_prompt.hip, and how a call's tiles are cut into workgroups.
#pragma once
#include <stddef.h>

#include <functional>
#include <queue>
#include <utility>
#include <vector>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define BARQ_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define BARQ_HOST_DEVICE inline
#endif

namespace barq {

constexpr int AP_NW = 4, AP_ROWS = 32 * AP_NW;   // waves of a workgroup, query rows of its tile

// Position blocks of 32 that tile `tile` of a kv head's flattened rows sees.
BARQ_HOST_DEVICE int ap_tile_blocks(int tile, int G, int q_len, int kv_len, long long start_pos) {
    const int row = tile * AP_ROWS + AP_ROWS - 1;
    const int i_last = row / G < q_len - 1 ? row / G : q_len - 1;
    const long long vis_last = start_pos + i_last + 1;
    const int j_end = (int)(vis_last < kv_len ? vis_last : kv_len);
    return (j_end + 31) / 32;
}

// Whether a chunk takes this kernel: head_dim 64 or 128, a kv head's rows
// addressable by the 32-bit buffer offsets of its K/V loads, and enough work
// for its longer fixed part.  The decode kernel (attention.hip) runs each
// query row by itself: a row costs its products at 5.5 Tera multiply-adds/s
// (QK and PV counted once) or its K and V rows from L2 at 14 TB/s (read once
// per kv head for groups of 2, 4 or 8 query heads, else once per query head).
// This kernel starts about 12 us later and reads K and V once, at 3.5 TB/s
// with the conversion.  Measured, us per call, decode kernel / this one:
// 32/8 heads of 128, 4000 cached, 6 / 8 / 12 rows 24.6 / 26.7, 30.0 / 27.2,
// 42.1 / 28.3; 500 cached, 24 / 40 rows 14.0 / 19.6, 21.5 / 21.2; 32/32 heads,
// 4000 cached, 4 / 6 rows 43.6 / 47.5, 69.5 / 47.4; 24/8 heads, 2 / 3 rows
// 24.4 / 25.6, 31.8 / 25.9; 32/8 heads of 64, 8 / 12 rows 19.1 / 19.6, 24.9 /
// 20.9; 40 rows from position 0: 7.7 / 15.8.  BARQ_ATTN_MFMA_MIN_Q: this
// kernel from that many rows on, whatever the work.
inline bool ap_path(size_t n_head, size_t n_head_kv, size_t head_dim, size_t q_len, size_t kv_len, int min_q) {
    if ((head_dim != 64 && head_dim != 128) || kv_len >= ((size_t)1 << 23)) return false;
    if (min_q > 0) return q_len >= (size_t)min_q;
    if (q_len < 2) return false;
    const size_t g = n_head_kv && n_head % n_head_kv == 0 ? n_head / n_head_kv : 1;
    const double reads = (double)(g == 2 || g == 4 || g == 8 ? n_head_kv : n_head);   // of K and V per query row
    const double seen = (double)kv_len - (q_len < kv_len ? 0.5 * (double)q_len : 0.5 * (double)kv_len);
    const double by_macs = (double)n_head / 5.5e6, by_bytes = reads * 8.0 / 14e6;   // us per position and dim
    const double rows_us = (double)q_len * seen * (double)head_dim * (by_macs > by_bytes ? by_macs : by_bytes);
    return rows_us > 1.2 * (12.0 + (double)kv_len * (double)(n_head_kv * head_dim) * 8.0 / 3.5e6);
}

// Launch plan: whole tiles, or pieces of `chunk` position blocks (partial
// states merged by attn_combine_few_kernel).  The plan assumes the chunk's queries are the
// last q_len of the kv_len positions (a prompt); at launch only the piece
// counts follow the actual start position, within `stride` pieces per tile
// (the workspace bound).
struct ApPlan {
    int G;        // query heads per kv head (1 when they do not divide)
    int groups;
    int tiles;    // per group
    int chunk;    // position blocks per piece; 0: whole tiles, no partial states
    int stride;   // partial states per (query row, head)
};

// pieces > 0: that many of the longest tile (tuning).
inline ApPlan ap_plan(size_t n_head, size_t n_head_kv, size_t head_dim, size_t q_len, size_t kv_len, size_t cus, int pieces) {
    ApPlan p{};
    p.G = (int)(n_head_kv && n_head % n_head_kv == 0 ? n_head / n_head_kv : 1);
    p.groups = (int)(n_head / p.G);
    p.tiles = (int)((q_len * p.G + AP_ROWS - 1) / AP_ROWS);
    p.chunk = 0;
    p.stride = 1;
    // where the tiles alone give every CU two workgroups, pieces only cost (2048
    // tokens, Llama-3-8B heads: 162 us whole, 200 us with the longer half cut in two)
    if ((size_t)p.tiles * p.groups >= 2 * cus) return p;
    const long long start = kv_len > q_len ? (long long)(kv_len - q_len) : 0;
    std::vector<int> nbs(p.tiles);
    int longest = 0;
    for (int t = 0; t < p.tiles; t++) {
        nbs[t] = ap_tile_blocks(t, p.G, (int)q_len, (int)kv_len, start);
        longest = nbs[t] > longest ? nbs[t] : longest;
    }
    // Choose the chunk by simulating the launch in units of one position block
    // (about 2 us): the pieces in the kernel's order (each costing its blocks
    // + FIXED for its fixed part: the query rows, the first loads, the partial
    // state), every CU holding up to two workgroups that share it equally,
    // each further piece going to the CU that frees a slot first; and the
    // partial states' way to memory and back (MERGE units per byte, about 4
    // TB/s).  Candidates cut the longest tile into k = 1, 2, ... pieces while
    // there are at most four pieces per CU in all (more never measured
    // faster); ties keep fewer pieces.
    constexpr double FIXED = 1.5, MERGE = 2.0 / 4e6 / 2.0;
    const double part_bytes = (double)AP_ROWS * p.groups * (head_dim + 2) * sizeof(float);
    auto simulate = [&](int c) {
        struct Cu { double t, w[2]; int n; };
        std::vector<Cu> cu(cus, Cu{0.0, {0.0, 0.0}, 0});
        auto event = [](const Cu& u) {
            return u.n == 2 ? u.t + 1.7 * (u.w[0] < u.w[1] ? u.w[0] : u.w[1]) : u.t + u.w[0];
        };
        typedef std::pair<double, size_t> Ev;
        std::priority_queue<Ev, std::vector<Ev>, std::greater<Ev>> heap;
        double end = 0.0, merged = 0.0;
        size_t placed = 0;
        auto finish = [&]() {   // the next piece to end; its CU has a slot free
            const Ev ev = heap.top();
            heap.pop();
            Cu& u = cu[ev.second];
            if (u.n == 2) {   // the shorter piece ends; the other has done as much
                const int done = u.w[0] < u.w[1] ? 0 : 1;
                u.w[0] = u.w[1 - done] - u.w[done];
                u.n = 1;
            } else {
                u.n = 0;
            }
            u.t = ev.first;
            end = ev.first > end ? ev.first : end;
            return ev.second;
        };
        for (int t = p.tiles - 1; t >= 0; t--) {   // the kernel's order: longest tiles first, then the head groups
            if (nbs[t] > c) merged += (nbs[t] + c - 1) / c * part_bytes;
            for (int b = 0; b < nbs[t]; b += c)
                for (int g = 0; g < p.groups; g++) {
                    const double len = (nbs[t] - b < c ? nbs[t] - b : c) + FIXED;
                    if (placed < 2 * cus) {   // the first round: one per CU, then a second
                        Cu& u = cu[placed % cus];
                        u.w[u.n++] = len;
                        if (++placed == 2 * cus)
                            for (size_t k = 0; k < cus; k++) heap.push(Ev(event(cu[k]), k));
                        continue;
                    }
                    const size_t k = finish();
                    cu[k].w[cu[k].n++] = len;
                    heap.push(Ev(event(cu[k]), k));
                }
        }
        if (placed < 2 * cus)
            for (size_t k = 0; k < cus; k++)
                if (cu[k].n) heap.push(Ev(event(cu[k]), k));
        while (!heap.empty()) {
            const size_t k = finish();
            if (cu[k].n) heap.push(Ev(event(cu[k]), k));
        }
        return end + MERGE * merged;
    };
    size_t chunk = (size_t)longest;
    double best = pieces > 0 ? 0.0 : simulate(longest);
    for (int k = 2; pieces <= 0 && k <= longest; k++) {
        const int c = (longest + k - 1) / k;
        if ((size_t)c >= chunk) continue;
        size_t n = 0;
        for (int nb : nbs) n += (size_t)((nb + c - 1) / c);
        if (n * p.groups > 4 * cus) break;   // smaller chunks only add pieces
        const double e = simulate(c);
        if (e < best - 1e-9) {
            best = e;
            chunk = (size_t)c;
        }
    }
    if (pieces > 0) chunk = ((size_t)longest + (size_t)pieces - 1) / (size_t)pieces;
    if (chunk < 1) chunk = 1;
    if (chunk >= (size_t)longest) return p;   // every tile in one piece
    const size_t nbmax = (kv_len + 31) / 32;
    p.chunk = (int)chunk;
    p.stride = (int)((nbmax + chunk - 1) / chunk);
    return p;
}

}  // namespace barq
