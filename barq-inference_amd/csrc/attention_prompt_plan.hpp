// Prompt attention on the host: which calls take the kernel of
// attention_prompt.hip, and how a call's tiles are cut into workgroups.
#pragma once
#include <stddef.h>

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
    double us;    // expected time of the kernel and the merge (0: whole tiles, two or more workgroups per CU)
};

// A launch's time, us, if the tiles (runs of equal length, shortest first) are
// cut into pieces of c position blocks: the last to end of the workgroups,
// which take pieces in the list's order, longest tile first, two to a CU, and
// the merge.  A block takes 2.7 us with 128 dims and 1.35 with 64, a piece as
// long as 1.4 blocks more for its fixed part (the query rows, the first loads,
// the partial state), and two pieces that share a CU 1.2 times as long as one;
// the merge reads a row's pieces one after the other (0.085 us each) and all
// states go to memory and back at 2.3 TB/s.  Fitted on MI355X to 108 launches
// of 14 shapes (2 to 1024 rows, 0 to 16000 cached, 1 to 32 kv heads): 11 % off
// root mean square, and its choice is the fastest chunk measured for each.
struct ApRun {
    int blocks, tiles;
    // pieces of c blocks, by 1 / c (an integer division takes several times as
    // long, and a plan forms some thousand quotients; blocks < 2^18)
    size_t pieces(double inv) const { return (size_t)(((double)blocks - 0.5) * inv + 1.0) * (size_t)tiles; }
};
inline double ap_time(const std::vector<ApRun>& runs, size_t groups, size_t head_dim, size_t cus, int c) {
    constexpr double FIXED = 1.4, SHARE = 1.2, MERGE_PIECE = 0.085, MERGE_BYTE = 2.0 / 4.6e6;
    const double block = head_dim == 128 ? 2.7 : 1.35;
    const double inv = 1.0 / (double)c;
    const auto length = [&](const ApRun& r) { return (double)(r.blocks < c ? r.blocks : c) + FIXED; };
    size_t n = 0, merged = 0, blocks = 0;
    for (const ApRun& r : runs) {
        const size_t k = r.pieces(inv);
        n += k;
        if (r.blocks > c) merged += k;
        blocks += (size_t)r.blocks * (size_t)r.tiles;
    }
    double t = length(runs.back());
    if (n * groups > cus) {   // the longest piece shares its CU with the one cus places down the list
        size_t left = cus / groups, i = runs.size() - 1;
        while (i > 0 && runs[i].pieces(inv) <= left) left -= runs[i--].pieces(inv);
        t += (SHARE - 1.0) * length(runs[i]);
        double all = ((double)blocks + FIXED * (double)n) * (double)groups * SHARE / 2.0 / (double)cus;
        if (n * groups > 2 * cus) all += 0.5 * SHARE * length(runs.front());   // the CUs end about half a last piece apart
        t = t > all ? t : all;
    }
    t *= block;
    if (merged)
        t += MERGE_PIECE * (double)((runs.back().blocks + c - 1) / c) +
             MERGE_BYTE * (double)(merged * AP_ROWS * groups * (head_dim + 2) * sizeof(float));
    return t;
}

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
    std::vector<ApRun> runs;
    runs.reserve((size_t)p.tiles);
    size_t total = 0;
    for (int t = 0; t < p.tiles; t++) {
        const int nb = ap_tile_blocks(t, p.G, (int)q_len, (int)kv_len, start);
        if (!runs.empty() && runs.back().blocks == nb) runs.back().tiles++;
        else runs.push_back(ApRun{nb, 1});
        total += (size_t)nb;
    }
    const int longest = runs.back().blocks;
    int chunk = longest;
    if (pieces > 0) {
        chunk = (longest + pieces - 1) / pieces;
        p.us = ap_time(runs, (size_t)p.groups, head_dim, cus, chunk);
    } else {
        // Candidates: the smallest chunks that leave at most 1/4, 1/2, ... 2, 2
        // 1/2, ... 4 pieces per CU (more never measured faster).  Smaller chunks of as many
        // rounds of pieces only add pieces to merge, larger ones make the pieces
        // longer.  Ties keep the larger chunk.
        double best = p.us = ap_time(runs, (size_t)p.groups, head_dim, cus, longest);
        for (int k = 1; k <= 16; k += k < 8 ? 1 : 2) {
            const size_t most = cus * (size_t)k / 4 / (size_t)p.groups;   // per head group
            if (most <= (size_t)p.tiles) continue;
            // n(c) = sum of ceil(blocks / c) lies between total / c and that + tiles
            int lo = (int)((total + most - 1) / most), hi = (int)(total / (most - (size_t)p.tiles)) + 1;
            if (lo < 1) lo = 1;
            if (hi > longest) hi = longest;
            while (lo < hi) {
                const int mid = (lo + hi) / 2;
                size_t n = 0;
                for (const ApRun& r : runs) n += r.pieces(1.0 / (double)mid);
                if (n <= most) hi = mid;
                else lo = mid + 1;
            }
            if (lo >= chunk) continue;
            const double e = ap_time(runs, (size_t)p.groups, head_dim, cus, lo);
            if (e < best - 1e-9) {
                best = p.us = e;
                chunk = lo;
            }
        }
    }
    if (chunk < 1) chunk = 1;
    if (chunk >= longest) return p;   // every tile in one piece
    const int nbmax = (int)((kv_len + 31) / 32);
    p.chunk = chunk;
    p.stride = (nbmax + chunk - 1) / chunk;
    return p;
}

// Expected time, us, of the decode kernel (attention.hip), which runs each
// query row by itself: its products at 4.8 Tera multiply-adds/s (QK and PV
// counted once; up to 30 % more of them for many rows), or its K and V rows,
// read once per kv head for groups of 2, 4 or 8 query heads, else once per query
// head, at 11.5 TB/s, or 31 TB/s when the layer's K and V are below 8 MB and
// stay in the L2s.
inline double ap_rows_time(size_t n_head, size_t n_head_kv, size_t head_dim, size_t q_len, size_t kv_len) {
    const size_t g = n_head_kv && n_head % n_head_kv == 0 ? n_head / n_head_kv : 1;
    const double reads = (double)(g == 2 || g == 4 || g == 8 ? n_head_kv : n_head);   // of K and V per query row
    const double seen = (double)kv_len - 0.5 * (double)(q_len < kv_len ? q_len : kv_len);
    const double by_macs = (double)n_head / 4.8e6 * (q_len > 8 ? 0.7 + 2.4 / (double)q_len : 1.0);
    const double by_bytes = reads * 8.0 / ((double)kv_len * (double)(n_head_kv * head_dim) * 8.0 < 8e6 ? 31e6 : 11.5e6);
    return 10.0 + (double)q_len * seen * (double)head_dim * (by_macs > by_bytes ? by_macs : by_bytes);
}

// Whether a chunk takes this kernel: head_dim 64 or 128, a kv head's rows
// addressable by the 32-bit buffer offsets of its K/V loads, and clearly less
// time expected than for the decode kernel; this one's launches cost 9.4 us
// beside ap_time.  Fitted on MI355X to both kernels' times at 560 calls (14 head
// counts, both dims, 2 to 512 rows, 0 to 16000 cached): the kernel it takes is
// 2.6 % slower than the faster one on average (always this one 8 %, always the
// decode kernel 145 %), and this one is taken where it is over 10 % slower in 3
// of them (without the factor 1.1 in 12).  Some calls, us, decode kernel / this
// one: 32/8 heads of 128, 4000 cached, 6 / 8 / 12 rows 25 / 31, 31 / 31, 44 / 33;
// 500 cached, 48 / 64 rows 23 / 24, 23 / 25; from position 0, 64 / 203 rows 7 /
// 17, 21 / 23; 32/8 heads of 64, 4000 cached, 8 / 12 rows 19 / 21, 25 / 22; 32/32
// heads of 128, 4000 cached, 4 / 6 rows 48 / 43, 70 / 43; 14/2 heads of 64, 4000
// cached, 8 rows 16 / 20.  (BARQ_ATTN_MFMA_MIN_Q: this kernel from that many
// rows on, whatever the times.)
inline bool ap_supported(size_t head_dim, size_t kv_len) {
    return (head_dim == 64 || head_dim == 128) && kv_len < ((size_t)1 << 23);
}
inline bool ap_path(size_t n_head, size_t n_head_kv, size_t head_dim, size_t q_len, size_t kv_len, const ApPlan& plan) {
    return ap_supported(head_dim, kv_len) && q_len >= 2 &&
           ap_rows_time(n_head, n_head_kv, head_dim, q_len, kv_len) > 1.1 * (9.4 + plan.us);
}

}  // namespace barq
