// Which path a multi-token attention call takes, in how many key splits, and what it needs of the
// handle's workspaces: host arithmetic without HIP, which the CPU tests build with g++.
#pragma once

#include <algorithm>
#include <cstddef>

namespace llmp {

// Tokens per group of the token-batched projections (the MFMA's N).
constexpr int kTokBatch = 16;
constexpr int kMaxPrefillSplits = 64;

// ---- the 16x16 path (prefill_kernels.h) -------------------------------------------------------
// Keys per tile and bytes per tile image (per KV head) for head_dim; 0 if unsupported.
constexpr int prefill_tile_keys(int head_dim) {
    return head_dim == 64 || head_dim == 96 || head_dim == 128 ? 64 : head_dim == 256 ? 32 : 0;
}
constexpr size_t prefill_tile_bytes(int head_dim) {
    // hi and lo parts of K rows (padded at head_dim 96) and of V^T, and the flag words
    const size_t tk = (size_t)prefill_tile_keys(head_dim), pitch = (size_t)(head_dim == 96 ? 112 : head_dim);
    return tk == 0 ? 0 : 4 * tk * (pitch + (size_t)head_dim) + 16;
}
// Launch shape of the attention kernel: one query head per wave (measured best at 32/8/64, 2048
// tokens: each wave's K/V fragments feed its MFMAs while occupancy stays at 4 waves/SIMD),
// 16 * NB query tokens per workgroup, at most 8 waves.  nb_big is used when the grid then still
// holds two workgroups per CU, else half of it (short prompts).
constexpr int nb_big(int group) { return group >= 8 ? 1 : (8 / group >= 4 ? 4 : 8 / group); }
// Workgroups per key split: query blocks of 16 * NB tokens times KV heads.
inline int prefill_items(int P, int n_kv_heads, int nb) { return ((P + 16 * nb - 1) / (16 * nb)) * n_kv_heads; }
// Query blocks per workgroup the launch uses for P tokens.
inline int prefill_nb(int P, int n_kv_heads, int group, int n_cu) {
    const int nb = nb_big(group);
    return nb > 1 && prefill_items(P, n_kv_heads, nb) < 2 * n_cu ? nb / 2 : nb;
}
// Key splits of a call: 1 unless the query blocks alone leave CUs idle (short prompts after a long
// cached prefix, speculative verification).
inline int prefill_key_splits(int P, int pos0, int window, int n_kv_heads, int group, int head_dim, int n_cu) {
    const int TK = prefill_tile_keys(head_dim);
    if (TK <= 0 || group <= 0) return 1;
    const int items = prefill_items(P, n_kv_heads, prefill_nb(P, n_kv_heads, group, n_cu));
    if (items >= n_cu) return 1;
    // Key tiles of the last query (the heaviest workgroup's range, up to one block's spread).
    const int last = pos0 + P - 1;
    const int kbeg = window > 0 ? std::max(0, last - window + 1) : 0;
    const int tiles = last / TK - kbeg / TK + 1;
    int ks = (2 * n_cu + items - 1) / items;          // about two workgroups per CU
    ks = std::min(ks, std::max(1, tiles / 2));        // at least two tiles per split
    return std::max(1, std::min(ks, kMaxPrefillSplits));
}

// ---- the wide path (prefill_wide_kernels.h) -----------------------------------------------------
constexpr int kWideCols = 128;   // columns (token, head) per workgroup
constexpr int prefill_wide_tile_keys(int head_dim) {
    return head_dim == 64 ? 64 : head_dim == 96 || head_dim == 128 ? 32 : 0;
}
constexpr size_t prefill_wide_tile_bytes(int head_dim) {
    // K and V, hi and lo, and the tile's flag word
    return (size_t)prefill_wide_tile_keys(head_dim) * (size_t)head_dim * 8 + sizeof(unsigned);
}
// The launch of a call: workgroups per key split, key splits, groups of 4 waves per workgroup and
// whether a workgroup takes a pair of blocks (prefill_wide_kernel).
struct WidePlan {
    int items, ksplit, groups, pairs;
};
inline WidePlan wide_plan(int P, int pos0, int window, int hkv, int group, int head_dim, int n_cu) {
    const int TK = prefill_wide_tile_keys(head_dim);
    const int nblk = (int)(((long long)P * group + kWideCols - 1) / kWideCols);
    const int last = pos0 + P - 1;
    const int tiles = last / TK - (window > 0 ? std::max(0, last - window + 1) : 0) / TK + 1;   // of the last block
    const int pair_items = (nblk + 1) / 2 * hkv;
    if (pair_items > n_cu) return {nblk * hkv, 1, 1, 0};
    if (2 * pair_items > n_cu) return {pair_items, 1, 2, 1};
    // Splits cost a combine launch and the partials' bytes: at least 12 tiles each, or 4 where the
    // blocks alone would leave seven CUs in eight idle.
    int ks = n_cu / (nblk * hkv);
    ks = std::max(1, std::min(std::min(ks, tiles / (nblk * hkv <= n_cu / 8 ? 4 : 12)), kMaxPrefillSplits));
    return {nblk * hkv, ks, 2, 0};
}
// A call takes the wide path when its matrix work pays for the image pass and the longer prologue
// (about 10 us together) and its key tiles feed enough column blocks.  Both paths measured over
// prompts of 70-1500 tokens after 0-12000 rows cross at 0.4-0.7 G multiply-adds of K Q^T at
// 24/8/128 and 32/8/64 (24/8/128 from position 0: 500 tokens 39.5 us against 40.7, 700 tokens 51.1
// against 48.3; after 3000 rows: 70 tokens 39.0 against 40.7, 100 tokens 54.9 against 46.3), and at
// 0.9-1.1 G at 16/8/128 (after 3000 rows: 150 tokens 42.8 against 50.0, 200 tokens 60.7 against
// 55.3), where the 16x16 kernel's eight waves share each tile.  The key splits of such a call, 0 of
// any other.
inline int prefill_wide_splits(int P, int pos0, int window, int n_kv_heads, int group, int head_dim, int n_cu) {
    if (prefill_wide_tile_keys(head_dim) == 0) return 0;
    const bool shared = head_dim >= 96 && group <= 2;
    const double avg = pos0 + (P + 1) / 2.0, keys = window > 0 ? std::min<double>(avg, window) : avg;
    const double work = (double)P * group * n_kv_heads * keys * head_dim;
    if ((long long)P * group < (shared ? 256 : 192) || work < (shared ? 1.0e9 : 5.0e8)) return 0;
    return wide_plan(P, pos0, window, n_kv_heads, group, head_dim, n_cu).ksplit;
}

// ---- workspaces -----------------------------------------------------------------------------------
// A layer's heads as the kernels run them: krep virtual KV heads of `group` query heads per cached
// KV head.
struct PrefillShape {
    int n_kv_heads, krep, group, head_dim, window, n_cu;
    int n_heads() const { return n_kv_heads * krep * group; }
};
// What a call of n tokens at pos0 needs on one of the two paths: its key tiles (from the first
// query's window start, or 0, to the last new row), the key splits (0: the wide path does not take
// the call), and the bytes of the tile images and of the split partials.
struct PrefillNeed {
    int TK, tile0, n_tiles, ksplit;
    size_t ws, part;
    size_t total() const { return ws + part; }
};
inline PrefillNeed prefill_need(const PrefillShape& s, int pos0, int n, bool wide) {
    const int D = s.head_dim;
    PrefillNeed r{};
    r.ksplit = wide ? prefill_wide_splits(n, pos0, s.window, s.n_kv_heads * s.krep, s.group, D, s.n_cu)
                    : prefill_key_splits(n, pos0, s.window, s.n_kv_heads * s.krep, s.group, D, s.n_cu);
    if (r.ksplit == 0) return r;
    r.TK = wide ? prefill_wide_tile_keys(D) : prefill_tile_keys(D);
    r.tile0 = (s.window > 0 ? std::max(0, pos0 - s.window + 1) : 0) / r.TK;
    r.n_tiles = (pos0 + n - 1) / r.TK - r.tile0 + 1;
    const size_t tiles = (size_t)s.n_kv_heads * (size_t)r.n_tiles;
    if (wide) r.ws = (tiles * prefill_wide_tile_bytes(D) + 255) & ~(size_t)255;
    else if (r.ksplit == 1) r.ws = tiles * prefill_tile_bytes(D);   // splits stage straight from the cache
    if (r.ksplit > 1) r.part = (size_t)r.ksplit * (size_t)n * (size_t)s.n_heads() * (size_t)(D + 2) * sizeof(float);
    return r;
}
// Bytes that the handle's workspaces hold: the wide path's, and the tile images and split partials
// of the other.
struct PrefillHave {
    size_t wide, ws, part;
};
// Whether a call runs in them as they are: on the wide path, or on the other in its own workspaces
// or, all of it, in the wide one.
inline bool prefill_fits(const PrefillShape& s, int pos0, int n, const PrefillHave& have) {
    const PrefillNeed w = prefill_need(s, pos0, n, true), p = prefill_need(s, pos0, n, false);
    return (w.ksplit > 0 && w.total() <= have.wide) || (p.ws <= have.ws && p.part <= have.part) ||
           p.total() <= have.wide;
}

// ---- passes of the attention half of many tokens (llmp_attn_block_batch) ---------------------------
// Tokens from which the projections run as tiled products (proj_gemm_kernels.h): about where the two
// cross at the 24/8/128 shape.  Whole calls there, groups against tiled, us: Q4_K_M 144 tokens 174
// against 184, 176 tokens 204 against 184; Q8_0 112 tokens 162 against 161; F32 80 tokens 162 against
// 178.  In groups a token costs 45-90 us per G weights by format, tiled a call has 55 us and 18 us per
// 1000 columns to spend first, so other widths cross elsewhere: 32/8/128 (dim 4096) at 50-90 tokens,
// 32/8/64 (dim 2048) at 110-170, but 16/8/128 (dim 1024) at 190-280 (144 tokens in Q4_K_M 86 against
// 122) and 4/1/256 (dim 1152) at 340-420 (144 tokens in Q8_0 61 against 97).
constexpr int kGemmTokens = 136;
// Tokens of one pass through the projections and the attention: bounds the scratch (about 120 MB
// at the 24/8/128 shape) at no cost, since a pass this long fills the chip many times over.
constexpr int kPassTokens = 2048;

// Tokens of a pass of K that run together, in one attention call; the rest, one token or none, runs
// as a single-token call behind them (27 against 49 us at 24/8/128 for a group of one token).  The
// tiled products have no such group.
inline int batch_together(int K, bool q8_input) {
    return K % kTokBatch == 1 && (q8_input || K < kGemmTokens) ? K - 1 : K;
}
// Whether the attention calls of n_tokens tokens in passes of `pass` fit the workspaces.  (Every
// call is looked at as it is made: fewer tokens can take more key splits and more partials.  After
// 8000 rows of 24/8/128, 33 tokens would take 22 splits, the 32 that run take 32.)
inline bool batch_fits(const PrefillShape& s, int pos0, int n_tokens, int pass, bool q8_input, const PrefillHave& have) {
    for (int t0 = 0; t0 < n_tokens; t0 += pass) {
        const int n = batch_together(std::min(pass, n_tokens - t0), q8_input);
        if (n > 0 && !prefill_fits(s, pos0 + t0, n, have)) return false;
    }
    return true;
}

}  // namespace llmp
