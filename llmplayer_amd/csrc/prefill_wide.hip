// Instantiation and dispatch of the wide multi-token attention (prefill_wide_kernels.h).
#include "prefill_wide_kernels.h"

#include <algorithm>

namespace llmp {
namespace {

int tile_keys(int head_dim) { return head_dim == 64 ? pk::WideTile<64>::TK : pk::WideTile<128>::TK; }

// The launch of a call: workgroups per key split, key splits, groups of 4 waves per workgroup and
// whether a workgroup takes a pair of blocks (prefill_wide_kernel).
struct WidePlan {
    int items, ksplit, groups, pairs;
};
WidePlan wide_plan(int P, int pos0, int window, int hkv, int group, int head_dim, int n_cu) {
    const int TK = tile_keys(head_dim);
    const int nblk = (int)(((long long)P * group + pk::kWideCols - 1) / pk::kWideCols);
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

template <int D>
hipError_t launch_wide_d(const pk::PrefillArgs& a, int group, void* ws, int tile0, int n_tiles, int row_end,
                         int n_cu, hipStream_t stream) {
    using T = pk::WideTile<D>;
    uint4* img = static_cast<uint4*>(ws);
    unsigned* flags = reinterpret_cast<unsigned*>(img + (size_t)a.Hkv * n_tiles * T::U4);
    const dim3 grid(n_tiles, a.Hkv), block(pk::wide_tile_threads<D>());
    if constexpr (D == 96) {   // fp32 caches only at head_dim 96
        if (a.kq != nullptr) return hipErrorInvalidValue;
        hipLaunchKernelGGL((pk::prefill_wide_tile_kernel<D, false>), grid, block, 0, stream, a, img, flags,
                           tile0, n_tiles, row_end);
    } else if (a.kq != nullptr) {
        hipLaunchKernelGGL((pk::prefill_wide_tile_kernel<D, true>), grid, block, 0, stream, a, img, flags,
                           tile0, n_tiles, row_end);
    } else {
        hipLaunchKernelGGL((pk::prefill_wide_tile_kernel<D, false>), grid, block, 0, stream, a, img, flags,
                           tile0, n_tiles, row_end);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const WidePlan p = wide_plan(a.P, a.pos0, a.window, a.Hkv * a.kv_rep, group, D, n_cu);
    const dim3 agrid(p.items, p.ksplit), ablock(p.groups * pk::kWideThreads);
    auto launch = [&](auto cap, auto groups) {
        hipLaunchKernelGGL((pk::prefill_wide_kernel<D, decltype(cap)::value, decltype(groups)::value>), agrid, ablock, 0,
                           stream, a, img, flags, tile0, n_tiles, p.ksplit, group, p.pairs);
    };
    using one = std::integral_constant<int, 1>;
    using two = std::integral_constant<int, 2>;
    if (a.softcap > 0.0f) {
        if (p.groups == 2) launch(std::true_type{}, two{});
        else launch(std::true_type{}, one{});
    } else {
        if (p.groups == 2) launch(std::false_type{}, two{});
        else launch(std::false_type{}, one{});
    }
    const int ksplit = p.ksplit;
    e = hipGetLastError();
    return e != hipSuccess || ksplit <= 1 ? e : launch_prefill_combine(a, D, ksplit, stream);
}

}  // namespace

int prefill_wide_tile_keys(int head_dim) {
    return head_dim == 64 || head_dim == 96 || head_dim == 128 ? tile_keys(head_dim) : 0;
}

size_t prefill_wide_tile_bytes(int head_dim) {
    // K and V, hi and lo, and the tile's flag word
    return (size_t)prefill_wide_tile_keys(head_dim) * head_dim * 8 + sizeof(unsigned);
}

// A call takes the wide path when its matrix work pays for the image pass and the longer prologue
// (about 10 us together) and its key tiles feed enough column blocks.  Both paths measured over
// prompts of 70-1500 tokens after 0-12000 rows cross at 0.4-0.7 G multiply-adds of K Q^T at
// 24/8/128 and 32/8/64 (24/8/128 from position 0: 500 tokens 39.5 us against 40.7, 700 tokens 51.1
// against 48.3; after 3000 rows: 70 tokens 39.0 against 40.7, 100 tokens 54.9 against 46.3), and at
// 0.9-1.1 G at 16/8/128 (after 3000 rows: 150 tokens 42.8 against 50.0, 200 tokens 60.7 against
// 55.3), where the 16x16 kernel's eight waves share each tile.
int prefill_wide_splits(int P, int pos0, int window, int n_kv_heads, int group, int head_dim, int n_cu) {
    if (prefill_wide_tile_keys(head_dim) == 0) return 0;
    const bool shared = head_dim >= 96 && group <= 2;
    const double avg = pos0 + (P + 1) / 2.0, keys = window > 0 ? std::min<double>(avg, window) : avg;
    const double work = (double)P * group * n_kv_heads * keys * head_dim;
    if ((long long)P * group < (shared ? 256 : 192) || work < (shared ? 1.0e9 : 5.0e8)) return 0;
    return wide_plan(P, pos0, window, n_kv_heads, group, head_dim, n_cu).ksplit;
}

hipError_t launch_prefill_wide(const pk::PrefillArgs& a, int head_dim, int group, void* ws, int tile0, int n_tiles,
                               int row_end, int n_cu, hipStream_t stream) {
    switch (head_dim) {
    case 64: return launch_wide_d<64>(a, group, ws, tile0, n_tiles, row_end, n_cu, stream);
    case 96: return launch_wide_d<96>(a, group, ws, tile0, n_tiles, row_end, n_cu, stream);
    case 128: return launch_wide_d<128>(a, group, ws, tile0, n_tiles, row_end, n_cu, stream);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace llmp
