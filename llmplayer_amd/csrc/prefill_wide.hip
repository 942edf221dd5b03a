// Instantiation and dispatch of the wide multi-token attention (prefill_wide_kernels.h).
#include "prefill_wide_kernels.h"

namespace llmp {
namespace {

template <int D>
constexpr bool tile_as_planned() {
    using T = pk::WideTile<D>;
    return prefill_wide_tile_keys(D) == T::TK && prefill_wide_tile_bytes(D) == T::U4 * sizeof(uint4) + sizeof(unsigned);
}
static_assert(tile_as_planned<64>() && tile_as_planned<96>() && tile_as_planned<128>(), "the plan's tiles are the kernel's");
static_assert(kWideCols == pk::kWideCols, "the plan's blocks are the kernel's");

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
