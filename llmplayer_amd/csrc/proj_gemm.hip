// Instantiation and dispatch of the many-token projection kernels (proj_gemm_kernels.h).
#include "proj_gemm_kernels.h"
#include "llmp_internal.h"

namespace llmp {
namespace {

template <class F1, class F2>
hipError_t launch_ff(const tk::ProjGemmArgs& a, hipStream_t st) {
    const int tiles = a.row_tiles * a.tok_tiles;
    hipLaunchKernelGGL((tk::proj_gemm_kernel<F1, F2>), dim3((tiles + 7) / 8 * 8), dim3(tk::kGemmThreads), 0, st, a);
    return hipGetLastError();
}

// A format as the product takes it.
template <class F> struct GemmFormat { using type = F; };
template <> struct GemmFormat<tk::PQ4K> { using type = tk::GQ4K; };
template <> struct GemmFormat<tk::PQ5K> { using type = tk::GQ5K; };
template <> struct GemmFormat<tk::PQ5_1> { using type = tk::GQ5_1; };
template <> struct GemmFormat<tk::PQ2_K> { using type = tk::GQ2_K; };

template <class Fn>
hipError_t with_format(int t, Fn fn) {
    switch (t) {
    case gk::kF32: return fn(tk::PF32{});
    case gk::kF16: return fn(tk::PF16{});
    case gk::kBF16: return fn(tk::PBF16{});
    case gk::kQ8_0: return fn(tk::PQ8_0{});
    case gk::kQ4_0: return fn(tk::PQ4_0{});
    case gk::kQ4_K: return fn(tk::PQ4K{});
    case gk::kQ6_K: return fn(tk::PQ6K{});
    case gk::kQ5_0: return fn(tk::PQ5_0{});
    case gk::kQ3_K: return fn(tk::PQ3K{});
    case gk::kQ5_K: return fn(tk::PQ5K{});
    case gk::kIQ4_NL: return fn(tk::PIQ4_NL{});
    case gk::kIQ4_XS: return fn(tk::PIQ4_XS{});
    case gk::kMXFP4: return fn(tk::PMXFP4{});
    case gk::kQ5_1: return fn(tk::PQ5_1{});
    case gk::kQ2_K: return fn(tk::PQ2_K{});
    case gk::kIQ3_XXS: return fn(tk::PIQ3_XXS{});
    case gk::kIQ3_S: return fn(tk::PIQ3_S{});
    case gk::kIQ2_S: return fn(tk::PIQ2_S{});
    default: return hipErrorInvalidValue;
    }
}

}  // namespace

hipError_t launch_weight_range(const gk::WPlanes& w, int ggml_type, int rows, int cols, int* rexp, hipStream_t st) {
    if (rows <= 0 || rows % 16 || cols <= 0 || cols % 32 || rexp == nullptr) return hipErrorInvalidValue;
    return with_format(ggml_type, [&](auto f) {
        hipLaunchKernelGGL((tk::weight_range_kernel<decltype(f)>), dim3(rows / 16), dim3(tk::kThreads), 0, st, w, cols, rexp);
        return hipGetLastError();
    });
}

int proj_gemm_steps(int cols) { return (cols + tk::kChunk - 1) / tk::kChunk * (tk::kChunk / 16); }

namespace {
int input_tiles(int n_tokens) { return (n_tokens + tk::kGemmToks - 1) / tk::kGemmToks * (tk::kGemmToks / 32); }
// The input sums, behind the fragments.
float* input_sums(const void* xs, int n_tokens, int steps) {
    return reinterpret_cast<float*>(static_cast<uint4*>(const_cast<void*>(xs)) + (size_t)input_tiles(n_tokens) * steps * 128);
}
}  // namespace

size_t proj_gemm_input_bytes(int n_tokens, int cols) {
    return (size_t)input_tiles(n_tokens) * (size_t)proj_gemm_steps(cols) * (128 * sizeof(uint4) + 32 * sizeof(float));
}

hipError_t launch_tok_split(const float* x, long long x_pitch, int cols, const float* norm_w, float eps, float* sc,
                            int n_tokens, void* xs, hipStream_t st) {
    if (x == nullptr || sc == nullptr || xs == nullptr || cols <= 0 || cols % 32 || (x_pitch & 3) || n_tokens < 1 ||
        (reinterpret_cast<uintptr_t>(x) & 15) || (reinterpret_cast<uintptr_t>(norm_w) & 15) ||
        (reinterpret_cast<uintptr_t>(xs) & 15))
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(tk::tok_scale_kernel<tk::kPrepThreads>, dim3(n_tokens), dim3(tk::kPrepThreads), 0, st, x,
                       x_pitch, cols, norm_w, eps, sc);
    const int steps = proj_gemm_steps(cols);
    hipLaunchKernelGGL(tk::tok_split_kernel<256>, dim3(input_tiles(n_tokens), (steps + 15) / 16), dim3(256), 0, st, x,
                       x_pitch, cols, norm_w, sc, n_tokens, steps, static_cast<uint4*>(xs),
                       input_sums(xs, n_tokens, steps));
    return hipGetLastError();
}

hipError_t launch_proj_gemm(tk::ProjGemmArgs a, int first_type, int second_type, hipStream_t st) {
    if (a.cols <= 0 || a.cols % 32 || a.K < 1 || a.nseg < 1 || a.nseg > 3 || a.xs == nullptr || a.tok_sc == nullptr)
        return hipErrorInvalidValue;
    a.row_tiles = 0;
    for (int i = 0; i < a.nseg; ++i) {
        if (a.seg[i].rows <= 0 || a.seg[i].rexp == nullptr) return hipErrorInvalidValue;
        a.seg[i].tile0 = a.row_tiles;
        a.row_tiles += (a.seg[i].rows + tk::kGemmRows - 1) / tk::kGemmRows;
    }
    a.tok_tiles = (a.K + tk::kGemmToks - 1) / tk::kGemmToks;
    a.steps = proj_gemm_steps(a.cols);
    a.xsum = input_sums(a.xs, a.K, a.steps);
    if (second_type >= 0) {
        if (!proj_tok_pair_supported(first_type, second_type)) return hipErrorInvalidValue;
        if (first_type == gk::kQ3_K) return launch_ff<tk::PQ3K, tk::GQ5K>(a, st);
        if (first_type == gk::kQ5_K) return launch_ff<tk::GQ5K, tk::PQ6K>(a, st);
        return launch_ff<tk::GQ4K, tk::PQ6K>(a, st);
    }
    return with_format(first_type, [&](auto f) {
        using F = typename GemmFormat<decltype(f)>::type;
        return launch_ff<F, F>(a, st);
    });
}

}  // namespace llmp
