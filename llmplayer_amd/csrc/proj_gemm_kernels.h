// Projections of many tokens (a prompt through llmp_attn_block_batch): Y[t][r] = sum_c W[r][c]
// x_t[c] as a tiled matrix product on v_mfma_f32_32x32x16_f16, from the weights' own GGUF planes.
//
// The 16-token kernel (proj_tok_kernels.h) decodes every weight and splits every input again for
// each group of 16 tokens; 63 groups of 1000 tokens took 63 x (22 + 12) us at the 24/8/128 shape with
// Q4_K_M weights.  Here a workgroup of 4 waves owns 64 rows x 128 tokens: the weights of a 32-column
// group are decoded once per 128 tokens, by the waves themselves, into LDS as fp16 operand
// fragments; the inputs were split once per call (tok_split_kernel) and stream through registers.
// Both are double buffered with one barrier per group, and two workgroups share a CU.
//
// Bound: neither memory nor the matrix units (a fifth busy) nor the vector units (a third), but the
// chain of a stage (operand reads, products beside the next group's decoding and the scaling, fragment
// writes, barrier) and the workgroup count: 640 for Q/K/V and 384 for Wo on 512 slots at 1000 tokens
// of that shape, where they take 160 and 108 us (64 and 39 GFLOP of products), against 1370 and 750 us
// in groups.  A 128 x 128 tile of 8 waves took 196 and 109 us where this one took 170 and 113 (with
// weights in two parts, then), and 226 against 178 us for the whole call at 96 tokens.
//
// Precision: no less than the 16-token kernel's.  Quantised weights are their exact integers, and a
// group's fp32 product is scaled afterwards (in two parts, hi + lo of the scaled weight, they lost
// 45 % to it: 1.66e-7 against 1.17e-7 from 64 bits with Q8_0 weights of 3072 columns; so 0.87e-7).
// Inputs are hi/lo parts brought into range by an exponent of their token, so both hold 2^-22 down
// to 2^-17 of its largest.  F32 weights are hi/lo parts, F16 and BF16 hi parts, in range by an
// exponent E_row of their row (weight_range_kernel, at upload), which the scales carry too.  Groups
// add up by FMA over a chunk of 128 columns and chunks in a compensated sum; F32, F16 and BF16 rows
// sum a chunk in the matrix unit and the chunks in fp32.
//
// Workgroups go to the XCDs in contiguous runs of a token-major order (block b runs on XCD b % 8),
// so an XCD's L2 holds the inputs of few token tiles while the much smaller quantised weights pass.
#pragma once

#include "proj_tok_kernels.h"

namespace llmp {
namespace tk {

typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int kGemmWaves = 4, kGemmThreads = kGemmWaves * 64;
constexpr int kGemmRows = 64, kGemmToks = 128;     // tile of a workgroup
constexpr int kGemmStage = 2;                      // 16-column steps per stage (one 32-column group)
constexpr int kGemmWFrags = 2 * kGemmStage * 2;    // 1 KB fragments per stage: weights (two 32-row tiles)
constexpr int kGemmXFrags = 4 * kGemmStage * 2;    // and inputs (four 32-token tiles)

struct GemmSeg {
    WPlanes w;
    int rows;
    int tile0;             // first row tile of the segment in the launch
    int fmt;               // launches over two formats: 0 = the first, 1 = the second
    const int* rexp;       // [rows] E_row
    const float* bias;     // [rows] or nullptr
    float* out;            // [K][out_pitch] (when resid is null)
    long long out_pitch;
};

struct ProjGemmArgs {
    GemmSeg seg[3];
    int nseg;
    int row_tiles, tok_tiles;
    int cols;              // a multiple of 32
    int K;                 // tokens
    const uint4* xs;       // tok_split_kernel: [32-token tile][16-column step][hi, lo][64 lanes]
    const float* xsum;     // and the sums of each step's inputs: [32-token tile][step][32 tokens]
    int steps;             // 16-column steps per tile in xs: whole 128-column chunks
    const float* tok_sc;   // [K][r, e]: the RMSNorm factor (1 without) and the input's exponent
    float* resid;          // resid[t*resid_pitch + row] += rscale? * value
    long long resid_pitch;
    float rscale;
};

// Factor 2^e, |e| <= 126.
__device__ __forceinline__ float exp2_int(int e) { return __uint_as_float((unsigned)(127 + e) << 23); }
// Exponent that brings a magnitude of these bits into [2^13, 2^14): 0 for zero.
__device__ __forceinline__ int gemm_exp(unsigned bits) {
    return bits == 0 ? 0 : max(-126, min(126, 140 - (int)(bits >> 23)));
}

// Scale and min of the 8 weights of lane (m, kq) in group gi of its chunk, from the chunk's table
// (1 and 0 for the formats without one).
template <class F>
__device__ __forceinline__ float2 weight_scale(const float* tab, int gi, int m, int kq) {
    const float* tr = tab + m * F::TAB;
    if constexpr (F::TAB == 0) return make_float2(1.0f, 0.0f);
    else if constexpr (F::MIN && F::HALVES) return reinterpret_cast<const float2*>(tr)[2 * gi + (kq >> 1)];
    else if constexpr (F::MIN) return reinterpret_cast<const float2*>(tr)[gi];
    else if constexpr (F::HALVES) return make_float2(tr[2 * gi + (kq >> 1)], 0.0f);
    else return make_float2(tr[gi], 0.0f);
}
// Those weights in fp32: scale * integer - min, rounded once (the range kernel's).
template <class F>
__device__ __forceinline__ void weight8(const typename F::Raw& raw, float2 sc, int gi, int kq, float (&v)[8]) {
    if constexpr (std::is_same<F, PF32>::value || std::is_same<F, PBF16>::value) {   // as they are
        const unsigned* u = reinterpret_cast<const unsigned*>(raw.w) + (std::is_same<F, PF32>::value ? 8 : 4) * gi;
#pragma unroll
        for (int e = 0; e < 8; ++e)
            v[e] = std::is_same<F, PF32>::value ? __uint_as_float(u[e])
                                                : bf2f((unsigned short)(u[e >> 1] >> (16 * (e & 1))));
        return;
    }
    uint4 a[F::NA];
    F::afrag(raw, gi, a, kq);
    uint4 u = a[0];
    if constexpr (F::HALVES) u = make_uint4(a[0].x | a[1].x, a[0].y | a[1].y, a[0].z | a[1].z, a[0].w | a[1].w);
    const f16x8_t h = as_f8(u);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = (float)h[e];
    if constexpr (F::TAB > 0) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = F::MIN ? __builtin_fmaf(v[e], sc.x, -sc.y) : v[e] * sc.x;
    }
}

template <class F, int NTHR>
__device__ __forceinline__ void stage_codebook(int tid) {
    constexpr int GRID = gk::FmtGrid<F>::BYTES;
    if constexpr (GRID > 0) {
        const uint4* src = static_cast<const uint4*>(gk::FmtGrid<F>::src());
        for (int i = tid; i < GRID / 16; i += NTHR) codebook_lds<GRID>()[i] = src[i];
        __syncthreads();
    }
}
template <class F>
__device__ __forceinline__ void chunk_table(const typename F::Raw& raw, float* tab, int m, int kq, int ch) {
    if constexpr (F::TAB > 0) {
        __builtin_amdgcn_wave_barrier();
        F::table(raw, tab, m, kq, ch);
        __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the table is written
        __builtin_amdgcn_wave_barrier();
    }
}

// E_row of rows 16 blockIdx.x .. +15 of a matrix (once per weight, at its upload).
template <class F>
__global__ __launch_bounds__(kThreads) void weight_range_kernel(WPlanes w, int cols, int* rexp) {
    __shared__ float s_tab[kWaves][16 * (F::TAB > 0 ? F::TAB : 1)];
    __shared__ unsigned s_max[kWaves][64];
    const int tid = threadIdx.x, lane = tid & 63, m = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), row = (int)blockIdx.x * 16 + m;
    stage_codebook<F, kThreads>(tid);
    unsigned mb = 0;
    for (int ch = wave; ch < (cols + kChunk - 1) / kChunk; ch += kWaves) {
        const int ng = min(kGroups, (cols >> 5) - ch * kGroups);
        typename F::Raw raw;
        F::load(raw, w, row, ch, kq, ng);
        chunk_table<F>(raw, s_tab[wave], m, kq, ch);
        for (int gi = 0; gi < kGroups; ++gi) {
            if (gi >= ng) break;
            float v[8];
            weight8<F>(raw, weight_scale<F>(s_tab[wave], gi, m, kq), gi, kq, v);
#pragma unroll
            for (int e = 0; e < 8; ++e) mb = max(mb, dk::abs_bits(v[e]));
        }
    }
    s_max[wave][lane] = mb;
    __syncthreads();
    if (tid < 16) {
        unsigned x = 0;
        for (int i = 0; i < kWaves * 4; ++i) x = max(x, s_max[i >> 2][16 * (i & 3) + tid]);
        rexp[blockIdx.x * 16 + tid] = gemm_exp(x);
    }
}

// Per token: sc[2t] = the RMSNorm factor r (tok_prep_kernel's), sc[2t + 1] = the exponent that
// brings its largest |x*w| (or |x|) into [2^13, 2^14).
template <int NTHR>
__global__ __launch_bounds__(NTHR) void tok_scale_kernel(const float* x, long long x_pitch, int cols, const float* w,
                                                         float eps, float* sc) {
    float r;
    unsigned m;
    tok_reduce<NTHR>(x + (long long)blockIdx.x * x_pitch, cols, w, eps, r, m);
    if (threadIdx.x == 0) {
        sc[2 * blockIdx.x] = r;
        sc[2 * blockIdx.x + 1] = (float)gemm_exp(m);
    }
}

// The inputs x*w * 2^e as hi/lo fragments, and their sums per 16 columns: blockIdx.x = 32-token
// tile, y = 256-column block.  Tokens past K and columns past cols are zeros.
template <int NTHR>
__global__ __launch_bounds__(NTHR) void tok_split_kernel(const float* x, long long x_pitch, int cols, const float* w,
                                                        const float* sc, int K, int steps, uint4* xs, float* xsum) {
#pragma unroll
    for (int i = 0; i < 1024 / NTHR; ++i) {
        const int p = threadIdx.x + NTHR * i, ks = 16 * (int)blockIdx.y + (p >> 6), lane = p & 63;
        if (ks >= steps) return;
        const int t = 32 * (int)blockIdx.x + (lane & 31), c = 16 * ks + 8 * (lane >> 5);
        float v[8] = {};
        if (t < K && c < cols) {
            const float4* xp = reinterpret_cast<const float4*>(x + (long long)t * x_pitch + c);
            const float4 a = xp[0], b = xp[1];
            const float xv[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
            float wv[8] = {1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f};
            if (w != nullptr) {
                const float4 w0 = reinterpret_cast<const float4*>(w + c)[0], w1 = reinterpret_cast<const float4*>(w + c)[1];
                wv[0] = w0.x; wv[1] = w0.y; wv[2] = w0.z; wv[3] = w0.w;
                wv[4] = w1.x; wv[5] = w1.y; wv[6] = w1.z; wv[7] = w1.w;
            }
            // (x*w) * 2^e; a factor below 1 goes to x, whose product with w may exceed fp32's range.
            const float f = exp2_int((int)sc[2 * t + 1]), fx = fminf(f, 1.0f), fv = fmaxf(f, 1.0f);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = ((xv[e] * fx) * wv[e]) * fv;
        }
        uint4 h, l;
        split8(v, h, l);
        const size_t step = (size_t)blockIdx.x * steps + ks;
        uint4* o = xs + step * 128 + lane;
        o[0] = h;
        o[64] = l;
        const float sum = dk::lane_step<32, false>(((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7])));
        if (lane < 32) xsum[step * 32 + lane] = sum;
    }
}

// A format with a scale s and a min m per block of 32 columns, w = s q - m, as the product takes it:
// w = s (q - z) - (m - s z), z the code nearest to zero weight.  q - z is exact in fp16 and both terms
// are as small as the weights, so nothing cancels.  Table per row: the chunk's 4 scales, 4 mins
// m - s z, and 4 zero points (zero_point_f16).
__device__ __forceinline__ float zero_code(float s, float m, float most) {
    const float z = __builtin_rintf(m * __builtin_amdgcn_rcpf(s));   // a code either way: any z is exact
    return s != 0.0f ? fminf(fmaxf(z, 0.0f), most) : 0.0f;
}
template <class P, int MOST>
struct Zeroed : P {
    static constexpr int TAB = 12, MINS = 4, ZEROS = 8;
    static __device__ __forceinline__ void table(const typename P::Raw& r, float* tab, int m, int kq, int ch) {
        const float2 e = P::entry(r, kq, ch);
        const float z = zero_code(e.x, e.y, (float)MOST);
        float* t = tab + m * TAB + kq;
        t[0] = e.x;
        t[MINS] = __builtin_fmaf(-z, e.x, e.y);
        t[ZEROS] = __uint_as_float(zero_point_f16(z));
    }
    static __device__ __forceinline__ uint4 integers(const typename P::Raw& r, unsigned zero, int gi, int kq) {
        unsigned c0, c1;
        P::codes(r, gi, kq, c0, c1);
        return f16x8_less(c0, c1, zero);
    }
    static __device__ __forceinline__ int zero_at(int gi, int) { return ZEROS + gi; }
};
using GQ4K = Zeroed<PQ4K, 15>;
using GQ5K = Zeroed<PQ5K, 31>;
using GQ5_1 = Zeroed<PQ5_1, 31>;
// Q2_K: the 4-bit sub-block scale times q - z is exact too (at most 45), so a group has one scale, d,
// and half the scaling of its 16-column sub-blocks.  Table per row: 8 mins, 8 zero points, d.
struct GQ2_K : PQ2_K {
    static constexpr int NA = 1, TAB = 20, MINS = 0, ZEROS = 8, SCALE = 16;
    static constexpr bool HALVES = false;
    static __device__ __forceinline__ void table(const Raw& r, float* tab, int m, int kq, int) {
        const unsigned wv = kq < 2 ? r.sc.x : r.sc.y;
        const float d = h2f(r.d), dm = h2f(r.dm);
        float* t = tab + m * TAB;
#pragma unroll
        for (int i = 0; i < 2; ++i) {   // sub-blocks 2 kq and 2 kq + 1 of the chunk
            const unsigned b = (wv >> (16 * (kq & 1) + 8 * i)) & 0xFFu;
            const float s = d * (float)(b & 15u), mn = dm * (float)(b >> 4), z = zero_code(s, mn, 3.0f);
            t[MINS + 2 * kq + i] = __builtin_fmaf(-z, s, mn);
            t[ZEROS + 2 * kq + i] = __uint_as_float(zero_point_f16(z));
        }
        if (kq == 0) t[SCALE] = d;
    }
    static __device__ __forceinline__ uint4 integers(const Raw& r, unsigned zero, int gi, int kq) {
        unsigned c0, c1;
        codes(r, gi, kq, c0, c1);
        const _Float16 sc = (_Float16)(float)(((gi < 2 ? r.sc.x : r.sc.y) >> (16 * (gi & 1) + 8 * (kq >> 1))) & 15u);
        return __builtin_bit_cast(uint4, as_f8(f16x8_less(c0, c1, zero)) * sc);
    }
    static __device__ __forceinline__ int zero_at(int gi, int kq) { return ZEROS + 2 * gi + (kq >> 1); }
};

// The formats with a scale table: their weights stay the exact integers.
template <class F>
constexpr bool integer_weights() { return F::TAB > 0; }
// Whether their mins are per 16 columns, not per 32.
template <class F>
constexpr bool half_mins() { return std::is_same<F, GQ2_K>::value; }
// The zero point of the 8 weights of lane (m, kq) in group gi, from its wave's table (formats with a min).
template <class F>
__device__ __forceinline__ unsigned group_zero(const float* tab, int gi, int m, int kq) {
    if constexpr (F::MIN) return __float_as_uint(tab[m * F::TAB + F::zero_at(gi, kq)]);
    else return 0u;
}
// Group gi of a chunk as fragments: the integers, or hi/lo parts scaled by the row's power of two fw.
template <class F>
__device__ __forceinline__ void decode_group(const typename F::Raw& raw, unsigned zero, int gi, int kq, float fw, uint4& h,
                                             uint4& l) {
    // groups past cols repeat the row's last (zero inputs)
    if constexpr (F::MIN) {
        h = F::integers(raw, zero, gi, kq);
    } else if constexpr (integer_weights<F>()) {
        uint4 a[F::NA];
        F::afrag(raw, gi, a, kq);
        h = a[0];
        if constexpr (F::HALVES) h = make_uint4(a[0].x | a[1].x, a[0].y | a[1].y, a[0].z | a[1].z, a[0].w | a[1].w);
    } else {
        float v[8];
        weight8<F>(raw, make_float2(1.0f, 0.0f), gi, kq, v);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = v[e] * fw;
        split8(v, h, l);
    }
}
// Its place in the stage buffer: lane (m, kq) of wave wv holds row 16 wv + m, columns 8 kq .. +7,
// i.e. row 16 (wv%2) + m of 32-row tile wv/2, half kq%2 of step kq/2.
template <bool WLO>
__device__ __forceinline__ void weight_put(const uint4& h, const uint4& l, uint4* __restrict__ dst, int wv, int m, int kq) {
    uint4* o = dst + (((wv >> 1) * kGemmStage + (kq >> 1)) * 2) * 64 + 32 * (kq & 1) + 16 * (wv & 1) + m;
    o[0] = h;
    if constexpr (WLO) o[64] = l;
}

// A wave's operands of one stage: its 32 tokens x 64 rows.
struct StageFrags {
    f16x8_t x[kGemmStage][2], w[2][kGemmStage][2];
};
template <bool WLO>
__device__ __forceinline__ void stage_read(StageFrags& f, const uint4* wst, const uint4* xst, int tt, int lane) {
#pragma unroll
    for (int s = 0; s < kGemmStage; ++s) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            f.x[s][p] = as_f8(xst[((tt * kGemmStage + s) * 2 + p) * 64 + lane]);
#pragma unroll
            for (int j = 0; j < 2; ++j)
                if (WLO || p == 0) f.w[j][s][p] = as_f8(wst[((j * kGemmStage + s) * 2 + p) * 64 + lane]);
        }
    }
}
template <bool WLO>
__device__ __forceinline__ void stage_products(const StageFrags& f, f32x16_t (&acc)[2]) {
#pragma unroll
    for (int s = 0; s < kGemmStage; ++s) {
        if constexpr (WLO)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.x[s][0], f.w[j][s][1], acc[j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.x[s][1], f.w[j][s][0], acc[j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.x[s][0], f.w[j][s][0], acc[j], 0, 0, 0);
    }
}

// The scales of a group of integer weights for this lane's two rows (row lane%32 of tile j), per 32
// or per 16 columns, times the row's power of two.
template <class F>
struct GroupScales {
    static_assert(!(F::HALVES && F::MIN), "one scale and min, or two scales, to a block");
    float s[2][F::HALVES ? 2 : 1];
};
template <class F>
__device__ __forceinline__ void group_scales(GroupScales<F>& g, const float* const (&tab)[2], int gi, const float (&fw)[2]) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        if constexpr (half_mins<F>()) {
            g.s[j][0] = tab[j][F::SCALE] * fw[j];
        } else if constexpr (F::HALVES) {
            const float2 t = reinterpret_cast<const float2*>(tab[j])[gi];
            g.s[j][0] = t.x * fw[j];
            g.s[j][1] = t.y * fw[j];
        } else {
            g.s[j][0] = tab[j][gi] * fw[j];
        }
        // an all-zero block may have any exponent: its zero sum must not meet an infinite scale
        if constexpr (std::is_same<F, PMXFP4>::value) g.s[j][0] = fminf(g.s[j][0], 3e38f);
    }
}
// The groups' sum so far into the row's; what rounding drops stays for the next (a compensated sum
// that needs no register of its own).
__device__ __forceinline__ void fold_sums(f32x16_t& sum, f32x16_t& acc) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const float s = sum[i] + acc[i];
        acc[i] = acc[i] - (s - sum[i]);
        sum[i] = s;
    }
}
// A group's exact products, summed from zero and scaled once, as the 16-token kernel does it.  The
// products of the hi parts come first: on top of a small sum (the lo parts') the matrix unit drops
// its low bits downwards, which left outputs 9e-8 of their root mean square too low.
template <class F>
__device__ __forceinline__ void group_products(const StageFrags& f, const GroupScales<F>& g, f32x16_t (&acc)[2]) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        auto add = [&](const f32x16_t& t, float s) {
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[j][i] = __builtin_fmaf(t[i], s, acc[j][i]);
        };
        f32x16_t t = {};
        if constexpr (F::HALVES) {
#pragma unroll
            for (int s = 0; s < kGemmStage; ++s) {
                t = f32x16_t{};
                t = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.x[s][0], f.w[j][s][0], t, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.x[s][1], f.w[j][s][0], t, 0, 0, 0);
                add(t, g.s[j][F::HALVES ? s : 0]);
            }
        } else {
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int s = 0; s < kGemmStage; ++s)
                    t = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.x[s][p], f.w[j][s][0], t, 0, 0, 0);
            add(t, g.s[j][0]);
        }
    }
}
// The min terms of a chunk, -(m - s z) sum(x) over its blocks of 32 or 16 columns, in fp32 on
// v_mfma_f32_32x32x2_f32 (lane l: token or row l%32 of block 2p + l/32): input sums, and their product.
template <class F>
constexpr int min_pairs() { return !F::MIN ? 1 : half_mins<F>() ? 4 : 2; }
template <class F>
struct MinSums {   // as loaded: adding them here would wait for every load before them
    float s[min_pairs<F>()][half_mins<F>() ? 1 : 2];
};
template <class F>
__device__ __forceinline__ void min_sums(MinSums<F>& x, const float* xsum, int ch, int lane) {
    constexpr int N = half_mins<F>() ? 1 : 2;
    const float* p = xsum + ch * (kChunk / 16) * 32 + (lane & 31);   // of the wave's token tile
#pragma unroll
    for (int i = 0; i < min_pairs<F>(); ++i)
#pragma unroll
        for (int k = 0; k < N; ++k) x.s[i][k] = p[(N * (2 * i + (lane >> 5)) + k) * 32];
}
// Stage g of a chunk takes a quarter of them (each product has the matrix unit for 64 cycles, which
// one after the other nothing covered): pair g / 2 of row tile g % 2, or pair g of both.
template <class F>
struct MinFactors {
    float c[half_mins<F>() ? 2 : 1];
};
template <class F>
__device__ __forceinline__ void min_factors(MinFactors<F>& m, const float* const (&tab)[2], const float (&fw)[2], int g,
                                            int lane) {
#pragma unroll
    for (int k = 0; k < (half_mins<F>() ? 2 : 1); ++k) {
        const int i = half_mins<F>() ? g : g >> 1, j = half_mins<F>() ? k : g & 1;
        m.c[k] = -tab[j][F::MINS + 2 * i + (lane >> 5)] * fw[j];
    }
}
template <class F>
__device__ __forceinline__ void min_products(const MinSums<F>& x, const MinFactors<F>& m, int g, f32x16_t (&acc)[2]) {
    if constexpr (half_mins<F>()) {
        acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(x.s[g][0], m.c[0], acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(x.s[g][0], m.c[1], acc[1], 0, 0, 0);
    } else {
        acc[g & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(x.s[g >> 1][0] + x.s[g >> 1][1], m.c[0], acc[g & 1], 0, 0, 0);
    }
}

// One stage of the workgroup's four token tiles, each wave its own tile: global memory to
// registers, registers to LDS.  (Copies straight into LDS would save the registers, but the wait
// counts then drain them at the next LDS access of the stage.)
constexpr int kGemmCopy = kGemmXFrags / kGemmWaves;
__device__ __forceinline__ void gemm_fetch(u32x4 (&r)[kGemmCopy], const uint4* xs, int steps, int stage, int wave,
                                           int lane) {
    const uint4* p = xs + ((size_t)wave * steps + kGemmStage * stage) * 128 + lane;
#pragma unroll
    for (int i = 0; i < kGemmCopy; ++i) r[i] = *reinterpret_cast<const u32x4*>(p + 64 * i);
}
__device__ __forceinline__ void gemm_put(const u32x4 (&r)[kGemmCopy], uint4* __restrict__ dst, int wave, int lane) {
#pragma unroll
    for (int i = 0; i < kGemmCopy; ++i) *reinterpret_cast<u32x4*>(dst + (wave * kGemmCopy + i) * 64 + lane) = r[i];
}

// Barrier of the workgroup that waits for its own LDS accesses only.
__device__ __forceinline__ void stage_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// `tabs`: the waves' tables, two chunks of tab_pitch floats each.
template <class F>
__device__ __forceinline__ void gemm_rows(const ProjGemmArgs& a, const GemmSeg& sg, int row0, const uint4* xs,
                                          const float* xsum, uint4 (*wb)[kGemmWFrags * 64], uint4 (*xb)[kGemmXFrags * 64],
                                          float* tabs, int tab_pitch, f32x16_t (&sum)[2], int wave, int lane) {
    constexpr bool INT = integer_weights<F>(), WLO = std::is_same<F, PF32>::value;
    const int m = lane & 15, kq = lane >> 4;
    const int row = min(row0 + 16 * wave + m, sg.rows - 1);   // rows past the segment repeat its last
    const float fw = exp2_int(sg.rexp[row]);                  // of the row this lane decodes,
    const float fr[2] = {exp2_int(sg.rexp[min(row0 + (lane & 31), sg.rows - 1)]),        // and of the rows whose
                         exp2_int(sg.rexp[min(row0 + 32 + (lane & 31), sg.rows - 1)])};  // products it holds
    const int ngroups = a.cols >> 5, nch = (ngroups + kGroups - 1) / kGroups, last = kGroups * nch - 1;
    auto groups = [&](int ch) { return min(kGroups, ngroups - ch * kGroups); };
    auto chunk = [&](int ch) { return min(ch, nch - 1); };     // past the end: the last again, unused
    float* const tab = tabs + wave * 2 * tab_pitch;
    const float* const row_tab[2] = {tabs + ((lane >> 4) & 1) * 2 * tab_pitch + m * F::TAB,
                                     tabs + (2 + ((lane >> 4) & 1)) * 2 * tab_pitch + m * F::TAB};
    // The inputs of stages s + 1 and s + 2 are in registers or on their way at stage s.
    u32x4 x[2][kGemmCopy];
    typename F::Raw r0, r1;   // the chunk being decoded, and the next one's, requested two stages before its table
    MinSums<F> sx, s1;        // of the same two chunks
    F::load(r0, sg.w, row, 0, kq, groups(0));
    gemm_fetch(x[0], xs, a.steps, 0, wave, lane);
    gemm_fetch(x[1], xs, a.steps, 1, wave, lane);
    if constexpr (F::MIN) min_sums<F>(sx, xsum, 0, lane);
    stage_codebook<F, kGemmThreads>(wave * 64 + lane);
    chunk_table<F>(r0, tab, m, kq, 0);
    uint4 h, l;
    decode_group<F>(r0, group_zero<F>(tab, 0, m, kq), 0, kq, fw, h, l);
    weight_put<WLO>(h, l, wb[0], wave, m, kq);
    gemm_put(x[0], xb[0], wave, lane);
    gemm_fetch(x[0], xs, a.steps, 2, wave, lane);
    f32x16_t acc[2] = {};
    for (int ch = 0; ch < nch; ++ch) {
        const int c1 = chunk(ch + 1);
        const int even = (ch & 1) * tab_pitch, odd = ((ch + 1) & 1) * tab_pitch;
        const float* const t0[2] = {row_tab[0] + even, row_tab[1] + even};
#pragma unroll
        for (int g = 0; g < kGroups; ++g) {
            // This stage's fragments are complete in every wave behind the barrier, and nobody reads
            // the other buffers any more.  (Its wait covers the LDS alone: the loads stay in flight.)
            stage_barrier();
            // A stage in three parts that the scheduler keeps apart: every read it needs; products
            // and the next group's decoding, dealt out between each other; the writes.  In the
            // compiler's order each product waited for its own operands (96 tokens: 194 us the
            // call, 178 so).
            StageFrags f;
            stage_read<WLO>(f, wb[g & 1], xb[g & 1], wave, lane);
            const int gn = (g + 1) % kGroups;
            if (g == 0) {
                F::load(r1, sg.w, row, c1, kq, groups(c1));
                if constexpr (F::MIN) min_sums<F>(s1, xsum, c1, lane);
            }
            if constexpr (INT) {
                GroupScales<F> gs;
                group_scales<F>(gs, t0, g, fr);
                const unsigned zero = group_zero<F>(tab + (gn == 0 ? odd : even), gn, m, kq);
                MinFactors<F> mc;
                if constexpr (F::MIN) min_factors<F>(mc, t0, fr, g, lane);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (F::MIN) min_products<F>(sx, mc, g, acc);
                // under the products of the other tile (at the end of the chunk, under nothing, it took
                // 200 tokens of the 24/8/128 shape in Q8_0 from 165 to 173 us)
                if (g == 1) fold_sums(sum[1], acc[1]);
                if (g == 2) fold_sums(sum[0], acc[0]);
                decode_group<F>(gn == 0 ? r1 : r0, zero, gn, kq, fw, h, l);
                group_products<F>(f, gs, acc);
#pragma unroll
                for (int i = 0; i < 4 * kGemmStage; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // a product
                    // decoding, scaling (with a min 4: 200 tokens in Q4_K 178.8 us, 182.4 with 8; without, 165
                    // against 166.9 in Q8_0)
                    __builtin_amdgcn_sched_group_barrier(0x002, F::MIN ? 4 : 8, 0);
                }
            } else {
                __builtin_amdgcn_sched_barrier(0);
                decode_group<F>(gn == 0 ? r1 : r0, 0u, gn, kq, fw, h, l);
                stage_products<WLO>(f, acc);
#pragma unroll
                for (int i = 0; i < 2 * kGemmStage * (WLO ? 3 : 2); ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // a product
                    __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);   // decoding
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            gemm_put(x[(g + 1) & 1], xb[(g + 1) & 1], wave, lane);
            gemm_fetch(x[(g + 1) & 1], xs, a.steps, min(kGroups * ch + g + 3, last), wave, lane);
            weight_put<WLO>(h, l, wb[(g + 1) & 1], wave, m, kq);
            if (g == 2 && F::TAB > 0) F::table(r1, tab + odd, m, kq, c1);
        }
        r0 = r1;
        if constexpr (F::MIN) sx = s1;
        if constexpr (!INT) {
            sum[0] += acc[0];
            sum[1] += acc[1];
            acc[0] = acc[1] = f32x16_t{};
        }
    }
    if constexpr (INT) {
        sum[0] += acc[0];
        sum[1] += acc[1];
    }
}

template <class F1, class F2>
__global__ __launch_bounds__(kGemmThreads) __attribute__((amdgpu_waves_per_eu(2)))
void proj_gemm_kernel(ProjGemmArgs a) {
    __shared__ uint4 s_w[2][kGemmWFrags * 64], s_x[2][kGemmXFrags * 64];
    constexpr int TP = 16 * tab_floats<F1, F2>();
    __shared__ float s_tab[kGemmWaves][2 * TP];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tiles = a.row_tiles * a.tok_tiles, per = (tiles + 7) / 8;
    const int tile = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || tile >= tiles) return;
    const int tok = tile / a.row_tiles, rt = tile - tok * a.row_tiles;
    const int si = a.nseg > 2 && rt >= a.seg[2].tile0 ? 2 : a.nseg > 1 && rt >= a.seg[1].tile0 ? 1 : 0;
    const GemmSeg& sg = a.seg[si];
    const int row0 = (rt - sg.tile0) * kGemmRows;
    const uint4* xs = a.xs + (size_t)tok * 4 * a.steps * 128;
    const float* xsum = a.xsum + ((size_t)tok * 4 + wave) * a.steps * 32;
    f32x16_t sum[2] = {};
    if (std::is_same<F1, F2>::value || sg.fmt == 0)
        gemm_rows<F1>(a, sg, row0, xs, xsum, s_w, s_x, &s_tab[0][0], TP, sum, wave, lane);
    else
        gemm_rows<F2>(a, sg, row0, xs, xsum, s_w, s_x, &s_tab[0][0], TP, sum, wave, lane);
    // D: lane = row l%32 of the tile, element i = token 8 (i/4) + 4 (l/32) + i%4.
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int row = row0 + 32 * j + (lane & 31);
        if (row >= sg.rows) continue;
        const int ew = sg.rexp[row];
        const float bias = sg.bias != nullptr ? sg.bias[row] : 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int t = kGemmToks * tok + 32 * wave + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
            if (t >= a.K) continue;
            const float2 f = reinterpret_cast<const float2*>(a.tok_sc)[t];
            float v = __builtin_amdgcn_ldexpf(sum[j][i], -(ew + (int)f.y)) * f.x;
            if (sg.bias != nullptr) v = v + bias;
            if (a.resid != nullptr) {
                if (a.rscale > 0.0f) v = v * a.rscale;
                float* x = a.resid + (long long)t * a.resid_pitch + row;
                *x = *x + v;
            } else {
                sg.out[(long long)t * sg.out_pitch + row] = v;
            }
        }
    }
}

}  // namespace tk
}  // namespace llmp
