// Projections of many tokens (a prompt through llmp_attn_block_batch): Y[t][r] = sum_c W[r][c]
// x_t[c] as a tiled matrix product on v_mfma_f32_32x32x16_f16, from the weights' own GGUF planes.
//
// The 16-token kernel (proj_tok_kernels.h) decodes every weight and splits every input again for
// each group of 16 tokens; 63 groups of 1000 tokens took 63 x (22 + 12) us at the 24/8/128 shape with
// Q4_K_M weights.  Here a workgroup of 4 waves owns 64 rows x 128 tokens: the weights of a 32-column
// group are decoded once per 128 tokens, by the waves themselves, into LDS as fp16 hi/lo operand
// fragments; the inputs were split once per call (tok_split_kernel) and stream through registers.
// Both are double buffered with one barrier per group, and two workgroups share a CU.
//
// Bound: neither the matrix units (about a third busy) nor memory, but the stage itself: operand
// reads, products beside the next group's decoding, fragment writes, barrier.  Measured at that shape,
// 1000 tokens: Q/K/V 170 us, Wo 113 us (48 GFLOP of products there, 97 for Q/K/V), against 1370 and
// 750 us in groups.  A 128 x 128 tile of 8 waves took 196 and 109 us at 1000 tokens, and 226 against
// 178 us for the whole call at 96 tokens, where a stage's latency is all there is.
//
// Precision.  A weight is w * 2^E_row = hi + lo with E_row from the row's largest magnitude
// (weight_range_kernel, at upload), so hi + lo holds it to 2^-22 down to 2^-17 of the row's
// largest; an input likewise with its token's exponent.  Products are hi*hi + hi*lo + lo*hi; each
// 128-column chunk is summed by the matrix unit from zero and added to the running sum in fp32,
// which keeps that chain as short as the 16-token kernel's.  F16 and BF16 rows have no lo part.
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
// Those weights in fp32: scale * integer - min, rounded once.
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

// The inputs x*w * 2^e as hi/lo fragments: blockIdx.x = 32-token tile, y = 256-column block.
// Tokens past K and columns past cols are zeros.
template <int NTHR>
__global__ __launch_bounds__(NTHR) void tok_split_kernel(const float* x, long long x_pitch, int cols, const float* w,
                                                        const float* sc, int K, int steps, uint4* xs) {
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
            const float f = exp2_int((int)sc[2 * t + 1]);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = (xv[e] * wv[e]) * f;
        }
        uint4 h, l;
        split8(v, h, l);
        uint4* o = xs + (((size_t)blockIdx.x * steps + ks) * 2) * 64 + lane;
        o[0] = h;
        o[64] = l;
    }
}

// Group gi of a chunk as hi/lo fragments, scaled by the row's power of two fw.
template <class F>
__device__ __forceinline__ void decode_group(const typename F::Raw& raw, float2 sc, int gi, int kq, float fw, uint4& h,
                                             uint4& l) {
    float v[8];
    weight8<F>(raw, sc, gi, kq, v);   // groups past cols repeat the row's last (zero inputs)
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = v[e] * fw;
    split8(v, h, l);
}
// Its place in the stage buffer: lane (m, kq) of wave wv holds row 16 wv + m, columns 8 kq .. +7,
// i.e. row 16 (wv%2) + m of 32-row tile wv/2, half kq%2 of step kq/2.
__device__ __forceinline__ void weight_put(const uint4& h, const uint4& l, uint4* __restrict__ dst, int wv, int m, int kq) {
    uint4* o = dst + (((wv >> 1) * kGemmStage + (kq >> 1)) * 2) * 64 + 32 * (kq & 1) + 16 * (wv & 1) + m;
    o[0] = h;
    o[64] = l;
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

template <class F>
__device__ __forceinline__ void gemm_rows(const ProjGemmArgs& a, const GemmSeg& sg, int row0, const uint4* xs,
                                          uint4 (*wb)[kGemmWFrags * 64], uint4 (*xb)[kGemmXFrags * 64], float* tab,
                                          int tab_pitch, f32x16_t (&sum)[2], int wave, int lane) {
    constexpr bool WLO = !(std::is_same<F, PF16>::value || std::is_same<F, PBF16>::value);
    const int m = lane & 15, kq = lane >> 4;
    const int row = min(row0 + 16 * wave + m, sg.rows - 1);   // rows past the segment repeat its last
    const float fw = exp2_int(sg.rexp[row]);
    const int ngroups = a.cols >> 5, nch = (ngroups + kGroups - 1) / kGroups, last = kGroups * nch - 1;
    auto groups = [&](int ch) { return min(kGroups, ngroups - ch * kGroups); };
    auto chunk = [&](int ch) { return min(ch, nch - 1); };     // past the end: the last again, unused
    // The inputs of stages s + 1 and s + 2 are in registers or on their way at stage s.
    u32x4 x[2][kGemmCopy];
    typename F::Raw r0, r1, r2;
    F::load(r0, sg.w, row, 0, kq, groups(0));
    F::load(r1, sg.w, row, chunk(1), kq, groups(chunk(1)));
    gemm_fetch(x[0], xs, a.steps, 0, wave, lane);
    gemm_fetch(x[1], xs, a.steps, 1, wave, lane);
    stage_codebook<F, kGemmThreads>(wave * 64 + lane);
    chunk_table<F>(r0, tab, m, kq, 0);
    uint4 h, l;
    decode_group<F>(r0, weight_scale<F>(tab, 0, m, kq), 0, kq, fw, h, l);
    weight_put(h, l, wb[0], wave, m, kq);
    gemm_put(x[0], xb[0], wave, lane);
    gemm_fetch(x[0], xs, a.steps, 2, wave, lane);
    for (int ch = 0; ch < nch; ++ch) {
        const int c1 = chunk(ch + 1), c2 = chunk(ch + 2);
        float* t0 = tab + (ch & 1) * tab_pitch;
        float* t1 = tab + ((ch + 1) & 1) * tab_pitch;
        f32x16_t acc[2] = {};
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
            const float2 sc = weight_scale<F>(gn == 0 ? t1 : t0, gn, m, kq);
            if (g == 3) F::load(r2, sg.w, row, c2, kq, groups(c2));
            __builtin_amdgcn_sched_barrier(0);
            decode_group<F>(gn == 0 ? r1 : r0, sc, gn, kq, fw, h, l);
            stage_products<WLO>(f, acc);
#pragma unroll
            for (int i = 0; i < 2 * kGemmStage * (WLO ? 3 : 2); ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // a product
                __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);   // decoding
            }
            __builtin_amdgcn_sched_barrier(0);
            gemm_put(x[(g + 1) & 1], xb[(g + 1) & 1], wave, lane);
            gemm_fetch(x[(g + 1) & 1], xs, a.steps, min(kGroups * ch + g + 3, last), wave, lane);
            weight_put(h, l, wb[(g + 1) & 1], wave, m, kq);
            if (g == 2 && F::TAB > 0) F::table(r1, t1, m, kq, c1);   // r1 was requested three stages ago
        }
        r0 = r1;
        r1 = r2;
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
    f32x16_t sum[2] = {};
    if (std::is_same<F1, F2>::value || sg.fmt == 0)
        gemm_rows<F1>(a, sg, row0, xs, s_w, s_x, s_tab[wave], TP, sum, wave, lane);
    else
        gemm_rows<F2>(a, sg, row0, xs, s_w, s_x, s_tab[wave], TP, sum, wave, lane);
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
