// Multi-token attention on 32x32 matrix tiles: the path of calls whose key tiles are each read
// by several workgroups (prefill_wide_splits); shorter chunks stay on prefill_kernels.h.
//
// One KV head's queries are flattened to columns c = token * G + head (G query heads per KV
// head), so a workgroup of 4 waves takes 128 consecutive columns whatever G is and no MFMA
// column is padding except in the last block.  A wave owns 32 columns: per key tile it forms
// S^T = K Q^T and O^T += V^T P^T with v_mfma_f32_32x32x16_f16, three products per term on fp16
// hi/lo parts as in prefill_kernels.h (hi*hi + hi*lo + lo*hi, ~2^-21 per term).
//
// Bound: matrix work and the softmax's vector work, with the LDS behind them.  A 32-column wave
// reads every operand of a tile once per 32 columns, half the LDS bytes per product of the 16x16
// form, which had the LDS two thirds busy at the matrix peak.  Key tiles are written once per
// call as images in operand order (each operand fragment one 1 KB run, lane l at 16 l): a tile
// goes from L2 to LDS by global_load_lds, 16 bytes per lane, through no register, and every
// operand read is a lane-linear ds_read_b128 (no bank conflicts).  Tiles of 32 KB (64 keys at
// head_dim 64, 32 keys at 128; 24 KB for 32 keys at 96) in two buffers leave two workgroups per CU, so one
// workgroup's softmax runs under the other's products.
//
// Measured (MI355X, attention kernel by rocprof, 16x16 kernel before): 24/8/128, 8192 fp32 tokens
// 1662 -> 1172 us (1.05 PFLOP/s of products issued; a library fp16 GEMM of 8192^3 reaches 1.20 on
// the same card, where the clock falls to about 1.6 GHz under either); 32/8/64, 2048 bf16 tokens
// 66.6 -> 59.1 us; 16/8/128, 777 tokens after 1501 rows 118 -> 63.7 us.  Steering the schedule
// (operand reads three products ahead, independent accumulators in turn, wave priorities)
// measured no faster at any of the three.
//
// Layout facts of v_mfma_f32_32x32x16_f16: lane l holds A[l%32][8*(l/32)+j] and
// B[8*(l/32)+j][l%32] (j < 8) and D[8*(i/4) + 4*(l/32) + i%4][l%32] (i < 16).  S^T's D fragment
// (lane: column l%32, keys 8*(i/4) + 4*(l/32) + i%4) is the B operand of the P V product as it
// is: step s of a 32-key tile takes i = 8s .. 8s+7, i.e. keys 16s + 8*(j/4) + 4*(l/32) + j%4,
// and the V^T fragments hold their keys in that order.
#pragma once

#include "prefill_kernels.h"

namespace llmp {
namespace pk {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kWideWaves = 4;
constexpr int kWideThreads = kWideWaves * 64;
constexpr int kWideCols = kWideWaves * 32;   // columns (token, head) per workgroup

// Tile image of TK keys: K fragments (key tile kt, 16-dim step s, part hi/lo), V^T hi fragments
// (16-key step v, 32-dim tile d), then the V^T lo fragments, each 64 uint4.
template <int D>
struct WideTile {
    static constexpr int TK = D <= 64 ? 64 : 32;
    static constexpr int KT = TK / 32, KS = D / 16, VS = TK / 16, DT = D / 32;
    static constexpr int NKF = KT * KS * 2, NVF = VS * DT;
    static constexpr int FRAGS = NKF + 2 * NVF;
    static constexpr int U4 = FRAGS * 64;
    static_assert(FRAGS % kWideWaves == 0, "the waves copy a tile in equal parts");
    static constexpr __device__ __host__ int kfrag(int kt, int s, int part) { return (kt * KS + s) * 2 + part; }
    static constexpr __device__ __host__ int vfrag(int v, int d, int part) { return NKF + part * NVF + v * DT + d; }
};

// Images of tiles tile0 + blockIdx.x of KV head blockIdx.y (fp32 or dequantised Q8_0 rows, scaled
// by 2^-E of the head's range exponents), and the tile's flag: nonzero when some V lo part
// exceeds 2^-24 (prefill_tile_kernel).  Rows at or past row_end repeat row row_end - 1.  A
// thread builds whole 16-byte lane pieces: 8 consecutive dims of one K row, or 8 keys of one dim
// of V (32 lanes read 128 consecutive bytes of a row).
template <int D>
constexpr int wide_tile_threads() { return D == 96 ? 192 : 256; }

template <int D, bool Q8>
__global__ __launch_bounds__(wide_tile_threads<D>()) void prefill_wide_tile_kernel(PrefillArgs a, uint4* ws, unsigned* flags,
                                                                int tile0, int n_tiles, int row_end) {
    using T = WideTile<D>;
    constexpr int NT = wide_tile_threads<D>();
    const int tid = threadIdx.x, kvh = blockIdx.y;
    const size_t slot = (size_t)kvh * n_tiles + blockIdx.x;
    uint4* img = ws + slot * T::U4;
    const int r0 = (tile0 + (int)blockIdx.x) * T::TK;
    const HeadRows kr = k_rows<Q8>(a, kvh), vr = v_rows<Q8>(a, kvh);
    const float fk = pow2i(-a.range[2 * kvh]), fv = pow2i(-a.range[2 * kvh + 1]);
    constexpr int NK = T::KT * T::KS * 64, NV = T::NVF * 64;   // pieces (hi and lo together)
    constexpr int KI = NK / NT, VI = NV / NT;
    static_assert(KI * NT == NK && VI * NT == NV, "tile pieces divide over the threads");
    floatx4 kx[KI][2];
    float vx[VI][8];
#pragma unroll
    for (int i = 0; i < KI; ++i) {
        const int e = tid + i * NT, f = e >> 6, l = e & 63;   // f = kt * KS + s
        const int row = min(r0 + 32 * (f / T::KS) + (l & 31), row_end - 1);
        const int c4 = 4 * (f % T::KS) + 2 * (l >> 5);
        kx[i][0] = load_chunk<D, Q8>(kr, row, c4);
        kx[i][1] = load_chunk<D, Q8>(kr, row, c4 + 1);
    }
#pragma unroll
    for (int i = 0; i < VI; ++i) {
        const int e = tid + i * NT, f = e >> 6, l = e & 63;   // f = v * DT + d
        const int k0 = r0 + 16 * (f / T::DT) + 4 * (l >> 5), dim = 32 * (f % T::DT) + (l & 31);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int row = min(k0 + 8 * (j >> 2) + (j & 3), row_end - 1);
            if constexpr (Q8)
                vx[i][j] = (float)vr.q[(long long)row * D + dim] * vr.s[(long long)row * (D / 32) + (dim >> 5)];
            else
                vx[i][j] = vr.f[(long long)row * D + dim];
        }
    }
#pragma unroll
    for (int i = 0; i < KI; ++i) {
        const int e = tid + i * NT, f = e >> 6, l = e & 63;
        const floatx4 x = chunk_values<Q8>(kx[i][0]) * fk, y = chunk_values<Q8>(kx[i][1]) * fk;
        uint4 h, lo;
        split_pair(x[0], x[1], h.x, lo.x);
        split_pair(x[2], x[3], h.y, lo.y);
        split_pair(y[0], y[1], h.z, lo.z);
        split_pair(y[2], y[3], h.w, lo.w);
        img[(2 * f) * 64 + l] = h;
        img[(2 * f + 1) * 64 + l] = lo;
    }
    bool vlo = false;
#pragma unroll
    for (int i = 0; i < VI; ++i) {
        const int e = tid + i * NT;
        uint4 h, lo;
        split_pair(vx[i][0] * fv, vx[i][1] * fv, h.x, lo.x);
        split_pair(vx[i][2] * fv, vx[i][3] * fv, h.y, lo.y);
        split_pair(vx[i][4] * fv, vx[i][5] * fv, h.z, lo.z);
        split_pair(vx[i][6] * fv, vx[i][7] * fv, h.w, lo.w);
        vlo = vlo || lo_significant(lo.x) || lo_significant(lo.y) || lo_significant(lo.z) || lo_significant(lo.w);
        img[T::NKF * 64 + e] = h;
        img[(T::NKF + T::NVF) * 64 + e] = lo;
    }
    const int any_vlo = __syncthreads_or(vlo ? 1 : 0);
    if (tid == 0) flags[slot] = any_vlo ? 1u : 0u;
}

// Copies a tile image into LDS: each wave moves FRAGS / kWideWaves fragments of 1 KB.
template <int D>
__device__ __forceinline__ void wide_copy(const uint4* __restrict__ src, uint4* __restrict__ dst, int wave, int lane) {
    using T = WideTile<D>;
#pragma unroll
    for (int i = 0; i < T::FRAGS / kWideWaves; ++i) {
        const int f = (i * kWideWaves + wave) * 64;
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) void*)(src + f + lane),
            (__attribute__((address_space(3))) void*)(dst + f), 16, 0, 0);
    }
}

// One wave's running state over its 32 columns.
template <int D>
struct WideState {
    f16x8 qh[D / 16], ql[D / 16];
    floatx16 o[D / 32];
    float m, l;     // running maximum and this lane's share of the sum
};

// The running maximum is raised, and the accumulators rescaled, only when some column's maximum
// grew by more than dk::kLazyMargin: P then stays below 2^8, far inside fp16's range.
template <int D, bool SOFTCAP>
__device__ __forceinline__ void wide_tile(const uint4* __restrict__ t, WideState<D>& w, const PrefillArgs& a,
                                          float fs, bool masked, bool v_lo, int lane, int t0, int qpos,
                                          int qstart) {
    using T = WideTile<D>;
    floatx16 st[T::KT];
#pragma unroll
    for (int kt = 0; kt < T::KT; ++kt) {
        floatx16 acc = {};
#pragma unroll
        for (int s = 0; s < T::KS; ++s) {
            const f16x8 kh = __builtin_bit_cast(f16x8, t[T::kfrag(kt, s, 0) * 64 + lane]);
            const f16x8 kl = __builtin_bit_cast(f16x8, t[T::kfrag(kt, s, 1) * 64 + lane]);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, w.ql[s], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(kl, w.qh[s], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(kh, w.qh[s], acc, 0, 0, 0);
        }
        st[kt] = acc;
    }
    if constexpr (SOFTCAP) {   // its tanh needs registers that the other layers do not have to spare
        const float isc = a.inv_softcap * fs, rfs = pow2_inv(fs);
#pragma unroll
        for (int kt = 0; kt < T::KT; ++kt)
#pragma unroll
            for (int i = 0; i < 16; ++i) st[kt][i] = (a.softcap_log2e * tanhf(st[kt][i] * isc)) * rfs;
    }
    if (masked) {
        const int k0 = t0 + 4 * (lane >> 5);
#pragma unroll
        for (int kt = 0; kt < T::KT; ++kt)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int key = k0 + 32 * kt + 8 * (i >> 2) + (i & 3);
                st[kt][i] = key <= qpos && key >= qstart ? st[kt][i] : -__builtin_inff();
            }
    }
    float mt = kNegBig;
#pragma unroll
    for (int kt = 0; kt < T::KT; ++kt)
#pragma unroll
        for (int i = 0; i < 16; ++i) mt = fmaxf(mt, st[kt][i]);
    mt = dk::lane_step<32, true>(mt) * fs;
    if (__any(mt > w.m + dk::kLazyMargin)) {
        const float mn = fmaxf(w.m, mt);
        const float alpha = dk::fast_exp2(w.m - mn);
        w.m = mn;
        w.l *= alpha;
#pragma unroll
        for (int d = 0; d < T::DT; ++d) w.o[d] *= alpha;
    }
    const float m = w.m;
#pragma unroll
    for (int kt = 0; kt < T::KT; ++kt)
#pragma unroll
        for (int i = 0; i < 16; ++i) st[kt][i] = dk::fast_exp2(__builtin_fmaf(st[kt][i], fs, -m));
    // The tile's sum first, pairwise, then one add to the running sum: a chain of one add per
    // tile instead of one per key.
    float part[T::KT];
#pragma unroll
    for (int kt = 0; kt < T::KT; ++kt) {
        float s8[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) s8[i] = st[kt][i] + st[kt][8 + i];
        part[kt] = ((s8[0] + s8[1]) + (s8[2] + s8[3])) + ((s8[4] + s8[5]) + (s8[6] + s8[7]));
    }
    w.l += T::KT == 2 ? part[0] + part[T::KT - 1] : part[0];
    auto pv = [&](auto has_lo) {
        constexpr bool HL = decltype(has_lo)::value;
#pragma unroll
        for (int v = 0; v < T::VS; ++v) {
            const int kt = v >> 1, b = 8 * (v & 1);
            uint4 h, lo;
            split_pair(st[kt][b], st[kt][b + 1], h.x, lo.x);
            split_pair(st[kt][b + 2], st[kt][b + 3], h.y, lo.y);
            split_pair(st[kt][b + 4], st[kt][b + 5], h.z, lo.z);
            split_pair(st[kt][b + 6], st[kt][b + 7], h.w, lo.w);
            const f16x8 ph = __builtin_bit_cast(f16x8, h), pl = __builtin_bit_cast(f16x8, lo);
#pragma unroll
            for (int d = 0; d < T::DT; ++d) {
                const f16x8 vh = __builtin_bit_cast(f16x8, t[T::vfrag(v, d, 0) * 64 + lane]);
                if constexpr (HL) {
                    const f16x8 vl = __builtin_bit_cast(f16x8, t[T::vfrag(v, d, 1) * 64 + lane]);
                    w.o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vl, ph, w.o[d], 0, 0, 0);
                }
                w.o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, pl, w.o[d], 0, 0, 0);
                w.o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vh, ph, w.o[d], 0, 0, 0);
            }
        }
    };
    if (v_lo) pv(std::true_type{});
    else pv(std::false_type{});
}

// One trip: the copy of tile i + 1 into the other buffer, then tile i's products.  The restrict
// qualifiers tell the compiler that the copy's buffer is not the one read here, so its wait
// counts leave the copy in flight.
template <int D, bool SOFTCAP>
__device__ __forceinline__ void wide_trip(const uint4* __restrict__ cur, uint4* __restrict__ nxt,
                                          const uint4* __restrict__ next_src, bool has_next, bool run,
                                          WideState<D>& w, const PrefillArgs& a, float fs, bool masked,
                                          bool v_lo, int wave, int lane, int t0, int qpos, int qstart) {
    if (has_next) wide_copy<D>(next_src, nxt, wave, lane);
    if (run) wide_tile<D, SOFTCAP>(cur, w, a, fs, masked, v_lo, lane, t0, qpos, qstart);
}

// The wave's columns of block `blk` (waves of a group 0 .. kWideWaves - 1).
struct WideCols {
    bool has_q, ok;          // the wave has columns; this lane's column exists
    int tok, hq, qpos, qstart;
    int w_lo, w_hi;          // every column attends keys <= w_lo, none a key > w_hi
    int w_beg, w_full;       // none attends a key < w_beg, every column attends keys >= w_full
};
__device__ __forceinline__ WideCols wide_cols(const PrefillArgs& a, int group, int vkh, int blk, int wave, int lane) {
    WideCols c;
    const int cols = a.P * group, cw = blk * kWideCols + 32 * wave, col = cw + (lane & 31);
    c.has_q = cw < cols;
    c.ok = col < cols;
    const int cc = min(col, cols - 1);
    c.tok = cc / group;
    c.hq = vkh * group + (cc - c.tok * group);
    c.qpos = a.pos0 + c.tok;
    c.qstart = a.window > 0 ? max(0, c.qpos - a.window + 1) : 0;
    c.w_lo = a.pos0 + min(cw, cols - 1) / group;
    c.w_hi = a.pos0 + min(cw + 31, cols - 1) / group;
    c.w_beg = a.window > 0 ? max(0, c.w_lo - a.window + 1) : 0;
    c.w_full = a.window > 0 ? max(0, c.w_hi - a.window + 1) : 0;
    return c;
}
// First key tile of a block and its tile count.
template <int D>
__device__ __forceinline__ void wide_range(const PrefillArgs& a, int group, int blk, int& first, int& n) {
    const int cols = a.P * group, c0 = blk * kWideCols, c1 = min(c0 + kWideCols, cols) - 1;
    const int kbeg = a.window > 0 ? max(0, a.pos0 + c0 / group - a.window + 1) : 0;
    first = kbeg / WideTile<D>::TK;
    n = (a.pos0 + c1 / group) / WideTile<D>::TK - first + 1;
}

// Attention of column blocks over the tile images; grid y: key splits (ksplit > 1 writes partials
// for prefill_combine_kernel).
//
// GROUPS = 1: 4 waves, two workgroups per CU, grid x: blocks x virtual KV heads, heaviest first:
// the form for many blocks, where each freed slot takes the next one.
// GROUPS = 2: two groups of 4 waves, each with its own tile stream, one workgroup per CU: the form
// for at most one workgroup per CU, where the heaviest block would outlast the rest.  With
// `pairs`, grid x runs over pairs of blocks (p, nblk - 1 - p) x heads: group 1 takes the heavy
// block's first tiles and group 0 the light block, then the heavy one's last tiles, half of the
// pair's tiles each, so every CU holds two busy waves per SIMD to the end; group 0 hands its part
// of the heavy block to group 1 through LDS.  Without `pairs` the groups halve the split's tiles
// of one block.
template <int D, bool SOFTCAP, int GROUPS>
__global__ __launch_bounds__(GROUPS * kWideThreads) __attribute__((amdgpu_waves_per_eu(2)))
void prefill_wide_kernel(PrefillArgs a, const uint4* __restrict__ ws, const unsigned* __restrict__ flags, int tile0,
                         int n_tiles, int ksplit, int group, int pairs) {
    using T = WideTile<D>;
    __shared__ uint4 buf[GROUPS * 2][T::U4];
    const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int g = GROUPS == 2 ? wave_all / kWideWaves : 0, wave = wave_all - g * kWideWaves;
    const int nblk = (a.P * group + kWideCols - 1) / kWideCols;
    const int hkv_v = a.Hkv * a.kv_rep, ks = blockIdx.y;
    const int vkh = (int)blockIdx.x % hkv_v, kvh = vkh / a.kv_rep, item = (int)blockIdx.x / hkv_v;
    const int heavy = nblk - 1 - item;

    // Tiles of the heavy block (its split's share), and in pairs the light block's before them.
    int first, n_all;
    wide_range<D>(a, group, heavy, first, n_all);
    const int per = (n_all + ksplit - 1) / ksplit;
    first += ks * per;
    const int n_heavy = max(0, min(per, n_all - ks * per));
    int l_first = 0, n_light = 0;
    if (GROUPS == 2 && pairs != 0 && item < heavy) wide_range<D>(a, group, item, l_first, n_light);
    // Group 1 runs heavy tiles [0, trips), group 0 the light tiles and heavy tiles [trips, n_heavy).
    const int trips = GROUPS == 2 ? (n_heavy + n_light + 1) / 2 : n_heavy;
    const int n0 = g == 0 ? n_light : 0;                     // light tiles of this group
    const int h_first = first + (GROUPS == 2 && g == 0 ? trips : 0);
    const int n = n0 + (GROUPS == 2 && g == 0 ? max(0, n_heavy - trips) : min(trips, n_heavy));
    const uint4* img = ws + (size_t)kvh * n_tiles * T::U4;
    const unsigned* fl = flags + (size_t)kvh * n_tiles;
    auto tile_of = [&](int it) { return it < n0 ? l_first + it : h_first + it - n0; };

    uint4* hb = buf[2 * g];
    if (n > 0) wide_copy<D>(img + (size_t)(tile_of(0) - tile0) * T::U4, hb, wave, lane);
    const int ek = a.range[2 * kvh];
    const float fvs = pow2i(a.range[2 * kvh + 1]);   // V's range factor, restored on the output (exact)
    WideState<D> w;
    WideCols c;
    float fs = 1.0f;
    int it = 0;
    auto begin = [&](int blk) {   // a block's queries and an empty state
        c = wide_cols(a, group, vkh, blk, wave, lane);
        int eq;
        query_fragment<D, 16>(a, c.tok, c.hq, c.qpos, lane >> 5, w.qh, w.ql, eq);
        // fs = 2^(ek + eq): the factor that restores the scores' scale (prefill_attn2_kernel); eq is
        // the column's own.
        fs = pow2i(min(ek + eq, 127));
#pragma unroll
        for (int d = 0; d < T::DT; ++d) w.o[d] = floatx16{};
        w.m = kNegBig;
        w.l = 0.0f;
    };
    auto run_to = [&](int end) {
        for (; it < end; ++it) {
            // The copies of this trip's tile (this wave's part) have landed; after the barrier
            // everybody's have, and nobody reads the other buffer any more.
            __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
            __syncthreads();
            const int tile = tile_of(it), t0 = tile * T::TK;
            const bool run = it < n && c.has_q && t0 <= c.w_hi && t0 + T::TK > c.w_beg;
            const bool masked = t0 + T::TK - 1 > c.w_lo || t0 < c.w_full;
            const bool v_lo = it < n && fl[tile - tile0] != 0;
            wide_trip<D, SOFTCAP>(hb + (it & 1) * T::U4, hb + ((it + 1) & 1) * T::U4,
                                  img + (size_t)(tile_of(it + 1) - tile0) * T::U4, it + 1 < n, run, w, a, fs, masked,
                                  v_lo, wave, lane, t0, c.qpos, c.qstart);
        }
    };
    auto finish = [&](bool partial) {
        if (!c.ok) return;
        const float lt = dk::lane_step<32, false>(w.l);
        const int h4 = 4 * (lane >> 5);
        if (partial) {
            const long long slot = ((long long)ks * a.P + c.tok) * a.Hq + c.hq;
#pragma unroll
            for (int d = 0; d < T::DT; ++d)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    *reinterpret_cast<float4*>(a.part_o + slot * D + 32 * d + 8 * q + h4) =
                        make_float4(w.o[d][4 * q] * fvs, w.o[d][4 * q + 1] * fvs, w.o[d][4 * q + 2] * fvs,
                                    w.o[d][4 * q + 3] * fvs);
            if (h4 == 0) *reinterpret_cast<float2*>(a.part_ml + 2 * slot) = make_float2(w.m, lt);
            return;
        }
        const long long row = (long long)c.tok * a.Hq * D + (long long)c.hq * D;
#pragma unroll
        for (int d = 0; d < T::DT; ++d)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int d0 = 32 * d + 8 * q + h4;
                float4 r;
                r.x = dk::finish_output(w.m, lt, w.o[d][4 * q], a.sinks, a.gate, c.hq, row + d0) * fvs;
                r.y = dk::finish_output(w.m, lt, w.o[d][4 * q + 1], a.sinks, a.gate, c.hq, row + d0 + 1) * fvs;
                r.z = dk::finish_output(w.m, lt, w.o[d][4 * q + 2], a.sinks, a.gate, c.hq, row + d0 + 2) * fvs;
                r.w = dk::finish_output(w.m, lt, w.o[d][4 * q + 3], a.sinks, a.gate, c.hq, row + d0 + 3) * fvs;
                *reinterpret_cast<float4*>(a.out + row + d0) = r;
            }
    };
    begin(n0 > 0 ? item : heavy);
    if constexpr (GROUPS == 2) {
        if (n_light > 0) {   // both groups make the same trips: one barrier each
            run_to(n_light);
            if (g == 0) {
                finish(false);
                begin(heavy);
            }
        }
    }
    run_to(trips);
    if constexpr (GROUPS == 2) {
        // Group 0's part of the heavy block to group 1 (the tile buffers are free behind the
        // barrier), which merges it into its own.
        constexpr int XS = 2 + 16 * T::DT;   // floats per lane, strided by the lanes
        static_assert((size_t)kWideThreads * XS * sizeof(float) <= sizeof(buf), "exchange fits the tiles");
        float* x = reinterpret_cast<float*>(&buf[0][0]) + wave * 64 + lane;
        __syncthreads();
        if (g == 0) {
            x[0] = w.m;
            x[kWideThreads] = w.l;
#pragma unroll
            for (int d = 0; d < T::DT; ++d)
#pragma unroll
                for (int i = 0; i < 16; ++i) x[(2 + 16 * d + i) * kWideThreads] = w.o[d][i];
        }
        __syncthreads();
        if (g == 0) return;
        const float mb = x[0], mn = fmaxf(w.m, mb);
        const float sa = dk::fast_exp2(w.m - mn), sb = dk::fast_exp2(mb - mn);
        w.l = __builtin_fmaf(w.l, sa, x[kWideThreads] * sb);
#pragma unroll
        for (int d = 0; d < T::DT; ++d)
#pragma unroll
            for (int i = 0; i < 16; ++i)
                w.o[d][i] = __builtin_fmaf(w.o[d][i], sa, x[(2 + 16 * d + i) * kWideThreads] * sb);
        w.m = mn;
    }
    finish(ksplit > 1);
}

}  // namespace pk
}  // namespace llmp
