// Kernels of the decode step that sit between the AWQ linears of a Qwen3 block:
// residual-add + RMSNorm, per-head q/k RMSNorm + rotary + KV-cache write, attention over
// the paged KV cache, and SiLU(gate)*up.  All of them are HBM/latency bound byte movers;
// arithmetic is fp32 with the rounding points of the torch modules they stand in for.
#include <type_traits>

#include "awq_common.hpp"
#include "step_epilogues.hpp"
#include "step_kernels.hpp"
#include "../../include/nq_engine_ops.h"

namespace awq {
namespace {

constexpr float kLog2e = 1.4426950408889634f;

template <typename T>
__device__ __forceinline__ void unpack8(u32x4 v, float (&f)[8]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t w = v[i];
        f[2 * i] = T::to_f32((uint16_t)(w & 0xFFFFu));
        f[2 * i + 1] = T::to_f32((uint16_t)(w >> 16));
    }
}
template <typename T>
__device__ __forceinline__ u32x4 pack8(const float (&f)[8]) {
    u32x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = (uint32_t)T::from_f32(f[2 * i]) | ((uint32_t)T::from_f32(f[2 * i + 1]) << 16);
    return v;
}
template <typename T>
__device__ __forceinline__ float round_to(float f) { return T::to_f32(T::from_f32(f)); }

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// ---------------------------------------------------------------------------------------------
// residual (+= delta); y = RMSNorm(residual) * weight.  One workgroup per row, 8 values per lane
// and pass, at most 4 passes (hidden <= 8192).  The sum of squares is built per 128-column tile
// (tile_ssq) and the tiles are added in index order: the order the AWQ GEMVs with a residual epilogue
// and an RMSNorm prologue use, so both routes give the same bits.
constexpr int kNormThreads = 256;
constexpr int kNormPasses = 4;
constexpr int kNormTiles = kNormPasses * kNormThreads / 16;

// Loads the row (adding and storing delta if given), leaves the tile sums in s_tile and returns their total.
template <typename T>
__device__ __forceinline__ float row_load_ssq(uint16_t* __restrict__ residual, const uint16_t* __restrict__ delta,
                                              int64_t base, int hidden, float (&v)[kNormPasses][8], float* s_tile) {
#pragma unroll
    for (int p = 0; p < kNormPasses; ++p) {
        const int i = (p * kNormThreads + threadIdx.x) * 8;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[p][e] = 0.f;
        if (i < hidden) {
            unpack8<T>(*reinterpret_cast<const u32x4*>(residual + base + i), v[p]);
            if (delta) {
                float d[8];
                unpack8<T>(*reinterpret_cast<const u32x4*>(delta + base + i), d);
#pragma unroll
                for (int e = 0; e < 8; ++e) v[p][e] = round_to<T>(v[p][e] + d[e]);
                *reinterpret_cast<u32x4*>(residual + base + i) = pack8<T>(v[p]);
            }
        }
        const float ts = tile_ssq(v[p]);   // every lane takes part; lanes past the row add zeros
        if ((threadIdx.x & 15) == 0) s_tile[p * (kNormThreads / 16) + (threadIdx.x >> 4)] = ts;
    }
    __syncthreads();
    const int tiles = (hidden + 127) >> 7;
    float tot = 0.f;
    for (int t = 0; t < tiles; ++t) tot += s_tile[t];
    return tot;
}

template <typename T>
__global__ __launch_bounds__(kNormThreads) void add_rmsnorm_kernel(uint16_t* __restrict__ residual,
                                                                  const uint16_t* __restrict__ delta,
                                                                  const uint16_t* __restrict__ weight,
                                                                  uint16_t* __restrict__ y, int hidden, float eps) {
    __shared__ float s_tile[kNormTiles];
    const int64_t base = (int64_t)blockIdx.x * hidden;
    float v[kNormPasses][8];
    u32x4 wraw[kNormPasses];   // the weight does not depend on the reduction: fetched up front
#pragma unroll
    for (int p = 0; p < kNormPasses; ++p) {
        const int i = (p * kNormThreads + threadIdx.x) * 8;
        if (i < hidden) wraw[p] = *reinterpret_cast<const u32x4*>(weight + i);
    }
    const float tot = row_load_ssq<T>(residual, delta, base, hidden, v, s_tile);
    const float r = rsqrtf(tot / (float)hidden + eps);
#pragma unroll
    for (int p = 0; p < kNormPasses; ++p) {
        const int i = (p * kNormThreads + threadIdx.x) * 8;
        if (i < hidden) {
            float w[8], o[8];
            unpack8<T>(wraw[p], w);
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = mul_round<T>(v[p][e], r) * w[e];
            *reinterpret_cast<u32x4*>(y + base + i) = pack8<T>(o);
        }
    }
}

// The same, bit for bit, a wave a row, four rows a workgroup: rows of up to 512 P columns.  A workgroup a row has half its lanes
// idle at 1024 columns and a barrier between reading and writing; with many rows a wave each keeps more of them on the way
// (8192 x 1024: 13.5 -> 8.2 us, 17.1 -> 11.9 with a delta; 8192 x 2048
// 15.5 -> 11.7, 8192 x 4096 27.8 -> 25.7).
template <typename T, int P>
__global__ __launch_bounds__(256) void add_rmsnorm_rows_kernel(uint16_t* __restrict__ residual, const uint16_t* __restrict__ delta,
                                                               const uint16_t* __restrict__ weight, uint16_t* __restrict__ y,
                                                               int64_t rows, int hidden, float eps) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const int64_t base = row * hidden;
    u32x4 x[P], d[P], w[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int i = (p * 64 + lane) * 8;
        x[p] = d[p] = w[p] = u32x4{0u, 0u, 0u, 0u};
        if (i < hidden) {
            x[p] = *reinterpret_cast<const u32x4*>(residual + base + i);
            if (delta) d[p] = *reinterpret_cast<const u32x4*>(delta + base + i);
            w[p] = *reinterpret_cast<const u32x4*>(weight + i);
        }
    }
    float v[P][8], tot = 0.f;
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int i = (p * 64 + lane) * 8;
        unpack8<T>(x[p], v[p]);
        if (delta) {
            float f[8];
            unpack8<T>(d[p], f);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[p][e] = round_to<T>(v[p][e] + f[e]);
            if (i < hidden) *reinterpret_cast<u32x4*>(residual + base + i) = pack8<T>(v[p]);
        }
        const float ts = tile_ssq(v[p]);       // tiles past the row add zeros
#pragma unroll
        for (int t = 0; t < 4; ++t) tot += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, ts), 16 * t));
    }
    const float r = rsqrtf(tot / (float)hidden + eps);
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int i = (p * 64 + lane) * 8;
        float f[8], o[8];
        unpack8<T>(w[p], f);
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = mul_round<T>(v[p][e], r) * f[e];
        if (i < hidden) *reinterpret_cast<u32x4*>(y + base + i) = pack8<T>(o);
    }
}

// ssq[tile][row] = sum of squares of x[row, 128 tile .. 128 tile + 127]: the statistics an AWQ GEMV with an
// RMSNorm prologue reads, for a residual stream that no GEMV with a residual epilogue has produced yet.
// With `ids` the row is gathered from a table first (row ids[r] of `x`, clamped to the table) and copied to x_out:
// the embedding lookup of a decode step and its statistics in one launch.
template <typename T>
__global__ __launch_bounds__(kNormThreads) void row_ssq_kernel(const uint16_t* __restrict__ x, float* __restrict__ ssq,
                                                              int rows, int hidden, const int64_t* __restrict__ ids,
                                                              int64_t table_rows, uint16_t* __restrict__ x_out) {
    __shared__ float s_tile[kNormTiles];
    float v[kNormPasses][8];
    int64_t src = blockIdx.x;
    if (ids) {
        src = ids[blockIdx.x];
        src = src < 0 ? 0 : (src >= table_rows ? table_rows - 1 : src);
    }
    row_load_ssq<T>(const_cast<uint16_t*>(x), nullptr, src * hidden, hidden, v, s_tile);
    const int tiles = (hidden + 127) >> 7;
    if ((int)threadIdx.x < tiles) ssq[(size_t)threadIdx.x * rows + blockIdx.x] = s_tile[threadIdx.x];
    if (x_out) {
#pragma unroll
        for (int p = 0; p < kNormPasses; ++p) {
            const int i = (p * kNormThreads + threadIdx.x) * 8;
            if (i < hidden) *reinterpret_cast<u32x4*>(x_out + (int64_t)blockIdx.x * hidden + i) = pack8<T>(v[p]);
        }
    }
}

// ---------------------------------------------------------------------------------------------
// One wave per (token row, head) of the fused q|k|v projection output.  q and k heads: RMSNorm over
// the head, then the half-split rotary at the row's position; q goes to q_out, k to its cache
// slot; v heads are copied to their cache slot.  A lane owns the rotary pairs (i, i + hd/2).
// Cache layout [blocks][kv heads][block_size][head_dim]: slot s is token s % block_size of block s / block_size.
constexpr int kMaxPairs = 2;  // head_dim <= 256

template <typename T>
__global__ __launch_bounds__(256) void qk_norm_rope_store_kernel(
    const uint16_t* __restrict__ qkv, const uint16_t* __restrict__ q_weight, const uint16_t* __restrict__ k_weight,
    const float* __restrict__ cos_sin, const int64_t* __restrict__ positions, const int64_t* __restrict__ slots,
    uint16_t* __restrict__ q_out, uint16_t* __restrict__ k_out, uint16_t* __restrict__ k_cache,
    uint16_t* __restrict__ v_cache, int rows, int nh, int nkv, int hd, int max_positions, int64_t num_slots,
    int block_size, float eps) {
    const int heads = nh + 2 * nkv;
    const int64_t item = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (item >= (int64_t)rows * heads) return;
    const int row = (int)(item / heads), h = (int)(item % heads), lane = threadIdx.x & 63, half = hd >> 1;
    const uint16_t* src = qkv + ((int64_t)row * heads + h) * hd;
    const int64_t slot = slots[row];
    const bool slot_ok = slot >= 0 && slot < num_slots;
    uint16_t* dst;
    uint16_t* dst2 = nullptr;   // dense copy of a normalised, rotated k head (prefill attention reads it)
    if (h < nh) {
        dst = q_out + ((int64_t)row * nh + h) * hd;
    } else if (h < nh + nkv) {
        if (k_out) dst2 = k_out + ((int64_t)row * nkv + (h - nh)) * hd;
        if (!slot_ok) {
            if (!dst2) return;
            dst = dst2;
            dst2 = nullptr;
        } else {
            dst = k_cache + (((slot / block_size) * nkv + (h - nh)) * block_size + slot % block_size) * hd;
        }
    } else {
        if (!slot_ok) return;
        dst = v_cache + (((slot / block_size) * nkv + (h - nh - nkv)) * block_size + slot % block_size) * hd;
    }
    float a[kMaxPairs], b[kMaxPairs];
    float ss = 0.f;
#pragma unroll
    for (int p = 0; p < kMaxPairs; ++p) {
        const int i = p * 64 + lane;
        a[p] = b[p] = 0.f;
        if (i < half) {
            a[p] = T::to_f32(src[i]);
            b[p] = T::to_f32(src[i + half]);
            ss += a[p] * a[p] + b[p] * b[p];
        }
    }
    if (h >= nh + nkv) {  // v: plain copy
#pragma unroll
        for (int p = 0; p < kMaxPairs; ++p) {
            const int i = p * 64 + lane;
            if (i < half) {
                dst[i] = src[i];
                dst[i + half] = src[i + half];
            }
        }
        return;
    }
    // norm weight and angles do not depend on the reduction: fetched before it
    const uint16_t* w = h < nh ? q_weight : k_weight;
    int64_t pos = positions[row];
    pos = pos < 0 ? 0 : (pos >= max_positions ? max_positions - 1 : pos);
    const float* cs = cos_sin + pos * hd;
    float w1[kMaxPairs], w2[kMaxPairs], cc[kMaxPairs], sn[kMaxPairs];
#pragma unroll
    for (int p = 0; p < kMaxPairs; ++p) {
        const int i = p * 64 + lane;
        w1[p] = w2[p] = cc[p] = sn[p] = 0.f;
        if (i < half) {
            w1[p] = T::to_f32(w[i]);
            w2[p] = T::to_f32(w[i + half]);
            cc[p] = cs[i];
            sn[p] = cs[i + half];
        }
    }
    const float r = rsqrtf(wave_sum(ss) / (float)hd + eps);
#pragma unroll
    for (int p = 0; p < kMaxPairs; ++p) {
        const int i = p * 64 + lane;
        if (i < half) {
            const float x1 = round_to<T>(round_to<T>(a[p] * r) * w1[p]);
            const float x2 = round_to<T>(round_to<T>(b[p] * r) * w2[p]);
            const uint16_t y1 = T::from_f32(as_f32_result(__fsub_rn(__fmul_rn(x1, cc[p]), __fmul_rn(x2, sn[p]))));
            const uint16_t y2 = T::from_f32(as_f32_result(__fadd_rn(__fmul_rn(x1, sn[p]), __fmul_rn(x2, cc[p]))));
            dst[i] = y1;
            dst[i + half] = y2;
            if (dst2) {
                dst2[i] = y1;
                dst2[i + half] = y2;
            }
        }
    }
}

// The word of lane ^ O.
template <int O>
__device__ __forceinline__ uint32_t lane_xor(uint32_t x) {
    if constexpr (O == 8) return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x128, 0xF, 0xF, false);        // row_ror:8
    else if constexpr (O == 2) return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x4E, 0xF, 0xF, false);   // quad_perm:[2,3,0,1]
    else if constexpr (O == 1) return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0xB1, 0xF, 0xF, false);   // quad_perm:[1,0,3,2]
    else if constexpr (O < 32) return (uint32_t)__builtin_amdgcn_ds_swizzle((int)x, O << 10 | 0x1F);
    else return (uint32_t)__shfl_xor((int)x, O);
}
template <int O>
__device__ __forceinline__ float add_lanes(float v) {       // the sum over O + O lanes, xor O first
    v += __builtin_bit_cast(float, lane_xor<O>(__builtin_bit_cast(uint32_t, v)));
    if constexpr (O > 1) return add_lanes<O / 2>(v);
    return v;
}

// RMSNorm of a head and half-split rotary: HD / 8 neighbouring lanes hold a head, lane dc of them the dims a[0..7] = 8 dc ..;
// cs: cos | sin of the head's position.  The summation order and rounding points of the q|k|v GEMV's fused epilogue (head_dim
// 128: tile_ssq), so that all routes give the same bits.  The vector ALU's work bounds the kernels around it, hence two values a word
// where both are rounded or change lanes, and the sine's sign taken once: both halves are x cos + other sin, a
// product and a fused multiply-add.
template <typename T, int HD>
struct Turn {
    static constexpr int LPH = HD / 8, HALF = HD / 2;
    float c[8], s[8];     // cos; -sin in the first half, sin in the second
    __device__ __forceinline__ Turn(const float* __restrict__ cs, int dc) {
        const int i0 = (dc % (LPH / 2)) * 8;   // index of this lane's first dim inside its half
        const bool first = dc < LPH / 2;
#pragma unroll
        for (int e = 0; e < 8; e += 4) {
            const f32x4 cv = *reinterpret_cast<const f32x4*>(cs + i0 + e), sv = *reinterpret_cast<const f32x4*>(cs + HALF + i0 + e);
#pragma unroll
            for (int i = 0; i < 4; ++i) c[e + i] = cv[i], s[e + i] = first ? -sv[i] : sv[i];
        }
    }
    __device__ __forceinline__ u32x4 operator()(const float (&a)[8], u32x4 weight, float eps) const {
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = __builtin_fmaf(a[e], a[e], ss);
        const float r = rsqrtf(add_lanes<LPH / 2>(ss) / (float)HD + eps);
        float w[8], x[8], other[8];
        unpack8<T>(weight, w);
        u32x4 xn, turned;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            xn[i] = T::pack2(mul_round<T>(a[2 * i], r) * w[2 * i], mul_round<T>(a[2 * i + 1], r) * w[2 * i + 1]);
        u32x4 across;
#pragma unroll
        for (int i = 0; i < 4; ++i) across[i] = lane_xor<LPH / 2>(xn[i]);
        unpack8<T>(xn, x);
        unpack8<T>(across, other);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float y[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int e = 2 * i + h;
                y[h] = as_f32_result(__builtin_fmaf(x[e], c[e], other[e] * s[e]));
            }
            turned[i] = T::pack2(y[0], y[1]);
        }
        return turned;
    }
};
template <typename T, int HD>
__device__ __forceinline__ u32x4 norm_rope(const float (&a)[8], const uint16_t* __restrict__ w, const float* __restrict__ cs,
                                           int dc, float eps) {
    return Turn<T, HD>(cs, dc)(a, *reinterpret_cast<const u32x4*>(w + dc * 8), eps);
}

// The same with 16-byte accesses, for head dims of 64, 128 or 256 and 16-byte aligned tensors (the scalar kernel
// above moves 2 bytes per lane and instruction: 260 us per layer for a 16,384-token prefill of Qwen3-0.6B).
// A lane owns 8 consecutive dims of a head, HD/8 lanes a head, a wave 64/(HD/8) heads; the rotary partner
// (dims i and i + HD/2) sits HD/16 lanes away.  The arithmetic per element is that of the scalar kernel.
template <typename T, int HD>
__global__ __launch_bounds__(256) void qk_norm_rope_store_vec_kernel(
    const uint16_t* __restrict__ qkv, const uint16_t* __restrict__ q_weight, const uint16_t* __restrict__ k_weight,
    const float* __restrict__ cos_sin, const int64_t* __restrict__ positions, const int64_t* __restrict__ slots,
    uint16_t* __restrict__ q_out, uint16_t* __restrict__ k_out, uint16_t* __restrict__ k_cache,
    uint16_t* __restrict__ v_cache, int rows, int nh, int nkv, int max_positions, int64_t num_slots, int block_size,
    float eps) {
    constexpr int LPH = HD / 8, HPW = 64 / LPH, HALF = HD / 2;
    const int heads = nh + 2 * nkv;
    const int lane = threadIdx.x & 63, sub = lane / LPH, dc = lane % LPH;
    const int64_t items = (int64_t)rows * heads;
    int64_t item = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * HPW + sub;
    const bool live = item < items;   // lanes past the end follow the last item (the shuffles need them) and store nothing
    item = live ? item : items - 1;
    const int row = (int)(item / heads), h = (int)(item % heads);
    const uint16_t* src = qkv + ((int64_t)row * heads + h) * HD + dc * 8;
    const int64_t slot = slots[row];
    const bool slot_ok = slot >= 0 && slot < num_slots;
    float a[8];
    const u32x4 raw = *reinterpret_cast<const u32x4*>(src);
    unpack8<T>(raw, a);
    if (h >= nh + nkv) {   // v: plain copy
        if (live && slot_ok)
            *reinterpret_cast<u32x4*>(v_cache + (((slot / block_size) * nkv + (h - nh - nkv)) * block_size +
                                                  slot % block_size) * HD + dc * 8) = raw;
        // no return: heads of one wave differ in kind, and the shuffles below need every lane
    }
    const bool is_q = h < nh, is_k = !is_q && h < nh + nkv;
    int64_t pos = positions[row];
    pos = pos < 0 ? 0 : (pos >= max_positions ? max_positions - 1 : pos);
    const u32x4 packed = norm_rope<T, HD>(a, is_q ? q_weight : k_weight, cos_sin + pos * HD, dc, eps);
    if (!live || !(is_q || is_k)) return;
    if (is_q) {
        *reinterpret_cast<u32x4*>(q_out + ((int64_t)row * nh + h) * HD + dc * 8) = packed;
        return;
    }
    if (k_out) *reinterpret_cast<u32x4*>(k_out + ((int64_t)row * nkv + (h - nh)) * HD + dc * 8) = packed;
    if (slot_ok)
        *reinterpret_cast<u32x4*>(k_cache + (((slot / block_size) * nkv + (h - nh)) * block_size + slot % block_size) * HD +
                                  dc * 8) = packed;
}

// The same for the outputs of separate q, k and v projections of `batch` sequences of `tokens` tokens: q stays [token][head],
// k and v become [sequence][kv head][token], where the attention over the sequences reads a head's tokens in a row.
// A workgroup takes a token and HD / 8 of its lanes a head, U heads at a time: nothing is divided per lane, and the norm's weights and the token's
// angles are read once for several heads.  Bound by memory and the vector ALU: 8192 tokens of 16 + 8 + 8
// heads of 128 (134 MB) 29.5 us, 4.5 TB/s; with a head for every HD / 8 lanes of the launch, whose token and place four 64-bit divisions found, a lane
// exchange and a rounding for every value and both halves' sums in every lane 40; 512 tokens 5.5 -> 5.1, 8192 sequences of one token 40 -> 29 (66 with
// four tokens of a sequence a workgroup, which gain nothing at any length); as torch operations, which pass over fp32 copies a dozen times, 560.
template <typename T, int HD, int U>
__global__ __launch_bounds__(512) void qkv_norm_rope_kernel(const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
                                                            const uint16_t* __restrict__ v, const uint16_t* __restrict__ q_weight,
                                                            const uint16_t* __restrict__ k_weight,
                                                            const float* __restrict__ cos_sin,
                                                            const int64_t* __restrict__ positions, bool per_sequence,
                                                            uint16_t* __restrict__ q_out, uint16_t* __restrict__ k_out,
                                                            uint16_t* __restrict__ v_out, int sequences, int tokens, int nh, int nkv, bool beside_tokens,
                                                            int64_t max_positions, float q_eps, float k_eps) {
    constexpr int LPH = HD / 8;
    const int heads = nh + 2 * nkv, groups = blockDim.x / LPH, group = threadIdx.x / LPH, dc = threadIdx.x % LPH;
    // U == 1: blockDim.y tokens or sequences a workgroup.  Lanes past the last one or the last head follow it (the shuffles need them) and store nothing.
    const int tokens_here = U == 1 && beside_tokens ? blockDim.y : 1, sequences_here = U == 1 && !beside_tokens ? blockDim.y : 1;
    const int own_t = blockIdx.x * tokens_here + (tokens_here > 1 ? threadIdx.y : 0), own_seq = blockIdx.y * sequences_here + (sequences_here > 1 ? threadIdx.y : 0);
    const int t = min(own_t, tokens - 1), seq = min(own_seq, sequences - 1);
    const int64_t row = (int64_t)seq * tokens + t;
    int64_t pos = positions[per_sequence ? row : t];
    pos += pos < 0 ? max_positions : 0;     // an index from the end, as the table's own indexing takes it
    const bool known = pos >= 0 && pos < max_positions;     // no angles for any other: not a number, rather than a wrong turn
    const float* angles = cos_sin + (known ? pos : 0) * HD;
    for (int h0 = blockIdx.z * U * groups; h0 < heads; h0 += gridDim.z * U * groups) {
        u32x4 raw[U], weight[U];
        uint16_t* dst[U];
        bool plain[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int h = min(h0 + u * groups + group, heads - 1), kv = h < nh + nkv ? h - nh : h - nh - nkv;
            const bool is_q = h < nh;
            plain[u] = h >= nh + nkv;
            raw[u] = *reinterpret_cast<const u32x4*>((is_q ? q + (row * nh + h) * HD : (plain[u] ? v : k) + (row * nkv + kv) * HD) + dc * 8);
            dst[u] = (is_q ? q_out + (row * nh + h) * HD : (plain[u] ? v_out : k_out) + (((int64_t)seq * nkv + kv) * tokens + t) * HD) + dc * 8;
            weight[u] = *reinterpret_cast<const u32x4*>((is_q ? q_weight : k_weight) + dc * 8);
        }
        const Turn<T, HD> turn(angles, dc);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int h = h0 + u * groups + group;
            float a[8];
            unpack8<T>(raw[u], a);
            const u32x4 turned = turn(a, weight[u], known ? (h < nh ? q_eps : k_eps) : __builtin_nanf(""));
            if (h < heads && own_t < tokens && own_seq < sequences) *reinterpret_cast<u32x4*>(dst[u]) = plain[u] ? raw[u] : turned;
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Attention of one new token per sequence over its paged KV cache (flash-decoding).
// Workgroup = (sequence, kv head, context split), WAVES waves (here 16 for up to 2 query heads per kv head, 8 for
// 4, 4 for 8: the wave merge buffer grows with G); with enough waves per workgroup a batch of sequences
// needs no context split and no second kernel.  A wave covers TPW = 64 / (HD/8) tokens
// per step: a lane holds 8 head dims of one token's K and V rows (one 16-byte load each), the G
// query heads of the kv group share those loads.  Every lane group keeps its own online-softmax
// state (running max, sum, 8 accumulators per query head); the states are merged across lane
// groups, then waves (LDS), then splits (fp32 partials + a second kernel).
constexpr float kNegBig = -3.0e38f;
constexpr int kMaxSplits = 16;
// Context splits of a (sequence, kv head) pair: workgroups are launched for `most`, split by split; a sequence of fewer than `from` tokens lies in the
// first `few`, and the workgroups of the others are done at once.
struct Splits {
    int pairs, most, few, from;
    __device__ __forceinline__ int of(int context) const { return context >= from ? most : few; }
};

template <typename T, int G, int HD, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void paged_attn_decode_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k_cache, const uint16_t* __restrict__ v_cache,
    const int32_t* __restrict__ block_table, const int32_t* __restrict__ context_lens, uint16_t* __restrict__ out,
    float* __restrict__ partial, int nkv, int block_size, int max_blocks, int num_blocks, Splits splits, float scale, int tiled) {
    constexpr int LPT = HD / 8;    // lanes per token
    constexpr int TPW = 64 / LPT;  // tokens per wave step
    constexpr int U = 2;           // token steps in flight
    constexpr bool kEarly = G == 4;   // block numbers of the first step beside the context length
    const int sp = blockIdx.x / (uint32_t)splits.pairs, pair = blockIdx.x % (uint32_t)splits.pairs;
    const int kvh = pair % (uint32_t)nkv, b = pair / (uint32_t)nkv;
    const int nh = nkv * G;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int dc = lane % LPT, ts = lane / LPT;

    // With four heads the first step's block numbers are asked for beside the context length where they don't hang on it: one trip to memory less before
    // the first keys, and registers that the compiler lays out better (us, blocks of 24 tokens, asked for step by step / so: 16 x 300 tokens of heads of
    // 128 21.1 / 18.3, 64 x 1300 119 / 88; heads of 64 24 x 4000 88 / 65).  Eight heads lose a fifth by it (heads of 64 31 x 4000 130 / 163, heads of 128 1 x
    // 140 17.6 / 22.4), one and two a twentieth up to 140 tokens (4.8 / 5.0, 7.2 / 7.6).
    const int32_t* table = block_table + (int64_t)b * max_blocks;
    int blocks[U], blocks0 = 0;
    if (kEarly && splits.most == 1) {
        blocks0 = table[0];
#pragma unroll
        for (int u = 0; u < U; ++u) blocks[u] = table[min((wave * TPW + ts + u * WAVES * TPW) / block_size, max_blocks - 1)];
    }
    int ctx = context_lens[b];
    ctx = ctx < 0 ? 0 : (ctx > max_blocks * block_size ? max_blocks * block_size : ctx);
    const int nsplit = splits.of(ctx);
    if (sp >= nsplit) return;
    const int per = (ctx + nsplit - 1) / nsplit;
    const int t0 = sp * per, t1 = min(ctx, t0 + per);

    float qf[G][8];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        unpack8<T>(*reinterpret_cast<const u32x4*>(q + ((int64_t)b * nh + kvh * G + g) * HD + dc * 8), qf[g]);
#pragma unroll
        for (int e = 0; e < 8; ++e) qf[g][e] *= scale * kLog2e;
    }
    float m[G], l[G], acc[G][8];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        m[g] = kNegBig;
        l[g] = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[g][e] = 0.f;
    }

    for (int t = t0 + wave * TPW + ts; t - ts < t1; t += WAVES * TPW * U) {
        u32x4 kr[U], vr[U];
        bool ok[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int tt = t + u * WAVES * TPW;
            ok[u] = tt < t1;
            const int tc = ok[u] ? tt : t0;
            int blk = kEarly && splits.most == 1 && t < WAVES * TPW * U ? (ok[u] ? blocks[u] : blocks0) : table[tc / block_size];
            blk = blk < 0 ? 0 : (blk >= num_blocks ? num_blocks - 1 : blk);
            const int64_t off = (((int64_t)blk * nkv + kvh) * block_size + tc % block_size) * HD + dc * 8;
            kr[u] = *reinterpret_cast<const u32x4*>(k_cache + off);
            vr[u] = *reinterpret_cast<const u32x4*>(v_cache + off);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float kf[8], vf[8];
            unpack8<T>(kr[u], kf);
            unpack8<T>(vr[u], vf);
#pragma unroll
            for (int g = 0; g < G; ++g) {
                float s = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) s += qf[g][e] * kf[e];
#pragma unroll
                for (int o = LPT / 2; o >= 1; o >>= 1) s += __shfl_xor(s, o);
                s = ok[u] ? s : kNegBig;
                const float mn = fmaxf(m[g], s);
                const float c = exp2f(m[g] - mn);
                const float p = ok[u] ? exp2f(s - mn) : 0.f;
                m[g] = mn;
                l[g] = l[g] * c + p;
#pragma unroll
                for (int e = 0; e < 8; ++e) acc[g][e] = acc[g][e] * c + p * vf[e];
            }
        }
    }

    // merge the TPW lane groups of this wave
#pragma unroll
    for (int g = 0; g < G; ++g) {
#pragma unroll
        for (int o = LPT; o < 64; o <<= 1) {
            const float mo = __shfl_xor(m[g], o), lo = __shfl_xor(l[g], o);
            const float mn = fmaxf(m[g], mo);
            const float ca = exp2f(m[g] - mn), cb = exp2f(mo - mn);
            l[g] = l[g] * ca + lo * cb;
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[g][e] = acc[g][e] * ca + __shfl_xor(acc[g][e], o) * cb;
            m[g] = mn;
        }
    }
    // merge the waves through LDS: [wave][g][HD + 2]
    __shared__ float s_acc[WAVES][G][HD + 2];
    if (ts == 0) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
#pragma unroll
            for (int e = 0; e < 8; ++e) s_acc[wave][g][dc * 8 + e] = acc[g][e];
            if (dc == 0) {
                s_acc[wave][g][HD] = m[g];
                s_acc[wave][g][HD + 1] = l[g];
            }
        }
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < G * HD; idx += 64 * WAVES) {
        const int g = idx / HD, d = idx % HD;
        float mn = kNegBig;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) mn = fmaxf(mn, s_acc[w][g][HD]);
        float lt = 0.f, at = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const float c = exp2f(s_acc[w][g][HD] - mn);
            lt += s_acc[w][g][HD + 1] * c;
            at += s_acc[w][g][d] * c;
        }
        const int64_t head = (int64_t)b * nh + kvh * G + g;
        if (nsplit == 1) {
            out[tiled ? tiled_at(b, (kvh * G + g) * HD + d, nh * HD) / 2 : head * HD + d] = T::from_f32(lt > 0.f ? at / lt : 0.f);
        } else {
            float* dst = partial + (head * splits.most + sp) * (HD + 2);
            dst[d] = at;
            if (d == 0) {
                dst[HD] = mn;
                dst[HD + 1] = lt;
            }
        }
    }
}

// The same for 2 or 4 query heads per kv head and 128 head dims, where the kernel above is bound by its
// vector-ALU dot products (8 FMAs, 4 shuffles and an online-softmax update per token, head and lane).
// A wave takes tiles of 16 tokens.  Scores: S^T = K q^T on the 16x16x32 MFMA (A = 16 token rows of K, 32 head dims
// per instruction; B = the G query heads as columns, the rest zero), so a lane ends up with 4 tokens of one head and
// the softmax bookkeeping is done once per tile and head, not per token and lane.  The probabilities cross to the
// value phase through a 16 x G array in LDS (private to the wave); there a lane holds 8 head dims of one token's V row
// as before and adds p * v for the G heads.  Tiles start at multiples of 16 tokens inside a context split and
// block_size % 16 == 0, so a tile never straddles a cache block.
// A lane holds the block of one of its wave's next 64 tiles each, so that a tile is one trip to memory and not two.  Rows past the context lie
// outside the buffer of their load: they are zero and cost no memory access.
// Bound by memory once 256 workgroups run; then the cache streams past the L2 (`full`: the rounds of workgroups on 256 CUs are three quarters full or
// more; and the workgroup's context is its share of 16 MB or more).  bf16, 8 kv heads, us, 28 layers' caches in turn; two heads, the vector kernel / this one:
// 1 x 1300 14.0 / 8.2, 8 x 320 11.2 / 7.8, 12 x 640 21.7 / 13.6, 32 x 640 21.0 / 16.5,
// 64 x 640 38 / 28.4, 64 x 1000 63.5 / 44.7 = 5.9 TB/s, 1 x 8000 24.9 / 14.7.  Four heads, this one with a tile
// behind its block number / now: 1 x 1300 13.5 / 8.7, 24 x 640 19.8 / 16.7, 32 x 640 20.2 / 18.2, 64 x 1000 52.4 / 44.9, 1 x 140 5.75 / 5.9.  Through the L2 32 x 640 takes 19.2 and
// 64 x 1000 50; part rounds and smaller caches are better off there (20 x 640 13.2, past it 14.3; 8 x 140 5.6, 6.2).  Two or more tiles on their way in a
// wave's registers take longer at every size (32 x 640 19.2 with two, 20.0 with four).  The last tile stands behind the loop, which asks for no tile that
// is not there: a workgroup waits for such loads before it adds its waves' sums (four heads, 32 x 64 6.1 -> 5.8 us, 24 x 300 10.8 -> 10.1, 64 x 140 11.8 -> 11.3).
template <typename T, int G, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void paged_attn_decode_mfma_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k_cache, const uint16_t* __restrict__ v_cache,
    const int32_t* __restrict__ block_table, const int32_t* __restrict__ context_lens, uint16_t* __restrict__ out,
    float* __restrict__ partial, int nkv, int block_size, int max_blocks, int num_blocks, Splits splits, float scale, int tiled,
    int full) {
    constexpr int HD = 128, TT = 16;
    static_assert(G == 2 || G == 4, "query heads per kv head");
    typedef float fG __attribute__((ext_vector_type(G)));
    const int sp = blockIdx.x / (uint32_t)splits.pairs, pair = blockIdx.x % (uint32_t)splits.pairs;
    const int kvh = pair % (uint32_t)nkv, b = pair / (uint32_t)nkv;
    const int nh = nkv * G;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lo = lane & 15, hi = lane >> 4;   // score phase: head lo, token quad hi; value phase: dims 8*lo.., token hi

    const int32_t* table = block_table + (int64_t)b * max_blocks;
    // blocks of the wave's tiles first, first + 1, .., one a lane
    const auto blocks_from = [&](int t0, int first) {
        // (a context is below 2^31, and the last of 64 tiles lies less than 2^14 behind its end)
        const uint32_t t = (uint32_t)t0 + ((uint32_t)(first + lane) * WAVES + wave) * TT, last = (uint32_t)max_blocks * block_size - 1;
        return table[min(t, last) / (uint32_t)block_size];
    };
    int blocks = splits.most == 1 ? blocks_from(0, 0) : 0;     // asked for beside the context length
    int ctx = context_lens[b];
    u32x4 bq[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        bq[i] = u32x4{0u, 0u, 0u, 0u};
        if (lo < G)
            bq[i] = *reinterpret_cast<const u32x4*>(q + ((int64_t)b * nh + kvh * G + lo) * HD + 32 * i + 8 * hi);
    }
    ctx = ctx < 0 ? 0 : (ctx > max_blocks * block_size ? max_blocks * block_size : ctx);
    const int nsplit = splits.of(ctx);
    if (sp >= nsplit) return;
    const int per = nsplit == 1 ? ctx : ((ctx + nsplit - 1) / nsplit + TT - 1) / TT * TT;
    const int t0 = sp * per, t1 = min(ctx, t0 + per);
    const int tiles = t1 - t0 > wave * TT ? (t1 - t0 - wave * TT + WAVES * TT - 1) / (WAVES * TT) : 0;
    if (splits.most > 1) blocks = blocks_from(t0, 0);
    int held = 0;

    __shared__ __align__(16) float s_p[WAVES][TT * G + G];   // per wave: p[token][head], then the rescale factor per head
    __shared__ float s_acc[WAVES][G][HD + 2];
    float* P = s_p[wave];

    u32x4 ka[4], va[4];
    const auto load = [&](int tile, auto policy) __attribute__((always_inline)) {
        constexpr int kPolicy = decltype(policy)::value;
        if (tile - held >= 64) {
            held = tile;
            blocks = blocks_from(t0, held);
        }
        int blk = __builtin_amdgcn_readlane(blocks, (tile - held) & 63);
        blk = blk < 0 ? 0 : (blk >= num_blocks ? num_blocks - 1 : blk);
        const int tb = t0 + (tile * WAVES + wave) * TT;
        const uint32_t bytes = (uint32_t)min(TT, t1 - tb) * (HD * 2);
        const int64_t base = (((int64_t)blk * nkv + kvh) * block_size + (uint32_t)tb % (uint32_t)block_size) * HD;
        const __amdgpu_buffer_rsrc_t k = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(k_cache + base), 0, bytes, 0x00020000);
        const __amdgpu_buffer_rsrc_t v = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(v_cache + base), 0, bytes, 0x00020000);
#pragma unroll
        for (int i = 0; i < 4; ++i) ka[i] = __builtin_amdgcn_raw_buffer_load_b128(k, lo * 256 + hi * 16 + 64 * i, 0, kPolicy);
#pragma unroll
        for (int u = 0; u < 4; ++u) va[u] = __builtin_amdgcn_raw_buffer_load_b128(v, hi * 256 + lo * 16 + 1024 * u, 0, kPolicy);
    };

    const float sc = scale * kLog2e;
    float m = kNegBig, lpart = 0.f;
    float acc[G][8];
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[g][e] = 0.f;

    const auto take = [&](int tile) __attribute__((always_inline)) {
        const int left = t1 - (t0 + (tile * WAVES + wave) * TT);
        f32x4 st = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) st = T::mfma16(ka[i], bq[i], st);
        // st[r]: head lo, token 4*hi + r of the tile
        float sv[4], mx = kNegBig;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            sv[r] = (4 * hi + r < left) ? st[r] * sc : kNegBig;
            mx = fmaxf(mx, sv[r]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float mn = fmaxf(m, mx);
        const float c = exp2f(m - mn);
        m = mn;
        float ps = 0.f;
        float pr[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            pr[r] = (4 * hi + r < left) ? exp2f(sv[r] - mn) : 0.f;
            ps += pr[r];
        }
        lpart = lpart * c + ps;
        if (lo < G) {
#pragma unroll
            for (int r = 0; r < 4; ++r) P[(4 * hi + r) * G + lo] = pr[r];
            if (hi == 0) P[TT * G + lo] = c;
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_wave_barrier();   // LDS operations of a wave execute in order: the reads below see these writes
        asm volatile("" ::: "memory");
        const fG cg = *reinterpret_cast<const fG*>(P + TT * G);
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[g][e] *= cg[g];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            float vf[8];
            unpack8<T>(va[u], vf);
            const fG pg = *reinterpret_cast<const fG*>(P + (4 * u + hi) * G);
#pragma unroll
            for (int g = 0; g < G; ++g)
#pragma unroll
                for (int e = 0; e < 8; ++e) acc[g][e] += pg[g] * vf[e];
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_wave_barrier();   // the next tile's writes come after these reads
        asm volatile("" ::: "memory");
    };
    const auto walk = [&](auto policy) {
        for (int tile = 0; tile + 1 < tiles; ++tile) {
            take(tile);
            load(tile + 1, policy);     // (behind a condition the loop takes half as long again, 32 x 640 25.1 us)
        }
    };
    if (tiles) {
        load(0, std::integral_constant<int, 0>{});
        if ((full >> (nsplit < splits.most) & 1) && (int64_t)(t1 - t0) * splits.pairs * nsplit >= 32768) walk(std::integral_constant<int, 2>{});      // nt
        else walk(std::integral_constant<int, 0>{});
        take(tiles - 1);
    }

    // the four token groups of the wave share m: their accumulators and partial sums just add
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            acc[g][e] += __shfl_xor(acc[g][e], 16);
            acc[g][e] += __shfl_xor(acc[g][e], 32);
        }
    lpart += __shfl_xor(lpart, 16);
    lpart += __shfl_xor(lpart, 32);
    if (hi == 0) {
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int e = 0; e < 8; ++e) s_acc[wave][g][lo * 8 + e] = acc[g][e];
        if (lo < G) {
            s_acc[wave][lo][HD] = m;
            s_acc[wave][lo][HD + 1] = lpart;
        }
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < G * HD; idx += 64 * WAVES) {
        const int g = idx / HD, d = idx % HD;
        float mn = kNegBig;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) mn = fmaxf(mn, s_acc[w][g][HD]);
        float lt = 0.f, at = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const float c = exp2f(s_acc[w][g][HD] - mn);
            lt += s_acc[w][g][HD + 1] * c;
            at += s_acc[w][g][d] * c;
        }
        const int64_t head = (int64_t)b * nh + kvh * G + g;
        if (nsplit == 1) {
            out[tiled ? tiled_at(b, (kvh * G + g) * HD + d, nh * HD) / 2 : head * HD + d] = T::from_f32(lt > 0.f ? at / lt : 0.f);
        } else {
            float* dst = partial + (head * splits.most + sp) * (HD + 2);
            dst[d] = at;
            if (d == 0) {
                dst[HD] = mn;
                dst[HD + 1] = lt;
            }
        }
    }
}

// Both products on the matrix cores, for 128 head dims and block sizes that are multiples of 16.  The query heads of
// a kv head are columns of a 16-column MFMA tile, so any count up to 16 fits: G > 0 fixes it at compile time (the
// launcher uses 8), G = 0 takes it from `heads_per_kv` -- the route of the head ratios the other kernels have no
// instantiation for (Qwen3-14B: 40 query heads on 8 kv heads).  The kernel above multiplies the probabilities with V on the vector ALU (G x 8
// FMAs per token and lane), which with 8 heads per kv head costs as much as fetching the cache: cache-resident it
// still takes 62 of the 102 us it needs from HBM at 64 sequences x 8 kv heads x 2060 tokens.  Here a wave takes
// tiles of 32 tokens:
//   scores   S^T = K q^T as above (two 16-token halves, four MFMAs each): a lane ends up with the scores of head
//            lane % 16 and tokens 4 * (lane / 16) + r of both halves -- which is where the B operand of the second
//            product wants the probabilities of that head, so they never leave their registers;
//   values   out^T[dims, heads] = V^T P^T, one MFMA per 16 head dims and tile.  Its A operand needs, per lane, eight
//            tokens of ONE head dim, but a V row has the dims side by side: the tile is brought to LDS (load-to-LDS,
//            16 lanes per row) and read back with the transposing LDS read (ds_read_b64_tr_b16: in each group of 16
//            lanes, lane 4q + c receives element c of the four 8-byte pieces that lanes q, q + 4, q + 8, q + 12 point
//            at).  Rows sit 256 bytes apart, i.e. on the same banks; each row is therefore stored rotated by its own
//            index in units of 32 bytes (the load's lanes simply fetch the rotated piece), and the 16 tokens of one
//            transposing read fall on all 64 banks twice.
// The online-softmax state (running maximum, rescale factor) is per head and lives in the lanes of that head, which
// are also the lanes that hold that head's output column: nothing crosses lanes but the maximum.
// Rows past the context may hold anything: their scores are replaced before the maximum, their probabilities are
// zero, and their V rows are fetched from the last valid token of the tile (0 x NaN would be NaN).
#define NQ_GPTR(p) ((__attribute__((address_space(1))) void*)(p))
#define NQ_LPTR(p) ((__attribute__((address_space(3))) void*)(p))
typedef short nq_s16x4 __attribute__((ext_vector_type(4)));

template <typename T, int G, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void paged_attn_decode_tr_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k_cache, const uint16_t* __restrict__ v_cache,
    const int32_t* __restrict__ block_table, const int32_t* __restrict__ context_lens, uint16_t* __restrict__ out,
    float* __restrict__ partial, int nkv, int block_size, int max_blocks, int num_blocks, int nsplit, float scale,
    int heads_per_kv) {
    constexpr int HD = 128, TT = 32, VBYTES = TT * HD * 2, WBYTES = 2 * VBYTES;   // a wave's K tile and V tile
    constexpr int GA = G ? G : 16;                                                // rows of the per-wave result
    static_assert(G >= 0 && G <= 16, "query heads per kv head");
    static_assert(GA * (HD + 2) * 4 <= WBYTES, "the per-wave results reuse the wave's tiles");
    const int Gv = G ? G : heads_per_kv;
    const int sp = blockIdx.x % nsplit;
    const int kvh = (blockIdx.x / nsplit) % nkv;
    const int b = blockIdx.x / (nsplit * nkv);
    const int nh = nkv * Gv;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lo = lane & 15, hi = lane >> 4;

    int ctx = context_lens[b];
    ctx = ctx < 0 ? 0 : (ctx > max_blocks * block_size ? max_blocks * block_size : ctx);
    const int per = ((ctx + nsplit - 1) / nsplit + TT - 1) / TT * TT;
    const int t0 = sp * per, t1 = min(ctx, t0 + per);

    __shared__ __attribute__((aligned(1024))) unsigned char s_raw[WAVES * WBYTES];
    unsigned char* kt = s_raw + wave * WBYTES;                       // this wave's K tile [32 tokens][256 B, rotated]
    unsigned char* vt = kt + VBYTES;                                 // and its V tile
    float (*s_acc)[GA][HD + 2] = reinterpret_cast<float (*)[GA][HD + 2]>(s_raw);   // after the loop

    u32x4 bq[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        bq[i] = u32x4{0u, 0u, 0u, 0u};
        if (lo < Gv)
            bq[i] = *reinterpret_cast<const u32x4*>(q + ((int64_t)b * nh + kvh * Gv + lo) * HD + 32 * i + 8 * hi);
    }
    const float sc = scale * kLog2e;
    float m = kNegBig, lpart = 0.f;
    f32x4 acc[8];
#pragma unroll
    for (int cb = 0; cb < 8; ++cb) acc[cb] = f32x4{0.f, 0.f, 0.f, 0.f};

    // load-to-LDS lane roles: instruction k fills rows 4k .. 4k + 3, 16 lanes a row (a whole 256-byte row per 16
    // lanes: 16 rows x 64 bytes per instruction, the A-operand layout of the score product, moves half as fast).
    // V: 16-byte position c' of row r holds the row's piece (window (c' / 2 - r) mod 8, half c' % 2); K: position c'
    // holds piece (c' - r) mod 16, so that the 16 token rows a b128 read of one piece index touches differ in bank.
    const int dma_row = lane >> 4, dma_piece = lane & 15;
    // transposing read: as a source, this lane points at token 4 * hi + lo / 4 (+ 16 for the second half), quad lo % 4
    const int tr_tok = 4 * hi + (lo >> 2), tr_quad = (lo & 3) * 8;

    const int32_t* table = block_table + (int64_t)b * max_blocks;
    for (int tb = t0 + wave * TT; tb < t1; tb += WAVES * TT) {
        int blk = table[tb / block_size];                         // wave-uniform
        blk = blk < 0 ? 0 : (blk >= num_blocks ? num_blocks - 1 : blk);
        const int64_t base = (((int64_t)blk * nkv + kvh) * block_size + tb % block_size) * HD;
        const int last = min(TT, t1 - tb) - 1;                    // last valid row of the tile
        // rows 16..31: in the same cache block 16 rows on, or (block sizes that are odd multiples of 16) at the start
        // of the next one; where the context ends before them, the first 16 rows stand in (their scores are replaced)
        int64_t base16 = base + 16 * HD;
        if (tb % block_size + 16 >= block_size) {                 // wave-uniform
            base16 = base;
            if (tb + 16 < t1) {
                int blk1 = table[(tb + 16) / block_size];
                blk1 = blk1 < 0 ? 0 : (blk1 >= num_blocks ? num_blocks - 1 : blk1);
                base16 = ((int64_t)blk1 * nkv + kvh) * block_size * HD;
            }
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {   // rows past the context are fetched as they are: their scores are replaced
            const int r = 4 * k + dma_row;
            const uint16_t* src = k_cache + (k < 4 ? base : base16) + (int64_t)(r & 15) * HD + 8 * ((dma_piece - r) & 15);
            __builtin_amdgcn_global_load_lds(NQ_GPTR(src), NQ_LPTR(kt + k * 1024), 16, 0, 0);
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int r = 4 * k + dma_row;
            const int w = ((dma_piece >> 1) - r) & 7;
            const int rr = min(r, last);
            const uint16_t* src = v_cache + (rr < 16 ? base : base16) + (int64_t)(rr & 15) * HD + 16 * w + 8 * (dma_piece & 1);
            __builtin_amdgcn_global_load_lds(NQ_GPTR(src), NQ_LPTR(vt + k * 1024), 16, 0, 0);
        }
        // the K tile has landed: a wave's loads return in order, the eight of the V tile are the newest
        asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        f32x4 st[2];
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            st[a] = f32x4{0.f, 0.f, 0.f, 0.f};
            const int r = 16 * a + lo;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const u32x4 ka = *reinterpret_cast<const u32x4*>(kt + r * 256 + ((4 * i + hi + r) & 15) * 16);
                st[a] = T::mfma16(ka, bq[i], st[a]);
            }
        }
        // st[a][r]: head lo, token tb + 16 a + 4 hi + r
        float sv[2][4], mx = kNegBig;
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                sv[a][r] = (16 * a + 4 * hi + r <= last) ? st[a][r] * sc : kNegBig;
                mx = fmaxf(mx, sv[a][r]);
            }
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float mn = fmaxf(m, mx);
        const float c = exp2f(m - mn);
        m = mn;
        float pr[2][4], ps = 0.f;
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                pr[a][r] = (16 * a + 4 * hi + r <= last) ? exp2f(sv[a][r] - mn) : 0.f;
                ps += pr[a][r];
            }
        lpart = lpart * c + ps;
        const u32x4 pb = u32x4{T::pack2(pr[0][0], pr[0][1]), T::pack2(pr[0][2], pr[0][3]),
                               T::pack2(pr[1][0], pr[1][1]), T::pack2(pr[1][2], pr[1][3])};
#pragma unroll
        for (int cb = 0; cb < 8; ++cb)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[cb][r] *= c;
        // the V tile has landed
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
        for (int cb = 0; cb < 8; ++cb) {
            u32x4 vf;
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                const int tok = 16 * a + tr_tok;
                const nq_s16x4 t4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (nq_s16x4 __attribute__((address_space(3)))*)(vt + tok * 256 + (((cb + tok) & 7) << 5) + tr_quad));
                const u32x2 t2 = __builtin_bit_cast(u32x2, t4);
                vf[2 * a] = t2[0];
                vf[2 * a + 1] = t2[1];
            }
            acc[cb] = T::mfma16(vf, pb, acc[cb]);   // rows: dims 16 cb + 4 hi + r, column: head lo
        }
        // the next tile's loads overwrite both tiles: every read of them has returned
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }

    lpart += __shfl_xor(lpart, 16);
    lpart += __shfl_xor(lpart, 32);
    __syncthreads();   // every wave is done with its tiles: the area now holds the per-wave results
    if (lo < Gv) {
#pragma unroll
        for (int cb = 0; cb < 8; ++cb)
#pragma unroll
            for (int r = 0; r < 4; ++r) s_acc[wave][lo][16 * cb + 4 * hi + r] = acc[cb][r];
        if (hi == 0) {
            s_acc[wave][lo][HD] = m;
            s_acc[wave][lo][HD + 1] = lpart;
        }
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < Gv * HD; idx += 64 * WAVES) {
        const int g = idx / HD, d = idx % HD;
        float mn = kNegBig;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) mn = fmaxf(mn, s_acc[w][g][HD]);
        float lt = 0.f, at = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const float c = exp2f(s_acc[w][g][HD] - mn);
            lt += s_acc[w][g][HD + 1] * c;
            at += s_acc[w][g][d] * c;
        }
        const int64_t head = (int64_t)b * nh + kvh * Gv + g;
        if (nsplit == 1) {
            out[head * HD + d] = T::from_f32(lt > 0.f ? at / lt : 0.f);
        } else {
            float* dst = partial + (head * nsplit + sp) * (HD + 2);
            dst[d] = at;
            if (d == 0) {
                dst[HD] = mn;
                dst[HD + 1] = lt;
            }
        }
    }
}

// Merge of the context splits: one workgroup of HD threads per (sequence, query head).
// MOST: at least their number (31 sequences x 64 heads of two parts: the whole call 29.3 us with four parts' values in registers, 30.5 with 16).
template <typename T, int HD, int MOST>
__global__ __launch_bounds__(HD) void paged_attn_merge_kernel(const float* __restrict__ partial,
                                                              const int32_t* __restrict__ context_lens, uint16_t* __restrict__ out,
                                                              Splits splits, int heads, int tiled) {
    const int b = blockIdx.x / heads, d = threadIdx.x, nsplit = splits.of(context_lens[b]);
    const float* src = partial + (int64_t)blockIdx.x * splits.most * (HD + 2);
    // every part's values are asked for before the first is used: one trip to memory whatever their number
    float m[MOST], l[MOST], v[MOST];
#pragma unroll
    for (int s = 0; s < MOST; ++s) {
        const float* p = src + (s < splits.most ? s : 0) * (HD + 2);
        m[s] = p[HD], l[s] = p[HD + 1], v[s] = p[d];
    }
    if (nsplit == 1) return;        // that workgroup has written the result
    float mn = kNegBig;
#pragma unroll
    for (int s = 0; s < MOST; ++s) mn = s < nsplit ? fmaxf(mn, m[s]) : mn;
    float lt = 0.f, at = 0.f;
#pragma unroll
    for (int s = 0; s < MOST; ++s) {
        const float c = exp2f(m[s] - mn);
        lt = s < nsplit ? lt + l[s] * c : lt;
        at = s < nsplit ? at + v[s] * c : at;
    }
    const int64_t at_row = (int64_t)blockIdx.x * HD + d;
    out[tiled ? tiled_at(b, (int)(blockIdx.x % heads) * HD + d, heads * HD) / 2 : at_row] = T::from_f32(lt > 0.f ? at / lt : 0.f);
}

// ---------------------------------------------------------------------------------------------
// out[r, i] = SiLU(gate_up[r, i]) * gate_up[r, inter + i], SiLU rounded to the tensor type first.
// Greedy sampler: out[r] = index of the largest logits[r, :] (the lowest index among equal maxima; NaNs are never
// selected).  One workgroup of 16 waves per row, 16-byte loads.  The vector ALU of the row's CU bounds it, so a thread only
// keeps the largest of each eight logits and looks for its place at the end: 32 rows of 151936 7.9 us, of 32768 4.3; with every
// logit compared and its place kept 15.5 and 5.9.
template <typename T>
__global__ __launch_bounds__(1024) void argmax_rows_kernel(const uint16_t* __restrict__ logits,
                                                           int64_t* __restrict__ out, int vocab) {
    const uint16_t* row = logits + (size_t)blockIdx.x * vocab;
    float best = -__builtin_inff();
    int bi = 0x7fffffff;
    auto take = [&](float f, int idx) {
        if (f > best || (f == best && idx < bi)) {
            best = f;
            bi = idx;
        }
    };
    const int nvec = (vocab & 7) == 0 ? vocab >> 3 : 0;   // rows are 16-byte aligned only then
    int bv = -1;                                          // the first of the thread's vectors that holds `best`
    for (int v0 = threadIdx.x; v0 < nvec; v0 += 4 * 1024) {
        u32x4 d[4];   // four loads in flight
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int v = v0 + u * 1024;
            d[u] = *reinterpret_cast<const u32x4*>(row + (size_t)(v < nvec ? v : v0) * 8);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int v = v0 + u * 1024;
            float f[8];
            unpack8<T>(d[u], f);
            const float m = fmaxf(fmaxf(fmaxf(f[0], f[1]), fmaxf(f[2], f[3])), fmaxf(fmaxf(f[4], f[5]), fmaxf(f[6], f[7])));
            if (v < nvec && (m > best || (bv < 0 && m == best))) {
                best = m;
                bv = v;
            }
        }
    }
    if (bv >= 0) {
        float f[8];
        unpack8<T>(*reinterpret_cast<const u32x4*>(row + (size_t)bv * 8), f);
#pragma unroll
        for (int i = 7; i >= 0; --i)
            if (f[i] == best) bi = bv * 8 + i;
    }
    for (int i = nvec * 8 + threadIdx.x; i < vocab; i += 1024) take(T::to_f32(row[i]), i);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) take(__shfl_xor(best, off), __shfl_xor(bi, off));
    __shared__ float s_best[16];
    __shared__ int s_idx[16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) {
        s_best[wave] = best;
        s_idx[wave] = bi;
    }
    __syncthreads();
    if (wave == 0) {
        best = lane < 16 ? s_best[lane] : -__builtin_inff();
        bi = lane < 16 ? s_idx[lane] : 0x7fffffff;
#pragma unroll
        for (int off = 8; off >= 1; off >>= 1) take(__shfl_xor(best, off), __shfl_xor(bi, off));
        if (lane == 0) out[blockIdx.x] = bi == 0x7fffffff ? 0 : bi;
    }
}

// Words of eight columns: word i of row r of gate and of up lies row_stride r + word_stride i elements from their starts.
template <typename T>
__global__ __launch_bounds__(256) void silu_mul_kernel(const uint16_t* __restrict__ gate, const uint16_t* __restrict__ up,
                                                       uint16_t* __restrict__ out, int64_t rows, int words, int64_t row_stride,
                                                       int word_stride) {
    const int64_t vec = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (vec >= rows * words) return;
    const int64_t at = vec / words * row_stride + vec % words * word_stride;
    float g[8], u[8], o[8];
    unpack8<T>(*reinterpret_cast<const u32x4*>(gate + at), g);
    unpack8<T>(*reinterpret_cast<const u32x4*>(up + at), u);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = round_to<T>(g[e] / (1.f + __expf(-g[e]))) * u[e];
    *reinterpret_cast<u32x4*>(out + vec * 8) = pack8<T>(o);
}

int bad(const char* fn, const char* what) {
    set_error("%s: %s", fn, what);
    return AWQ_ERR_INVALID_ARG;
}
bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// The kernel with both products on the matrix cores takes 128 head dims and block sizes that are multiples of 16; it
// is used at 8 query heads per kv head, where the vector-ALU value product of the other kernels costs the most
// (bf16, against them: 128 sequences x 8 kv heads x 1024 tokens 120 -> 102 us, 32 x 8 x 512 23.2 -> 19.9, 1 x 8 x 8000
// 31.7 -> 24.6, 64 x 8 x 2060 the same 102 us = 5.3 TB/s; at 4 and 2 heads per kv head it measured equal or slower:
// 16 x 8 x 4000 at 4 heads 52.6 -> 55.0 us, the Qwen3-0.6B decode step 1.615 -> 1.673 ms).
// Head ratios other than 1, 2, 4 and 8 (up to 16) have no other kernel and take it as well.
bool attn_tr(int G, int64_t head_dim, int64_t block_size) {
    return (G == 8 || (G != 1 && G != 2 && G != 4 && G >= 1 && G <= 16)) && head_dim == 128 && block_size % 16 == 0;
}
// the vector kernel's waves, and those of the kernel with both products on the matrix cores (two and four heads on the matrix cores: launch_attn)
int attn_waves(int G, bool tr) { return tr ? 4 : (G <= 2 ? 16 : (G <= 4 ? 8 : 4)); }

// Context splits of a (sequence, kv head) pair. A launch lasts as long as the CU with the most workgroups, each of its workgroups costs what 250 tokens
// cost beside the tokens of its split, and the merge what 400 do: the split count with the smallest such sum. Over batches of 1 to 31, contexts of 140 to
// 8000 tokens and two or four heads per kv head (8 kv heads, bf16) it is 0.3 % from the best of eight counts on average. 256 pairs or more are not split.
// The host knows the table's length and not the contexts.  Several rounds of workgroups pay near that length alone, so that sequences shorter
// than where the sums meet keep to one round (four heads, 24 sequences with a table of 4096 tokens, at 64 / 300 / 900 / 4000 tokens: four splits, three
// rounds, 15.5, 20.2, 29.9, 76 us; two, as a rule of waves on the chip has it, 10.0, 14.4, 26.3, 87; now 8.2, 11.4, 22.7, 75).
// Four-wave workgroups (eight heads per kv head, with or without the matrix cores) run best at about 2048 waves on the chip with 128 tokens or more per
// split (64 sequences x 8 kv heads x 2060 tokens at 8 heads per kv head 124 us in two splits + merge, 105 unsplit).
Splits pick_splits(int64_t batch, int64_t nkv, int64_t max_context, int G, bool tr) {
    const int64_t pairs = batch * nkv, waves = attn_waves(G, tr);
    if (waves == 4) {
        const int64_t s = cdiv(2048, pairs * waves), cap = max_context / 128 > 1 ? max_context / 128 : 1;
        const int64_t m = s < cap ? s : cap;
        const int n = (int)(m > kMaxSplits ? kMaxSplits : (m < 1 ? 1 : m));
        return Splits{(int)pairs, n, n, 0};
    }
    int best = 1;
    if (pairs < 256) {
        int64_t least = 250 + max_context;
        for (int s = 2; s <= kMaxSplits && (int64_t)s * 64 <= max_context; ++s) {
            const int64_t cost = cdiv(pairs * s, 256) * (250 + cdiv(max_context, s)) + 400;
            if (cost < least) least = cost, best = s;
        }
    }
    const int one = (int)std::max<int64_t>(1, std::min<int64_t>(best, 256 / pairs));
    if (one == best) return Splits{(int)pairs, best, best, 0};
    const double rounds = (double)cdiv(pairs * best, 256), gain = 1.0 / one - rounds / best;     // a token
    const double from = gain > 0 ? ((rounds - 1) * 250 + (one == 1 ? 400 : 0)) / gain : (double)max_context;
    return Splits{(int)pairs, best, one, (int)std::min(from + 1, (double)max_context)};
}

template <typename T, int HD>
void launch_merge(const float* partial, const int32_t* ctx, void* out, Splits splits, int64_t batch, int heads, int tiled, hipStream_t st) {
    if (splits.most == 1) return;
    const auto kernel = splits.most <= 4 ? paged_attn_merge_kernel<T, HD, 4> : paged_attn_merge_kernel<T, HD, kMaxSplits>;
    kernel<<<dim3((unsigned)(batch * heads)), dim3(HD), 0, st>>>(partial, ctx, (uint16_t*)out, splits, heads, tiled);
}

template <typename T, int G, int HD>
void launch_attn(const void* q, const void* kc, const void* vc, const int32_t* table, const int32_t* ctx, void* out,
                 float* partial, int64_t batch, int nkv, int bs, int max_blocks, int num_blocks, Splits splits,
                 float scale, int tiled, hipStream_t st) {
    constexpr int WAVES = G <= 2 ? 16 : (G <= 4 ? 8 : 4);
    if constexpr (HD == 128 && G == 8) {
        if (attn_tr(G, HD, bs)) {
            paged_attn_decode_tr_kernel<T, G, 4><<<dim3((unsigned)(batch * nkv * splits.most)), dim3(256), 0, st>>>(
                (const uint16_t*)q, (const uint16_t*)kc, (const uint16_t*)vc, table, ctx, (uint16_t*)out, partial, nkv,
                bs, max_blocks, num_blocks, splits.most, scale, G);
            launch_merge<T, HD>(partial, ctx, out, splits, batch, nkv * G, 0, st);
            return;
        }
    }
    if constexpr (HD == 128 && (G == 2 || G == 4)) {
        if (bs % 16 == 0) {
            // a CU holds one workgroup of eight waves or, where there are more than CUs, several of four, whose last round is shorter (two heads, 40 x
            // 640 tokens 23.9 us, 26.2 with eight; four heads, 64 x 640 29.5, 32.5; 24 x 640 14.9, 17.1 with four)
            const int64_t groups = batch * nkv * splits.most;
            const auto fills = [](int64_t n) { return n * 4 >= cdiv(n, 256) * 256 * 3; };
            const int full = fills(groups) | fills(batch * nkv * splits.few) << 1;
            const auto go = [&](auto waves) {
                constexpr int W = decltype(waves)::value;
                paged_attn_decode_mfma_kernel<T, G, W><<<dim3((unsigned)groups), dim3(64 * W), 0, st>>>(
                    (const uint16_t*)q, (const uint16_t*)kc, (const uint16_t*)vc, table, ctx, (uint16_t*)out, partial, nkv, bs, max_blocks,
                    num_blocks, splits, scale, tiled, full);
            };
            if (batch * nkv > 256) go(std::integral_constant<int, 4>{});
            else go(std::integral_constant<int, 8>{});
            launch_merge<T, HD>(partial, ctx, out, splits, batch, nkv * G, tiled, st);
            return;
        }
    }
    paged_attn_decode_kernel<T, G, HD, WAVES><<<dim3((unsigned)(batch * nkv * splits.most)), dim3(64 * WAVES), 0, st>>>(
        (const uint16_t*)q, (const uint16_t*)kc, (const uint16_t*)vc, table, ctx, (uint16_t*)out, partial, nkv, bs,
        max_blocks, num_blocks, splits, scale, tiled);
    launch_merge<T, HD>(partial, ctx, out, splits, batch, nkv * G, tiled, st);
}

template <typename T, int HD>
int launch_attn_g(int G, const void* q, const void* kc, const void* vc, const int32_t* table, const int32_t* ctx,
                  void* out, float* partial, int64_t batch, int nkv, int bs, int max_blocks, int num_blocks,
                  Splits splits, float scale, int tiled, hipStream_t st) {
    switch (G) {
#define NQ_CASE(g)                                                                                              \
    case g:                                                                                                     \
        launch_attn<T, g, HD>(q, kc, vc, table, ctx, out, partial, batch, nkv, bs, max_blocks, num_blocks,      \
                              splits, scale, tiled, st);                                                        \
        return AWQ_OK;
        NQ_CASE(1) NQ_CASE(2) NQ_CASE(4) NQ_CASE(8)
#undef NQ_CASE
    }
    if constexpr (HD == 128) {
        if (attn_tr(G, HD, bs)) {   // any other ratio up to 16: the matrix-core kernel with the count at run time
            paged_attn_decode_tr_kernel<T, 0, 4><<<dim3((unsigned)(batch * nkv * splits.most)), dim3(256), 0, st>>>(
                (const uint16_t*)q, (const uint16_t*)kc, (const uint16_t*)vc, table, ctx, (uint16_t*)out, partial, nkv,
                bs, max_blocks, num_blocks, splits.most, scale, G);
            launch_merge<T, HD>(partial, ctx, out, splits, batch, nkv * G, 0, st);
            return AWQ_OK;
        }
    }
    set_error("nq_paged_attention_decode: query heads per kv head must be 1, 2, 4 or 8 (or, with head_dim 128 and a "
              "block size that is a multiple of 16, any count up to 16), got %d", G);
    return AWQ_ERR_UNSUPPORTED;
}

}  // namespace
}  // namespace awq

using namespace awq;

extern "C" int nq_add_rmsnorm(void* residual, const void* delta, const void* weight, void* y, int64_t rows,
                              int64_t hidden, float eps, int dtype, void* stream) {
    const char* fn = "nq_add_rmsnorm";
    if (!residual || !weight || !y) return bad(fn, "null pointer argument");
    if (!aligned16(residual) || !aligned16(weight) || !aligned16(y) || !aligned16(delta))
        return bad(fn, "every tensor must be 16-byte aligned");
    if (dtype != AWQ_F16 && dtype != AWQ_BF16) return bad(fn, "dtype must be AWQ_F16 or AWQ_BF16");
    if (rows <= 0 || hidden <= 0 || hidden % 8 != 0) return bad(fn, "rows > 0 and hidden a positive multiple of 8");
    if (hidden > kNormThreads * 8 * kNormPasses || rows > 0x7fffffff) {
        set_error("%s: hidden=%lld exceeds %d", fn, (long long)hidden, kNormThreads * 8 * kNormPasses);
        return AWQ_ERR_UNSUPPORTED;
    }
    hipStream_t st = (hipStream_t)stream;
    (void)hipGetLastError();
    // a wave a row from 1024 rows on (256 workgroups), longer rows than 2560 from 2048 on (1500 x 4096 8.0 us with a workgroup each, 8.8 with
    // a wave; 2048 rows 10.2 and 10.1, x 3072 9.1 and 8.5); with a delta those beyond 1024 are as well or better off with a workgroup each (8192 x 2048 25.7 us
    // there, 29.6 with a wave)
    if (rows >= (hidden <= 2560 ? 1024 : 2048) && hidden <= (delta ? 1024 : 4096)) {
        const auto go = [&](auto kernel) {
            kernel<<<dim3((unsigned)cdiv(rows, 4)), dim3(256), 0, st>>>((uint16_t*)residual, (const uint16_t*)delta, (const uint16_t*)weight,
                                                                        (uint16_t*)y, rows, (int)hidden, eps);
        };
        const auto passes = [&](auto p) {
            constexpr int P = decltype(p)::value;
            dtype == AWQ_F16 ? go(add_rmsnorm_rows_kernel<F16, P>) : go(add_rmsnorm_rows_kernel<BF16, P>);
        };
        if (hidden <= 512) passes(std::integral_constant<int, 1>{});
        else if (hidden <= 1024) passes(std::integral_constant<int, 2>{});
        else if (hidden <= 2048) passes(std::integral_constant<int, 4>{});
        else if (hidden <= 2560) passes(std::integral_constant<int, 5>{});
        else passes(std::integral_constant<int, 8>{});
    } else if (dtype == AWQ_F16)
        add_rmsnorm_kernel<F16><<<dim3((unsigned)rows), dim3(kNormThreads), 0, st>>>(
            (uint16_t*)residual, (const uint16_t*)delta, (const uint16_t*)weight, (uint16_t*)y, (int)hidden, eps);
    else
        add_rmsnorm_kernel<BF16><<<dim3((unsigned)rows), dim3(kNormThreads), 0, st>>>(
            (uint16_t*)residual, (const uint16_t*)delta, (const uint16_t*)weight, (uint16_t*)y, (int)hidden, eps);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? AWQ_OK : hip_fail(fn, e);
}

static int row_ssq_entry(const char* fn, const void* x, float* ssq, int64_t rows, int64_t hidden, const int64_t* ids,
                         int64_t table_rows, void* x_out, int dtype, void* stream);

extern "C" int nq_row_ssq(const void* x, float* ssq, int64_t rows, int64_t hidden, int dtype, void* stream) {
    return row_ssq_entry("nq_row_ssq", x, ssq, rows, hidden, nullptr, 0, nullptr, dtype, stream);
}

extern "C" int nq_embed_row_ssq(const int64_t* ids, const void* table, void* x_out, float* ssq, int64_t rows,
                                int64_t hidden, int64_t table_rows, int dtype, void* stream) {
    const char* fn = "nq_embed_row_ssq";
    if (!ids || !x_out) return bad(fn, "null pointer argument");
    if (!aligned16(x_out)) return bad(fn, "x_out must be 16-byte aligned");
    if (table_rows <= 0) return bad(fn, "table_rows must be positive");
    return row_ssq_entry(fn, table, ssq, rows, hidden, ids, table_rows, x_out, dtype, stream);
}

static int row_ssq_entry(const char* fn, const void* x, float* ssq, int64_t rows, int64_t hidden, const int64_t* ids,
                         int64_t table_rows, void* x_out, int dtype, void* stream) {
    if (!x || !ssq) return bad(fn, "null pointer argument");
    if (!aligned16(x) || (reinterpret_cast<uintptr_t>(ssq) & 3u)) return bad(fn, "x must be 16-byte, ssq 4-byte aligned");
    if (dtype != AWQ_F16 && dtype != AWQ_BF16) return bad(fn, "dtype must be AWQ_F16 or AWQ_BF16");
    if (rows <= 0 || hidden <= 0 || hidden % 8 != 0) return bad(fn, "rows > 0 and hidden a positive multiple of 8");
    if (hidden > kNormThreads * 8 * kNormPasses || rows > 0x7fffffff) {
        set_error("%s: hidden=%lld exceeds %d", fn, (long long)hidden, kNormThreads * 8 * kNormPasses);
        return AWQ_ERR_UNSUPPORTED;
    }
    hipStream_t st = (hipStream_t)stream;
    (void)hipGetLastError();
    if (dtype == AWQ_F16)
        row_ssq_kernel<F16><<<dim3((unsigned)rows), dim3(kNormThreads), 0, st>>>((const uint16_t*)x, ssq, (int)rows, (int)hidden,
                                                                                ids, table_rows, (uint16_t*)x_out);
    else
        row_ssq_kernel<BF16><<<dim3((unsigned)rows), dim3(kNormThreads), 0, st>>>((const uint16_t*)x, ssq, (int)rows, (int)hidden,
                                                                                 ids, table_rows, (uint16_t*)x_out);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? AWQ_OK : hip_fail(fn, e);
}

extern "C" int nq_qk_norm_rope_store(const void* qkv, const void* q_weight, const void* k_weight, const float* cos_sin,
                                     const int64_t* positions, const int64_t* slots, void* q_out, void* k_out,
                                     void* k_cache, void* v_cache, int64_t rows, int64_t num_heads, int64_t num_kv_heads,
                                     int64_t head_dim, int64_t max_positions, int64_t num_slots, int64_t block_size,
                                     float eps, int dtype, void* stream) {
    const char* fn = "nq_qk_norm_rope_store";
    if (!qkv || !q_weight || !k_weight || !cos_sin || !positions || !slots || !q_out || !k_cache || !v_cache)
        return bad(fn, "null pointer argument");
    if (dtype != AWQ_F16 && dtype != AWQ_BF16) return bad(fn, "dtype must be AWQ_F16 or AWQ_BF16");
    if (rows <= 0 || num_heads <= 0 || num_kv_heads <= 0 || max_positions <= 0 || num_slots <= 0 || block_size <= 0 ||
        block_size > 0x7fffffff || num_slots % block_size != 0)
        return bad(fn, "rows, head counts, max_positions, block_size must be positive and num_slots a multiple of block_size");
    if (head_dim <= 0 || head_dim % 2 != 0 || head_dim > 128 * kMaxPairs) {
        set_error("%s: head_dim must be even and at most %d, got %lld", fn, 128 * kMaxPairs, (long long)head_dim);
        return AWQ_ERR_UNSUPPORTED;
    }
    const int64_t items = rows * (num_heads + 2 * num_kv_heads);
    if (items > ((int64_t)1 << 32)) return bad(fn, "too many rows");
    hipStream_t st = (hipStream_t)stream;
    (void)hipGetLastError();
    const bool vec = (head_dim == 64 || head_dim == 128 || head_dim == 256) && aligned16(qkv) && aligned16(q_weight) &&
                     aligned16(k_weight) && aligned16(cos_sin) && aligned16(q_out) && aligned16(k_out) &&
                     aligned16(k_cache) && aligned16(v_cache);
    if (vec) {
#define NQ_ROPE_VEC(TT, HH)                                                                                          \
    qk_norm_rope_store_vec_kernel<TT, HH><<<dim3((unsigned)cdiv(items, 4 * (64 / (HH / 8)))), dim3(256), 0, st>>>(  \
        (const uint16_t*)qkv, (const uint16_t*)q_weight, (const uint16_t*)k_weight, cos_sin, positions, slots,      \
        (uint16_t*)q_out, (uint16_t*)k_out, (uint16_t*)k_cache, (uint16_t*)v_cache, (int)rows, (int)num_heads,       \
        (int)num_kv_heads, (int)max_positions, num_slots, (int)block_size, eps)
        if (dtype == AWQ_F16) {
            if (head_dim == 64) NQ_ROPE_VEC(F16, 64);
            else if (head_dim == 128) NQ_ROPE_VEC(F16, 128);
            else NQ_ROPE_VEC(F16, 256);
        } else {
            if (head_dim == 64) NQ_ROPE_VEC(BF16, 64);
            else if (head_dim == 128) NQ_ROPE_VEC(BF16, 128);
            else NQ_ROPE_VEC(BF16, 256);
        }
#undef NQ_ROPE_VEC
        const hipError_t ev = hipGetLastError();
        return ev == hipSuccess ? AWQ_OK : hip_fail(fn, ev);
    }
    const dim3 grid((unsigned)cdiv(items, 4)), block(256);
    if (dtype == AWQ_F16)
        qk_norm_rope_store_kernel<F16><<<grid, block, 0, st>>>(
            (const uint16_t*)qkv, (const uint16_t*)q_weight, (const uint16_t*)k_weight, cos_sin, positions, slots,
            (uint16_t*)q_out, (uint16_t*)k_out, (uint16_t*)k_cache, (uint16_t*)v_cache, (int)rows, (int)num_heads,
            (int)num_kv_heads,
            (int)head_dim, (int)max_positions, num_slots, (int)block_size, eps);
    else
        qk_norm_rope_store_kernel<BF16><<<grid, block, 0, st>>>(
            (const uint16_t*)qkv, (const uint16_t*)q_weight, (const uint16_t*)k_weight, cos_sin, positions, slots,
            (uint16_t*)q_out, (uint16_t*)k_out, (uint16_t*)k_cache, (uint16_t*)v_cache, (int)rows, (int)num_heads,
            (int)num_kv_heads,
            (int)head_dim, (int)max_positions, num_slots, (int)block_size, eps);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? AWQ_OK : hip_fail(fn, e);
}

extern "C" size_t nq_paged_attention_workspace_bytes(int64_t batch, int64_t num_heads, int64_t num_kv_heads,
                                                     int64_t head_dim, int64_t max_context) {
    if (batch <= 0 || num_heads <= 0 || num_kv_heads <= 0 || head_dim <= 0 || max_context <= 0) return 0;
    // the block size decides the kernel and with it the split count: room for either
    const int G = (int)(num_heads / num_kv_heads);
    int s = pick_splits(batch, num_kv_heads, max_context, G, false).most;
    if (attn_tr(G, head_dim, 32)) s = std::max(s, pick_splits(batch, num_kv_heads, max_context, G, true).most);
    return s > 1 ? (size_t)(batch * num_heads * s * (head_dim + 2)) * sizeof(float) : 0;
}

static int paged_attention_decode(const char* fn, const void* q, const void* k_cache, const void* v_cache, const int32_t* block_table,
                                  const int32_t* context_lens, void* out, int64_t batch, int64_t num_heads, int64_t num_kv_heads,
                                  int64_t head_dim, int64_t block_size, int64_t max_blocks_per_seq, int64_t num_blocks, float scale, int dtype,
                                  int tiled, void* workspace, size_t workspace_bytes, void* stream) {
    if (!q || !k_cache || !v_cache || !block_table || !context_lens || !out) return bad(fn, "null pointer argument");
    if (!aligned16(q) || !aligned16(k_cache) || !aligned16(v_cache) || !aligned16(out))
        return bad(fn, "q, caches and out must be 16-byte aligned");
    if (dtype != AWQ_F16 && dtype != AWQ_BF16) return bad(fn, "dtype must be AWQ_F16 or AWQ_BF16");
    if (batch <= 0 || num_heads <= 0 || num_kv_heads <= 0 || block_size <= 0 || max_blocks_per_seq <= 0 ||
        num_blocks <= 0 || num_heads % num_kv_heads != 0)
        return bad(fn, "sizes must be positive and num_heads a multiple of num_kv_heads");
    if (head_dim != 64 && head_dim != 128) {
        set_error("%s: head_dim must be 64 or 128, got %lld", fn, (long long)head_dim);
        return AWQ_ERR_UNSUPPORTED;
    }
    const int64_t max_context = block_size * max_blocks_per_seq;
    if (max_context > 0x7fffffff || num_blocks * block_size > 0x7fffffff || batch * num_kv_heads * 16 > 0x7fffffff)
        return bad(fn, "problem too large");
    const Splits splits = pick_splits(batch, num_kv_heads, max_context, (int)(num_heads / num_kv_heads),
                                   attn_tr((int)(num_heads / num_kv_heads), head_dim, block_size));
    const size_t need = splits.most > 1 ? (size_t)(batch * num_heads * splits.most * (head_dim + 2)) * sizeof(float) : 0;
    if (need && (!workspace || workspace_bytes < need || !aligned16(workspace))) {
        set_error("%s: workspace of %zu bytes needed, %zu given", fn, need, workspace ? workspace_bytes : (size_t)0);
        return AWQ_ERR_WORKSPACE;
    }
    hipStream_t st = (hipStream_t)stream;
    (void)hipGetLastError();
    const int G = (int)(num_heads / num_kv_heads);
    int rc;
    if (dtype == AWQ_F16)
        rc = head_dim == 128
                 ? launch_attn_g<F16, 128>(G, q, k_cache, v_cache, block_table, context_lens, out, (float*)workspace,
                                           batch, (int)num_kv_heads, (int)block_size, (int)max_blocks_per_seq,
                                           (int)num_blocks, splits, scale, tiled, st)
                 : launch_attn_g<F16, 64>(G, q, k_cache, v_cache, block_table, context_lens, out, (float*)workspace,
                                          batch, (int)num_kv_heads, (int)block_size, (int)max_blocks_per_seq,
                                          (int)num_blocks, splits, scale, tiled, st);
    else
        rc = head_dim == 128
                 ? launch_attn_g<BF16, 128>(G, q, k_cache, v_cache, block_table, context_lens, out, (float*)workspace,
                                            batch, (int)num_kv_heads, (int)block_size, (int)max_blocks_per_seq,
                                            (int)num_blocks, splits, scale, tiled, st)
                 : launch_attn_g<BF16, 64>(G, q, k_cache, v_cache, block_table, context_lens, out, (float*)workspace,
                                           batch, (int)num_kv_heads, (int)block_size, (int)max_blocks_per_seq,
                                           (int)num_blocks, splits, scale, tiled, st);
    if (rc != AWQ_OK) return rc;
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? AWQ_OK : hip_fail(fn, e);
}

extern "C" int nq_paged_attention_decode(const void* q, const void* k_cache, const void* v_cache,
                                         const int32_t* block_table, const int32_t* context_lens, void* out,
                                         int64_t batch, int64_t num_heads, int64_t num_kv_heads, int64_t head_dim,
                                         int64_t block_size, int64_t max_blocks_per_seq, int64_t num_blocks, float scale,
                                         int dtype, void* workspace, size_t workspace_bytes, void* stream) {
    return paged_attention_decode("nq_paged_attention_decode", q, k_cache, v_cache, block_table, context_lens, out, batch, num_heads, num_kv_heads,
                                  head_dim, block_size, max_blocks_per_seq, num_blocks, scale, dtype, 0, workspace, workspace_bytes, stream);
}

extern "C" int nq_paged_attention_decode_tiled(const void* q, const void* k_cache, const void* v_cache,
                                               const int32_t* block_table, const int32_t* context_lens, void* out,
                                               int64_t batch, int64_t num_heads, int64_t num_kv_heads, int64_t head_dim,
                                               int64_t block_size, int64_t max_blocks_per_seq, int64_t num_blocks, float scale,
                                               int dtype, void* workspace, size_t workspace_bytes, void* stream) {
    const char* fn = "nq_paged_attention_decode_tiled";
    if (head_dim != 128 || num_kv_heads <= 0 || (num_heads != num_kv_heads && num_heads != 2 * num_kv_heads)) {
        set_error("%s: head_dim 128, one or two query heads per kv head", fn);
        return AWQ_ERR_UNSUPPORTED;
    }
    return paged_attention_decode(fn, q, k_cache, v_cache, block_table, context_lens, out, batch, num_heads, num_kv_heads, head_dim, block_size,
                                  max_blocks_per_seq, num_blocks, scale, dtype, 1, workspace, workspace_bytes, stream);
}

extern "C" int nq_argmax_rows(const void* logits, int64_t* out, int64_t rows, int64_t vocab, int dtype,
                              void* stream) {
    const char* fn = "nq_argmax_rows";
    if (!logits || !out) return bad(fn, "null pointer argument");
    if (!aligned16(logits)) return bad(fn, "logits must be 16-byte aligned");
    if (dtype != AWQ_F16 && dtype != AWQ_BF16) return bad(fn, "dtype must be AWQ_F16 or AWQ_BF16");
    if (rows <= 0 || vocab <= 0 || rows > 0x7fffffff || vocab > 0x7ffffff0) return bad(fn, "rows and vocab must be positive 31-bit counts");
    hipStream_t st = (hipStream_t)stream;
    (void)hipGetLastError();
    if (dtype == AWQ_F16)
        argmax_rows_kernel<F16><<<dim3((unsigned)rows), dim3(1024), 0, st>>>((const uint16_t*)logits, out, (int)vocab);
    else
        argmax_rows_kernel<BF16><<<dim3((unsigned)rows), dim3(1024), 0, st>>>((const uint16_t*)logits, out, (int)vocab);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? AWQ_OK : hip_fail(fn, e);
}

extern "C" int nq_decode_prepare(const int64_t* positions, const uint8_t* active, const int32_t* block_table,
                                 int64_t* slots, int32_t* context_lens, int64_t rows, int64_t max_blocks,
                                 int64_t block_size, void* stream) {
    const char* fn = "nq_decode_prepare";
    if (!positions || !active || !block_table || !slots || !context_lens) return bad(fn, "null pointer argument");
    if (rows <= 0 || max_blocks <= 0 || block_size <= 0 || rows > 0x7fffffff || max_blocks > 0x7fffffff ||
        block_size > 0x7fffffff)
        return bad(fn, "rows, max_blocks and block_size must be positive 31-bit counts");
    (void)hipGetLastError();
    decode_prepare_kernel<<<dim3((unsigned)cdiv(rows, 256)), dim3(256), 0, (hipStream_t)stream>>>(
        positions, active, block_table, slots, context_lens, (int)rows, (int)max_blocks, (int)block_size);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? AWQ_OK : hip_fail(fn, e);
}

extern "C" int nq_decode_advance(const int64_t* next_tokens, const uint8_t* active, int64_t* out_log, int64_t* ids,
                                 int64_t* positions, int64_t* step, int64_t rows, int64_t out_rows, void* stream) {
    const char* fn = "nq_decode_advance";
    if (!next_tokens || !active || !out_log || !ids || !positions || !step) return bad(fn, "null pointer argument");
    if (rows <= 0 || rows > 0x7fffffff || out_rows <= 0) return bad(fn, "rows and out_rows must be positive");
    (void)hipGetLastError();
    decode_advance_kernel<<<dim3(1), dim3(1024), 0, (hipStream_t)stream>>>(next_tokens, active, out_log, ids, positions,
                                                                         step, (int)rows, out_rows);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? AWQ_OK : hip_fail(fn, e);
}

static int silu_mul_entry(const char* fn, const void* gate, const void* up, void* out, int64_t rows, int64_t inter,
                          int64_t row_stride, int word_stride, int dtype, void* stream) {
    if (!gate || !up || !out) return bad(fn, "null pointer argument");
    if (!aligned16(gate) || !aligned16(up) || !aligned16(out)) return bad(fn, "tensors must be 16-byte aligned");
    if (dtype != AWQ_F16 && dtype != AWQ_BF16) return bad(fn, "dtype must be AWQ_F16 or AWQ_BF16");
    if (rows <= 0 || inter <= 0 || inter % 8 != 0) return bad(fn, "rows > 0 and inter a positive multiple of 8");
    const int64_t vecs = rows * (inter / 8);
    if (cdiv(vecs, 256) > 0x7fffffff || inter > 0x3fffffff) return bad(fn, "problem too large");
    hipStream_t st = (hipStream_t)stream;
    (void)hipGetLastError();
    const dim3 grid((unsigned)cdiv(vecs, 256)), block(256);
    if (dtype == AWQ_F16)
        silu_mul_kernel<F16><<<grid, block, 0, st>>>((const uint16_t*)gate, (const uint16_t*)up, (uint16_t*)out, rows,
                                                     (int)(inter / 8), row_stride, word_stride);
    else
        silu_mul_kernel<BF16><<<grid, block, 0, st>>>((const uint16_t*)gate, (const uint16_t*)up, (uint16_t*)out, rows,
                                                      (int)(inter / 8), row_stride, word_stride);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? AWQ_OK : hip_fail(fn, e);
}

extern "C" int nq_silu_mul(const void* gate_up, void* out, int64_t rows, int64_t inter, int dtype, void* stream) {
    return silu_mul_entry("nq_silu_mul", gate_up, (const uint16_t*)gate_up + (inter > 0 ? inter : 0), out, rows, inter, 2 * inter, 8,
                          dtype, stream);
}

extern "C" int nq_silu_mul_interleaved(const void* gate_up, void* out, int64_t rows, int64_t inter, int dtype,
                                       void* stream) {
    return silu_mul_entry("nq_silu_mul_interleaved", gate_up, (const uint16_t*)gate_up + 8, out, rows, inter, 2 * inter, 16, dtype,
                          stream);
}

extern "C" int nq_silu_mul_pair(const void* gate, const void* up, void* out, int64_t rows, int64_t inter, int dtype,
                                void* stream) {
    return silu_mul_entry("nq_silu_mul_pair", gate, up, out, rows, inter, inter, 8, dtype, stream);
}

extern "C" int nq_qkv_norm_rope(const void* q, const void* k, const void* v, const void* q_weight, const void* k_weight,
                                const float* cos_sin, const int64_t* positions, int per_sequence, void* q_out, void* k_out,
                                void* v_out, int64_t batch, int64_t tokens, int64_t num_heads, int64_t num_kv_heads,
                                int64_t head_dim, int64_t max_positions, float q_eps, float k_eps, int dtype, void* stream) {
    const char* fn = "nq_qkv_norm_rope";
    if (!q || !k || !v || !q_weight || !k_weight || !cos_sin || !positions || !q_out || !k_out || !v_out)
        return bad(fn, "null pointer argument");
    for (const void* p : {q, k, v, q_weight, k_weight, (const void*)cos_sin, (const void*)q_out, (const void*)k_out, (const void*)v_out})
        if (!aligned16(p)) return bad(fn, "every tensor must be 16-byte aligned");
    if (dtype != AWQ_F16 && dtype != AWQ_BF16) return bad(fn, "dtype must be AWQ_F16 or AWQ_BF16");
    if (batch <= 0 || tokens <= 0 || num_heads <= 0 || num_kv_heads <= 0 || max_positions <= 0 || tokens > 0x7fffffff ||
        num_heads + 2 * num_kv_heads > 0x7fffffff)
        return bad(fn, "sizes must be positive 31-bit counts");
    if (head_dim != 64 && head_dim != 128 && head_dim != 256) {
        set_error("%s: head_dim must be 64, 128 or 256, got %lld", fn, (long long)head_dim);
        return AWQ_ERR_UNSUPPORTED;
    }
    const int64_t items = batch * tokens * (num_heads + 2 * num_kv_heads);
    if (cdiv(items, 4 * (512 / head_dim)) > 0x7fffffff) return bad(fn, "problem too large");
    // Two heads a group of lanes and pass, passes of up to 512 lanes equally full.  One head, and not two behind one another, where a wave has lanes for all
    // of them (then with several tokens or sequences a workgroup: 8192 x 1 token of 4 + 1 + 1 heads of 64 6.6 us, 8.6 with two heads in a
    // wave of its own) and where the launch has fewer waves than the chip holds at a time (then over several workgroups of 128 lanes: 64 tokens of
    // 16 + 8 + 8 heads of 128 3.6 us, of 64 + 8 + 8 3.9; 4.1 and 5.3).
    const int64_t heads = num_heads + 2 * num_kv_heads, each = head_dim / 8;
    const bool few = heads * each <= 64, small = !few && batch * tokens * heads * each <= 2048 * 64;
    const int64_t parts = cdiv(heads, 2), passes = cdiv(parts * each, 512);
    const int64_t lanes = few ? heads * each : small ? 128 : cdiv(cdiv(parts, passes) * each, 64) * 64, shares = small ? cdiv(heads * each, lanes) : 1;
    const bool beside_tokens = few && tokens >= 256 / lanes;
    const int64_t tokens_beside = beside_tokens ? 256 / lanes : 1, sequences_beside = few && !beside_tokens ? std::min<int64_t>(batch, 256 / lanes) : 1;
    hipStream_t st = (hipStream_t)stream;
    (void)hipGetLastError();
    const auto go = [&](auto type, auto dim, auto wide) {
        using T = decltype(type);
        constexpr int HD = decltype(dim)::value, U = decltype(wide)::value;
        const int64_t most = 65535 * sequences_beside;
        for (int64_t b = 0; b < batch; b += most) {     // the grid's second dimension
            const int64_t some = std::min<int64_t>(batch - b, most), r = b * tokens;
            const auto at = [&](const void* x, int64_t heads) { return (uint16_t*)x + r * heads * HD; };
            qkv_norm_rope_kernel<T, HD, U><<<dim3((unsigned)cdiv(tokens, tokens_beside), (unsigned)cdiv(some, sequences_beside), (unsigned)shares),
                                             dim3((unsigned)lanes, (unsigned)(tokens_beside * sequences_beside)), 0, st>>>(
                at(q, num_heads), at(k, num_kv_heads), at(v, num_kv_heads), (const uint16_t*)q_weight, (const uint16_t*)k_weight, cos_sin,
                positions + (per_sequence ? r : 0), per_sequence != 0, at(q_out, num_heads), at(k_out, num_kv_heads), at(v_out, num_kv_heads),
                (int)some, (int)tokens, (int)num_heads, (int)num_kv_heads, beside_tokens, max_positions, q_eps, k_eps);
        }
    };
    const auto of = [&](auto type, auto wide) {
        if (head_dim == 64) go(type, std::integral_constant<int, 64>{}, wide);
        else if (head_dim == 128) go(type, std::integral_constant<int, 128>{}, wide);
        else go(type, std::integral_constant<int, 256>{}, wide);
    };
    const auto with = [&](auto wide) { dtype == AWQ_F16 ? of(F16{}, wide) : of(BF16{}, wide); };
    if (few || small) with(std::integral_constant<int, 1>{});
    else with(std::integral_constant<int, 2>{});
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? AWQ_OK : hip_fail(fn, e);
}
