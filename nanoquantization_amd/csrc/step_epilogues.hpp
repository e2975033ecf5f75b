// Epilogues of the decode step's linears that several kernels share: q/k norm, rotary and cache write behind q|k|v, and
// SiLU(gate) * up.
#pragma once

#include "awq_common.hpp"

namespace awq {

// Byte offset of column k of a row in the input layout of nq_block_step's linears: pieces of 1 KiB (16 rows x 32 columns) in the order of the
// matrix instruction's operand.
__host__ __device__ __forceinline__ constexpr uint32_t tiled_at(int row, int k, int width) {
    return (uint32_t)(((row >> 4) * (width >> 5) + (k >> 5)) * 1024 + ((k >> 3 & 3) * 16 + (row & 15)) * 16 + (k & 7) * 2);
}

// Epilogue of the fused q|k|v projection of a decode step (act == 2): the 128 columns of a column tile are one
// head (head_dim 128).  q and k heads: RMSNorm over the head, half-split rotary at the row's position; q goes
// to q_out, k to its paged-cache slot; v heads are written to their cache slot as they are.  The arithmetic per
// element is that of the stand-alone kernel behind nq_qk_norm_rope_store (the GEMV's fp32 sum is rounded to T first,
// as a separate projection would round it).  Cache layout [blocks][kv heads][block_size][128].
struct QkvEpilogue {
    const uint16_t* q_weight;
    const uint16_t* k_weight;
    const float* cos_sin;        // [max_positions][128]: 64 cosines, then 64 sines
    const int64_t* positions;    // [M]
    const int64_t* slots;        // [M], negative = the row owns no cache slot
    uint16_t* q_out;             // [M][nh][128]
    uint16_t* k_cache;
    uint16_t* v_cache;
    int nh, nkv, max_positions, block_size;
    int64_t num_slots;
    float eps;
};

// The 16 lanes that hold the 16 words of (row m, head n0 / 128) call this together; `valid` masks the stores.
template <typename T>
__device__ __forceinline__ void qkv_rope_store(const float (&out)[8], int m, size_t n0, bool valid,
                                               const QkvEpilogue& qe) {
    const int head = (int)(n0 >> 7), dc = (int)((n0 & 127) >> 3);
    const int row = valid ? m : 0;
    float a[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) a[e] = T::to_f32(T::from_f32(out[e]));
    const int64_t slot = qe.slots[row];
    const bool slot_ok = slot >= 0 && slot < qe.num_slots;
    const bool is_q = head < qe.nh, is_k = !is_q && head < qe.nh + qe.nkv;
    if (!is_q && !is_k) {   // v (uniform over the 16 lanes: no shuffle below is reached by a partial group)
        if (valid && slot_ok) {
            u32x4 o;
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = T::pack2(a[2 * i], a[2 * i + 1]);
            *reinterpret_cast<u32x4*>(qe.v_cache + (((slot / qe.block_size) * qe.nkv + (head - qe.nh - qe.nkv)) *
                                                        qe.block_size + slot % qe.block_size) * 128 + dc * 8) = o;
        }
        return;
    }
    const uint16_t* w = is_q ? qe.q_weight : qe.k_weight;
    const u32x4 wraw = *reinterpret_cast<const u32x4*>(w + dc * 8);
    int64_t pos = qe.positions[row];
    pos = pos < 0 ? 0 : (pos >= qe.max_positions ? qe.max_positions - 1 : pos);
    const int i0 = (dc & 7) * 8;
    const float* cs = qe.cos_sin + pos * 128;
    const f32x4 c0 = *reinterpret_cast<const f32x4*>(cs + i0), c1 = *reinterpret_cast<const f32x4*>(cs + i0 + 4);
    const f32x4 s0 = *reinterpret_cast<const f32x4*>(cs + 64 + i0), s1 = *reinterpret_cast<const f32x4*>(cs + 64 + i0 + 4);
    const float ss = tile_ssq(a);
    const float r = rsqrtf(ss / 128.f + qe.eps);
    const bool first = dc < 8;
    uint32_t packed[4];
    float y[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float wf = T::to_f32((uint16_t)((e & 1) ? wraw[e >> 1] >> 16 : wraw[e >> 1] & 0xFFFFu));
        const float xn = T::to_f32(T::from_f32(mul_round<T>(a[e], r) * wf));
        const float other = __shfl_xor(xn, 8);
        const float cc = e < 4 ? c0[e] : c1[e - 4], sn = e < 4 ? s0[e] : s1[e - 4];
        const float x1 = first ? xn : other, x2 = first ? other : xn;
        y[e] = as_f32_result(first ? __fsub_rn(__fmul_rn(x1, cc), __fmul_rn(x2, sn))
                                   : __fadd_rn(__fmul_rn(x1, sn), __fmul_rn(x2, cc)));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) packed[i] = T::pack2(y[2 * i], y[2 * i + 1]);
    const u32x4 o = u32x4{packed[0], packed[1], packed[2], packed[3]};
    if (!valid) return;
    if (is_q) {
        *reinterpret_cast<u32x4*>(qe.q_out + ((int64_t)m * qe.nh + head) * 128 + dc * 8) = o;
    } else if (slot_ok) {
        *reinterpret_cast<u32x4*>(qe.k_cache + (((slot / qe.block_size) * qe.nkv + (head - qe.nh)) * qe.block_size +
                                                slot % qe.block_size) * 128 + dc * 8) = o;
    }
}

template <typename T>
__device__ __forceinline__ float silu_times_up(float gate, float up) {
    const float g = T::to_f32(T::from_f32(gate));
    return T::to_f32(T::from_f32(g / (1.f + __expf(-g)))) * T::to_f32(T::from_f32(up));
}

}  // namespace awq
