// Mixture of experts: router, grouping of (row, choice) pairs by expert, and the two grouped products.
//
// The grouped products exist in four forms, chosen by pairs per expert and operand alignment (moe_form):
//   few pairs    tiles of 16, 32 or 64 pairs on the skinny core: the weights stream once, straight into MFMA operands
//   many pairs   tiles of 64 or 128 pairs x 128 weight rows staged through LDS by load-to-LDS, double-buffered, MFMA 16x16x32
//   most pairs   tiles of 128 or 256 pairs x 256 weight rows on the product core of pingpong.hpp (rows in whole stages of 64)
//   any sizes    32 x 32 tiles in fp32 on the vector ALU (fp32 operands, rows that are not multiples of 8)
#include <algorithm>
#include <cmath>

#include "../pingpong.hpp"
#include "moe_route.hpp"
#include "skinny.hpp"

namespace nqh {
namespace {

// ---- router, any sizes: one wave per row -----------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void router_rows_kernel(const typename T::elem* __restrict__ h,
                                                          const typename T::elem* __restrict__ router,
                                                          int32_t* __restrict__ expert, float* __restrict__ weight,
                                                          int64_t rows, int width, int experts, int top) {
    extern __shared__ float s_score[];   // [4][experts]
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + wave;
    if (row >= rows) return;             // no barriers below: a wave works alone
    float* sc = s_score + wave * experts;
    for (int e = 0; e < experts; ++e) {
        float z = 0.f;
        for (int d = lane; d < width; d += 64) z += T::load(h + row * width + d) * T::load(router + (int64_t)e * width + d);
        z = wave_sum(z);
        if (lane == 0) sc[e] = sigmoid_f32(z);
    }
    wave_lds_fence();
    wave_topk(sc, experts, top, [&](int t, int e, float s) {
        expert[row * top + t] = e;
        weight[row * top + t] = s;
    });
}

// ---- router in bf16: 16 rows per workgroup, the waves split the width, experts 16 to an MFMA -----------------
// Products of bf16 operands are exact in the fp32 accumulation.
constexpr int kRouterTiles = 8;          // expert tiles per pass over the rows
__global__ __launch_bounds__(256) void router_mfma_kernel(const uint16_t* __restrict__ h, const uint16_t* __restrict__ router,
                                                          int32_t* __restrict__ expert, float* __restrict__ weight,
                                                          int rows, int width, int experts, int top) {
    extern __shared__ float s_mem[];     // scores [16][experts], then partial sums [4][tiles * 256]
    const int lane = threadIdx.x & 63, lo = lane & 15, hi = lane >> 4, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r0 = blockIdx.x * 16;
    float* s_part = s_mem + 16 * experts;
    const uint16_t* x_row = h + (int64_t)min(r0 + lo, rows - 1) * width;
    for (int e0 = 0; e0 < experts; e0 += 16 * kRouterTiles) {
        const int tiles = min(kRouterTiles, (experts - e0 + 15) / 16);
        f32x4 acc[kRouterTiles];
#pragma unroll
        for (int j = 0; j < kRouterTiles; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int k0 = wave * kPiece; k0 < width; k0 += 4 * kPiece) {
            u32x4 x[4];
            load_piece(x, x_row, k0, hi, width);
#pragma unroll
            for (int j = 0; j < kRouterTiles; ++j)
                if (j < tiles) {
                    u32x4 w[4];
                    load_piece_clamped(w, router + (int64_t)min(e0 + 16 * j + lo, experts - 1) * width, k0, hi, width);
#pragma unroll
                    for (int s = 0; s < 4; ++s) acc[j] = Bf::mfma16(w[s], x[s], acc[j]);
                }
        }
        __syncthreads();                 // the previous pass has read its sums
#pragma unroll
        for (int j = 0; j < kRouterTiles; ++j)
            if (j < tiles)
                *reinterpret_cast<f32x4*>(s_part + (wave * kRouterTiles + j) * 256 + lo * 16 + 4 * hi) = acc[j];
        __syncthreads();
        for (int i = threadIdx.x; i < tiles * 256; i += 256) {
            const int j = i >> 8, t = i >> 4 & 15, e = e0 + 16 * j + (i & 15);
            if (e >= experts) continue;
            float z = 0.f;
#pragma unroll
            for (int w = 0; w < 4; ++w) z += s_part[(w * kRouterTiles + j) * 256 + (i & 255)];
            s_mem[t * experts + e] = sigmoid_f32(z);
        }
    }
    __syncthreads();
    for (int t = wave; t < 16; t += 4) {
        const int row = r0 + t;
        if (row < rows)
            wave_topk(s_mem + t * experts, experts, top, [&](int i, int e, float s) {
                expert[(int64_t)row * top + i] = e;
                weight[(int64_t)row * top + i] = s;
            });
    }
}

// ---- plan ------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(1024) void moe_plan_kernel(const int32_t* __restrict__ expert, int32_t* __restrict__ order,
                                                        int32_t* __restrict__ tiles, int64_t pairs, int experts,
                                                        int tile_rows, int max_tiles) {
    __shared__ PlanShared s;
    plan_pairs(s, [&](int64_t p) { return expert[p]; }, order, tiles, pairs, experts, tile_rows, max_tiles);
}

// ---- grouped products, any sizes, fp32 arithmetic on the vector ALU ---------------------------------------
// Tiles of 32 pairs x 32 output columns.  GATED: two weight rows per column (gate and up) and the gated epilogue;
// otherwise rows come from `act` in plan order and go to y in pair order.
constexpr int kSimpleTile = 32;
template <typename T, bool GATED>
__global__ __launch_bounds__(256) void moe_tile_kernel(const typename T::elem* __restrict__ in,
                                                       const typename T::elem* __restrict__ w,
                                                       const float* __restrict__ weight, const int32_t* __restrict__ order,
                                                       const int32_t* __restrict__ tiles, typename T::elem* __restrict__ out,
                                                       int max_tiles, int top, int n_out, int n_in) {
    __shared__ float s_x[32][33], s_a[32][33], s_b[GATED ? 32 : 1][33];
    if ((int)blockIdx.x >= tiles[3 * max_tiles]) return;
    const int e = tiles[blockIdx.x], first = tiles[max_tiles + blockIdx.x], count = tiles[2 * max_tiles + blockIdx.x];
    const int n0 = blockIdx.y * 32, tid = threadIdx.x, col = tid & 31, r0 = tid >> 5;
    const typename T::elem* we = w + (int64_t)e * (GATED ? 2 : 1) * n_out * n_in;
    float a[4] = {0.f, 0.f, 0.f, 0.f}, b[4] = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < n_in; k0 += 32) {
        __syncthreads();
        const int kk = k0 + col;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = r0 + 8 * i;
            float x = 0.f, wa = 0.f, wb = 0.f;
            if (kk < n_in) {
                if (r < count) x = T::load(in + (int64_t)(GATED ? order[first + r] / top : first + r) * n_in + kk);
                if (n0 + r < n_out) {
                    wa = T::load(we + (int64_t)(n0 + r) * n_in + kk);
                    if constexpr (GATED) wb = T::load(we + (int64_t)(n_out + n0 + r) * n_in + kk);
                }
            }
            s_x[r][col] = x;
            s_a[r][col] = wa;
            if constexpr (GATED) s_b[r][col] = wb;
        }
        __syncthreads();
#pragma unroll 8
        for (int k = 0; k < 32; ++k) {
            const float wa = s_a[col][k], wb = GATED ? s_b[col][k] : 0.f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float x = s_x[r0 + 8 * i][k];
                a[i] += x * wa;
                if constexpr (GATED) b[i] += x * wb;
            }
        }
    }
    if (n0 + col >= n_out) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = r0 + 8 * i;
        if (r >= count) continue;
        const int32_t pair = order[first + r];
        if constexpr (GATED) {
            const float s = weight[pair];
            T::store(out + (int64_t)(first + r) * n_out + n0 + col, silu_f32(s * a[i]) * (s * b[i]));
        } else {
            T::store(out + (int64_t)pair * n_out + n0 + col, a[i]);
        }
    }
}

// ---- few pairs per expert: a tile of 16 MT pairs and 16 output columns per workgroup ------------------------
template <bool GATED, int MT>
__global__ __launch_bounds__(skinny_max_threads(MT)) void moe_skinny_kernel(const uint16_t* __restrict__ in, const uint16_t* __restrict__ w,
                                                          const float* __restrict__ weight,
                                                          const int32_t* __restrict__ order,
                                                          const int32_t* __restrict__ tiles, uint16_t* __restrict__ out,
                                                          int max_tiles, int top, int n_out, int n_in) {
    extern __shared__ __attribute__((aligned(16))) float s_sum[];
    constexpr int NW = GATED ? 2 : 1;
    if ((int)blockIdx.y >= tiles[3 * max_tiles]) return;
    const int e = tiles[blockIdx.y], first = tiles[max_tiles + blockIdx.y], count = tiles[2 * max_tiles + blockIdx.y];
    const int lane = threadIdx.x & 63, lo = lane & 15, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int waves = blockDim.x >> 6, n0 = blockIdx.x * 16;
    const uint16_t* we = w + (int64_t)e * NW * n_out * n_in + (int64_t)min(n0 + lo, n_out - 1) * n_in;
    const uint16_t* w_row[NW];
    w_row[0] = we;
    if constexpr (GATED) w_row[1] = we + (int64_t)n_out * n_in;
    const uint16_t* x_row[MT];
    f32x4 acc[MT][NW];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int place = first + min(16 * m + lo, count - 1);
        x_row[m] = in + (int64_t)(GATED ? order[place] / top : place) * n_in;
#pragma unroll
        for (int j = 0; j < NW; ++j) acc[m][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    skinny_accumulate<MT, NW>(acc, w_row, x_row, n_in, wave, waves);
    skinny_reduce<MT, NW>(acc, s_sum, wave, waves);
    for (int i = threadIdx.x; i < MT * 256; i += blockDim.x) {
        const int t = i >> 4, n = n0 + (i & 15);
        if (t >= count || n >= n_out) continue;
        const int32_t pair = order[first + t];
        const float* v = s_sum + (i >> 8) * NW * 256 + (i & 255);
        if constexpr (GATED) {
            const float s = weight[pair];
            out[(int64_t)(first + t) * n_out + n] = Bf::from_f32(silu_f32(s * v[0]) * (s * v[256]));
        } else {
            out[(int64_t)pair * n_out + n] = Bf::from_f32(v[0]);
        }
    }
}

// ---- many pairs per expert: PT = 64 or 128 pairs x 128 weight rows per workgroup -------------------------------
// Four waves of 64 weight rows x PT / 2 pairs.  A stage is 64 contraction elements of both operands, 128 bytes a row in LDS; a row's eight
// 16-byte pieces are stored at position piece ^ (row / 2 % 8), so that the 16 rows one operand read touches fall on all
// banks once (rows r and r + 1 sit in the two halves of the banks).  Load-to-LDS writes linearly, so the swizzle is in
// the lanes' source addresses.  Weight rows are the A operand: a lane ends up with four consecutive output columns of
// one pair.  GATED: 64 gate rows and their 64 up rows; every wave holds both of a column.
#define NQH_GPTR(p) ((__attribute__((address_space(1))) void*)(p))
#define NQH_LPTR(p) ((__attribute__((address_space(3))) void*)(p))
constexpr int kTile = 128, kStage = 64, kRowBytes = kStage * 2;
__device__ const u32x4 g_zero_piece = {0u, 0u, 0u, 0u};   // what lies past the end of a row

template <bool GATED, int PT>
__global__ __launch_bounds__(256) void moe_gemm_kernel(const uint16_t* __restrict__ in, const uint16_t* __restrict__ w,
                                                       const float* __restrict__ weight,
                                                       const int32_t* __restrict__ order,
                                                       const int32_t* __restrict__ tiles, uint16_t* __restrict__ out,
                                                       int max_tiles, int top, int n_out, int n_in, int n_groups) {
    constexpr int NJ = PT / 32;            // pair tiles of 16 per wave
    // one array: with an array per operand the compiler waits for every load-to-LDS in flight before any LDS read
    constexpr int kBuf = (kTile + PT) * kRowBytes, kX = kTile * kRowBytes;
    __shared__ __attribute__((aligned(1024))) unsigned char s_mem[2 * kBuf];   // [buffer][weights | pairs]
    // workgroups go round-robin over the 8 XCDs: give every XCD a contiguous run of the work, pair tiles fastest inside
    // blocks of 8 tiles so that both operands are reused in that XCD's L2
    const int total = gridDim.x, per = total >> 3;
    const int id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    const int block = id / (8 * n_groups), in_block = id - block * 8 * n_groups;
    const int tile = block * 8 + (in_block & 7), group = in_block >> 3;
    if (tile >= tiles[3 * max_tiles]) return;
    const int e = tiles[tile], first = tiles[max_tiles + tile], count = tiles[2 * max_tiles + tile];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lo = lane & 15, hi = lane >> 4, wm = wave & 1, wn = wave >> 1;
    const int n0 = group * (GATED ? kTile / 2 : kTile);
    const uint16_t* we = w + (int64_t)e * (GATED ? 2 : 1) * n_out * n_in;

    // staging roles: instruction i of this wave fills rows 8 (4 i + wave) .. + 7 of the tile, eight lanes a row
    const int piece_pos = lane & 7;
    const uint16_t *src_w[4], *src_x[NJ];
    int piece_k[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 8 * (4 * i + wave) + (lane >> 3);
        piece_k[i] = 8 * (piece_pos ^ ((r >> 1) & 7));
        int row;
        if constexpr (GATED) row = min(n0 + (r & 63), n_out - 1) + (r >= 64 ? n_out : 0);
        else row = min(n0 + r, n_out - 1);
        src_w[i] = we + (int64_t)row * n_in;
        if (i < NJ) {
            const int place = first + min(r, count - 1);
            src_x[i] = in + (int64_t)(GATED ? order[place] / top : place) * n_in;
        }
    }
    auto stage = [&](int k0, int buf) {
        unsigned char* base = s_mem + buf * kBuf;
        if (k0 + kStage <= n_in) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int dst = (4 * i + wave) * 1024;
                __builtin_amdgcn_global_load_lds(NQH_GPTR(src_w[i] + k0 + piece_k[i]), NQH_LPTR(base + dst), 16, 0, 0);
                if (i < NJ)
                    __builtin_amdgcn_global_load_lds(NQH_GPTR(src_x[i] + k0 + piece_k[i]), NQH_LPTR(base + kX + dst), 16, 0, 0);
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {    // the last stage of a row that is no multiple of 64: zeros past its end
            const int k = k0 + piece_k[i], dst = (4 * i + wave) * 1024;
            const void* zero = &g_zero_piece;
            const void* pw = k < n_in ? (const void*)(src_w[i] + k) : zero;
            __builtin_amdgcn_global_load_lds(NQH_GPTR(pw), NQH_LPTR(base + dst), 16, 0, 0);
            if (i < NJ) {
                const void* px = k < n_in ? (const void*)(src_x[i] + k) : zero;
                __builtin_amdgcn_global_load_lds(NQH_GPTR(px), NQH_LPTR(base + kX + dst), 16, 0, 0);
            }
        }
    };
    auto row_w = [&](int i) { return GATED ? (i < 2 ? wm * 32 + 16 * i : 64 + wm * 32 + 16 * (i - 2)) : wm * 64 + 16 * i; };
    f32x4 acc[4][NJ];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    stage(0, 0);
    int buf = 0;
    for (int k0 = 0; k0 < n_in; k0 += kStage) {
        __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): this wave's part of the stage has landed
        __syncthreads();                      // and everyone else's; the other buffer is free
        if (k0 + kStage < n_in) stage(k0 + kStage, buf ^ 1);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            u32x4 a[4], b[NJ];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int ra = row_w(i) + lo;
                a[i] = *reinterpret_cast<const u32x4*>(s_mem + buf * kBuf + ra * kRowBytes + (((4 * s + hi) ^ ((ra >> 1) & 7)) * 16));
            }
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int rb = wn * (PT / 2) + 16 * j + lo;
                b[j] = *reinterpret_cast<const u32x4*>(s_mem + buf * kBuf + kX + rb * kRowBytes + (((4 * s + hi) ^ ((rb >> 1) & 7)) * 16));
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < NJ; ++j) acc[i][j] = Bf::mfma16(a[i], b[j], acc[i][j]);
        }
        buf ^= 1;
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int t = wn * (PT / 2) + 16 * j + lo;
        if (t >= count) continue;
        const int32_t pair = order[first + t];
        if constexpr (GATED) {
            const float s = weight[pair];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int n = n0 + wm * 32 + 16 * i + 4 * hi;
                float v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = silu_f32(s * acc[i][j][r]) * (s * acc[i + 2][j][r]);
                if (n < n_out) store_vec<Bf, 4>(out + (int64_t)(first + t) * n_out + n, v);   // n_out % 8 == 0
            }
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int n = n0 + wm * 64 + 16 * i + 4 * hi;
                float v[4] = {acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
                if (n < n_out) store_vec<Bf, 4>(out + (int64_t)pair * n_out + n, v);
            }
        }
    }
}

// ---- most pairs per expert: XR = 128 or 256 pairs x 256 weight rows per workgroup -------------------------------
// A gathered row is one 32-bit offset per lane and load, so the gather costs nothing in the loop.  GATED: 128 gate rows and
// their 128 up rows; a wave's first tiles are gate, the others the up rows of the same columns.  The same sums in the same
// order as moe_gemm_kernel.  16,384 pairs of 8 experts, 4096 -> 2 x 6144 and back: 2890 us
// with moe_gemm_kernel, 1950 like this.
template <bool GATED, int XR>
__global__ __launch_bounds__(512, 2) void moe_pingpong_kernel(const uint16_t* __restrict__ in, const uint16_t* __restrict__ w,
                                                              const float* __restrict__ weight,
                                                              const int32_t* __restrict__ order,
                                                              const int32_t* __restrict__ tiles, uint16_t* __restrict__ out,
                                                              int max_tiles, int top, int n_out, int n_in, int n_groups,
                                                              int in_rows) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char s_stage[];
    using P = awq::PingPong<Bf, XR>;
    constexpr int kCols = GATED ? 128 : 256;
    int tile, group;
    if (!awq::xcd_tile((int)blockIdx.x, tiles[3 * max_tiles], n_groups, tile, group)) return;
    const int e = tiles[tile], first = tiles[max_tiles + tile], count = tiles[2 * max_tiles + tile];
    const int n0 = group * kCols;
    const uint32_t row_bytes = (uint32_t)n_in * 2, w_bytes = (GATED ? 2 : 1) * (uint32_t)n_out * row_bytes;
    P p;
    uint32_t vw[4], vx[P::kXLoads];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int r = P::w_row(q, p.wave, p.lane);
        int row = min(n0 + r, n_out - 1);
        if (GATED) row = min(n0 + r / (2 * P::kHalf) * P::kHalf + r % P::kHalf, n_out - 1) + (r / P::kHalf & 1) * n_out;
        vw[q] = P::source(row, (GATED ? 2 : 1) * n_out, row_bytes, r, p.lane);
    }
#pragma unroll
    for (int q = 0; q < P::kXLoads; ++q) {
        const int r = P::x_row(q, p.wave, p.lane), place = first + min(r, count - 1);
        vx[q] = P::source(GATED ? order[place] / top : place, in_rows, row_bytes, r, p.lane);
    }
    const auto rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(w) + (int64_t)e * (GATED ? 2 : 1) * n_out * n_in, 0,
                                                      w_bytes, 0x00020000);
    const auto rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(in), 0, (uint32_t)in_rows * row_bytes, 0x00020000);
    p.run(s_stage, rw, vw, rx, vx, n_in / P::kStage);
    if constexpr (GATED) {
        float score[P::NJ];
#pragma unroll
        for (int j = 0; j < P::NJ; ++j) score[j] = weight[order[first + min(p.wn * (XR / P::kWN) + 16 * j + p.lo, count - 1)]];
        p.template write<kCols>(s_stage, [&](int i, int j) {
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = silu_f32(score[j] * p.acc[i][j][r]) * (score[j] * p.acc[i + P::MI / 2][j][r]);
            return u32x2{Bf::pack2(v[0], v[1]), Bf::pack2(v[2], v[3])};
        }, [&](int r, int c, u32x4 v) {
            if (r < count && n0 + c < n_out) *reinterpret_cast<u32x4*>(out + (int64_t)(first + r) * n_out + n0 + c) = v;
        });
    } else {
        p.template write<kCols>(s_stage, [&](int i, int j) {
            const f32x4 v = p.acc[i][j];
            return u32x2{Bf::pack2(v[0], v[1]), Bf::pack2(v[2], v[3])};
        }, [&](int r, int c, u32x4 v) {
            if (r < count && n0 + c < n_out) *reinterpret_cast<u32x4*>(out + (int64_t)order[first + r] * n_out + n0 + c) = v;
        });
    }
}

template <bool GATED, int XR>
void launch_pingpong(const uint16_t* in, const uint16_t* w, const float* weight, const int32_t* order, const int32_t* tiles,
                     uint16_t* out, int64_t in_rows, int max_tiles, int top, int n_out, int n_in, hipStream_t st) {
    using P = awq::PingPong<Bf, XR>;
    auto kern = moe_pingpong_kernel<GATED, XR>;
    static bool raised = false;          // once per process and instantiation
    if (!raised) {
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, P::kLds) != hipSuccess)
            return;                      // launched() reports it
        raised = true;
    }
    const int64_t groups = cdiv(n_out, GATED ? 128 : 256);
    kern<<<dim3((unsigned)(cdiv(max_tiles * groups, 8) * 8)), dim3(P::kThreads), P::kLds, st>>>(
        in, w, weight, order, tiles, out, max_tiles, top, n_out, n_in, (int)groups, (int)in_rows);
}

enum class MoeForm { simple, skinny16, skinny32, skinny64, gemm64, gemm128, pingpong128, pingpong256 };
// Expected tiles of `rows` pairs: the pairs of an expert vary around their mean, here evenly over 2.2 of its roots to either side
// (routers are less even than chance), and near whole tiles some of the experts have one more.
double expected_tiles(int64_t pairs, int64_t experts, int rows) {
    if (pairs < experts) return (double)pairs;
    const double mean = (double)pairs / (double)experts, spread = 2.2 * std::sqrt(mean);
    const double low = std::max(0.0, mean - spread), high = mean + spread;
    const auto below = [&](double x) {          // the integral of ceil(u / rows) from 0 to x
        const double k = std::floor(x / rows);
        return rows * k * (k + 1) / 2 + (k + 1) * (x - k * rows);
    };
    return (double)experts * (below(high) - below(low)) / (high - low);
}

// Microseconds of both products: a stage of 64 of the contraction, in fuller rounds of the CUs a longer one, and the ends of a tile; no
// less than the weights take from memory.  Fitted to 16 sizes (2 to 128 experts, 512 to 4096 -> 2 x 384 to 2 x 6144) at 20 to 1000 pairs
// an expert, all forms timed: the least estimate is 0.7 % from the fastest form on average, more than a tenth in one of 30.
double moe_form_us(MoeForm form, int64_t pairs, int64_t experts, int64_t width, int64_t ff) {
    const bool gemm = form == MoeForm::gemm64, large = form == MoeForm::pingpong256;
    const double tiles = expected_tiles(pairs, experts, gemm ? 64 : (large ? 256 : 128)), columns = gemm ? 128 : 256;
    const auto product = [&](int64_t n_out, int64_t n_in) {
        const double rounds = tiles * std::ceil((double)n_out / columns) / 256, full = std::floor(rounds), part = rounds - full;
        const double stages = (double)n_in / 64;
        if (gemm) return 4.9 + stages * std::max(0.53, 0.23 + 0.436 * rounds);
        const double alone = large ? 0.744 : 0.53, shared = large ? 0.748 : 0.487;
        return std::ceil(rounds) * (large ? 10.4 : 6.6) + stages * (full * (alone + shared) + (part > 0 ? alone + shared * part : 0));
    };
    const double streamed = (double)(std::min(experts, pairs) * width * ff * 6) / ((gemm ? 3.34 : (large ? 3.6 : 4.23)) * 1e6);
    return std::max(product(2 * ff, width) + product(width, ff), streamed);
}

MoeForm moe_form(int64_t pairs, int64_t experts, int64_t width, int64_t ff, int dtype) {
    if (dtype != NQH_BF16 || width % 8 != 0 || ff % 8 != 0) return MoeForm::simple;
    // by pairs per expert, so that one tile usually holds all pairs of an expert while there are few
    if (pairs <= 6 * experts || pairs <= 16) return MoeForm::skinny16;
    if (pairs <= 16 * experts || pairs <= 32) return MoeForm::skinny32;
    // few experts and short rows: more workgroups (2 experts, 1024 -> 2 x 4096, 20 pairs each: 31 us, 50 with 64 x 128 tiles)
    const int64_t used = std::min(experts, pairs);
    if ((pairs <= 40 * experts || pairs <= 64) && used * cdiv(std::min(width, 2 * ff), 128) < 64) return MoeForm::skinny64;
    // The ping-pong core wants whole stages and 32-bit offsets into the rows and into an expert's weights.  Its tiles stream an expert's
    // weights once and faster; the 64 x 128 tiles have less to fill.  Both products, 64 x 128 / ping-pong 128 / 256 pairs a tile, us:
    //   8 experts, 4096 -> 2 x 6144, 20 pairs each 291 / 262 / 315, 115 each 430 / 297 / 330, 250 each 682 / 476 / 372;
    //   8 experts, 2048 -> 2 x 3072, 28 each 98 / 84 / 110, 100 each 130 / 98 / 108, 130 each 133 / 130 / 111;
    //   8 experts, 1024 -> 2 x 1536, 20 each 33 / 38 / 56, 160 each 39 / 43 / 58, 600 each 87 / 68 / 95;
    //   64 experts, 1024 -> 2 x 512, 40 each 57 / 43 / 57; 16 experts, 40 each 24 / 28 / 41, 115 each 26 / 30 / 42, 325 each 48 / 35 / 48;
    //   4 experts, 4096 -> 2 x 1536, 20 each 56 / 64 / 96, 200 each 64 / 70 / 100, 400 each 101 / 80 / 108.
    const bool stages = width % 64 == 0 && ff % 64 == 0 && pairs * std::max(width, ff) * 2 < (1ll << 32) &&
                        width * ff * 4 < (1ll << 32);
    if (!stages) return pairs <= 256 * experts ? MoeForm::gemm64 : MoeForm::gemm128;
    // (many pairs, a workgroup for half of the CUs in the smaller product: whatever the estimate, which was not fitted to shorter rows)
    const bool many = pairs > 160 * experts && pairs * std::min(cdiv(width, 256), cdiv(ff, 128)) >= 128 * 128;
    MoeForm best = MoeForm::pingpong128;
    for (const MoeForm form : {MoeForm::pingpong256, MoeForm::gemm64})
        if (!(many && form == MoeForm::gemm64) &&
            moe_form_us(form, pairs, experts, width, ff) < moe_form_us(best, pairs, experts, width, ff))
            best = form;
    return best;
}
int moe_form_rows(MoeForm f) {
    switch (f) {
        case MoeForm::skinny16: return 16;
        case MoeForm::skinny64: case MoeForm::gemm64: return 64;
        case MoeForm::gemm128: case MoeForm::pingpong128: return 128;
        case MoeForm::pingpong256: return 256;
        default: return 32;
    }
}

}  // namespace
}  // namespace nqh

using namespace nqh;

extern "C" int nqh_router_topk(const void* h, const void* router, int32_t* expert, float* weight, int64_t rows,
                               int64_t width, int64_t experts, int64_t top, int dtype, void* stream) {
    const char* fn = "nqh_router_topk";
    if (!h || !router || !expert || !weight) return fail(NQH_ERR_ARG, fn, "null pointer");
    if (!dtype_ok(dtype)) return fail(NQH_ERR_ARG, fn, "dtype must be NQH_BF16 or NQH_F32");
    if (rows <= 0 || width <= 0 || width > kMaxI32 || rows > kMaxI32 - 16 || top <= 0 || top > experts)
        return fail(NQH_ERR_ARG, fn, "sizes must be positive and top <= experts");
    if (experts > kMaxExperts) return fail(NQH_ERR_UNSUPPORTED, fn, "more than %d experts", kMaxExperts);
    (void)hipGetLastError();
    if (dtype == NQH_BF16 && width % 8 == 0 && experts <= 512 && aligned(h, 16) && aligned(router, 16)) {
        router_mfma_kernel<<<dim3((unsigned)cdiv(rows, 16)), dim3(256),
                             (size_t)(16 * experts + 4 * kRouterTiles * 256) * sizeof(float), (hipStream_t)stream>>>(
            (const uint16_t*)h, (const uint16_t*)router, expert, weight, (int)rows, (int)width, (int)experts, (int)top);
        return launched(fn);
    }
    NQH_WITH_TYPE(dtype, {
        using E = typename T::elem;
        router_rows_kernel<T><<<dim3((unsigned)cdiv(rows, 4)), dim3(256), (size_t)experts * 4 * sizeof(float),
                                (hipStream_t)stream>>>((const E*)h, (const E*)router, expert, weight, rows, (int)width,
                                                       (int)experts, (int)top);
    });
    return launched(fn);
}

extern "C" int64_t nqh_moe_max_tiles(int64_t pairs, int64_t experts, int64_t tile_rows) {
    if (pairs <= 0 || experts <= 0 || tile_rows <= 0) return 0;
    // full tiles plus one partial tile per expert that has pairs
    return pairs / tile_rows + (experts < pairs ? experts : pairs);
}

extern "C" int nqh_moe_plan(const int32_t* expert, int32_t* order, int32_t* tiles, int64_t pairs, int64_t experts,
                            int64_t tile_rows, int64_t max_tiles, void* stream) {
    const char* fn = "nqh_moe_plan";
    if (!expert || !order || !tiles) return fail(NQH_ERR_ARG, fn, "null pointer");
    if (pairs <= 0 || pairs > kMaxI32 || experts <= 0 || tile_rows <= 0 || tile_rows > kMaxI32 || 3 * max_tiles > kMaxI32)
        return fail(NQH_ERR_ARG, fn, "sizes must be positive 31-bit counts");
    if (experts > kMaxExperts) return fail(NQH_ERR_UNSUPPORTED, fn, "more than %d experts", kMaxExperts);
    if (max_tiles < nqh_moe_max_tiles(pairs, experts, tile_rows))
        return fail(NQH_ERR_ARG, fn, "max_tiles %lld is too small", (long long)max_tiles);
    (void)hipGetLastError();
    moe_plan_kernel<<<dim3(1), dim3(1024), 0, (hipStream_t)stream>>>(expert, order, tiles, pairs, (int)experts,
                                                                   (int)tile_rows, (int)max_tiles);
    return launched(fn);
}

static int check_moe(const char* fn, const void* in, const void* w, const int32_t* order, const int32_t* tiles,
                     const void* out, int64_t pairs, int64_t top, int64_t experts, int64_t width, int64_t ff,
                     int64_t tile_rows, int64_t max_tiles, int dtype) {
    if (!in || !w || !order || !tiles || !out) return fail(NQH_ERR_ARG, fn, "null pointer");
    if (!dtype_ok(dtype)) return fail(NQH_ERR_ARG, fn, "dtype must be NQH_BF16 or NQH_F32");
    if (pairs <= 0 || pairs > kMaxI32 || top <= 0 || experts <= 0 || width <= 0 || ff <= 0 || width > kMaxI32 ||
        2 * ff > kMaxI32 || max_tiles <= 0 || 3 * max_tiles > kMaxI32 || cdiv(width, 32) > 65535 || cdiv(ff, 32) > 65535 ||
        (max_tiles + 8) * (cdiv(std::max(width, ff), 64) + 1) > kMaxI32)
        return fail(NQH_ERR_ARG, fn, "sizes must be positive 31-bit counts");
    if (dtype == NQH_BF16 && (!aligned(in, 16) || !aligned(w, 16) || !aligned(out, 16)))
        return fail(NQH_ERR_ARG, fn, "bf16 operands must be 16-byte aligned");
    if (tile_rows != nqh_moe_tile_rows(pairs, experts, width, ff, dtype))
        return fail(NQH_ERR_ARG, fn, "the plan's tile_rows is not nqh_moe_tile_rows of this problem");
    return NQH_OK;
}

// Launches the bf16 form of this problem; false if it is the simple kernels' (nothing launched).
template <bool GATED>
static bool launch_fast(const void* in, const void* w, const float* weight, const int32_t* order, const int32_t* tiles,
                        void* out, int64_t pairs, int64_t top, int64_t experts, int64_t width, int64_t ff, int64_t n_out,
                        int64_t n_in, int64_t max_tiles, int dtype, void* stream) {
    const MoeForm form = moe_form(pairs, experts, width, ff, dtype);
    if (form == MoeForm::simple) return false;
    hipStream_t st = (hipStream_t)stream;
    (void)hipGetLastError();
#define NQH_ARGS                                                                                                        \
    (const uint16_t*)in, (const uint16_t*)w, weight, order, tiles, (uint16_t*)out, (int)max_tiles, (int)top, (int)n_out, \
        (int)n_in
    if (form == MoeForm::gemm64 || form == MoeForm::gemm128) {
        const int64_t groups = cdiv(n_out, GATED ? kTile / 2 : kTile);
        // whole blocks of 8 tiles x groups: a multiple of 8 workgroups
        const dim3 grid((unsigned)(cdiv(max_tiles, 8) * 8 * groups));
        if (form == MoeForm::gemm64) moe_gemm_kernel<GATED, 64><<<grid, dim3(256), 0, st>>>(NQH_ARGS, (int)groups);
        else moe_gemm_kernel<GATED, 128><<<grid, dim3(256), 0, st>>>(NQH_ARGS, (int)groups);
        return true;
    }
    if (form == MoeForm::pingpong128 || form == MoeForm::pingpong256) {
        const int64_t in_rows = GATED ? pairs / top : pairs;
        if (form == MoeForm::pingpong128)
            launch_pingpong<GATED, 128>((const uint16_t*)in, (const uint16_t*)w, weight, order, tiles, (uint16_t*)out, in_rows,
                                        (int)max_tiles, (int)top, (int)n_out, (int)n_in, st);
        else
            launch_pingpong<GATED, 256>((const uint16_t*)in, (const uint16_t*)w, weight, order, tiles, (uint16_t*)out, in_rows,
                                        (int)max_tiles, (int)top, (int)n_out, (int)n_in, st);
        return true;
    }
    const int64_t groups = cdiv(n_out, 16);
    const int mt = moe_form_rows(form) / 16;
    int waves = skinny_waves(groups * (pairs < experts ? pairs : experts), n_in);
    waves = std::min(waves, skinny_max_threads(mt) / 64);
    const size_t lds = (size_t)waves * mt * (GATED ? 512 : 256) * sizeof(float);     // at most 64 KiB
    const dim3 grid((unsigned)groups, (unsigned)max_tiles), block((unsigned)waves * 64);
    if (mt == 1) moe_skinny_kernel<GATED, 1><<<grid, block, lds, st>>>(NQH_ARGS);
    else if (mt == 2) moe_skinny_kernel<GATED, 2><<<grid, block, lds, st>>>(NQH_ARGS);
    else moe_skinny_kernel<GATED, 4><<<grid, block, lds, st>>>(NQH_ARGS);
#undef NQH_ARGS
    return true;
}

extern "C" int64_t nqh_moe_tile_rows(int64_t pairs, int64_t experts, int64_t width, int64_t ff, int dtype) {
    return moe_form_rows(moe_form(pairs, experts, width, ff, dtype));
}

extern "C" int nqh_moe_gate_up(const void* h, const void* gate_up, const float* weight, const int32_t* order,
                               const int32_t* tiles, void* act, int64_t pairs, int64_t top, int64_t experts,
                               int64_t width, int64_t ff, int64_t tile_rows, int64_t max_tiles, int dtype, void* stream) {
    const char* fn = "nqh_moe_gate_up";
    const int rc = check_moe(fn, h, gate_up, order, tiles, act, pairs, top, experts, width, ff, tile_rows, max_tiles, dtype);
    if (rc != NQH_OK) return rc;
    if (!weight) return fail(NQH_ERR_ARG, fn, "null pointer");
    if (launch_fast<true>(h, gate_up, weight, order, tiles, act, pairs, top, experts, width, ff, ff, width, max_tiles, dtype,
                          stream))
        return launched(fn);
    (void)hipGetLastError();
    NQH_WITH_TYPE(dtype, {
        using E = typename T::elem;
        moe_tile_kernel<T, true><<<dim3((unsigned)max_tiles, (unsigned)cdiv(ff, 32)), dim3(256), 0, (hipStream_t)stream>>>(
            (const E*)h, (const E*)gate_up, weight, order, tiles, (E*)act, (int)max_tiles, (int)top, (int)ff, (int)width);
    });
    return launched(fn);
}

extern "C" int nqh_moe_down(const void* act, const void* down, const int32_t* order, const int32_t* tiles, void* y,
                            int64_t pairs, int64_t experts, int64_t width, int64_t ff, int64_t tile_rows,
                            int64_t max_tiles, int dtype, void* stream) {
    const char* fn = "nqh_moe_down";
    const int rc = check_moe(fn, act, down, order, tiles, y, pairs, 1, experts, width, ff, tile_rows, max_tiles, dtype);
    if (rc != NQH_OK) return rc;
    if (launch_fast<false>(act, down, nullptr, order, tiles, y, pairs, 1, experts, width, ff, width, ff, max_tiles, dtype,
                           stream))
        return launched(fn);
    (void)hipGetLastError();
    NQH_WITH_TYPE(dtype, {
        using E = typename T::elem;
        moe_tile_kernel<T, false><<<dim3((unsigned)max_tiles, (unsigned)cdiv(width, 32)), dim3(256), 0,
                                    (hipStream_t)stream>>>((const E*)act, (const E*)down, nullptr, order, tiles, (E*)y,
                                                           (int)max_tiles, 1, (int)width, (int)ff);
    });
    return launched(fn);
}
