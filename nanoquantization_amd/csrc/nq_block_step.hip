// The linears between two attentions of a decode step in one launch: o_proj + residual, RMSNorm + gate|up + SiLU(gate) * up,
// down_proj + residual, RMSNorm + q|k|v of the next layer with q/k norm, rotary and cache write.
//
// At these sizes a linear is latency and not work (1 to 3 MB of weights): a launch of its own takes 7 to 9 us, of which a launch that does nothing
// takes 4.  Here 256 workgroups stay for the four phases.  While the first runs, the weights of the others come in (LDS and registers), so that
// a phase is: the phase before is known to be over, x arrives, some matrix instructions, the sums of the chunks of K, the result leaves.  Times
// inside a launch, Qwen3-0.6B, 32 rows, us: o_proj 6.9 (its weights and x come from memory), the others 4.2 to 5; of a phase 1.3 go by until the phase
// before is known to be over, 1.2 for x, 0.6 for the norm, 0.5 for the product, 0.9 for the sums and the epilogue, 0.4 until the results are out.
// Whole decode steps, the attention beside it unchanged, before (five launches a layer) / now, us: Qwen3-0.6B, 28 layers, 32 sequences of 640 tokens 1576 / 1287; six layers, 1 / 16 / 64
// rows 283 / 244, 333 / 277, 479 / 423; six layers of Qwen3-1.7B, 1 / 16 / 32 rows 346 / 333, 402 / 353, 451 / 406.
//
// Weights lie in pieces of 128 rows x 16 columns in operand order (nq_tile_weight): a load is 1 KiB without gaps, where the packed
// layout gives a CU 64 bytes of a row at a time, and eight codes of a lane unpack with seven instructions.  A task is a row tile of 16 (or two) by one
// column tile (three of gate|up, the eight of a head of q|k|v); the eight waves of a workgroup share its K.  Narrow tiles because 1024
// columns have to keep as many CUs busy as there are.  Between phases x lies in operand order too: rows as they are cost 2.7 us instead of 1.3.
// The sums are added in the GEMVs' order (hidden 2048: as they have it at 5 to 16 rows) and the norm rounds where theirs does, so that a model of 28 layers gives the same logits (with the norm
// round the sums, 1 / rms behind the product, a step takes 30 us less and its logits are 4.6 % of their norm away, as far as both are from
// 64 bits).
//
// Phases.  The tasks of a phase are dealt to shares, share = workgroup; XCD i (workgroups i, i + 8, ..) takes the i-th eighth, so that a line of the
// result is written from one XCD.  A share that is done sets its bit in the word of its XCD, the last of a word its bit in the root, the last
// of all rings 32 bells, each looked at by eight workgroups.  (All workgroups looking at the eight words delays the bits by up to 1.5 us, a
// word whose bits come from several XCDs by 3, and so do loads in flight in the wave that looks, whose answers come in order: hence the weights
// are asked for at the beginning.)  What crosses workgroups is stored past the L2 (sc1) and its lines, which hold nothing else, were read by nobody earlier in
// the launch, so that ordinary loads, which the XCD's L2 shares, find no older one.  A workgroup never relies on another one to start: after `spin` looks it
// takes the first share that is missing itself; shares read only what earlier phases have written and write the same values whoever runs them.
#include <type_traits>

#include "awq_common.hpp"
#include "step_epilogues.hpp"

#include "../../include/nq_engine_ops.h"

namespace awq {
namespace {

constexpr int kBlockWaves = 8, kBlockThreads = 64 * kBlockWaves, kShares = 256;
// flags of a phase, a line each: a word per XCD, the root, the bells
constexpr int kWordPitch = 32, kBells = 32, kRootAt = 8, kBellAt = 9, kPhaseWords = (kBellAt + kBells) * kWordPitch;
constexpr int kShared = 0, kAgent = 16;      // cache policy of buffer accesses; 16: sc1, the agent's point of coherence

struct Tiled {
    const u32x4* words;
    const uint32_t* affine;
    int chunks, tiles;
};

struct BlockStep {
    Tiled o, gate_up, down, qkv;
    const uint16_t* attn;
    const uint16_t* res_in;
    uint16_t* res_out;
    uint16_t *act, *tiled_mid, *tiled_out;
    float *squares_mid, *squares_out;
    const uint16_t* norm_mid;
    const uint16_t* norm_next;
    uint32_t* done;
    uint32_t* clear;
    float eps;
    int rows, spin;
    QkvEpilogue qe;
    const char* next[4];
    int64_t next_lines[4];
};

typedef __amdgpu_buffer_rsrc_t Rsrc;
__device__ __forceinline__ Rsrc rsrc_of(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}

#define NQ_GPTR(p) ((const __attribute__((address_space(1))) void*)(p))
#define NQ_LPTR(p) ((__attribute__((address_space(3))) void*)(p))

constexpr int kPiece = 1024 + 64;       // words, scales and zero points of 128 rows x 16 columns
constexpr int max_of(int a, int b) { return a > b ? a : b; }

// What a wave keeps in LDS: the sums of its chunks of the current task (1 KiB a chunk, column tile and row tile) and its pieces of gate|up and
// down_proj.  The sums of gate|up also lie over the pieces they are of, those of q|k|v over all.  MT: row tiles of a task of gate|up
// (of the others one); CO, CH, CI: chunks of 128 of a wave's part of heads * 128, hidden, inter.
template <int MT, int CO, int CH, int CI>
struct Form {
    static constexpr int CG = 3;
    static constexpr int head = 8 * CH * 1024, head_rows = 2 * 132 * 4;      // q|k|v: sums, and behind them two rows of the head
    static constexpr int at_g = (max_of(max_of(CO * 1024, CG * CH * (MT * 1024 - kPiece)), head + head_rows - (CG * CH + CI) * kPiece) + 63) / 64 * 64;
    static constexpr int at_d = at_g + CG * CH * kPiece, bytes = at_d + CI * kPiece;
};

// Pieces of chunks wave, wave + 8, .. of CT column tiles to LDS, [tile][chunk].
template <int CT, int C>
__device__ __forceinline__ void bring(char* to, const Tiled& t, int tile0, int lane, int wave) {
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int d = 0; d < C; ++d) {
            const size_t piece = (size_t)min(tile0 + c, t.tiles - 1) * t.chunks + wave + kBlockWaves * d;
            __builtin_amdgcn_global_load_lds(NQ_GPTR(t.words + piece * 64 + lane), NQ_LPTR(to + (c * C + d) * kPiece), 16, 0, 0);
            if (lane < 16)
                __builtin_amdgcn_global_load_lds(NQ_GPTR(t.affine + piece * 16 + lane), NQ_LPTR(to + (c * C + d) * kPiece + 1024), 4, 0, 0);
        }
}

// Rows of x as the matrix instruction takes them, of this wave's C chunks of K.
template <int MT, int C>
__device__ __forceinline__ void load_x(u32x4 (&v)[C][MT][4], const Rsrc& x, int row0, int chunks, int chunk0, int lane, int wave) {
#pragma unroll
    for (int d = 0; d < C; ++d)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int s = 0; s < 4; ++s)
                v[d][m][s] = __builtin_amdgcn_raw_buffer_load_b128(x, (uint32_t)(row0 / 16 + m) * (chunks * 4096) + 16 * lane + 1024 * s,
                                                                   (uint32_t)(wave + kBlockWaves * (chunk0 + d)) * 4096, kShared);
}

// y = x W of each of this wave's chunks for 16 MT rows and 16 CT columns; piece(c, d, ..) gives the lane's words and its column's scale and zero point.
// Codes go into the mantissa of a bf16, 128 + q or (columns 2, 3, 6, 7 of a word) 16 + q; the sums of a chunk and what is folded into them are
// those of the GEMVs (awq_gemv.hip), bit for bit.
template <typename T, int CT, int MT, int C, typename Piece>
__device__ __forceinline__ void multiply(const u32x4 (&v)[C][MT][4], f32x4 (&y)[C][CT][MT], int lane, Piece piece) {
    const bool high = lane & 2;
    const uint32_t mask = high ? 0x00780078u : 0x000F000Fu, magic = high ? 0x41804180u : 0x43004300u;
    const float offset = high ? 16.f : 128.f;
    const u32x4 ones = u32x4{T::ones2, T::ones2, T::ones2, T::ones2};
    const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < C; ++d) {
        f32x4 sum[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            sum[m] = zero;
#pragma unroll
            for (int s = 0; s < 4; ++s) sum[m] = T::mfma16(v[d][m][s], ones, sum[m]);
        }
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            u32x4 words;
            uint32_t affine;
            piece(c, d, words, affine);
            f32x4 acc[MT];
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                u32x4 b;
#pragma unroll
                for (int p = 0; p < 4; ++p) b[p] = (__builtin_amdgcn_alignbit(words[s], words[s], 4 * p) & mask) | magic;
#pragma unroll
                for (int m = 0; m < MT; ++m) acc[m] = T::mfma16(v[d][m][s], b, s == 0 ? zero : acc[m]);
            }
            const float step = T::to_f32((uint16_t)(affine & 0xFFFFu));
            const float z = (float)(affine >> 16) + offset;
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float t = step * (acc[m][i] - z * sum[m][i]);
                    y[d][c][m][i] = 0.f + t;
                }
        }
    }
}

// The sums of the wave's chunks to its part of LDS; then, behind a barrier, lane (column, 4 rows) of tile t = (c, m) adds those of all chunks: up to
// eight one after the other, more in fours whose sums are added one after the other (the order of the GEMVs' waves and K splits, of the
// second size at 5 to 16 rows).
template <int CT, int MT, int C>
__device__ __forceinline__ void sums_to_lds(const f32x4 (&y)[C][CT][MT], char* mine, int lane) {
#pragma unroll
    for (int d = 0; d < C; ++d)
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int m = 0; m < MT; ++m) *reinterpret_cast<f32x4*>(mine + ((d * CT + c) * MT + m) * 1024 + lane * 16) = y[d][c][m];
    __syncthreads();
}
template <int BYTES, int TILES, int C>
__device__ __forceinline__ f32x4 add_sums(const char* arena, int tile, int lane) {
    constexpr int kRun = C == 1 ? 8 : 4;
    f32x4 out = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int g = 0; g < kBlockWaves * C / kRun; ++g) {
        f32x4 v[kRun], s = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < kRun; ++j) {
            const int chunk = g * kRun + j;
            v[j] = *reinterpret_cast<const f32x4*>(arena + chunk % kBlockWaves * BYTES + (chunk / kBlockWaves * TILES + tile) * 1024 + lane * 16);
        }
#pragma unroll
        for (int j = 0; j < kRun; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) s[i] += v[j][i];
#pragma unroll
        for (int i = 0; i < 4; ++i) out[i] += s[i];
    }
    return out;
}

// Where the sum of a row's squares of columns n .. n + 7 lies, in bytes: the 16 of 128 columns are half a line, and the line is of two rows of the same
// columns, which one XCD writes.
__device__ __forceinline__ uint32_t square_at(int row, int n, int width) {
    return (uint32_t)((((row >> 4) * (width >> 7) + (n >> 7)) * 16 + (row & 15)) * 64 + (n >> 3 & 15) * 4);
}

// RMSNorm of what this wave has of 16 MT rows, x = T(T(x * r) * weight).  `squares` holds the sums of the rows' squares eight columns at a time: a wave
// adds those of a tile of 128 (in the order of tile_ssq, awq_common.hpp), the tiles meet in LDS and are added in their order.
template <typename T, int MT, int C>
__device__ __forceinline__ void normalise(u32x4 (&v)[C][MT][4], const Rsrc& squares, const uint16_t* weight, int row0, float eps, float* s_tiles, int lane,
                                          int wave) {
    constexpr int kTiles = kBlockWaves * C, kPitch = kTiles + 4;
    f32x4 part[C][MT];
    u32x4 w[C][4];
#pragma unroll
    for (int d = 0; d < C; ++d) {
        const int tile = wave + kBlockWaves * d;
#pragma unroll
        for (int m = 0; m < MT; ++m)
            part[d][m] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                       squares, square_at(row0 + 16 * m + (lane & 15), tile * 128, kTiles * 128) + (lane >> 4) * 16, 0,
                                                       kShared));
#pragma unroll
        for (int s = 0; s < 4; ++s) w[d][s] = *reinterpret_cast<const u32x4*>(weight + tile * 128 + 32 * s + 8 * (lane >> 4));
    }
#pragma unroll
    for (int d = 0; d < C; ++d)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            f32x4 p = part[d][m];
#pragma unroll
            for (int i = 0; i < 4; ++i) p[i] += __shfl_xor(p[i], 32);
#pragma unroll
            for (int i = 0; i < 4; ++i) p[i] += __shfl_xor(p[i], 16);
            const float ss = (p[0] + p[2]) + (p[1] + p[3]);
            if (lane < 16) s_tiles[(16 * m + lane) * kPitch + wave + kBlockWaves * d] = ss;
        }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        float total = 0.f;
#pragma unroll
        for (int t = 0; t < kTiles; t += 4) {
            const f32x4 p = *reinterpret_cast<const f32x4*>(s_tiles + (16 * m + (lane & 15)) * kPitch + t);
#pragma unroll
            for (int i = 0; i < 4; ++i) total += p[i];
        }
        const float r = rsqrtf(total / (float)(kTiles * 128) + eps);
#pragma unroll
        for (int d = 0; d < C; ++d)
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t xv = v[d][m][s][i], wv = w[d][s][i];
                    const float lo = mul_round<T>(T::to_f32((uint16_t)(xv & 0xFFFFu)), r) * T::to_f32((uint16_t)(wv & 0xFFFFu));
                    const float hi = mul_round<T>(T::to_f32((uint16_t)(xv >> 16)), r) * T::to_f32((uint16_t)(wv >> 16));
                    v[d][m][s][i] = T::pack2(lo, hi);
                }
    }
}

// The bits of a word when all shares (a multiple of eight) are done.
__device__ __forceinline__ uint32_t full_word(int shares) { return shares >= kShares ? ~0u : (1u << (shares >> 3)) - 1; }
// All shares of a phase done: -1; after `spin` looks the first one that is not.
__device__ __forceinline__ int await_shares(const uint32_t* done, int shares, int spin, int* s_missing, int lane, int wave) {
    if (wave == 0) {
        int missing = -1;
        for (int look = 0;; ++look) {
            if (__hip_atomic_load(done + (kBellAt + blockIdx.x % kBells) * kWordPitch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
            if (look >= spin) {
                const uint32_t open =
                    lane < 8 ? full_word(shares) & ~__hip_atomic_load(done + lane * kWordPitch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
                const uint64_t any = __ballot(open != 0);
                if (any == 0) break;
                const int l = __builtin_ctzll(any);
                missing = l + 8 * __builtin_ctz(__shfl(open, l));
                break;
            }
            __builtin_amdgcn_s_sleep(2);
        }
        if (lane == 0) *s_missing = missing;
    }
    __syncthreads();
    const int missing = *s_missing;
    __syncthreads();        // the next look may write it
    return missing;
}
// The share's results are out: its bit, and what the last bit of all sets off.
__device__ __forceinline__ void share_done(uint32_t* done, int share, int shares, int lane, int wave) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0x0F70);     // vmcnt(0)
    __syncthreads();
    if (wave == 0) {
        bool all = false;
        if (lane == 0) {
            const uint32_t bit = 1u << (share >> 3);
            const uint32_t word = __hip_atomic_fetch_or(done + (share & 7) * kWordPitch, bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) | bit;
            if (word == full_word(shares)) {
                const uint32_t mine = 1u << (share & 7);
                all = (__hip_atomic_fetch_or(done + kRootAt * kWordPitch, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) | mine) == 0xFF;
            }
        }
        if (__ballot(all) && lane < kBells)
            __hip_atomic_store(done + (kBellAt + lane) * kWordPitch, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

template <int MT, int CO, int CH, int CI>
__global__ __launch_bounds__(kBlockThreads) void block_step_kernel(const BlockStep a) {
    using T = BF16;
    using F = Form<MT, CO, CH, CI>;
    constexpr int CG = F::CG, kTurn = 20;
    constexpr bool kLate = CH * MT > 2;      // no registers for q|k|v's weights while gate|up runs: they come with down_proj
    extern __shared__ __align__(16) char arena[];
    __shared__ int s_missing;
    __shared__ __align__(16) float s_tiles[16 * MT * (kBlockWaves * CH + 4)];
    __shared__ __align__(16) float s_turn[16 * kTurn];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), own = blockIdx.x;
    const int column = lane & 15, row4 = (lane >> 4) * 4;
    const bool odd = lane & 1;
    char* mine = arena + wave * F::bytes;
    constexpr int wide = kBlockWaves * 128 * CO, width = kBlockWaves * 128 * CH, inter = kBlockWaves * 128 * CI;
    constexpr int tiles0 = width / 16, tiles1 = inter / 8;
    const int m_tiles = (a.rows + 15) / 16, groups1 = (m_tiles + MT - 1) / MT;
    const int tasks0 = tiles0 * m_tiles, tasks1 = tiles1 / CG * groups1, tasks3 = a.qkv.tiles / 8 * m_tiles;
    const int per0 = tasks0 / 8, per1 = tasks1 / 8, per3 = (tasks3 + 7) / 8;
    const int shares0 = min(8 * per0, kShares), shares1 = min(8 * per1, kShares);
    const auto first = [](int share, int per) { return (share & 7) * per + (share >> 3); };
    const auto end = [](int share, int per, int tasks) { return min(((share & 7) + 1) * per, tasks); };
    const uint32_t all = (uint32_t)a.rows * width * 2, padded = (uint32_t)m_tiles * 16 * width * 2, square_bytes = (uint32_t)m_tiles * 16 * (width / 8) * 4;
    const auto over = [](int task, int groups) { return task * (groups == 1 ? 65536 : groups == 2 ? 32768 : groups == 3 ? 21846 : 16384) >> 16; };

    u32x4 w0[CO], w3[8][CH];
    uint32_t affine0[CO], affine3[8][CH];
    const auto bring0 = [&](int task) {
#pragma unroll
        for (int d = 0; d < CO; ++d) {
            const size_t piece = (size_t)over(task, m_tiles) * a.o.chunks + wave + kBlockWaves * d;
            w0[d] = a.o.words[piece * 64 + lane];
            affine0[d] = a.o.affine[piece * 16 + column];
        }
    };
    const auto bring3 = [&](int task) {
#pragma unroll
        for (int c = 0; c < 8; ++c)
#pragma unroll
            for (int d = 0; d < CH; ++d) {
                const size_t piece = (size_t)(over(task, m_tiles) * 8 + c) * a.qkv.chunks + wave + kBlockWaves * d;
                w3[c][d] = a.qkv.words[piece * 64 + lane];
                affine3[c][d] = a.qkv.affine[piece * 16 + column];
            }
    };
    const auto piece_of = [&](int at, u32x4& words, uint32_t& affine) {
        words = *reinterpret_cast<const u32x4*>(mine + at + lane * 16);
        affine = *reinterpret_cast<const uint32_t*>(mine + at + 1024 + column * 4);
    };
    // what this wave has asked for by load-to-LDS is there (the compiler does not count it against the reads)
    const auto drain = [] { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); };
    const int own0 = first(own, per0), own1 = first(own, per1), own3 = first(own, per3), end3 = end(own, per3, tasks3);
    const auto ahead = [&] {        // what the later phases multiply first, on its way while the first phase runs
        if (own < shares1) bring<CG, CH>(mine + F::at_g, a.gate_up, over(own1, groups1) * CG, lane, wave);
        if (own < shares0) bring<1, CI>(mine + F::at_d, a.down, over(own0, m_tiles), lane, wave);
        if (!kLate && own3 < end3) bring3(own3);
    };
    if (own == 0)
        for (int i = threadIdx.x; i < 3 * kPhaseWords / kWordPitch; i += kBlockThreads) a.clear[i * kWordPitch] = 0;

    // What a task of o_proj or down_proj leaves, behind its multiplication: lane (row, half) of a row tile takes eight columns of the new
    // residual: the residual as rows (down_proj) and as the next linear's input, and the sum of the eight squares.
    struct Residual {
        Rsrc before, rows, tiled, squares;
        bool before_tiled, to_rows, to_tiled;
    };
    const auto old_of = [&](const Residual& r, int tile, int row0) {
        const int row = row0 + (lane >> 1 & 15), n = 16 * tile + (lane & 1) * 8;
        return __builtin_amdgcn_raw_buffer_load_b128(r.before, r.before_tiled ? tiled_at(row, n, width) : (uint32_t)(row * width + n) * 2, 0, kShared);
    };
    const auto leave = [&](const Residual& r, const f32x4& sum, const u32x4& old, int tile, int row0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) s_turn[(row4 + i) * kTurn + column] = sum[i];
        if (lane >= 32) return;
        const int r16 = lane >> 1, half = (lane & 1) * 8, row = row0 + r16, n = 16 * tile + half;
        const f32x4 lo = *reinterpret_cast<const f32x4*>(s_turn + r16 * kTurn + half), hi = *reinterpret_cast<const f32x4*>(s_turn + r16 * kTurn + half + 4);
        float v[8], ss = 0.f;
        u32x4 out;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float x = e < 4 ? lo[e] : hi[e - 4], before = T::to_f32((uint16_t)((e & 1) ? old[e >> 1] >> 16 : old[e >> 1] & 0xFFFFu));
            v[e] = T::to_f32(T::from_f32(before + T::to_f32(T::from_f32(x))));
            ss = __builtin_fmaf(v[e], v[e], ss);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) out[i] = T::pack2(v[2 * i], v[2 * i + 1]);
        // rows past the end are outside the row-by-row residual
        if (r.to_rows) __builtin_amdgcn_raw_buffer_store_b128(out, r.rows, (uint32_t)(row * width + n) * 2, 0, kAgent);
        if (r.to_tiled) {
            __builtin_amdgcn_raw_buffer_store_b128(out, r.tiled, tiled_at(row, n, width), 0, kAgent);
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, ss), r.squares, square_at(row, n, width), 0, kAgent);
        }
    };
    const auto o_proj = [&](int task, bool reload, auto hook) {
        const int tile = over(task, m_tiles), row0 = (task - tile * m_tiles) * 16;
        const Residual r{rsrc_of(a.res_in, all), rsrc_of(a.res_in, 0), rsrc_of(a.tiled_mid, padded), rsrc_of(a.squares_mid, square_bytes), false, false, true};
        if (reload) bring0(task);
        u32x4 v[CO][1][4], old = u32x4{0, 0, 0, 0};
        f32x4 y[CO][1][1];
        load_x<1, CO>(v, rsrc_of(a.attn, (uint32_t)m_tiles * 16 * wide * 2), row0, wide / 128, 0, lane, wave);
        if (wave == 0) old = old_of(r, tile, row0);
        hook();
        multiply<T, 1, 1, CO>(v, y, lane, [&](int, int d, u32x4& words, uint32_t& affine) { words = w0[d], affine = affine0[d]; });
        sums_to_lds<1, 1, CO>(y, mine, lane);
        if (wave == 0) leave(r, add_sums<F::bytes, 1, CO>(arena, 0, lane), old, tile, row0);
    };
    const auto gate = [&](int task, bool reload) {
        const int group = over(task, groups1), tile = group * CG, row0 = (task - group * groups1) * 16 * MT;
        const Rsrc act = rsrc_of(a.act, (uint32_t)m_tiles * 16 * inter * 2);
        if (reload) bring<CG, CH>(mine + F::at_g, a.gate_up, tile, lane, wave);
        drain();
        u32x4 v[CH][MT][4];
        f32x4 y[CH][CG][MT];
        load_x<MT, CH>(v, rsrc_of(a.tiled_mid, padded), row0, width / 128, 0, lane, wave);
        normalise<T, MT, CH>(v, rsrc_of(a.squares_mid, square_bytes), a.norm_mid, row0, a.eps, s_tiles, lane, wave);
        multiply<T, CG, MT, CH>(v, y, lane,
                                 [&](int c, int d, u32x4& words, uint32_t& affine) { piece_of(F::at_g + (c * CH + d) * kPiece, words, affine); });
        sums_to_lds<CG, MT, CH>(y, mine, lane);
        if (wave < CG * MT) {      // lanes of gate columns take the first two rows, those of up columns the others
            const f32x4 sum = add_sums<F::bytes, CG * MT, CH>(arena, wave, lane);
            const int c = wave / MT, row = row0 + wave % MT * 16 + row4;
            const bool up = column >= 8;
            float out[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const float own_sum = up ? sum[2 + i] : sum[i], other = __shfl_xor(up ? sum[i] : sum[2 + i], 8);
                out[i] = silu_times_up<T>(up ? other : own_sum, up ? own_sum : other);
            }
            const float other = __shfl_xor(odd ? out[0] : out[1], 1);
            const uint32_t pair = odd ? T::pack2(other, out[1]) : T::pack2(out[0], other);
            __builtin_amdgcn_raw_buffer_store_b32(pair, act, tiled_at(row + (up ? 2 : 0) + odd, (tile + c) * 8 + (column & 6), inter), 0, kAgent);
        }
    };
    const auto down_proj = [&](int task, bool reload, auto hook) {
        constexpr int D = 3;       // chunks of x in registers at a time
        static_assert(CI % D == 0, "whole runs of chunks");
        const int tile = over(task, m_tiles), row0 = (task - tile * m_tiles) * 16;
        const Residual r{rsrc_of(a.tiled_mid, padded), rsrc_of(a.res_out, all), rsrc_of(a.tiled_out, padded), rsrc_of(a.squares_out, square_bytes), true, true,
                         a.norm_next != nullptr};
        if (reload) bring<1, CI>(mine + F::at_d, a.down, tile, lane, wave);
        drain();
        const Rsrc x = rsrc_of(a.act, (uint32_t)m_tiles * 16 * inter * 2);
        u32x4 old = u32x4{0, 0, 0, 0};
        f32x4 y[CI][1][1];
#pragma unroll
        for (int base = 0; base < CI; base += D) {
            u32x4 v[D][1][4];
            load_x<1, D>(v, x, row0, inter / 128, base, lane, wave);
            if (base == 0 && wave == 0) old = old_of(r, tile, row0);
            if (base + D == CI) hook();
            f32x4 part[D][1][1];
            multiply<T, 1, 1, D>(v, part, lane,
                                   [&](int, int d, u32x4& words, uint32_t& affine) { piece_of(F::at_d + (base + d) * kPiece, words, affine); });
#pragma unroll
            for (int d = 0; d < D; ++d) y[base + d][0][0] = part[d][0][0];
        }
        sums_to_lds<1, 1, CI>(y, mine, lane);
        if (wave == 0) leave(r, add_sums<F::bytes, 1, CI>(arena, 0, lane), old, tile, row0);
    };
    // a phase: the first task of the own share with what `ahead` brought, then the rest of it, then what is missing
    const auto phase = [&](int per, int tasks, int shares, uint32_t* done, bool last, auto begin, auto task_of) {
        int share = own < shares ? own : -1, task = 0, stop = 0;
        if (share >= 0) {
            task = first(own, per), stop = end(own, per, tasks);
            begin(task);
            task += 32;
        }
        for (;;) {
            if (share >= 0) {
                for (; task < stop; task += 32) {
                    __syncthreads();
                    task_of(task);
                }
                share_done(done, share, shares, lane, wave);
            }
            if (last) return;
            share = await_shares(done, shares, a.spin, &s_missing, lane, wave);
            if (share < 0) return;
            task = first(share, per), stop = end(share, per, tasks);
        }
    };

    if (own < shares0) bring0(own0);
    else ahead();
    phase(per0, tasks0, shares0, a.done, false, [&](int task) { o_proj(task, false, ahead); }, [&](int task) { o_proj(task, true, [] {}); });
    phase(per1, tasks1, shares1, a.done + kPhaseWords, false, [&](int task) { gate(task, false); }, [&](int task) { gate(task, true); });
    const auto late = [&] {
        if (kLate && own3 < end3) bring3(own3);
    };
    if (own >= shares0) late();
    phase(per0, tasks0, shares0, a.done + 2 * kPhaseWords, !a.norm_next, [&](int task) { down_proj(task, false, late); },
          [&](int task) { down_proj(task, true, [] {}); });
    if (!a.norm_next) return;
    if (own >= 8 * per3) {
        // Workgroups without a head touch the lines of the weights that the launch behind the next attention reads, which then finds them in the
        // memory-side cache (28 layers, 32 rows: 1295 -> 1268 us a step).
        const int64_t threads = (int64_t)(kShares - 8 * per3) * kBlockThreads, at = (int64_t)(own - 8 * per3) * kBlockThreads + threadIdx.x;
        uint32_t seen = 0;
        for (int r = 0; r < 4; ++r)
            for (int64_t line = at; line < a.next_lines[r]; line += threads)
                seen |= *reinterpret_cast<const volatile uint32_t*>(a.next[r] + line * 128);
        asm volatile("" ::"v"(seen));
        return;
    }
    // q|k|v of the next layer, one head and 16 rows a task
    for (int task = own3; task < end3; task += 32) {
        const int head = over(task, m_tiles), row0 = (task - head * m_tiles) * 16;
        if (task != own3) {
            __syncthreads();
            bring3(task);
        }
        u32x4 v[CH][1][4];
        f32x4 y[CH][8][1];
        load_x<1, CH>(v, rsrc_of(a.tiled_out, padded), row0, width / 128, 0, lane, wave);
        normalise<T, 1, CH>(v, rsrc_of(a.squares_out, square_bytes), a.norm_next, row0, a.eps, s_tiles, lane, wave);
        multiply<T, 8, 1, CH>(v, y, lane, [&](int c, int d, u32x4& words, uint32_t& affine) { words = w3[c][d], affine = affine3[c][d]; });
        sums_to_lds<8, 1, CH>(y, mine, lane);
        const auto row_of = [&](int r) { return reinterpret_cast<float*>(arena + (r >> 1) * F::bytes + F::head + (r & 1) * 528); };
        const f32x4 sum = add_sums<F::bytes, 8, CH>(arena, wave, lane);
#pragma unroll
        for (int i = 0; i < 4; ++i) row_of(row4 + i)[16 * wave + column] = sum[i];
        __syncthreads();
        if (threadIdx.x < 256) {
            const int r = threadIdx.x >> 4, c = (threadIdx.x & 15) * 8;
            const float* p = row_of(r) + c;
            float out[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) out[i] = p[i];
            qkv_rope_store<T>(out, row0 + r, (size_t)head * 128 + c, row0 + r < a.rows, a.qe);
        }
    }
}

__global__ __launch_bounds__(256) void tile_weight_kernel(const uint32_t* __restrict__ qweight, const uint16_t* __restrict__ qscales,
                                                          const uint32_t* __restrict__ qzeros, u32x4* __restrict__ words,
                                                          uint32_t* __restrict__ affine, int K, int N, int g) {
    const int chunks = K / 128, row_words = N / 8;
    const int64_t item = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (item >= (int64_t)(N / 16) * chunks) return;
    const int tile = (int)(item / chunks), chunk = (int)(item % chunks), lane = threadIdx.x & 63;
    const int n = tile * 16 + (lane & 15), shift = nibble_shift(n & 7);
    const uint32_t* column = qweight + (size_t)(chunk * 128 + 8 * (lane >> 4)) * row_words + (n >> 3);
    u32x4 out;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        uint32_t w = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) w |= (column[(size_t)(32 * s + j) * row_words] >> shift & 15u) << (j & 1 ? 16 + 2 * (j - 1) : 2 * j);
        out[s] = n & 2 ? w << 3 | w >> 29 : w;      // where the kernel's 16 + q has its code
    }
    words[item * 64 + lane] = out;
    if (lane < 16) {
        const int group = chunk * 128 / g;
        affine[item * 16 + lane] = (qzeros[(size_t)group * row_words + (n >> 3)] >> shift & 15u) << 16 | qscales[(size_t)group * N + n];
    }
}

}  // namespace
}  // namespace awq

using namespace awq;

static int bad(const char* fn, const char* what) {
    set_error("%s: %s", fn, what);
    return AWQ_ERR_INVALID_ARG;
}

extern "C" size_t nq_tiled_weight_bytes(int64_t N, int64_t K) {
    return N <= 0 || K <= 0 || N % 16 || K % 128 ? 0 : (size_t)N * (K / 128) * (64 + 4);
}

extern "C" int nq_tile_weight(const int32_t* qweight, const void* qscales, const int32_t* qzeros, void* out, int64_t N, int64_t K,
                              int64_t group_size, int dtype, void* stream) {
    const char* fn = "nq_tile_weight";
    if (!qweight || !qscales || !qzeros || !out) return bad(fn, "null pointer argument");
    if (dtype != AWQ_F16 && dtype != AWQ_BF16) return bad(fn, "dtype must be AWQ_F16 or AWQ_BF16");
    if (N <= 0 || K <= 0 || N % 16 || K % 128 || group_size <= 0 || group_size % 128 || K % group_size || N > 0x7fffffff || K > 0x7fffffff)
        return bad(fn, "needs N % 16 == 0, K % 128 == 0 and a group size that 128 divides");
    if (reinterpret_cast<uintptr_t>(out) & 15u) return bad(fn, "the result must be 16-byte aligned");
    const int64_t items = N / 16 * (K / 128);
    if (cdiv(items, 4) > 0x7fffffff) return bad(fn, "problem too large");
    (void)hipGetLastError();
    tile_weight_kernel<<<dim3((unsigned)cdiv(items, 4)), 256, 0, (hipStream_t)stream>>>(
        (const uint32_t*)qweight, (const uint16_t*)qscales, (const uint32_t*)qzeros, (u32x4*)out,
        (uint32_t*)((char*)out + (size_t)N * (K / 128) * 64), (int)K, (int)N, (int)group_size);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? AWQ_OK : hip_fail(fn, e);
}

namespace awq {
namespace {

Tiled tiled(const void* p, int64_t N, int64_t K) {
    return Tiled{(const u32x4*)p, (const uint32_t*)((const char*)p + (size_t)N * (K / 128) * 64), (int)(K / 128), (int)(N / 16)};
}

template <int MT, int CO, int CH, int CI>
hipError_t launch_block_step(const BlockStep& a, hipStream_t st) {
    constexpr int lds = kBlockWaves * Form<MT, CO, CH, CI>::bytes;
    const auto kernel = block_step_kernel<MT, CO, CH, CI>;
    if (lds > 65536) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return e;
    }
    kernel<<<dim3(kShares), dim3(kBlockThreads), lds, st>>>(a);
    return hipGetLastError();
}

}  // namespace
}  // namespace awq

extern "C" size_t nq_block_step_supported(int64_t rows, int64_t hidden, int64_t inter, int64_t heads, int64_t kv_heads) {
    // (more rows of the second size have no registers left for their sums: six layers at 40 / 64 rows 560 / 610 us in launches one by one, 584 / 623)
    // head ratios: those whose attention leaves its result in the layout that o_proj reads (nq_paged_attention_decode_tiled)
    return rows >= 1 && heads == 16 && (kv_heads == heads || 2 * kv_heads == heads) &&
           ((hidden == 1024 && inter == 3072 && rows <= 64) || (hidden == 2048 && inter == 6144 && rows <= 32));
}

extern "C" size_t nq_block_step_flag_words(void) { return 3 * kPhaseWords; }

extern "C" int nq_block_step(const nq_block_step_args* p, void* stream) {
    const char* fn = "nq_block_step";
    if (!p) return bad(fn, "null pointer argument");
    const nq_block_step_args& q = *p;
    if (!q.o || !q.gate_up || !q.down || !q.attn || !q.res_in || !q.res_out || !q.act ||
        !q.norm_mid || !q.tiled_mid || !q.squares_mid || !q.done || !q.clear)
        return bad(fn, "null pointer argument");
    if (q.qkv && (!q.norm_next || !q.tiled_out || !q.squares_out || !q.q_weight || !q.k_weight || !q.cos_sin || !q.positions || !q.slots || !q.q_out || !q.k_cache || !q.v_cache))
        return bad(fn, "null pointer argument");
    const uintptr_t bits = (uintptr_t)q.o | (uintptr_t)q.gate_up | (uintptr_t)q.down | (uintptr_t)q.qkv | (uintptr_t)q.attn | (uintptr_t)q.res_in |
                           (uintptr_t)q.res_out | (uintptr_t)q.act | (uintptr_t)q.tiled_mid | (uintptr_t)q.tiled_out | (uintptr_t)q.squares_mid | (uintptr_t)q.squares_out |
                           (uintptr_t)q.norm_mid | (uintptr_t)q.norm_next | (uintptr_t)q.done | (uintptr_t)q.clear | (uintptr_t)q.q_weight |
                           (uintptr_t)q.k_weight | (uintptr_t)q.cos_sin | (uintptr_t)q.q_out | (uintptr_t)q.k_cache | (uintptr_t)q.v_cache;
    if (bits & 15u) return bad(fn, "every tensor must be 16-byte aligned");
    // What one phase writes and a later one reads through the L2 has lines of its own (their sizes are whole lines at any number of rows): nobody
    // brings one in by reading its neighbour before it is written.  The flags of another launch are cleared beside this one's.
    const uintptr_t lines = (uintptr_t)q.act | (uintptr_t)q.tiled_mid | (uintptr_t)q.tiled_out | (uintptr_t)q.squares_mid | (uintptr_t)q.squares_out |
                            (uintptr_t)q.done | (uintptr_t)q.clear | (uintptr_t)q.attn | (uintptr_t)q.res_out | (uintptr_t)q.q_out;
    if (lines & 127u) return bad(fn, "attn, res_out, act, q_out, the tiled residuals, the squares and the flags must be 128-byte aligned");
    if (!nq_block_step_supported(q.rows, q.hidden, q.inter, q.heads, q.kv_heads)) {
        set_error("%s: no form for these sizes", fn);
        return AWQ_ERR_UNSUPPORTED;
    }
    if (q.res_out == q.res_in || q.tiled_mid == q.tiled_out || q.done == q.clear)
        return bad(fn, "the residual buffers and the flags must be distinct");
    if (q.qkv && (q.max_positions <= 0 || q.max_positions > 0x7fffffff || q.block_size <= 0 || q.block_size > 0x7fffffff || q.num_slots <= 0 ||
                  q.num_slots % q.block_size))
        return bad(fn, "needs positive max_positions and block_size, and num_slots a multiple of block_size");
    if (q.spin < 0 || q.spin > (1 << 24)) return bad(fn, "spin outside 0 .. 2^24");
    BlockStep a = {};
    const int64_t wide = q.heads * 128;
    a.o = tiled(q.o, q.hidden, wide);
    a.gate_up = tiled(q.gate_up, 2 * q.inter, q.hidden);
    a.down = tiled(q.down, q.hidden, q.inter);
    if (q.qkv) a.qkv = tiled(q.qkv, wide + 2 * q.kv_heads * 128, q.hidden);
    a.attn = (const uint16_t*)q.attn, a.res_in = (const uint16_t*)q.res_in;
    a.res_out = (uint16_t*)q.res_out, a.act = (uint16_t*)q.act;
    a.tiled_mid = (uint16_t*)q.tiled_mid, a.tiled_out = (uint16_t*)q.tiled_out, a.squares_mid = q.squares_mid, a.squares_out = q.squares_out;
    a.norm_mid = (const uint16_t*)q.norm_mid, a.norm_next = q.qkv ? (const uint16_t*)q.norm_next : nullptr;
    a.done = q.done, a.clear = q.clear;
    a.eps = q.eps, a.rows = (int)q.rows, a.spin = (int)q.spin;
    a.qe.q_weight = (const uint16_t*)q.q_weight, a.qe.k_weight = (const uint16_t*)q.k_weight;
    a.qe.cos_sin = q.cos_sin, a.qe.positions = q.positions, a.qe.slots = q.slots;
    a.qe.q_out = (uint16_t*)q.q_out, a.qe.k_cache = (uint16_t*)q.k_cache, a.qe.v_cache = (uint16_t*)q.v_cache;
    a.qe.nh = (int)q.heads, a.qe.nkv = (int)q.kv_heads, a.qe.max_positions = (int)q.max_positions, a.qe.block_size = (int)q.block_size;
    a.qe.num_slots = q.num_slots, a.qe.eps = q.head_eps;
    for (int i = 0; i < 4; ++i) a.next[i] = (const char*)q.next[i], a.next_lines[i] = q.next[i] ? (int64_t)(q.next_bytes[i] / 128) : 0;
    const hipStream_t st = (hipStream_t)stream;
    (void)hipGetLastError();
    const int mt = (int)((q.rows + 15) / 16);
    hipError_t e;
    if (q.hidden == 1024)
        e = mt <= 2 ? launch_block_step<1, 2, 1, 3>(a, st) : launch_block_step<2, 2, 1, 3>(a, st);
    else
        e = mt <= 1 ? launch_block_step<1, 2, 2, 6>(a, st) : launch_block_step<2, 2, 2, 6>(a, st);
    return e == hipSuccess ? AWQ_OK : hip_fail(fn, e);
}
