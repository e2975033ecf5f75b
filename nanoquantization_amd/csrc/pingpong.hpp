// The dense 16-bit matrix product core: a workgroup's tile of 256 weight rows x XR (256 or 128) rows of x, both operands in
// memory with the contraction index contiguous, fp32 accumulation.
//
// What bounds it: the matrix cores at the clock that the chip holds under them (a loop of nothing but MFMAs on random bf16
// operands reaches 2.0 PFLOP/s here).  A SIMD has two waves, w and w + 4, that run the same program half a phase apart:
// while one issues 16 MFMAs the other reads its next operands from LDS and asks for a later stage, and a barrier hands the
// roles over.  A wave's part of the tile is four quadrants, so a stage of 64 contraction elements is four phases; the
// operand reads are dealt out 8, 4, 8, 4 (one half of a stage's x rows is read a phase early, into registers of its own) --
// with 12, 4, 8, 0 the phase of twelve lasts longer than the other wave's MFMAs: 1.44 -> 1.47 PFLOP/s.  Loads go straight
// to LDS and are waited for by count, three phases after they were asked for; a part of a buffer is asked for again as soon as both waves of
// every SIMD have read it.  XR = 128 has half the x rows, two phases a stage and room for a third buffer.
//
// Measured on 12288 x 4096 bf16 weights: 8192 rows 560-570 us (1.45-1.47 PFLOP/s; the same tiles with one barrier a stage and
// operand reads mixed between a wave's own MFMAs 630 us), 8192^3 740 us (1.49); 1024 rows 80 us with XR = 256 and 96 with
// 128, 512 rows 66 and 48: the smaller tile where the larger one leaves CUs without a tile.
#pragma once

#include "awq_common.hpp"

namespace awq {

template <typename T, int XR>
struct PingPong {
    static_assert(XR == 256 || XR == 128, "x rows of a tile");
    static constexpr int kThreads = 512, kWR = 256, kStage = 64;
    static constexpr int kWM = XR == 256 ? 2 : 4, kWN = 8 / kWM;              // waves along the weight rows, along the x rows
    static constexpr int MI = kWR / kWM / 16, NJ = XR / kWN / 16;             // 16 x 16 tiles of a wave
    static constexpr int kBufs = XR == 256 ? 2 : 3;
    static constexpr int kX = kWR * 128, kBuf = kX + XR * 128;                // [buffer][weight rows | x rows], 128 bytes a row
    static constexpr int kLds = kBufs * kBuf;
    static constexpr int kHalf = kWR / kWM / 2;                               // weight rows of the first half of a wave's tiles
    static constexpr int kXLoads = XR / 64;

    int lane, wave, lo, hi, wm, wn;
    f32x4 acc[MI][NJ];

    __device__ __forceinline__ PingPong() {
        lane = threadIdx.x & 63;
        wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        lo = lane & 15, hi = lane >> 4, wm = wave % kWM, wn = wave / kWM;
    }

    // Rows of the tile that load q of a stage brings for a lane, eight lanes a row, and the 16-byte piece of the stage's
    // 128 bytes: pieces are stored at position piece ^ (row / 2 % 8), which spreads the 16 rows of an operand read over all
    // banks; load-to-LDS writes linearly, so the swizzle is in the source addresses.
    static __host__ __device__ __forceinline__ int w_row(int q, int wave, int lane) { return 64 * q + 8 * wave + (lane >> 3); }     // q < 4
    static __host__ __device__ __forceinline__ int x_row(int q, int wave, int lane) {                                                // q < kXLoads
        // XR = 256: loads 0 and 2 bring the first 32 rows of every wave's 64, loads 1 and 3 the others
        if (XR == 256) return 64 * ((q & 2) + (wave >> 2)) + 32 * (q & 1) + 8 * (wave & 3) + (lane >> 3);
        return 64 * q + 8 * wave + (lane >> 3);
    }
    // Byte offset in an operand of `rows` rows of the piece that comes to `tile_row` from source row `row`: past the end the
    // last row again, of which nothing is stored.
    static __host__ __device__ __forceinline__ uint32_t source(int row, int rows, uint32_t row_bytes, int tile_row, int lane) {
        return (uint32_t)(row < rows ? row : rows - 1) * row_bytes + ((lane & 7) ^ ((tile_row >> 1) & 7)) * 16;
    }
    // Byte offset of stage t in a row.  The pipeline asks for two stages past the last one, which nobody reads: the last one
    // again.  With `source` no request leaves an operand; the count of requests, which the waits rely on, stays.
    static __host__ __device__ __forceinline__ int stage_bytes(int t, int steps) { return (t < steps ? t : steps - 1) * (kStage * 2); }

    // vw[q], vx[q]: `source` of this lane's piece of its rows in the buffers rw and rx.
    __device__ __forceinline__ void run(unsigned char* s_mem, __amdgpu_buffer_rsrc_t rw, const uint32_t (&vw)[4],
                                        __amdgpu_buffer_rsrc_t rx, const uint32_t (&vx)[kXLoads], int steps) {
        const auto load = [&](__amdgpu_buffer_rsrc_t r, uint32_t v, int first_row, int at, int t) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)(s_mem + at + first_row * 128),
                                                     16, v, stage_bytes(t, steps), 0, 0);
        };
        const auto load_w = [&](int q, int t, int at) { load(rw, vw[q], 64 * q + 8 * wave, at, t); };
        const auto load_x = [&](int q, int t, int at) {
            load(rx, vx[q], XR == 256 ? 64 * ((q & 2) + (wave >> 2)) + 32 * (q & 1) + 8 * (wave & 3) : 64 * q + 8 * wave,
                 at + kX, t);
        };
        const int swz = ((hi ^ (lo >> 1)) & 7) * 16;
        const int a_at = (wm * (kWR / kWM) + lo) * 128 + swz, b_at = kX + (wn * (XR / kWN) + lo) * 128 + swz;
        const auto read = [&](int at, int tile, int s) {
            return *reinterpret_cast<const u32x4*>(s_mem + ((at ^ (64 * s)) + tile * 2048));
        };
        // this wave's LDS reads are in registers; then the barrier that hands the matrix cores to the other wave.  Nothing is
        // scheduled across.
        const auto hand_over = [] {
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
        };
        const auto operands_there = [&] {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            hand_over();
        };
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

        if constexpr (XR == 256) {
            // the parts of a stage: weight rows 64 .. 127 and 192 .. 255 (loads 1, 3), the others (0, 2), and the two halves of
            // every wave's x rows.  They are asked for in the order in which they are read first.
            const auto load_a = [&](int h, int t, int at) { load_w(h, t, at), load_w(2 + h, t, at); };
            const auto load_b = [&](int h, int t, int at) { load_x(h, t, at), load_x(2 + h, t, at); };
            u32x4 a[2][4], b_even[2][2], b_odd[2][2], b1[2][2];
            const auto read_a = [&](int h, int at) {
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int i = 0; i < 4; ++i) a[s][i] = read(at + a_at, 4 * h + i, s);
            };
            const auto read_b = [&](u32x4 (&b)[2][2], int h, int at) {
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int j = 0; j < 2; ++j) b[s][j] = read(at + b_at, 2 * h + j, s);
            };
            const auto multiply = [&](int ha, int hb, const u32x4 (&b)[2][2]) {
#pragma unroll
                for (int s = 0; s < 2; ++s)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int j = 0; j < 2; ++j)
                            acc[4 * ha + i][2 * hb + j] = T::mfma16(a[s][i], b[s][j], acc[4 * ha + i][2 * hb + j]);
            };
            load_b(0, 0, 0), load_a(0, 0, 0), load_b(1, 0, 0), load_a(1, 0, 0);
            load_b(0, 1, kBuf), load_a(0, 1, kBuf), load_b(1, 1, kBuf);
            __builtin_amdgcn_s_waitcnt(0x0F76);         // vmcnt(6): stage 0 is there
            __builtin_amdgcn_s_barrier();
            if (wave >= 4) __builtin_amdgcn_s_barrier();    // half a phase behind from here on
            int at = 0;
            read_b(b_even, 0, 0);
            const auto stage = [&](int t, const u32x4 (&b0)[2][2], u32x4 (&next)[2][2]) {
                read_a(0, at);
                load_a(1, t + 1, at ^ kBuf);
                operands_there();
                multiply(0, 0, b0);
                hand_over();
                read_b(b1, 1, at);
                load_b(0, t + 2, at);
                operands_there();
                multiply(0, 1, b1);
                hand_over();
                read_a(1, at);
                load_a(0, t + 2, at);
                __builtin_amdgcn_s_waitcnt(0x0F7A);     // vmcnt(10): the next stage's first x rows
                operands_there();
                multiply(1, 1, b1);
                hand_over();
                read_b(next, 0, at ^ kBuf);
                load_b(1, t + 2, at);
                __builtin_amdgcn_s_waitcnt(0x0F76);     // vmcnt(6): all of the next stage
                operands_there();
                multiply(1, 0, b0);
                hand_over();
                at ^= kBuf;
            };
            static_assert((kBuf & (kBuf - 1)) == 0, "buffers alternate by an exclusive or");
            int t = 0;
#pragma unroll 1
            for (; t + 1 < steps; t += 2) {
                stage(t, b_even, b_odd);
                stage(t + 1, b_odd, b_even);
            }
            if (t < steps) stage(t, b_even, b_odd);
        } else {
            u32x4 a[4], b[4];
            const auto read_ab = [&](int s, int at) {
#pragma unroll
                for (int i = 0; i < 4; ++i) a[i] = read(at + a_at, i, s), b[i] = read(at + b_at, i, s);
            };
            const auto multiply = [&] {
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) acc[i][j] = T::mfma16(a[i], b[j], acc[i][j]);
            };
            const auto first_half = [&](int t, int at) { load_w(0, t, at), load_w(1, t, at), load_x(0, t, at); };
            const auto second_half = [&](int t, int at) { load_w(2, t, at), load_w(3, t, at), load_x(1, t, at); };
            first_half(0, 0), second_half(0, 0), first_half(1, kBuf), second_half(1, kBuf);
            __builtin_amdgcn_s_waitcnt(0x0F76);         // vmcnt(6): stage 0 is there
            __builtin_amdgcn_s_barrier();
            if (wave >= 4) __builtin_amdgcn_s_barrier();
            int at = 0, next = 2 * kBuf;                // stage t + 2 goes where stage t - 1 was
#pragma unroll 1
            for (int t = 0; t < steps; ++t) {
                read_ab(0, at);
                first_half(t + 2, next);
                operands_there();
                multiply();
                hand_over();
                read_ab(1, at);
                second_half(t + 2, next);
                __builtin_amdgcn_s_waitcnt(0x0F76);     // vmcnt(6): the next stage
                operands_there();
                multiply();
                hand_over();
                at = at == 2 * kBuf ? 0 : at + kBuf;
                next = next == 2 * kBuf ? 0 : next + kBuf;
            }
        }
        if (wave < 4) __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_s_waitcnt(0x0F70);             // the stages past the end have landed: the LDS is the caller's
        __syncthreads();
    }

    // The tile as 16-bit values, through LDS in whole rows of COLS consecutive values.  value(i, j) gives four consecutive
    // columns (two words) of tile pair (i, j), i < COLS / 16 / kWM; store(row, column, eight values) writes 16 bytes of a row.
    template <int COLS, typename V, typename S>
    __device__ __forceinline__ void write(unsigned char* s_mem, V&& value, S&& store) {
        to_lds<COLS>(s_mem, value);
#pragma unroll 4
        for (int q = threadIdx.x; q < XR * COLS / 8; q += kThreads) {
            const int r = q / (COLS / 8), c = q % (COLS / 8) * 8;
            store(r, c, stored<COLS>(s_mem, r, c));
        }
    }
    template <int COLS, typename V>
    __device__ __forceinline__ void to_lds(unsigned char* s_mem, V&& value) {
        constexpr int kTiles = COLS / 16 / kWM, kBytes = COLS * 2;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int i = 0; i < kTiles; ++i) {
                const int r = wn * (XR / kWN) + 16 * j + lo, c = wm * (COLS / kWM) + 16 * i + 4 * hi;
                *reinterpret_cast<u32x2*>(s_mem + r * kBytes + ((c * 2) ^ ((r & 15) << 4))) = value(i, j);
            }
        __syncthreads();
    }
    template <int COLS>
    static __device__ __forceinline__ u32x4 stored(const unsigned char* s_mem, int r, int c) {
        return *reinterpret_cast<const u32x4*>(s_mem + r * COLS * 2 + ((c * 2) ^ ((r & 15) << 4)));
    }

    // Eight values a thread and store of `write<256>`: how many, and which store n of this thread is.
    static constexpr int kStores = XR * 32 / kThreads;
    static __device__ __forceinline__ int store_row(int n) { return (threadIdx.x + n * kThreads) >> 5; }
    static __device__ __forceinline__ int store_column() { return (threadIdx.x & 31) * 8; }
};

// Workgroups go round-robin over the 8 XCDs, each with its own L2: every XCD takes a contiguous run of the tiles, in blocks
// of 8 x tiles with the weight tiles outside, so that both operands are met again in that L2.  Any grid of a multiple of 8
// that has a workgroup per tile; false for the workgroups that get none.  (`workgroup`: blockIdx.x, an argument so that the
// host can enumerate the map.)
__host__ __device__ __forceinline__ bool xcd_tile(int workgroup, int x_tiles, int w_tiles, int& xt, int& wt) {
    const int total = x_tiles * w_tiles, per = (total + 7) >> 3;
    // past the end of its XCD's run: in a larger grid the sum below would be a tile of the next XCD's
    if (workgroup >> 3 >= per) return false;
    const int id = (workgroup & 7) * per + (workgroup >> 3);
    if (id >= total) return false;
    const int block = id / (8 * w_tiles), in_block = id - block * 8 * w_tiles;
    const int rows = x_tiles - 8 * block < 8 ? x_tiles - 8 * block : 8;
    xt = 8 * block + in_block % rows;
    wt = in_block / rows;
    return true;
}

}  // namespace awq
