// y[M, N] = x[M, K] . dequantised W[K, N] (+ bias) for 17 to about 1000 rows: too many for the GEMV, too few for 256 x 256 tiles
// to cover the CUs (333 rows by 9720 columns are 76 of them) and for a dequantised weight to pay for its trip through memory.
//
// Workgroup: 16 MT rows (MT 2..8) by 128 columns, eight waves.  Wave (turn, kh, bh): the even (bh 0) or odd columns of the tile,
// the first (kh 0) or second 32 rows of K of every second stage of 64 (turn); the four parts of K meet in LDS at the end.  That
// way no word is unpacked twice in a workgroup.  A SIMD has one wave of either turn, half a round apart: while one multiplies,
// the other reads its next words and rows of x from LDS and unpacks the words to operands, and a barrier hands the roles over;
// the unpacking (22 vector instructions in bf16, 14 in fp16 for 8 x 1 weights a lane) is as long as the matrix instructions of
// seven (five) row tiles.  Up to four row tiles leave registers and LDS for two workgroups on a CU, which fill each other's waits.
// Stage (64 rows of K): x [16 MT rows][128 B], words [2 halves][32 rows][16], scales and zero words of the two halves; all
// load-to-LDS in pieces of 1 KiB, 16 bytes a lane, in a ring of kDepth stages.
// Unpacked values are those of awq_dequantize, bit for bit; bf16 scales of 2^113 and more, whose quick way to them overflows, in a
// second pass of the waves that meet one.
// What bounds it: the phases, 0.38 us a stage at five row tiles and 0.46 at eight in fp16, 0.44 and 0.51 in bf16.  333 x 2816 x 9720 in
// fp16, over the time a CU is busy: the matrix cores 34 %, the vector units 39 %, the LDS 20 % without conflicts; of a wave's time a
// third goes by at hand-overs and for LDS reads, a third for the issue of its next instruction.  (With the loads from memory answered
// by zeros the time is the same.)  The end, where the four parts of K meet, takes 1.2 us with five row tiles and 1.5 with eight more than
// without the exchange; few stages are left to awq_gemm_rows4.hip, where two parts meet.
// Measured: 333 x 2816 x 9720 in fp16, groups of 64, 29.8 -> 26.7 us against those four waves, in bf16 34.9 -> 30.4; 640 x 2048 x 6144
// in bf16 28 -> 26.  5120 x 25600 in groups of 64 at 64 rows, bf16, 46 -> 41 us
// against the 64 x 256 tiles of awq_gemm.hip, 5120 x 17408 at 57 rows 44 -> 31 and at 32 rows 29 -> 25, 15296 x 4680 at 18 rows
// 33 -> 23; 5120 x 25600 at 100 rows 69 -> 47 against its 128 x 128 tiles.
#include "awq_common.hpp"
#include "awq_gemm_parts.hpp"

#include <algorithm>
#include <type_traits>

#define AWQ_LPTR(p) ((__attribute__((address_space(3))) void*)(p))
#define AWQ_GPTR(p) ((__attribute__((address_space(1))) const void*)(p))

namespace awq {
namespace {

constexpr int kThreads = 512, kPad = 132;                 // kPad: floats a row of the fp32 tile at the end
constexpr int stage_bytes(int MT) { return MT * 2048 + 4096 + 1024; }      // x, words, scales and zero words of 64 rows of K
constexpr int per_cu(int MT) { return MT <= 4 ? 2 : 1; }                      // workgroups that share a CU
// Four stages on the way while one is read: more take longer to ask for than they save (128 rows of 16384 columns, fp16, K of 128 /
// 1024 / 4096: 9.5 / 16.8 / 38.8 us with seven to ten, 9.2 / 15.5 / 37.4 with four, 9.1 / 15.5 / 37.2 with three).
constexpr int kDepth = 5;
// 16 x 64 tiles that a wave gives away at the end, in the first and in the second exchange
constexpr int pairs(int MT) { return (MT + 1) / 2; }
constexpr int fours(int MT) { return (MT + 3) / 4; }
constexpr int lds_bytes(int MT) {
    return std::max({kDepth * stage_bytes(MT), 8 * 4096 * pairs(MT), 8 * 4096 * fours(MT) + 16 * MT * kPad * 4});
}
static_assert(2 * lds_bytes(2) <= 160 * 1024 && 2 * lds_bytes(3) <= 160 * 1024 && 2 * lds_bytes(4) <= 160 * 1024, "two on a CU");
static_assert(lds_bytes(5) <= 160 * 1024 && lds_bytes(6) <= 160 * 1024 && lds_bytes(7) <= 160 * 1024 && lds_bytes(8) <= 160 * 1024, "LDS");

// The even (bh 0) or odd columns 2 f + bh of word pairs.  A nibble is put under the exponent that gives it the weight 1 --
// (w & mask) | magic is a float's (half's) 2^e + q -- so unpacking takes one instruction a nibble, and a shift for those that
// lie too high or low.  bh is a register and not a template argument: the four roles of waves share one piece of code.
template <typename T>
struct Columns;

template <>
struct Columns<F16> {
    AndOr low, high;     // nibbles 0 and 1 of a 16-bit half: 1024 + q, 64 + q
    uint32_t zp[4], sc[4], pick, pick_scale;
    __device__ __forceinline__ explicit Columns(int bh)
        : low(0x000F000Fu, 0x64006400u), high(0x00F000F0u, 0x54005400u), pick(bh ? 0x07060302u : 0x05040100u),
          pick_scale(bh ? 0x03020302u : 0x01000100u) {}
    __device__ __forceinline__ void embed(uint32_t w1, uint32_t w0, uint32_t (&q)[4]) const {
        const uint32_t v = __builtin_amdgcn_perm(w1, w0, pick), u = v >> 8;
        q[0] = low(v), q[1] = high(v), q[2] = low(u), q[3] = high(u);
    }
    __device__ __forceinline__ void set_group(uint32_t zw, u32x4 sv) {
        embed(zw, zw, zp);
#pragma unroll
        for (int f = 0; f < 4; ++f) sc[f] = __builtin_amdgcn_perm(sv[f], sv[f], pick_scale);
    }
    __device__ __forceinline__ void pair(uint32_t w0, uint32_t w1, uint32_t (&out)[4]) const {
        uint32_t q[4];
        embed(w1, w0, q);
#pragma unroll
        for (int f = 0; f < 4; ++f) out[f] = as_u32((as_f16x2(q[f]) - as_f16x2(zp[f])) * as_f16x2(sc[f]));
    }
};

template <>
struct Columns<BF16> {
    AndOr at8, at12;         // nibble at that bit of a float: 2^15 + q, 2^11 + q
    float sc[4], nzs[4];     // the scale, and minus scale times what a nibble of the zero point gives
    int up, down;
    __device__ __forceinline__ explicit Columns(int bh) : at8(0xF00u, 0x47000000u), at12(0xF000u, 0x45000000u), up(bh ? 0 : 16), down(bh ? 16 : 0) {}
    __device__ __forceinline__ void embed(uint32_t word, float (&q)[4]) const {
        const uint32_t w = word >> down, u = w << 8;
        q[0] = __builtin_bit_cast(float, at8(u)), q[1] = __builtin_bit_cast(float, at12(u));
        q[2] = __builtin_bit_cast(float, at8(w)), q[3] = __builtin_bit_cast(float, at12(w));
    }
    __device__ __forceinline__ void set_group(uint32_t zw, u32x4 sv) {
        embed(zw, nzs);
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            sc[f] = __builtin_bit_cast(float, (sv[f] << up) & 0xFFFF0000u);
            nzs[f] *= -sc[f];
        }
    }
    __device__ __forceinline__ void pair(uint32_t w0, uint32_t w1, uint32_t (&out)[4]) const {
        float q0[4], q1[4];
        embed(w0, q0);
        embed(w1, q1);
        // 2^15 + z has 16 bits and the scale 8: the product kept in nzs is exact, and so is the sum, (q - z) * s; unless it leaves the
        // range of a float, and no weight of the column is a number
#pragma unroll
        for (int f = 0; f < 4; ++f)
            out[f] = BF16::pack2(__builtin_fmaf(q0[f], sc[f], nzs[f]), __builtin_fmaf(q1[f], sc[f], nzs[f]));
    }
    // The same for any scale.
    __device__ __forceinline__ void pair_exact(uint32_t w0, uint32_t w1, uint32_t zw, uint32_t (&out)[4]) const {
        float q0[4], q1[4], z[4];
        embed(w0, q0);
        embed(w1, q1);
        embed(zw, z);
#pragma unroll
        for (int f = 0; f < 4; ++f) out[f] = BF16::pack2((q0[f] - z[f]) * sc[f], (q1[f] - z[f]) * sc[f]);
    }
};

template <typename T, int MT>
__device__ __forceinline__ void rows_tile(
    const uint16_t* __restrict__ x, const Parts& parts, const uint16_t* __restrict__ bias, float* __restrict__ partials, int M, int K,
    int g, int m_tiles, int items, int steps_per_split, int splits, bool gated) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char s_mem[];
    constexpr int kStage = stage_bytes(MT), kWords = MT * 2048, kScales = kWords + 4096;
    constexpr int kPairs = pairs(MT), kFours = fours(MT), kGiven = 8 * 4096 * kFours;
    // runs of consecutive items to each XCD: the row tiles of a column tile read its words through one L2
    const int per = gridDim.x >> 3, id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (id >= items) return;
    const int split = id % splits, tile = id / splits;
    const int m0 = tile % m_tiles * (16 * MT), column = tile / m_tiles * 128, part = parts.of(column);
    const uint32_t* __restrict__ qweight = pick_part(parts.qweight, part);
    const uint16_t* __restrict__ scales = pick_part(parts.scales, part);
    const uint32_t* __restrict__ qzeros = pick_part(parts.qzeros, part);
    uint16_t* __restrict__ y = pick_part(parts.y, part);
    const int N = pick_part(parts.columns, part), first = pick_part(parts.first, part), tn = (column - first) >> 7;
    partials += (size_t)splits * M * first;        // a part's partials [split][M][its columns] behind those of the parts before it
    const int words = N >> 3;
    const int word0 = min(16 * tn, words - 16);     // a last tile that is not whole begins earlier (N >= 128) and stores some columns again
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 15, kb = lane >> 4, bh = wave & 1, kh = (wave >> 1) & 1, turn = wave >> 2;
    const int begin = split * steps_per_split, n = min(begin + steps_per_split, K >> 6) - begin;   // 64-row steps
    const int k0 = 64 * begin;

    f32x4 acc[MT][4];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int f = 0; f < 4; ++f) acc[mt][f] = f32x4{0.f, 0.f, 0.f, 0.f};

    // A stage in pieces of 1024 bytes, piece i to wave i % 8: 2 MT of x (eight rows, 128 bytes each), four of words (16 rows of
    // 64 bytes), and the scales and zero words of its two groups of 32 rows, which come in one.
    constexpr int kPieces = 2 * MT + 5, kMost = (kPieces + 7) / 8, kFull = kPieces % 8 ? kPieces % 8 : 8;   // waves below kFull bring kMost
    constexpr int kGroupPiece = 2 * MT + 4;
    static_assert((kDepth - 2) * kMost < 64, "the wait counts to 63");
    uint32_t source[kMost], offset[kMost], step[kMost];      // bytes: of a lane, of the next stage to be asked for, from stage to stage
    uint64_t operand[kMost];
#pragma unroll
    for (int q = 0; q < kMost; ++q) {
        const int i = 8 * q + wave;
        const uint64_t p = i < 2 * MT ? reinterpret_cast<uint64_t>(x) : reinterpret_cast<uint64_t>(qweight);
        // (a descriptor that the compiler does not see to be the same in all lanes costs a loop over the lanes)
        operand[q] = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(p >> 32)) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane((int)p);
        if (i < 2 * MT) {
            // 16-byte piece p of a row lies at p ^ row / 2: an operand read meets all banks
            const int row = 8 * i + (lane >> 3);
            source[q] = ((uint32_t)min(m0 + row, M - 1) * (uint32_t)K + (uint32_t)((lane & 7) ^ ((row >> 1) & 7)) * 8u) * 2u;
            offset[q] = (uint32_t)k0 * 2u, step[q] = 128u;
        } else {
            // row 8 a + b of a half's 32 lies at 4 b + a: the lanes of an operand read lie side by side
            const int at = 16 * ((i - 2 * MT) & 1) + (lane >> 2);
            source[q] = ((uint32_t)((at & 3) * 8 + (at >> 2)) * (uint32_t)words + (uint32_t)(word0 + 4 * (lane & 3))) * 4u;
            offset[q] = (uint32_t)(k0 + 32 * ((i - 2 * MT) >> 1)) * (uint32_t)words * 4u, step[q] = 64u * (uint32_t)words * 4u;
        }
    }
    // Scales: lanes 0 .. 15 of the first 32 rows, 16 .. 31 of the second; zero words: lanes 32 .. 35 and 36 .. 39 (and again).
    const bool second = lane < 32 ? lane & 16 : lane & 4;
    const unsigned char* group_base = lane < 32 ? reinterpret_cast<const unsigned char*>(scales) + 16 * (size_t)(word0 + j)
                                                : reinterpret_cast<const unsigned char*>(qzeros) + 4 * (size_t)(word0 + 4 * (lane & 3));
    const uint32_t group_bytes = (uint32_t)words * (lane < 32 ? 16u : 4u);
    uint32_t group = (uint32_t)((k0 + (second ? 32 : 0)) / g);              // of this lane, in the next stage to be asked for
    int left = (int)(group + 1) * g - (k0 + (second ? 32 : 0));             // rows of K until it ends
    const uint32_t last_group = (uint32_t)(K / g) - 1u;

    // stages asked for, the ring's place (in bytes) of the next one, and the size that the operands' descriptors give: none past the end
    int asked = 0, ask_at = 0, open = -1;
    // piece q of the stage `asked`; past the last stage nothing is read (the count of requests, which the waits rely on, stays)
    auto ask = [&](int q) {
        const int i = 8 * q + wave;
        if (q < kMost - 1 || wave < kFull) {
            if (q == kGroupPiece / 8 && wave == kGroupPiece % 8) {
                __builtin_amdgcn_global_load_lds(AWQ_GPTR(group_base + (size_t)min(group, last_group) * group_bytes),
                                                 AWQ_LPTR(s_mem + ask_at + kScales), 16, 0, 0);
                left -= 64;
#pragma unroll
                for (int c = 0; c < 2; ++c) {     // twice over at groups of 32
                    const bool over = left <= 0;
                    group += over, left += over ? g : 0;
                }
            } else {
                const auto r = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(operand[q]), 0, __builtin_amdgcn_readfirstlane(open), 0x00020000);
                __builtin_amdgcn_raw_ptr_buffer_load_lds(r, AWQ_LPTR(s_mem + ask_at + i * 1024), 16, source[q], offset[q], 0, 0);
                offset[q] += step[q];
            }
        }
    };
    auto asked_all = [&] {
        open = __builtin_amdgcn_readfirstlane(++asked < n ? -1 : 0);
        asm volatile("" : "+s"(open));
        ask_at = ask_at + kStage == kDepth * kStage ? 0 : ask_at + kStage;
    };
    // Where the registers suffice, the words of a wave's next stage come beside its matrix instructions, a phase before its rows.
    constexpr bool kEarly = MT != 4;
    constexpr int kOnTheWay = kDepth - (kEarly ? 3 : 2);
    // This wave's share of all stages but the kOnTheWay last asked for is there; then the barrier that hands the matrix cores
    // to the other wave of the SIMD.  Nothing is scheduled across.
    auto hand_over = [&] {
        __builtin_amdgcn_sched_barrier(0);
        constexpr int most = kOnTheWay * kMost, fewer = kOnTheWay * (kMost - 1);
        if (wave < kFull) __builtin_amdgcn_s_waitcnt(0x0F70 | (most & 15) | ((most >> 4) << 14));
        else __builtin_amdgcn_s_waitcnt(0x0F70 | (fewer & 15) | ((fewer >> 4) << 14));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll 1
    for (int t = 0; t < kDepth - 1; ++t) {
#pragma unroll
        for (int q = 0; q < kMost; ++q) ask(q);
        asked_all();
    }
    hand_over();
    if (turn == 1) {       // half a round behind from here on
#pragma unroll
        for (int q = 0; q < kMost; ++q) ask(q);
        asked_all();
        hand_over();
    }
    Columns<T> cols(bh);
    const int x_at = j * 128 + (((4 * kh + kb) ^ (j >> 1)) & 7) * 16;
    const int w_at = kWords + kh * 2048 + lane * 4;
    const int z_at = kScales + 512 + kh * 64 + j * 4, s_at = kScales + kh * 256 + j * 16;
    int at = turn * kStage;       // of the stage this wave reads next
    uint32_t w[8], zw;
    u32x4 sv;
    auto read_words = [&](int at) {
        const unsigned char* base = s_mem + at;
#pragma unroll
        for (int r = 0; r < 8; ++r) w[r] = *reinterpret_cast<const uint32_t*>(base + w_at + r * 256);
        zw = *reinterpret_cast<const uint32_t*>(base + z_at);
        sv = *reinterpret_cast<const u32x4*>(base + s_at);
    };
    auto read_rows = [&](int at, u32x4 (&a)[MT]) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) a[mt] = *reinterpret_cast<const u32x4*>(s_mem + at + x_at + mt * 2048);
    };
    if (kEarly) read_words(at);
    __builtin_amdgcn_s_waitcnt(0xC07F);     // LDS and scalar reads: one still open here would be waited for in every round of the loop
#pragma unroll 1
    for (int t = turn; t < n; t += 2) {
        u32x4 a[MT], b[4];
        if (!kEarly) read_words(at);
        read_rows(at, a);
        // (without this the compiler mixes the group's constants into the unpacking: 64 rows of 16384 columns, K of 4096, 35 -> 37 us)
        if (!kEarly && T::id == AWQ_BF16) __builtin_amdgcn_sched_barrier(0);
        cols.set_group(zw, sv);
#pragma unroll
        for (int rp = 0; rp < 4; ++rp) {
            if (rp == 2) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int q = 0; q < kMost; ++q) ask(q);
                asked_all();
                __builtin_amdgcn_sched_barrier(0);
            }
            uint32_t v[4];
            cols.pair(w[2 * rp], w[2 * rp + 1], v);
#pragma unroll
            for (int f = 0; f < 4; ++f) b[f][rp] = v[f];
        }
        // (or the compiler moves the unpacking to its use, behind the barrier)
#pragma unroll
        for (int f = 0; f < 4; ++f) asm volatile("" : "+v"(b[f]));
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) asm volatile("" : "+v"(a[mt]));
        at = at + 2 * kStage >= kDepth * kStage ? at + (2 - kDepth) * kStage : at + 2 * kStage;
        hand_over();
        if (kEarly) read_words(at);     // past the last stage whatever lies there, and nothing uses it
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < kMost; ++q) {
#pragma unroll
            for (int i = 4 * MT * q / kMost; i < 4 * MT * (q + 1) / kMost; ++i) acc[i % MT][i / MT] = T::mfma16(a[i % MT], b[i / MT], acc[i % MT][i / MT]);
            __builtin_amdgcn_sched_barrier(0);
            ask(q);
            __builtin_amdgcn_sched_barrier(0);
        }
        asked_all();
        hand_over();
    }
    if ((n & 1) == turn) __builtin_amdgcn_s_barrier();      // the turn that had one phase fewer
    __builtin_amdgcn_s_waitcnt(0x0F70);                     // what was asked for past the end has come: the LDS is free

    if constexpr (T::id == AWQ_BF16) {
        // A weight that was no number has made all rows of its column none, whatever x holds: this wave's part of the tile once more,
        // straight from memory.  (A branch among the unpacking that looks at the scales costs a third of the whole kernel's time.)
        const auto none = [&](int f, int r) { return !(__builtin_fabsf(acc[0][f][r]) <= 3.402823466e38f); };
        bool some = false;
#pragma unroll
        for (int f = 0; f < 4; ++f) some |= none(f, 0);
        uint64_t off = 0;       // columns that hold none in all of the first 16 rows: a row of x that is none leaves the others
        if (__builtin_amdgcn_ballot_w64(some)) {
#pragma unroll
            for (int f = 0; f < 4; ++f) {
                uint64_t lanes = __builtin_amdgcn_ballot_w64(none(f, 0) && none(f, 1) && none(f, 2) && none(f, 3));
                lanes &= lanes >> 32;
                off |= lanes & (lanes >> 16) & 0xFFFFu;
            }
        }
        if (off != 0) {
            int row = j, part_k = 8 * kb;       // (hidden from the compiler, which would keep what the two passes share through the first)
            asm volatile("" : "+v"(row), "+v"(part_k));
            const int word = word0 + row;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int f = 0; f < 4; ++f) acc[mt][f] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
            for (int t = turn; t < n; t += 2) {
                const int k = k0 + 64 * t + 32 * kh;
                const size_t at_group = (size_t)(k / g) * words + word;
                const uint32_t zero = qzeros[at_group];
                cols.set_group(zero, *reinterpret_cast<const u32x4*>(scales + 8 * at_group));
                u32x4 b[4];
#pragma unroll
                for (int rp = 0; rp < 4; ++rp) {
                    const uint32_t* p = qweight + (size_t)(k + part_k + 2 * rp) * words + word;
                    uint32_t v[4];
                    cols.pair_exact(p[0], p[words], zero, v);
#pragma unroll
                    for (int f = 0; f < 4; ++f) b[f][rp] = v[f];
                }
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    const u32x4 a = *reinterpret_cast<const u32x4*>(x + (size_t)min(m0 + 16 * mt + row, M - 1) * K + k + part_k);
#pragma unroll
                    for (int f = 0; f < 4; ++f) acc[mt][f] = T::mfma16(a, b[f], acc[mt][f]);
                }
            }
        }
    }

    // The four parts of K meet, (0 + 1) + (2 + 3), and every wave ends with a quarter of the row tiles: the two of a turn give each
    // other every second tile, then the turns every second of those, in the layout of the registers; the sums go to an fp32 tile
    // [16 MT][column c of word j at 16 c + j], written and read without bank conflicts.  (All through such tiles, of which LDS
    // holds two, the end took 2.2 us with 128 rows; so 1.7.)
    float* tile_f = reinterpret_cast<float*>(s_mem + kGiven);
    const auto meet = [&](auto khc, auto turnc) {
        constexpr int KH = decltype(khc)::value, TURN = decltype(turnc)::value;
        f32x4* mine = reinterpret_cast<f32x4*>(s_mem) + wave * (kPairs * 256) + lane;
        const f32x4* first = reinterpret_cast<const f32x4*>(s_mem) + (wave ^ 2) * (kPairs * 256) + lane;
        f32x4* mine2 = reinterpret_cast<f32x4*>(s_mem) + wave * (kFours * 256) + lane;
        const f32x4* other = reinterpret_cast<const f32x4*>(s_mem) + (wave ^ 4) * (kFours * 256) + lane;
#pragma unroll
        for (int mt = 1 - KH; mt < MT; mt += 2)
#pragma unroll
            for (int f = 0; f < 4; ++f) mine[(mt / 2 * 4 + f) * 64] = acc[mt][f];
        __syncthreads();
#pragma unroll
        for (int mt = KH; mt < MT; mt += 2)
#pragma unroll
            for (int f = 0; f < 4; ++f) acc[mt][f] += first[(mt / 2 * 4 + f) * 64];
        __syncthreads();
#pragma unroll
        for (int mt = KH + 2 * (1 - TURN); mt < MT; mt += 4)
#pragma unroll
            for (int f = 0; f < 4; ++f) mine2[(mt / 4 * 4 + f) * 64] = acc[mt][f];
        __syncthreads();
#pragma unroll
        for (int mt = KH + 2 * TURN; mt < MT; mt += 4)
#pragma unroll
            for (int f = 0; f < 4; ++f) {
                const f32x4 sum = acc[mt][f] + other[(mt / 4 * 4 + f) * 64];
#pragma unroll
                for (int r = 0; r < 4; ++r) tile_f[(16 * mt + 4 * kb + r) * kPad + (2 * f + bh) * 16 + j] = sum[r];
            }
    };
    __syncthreads();
    using Zero = std::integral_constant<int, 0>;
    using One = std::integral_constant<int, 1>;
    if (kh == 0 && turn == 0) meet(Zero{}, Zero{});
    else if (kh == 0) meet(Zero{}, One{});
    else if (turn == 0) meet(One{}, Zero{});
    else meet(One{}, One{});
    __syncthreads();
    const int wc = word0 + j;
    for (int p = wave; p < 4 * MT; p += 8) {
        const int row = 16 * (p >> 2) + 4 * kb + (p & 3), m = m0 + row;
        if (m >= M) continue;
        float v[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) v[c] = tile_f[row * kPad + 16 * c + j];
        if (splits > 1) {
            float* dst = partials + ((size_t)split * M + m) * N + 8 * (size_t)wc;
            *reinterpret_cast<f32x4*>(dst) = f32x4{v[0], v[1], v[2], v[3]};
            *reinterpret_cast<f32x4*>(dst + 4) = f32x4{v[4], v[5], v[6], v[7]};
            continue;
        }
        if (bias) {
            const u32x4 bv = *reinterpret_cast<const u32x4*>(bias + 8 * (size_t)wc);
#pragma unroll
            for (int c = 0; c < 8; ++c)
                v[c] = add_bias<T>(v[c], T::to_f32((uint16_t)((c & 1) ? (bv[c >> 1] >> 16) : (bv[c >> 1] & 0xFFFFu))));
        }
        u32x4 o;
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = T::pack2(v[2 * i], v[2 * i + 1]);
        if (gated) swiglu_word_store<T>(o, y + (size_t)m * (N >> 1), wc);
        else *reinterpret_cast<u32x4*>(y + (size_t)m * N + 8 * (size_t)wc) = o;
    }
}

template <typename T, int MT>
__global__ __launch_bounds__(kThreads, 2 * per_cu(MT)) void rows_kernel(
    const uint16_t* __restrict__ x, Parts parts, const uint16_t* __restrict__ bias, float* __restrict__ partials, int M, int K,
    int g, int m_tiles, int items, int steps_per_split, int splits, bool gated) {
    rows_tile<T, MT>(x, parts, bias, partials, M, K, g, m_tiles, items, steps_per_split, splits, gated);
}

// y = dtype(sum over splits, in split order) of every part; a thread owns 8 consecutive columns of one row.
template <typename T>
__global__ __launch_bounds__(256) void rows_sum_kernel(const float* __restrict__ partials, Parts parts, int64_t M, int splits) {
    const int64_t vec = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int per_row = parts.total >> 3;
    if (vec >= M * per_row) return;
    const int64_t m = vec / per_row;
    const int column = (int)(vec % per_row) * 8, part = parts.of(column);
    const int N = pick_part(parts.columns, part), first = pick_part(parts.first, part);
    f32x4 lo, hi;
    add_splits(partials + (size_t)splits * M * first + (size_t)m * N + (column - first), (size_t)M * N, splits, lo, hi);
    *reinterpret_cast<u32x4*>(pick_part(parts.y, part) + (size_t)m * N + (column - first)) =
        u32x4{T::pack2(lo[0], lo[1]), T::pack2(lo[2], lo[3]), T::pack2(hi[0], hi[1]), T::pack2(hi[2], hi[3])};
}

template <typename T, int MT>
hipError_t launch(const RowsPlan& p, const void* x, const Parts& parts, const void* bias, float* partials, int M, int K, int g,
                  bool gated, hipStream_t st) {
    auto kern = rows_kernel<T, MT>;
    static bool raised = false;      // once per process and instantiation
    if (!raised) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 lds_bytes(MT));
        if (e != hipSuccess) return e;
        raised = true;
    }
    (void)hipGetLastError();
    const int items = p.m_tiles * p.n_tiles * p.splits;
    kern<<<dim3((unsigned)(cdiv(items, 8) * 8)), dim3(kThreads), lds_bytes(MT), st>>>(
        (const uint16_t*)x, parts, (const uint16_t*)bias, partials, M, K, g, p.m_tiles, items, p.steps_per_split, p.splits, gated);
    return hipGetLastError();
}

}  // namespace

RowsPlan make_rows_plan(int64_t M, int64_t N, int64_t K, int64_t g, int dtype, int split_k) {
    RowsPlan p{};
    // 32-bit offsets into x, the words and the scales
    if (M < 1 || N < 8 || N % 8 != 0 || K < 64 || K % 64 != 0 || g < 32 || g % 32 != 0 || K % g != 0 ||
        M * K >= (1ll << 31) || (K + 64) * N >= (1ll << 32) || cdiv(M, 128) * cdiv(N, 128) * 16 >= (1ll << 31))
        return p;
    const int64_t m_tiles = cdiv(M, 128), n_tiles = cdiv(N, 128), steps = K / 64;
    p.m_tiles = (int)m_tiles, p.n_tiles = (int)n_tiles;
    const bool narrow = N < 128;      // less than a tile's columns: the four waves alone take that
    p.mt = (int)std::max<int64_t>(narrow ? 5 : 2, cdiv(cdiv(M, m_tiles), 16));
    // From 65 rows on the four waves are the faster ones up to 18 stages a split in fp16 and 14 in bf16: their end takes 1.2 to 1.5 us
    // less, a stage 0.1 more.  Against the eight, by stages: fp16 0.83 of the time with 2, 0.91 with 8, 0.97 with 16, 0.99 to 1.02
    // with 20, 1.02 with 24; bf16 0.87, 0.94, 1.01 with 16, 1.02 with 20.
    const int few = dtype == AWQ_F16 ? 18 : 14, t = dtype == AWQ_F16 ? 0 : 1;
    // Microseconds, by type and MT: a stage of the four waves; of the eight with a CU to itself and with two workgroups on it; and of
    // filling the ring, the tile's sums and the launch.  A K split writes its fp32 sums and reads them again in a second launch.
    // From five row tiles on within 10 % of 96 of 100 measured times (42 weights, 130 to 2048 rows, every split).
    constexpr double kFour[2][4] = {{0.45, 0.445, 0.485, 0.515}, {0.56, 0.56, 0.595, 0.59}};     // [fp16, bf16][MT - 5]
    constexpr double kAlone[2][7] = {{0.28, 0.295, 0.38, 0.375, 0.38, 0.405, 0.46}, {0.345, 0.37, 0.445, 0.44, 0.465, 0.485, 0.515}};   // [MT - 2]
    constexpr double kShared[2][3] = {{0.455, 0.45, 0.495}, {0.52, 0.53, 0.575}};
    const auto four = [&](int64_t s) { return narrow || (p.mt >= 5 && cdiv(steps, s) <= few); };
    const auto us = [&](int64_t s) {
        const int64_t items = m_tiles * n_tiles * s, n = cdiv(steps, s);
        const double moved = (double)s * (double)(M * N) * 8;
        if (p.mt <= 4) {
            const int64_t last = items % 512;
            const double fixed = 4.6 + 0.95 * p.mt, alone = kAlone[t][p.mt - 2] * (double)n + fixed;
            const double whole = kShared[t][p.mt - 2] * (double)n + fixed;
            return (double)(items / 512) * whole + (last == 0 ? 0 : last > 256 ? whole : alone) + (s > 1 ? 2.5 + moved / 5.0e6 : 0);
        }
        const double round = four(s) ? kFour[t][p.mt - 5] * (double)n + 4.1 + 0.31 * p.mt : kAlone[t][p.mt - 2] * (double)n + 5.5 + 0.26 * p.mt;
        // (full rounds take longer once a launch lasts: 512 x 4096 x 24576, three of them, 128 us in fp16 where this alone says 111)
        const double rounds = (double)cdiv(items, 256), all = rounds * round, full = (double)items / (256 * rounds);
        const double held = full > 0.9 ? (t == 0 ? 0.17 : 0.07) * std::max(0.0, all - 24) : 0;
        return all + held + (s > 1 ? 2 + moved / 3.6e6 : 0);
    };
    int64_t best = 1;
    // (splits of more than a round of the CUs were not timed from five row tiles on)
    for (int64_t s = 2; s <= 16 && s * 4 <= steps && (p.mt <= 4 || m_tiles * n_tiles * s <= 256); ++s)
        if (us(s) < us(best)) best = s;
    if (split_k > 0) best = std::min<int64_t>(split_k, steps);
    p.steps_per_split = (int)cdiv(steps, best);
    p.splits = (int)cdiv(steps, p.steps_per_split);
    p.four = four(p.splits);
    p.us = us(p.splits);
    return p;
}

hipError_t launch_rows(const RowsPlan& p, int dtype, const void* x, const Parts& parts, const void* bias, int M, int K, int g,
                       void* workspace, bool gated, hipStream_t st) {
    float* partials = p.splits > 1 ? reinterpret_cast<float*>(reinterpret_cast<char*>(workspace) + kCounterBytes) : nullptr;
#define AWQ_ROWS(T, MT) \
    if (p.mt == MT) e = launch<T, MT>(p, x, parts, bias, partials, M, K, g, gated, st);
    hipError_t e = hipErrorInvalidValue;
    if (p.four) {
        e = launch_rows4(p, dtype, x, parts, bias, partials, M, K, g, gated, st);
    } else if (dtype == AWQ_F16) {
        AWQ_ROWS(F16, 2) AWQ_ROWS(F16, 3) AWQ_ROWS(F16, 4)
        AWQ_ROWS(F16, 5) AWQ_ROWS(F16, 6) AWQ_ROWS(F16, 7) AWQ_ROWS(F16, 8)
    } else {
        AWQ_ROWS(BF16, 2) AWQ_ROWS(BF16, 3) AWQ_ROWS(BF16, 4)
        AWQ_ROWS(BF16, 5) AWQ_ROWS(BF16, 6) AWQ_ROWS(BF16, 7) AWQ_ROWS(BF16, 8)
    }
#undef AWQ_ROWS
    if (e != hipSuccess || p.splits == 1) return e;
    if (parts.count == 1) return launch_splitk_reduce(dtype, partials, bias, parts.y[0], M, parts.total, p.splits, st, gated);
    const dim3 grid((unsigned)cdiv((int64_t)M * (parts.total >> 3), 256)), block(256);
    if (dtype == AWQ_F16) rows_sum_kernel<F16><<<grid, block, 0, st>>>(partials, parts, M, p.splits);
    else rows_sum_kernel<BF16><<<grid, block, 0, st>>>(partials, parts, M, p.splits);
    return hipGetLastError();
}

}  // namespace awq
