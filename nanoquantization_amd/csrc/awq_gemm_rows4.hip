// The tiles of awq_gemm_rows.hip for few stages of K, and for widths of less than a tile: y[M, N] = x[M, K] . dequantised W[K, N] (+ bias).
//
// Workgroup: 16 MT rows (MT 5..8) by 128 columns, four waves, one a SIMD.  Wave (bh, kh): the even (bh 0) or odd columns of the
// tile, the first (kh 0) or second 32 of every 64 rows of K; the two meet in LDS at the end.  That way no word is unpacked
// twice in a workgroup, and a wave reads 16 MT rows of x from LDS for 64 columns: 64 of the 128 bytes a cycle at the full
// matrix rate, where four waves side by side would need them all.
// Stage (64 rows of K): x [16 MT rows][128 B], and per half words [32 rows][16], zero words and scales of the 16 word columns;
// all load-to-LDS, kDepth stages in a ring, so five are on their way while one is multiplied (a stage is 0.2 us of matrix
// instructions, a trip to HBM five times that).  The words of the stage after are unpacked to operands beside the matrix
// instructions of this one: a wave alone on its SIMD has only its own instructions to put there.
// Unpacked values are those of awq_dequantize, bit for bit.
// Against the eight waves of awq_gemm_rows.hip a stage takes longer (0.44-0.56 us in fp16 and 0.56-0.62 in bf16 by MT, there 0.38-0.46 and
// 0.43-0.51), but two parts of K meet at the end and not four: 1.2 us less with 80 rows, 1.5 with 128.  160 x 1024 x 1024 in
// four splits, fp16, 11.4 -> 9.6 us; 144 x 2048 x 2048 in four 14.5 -> 13.2; 256 x 5120 x 2048 in eight 23.3 -> 21.6.
#include "awq_common.hpp"
#include "awq_gemm_parts.hpp"

#include <algorithm>

#define AWQ_LPTR(p) ((__attribute__((address_space(3))) void*)(p))

namespace awq {
namespace {

constexpr int kDepth = 6, kThreads = 256, kPad = 132;   // kPad: floats a row of the fp32 tile at the end
constexpr int kHalf = 2048 + 256 + 1024;                 // words, zero words, scales of 32 rows of K
constexpr int stage_bytes(int MT) { return MT * 2048 + 2 * kHalf; }
constexpr int lds_bytes(int MT) { return kDepth * stage_bytes(MT); }
static_assert(lds_bytes(5) >= 80 * kPad * 4 && lds_bytes(8) >= 128 * kPad * 4 && lds_bytes(8) <= 160 * 1024, "LDS");

__device__ __forceinline__ __amdgpu_buffer_rsrc_t resource(const void* p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)0xFFFFFFFFu, 0x00020000);
}

// Four columns (2 f + BH) of word pairs.  A nibble is put under the exponent that gives it the weight 1 -- (w & mask) | magic is
// a float's (half's) 2^e + q -- so unpacking takes one instruction a nibble, and a shift for those that lie too high or low.
template <typename T, int BH>
struct Columns;

template <int BH>
struct Columns<F16, BH> {
    AndOr low, high;     // nibbles 0 and 1 of a 16-bit half: 1024 + q, 64 + q
    uint32_t zp[4], sc[4];
    __device__ __forceinline__ Columns() : low(0x000F000Fu, 0x64006400u), high(0x00F000F0u, 0x54005400u) {}
    __device__ __forceinline__ void embed(uint32_t w1, uint32_t w0, uint32_t (&q)[4]) const {
        const uint32_t v = __builtin_amdgcn_perm(w1, w0, BH ? 0x07060302u : 0x05040100u), u = v >> 8;
        q[0] = low(v), q[1] = high(v), q[2] = low(u), q[3] = high(u);
    }
    __device__ __forceinline__ void set_group(uint32_t zw, u32x4 sv) {
        embed(zw, zw, zp);
#pragma unroll
        for (int f = 0; f < 4; ++f) sc[f] = __builtin_amdgcn_perm(sv[f], sv[f], BH ? 0x03020302u : 0x01000100u);
    }
    __device__ __forceinline__ void pair(uint32_t w0, uint32_t w1, uint32_t (&out)[4]) const {
        uint32_t q[4];
        embed(w1, w0, q);
#pragma unroll
        for (int f = 0; f < 4; ++f) out[f] = as_u32((as_f16x2(q[f]) - as_f16x2(zp[f])) * as_f16x2(sc[f]));
    }
};

template <int BH>
struct Columns<BF16, BH> {
    AndOr at8, at12, at16;   // nibble at that bit of a float: 2^15 + q, 2^11 + q, 2^7 + q
    float sc[4], zp[4];
    __device__ __forceinline__ Columns()
        : at8(0xF00u, 0x47000000u), at12(0xF000u, 0x45000000u), at16(0xF0000u, 0x43000000u) {}
    __device__ __forceinline__ void embed(uint32_t w, float (&q)[4]) const {
        uint32_t b[4];
        if constexpr (BH == 0) {
            const uint32_t u = w << 8;
            b[0] = at8(u), b[1] = at12(u), b[2] = at8(w), b[3] = at12(w);
        } else {
            const uint32_t u = w >> 12;
            b[0] = at16(w), b[1] = at8(u), b[2] = at12(u), b[3] = at16(u);
        }
#pragma unroll
        for (int f = 0; f < 4; ++f) q[f] = __builtin_bit_cast(float, b[f]);
    }
    __device__ __forceinline__ void set_group(uint32_t zw, u32x4 sv) {
        embed(zw, zp);
#pragma unroll
        for (int f = 0; f < 4; ++f) sc[f] = __builtin_bit_cast(float, BH ? sv[f] & 0xFFFF0000u : sv[f] << 16);
    }
    __device__ __forceinline__ void pair(uint32_t w0, uint32_t w1, uint32_t (&out)[4]) const {
        float q0[4], q1[4];
        embed(w0, q0);
        embed(w1, q1);
        // q - z and its product with the scale are exact
#pragma unroll
        for (int f = 0; f < 4; ++f) out[f] = BF16::pack2((q0[f] - zp[f]) * sc[f], (q1[f] - zp[f]) * sc[f]);
    }
};

template <typename T, int MT>
__device__ __forceinline__ void rows_tile(
    const uint16_t* __restrict__ x, const Parts& parts, const uint16_t* __restrict__ bias, float* __restrict__ partials, int M, int K,
    int g, int m_tiles, int items, int steps_per_split, int splits, bool gated) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char s_mem[];
    constexpr int kStage = stage_bytes(MT);
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
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 15, kb = lane >> 4, bh = wave & 1, kh = wave >> 1;
    const int begin = split * steps_per_split, n = min(begin + steps_per_split, K >> 6) - begin;   // 64-row steps
    const int k0 = 64 * begin;
    const int words_at = MT * 2048 + kh * kHalf, zeros_at = words_at + 2048, scales_at = zeros_at + 256;

    f32x4 acc[MT][4];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int f = 0; f < 4; ++f) acc[mt][f] = f32x4{0.f, 0.f, 0.f, 0.f};

    auto run = [&](auto half) {
        constexpr int BH = decltype(half)::value;
        // Pieces of x: eight rows, 128 bytes each; piece i goes to wave i % 4, of an odd MT's the last two to the waves of kh 0.
        constexpr int XP = MT / 2, kLoads = XP + 4 + 1;     // loads a stage of this wave, but for those two
        constexpr bool ODD = MT % 2;
        static_assert((kDepth - 3) * (kLoads + 1) < 64, "the wait counts to 63");
        uint32_t xsrc[XP + ODD];      // bytes
#pragma unroll
        for (int i = 0; i < XP + ODD; ++i) {
            // 16-byte piece p of a row lies at p ^ row / 2: an operand read meets all banks
            const int row = 8 * (4 * i + wave) + (lane >> 3);
            xsrc[i] = ((uint32_t)min(m0 + row, M - 1) * (uint32_t)K + (uint32_t)((lane & 7) ^ ((row >> 1) & 7)) * 8u) * 2u;
        }
        // columns past the last word read it again; nothing of them is stored
        const uint32_t word = (uint32_t)min(tn * 16 + j, words - 1);
        const uint32_t wsrc = ((uint32_t)(8 * kb + 4 * BH) * (uint32_t)words + word) * 4u, zsrc = word * (BH == 0 ? 4u : 16u);
        // of the next stage to be issued: its rows of x and words in bytes, the group of this half and the rows left of it
        uint32_t x_off = (uint32_t)k0 * 2u, w_off = (uint32_t)(k0 + 32 * kh) * (uint32_t)words * 4u;
        int group = __builtin_amdgcn_readfirstlane((k0 + 32 * kh) / g), left = (group + 1) * g - (k0 + 32 * kh);
        const auto rx = resource(x), rw = resource(qweight), rz = resource(BH == 0 ? (const void*)qzeros : (const void*)scales);
        auto issue_x = [&](int slot, int i) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, AWQ_LPTR(s_mem + slot * kStage + (4 * i + wave) * 1024), 16, xsrc[i], x_off, 0, 0);
        };
        // load `i` of a stage but for the odd piece of x
        auto issue = [&](int slot, int i) {
            unsigned char* base = s_mem + slot * kStage;
            if (i < XP) {
                issue_x(slot, i);
            } else if (i < XP + 4) {
                const int p = i - XP;     // piece 4 BH + p: rows p, 8 + p, 16 + p, 24 + p, so that the lanes of an operand read side by side
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, AWQ_LPTR(base + words_at + (4 * BH + p) * 256), 4, wsrc,
                                                         w_off + (uint32_t)(p * words) * 4u, 0, 0);
            } else if (BH == 0) {         // (four times over, which spares a branch)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rz, AWQ_LPTR(base + zeros_at), 4, zsrc, (uint32_t)(group * words) * 4u, 0, 0);
            } else {
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rz, AWQ_LPTR(base + scales_at), 16, zsrc, (uint32_t)(group * words) * 16u, 0, 0);
            }
        };
        auto issued = [&] {
            x_off += 128;
            w_off += 64u * (uint32_t)words * 4u;
            left -= 64;
#pragma unroll
            for (int i = 0; i < 2; ++i) {     // twice over at groups of 32
                const bool over = left <= 0;
                group += over, left += over ? g : 0;
            }
        };
        struct Operands {
            u32x4 a[MT], b[4];
        };
        Columns<T, BH> cols;
        uint32_t w[8], zw;
        u32x4 sv;
        auto read_words = [&](int slot) {
            const unsigned char* base = s_mem + slot * kStage;
#pragma unroll
            for (int r = 0; r < 8; ++r) w[r] = *reinterpret_cast<const uint32_t*>(base + words_at + r * 256 + lane * 4);
            zw = *reinterpret_cast<const uint32_t*>(base + zeros_at + j * 4);
            sv = *reinterpret_cast<const u32x4*>(base + scales_at + j * 16);
        };
        auto read_rows = [&](int slot, Operands& o) {
            const unsigned char* base = s_mem + slot * kStage + j * 128 + (((4 * kh + kb) ^ (j >> 1)) & 7) * 16;
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) o.a[mt] = *reinterpret_cast<const u32x4*>(base + mt * 2048);
        };
        auto unpack = [&](int rp, Operands& o) {
            uint32_t v[4];
            cols.pair(w[2 * rp], w[2 * rp + 1], v);
#pragma unroll
            for (int f = 0; f < 4; ++f) o.b[f][rp] = v[f];
        };
        auto landed = [&](auto newer) {   // all stages but the `newer` last issued
            constexpr int c = decltype(newer)::value * kLoads, more = decltype(newer)::value * (kLoads + ODD);
            if (ODD && kh == 0) __builtin_amdgcn_s_waitcnt(0x0F70 | (more & 15) | ((more >> 4) << 14));
            else __builtin_amdgcn_s_waitcnt(0x0F70 | (c & 15) | ((c >> 4) << 14));
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        int next = 0;    // ring slot of the next stage to be read
        // FULL: a stage is issued, into the slot before the one being multiplied, which every wave had read before it came to
        // this barrier.
        auto stage = [&](auto full, int t, const Operands& cur, Operands& nxt) {
            constexpr bool FULL = decltype(full)::value;
            landed(std::integral_constant<int, FULL ? kDepth - 3 : 0>{});
            // Seven pieces, each with its share of the matrix instructions and what fills their time: the words and rows of the
            // next stage from LDS, the loads of a later one, then the words, which are there by now.
            constexpr int kAll = 4 * MT, kFirst = kAll / 3, kPer = (kAll - kFirst) / 4;
            auto multiply = [&](int from, int to) {
#pragma unroll
                for (int i = 0; i < kAll; ++i)
                    if (i >= from && i < to) acc[i % MT][i / MT] = T::mfma16(cur.a[i % MT], cur.b[i / MT], acc[i % MT][i / MT]);
            };
            const int slot = next >= 2 ? next - 2 : next + kDepth - 2;
            if (FULL && ODD && kh == 0) issue_x(slot, XP);
            __builtin_amdgcn_sched_barrier(0);
            read_words(next);     // past the last stage what an earlier one left there, and nothing uses it
            multiply(0, 2);
            __builtin_amdgcn_sched_barrier(0);
            read_rows(next, nxt);
            multiply(2, kFirst - 3);
#pragma unroll
            for (int i = 2; i < kFirst - 3; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            cols.set_group(zw, sv);
            multiply(kFirst - 3, kFirst);
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int rp = 0; rp < 4; ++rp) {
                // a load to every second or third matrix instruction: four waves' loads take the CU that long
                constexpr int kShare = (kLoads + 3) / 4;
#pragma unroll
                for (int i = 0; i < kShare; ++i)
                    if (FULL && rp * kShare + i < kLoads) issue(slot, rp * kShare + i);
                unpack(rp, nxt);
                multiply(kFirst + rp * kPer, rp == 3 ? kAll : kFirst + (rp + 1) * kPer);
#pragma unroll
                for (int i = 0; i < kPer; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, T::id == AWQ_F16 ? 3 : 6, 0);
                    if (FULL && i < kShare) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (FULL) issued();
            // (or the compiler moves the unpacking to its use, in front of the next stage's matrix instructions)
#pragma unroll
            for (int f = 0; f < 4; ++f) asm volatile("" : "+v"(nxt.b[f]));
            next = next + 1 == kDepth ? 0 : next + 1;
        };
        Operands even, odd;
        for (int t = 0; t < kDepth - 1 && t < n; ++t) {
            if (ODD && kh == 0) issue_x(t, XP);
#pragma unroll
            for (int i = 0; i < kLoads; ++i) issue(t, i);
            issued();
        }
        landed(std::integral_constant<int, 0>{});
        read_words(0);
        read_rows(0, even);
        cols.set_group(zw, sv);
#pragma unroll
        for (int rp = 0; rp < 4; ++rp) unpack(rp, even);
        __builtin_amdgcn_s_waitcnt(0xC07F);   // the LDS reads: one still open here would be waited for in every round of the loop
        next = 1;
        int t = 0;
        for (; t + kDepth < n; t += 2) {
            stage(std::true_type{}, t, even, odd);
            stage(std::true_type{}, t + 1, odd, even);
        }
        if (t + kDepth - 1 < n) {
            stage(std::true_type{}, t, even, odd);
            even = odd;
            ++t;
        }
        for (; t < n; t += 2) {
            stage(std::false_type{}, t, even, odd);
            if (t + 1 < n) stage(std::false_type{}, t + 1, odd, even);
        }
    };
    if (bh == 0) run(std::integral_constant<int, 0>{});
    else run(std::integral_constant<int, 1>{});

    // The halves of K meet.  fp32 tile [16 MT][column c of word j at 16 c + j], written and read without bank conflicts.
    float* tile_f = reinterpret_cast<float*>(s_mem);
    auto at = [&](int mt, int f, int r) { return (16 * mt + 4 * kb + r) * kPad + (2 * f + bh) * 16 + j; };
    __syncthreads();
    if (kh == 1) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int f = 0; f < 4; ++f)
#pragma unroll
                for (int r = 0; r < 4; ++r) tile_f[at(mt, f, r)] = acc[mt][f][r];
    }
    __syncthreads();
    if (kh == 0) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int f = 0; f < 4; ++f)
#pragma unroll
                for (int r = 0; r < 4; ++r) tile_f[at(mt, f, r)] += acc[mt][f][r];
    }
    __syncthreads();
    const int wc = tn * 16 + j;
    if (wc >= words) return;
    for (int p = wave; p < 4 * MT; p += 4) {
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
__global__ __launch_bounds__(kThreads, 2) void rows4_kernel(
    const uint16_t* __restrict__ x, Parts parts, const uint16_t* __restrict__ bias, float* __restrict__ partials, int M, int K,
    int g, int m_tiles, int items, int steps_per_split, int splits, bool gated) {
    rows_tile<T, MT>(x, parts, bias, partials, M, K, g, m_tiles, items, steps_per_split, splits, gated);
}

template <typename T, int MT>
hipError_t launch(const RowsPlan& p, const void* x, const Parts& parts, const void* bias, float* partials, int M, int K, int g,
                  bool gated, hipStream_t st) {
    auto kern = rows4_kernel<T, MT>;
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

hipError_t launch_rows4(const RowsPlan& p, int dtype, const void* x, const Parts& parts, const void* bias, float* partials, int M,
                        int K, int g, bool gated, hipStream_t st) {
#define AWQ_ROWS(T, MT) \
    if (p.mt == MT) return launch<T, MT>(p, x, parts, bias, partials, M, K, g, gated, st);
    if (dtype == AWQ_F16) {
        AWQ_ROWS(F16, 5) AWQ_ROWS(F16, 6) AWQ_ROWS(F16, 7) AWQ_ROWS(F16, 8)
    } else {
        AWQ_ROWS(BF16, 5) AWQ_ROWS(BF16, 6) AWQ_ROWS(BF16, 7) AWQ_ROWS(BF16, 8)
    }
#undef AWQ_ROWS
    return hipErrorInvalidValue;
}

}  // namespace awq
