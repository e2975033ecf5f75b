// Offline path on the device: per-group asymmetric 4-bit min/max quantisation of an fp32 weight
// [N, K] fused with the AWQ packing, producing qweight [K, N/8], qzeros [K/g, N/8] and qscales
// [K/g, N] directly.  The words equal those of the reference's quantise -> transpose -> pack chain in fp32 (round half
// to even): step size and zero point by its operations, codes by a product with the reciprocal that is decided by the
// division wherever the two could round apart (code_of).
#include <chrono>
#include <type_traits>

#include "awq_common.hpp"

namespace awq {
namespace {

__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = fminf(v, __shfl_xor(v, o));
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}

// The group's step size and zero point: RN((hi - lo) / 15) from 1e-5 up, and -rint(lo / s) in 0..15.
__device__ __forceinline__ float group_scale(float lo, float hi) {
    return __fdiv_rn(fmaxf(__fsub_rn(hi, lo), 1e-5f), 15.f);
}
__device__ __forceinline__ float group_zero(float lo, float s) {
    return fminf(fmaxf(-rintf(__fdiv_rn(lo, s)), 0.f), 15.f);
}
// The code of a weight: rint(RN(v / s)) + z in 0..15.  The packer's own pass over the fake-quantised weight,
// rint(RN(RN((q - z) s) / s) + z), gives q back: both roundings move the quotient by less than 2^-23 of a whole number of
// at most 15, and where s is infinite or the product overflows the conversion of the infinity ends in the same nibble.
//
// r = RN(1 / s): v r is within 2^-22 of RN(v / s), relatively, so that the two round to the same whole number unless v r is
// that close to halfway between two; only there (and for quotients that have no fraction bits to speak of, infinities and
// NaN, which fail the comparison) the division is done.  Two divisions a weight were 50 vector instructions and the
// vector ALU's 80 us for 50 M weights.
__device__ __forceinline__ float code_of(float v, float s, float r, float z) {
    float t = __fmul_rn(v, r), n = rintf(t);
    if (!(fabsf(fabsf(t - n) - 0.5f) > 0x1p-21f * fmaxf(fabsf(t), 1.f))) n = rintf(__fdiv_rn(v, s));
    return fminf(fmaxf(__fadd_rn(n, z), 0.f), 15.f);
}

// min / max over the 16 lanes of a DPP row (over each half of it if HALF)
template <bool HALF>
__device__ __forceinline__ void row_min_max(float& lo, float& hi) {
    const auto at = [](float v, auto ctrl) {
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), decltype(ctrl)::value, 0xF,
                                                                     0xF, true));
    };
    const auto step = [&](auto ctrl) {
        lo = fminf(lo, at(lo, ctrl));
        hi = fmaxf(hi, at(hi, ctrl));
    };
    step(std::integral_constant<int, 0xB1>{});      // quad_perm 1,0,3,2
    step(std::integral_constant<int, 0x4E>{});      // quad_perm 2,3,0,1
    step(std::integral_constant<int, 0x141>{});     // row_half_mirror
    if (!HALF) step(std::integral_constant<int, 0x140>{});     // row_mirror
}

// Group sizes 32, 64 and 128, 16-byte aligned weights: read once, written in whole lines.  A workgroup of four waves takes
// 4 * WPW words (8 weight rows each) x 128 columns of the weight.  A wave loads the 8 rows of a word at once: lane (p, j) =
// (lane / 16, lane % 16) holds columns 4 j .. 4 j + 3 and 64 + 4 j .. of rows p and p + 4, so that a group's minimum and
// maximum are a reduction over the 16 lanes of a DPP row and no lane ever needs another row's scale.  The nibbles of a
// word come together across the four DPP rows with the row-swapping permutes (reduce-scatter: lane (p, j) ends up with the
// words of columns 4 j + p and 64 + 4 j + p) and leave through LDS, 4 * WPW consecutive words of a packed row at a time.
//
// Bound by memory (4 B read, 0.52 B written per weight).  12288 x 4096, g = 128: 147 us with one wave per word and group,
// 64-byte pieces of packed rows written 4 B at a time and the weight read twice, 48.5 us like this (4.7 TB/s; a large copy runs at 5.0 here).  WPW = 8 writes
// 128-byte pieces; small weights take WPW = 2 to reach more CUs.
template <typename T, int G, int WPW>
__global__ __launch_bounds__(256) void quantize_tile_kernel(const float* __restrict__ w, uint32_t* __restrict__ qweight,
                                                            uint32_t* __restrict__ qzeros, uint16_t* __restrict__ qscales,
                                                            int N, int K, int* __restrict__ nan_flag) {
    constexpr int W = 4 * WPW, GROUPS = 128 / G;        // words and groups of a tile
    __shared__ uint32_t s_word[128][W + 1];
    __shared__ uint32_t s_zero[GROUPS][W];
    __shared__ uint16_t s_scale[GROUPS][8 * W];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, p = lane >> 4, j = lane & 15;
    const int words = N >> 3, k0 = blockIdx.x * 128, i0 = blockIdx.y * W;
    // columns past the end (K is a multiple of G only) read a group that exists; what comes of them is not stored
    int col[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int c = k0 + 64 * h + 4 * j;
        col[h] = c < K ? c : 4 * j % G;
    }
    const int shift = 16 * (p & 1) + 4 * (p >> 1);      // nibble of column p; column p + 4 is 8 bits further
    bool nan = false;
    f32x4 v[2][2], next[2][2];                          // [row p, p + 4][column half]
    const auto load = [&](int u, f32x4 (&to)[2][2]) {
        const int i = min(i0 + wave * WPW + u, words - 1);
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                to[r][h] = *reinterpret_cast<const f32x4*>(w + (size_t)(8 * i + p + 4 * r) * K + col[h]);
    };
    load(0, next);
#pragma unroll 2
    for (int u = 0; u < WPW; ++u) {
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
            for (int h = 0; h < 2; ++h) v[r][h] = next[r][h];
        if (u + 1 < WPW) load(u + 1, next);
        const int x = wave * WPW + u;
        uint32_t part[2][4];
        float code[2][2][4];
        uint32_t zbits[2] = {0, 0};
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            float lo[2], hi[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const f32x4 e = v[r][h];
                nan |= (e[0] != e[0]) | (e[1] != e[1]) | (e[2] != e[2]) | (e[3] != e[3]);
                lo[h] = fminf(fminf(e[0], e[1]), fminf(e[2], e[3]));
                hi[h] = fmaxf(fmaxf(e[0], e[1]), fmaxf(e[2], e[3]));
            }
            if (G == 128) {
                lo[0] = fminf(lo[0], lo[1]);
                hi[0] = fmaxf(hi[0], hi[1]);
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (G == 128 && h == 1) break;
                row_min_max<G == 32>(lo[h], hi[h]);
            }
            float s[2], rs[2], z[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (G == 128 && h == 1) {
                    s[1] = s[0], rs[1] = rs[0], z[1] = z[0];
                    break;
                }
                s[h] = group_scale(lo[h], hi[h]);
                rs[h] = __fdiv_rn(1.f, s[h]);
                z[h] = group_zero(lo[h], s[h]);
                zbits[h] |= (uint32_t)z[h] << (shift + 8 * r);
                const int group = G == 128 ? 0 : G == 64 ? h : 2 * h + (j >> 3);
                if (j % (G == 32 ? 8 : 16) == 0) s_scale[group][8 * x + p + 4 * r] = T::from_f32(s[h]);
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int e = 0; e < 4; ++e) code[r][h][e] = code_of(v[r][h][e], s[h], rs[h], z[h]);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                part[h][e] = (uint32_t)__builtin_fmaf(code[1][h][e], 256.f, code[0][h][e]) << shift;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const auto a = __builtin_amdgcn_permlane16_swap(part[h][0], part[h][1], false, false);
            const auto b = __builtin_amdgcn_permlane16_swap(part[h][2], part[h][3], false, false);
            const auto c = __builtin_amdgcn_permlane32_swap(a[0] | a[1], b[0] | b[1], false, false);
            s_word[64 * h + 4 * j + p][x] = c[0] | c[1];
            if (G == 128 && h == 1) continue;
            const auto y = __builtin_amdgcn_permlane16_swap(zbits[h], zbits[h], false, false);
            const auto q = __builtin_amdgcn_permlane32_swap(y[0] | y[1], y[0] | y[1], false, false);
            if (p == 0 && j % (G == 32 ? 8 : 16) == 0) s_zero[G == 32 ? 2 * h + (j >> 3) : h][x] = q[0] | q[1];
        }
    }
    if (nan_flag && nan) __hip_atomic_store(nan_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __syncthreads();
    const int x = threadIdx.x % W, rows = min(128, K - k0), groups = rows / G;
    if (i0 + x < words) {
        for (int k = threadIdx.x / W; k < rows; k += 256 / W) qweight[(size_t)(k0 + k) * words + i0 + x] = s_word[k][x];
        for (int q = threadIdx.x / W; q < groups; q += 256 / W) qzeros[(size_t)(k0 / G + q) * words + i0 + x] = s_zero[q][x];
    }
    for (int c = threadIdx.x; c < 8 * W * groups; c += 256) {
        const int q = c / (8 * W), n = c % (8 * W);
        if (8 * i0 + n < N) qscales[(size_t)(k0 / G + q) * N + 8 * i0 + n] = s_scale[q][n];
    }
}

// Any group size and alignment.  One wave per (word column i, group kg): 8 output columns n = 8i..8i+7, g input rows k.
// Weight rows are read 64 consecutive floats at a time (coalesced); a lane ends up with the 8 nibbles of one packed word
// per k it owns.
template <typename T>
__global__ __launch_bounds__(256) void quantize_pack_kernel(const float* __restrict__ w,
                                                            uint32_t* __restrict__ qweight,
                                                            uint32_t* __restrict__ qzeros,
                                                            uint16_t* __restrict__ qscales, int N, int K, int g,
                                                            int* __restrict__ nan_flag) {
    const int lane = threadIdx.x & 63;
    const int words = N >> 3, groups = K / g;
    const int64_t item = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (item >= (int64_t)words * groups) return;
    const int i = (int)(item % words), kg = (int)(item / words);
    const float* base = w + (size_t)(8 * i) * K + (size_t)kg * g;

    float s[8], r[8], z[8];
    bool nan = false;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        float lo = INFINITY, hi = -INFINITY;
        for (int kk = lane; kk < g; kk += 64) {
            const float v = base[(size_t)c * K + kk];
            nan |= v != v;
            lo = fminf(lo, v);
            hi = fmaxf(hi, v);
        }
        lo = wave_min(lo);
        hi = wave_max(hi);
        s[c] = group_scale(lo, hi);
        r[c] = __fdiv_rn(1.f, s[c]);
        z[c] = group_zero(lo, s[c]);
    }
    if (nan_flag && nan) __hip_atomic_store(nan_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    for (int kk = lane; kk < g; kk += 64) {
        uint32_t word = 0;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const float v = base[(size_t)c * K + kk];
            word |= (uint32_t)code_of(v, s[c], r[c], z[c]) << nibble_shift(c);
        }
        qweight[(size_t)(kg * g + kk) * words + i] = word;
    }
    if (lane == 0) {
        uint32_t zw = 0;
#pragma unroll
        for (int c = 0; c < 8; ++c) zw |= ((uint32_t)(int)z[c] & 15u) << nibble_shift(c);
        qzeros[(size_t)kg * words + i] = zw;
    }
    if (lane < 8) {
        float sv = s[0];
#pragma unroll
        for (int c = 1; c < 8; ++c) sv = lane == c ? s[c] : sv;
        qscales[(size_t)kg * N + 8 * i + lane] = T::from_f32(sv);
    }
}

template <typename T, int G>
void launch_tiles(const float* w, uint32_t* qw, uint32_t* qz, uint16_t* qs, int N, int K, int* nan_flag, hipStream_t st) {
    const unsigned kt = (unsigned)cdiv(K, 128);
    // two workgroups a CU with the wide tile, or the narrow one
    if (cdiv(N, 256) * kt >= 512)
        quantize_tile_kernel<T, G, 8><<<dim3(kt, (unsigned)cdiv(N, 256)), 256, 0, st>>>(w, qw, qz, qs, N, K, nan_flag);
    else
        quantize_tile_kernel<T, G, 2><<<dim3(kt, (unsigned)cdiv(N, 64)), 256, 0, st>>>(w, qw, qz, qs, N, K, nan_flag);
}

template <typename T>
void launch_quantize(const float* w, uint32_t* qw, uint32_t* qz, uint16_t* qs, int N, int K, int g, int* nan_flag,
                     hipStream_t st) {
    // the tile kernel's 16-byte loads need aligned rows (K is a multiple of g), its grid at most 65535 tiles of rows
    const bool tiles = ((uintptr_t)w & 15) == 0 && cdiv(N, 64) <= 65535;
    if (tiles && g == 128) return launch_tiles<T, 128>(w, qw, qz, qs, N, K, nan_flag, st);
    if (tiles && g == 64) return launch_tiles<T, 64>(w, qw, qz, qs, N, K, nan_flag, st);
    if (tiles && g == 32) return launch_tiles<T, 32>(w, qw, qz, qs, N, K, nan_flag, st);
    const int64_t items = (int64_t)(N / 8) * (K / g);
    quantize_pack_kernel<T><<<dim3((unsigned)cdiv(items, 4)), 256, 0, st>>>(w, qw, qz, qs, N, K, g, nan_flag);
}

}  // namespace
}  // namespace awq

using namespace awq;

static int quantize_pack(const char* fn, const float* weight, int32_t* qweight, void* qscales, int32_t* qzeros, int64_t N,
                         int64_t K, int64_t group_size, int dtype, int32_t* nan_flag, void* stream) {
    if (!weight || !qweight || !qscales || !qzeros) {
        set_error("%s: null pointer argument", fn);
        return AWQ_ERR_INVALID_ARG;
    }
    if (dtype != AWQ_F16 && dtype != AWQ_BF16) {
        set_error("%s: dtype must be AWQ_F16 (0) or AWQ_BF16 (1), got %d", fn, dtype);
        return AWQ_ERR_INVALID_ARG;
    }
    if (N <= 0 || K <= 0 || group_size <= 0 || N % 8 != 0 || K % group_size != 0) {
        set_error("%s: need N %% 8 == 0 and K %% group_size == 0 (N=%lld K=%lld g=%lld)", fn, (long long)N,
                  (long long)K, (long long)group_size);
        return AWQ_ERR_INVALID_ARG;
    }
    const int64_t items = (N / 8) * (K / group_size);
    if (N > 0x7fffffff || K > 0x7fffffff || cdiv(items, 4) > 0x7fffffff) {
        set_error("%s: problem too large", fn);
        return AWQ_ERR_UNSUPPORTED;
    }
    hipStream_t st = (hipStream_t)stream;
    (void)hipGetLastError();
    if (dtype == AWQ_F16)
        launch_quantize<F16>(weight, (uint32_t*)qweight, (uint32_t*)qzeros, (uint16_t*)qscales, (int)N, (int)K,
                             (int)group_size, nan_flag, st);
    else
        launch_quantize<BF16>(weight, (uint32_t*)qweight, (uint32_t*)qzeros, (uint16_t*)qscales, (int)N, (int)K,
                              (int)group_size, nan_flag, st);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? AWQ_OK : hip_fail(fn, e);
}

extern "C" int awq_quantize_pack(const float* weight, int32_t* qweight, void* qscales, int32_t* qzeros, int64_t N,
                                 int64_t K, int64_t group_size, int dtype, void* stream) {
    return quantize_pack("awq_quantize_pack", weight, qweight, qscales, qzeros, N, K, group_size, dtype, nullptr, stream);
}

extern "C" int awq_quantize_pack_flagged(const float* weight, int32_t* qweight, void* qscales, int32_t* qzeros, int64_t N,
                                         int64_t K, int64_t group_size, int dtype, int32_t* nan_flag, void* stream) {
    return quantize_pack("awq_quantize_pack_flagged", weight, qweight, qscales, qzeros, N, K, group_size, dtype, nan_flag,
                         stream);
}

namespace awq {
namespace {

__global__ void announce_kernel(int* word) { __hip_atomic_store(word, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM); }

}  // namespace
}  // namespace awq

// The caller needs the NaN flag at once.  A kernel behind the first one writes a word that the host looks at: 4 us sooner than the stream's
// signal (1024 x 2048 24.2 us a call with the signal, 20.2 with the word; 4096 x 12288 64.1 and 60.1).  After a millisecond (work queued
// before, an error, a stream that is being captured) the stream is asked instead.
extern "C" int awq_quantize_pack_checked(const float* weight, int32_t* qweight, void* qscales, int32_t* qzeros, int64_t N,
                                         int64_t K, int64_t group_size, int dtype, int32_t* words, void* stream) {
    const char* fn = "awq_quantize_pack_checked";
    if (!words) {
        set_error("%s: null pointer argument", fn);
        return AWQ_ERR_INVALID_ARG;
    }
    const int rc = quantize_pack(fn, weight, qweight, qscales, qzeros, N, K, group_size, dtype, words, stream);
    if (rc != AWQ_OK) return rc;
    hipStream_t st = (hipStream_t)stream;
    int32_t* done = words + 1;
    announce_kernel<<<1, 1, 0, st>>>(done);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) {
        const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(1);
        do {
            for (int look = 0; look < 64; ++look)
                if (__atomic_load_n(done, __ATOMIC_ACQUIRE)) return AWQ_OK;
        } while (std::chrono::steady_clock::now() < until);
    }
    const hipError_t waited = hipStreamSynchronize(st);
    if (e == hipSuccess) e = waited;
    return e == hipSuccess ? AWQ_OK : hip_fail(fn, e);
}
