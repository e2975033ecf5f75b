// Kernel (c) for many rows: the weight dequantised once into scratch memory, [columns][K] (the exact RN_dtype((q - z) s) that
// every other path multiplies), then the dense product of pingpong.hpp.
//
// The fused kernels unpack a weight tile for every 256 rows of x, which costs the SIMD's issue port as much as a third of the
// MFMAs do (awq_gemm_regb.hip); from about a thousand rows on, one pass that writes the weight out (2.5 bytes a weight, and
// the product then finds it in the Infinity Cache) is the cheaper way.  Scratch is a slab of columns of at most 256 MiB (the
// size of that cache), wider weights are taken slab by slab.
#include <algorithm>

#include "awq_gemm_parts.hpp"
#include "pingpong.hpp"

namespace awq {
namespace {

constexpr int64_t kSlabBytes = 256ll << 20;

// Where a slab's columns go: rows of ldy values from column `first` on; a tile lies in one output.
struct Outputs {
    uint16_t* y[kMaxParts];
    int ldy[kMaxParts], first[kMaxParts];
    Outputs(void* to, int ld) {
        for (int i = 0; i < kMaxParts; ++i) y[i] = static_cast<uint16_t*>(to), ldy[i] = ld, first[i] = i ? 0x7fffffff : 0;
    }
    explicit Outputs(const Parts& p) {
        for (int i = 0; i < kMaxParts; ++i) y[i] = p.y[i], ldy[i] = p.columns[i], first[i] = p.first[i];
    }
};

// GATED: the slab's columns are gate and up words in turn; a tile is 128 gate columns and their up columns, a wave's first
// tiles gate, the others up.
// ADD: y = residual + dtype(product), rounded once more, as a separate addition leaves it; residual lies as y does.  Its rows are asked for in
// front of the product (256-row tiles have no registers left for that: behind it), and the addition's own pass over three tensors is gone: 8192 x
// 1024 of K 2048 / 3072 with a pass of its own 50.6 / 62.1 us, so 43.0 / 56.1; 8192 x 2560 of K 4096 198 and 180.
template <typename T, int XR, bool GATED, bool ADD>
__global__ __launch_bounds__(512, 2) void dense_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ wt,
                                                       const uint16_t* __restrict__ bias, const uint16_t* residual,
                                                       Outputs out, int M, int cols, int K, int x_tiles, int w_tiles) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char s_mem[];
    using P = PingPong<T, XR>;
    int xt, nt;
    if (!xcd_tile((int)blockIdx.x, x_tiles, w_tiles, xt, nt)) return;
    P p;
    const int m0 = xt * XR, n0 = nt * (GATED ? 128 : 256), out_cols = GATED ? cols / 2 : cols;
    const uint32_t row_bytes = (uint32_t)K * 2;
    uint32_t vw[4], vx[P::kXLoads];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int r = P::w_row(q, p.wave, p.lane);
        int col = n0 + r;
        if (GATED) {
            const int c = n0 + r / (2 * P::kHalf) * P::kHalf + r % P::kHalf;
            col = 16 * (c >> 3) + (c & 7) + 8 * (r / P::kHalf & 1);
        }
        vw[q] = P::source(col, cols, row_bytes, r, p.lane);
    }
    const int rows = min(XR, M - m0);
#pragma unroll
    for (int q = 0; q < P::kXLoads; ++q) {
        const int r = P::x_row(q, p.wave, p.lane);
        vx[q] = P::source(r, rows, row_bytes, r, p.lane);
    }
    const auto rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(wt), 0, cols * row_bytes, 0x00020000);
    const auto rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(x) + (size_t)m0 * K, 0,
                                                      rows * row_bytes, 0x00020000);
    u32x4 old[ADD ? P::kStores : 1];
    const auto ask = [&] {
        const auto ro = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(residual) + (size_t)m0 * out.ldy[0] + n0, 0,
                                                          (uint32_t)((rows - 1) * out.ldy[0] + min(256, cols - n0)) * 2, 0x00020000);
#pragma unroll
        for (int n = 0; n < P::kStores; ++n)        // past the tile's end: zero, or the next row's
            old[n] = __builtin_amdgcn_raw_buffer_load_b128(ro, (uint32_t)(P::store_row(n) * out.ldy[0] + P::store_column()) * 2, 0, 0);
    };
    if constexpr (ADD && XR == 128) ask();
    p.run(s_mem, rw, vw, rx, vx, K / P::kStage);
    if constexpr (ADD && XR != 128) ask();
    const int part = (n0 >= out.first[1]) + (n0 >= out.first[2]), ldy = pick_part(out.ldy, part);
    using Result = std::conditional_t<ADD, uint16_t*, uint16_t* __restrict__>;       // the residual may be the result
    const Result y = pick_part(out.y, part) + (n0 - pick_part(out.first, part));
    const auto store = [&](int r, int c, u32x4 v) {
        if (m0 + r < M && n0 + c < out_cols) *reinterpret_cast<u32x4*>(y + (size_t)(m0 + r) * ldy + c) = v;
    };
    if constexpr (ADD) {
        p.template to_lds<256>(s_mem, [&](int i, int j) {
            const f32x4 v = p.acc[i][j];
            return u32x2{T::pack2(v[0], v[1]), T::pack2(v[2], v[3])};
        });
#pragma unroll
        for (int n = 0; n < P::kStores; ++n) {
            const int row = P::store_row(n), c = P::store_column();
            const u32x4 v = p.template stored<256>(s_mem, row, c);
            u32x4 sum;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const auto half = [&](uint32_t w, int h) { return T::to_f32((uint16_t)(w >> (16 * h))); };
                sum[i] = T::pack2(half(old[n][i], 0) + half(v[i], 0), half(old[n][i], 1) + half(v[i], 1));
            }
            store(row, c, sum);
        }
    } else if constexpr (GATED) {
        p.template write<128>(s_mem, [&](int i, int j) {
            const f32x4 g4 = p.acc[i][j], u4 = p.acc[i + P::MI / 2][j];
            float o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {       // dtype(SiLU(gate)) * up of the rounded products, as swiglu_pair_store
                const float g = T::to_f32(T::from_f32(g4[e])), u = T::to_f32(T::from_f32(u4[e]));
                o[e] = T::to_f32(T::from_f32(g / (1.f + __expf(-g)))) * u;
            }
            return u32x2{T::pack2(o[0], o[1]), T::pack2(o[2], o[3])};
        }, store);
    } else if (bias) {
        p.template write<256>(s_mem, [&](int i, int j) {
            const f32x4 v = p.acc[i][j];
            const int c = min(n0 + p.wm * (256 / P::kWM) + 16 * i + 4 * p.hi, cols - 4);
            const u32x2 b = *reinterpret_cast<const u32x2*>(bias + c);
            float o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = add_bias<T>(v[e], T::to_f32((uint16_t)(b[e >> 1] >> (16 * (e & 1)))));
            return u32x2{T::pack2(o[0], o[1]), T::pack2(o[2], o[3])};
        }, store);
    } else {
        p.template write<256>(s_mem, [&](int i, int j) {
            const f32x4 v = p.acc[i][j];
            return u32x2{T::pack2(v[0], v[1]), T::pack2(v[2], v[3])};
        }, store);
    }
}

// Columns of a slab: all, or equal parts of at most kSlabBytes, in whole tiles.
int64_t slab_columns(int64_t N, int64_t K) {
    const int64_t most = std::max<int64_t>(256, kSlabBytes / (2 * K) / 256 * 256);
    return std::min(cdiv(cdiv(N, cdiv(N, most)), 256) * 256, cdiv(N, 256) * 256);
}

// Microseconds of the product over one slab: rounds of 256 workgroups, a stage of 1.42 us with 256-row tiles and 0.8 with
// 128-row ones (measured with full rounds; 8192 x 4096 x 12288 six rounds of 64 stages 560 us, 512 x 4096 x 12288 one round
// of the small tile 48 us), and filling and storing a tile.
double product_us(int64_t M, int64_t slab, int64_t K, int xr) {
    return (double)cdiv(cdiv(M, xr) * cdiv(slab, 256), 256) * ((double)(K / 64) * (xr == 256 ? 1.42 : 0.8) + (xr == 256 ? 5 : 4));
}

int product_tile(int64_t M, int64_t slab, int64_t K) { return product_us(M, slab, K, 128) < product_us(M, slab, K, 256) ? 128 : 256; }

// The same for the comparison with other ways, fitted to the times of 42 weights by 130 to 2048 rows (within 10 % in 94 of 100; the
// terms have to be taken together): rounds with their ends, the last of which has shorter stages where it leaves CUs idle.
double rounds_us(int64_t M, int64_t slab, int64_t K) {
    const int xr = product_tile(M, slab, K);
    const int64_t tiles = cdiv(M, xr) * cdiv(slab, 256), full = tiles / 256;
    const double steps = (double)(K / 64), part = (double)(tiles % 256) / 256, ends = xr == 256 ? 0 : 1.6;
    const double stage = xr == 256 ? 0.62 + 0.6 * part : 0.57 + 0.1 * part;
    return (double)full * (steps * (xr == 256 ? 1.25 : 0.76) + ends) + (part > 0 ? steps * stage + ends : 0);
}

template <typename T, int XR, bool GATED, bool ADD = false>
hipError_t launch(const void* x, const void* wt, const void* bias, const void* residual, const Outputs& out, int M, int cols, int K, hipStream_t st) {
    using P = PingPong<T, XR>;
    auto kern = dense_kernel<T, XR, GATED, ADD>;
    static bool raised = false;      // once per process and instantiation
    if (!raised) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 P::kLds);
        if (e != hipSuccess) return e;
        raised = true;
    }
    const int x_tiles = (int)cdiv(M, XR), w_tiles = (int)cdiv(cols, 256);
    (void)hipGetLastError();
    kern<<<dim3((unsigned)(cdiv((int64_t)x_tiles * w_tiles, 8) * 8)), dim3(P::kThreads), P::kLds, st>>>(
        (const uint16_t*)x, (const uint16_t*)wt, (const uint16_t*)bias, (const uint16_t*)residual, out, M, cols, K, x_tiles, w_tiles);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_dense(const void* x, const void* wt, const void* bias, const void* residual, const Outputs& out, int M, int cols, int K,
                        int xr, bool gated, hipStream_t st) {
    const auto go = [&](auto rows) {
        constexpr int XR = decltype(rows)::value;
        return residual ? launch<T, XR, false, true>(x, wt, nullptr, residual, out, M, cols, K, st)
               : gated  ? launch<T, XR, true>(x, wt, bias, nullptr, out, M, cols, K, st)
                        : launch<T, XR, false>(x, wt, bias, nullptr, out, M, cols, K, st);
    };
    return xr == 256 ? go(std::integral_constant<int, 256>{}) : go(std::integral_constant<int, 128>{});
}

// Sizes and group sizes the path takes; 32-bit offsets inside a tile's rows of x and inside a slab.
bool takes(int64_t M, int64_t N, int64_t K, int64_t g) {
    return M >= 1 && N >= 8 && N % 8 == 0 && K >= 64 && K % 64 == 0 && g > 0 && K % g == 0 && (g % 64 == 0 || (64 % g == 0 && g % 8 == 0)) &&
           K <= (1 << 20) && M < (1ll << 31) - 256 && N < (1ll << 31) - 256 && cdiv(M, 128) * cdiv(N, 256) < (1ll << 31) - 8;
}

}  // namespace

double dense_linear_us(int64_t M, int64_t N, int64_t K, int64_t g) {
    if (!takes(M, N, K, g)) return -1;
    const int64_t slab = slab_columns(N, K);
    // the dequantise pass moves 2.5 bytes a weight at 6.4 TB/s (4096 x 12288 20.5 us, 5120 x 25600 62); a slab that the 256 MB cache
    // does not hold is read from memory (5120 x 25600, 262 MB: 640 rows 242 us, 1500 rows 446); the result is written at 2.7 TB/s
    const double cold = slab * K * 2 > (192ll << 20) ? 2.3 * (double)(K * N) / 6.0e6 : 0;
    return 6.9 + 2.5 * (double)(K * N) / 6.4e6 + cold + (double)cdiv(N, slab) * rounds_us(M, slab, K) + (double)(M * N) * 2 / 2.7e6;
}

size_t dense_parts_scratch_bytes(const int64_t* N, int count, int64_t M, int64_t K, int64_t g) {
    int64_t total = 0;
    for (int i = 0; i < count; ++i) {
        if (N[i] <= 0 || N[i] % 256 != 0) return 0;      // a tile lies in one output
        total += N[i];
    }
    return takes(M, total, K, g) && slab_columns(total, K) == total ? (size_t)(total * K * 2) : 0;
}

int dense_parts(const char* fn, const void* x, const Parts& parts, int64_t M, int64_t K, int64_t g, int dtype, void* scratch,
                size_t scratch_bytes, hipStream_t st) {
    const int64_t N[kMaxParts] = {parts.columns[0], parts.columns[1], parts.columns[2]};
    const size_t need = dense_parts_scratch_bytes(N, parts.count, M, K, g);
    if (!need || !scratch || scratch_bytes < need || (reinterpret_cast<uintptr_t>(scratch) & 15u)) {
        set_error("%s: 16-byte aligned scratch of %zu bytes needed, %zu given", fn, need, scratch ? scratch_bytes : (size_t)0);
        return AWQ_ERR_WORKSPACE;
    }
    const int xr = product_tile(M, parts.total, K);
    hipError_t e = launch_dequant_transpose_parts(dtype, parts, scratch, (int)K, (int)g, st);
    if (e == hipSuccess)
        e = dtype == AWQ_F16 ? launch_dense<F16>(x, scratch, nullptr, nullptr, Outputs(parts), (int)M, parts.total, (int)K, xr, false, st)
                             : launch_dense<BF16>(x, scratch, nullptr, nullptr, Outputs(parts), (int)M, parts.total, (int)K, xr, false, st);
    return e == hipSuccess ? AWQ_OK : hip_fail(fn, e);
}

}  // namespace awq

using namespace awq;

extern "C" size_t awq_linear_dense_scratch_bytes(int64_t M, int64_t N, int64_t K, int64_t group_size) {
    return takes(M, N, K, group_size) ? (size_t)(std::min(slab_columns(N, K), N) * K * 2) : 0;
}

// `second`: the up weight beside `w`, the gate weight, N columns of each.
static int dense_entry(const char* fn, const void* x, const PackedWeight& w, const PackedWeight* second, const void* bias, const void* residual,
                       void* y, int64_t M, int64_t N, int64_t K, int64_t g, int dtype, bool gated, void* scratch, size_t scratch_bytes,
                       void* stream) {
    const int64_t cols_in_all = second ? 2 * N : N;
    if (!takes(M, cols_in_all, K, g) || (gated && (bias || cols_in_all % 16 != 0))) {
        set_error("%s: needs K %% 64 == 0, a group size of 8, 16, 32 or a multiple of 64, and for a gated product N %% 16 == 0 "
                  "and no bias (M=%lld N=%lld K=%lld g=%lld)", fn, (long long)M, (long long)N, (long long)K, (long long)g);
        return AWQ_ERR_UNSUPPORTED;
    }
    if ((reinterpret_cast<uintptr_t>(bias) | reinterpret_cast<uintptr_t>(scratch) | reinterpret_cast<uintptr_t>(residual)) & 15u) {
        set_error("%s: bias, residual and scratch must be 16-byte aligned", fn);
        return AWQ_ERR_INVALID_ARG;
    }
    const size_t need = awq_linear_dense_scratch_bytes(M, cols_in_all, K, g);
    if (!scratch || scratch_bytes < need) {
        set_error("%s: scratch of %zu bytes needed, %zu given", fn, need, scratch ? scratch_bytes : (size_t)0);
        return AWQ_ERR_WORKSPACE;
    }
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const int64_t slab = slab_columns(cols_in_all, K);
    const int xr = product_tile(M, slab, K);
    for (int64_t n = 0; n < cols_in_all; n += slab) {
        const int64_t cols = std::min(slab, cols_in_all - n), each = second ? 2 : 1;
        hipError_t e = launch_dequant_transpose(dtype, w, second, scratch, (int)N, (int)K, (int)g, st, n / each, cols / each);
        const void* b = bias ? static_cast<const uint16_t*>(bias) + n : nullptr;
        const void* res = residual ? static_cast<const uint16_t*>(residual) + n : nullptr;
        const Outputs out(static_cast<uint16_t*>(y) + (gated ? n / 2 : n), (int)(gated ? cols_in_all / 2 : N));
        if (e == hipSuccess)
            e = dtype == AWQ_F16 ? launch_dense<F16>(x, scratch, b, res, out, (int)M, (int)cols, (int)K, xr, gated, st)
                                 : launch_dense<BF16>(x, scratch, b, res, out, (int)M, (int)cols, (int)K, xr, gated, st);
        if (e != hipSuccess) return hip_fail(fn, e);
    }
    return AWQ_OK;
}

extern "C" int awq_linear_dense(const void* x, const int32_t* qweight, const void* qscales, const int32_t* qzeros,
                                const void* bias, void* y, int64_t M, int64_t N, int64_t K, int64_t group_size, int dtype,
                                int gated, void* scratch, size_t scratch_bytes, void* stream) {
    const char* fn = "awq_linear_dense";
    PrefetchRegions dropped;            // hints of this thread were meant for this call; the product fills the chip
    take_prefetch_hint(&dropped);
    const int rc = check_linear_args(fn, x, qweight, qscales, qzeros, y, M, N, K, group_size, dtype);
    if (rc != AWQ_OK) return rc;
    return dense_entry(fn, x, {qweight, qscales, qzeros}, nullptr, bias, nullptr, y, M, N, K, group_size, dtype, gated != 0, scratch,
                       scratch_bytes, stream);
}

extern "C" int awq_linear_dense_add(const void* x, const int32_t* qweight, const void* qscales, const int32_t* qzeros,
                                    const void* residual, void* y, int64_t M, int64_t N, int64_t K, int64_t group_size, int dtype,
                                    void* scratch, size_t scratch_bytes, void* stream) {
    const char* fn = "awq_linear_dense_add";
    PrefetchRegions dropped;
    take_prefetch_hint(&dropped);
    const int rc = check_linear_args(fn, x, qweight, qscales, qzeros, y, M, N, K, group_size, dtype);
    if (rc != AWQ_OK) return rc;
    if (!residual) {
        set_error("%s: null pointer argument", fn);
        return AWQ_ERR_INVALID_ARG;
    }
    if (N > (1 << 22)) {        // a tile's rows of the residual lie within 32-bit offsets
        set_error("%s: too many columns", fn);
        return AWQ_ERR_UNSUPPORTED;
    }
    return dense_entry(fn, x, {qweight, qscales, qzeros}, nullptr, nullptr, residual, y, M, N, K, group_size, dtype, false, scratch,
                       scratch_bytes, stream);
}

extern "C" int awq_linear_dense_pair(const void* x, const int32_t* gate_qweight, const void* gate_qscales,
                                     const int32_t* gate_qzeros, const int32_t* up_qweight, const void* up_qscales,
                                     const int32_t* up_qzeros, void* y, int64_t M, int64_t N, int64_t K, int64_t group_size,
                                     int dtype, void* scratch, size_t scratch_bytes, void* stream) {
    const char* fn = "awq_linear_dense_pair";
    PrefetchRegions dropped;
    take_prefetch_hint(&dropped);
    int rc = check_linear_args(fn, x, gate_qweight, gate_qscales, gate_qzeros, y, M, N, K, group_size, dtype);
    if (rc == AWQ_OK) rc = check_linear_args(fn, x, up_qweight, up_qscales, up_qzeros, y, M, N, K, group_size, dtype);
    if (rc != AWQ_OK) return rc;
    const PackedWeight up(up_qweight, up_qscales, up_qzeros);
    return dense_entry(fn, x, {gate_qweight, gate_qscales, gate_qzeros}, &up, nullptr, nullptr, y, M, N, K, group_size, dtype, true, scratch,
                       scratch_bytes, stream);
}
