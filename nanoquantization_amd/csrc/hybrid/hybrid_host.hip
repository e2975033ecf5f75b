// Error plumbing of libnq_hybrid.so and the bookkeeping entry points of a decode step.
#include <cstdarg>
#include <cstdio>

#include "../step_kernels.hpp"
#include "hybrid_common.hpp"

namespace nqh {
namespace {
thread_local char g_error[512] = "";

// Largest logit per row, the lowest index among equal ones; NaNs are never selected.  As argmax_rows_kernel (nq_decode_ops.hip): a thread
// keeps the largest of four logits at a time and looks for its place at the end (16 rows of 32768 6.0 -> 4.6 us, of 151936 16.2 -> 8.9).  Of
// up to 16384 (FEW: a thread has four vectors) that look costs more than it saves, 2048 3.2 -> 3.35 us, 8200 3.85 -> 4.0.
template <bool FEW>
__global__ __launch_bounds__(1024) void argmax_f32_kernel(const float* __restrict__ logits, int64_t* __restrict__ out,
                                                          int vocab) {
    const float* row = logits + (size_t)blockIdx.x * vocab;
    float best = -__builtin_inff();
    int bi = 0x7fffffff;
    auto take = [&](float f, int idx) {
        if (f > best || (f == best && idx < bi)) {
            best = f;
            bi = idx;
        }
    };
    const int nvec = (vocab & 3) == 0 ? vocab >> 2 : 0;   // rows are 16-byte aligned only then
    int bv = -1;                                          // the first of the thread's vectors that holds `best`
    constexpr int kLoads = FEW ? 4 : 8;                   // in flight
    for (int v0 = threadIdx.x; v0 < nvec; v0 += kLoads * 1024) {
        f32x4 d[kLoads];
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const int v = v0 + u * 1024;
            d[u] = *reinterpret_cast<const f32x4*>(row + (size_t)(v < nvec ? v : v0) * 4);
        }
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
            const int v = v0 + u * 1024;
            if constexpr (FEW) {
                if (v < nvec) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) take(d[u][i], v * 4 + i);
                }
                continue;
            }
            const float m = fmaxf(fmaxf(d[u][0], d[u][1]), fmaxf(d[u][2], d[u][3]));
            if (v < nvec && (m > best || (bv < 0 && m == best))) {
                best = m;
                bv = v;
            }
        }
    }
    if (bv >= 0) {
        const f32x4 f = *reinterpret_cast<const f32x4*>(row + (size_t)bv * 4);
#pragma unroll
        for (int i = 3; i >= 0; --i)
            if (f[i] == best) bi = bv * 4 + i;
    }
    for (int i = nvec * 4 + threadIdx.x; i < vocab; i += 1024) take(row[i], i);
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
}  // namespace

int fail(int status, const char* fn, const char* fmt, ...) {
    const int n = snprintf(g_error, sizeof g_error, "%s: ", fn);
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_error + n, sizeof g_error - n, fmt, ap);
    va_end(ap);
    return status;
}
int launched(const char* fn) {
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? NQH_OK : fail(NQH_ERR_HIP, fn, "%s", hipGetErrorString(e));
}
}  // namespace nqh

using namespace nqh;

extern "C" const char* nqh_last_error(void) { return g_error; }

extern "C" int nqh_argmax_rows(const float* logits, int64_t* out, int64_t rows, int64_t vocab, void* stream) {
    const char* fn = "nqh_argmax_rows";
    if (!logits || !out || !aligned(logits, 16)) return fail(NQH_ERR_ARG, fn, "null or misaligned pointer");
    if (rows <= 0 || vocab <= 0 || rows > kMaxI32 || vocab > 0x7ffffff0)
        return fail(NQH_ERR_ARG, fn, "rows and vocab must be positive 31-bit counts");
    (void)hipGetLastError();
    (vocab <= 16384 ? argmax_f32_kernel<true> : argmax_f32_kernel<false>)<<<dim3((unsigned)rows), dim3(1024), 0, (hipStream_t)stream>>>(logits, out, (int)vocab);
    return launched(fn);
}

extern "C" int nqh_decode_prepare(const int64_t* positions, const uint8_t* active, const int32_t* block_table,
                                  int64_t* slots, int32_t* context_lens, int64_t rows, int64_t max_blocks,
                                  int64_t block_size, void* stream) {
    const char* fn = "nqh_decode_prepare";
    if (!positions || !active || !block_table || !slots || !context_lens) return fail(NQH_ERR_ARG, fn, "null pointer");
    if (rows <= 0 || max_blocks <= 0 || block_size <= 0 || rows > kMaxI32 || max_blocks > kMaxI32 || block_size > kMaxI32)
        return fail(NQH_ERR_ARG, fn, "rows, max_blocks and block_size must be positive 31-bit counts");
    (void)hipGetLastError();
    awq::decode_prepare_kernel<<<dim3((unsigned)cdiv(rows, 256)), dim3(256), 0, (hipStream_t)stream>>>(
        positions, active, block_table, slots, context_lens, (int)rows, (int)max_blocks, (int)block_size);
    return launched(fn);
}

extern "C" int nqh_decode_advance(const int64_t* next_tokens, const uint8_t* active, int64_t* out_log, int64_t* ids,
                                  int64_t* positions, int64_t* step, int64_t rows, int64_t out_rows, void* stream) {
    const char* fn = "nqh_decode_advance";
    if (!next_tokens || !active || !out_log || !ids || !positions || !step) return fail(NQH_ERR_ARG, fn, "null pointer");
    if (rows <= 0 || rows > kMaxI32 || out_rows <= 0) return fail(NQH_ERR_ARG, fn, "rows and out_rows must be positive");
    (void)hipGetLastError();
    awq::decode_advance_kernel<<<dim3(1), dim3(1024), 0, (hipStream_t)stream>>>(next_tokens, active, out_log, ids,
                                                                              positions, step, (int)rows, out_rows);
    return launched(fn);
}
