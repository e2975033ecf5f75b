// Dense linears.  For few rows: y = act(x W^T (+ bias)), bf16 operands, fp32 accumulation.
//   skinny_linear_kernel   both operands straight from memory, 16 rows at a time, the waves split the contraction
//   stream_linear_kernel   up to 64 rows at once: the activations go through LDS; the contraction may be split over workgroups,
//                          whose sums the reader adds (nqh_skinny_linear_parts) or sum_parts_kernel
// plan_linear says which.  For more rows dense_linear_kernel, an activation or a bias in its epilogue, the contraction split likewise
// (plan_dense), where it is done before a library product that the host issues.
#include <algorithm>
#include <atomic>
#include <cmath>

#include "../pingpong.hpp"
#include "skinny.hpp"

namespace nqh {
namespace {

template <bool F32OUT>
__global__ __launch_bounds__(1024) void skinny_linear_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                                             const uint16_t* __restrict__ bias, void* __restrict__ y,
                                                             int rows, int n_out, int n_in, int act, float param) {
    extern __shared__ __attribute__((aligned(16))) float s_sum[];
    const int lane = threadIdx.x & 63, lo = lane & 15, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int waves = blockDim.x >> 6, n0 = blockIdx.x * 16, r0 = blockIdx.y * 16;
    rows -= r0;
    x += (int64_t)r0 * n_in;
    const uint16_t* w_row[1] = {w + (int64_t)min(n0 + lo, n_out - 1) * n_in};
    const uint16_t* x_row[1] = {x + (int64_t)min(lo, rows - 1) * n_in};
    f32x4 acc[1][1] = {{f32x4{0.f, 0.f, 0.f, 0.f}}};
    skinny_accumulate<1, 1>(acc, w_row, x_row, n_in, wave, waves);
    skinny_reduce<1, 1>(acc, s_sum, wave, waves);
    const int t = threadIdx.x >> 4, n = n0 + (threadIdx.x & 15);
    if (threadIdx.x < 256 && t < rows && n < n_out) {
        const float v = activation_f32(s_sum[threadIdx.x] + (bias ? Bf::to_f32(bias[n]) : 0.f), act, param);
        if constexpr (F32OUT) reinterpret_cast<float*>(y)[(int64_t)(r0 + t) * n_out + n] = v;
        else reinterpret_cast<uint16_t*>(y)[(int64_t)(r0 + t) * n_out + n] = Bf::from_f32(v);
    }
}

// 16 MT rows, 16 NT output features and a part of the contraction per workgroup; its waves are NT features tiles x KS parts of every
// stage of KS * 128 contraction elements.  The weights go straight into registers, kAhead stages ahead; the activations, which all
// waves read, are brought to LDS once, as far ahead (rows of 256 bytes, 16-byte piece p of row r at position (p + r) % 16: the 16
// rows of an operand read fall on all banks once).  A stage is waited for by the count of the requests behind it, so that the one
// barrier a stage stops nobody's stream.  Workgroups begin at different stages: in step they would ask the same memory channels,
// the rows of a weight being a power of two apart as often as not.
//
// Bound by the stream of the weights (5 to 5.6 TB/s) and by what a CU takes in, some 45 KB/us of weights and activations alike.  That
// is why the contraction is split until there is a workgroup for each CU, and why workgroups are wider where there are more rows.
// Weights from memory, us, before (all of the contraction in one workgroup, one stage ahead, waited for in full) / this with the sums
// left to the reader: 18432 -> 4096 at 64, 16 rows and one 87 / 34, 41 / 28, 33.8 / 27.4; unsplit: 64 rows 4096 -> 32768 70 / 53 (63 with
// all workgroups in step).  Seven stages ahead are no faster than three.
#define NQH_LPTR(p) ((__attribute__((address_space(3))) void*)(p))

template <int N, typename F>
__device__ __forceinline__ void each_of(F&& f) {      // f(0) .. f(N - 1), the numbers known to the compiler
    if constexpr (N > 0) {
        each_of<N - 1>(f);
        f(Int<N - 1>());
    }
}

// SPLIT: y takes the sums of every part, fp32 [rows, parts, n_out], n_out % 4 == 0; bias and activation are the reader's.
template <int MT, int NT, int KS, int kAhead, bool F32OUT, bool SPLIT>
__global__ __launch_bounds__(64 * NT * KS, NT == 8 ? 4 : 2) void stream_linear_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, const uint16_t* __restrict__ bias, void* __restrict__ y, int rows,
    int n_out, int n_in, int act, float param, int pieces_each) {
    constexpr int NW = NT * KS, kPart = 16 * MT * 256, kBuf = KS * kPart, kLoads = kBuf / 1024 / NW;
    constexpr int kStageLoads = 4 + kLoads, kStageBufs = kAhead + 1;
    static_assert(kLoads >= 1 && kLoads * NW * 1024 == kBuf, "every wave brings the same");
    extern __shared__ __attribute__((aligned(1024))) unsigned char s_x[];   // [buffer][row][256 bytes]
    const int lane = threadIdx.x & 63, lo = lane & 15, hi = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nt = wave % NT, part = wave / NT, n0 = (blockIdx.x * NT + nt) * 16, first = blockIdx.y * pieces_each;
    const int pieces = min(pieces_each, (n_in + kPiece - 1) / kPiece - first), count = (pieces + KS - 1) / KS;
    // This wave's rows of the weight, past the end the last one.  What lies past the end of a row or behind the last stage is
    // outside the buffer: zeros without traffic, and the count of requests stays.
    const int w0 = min(n0, n_out - 1), own = min(n0 + lo, n_out - 1) - w0;
    const auto rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(w) + (int64_t)w0 * n_in, 0,
                                                      (uint32_t)min(16, n_out - w0) * (uint32_t)n_in * 2, 0x00020000);
    const uint32_t own_at = (uint32_t)own * (uint32_t)n_in * 2;
    const auto rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(x), 0, (uint32_t)rows * (uint32_t)n_in * 2, 0x00020000);
    constexpr uint32_t kOutside = 0x80000000u;
    const int turn = (int)(((blockIdx.x * 5) & 31) * (unsigned)count >> 5);      // the stage that comes first here
    const auto turned = [&](int t) { const int u = t + turn; return t >= count ? t : u >= count ? u - count : u; };
    const auto load_w = [&](u32x4 (&f)[4], int t0) {
        const int t = turned(t0);
        const int k0 = (first + t * KS + part) * kPiece + 8 * hi, end = t * KS + part < pieces ? n_in : 0;
#pragma unroll
        for (int s = 0; s < 4; ++s)
            f[s] = __builtin_amdgcn_raw_buffer_load_b128(rw, k0 + 32 * s < end ? own_at + (uint32_t)(k0 + 32 * s) * 2 : kOutside, 0, 0);
    };
    const auto load_x = [&](int t0, int at) {
        const int t = turned(t0);
        unsigned char* buf = s_x + at * kBuf;
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int block = i * NW + wave, p = block / (4 * MT), row = block % (4 * MT) * 4 + (lane >> 4);       // 1 KiB: four rows
            const int end = t * KS + p < pieces ? n_in : 0;
            const int k = (first + t * KS + p) * kPiece + 8 * (((lane & 15) - row) & 15);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, NQH_LPTR(buf + block * 1024), 16,
                                                     k < end ? (uint32_t)(min(row, rows - 1) * n_in + k) * 2 : kOutside, 0, 0, 0);
        }
    };
    f32x4 acc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 f[kStageBufs][4];
#pragma unroll
    for (int t = 0; t < kAhead; ++t) {
        load_x(t, t);
        load_w(f[t], t);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_wave_barrier();
    }
    // stage t lies in buffer and registers `at`; `behind` stages have been asked for since
    const auto landed = [&](auto behind) {
        constexpr int c = behind * kStageLoads;
        static_assert(c < 64, "what the counter holds");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0x0F70 | (c & 15) | ((c >> 4) << 14));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    const auto multiply = [&](const u32x4 (&cur)[4], int at) {
        const unsigned char* base = s_x + at * kBuf + part * kPart + lo * 256;
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const u32x4 xf = *reinterpret_cast<const u32x4*>(base + m * 4096 + ((4 * s + hi + lo) & 15) * 16);
                acc[m] = Bf::mfma16(cur[s], xf, acc[m]);
            }
    };
    int t = 0;
#pragma unroll 1
    for (; t + kStageBufs <= count; t += kStageBufs) {
        each_of<kStageBufs>([&](auto u) {
            landed(Int<kAhead - 1>());
            load_x(t + u + kAhead, (u + kAhead) % kStageBufs);          // where everybody has read the stage before this one
            load_w(f[(u + kAhead) % kStageBufs], t + u + kAhead);
            __builtin_amdgcn_sched_barrier(0);
            multiply(f[u], u);
        });
    }
    each_of<kAhead>([&](auto u) {
        if (t + u >= count) return;
        landed(Int<kAhead - 1 - u>());
        multiply(f[u], u);
    });
    __builtin_amdgcn_s_waitcnt(0x0F70);       // what was asked for past the end has come: the LDS may be given back
    if constexpr (KS > 1) {
        __syncthreads();
        float* sums = reinterpret_cast<float*>(s_x);
        if (part > 0) {
#pragma unroll
            for (int m = 0; m < MT; ++m) *reinterpret_cast<f32x4*>(sums + (((part - 1) * NT + nt) * MT + m) * 256 + lane * 4) = acc[m];
        }
        __syncthreads();
        if (part > 0) return;
#pragma unroll
        for (int p = 0; p < KS - 1; ++p)
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[m] += *reinterpret_cast<const f32x4*>(sums + ((p * NT + nt) * MT + m) * 256 + lane * 4);
    }
    const int n = n0 + 4 * hi;
    if (n >= n_out) return;
    const bool whole = n_out % 4 == 0 && ((uintptr_t)y & 15) == 0;        // a lane's four features: one aligned access
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int row = 16 * m + lo;
        if (row >= rows) continue;
        if constexpr (SPLIT) {
            *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(y) + ((int64_t)row * gridDim.y + blockIdx.y) * n_out + n) = acc[m];
        } else {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = activation_f32(acc[m][e] + (bias ? Bf::to_f32(bias[min(n + e, n_out - 1)]) : 0.f), act, param);
            const int64_t at = (int64_t)row * n_out + n;
            if (whole) {
                if constexpr (F32OUT) store_vec<Fp, 4>(reinterpret_cast<float*>(y) + at, v);
                else store_vec<Bf, 4>(reinterpret_cast<uint16_t*>(y) + at, v);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < n_out) {
                        if constexpr (F32OUT) reinterpret_cast<float*>(y)[at + e] = v[e];
                        else reinterpret_cast<uint16_t*>(y)[at + e] = Bf::from_f32(v[e]);
                    }
            }
        }
    }
}

// y = act(sum over the parts of the contraction (+ bias)): parts [rows, splits, n_out], four features a thread.
template <bool F32OUT>
__global__ __launch_bounds__(256) void sum_parts_kernel(const float* __restrict__ parts, const uint16_t* __restrict__ bias,
                                                        void* __restrict__ y, int n_out, int splits, int act, float param) {
    const int n = (blockIdx.y * 256 + threadIdx.x) * 4, row = blockIdx.x;
    if (n >= n_out) return;
    const float* src = parts + (int64_t)row * splits * n_out + n;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int s = 0; s < splits; ++s) {
        const f32x4 p = *reinterpret_cast<const f32x4*>(src + (int64_t)s * n_out);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += p[e];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = activation_f32(v[e] + (bias ? Bf::to_f32(bias[n + e]) : 0.f), act, param);
    const int64_t at = (int64_t)row * n_out + n;
    if constexpr (F32OUT) store_vec<Fp, 4>(reinterpret_cast<float*>(y) + at, v);
    else store_vec<Bf, 4>(reinterpret_cast<uint16_t*>(y) + at, v);
}

int launch_sum_parts(const char* fn, const void* parts, const void* bias, void* y, int64_t rows, int64_t n_out, int64_t splits, int out_f32,
                     int act, float param, hipStream_t stream) {
    const auto kernel = out_f32 ? sum_parts_kernel<true> : sum_parts_kernel<false>;
    kernel<<<dim3((unsigned)rows, (unsigned)cdiv(n_out, 1024)), dim3(256), 0, stream>>>((const float*)parts, (const uint16_t*)bias, y, (int)n_out,
                                                                                  (int)splits, act, param);
    return launched(fn);
}

// Lets a kernel use `lds` bytes; `raised`: the devices where that has been done.
int allow_lds(const char* fn, const void* kernel, int lds, std::atomic<uint64_t>& raised) {
    int device = 0;
    hipError_t e = hipGetDevice(&device);
    if (e == hipSuccess && (device > 63 || !(raised.load(std::memory_order_relaxed) >> device & 1))) {
        e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e == hipSuccess && device < 64) raised.fetch_or(1ull << device, std::memory_order_relaxed);
    }
    return e == hipSuccess ? NQH_OK : fail(NQH_ERR_HIP, fn, "%s", hipGetErrorString(e));
}

template <int MT, int NT, int KS, int kAhead, bool F32OUT, bool SPLIT>
int launch_stream(const char* fn, const void* x, const void* w, const void* bias, void* y, int64_t rows, int64_t n_out, int64_t n_in,
                  int act, float param, int64_t splits, hipStream_t stream) {
    const int64_t each = cdiv(cdiv(n_in, kPiece), splits);
    constexpr int lds = (kAhead + 1) * KS * 16 * MT * 256;
    const auto kernel = stream_linear_kernel<MT, NT, KS, kAhead, F32OUT, SPLIT>;
    static std::atomic<uint64_t> raised{0};
    const int rc = lds > 65536 ? allow_lds(fn, (const void*)kernel, lds, raised) : NQH_OK;
    if (rc != NQH_OK) return rc;
    kernel<<<dim3((unsigned)cdiv(n_out, 16 * NT), (unsigned)splits), dim3(64 * NT * KS), lds, stream>>>(
        (const uint16_t*)x, (const uint16_t*)w, (const uint16_t*)bias, y, (int)rows, (int)n_out, (int)n_in, act, param, (int)each);
    return launched(fn);
}

// What a call runs: skinny_linear_kernel, or stream_linear_kernel with 2 (x 2 parts of a stage), 4 or 8 features tiles to a workgroup
// and the contraction in `splits` parts.
enum Form { kSkinny, kTwo, kFour, kEight };
struct LinearPlan {
    Form form;
    int splits;
};
// Who may add the parts: nobody, sum_parts_kernel, the same where the host issues call after call, the reader of the result.
enum class Sums { kNone, kOwnPass, kIssuedPass, kReader };
Sums sums_of(int adds) { return adds == NQH_ADDS_NOBODY ? Sums::kNone : adds == NQH_ADDS_PASS ? Sums::kOwnPass : Sums::kReader; }

// The least estimated time.  In us: a launch with its first data; what the fullest CU takes in (KB, at a rate of its own per form) and
// the weights from memory (MB), the root of the sum of their squares; parts written, and read by a pass of their own or by a reader
// whose row is one workgroup.  A pass that the host issues takes its 8 us, by which prompts of 40 tokens through small layers were 5 to
// 12 % longer.  Fitted to 32 weights (544 to 32768 x 1024 to 18432) at 1 to 64 rows, every form and split, from
// memory: 3.6 % off in the middle, 9.5 % in one of ten; the chosen form takes 0.4 % (nobody adds), 1.6 % (own pass) and 1.1 % (reader)
// longer than the fastest on average, 16 % at worst.  Long contractions and, the other way, few rows of many features are
// where skinny_linear_kernel is off the estimate; so are few rows where the rows of the weight are a power of two of 8 KB and more
// apart, which costs the streams a tenth and it nothing (4096 -> 32768 at 4 rows 48.6 us, as streams 51 to 54; 4096 -> 65536 90, 97
// to 100).  Over 163 weights (96 to 151936 x 512 to 18432) at 1 to 16 rows, nobody adding, the choice is 0.7 % from the fastest on
// average; with no such factor and 1.12 for long contractions it was 1.2 %, and 16 rows of 12288 -> 1024 took 30.6 us as a stream, 24.9 here.
LinearPlan make_linear_plan(int64_t rows, int64_t n_out, int64_t n_in, Sums sums) {
    struct Of {
        double launch, memory, rate, more;       // us, MB/us, KB/us for one tile of rows and so many more for four
        int tiles, parts;
    };
    static constexpr Of kOf[] = {{2.95, 7.95, 30.7, 5.6, 1, 1}, {2.67, 7.05, 48.1, 0, 2, 2}, {2.62, 7.15, 44.0, 3.3, 4, 1}, {3.02, 8.0, 39.8, 2.1, 8, 1}};
    const auto hypot2 = [](double a, double b) { return std::sqrt(a * a + b * b); };
    const double mb = 2e-6 * n_out * n_in;
    const int64_t groups = cdiv(n_out, 16) * cdiv(rows, 16), few = std::min<int64_t>(rows, 16), pieces = cdiv(n_in, kPiece);
    LinearPlan best{kSkinny, 1};
    double least = kOf[0].launch + hypot2(cdiv(groups, 256) * n_in * 2e-3 * (16 + few) / (kOf[0].rate + kOf[0].more * few / 16), mb / kOf[0].memory);
    if (rows <= 5 && n_out >= 16384) least *= 0.93;
    if (rows <= 6 && n_out >= 16384 && n_in >= 4096 && (n_in & (n_in - 1)) == 0) least *= 0.9;
    if (n_in >= 8192) least *= 1.06;
    if (n_in > (1 << 24)) return best;             // 32-bit offsets into 16 rows of the weight and all of x
    const int mt = rows <= 16 ? 1 : rows <= 32 ? 2 : 4;
    for (const Form form : {kTwo, kFour, kEight}) {
        if (form == kEight && mt == 1) continue;
        const Of& of = kOf[form];
        const int64_t columns = cdiv(n_out, 16 * of.tiles);
        const double rate = of.rate + of.more * (mt - 1) / 3;
        for (int64_t s = 1; s <= 16; ++s) {
            const int64_t each = cdiv(pieces, s);
            if (s > 1 && (sums == Sums::kNone || n_out % 4 != 0 || each < 2 || columns * s > 1024)) break;
            if (cdiv(pieces, each) != s) continue;             // the last part would be empty
            double us = of.launch + hypot2(cdiv(columns * s, 256) * cdiv(each, of.parts) * of.parts * 4.096 * (of.tiles + mt) / rate, mb / of.memory);
            if (s > 1) {
                const double parts = 4e-6 * s * rows * n_out;
                us += parts / 3.2 + (sums == Sums::kReader ? 0.3 + 4e-3 * s * n_out / 60 : parts / 6 + (sums == Sums::kOwnPass ? 2.65 : 8));
            }
            if (us < least) least = us, best = {form, (int)s};
        }
    }
    return best;
}

// What `make` says, remembered per thread: some 50 estimates take the host 3 us, as long as a launch.
template <typename Plan, typename F>
Plan remembered(int64_t rows, int64_t n_out, int64_t n_in, Sums sums, F make) {
    struct Entry {
        int64_t rows, n_out, n_in;
        Sums sums;
        Plan plan;
    };
    thread_local Entry kept[64] = {};                  // rows 0: empty
    Entry& e = kept[(uint64_t)(n_out * 31 + n_in * 7 + rows * 3 + (int)sums) * 0x9E3779B97F4A7C15ull >> 58];
    if (e.rows != rows || e.n_out != n_out || e.n_in != n_in || e.sums != sums)
        e = {rows, n_out, n_in, sums, make(rows, n_out, n_in, sums)};
    return e.plan;
}

LinearPlan plan_linear(int64_t rows, int64_t n_out, int64_t n_in, Sums sums) {
    return remembered<LinearPlan>(rows, n_out, n_in, sums, make_linear_plan);
}

size_t parts_bytes(LinearPlan plan, int64_t rows, int64_t n_out) {
    return plan.splits > 1 ? (size_t)plan.splits * rows * n_out * sizeof(float) : 0;
}

int run_skinny(const char* fn, const void* x, const void* w, const void* bias, void* y, int64_t rows, int64_t n_out, int64_t n_in,
               int out_f32, int act, float param, hipStream_t stream) {
    const int64_t groups = cdiv(n_out, 16);
    const int waves = skinny_waves(groups * cdiv(rows, 16), n_in);
    const size_t lds = (size_t)waves * 256 * sizeof(float);
    const auto kernel = out_f32 ? skinny_linear_kernel<true> : skinny_linear_kernel<false>;
    kernel<<<dim3((unsigned)groups, (unsigned)cdiv(rows, 16)), dim3((unsigned)waves * 64), lds, stream>>>(
        (const uint16_t*)x, (const uint16_t*)w, (const uint16_t*)bias, y, (int)rows, (int)n_out, (int)n_in, act, param);
    return launched(fn);
}

// The product as planned; with parts y takes their sums.
int run_plan(const char* fn, LinearPlan plan, const void* x, const void* w, const void* bias, void* y, int64_t rows, int64_t n_out,
             int64_t n_in, int out_f32, int act, float param, hipStream_t stream) {
    if (plan.form == kSkinny) return run_skinny(fn, x, w, bias, y, rows, n_out, n_in, out_f32, act, param, stream);
    const auto go = [&](auto mt, auto nt, auto ks, auto ahead) {
        if (plan.splits > 1)
            return launch_stream<mt, nt, ks, ahead, true, true>(fn, x, w, bias, y, rows, n_out, n_in, act, param, plan.splits, stream);
        return out_f32 ? launch_stream<mt, nt, ks, ahead, true, false>(fn, x, w, bias, y, rows, n_out, n_in, act, param, 1, stream)
                       : launch_stream<mt, nt, ks, ahead, false, false>(fn, x, w, bias, y, rows, n_out, n_in, act, param, 1, stream);
    };
    const auto of_rows = [&](auto mt) {
        if (plan.form == kTwo) return go(mt, Int<2>(), Int<2>(), Int<2>());
        if constexpr (mt > 1)
            if (plan.form == kEight) return go(mt, Int<8>(), Int<1>(), Int<3>());
        return go(mt, Int<4>(), Int<1>(), Int<3>());
    };
    return rows <= 16 ? of_rows(Int<1>()) : rows <= 32 ? of_rows(Int<2>()) : of_rows(Int<4>());
}

bool skinny_takes(int64_t rows, int64_t n_out, int64_t n_in) {
    return rows > 0 && rows <= 64 && n_out > 0 && n_in > 0 && n_in % 8 == 0 && n_out <= kMaxI32 - 16 && n_in <= (1 << 30);
}

// ---- many rows: activation(x @ weight^T (+ bias)) on the tiles of pingpong.hpp -----------------------------------------
// The activation of a library product is a pass of its own that reads and writes the result once more.  Here it is applied
// on the way out of the tile, to the value rounded to bf16 as that pass finds it: the same results but for the order of the sums.
// Bound by the matrix cores from a few hundred rows on, by the fill and store of its one tile below.  SPLIT: blockIdx.y is a part of
// steps_each stages of the contraction, and y takes its sums, fp32 [rows, parts, n_out], n_out % 4 == 0; bias and activation are the
// reader's.
template <int XR, bool SPLIT, bool BIAS>
__global__ __launch_bounds__(512, 2) void dense_linear_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                                              const uint16_t* __restrict__ bias, void* __restrict__ y, int rows, int n_out,
                                                              int n_in, int x_stride, int act, float param, int x_tiles, int w_tiles,
                                                              int steps_each) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char s_stage[];
    using P = awq::PingPong<Bf, XR>;
    int xt, wt;
    if (!awq::xcd_tile((int)blockIdx.x, x_tiles, w_tiles, xt, wt)) return;
    P p;
    const int m0 = xt * XR, n0 = wt * 256, count = min(XR, rows - m0);
    const uint32_t row_bytes = (uint32_t)n_in * 2, x_bytes = (uint32_t)x_stride * 2;
    const int first = SPLIT ? (int)blockIdx.y * steps_each : 0, steps = min(steps_each, n_in / P::kStage - first);
    uint32_t vw[4], vx[P::kXLoads];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int r = P::w_row(q, p.wave, p.lane);
        vw[q] = P::source(n0 + r, n_out, row_bytes, r, p.lane) + first * (P::kStage * 2);
    }
#pragma unroll
    for (int q = 0; q < P::kXLoads; ++q) {
        const int r = P::x_row(q, p.wave, p.lane);
        vx[q] = P::source(r, count, x_bytes, r, p.lane) + first * (P::kStage * 2);
    }
    const auto rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(w), 0, (uint32_t)n_out * row_bytes, 0x00020000);
    const auto rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(x) + (int64_t)m0 * x_stride, 0,
                                                      (uint32_t)(count - 1) * x_bytes + row_bytes, 0x00020000);
    p.run(s_stage, rw, vw, rx, vx, steps);
    if constexpr (SPLIT) {
#pragma unroll
        for (int j = 0; j < P::NJ; ++j) {
            const int r = p.wn * (XR / P::kWN) + 16 * j + p.lo;
            if (r >= count) continue;
            float* to = reinterpret_cast<float*>(y) + ((int64_t)(m0 + r) * gridDim.y + blockIdx.y) * n_out;
#pragma unroll
            for (int i = 0; i < P::MI; ++i) {
                const int n = n0 + p.wm * (256 / P::kWM) + 16 * i + 4 * p.hi;
                if (n < n_out) *reinterpret_cast<f32x4*>(to + n) = p.acc[i][j];
            }
        }
    } else {
        p.template write<256>(s_stage, [&](int i, int j) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float a = p.acc[i][j][e];
                if constexpr (BIAS) a += Bf::to_f32(bias[min(n0 + p.wm * (256 / P::kWM) + 16 * i + 4 * p.hi + e, n_out - 1)]);
                v[e] = activation_f32(Bf::round(a), act, param);
            }
            return u32x2{Bf::pack2(v[0], v[1]), Bf::pack2(v[2], v[3])};
        }, [&](int r, int c, u32x4 v) {
            if (r < count && n0 + c < n_out)
                *reinterpret_cast<u32x4*>(reinterpret_cast<uint16_t*>(y) + (int64_t)(m0 + r) * n_out + n0 + c) = v;
        });
    }
}

template <int XR, bool SPLIT, bool BIAS>
int launch_dense_as(const char* fn, const void* x, const void* w, const void* bias, void* y, int64_t rows, int64_t n_out, int64_t n_in,
                    int64_t x_stride, int act, float param, int64_t splits, void* stream) {
    using P = awq::PingPong<Bf, XR>;
    const auto kernel = dense_linear_kernel<XR, SPLIT, BIAS>;
    static std::atomic<uint64_t> raised{0};
    const int rc = allow_lds(fn, (const void*)kernel, P::kLds, raised);
    if (rc != NQH_OK) return rc;
    const int64_t x_tiles = cdiv(rows, XR), w_tiles = cdiv(n_out, 256);
    kernel<<<dim3((unsigned)(cdiv(x_tiles * w_tiles, 8) * 8), (unsigned)splits), dim3(P::kThreads), P::kLds, (hipStream_t)stream>>>(
        (const uint16_t*)x, (const uint16_t*)w, (const uint16_t*)bias, y, (int)rows, (int)n_out, (int)n_in, (int)x_stride, act,
        param, (int)x_tiles, (int)w_tiles, (int)cdiv(n_in / P::kStage, splits));
    return launched(fn);
}

// (The bias is a form of its own: asked for in the epilogue of the others it cost them 3 to 5 %, 1000 rows of 2048 -> 9216 44.2 -> 46.6 us.)
template <int XR, bool SPLIT>
int launch_dense(const char* fn, const void* x, const void* w, const void* bias, void* y, int64_t rows, int64_t n_out, int64_t n_in,
                 int64_t x_stride, int act, float param, int64_t splits, void* stream) {
    if constexpr (!SPLIT)
        if (bias) return launch_dense_as<XR, SPLIT, true>(fn, x, w, bias, y, rows, n_out, n_in, x_stride, act, param, splits, stream);
    return launch_dense_as<XR, SPLIT, false>(fn, x, w, nullptr, y, rows, n_out, n_in, x_stride, act, param, splits, stream);
}

// Whole stages, 16-byte rows of y, 32-bit offsets into the weight and into a tile's rows of x, a launchable grid.
bool dense_activation_takes(int64_t rows, int64_t n_out, int64_t n_in) {
    return rows >= 1 && rows <= kMaxI32 - 256 && n_out >= 8 && n_out % 8 == 0 && n_in >= 64 && n_in % 64 == 0 && n_in <= (1 << 20) &&
           n_out < (1ll << 31) / n_in && cdiv(rows, 128) * cdiv(n_out, 256) <= kMaxI32 / 512;
}

// Estimated microseconds with tiles of xr rows: rounds of 256 workgroups, a stage of 1.42 and 0.8 us in a full one and less in one
// that leaves CUs idle (measured with 100 to 256 tiles of 64 stages), filling and storing a tile.
double dense_activation_us(int64_t rows, int64_t n_out, int64_t n_in, int xr) {
    const int64_t tiles = cdiv(rows, xr) * cdiv(n_out, 256), full = tiles / 256;
    const double steps = (double)(n_in / 64), part = (double)(tiles % 256) / 256, ends = xr == 256 ? 5 : 4;
    const double stage = xr == 256 ? std::max(0.7, 0.45 + 0.97 * part) : 0.6 + 0.2 * part;
    return full * (steps * (xr == 256 ? 1.42 : 0.8) + ends) + (part > 0 ? steps * stage + ends : 0);
}

int dense_activation_tile(int64_t rows, int64_t n_out, int64_t n_in) {
    return dense_activation_us(rows, n_out, n_in, 128) < dense_activation_us(rows, n_out, n_in, 256) ? 128 : 256;
}

// ---- the same without an activation, instead of a library product -----------------------------------------------------------
struct DensePlan {
    int xr, splits;
    double us;
};

// Estimated microseconds: rounds of 256 workgroups as above, by stages and ends, the weights from memory, parts written and read as in
// plan_linear (a reader of more rows than CUs: 5.5 TB/s; it reads sums instead of a 16-bit result).  Fitted to 33 weights (96 to 18432 x 1024 to
// 18432) at 80 to 8192 rows: 5 % off in the middle, 14 % in one of ten; the chosen form 1.2 % from the fastest on average.
DensePlan make_dense_plan(int64_t rows, int64_t n_out, int64_t n_in, Sums sums) {
    const double memory = 3.2 + 2e-6 * n_out * n_in / 3.6;
    DensePlan best{0, 1, 1e30};
    for (const int xr : {128, 256}) {
        const int64_t tiles = cdiv(rows, xr) * cdiv(n_out, 256), steps = n_in / 64;
        for (int64_t s = 1; s <= 16; ++s) {
            const int64_t each = cdiv(steps, s), work = tiles * s;
            const double parts = 4e-6 * s * rows * n_out;
            if (s > 1 && (sums == Sums::kNone || n_out % 4 != 0 || each < 2 || work > 520 || parts > 268)) break;
            if (cdiv(steps, each) != s) continue;
            const double part = (double)(work % 256) / 256, whole = (double)(work / 256);
            const double stage = xr == 256 ? std::max(0.52, 0.91 + 0.37 * part) : std::max(0.59, 0.6 + 0.32 * part), end = xr == 256 ? 5.4 : 3.3;
            double us = std::max(memory, 3.2 + whole * (each * (xr == 256 ? 1.36 : 0.85) + end) + (part > 0 ? each * stage + end : 0));
            if (s > 1)
                us += parts / 8 + (sums == Sums::kReader ? std::max((parts - 2e-6 * rows * n_out) / 5.5, 4e-3 * s * n_out / 60) : 2.65 + parts / 6);
            if (us < best.us) best = {xr, (int)s, us};
        }
    }
    return best;
}

DensePlan plan_dense(int64_t rows, int64_t n_out, int64_t n_in, Sums sums) {
    return remembered<DensePlan>(rows, n_out, n_in, sums, make_dense_plan);
}

// What a library product is worth waiting for: the time that it takes on the GPU, less a margin for being ahead of the estimate in a
// pass (contractions of 12288 and more it does not split well), or most of the 21 us that it takes the host to issue; busy: of a pass
// with other work that the GPU takes longer for than the host, which hides a part of that, as many rows do in any layer (the figures are
// beside nqh_dense_linear_wanted).
double library_us(int64_t rows, int64_t n_out, int64_t n_in, bool busy) {
    const double size = (double)rows * (double)n_out;
    return std::max(busy || rows > 2400 ? 15.0 : 20.0, (n_in >= 12288 ? 0.9 : 0.8) * (6.2 + 2e-9 * size * n_in / (1.4 * size / (size + 1.57e6))));
}

}  // namespace
}  // namespace nqh

using namespace nqh;

extern "C" int64_t nqh_skinny_linear_parts(int64_t rows, int64_t out_features, int64_t in_features) {
    return skinny_takes(rows, out_features, in_features) ? plan_linear(rows, out_features, in_features, Sums::kReader).splits : 1;
}

extern "C" int nqh_skinny_linear_sums(const void* x, const void* weight, float* sums, int64_t rows, int64_t out_features,
                                      int64_t in_features, void* stream) {
    const char* fn = "nqh_skinny_linear_sums";
    if (!x || !weight || !sums || !aligned(x, 16) || !aligned(weight, 16) || !aligned(sums, 16))
        return fail(NQH_ERR_ARG, fn, "null or misaligned pointer");
    if (!skinny_takes(rows, out_features, in_features))
        return fail(NQH_ERR_ARG, fn, "1 to 64 rows and an in_features that is a multiple of 8");
    (void)hipGetLastError();
    return run_plan(fn, plan_linear(rows, out_features, in_features, Sums::kReader), x, weight, nullptr, sums, rows, out_features,
                    in_features, 1, NQH_ACT_NONE, 0.f, (hipStream_t)stream);
}

extern "C" int nqh_skinny_linear_form(int64_t rows, int64_t out_features, int64_t in_features, int adds, int64_t* parts) {
    if (!skinny_takes(rows, out_features, in_features) || adds < NQH_ADDS_NOBODY || adds > NQH_ADDS_READER) return 0;
    const LinearPlan plan = plan_linear(rows, out_features, in_features, sums_of(adds));
    if (parts) *parts = plan.splits;
    return 1 << plan.form;
}

extern "C" size_t nqh_skinny_linear_scratch_bytes(int64_t rows, int64_t out_features, int64_t in_features, int captured) {
    if (!skinny_takes(rows, out_features, in_features) ||
        plan_linear(rows, out_features, in_features, captured ? Sums::kOwnPass : Sums::kIssuedPass).splits == 1)
        return 0;
    return parts_bytes(plan_linear(rows, out_features, in_features, Sums::kOwnPass), rows, out_features);
}

extern "C" int nqh_skinny_linear_ex(const void* x, const void* weight, const void* bias, void* y, int64_t rows, int64_t out_features,
                                    int64_t in_features, int out_f32, int act, float param, void* scratch, size_t scratch_bytes,
                                    void* stream) {
    const char* fn = "nqh_skinny_linear";
    if (!x || !weight || !y || !aligned(x, 16) || !aligned(weight, 16) || !aligned(scratch, 16))
        return fail(NQH_ERR_ARG, fn, "null or misaligned pointer");
    if (!skinny_takes(rows, out_features, in_features))
        return fail(NQH_ERR_ARG, fn, "1 to 64 rows and an in_features that is a multiple of 8");
    if (act < NQH_ACT_NONE || act > NQH_ACT_SOFTCAP || (act == NQH_ACT_SOFTCAP && !(param > 0.f)))
        return fail(NQH_ERR_ARG, fn, "unknown activation, or a cap that is not positive");
    (void)hipGetLastError();
    const hipStream_t st = (hipStream_t)stream;
    LinearPlan plan = plan_linear(rows, out_features, in_features, scratch && aligned(y, 16) ? Sums::kOwnPass : Sums::kNone);
    if (scratch_bytes < parts_bytes(plan, rows, out_features)) plan = plan_linear(rows, out_features, in_features, Sums::kNone);
    if (plan.splits == 1) return run_plan(fn, plan, x, weight, bias, y, rows, out_features, in_features, out_f32, act, param, st);
    const int rc = run_plan(fn, plan, x, weight, nullptr, scratch, rows, out_features, in_features, 1, NQH_ACT_NONE, 0.f, st);
    if (rc != 0) return rc;
    return launch_sum_parts(fn, scratch, bias, y, rows, out_features, plan.splits, out_f32, act, param, st);
}

extern "C" int nqh_skinny_linear(const void* x, const void* weight, const void* bias, void* y, int64_t rows,
                                 int64_t out_features, int64_t in_features, int out_f32, int act, float param,
                                 void* stream) {
    return nqh_skinny_linear_ex(x, weight, bias, y, rows, out_features, in_features, out_f32, act, param, nullptr, 0, stream);
}

// 1 where the tiles are one round of the 256 CUs and estimated to take less time than the library's product and the activation's pass
// do when a python program issues them: 1.3 PFLOP/s and 5 TB/s, 28 us at least, the two launches.  On the GPU alone, from a graph, the
// library's smaller tiles are ahead up to some 1000 rows: relu2, this kernel / those two, us, 2048 -> 9216 at 100 rows 26 / 17, 2048 ->
// 1536 at 1000 rows 27 / 18.  What counts is the pass, which the host issues more slowly than the GPU works it off: Roletar prompts through
// three layers with this kernel / without, wall time, 1.7B, 128 tokens 646 / 751, 1000 tokens 860 / 872; 8B 0 to 2 % less.
// Several rounds of short contractions stay with the library: in a pass its products lose less to the writes between the rounds (0.6B,
// 8192 tokens, 576 tiles: 110 here, 83 + 24 there, though 89 / 103 when repeated alone).  Of 4096 and more the ends of the tiles weigh less
// (4000 rows, 4096 -> 18432: 453 here, 365 to 564 + 48 there).
extern "C" int nqh_dense_activation_wanted(int64_t rows, int64_t out_features, int64_t in_features) {
    if (!dense_activation_takes(rows, out_features, in_features)) return 0;
    const int xr = dense_activation_tile(rows, out_features, in_features);
    const double work = (double)rows * (double)out_features;
    if (cdiv(rows, xr) * cdiv(out_features, 256) > 256)
        return in_features >= 4096 && plan_dense(rows, out_features, in_features, Sums::kNone).us <
                                          0.92 * (6.2 + 2e-9 * work * (double)in_features / (1.4 * work / (work + 1.57e6)) + 4e-6 * work / 5);
    return dense_activation_us(rows, out_features, in_features, xr) <
           std::max(28.0, 2 * work * (double)in_features / 1.3e9 + 4 * work / 5e6 + 5);
}

extern "C" int nqh_dense_activation(const void* x, const void* weight, void* y, int64_t rows, int64_t out_features, int64_t in_features,
                                    int act, float param, void* stream) {
    const char* fn = "nqh_dense_activation";
    if (!x || !weight || !y || !aligned(x, 16) || !aligned(weight, 16) || !aligned(y, 16))
        return fail(NQH_ERR_ARG, fn, "null or misaligned pointer");
    if (!dense_activation_takes(rows, out_features, in_features))
        return fail(NQH_ERR_UNSUPPORTED, fn, "needs an in_features that is a multiple of 64, an out_features that is one of 8, and a "
                                             "weight of less than 2^31 elements");
    if (act < NQH_ACT_NONE || act > NQH_ACT_SOFTCAP || (act == NQH_ACT_SOFTCAP && !(param > 0.f)))
        return fail(NQH_ERR_ARG, fn, "unknown activation, or a cap that is not positive");
    (void)hipGetLastError();
    return dense_activation_tile(rows, out_features, in_features) == 128
               ? launch_dense<128, false>(fn, x, weight, nullptr, y, rows, out_features, in_features, in_features, act, param, 1, stream)
               : launch_dense<256, false>(fn, x, weight, nullptr, y, rows, out_features, in_features, in_features, act, param, 1, stream);
}

// Products of prompts.  A library product takes the host 21 us to issue (measured from python on one machine: on a faster one the line lies
// lower), this one 6, and a pass of some hundred rows through small layers is 11 of them; on the GPU the library is ahead by up to a
// third there.  Where its tiles leave CUs idle over a long contraction it falls far behind (1000 rows of 18432 -> 4096: 217 us, this with
// the sums left to the reader 114; 160 of 8192 -> 4096 48 / 25), and with many rows it is ahead by 3 to 10 %.  Prompts through three
// layers, before / with this kernel, us: Roletar 0.6B, 300 tokens 650 / 434, 8B, 2000 tokens 3157 / 2682; Gafulix 0.6B, 300 tokens 635 / 472.
// Where experts' weights take the GPU longer than the host is ahead by (Gafulix 1.7B and 8B, 200 to 900 us) a product of 15 to 20 us is
// the library's (busy; 1700 rows, 2048 -> 2048: 27 here, 17 there); of Gafulix 0.6B, 16 us of weights a layer, it is not (500 tokens 572 busy, 500 not).
extern "C" int nqh_dense_linear_wanted(int64_t rows, int64_t out_features, int64_t in_features, int reader, int busy) {
    return dense_activation_takes(rows, out_features, in_features) &&
           plan_dense(rows, out_features, in_features, reader ? Sums::kReader : Sums::kOwnPass).us <
               library_us(rows, out_features, in_features, busy != 0);
}

extern "C" int nqh_dense_linear_form(int64_t rows, int64_t out_features, int64_t in_features, int adds, int64_t* parts) {
    if (!dense_activation_takes(rows, out_features, in_features) || adds < NQH_ADDS_NOBODY || adds > NQH_ADDS_READER) return 0;
    const DensePlan plan = plan_dense(rows, out_features, in_features, sums_of(adds));
    if (parts) *parts = plan.splits;
    return plan.xr;
}

extern "C" size_t nqh_dense_linear_scratch_bytes(int64_t rows, int64_t out_features, int64_t in_features) {
    if (!dense_activation_takes(rows, out_features, in_features)) return 0;
    const DensePlan plan = plan_dense(rows, out_features, in_features, Sums::kOwnPass);
    return plan.splits > 1 ? (size_t)plan.splits * rows * out_features * sizeof(float) : 0;
}

extern "C" int nqh_dense_linear(const void* x, const void* weight, const void* bias, void* y, int64_t rows, int64_t out_features,
                                int64_t in_features, int64_t x_stride, void* scratch, size_t scratch_bytes, void* stream) {
    const char* fn = "nqh_dense_linear";
    if (!x || !weight || !y || !aligned(x, 16) || !aligned(weight, 16) || !aligned(y, 16) || !aligned(scratch, 16))
        return fail(NQH_ERR_ARG, fn, "null or misaligned pointer");
    if (!dense_activation_takes(rows, out_features, in_features))
        return fail(NQH_ERR_UNSUPPORTED, fn, "needs an in_features that is a multiple of 64, an out_features that is one of 8, and a "
                                             "weight of less than 2^31 elements");
    if (x_stride < in_features || x_stride % 8 != 0 || x_stride > (1 << 20))
        return fail(NQH_ERR_ARG, fn, "rows of x must be a multiple of 8 elements apart, at least in_features and at most 2^20");
    (void)hipGetLastError();
    DensePlan plan = plan_dense(rows, out_features, in_features, scratch ? Sums::kOwnPass : Sums::kNone);
    if (plan.splits > 1 && scratch_bytes < (size_t)plan.splits * rows * out_features * sizeof(float))
        plan = plan_dense(rows, out_features, in_features, Sums::kNone);
    if (plan.splits == 1)
        return plan.xr == 128 ? launch_dense<128, false>(fn, x, weight, bias, y, rows, out_features, in_features, x_stride, NQH_ACT_NONE, 0.f, 1, stream)
                              : launch_dense<256, false>(fn, x, weight, bias, y, rows, out_features, in_features, x_stride, NQH_ACT_NONE, 0.f, 1, stream);
    const int rc = plan.xr == 128 ? launch_dense<128, true>(fn, x, weight, nullptr, scratch, rows, out_features, in_features, x_stride, NQH_ACT_NONE, 0.f, plan.splits, stream)
                                  : launch_dense<256, true>(fn, x, weight, nullptr, scratch, rows, out_features, in_features, x_stride, NQH_ACT_NONE, 0.f, plan.splits, stream);
    return rc != NQH_OK ? rc : launch_sum_parts(fn, scratch, bias, y, rows, out_features, plan.splits, 0, NQH_ACT_NONE, 0.f, (hipStream_t)stream);
}

extern "C" int64_t nqh_dense_linear_parts(int64_t rows, int64_t out_features, int64_t in_features) {
    return dense_activation_takes(rows, out_features, in_features) ? plan_dense(rows, out_features, in_features, Sums::kReader).splits : 1;
}

extern "C" int nqh_dense_linear_sums(const void* x, const void* weight, float* sums, int64_t rows, int64_t out_features,
                                     int64_t in_features, void* stream) {
    const char* fn = "nqh_dense_linear_sums";
    if (!x || !weight || !sums || !aligned(x, 16) || !aligned(weight, 16) || !aligned(sums, 16))
        return fail(NQH_ERR_ARG, fn, "null or misaligned pointer");
    if (!dense_activation_takes(rows, out_features, in_features))
        return fail(NQH_ERR_UNSUPPORTED, fn, "needs an in_features that is a multiple of 64, an out_features that is one of 8, and a "
                                             "weight of less than 2^31 elements");
    (void)hipGetLastError();
    const DensePlan plan = plan_dense(rows, out_features, in_features, Sums::kReader);
    return plan.xr == 128 ? launch_dense<128, true>(fn, x, weight, nullptr, sums, rows, out_features, in_features, in_features, NQH_ACT_NONE, 0.f, plan.splits, stream)
                          : launch_dense<256, true>(fn, x, weight, nullptr, sums, rows, out_features, in_features, in_features, NQH_ACT_NONE, 0.f, plan.splits, stream);
}
