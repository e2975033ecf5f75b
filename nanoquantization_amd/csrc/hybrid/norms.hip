// The step between two sublayers on an fp32 residual stream, and the q/k norm + rotary + cache write of an attention
// layer whose norm spans the whole projection.  Byte movers: one workgroup per token row.
#include <algorithm>

#include "moe_route.hpp"

namespace nqh {
namespace {

constexpr int kRowThreads = 256;
constexpr int kMaxWidth = 8192;
constexpr int kRoutedExperts = 128, kRoutedRows = 256;   // limits of the routed form

// What the routed form does behind the norm: router scores of the row, its top experts, and -- by the workgroup that
// comes last -- the plan of all rows (moe_route.hpp).
struct RouteArgs {
    const void* router;
    int32_t* expert;
    float* weight;
    int32_t *order, *tiles;
    int* counter;                        // zero before and after
    int experts, top, tile_rows, max_tiles;
};

template <typename T, typename Y, int V, int THREADS, int P, bool ROUTED>
__global__ __launch_bounds__(THREADS) void residual_norm_kernel(
    float* __restrict__ x, int init, const typename Y::elem* __restrict__ y, int parts, const typename T::elem* __restrict__ post_w, const int64_t* __restrict__ ids,
    const typename T::elem* __restrict__ table, int64_t table_rows, const typename T::elem* __restrict__ next_w,
    typename T::elem* __restrict__ h, int width, float eps, RouteArgs route) {
    constexpr int WAVES = THREADS / 64;
    __shared__ float s_a[WAVES], s_b[WAVES];
    const int64_t row = blockIdx.x, base = row * width;
    float v[P][V], wp[P][V], wn[P][V];
    typename Raw4<T>::type rw[ROUTED ? 8 : 1][P];        // the router's first eight rows
    if constexpr (ROUTED) {
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
            for (int p = 0; p < P; ++p)
                rw[u][p] = *reinterpret_cast<const typename Raw4<T>::type*>(
                    (const typename T::elem*)route.router + (int64_t)min(u, route.experts - 1) * width +
                    min((int)(p * THREADS + threadIdx.x) * 4, width - 4));
    }
    int64_t src = 0;
    if (ids) {
        src = ids[row];
        src = (src < 0 ? 0 : (src >= table_rows ? table_rows - 1 : src)) * width;
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {        // everything that no reduction has to wait for
        const int i = (p * THREADS + threadIdx.x) * V;
#pragma unroll
        for (int e = 0; e < V; ++e) v[p][e] = wp[p][e] = wn[p][e] = 0.f;
        if (i < width) {
            if (!init) load_vec<Fp, V>(x + base + i, v[p]);
            if (post_w) load_vec<T, V>(post_w + i, wp[p]);
            if (h) load_vec<T, V>(next_w + i, wn[p]);
        }
    }
    if (y) {
        float s[P][V], ss = 0.f;
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const int i = (p * THREADS + threadIdx.x) * V;
#pragma unroll
            for (int e = 0; e < V; ++e) s[p][e] = 0.f;
            if (i < width) {
                load_parts<Y, V>(y + row * parts * width + i, parts, width, s[p]);
#pragma unroll
                for (int e = 0; e < V; ++e) ss += s[p][e] * s[p][e];
            }
        }
        if (post_w) {
            const float r = rsqrtf(block_sum<WAVES>(ss, s_a) / (float)width + eps);
#pragma unroll
            for (int p = 0; p < P; ++p)
#pragma unroll
                for (int e = 0; e < V; ++e) v[p][e] += s[p][e] * r * wp[p][e];
        } else {
#pragma unroll
            for (int p = 0; p < P; ++p)
#pragma unroll
                for (int e = 0; e < V; ++e) v[p][e] += s[p][e];
        }
    }
    float ss = 0.f;
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int i = (p * THREADS + threadIdx.x) * V;
        if (i < width) {
            if (ids) {
                float t[V];
                load_vec<T, V>(table + src + i, t);
#pragma unroll
                for (int e = 0; e < V; ++e) v[p][e] += t[e];
            }
            store_vec<Fp, V>(x + base + i, v[p]);
#pragma unroll
            for (int e = 0; e < V; ++e) ss += v[p][e] * v[p][e];
        }
    }
    if (!h) return;
    const float r = rsqrtf(block_sum<WAVES>(ss, s_b) / (float)width + eps);
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int i = (p * THREADS + threadIdx.x) * V;
#pragma unroll
        for (int e = 0; e < V; ++e) v[p][e] *= r * wn[p][e];
        if (i < width) store_vec<T, V>(h + base + i, v[p]);
    }
    if constexpr (ROUTED) {
        __shared__ PlanShared s_plan;
        __shared__ float s_z[kRoutedExperts][WAVES + 1], s_score[kRoutedExperts];
        __shared__ int s_last;
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
        for (int p = 0; p < P; ++p)      // the router reads h as it was stored
#pragma unroll
            for (int e = 0; e < V; ++e) v[p][e] = T::round(v[p][e]);
        for (int x0 = 0; x0 < route.experts; x0 += 8) {   // eight experts' loads and reductions in flight
            float z[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                z[u] = 0.f;
#pragma unroll
                for (int p = 0; p < P; ++p) {
                    const int i = (p * THREADS + threadIdx.x) * V;
                    if (x0 > 0)
                        rw[u][p] = *reinterpret_cast<const typename Raw4<T>::type*>(
                            (const typename T::elem*)route.router + (int64_t)min(x0 + u, route.experts - 1) * width +
                            min(i, width - 4));
                    if (i < width) {
#pragma unroll
                        for (int e = 0; e < V; ++e) z[u] += v[p][e] * Raw4<T>::get(rw[u][p], e);
                    }
                }
            }
#pragma unroll
            for (int o = 32; o >= 1; o >>= 1)
#pragma unroll
                for (int u = 0; u < 8; ++u) z[u] += __shfl_xor(z[u], o);
            if (lane < 8 && x0 + lane < route.experts) {
                float mine = z[0];
#pragma unroll
                for (int u = 1; u < 8; ++u) mine = lane == u ? z[u] : mine;
                s_z[x0 + lane][wave] = mine;
            }
        }
        __syncthreads();
        for (int e = threadIdx.x; e < route.experts; e += THREADS) {
            float z = 0.f;
#pragma unroll
            for (int w = 0; w < WAVES; ++w) z += s_z[e][w];
            s_score[e] = sigmoid_f32(z);
        }
        __syncthreads();
        const int pairs = gridDim.x * route.top;
        __shared__ int s_top[64];
        if (wave == 0)
            wave_topk(s_score, route.experts, route.top, [&](int t, int e, float s) {
                // read by another workgroup of this launch: through the agent's point of coherence
                __hip_atomic_store(route.expert + row * route.top + t, e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                route.weight[row * route.top + t] = s;
                if (t < 64) s_top[t] = e;
            });
        if (gridDim.x == 1 && pairs <= 64) {             // one row: no other workgroup to wait for
            if (wave == 0) {
                wave_lds_fence();
                wave_plan(s_top[min(lane, pairs - 1)], route.order, route.tiles, pairs, route.experts, route.tile_rows,
                          route.max_tiles);
            }
            return;
        }
        if (!awq::arrive_last(route.counter, gridDim.x, &s_last)) return;
        if (threadIdx.x == 0) __hip_atomic_store(route.counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        auto expert_of = [&](int64_t p) {
            return __hip_atomic_load(route.expert + p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        };
        if (pairs <= 64) {
            if (wave == 0)
                wave_plan(expert_of(min(lane, pairs - 1)), route.order, route.tiles, pairs, route.experts, route.tile_rows,
                          route.max_tiles);
            return;
        }
        plan_pairs(s_plan, expert_of, route.order, route.tiles, pairs, route.experts, route.tile_rows, route.max_tiles);
    }
}

// V consecutive elements of a head per lane (V even: rotary pairs never straddle lanes).
template <typename T, int V>
__global__ __launch_bounds__(kRowThreads) void qk_norm_rope_store_kernel(
    const typename T::elem* __restrict__ qkv, const typename T::elem* __restrict__ q_w,
    const typename T::elem* __restrict__ k_w, const float* __restrict__ cos_sin, const int64_t* __restrict__ positions,
    const int64_t* __restrict__ slots, typename T::elem* __restrict__ q_out, typename T::elem* __restrict__ k_cache,
    typename T::elem* __restrict__ v_cache, int heads, int kv_heads, int dim, int vdim, int rot_dims, int k_row,
    int v_row, int64_t max_positions, int64_t num_slots, int block_size, float eps, uint32_t inv_dim, uint32_t inv_vdim) {
    __shared__ float s_q[4], s_k[4];
    // i / n for i * n < 2^32 (checked on the host) as the high half of i * ceil(2^32 / n)
    auto div_by = [](int i, uint32_t inv) { return (int)__umulhi((uint32_t)i, inv); };
    const int64_t row = blockIdx.x;
    const int nq = heads * dim, nk = kv_heads * dim, nv = kv_heads * vdim;
    const typename T::elem* src = qkv + row * (nq + nk + nv);
    float rq = 1.f, rk = 1.f;
    float keep_q[2][V], keep_k[V];       // the first elements stay in registers for the second pass over the row
    if (q_w) {
        float sq = 0.f, sk = 0.f;
        auto square = [&](const typename T::elem* p, int i, int n, float (&a)[V]) {
            float t = 0.f;
#pragma unroll
            for (int e = 0; e < V; ++e) a[e] = 0.f;
            if (i < n) load_vec<T, V>(p + i, a);
#pragma unroll
            for (int e = 0; e < V; ++e) t += a[e] * a[e];
            return t;
        };
        const int i0 = threadIdx.x * V;
        sq = square(src, i0, nq, keep_q[0]);
        sq += square(src, i0 + kRowThreads * V, nq, keep_q[1]);
        sk = square(src + nq, i0, nk, keep_k);
        float a[V];
        for (int i = i0 + 2 * kRowThreads * V; i < nq; i += kRowThreads * V) sq += square(src, i, nq, a);
        for (int i = i0 + kRowThreads * V; i < nk; i += kRowThreads * V) sk += square(src + nq, i, nk, a);
        sk = wave_sum(sk);
        if ((threadIdx.x & 63) == 0) s_k[threadIdx.x >> 6] = sk;
        rq = rsqrtf(block_sum<4>(sq, s_q) / (float)nq + eps);   // its barrier covers s_k
        rk = rsqrtf((s_k[0] + s_k[1] + s_k[2] + s_k[3]) / (float)nk + eps);
    }
    const int64_t slot = slots[row];
    const bool slot_ok = slot >= 0 && slot < num_slots;
    const int64_t blk = slot_ok ? slot / block_size : 0, off = slot_ok ? slot % block_size : 0;
    int64_t pos = positions[row];
    pos = pos < 0 ? 0 : (pos >= max_positions ? max_positions - 1 : pos);
    const float* cs = cos_sin + pos * rot_dims;
    const int half = rot_dims >> 1;

    auto normed_rotated = [&](float (&a)[V], const typename T::elem* w, float r, int d, float (&o)[V]) {
        if (w) {
            float g[V];
            load_vec<T, V>(w, g);
#pragma unroll
            for (int e = 0; e < V; ++e) a[e] = a[e] * r * g[e];
        }
        float cv[V / 2], sv[V / 2];
        const bool whole = V == 8 && rot_dims % 8 == 0 && d + V <= rot_dims;   // aligned quads of cosines and sines
        if constexpr (V == 8) {
            if (whole) {
                load_vec<Fp, 4>(cs + (d >> 1), cv);
                load_vec<Fp, 4>(cs + half + (d >> 1), sv);
            }
        }
#pragma unroll
        for (int e = 0; e < V; e += 2) {
            if (d + e < rot_dims) {
                const float c = whole ? cv[e / 2] : cs[(d + e) >> 1], s = whole ? sv[e / 2] : cs[half + ((d + e) >> 1)];
                o[e] = a[e] * c - a[e + 1] * s;
                o[e + 1] = a[e + 1] * c + a[e] * s;
            } else {
                o[e] = a[e];
                o[e + 1] = a[e + 1];
            }
        }
    };
    auto put_q = [&](int i, float (&a)[V]) {
        const int hd = div_by(i, inv_dim), d = i - hd * dim;
        float o[V];
        normed_rotated(a, q_w ? q_w + i : nullptr, rq, d, o);
        store_vec<T, V>(q_out + (row * heads + hd) * k_row + d, o);
    };
    auto put_k = [&](int i, float (&a)[V]) {
        const int hd = div_by(i, inv_dim), d = i - hd * dim;
        float o[V];
        normed_rotated(a, k_w ? k_w + i : nullptr, rk, d, o);
        store_vec<T, V>(k_cache + ((blk * kv_heads + hd) * block_size + off) * k_row + d, o);
    };
    const int i0 = threadIdx.x * V;
    int kept_q = 0, kept_k = 0;
    if (q_w) {
        if (i0 < nq) put_q(i0, keep_q[0]);
        if (i0 + kRowThreads * V < nq) put_q(i0 + kRowThreads * V, keep_q[1]);
        if (slot_ok && i0 < nk) put_k(i0, keep_k);
        kept_q = 2 * kRowThreads * V;
        kept_k = kRowThreads * V;
    }
    for (int i = i0 + kept_q; i < nq; i += kRowThreads * V) {
        float a[V];
        load_vec<T, V>(src + i, a);
        put_q(i, a);
    }
    const int pad = k_row - dim;
    for (int i = threadIdx.x; i < heads * pad; i += kRowThreads)
        T::store(q_out + (row * heads + i / pad) * k_row + dim + i % pad, 0.f);
    if (!slot_ok) return;
    for (int i = i0 + kept_k; i < nk; i += kRowThreads * V) {
        float a[V];
        load_vec<T, V>(src + nq + i, a);
        put_k(i, a);
    }
    for (int i = threadIdx.x * V; i < nv; i += kRowThreads * V) {
        const int hd = div_by(i, inv_vdim), d = i - hd * vdim;
        float a[V];
        load_vec<T, V>(src + nq + nk + i, a);
        store_vec<T, V>(v_cache + ((blk * kv_heads + hd) * block_size + off) * v_row + d, a);
    }
}

// RMS norm of a head's output, weight, gate.  LANES lanes per (row, head), V columns each and step.
template <typename T, int V, int LANES>
__global__ __launch_bounds__(256) void head_norm_gate_kernel(const float* __restrict__ o,
                                                             const typename T::elem* __restrict__ gate,
                                                             int64_t gate_stride,
                                                             const typename T::elem* __restrict__ w,
                                                             typename T::elem* __restrict__ out, int64_t items, int heads,
                                                             int vdim, float eps) {
    const int64_t want = (int64_t)blockIdx.x * (256 / LANES) + threadIdx.x / LANES;
    const bool live = want < items;      // lanes past the end follow the last item (the shuffles need them)
    const int64_t item = live ? want : items - 1, row = item / heads;
    const int sub = threadIdx.x % LANES, hd = (int)(item % heads);
    const float* src = o + item * vdim;
    float ss = 0.f;
    for (int c = sub * V; c < vdim; c += LANES * V) {
        float a[V];
        load_vec<Fp, V>(src + c, a);
#pragma unroll
        for (int e = 0; e < V; ++e) ss += a[e] * a[e];
    }
#pragma unroll
    for (int x = LANES / 2; x >= 1; x >>= 1) ss += __shfl_xor(ss, x);
    const float r = rsqrtf(ss / (float)vdim + eps);
    const typename T::elem* g = gate + row * gate_stride + (int64_t)hd * vdim;
    if (!live) return;
    for (int c = sub * V; c < vdim; c += LANES * V) {
        float a[V], b[V], n[V];
        load_vec<Fp, V>(src + c, a);
        load_vec<T, V>(g + c, b);
        load_vec<T, V>(w + c, n);
#pragma unroll
        for (int e = 0; e < V; ++e) a[e] = a[e] * r * n[e] * silu_f32(b[e]);
        store_vec<T, V>(out + item * vdim + c, a);
    }
}

}  // namespace
}  // namespace nqh

using namespace nqh;

static int check_residual(const char* fn, const float* x, const void* y, int64_t y_parts, const int64_t* ids,
                          const void* table, int64_t table_rows, const void* next_weight, const void* h, int64_t rows,
                          int64_t width, int dtype) {
    if (!x || (ids && !table) || (h && !next_weight)) return fail(NQH_ERR_ARG, fn, "null pointer");
    if (!dtype_ok(dtype)) return fail(NQH_ERR_ARG, fn, "dtype must be NQH_BF16 or NQH_F32");
    if (rows <= 0 || rows > kMaxI32 || width <= 0 || (y && (y_parts <= 0 || y_parts > kMaxI32)) || (ids && table_rows <= 0))
        return fail(NQH_ERR_ARG, fn, "sizes must be positive 31-bit counts");
    if (width > kMaxWidth) return fail(NQH_ERR_UNSUPPORTED, fn, "width %lld exceeds %d", (long long)width, kMaxWidth);
    return NQH_OK;
}

static bool residual_vec(const void* x, const void* y, const void* post_weight, const void* table, const void* next_weight,
                         const void* h, int64_t width) {
    return width % 4 == 0 && aligned(x, 16) && aligned(y, 16) && aligned(post_weight, 16) && aligned(table, 16) &&
           aligned(next_weight, 16) && aligned(h, 16);
}

#define NQH_ARGS                                                                                                          \
    x, init, (const typename Y::elem*)y, (int)y_parts, (const E*)post_weight, ids, (const E*)table, table_rows, (const E*)next_weight,   \
        (E*)h, (int)width, eps
extern "C" int nqh_residual_norm(float* x, int init, const void* y, int64_t y_parts, const void* post_weight,
                                 const int64_t* ids, const void* table, int64_t table_rows, const void* next_weight,
                                 void* h, int64_t rows, int64_t width, float eps, int dtype, void* stream) {
    const char* fn = "nqh_residual_norm";
    const bool y_f32 = (dtype & NQH_Y_F32) != 0;
    dtype &= ~NQH_Y_F32;
    const int rc = check_residual(fn, x, y, y_parts, ids, table, table_rows, next_weight, h, rows, width, dtype);
    if (rc != NQH_OK) return rc;
    const bool vec = residual_vec(x, y, post_weight, table, next_weight, h, width);
    hipStream_t st = (hipStream_t)stream;
    (void)hipGetLastError();
#define NQH_GO(V, THREADS, P)                                                                                     \
    residual_norm_kernel<T, Y, V, THREADS, P, false><<<dim3((unsigned)rows), dim3(THREADS), 0, st>>>(NQH_ARGS, RouteArgs{})
    NQH_WITH_TYPE(dtype, {
        using E = typename T::elem;
        NQH_WITH_Y(y_f32, {
            if (!vec) NQH_GO(1, 1024, 8);
            else if (width <= 1024) NQH_GO(4, 256, 1);
            else if (rows <= 256 && width <= 4096) NQH_GO(4, 1024, 1);   // few rows: more loads in flight per row
            else if (rows <= 256) NQH_GO(4, 1024, 2);
            else if (width <= 2048) NQH_GO(4, 256, 2);
            else if (width <= 4096) NQH_GO(4, 256, 4);
            else NQH_GO(4, 256, 8);
        });
    });
#undef NQH_GO
    return launched(fn);
}

extern "C" int nqh_residual_norm_route_supported(int64_t rows, int64_t width, int64_t experts) {
    return rows >= 1 && rows <= kRoutedRows && width % 4 == 0 && width <= kMaxWidth && experts <= kRoutedExperts;
}

extern "C" int nqh_residual_norm_route(float* x, int init, const void* y, int64_t y_parts, const void* post_weight,
                                       const int64_t* ids, const void* table, int64_t table_rows, const void* next_weight,
                                       void* h, const void* router, int32_t* expert, float* weight, int32_t* order,
                                       int32_t* tiles, int32_t* counter, int64_t rows, int64_t width, int64_t experts,
                                       int64_t top, int64_t tile_rows, int64_t max_tiles, float eps, int dtype,
                                       void* stream) {
    const char* fn = "nqh_residual_norm_route";
    const bool y_f32 = (dtype & NQH_Y_F32) != 0;
    dtype &= ~NQH_Y_F32;
    const int rc = check_residual(fn, x, y, y_parts, ids, table, table_rows, next_weight, h, rows, width, dtype);
    if (rc != NQH_OK) return rc;
    if (!h || !router || !expert || !weight || !order || !tiles || !counter) return fail(NQH_ERR_ARG, fn, "null pointer");
    if (!nqh_residual_norm_route_supported(rows, width, experts) || !aligned(router, 16) ||
        !residual_vec(x, y, post_weight, table, next_weight, h, width))
        return fail(NQH_ERR_UNSUPPORTED, fn, "at most %d rows and %d experts, width a multiple of 4, 16-byte aligned tensors",
                    kRoutedRows, kRoutedExperts);
    if (experts <= 0 || top <= 0 || top > experts || tile_rows <= 0 || tile_rows > kMaxI32 || 3 * max_tiles > kMaxI32 ||
        max_tiles < nqh_moe_max_tiles(rows * top, experts, tile_rows))
        return fail(NQH_ERR_ARG, fn, "top must be 1 .. experts and max_tiles nqh_moe_max_tiles or more");
    const RouteArgs route{router, expert, weight, order, tiles, counter, (int)experts, (int)top, (int)tile_rows, (int)max_tiles};
    hipStream_t st = (hipStream_t)stream;
    (void)hipGetLastError();
#define NQH_GO(V, THREADS, P)                                                                                     \
    residual_norm_kernel<T, Y, V, THREADS, P, true><<<dim3((unsigned)rows), dim3(THREADS), 0, st>>>(NQH_ARGS, route)
    NQH_WITH_TYPE(dtype, {
        using E = typename T::elem;
        NQH_WITH_Y(y_f32, {
            if (width <= 1024) NQH_GO(4, 256, 1);
            else if (width <= 4096) NQH_GO(4, 1024, 1);
            else NQH_GO(4, 1024, 2);
        });
    });
#undef NQH_GO
    return launched(fn);
}
#undef NQH_ARGS

extern "C" int nqh_qk_norm_rope_store(const void* qkv, const void* q_weight, const void* k_weight, const float* cos_sin,
                                      const int64_t* positions, const int64_t* slots, void* q_out, void* k_cache,
                                      void* v_cache, int64_t rows, int64_t heads, int64_t kv_heads, int64_t dim,
                                      int64_t vdim, int64_t rot_dims, int64_t k_row, int64_t v_row,
                                      int64_t max_positions, int64_t num_slots, int64_t block_size, float eps, int dtype,
                                      void* stream) {
    const char* fn = "nqh_qk_norm_rope_store";
    if (!qkv || !positions || !slots || !q_out || !k_cache || !v_cache || (rot_dims > 0 && !cos_sin) ||
        (!q_weight != !k_weight))
        return fail(NQH_ERR_ARG, fn, "null pointer");
    if (!dtype_ok(dtype)) return fail(NQH_ERR_ARG, fn, "dtype must be NQH_BF16 or NQH_F32");
    if (rows <= 0 || rows > kMaxI32 || heads <= 0 || kv_heads <= 0 || dim <= 0 || vdim <= 0 || max_positions <= 0 ||
        num_slots <= 0 || block_size <= 0 || block_size > kMaxI32 || num_slots % block_size != 0 ||
        heads * k_row > kMaxI32 || kv_heads * v_row > kMaxI32)
        return fail(NQH_ERR_ARG, fn, "sizes must be positive and num_slots a multiple of block_size");
    if (dim % 2 != 0 || rot_dims < 0 || rot_dims % 2 != 0 || rot_dims > dim || k_row < dim || v_row < vdim)
        return fail(NQH_ERR_ARG, fn, "dim and rot_dims must be even, rot_dims <= dim, and rows at least as wide as heads");
    const bool vec = dim % 8 == 0 && vdim % 8 == 0 && k_row % 8 == 0 && v_row % 8 == 0 && aligned(qkv, 16) &&
                     aligned(q_weight, 16) && aligned(k_weight, 16) && aligned(q_out, 16) && aligned(k_cache, 16) &&
                     aligned(v_cache, 16);
    const uint32_t inv_dim = (uint32_t)((((uint64_t)1 << 32) + dim - 1) / dim), inv_vdim = (uint32_t)((((uint64_t)1 << 32) + vdim - 1) / vdim);
    if ((heads + kv_heads) * std::max(dim, vdim) * std::max(dim, vdim) >= ((int64_t)1 << 32) || dim < 2 || vdim < 2)
        return fail(NQH_ERR_UNSUPPORTED, fn, "heads too wide");
    if (!vec && vdim % 2 != 0) return fail(NQH_ERR_UNSUPPORTED, fn, "vdim must be even");
    (void)hipGetLastError();
#define NQH_ARGS (const E*)qkv, (const E*)q_weight, (const E*)k_weight, cos_sin, positions, slots, (E*)q_out,           \
                  (E*)k_cache, (E*)v_cache, (int)heads, (int)kv_heads, (int)dim, (int)vdim, (int)rot_dims, (int)k_row,   \
                  (int)v_row, max_positions, num_slots, (int)block_size, eps, inv_dim, inv_vdim
    NQH_WITH_TYPE(dtype, {
        using E = typename T::elem;
        if (vec)
            qk_norm_rope_store_kernel<T, 8><<<dim3((unsigned)rows), dim3(kRowThreads), 0, (hipStream_t)stream>>>(NQH_ARGS);
        else
            qk_norm_rope_store_kernel<T, 2><<<dim3((unsigned)rows), dim3(kRowThreads), 0, (hipStream_t)stream>>>(NQH_ARGS);
    });
#undef NQH_ARGS
    return launched(fn);
}

extern "C" int nqh_head_norm_gate(const float* o, const void* gate, int64_t gate_stride, const void* weight, void* out,
                                  int64_t rows, int64_t heads, int64_t vdim, float eps, int dtype, void* stream) {
    const char* fn = "nqh_head_norm_gate";
    if (!o || !gate || !weight || !out) return fail(NQH_ERR_ARG, fn, "null pointer");
    if (!dtype_ok(dtype)) return fail(NQH_ERR_ARG, fn, "dtype must be NQH_BF16 or NQH_F32");
    if (rows <= 0 || heads <= 0 || vdim <= 0 || heads > kMaxI32 || vdim > kMaxI32 || cdiv(rows * heads, 4) > kMaxI32 ||
        gate_stride < heads * vdim)
        return fail(NQH_ERR_ARG, fn, "sizes must be positive and the gate row at least heads * vdim wide");
    (void)hipGetLastError();
    NQH_WITH_TYPE(dtype, {
        using E = typename T::elem;
        const bool vec = vdim % 4 == 0 && gate_stride % 4 == 0 && aligned(o, 16) && aligned(gate, 4 * sizeof(E)) &&
                         aligned(weight, 4 * sizeof(E)) && aligned(out, 4 * sizeof(E));
        const int64_t items = rows * heads;
        if (vec && vdim <= 64)
            head_norm_gate_kernel<T, 4, 16><<<dim3((unsigned)cdiv(items, 16)), dim3(256), 0, (hipStream_t)stream>>>(
                o, (const E*)gate, gate_stride, (const E*)weight, (E*)out, items, (int)heads, (int)vdim, eps);
        else if (vec)
            head_norm_gate_kernel<T, 4, 32><<<dim3((unsigned)cdiv(items, 8)), dim3(256), 0, (hipStream_t)stream>>>(
                o, (const E*)gate, gate_stride, (const E*)weight, (E*)out, items, (int)heads, (int)vdim, eps);
        else
            head_norm_gate_kernel<T, 1, 64><<<dim3((unsigned)cdiv(items, 4)), dim3(256), 0, (hipStream_t)stream>>>(
                o, (const E*)gate, gate_stride, (const E*)weight, (E*)out, items, (int)heads, (int)vdim, eps);
    });
    return launched(fn);
}
