// PyTorch-ROCm operator binding over the C ABI of libawq_hip.so (include/awq_hip.h).
//
// No kernels here: every operator checks its arguments the way the reference's Python entry points do
// (nanoquantization/layers/gemm.py:126-180 awq_dequantize, :329-379 awq_gemm, :552-567 WQLinear_GEMM.forward),
// allocates the output with torch, and calls the C entry point on torch's current HIP stream -- where the
// reference's Triton launches go (layers/gemm.py:363-377).  Registered as
//   torch.ops.nanoquantization_amd.awq_dequantize(qweight, qscales, qzeros) -> Tensor [K, N]
//   torch.ops.nanoquantization_amd.awq_linear(x, qweight, qscales, qzeros, bias?) -> Tensor [M, N]
//   torch.ops.nanoquantization_amd.awq_linear_swiglu(x, qweight, qscales, qzeros) -> Tensor [M, N / 2]
// and the steps between the linears of the Qwen3 modules (nanoquantization/layers/norm.py:18-32, layers/rope.py:24-45,
// models/qwen3_quantized.py:79-99, 147-152), inference only (none has a derivative):
//   awq_swiglu_pair, awq_linear_three, awq_linear_add, rms_norm, silu_mul, qkv_norm_rope, causal_attention
// with Meta kernels (shapes only), so the operators are visible to the dispatcher and to tracing.
#include <dlfcn.h>

#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <torch/library.h>

#include <array>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "../../include/awq_hip.h"
#include "../../include/nq_engine_ops.h"
#include "../../include/nq_hybrid_ops.h"

namespace {

// PyTorch-ROCm labels HIP tensors and streams with the device type "cuda"; these are the HIP guard and stream
// getters for that labelling.
using DeviceGuard = c10::hip::HIPGuardMasqueradingAsCUDA;
hipStream_t current_stream(c10::DeviceIndex index) {
    return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(index).stream();
}

struct Packed {
    int64_t K, N, g;
    int dtype;
};

Packed check_packed(const at::Tensor& qweight, const at::Tensor& qscales, const at::Tensor& qzeros) {
    TORCH_CHECK(qweight.dim() == 2 && qscales.dim() == 2 && qzeros.dim() == 2,
                "qweight, qscales and qzeros must be 2-D");
    TORCH_CHECK(qweight.scalar_type() == at::kInt && qzeros.scalar_type() == at::kInt,
                "qweight and qzeros must be int32");
    TORCH_CHECK(qscales.scalar_type() == at::kHalf || qscales.scalar_type() == at::kBFloat16,
                "qscales dtype must be float16 or bfloat16, got ", qscales.scalar_type());
    Packed p;
    p.K = qweight.size(0);
    p.N = qscales.size(1);
    TORCH_CHECK(p.K > 0 && p.N > 0 && qscales.size(0) > 0, "empty packed weight");
    p.g = p.K / qscales.size(0);
    TORCH_CHECK(qweight.size(1) * 8 == p.N, "qweight must be [K, N/8]");
    TORCH_CHECK(qscales.size(0) * p.g == p.K, "qscales must be [K/g, N]");
    TORCH_CHECK(qzeros.size(0) == qscales.size(0) && qzeros.size(1) * 8 == p.N, "qzeros must be [K/g, N/8]");
    TORCH_CHECK(p.g == 32 || p.g == 64 || p.g == 128 || p.g == p.K, "unsupported group size ", p.g);
    p.dtype = qscales.scalar_type() == at::kHalf ? AWQ_F16 : AWQ_BF16;
    return p;
}

void check_device(const at::Tensor& ref, std::initializer_list<const at::Tensor*> others) {
    TORCH_CHECK(ref.is_cuda(), "AWQ kernels run on a HIP device only (tensor is on ", ref.device(),
                "); there is no CPU fallback");
    for (const at::Tensor* t : others)
        TORCH_CHECK(t->device() == ref.device(), "tensors on different devices: ", t->device(), " vs ", ref.device());
}

void check_status(int status, const char* entry) {
    TORCH_CHECK(status == AWQ_OK, "libawq_hip: ", entry, " failed (status ", status, "): ", awq_hip_last_error());
}

// One zero-filled split-K workspace per (device, stream).  The kernels leave it zeroed and calls on one stream are
// ordered, so every layer shares it.  A workspace is never freed: a HIP graph captured while it was current keeps
// its address, so a larger request retires the old tensor instead of releasing it.
struct WsKey {
    int device;
    void* stream;
    bool operator==(const WsKey& o) const { return device == o.device && stream == o.stream; }
};
struct WsHash {
    size_t operator()(const WsKey& k) const { return std::hash<void*>()(k.stream) ^ (size_t)k.device * 0x9E3779B97F4A7C15ull; }
};
std::mutex g_ws_mutex;
std::unordered_map<WsKey, at::Tensor, WsHash> g_ws;
std::vector<at::Tensor> g_ws_retired;

at::Tensor workspace(const at::Device& dev, void* stream, size_t nbytes) {
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    const WsKey key{dev.index(), stream};
    auto it = g_ws.find(key);
    if (it != g_ws.end() && (size_t)it->second.numel() >= nbytes) return it->second;
    if (it != g_ws.end()) g_ws_retired.push_back(it->second);
    const int64_t size = (int64_t)std::max<size_t>(nbytes, (size_t)8 << 20);
    at::Tensor ws = at::zeros({size}, at::TensorOptions().dtype(at::kByte).device(dev));
    g_ws[key] = ws;
    return ws;
}

// Memory from the caching allocator for one call (ordered on the current stream like any temporary); undefined without room.
at::Tensor bytes_or_none(const at::Device& dev, size_t nbytes) {
    try {
        return at::empty({(int64_t)nbytes}, at::TensorOptions().dtype(at::kByte).device(dev));
    } catch (const c10::OutOfMemoryError&) {
        return {};
    }
}

// Scratch for awq_linear_dense where that is the fastest way, else undefined; without room for it the fused kernels run.
at::Tensor dense_scratch(const at::Device& dev, int64_t M, const Packed& p) {
    const size_t nbytes = M > 128 ? awq_linear_scratch_bytes(M, p.N, p.K, p.g, p.dtype) : 0;
    return nbytes ? bytes_or_none(dev, nbytes) : at::Tensor();
}

at::Tensor awq_dequantize_op(const at::Tensor& qweight, const at::Tensor& qscales, const at::Tensor& qzeros) {
    const Packed p = check_packed(qweight, qscales, qzeros);
    check_device(qweight, {&qscales, &qzeros});
    const DeviceGuard guard(qweight.device());
    const at::Tensor qw = qweight.contiguous(), qs = qscales.contiguous(), qz = qzeros.contiguous();
    at::Tensor out = at::empty({p.K, p.N}, qs.options());
    hipStream_t stream = current_stream(qw.device().index());
    check_status(awq_dequantize(qw.data_ptr<int32_t>(), qs.data_ptr(), qz.data_ptr<int32_t>(), out.data_ptr(), p.K,
                                p.N, p.g, p.dtype, stream),
                 "awq_dequantize");
    return out;
}

at::Tensor awq_dequantize_meta(const at::Tensor& qweight, const at::Tensor& qscales, const at::Tensor& qzeros) {
    return at::empty({qweight.size(0), qscales.size(1)}, qscales.options());
}

using LinearEntry = int (*)(const void*, const int32_t*, const void*, const int32_t*, const void*, void*, int64_t,
                            int64_t, int64_t, int64_t, int, void*, size_t, void*);

at::Tensor awq_linear_op(const at::Tensor& x, const at::Tensor& qweight, const at::Tensor& qscales,
                         const at::Tensor& qzeros, const c10::optional<at::Tensor>& bias) {
    const Packed p = check_packed(qweight, qscales, qzeros);
    TORCH_CHECK(x.dim() == 2 && x.size(1) == p.K, "x must be [M, ", p.K, "], got ", x.sizes());
    check_device(x, {&qweight, &qscales, &qzeros});
    const DeviceGuard guard(x.device());
    const at::ScalarType dt = qscales.scalar_type();
    // the reference casts x to the output dtype on load (layers/gemm.py:259)
    const at::Tensor xc = (x.scalar_type() == dt ? x : x.to(dt)).contiguous();
    const at::Tensor qw = qweight.contiguous(), qs = qscales.contiguous(), qz = qzeros.contiguous();
    at::Tensor b;
    if (bias.has_value() && bias->defined()) {
        TORCH_CHECK(bias->numel() == p.N, "bias must have ", p.N, " elements");
        b = bias->to(x.device(), dt).contiguous();
    }
    const int64_t M = xc.size(0);
    at::Tensor out = at::empty({M, p.N}, qs.options());
    if (M == 0) return out;
    hipStream_t stream = current_stream(x.device().index());
    if (const at::Tensor scratch = dense_scratch(x.device(), M, p); scratch.defined()) {
        check_status(awq_linear_dense(xc.data_ptr(), qw.data_ptr<int32_t>(), qs.data_ptr(), qz.data_ptr<int32_t>(),
                                      b.defined() ? b.data_ptr() : nullptr, out.data_ptr(), M, p.N, p.K, p.g, p.dtype, 0,
                                      scratch.data_ptr(), (size_t)scratch.numel(), stream),
                     "awq_linear_dense");
        return out;
    }
    const size_t nbytes = awq_linear_workspace_bytes(M, p.N, p.K);
    at::Tensor ws;
    if (nbytes) ws = workspace(x.device(), stream, nbytes);
    check_status(awq_linear(xc.data_ptr(), qw.data_ptr<int32_t>(), qs.data_ptr(), qz.data_ptr<int32_t>(),
                            b.defined() ? b.data_ptr() : nullptr, out.data_ptr(), M, p.N, p.K, p.g, p.dtype,
                            nbytes ? ws.data_ptr() : nullptr, nbytes ? (size_t)ws.numel() : 0, stream),
                 "awq_linear");
    return out;
}

// residual + awq_linear(x): in the product's last step where the weight is dequantised first, else an addition of its own.
at::Tensor awq_linear_add_op(const at::Tensor& x, const at::Tensor& qweight, const at::Tensor& qscales, const at::Tensor& qzeros,
                             const at::Tensor& residual) {
    const Packed p = check_packed(qweight, qscales, qzeros);
    TORCH_CHECK(x.dim() == 2 && x.size(1) == p.K, "x must be [M, ", p.K, "], got ", x.sizes());
    const int64_t M = x.size(0);
    TORCH_CHECK(residual.dim() == 2 && residual.size(0) == M && residual.size(1) == p.N && residual.scalar_type() == qscales.scalar_type(),
                "residual must be [", M, ", ", p.N, "] of the scales' type, got ", residual.sizes());
    check_device(x, {&qweight, &qscales, &qzeros, &residual});
    const DeviceGuard guard(x.device());
    const bool dense = residual.is_contiguous() && !(reinterpret_cast<uintptr_t>(residual.data_ptr()) & 15u) && p.N <= (1 << 22);
    if (const at::Tensor scratch = dense ? dense_scratch(x.device(), M, p) : at::Tensor(); scratch.defined()) {
        const at::ScalarType dt = qscales.scalar_type();
        const at::Tensor xc = (x.scalar_type() == dt ? x : x.to(dt)).contiguous();
        const at::Tensor qw = qweight.contiguous(), qs = qscales.contiguous(), qz = qzeros.contiguous();
        at::Tensor out = at::empty({M, p.N}, qs.options());
        check_status(awq_linear_dense_add(xc.data_ptr(), qw.data_ptr<int32_t>(), qs.data_ptr(), qz.data_ptr<int32_t>(), residual.data_ptr(),
                                          out.data_ptr(), M, p.N, p.K, p.g, p.dtype, scratch.data_ptr(), (size_t)scratch.numel(),
                                          current_stream(x.device().index())),
                     "awq_linear_dense_add");
        return out;
    }
    return at::add(residual, awq_linear_op(x, qweight, qscales, qzeros, c10::nullopt));
}
at::Tensor awq_linear_add_meta(const at::Tensor&, const at::Tensor&, const at::Tensor&, const at::Tensor&, const at::Tensor& residual) {
    return at::empty(residual.sizes(), residual.options());
}

at::Tensor awq_linear_meta(const at::Tensor& x, const at::Tensor& qweight, const at::Tensor& qscales,
                           const at::Tensor& qzeros, const c10::optional<at::Tensor>& bias) {
    return at::empty({x.size(0), qscales.size(1)}, qscales.options());
}

at::Tensor awq_linear_swiglu_op(const at::Tensor& x, const at::Tensor& qweight, const at::Tensor& qscales,
                                const at::Tensor& qzeros) {
    const Packed p = check_packed(qweight, qscales, qzeros);
    TORCH_CHECK(x.dim() == 2 && x.size(1) == p.K, "x must be [M, ", p.K, "], got ", x.sizes());
    TORCH_CHECK(p.N % 16 == 0, "gate|up interleaved by words needs N % 16 == 0");
    check_device(x, {&qweight, &qscales, &qzeros});
    const DeviceGuard guard(x.device());
    const at::ScalarType dt = qscales.scalar_type();
    const at::Tensor xc = (x.scalar_type() == dt ? x : x.to(dt)).contiguous();
    const at::Tensor qw = qweight.contiguous(), qs = qscales.contiguous(), qz = qzeros.contiguous();
    const int64_t M = xc.size(0);
    at::Tensor out = at::empty({M, p.N / 2}, qs.options());
    if (M == 0) return out;
    hipStream_t stream = current_stream(x.device().index());
    if (const at::Tensor scratch = dense_scratch(x.device(), M, p); scratch.defined()) {
        check_status(awq_linear_dense(xc.data_ptr(), qw.data_ptr<int32_t>(), qs.data_ptr(), qz.data_ptr<int32_t>(), nullptr,
                                      out.data_ptr(), M, p.N, p.K, p.g, p.dtype, 1, scratch.data_ptr(),
                                      (size_t)scratch.numel(), stream),
                     "awq_linear_dense");
        return out;
    }
    const size_t nbytes = awq_linear_swiglu_workspace_bytes(M, p.N, p.K);
    at::Tensor ws;
    if (nbytes) ws = workspace(x.device(), stream, nbytes);
    check_status(awq_linear_swiglu(xc.data_ptr(), qw.data_ptr<int32_t>(), qs.data_ptr(), qz.data_ptr<int32_t>(),
                                   out.data_ptr(), M, p.N, p.K, p.g, p.dtype, nbytes ? ws.data_ptr() : nullptr,
                                   nbytes ? (size_t)ws.numel() : 0, stream),
                 "awq_linear_swiglu");
    return out;
}

at::Tensor awq_linear_swiglu_meta(const at::Tensor& x, const at::Tensor& qweight, const at::Tensor& qscales,
                                  const at::Tensor& qzeros) {
    return at::empty({x.size(0), qscales.size(1) / 2}, qscales.options());
}

// ---- the steps between the linears -------------------------------------------------------------------------------------
int dtype_of(const at::Tensor& t) {
    TORCH_CHECK(t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16, "float16 or bfloat16 expected, got ",
                t.scalar_type());
    return t.scalar_type() == at::kHalf ? AWQ_F16 : AWQ_BF16;
}

// Dense and 16-byte aligned, as the kernels' accesses want it: a view into the middle of a buffer may be neither.
at::Tensor dense16(const at::Tensor& t) {
    const at::Tensor d = t.contiguous();
    return reinterpret_cast<uintptr_t>(d.data_ptr()) & 15u ? d.clone() : d;
}

// The result has the strides that elementwise operations on x give (x's own, where x is dense in some order of its dimensions).
at::Tensor rms_norm_op(const at::Tensor& x, const at::Tensor& weight, double eps) {
    const int dtype = dtype_of(x);
    TORCH_CHECK(x.dim() >= 1 && weight.dim() == 1 && x.size(-1) == weight.size(0) && weight.scalar_type() == x.scalar_type(),
                "weight must be [x.size(-1)] of x's dtype");
    check_device(x, {&weight});
    const DeviceGuard guard(x.device());
    at::Tensor y = at::empty_like(x);
    if (x.numel() == 0) return y;
    const at::Tensor out = y.is_contiguous() ? y : at::empty(x.sizes(), x.options());
    const at::Tensor xd = dense16(x), w = dense16(weight);
    const int64_t hidden = x.size(-1);
    check_status(nq_add_rmsnorm(xd.data_ptr(), nullptr, w.data_ptr(), out.data_ptr(), x.numel() / hidden, hidden, (float)eps,
                                dtype, current_stream(x.device().index())),
                 "nq_add_rmsnorm");
    if (!out.is_same(y)) y.copy_(out);
    return y;
}
at::Tensor rms_norm_meta(const at::Tensor& x, const at::Tensor&, double) { return at::empty_like(x); }

at::Tensor silu_mul_op(const at::Tensor& gate, const at::Tensor& up) {
    const int dtype = dtype_of(gate);
    TORCH_CHECK(gate.dim() >= 1 && gate.sizes() == up.sizes() && gate.scalar_type() == up.scalar_type(),
                "gate and up must be alike");
    check_device(gate, {&up});
    const DeviceGuard guard(gate.device());
    at::Tensor y = at::empty(gate.sizes(), gate.options());
    if (gate.numel() == 0) return y;
    const at::Tensor g = dense16(gate), u = dense16(up);
    const int64_t inter = gate.size(-1);
    check_status(nq_silu_mul_pair(g.data_ptr(), u.data_ptr(), y.data_ptr(), gate.numel() / inter, inter, dtype,
                                  current_stream(gate.device().index())),
                 "nq_silu_mul_pair");
    return y;
}
at::Tensor silu_mul_meta(const at::Tensor& gate, const at::Tensor&) { return at::empty(gate.sizes(), gate.options()); }

// Linears without bias of one input, by triples of packed weight, scales and zero points: one launch where that is the fastest
// way, else one each.
std::vector<at::Tensor> linear_parts(const at::Tensor& x, const std::vector<std::array<at::Tensor, 3>>& in) {
    const int count = (int)in.size();
    Packed p[3];
    int64_t N[3];
    TORCH_CHECK(count >= 1 && count <= 3, "one to three weights");
    for (int i = 0; i < count; ++i) {
        p[i] = check_packed(in[i][0], in[i][1], in[i][2]);
        TORCH_CHECK(p[i].K == p[0].K && p[i].g == p[0].g && p[i].dtype == p[0].dtype, "the weights must have one K, group size and type");
        check_device(x, {&in[i][0], &in[i][1], &in[i][2]});
        N[i] = p[i].N;
    }
    TORCH_CHECK(x.dim() == 2 && x.size(1) == p[0].K, "x must be [M, ", p[0].K, "], got ", x.sizes());
    const DeviceGuard guard(x.device());
    const int64_t M = x.size(0);
    size_t nbytes = 0, scratch_bytes = 0;
    at::Tensor scratch;
    std::vector<at::Tensor> out(count);
    bool one = awq_linear_parts_wanted(N, count, M, p[0].K, p[0].g, p[0].dtype, &nbytes, &scratch_bytes) != 0;
    if (one && scratch_bytes) one = (scratch = bytes_or_none(x.device(), scratch_bytes)).defined();
    if (!one) {
        for (int i = 0; i < count; ++i) out[i] = awq_linear_op(x, in[i][0], in[i][1], in[i][2], c10::nullopt);
        return out;
    }
    const at::ScalarType dt = in[0][1].scalar_type();
    const at::Tensor xc = (x.scalar_type() == dt ? x : x.to(dt)).contiguous();
    at::Tensor dense[3][3];
    const int32_t* words[3];
    const void* scales[3];
    const int32_t* zeros[3];
    void* y[3];
    for (int i = 0; i < count; ++i) {
        for (int j = 0; j < 3; ++j) dense[i][j] = in[i][j].contiguous();
        out[i] = at::empty({M, N[i]}, in[0][1].options());
        words[i] = dense[i][0].data_ptr<int32_t>(), scales[i] = dense[i][1].data_ptr(), zeros[i] = dense[i][2].data_ptr<int32_t>();
        y[i] = out[i].data_ptr();
    }
    hipStream_t stream = current_stream(x.device().index());
    at::Tensor ws;
    if (nbytes) ws = workspace(x.device(), stream, nbytes);
    check_status(awq_linear_parts(xc.data_ptr(), words, scales, zeros, y, N, count, M, p[0].K, p[0].g, p[0].dtype,
                                  nbytes ? ws.data_ptr() : nullptr, nbytes ? (size_t)ws.numel() : 0,
                                  scratch.defined() ? scratch.data_ptr() : nullptr, scratch_bytes, stream),
                 "awq_linear_parts");
    return out;
}

// gate and up of an MLP that lie apart: one product where the rows are many, else two and the activation.
at::Tensor awq_swiglu_pair_op(const at::Tensor& x, const at::Tensor& gate_qweight, const at::Tensor& gate_qscales,
                              const at::Tensor& gate_qzeros, const at::Tensor& up_qweight, const at::Tensor& up_qscales,
                              const at::Tensor& up_qzeros) {
    Packed p = check_packed(gate_qweight, gate_qscales, gate_qzeros);
    const Packed up = check_packed(up_qweight, up_qscales, up_qzeros);
    TORCH_CHECK(p.K == up.K && p.N == up.N && p.g == up.g && p.dtype == up.dtype, "gate and up must be alike");
    TORCH_CHECK(x.dim() == 2 && x.size(1) == p.K, "x must be [M, ", p.K, "], got ", x.sizes());
    check_device(x, {&gate_qweight, &gate_qscales, &gate_qzeros, &up_qweight, &up_qscales, &up_qzeros});
    const DeviceGuard guard(x.device());
    const int64_t M = x.size(0);
    p.N *= 2;
    const at::Tensor scratch = M > 0 ? dense_scratch(x.device(), M, p) : at::Tensor();
    if (!scratch.defined()) {
        const std::vector<at::Tensor> y = linear_parts(x, {{gate_qweight, gate_qscales, gate_qzeros}, {up_qweight, up_qscales, up_qzeros}});
        return silu_mul_op(y[0], y[1]);
    }
    const at::ScalarType dt = gate_qscales.scalar_type();
    const at::Tensor xc = (x.scalar_type() == dt ? x : x.to(dt)).contiguous();
    const at::Tensor gw = gate_qweight.contiguous(), gs = gate_qscales.contiguous(), gz = gate_qzeros.contiguous(),
                     uw = up_qweight.contiguous(), us = up_qscales.contiguous(), uz = up_qzeros.contiguous();
    at::Tensor out = at::empty({M, up.N}, gs.options());
    check_status(awq_linear_dense_pair(xc.data_ptr(), gw.data_ptr<int32_t>(), gs.data_ptr(), gz.data_ptr<int32_t>(),
                                       uw.data_ptr<int32_t>(), us.data_ptr(), uz.data_ptr<int32_t>(), out.data_ptr(), M, up.N, p.K,
                                       p.g, p.dtype, scratch.data_ptr(), (size_t)scratch.numel(),
                                       current_stream(x.device().index())),
                 "awq_linear_dense_pair");
    return out;
}
at::Tensor awq_swiglu_pair_meta(const at::Tensor& x, const at::Tensor&, const at::Tensor& gate_qscales, const at::Tensor&,
                                const at::Tensor&, const at::Tensor&, const at::Tensor&) {
    return at::empty({x.size(0), gate_qscales.size(1)}, gate_qscales.options());
}

using Three = std::tuple<at::Tensor, at::Tensor, at::Tensor>;

// Three linears without bias of one input.
Three awq_linear_three_op(const at::Tensor& x, const at::Tensor& qweight0, const at::Tensor& qscales0, const at::Tensor& qzeros0,
                          const at::Tensor& qweight1, const at::Tensor& qscales1, const at::Tensor& qzeros1,
                          const at::Tensor& qweight2, const at::Tensor& qscales2, const at::Tensor& qzeros2) {
    std::vector<at::Tensor> y = linear_parts(x, {{qweight0, qscales0, qzeros0}, {qweight1, qscales1, qzeros1}, {qweight2, qscales2, qzeros2}});
    return {y[0], y[1], y[2]};
}
Three awq_linear_three_meta(const at::Tensor& x, const at::Tensor&, const at::Tensor& qscales0, const at::Tensor&, const at::Tensor&,
                            const at::Tensor& qscales1, const at::Tensor&, const at::Tensor&, const at::Tensor& qscales2,
                            const at::Tensor&) {
    const auto like = [&](const at::Tensor& s) { return at::empty({x.size(0), s.size(1)}, s.options()); };
    return {like(qscales0), like(qscales1), like(qscales2)};
}

Three qkv_outputs(const at::Tensor& q, int64_t heads, int64_t kv_heads) {
    const int64_t b = q.size(0), s = q.size(1), hd = q.size(2) / heads;
    return {at::empty({b, s, heads, hd}, q.options()), at::empty({b, kv_heads, s, hd}, q.options()),
            at::empty({b, kv_heads, s, hd}, q.options())};
}

Three qkv_norm_rope_op(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& q_weight,
                       const at::Tensor& k_weight, const at::Tensor& cos_sin, const at::Tensor& positions, int64_t heads,
                       int64_t kv_heads, double q_eps, double k_eps) {
    const int dtype = dtype_of(q);
    TORCH_CHECK(q.dim() == 3 && k.dim() == 3 && v.dim() == 3 && heads > 0 && kv_heads > 0 && q.size(2) % heads == 0,
                "q, k and v must be [batch, tokens, heads * head_dim]");
    const int64_t b = q.size(0), s = q.size(1), hd = q.size(2) / heads;
    TORCH_CHECK(k.sizes() == v.sizes() && k.size(0) == b && k.size(1) == s && k.size(2) == kv_heads * hd, "k and v do not go with q");
    TORCH_CHECK(q_weight.dim() == 1 && q_weight.size(0) == hd && k_weight.dim() == 1 && k_weight.size(0) == hd,
                "norm weights must be [head_dim]");
    for (const at::Tensor* t : {&k, &v, &q_weight, &k_weight})
        TORCH_CHECK(t->scalar_type() == q.scalar_type(), "one dtype expected");
    TORCH_CHECK(cos_sin.scalar_type() == at::kFloat && cos_sin.is_contiguous() && cos_sin.numel() > 0 && cos_sin.numel() % hd == 0,
                "cos_sin must be a dense float32 table of head_dim columns");
    TORCH_CHECK(positions.scalar_type() == at::kLong && positions.dim() == 2 && positions.size(1) == s &&
                    (positions.size(0) == 1 || positions.size(0) == b),
                "positions must be int64 [1 or batch, tokens]");
    check_device(q, {&k, &v, &q_weight, &k_weight, &cos_sin, &positions});
    const DeviceGuard guard(q.device());
    Three out = qkv_outputs(q, heads, kv_heads);
    if (b * s == 0) return out;
    const at::Tensor qd = dense16(q), kd = dense16(k), vd = dense16(v), qw = dense16(q_weight), kw = dense16(k_weight),
                     table = dense16(cos_sin), pos = positions.contiguous();
    check_status(nq_qkv_norm_rope(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), qw.data_ptr(), kw.data_ptr(),
                                  table.data_ptr<float>(), pos.data_ptr<int64_t>(), pos.size(0) > 1, std::get<0>(out).data_ptr(),
                                  std::get<1>(out).data_ptr(), std::get<2>(out).data_ptr(), b, s, heads, kv_heads, hd,
                                  table.numel() / hd, (float)q_eps, (float)k_eps, dtype, current_stream(q.device().index())),
                 "nq_qkv_norm_rope");
    return out;
}
Three qkv_norm_rope_meta(const at::Tensor& q, const at::Tensor&, const at::Tensor&, const at::Tensor&, const at::Tensor&,
                         const at::Tensor&, const at::Tensor&, int64_t heads, int64_t kv_heads, double, double) {
    return qkv_outputs(q, heads, kv_heads);
}

// libnq_hybrid.so lies beside this library and is opened by the first call that needs it: a process that only runs linears
// does not register its kernels, and launches half a microsecond faster (a 16-row linear, host time, 6.9 -> 6.3 us).
struct HybridEntries {
    decltype(&nqh_causal_attention) causal_attention = nullptr;
    decltype(&nqh_last_error) last_error = nullptr;
    HybridEntries() {
        if (void* lib = dlopen("libnq_hybrid.so", RTLD_NOW | RTLD_LOCAL)) {
            causal_attention = reinterpret_cast<decltype(causal_attention)>(dlsym(lib, "nqh_causal_attention"));
            last_error = reinterpret_cast<decltype(last_error)>(dlsym(lib, "nqh_last_error"));
        }
    }
};

at::Tensor causal_attention_op(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, double scale) {
    TORCH_CHECK(q.scalar_type() == at::kBFloat16 && k.scalar_type() == at::kBFloat16 && v.scalar_type() == at::kBFloat16,
                "bfloat16 expected");
    TORCH_CHECK(q.dim() == 4 && k.dim() == 4 && k.sizes() == v.sizes() && k.size(0) == q.size(0) && k.size(2) == q.size(1) &&
                    k.size(3) == q.size(3) && k.size(1) > 0 && q.size(2) % k.size(1) == 0,
                "q must be [batch, tokens, heads, dim], k and v [batch, kv_heads, tokens, dim]");
    check_device(q, {&k, &v});
    const DeviceGuard guard(q.device());
    at::Tensor out = at::empty({q.size(0), q.size(1), q.size(2) * q.size(3)}, q.options());
    if (out.numel() == 0) return out;
    static const HybridEntries hybrid;
    TORCH_CHECK(hybrid.causal_attention && hybrid.last_error, "libnq_hybrid.so cannot be loaded");
    const at::Tensor qd = dense16(q), kd = dense16(k), vd = dense16(v);
    const int status = hybrid.causal_attention(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), out.data_ptr(), q.size(0), q.size(1),
                                            q.size(2), k.size(1), q.size(3), (float)scale, NQH_BF16,
                                            current_stream(q.device().index()));
    TORCH_CHECK(status == NQH_OK, "libnq_hybrid: nqh_causal_attention failed (status ", status, "): ", hybrid.last_error());
    return out;
}
at::Tensor causal_attention_meta(const at::Tensor& q, const at::Tensor&, const at::Tensor&, double) {
    return at::empty({q.size(0), q.size(1), q.size(2) * q.size(3)}, q.options());
}

}  // namespace

TORCH_LIBRARY(nanoquantization_amd, m) {
    m.def("awq_dequantize(Tensor qweight, Tensor qscales, Tensor qzeros) -> Tensor");
    m.def("awq_linear(Tensor x, Tensor qweight, Tensor qscales, Tensor qzeros, Tensor? bias=None) -> Tensor");
    m.def("awq_linear_swiglu(Tensor x, Tensor qweight, Tensor qscales, Tensor qzeros) -> Tensor");
    m.def("awq_swiglu_pair(Tensor x, Tensor gate_qweight, Tensor gate_qscales, Tensor gate_qzeros, Tensor up_qweight, "
          "Tensor up_qscales, Tensor up_qzeros) -> Tensor");
    m.def("awq_linear_add(Tensor x, Tensor qweight, Tensor qscales, Tensor qzeros, Tensor residual) -> Tensor");
    m.def("awq_linear_three(Tensor x, Tensor qweight0, Tensor qscales0, Tensor qzeros0, Tensor qweight1, Tensor qscales1, Tensor "
          "qzeros1, Tensor qweight2, Tensor qscales2, Tensor qzeros2) -> (Tensor, Tensor, Tensor)");
    m.def("rms_norm(Tensor x, Tensor weight, float eps) -> Tensor");
    m.def("silu_mul(Tensor gate, Tensor up) -> Tensor");
    m.def("qkv_norm_rope(Tensor q, Tensor k, Tensor v, Tensor q_weight, Tensor k_weight, Tensor cos_sin, Tensor positions, "
          "int heads, int kv_heads, float q_eps, float k_eps) -> (Tensor, Tensor, Tensor)");
    m.def("causal_attention(Tensor q, Tensor k, Tensor v, float scale) -> Tensor");
}

TORCH_LIBRARY_IMPL(nanoquantization_amd, CUDA, m) {   // the dispatch key of HIP tensors in PyTorch-ROCm
    m.impl("awq_dequantize", &awq_dequantize_op);
    m.impl("awq_linear", &awq_linear_op);
    m.impl("awq_linear_swiglu", &awq_linear_swiglu_op);
    m.impl("awq_swiglu_pair", &awq_swiglu_pair_op);
    m.impl("awq_linear_three", &awq_linear_three_op);
    m.impl("awq_linear_add", &awq_linear_add_op);
    m.impl("rms_norm", &rms_norm_op);
    m.impl("silu_mul", &silu_mul_op);
    m.impl("qkv_norm_rope", &qkv_norm_rope_op);
    m.impl("causal_attention", &causal_attention_op);
}

TORCH_LIBRARY_IMPL(nanoquantization_amd, Meta, m) {
    m.impl("awq_dequantize", &awq_dequantize_meta);
    m.impl("awq_linear", &awq_linear_meta);
    m.impl("awq_linear_swiglu", &awq_linear_swiglu_meta);
    m.impl("awq_swiglu_pair", &awq_swiglu_pair_meta);
    m.impl("awq_linear_three", &awq_linear_three_meta);
    m.impl("awq_linear_add", &awq_linear_add_meta);
    m.impl("rms_norm", &rms_norm_meta);
    m.impl("silu_mul", &silu_mul_meta);
    m.impl("qkv_norm_rope", &qkv_norm_rope_meta);
    m.impl("causal_attention", &causal_attention_meta);
}
