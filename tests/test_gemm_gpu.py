"""Kernel (c): fused dequant + MFMA GEMM through the C ABI against the fp32-accumulation oracle."""
import ctypes

import numpy as np
import pytest
import torch

import nanoquantization_amd as nq
from nanoquantization_amd import _lib
from nanoquantization_amd.layers.gemm import awq_gemm_variant
from conftest import make_case, make_x, random_packed, to_bits, to_dev
from oracle import awq_oracle as o

pytestmark = pytest.mark.gpu

TOL = 1e-2
# with a bias the reference rounds twice (the product, then out.add_(bias), layers/gemm.py:561-566): one more half ulp
BIAS_STEP = {"f16": 2.0 ** -11, "bf16": 2.0 ** -8}
TIGHT = {"f16": 1.5e-3, "bf16": 6e-3}


def _check(y, xb, p, dtype, bias=None):
    ref = o.linear_fp32(xb, p["qweight"], p["qzeros"], p["qscales"], dtype, bias)
    err = o.max_rel_err(o.from_bits16(to_bits(y), dtype), ref)
    assert err <= TOL, f"max rel err {err}"
    assert err <= TIGHT[dtype] + BIAS_STEP[dtype] * (bias is not None), f"max rel err {err}"
    return err


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_gemm_every_variant_and_split(dtype):
    L = _lib.lib()
    K, N = 512, 520            # N not a multiple of any tile: exercises the column masks
    p = random_packed(K, N, 128, dtype, seed=60)
    dev = [to_dev(p["qweight"]), to_dev(p["qscales"], dtype), to_dev(p["qzeros"])]
    for M in (17, 128, 300):
        xb = make_x(M, K, dtype, seed=61 + M)
        xd = to_dev(xb, dtype)
        for v in range(L.awq_gemm_variant_count()):
            for split in (1, 3):
                print(f"gemm variant {L.awq_gemm_variant_name(v).decode()} split={split} M={M} {dtype}", flush=True)
                y = awq_gemm_variant(xd, *dev, v, split)
                torch.cuda.synchronize()
                _check(y, xb, p, dtype)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("M,K,N,g", [(32, 1024, 3072, 128), (64, 3072, 1024, 128), (256, 1024, 2048, 32),
                                      (512, 4096, 1024, 128), (130, 256, 8, 64), (1000, 2048, 264, 128)])
def test_gemm_default_dispatch(dtype, M, K, N, g):
    print(f"gemm default {dtype} M={M} K={K} N={N} g={g}", flush=True)
    p = make_case(K, N, g, dtype, seed=M + K)
    xb = make_x(M, K, dtype, seed=M)
    y = nq.awq_gemm(to_dev(xb, dtype), to_dev(p["qweight"]), to_dev(p["qscales"], dtype), to_dev(p["qzeros"]), 8)
    torch.cuda.synchronize()
    assert tuple(y.shape) == (M, N)
    _check(y, xb, p, dtype)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_gemm_equals_dequant_then_matmul(dtype):
    # the reference's M >= 256 branch: awq_dequantize + torch.matmul (layers/gemm.py:559-561); the fused
    # kernel multiplies the very same rounded weights, so it must agree with that path to fp32-sum accuracy
    print(f"gemm vs dequant+matmul {dtype}", flush=True)
    M, K, N = 384, 1024, 1024
    p = make_case(K, N, 128, dtype, seed=70)
    xb = make_x(M, K, dtype, seed=71)
    qw, qs, qz = to_dev(p["qweight"]), to_dev(p["qscales"], dtype), to_dev(p["qzeros"])
    xd = to_dev(xb, dtype)
    w = nq.awq_dequantize(qw, qs, qz)
    y_unfused = torch.matmul(xd.float(), w.float())
    y = nq.awq_gemm(xd, qw, qs, qz, 8)
    err = (y.float() - y_unfused).abs().max().item() / y_unfused.abs().max().item()
    assert err <= (1e-3 if dtype == "f16" else 5e-3), err


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_gemm_bias_and_determinism(dtype):
    print(f"gemm bias {dtype}", flush=True)
    M, K, N = 200, 1024, 512
    p = make_case(K, N, 128, dtype, seed=80)
    dev = [to_dev(p["qweight"]), to_dev(p["qscales"], dtype), to_dev(p["qzeros"])]
    xb = make_x(M, K, dtype, seed=81)
    xd = to_dev(xb, dtype)
    bias = np.linspace(-2, 2, N).astype(np.float32)
    v = 0   # the 128 x 128 tile
    for split in (1, 4):
        y = awq_gemm_variant(xd, *dev, v, split, bias=to_dev(o.to_bits16(bias, dtype), dtype))
        _check(y, xb, p, dtype, o.to_dtype_f32(bias, dtype))
    y1 = awq_gemm_variant(xd, *dev, v, 4)
    y2 = awq_gemm_variant(xd, *dev, v, 4)
    assert torch.equal(y1, y2)
    assert torch.count_nonzero(awq_gemm_variant(torch.zeros_like(xd), *dev, v, 4)) == 0


@pytest.mark.parametrize("form", ["p", "r"])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_gemm_tail_tiles_split(dtype, form):
    # 9 x 30 = 270 tiles of 256 x 256 (ragged in M and N): 256 whole tiles and a tail of 14 whose K range is cut;
    # the mixed launch must agree with the oracle, with the uncut launch bit for bit where no cut applies,
    # and be bit-stable -- for the pipelined kernel (p) and the one that builds its B operands in registers (r)
    L = _lib.lib()
    names = [L.awq_gemm_variant_name(i).decode() for i in range(L.awq_gemm_variant_count())]
    tail, whole = names.index(f"256x256{form}t"), names.index(f"256x256{form}")
    # (the register-operand kernel takes widths that are multiples of 128; other widths run the pipelined one under
    # its name: its case has the last tile half empty instead of ragged)
    M, K, N = 2300, 256, (7672 if form == "p" else 7552)
    p = random_packed(K, N, 128, dtype, seed=95)
    dev = [to_dev(p["qweight"]), to_dev(p["qscales"], dtype), to_dev(p["qzeros"])]
    xb = make_x(M, K, dtype, seed=96)
    xd = to_dev(xb, dtype)
    bias = np.linspace(-1, 1, N).astype(np.float32)
    bd = to_dev(o.to_bits16(bias, dtype), dtype)
    y1 = awq_gemm_variant(xd, *dev, whole, 1, bias=bd)
    _check(y1, xb, p, dtype, o.to_dtype_f32(bias, dtype))
    for split in (2, 4):
        print(f"gemm tail {form} split={split} {dtype}", flush=True)
        y = awq_gemm_variant(xd, *dev, tail, split, bias=bd)
        torch.cuda.synchronize()
        _check(y, xb, p, dtype, o.to_dtype_f32(bias, dtype))
        assert torch.equal(y, awq_gemm_variant(xd, *dev, tail, split, bias=bd))
        # tiles 0..255 in n-fastest order: tile rows 0..7 entirely (8 x 30 = 240) and 16 tiles of row 8
        assert torch.equal(y[:2048], y1[:2048])
        assert torch.equal(y[2048:, :16 * 256], y1[2048:, :16 * 256])


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("K,N,g", [(1024, 1032, 128), (256, 8, 64), (512, 264, 32), (128, 4096, 128), (1024, 520, 1024)])
def test_dequantize_transposed_bit_exact(dtype, K, N, g):
    # out [N, K] must be awq_dequantize's [K, N] transposed, bit for bit (and so the oracle's RN((q - z) * s))
    print(f"dequantize transposed {dtype} K={K} N={N} g={g}", flush=True)
    p = random_packed(K, N, g, dtype, seed=K + N + g)
    dev = [to_dev(p["qweight"]), to_dev(p["qscales"], dtype), to_dev(p["qzeros"])]
    wt = nq.awq_dequantize_transposed(*dev)
    assert tuple(wt.shape) == (N, K)
    assert torch.equal(wt, nq.awq_dequantize(*dev).t())
    ref_bits = o.dequant(p["qweight"], p["qzeros"], p["qscales"], dtype)
    assert np.array_equal(to_bits(wt).T, ref_bits)


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("M,K,N,g", [(1024, 1024, 1032, 128), (1500, 512, 2048, 64), (2048, 256, 264, 32)])
def test_linear_large_m_equals_dequantise_then_matmul(dtype, M, K, N, g):
    # 1024 rows and more, the regime of the reference's awq_dequantize + torch.matmul (layers/gemm.py:558-561): the
    # default dispatch (fused kernel) against the fp32 oracle, with and without bias, against the forced whole-tile
    # variant, and against that two-step structure built from awq_dequantize_transposed + a dense matmul
    from nanoquantization_amd.layers.gemm import _linear
    print(f"large-M linear {dtype} M={M} K={K} N={N} g={g}", flush=True)
    p = make_case(K, N, g, dtype, seed=M + N)
    xb = make_x(M, K, dtype, seed=M)
    dev = [to_dev(p["qweight"]), to_dev(p["qscales"], dtype), to_dev(p["qzeros"])]
    xd = to_dev(xb, dtype)
    y = nq.awq_gemm(xd, *dev, 8)
    _check(y, xb, p, dtype)
    bias = np.linspace(-1, 1, N).astype(np.float32)
    yb = _linear("awq_linear", xd, *dev, to_dev(o.to_bits16(bias, dtype), dtype))
    _check(yb, xb, p, dtype, o.to_dtype_f32(bias, dtype))
    L = _lib.lib()
    names = [L.awq_gemm_variant_name(i).decode() for i in range(L.awq_gemm_variant_count())]
    fused = awq_gemm_variant(xd, *dev, names.index("256x256p"), 1)
    fused_r = awq_gemm_variant(xd, *dev, names.index("256x256r"), 1)
    two_step = torch.matmul(xd, nq.awq_dequantize_transposed(*dev).t())
    for other in (fused, fused_r, two_step):
        err = (y.float() - other.float()).abs().max().item() / other.float().abs().max().item()
        assert err <= (2e-3 if dtype == "f16" else 1.6e-2), err     # both round an fp32 sum of the same products once


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("M,K,N,g,split", [(300, 1024, 520, 128, 1), (777, 2048, 1032, 64, 3), (256, 64, 256, 64, 1),
                                            (1000, 768, 2048, 768, 2), (513, 512, 264, 32, 1)])
def test_gemm_register_b_kernel_equals_pipelined(dtype, M, K, N, g, split):
    # the two 256 x 256 kernels multiply the same rounded weights (on MFMAs of different depth, so the fp32 sums may
    # differ in their last bits): ragged M and N, K of one step, odd K slices, every group size (g = 32 runs the
    # pipelined kernel under the r names, bit for bit), with bias
    print(f"gemm r vs p {dtype} M={M} K={K} N={N} g={g} split={split}", flush=True)
    L = _lib.lib()
    names = [L.awq_gemm_variant_name(i).decode() for i in range(L.awq_gemm_variant_count())]
    p = random_packed(K, N, g, dtype, seed=K + N + g)
    dev = [to_dev(p["qweight"]), to_dev(p["qscales"], dtype), to_dev(p["qzeros"])]
    xb = make_x(M, K, dtype, seed=M)
    xd = to_dev(xb, dtype)
    bias = np.linspace(-1, 1, N).astype(np.float32)
    bd = to_dev(o.to_bits16(bias, dtype), dtype)
    for form in ("", "t"):
        yp = awq_gemm_variant(xd, *dev, names.index("256x256p" + form), split, bias=bd)
        yr = awq_gemm_variant(xd, *dev, names.index("256x256r" + form), split, bias=bd)
        torch.cuda.synchronize()
        if g % 64 != 0:
            assert torch.equal(yp, yr), form
        diff = (yp.float() - yr.float()).abs().max().item() / yp.float().abs().max().item()
        assert diff <= (1e-3 if dtype == "f16" else 8e-3), (form, diff)
        _check(yr, xb, p, dtype, o.to_dtype_f32(bias, dtype))


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("M,K,N", [(4096, 512, 4352), (4096, 1024, 4096), (2048, 1024, 4096), (4096, 4096, 4096),
                                   (1024, 1024, 4096)])
def test_gemm_default_kernel_by_work_items(dtype, M, K, N):
    # awq_gemm runs the register-operand kernel (r) where the plan's work items -- whole tiles plus the
    # K slices of the tail tiles -- outnumber the 256 CUs (16 x 17 = 272 tiles); at exactly 256 items (16 x 16 tiles, or
    # 8 x 16 cut in two) in fp16, and in bf16 if an item has 64 K steps at least; the pipelined kernel (p) otherwise
    # (4 x 16 tiles cut in two).  awq_gemm_plan names that kernel, and forcing the planned pair gives the same bits.
    import ctypes
    from nanoquantization_amd.layers import gemm as gemm_layer
    L = _lib.lib()
    names = [L.awq_gemm_variant_name(i).decode() for i in range(L.awq_gemm_variant_count())]
    v, sp = ctypes.c_int(), ctypes.c_int()
    dt = _lib.AWQ_F16 if dtype == "f16" else _lib.AWQ_BF16
    assert L.awq_gemm_plan(M, N, K, 128, dt, ctypes.byref(v), ctypes.byref(sp)) == 0
    name = names[v.value]
    tiles = (M // 256) * (N // 256)
    tail = tiles % 256 if name.endswith("t") else (tiles if sp.value > 1 else 0)
    items = tiles - tail + tail * sp.value
    print(f"gemm default {dtype} M={M} K={K} N={N}: plan {name} split {sp.value}, {items} items", flush=True)
    steps = K // 64 // (sp.value if tail == tiles else 1)
    use_r = items > 256 or (items == 256 and (dtype == "f16" or steps >= 64))
    assert name in (("256x256r", "256x256rt") if use_r else ("256x256p", "256x256pt")), (name, items, steps)
    p = random_packed(K, N, 128, dtype, seed=123)
    dev = [to_dev(p["qweight"]), to_dev(p["qscales"], dtype), to_dev(p["qzeros"])]
    xd = to_dev(make_x(M, K, dtype, seed=124), dtype)
    # (the entry itself: the default linear takes other ways on some of these sizes, 1024 x 4096 at 1024 rows 31 -> 18 us)
    y = gemm_layer._linear("awq_gemm", xd, *dev, None)
    assert torch.equal(y, awq_gemm_variant(xd, *dev, v.value, sp.value)), name
    rows = torch.arange(0, M, 97, device="cuda")
    ref = xd[rows].float() @ nq.awq_dequantize(*dev).float()
    assert ((y[rows].float() - ref).abs().max() / ref.abs().max()).item() <= TIGHT[dtype]


def test_gemm_prefill_full_size_bf16():
    # Qwen3-8B MLP gate/up at M=512, its real size (oracle: numpy float64 matmul, a few seconds)
    print("gemm full size M=512 4096x12288 bf16", flush=True)
    M, K, N = 512, 4096, 12288
    p = random_packed(K, N, 128, "bf16", seed=90)
    xb = make_x(M, K, "bf16", seed=91)
    y = nq.awq_gemm(to_dev(xb, "bf16"), to_dev(p["qweight"]), to_dev(p["qscales"], "bf16"), to_dev(p["qzeros"]), 8)
    _check(y, xb, p, "bf16")


@pytest.mark.parametrize("M,K,N", [(8192, 4096, 12288), (8192, 12288, 4096), (2048, 4096, 12288), (2048, 12288, 4096),
                                   (512, 12288, 4096), (4096, 8192, 5120), (300, 5120, 25600)])
def test_gemm_largest_shapes_properties(M, K, N):
    """The prefill shapes at their real sizes (Qwen3-8B MLP at M = 512 / 2048 / 8192, Qwen3-32B o_proj at a 4096-token
    prefill and gate/up at a ragged M), too big for the CPU oracle: checked through size-independent properties, on
    the default dispatch and on both 256 x 256 fused kernels (the pipelined one, p, and the one that builds its B
    operands in registers, r) forced in both of their forms (every tile whole; the tiles of the last round cut along K
    with the plan's split).  (1) rows sampled across every workgroup tile equal the
    fp32 matmul of those rows with the dequantised weight (itself bit-exact against the oracle); (2) the same rows
    pushed through alone (another tile shape) agree too; (3) run-to-run bit-stable; (4) a zero row gives exact zeros."""
    print(f"gemm properties M={M} K={K} N={N} bf16", flush=True)
    L = _lib.lib()
    names = [L.awq_gemm_variant_name(i).decode() for i in range(L.awq_gemm_variant_count())]
    import ctypes
    v, sp = ctypes.c_int(), ctypes.c_int()
    assert L.awq_gemm_plan(M, N, K, 128, _lib.AWQ_BF16, ctypes.byref(v), ctypes.byref(sp)) == 0
    g = torch.Generator(device="cuda").manual_seed(M + K)
    qw = torch.randint(-2 ** 31, 2 ** 31 - 1, (K, N // 8), dtype=torch.int32, device="cuda", generator=g)
    qz = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 128, N // 8), dtype=torch.int32, device="cuda", generator=g)
    sc = (torch.rand(K // 128, N, device="cuda", generator=g) * 0.01 + 0.002).to(torch.bfloat16)
    x = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
    x[5] = 0
    rows = torch.arange(3, M, max(1, M // 61), device="cuda")[:64]          # one or two rows of every 256-row tile
    w = nq.awq_dequantize(qw, sc, qz).float()
    ref = x[rows].float() @ w
    runs = [("default " + names[v.value] + f" split {sp.value}", lambda: nq.awq_gemm(x, qw, sc, qz, 8)),
            ("256x256p split 1", lambda: awq_gemm_variant(x, qw, sc, qz, names.index("256x256p"), 1)),
            (f"256x256pt split {max(sp.value, 2)}",
             lambda: awq_gemm_variant(x, qw, sc, qz, names.index("256x256pt"), max(sp.value, 2))),
            ("256x256r split 1", lambda: awq_gemm_variant(x, qw, sc, qz, names.index("256x256r"), 1)),
            (f"256x256rt split {max(sp.value, 2)}",
             lambda: awq_gemm_variant(x, qw, sc, qz, names.index("256x256rt"), max(sp.value, 2)))]
    for what, run in runs:
        print(f"  {what}", flush=True)
        y = run()
        torch.cuda.synchronize()
        assert torch.equal(y, run()), what
        assert torch.count_nonzero(y[5]) == 0, what
        err = ((y[rows].float() - ref).abs().max() / ref.abs().max()).item()
        assert err <= TIGHT["bf16"], (what, err)
        del y
    sub = nq.awq_gemm(x[rows].contiguous(), qw, sc, qz, 8).float()          # another kernel / tile shape
    assert ((sub - ref).abs().max() / ref.abs().max()).item() <= TIGHT["bf16"]


# one and several tiles of 256 and of 128 rows, rows and columns past the last tile, one, two and three stages of K (the
# buffers in flight at the start), every group size form, a weight of two slabs (131072 x 1032: 270 MB)
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("M,K,N,g", [(1, 64, 8, 64), (129, 128, 264, 32), (300, 192, 520, 64), (256, 256, 256, 128),
                                      (4352, 320, 4104, 64), (8200, 320, 4104, 64), (700, 1024, 1032, 1024), (40, 131072, 1032, 128)])
def test_linear_dense(dtype, M, K, N, g):
    """The weight dequantised first, with bias and with the gated epilogue, against the fp64 product of the dequantised
    weight and against the separate activation kernel; rows of zeros stay zero, two runs give the same bits."""
    from nanoquantization_amd.engine import ops
    print(f"linear dense {dtype} M={M} K={K} N={N} g={g}", flush=True)
    tdt = torch.float16 if dtype == "f16" else torch.bfloat16
    gen = torch.Generator(device="cuda").manual_seed(M + N)
    qw = torch.randint(-2 ** 31, 2 ** 31 - 1, (K, N // 8), dtype=torch.int32, device="cuda", generator=gen)
    qz = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // g, N // 8), dtype=torch.int32, device="cuda", generator=gen)
    qs = (torch.rand(K // g, N, device="cuda", generator=gen) * 0.02 + 0.001).to(tdt)
    x = torch.randn(M, K, device="cuda", generator=gen).to(tdt)
    bias = torch.randn(N, device="cuda", generator=gen).to(tdt)
    if M > 1:
        x[M // 2] = 0
    L = _lib.lib()
    scratch = torch.full((L.awq_linear_dense_scratch_bytes(M, N, K, g),), 0xFF, dtype=torch.uint8, device="cuda")   # NaN

    def dense(b, gated):
        y = torch.empty(M, N // 2 if gated else N, dtype=tdt, device="cuda")
        _lib.check(L.awq_linear_dense(x.data_ptr(), qw.data_ptr(), qs.data_ptr(), qz.data_ptr(),
                                      None if b is None else b.data_ptr(), y.data_ptr(), M, N, K, g, _lib.dtype_id(tdt),
                                      int(gated), scratch.data_ptr(), scratch.numel(), _lib.current_stream_ptr(y.device)))
        return y
    y, yb = dense(None, False), dense(bias, False)
    ref = x.double() @ nq.awq_dequantize(qw, qs, qz).double()
    top = ref.abs().max().item()
    assert (y.double() - ref).abs().max().item() <= TIGHT[dtype] * top
    assert (yb.double() - ref - bias.double()).abs().max().item() <= (TIGHT[dtype] + BIAS_STEP[dtype]) * (top + 4)
    assert torch.equal(y, dense(None, False))
    assert M == 1 or torch.count_nonzero(y[M // 2]) == 0
    if N % 16 == 0:
        assert torch.equal(dense(None, True), ops.silu_mul(y, interleaved=True))
    # with a residual, in a tensor of its own and in place: the bits of an addition behind the product, and nothing behind the rows
    r = torch.randn(M + 1, N, device="cuda", generator=gen).to(tdt)
    for out in (torch.full_like(r, 3.0), r.clone()):
        last, res = out[M].clone(), out if torch.equal(out, r) else r
        _lib.check(L.awq_linear_dense_add(x.data_ptr(), qw.data_ptr(), qs.data_ptr(), qz.data_ptr(), res.data_ptr(), out.data_ptr(), M, N, K, g,
                                          _lib.dtype_id(tdt), scratch.data_ptr(), scratch.numel(), _lib.current_stream_ptr(y.device)))
        assert torch.equal(out[:M], r[:M] + y) and torch.equal(out[M], last)


def test_linear_dense_routes():
    """The default linear takes the dense path where its estimate is the lower one, with the bits of the forced call, also
    under graph capture; the fused kernels keep short prompts, few rows of a short K and what the path refuses."""
    L = _lib.lib()
    wanted = L.awq_linear_dense_wanted_bytes
    assert wanted(8192, 12288, 4096, 128) == 2 * 12288 * 4096 and wanted(2048, 4096, 12288, 128) > 0
    assert wanted(128, 12288, 4096, 128) == 0 and wanted(512, 4096, 12288, 128) == 0
    assert wanted(2048, 4096, 1024, 128) > 0 and wanted(200, 25600, 512, 128) == 0      # 31 us, fused 41; 25, fused 20
    assert wanted(8192, 4096, 4096 + 32, 32) == 0
    assert wanted(8192, 51200, 5120, 128) <= 256 << 20
    M, K, N = 2100, 2048, 2056
    p = random_packed(K, N, 128, "bf16", seed=7)
    dev = [to_dev(p["qweight"]), to_dev(p["qscales"], "bf16"), to_dev(p["qzeros"])]
    assert wanted(M, N, K, 128) > 0
    xb = make_x(M, K, "bf16", seed=8)
    x = to_dev(xb, "bf16")
    want = torch.empty(M, N, dtype=torch.bfloat16, device="cuda")
    scratch = torch.empty(L.awq_linear_dense_scratch_bytes(M, N, K, 128), dtype=torch.uint8, device="cuda")
    _lib.check(L.awq_linear_dense(x.data_ptr(), *(t.data_ptr() for t in dev), None, want.data_ptr(), M, N, K, 128, _lib.AWQ_BF16, 0,
                                  scratch.data_ptr(), scratch.numel(), _lib.current_stream_ptr(want.device)))
    _check(want, xb, p, "bf16")
    assert L.awq_linear_route(M, N, K, 128, _lib.AWQ_BF16, 0, None) == b"dense"
    assert torch.equal(nq.awq_gemm(x, *dev, 8), want)
    assert torch.equal(_lib.torch_ops().awq_linear(x, *dev, None), want)
    s, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        assert torch.equal(nq.awq_gemm(x, *dev, 8), want)
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=s):
            y = nq.awq_gemm(x, *dev, 8)
    torch.cuda.synchronize()
    for rep in range(3):
        y.zero_()
        graph.replay()
        other = nq.awq_gemm(x * 2, *dev, 8)         # eager work with scratch of its own between the replays
        torch.cuda.synchronize()
        assert torch.equal(y, want) and torch.equal(other, nq.awq_gemm(x * 2, *dev, 8)), rep


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("M,K,N,g", [(48, 288, 512, 32), (200, 224, 384, 32), (65, 544, 1280, 32), (32, 32, 256, 32)])
def test_linear_k_not_a_multiple_of_64(dtype, M, K, N, g):
    """K = 32 * odd (the reference admits any multiple of its 32-row K block) above 16 rows: awq_linear serves it
    with the GEMV, 16 rows at a time."""
    from nanoquantization_amd.layers import gemm as gemm_layer
    print(f"linear K%64!=0 M={M} K={K} N={N} g={g} {dtype}", flush=True)
    p = make_case(K, N, g, dtype, seed=M + K)
    xb = make_x(M, K, dtype, seed=M)
    bias = np.random.default_rng(M).standard_normal(N).astype(np.float32)
    bias_bits = o.to_bits16(bias, dtype)
    y = gemm_layer._linear("awq_linear", to_dev(xb, dtype), to_dev(p["qweight"]), to_dev(p["qscales"], dtype),
                           to_dev(p["qzeros"]), to_dev(bias_bits, dtype))
    _check(y, xb, p, dtype, o.from_bits16(bias_bits, dtype))


def test_linear_random_shapes_default_dispatch():
    """Seeded sweep over odd shape combinations (row counts either side of every dispatch boundary, K = group x small
    and large factors, N with and without whole 128-column tiles, three group sizes, optional bias): whatever kernel
    the default dispatch picks must meet the tight error bound and be bit-stable run to run."""
    import random
    from nanoquantization_amd.layers import gemm as gemm_layer
    rnd = random.Random(1234)
    cases = 0
    while cases < 60:
        tdt = rnd.choice([torch.float16, torch.bfloat16])
        g = rnd.choice([128, 128, 128, 64, 32])
        K = g * rnd.choice([1, 2, 3, 4, 5, 7, 8, 9, 12, 16, 17, 24, 31, 32, 40, 48, 64, 100])
        N = 8 * rnd.choice([1, 3, 16, 17, 32, 48, 64, 96, 128, 136, 160, 256, 272, 384, 512, 640, 1000, 1024, 1280])
        M = rnd.choice([1, 2, 3, 4, 5, 7, 8, 15, 16, 17, 24, 31, 32, 33, 48, 63, 64, 65, 100, 128, 129, 200, 256, 300, 1024, 1100])
        if K % 32 or K * N * max(M, 64) > 2e10:
            continue
        cases += 1
        gen = torch.Generator(device="cuda").manual_seed(cases)
        qw = torch.randint(-2 ** 31, 2 ** 31 - 1, (K, N // 8), dtype=torch.int32, device="cuda", generator=gen)
        qz = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // g, N // 8), dtype=torch.int32, device="cuda", generator=gen)
        qs = (torch.rand(K // g, N, device="cuda", generator=gen) * 0.02 + 0.001).to(tdt)
        x = torch.randn(M, K, device="cuda", generator=gen).to(tdt)
        bias = torch.randn(N, device="cuda", generator=gen).to(tdt) if rnd.random() < 0.3 else None
        print(f"random linear {cases}: M={M} K={K} N={N} g={g} {tdt} bias={bias is not None}", flush=True)
        y = gemm_layer._linear("awq_linear", x, qw, qs, qz, bias)
        ref = x.float() @ nq.awq_dequantize(qw, qs, qz).float()
        if bias is not None:
            ref = ref + bias.float()
        err = ((y.float() - ref).abs().max() / ref.abs().max().clamp_min(1e-6)).item()
        assert err <= (1.5e-3 if tdt == torch.float16 else 6e-3), err
        assert torch.equal(y, gemm_layer._linear("awq_linear", x, qw, qs, qz, bias))


# a row, tiles of five to eight 16-row blocks, one row past a tile; less and more stages of K than the ring holds, also cut in
# three; columns past the last tile; groups of less, as much and more than a stage; from the third line on both sides of the stages
# where four waves hand over to eight (14 and 15 in bf16, 18 and 19 in fp16), and more, odd and even
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("M,K,N,g", [(1, 64, 8, 32), (81, 320, 136, 64), (113, 384, 520, 128), (128, 448, 256, 32), (129, 512, 8, 512),
                                      (270, 192, 264, 192), (333, 1088, 1032, 64),
                                      (1, 1280, 128, 64), (80, 896, 136, 32), (81, 960, 256, 64), (112, 1152, 264, 128), (113, 1216, 392, 64),
                                      (128, 1344, 256, 32), (257, 3712, 136, 64), (66, 4096, 1032, 128), (96, 4160, 120, 64)])
def test_gemm_rows128(dtype, M, K, N, g):
    print(f"gemm rows128 {dtype} M={M} K={K} N={N} g={g}", flush=True)
    L = _lib.lib()
    v = [L.awq_gemm_variant_name(i).decode() for i in range(L.awq_gemm_variant_count())].index("rows128")
    p = random_packed(K, N, g, dtype, seed=M + K)
    dev = [to_dev(p["qweight"]), to_dev(p["qscales"], dtype), to_dev(p["qzeros"])]
    xb = make_x(M, K, dtype, seed=M)
    xd = to_dev(xb, dtype)
    bias = np.linspace(-2, 2, N).astype(np.float32)
    bd = to_dev(o.to_bits16(bias, dtype), dtype)
    for split in (1, 3):
        y = awq_gemm_variant(xd, *dev, v, split)
        torch.cuda.synchronize()
        _check(y, xb, p, dtype)
        assert torch.equal(y, awq_gemm_variant(xd, *dev, v, split))
        _check(awq_gemm_variant(xd, *dev, v, split, bias=bd), xb, p, dtype, o.to_dtype_f32(bias, dtype))
    # the unpacked weight is awq_dequantize's, bit for bit: rows of the identity
    n = min(M, K)
    eye = torch.eye(n, K, device="cuda", dtype=xd.dtype)
    assert torch.equal(awq_gemm_variant(eye, *dev, v, 1), nq.awq_dequantize(*dev)[:n])


# the tiles of which two share a CU, at the first and last row of each; fewer stages than the ring holds, odd and even counts,
# the last K split one stage long; widths of one tile, a word more, a word less than two, not a multiple of four words
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("M,K,N,g,split", [(17, 64, 128, 32, 1), (32, 1344, 136, 64, 4), (33, 1088, 248, 32, 3), (48, 576, 1032, 576, 1),
                                           (49, 640, 264, 128, 5), (64, 2112, 1240, 64, 2), (65, 1152, 520, 1152, 1), (80, 704, 264, 64, 3)])
def test_gemm_rows128_few_rows(dtype, M, K, N, g, split):
    print(f"gemm rows128 few rows {dtype} M={M} K={K} N={N} g={g} split={split}", flush=True)
    L = _lib.lib()
    v = [L.awq_gemm_variant_name(i).decode() for i in range(L.awq_gemm_variant_count())].index("rows128")
    p = random_packed(K, N, g, dtype, seed=M + K)
    dev = [to_dev(p["qweight"]), to_dev(p["qscales"], dtype), to_dev(p["qzeros"])]
    xb = make_x(M, K, dtype, seed=M)
    xd = to_dev(xb, dtype)
    bias = np.linspace(-2, 2, N).astype(np.float32)
    y = awq_gemm_variant(xd, *dev, v, split)
    _check(y, xb, p, dtype)
    assert torch.equal(y, awq_gemm_variant(xd, *dev, v, split))
    _check(awq_gemm_variant(xd, *dev, v, split, bias=to_dev(o.to_bits16(bias, dtype), dtype)), xb, p, dtype, o.to_dtype_f32(bias, dtype))
    eye = torch.eye(min(M, K), K, device="cuda", dtype=xd.dtype)
    assert torch.equal(awq_gemm_variant(eye, *dev, v, 1), nq.awq_dequantize(*dev)[:min(M, K)])
    # the default linear of these rows: the GEMV where it takes the sizes, else these tiles with their own split
    chosen = ctypes.c_int()
    name = L.awq_linear_route(M, N, K, g, _lib.dtype_id(xd.dtype), 0, ctypes.byref(chosen))
    assert name == b"rows128" or (name == b"gemv" and g % 128 == 0)
    if name != b"gemv":
        assert torch.equal(nq.awq_gemm(xd, *dev, 8), awq_gemm_variant(xd, *dev, v, chosen.value))


# scales up to the largest for which 15 times one is a number; the quick way to a weight leaves the range of a float from 2^113 on
@pytest.mark.parametrize("M,K,N,g,split", [(40, 704, 264, 32, 1), (128, 1088, 128, 64, 3), (200, 576, 392, 64, 1)])
def test_gemm_rows128_large_scales(M, K, N, g, split):
    print(f"gemm rows128 large scales M={M} K={K} N={N} g={g} split={split}", flush=True)
    L = _lib.lib()
    v = [L.awq_gemm_variant_name(i).decode() for i in range(L.awq_gemm_variant_count())].index("rows128")
    gen = torch.Generator(device="cuda").manual_seed(M)
    words = lambda r: torch.randint(-2 ** 31, 2 ** 31 - 1, (r, N // 8), dtype=torch.int32, device="cuda", generator=gen)
    qw, qz = words(K), words(K // g)
    # every 37th column in the middle group alone, at 2^112, 2^113, .. 2^123
    qs = (torch.rand(K // g, N, device="cuda", generator=gen) * 0.02 + 0.001).to(torch.bfloat16)
    for i, c in enumerate(range(3, N, 37)):
        qs[K // g // 2, c] = 2.0 ** (112 + i % 12) * (1 + i % 2 / 2)
    w = nq.awq_dequantize(qw, qs, qz)
    assert w.isfinite().all()
    eye = torch.eye(min(M, K), K, device="cuda", dtype=torch.bfloat16)
    eye = torch.roll(eye, K // g // 2 * g, dims=1)           # rows of the group with the large scales
    assert torch.equal(awq_gemm_variant(eye, qw, qs, qz, v, split), torch.roll(w, -(K // g // 2 * g), dims=0)[:min(M, K)])
    x = (torch.randn(M, K, device="cuda", generator=gen) * 2.0 ** -20).to(torch.bfloat16)
    y = awq_gemm_variant(x, qw, qs, qz, v, split)
    ref = x.double() @ w.double()
    bound = TIGHT["bf16"] * ref.abs().amax(dim=0)            # a column at a time
    assert y.isfinite().all() and ((y.double() - ref).abs() <= bound).all()
    # an element of x that is no number concerns its own row
    xn = x.clone()
    xn[0, 5] = float("nan")
    z = awq_gemm_variant(xn, qw, qs, qz, v, split)
    assert z[0].isnan().all() and torch.equal(z[1:], y[1:])
    # a scale that is no number concerns its own column
    qs[0, 1] = float("inf")
    z = awq_gemm_variant(x, qw, qs, qz, v, split)
    other = [c for c in range(N) if c != 1]
    assert not z[:, 1].isfinite().any() and torch.equal(z[:, other], y[:, other])


# tiles of few rows unsplit and in K splits, dequantised first with tiles of 128 and of 256 rows; widths that are no whole tiles, a K
# and rows that the one launch does not take
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("M,K,N,g,way", [(129, 1024, (2048, 1024, 1024), 128, "rows"), (200, 4096, (1024, 256, 128), 64, "rows"), (40, 512, (128, 384, 128), 32, "rows"),
                                         (1700, 2048, (2048, 1024, 1024), 128, "dense"), (4096, 1024, (512, 256, 1280), 64, "dense"),
                                         (300, 512, (256, 136, 128), 64, ""), (300, 96, (256, 128, 128), 32, ""), (100, 1024, (256, 128, 128), 128, ""), (1, 1024, (256, 128, 128), 64, "")])
def test_linear_parts(dtype, M, K, N, g, way):
    """Three weights in one launch: the bits of the same kernel on the weights side by side; else those of three linears."""
    print(f"linear parts {dtype} M={M} K={K} N={N} g={g} {way}", flush=True)
    L, tdt = _lib.lib(), torch.float16 if dtype == "f16" else torch.bfloat16
    gen = torch.Generator(device="cuda").manual_seed(M + K)
    words = lambda r, n: torch.randint(-2 ** 31, 2 ** 31 - 1, (r, n // 8), dtype=torch.int32, device="cuda", generator=gen)
    parts = [(words(K, n), ((torch.rand(K // g, n, device="cuda", generator=gen) + 0.1) * 0.2 / K ** 0.5).to(tdt), words(K // g, n)) for n in N]
    x = torch.randn(M, K, device="cuda", generator=gen).to(tdt)
    ws, scratch = ctypes.c_size_t(), ctypes.c_size_t()
    wanted = L.awq_linear_parts_wanted((ctypes.c_int64 * 3)(*N), 3, M, K, g, _lib.dtype_id(tdt), ctypes.byref(ws), ctypes.byref(scratch))
    assert bool(wanted) == bool(way) and bool(scratch.value) == (way == "dense")
    y = _lib.torch_ops().awq_linear_three(x, *(t for p in parts for t in p))
    assert [tuple(t.shape) for t in y] == [(M, n) for n in N] and all(t.is_contiguous() for t in y)
    if not way:
        for t, p in zip(y, parts):
            assert torch.equal(t, nq.awq_gemm(x, *p, 8))
        return
    side = [torch.cat(t, dim=1).contiguous() for t in zip(*parts)]
    if way == "dense":
        want, room = torch.empty(M, sum(N), dtype=tdt, device="cuda"), torch.empty(scratch.value, dtype=torch.uint8, device="cuda")
        _lib.check(L.awq_linear_dense(x.data_ptr(), *(t.data_ptr() for t in side), None, want.data_ptr(), M, sum(N), K, g, _lib.dtype_id(tdt), 0,
                                      room.data_ptr(), room.numel(), _lib.current_stream_ptr(x.device)))
    else:
        v = [L.awq_gemm_variant_name(i).decode() for i in range(L.awq_gemm_variant_count())].index("rows128")
        split = 1
        while ws.value and L.awq_gemm_ex_workspace_bytes(M, sum(N), K, v, split) != ws.value:
            split += 1
        want = awq_gemm_variant(x, *side, v, split)
    assert torch.equal(torch.cat(y, dim=1), want)
    ref = x.double() @ nq.awq_dequantize(*side).double()
    assert (want.double() - ref).abs().max().item() <= TIGHT[dtype] * ref.abs().max().item()


def test_gemm_rows128_routes():
    """The default linear takes these tiles for a few hundred rows, with the bits of the forced variant; what they refuse, short
    K and the plan of awq_gemm stay with the other kernels."""
    L = _lib.lib()
    names = [L.awq_gemm_variant_name(i).decode() for i in range(L.awq_gemm_variant_count())]
    v = names.index("rows128")
    for M, K, N, g, split in ((333, 2816, 1304, 64, 5), (200, 2048, 2048, 128, 4)):
        p = random_packed(K, N, g, "bf16", seed=9)
        dev = [to_dev(p["qweight"]), to_dev(p["qscales"], "bf16"), to_dev(p["qzeros"])]
        x = to_dev(make_x(M, K, "bf16", seed=10), "bf16")
        y = nq.awq_gemm(x, *dev, 8)
        chosen = ctypes.c_int()
        assert L.awq_linear_route(M, N, K, g, _lib.AWQ_BF16, 0, ctypes.byref(chosen)) == b"rows128"
        assert torch.equal(y, awq_gemm_variant(x, *dev, v, chosen.value)), (M, K, N)
        assert L.awq_linear_workspace_bytes(M, N, K) >= L.awq_gemm_ex_workspace_bytes(M, N, K, v, split)
    # groups of 16 rows end inside a wave's 32: an error, before anything is launched
    args = (x.data_ptr(), dev[0].data_ptr(), dev[1].data_ptr(), dev[2].data_ptr(), None, y.data_ptr())
    assert L.awq_gemm_ex(*args, M, N, K, 16, _lib.AWQ_BF16, None, 0, None, v, 1) != 0
    assert b"group size" in L.awq_hip_last_error()


# unsplit and in two to five K splits, rows past the last tile, columns past the last tile (2 x 1032: 16.1 of them)
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("M,K,inter,g,split", [(200, 2048, 8192, 128, False), (160, 12288, 1024, 128, True), (333, 2816, 1032, 64, True),
                                               (513, 4096, 1024, 128, True)])
def test_swiglu_rows128(dtype, M, K, inter, g, split):
    """The gated epilogue of the 128-row tiles, in the tile and in the sum of the K splits: the bits of the same tiles' product
    and the separate activation."""
    from nanoquantization_amd.engine import ops
    print(f"swiglu rows128 {dtype} M={M} K={K} inter={inter}", flush=True)
    tdt, L, N = torch.float16 if dtype == "f16" else torch.bfloat16, _lib.lib(), 2 * inter
    chosen = ctypes.c_int()
    assert L.awq_linear_route(M, N, K, g, _lib.dtype_id(tdt), 1, ctypes.byref(chosen)) == b"rows128"
    assert (chosen.value > 1) == split
    gen = torch.Generator(device="cuda").manual_seed(M + K)
    qw = torch.randint(-2 ** 31, 2 ** 31 - 1, (K, N // 8), dtype=torch.int32, device="cuda", generator=gen)
    qz = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // g, N // 8), dtype=torch.int32, device="cuda", generator=gen)
    qs = ((torch.rand(K // g, N, device="cuda", generator=gen) + 0.1) * 0.2 / K ** 0.5).to(tdt)
    x = torch.randn(M, K, device="cuda", generator=gen).to(tdt)
    names = [L.awq_gemm_variant_name(i).decode() for i in range(L.awq_gemm_variant_count())]
    plain = awq_gemm_variant(x, qw, qs, qz, names.index("rows128"), chosen.value)
    assert torch.equal(ops.awq_linear_swiglu(x, qw, qs, qz), ops.silu_mul(plain, interleaved=True))
    assert torch.equal(_lib.torch_ops().awq_linear_swiglu(x, qw, qs, qz), ops.silu_mul(plain, interleaved=True))
    ref = x.double() @ nq.awq_dequantize(qw, qs, qz).double()
    assert (plain.double() - ref).abs().max().item() <= TIGHT[dtype] * ref.abs().max().item()


# a row, columns past the last tile, an odd number of words, two slabs (131072 x 1040: 273 MB)
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("M,K,N,g", [(1, 64, 8, 64), (300, 192, 264, 32), (257, 256, 1024, 128), (30, 131072, 520, 128)])
def test_linear_dense_pair(dtype, M, K, N, g):
    """Gate and up that lie apart, in one product: the bits of two products and the activation."""
    from nanoquantization_amd.engine import ops
    print(f"linear dense pair {dtype} M={M} K={K} N={N} g={g}", flush=True)
    tdt, L = torch.float16 if dtype == "f16" else torch.bfloat16, _lib.lib()
    gen = torch.Generator(device="cuda").manual_seed(M + N)
    words = lambda r: torch.randint(-2 ** 31, 2 ** 31 - 1, (r, N // 8), dtype=torch.int32, device="cuda", generator=gen)
    weights = [(words(K), (torch.rand(K // g, N, device="cuda", generator=gen) * 0.02 / K ** 0.5 * 8).to(tdt), words(K // g)) for _ in range(2)]
    x = torch.randn(M, K, device="cuda", generator=gen).to(tdt)
    scratch = torch.full((L.awq_linear_dense_scratch_bytes(M, 2 * N, K, g),), 0xFF, dtype=torch.uint8, device="cuda")   # NaN
    tail = (M, N, K, g, _lib.dtype_id(tdt))
    end = (scratch.data_ptr(), scratch.numel(), _lib.current_stream_ptr(x.device))
    parts = []
    for w in weights:
        parts.append(torch.empty(M, N, dtype=tdt, device="cuda"))
        _lib.check(L.awq_linear_dense(x.data_ptr(), *(t.data_ptr() for t in w), None, parts[-1].data_ptr(), *tail, 0, *end))
    y = torch.empty(M, N, dtype=tdt, device="cuda")
    scratch.fill_(0xFF)
    _lib.check(L.awq_linear_dense_pair(x.data_ptr(), *(t.data_ptr() for w in weights for t in w), y.data_ptr(), *tail, *end))
    assert torch.equal(y, _lib.torch_ops().silu_mul(*parts)) and not y.isnan().any()
    got = _lib.torch_ops().awq_swiglu_pair(x, *weights[0], *weights[1])
    assert (got.float() - y.float()).norm() <= 2.0 ** -7 * y.float().norm()
