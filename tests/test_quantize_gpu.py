"""The device quantise+pack kernel against the CPU oracle's quantise -> transpose -> int-quantise -> pack
chain (utils/quantization.py:5-58, awq/quantizer.py:156-158, layers/gemm.py:474-548 of the reference):
packed words, zero words and scales must be bit-identical."""
import numpy as np
import pytest
import torch

from oracle import awq_oracle as o

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("N,K,g", [(3072, 1024, 128), (64, 256, 32), (8, 128, 128), (1000, 384, 64), (40, 512, 512)])
def test_quantize_pack_bit_exact(dtype, N, K, g):
    import nanoquantization_amd as nq
    rng = np.random.default_rng(N * 7 + K + g)
    w = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
    w[0, :g] = 0.125            # a constant group: max == min, scale = 1e-5 / 15
    w[1 % N, g - 1] = 3.0       # an outlier that stretches one group
    w[2 % N, :g] = np.linspace(-1.0, 2.0, g, dtype=np.float32)
    ref = o.make_packed(w, g, dtype)
    tdt = torch.float16 if dtype == "f16" else torch.bfloat16
    print(f"quantize_pack N={N} K={K} g={g} {dtype}", flush=True)
    qw, qs, qz = nq.quantize_pack(torch.from_numpy(w).cuda(), g, tdt)
    assert np.array_equal(qw.cpu().numpy(), ref["qweight"])
    assert np.array_equal(qz.cpu().numpy(), ref["qzeros"])
    assert np.array_equal(qs.cpu().view(torch.int16).numpy().view(np.uint16), ref["qscales"])


# both tile widths at their edges: words past the last tile, columns past K, the switch between the widths (4096 x 4096),
# and rows that are not 16-byte aligned, which take the general kernel
@pytest.mark.parametrize("N,K,g,offset", [(264, 192, 64, 0), (72, 96, 32, 0), (520, 160, 32, 0), (248, 128, 128, 0),
                                          (4088, 4096, 128, 0), (4096, 4128, 32, 0), (264, 256, 128, 1)])
def test_quantize_tiles_bit_exact(N, K, g, offset):
    """Quotients exactly halfway between two codes, ones next to them, huge and tiny groups, infinities."""
    import nanoquantization_amd as nq
    rng = np.random.default_rng(N + K + g)
    w = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
    half = (np.arange(g) % 31 - 0.5).astype(np.float32)      # lo = -0.5, hi = 29.5: s = 2, v / s in quarters
    w[0, :g] = half
    w[3, -g:] = np.nextafter(half, np.float32(np.inf))
    w[5, -g:] = np.nextafter(half, np.float32(-np.inf))
    w[N - 1, -g:] = 1000.0 + half * 1e-4                     # quotients with few fraction bits
    w[N - 2, :g] *= np.float32(1e-30)
    w[N - 3, :g] *= np.float32(1e30)
    w[N - 4, :g] = np.where(np.arange(g) % 2, np.float32(3e38), np.float32(-3e38))     # hi - lo overflows
    w[N - 5, g - 1] = np.inf
    with np.errstate(all="ignore"):
        ref = o.make_packed(w, g, "bf16")
    buf = torch.zeros(N * K + offset, device="cuda")
    wd = buf[offset:].view(N, K)
    wd.copy_(torch.from_numpy(w))
    qw, qs, qz = nq.quantize_pack(wd, g, torch.bfloat16)
    finite = np.ones(N, bool)
    finite[[N - 4, N - 5]] = False        # what the oracle makes of a NaN quotient is the host's conversion of a NaN
    words = finite.reshape(-1, 8).all(axis=1)
    assert np.array_equal(qw.cpu().numpy()[:, words], ref["qweight"][:, words])
    assert np.array_equal(qz.cpu().numpy()[:, words], ref["qzeros"][:, words])
    assert np.array_equal(qs.cpu().view(torch.int16).numpy().view(np.uint16)[:, finite], ref["qscales"][:, finite])
    for at in ((0, 0), (N - 1, K - 1), (N // 2, g - 1)):
        bad = wd.clone()
        bad[at] = float("nan")
        with pytest.raises(AssertionError, match="nan"):
            nq.quantize_pack(bad, g, torch.bfloat16)


def test_quantize_pack_feeds_the_linear():
    import nanoquantization_amd as nq
    torch.manual_seed(0)
    w = torch.randn(512, 256) * 0.02
    x = torch.randn(5, 256).half()
    qw, qs, qz = nq.quantize_pack(w.cuda(), 128, torch.float16)
    y = nq.awq_gemm(x.cuda(), qw, qs, qz, 8).float().cpu()
    dq, _, _ = nq.pseudo_quantize(w, 128, 4, True)
    ref = x.float() @ dq.t()
    assert (y - ref).abs().max() <= 1e-2 * ref.abs().max()


def test_quantize_pack_rejects_bad_input():
    import nanoquantization_amd as nq
    from nanoquantization_amd import _lib
    with pytest.raises(_lib.AwqHipError, match="HIP device only"):
        nq.quantize_pack(torch.zeros(8, 128), 128)
    with pytest.raises(AssertionError, match="nan"):
        nq.quantize_pack(torch.full((8, 128), float("nan")).cuda(), 128)


def test_quantize_pack_under_a_default_device():
    """The caller's default device is where torch puts what names none: the word for NaN, in pinned host memory, names its own."""
    import nanoquantization_amd as nq
    w = torch.randn(16, 256, generator=torch.Generator().manual_seed(3)).cuda()
    want = nq.quantize_pack(w, 128, torch.bfloat16)
    with torch.device("cuda"):
        got = nq.quantize_pack(w, 128, torch.bfloat16)
        with pytest.raises(AssertionError, match="nan"):
            nq.quantize_pack(torch.full((8, 128), float("nan"), device="cuda"), 128)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("nan", [False, True])
def test_quantize_behind_queued_work(nan):
    """Work in front of the kernel that lasts longer than the host looks for its word, on a stream of the caller's: the call then waits for the stream."""
    import nanoquantization_amd as nq
    w = torch.randn(256, 512, generator=torch.Generator().manual_seed(5)).cuda()
    if nan:
        w[17, 300] = float("nan")
    torch.cuda.synchronize()
    big = torch.ones(1 << 28, device="cuda")
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        for _ in range(20):             # 2 GiB each
            big.mul_(1.0)
        if nan:
            with pytest.raises(AssertionError, match="nan"):
                nq.quantize_pack(w, 128)
        else:
            got = nq.quantize_pack(w, 128)
            assert stream.query(), "the call waits"
    torch.cuda.synchronize()
    if not nan:
        for a, b in zip(got, nq.quantize_pack(w, 128)):
            assert torch.equal(a, b)
