"""Kernels of the hybrid decoders against the plain oracle, each mechanism alone, in bf16 and in fp32."""
import pytest
import torch

from hybrid_cases import STREAM_SIZES, TALL_TILE_SIZES
from nanoquantization_amd import _lib
from nanoquantization_amd.engine import hybrid_ops as ops
from oracle import hybrid_oracle as o

pytestmark = pytest.mark.gpu
DTYPES = [torch.float32, torch.bfloat16]
TOL = {torch.float32: 2e-5, torch.bfloat16: 1.5e-2}


def rand(*shape, seed=0, dtype=torch.float32, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(dtype)


def close(got, want, dtype, what=""):
    got, want = got.double().cpu(), want.double()
    assert got.shape == want.shape, (what, got.shape, want.shape)
    err, ref = (got - want).abs().max().item(), want.abs().max().item()
    assert err <= TOL[dtype] * max(ref, 1e-3), (what, dtype, err, ref)


# ---- the step between two sublayers ----------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,width,parts", [(3, 72, 1), (5, 1024, 3), (2, 8192, 2), (4, 50, 2), (1, 7, 1)])
def test_residual_norm(dtype, rows, width, parts):
    print(f"residual_norm {rows}x{width} parts={parts} {dtype}", flush=True)
    x0, y = rand(rows, width, seed=1), rand(rows, parts, width, seed=2, dtype=dtype)
    wb, wn = rand(width, seed=3, dtype=dtype), rand(width, seed=4, dtype=dtype)
    table, ids = rand(9, width, seed=5, dtype=dtype), torch.tensor([i % 9 for i in range(rows)])
    c = lambda t: t.cuda().contiguous()
    eps = 1e-3
    # everything at once
    x = c(x0)
    h = ops.residual_norm(x, eps, y=c(y), post_weight=c(wb), ids=c(ids), table=c(table), next_weight=c(wn))
    want = x0.double() + o.rms(y.double().sum(1), wb.double(), eps) + table.double()[ids]
    close(x, want, torch.float32, "x")
    close(h, o.rms(want, wn.double(), eps), dtype, "h")
    # start of a pass over the layers
    x = torch.full((rows, width), float("nan"), device="cuda")
    h = ops.residual_norm(x, eps, init=True, ids=c(ids), table=c(table), next_weight=c(wn))
    close(x, table.double()[ids], torch.float32)
    close(h, o.rms(table.double()[ids], wn.double(), eps), dtype)
    # addition without a norm of its own, no successor
    x = c(x0)
    assert ops.residual_norm(x, eps, y=c(y)) is None
    close(x, x0.double() + y.double().sum(1), torch.float32)


# ---- q/k norm, rotary, cache write --------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,G,dim,vdim,rot,norm", [(6, 2, 40, 24, 24, True), (4, 4, 64, 64, 64, True), (3, 1, 22, 26, 10, True),
                                                  (4, 2, 128, 96, 0, True), (8, 2, 32, 48, 32, False)])
def test_qk_norm_rope_store(dtype, H, G, dim, vdim, rot, norm):
    print(f"qk_norm_rope_store H={H} G={G} dim={dim} vdim={vdim} rot={rot} {dtype}", flush=True)
    rows, bs, blocks, eps, base = 5, 4, 6, 1e-4, 300.0
    kr, vr = ((dim + 31) // 32 * 32, (vdim + 31) // 32 * 32) if dtype == torch.bfloat16 else (dim, vdim)
    qkv = rand(rows, H * dim + G * (dim + vdim), seed=1, dtype=dtype)
    qw, kw = rand(H * dim, seed=2, dtype=dtype), rand(G * dim, seed=3, dtype=dtype)
    pos = torch.tensor([0, 3, 17, 40, 41])
    slots = torch.tensor([5, 23, -1, 0, 10])
    freqs, mag = o.rotary_frequencies(rot, base, dict(factor=2.0, original=32, fast=4.0, slow=0.5)) if rot else ([], 1.0)
    table = None
    if rot:
        ang = torch.arange(64, dtype=torch.float64).unsqueeze(1) * torch.tensor(freqs, dtype=torch.float64)
        table = torch.cat([ang.cos() * mag, ang.sin() * mag], 1).float().cuda()
    kc = torch.zeros(blocks, G, bs, kr, dtype=dtype, device="cuda")
    vc = torch.zeros(blocks, G, bs, vr, dtype=dtype, device="cuda")
    q = ops.qk_norm_rope_store(qkv.cuda(), qw.cuda() if norm else None, kw.cuda() if norm else None, table, pos.cuda(),
                               slots.cuda(), kc, vc, H, dim, vdim, eps)
    d = qkv.double()
    wq, wk = d[:, :H * dim], d[:, H * dim:(H + G) * dim]
    if norm:
        wq, wk = o.rms(wq, qw.double(), eps), o.rms(wk, kw.double(), eps)
    wq, wk = wq.reshape(rows, H, dim), wk.reshape(rows, G, dim)
    if rot:
        wq = torch.stack([o.rotate_interleaved(wq[t], int(pos[t]), freqs, mag, rot) for t in range(rows)])
        wk = torch.stack([o.rotate_interleaved(wk[t], int(pos[t]), freqs, mag, rot) for t in range(rows)])
    close(q[..., :dim], wq, dtype, "q")
    assert torch.count_nonzero(q[..., dim:]) == 0
    wv = d[:, (H + G) * dim:].reshape(rows, G, vdim)
    ek, ev = torch.zeros(kc.shape, dtype=torch.float64), torch.zeros(vc.shape, dtype=torch.float64)
    for t, s in enumerate(slots.tolist()):
        if s >= 0:
            ek[s // bs, :, s % bs, :dim], ev[s // bs, :, s % bs, :vdim] = wk[t], wv[t]
    close(kc, ek, dtype, "k")
    close(vc, ev, dtype, "v")


# ---- attention ----------------------------------------------------------------------------------------------------
def paged(k, v, bs, dtype, spare=3, seed=9):
    """One sequence's keys and values [T, G, d] scattered over cache blocks; unused rows hold garbage."""
    T, G, dim = k.shape
    vdim = v.shape[2]
    kr, vr = ops.cache_rows(dim, vdim, dtype)
    nb = -(-T // bs)
    table = torch.randperm(nb + spare, generator=torch.Generator().manual_seed(seed))[:nb]
    kc = torch.full((nb + spare, G, bs, kr), 1e4, dtype=dtype)
    vc = torch.full((nb + spare, G, bs, vr), 1e4, dtype=dtype)
    kc[..., dim:], vc[..., vdim:] = 0, 0
    for t in range(T):
        b, i = int(table[t // bs]), t % bs
        kc[b, :, i, :dim], vc[b, :, i, :vdim] = k[t].to(dtype), v[t].to(dtype)
    return kc.cuda(), vc.cuda(), table.to(torch.int32).cuda()


def span(start, rows, table, bs):
    """The pass of one portion of the sequence whose block table is `table`."""
    return ops.PromptPass([(start, rows, table.tolist(), 0)], bs, torch.device("cuda"))


def padded_q(q, width, dtype):
    out = torch.zeros(q.shape[0], q.shape[1], width, dtype=dtype)
    out[..., :q.shape[2]] = q.to(dtype)
    return out.cuda()


ATTENTION = [  # T, H, G, dim, vdim, block, chunk
    (70, 4, 2, 40, 24, 16, 20), (130, 2, 1, 64, 64, 32, 0), (150, 3, 3, 96, 96, 64, 48), (65, 6, 1, 32, 48, 16, 7),
    (200, 4, 2, 128, 128, 64, 128), (100, 8, 1, 128, 64, 16, 64), (90, 2, 1, 192, 160, 32, 33), (80, 2, 2, 256, 256, 64, 0),
    (140, 16, 1, 64, 96, 16, 100), (75, 40, 2, 32, 32, 16, 50), (40, 2, 2, 22, 18, 16, 5), (33, 1, 1, 16, 16, 16, 1), (600, 2, 1, 64, 64, 64, 512)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("T,H,G,dim,vdim,bs,chunk", ATTENTION)
def test_attention_prefill_portions_and_decode(dtype, T, H, G, dim, vdim, bs, chunk):
    print(f"attention T={T} H={H} G={G} dim={dim} vdim={vdim} bs={bs} chunk={chunk} {dtype}", flush=True)
    q, k, v = (rand(T, H, dim, seed=1, dtype=dtype), rand(T, G, dim, seed=2, dtype=dtype), rand(T, G, vdim, seed=3, dtype=dtype))
    scale = dim ** -0.5 * 1.7
    want = o.attend(q.double(), k.double(), v.double(), scale, chunk).reshape(T, H * vdim)
    kc, vc, table = paged(k, v, bs, dtype)
    qd = padded_q(q, kc.shape[3], dtype)
    close(ops.attention_prefill(qd, kc, vc, span(0, T, table, bs), dim, vdim, scale, chunk), want, dtype, "whole")
    at = 0
    for n in (2, 3, 17, 16, 1, 31, T):      # portions that start and end anywhere
        n = min(n, T - at)
        if n:
            got = ops.attention_prefill(qd[at:at + n].contiguous(), kc, vc, span(at, n, table, bs), dim, vdim, scale, chunk)
            close(got, want[at:at + n], dtype, f"portion {at}+{n}")
        at += n
    # decode: every position at once, one row each
    rows = torch.tensor(sorted({0, 1, T // 2, T - 1, T - 2} | {c for e in range(0, T, max(chunk, 16)) for c in (e - 1, e, e + 1)
                                                           if 0 <= c < T}))
    tables = table.repeat(len(rows), 1).contiguous()
    got = ops.attention_decode(qd[rows.cuda()].contiguous(), kc, vc, tables, (rows + 1).to(torch.int32).cuda(), dim, vdim,
                               scale, chunk)
    close(got, want[rows], dtype, "decode")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("chunk,bs", [(48, 16), (50, 16), (0, 32), (300, 64)])
def test_attention_one_key_stands_out(dtype, chunk, bs):
    """A key that only one query points at, placed at the chunk's first token, just before it, at block borders and far
    away: the output must be that key's value exactly when the mask lets it through."""
    T, dim = 400, 64
    print(f"attention needle chunk={chunk} bs={bs} {dtype}", flush=True)
    for i in (399, 349, 200, 150):
        first = i // chunk * chunk if chunk else 0
        spots = {first, first + 1, first - 1, i, i - 1, i // bs * bs, i // bs * bs - 1, first + (i - first) // 2, 0}
        for j in sorted(s for s in spots if 0 <= s <= i):
            k, v = rand(T, 1, dim, seed=4, scale=0.1), rand(T, 1, dim, seed=5)
            q = rand(T, 1, dim, seed=6, scale=0.1)
            e = torch.zeros(dim)
            e[7] = 20.0
            q[i, 0], k[j, 0] = e, e
            kc, vc, table = paged(k, v, bs, dtype)
            qd = padded_q(q, dim, dtype)
            seen = o.visible(i, j, chunk)
            # alone, from a portion cut right in front of it, and decoded
            outs = [ops.attention_prefill(qd[i:i + 1].contiguous(), kc, vc, span(i, 1, table, bs), dim, dim, 0.125, chunk)[0],
                    ops.attention_prefill(qd[max(0, i - 40):i + 1].contiguous(), kc, vc,
                                          span(max(0, i - 40), min(i, 40) + 1, table, bs), dim, dim, 0.125, chunk)[-1],
                    ops.attention_decode(qd[i:i + 1].contiguous(), kc, vc, table.unsqueeze(0).contiguous(),
                                         torch.tensor([i + 1], dtype=torch.int32).cuda(), dim, dim, 0.125, chunk)[0]]
            for n, got in enumerate(outs):
                diff = (got.float().cpu() - v[j, 0]).abs().max().item()
                assert (diff < 2e-2) == seen, (i, j, chunk, n, diff, seen)


def test_attention_decode_long_context():
    """Contexts long enough for the context split, ragged over the batch."""
    dtype, T, G, H, dim, bs = torch.bfloat16, 3000, 2, 8, 64, 64
    k, v = rand(T, G, dim, seed=1, dtype=dtype), rand(T, G, dim, seed=2, dtype=dtype)
    kc, vc, table = paged(k, v, bs, dtype)
    ctx = torch.tensor([3000, 2999, 1, 65, 2049, 700], dtype=torch.int32)
    q = rand(len(ctx), H, dim, seed=3, dtype=dtype)
    for chunk in (0, 2048, 100):
        print(f"long decode chunk={chunk}", flush=True)
        got = ops.attention_decode(q.cuda(), kc, vc, table.repeat(len(ctx), 1).contiguous(), ctx.cuda(), dim, dim, 0.2, chunk)
        for b, n in enumerate(ctx.tolist()):
            lo = (n - 1) // chunk * chunk if chunk else 0
            kk, vv = k[lo:n].double(), v[lo:n].double()
            for h in range(H):
                s = kk[:, h // 4] @ q[b, h].double() * 0.2
                close(got[b, h * dim:(h + 1) * dim], torch.softmax(s, 0) @ vv[:, h // 4], dtype, (chunk, b, h))


# ---- gated linear attention ------------------------------------------------------------------------------------------
GLA_CASES = [(1, 2, 24, 40), (37, 3, 24, 40), (64, 2, 64, 64), (150, 2, 32, 32), (130, 1, 128, 128), (100, 2, 96, 48),
             (70, 1, 256, 256), (45, 2, 20, 12), (700, 1, 64, 96)]


def gla_inputs(T, H, dim, vdim, rank, dtype, seed=0, zshift=2.0):
    proj = rand(T, 2 * H * dim + 2 * H * vdim + rank, seed=seed, dtype=dtype)
    up = rand(H * dim, rank, seed=seed + 1, dtype=dtype, scale=rank ** -0.5)
    bias = (rand(H * dim, seed=seed + 2) + zshift).to(dtype)
    norm = (1 + 0.3 * rand(vdim, seed=seed + 3)).to(dtype)
    return proj, up, bias, norm


def gla_want(proj, up, bias, H, dim, vdim, tau, state=None):
    T = proj.shape[0]
    d = proj.double()
    q, k, v, g, low = d.split([H * dim, H * dim, H * vdim, H * vdim, up.shape[1]], dim=1)
    decay = o.channel_decay(low @ up.double().T + bias.double(), tau).view(T, H, dim)
    out, S = o.gla_scan(q.view(T, H, dim) * dim ** -0.5, k.view(T, H, dim), v.view(T, H, vdim), decay, state)
    return out, S, decay, g


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("T,H,dim,vdim", GLA_CASES)
@pytest.mark.parametrize("tau,zshift", [(4.0, 2.0), (1.0, -6.0)])
def test_gla_prefill_portions_and_decode(dtype, T, H, dim, vdim, tau, zshift):
    """zshift -6 at tau 1: decays of e^-6 and below a token, where a factored form of the decay would overflow."""
    rank, slots, eps = 10, 3, 1e-4
    print(f"gla T={T} H={H} dim={dim} vdim={vdim} tau={tau} {dtype}", flush=True)
    proj, up, bias, norm = gla_inputs(T, H, dim, vdim, rank, dtype, zshift=zshift)
    want, S, decay, g = gla_want(proj, up, bias, H, dim, vdim, tau)
    pd, ud, bd = proj.cuda(), up.cuda(), bias.cuda()
    dec = ops.gla_decay(pd, ud, bd, H, dim, vdim, tau)
    close(dec, decay.reshape(T, -1), torch.float32, "decay")
    # fp32 arithmetic on the given operands in either type: the tolerance is fp32's
    for cuts in ([T], [2] * (T // 2) + [T % 2], [T // 3, 16, T]):
        state = torch.full((slots, H, dim, vdim), 1e3, device="cuda")       # a slot is taken over as it is
        out = torch.empty(T, H * vdim, device="cuda")
        at = 0
        for n in cuts:
            n = min(n, T - at)
            if n > 0:
                one = ops.PromptPass([(at, n, range(T), 1)], 1, torch.device("cuda"))
                out[at:at + n] = ops.gla_prefill(pd[at:at + n], dec[at:at + n], state, one, H, dim, vdim, rank)
                at += n
        assert at == T
        close(out, want.reshape(T, -1), torch.float32, f"o {cuts[:2]}")
        close(state[1], S, torch.float32, "state")
        assert (state[0] == 1e3).all() and (state[2] == 1e3).all()
    gated = ops.head_norm_gate(out, pd, norm.cuda(), H, dim, vdim, rank, eps)
    wg = o.rms(want, norm.double(), eps).reshape(T, -1) * o.silu(g)
    close(gated, wg, dtype, "gated")
    # token by token, an idle row and a foreign slot beside it
    state = torch.full((slots, H, dim, vdim), 1e3, device="cuda")
    active = torch.tensor([True, False], device="cuda")
    slot = torch.tensor([2, 0], dtype=torch.int32, device="cuda")
    steps = min(T, 40)
    for t in range(steps):
        got = ops.gla_decode(pd[t:t + 1].repeat(2, 1), ud, bd, norm.cuda(), state, slot,
                             torch.tensor([t, t], device="cuda"), active, H, dim, vdim, tau, eps)
        close(got[0], wg[t], dtype, f"decode {t}")
        assert torch.count_nonzero(got[1]) == 0
    close(state[2], gla_want(proj[:steps], up, bias, H, dim, vdim, tau)[1], torch.float32, "decode state")
    assert (state[0] == 1e3).all() and (state[1] == 1e3).all()


@pytest.mark.parametrize("T", [300, 2100])
def test_gla_remembers_one_far_token(T):
    """Decays near 1 and one large key/value at the start, in the middle, at piece borders: the last token reads it."""
    H, dim, vdim, rank = 1, 32, 32, 4
    for j in (0, 15, 16, 63, 64, 255, 256, T - 1):
        print(f"gla needle T={T} j={j}", flush=True)
        proj = rand(T, 2 * dim + 2 * vdim + rank, seed=3, scale=0.01)
        proj[j, dim + 5] = proj[T - 1, 5] = 30.0
        up, bias = rand(dim, rank, seed=1), torch.full((dim,), 9.0)
        pd = proj.cuda()
        dec = ops.gla_decay(pd, up.cuda(), bias.cuda(), H, dim, vdim, 16.0)
        state = torch.zeros(1, H, dim, vdim, device="cuda")
        out = ops.gla_prefill(pd, dec, state, ops.PromptPass([(0, T, range(T), 0)], 1, torch.device("cuda")), H, dim, vdim, rank)
        q, k, v, _, _ = proj.double().split([dim, dim, vdim, vdim, rank], dim=1)
        d = dec.double().cpu()
        w = torch.cat([torch.flip(torch.cumprod(torch.flip(d[1:], [0]), 0), [0]), torch.ones(1, dim).double()])
        want = ((q[T - 1] * dim ** -0.5 * w * k).sum(-1, keepdim=True) * v).sum(0)
        close(out[T - 1], want, torch.float32, j)


@pytest.mark.parametrize("dtype", DTYPES)
def test_ragged_pass_equals_each_sequence_alone(dtype):
    """Portions of several sequences, some in their middle, long enough for several pieces and tiles, in one launch."""
    H, G, dim, vdim, bs, chunk, rank = 4, 2, 64, 48, 16, 100, 8
    portions = [(0, 300), (37, 150), (0, 1), (250, 2), (128, 128)]           # (start, rows)
    total = [s + n for s, n in portions]
    kr, vr = ops.cache_rows(dim, vdim, dtype)
    nb = [-(-t // bs) for t in total]
    order = torch.randperm(sum(nb), generator=torch.Generator().manual_seed(2)).tolist()
    kc, vc = (rand(sum(nb), G, bs, w, seed=7 + w, dtype=dtype).cuda() for w in (kr, vr + 0))
    blocks = [[order.pop() for _ in range(n)] for n in nb]
    segs = [(s, n, b, i) for i, ((s, n), b) in enumerate(zip(portions, blocks))]
    q = rand(sum(n for _, n in portions), H, kr, seed=3, dtype=dtype).cuda()
    print(f"ragged pass {dtype}", flush=True)
    dev = torch.device("cuda")
    got = ops.attention_prefill(q, kc, vc, ops.PromptPass(segs, bs, dev), dim, vdim, 0.1, chunk)
    HG, dg, vg = 16, 64, 80
    proj, up, bias, _ = gla_inputs(q.shape[0], HG, dg, vg, rank, dtype)
    proj, dec = proj.cuda(), None
    dec = ops.gla_decay(proj, up.cuda(), bias.cuda(), HG, dg, vg, 8.0)
    s0 = rand(len(segs), HG, dg, vg, seed=5).cuda()
    state = s0.clone()
    layout = ops.PromptPass(segs, bs, dev)
    assert layout.pieces(_lib.hybrid_lib().nqh_gla_piece_rows(q.shape[0], HG, dg, vg))[2]     # a sequence of several pieces
    o = ops.gla_prefill(proj, dec, state, layout, HG, dg, vg, rank)
    at = 0
    for i, seg in enumerate(segs):
        n = seg[1]
        one = ops.PromptPass([seg], bs, dev)
        alone = ops.attention_prefill(q[at:at + n].contiguous(), kc, vc, one, dim, vdim, 0.1, chunk)
        close(got[at:at + n], alone.double().cpu(), dtype, i)
        st = s0.clone()
        oi = ops.gla_prefill(proj[at:at + n].contiguous(), dec[at:at + n].contiguous(), st, one, HG, dg, vg, rank)
        close(o[at:at + n], oi.double().cpu(), torch.float32, i)
        close(state[i], st[i].double().cpu(), torch.float32, i)
        at += n


@pytest.mark.parametrize("dim,block", [(32, 16), (64, 24), (96, 64), (128, 7), (128, 64), (192, 32), (256, 64)])
def test_attention_prefill_tile_edges(dim, block):
    """Contexts around the key tiles (32 and 64) and the query tiles (128), one to five tiles, blocks of any size; scores
    that grow from tile to tile, a row whose first tiles are masked, scales of any sign."""
    H, G, bf = 4, 2, torch.bfloat16
    row = ops.cache_rows(dim, dim, bf)[0]
    lens = [1, 31, 33, 63, 64, 65, 127, 128, 129, 190, 257, 320]
    per = [(n + block - 1) // block for n in lens]
    first = [sum(per[:i]) for i in range(len(per))]
    blocks = torch.randperm(sum(per), generator=torch.Generator().manual_seed(1)).tolist()
    segs = [(0, n, blocks[f:f + p], 0) for n, f, p in zip(lens, first, per)]
    k = torch.zeros(sum(per), G, block, row, dtype=bf)
    v = torch.zeros_like(k)
    ks, vs, qs = [], [], []
    for i, (n, f, p) in enumerate(zip(lens, first, per)):
        kk, vv, qq = rand(p * block, G, dim, seed=3 * i, dtype=bf), rand(p * block, G, dim, seed=3 * i + 1, dtype=bf), rand(n, H, dim, seed=3 * i + 2, dtype=bf)
        kk *= (1 + torch.arange(p * block) / 40.0).view(-1, 1, 1).to(bf)       # later keys score higher and higher
        for j, b in enumerate(blocks[f:f + p]):
            k[b, :, :, :dim], v[b, :, :, :dim] = (x[j * block:(j + 1) * block].transpose(0, 1) for x in (kk, vv))
        ks.append(kk[:n].double()), vs.append(vv[:n].double()), qs.append(qq)
    q = torch.zeros(sum(lens), H, row, dtype=bf)
    q[:, :, :dim] = torch.cat(qs)
    lay = ops.PromptPass(segs, block, torch.device("cuda"))
    for scale, window in ((dim ** -0.5, 0), (-dim ** -0.5, 0), (0.0, 0), (dim ** -0.5, 70)):
        print(f"attention tiles dim={dim} block={block} scale={scale:.3f} window={window}", flush=True)
        got = ops.attention_prefill(q.cuda(), k.cuda(), v.cuda(), lay, dim, dim, scale, window=window).cpu()
        at = 0
        for n, kk, vv, qq in zip(lens, ks, vs, qs):
            s = torch.einsum("thd,shd->hts", qq.double(), kk.repeat_interleave(H // G, dim=1)) * scale
            i, j = torch.arange(n).view(-1, 1), torch.arange(n).view(1, -1)
            s = s.masked_fill((j > i) | (i - j >= (window or n + 1)), float("-inf"))
            want = torch.einsum("hts,shd->thd", s.softmax(dim=2), vv.repeat_interleave(H // G, dim=1)).reshape(n, H * dim)
            close(got[at:at + n], want, bf, (n, scale))
            at += n


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("heads", [10, 16])      # 640 workgroups, which all start at once, and more, whose waves go before one another
def test_prompt_attention_of_many_workgroups(dim, heads):
    """Dense, paged and latent prompts of many workgroups give the bits of each sequence alone, whichever wave goes first."""
    gen, bf, dev = torch.Generator(device="cuda").manual_seed(heads), torch.bfloat16, torch.device("cuda")
    randn = lambda *n: torch.randn(*n, generator=gen, device="cuda").to(bf)
    G, bs, scale = 2, 64, dim ** -0.5
    causal = _lib.torch_ops().causal_attention
    q, k, v = randn(8, 1000, heads, dim), randn(8, G, 1000, dim), randn(8, G, 1000, dim)
    print(f"many workgroups dim={dim} heads={heads}", flush=True)
    got = causal(q, k, v, scale)
    for b in range(8):
        assert torch.equal(got[b:b + 1], causal(q[b:b + 1], k[b:b + 1], v[b:b + 1], scale)), b
    # 65 tiles of queries, sequences on both sides of where the host's line for keys and the kernel's for dense keys lie
    lens = [1500, 1100, 1000, 900, 770, 640, 300, 129, 128, 1200]
    nb = [-(-n // bs) for n in lens]
    first = [sum(nb[:i]) for i in range(len(nb))]
    segs = [(0, n, list(range(f, f + m)), 0) for n, f, m in zip(lens, first, nb)]
    kc, vc, q = randn(sum(nb), G, bs, dim), randn(sum(nb), G, bs, dim), randn(sum(lens), heads, dim)
    kv, rot = randn(sum(lens), heads * (dim + 64)), randn(sum(lens), 32)
    width = _lib.hybrid_lib().nqh_latent_attention_prefill_query_row(dim, 32, 64, 1)
    ql = torch.zeros(sum(lens), heads, width, dtype=bf, device="cuda")
    ql[..., :dim + 32] = randn(sum(lens), heads, dim + 32)
    lay = ops.PromptPass(segs, bs, dev)
    paged = ops.attention_prefill(q, kc, vc, lay, dim, dim, scale)
    windowed = ops.attention_prefill(q, kc, vc, lay, dim, dim, scale, window=500)
    latent = ops.latent_attention_prefill(ql, kv, rot, lay, dim, 64, scale)
    at = 0
    for seg in segs:
        one, part = ops.PromptPass([seg], bs, dev), slice(at, at + seg[1])
        assert torch.equal(paged[part], ops.attention_prefill(q[part], kc, vc, one, dim, dim, scale)), seg[1]
        assert torch.equal(windowed[part], ops.attention_prefill(q[part], kc, vc, one, dim, dim, scale, window=500)), seg[1]
        assert torch.equal(latent[part], ops.latent_attention_prefill(ql[part], kv[part], rot[part], one, dim, 64, scale)), seg[1]
        at += seg[1]


# ---- mixture of experts --------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,width,experts,top,ff", [(1, 72, 5, 2, 48), (37, 64, 9, 1, 40), (20, 128, 7, 7, 64),
                                                      (300, 96, 4, 2, 36), (3, 50, 3, 1, 21), (64, 256, 64, 6, 128), (5, 64, 200, 3, 32), (90, 96, 300, 4, 16), (6, 80, 1, 1, 24),
                                                      (1500, 128, 6, 2, 160), (700, 256, 3, 1, 96),
                                                      (40, 264, 4, 2, 72), (100, 128, 8, 2, 64), (120, 136, 4, 1, 200)])
def test_router_and_experts(dtype, rows, width, experts, top, ff):
    print(f"moe rows={rows} width={width} experts={experts} top={top} ff={ff} {dtype}", flush=True)
    h = rand(rows, width, seed=1, dtype=dtype)
    router = rand(experts, width, seed=2, dtype=dtype, scale=2 * width ** -0.5)
    gu, dn = rand(experts, 2 * ff, width, seed=3, dtype=dtype, scale=width ** -0.5), rand(experts, width, ff, seed=4, dtype=dtype, scale=ff ** -0.5)
    expert, weight = ops.router_topk(h.cuda(), router.cuda(), top)
    s = torch.sigmoid(h.double() @ router.double().T)
    ws, we = s.topk(top, dim=1)
    close(weight, ws, torch.float32, "scores")
    gap = s.sort(dim=1, descending=True).values[:, :top + 1]
    clear = (gap[:, :-1] - gap[:, 1:]).min(dim=1).values > 1e-5 if experts > 1 else torch.ones(rows, dtype=torch.bool)
    assert torch.equal(expert.cpu().long()[clear], we[clear]) and clear.float().mean() > 0.8
    y = ops.moe_experts(h.cuda(), gu.cuda(), dn.cuda(), ops.route(h.cuda(), router.cuda(), top, ff))
    assert y.shape == (rows, top, width)
    e, w = expert.cpu().long(), weight.cpu().double()
    u = h.double().unsqueeze(1) * w.unsqueeze(-1)                              # [rows, top, width]
    want = torch.empty(rows, top, width, dtype=torch.float64)
    for x in range(experts):
        at = (e == x).nonzero(as_tuple=True)
        if len(at[0]):
            a, b = u[at] @ gu[x, :ff].double().T, u[at] @ gu[x, ff:].double().T
            want[at] = (o.silu(a) * b) @ dn[x].double().T
    close(y, want, dtype, "experts")


# the two tile sizes of the product core, output widths past the last tile, one stage of contraction and an odd number of them
@pytest.mark.parametrize("rows,width,experts,top,ff,tile", [(1200, 1600, 8, 2, 832, 128), (2500, 1600, 6, 2, 832, 256),
                                                            (17000, 64, 8, 2, 192, 256), (17000, 192, 60, 1, 64, 128)])
def test_experts_with_many_pairs(rows, width, experts, top, ff, tile):
    """An expert without pairs, one with a single pair, one with exactly a tile, the others unequal."""
    print(f"moe rows={rows} width={width} experts={experts} top={top} ff={ff}", flush=True)
    bf = torch.bfloat16
    h = rand(rows, width, seed=1, dtype=bf).cuda()
    gu = rand(experts, 2 * ff, width, seed=3, dtype=bf, scale=width ** -0.5).cuda()
    dn = rand(experts, width, ff, seed=4, dtype=bf, scale=ff ** -0.5).cuda()
    r = ops.Routing(rows, experts, top, width, ff, 1, h.device)
    assert r.tile_rows == tile
    pairs = rows * top
    e = 3 + (torch.rand(pairs, generator=torch.Generator().manual_seed(5)) ** 2 * (experts - 3)).int()
    e[7], e[tile:2 * tile] = 1, 2
    r.expert.copy_(e.view(rows, top))
    r.weight.copy_(torch.rand(rows, top, generator=torch.Generator().manual_seed(6)))
    r.order, r.tiles = ops.moe_plan(r.expert, experts, r.tile_rows)
    y = ops.moe_experts(h, gu, dn, r)
    u = h.double().unsqueeze(1) * r.weight.double().unsqueeze(-1)
    want = torch.empty(rows, top, width, dtype=torch.float64, device="cuda")
    for x in range(experts):
        at = (r.expert == x).nonzero(as_tuple=True)
        a, b = u[at] @ gu[x, :ff].double().T, u[at] @ gu[x, ff:].double().T
        want[at] = (a * torch.sigmoid(a) * b) @ dn[x].double().T
    close(y, want.cpu(), bf, "experts")
    assert torch.equal(y, ops.moe_experts(h, gu, dn, r))


# few pairs on large tiles: just past the skinny tiles, some 100 pairs an expert, near 128 where 256 pairs a tile are the faster; the same
# with weights too small for them; short rows, where the larger tiles come later; few experts, which keep the skinny tiles longer
@pytest.mark.parametrize("rows,width,experts,top,ff,tile", [(70, 1856, 20, 6, 960, 128), (300, 1024, 64, 20, 640, 128), (560, 1024, 40, 10, 640, 256),
                                                            (65, 1856, 8, 2, 960, 64), (353, 1856, 8, 2, 960, 64), (600, 1856, 8, 2, 960, 64),
                                                            (65, 512, 8, 2, 320, 64), (1000, 512, 8, 2, 320, 64), (3000, 1024, 8, 2, 512, 128),
                                                            (70, 1024, 4, 1, 320, 64), (33, 4096, 1, 1, 4096, 64)])
def test_experts_with_few_pairs_on_large_tiles(rows, width, experts, top, ff, tile):
    bf = torch.bfloat16
    print(f"moe rows={rows} width={width} experts={experts} top={top} ff={ff}", flush=True)
    h = rand(rows, width, seed=1, dtype=bf).cuda()
    gu = rand(experts, 2 * ff, width, seed=3, dtype=bf, scale=width ** -0.5).cuda()
    dn = rand(experts, width, ff, seed=4, dtype=bf, scale=ff ** -0.5).cuda()
    r = ops.Routing(rows, experts, top, width, ff, 1, h.device)
    assert r.tile_rows == tile
    r.expert.copy_(((torch.rand(rows, top, generator=torch.Generator().manual_seed(5)) ** 2) * experts).int())
    r.weight.copy_(torch.rand(rows, top, generator=torch.Generator().manual_seed(6)))
    r.order, r.tiles = ops.moe_plan(r.expert, experts, r.tile_rows)
    u = h.double().unsqueeze(1) * r.weight.double().unsqueeze(-1)
    want = torch.empty(rows, top, width, dtype=torch.float64, device="cuda")
    for x in range(experts):
        at = (r.expert == x).nonzero(as_tuple=True)
        a, b = u[at] @ gu[x, :ff].double().T, u[at] @ gu[x, ff:].double().T
        want[at] = (a * torch.sigmoid(a) * b) @ dn[x].double().T
    close(ops.moe_experts(h, gu, dn, r), want.cpu(), bf, "experts")


@pytest.mark.parametrize("streams,width,parts", [(1, 1024, 1), (2, 1024, 2), (4, 50, 5), (8, 4100, 7)])
def test_norms_add_parts_of_either_type(streams, width, parts):
    """Parts of the call's type and the same values as fp32 sums, one part and several: kernels of their own, which may contract their
    products differently.  At most streams + parts fp32 operations on values of the result's size: 15 x 2^-24, a twentieth of the bound."""
    print(f"parts of either type {streams} x {width}, {parts}", flush=True)
    bf, rows = torch.bfloat16, 5
    y = rand(rows, parts, width, seed=1, dtype=bf).cuda()
    wn, mix, write = (rand(*s, seed=2 + i, dtype=bf).cuda() for i, s in enumerate([(width,), (streams, streams), (streams,)]))
    x0 = rand(rows, streams, width, seed=7).cuda()
    rms = lambda t, w: t / (t.square().mean(-1, keepdim=True) + 1e-3).sqrt() * w.double()
    total = y.double().sum(1)
    mixed = torch.einsum("st,rsw->rtw", mix.double(), x0.double()) + write.double().view(1, -1, 1) * total.unsqueeze(1)
    for v in (y, y.float()):
        x, r = x0.clone(), x0[:, 0].clone()
        h = ops.hyper_norm(x, 1e-3, y=v, mix=mix, write=write, next_weight=wn)
        close(x, mixed.cpu(), torch.float32, v.dtype)
        close(h, rms(mixed.sum(1), wn).cpu(), bf, v.dtype)
        ops.residual_norm(r, 1e-3, y=v, post_weight=wn, next_weight=wn)
        close(r, (x0[:, 0].double() + rms(total, wn)).cpu(), torch.float32, v.dtype)


@pytest.mark.parametrize("rows,width,parts", [(1, 72, 1), (16, 2048, 7), (5, 50, 3)])
def test_residual_norm_route_adds_the_parts_of_a_product(rows, width, parts):
    """fp32 parts beside bf16 weights, as residual_norm and route take them."""
    print(f"norm + route of fp32 parts {rows} x {parts} x {width}", flush=True)
    bf = torch.bfloat16
    x0, y = rand(rows, width, seed=1).cuda(), rand(rows, parts, width, seed=2).cuda()
    wb, wn, router = (rand(*s, seed=3 + i, dtype=bf).cuda() for i, s in enumerate([(width,), (width,), (8, width)]))
    x1, x2 = x0.clone(), x0.clone()
    h1 = ops.residual_norm(x1, 1e-5, y=y, post_weight=wb, next_weight=wn)
    h2, r = ops.residual_norm_route(x2, 1e-5, router, 2, 64, wn, y=y, post_weight=wb)
    assert torch.equal(x1, x2) and torch.equal(h1, h2) and torch.equal(r.expert, ops.route(h1, router, 2, 64).expert)
    total = y.double().sum(1)
    close(x1, (x0 + total / (total.square().mean(-1, keepdim=True) + 1e-5).sqrt() * wb).double().cpu(), torch.float32)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,width,experts,top,ff", [(1, 72, 5, 2, 48), (16, 2048, 8, 2, 64), (64, 256, 64, 6, 128),
                                                      (200, 1028, 128, 8, 32), (33, 4096, 3, 3, 24), (300, 64, 8, 2, 32)])
def test_residual_norm_route_equals_separate_launches(dtype, rows, width, experts, top, ff):
    print(f"norm + route rows={rows} width={width} experts={experts} top={top} {dtype}", flush=True)
    x0, y = rand(rows, width, seed=1).cuda(), rand(rows, 2, width, seed=2, dtype=dtype).cuda()
    wb, wn = rand(width, seed=3, dtype=dtype).cuda(), rand(width, seed=4, dtype=dtype).cuda()
    router = rand(experts, width, seed=5, dtype=dtype, scale=2 * width ** -0.5).cuda()
    for again in range(3):                 # the arrival counter is left as it was found
        x1, x2 = x0.clone(), x0.clone()
        h1 = ops.residual_norm(x1, 1e-5, y=y, post_weight=wb, next_weight=wn)
        h2, r = ops.residual_norm_route(x2, 1e-5, router, top, ff, wn, y=y, post_weight=wb)
        assert torch.equal(x1, x2) and torch.equal(h1, h2)
        s = torch.sigmoid(h1.double() @ router.double().T).cpu()
        ws, we = s.topk(top, dim=1)
        close(r.weight, ws, torch.float32, "scores")
        gap = s.sort(dim=1, descending=True).values[:, :top + 1]
        clear = (gap[:, :-1] - gap[:, 1:]).min(dim=1).values > 1e-5
        assert torch.equal(r.expert.cpu().long()[clear], we[clear]) and clear.float().mean() > 0.8
        e, order, tiles = r.expert.cpu().reshape(-1), r.order.cpu().long(), r.tiles.cpu()
        n, seen = r.max_tiles, 0
        assert sorted(order.tolist()) == list(range(rows * top))
        for t in range(int(tiles[-1])):
            ex, first, count = int(tiles[t]), int(tiles[n + t]), int(tiles[2 * n + t])
            assert 1 <= count <= r.tile_rows and first == seen and (e[order[first:first + count]] == ex).all()
            seen += count
        assert seen == rows * top


def test_moe_plan_groups_every_pair_once():
    for pairs, experts, rows in ((1, 1, 16), (1000, 7, 16), (5000, 64, 128), (300, 1000, 32)):
        print(f"plan pairs={pairs} experts={experts}", flush=True)
        e = torch.randint(0, experts, (pairs, 1), generator=torch.Generator().manual_seed(pairs), dtype=torch.int32)
        e[: pairs // 3] = e[0]
        order, tiles = ops.moe_plan(e.cuda(), experts, rows)
        order, tiles = order.cpu().long(), tiles.cpu()
        n = (tiles.numel() - 1) // 3
        assert sorted(order.tolist()) == list(range(pairs))
        seen = 0
        for t in range(int(tiles[-1])):
            ex, first, count = int(tiles[t]), int(tiles[n + t]), int(tiles[2 * n + t])
            assert 1 <= count <= rows and (e[order[first:first + count], 0] == ex).all() and first == seen
            seen += count
        assert seen == pairs


# ---- dense products, sampling ----------------------------------------------------------------------------------------
@pytest.mark.parametrize("rows,n_out,n_in", [(1, 440, 200), (3, 50, 8), (16, 1000, 1024), (17, 96, 136), (33, 256, 512),
                                             (64, 640, 4096), (5, 16, 128), (48, 33, 72)])
def test_skinny_linear(rows, n_out, n_in):
    print(f"skinny {rows} x {n_in} -> {n_out}", flush=True)
    x, w = rand(rows, n_in, seed=1, dtype=torch.bfloat16), rand(n_out, n_in, seed=2, dtype=torch.bfloat16)
    b = rand(n_out, seed=3, dtype=torch.bfloat16)
    want = x.double() @ w.double().T
    close(ops.skinny_linear(x.cuda(), w.cuda(), out_f32=True), want, torch.float32)
    close(ops.skinny_linear(x.cuda(), w.cuda(), b.cuda(), out_f32=True), want + b.double(), torch.float32)
    close(ops.skinny_linear(x.cuda(), w.cuda(), b.cuda()), want + b.double(), torch.bfloat16)


# whole and split contractions, ends inside a stage, a wave's features, a workgroup; what a former launch left in LDS (NaN here)
# reaches nothing.  Bounds as for any fp32 sum of these lengths: `close`.  Every tile height and workgroup width: test_stream_linear_forms
@pytest.mark.parametrize("rows,n_out,n_in", [(1, 64, 8), (5, 132, 1000), (16, 2048, 2048), (16, 544, 4096), (17, 1028, 136), (20, 4608, 1024),
                                             (32, 2052, 9224), (33, 4096, 4608), (64, 4100, 2056), (64, 12288, 1024), (40, 1030, 520),
                                             (64, 18432, 2048)])
def test_skinny_linear_parts(rows, n_out, n_in):
    print(f"skinny parts {rows} x {n_in} -> {n_out}", flush=True)
    x, w, b = (rand(*s, seed=i, dtype=torch.bfloat16) for i, s in enumerate([(rows, n_in), (n_out, n_in), (n_out,)]))
    xd, wd = x.cuda(), w.cuda()
    want = x.double() @ w.double().T
    for poison in (False, True):
        if poison:
            ops.skinny_linear(torch.full_like(xd, float("nan")), wd)
        sums = ops.skinny_linear_sums(xd, wd)
        assert sums.shape[::2] == (rows, n_out)
        close(sums.double().sum(1), want, torch.float32)
        close(ops.skinny_linear(xd, wd, b.cuda(), out_f32=True), want + b.double(), torch.float32)
    close(ops.skinny_linear(xd, wd, b.cuda(), activation="relu2"), (want + b.double()).clamp(min=0) ** 2, torch.bfloat16)
    # without scratch memory, and where the result does not lie on 16 bytes
    y = torch.empty(rows * n_out + 1, dtype=torch.bfloat16, device="cuda")[1:].view(rows, n_out)
    for scratch, nbytes in ((None, 0), (torch.empty(64 << 20, dtype=torch.uint8, device="cuda"), 64 << 20)):
        ops._call(xd.device, "nqh_skinny_linear_ex", xd.data_ptr(), wd.data_ptr(), None, y.data_ptr(), rows, n_out, n_in, 0, 0, 0.0,
                  ops._ptr(scratch), nbytes)
        close(y, want, torch.bfloat16)


@pytest.mark.parametrize("rows,n_out,n_in", STREAM_SIZES)
def test_stream_linear_forms(rows, n_out, n_in):
    """Every form (test_hybrid_host.py checks that the sizes reach them all): into bf16 and fp32, with a bias and an activation, without
    scratch memory, with it and for a reader.  Bounds as above."""
    print(f"stream linear {rows} x {n_in} -> {n_out}", flush=True)
    x, w, b = (rand(*s, seed=i, dtype=torch.bfloat16).cuda() for i, s in enumerate([(rows, n_in), (n_out, n_in), (n_out,)]))
    want = x.double() @ w.double().T
    full = ((want + b.double()).clamp(min=0) ** 2).cpu()
    scratch = torch.full((16 * rows * n_out,), float("nan"), device="cuda")
    for room in (None, scratch):
        for f32, dtype in ((0, torch.bfloat16), (1, torch.float32)):
            y = torch.full((rows, n_out), float("nan"), dtype=dtype, device="cuda")
            ops._call(x.device, "nqh_skinny_linear_ex", x.data_ptr(), w.data_ptr(), b.data_ptr(), y.data_ptr(), rows, n_out, n_in, f32, 1, 0.0,
                      ops._ptr(room), 0 if room is None else 4 * room.numel())
            close(y, full, dtype, (room is None, f32))
    close(ops.skinny_linear_sums(x, w).double().sum(1), want.cpu(), torch.float32)


def test_linear_of_many_rows_with_a_strided_bias():
    """The library's product takes what dense_linear does not."""
    from nanoquantization_amd.engine.hybrid_engine import HybridEngine
    print("linear of 300 rows, strided bias", flush=True)
    x, w, b = (rand(*s, seed=i, dtype=torch.bfloat16).cuda() for i, s in enumerate([(300, 1024), (2048, 1024), (2048, 2)]))
    engine = HybridEngine.__new__(HybridEngine)
    engine._busy = False
    assert ops.dense_linear_wanted(x, w, False, False)
    want = (x.double() @ w.double().T + b[:, 1].double()).cpu()
    close(engine._linear(x, w, b[:, 1]), want, torch.bfloat16)
    close(engine._linear(x, w, b[:, 1].contiguous()), want, torch.bfloat16)


@pytest.mark.parametrize("rows", [16, 65])
def test_linears_without_memory_for_parts(rows, monkeypatch):
    """Where no memory is left for the sums of parts, a linear of an engine runs unsplit into its plain result."""
    from nanoquantization_amd.engine.hybrid_engine import HybridEngine
    print(f"linear without memory for parts, {rows} rows", flush=True)
    n_out, n_in = 4096, 18432
    x, w = (rand(*s, seed=i, dtype=torch.bfloat16) for i, s in enumerate([(rows, n_in), (n_out, n_in)]))
    xd, wd = x.cuda(), w.cuda()
    want = (xd.double() @ wd.double().T).cpu()
    engine = HybridEngine.__new__(HybridEngine)
    engine._busy = False
    parts = engine._sublayer_linear(xd, wd)
    assert parts.dim() == 3 and parts.shape[1] > 1                 # there is something to do without
    empty = torch.empty

    def little(*size, **kw):
        t = empty(*size, **kw)
        if t.numel() * t.element_size() > rows * n_out * 2:
            raise torch.cuda.OutOfMemoryError("only the result fits")
        return t
    with monkeypatch.context() as m:
        m.setattr(torch, "empty", little)
        y, alone = engine._sublayer_linear(xd, wd), engine._linear(xd, wd)
    assert y.shape == (rows, n_out) and y.dtype == torch.bfloat16
    close(y, want, torch.bfloat16)
    close(alone, want, torch.bfloat16)


@pytest.mark.parametrize("rows,width,parts", [(1, 64, 1), (3, 1024, 2), (2, 50, 3), (5, 2052, 7), (2, 4096, 16), (300, 72, 5)])
def test_norms_add_the_parts_of_a_product(rows, width, parts):
    """The residual's next read with fp32 parts equals the one with their sum."""
    print(f"parts {rows} x {parts} x {width}", flush=True)
    y = rand(rows, parts, width, seed=1).cuda()
    total = y.double().sum(1)
    x0, wn, wp = rand(rows, width, seed=2), rand(width, seed=3, dtype=torch.bfloat16), rand(width, seed=4, dtype=torch.bfloat16)
    rms = lambda t, w: t / (t.square().mean(-1, keepdim=True) + 1e-3).sqrt() * w.double()
    x = x0.cuda()
    h = ops.residual_norm(x, 1e-3, y=y, post_weight=wp.cuda(), next_weight=wn.cuda())
    want = x0.double() + rms(total.cpu(), wp)
    close(x, want, torch.float32)
    close(h, rms(want, wn), torch.bfloat16)
    x, mix, write = torch.stack([x0, 2 * x0], 1).cuda(), torch.tensor([[0.5, 0.25], [1.0, 2.0]]), torch.tensor([1.0, 0.5])
    h = ops.hyper_norm(x, 1e-3, y=y, mix=mix.bfloat16().cuda(), write=write.bfloat16().cuda(), next_weight=wn.cuda())
    want = torch.einsum("st,rsw->rtw", mix.double(), torch.stack([x0, 2 * x0], 1).double()) + write.double().view(1, 2, 1) * total.cpu().unsqueeze(1)
    close(x, want, torch.float32)
    close(h, rms(want.sum(1), wn), torch.bfloat16)


# one row, both tile heights, rows and columns past their tiles (also fewer than a tile), one stage to many; several rounds of tiles
@pytest.mark.parametrize("rows,n_out,n_in", [(1, 8, 64), (130, 264, 128), (127, 4608, 192), (257, 8, 320), (256, 512, 1024),
                                             (2049, 4616, 1024), (4000, 1032, 64)])
def test_dense_activation(rows, n_out, n_in):
    print(f"dense activation {rows} x {n_in} -> {n_out}", flush=True)
    x, w = rand(rows, n_in, seed=1, dtype=torch.bfloat16), rand(n_out, n_in, seed=2, dtype=torch.bfloat16, scale=n_in ** -0.5)
    want = x.double() @ w.double().T
    got = ops.dense_activation(x.cuda(), w.cuda(), "relu2").cpu()
    close(got, want.clamp(min=0) ** 2, torch.bfloat16)
    y = ops.dense_activation(x.cuda(), w.cuda(), None)
    close(y, want, torch.bfloat16)
    assert torch.equal(got, ops.activate_(y, "relu2").cpu())      # of the product rounded to bf16


# whole and split contractions (the last part shorter), rows and columns past their tiles, fewer than a tile, on tiles of 128 rows; of 256: below
@pytest.mark.parametrize("rows,n_out,n_in", [(65, 8, 64), (130, 96, 2048), (127, 4608, 192), (257, 264, 4672), (1000, 1024, 4608),
                                             (2049, 2056, 1024), (300, 4096, 18432)])
def test_dense_linear(rows, n_out, n_in):
    print(f"dense linear {rows} x {n_in} -> {n_out}", flush=True)
    x, w, b = (rand(*s, seed=i, dtype=torch.bfloat16) for i, s in enumerate([(rows, n_in), (n_out, n_in), (n_out,)]))
    xd, wd = x.cuda(), w.cuda()
    want = (xd.double() @ wd.double().T).cpu()
    close(ops.dense_linear(xd, wd), want, torch.bfloat16)
    close(ops.dense_linear(xd, wd, b.cuda()), want + b.double(), torch.bfloat16)
    y = torch.empty(rows, n_out, dtype=torch.bfloat16, device="cuda")           # without scratch memory: one part
    ops._call(xd.device, "nqh_dense_linear", xd.data_ptr(), wd.data_ptr(), None, y.data_ptr(), rows, n_out, n_in, n_in, None, 0)
    close(y, want, torch.bfloat16)
    wide = torch.full((rows, n_in + 24), float("nan"), dtype=torch.bfloat16, device="cuda")      # columns of a wider tensor
    wide[:, 8:8 + n_in] = xd
    assert torch.equal(ops.dense_linear(wide[:, 8:8 + n_in], wd), ops.dense_linear(xd, wd))
    sums = ops.dense_linear_sums(xd, wd)
    assert (sums is None) == (ops._of_sizes("nqh_dense_linear_parts", rows, n_out, n_in) == 1)
    if sums is not None:
        close(sums.double().sum(1), want, torch.float32)


@pytest.mark.parametrize("rows,n_out,n_in", TALL_TILE_SIZES)
def test_dense_linear_on_tall_tiles(rows, n_out, n_in):
    """256-row tiles whole and in parts, with rows and columns past the last tile: a bias, a row stride, parts added by a pass and by
    a reader."""
    print(f"dense linear on tall tiles {rows} x {n_in} -> {n_out}", flush=True)
    x, w, b = (rand(*s, seed=i, dtype=torch.bfloat16).cuda() for i, s in enumerate([(rows, n_in), (n_out, n_in), (n_out,)]))
    want = (x.double() @ w.double().T).cpu()
    wide = torch.full((rows, n_in + 24), float("nan"), dtype=torch.bfloat16, device="cuda")
    wide[:, 8:8 + n_in] = x
    close(ops.dense_linear(x, w, b), want + b.double().cpu(), torch.bfloat16)
    assert torch.equal(ops.dense_linear(wide[:, 8:8 + n_in], w, b), ops.dense_linear(x, w, b))
    y = torch.empty(rows, n_out, dtype=torch.bfloat16, device="cuda")           # without scratch memory
    ops._call(x.device, "nqh_dense_linear", wide[:, 8:].data_ptr(), w.data_ptr(), b.data_ptr(), y.data_ptr(), rows, n_out, n_in, n_in + 24, None, 0)
    close(y, want + b.double().cpu(), torch.bfloat16)
    sums = torch.full((rows, ops._of_sizes("nqh_dense_linear_parts", rows, n_out, n_in), n_out), float("nan"), device="cuda")
    ops._call(x.device, "nqh_dense_linear_sums", x.data_ptr(), w.data_ptr(), sums.data_ptr(), rows, n_out, n_in)
    close(sums.double().sum(1), want, torch.float32)


def test_argmax_and_bookkeeping():
    for rows, vocab in ((1, 5), (3, 131), (4, 32000), (2, 4098)):
        x = rand(rows, vocab, seed=vocab)
        x[0, vocab - 1] = x[0, 1] = 99.0
        assert torch.equal(ops.argmax_rows(x.cuda()).cpu(), x.argmax(-1).where(torch.arange(rows) > 0, torch.tensor(1)))
    pos, act = torch.tensor([0, 5, 9]).cuda(), torch.tensor([True, True, False]).cuda()
    table = torch.tensor([[3, 1, 0], [2, 4, 0], [5, 5, 5]], dtype=torch.int32).cuda()
    slots, ctx = ops.decode_prepare(pos, act, table, 4)
    assert slots.tolist() == [12, 17, -1] and ctx.tolist() == [1, 6, 10]
    log, ids, step = torch.zeros(2, 3, dtype=torch.long).cuda(), torch.zeros(3, dtype=torch.long).cuda(), torch.zeros(1, dtype=torch.long).cuda()
    ops.decode_advance(torch.tensor([7, 8, 9]).cuda(), act, log, ids, pos, step)
    assert log.tolist() == [[7, 8, 9], [0, 0, 0]] and ids.tolist() == [7, 8, 9] and pos.tolist() == [1, 6, 9] and step.item() == 1


def test_argument_checks_raise():
    q = torch.zeros(4, 2, 32, dtype=torch.bfloat16, device="cuda")
    kc = torch.zeros(2, 1, 16, 32, dtype=torch.bfloat16, device="cuda")
    table = torch.tensor([0], dtype=torch.int32, device="cuda")
    with pytest.raises(_lib.AwqHipError):                  # positions past the block table
        ops.attention_prefill(q, kc, kc, span(13, 4, table, 16), 32, 32, 1.0)
    with pytest.raises(_lib.AwqHipError):
        ops.skinny_linear(torch.zeros(65, 32, dtype=torch.bfloat16, device="cuda"), torch.zeros(8, 32, dtype=torch.bfloat16, device="cuda"))
    with pytest.raises(_lib.AwqHipError):
        ops.router_topk(torch.zeros(1, 8, device="cuda"), torch.zeros(2, 8, device="cuda"), 3)
    with pytest.raises(_lib.AwqHipError):
        ops.argmax_rows(torch.zeros(1, 8))
