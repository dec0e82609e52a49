"""The Sabezen decoder on the GPU against the plain implementation: the new kernels alone, each
mechanism as a model of one layer, the whole model under four ways of cutting the same requests into
steps (whole, bulk then single tokens, portions down to two tokens, mixed batches on a small page pool
with four state slots, pages and slots used again), in 32-bit and in bfloat16, on configurations with
even and with odd sizes and on one without any attention; keys far away and at the edges of a chunk;
long decoding through graph replays; greedy generation through the entry point and its scheduler; the
trace runner and the command line as subprocesses."""
import json
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

import plain_sabezen as ps
import sabezen_util as su
import trace_util as tu
from conftest import ROOT

pytestmark = pytest.mark.gpu

TOL = {"float32": 3e-5, "bfloat16": 8e-2}
DT = {"float32": torch.float32, "bfloat16": torch.bfloat16}
LENGTHS = {"A": [5, 17, 64, 1, 100, 33, 129, 49, 2], "B": [40, 3, 100, 65, 2, 31], "C": [90, 3, 41, 1, 130],
           "D": [700, 47, 313, 1, 161]}


def dev(a, dtype=None):
    t = torch.as_tensor(np.asarray(a))
    if dtype is not None:
        t = t.to(dtype)
    return t.cuda().contiguous()


def i32(a):
    return torch.as_tensor(np.asarray(a, dtype=np.int32)).cuda()


# ------------------------------------------------------------------ kernels alone

@pytest.mark.parametrize("d", [4, 60, 260, 4096, 4100, 8192, 8196])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_layernorm_in_fours(d, dt):
    """Widths of whole fours: less than a wave's, one and two fours a thread, and the first that goes back to one value at a
    time; rows far from zero, gathered.  A float32 mean and variance of d numbers are off by some roundings each."""
    from hfee_amd.kernels import ops
    g = torch.Generator().manual_seed(d)
    x, w = torch.randn(5, d, generator=g) * 2 + 9, (1 + torch.randn(d, generator=g) * 0.3).to(dt)
    out = torch.zeros(3, d, dtype=dt, device="cuda")
    ops.layernorm(out, x.cuda(), w.cuda(), 1e-5, i32([4, 0, 4]))
    assert su.rel(out.double().cpu(), ps.layer_norm(x.double(), w.double(), 1e-5)[[4, 0, 4]]) < (2e-6 if dt == torch.float32 else 6e-3)


@pytest.mark.parametrize("d", [4, 60, 90, 260, 1028, 4095, 4096, 4100, 8192, 8196])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_layernorm_has_one_order_of_additions(d, dt):
    """Widths that go through fours and widths that do not: 256 shares, each its every 256th value in order, four waves of
    them in a butterfly each, the waves in order.  The same sums in numpy give the same bits."""
    from hfee_amd.kernels import ops
    g = torch.Generator().manual_seed(d)
    x, w = torch.randn(4, d, generator=g) * 2 + 9, (1 + torch.randn(d, generator=g) * 0.3).to(dt)
    out = torch.zeros(4, d, dtype=dt, device="cuda")
    ops.layernorm(out, x.cuda(), w.cuda(), 1e-5)

    def workgroup(shares):                          # [rows, 256]
        lanes = shares.reshape(-1, 4, 64)
        for off in (32, 16, 8, 4, 2, 1):
            lanes = lanes + lanes[:, :, np.arange(64) ^ off]
        total = np.zeros(len(lanes), np.float32)
        for wave in range(4):
            total = total + lanes[:, wave, 0]
        return total

    f = np.float32
    rows = np.zeros((4, -(-d // 256) * 256), f)
    rows[:, :d] = x.numpy()
    inside = np.arange(rows.shape[1]) < d
    shares = np.zeros((4, 256), f)
    for i in range(0, rows.shape[1], 256):
        shares = shares + rows[:, i:i + 256]
    off = np.where(inside, rows - (workgroup(shares) / f(d))[:, None], f(0))
    squares = np.zeros((4, 256), f)
    for i in range(0, rows.shape[1], 256):          # (one rounding a step: the product is exact in the wider type)
        own = off[:, i:i + 256].astype(np.longdouble)
        squares = (own * own + squares).astype(f)
    inv = f(1) / np.sqrt(workgroup(squares) / f(d) + f(1e-5))
    want = torch.from_numpy(off[:, :d] * inv[:, None] * w.float().numpy()).to(dt)
    assert torch.equal(out.cpu(), want)


@pytest.mark.parametrize("d", [1024, 1028, 2048, 4096, 4100])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_layernorm_rows_have_the_same_bits_among_many(d, dt):
    """From some number of rows on, another one for either type, rows of 1,025 to 4,096 go through another kernel."""
    from hfee_amd.kernels import ops
    x = torch.randn(2049, d, generator=torch.Generator().manual_seed(d)).cuda()
    w, outs = torch.full((d,), 0.7, device="cuda"), []
    for n in (3, 256, 257, 512, 513, 1024, 1025, 2049):
        outs.append(torch.zeros(n, d, dtype=dt, device="cuda"))
        ops.layernorm(outs[-1], x[:n], w, 1e-5)
    assert all(torch.equal(o, outs[-1][:len(o)]) for o in outs) and float(outs[-1].float().std()) > 0.5


def test_layernorm_and_scaled_embedding():
    from hfee_amd.kernels import ops
    g = torch.Generator().manual_seed(0)
    x = torch.randn(7, 90, generator=g) * 3 + 1.5
    w = 1 + torch.randn(90, generator=g) * 0.3
    for dt in (torch.float32, torch.bfloat16):
        out = torch.zeros(7, 90, dtype=dt, device="cuda")
        ops.layernorm(out, x.cuda(), w.to(dt).cuda(), 1e-5)
        want = ps.layer_norm(x.double(), w.to(dt).double(), 1e-5)
        assert su.rel(out.double().cpu(), want) < (2e-6 if dt == torch.float32 else 6e-3)
    rows = i32([5, 0, 5])
    out = torch.zeros(3, 90, device="cuda")
    ops.layernorm(out, x.cuda(), w.cuda(), 1e-5, rows)
    assert su.rel(out.cpu(), ps.layer_norm(x.double(), w.double(), 1e-5)[[5, 0, 5]]) < 2e-6
    table = torch.randn(20, 24, generator=g)
    for dt in (torch.float32, torch.bfloat16):
        emb = torch.zeros(4, 24, device="cuda")
        ops.embed(emb, table.to(dt).cuda(), i32([3, 19, 0, 3]), scale=7.5)
        assert torch.equal(emb.cpu(), table.to(dt).float()[[3, 19, 0, 3]] * 7.5)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_xielu(dtype):
    from hfee_amd.kernels import ops
    dt = DT[dtype]
    z = torch.linspace(-6, 6, 333).reshape(3, 111).to(dt)
    p, q = torch.tensor(0.7, dtype=torch.float64), torch.tensor(-0.4, dtype=torch.float64)
    a, b = float(torch.nn.functional.softplus(p)), 0.5 + float(torch.nn.functional.softplus(q))
    out = torch.zeros(3, 111, dtype=dt, device="cuda")
    ops.bias_act(out, z.cuda(), None, "xielu", (a, b))
    want = ps.xielu(z.double(), p, q)
    assert su.rel(out.double().cpu(), want) < (1e-6 if dtype == "float32" else 5e-3)


def _paged(positions_of_segments, page_size=16, seed=0):
    """positions [n], token_segment [n], tables [segments, blocks] with pages in a shuffled order."""
    rng = np.random.default_rng(seed)
    most = max(p[-1] for p in positions_of_segments) + 1
    blocks = -(-most // page_size)
    pages = rng.permutation(len(positions_of_segments) * blocks + 2)
    tables = pages[:len(positions_of_segments) * blocks].reshape(len(positions_of_segments), blocks)
    pos = np.concatenate(positions_of_segments)
    seg = np.concatenate([np.full(len(p), s) for s, p in enumerate(positions_of_segments)])
    return i32(pos), i32(seg), i32(tables), len(pages)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("chunk,H,G,D,half", [(24, 4, 2, 16, 4), (70, 3, 3, 20, 10), (0, 2, 1, 8, 0)])
def test_mixed_attention_kernels_with_a_key_that_stands_out(dtype, chunk, H, G, D, half):
    """One key far back in the query's chunk, one just outside it and the chunk's first and last keys are
    made to stand out (their key and the queries behind them scaled up): a kernel that loses a far key,
    reads one key too many at the chunk's edge or one too few shows.  The cache is written in portions
    (one of them two tokens) and the last tokens one by one."""
    from hfee_amd.kernels import ops
    from hfee_amd.parts.rotary import rope_frequencies
    dt, T, page = DT[dtype], 150, 16
    g = torch.Generator().manual_seed(chunk + H)
    size = chunk or T
    q = torch.randn(T, H, D, generator=g)
    k = torch.randn(T, G, D, generator=g)
    last = T - 1
    first = last // size * size
    marked = [first, max(first - 1, 0), first + 1, last, 2]
    for j in marked:
        k[j] *= 3.0
    q[last] = k[marked[0]].repeat_interleave(H // G, dim=0) * 1.5 + q[last] * 0.1      # looks at its chunk's first key
    if first > 0:
        q[last - 1] = k[first - 1].repeat_interleave(H // G, dim=0) * 1.5                  # looks just outside: must not see it
    q, k = q.to(dt), k.to(dt)
    talk = torch.eye(H) + torch.randn(H, H, generator=g) * 0.3
    m = {"heads": H, "kv_heads": G, "dim": D, "scale": 0.3, "mask": {"size": size}, "rot": {"dims": 2 * half, "base": 100.0}}
    # the plain mixer with identity projections: its input is [q | k]
    hidden = (H + G) * D
    w = {"m.q": torch.eye(hidden)[:H * D], "m.k": torch.eye(hidden)[H * D:], "m.talk": talk, "m.o": torch.eye(H * D)}
    want = ps.chunked_talking_attention(torch.cat([q.reshape(T, -1), k.reshape(T, -1)], dim=1).double(),
                                        {n: t.double() for n, t in w.items()}, "m.", m, 1e-6)
    inv = rope_frequencies(2 * half, 100.0) if half else np.zeros(0)
    ang = np.arange(T)[:, None] * inv[None, :]
    cos, sin = (dev(np.cos(ang), torch.float32), dev(np.sin(ang), torch.float32)) if half else (None, None)
    got = torch.zeros(T, H * D, dtype=dt, device="cuda")
    cuts = [0, 37, 39, 100, 140] + list(range(141, T + 1))
    pos_all, seg_all, tables, pages = _paged([np.arange(T)], page, seed=1)
    cache = torch.full((pages, G, page * 2 * D), float("nan"), dtype=dt, device="cuda")
    for lo, hi in zip(cuts[:-1], cuts[1:]):
        qs, ks = q[lo:hi].reshape(hi - lo, -1).cuda().contiguous(), k[lo:hi].reshape(hi - lo, -1).cuda().contiguous()
        pos, seg = pos_all[lo:hi].contiguous(), seg_all[lo:hi].contiguous()
        ops.attention_mix_prepare(qs, ks, pos, seg, tables, cos, sin, cache, H, G, D, page, hi - 1, norm=True, eps=1e-6)
        out = torch.zeros(hi - lo, H * D, dtype=dt, device="cuda")
        ops.attention_mix(out, qs, cache, pos, seg, tables, H, G, D, page, 0.3, mix=talk.cuda(), chunk=chunk, sink="zero")
        got[lo:hi] = out
    tol = 3e-5 if dtype == "float32" else 3e-2
    assert su.rel(got.double().cpu(), want) < tol
    for t in (last, last - 1, first, min(first + 1, last)):
        assert su.rel(got[t].double().cpu(), want[t]) < tol, f"token {t}"


@pytest.mark.parametrize("chunk,H,G,D,half", [(24, 4, 2, 32, 8), (70, 8, 2, 64, 16), (0, 4, 4, 32, 0), (16, 8, 8, 32, 16)])
def test_mixed_attention_on_the_matrix_cores(chunk, H, G, D, half):
    """The matrix-core kernel against the plain mixer in float64 and against the plain kernel, with keys
    that stand out at the chunk's first and last place and just outside it; the sequence comes in
    portions whose items end at every chunk's edge, then token by token, beside a second sequence."""
    from hfee_amd.kernels import ops
    from hfee_amd.parts.rotary import rope_frequencies
    T, page = 150, 16
    g = torch.Generator().manual_seed(chunk + H)
    size = chunk or T
    q = torch.randn(2, T, H, D, generator=g)
    k = torch.randn(2, T, G, D, generator=g)
    last = T - 1
    first = last // size * size
    for j in (first, max(first - 1, 0), min(first + 1, last), last, 2):
        k[:, j] *= 3.0
    q[0, last] = k[0, first].repeat_interleave(H // G, dim=0) * 1.5 + q[0, last] * 0.1
    if first > 0:
        q[0, last - 1] = k[0, first - 1].repeat_interleave(H // G, dim=0) * 1.5
    q, k = q.bfloat16(), k.bfloat16()
    talk = torch.eye(H) + torch.randn(H, H, generator=g) * 0.3
    m = {"heads": H, "kv_heads": G, "dim": D, "scale": 0.3, "mask": {"size": size}, "rot": {"dims": 2 * half, "base": 100.0}}
    hidden = (H + G) * D
    w = {"m.q": torch.eye(hidden)[:H * D].double(), "m.k": torch.eye(hidden)[H * D:].double(), "m.talk": talk.double(),
         "m.o": torch.eye(H * D).double()}
    want = [ps.chunked_talking_attention(torch.cat([q[s].reshape(T, -1), k[s].reshape(T, -1)], dim=1).double(), w, "m.", m, 1e-6)
            for s in range(2)]
    inv = rope_frequencies(2 * half, 100.0) if half else np.zeros(0)
    ang = np.arange(T)[:, None] * inv[None, :]
    cos, sin = (dev(np.cos(ang), torch.float32), dev(np.sin(ang), torch.float32)) if half else (None, None)
    _, _, tables, pages = _paged([np.arange(T), np.arange(T)], page, seed=2)
    cache = torch.zeros((pages, G, page * 2 * D), dtype=torch.bfloat16, device="cuda")
    got = torch.zeros(2, T, H * D, dtype=torch.bfloat16, device="cuda")
    plain = torch.zeros(2, T, H * D, dtype=torch.bfloat16, device="cuda")
    fed = [0, 0]
    steps = [(37, 5), (2, 60), (61, 0), (40, 45), (0, 30)] + [(1, 1)] * 10
    for sizes in steps:
        segs = [(s, n) for s, n in enumerate(sizes) if n]
        pos = np.concatenate([np.arange(fed[s], fed[s] + n) for s, n in segs])
        seg = np.concatenate([np.full(n, s) for s, n in segs])        # (the block table's row is the sequence)
        qs = torch.cat([q[s, fed[s]:fed[s] + n].reshape(n, -1) for s, n in segs]).cuda().contiguous()
        ks = torch.cat([k[s, fed[s]:fed[s] + n].reshape(n, -1) for s, n in segs]).cuda().contiguous()
        ops.attention_mix_prepare(qs, ks, i32(pos), i32(seg), tables, cos, sin, cache, H, G, D, page, int(pos.max()),
                                  norm=True, eps=1e-6)
        items, row = [], 0
        for s, n in segs:
            off = 0
            while off < n:
                p = fed[s] + off
                room = min(16, n - off, (chunk - p % chunk) if chunk else 16)
                items.append((row + off, room, p, s))
                off += room
            row += n
        out = torch.zeros(len(pos), H * D, dtype=torch.bfloat16, device="cuda")
        splits = 1 + len(pos) % 4                      # (the key tiles of an item over one to four workgroups)
        partial = torch.full((ops.attention_mix_partial_words(len(items), H, D, splits),), float("nan"), device="cuda")
        ops.attention_mix_bf16(out, qs, cache, i32(np.asarray(items).reshape(-1, 4)), tables, H, G, D, page, 0.3,
                               mix_t=talk.t().contiguous().cuda(), chunk=chunk, sink="zero", splits=splits,
                               partial=partial if splits > 1 else None)
        ref = torch.zeros_like(out)
        ops.attention_mix(ref, qs, cache, i32(pos), i32(seg), tables, H, G, D, page, 0.3, mix=talk.cuda(), chunk=chunk, sink="zero")
        row = 0
        for s, n in segs:
            got[s, fed[s]:fed[s] + n] = out[row:row + n]
            plain[s, fed[s]:fed[s] + n] = ref[row:row + n]
            row += n
            fed[s] += n
    assert fed == [T, T]
    for s in range(2):
        assert su.rel(plain[s].double().cpu(), want[s]) < 3e-2
        assert su.rel(got[s].double().cpu(), want[s]) < 3e-2
        assert su.rel(got[s].double().cpu(), plain[s].double().cpu()) < 2e-2
        for t in (last, last - 1, first, min(first + 1, last), 0, 1, 15, 16, 17):
            assert su.rel(got[s, t].double().cpu(), want[s][t]) < 3e-2, f"sequence {s} token {t}"


@pytest.mark.parametrize("H,G,D", [(8, 2, 64), (16, 4, 128), (32, 8, 128), (8, 8, 64), (12, 3, 32), (24, 6, 64), (40, 10, 32),
                                   (40, 40, 64), (32, 8, 64), (32, 32, 128), (64, 16, 64), (64, 64, 64)])
def test_mixed_attention_over_several_workgroups(H, G, D):
    """Items of unequal lengths whole and over several workgroups, some without a tile, against the plain kernel (bfloat16
    results of the same inputs: a few rounding steps of 2^-9); four, eight and other numbers of heads a wave, mixed on the matrix
    unit or the vector units, queries in registers, in LDS or read again, keys and values early or late.  The chunk begins inside a
    tile.  (64 heads are mixed within each half of them: the plain kernel takes the halves one by one.)"""
    from hfee_amd.kernels import ops
    page, chunk, starts, counts = 16, 88, (0, 100, 89, 263), (70, 30, 1, 1)
    g = torch.Generator().manual_seed(H)
    pages = [-(-(a + n) // page) for a, n in zip(starts, counts)]
    tables = torch.zeros(len(starts), max(pages), dtype=torch.int32)
    order, at = torch.randperm(sum(pages), generator=g), 0
    for s, n in enumerate(pages):
        tables[s, :n] = order[at:at + n]
        at += n
    tables = tables.cuda()
    cache = torch.randn(sum(pages), G, page * 2 * D, generator=g).bfloat16().cuda()
    q = (torch.randn(sum(counts), H * D, generator=g) * 2).bfloat16().cuda()
    halves = 2 if H == 64 else 1
    h, k = H // halves, G // halves
    talk = torch.block_diag(*(torch.eye(h) + torch.randn(h, h, generator=g) * 0.2 for _ in range(halves))).cuda()
    items, row = [], 0
    for s, (start, n) in enumerate(zip(starts, counts)):
        off = 0
        while off < n:
            p = start + off
            room = min(16, n - off, chunk - p % chunk)
            items.append((row + off, room, p, s))
            off += room
        row += n
    i32 = lambda a: torch.as_tensor(np.asarray(a), dtype=torch.int32, device="cuda")      # noqa: E731
    pos = np.concatenate([np.arange(a, a + n) for a, n in zip(starts, counts)])
    want = torch.zeros_like(q)
    kw = dict(chunk=chunk, sink="zero")
    for i in range(halves):
        mine, heads = torch.zeros_like(q[:, :h * D]).contiguous(), slice(i * h, (i + 1) * h)
        ops.attention_mix(mine, q[:, i * h * D:(i + 1) * h * D].contiguous(), cache[:, i * k:(i + 1) * k].contiguous(), i32(pos),
                          i32(np.repeat(np.arange(4), counts)), tables, h, k, D, page, D ** -0.5, mix=talk[heads, heads].contiguous(), **kw)
        want[:, i * h * D:(i + 1) * h * D] = mine
    for splits in (1, 2, 3, 16):
        partial = torch.full((max(1, ops.attention_mix_partial_words(len(items), H, D, splits)),), float("nan"), device="cuda")
        got = torch.full_like(q, float("nan"))
        ops.attention_mix_bf16(got, q, cache, i32(items), tables, H, G, D, page, D ** -0.5, mix_t=talk.t().contiguous(),
                               splits=splits, partial=partial if splits > 1 else None, **kw)
        for t in range(len(pos)):
            assert su.rel(got[t].double().cpu(), want[t].double().cpu()) < 1e-2, f"row {t} over {splits} workgroups"


@pytest.mark.parametrize("H,G,D", [(16, 4, 128), (32, 8, 64), (64, 16, 64)])
def test_mixing_on_the_matrix_unit_adds_as_the_vector_units_do(H, G, D, monkeypatch):
    """Four and eight heads of a wave mixed by the matrix unit give to the bit what the vector units give: the same
    multiply-adds in the order of the heads."""
    from hfee_amd.kernels import lib, ops
    page, n, g = 16, 75, torch.Generator().manual_seed(H)
    table = torch.randperm(-(-n // page), generator=g).to(torch.int32).cuda()[None]
    cache = torch.randn(table.numel(), G, page * 2 * D, generator=g).bfloat16().cuda()
    q = (torch.randn(n, H * D, generator=g) * 3).bfloat16().cuda()
    talk = torch.randn(H, H, generator=g).cuda()
    items = i32([[p, min(16, n - p), p, 0] for p in range(0, n, 16)])
    results = []
    for kernels in (lib.attention_mix_bf16, lambda h, k, d: lib.load(f"attention_mix_bf16_h{h}_g{k}_d{d}_vectors")):
        monkeypatch.setattr(lib, "attention_mix_bf16", kernels)
        out = torch.full_like(q, float("nan"))
        ops.attention_mix_bf16(out, q, cache, items, table, H, G, D, page, D ** -0.5, mix_t=talk, sink="zero")
        results.append(out)
    assert torch.equal(*results) and bool(torch.isfinite(results[0]).all())


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("lengths", [(1,), (1, 1, 1), (9, 1, 2), (70, 17), (2755, 17, 3)])
@pytest.mark.parametrize("D", [4, 32, 128, 256])
def test_inputs_with_decays_a_channel_in_one_launch(dtype, lengths, D):
    """Decays a channel beside the convolution, the unit vectors and the strengths, to the bit what a launch a mechanism gives
    (values by one, as odd widths have them); a token a workgroup, and of the many tokens eight."""
    from hfee_amd.kernels import ops
    dt = getattr(torch, dtype)
    H, G, V, K = 6, 2, 24, 4
    qk, C, n = G * D, 2 * G * D + H * V, sum(lengths)
    assert ops.delta_inputs_fit(C, D, K)
    g = torch.Generator().manual_seed(n)
    rand = lambda *shape: torch.randn(*shape, generator=g).cuda()      # noqa: E731
    proj = rand(n, C + 8).to(dt)
    x, b = proj[:, :C], proj[:, C:C + H]
    step, taps, state = rand(n, H * D).to(dt), rand(C, K), rand(5, K - 1, C).to(dt)
    bias, a_log = rand(H * D), rand(H)
    i32 = lambda a: torch.tensor(a, dtype=torch.int32, device="cuda")      # noqa: E731
    rows, lens, slots = i32(np.cumsum((0,) + lengths)[:-1].tolist()), i32(lengths), i32([4, 1, 2][:len(lengths)])
    seg = i32(np.repeat(np.arange(len(lengths)), lengths).tolist())
    want, states = torch.zeros(n, C, device="cuda"), [state.clone(), state.clone()]
    ops.short_conv_silu(want, x, states[0], taps, seg, rows, slots)
    ops.short_conv_keep(states[0], x, rows, lens, slots)
    ops.unit_heads(want[:, :qk], G, D, 1e-6, 0.5)
    ops.unit_heads(want[:, qk:2 * qk], G, D, 1e-6, 1.0)
    wide = torch.zeros(n, H * D + 1, device="cuda")[:, :H * D]      # (rows that are no aligned fours: a value a thread)
    beta = torch.zeros(n, H, device="cuda")
    ops.scan_gate(wide, step, "step_decay", bias=bias, per_head=a_log, head_width=D)
    ops.scan_gate(beta, b, "sigmoid")
    got, decay, strength = torch.zeros(n, C, device="cuda"), torch.zeros(n, H * D, device="cuda"), torch.zeros(n, H, device="cuda")
    singles = max(lengths) == 1
    ops.delta_inputs(got, decay, strength, x, step, b, states[1], taps, bias, a_log, seg, rows, slots, qk, D, H, 1e-6, 0.5, keep=singles)
    if not singles:
        ops.short_conv_keep(states[1], x, rows, lens, slots)
    assert torch.equal(decay, wide) and torch.equal(strength, beta) and torch.equal(states[0], states[1])
    assert torch.equal(got, want)
    for kind, kw in (("cast", dict(number=0.3, first_columns=D + 1)), ("silu", {}), ("root_sigmoid", dict(number=16.0, bias=bias)), ("softplus", {})):
        fours = torch.zeros(n, H * D, device="cuda")
        ops.scan_gate(fours, step, kind, **kw)
        ops.scan_gate(wide, step, kind, **kw)
        assert torch.equal(fours, wide), kind


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("n,width", [(512, 4096), (2049, 1028)])
def test_gates_of_many_values_in_fours(dtype, n, width):
    """Four values a thread give what one gives (rows that are no aligned fours go one by one), through every function."""
    from hfee_amd.kernels import ops
    g = torch.Generator(device="cuda").manual_seed(n)
    z = (torch.randn(n, width, device="cuda", generator=g) * 4).to(getattr(torch, dtype))
    bias, a_log = torch.randn(width, device="cuda", generator=g), torch.randn(width // 4, device="cuda", generator=g)
    for kind, kw in (("cast", dict(number=0.3, first_columns=width // 2 + 1)), ("silu", {}), ("sigmoid", {}), ("softplus", dict(bias=bias)),
                     ("root_sigmoid", dict(number=16.0, bias=bias)), ("step_decay", dict(bias=bias, per_head=a_log, head_width=4))):
        fours, ones = torch.zeros(n, width, device="cuda"), torch.zeros(n, width + 1, device="cuda")[:, :width]
        ops.scan_gate(fours, z, kind, **kw)
        ops.scan_gate(ones, z, kind, **kw)
        assert torch.equal(fours, ones) and int((fours != 0).sum()) > n * width // 2, kind


@pytest.mark.parametrize("per_channel", [True, False])
@pytest.mark.parametrize("at", [0, 1, 2, 7])
def test_inputs_whose_bias_begins_at_any_number(at, per_channel):
    """The decays' bias is a model's own tensor, which may be a view of a larger one: where it begins moves no bit."""
    from hfee_amd.kernels import ops
    H, D, n, K = 6, 16, 5, 4
    C, W, g = 3 * H * D, H * D if per_channel else H, torch.Generator().manual_seed(at)
    rand = lambda *shape: torch.randn(*shape, generator=g).cuda()      # noqa: E731
    proj, step, taps, a_log = rand(n, C + 8), rand(n, W), rand(C, K), rand(H)
    bias, held = rand(W), torch.full((W + 8,), float("nan"), device="cuda")
    held[at:at + W] = bias
    decays = []
    for b in (bias, held[at:at + W]):
        y, decay, beta = (torch.full((n, w), float("nan"), device="cuda") for w in (C, W, H))
        ops.delta_inputs(y, decay, beta, proj[:, :C], step, proj[:, C:C + H], torch.zeros(2, K - 1, C, device="cuda"), taps, b, a_log,
                         i32([0] * n), i32([0]), i32([1]), H * D, D, H, 1e-6, 0.5, keep=False)
        decays.append(decay)
    assert torch.equal(*decays) and bool(torch.isfinite(decays[0]).all())


@pytest.mark.parametrize("rule", ["delta", "decay_add"])
@pytest.mark.parametrize("H,G,D,V", [(4, 2, 8, 16), (3, 3, 20, 12), (2, 1, 33, 70)])
def test_linear_scan_in_portions(rule, H, G, D, V):
    """The recurrence by its definition, token by token in float64, against the kernel fed the same
    sequence in portions of unequal size for two requests side by side in other slots."""
    from hfee_amd.kernels import ops
    if rule == "decay_add":
        G = H
    g = torch.Generator().manual_seed(D)
    T = [45, 23]
    data = []
    for t in T:
        q, k = torch.randn(t, G, D, generator=g) * 0.4, torch.randn(t, G, D, generator=g) * 0.4
        v = torch.randn(t, H, V, generator=g)
        a = torch.rand(t, H, D, generator=g) * 0.3 + 0.7
        b = torch.rand(t, H, generator=g)
        data.append((q, k, v, a, b))
    want, final = [], []
    for q, k, v, a, b in data:
        o = torch.zeros(q.shape[0], H, V, dtype=torch.float64)
        final.append([])
        for h in range(H):
            S = torch.zeros(D, V, dtype=torch.float64)
            for t in range(q.shape[0]):
                qt, kt = q[t, h // (H // G)].double(), k[t, h // (H // G)].double()
                S = a[t, h].double()[:, None] * S
                u = b[t, h].double() * (v[t, h].double() - S.T @ kt) if rule == "delta" else v[t, h].double()
                S = S + kt[:, None] * u[None, :]
                o[t, h] = S.T @ qt
            final[-1].append(S)
        want.append(o.reshape(q.shape[0], -1))
    state = torch.zeros(5, H, *ops.scan_state_shape(D, V), device="cuda")
    state[1].fill_(float("nan"))                    # a slot that nobody uses
    slots = [3, 0]
    fed = [0, 0]
    got = [torch.zeros(t, H * V) for t in T]
    for sizes in ([7, 2], [1, 1], [20, 0], [2, 13], [15, 7]):
        segs = [(s, n) for s, n in enumerate(sizes) if n]
        parts = [tuple(x[fed[s]:fed[s] + n] for x in data[s]) for s, n in segs]
        cat = [torch.cat([p[i].reshape(p[i].shape[0], -1) for p in parts]).cuda().contiguous() for i in range(5)]
        rows = np.cumsum([0] + [n for _, n in segs])[:-1]
        out = torch.zeros(sum(n for _, n in segs), H * V, device="cuda")
        ops.linear_scan(out, state, cat[0], cat[1], cat[2], cat[3], cat[4] if rule == "delta" else None, i32(rows),
                        i32([n for _, n in segs]), i32([slots[s] for s, _ in segs]), H, G, D, V, rule)
        for (s, n), r in zip(segs, rows):
            got[s][fed[s]:fed[s] + n] = out[r:r + n].cpu()
            fed[s] += n
    assert fed == T
    for s in range(2):
        assert su.rel(got[s], want[s]) < 2e-5
        assert su.rel(ops.scan_state_matrix(state[slots[s]], D, V).cpu(), torch.stack(final[s])) < 2e-5
    assert bool(torch.isnan(state[1]).all()) and float(state[2].abs().sum()) == 0.0


@pytest.mark.parametrize("rule", ["delta", "decay_add", "scaled_add"])
@pytest.mark.parametrize("D,V,pad", [(64, 20, 0), (128, 17, 4), (128, 32, 1), (256, 16, 0), (512, 8, 4)])
def test_linear_scan_around_its_blocks(rule, D, V, pad):
    """Key sizes that fill a lane's rows, whose numbers come in loads of sixteen bytes (rows padded by a multiple of four
    numbers) or one by one (padded by one), portions that end in front of, on and behind a block of tokens and of
    blocks, then steps of single tokens, against the recurrence in float64."""
    from hfee_amd.kernels import ops
    H, G, block = 2, (2 if rule == "decay_add" else 1), 16 if D <= 128 else 8 if D == 256 else 4
    T = [1, block - 1, block, block + 1, 2 * block, 3 * block + 1]
    singles, g = 2, torch.Generator().manual_seed(D + V)
    slots = [3, 0, 5, 1, 6, 2]
    state = torch.zeros(7, H, *ops.scan_state_shape(D, V), device="cuda")
    want_S = torch.zeros(len(T), H, D, V, dtype=torch.float64)

    def step(lengths):
        n = sum(lengths)
        q, k = torch.randn(n, G, D, generator=g) * D ** -0.5, torch.randn(n, G, D, generator=g) * D ** -0.5
        v, a, b = torch.randn(n, H, V, generator=g), torch.rand(n, H, D, generator=g) * 0.3 + 0.7, torch.rand(n, H, generator=g)
        want = torch.zeros(n, H, V, dtype=torch.float64)
        rows = np.cumsum([0] + lengths)[:-1]
        for s, (row, length) in enumerate(zip(rows, lengths)):
            for h in range(H):
                S = want_S[s, h]
                for t in range(row, row + length):
                    qt, kt, vt = q[t, h * G // H].double(), k[t, h * G // H].double(), v[t, h].double()
                    S = a[t, h].double()[:, None] * S
                    u = {"delta": lambda: b[t, h].double() * (vt - S.T @ kt), "decay_add": lambda: vt,
                         "scaled_add": lambda: b[t, h].double() * vt}[rule]()
                    S = S + kt[:, None] * u[None, :]
                    want[t, h] = S.T @ qt
                want_S[s, h] = S

        def rows_of(x):          # rows that begin `pad` numbers apart from where they end
            wide = torch.full((n, x[0].numel() + pad), float("nan"), device="cuda")
            wide[:, :x[0].numel()] = x.reshape(n, -1).cuda()
            return wide[:, :x[0].numel()]
        out = torch.full((n, H * V + pad), float("nan"), device="cuda")[:, :H * V]
        ops.linear_scan(out, state, rows_of(q), rows_of(k), rows_of(v), rows_of(a), b.cuda() if rule != "decay_add" else None,
                        i32(rows), i32(lengths), i32(slots), H, G, D, V, rule, singles=max(lengths) == 1)
        assert su.rel(out.cpu(), want.reshape(n, -1)) < 2e-5

    for lengths in [T] + [[1] * len(T)] * singles + [T[::-1]]:
        step(list(lengths))
    for s, slot in enumerate(slots):
        assert su.rel(ops.scan_state_matrix(state[slot], D, V).cpu(), want_S[s]) < 2e-5
    assert float(state[4].abs().sum()) == 0.0


@pytest.mark.parametrize("rule", ["delta", "decay_add", "scaled_add"])
@pytest.mark.parametrize("D", [12, 20, 64, 96, 128, 256, 400, 512])
def test_linear_scan_with_a_decay_a_head(rule, D):
    """One decay a head, of each token or the same for all, gives to the bit what it gives spelled out a channel: portions of a
    few tokens, which are one block and ask for none behind it, and around the blocks of every key size."""
    from hfee_amd.kernels import ops
    H, V, block = 2, 20, 16 if D <= 128 else 8 if D <= 256 else 4
    lengths = [2, 3, block - 1, block, block + 1, 2 * block + 3, 1]
    G, n, g = (H if rule == "decay_add" else 1), sum(lengths), torch.Generator().manual_seed(D)
    rand = lambda *shape: torch.randn(*shape, generator=g).cuda()      # noqa: E731
    q, k, v, b = rand(n, G * D) * D ** -0.5, rand(n, G * D) * D ** -0.5, rand(n, H * V), rand(n, H).sigmoid()
    start = rand(len(lengths) + 1, H, *ops.scan_state_shape(D, V))
    rows, lens, slots = i32(np.cumsum([0] + lengths)[:-1]), i32(lengths), i32([3, 0, 5, 1, 6, 2, 7])
    for a in (rand(n, H).sigmoid(), rand(H).sigmoid()):
        got = []
        for decay, per_head in ((a, True), (a.expand(n, H).repeat_interleave(D, 1).contiguous(), False)):
            state, out = start.clone(), torch.full((n, H * V), float("nan"), device="cuda")
            ops.linear_scan(out, state, q, k, v, decay, None if rule == "decay_add" else b, rows, lens, slots, H, G, D, V, rule,
                            decay_per_head=per_head)
            got.append((out, state))
        assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
        assert bool(torch.isfinite(got[0][0]).all()) and torch.equal(got[0][1][4], start[4])


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("K", [1, 2, 4, 5])
def test_short_convolution_carries_its_inputs(dtype, K):
    from hfee_amd.kernels import ops
    dt = DT[dtype]
    g = torch.Generator().manual_seed(K)
    C, T = 37, 30
    x = torch.randn(T, C, generator=g).to(dt)
    taps = torch.randn(C, K, generator=g)
    want = ps.short_conv_silu(x.double(), taps.double())
    state = torch.zeros(3, K - 1, C, dtype=dt, device="cuda")
    got = torch.zeros(T, C)
    at = 0
    for n in (1, 1, 2, 9, 1, 3, 13):       # (portions shorter than the taps keep a part of the old state)
        xs = x[at:at + n].cuda().contiguous()
        y = torch.zeros(n, C, device="cuda")
        ops.short_conv_silu(y, xs, state, taps.cuda(), i32([0] * n), i32([0]), i32([2]))
        ops.short_conv_keep(state, xs, i32([0]), i32([n]), i32([2]))
        got[at:at + n] = y.cpu()
        at += n
    assert at == T and su.rel(got, want) < 2e-6
    assert float(state[:2].abs().sum()) == 0.0


@pytest.mark.parametrize("users,width,ff", [((1, 2, 3, 4, 5, 9), 64, 50), ((64,), 520, 16), ((0, 7, 0, 1), 1032, 33)])
@pytest.mark.parametrize("numbers", [None, (7.0, 1.702)])
def test_few_tokens_expert_by_expert(users, width, ff, numbers):
    """The first product of up to 64 (token, expert) pairs, an expert's rows once for all its tokens: every number of
    tokens that are taken together, rows that fill no block, and pairs whose expert number stands for no matrix, whose
    rows stay as they were.  Against float64: an activation is off by half a bfloat16 ulp and its sums' roundings."""
    from hfee_amd.kernels import ops
    g = torch.Generator().manual_seed(width + ff)
    E = len(users)
    chosen = torch.cat([torch.full((c,), e) for e, c in enumerate(users)] + ([] if sum(users) == 64 else [torch.full((2,), E + 1)]))
    n = len(chosen)
    chosen = chosen[torch.randperm(n, generator=g)].to(torch.int32).view(n, 1)
    rand = lambda *shape: (torch.randn(*shape, generator=g) * 0.3).to(torch.bfloat16).cuda()      # noqa: E731
    h, wg, wu = rand(n, width), rand(E, ff, width), rand(E, ff, width)
    act = torch.full((n, ff), 5.0, dtype=torch.bfloat16, device="cuda")
    ops.moe_up(act, h, wg, wu, 1, chosen=chosen.cuda(), **(dict(activation="clipped", numbers=numbers) if numbers else {}))
    for t in range(n):
        e = int(chosen[t, 0])
        if e >= E:
            assert (act[t] == 5.0).all()
            continue
        gate, up = wg[e].double() @ h[t].double(), wu[e].double() @ h[t].double()
        if numbers:
            gate, up = gate.clamp(max=numbers[0]), up.clamp(-numbers[0], numbers[0])
            want = gate * torch.sigmoid(numbers[1] * gate) * (up + 1)
        else:
            want = gate * torch.sigmoid(gate) * up
        size = (wg[e].double().abs() @ h[t].double().abs() + 1) * (wu[e].double().abs() @ h[t].double().abs() + 1)
        assert ((act[t].double() - want).abs() <= 2.0 ** -8 * want.abs() + width * 2.0 ** -23 * size).all(), t


@pytest.mark.parametrize("n,top,E,width,ff", [(1, 2, 5, 64, 40), (8, 2, 3, 70, 520), (16, 4, 9, 33, 16), (64, 1, 2, 6, 1032), (21, 3, 4, 4, 8),
                                              (1, 3, 9, 33, 16), (2, 4, 6, 70, 40), (5, 3, 20, 66, 64), (21, 3, 3, 1023, 264)])
@pytest.mark.parametrize("accumulate", [True, False])
def test_few_tokens_second_product(n, top, E, width, ff, accumulate):
    """The second product of up to 64 pairs, expert by expert: tokens that share experts and ones that name one beyond the
    last (left out), widths that fill no four.  Against float64 over the same bfloat16 numbers: a float32 sum of ff products
    a pair, added up over the pairs; and a token's numbers stay the same, bit for bit, alone."""
    from hfee_amd.kernels import ops
    g = torch.Generator().manual_seed(n * width + ff)
    chosen = torch.rand(n, E + 2, generator=g).topk(top, dim=1).indices.to(torch.int32).cuda()
    act, wd = torch.randn(n * top, ff, generator=g).bfloat16().cuda(), torch.randn(E, width, ff, generator=g).bfloat16().cuda()
    weights = torch.rand(n, top, generator=g).cuda()
    x0 = torch.randn(n, width, generator=g).cuda()

    def run(rows):
        x = x0[rows].clone()
        a = act.view(n, top, ff)[rows].reshape(-1, ff).contiguous()
        ops.moe_down(x, a, wd, top, pair_weights=weights[rows].contiguous(), chosen=chosen[rows].contiguous(), accumulate=accumulate)
        return x
    out = run(list(range(n)))
    for t in range(n):
        want, size = (x0[t].double() if accumulate else torch.zeros(width, dtype=torch.float64, device="cuda")), x0[t].double().abs()
        for j in range(top):
            e = int(chosen[t, j])
            if e < E:
                want = want + weights[t, j].double() * (wd[e].double() @ act[t * top + j].double())
                size = size + wd[e].double().abs() @ act[t * top + j].double().abs()
        assert ((out[t].double() - want).abs() <= (ff / 32 + 24) * 2.0 ** -24 * size).all(), t
    assert torch.equal(run([n - 1])[0], out[n - 1])


@pytest.mark.parametrize("n,top,E,width,ff", [(5, 1, 48, 96, 64), (6, 1, 47, 96, 64), (2, 1, 16, 4100, 16), (7, 1, 7, 2500, 24),
                                              (8, 8, 300, 1100, 40), (3, 2, 300, 4096, 8), (64, 1, 300, 64, 64),
                                              (2, 4, 6, 72, 40), (5, 3, 20, 64, 64), (40, 1, 2, 4096, 512), (64, 1, 64, 2048, 520),
                                              (21, 3, 3, 1024, 264), (12, 1, 4, 8192, 16), (2, 2, 16, 64, 4096), (17, 1, 2, 64, 64)])
def test_few_tokens_have_the_same_bits_alone(n, top, E, width, ff):
    """Every reason for which a second product goes expert by expert, with four, eight and sixteen waves a workgroup, and sizes
    for which it goes token by token; groups of one to four pairs of an expert and several groups of one; more experts than
    pairs, among them numbers that stand for none; many pairs of next to no work: what a token alone gives, bit for bit."""
    from hfee_amd.kernels import ops
    g = torch.Generator().manual_seed(n * E)
    rand = lambda *shape: (torch.randn(*shape, generator=g) * shape[-1] ** -0.5).to(torch.bfloat16).cuda()      # noqa: E731
    h, wg, wu, wd = rand(n, width) * 16, rand(E, ff, width), rand(E, ff, width), rand(E, width, ff)
    chosen = torch.stack([torch.randperm(E + 1, generator=g)[:top] for _ in range(n)]).to(torch.int32).cuda()     # (E: no expert)
    weights = torch.rand(n, top, generator=g).cuda()

    def run(rows):
        act = torch.zeros(len(rows) * top, ff, dtype=torch.bfloat16, device="cuda")
        x = torch.ones(len(rows), width, device="cuda")
        some = chosen[rows].contiguous()
        ops.moe_up(act, h[rows].contiguous(), wg, wu, top, chosen=some)
        ops.moe_down(x, act, wd, top, pair_weights=weights[rows].contiguous(), chosen=some)
        return act.view(len(rows), top, ff), x
    act, x = run(list(range(n)))
    assert float(act.float().std()) > 0 and float(x.std()) > 0
    for t in range(n):
        one_act, one_x = run([t])
        assert torch.equal(one_act[0], act[t]) and torch.equal(one_x[0], x[t])


@pytest.mark.parametrize("counts,width,ff", [((1, 0, 64, 65, 128, 129, 300), 128, 192), ((16, 17, 0, 2), 64, 64), ((100, 30), 64, 128),
                                             ((129, 63), 256, 64), ((700, 300), 64, 64),
                                             ((200, 3), 576, 320), ((70, 129, 31), 96, 160)])
@pytest.mark.parametrize("gated", [True, False])
def test_grouped_experts_at_the_edges_of_their_tiles(counts, width, ff, gated):
    """Tiles of up to 128 pairs and 256 weight rows (sizes in multiples of 64; the last sizes go through the tiles of 64
    pairs): experts with none, one, a tile's and a tile's and one more pairs, rows that fill no block, a single step of
    K.  Against the sums in float64 over the bfloat16 operands and activations: a float32 sum of K products is off by at
    most K roundings of its terms' sizes, an activation by half a bfloat16 ulp more.  A pair's numbers stay the same,
    bit for bit, among fewer pairs."""
    from hfee_amd.kernels import ops
    g = torch.Generator().manual_seed(sum(counts) + width)
    E, n = len(counts), sum(counts)
    chosen = torch.cat([torch.full((c,), e) for e, c in enumerate(counts)])[torch.randperm(n, generator=g)].to(torch.int32).view(n, 1)
    rand = lambda *shape: (torch.randn(*shape, generator=g) * shape[-1] ** -0.5).to(torch.bfloat16).cuda()      # noqa: E731
    h, wg, wu, wd = rand(n, width) * width ** 0.5, rand(E, ff, width), rand(E, ff, width), rand(E, width, ff)
    h = h.to(torch.bfloat16)

    def run(rows):
        m = len(rows)
        order = torch.zeros(m, dtype=torch.int32, device="cuda")
        tiles = torch.zeros(3 * ops.moe_group_tiles(m, 1, E) + 1, dtype=torch.int32, device="cuda")
        act = torch.zeros(m, ff, dtype=torch.bfloat16, device="cuda")
        y = torch.full((m, width), 7.0, dtype=torch.float32, device="cuda")
        ops.moe_grouped(None, h[rows].contiguous(), wg if gated else None, wu, wd, 1, order, tiles, act, y, chosen=chosen[rows.cpu()].cuda())
        return act, y
    everything = torch.arange(n, device="cuda")
    act, y = run(everything)
    e = chosen.view(-1).long().cuda()
    up = torch.einsum("nfw,nw->nf", wu[e].double(), h.double())
    if gated:
        gate = torch.einsum("nfw,nw->nf", wg[e].double(), h.double())
        want = gate / (1 + torch.exp(-gate)) * up
    else:
        want = torch.relu(up) ** 2
    assert ((act.double() - want).abs() <= 2.0 ** -8 * want.abs() + width * 2.0 ** -24 * 30).all()
    down = torch.einsum("nwf,nf->nw", wd[e].double(), act.double())
    size = torch.einsum("nwf,nf->nw", wd[e].double().abs(), act.double().abs())
    assert ((y.double() - down).abs() <= (ff + 2) * 2.0 ** -24 * size).all()
    some = everything[::3]
    act2, y2 = run(some)
    assert torch.equal(act2, act[some]) and torch.equal(y2, y[some])


@pytest.mark.parametrize("E,width,ff,gated", [(24, 1344, 1472, True), (24, 1344, 2944, False), (186, 128, 64, True), (186, 192, 192, False),
                                              (330, 128, 64, True), (330, 192, 192, False)])
def test_grouped_experts_with_many_pairs_each(E, width, ff, gated):
    """Enough tiles to fill the GPU with up to 192 pairs each (the last two: 128), at every number of 32s of them and at the edges
    between, of which one and two tiles and more are made; two, four, six and many steps of K.  Every value against the sums in float64 (a float32 sum
    of K products is off by at most K roundings of its terms' sizes, an activation by half a bfloat16 ulp more); a pair's numbers
    stay the same, bit for bit, where few others have its expert."""
    from hfee_amd.kernels import ops
    g = torch.Generator().manual_seed(width)
    edges = (129, 160, 161, 192, 193, 224, 225, 256, 257, 383, 384, 385, 96, 97, 128, 65, 64, 33, 32, 1, 0, 150, 180, 190)
    counts = [edges[e % len(edges)] for e in range(E)]
    n = sum(counts)
    chosen = torch.cat([torch.full((c,), e) for e, c in enumerate(counts)])[torch.randperm(n, generator=g)].to(torch.int32).view(n, 1).cuda()
    gen = torch.Generator(device="cuda").manual_seed(ff)
    rand = lambda *shape: (torch.randn(*shape, generator=gen, device="cuda") * shape[-1] ** -0.5).to(torch.bfloat16)      # noqa: E731
    h, wg, wu, wd = (rand(n, width).float() * width ** 0.5).to(torch.bfloat16), rand(E, ff, width), rand(E, ff, width), rand(E, width, ff)

    def run(rows):
        m = len(rows)
        order = torch.zeros(m, dtype=torch.int32, device="cuda")
        tiles = torch.zeros(3 * ops.moe_group_tiles(m, 1, E) + 1, dtype=torch.int32, device="cuda")
        act = torch.zeros(m, ff, dtype=torch.bfloat16, device="cuda")
        y = torch.full((m, width), 7.0, dtype=torch.float32, device="cuda")
        ops.moe_grouped(None, h[rows].contiguous(), wg if gated else None, wu, wd, 1, order, tiles, act, y, chosen=chosen[rows].contiguous())
        return act, y, tiles
    everything = torch.arange(n, device="cuda")
    act, y, tiles = run(everything)
    most = 3 * ((n + 127) // 128 + E)
    assert int(tiles[:most].view(-1, 3)[:int(tiles[most]), 2].max()) == (128 if E == 330 else 192)
    for e in range(min(E, len(edges))):
        at = (chosen.view(-1) == e).nonzero().squeeze(1)
        up = h[at].double() @ wu[e].double().t().contiguous()
        gate = h[at].double() @ wg[e].double().t().contiguous()
        want = gate / (1 + torch.exp(-gate)) * up if gated else torch.relu(up) ** 2
        assert ((act[at].double() - want).abs() <= 2.0 ** -8 * want.abs() + width * 2.0 ** -24 * 30).all()
        down = act[at].double() @ wd[e].double().t().contiguous()
        size = act[at].double().abs() @ wd[e].double().abs().t().contiguous()
        assert ((y[at].double() - down).abs() <= (ff + 2) * 2.0 ** -24 * size).all()
    some = everything[::5]
    act2, y2, _ = run(some)
    assert torch.equal(act2, act[some]) and torch.equal(y2, y[some])


@pytest.mark.parametrize("size,experts,counts", [
    (1024, 16, (192, [300] * 16)), (1024, 16, (128, [4800] + [0] * 15)), (1024, 16, (192, [0, 600] * 8)), (1024, 18, (192, [0] + [300] * 16)),
    (1024, 16, (128, [1600, 800, 530, 400, 320, 265, 228, 200, 178, 160, 145, 133, 123, 114, 106, 100])), (1024, 1, (128, [300])),
    (512, 64, (192, [300] * 64)), (512, 65, (128, [128] * 65)), (512, 65, (128, [0] * 64 + [7200])), (256, 129, (192, [0] + [300] * 128)),
    (256, 200, (192, list(range(200)))), (256, 200, (192, [3000 // (e + 1) for e in range(200)]))])
@pytest.mark.parametrize("top", [1, 3])
def test_tiles_of_grouped_experts_go_by_how_the_pairs_lie(size, experts, counts, top):
    """What the device makes of a step's pairs: every pair in the order once, among its expert's; an expert's tiles as few as their size
    allows, of whole 32s and alike; and the larger size where the rule expects it to be faster: rounds of 256 workgroups times the
    largest tile, 7 % less.  The same number of pairs spread evenly and on one expert go two ways."""
    from hfee_amd.kernels import ops
    E, width, ff, (most_pairs, counts) = experts, size, size, counts
    counts = list(counts) + [0] * (E - len(counts))
    none = -sum(counts) % top                              # (pairs of no expert)
    g = torch.Generator().manual_seed(E + top)
    flat = torch.cat([torch.full((c,), e) for e, c in enumerate(counts + [none])])
    chosen = flat[torch.randperm(len(flat), generator=g)].to(torch.int32).view(-1, top)
    n = chosen.shape[0]

    def cost(pairs):
        made = [(-(-c // pairs), -(-c // 32)) for c in counts if c]
        tiles, largest = sum(t for t, _ in made), max(2, *(-(-groups // t) for t, groups in made), 2)
        return (-(-tiles * (ff // 128) // 256) * width + -(-tiles * (width // 256) // 256) * ff) * (largest + 0.5)
    assert most_pairs == (192 if cost(192) < 0.93 * cost(128) else 128)
    h = torch.zeros(n, width, dtype=torch.bfloat16, device="cuda")
    w = torch.zeros(E, ff, width, dtype=torch.bfloat16, device="cuda")
    order = torch.full((n * top,), -1, dtype=torch.int32, device="cuda")
    tiles = torch.zeros(3 * ops.moe_group_tiles(n, top, E) + 1, dtype=torch.int32, device="cuda")
    act, y = torch.zeros(n * top, ff, dtype=torch.bfloat16, device="cuda"), torch.zeros(n * top, width, device="cuda")
    ops.moe_grouped(None, h, w, w, w, top, order, tiles, act, y, chosen=chosen.cuda())
    lie, most = tiles.tolist(), 3 * ((n * top + 127) // 128 + E)
    want, start = [], 0
    for e, count in enumerate(counts):
        n_tiles, groups, at = -(-count // most_pairs), -(-count // 32), 0
        for i in range(n_tiles):
            mine = min(32 * (groups // n_tiles + (i < groups % n_tiles)), count - at)
            want.append((e, start + at, mine))
            at += mine
        assert at == count
        start += count
    assert [tuple(lie[3 * i:3 * i + 3]) for i in range(lie[most])] == want
    order, of = order.tolist(), chosen.view(-1).tolist()
    assert sorted(order[:start]) == [p for p, e in enumerate(of) if e < E] and set(order[start:]) <= {-1}
    assert all(of[p] == e for e, first, count in want for p in order[first:first + count])


@pytest.mark.parametrize("n,top,width", [(70, 2, 32), (33, 3, 1024), (300, 5, 1056), (17, 4, 4128)])
@pytest.mark.parametrize("weighted", [True, False])
def test_experts_outputs_add_up_to_the_same_bits_in_any_rows(n, top, width, weighted):
    """The kernel that adds up a token's experts, by fours into rows on 16 bytes and by single values into others: the weighted sums in
    the order of the experts, rounded where a float32 multiply-add rounds, then added to the stream."""
    from hfee_amd.kernels import ops
    E, ff = 7, 32
    g = torch.Generator().manual_seed(n)
    rand = lambda *shape: (torch.randn(*shape, generator=g) * shape[-1] ** -0.5).to(torch.bfloat16).cuda()      # noqa: E731
    h, wg, wu, wd = rand(n, width) * 16, rand(E, ff, width), rand(E, ff, width), rand(E, width, ff)
    chosen = torch.rand(n, E, generator=g).topk(top).indices.to(torch.int32).cuda()
    weights = torch.rand(n, top, generator=g).cuda() if weighted else None
    results = []
    for pad, at in ((0, 0), (4, 0), (3, 0), (4, 1)):
        x = torch.ones(n, width + pad, device="cuda")[:, at:at + width]
        order = torch.zeros(n * top, dtype=torch.int32, device="cuda")
        tiles = torch.zeros(3 * ops.moe_group_tiles(n, top, E) + 1, dtype=torch.int32, device="cuda")
        act = torch.zeros(n * top, ff, dtype=torch.bfloat16, device="cuda")
        y = torch.zeros(n * top, width, device="cuda")
        ops.moe_grouped(x, h, wg, wu, wd, top, order, tiles, act, y, weight=1.0 / top, chosen=chosen, pair_weights=weights)
        results.append(x.clone())
    assert all(torch.equal(results[0], r) for r in results[1:])
    total = torch.zeros(n, width, dtype=torch.float64, device="cuda")
    for j in range(top):
        w = weights[:, j:j + 1].double() if weighted else torch.tensor(1.0 / top, dtype=torch.float32).double().item()
        total = (total + y.view(n, top, width)[:, j].double() * w).float().double()
    # (a float64 sum that is then rounded may round twice: one ulp of the sum's largest part)
    assert ((results[0].double() - (1.0 + total)).abs() <= 2.0 ** -22 * (1 + y.view(n, top, width).double().abs().sum(1))).all()
    assert float((results[0] - 1).std()) > 0


@pytest.mark.parametrize("form", ["gated", "clipped", "not gated"])
@pytest.mark.parametrize("top", [1, 2])
def test_grouped_experts_have_one_order_of_additions(form, top):
    """Rows so far apart that an offset of 32 bits does not reach them all go through tiles of 64 pairs by way of registers,
    rows side by side through tiles of 128 pairs straight into LDS: the same bits, in activations, pairs' outputs and the
    stream that they are added to."""
    from hfee_amd.kernels import ops
    E, width, ff, n = 3, 320, 448, 259
    g = torch.Generator().manual_seed(top)
    rand = lambda *shape: (torch.randn(*shape, generator=g) * shape[-1] ** -0.5).to(torch.bfloat16).cuda()      # noqa: E731
    near, wg, wu, wd = rand(n, width) * 16, rand(E, ff, width), rand(E, ff, width), rand(E, width, ff)
    apart = -(-(1 << 30) // n // 8) * 8 + 8
    far = torch.empty(n, apart, dtype=torch.bfloat16, device="cuda")[:, :width]
    far.copy_(near)
    chosen = torch.rand(n, E, generator=g).topk(top).indices.to(torch.int32).cuda()
    weights = torch.rand(n, top, generator=g).cuda()
    more = dict(activation="clipped", numbers=(7.0, 1.702)) if form == "clipped" else {}
    results = []
    for h in (near, far):
        order = torch.zeros(n * top, dtype=torch.int32, device="cuda")
        tiles = torch.zeros(3 * ops.moe_group_tiles(n, top, E) + 1, dtype=torch.int32, device="cuda")
        act = torch.zeros(n * top, ff, dtype=torch.bfloat16, device="cuda")
        y = torch.zeros(n * top, width, device="cuda")
        x = torch.ones(n, width, device="cuda")
        which = dict(in_weights=weights) if form == "not gated" else dict(pair_weights=weights)
        ops.moe_grouped(x, h, None if form == "not gated" else wg, wu, wd, top, order, tiles, act, y, chosen=chosen, **which, **more)
        results.append((act, y, x))
    for a, b in zip(*results):
        assert torch.equal(a, b)
    assert results[0][2].std() > 0


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_experts_by_table(dtype):
    from hfee_amd.kernels import ops
    dt = DT[dtype]
    g = torch.Generator().manual_seed(4)
    n, width, F, E, top, vocab = 9, 40, 22, 5, 3, 30
    h = torch.randn(n, width, generator=g).to(dt)
    wg, wu = (torch.randn(E, F, width, generator=g) * 0.2).to(dt), (torch.randn(E, F, width, generator=g) * 0.2).to(dt)
    wd = (torch.randn(E, width, F, generator=g) * 0.2).to(dt)
    table = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(vocab)]).to(torch.int32)
    ids = torch.randint(0, vocab, (n,), generator=g)
    w = {"m.table": table}
    for e in range(E):
        w.update({f"m.e{e}.gate": wg[e].double(), f"m.e{e}.up": wu[e].double(), f"m.e{e}.down": wd[e].double()})
    want = ps.table_moe(h.double(), ids, w, "m.", {"router": {"top": top}})
    x = torch.ones(n, width, device="cuda")
    act = torch.zeros(n * top, F, dtype=dt, device="cuda")
    ops.moe_up(act, h.cuda(), wg.cuda(), wu.cuda(), top, table=table.cuda(), token_ids=i32(ids))
    ops.moe_down(x, act, wd.cuda(), top, weight=1.0 / top, table=table.cuda(), token_ids=i32(ids))
    assert su.rel(x.double().cpu() - 1.0, want) < (1e-5 if dtype == "float32" else 2e-2)


@pytest.mark.parametrize("n,top,E,F,width", [(300, 2, 5, 96, 64), (70, 1, 3, 32, 96), (9, 3, 4, 64, 32), (129, 4, 40, 320, 128)])
def test_experts_grouped_on_the_matrix_cores(n, top, E, F, width):
    """Pairs grouped by expert against the token-by-token kernels and the plain sum: experts with no
    token, with one, with more than a tile of 64; every token's own result whatever shares its tile."""
    from hfee_amd.kernels import ops
    g = torch.Generator().manual_seed(n)
    vocab = 50
    h = torch.randn(n, width, generator=g).bfloat16()
    wg, wu = (torch.randn(E, F, width, generator=g) * 0.2).bfloat16(), (torch.randn(E, F, width, generator=g) * 0.2).bfloat16()
    wd = (torch.randn(E, width, F, generator=g) * 0.2).bfloat16()
    table = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(vocab)]).to(torch.int32)
    if E > 4:
        table[table == 1] = 0 if top == 1 else table[table == 1]        # (an expert that nobody uses, where rows stay distinct)
    ids = torch.randint(0, vocab, (n,), generator=g)
    x0 = torch.randn(n, width, generator=g)
    one = x0.clone().cuda()
    act = torch.zeros(n * top, F, dtype=torch.bfloat16, device="cuda")
    ops.moe_up(act, h.cuda(), wg.cuda(), wu.cuda(), top, table=table.cuda(), token_ids=i32(ids))
    ops.moe_down(one, act, wd.cuda(), top, weight=1.0 / top, table=table.cuda(), token_ids=i32(ids))
    grouped = x0.clone().cuda()
    order = torch.zeros(n * top, dtype=torch.int32, device="cuda")
    tiles = torch.zeros(3 * ops.moe_group_tiles(n, top, E) + 1, dtype=torch.int32, device="cuda")
    act2 = torch.zeros(n * top, F, dtype=torch.bfloat16, device="cuda")
    y = torch.zeros(n * top, width, device="cuda") if top > 1 else None
    ops.moe_grouped(grouped, h.cuda(), wg.cuda(), wu.cuda(), wd.cuda(), top, order, tiles, act2, y, weight=1.0 / top,
                    table=table.cuda(), token_ids=i32(ids))
    assert sorted(order.cpu().tolist()) == list(range(n * top))
    assert su.rel((grouped - x0.cuda()).cpu(), (one - x0.cuda()).cpu()) < 1e-2
    # the same tokens in another company: a token's numbers stay what they were, bit for bit
    keep = torch.arange(0, n, 3)
    again = x0[keep].clone().cuda()
    ops.moe_grouped(again, h[keep].cuda().contiguous(), wg.cuda(), wu.cuda(), wd.cuda(), top, order, tiles, act2, y,
                    weight=1.0 / top, table=table.cuda(), token_ids=i32(ids[keep]))
    assert torch.equal(again.cpu(), grouped.cpu()[keep])


# ------------------------------------------------------------------ the whole model

@pytest.fixture(scope="module")
def folders(tmp_path_factory):
    base = tmp_path_factory.mktemp("sabezen")
    out = {(name, dtype): su.make_folder(base / f"{name}_{dtype}", cj, seed=7 + ord(name[0]), dtype=dtype)
           for name, cj in list(su.CONFIGS.items()) + list(su.SINGLE.items()) for dtype in ("float32", "bfloat16")}
    return out


def plain_logits(folder, tokens):
    cj, w = su.load_plain(folder)
    return ps.forward(cj, w, tokens, dtype=torch.float64).numpy()


@pytest.fixture(scope="module")
def plain_rows(folders):
    cache = {}

    def get(name, dtype, lengths=None):
        key = (name, dtype, tuple(lengths or LENGTHS[name]))
        if key not in cache:
            cj = (su.CONFIGS.get(name) or su.SINGLE[name])
            reqs = tu.make_requests(cj["vocab"], list(key[2]), seed=ord(name[0]))
            rows = {}
            for rid, toks in reqs.items():
                logits = plain_logits(folders[(name, dtype)], toks)
                rows.update({(rid, i): logits[i] for i in range(len(toks))})
            cache[key] = (reqs, rows)
        return cache[key]
    return get


def compare(got, want, tol, what):
    assert set(got) == set(want), f"{what}: positions differ"
    worst, where, errors = 0.0, None, []
    for key in want:
        e = su.rel(got[key], want[key])
        errors.append(e)
        if not e <= worst:
            worst, where = e, key
    assert worst < tol, f"{what}: worst relative error {worst:.3e} at {where}"
    assert np.median(errors) < tol / 2, f"{what}: median relative error {np.median(errors):.3e}"


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", sorted(su.SINGLE))
def test_each_mechanism_as_a_model_of_one_layer(folders, plain_rows, name, dtype):
    from hfee_amd.trace_replay import Replayer
    reqs, want = plain_rows(name, dtype, [37, 2, 11])
    for what, steps in (("whole", tu.whole(reqs)), ("bulk then single tokens", tu.bulk_then_tail(reqs, 9)),
                        ("portions", tu.portions(reqs, sizes=(2, 5, 3, 2, 7)))):
        rep = Replayer(folders[(name, dtype)], dtype, 64, max_requests=2)
        compare(tu.run(rep, steps), want, TOL[dtype], f"{name} {dtype} {what}")


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", ["A", "B", "C", "D"])
def test_every_way_of_cutting_gives_the_plain_logits(folders, plain_rows, name, dtype):
    from hfee_amd.trace_replay import Replayer
    reqs, want = plain_rows(name, dtype)
    longest = max(len(t) for t in reqs.values())
    one = (longest + 63) // 64 * 64
    for what, steps, room in (("whole", tu.whole(reqs), one), ("bulk then single tokens", tu.bulk_then_tail(reqs, 40), one),
                              ("portions", tu.portions(reqs), one), ("mixed", *tu.mixed(reqs, seed=len(name)))):
        rep = Replayer(folders[(name, dtype)], dtype, room, max_requests=4)
        got = tu.run(rep, steps)
        compare(got, want, TOL[dtype], f"{name} {dtype} {what}")
        rep.engine.cache.check()
        assert not rep.engine.cache.requests


def test_cuts_agree_closely_in_32_bit(folders, plain_rows):
    """Whole prompts against portions and single tokens: rounding apart, the same logits."""
    from hfee_amd.trace_replay import Replayer
    reqs, _ = plain_rows("A", "float32")
    runs = []
    for steps in (tu.whole(reqs), tu.portions(reqs, sizes=(2, 3, 16, 1, 15, 17, 2)), tu.bulk_then_tail(reqs, 20)):
        runs.append(tu.run(Replayer(folders[("A", "float32")], "float32", 192, max_requests=4), steps))
    for other in runs[1:]:
        for key in runs[0]:
            assert su.rel(other[key], runs[0][key]) < 3e-6


@pytest.mark.parametrize("name", ["A", "C"])
def test_a_slot_that_is_used_again_starts_from_nothing(folders, plain_rows, name):
    """One state slot and a pool of one request's pages: every request inherits the slot and the pages of
    the one before, whose state and convolution inputs must be gone."""
    from hfee_amd.trace_replay import Replayer
    reqs, want = plain_rows(name, "float32")
    longest = max(len(t) for t in reqs.values())
    rep = Replayer(folders[(name, "float32")], "float32", (longest + 63) // 64 * 64, max_requests=1)
    got = tu.run(rep, tu.portions(reqs, sizes=(9, 2, 30)))
    compare(got, want, TOL["float32"], f"{name}: one slot for all")


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_long_decoding(folders, dtype):
    """300 single tokens after a short prompt: decode steps replayed from captured graphs, across page
    borders and across several chunks, the states carried through every replay."""
    from hfee_amd.trace_replay import Replayer
    rng = np.random.default_rng(9)
    toks = rng.integers(0, 500, size=330).tolist()
    rep = Replayer(folders[("D", dtype)], dtype, 384, max_requests=4)
    steps = [{"entries": [("a", toks[:30], [29])], "end": []}]
    steps += [{"entries": [("a", toks[i:i + 1], [0])], "end": ["a"] if i == 329 else []} for i in range(30, 330)]
    got = tu.run(rep, steps)
    assert rep.engine.graph_replays > 250
    want = plain_logits(folders[("D", dtype)], toks)
    compare(got, {("a", i): want[i] for i in range(29, 330)}, TOL[dtype], f"long decoding {dtype}")


def test_grouped_experts_inside_replayed_decode_steps(tmp_path):
    """Three requests decode side by side on a model of two experts, both for every token: more pairs than
    experts, so the grouped kernels (their ordering on the device included) run inside the recorded graphs."""
    from hfee_amd.trace_replay import Replayer
    cj = su.config(70, 64, 1e-6, 2.0, [su.moe(su.gla(2, 16, 16, 6.0, 8), 32, 2, 2), su.moe(su.attention(4, 2, 32, 16, 24, 0.2), 64, 3, 2)])
    folder = su.make_folder(tmp_path / "few", cj, seed=5, dtype="bfloat16")
    reqs = tu.make_requests(70, [50, 47, 44], seed=1)
    steps = [{"entries": [(rid, toks[:4], [3]) for rid, toks in reqs.items()], "end": []}]
    for i in range(4, 44):
        steps.append({"entries": [(rid, toks[i:i + 1], [0]) for rid, toks in reqs.items()], "end": []})
    steps.append({"entries": [(rid, toks[44:], [len(toks) - 45]) for rid, toks in reqs.items() if len(toks) > 44],
                  "end": list(reqs)})
    rep = Replayer(folder, "bfloat16", 256, max_requests=4)
    got = tu.run(rep, steps)
    assert rep.engine.graph_replays > 30
    want = {}
    for rid, toks in reqs.items():
        logits = plain_logits(folder, toks)
        want.update({(rid, i): logits[i] for i in range(3, 44)})
        if len(toks) > 44:
            want[(rid, len(toks) - 1)] = logits[len(toks) - 1]
    compare(got, want, TOL["bfloat16"], "grouped experts in graphs")


@pytest.mark.parametrize("name", ["A", "D"])
def test_a_prompts_recurrences_have_the_bits_of_single_tokens(folders, name, monkeypatch):
    """What the recurrences of a bfloat16 step make of whole prompts, outputs and states, is what the same tokens give one
    at a time: ids chosen among close candidates do not depend on how long a portion is."""
    from hfee_amd.kernels import ops
    from hfee_amd.trace_replay import Replayer
    scan, seen = ops.linear_scan, []

    def record(out, state, q, k, v, decay, beta, rows, lengths, slots, *sizes, **more):
        before = state.clone()
        scan(out, state, q, k, v, decay, beta, rows, lengths, slots, *sizes, **more)
        seen.append((out.clone(), before, state.clone(), q.clone(), k.clone(), v.clone(), decay.clone(),
                     None if beta is None else beta.clone(), lengths.tolist(), slots.clone(), sizes))

    monkeypatch.setattr(ops, "linear_scan", record)
    reqs = tu.make_requests(60, [100, 17, 70, 1], seed=3)
    tu.run(Replayer(folders[(name, "bfloat16")], "bfloat16", 192, max_requests=4), tu.whole(reqs))
    assert any(max(s[8]) == 100 for s in seen) and len(seen) >= 2
    for out, state, after, q, k, v, decay, beta, lengths, slots, sizes in seen:
        row0 = 0
        for i, n in enumerate(lengths):
            for t in range(row0, row0 + n):
                one = torch.zeros_like(out[t:t + 1])
                scan(one, state, *(x[t:t + 1].contiguous() for x in (q, k, v, decay)),
                     None if beta is None else beta[t:t + 1].contiguous(), i32([0]), i32([1]), slots[i:i + 1].contiguous(), *sizes)
                assert torch.equal(one, out[t:t + 1]), f"request {i}, token {t - row0}"
            row0 += n
        assert torch.equal(state, after)


def test_a_far_token_shows_through_the_states(folders):
    """Two sequences that differ in their first token only: hundreds of tokens later the recurrent layers
    still carry the difference (no attention layer could: the chunks are long past), and the engine's
    logits follow the plain ones in both."""
    from hfee_amd.trace_replay import Replayer
    rng = np.random.default_rng(2)
    a = rng.integers(0, 60, size=260).tolist()
    b = [(a[0] + 7) % 60] + a[1:]
    rep = Replayer(folders[("C", "float32")], "float32", 640, max_requests=2)
    got = tu.run(rep, [{"entries": [("a", a[:200], []), ("b", b[:200], [])], "end": []},
                       {"entries": [("a", a[200:], [59]), ("b", b[200:], [59])], "end": ["a", "b"]}])
    wa, wb = plain_logits(folders[("C", "float32")], a)[259], plain_logits(folders[("C", "float32")], b)[259]
    assert su.rel(got[("a", 259)], wa) < TOL["float32"] and su.rel(got[("b", 259)], wb) < TOL["float32"]


def greedy(folder, prompt, count):
    seq = list(prompt)
    for _ in range(count):
        seq.append(int(np.argmax(plain_logits(folder, seq)[-1])))
    return seq[len(prompt):]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_greedy_generation_through_the_entry_point(folders, dtype):
    from hfee_amd import LLM, SamplingParams
    folder = folders[("A", dtype)]
    llm = LLM(folder, dtype=dtype, num_ctx=128, num_parallel=3, max_batch_tokens=24)
    g = np.random.default_rng(5)
    prompts = [g.integers(0, 131, size=n).tolist() for n in (5, 40, 1, 17, 33)]
    outs = llm.generate(prompts, SamplingParams.greedy(num_predict=8))
    for p, o in zip(prompts, outs):
        want = greedy(folder, p, 8)
        if dtype == "float32":
            assert o.token_ids == want
        else:
            logits = plain_logits(folder, p + want)
            margins = []
            for i in range(8):
                row = np.sort(logits[len(p) - 1 + i])
                margins.append(float((row[-1] - row[-2]) / np.abs(row).max()))
            tu.agree_until_a_near_tie(o.token_ids, want, margins, f"greedy {dtype}")


def test_trace_runner_as_a_subprocess(folders, tmp_path):
    folder = folders[("B", "float32")]
    toks = list(range(1, 40))
    lines = [{"step": 0, "entries": [{"id": "x", "tokens": toks[:21], "want": [0, 20]}], "end": []},
             {"step": 1, "entries": [{"id": "x", "tokens": toks[21:22], "want": []}], "end": []},
             {"step": 2, "entries": [{"id": "x", "tokens": toks[22:], "want": [16]}, {"id": "y", "tokens": toks[:2], "want": [1]}],
              "end": ["x", "y"]}]
    out = tmp_path / "out"
    p = subprocess.run([sys.executable, os.path.join(ROOT, "bin", "trace_run"), "--model", folder, "--dtype", "float32",
                        "--out", str(out), "--max-tokens", "128"], input="\n".join(json.dumps(l) for l in lines) + "\n",
                       capture_output=True, text=True, timeout=600)
    assert p.returncode == 0, p.stderr[-2000:]
    assert [l for l in p.stdout.splitlines() if l.startswith("done")] == ["done 0", "done 1", "done 2"]
    want = plain_logits(folder, toks)
    a = np.fromfile(out / "0.f32", dtype="<f4").reshape(2, -1)
    c = np.fromfile(out / "2.f32", dtype="<f4").reshape(2, -1)
    assert not (out / "1.f32").exists()
    assert su.rel(a[0], want[0]) < 3e-5 and su.rel(a[1], want[20]) < 3e-5
    assert su.rel(c[0], want[38]) < 3e-5 and su.rel(c[1], want[1]) < 3e-5


def test_the_command_line_runs_the_design(folders):
    """`hfee run <folder> --tokens ...`: the greedy continuation's ids."""
    folder = folders[("B", "float32")]
    prompt = tu.make_requests(97, [11], seed=8)["r0"]
    want = greedy(folder, prompt, 7)
    p = subprocess.run([sys.executable, os.path.join(ROOT, "bin", "hfee"), "run", folder, "--tokens",
                        ",".join(map(str, prompt)), "--dtype", "float32", "--temperature", "0", "--repeat-penalty", "1",
                        "--num-predict", "7", "--num-ctx", "128", "--verbose"],
                       capture_output=True, text=True, timeout=300, stdin=subprocess.DEVNULL)
    assert p.returncode == 0, p.stderr[-2000:]
    assert [int(t) for t in p.stdout.strip().splitlines()[0].split()] == want


def test_seeded_sampling_does_not_depend_on_the_batch(folders):
    from hfee_amd import LLM, SamplingParams
    folder = folders[("A", "float32")]
    g = np.random.default_rng(3)
    prompts = [g.integers(0, 131, size=n).tolist() for n in (9, 30, 2)]
    params = [SamplingParams(temperature=0.9, top_k=20, top_p=0.95, seed=100 + i, num_predict=10) for i in range(3)]
    together = LLM(folder, dtype="float32", num_ctx=128, num_parallel=3).generate(prompts, params)
    for i in range(3):
        alone = LLM(folder, dtype="float32", num_ctx=128, num_parallel=1).generate([prompts[i]], [params[i]])[0]
        assert alone.token_ids == together[i].token_ids
