"""The prefill kernels at the sizes where their dispatch or tiling changes
(GPU): runs, tiles and remainders, and rows that break 16-byte alignment."""
from dataclasses import fields

import pytest
import torch

from oracle import anchor as oracle_memory
from oracle import glue
from yanchor_amd import _native
from yanchor_amd import gdn
from yanchor_amd import independent_memory as im
from yanchor_amd import layers

pytestmark = pytest.mark.gpu


def _cu(lengths, dev):
    return torch.tensor([0, *torch.tensor(lengths).cumsum(0).tolist()], dtype=torch.int32, device=dev)


@pytest.mark.parametrize("lengths,channels,pad", [
    ([1, 2, 0, 3, 5, 64, 65, 1], 2048, 8),          # short runs, whole channel blocks
    ([700, 1, 2, 0, 900, 3], 12288, 64),            # long runs: pieces end inside a run
    ([130, 7], 2056, 8),                            # a last channel block of one group
    ([130, 7], 2052, 0),                            # rows off 16-byte alignment: one channel a thread
])
def test_conv_prefill_runs(gpu, lengths, channels, pad):
    """One bf16 ulp of the oracle's float32 form (its taps sum in another
    order, so a value may round to the next bf16), the window exactly."""
    g = torch.Generator().manual_seed(11)
    n = sum(lengths)
    proj = torch.randn(n, channels + pad, generator=g).to(torch.bfloat16)
    window = torch.randn(len(lengths), 3, channels, generator=g).to(torch.bfloat16)
    w = (torch.randn(channels, 4, generator=g) * 0.5).to(torch.bfloat16)
    win = window.to(gpu)
    args = (proj.to(gpu), win, w.to(gpu), _cu(lengths, gpu), channels)
    planes = layers.conv_prefill(args[0], window.to(gpu), *args[2:], planes=4).cpu()
    out = layers.conv_prefill(*args).cpu()
    assert torch.equal(planes, out.view(n, 4, channels // 4).transpose(0, 1))
    off = 0
    for r, length in enumerate(lengths):
        y, new = glue.causal_conv1d_prefill(proj[off: off + length, :channels], window[r], w)
        if length:
            assert torch.allclose(out[off: off + length].float(), y.float(), rtol=2 ** -7, atol=2 ** -7), r
        assert torch.equal(win[r].cpu(), new), r
        off += length


def _swa_reference(q, k, v, lengths, starts, rk, rv, window, gate):
    """float64 sliding-window attention of each piece over [ring | piece]."""
    out, off = torch.zeros(q.shape, dtype=torch.float64), 0
    for r, n in enumerate(lengths):
        ctx = min(starts[r], window - 1)
        pos = torch.arange(starts[r] - ctx, starts[r]) % window
        kc = torch.cat((rk[r][:, pos].transpose(0, 1), k[off: off + n]), 0).double()
        vc = torch.cat((rv[r][:, pos].transpose(0, 1), v[off: off + n]), 0).double()
        if n:
            out[off: off + n] = glue.swa_prefill_attention(q[None, off: off + n].double(), kc[None], vc[None], window,
                                                           query_start=ctx)[0]
        off += n
    return out if gate is None else out * torch.sigmoid(gate.double())


@pytest.mark.parametrize("heads,groups,window,lengths,starts", [
    (32, 8, 64, [1, 31, 32, 33, 0, 200, 5], [0, 63, 64, 1000, 7, 30, 64]),   # an odd number of tiles, two pieces a group
    (6, 6, 100, [130, 3], [99, 250]),              # one head a group: 64 tokens a tile, a window off the tile size
    (16, 2, 1024, [9, 70, 8], [2000, 1, 0]),       # 8 heads a group
    (64, 1, 65, [3, 2], [64, 0]),                  # 64 heads a group: one token a tile
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_swa_prefill_tiles(gpu, heads, groups, window, lengths, starts, dtype):
    """Bound: the result's own rounding and P's (half an ulp each, 2^-9 in
    bf16) with the gate's two products: 2e-2 as for the other swa tests."""
    gen = torch.Generator().manual_seed(5)
    n, r = sum(lengths), len(lengths)
    q = torch.randn(n, heads, 128, generator=gen).to(dtype)
    k = torch.randn(n, groups, 128, generator=gen).to(dtype)
    v = torch.randn(n, groups, 128, generator=gen).to(dtype)
    rk = torch.randn(r, groups, window, 128, generator=gen).to(dtype)
    rv = torch.randn(r, groups, window, 128, generator=gen).to(dtype)
    gate = torch.randn(n, heads, 130, generator=gen).to(dtype)[..., :128]      # rows off 16-byte alignment
    wide = torch.zeros(n, (1 << 23) + groups * 128, dtype=dtype) if n < 16 else None
    kd = k.to(gpu)
    if wide is not None:                                     # a token stride past the 32-bit tile offsets
        kd = wide.to(gpu)[:, : groups * 128].view(n, groups, 128)
        kd.copy_(k)
    ref = _swa_reference(q, k, v, lengths, starts, rk, rv, window, gate)
    args = (q.to(gpu), kd, v.to(gpu), _cu(lengths, gpu), torch.tensor(starts, device=gpu), rk.to(gpu), rv.to(gpu),
            torch.arange(r, device=gpu))
    out = layers.swa_prefill(*args, gate=gate.to(gpu))
    assert ((out.cpu().double() - ref).norm() / ref.norm()).item() < 2e-2
    # the caller's own tile list, in another order and in part: the same rows
    tiles = layers.prefill_tiles(lengths, 64 // (heads // groups), "cpu")
    pick = torch.randperm(len(tiles), generator=gen)
    again = layers.swa_prefill(*args, gate=gate.to(gpu), tiles=tiles[pick])
    assert ((again.cpu().double() - ref).norm() / ref.norm()).item() < 2e-2


@pytest.mark.parametrize("heads,groups,tt", [(32, 8, 16), (2, 2, 64), (16, 2, 8)])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_swa_prefill_unseen_values(gpu, heads, groups, tt, bad):
    """A value that is not finite reaches no token before the tile of ``tt``
    tokens it lies in and none after the last tile with a token that sees it,
    whatever shares the workgroup: those rows are bit for bit what they are
    without it."""
    gen = torch.Generator().manual_seed(9)
    n, window, bf = 6 * tt + 200, 64, torch.bfloat16
    q, k, v = (torch.randn(n, h, 128, generator=gen).to(bf) for h in (heads, groups, groups))
    ring = torch.randn(1, groups, window, 128, generator=gen).to(bf)

    def run(x):
        return layers.swa_prefill(q.to(gpu), k.to(gpu), x.to(gpu), _cu([n], gpu), torch.tensor([70], device=gpu),
                                  ring.to(gpu), ring.to(gpu), torch.zeros(1, dtype=torch.long, device=gpu)).cpu()
    clean = run(v)
    for at in (0, tt, 2 * tt + 1, 3 * tt, 4 * tt - 1):
        x = v.clone()
        x[at] = bad
        got = run(x)
        first, last = at // tt * tt, (at + window - 1) // tt * tt + tt
        assert not torch.isfinite(got[at].float()).any()
        assert torch.equal(got[:first], clean[:first]), at
        assert torch.equal(got[last:], clean[last:]), at


def test_swa_prefill_past_a_grid_row(gpu):
    """More tiles than one grid row holds threads for: the first of two pieces
    over and over, then the second once."""
    n, g, bf = 3, 8, torch.bfloat16
    q, k, v = (torch.randn(n, g, 128, device=gpu).to(bf) for _ in range(3))
    ring, at = torch.zeros(2, g, 64, 128, dtype=bf, device=gpu), torch.zeros(2, dtype=torch.long, device=gpu)
    rows, cu = torch.arange(2, device=gpu), _cu([1, 2], gpu)
    want = layers.swa_prefill(q, k, v, cu, at, ring, ring, rows)
    tiles = torch.zeros((1 << 22) + 5, 2, dtype=torch.int32, device=gpu)
    tiles[-1, 0] = 1
    out = torch.full_like(q, 7.0)
    _native.call("yh_swa_prefill", q.data_ptr(), g * 128, k.data_ptr(), g * 128, v.data_ptr(), g * 128,
                 ring.data_ptr(), ring.data_ptr(), rows.data_ptr(), at.data_ptr(), cu.data_ptr(), tiles.data_ptr(),
                 len(tiles), None, 0, 0, out.data_ptr(), 2, 2, g, g, 128, 64, _native.BF16, _native.stream_of(q))
    assert torch.equal(out, want)


def test_swa_prefill_scattered_tiles(gpu):
    """A caller's tile list whose neighbours lie far apart costs about what the
    sorted list does (each tile its own window, at most twice the copies): the
    keys between two tiles of a piece are not walked.  Walking them took 8 times
    as long here; the bound is 5."""
    n, window, bf = 16000, 64, torch.bfloat16
    q, k, v = (torch.randn(n, h, 128, device=gpu).to(bf) for h in (32, 8, 8))
    ring = torch.zeros(1, 8, window, 128, dtype=bf, device=gpu)
    at = torch.zeros(1, dtype=torch.long, device=gpu)
    tiles = layers.prefill_tiles([n], 16, "cpu")
    mixed = tiles[torch.randperm(len(tiles), generator=torch.Generator().manual_seed(0))]
    launch, times, outs = _native.call, [], []

    def timed(name, *args):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        launch(name, *args)
        b.record()
        b.synchronize()
        times.append(a.elapsed_time(b))
    try:
        _native.call = timed
        for _ in range(5):
            for order in (tiles, mixed):
                outs.append(layers.swa_prefill(q, k, v, _cu([n], gpu), at, ring, ring, at, tiles=order))
    finally:
        _native.call = launch
    assert torch.equal(outs[-1], outs[-2]) or (outs[-1].float() - outs[-2].float()).abs().max() < 0.05
    assert min(times[1::2]) <= 5 * min(times[::2]), times


def _one_key(dtype, tail):
    """Queries of 25 lengths and 1024 keys along one dim: score 8 a / sqrt(128)
    for key 0, 0 for the others, so that those weigh exp(-5.3) .. exp(-7.3) each
    (tail: exp(-9.5) .. exp(-10.5), subnormal in float16)."""
    a = torch.linspace(13.5, 15.0, 25) if tail else torch.linspace(7.5, 10.5, 25)
    q, k = torch.zeros(25, 128, dtype=dtype), torch.zeros(1024, 128, dtype=dtype)
    q[:, 0], k[0, 0] = a, 8.0
    p = torch.exp(q[:, :1].double() * -8.0 / 128 ** 0.5)
    return q, k, p


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_softmax_denominator_keeps_float32(gpu, dtype):
    """Only key 0 has a value, so a row is value / (1 + 1023 p), and with the sum
    in float32 it is that to about 2e-6 before its one rounding: all but the
    values so near a rounding boundary (1 % in float16, whose steps are 2^-11)
    are the rounded reference.  Sums of rounded p miss it in 16 % of the values."""
    gen = torch.Generator().manual_seed(1)
    q, k, p = _one_key(dtype, False)
    v = (1 + torch.rand(1, 128, generator=gen)).to(dtype)
    want = v[0].double() / (1 + 1023 * p)
    # key 0 lies in the first key tile, so the others are weighed against it: in
    # the ring, 30 keys after the oldest of a piece at position 5000
    rk, rv = torch.zeros(2, 1, 1, 1024, 128, dtype=dtype)
    rk[0, 0, (5000 - 1023 + 30) % 1024], rv[0, 0, (5000 - 1023 + 30) % 1024] = k[0], v[0]
    zero = torch.zeros(25, 1, 128, dtype=dtype, device=gpu)
    got = layers.swa_prefill(q[:, None].to(gpu), zero, zero, _cu([25], gpu), torch.tensor([5000], device=gpu),
                             rk.to(gpu), rv.to(gpu), torch.zeros(1, dtype=torch.long, device=gpu)).cpu()[:, 0].double()
    assert (got != want.to(dtype).double()).double().mean().item() <= 0.02


@pytest.mark.parametrize("form", ["window", "memory"])
def test_subnormal_float16_weights(gpu, form):
    """One dominant key over 1023 keys whose weights (and their lo parts) are
    subnormal in float16, a few per cent of the sum.  Bound: the result's own
    rounding, 2^-11, and that of p to steps of 2^-24 (half a step against 2.6e-5,
    2^-9.8, of the 4 % they add up to): 2^-10."""
    gen = torch.Generator().manual_seed(2)
    q, k, p = _one_key(torch.float16, True)
    v = (1 + torch.rand(1024, 128, generator=gen)).to(torch.float16)
    if form == "window":   # query t reads 999 ring slots and the piece up to t
        rk, rv = torch.zeros(2, 1, 1, 1024, 128, dtype=torch.float16)
        rk[0, 0, 0], rv[0, 0, :999] = k[0], v[:999]
        got = layers.swa_prefill(q[:, None].to(gpu), k[999:, None].to(gpu), v[999:, None].to(gpu), _cu([25], gpu),
                                 torch.tensor([999], device=gpu), rk.to(gpu), rv.to(gpu),
                                 torch.zeros(1, dtype=torch.long, device=gpu)).cpu()[:, 0].double()
        tail = v[1:999].double().sum(0) + v[999:].double().cumsum(0)
        want = (v[0].double() + p * tail) / (1 + p * (999 + torch.arange(25)[:, None]))
    else:                  # the sink's logit is 0 as well
        refs = torch.arange(1024, dtype=torch.int32).view(1, 1, 1, 1024).to(gpu)
        got = im.indexed_gqa(q.view(1, 1, 25, 1, 128).to(gpu), k.view(1, 1024, 1, 128).to(gpu),
                             v.view(1, 1024, 1, 128).to(gpu), refs).cpu().view(25, 128).double()
        want = (v[0].double() + p * v[1:].double().sum(0)) / (1 + p * 1024)
    assert ((got - want).norm() / want.norm()).item() <= 2 ** -10


def _memory_state(gen, b, g, cap, chunk, counts, base, dtype, odd):
    """A memory state with committed slots in no particular order, ``counts``
    pending tokens a row and positions below ``base``.  odd: tied scores, empty
    slots with finite scores and slots at positions past the new tokens."""
    st = im.IndependentMemoryState.empty(b, g, cap, chunk, 128, "cpu", dtype)
    for x in (st.keys, st.values, st.pending_keys, st.pending_values):
        x.copy_(torch.randn(x.shape, generator=gen))
    pos = torch.stack([torch.randperm(base, generator=gen)[:cap] for _ in range(b * g)]).view(b, g, cap)
    sc = torch.randn(b, g, cap, generator=gen)
    if odd:
        sc = sc.round()
        pos = torch.where(torch.rand(pos.shape, generator=gen) < 0.2, -1, pos)
        pos = torch.where(torch.rand(pos.shape, generator=gen) < 0.1, pos + 1000000, pos).clamp(min=-1)
    st.positions.copy_(pos)
    st.scores.copy_(sc)
    st.pending_scores.copy_(torch.randn(st.pending_scores.shape, generator=gen))
    st.count.copy_(torch.tensor(counts))
    st.total.copy_(torch.tensor([base + c for c in counts]))
    return st


def _clone(st, dev):
    return im.IndependentMemoryState(**{f.name: getattr(st, f.name).to(dev, copy=True) for f in fields(st)})


@pytest.mark.parametrize("cap,chunk,length,heads,groups,odd", [
    (16, 8, 40, 4, 2, True),           # many small blocks, ties
    (256, 64, 100, 32, 8, False),      # less than two blocks
    (256, 64, 4200, 4, 1, True),       # more tokens than one sort holds
    (1030, 5, 3100, 3, 1, True),       # sizes off every power of two, a second sort of a few blocks
    (3, 64, 1, 8, 8, False),           # one token, fewer slots than a run
])
def test_memory_sequence_segments(gpu, cap, chunk, length, heads, groups, odd):
    """The state bit for bit against the oracle's token order, the read within
    1e-2 of it; masked rows and packed rows alike."""
    gen = torch.Generator().manual_seed(cap + length)
    b, dt = 3, torch.bfloat16
    st = _memory_state(gen, b, groups, cap, chunk, [0, chunk - 1, chunk // 2], max(2 * cap, 64), dt, odd)
    q = torch.randn(b, length, heads, 128, generator=gen).to(dt)
    k = torch.randn(b, length, groups, 128, generator=gen).to(dt)
    v = torch.randn(b, length, 2 * groups, 128, generator=gen).to(dt)[:, :, groups:]      # a column view
    sc = torch.randn(b, length, groups, generator=gen)
    if odd:
        sc = sc.round()
    lens = [length, max(1, length // 3), max(1, length - 1)]
    valid = torch.arange(length)[None] < torch.tensor(lens)[:, None]
    if odd and length > 2:
        valid[0, 1] = False                                                               # a hole
    want_state = oracle_memory.MemoryState(**{f.name: getattr(st, f.name).clone() for f in fields(st)})
    want = oracle_memory.sequence(q, k, v, sc, valid, chunk, want_state)
    got_state = _clone(st, gpu)
    got = im.sequence(q.to(gpu), k.to(gpu), v.to(gpu), sc.to(gpu), valid.to(gpu), chunk, got_state)
    for f in fields(st):
        a, w = getattr(got_state, f.name).cpu(), getattr(want_state, f.name)
        assert torch.equal(a.double(), w.double()), f.name
    assert (got.cpu().double() - want.double()).norm() <= 1e-2 * want.double().norm() + 1e-6
    assert not got.cpu()[~valid].any()
    # packed: the same tokens without padding
    lens = valid.sum(1).tolist()
    pack = [x.to(gpu)[valid.to(gpu)] for x in (q, k, v, sc)]
    packed_state = _clone(st, gpu)
    again = im.sequence_packed(*pack, _cu(lens, gpu), lens, chunk, packed_state)
    for f in fields(st):
        assert torch.equal(getattr(packed_state, f.name), getattr(got_state, f.name)), f.name
    assert torch.equal(again, got[valid.to(gpu)])


@pytest.mark.parametrize("cap,chunk,length,heads,groups", [(16, 8, 40, 4, 2), (256, 64, 300, 32, 8), (130, 5, 33, 3, 1)])
def test_assembled_sequence_calls(gpu, cap, chunk, length, heads, groups):
    """The C calls that take assembled sources [slots | pending | new tokens] --
    yh_anchor_prefix, yh_anchor_sequence_read, yh_anchor_sequence_commit -- leave
    the oracle's state and read, as the calls on tokens in place do."""
    gen = torch.Generator().manual_seed(cap)
    b, dt, counts = 3, torch.bfloat16, [length, length // 3, 1]
    st = _memory_state(gen, b, groups, cap, chunk, [0, chunk - 1, chunk // 2], 2 * cap, dt, True)
    q, k, v = (torch.randn(b, length, h, 128, generator=gen).to(dt) for h in (heads, groups, groups))
    sc = torch.randn(b, length, groups, generator=gen)
    valid = torch.arange(length)[None] < torch.tensor(counts)[:, None]
    want_state = oracle_memory.MemoryState(**{f.name: getattr(st, f.name).clone() for f in fields(st)})
    want = oracle_memory.sequence(q, k, v, sc, valid, chunk, want_state)
    src = [torch.cat((c.transpose(1, 2), p[:, :, :chunk].transpose(1, 2), x), 1).contiguous().to(gpu)
           for c, p, x in ((st.keys, st.pending_keys, k), (st.values, st.pending_values, v))]
    got = _clone(st, gpu)
    q, sc, n = q.to(gpu), sc.to(gpu), torch.tensor(counts, device=gpu)
    blocks, total = -(-length // chunk) + 1, cap + chunk + length
    block_refs = torch.empty(b, blocks, groups, cap, dtype=torch.int32, device=gpu)
    final, pending = torch.empty_like(block_refs[:, 0]), torch.empty(b, groups, chunk, dtype=torch.int32, device=gpu)
    out, stream = torch.empty_like(q), _native.stream_of(q)
    _native.call("yh_anchor_prefix", sc.data_ptr(), n.data_ptr(), got.scores.data_ptr(), got.positions.data_ptr(),
                 got.pending_scores.data_ptr(), got.count.data_ptr(), got.total.data_ptr(), block_refs.data_ptr(),
                 final.data_ptr(), pending.data_ptr(), b, length, groups, cap, chunk, chunk, blocks, stream)
    _native.call("yh_anchor_sequence_read", q.data_ptr(), src[0].data_ptr(), src[1].data_ptr(), block_refs.data_ptr(),
                 _native.I32, got.count.data_ptr(), out.data_ptr(), b, length, blocks, chunk, heads, groups, 128, total,
                 cap, _native.BF16, stream)
    _native.call("yh_anchor_sequence_commit", src[0].data_ptr(), src[1].data_ptr(), final.data_ptr(),
                 pending.data_ptr(), n.data_ptr(), got.keys.data_ptr(), got.values.data_ptr(),
                 got.pending_keys.data_ptr(), got.pending_values.data_ptr(), got.count.data_ptr(),
                 got.total.data_ptr(), b, total, length, groups, cap, chunk, chunk, 128, _native.BF16, stream)
    for f in fields(st):
        assert torch.equal(getattr(got, f.name).cpu().double(), getattr(want_state, f.name).double()), f.name
    diff = (out.cpu().double() - want.double())[valid]
    assert diff.norm() <= 1e-2 * want.double()[valid].norm()


def test_prefix_past_a_grid_row(gpu):
    """More memories than one grid row of its workgroups holds threads for: one
    slot and one token each, the better of the two stays."""
    b, g = (1 << 22) // 8 + 3, 8
    score, pos = torch.randn(b, g, 1, device=gpu), torch.zeros(b, g, 1, dtype=torch.int32, device=gpu)
    new, old = torch.randn(b, 1, g, device=gpu), score.clone()
    pend, count, total = torch.zeros(b, g, 1, device=gpu), torch.zeros(b, dtype=torch.long, device=gpu), \
        torch.full((b,), 5, dtype=torch.long, device=gpu)
    ones = torch.ones_like(count)
    refs = torch.full((3, b, g, 1), -7, dtype=torch.int32, device=gpu)     # of the block, final, pending
    _native.call("yh_anchor_prefix", new.data_ptr(), ones.data_ptr(), score.data_ptr(), pos.data_ptr(), pend.data_ptr(),
                 count.data_ptr(), total.data_ptr(), refs[0].data_ptr(), refs[1].data_ptr(), refs[2].data_ptr(), b, 1,
                 g, 1, 1, 1, 1, _native.stream_of(new))
    fresh = new.transpose(1, 2)
    kept = (fresh > old)
    sure = fresh != old
    assert torch.equal(score, torch.maximum(fresh, old))
    assert torch.equal(pos[sure], (kept * 5).to(torch.int32)[sure])
    assert not refs[0].any() and torch.equal(refs[1][sure], (kept * 2).to(torch.int32)[sure])
    assert (refs[2] == -1).all() and torch.isinf(pend).all()


@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 128), (torch.float32, 20)])
@pytest.mark.parametrize("cap,pc,chunk", [(4090, 20, 16), (4096, 4200, 7), (4095, 1, 1), (31, 70, 64)])
def test_commit_from_other_sources(gpu, cap, pc, chunk, dtype, d):
    """Rows past one stage of the commit (4096), exactly: every slot takes the
    source row it names, or zeros; the counters advance."""
    gen = torch.Generator().manual_seed(cap + pc)
    b, g, s, length = 2, 3, 500, 9
    src = torch.randn(2, b, s, g, d, generator=gen).to(dtype)
    refs = [torch.randint(-40, s + 40, (b, g, n), generator=gen).to(torch.int32) for n in (cap, pc)]
    rows, counts = torch.full((2, b, g, cap, d), 7.0).to(dtype), torch.tensor([length, 4])
    pend, count, total = torch.full((2, b, g, pc, d), 7.0).to(dtype), torch.tensor([chunk - 1, 0]), torch.tensor([90, 80])

    def take(which, ref):
        at = ref.clamp(0, s - 1).long()
        x = src[which][torch.arange(b)[:, None, None], at, torch.arange(g)[None, :, None]]
        return x.masked_fill(((ref < 0) | (ref >= s))[..., None], 0)
    dev = [x.to(gpu) for x in (src[0], src[1], *refs, counts, rows[0], rows[1], pend[0], pend[1], count, total)]
    _native.call("yh_anchor_sequence_commit", *[x.data_ptr() for x in dev], b, s, length, g, cap, pc, chunk, d,
                 _native.code(src), _native.stream_of(dev[0]))
    for x, want in zip(dev[5:9], (take(0, refs[0]), take(1, refs[0]), take(0, refs[1]), take(1, refs[1]))):
        assert torch.equal(x.cpu(), want)
    assert torch.equal(dev[9].cpu(), (count + counts) % chunk) and torch.equal(dev[10].cpu(), total + counts)


@pytest.mark.parametrize("case", ["float32", "heads of 64", "5 heads on 2 groups", "no tokens", "unaligned keys"])
@pytest.mark.parametrize("packed", [False, True])
def test_memory_sequence_refusals_leave_the_state(gpu, case, packed):
    """What the read or the state rewrite cannot take is refused before the scan
    rewrites the state's scores and positions."""
    gen = torch.Generator().manual_seed(6)
    dt, d = torch.float32 if case == "float32" else torch.bfloat16, 64 if case == "heads of 64" else 128
    h, n = 5 if case[0] == "5" else 4, 0 if case == "no tokens" else 6
    if packed and n == 0:
        pytest.skip("packed rows hold at least one token")
    state = im.IndependentMemoryState.empty(1, 2, 16, 4, d, gpu, dt)
    state.scores.copy_(torch.randn(state.scores.shape, generator=gen))
    state.positions.copy_(torch.randint(0, 50, state.positions.shape, generator=gen))
    state.total.fill_(60)
    if case == "unaligned keys":
        state.keys = torch.zeros(state.keys.numel() + 1, dtype=dt, device=gpu)[1:].view(state.keys.shape)
    before = _clone(state, "cpu")
    toks = [torch.randn(1, n, x, d, generator=gen).to(dt).to(gpu) for x in (h, 2, 2)] + \
        [torch.randn(1, n, 2, generator=gen).to(gpu)]
    with pytest.raises(ValueError):
        if packed:
            im.sequence_packed(*[x[0] for x in toks], _cu([n], gpu), [n], 4, state)
        else:
            im.sequence(*toks, None, 4, state)
    for f in fields(state):
        assert torch.equal(getattr(state, f.name).cpu(), getattr(before, f.name)), f.name


@pytest.mark.parametrize("offsets", [[0, 8, 10], [0, 5, 9], [0, 5], [1, 5, 10], [0, 5, 11]])
def test_memory_sequence_packed_offsets(gpu, offsets):
    """Offsets that are not those of ``lengths`` are refused before anything is
    written; offsets on the host give what those on the device give."""
    gen = torch.Generator().manual_seed(4)
    dt, lens = torch.bfloat16, [5, 5]
    st = _memory_state(gen, 2, 2, 16, 4, [0, 3], 40, dt, False)
    toks = [torch.randn(10, h, 128, generator=gen).to(dt).to(gpu) for h in (4, 2, 2)] + \
        [torch.randn(10, 2, generator=gen).to(gpu)]
    state = _clone(st, gpu)
    with pytest.raises(ValueError, match="offsets"):
        im.sequence_packed(*toks, torch.tensor(offsets, dtype=torch.int32, device=gpu), lens, 4, state)
    for f in fields(st):
        assert torch.equal(getattr(state, f.name).cpu(), getattr(st, f.name)), f.name
    outs, states = [], []
    for cu in (_cu(lens, gpu), _cu(lens, "cpu")):
        states.append(_clone(st, gpu))
        outs.append(im.sequence_packed(*toks, cu, lens, 4, states[-1]))
    for o, s in zip(outs[1:], states[1:]):
        assert torch.equal(o, outs[0])
        assert all(torch.equal(getattr(s, f.name), getattr(states[0], f.name)) for f in fields(st))


@pytest.mark.parametrize("lengths,h,hv,v,h0,gates", [
    ([3001], 4, 4, 128, True, torch.float32),        # one tile a workgroup, a ragged last chunk
    ([129, 0, 64, 700], 2, 8, 128, False, torch.bfloat16),   # an empty sequence, slots between chunks, GQA
    ([500, 1], 3, 27, 128, True, torch.float32),     # two tiles a workgroup
    ([191, 257], 16, 32, 64, True, torch.float32),   # 64 value columns
    ([300, 200, 257], 8, 32, 64, True, torch.float32),   # two tiles of them a workgroup
])
def test_gdn_few_sequences(gpu, lengths, h, hv, v, h0, gates):
    """The same operations in the same order as the one-launch form: the same
    bits as that form gives the same sequences among many."""
    gen = torch.Generator().manual_seed(3)
    n, copies = sum(lengths), -(-300 // (len(lengths) * hv * v // 32)) + 1
    q, k = (torch.randn(1, n, h, 128, generator=gen).to(torch.bfloat16).to(gpu) for _ in range(2))
    val = torch.randn(1, n, hv, v, generator=gen).to(torch.bfloat16).to(gpu)
    g = torch.nn.functional.logsigmoid(torch.randn(1, n, hv, generator=gen) + 3).to(gates).to(gpu)
    beta = torch.rand(1, n, hv, generator=gen).to(gates).to(gpu)
    s0 = torch.randn(len(lengths), hv, 128, v, generator=gen).to(gpu) * 0.02 if h0 else None
    need = _native.lib().yh_gdn_chunk_workspace_bytes
    assert need(n, len(lengths), hv, v) > 0 and need(copies * n, copies * len(lengths), hv, v) == 0

    def run(c):
        x = [t.repeat(1, c, 1, 1) for t in (q, k, val)] + [t.repeat(1, c, 1) for t in (g, beta)]
        return gdn.chunk_gated_delta_rule(*x[:3], g=x[3], beta=x[4], use_qk_l2norm_in_kernel=True,
                                          initial_state=None if s0 is None else s0.repeat(c, 1, 1, 1),
                                          output_final_state=True, cu_seqlens=_cu(lengths * c, gpu))
    o, st = run(1)
    many_o, many_st = run(copies)
    assert torch.equal(o, many_o[:, :n]) and torch.equal(st, many_st[: len(lengths)])
    assert torch.equal(o, many_o[:, -n:]) and torch.equal(st, many_st[-len(lengths):])


def test_gdn_no_room_for_scratch(gpu, monkeypatch):
    """The few-sequences form's scratch is not a condition of the call: without
    room for it the call gives the same bits."""
    x = torch.randn(1, 700, 4, 128, device=gpu).to(torch.bfloat16)
    g = -torch.rand(1, 700, 4, device=gpu)
    args = dict(g=g, beta=-g, output_final_state=True, cu_seqlens=_cu([700], gpu), use_qk_l2norm_in_kernel=True)
    want = gdn.chunk_gated_delta_rule(x, x, x, **args)
    need = _native.lib().yh_gdn_chunk_workspace_bytes(700, 1, 4, 128)
    empty, refused = torch.empty, []

    def no_scratch(*size, **kw):
        if size == (need,):
            refused.append(size)
            raise torch.OutOfMemoryError("no room")
        return empty(*size, **kw)
    monkeypatch.setattr(torch, "empty", no_scratch)
    got = gdn.chunk_gated_delta_rule(x, x, x, **args)
    monkeypatch.undo()
    assert refused and all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("lens", [[300], [300, 200], [10] * 9])
def test_gdn_lengths_of_every_sequence(gpu, lens):
    """A ``lengths`` that misses a sequence is refused whichever form runs."""
    total, hv = sum(lens), 32
    x = torch.zeros(1, total, hv, 128, dtype=torch.bfloat16, device=gpu)
    g = torch.zeros(1, total, hv, device=gpu)
    with pytest.raises(IndexError):
        gdn.chunk_gated_delta_rule(x, x, x, g=g, beta=g, cu_seqlens=_cu(lens, gpu), lengths=lens[:-1])


@pytest.mark.parametrize("n,length,hv", [(64, 200, 1), (32, 130, 1), (8, 140, 4), (2, 150, 32), (1, 129, 32)])
def test_gdn_few_sequences_time(gpu, n, length, hv):
    """At the edge of its rule (short sequences, many of few heads) the split form
    is no slower than the one launch it stands for (best of 40, 4 % for the
    clock)."""
    total = n * length
    q, k, v = (torch.randn(total, hv, 128, device=gpu).to(torch.bfloat16) for _ in range(3))
    g, beta = -0.1 * torch.rand(total, hv, device=gpu), torch.rand(total, hv, device=gpu)
    cu, o = _cu([length] * n, gpu), torch.empty_like(v)
    state = torch.empty(n, hv, 128, 128, device=gpu)
    need = _native.lib().yh_gdn_chunk_workspace_bytes(total, n, hv, 128)
    ws = torch.empty(need, dtype=torch.uint8, device=gpu)
    assert need > 0

    def best(scratch, size):
        times = []
        for _ in range(40):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(5):
                _native.call("yh_gdn_chunk_varlen", q.data_ptr(), k.data_ptr(), v.data_ptr(), g.data_ptr(),
                             beta.data_ptr(), None, state.data_ptr(), o.data_ptr(), cu.data_ptr(), None, n, total, hv,
                             hv, 128, 128, 128 ** -0.5, 1, _native.BF16, _native.F32, _native.F32, scratch, size,
                             _native.stream_of(q))
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)
    best(ws.data_ptr(), need)
    split, one = best(ws.data_ptr(), need), best(None, 0)
    print(n, length, hv, 'us:', split * 200, one * 200, flush=True)
    assert split <= 1.04 * one
