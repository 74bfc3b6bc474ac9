"""The prefill kernels at the sizes where their dispatch or tiling changes
(GPU): runs, tiles and remainders, and rows that break 16-byte alignment."""
import pytest
import torch

from oracle import glue
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
    out = layers.conv_prefill(proj.to(gpu), win, w.to(gpu), _cu(lengths, gpu), channels).cpu()
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
