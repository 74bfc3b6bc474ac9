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
