"""The decode reads of four heads a memory at every number of waves the
launcher gives them (GPU), against float64."""
import pytest
import torch

from yanchor_amd import independent_memory as im

pytestmark = pytest.mark.gpu

D = 128


def _reference(q, keys, values, live, sink):
    b, h, g = q.shape[0], q.shape[1], keys.shape[1]
    logits = torch.einsum("bgrd,bgsd->bgrs", q.double().view(b, g, h // g, D), keys.double()) / D ** 0.5
    logits = logits.masked_fill(~live[:, :, None], float("-inf"))
    if sink:
        logits = torch.nn.functional.pad(logits, (0, 1))
    w = logits.softmax(-1).nan_to_num(0.0)[..., : keys.shape[2]]
    return torch.einsum("bgrs,bgsd->bgrd", w, values.double().masked_fill(~live[..., None], 0)).reshape(b, h, D)


@pytest.mark.parametrize("b,g,slots", [
    (1, 8, 1024),    # a CU's worth of waves on each memory
    (1, 8, 256),     # six
    (2, 3, 80),      # an odd multiple of 16: fewer blocks than waves
    (2, 2, 48),      # too few blocks to share out
    (33, 8, 256),    # past one memory a CU: four
    (97, 8, 64),     # past three: two
])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_read_waves(gpu, b, g, slots, dtype):
    """bf16 2e-2, float32 1e-3 (the bounds of the other read tests)."""
    gen = torch.Generator().manual_seed(b + slots)
    q = torch.randn(b, 4 * g, D, generator=gen).to(dtype)
    keys, values = (torch.randn(b, g, slots, D, generator=gen).to(dtype) for _ in range(2))
    live = torch.rand(b, g, slots, generator=gen) < 0.7
    live[0, 0, slots // 2:] = False          # whole blocks dead
    live[-1, -1] = False                     # nothing live
    keys[~live] = float("nan")               # never reaches the sum
    values[~live] = float("inf")
    pos = torch.where(live, torch.arange(slots), -1).to(torch.int32)
    tol = 2e-2 if dtype == torch.bfloat16 else 1e-3

    def close(got, want):
        return ((got.cpu().double() - want).norm() / want.norm()).item() <= tol
    clean = keys.masked_fill(~live[..., None], 0)
    got = im.ring_decode_attention(q[:, None].to(gpu), keys.to(gpu), values.to(gpu), pos.to(gpu))
    assert close(got[:, 0], _reference(q, clean, values, live, False))
    st = im.IndependentMemoryState.empty(b, g, slots, 64, D, gpu, dtype)
    st.keys.copy_(keys)
    st.values.copy_(values)
    st.positions.copy_(pos)
    got = im.committed_gqa(q[:, None].to(gpu), st)
    assert close(got[:, 0], _reference(q, clean, values, live, True))
