"""The full-vocabulary draws where their digits, lists and ties decide (GPU):
the same tokens as a host selection over exact integer masses."""
import numpy as np
import pytest
import torch

from oracle import sampling
from yanchor_amd import inference_kernels as ik

pytestmark = pytest.mark.gpu


def _select(order, mass, t):
    """The first element of ``order`` whose inclusive mass reaches t, and that mass."""
    cum, last = 0, None
    for i in order:
        cum, last = cum + int(mass[i]), i
        if cum >= t:
            return i, cum
    return last, cum


@pytest.mark.parametrize("v", [1, 63, 1024, 5000])
@pytest.mark.parametrize("k,p", [(0, 1.0), (0, 0.9), (80, 0.7)])
@pytest.mark.parametrize("ties", ["none", "few_values", "one_value"])
def test_full_draws(gpu, v, k, p, ties):
    """Rows of every number of elements around the lists' 512; tied scores go
    by index.  A draw within 1e-6 of a boundary may fall on either side: the
    masses' exponentials are float32."""
    if k > v:
        pytest.skip("top_k above the vocabulary")
    gen = torch.Generator().manual_seed(v + k)
    b = 6
    x = torch.randn(b, v, generator=gen) * 2
    if ties == "few_values":
        x = x.round()
    if ties == "one_value":
        x.fill_(0.25)
    ids, steps = torch.arange(b) * 3, torch.arange(b) + 11
    got = ik.topk_sample(x.to(gpu), ids.to(gpu), steps.to(gpu), seed=77, temperature=0.7, top_k=k, top_p=p,
                         mode=ik.SAMPLE_TORCH).cpu().flatten().tolist()
    u = sampling.counter_uniform(ids, steps, seed=77).double().flatten().tolist()
    for r in range(b):
        xr = x[r].numpy()
        value_order = np.argsort(-xr, kind="stable")
        kept = value_order[: k if 1 < k < v else v]
        e = np.exp((xr.astype(np.float64) - xr.max()) / 0.7)
        mass = np.zeros(v, dtype=object)
        mass[kept] = [int(z) for z in e[kept] / e[kept].sum() * 2.0 ** 62]
        total = int(sum(mass[kept]))
        near = set()
        for shift in (-1e-6, 0.0, 1e-6):
            if k <= 0 and p == 1.0:
                near.add(_select(range(v), mass, max(1, int((u[r] + shift) * total)))[0])
            else:
                _, cut = _select(kept, mass, max(1, int(min(p + shift, 1.0) * total)))
                for s2 in (-1e-6, 0.0, 1e-6):
                    near.add(_select(kept, mass, max(1, int((u[r] + s2) * cut)))[0])
        assert got[r] in near, (r, got[r], near)


@pytest.mark.parametrize("v", [90, 600, 5000])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("k,p", [(0, 1.0), (0, 0.9), (80, 0.7)])
def test_rows_without_probabilities(gpu, v, dtype, k, p):
    """A NaN, +infinity or nothing above -infinity leaves no mass to draw from:
    the first element of the order, among rows that draw as they would alone."""
    gen = torch.Generator().manual_seed(v)
    x = torch.randn(6, v, generator=gen).to(dtype)
    x[1, [v // 2, v // 2 + 3]] = float("nan")
    x[2, [v - 1, 40]] = float("inf")
    x[3] = float("-inf")
    x[4, 5:] = float("-inf")          # five finite scores
    x = x.to(gpu)
    ids, steps = torch.arange(6, device=gpu) * 5, torch.arange(6, device=gpu)

    def draw(rows):
        return ik.topk_sample(x[rows], ids[rows], steps[rows], seed=3, temperature=0.8, top_k=k, top_p=p,
                              mode=ik.SAMPLE_TORCH).flatten().tolist()
    got = draw(list(range(6)))
    in_order = k <= 0 and p == 1.0
    assert got[1:4] == ([0, 0, 0] if in_order else [v // 2, 40, 0])
    assert 0 <= got[4] < 5
    assert [got[0], got[4], got[5]] == draw([0]) + draw([4]) + draw([5])
