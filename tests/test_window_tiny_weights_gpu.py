"""Softmax weights below 2^-126 of a row's largest count where their values are large: prompt rows of window attention on the bf16
kernels, within a tile of 32 keys and across tiles (the rescaling of what was summed before)."""
import math

import pytest
import torch

from vgate.ops import seq

pytestmark = pytest.mark.gpu


def _run(scores, values, device, kernel):
    """One sequence of one head; the score of key j is ln 2 times scores[j] for every query, its value values[j]."""
    n, D, page = len(scores), 32, 16
    pages = n // page
    kc, vc = (torch.zeros(pages, 1, page, D, dtype=torch.bfloat16) for _ in range(2))
    kc[:, 0, :, 0] = torch.tensor(scores, dtype=torch.bfloat16).view(pages, page)
    vc[:, 0] = torch.tensor(values, dtype=torch.bfloat16).view(pages, page, 1)
    q = torch.zeros(n, D, dtype=torch.bfloat16)
    q[:, 0] = 1
    out = torch.zeros(n, D, dtype=torch.bfloat16, device=device)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=device)  # noqa: E731
    vt = vc.transpose(2, 3).contiguous().to(device) if device == "cuda" else None
    seq.window_attn(q.to(device), kc.to(device), vc.to(device), None, None, i32([list(range(pages))]), i32([n]), i32([0, n]), out, math.log(2.0), 1,
                    4 * n, 0, None, None, vt=vt, prefill_kernel=kernel)
    return out.float().cpu()


@pytest.mark.parametrize("kernel", [0, 1])
@pytest.mark.parametrize("least", [-127, -130, -140])
def test_rescaled_sum_below_the_normal_range(least, kernel):
    n = 96
    scores, values = [-1000] * n, [0.0] * n
    scores[0], values[0] = 0, 2.0 ** 120
    scores[40] = -least                                       # from here on the first key's weight is 2^least
    got, want = _run(scores, values, "cuda", kernel), _run(scores, values, "cpu", kernel)
    assert (want[40:] > 0).all()
    # weights are exact powers of two but for the score's rounding: 2^-24 x 140 ln 2 ...; a weight below 2^-126 has at least 9 bits here
    assert ((got - want).abs() <= 2.0 ** -7 * want.abs()).all()


@pytest.mark.parametrize("kernel", [0, 1])
def test_weights_below_the_normal_range(kernel):
    n = 96
    scores, values = [-1000] * n, [0.0] * n
    scores[0] = 0
    scores[5], values[5] = -130, 2.0 ** 120
    got, want = _run(scores, values, "cuda", kernel), _run(scores, values, "cpu", kernel)
    assert ((got - want).abs() <= 2.0 ** -7 * want.abs()).all()
