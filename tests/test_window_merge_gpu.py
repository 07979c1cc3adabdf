"""Window attention of decoded tokens whose keys several workgroups share: what the merge of their results makes of infinite values."""
import pytest
import torch

from vgate.ops import seq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("window,n,parts", [(400, 400, 2), (1000, 992, 4)])
@pytest.mark.parametrize("key", [3, -20])
def test_infinite_value_in_one_column_of_a_turned_pair(window, n, parts, key):
    """Both columns of the pair are infinite, as the turn makes them, not NaN; the others are as they would be without it. Values are at most
    4: a softmax weight's rounding to bf16 moves a sum by 2^-9 of them, the result's by as much again."""
    H, G, D, V, page = 4, 2, 32, 32, 16
    assert seq._C().window_attn_split(1, 1, H, G, D, V, False, page, window, 0, 0, 0)[0] == parts
    key %= n   # (of the first part, of the last)
    g = torch.Generator().manual_seed(window + key)
    kc, vc = (torch.randn(n // page, G, page, D, generator=g).clamp(-4, 4).bfloat16() for _ in range(2))
    vc[key // page, :, key % page, 5] = float("inf")
    q, freq = torch.randn(1, H * D, generator=g).bfloat16(), seq.rope_inv_freq(V, 10000.0, "cpu")

    def run(dev, dt):
        i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)  # noqa: E731
        out = torch.empty(1, H * V, dtype=dt, device=dev)
        vt = vc.transpose(2, 3).contiguous().cuda() if dev == "cuda" else None
        seq.window_attn(q.to(dev, dt), kc.to(dev, dt), vc.to(dev, dt), None, None, i32([list(range(n // page))]), i32([n]), i32([0, 1]), out,
                        D ** -0.5, H, window, 0, None, freq.to(dev), vt=vt)
        return out.float().cpu().view(H, V)

    got, want = run("cuda", torch.bfloat16), run("cpu", torch.float32)
    pair = torch.zeros(V, dtype=torch.bool)
    pair[4:6] = True
    assert torch.isinf(want[:, pair]).all() and torch.equal(got[:, pair], want[:, pair])
    assert ((got - want)[:, ~pair].abs() <= 4 * 2.0 ** -8 + 1e-4).all()
