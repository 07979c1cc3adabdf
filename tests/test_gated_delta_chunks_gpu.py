"""The gated delta rule's two forms (chunks, tokens one by one in one launch) against the op's CPU form, at the sizes where
chunks, staged tokens and tiles end, where one form hands over to the other, and with rows of padding."""
import pytest
import torch

from vgate.ops import seq

pytestmark = pytest.mark.gpu


def _run(H, G, D, V, taps, lens, pos, dt, seed, device, pad):
    g = torch.Generator().manual_seed(seed)
    T, S, n = sum(lens), len(lens), G * D
    rows = torch.randn(T + pad, 2 * n + H * V + H + 8, generator=g).to(dt)      # columns of one fused projection
    zg = torch.randn(T + pad, H * (D + V), generator=g)
    decay, nw = torch.rand(H, generator=g), 1 + 0.1 * torch.randn(V, generator=g)
    conv_w = torch.randn(taps, 2 * n + H * V, generator=g) * taps ** -0.5
    state, kept = torch.randn(S + 2, H, D, V, generator=g), torch.randn(S + 2, taps - 1, 2 * n + H * V, generator=g)
    slots = torch.randperm(S + 2, generator=g)[:S].int()
    ctx = torch.tensor([p + m for p, m in zip(pos, lens)], dtype=torch.int32)
    qs = torch.tensor([0] + lens, dtype=torch.int32).cumsum(0).int()
    rows, zg, decay, nw, conv_w, state, kept, slots, ctx, qs = (
        x.to(device) for x in (rows, zg, decay, nw, conv_w, state, kept, slots, ctx, qs))
    out = torch.zeros(T + pad, H * V, dtype=dt, device=device)
    a, b = 2 * n, 2 * n + H * V
    seq.gated_delta(rows[:, :n], rows[:, n:a], rows[:, a:b], rows[:, b: b + H], zg[:, : H * D], zg[:, H * D:], decay, nw, conv_w, state,
                    kept, slots, ctx, qs, out, 1e-6, D ** -0.5, 1e-6)
    return out[:T].float().cpu(), state.cpu(), kept.cpu()


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,G,D,V,taps", [(2, 2, 5, 7, 4), (3, 3, 32, 32, 2), (2, 2, 33, 20, 1), (3, 3, 64, 48, 4), (2, 2, 24, 100, 3),
                                          (5, 5, 128, 128, 4), (4, 2, 32, 64, 4)])
@pytest.mark.parametrize("lens,pos,pad", [([1], [0], 0), ([1] * 9, [3] * 9, 7), ([7, 1, 8, 9, 2], [5, 1, 0, 0, 2], 3), ([64], [3], 0),
                                          ([65], [1], 5), ([1] * 24 + [31, 32, 33, 40, 7, 8, 9, 95], [2] * 32, 5), ([48, 49, 1, 64], [0, 3, 40, 0], 9), ([20], [3], 200), ([1], [6], 300),
                                          ([1] * 6 + [161], [9] * 7, 0), ([3, 30], [0, 2], 130)])
def test_matches_cpu_form(H, G, D, V, taps, lens, pos, pad, dt):
    got, want = (_run(H, G, D, V, taps, lens, pos, dt, 3 * H + D, d, pad) for d in ("cuda", "cpu"))
    # both sum fp32 products in other orders: a state entry gathers up to 161 updates of size ~ 1 and D-term sums under decays
    # < 1, relative error of the whole below 2^-24 x (161 + D) x a few; a bf16 result rounds by 2^-8
    rel = lambda a, b: float((a - b).norm() / b.norm())  # noqa: E731
    assert rel(got[0], want[0]) < (2e-5 if dt == torch.float32 else 2.0 ** -8)
    assert rel(got[1], want[1]) < 2e-5
    assert torch.equal(got[2], want[2])    # (copies of inputs)
