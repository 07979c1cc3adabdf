"""The generalized delta rule's two forms (chunks, tokens one by one) against the op's CPU form, at the sizes where chunks,
staged tokens and tiles end and where one form hands over to the other."""
import pytest
import torch

from vgate.ops import seq

pytestmark = pytest.mark.gpu


def _inputs(H, D, lens, pos, dt, seed, device, pad=3):
    g = torch.Generator().manual_seed(seed)
    T, n, S = sum(lens), H * D, len(lens)
    P = torch.randn(T + pad, 5 * n + 8, generator=g).to(dt)     # columns of one fused projection, with padding rows
    cols = [P[:, i * n: (i + 1) * n] for i in range(5)]
    t = dict(r=cols[0], k=cols[1], v=cols[2], g=cols[3], a=cols[4], wl=torch.randn(T + pad, n, generator=g).to(dt),
             w0=torch.randn(n, generator=g), ab=torch.randn(n, generator=g), nw=1 + 0.1 * torch.randn(n, generator=g),
             state=torch.randn(S + 2, H, D, D, generator=g))
    slots = torch.randperm(S + 2, generator=g)[:S].int()
    ctx = torch.tensor([p + m for p, m in zip(pos, lens)], dtype=torch.int32)
    qs = torch.tensor([0] + lens, dtype=torch.int32).cumsum(0).int()
    P = P.to(device)
    moved = {k: P[:, i * n: (i + 1) * n] for i, k in enumerate("rkvga")}
    moved.update({k: v.to(device) for k, v in t.items() if k not in moved})
    return moved, slots.to(device), ctx.to(device), qs.to(device), torch.zeros(T + pad, n, dtype=dt, device=device)


def _run(H, D, lens, pos, dt, seed, device, pad=3):
    t, slots, ctx, qs, out = _inputs(H, D, lens, pos, dt, seed, device, pad)
    seq.delta_rule(t["r"], t["k"], t["v"], t["g"], t["a"], t["wl"], t["w0"], t["ab"], t["nw"], t["state"], slots, ctx, qs, out,
                   0.6, 1e-6, 1e-6)
    return out[: sum(lens)].float().cpu(), t["state"].cpu()


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,D", [(1, 1), (2, 5), (3, 32), (2, 33), (3, 64), (1, 100), (9, 128)])
@pytest.mark.parametrize("lens,pos", [([128], [0]), ([161], [7]), ([48, 49, 1, 64], [0, 3, 40, 0]), ([1] * 12 + [117], [9] * 13),
                                      ([33, 95], [1, 0]), ([1], [0]), ([7, 1, 8, 9], [5, 1, 0, 0]), ([64], [3]), ([1] * 70, [2] * 70)])
def test_matches_cpu_form(H, D, lens, pos, dt):
    out, state = _run(H, D, lens, pos, dt, 3 * H + D, "cuda")
    want, state_w = _run(H, D, lens, pos, dt, 3 * H + D, "cpu")
    # both sum fp32 products in other orders: a state entry gathers up to 161 updates of size ~ 1 and D-term sums under decays
    # < 1, relative error of the whole below 2^-24 x (161 + D) x a few; a bf16 result rounds by 2^-8
    rel = lambda a, b: float((a - b).norm() / b.norm())  # noqa: E731
    assert rel(state, state_w) < 2e-5
    assert rel(out, want) < (2e-5 if dt == torch.float32 else 2.0 ** -8)


@pytest.mark.parametrize("lens,pos,pad", [([20], [3], 80), ([1], [0], 300), ([48], [1], 17), ([49], [0], 64), ([3, 30], [0, 2], 130)])
def test_fewer_tokens_than_rows(lens, pos, pad):
    """A step's rows are padded to a size of their own: few tokens among many rows."""
    out, state = _run(3, 64, lens, pos, torch.float32, 11, "cuda", pad)
    want, state_w = _run(3, 64, lens, pos, torch.float32, 11, "cpu", pad)
    assert float((state - state_w).norm() / state_w.norm()) < 2e-5   # (as above)
    assert float((out - want).norm() / want.norm()) < 2e-5


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,D", [(1, 1), (2, 5), (3, 33), (3, 64), (1, 100), (5, 128)])
@pytest.mark.parametrize("lens,pos", [([9], [0]), ([16], [7]), ([92], [3]), ([125], [0]), ([1, 11], [5, 0]), ([17, 30, 1, 9], [0, 3, 40, 1]), ([96, 1, 95], [0, 2, 9]),
                                      ([1, 129, 3], [4, 0, 9]), ([97, 96, 1], [0, 5, 2]), ([130, 128, 1, 20], [0, 1, 2, 3])])
def test_token_scan(H, D, lens, pos, dt):
    """Steps around the lines of the token scan, with staged tokens that fill their eight and do not, and with a longer portion in
    chunks beside it."""
    out, state = _run(H, D, lens, pos, dt, H + D, "cuda")
    want, state_w = _run(H, D, lens, pos, dt, H + D, "cpu")
    rel = lambda a, b: float((a - b).norm() / b.norm())  # noqa: E731
    assert rel(state, state_w) < 2e-5   # (as above)
    assert rel(out, want) < (2e-5 if dt == torch.float32 else 2.0 ** -8)


@pytest.mark.parametrize("S", [97, 128, 200])
def test_many_decoded_tokens(S):
    """One token each, after others: at position 0 the output is (k . r) v and its norm blows up what rounding leaves of a k . r near
    zero (fp32 on the CPU is off by 3e-4 of a token's output at S = 200 then, by 3e-7 here)."""
    out, state = _run(2, 64, [1] * S, [3] * S, torch.float32, S, "cuda", 0)
    want, state_w = _run(2, 64, [1] * S, [3] * S, torch.float32, S, "cpu", 0)
    assert float((state - state_w).norm() / state_w.norm()) < 2e-5   # (as above)
    assert float((out - want).norm() / want.norm()) < 2e-5


def test_scratch_of_the_scan_alone():
    """With no more scratch than the token scan's, a step that would take chunks takes the scan."""
    from vgate import ops
    lens, pos, H, D = [200], [4], 3, 64
    t, slots, ctx, qs, out = _inputs(H, D, lens, pos, torch.float32, 1, "cuda")
    scratch = torch.empty(6 * out.numel(), device="cuda")
    assert scratch.numel() < ops.native().delta_rule_scratch(out.shape[0], H, D)
    ops.native().delta_rule(t["r"], t["k"], t["v"], t["g"], t["a"], t["wl"], t["w0"], t["ab"], t["nw"], t["state"], slots, ctx, qs, out,
                            0.6, 1e-6, 1e-6, scratch)
    want, state_w = _run(H, D, lens, pos, torch.float32, 1, "cpu")
    assert float((t["state"].cpu() - state_w).norm() / state_w.norm()) < 2e-5   # (as above)
    assert float((out[:200].cpu() - want).norm() / want.norm()) < 2e-5
