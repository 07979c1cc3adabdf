"""A step whose tokens fill its rows exactly, beside padding sequences that start where the rows end: the padding changes no
result and reads nothing of what lies behind the queries."""
import pytest
import torch

from vgate import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Hq,Hkv", [(12, 2), (32, 8)])
@pytest.mark.parametrize("lens,ctxs", [([1, 1, 1], [5, 70, 300]), ([1, 40, 23], [700, 40, 90]), ([500, 9], [500, 30])])
def test_padding_sequences_behind_full_rows(Hq, Hkv, lens, ctxs):
    D, dev, n, T = 128, "cuda", len(lens), sum(lens)
    g = torch.Generator(dev).manual_seed(T)
    rand = lambda *s: torch.randn(*s, device=dev, generator=g).bfloat16()  # noqa: E731
    blocks = 50
    kc, vc = rand(n * blocks, Hkv, 16, D), rand(n * blocks, Hkv, 16, D)
    behind = rand(T + 1, Hq * D)
    behind[T] = float("nan")
    q = behind[:T]
    ts, tq = ops.prefill_tiles([m if m > 1 else 0 for m in lens], ops.flash_lead(Hq, Hkv))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=dev)  # noqa: E731
    ts, tq = i32(ts + [-1]), i32(tq + [0])
    outs = []
    for pad in (0, 3):
        S = n + pad
        bt = torch.zeros(S, blocks, dtype=torch.int32, device=dev)
        bt[:n] = torch.arange(n * blocks, device=dev).int().view(n, blocks)
        cl, qs = i32(ctxs + [0] * pad), i32([sum(lens[:i]) for i in range(n + 1)] + [T] * pad)
        po, pml = torch.zeros(S, Hq, 2, D, device=dev), torch.zeros(S, Hq, 2, 2, device=dev)
        out = torch.zeros(T, Hq * D, device=dev).bfloat16()
        ops.attention(q, Hq * D, kc, vc, bt, cl, qs, ts, tq, out, po, pml, Hq, Hkv, 512, D ** -0.5)
        outs.append(out)
    assert torch.isfinite(outs[0].float()).all() and torch.equal(outs[0], outs[1])
