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


@pytest.mark.parametrize("S", [1, 5, 300])
@pytest.mark.parametrize("part", [64, 512])
def test_equal_and_whole_partitions(S, part):
    """Contexts around one, two and three partitions, in launches few enough for equal parts and too many: one partition's result."""
    Hq, Hkv, D, dev = 12, 2, 128, "cuda"
    g = torch.Generator(dev).manual_seed(S + part)
    rand = lambda *s: torch.randn(*s, device=dev, generator=g).bfloat16()  # noqa: E731
    lens = [part - 1, part, part + 1, 2 * part - 31, 2 * part, 2 * part + 1, 3 * part - 1, 1]
    ctx = [lens[i % len(lens)] for i in range(S)] if S > 1 else [2 * part + 1]
    blocks = 3 * part // 16
    kc, vc = rand(64, Hkv, 16, D), rand(64, Hkv, 16, D)
    bt = torch.randint(0, 64, (S, blocks), device=dev, generator=g).int()
    cl, qs = torch.tensor(ctx, dtype=torch.int32, device=dev), torch.arange(S + 1, device=dev).int()
    q, none = rand(S, Hq * D), torch.empty(0, dtype=torch.int32, device=dev)
    outs = []
    for size in (part, 1024 if part == 64 else 512):
        P = -(-blocks * 16 // size)
        po, pml = torch.zeros(S, Hq, P, D, device=dev), torch.zeros(S, Hq, P, 2, device=dev)
        out = torch.zeros(S, Hq * D, device=dev).bfloat16()
        ops.attention(q, Hq * D, kc, vc, bt, cl, qs, none, none, out, po, pml, Hq, Hkv, size, D ** -0.5)
        outs.append(out.float())
    n = [c for c in ctx]
    k = torch.stack([kc[bt[i].long()].transpose(1, 2).reshape(-1, Hkv, D)[: max(n)] for i in range(S)]).float()
    v = torch.stack([vc[bt[i].long()].transpose(1, 2).reshape(-1, Hkv, D)[: max(n)] for i in range(S)]).float()
    qq = q.float().view(S, Hkv, Hq // Hkv, D)
    sc = torch.matmul(qq, k.permute(0, 2, 3, 1).contiguous()) * D ** -0.5
    sc = sc.masked_fill(torch.arange(max(n), device=dev) >= cl.view(S, 1, 1, 1), float("-inf"))
    want = torch.matmul(sc.softmax(-1), v.permute(0, 2, 1, 3).contiguous()).reshape(S, Hq * D)
    for out in outs:   # weights rounded to bf16 (2^-9 each, of values of size ~ 1 that average out) and a bf16 result
        assert float((out - want).norm() / want.norm()) < 2.0 ** -7


@pytest.mark.parametrize("S,Hq,Hkv,ctx", [(64, 32, 8, 600), (64, 12, 2, 1300), (16, 32, 8, 600), (64, 12, 2, 600), (300, 12, 2, 600)])
def test_partitions_do_not_depend_on_the_room_for_longer_contexts(S, Hq, Hkv, ctx):
    """The same contexts with block tables (and partial results) for 1, 4 and 16 times as many tokens: the same bits."""
    D, part, dev = 128, 512, "cuda"
    g = torch.Generator(dev).manual_seed(S)
    rand = lambda *s: torch.randn(*s, device=dev, generator=g).bfloat16()  # noqa: E731
    used = -(-ctx // 16)
    kc, vc = rand(256, Hkv, 16, D), rand(256, Hkv, 16, D)
    pages = torch.randint(0, 256, (S, used), device=dev, generator=g).int()
    cl = torch.tensor([ctx - i % 7 for i in range(S)], dtype=torch.int32, device=dev)
    q, qs, none = rand(S, Hq * D), torch.arange(S + 1, device=dev).int(), torch.empty(0, dtype=torch.int32, device=dev)
    outs = []
    for room in (1, 4, 16):
        bt = torch.zeros(S, used * room, dtype=torch.int32, device=dev)
        bt[:, :used] = pages
        P = -(-used * room * 16 // part)
        po, pml = torch.zeros(S, Hq, P, D, device=dev), torch.zeros(S, Hq, P, 2, device=dev)
        out = torch.zeros(S, Hq * D, device=dev).bfloat16()
        ops.attention(q, Hq * D, kc, vc, bt, cl, qs, none, none, out, po, pml, Hq, Hkv, part, D ** -0.5)
        outs.append(out)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
