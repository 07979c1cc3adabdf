"""Decoded tokens of hybrid models: latent attention whose keys several workgroups share, routing with its sort, narrow products and short
convolutions, against the ops' other forms; linear attention's chunks against 64 bits."""
import pytest
import torch

from vgate.ops import seq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rank,rot,H", [(128, 64, 8), (256, 64, 16), (512, 64, 12), (512, 64, 1), (512, 128, 16), (264, 64, 12), (200, 24, 5), (100, 64, 16), (96, 32, 3)])
@pytest.mark.parametrize("S", [1, 3, 40, 300])
def test_latent_attn_of_decoded_tokens(rank, rot, H, S):
    """Whole tiles (nothing clamped) and others, contexts from one key to some tiles per wave, one to eight workgroups per sequence. Values are
    at most 4: a softmax weight's rounding to bf16 moves a sum by 2^-9 of them, the result's by as much again."""
    g = torch.Generator().manual_seed(rank + H + S)
    E, lens = rank + rot, [1 + (i * 317 + 40 * (i % 3)) % 1100 if S < 100 else 1 + i % 70 for i in range(S)]
    pages = [-(-n // 16) for n in lens]
    cache = (torch.randn(sum(pages), 16, E, generator=g).clamp(-4, 4)).bfloat16()
    tables, at = torch.zeros(S, max(pages), dtype=torch.int32), 0
    order = torch.randperm(sum(pages), generator=g).int()
    for i, n in enumerate(pages):
        tables[i, :n] = order[at: at + n]
        at += n
    qa = torch.randn(S, H, E, generator=g).bfloat16()
    sink, start = torch.randn(H, generator=g), torch.arange(S + 1, dtype=torch.int32)
    ctx, scale = torch.tensor(lens, dtype=torch.int32), E ** -0.5
    tr = cache[:, :, :rank].transpose(1, 2).contiguous()
    for window in (seq.LATENT_FULL, 70):
        got, want = torch.empty(S, H, rank, dtype=torch.bfloat16, device="cuda"), torch.empty(S, H, rank)
        seq.latent_attn(qa.cuda(), cache.cuda(), tables.cuda(), ctx.cuda(), start.cuda(), got, scale, H, rank, rot, num_seqs=S, cache_t=tr.cuda(),
                        window=window, sink=sink.cuda())
        seq.latent_attn(qa.float(), cache.float(), tables, ctx, start, want, scale, H, rank, rot, num_seqs=S, window=window, sink=sink)
        assert ((got.float().cpu() - want).abs() <= 4 * 2.0 ** -8 + 1e-4).all()


@pytest.mark.parametrize("rank,rot", [(128, 64), (256, 64), (512, 64), (264, 64), (96, 32)])
def test_latent_attn_adds_its_waves_by_fused_steps(rank, rot, monkeypatch):
    """Two waves whose sums are A and -A, a third with the row's maximum, so that both are scaled by the same inexact f: o0 f rounded, then
    fma(o1, f, .) leaves the rounding of A f, at most 2^-24 of it and seldom none. (Both rounded ahead of the sum would leave zeros.)"""
    monkeypatch.setattr(seq, "LATENT_SPLIT", False)   # (one workgroup: waves take tiles of 32 keys in turn)
    H, E = 2, rank + rot
    g = torch.Generator().manual_seed(rank)
    A = torch.randn(rank, generator=g).bfloat16()
    cache = torch.zeros(6, 16, E, dtype=torch.bfloat16)
    cache[0, 0, :rank], cache[2, 0, :rank], cache[4, 0, rank] = A, -A, 1.3
    qa = torch.zeros(1, H, E, dtype=torch.bfloat16)
    qa[:, :, rank] = 1.0
    out = torch.empty(1, H, rank, dtype=torch.bfloat16, device="cuda")
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    seq.latent_attn(qa.cuda(), cache.cuda(), i32([[0, 1, 2, 3, 4, 5]]), i32([96]), i32([0, 1]), out, 1.0, H, rank, rot,
                    cache_t=cache[:, :, :rank].transpose(1, 2).contiguous().cuda())
    out = out.float().cpu()
    assert (out.abs() <= 2.0 ** -23 * A.float().abs()).all() and (out != 0).float().mean().item() > 0.8


@pytest.mark.parametrize("rank", [128, 256, 264, 512])
@pytest.mark.parametrize("T,S", [(1, 1), (32, 32), (48, 64), (64, 64), (96, 128), (128, 128), (256, 256), (300, 512)])
def test_latent_attn_parts(T, S, rank):
    """Two workgroups per CU in all, whatever the latent's size."""
    H, wg = 12, (T * 12 + 63) // 64 + S
    assert seq._C().latent_attn_split(T, S, H, rank, 64, False, 16)[0] == max(1, min(8, 512 // wg))


@pytest.mark.parametrize("rank,rot,H", [(256, 64, 8), (512, 64, 12), (264, 64, 12), (96, 32, 8)])
@pytest.mark.parametrize("lens", [[1] * 8 + [3], [1, 1, 4, 1, 1, 1, 1, 0] + [1] * 20, [1] * 60 + [9, 1, 0, 7], [0] * 300 + [1, 5, 1, 3] + [0] * 300])
def test_latent_attn_of_short_portions_among_decodes(rank, rot, H, lens):
    """Steps that count as decoding (at most 16 rows to a slot) with portions of more than 16 rows, whose waves take rows and not keys, beside
    sequences that several workgroups share (eight at first, one in the last list), and slots without tokens. Tolerance as above."""
    g = torch.Generator().manual_seed(rank + len(lens))
    S, T, E = len(lens), sum(lens), rank + rot
    if T * H > 16 * S:
        lens, S = lens + [0] * (T * H // 16 + 1 - S), T * H // 16 + 1
    ctx = [n + (i * 131) % 700 if n else 0 for i, n in enumerate(lens)]
    pages = [-(-c // 16) for c in ctx]
    cache = torch.randn(sum(pages), 16, E, generator=g).clamp(-4, 4).bfloat16()
    tables, at, start = torch.zeros(S, max(pages), dtype=torch.int32), 0, [0]
    for i, n in enumerate(pages):
        tables[i, :n] = torch.arange(at, at + n, dtype=torch.int32)
        at += n
        start.append(start[-1] + lens[i])
    assert (seq._C().latent_attn_split(T, S, H, rank, rot, False, 16)[0] == 1) == (S > 500) and max(lens) * H > 16
    qa, sink, scale = torch.randn(T, H, E, generator=g).bfloat16(), torch.randn(H, generator=g), E ** -0.5
    ctx, start = torch.tensor(ctx, dtype=torch.int32), torch.tensor(start, dtype=torch.int32)
    tr = cache[:, :, :rank].transpose(1, 2).contiguous()
    for window in (seq.LATENT_FULL, 70):
        got, want = torch.empty(T, H, rank, dtype=torch.bfloat16, device="cuda"), torch.empty(T, H, rank)
        seq.latent_attn(qa.cuda(), cache.cuda(), tables.cuda(), ctx.cuda(), start.cuda(), got, scale, H, rank, rot, num_seqs=S, cache_t=tr.cuda(),
                        window=window, sink=sink.cuda())
        seq.latent_attn(qa.float(), cache.float(), tables, ctx, start, want, scale, H, rank, rot, num_seqs=S, window=window, sink=sink)
        assert ((got.float().cpu() - want).abs() <= 4 * 2.0 ** -8 + 1e-4).all()


@pytest.mark.parametrize("score", [seq.ROUTE_SIGMOID, seq.ROUTE_SOFTMAX, seq.ROUTE_TOP_SOFTMAX])
@pytest.mark.parametrize("T,E,top", [(1, 1, 1), (7, 8, 2), (16, 64, 6), (16, 65, 4), (17, 60, 60), (16, 64, 4), (16, 64, 5), (2, 64, 32), (1, 64, 64), (65, 8, 2), (40, 65, 4), (33, 512, 8), (5, 600, 3)])
def test_moe_route_sort(T, E, top, score):
    """One launch and two, on either side of their line: the choice and weights of the CPU form, every pair in its expert's stretch once."""
    g = torch.Generator().manual_seed(T + E)
    z, corr = torch.randn(T, E, generator=g), 0.1 * torch.randn(E, generator=g)

    def run(dev):
        idx, wts = torch.empty(T, top, dtype=torch.int32, device=dev), torch.empty(T, top, device=dev)
        rows, pos, off = (torch.full((n,), -1, dtype=torch.int32, device=dev) for n in (T * top, T * top, E + 1))
        seq.moe_route_sort(z.to(dev), corr.to(dev), top, 1e-20, idx, wts, rows, pos, off, score=score, scale=1.5)
        return [t.cpu() for t in (idx, wts, rows, pos, off)]

    (idx, wts, rows, pos, off), want = run("cuda"), run("cpu")
    assert torch.equal(idx, want[0]) and torch.allclose(wts, want[1], rtol=1e-5, atol=1e-7) and torch.equal(off, want[4])
    assert sorted(pos.tolist()) == list(range(T * top))
    token = torch.arange(T * top) // top
    assert torch.equal(rows[pos.long()], token.int())
    assert (off[idx.flatten().long()] <= pos).all() and (pos < off[idx.flatten().long() + 1]).all()


@pytest.mark.parametrize("M", [1, 15, 16, 17, 33, 2047, 4096, 4097])
@pytest.mark.parametrize("N,K", [(1, 264), (8, 1024), (16, 520), (72, 512), (17, 1000), (128, 2056)])
def test_narrow_products(M, N, K):
    """Workgroups of 16 rows and of 64, on either side of their line, ragged columns and k. fp32 sums of products of bf16: |error| below
    K 2^-24 of the sum of the products' sizes."""
    g = torch.Generator().manual_seed(M + N)
    a, w, w2 = (torch.randn(r, K, generator=g).bfloat16().cuda() for r in (M, N, N))
    bias = torch.randn(N, generator=g).cuda()
    bound = (a.float().abs() @ w.float().abs().t()).max().item() * K * 2.0 ** -24 + 1e-6
    out = torch.empty(M, N, device="cuda")
    seq.gemm(a, w, out, bias=bias)
    want = a.double() @ w.double().t() + bias
    assert (out - want).abs().max().item() <= bound
    seq.gemm(a, w, out, w2=w2, act=seq.ACT_SILU_MUL)
    gate, up = a.double() @ w.double().t(), a.double() @ w2.double().t()
    assert (out - torch.nn.functional.silu(gate) * up).abs().max().item() <= bound * (1.1 * up.abs().max().item() + gate.abs().max().item())


@pytest.mark.parametrize("C", [8, 2056])
@pytest.mark.parametrize("taps", [1, 3, 4])
@pytest.mark.parametrize("lens", [[1] * 70, [1] * 64 + [0, 3, 0], [5] * 110, [0, 700, 0, 9, 3], [1]])
def test_short_conv_runs(C, taps, lens):
    """Workgroups of one token, one and several of channels, sequences of one token to hundreds, some without a slot or without tokens, rows
    past the last sequence: the bits of the kernel for rows that are not of whole pieces."""
    g = torch.Generator().manual_seed(C + taps + len(lens))
    T, S = sum(lens), len(lens)
    x = torch.randn(T + 5, 2 * C, generator=g).bfloat16().cuda()[:, C:]
    w, b, kept = (torch.randn(s, generator=g).cuda() for s in ((taps, C), (C,), (S, taps - 1, C)))
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    slots = i32([-1 if s % 5 == 3 else S - 1 - s for s in range(S)])
    ctx, start = i32([n + (13 if s % 2 else 0) for s, n in enumerate(lens)]), i32([sum(lens[:s]) for s in range(S + 1)])
    a, o = torch.full((T + 5, C), 7.0, dtype=torch.bfloat16, device="cuda"), torch.full((T + 5, C + 1), 7.0, dtype=torch.bfloat16, device="cuda")[:, 1:]
    for silu in (False, True):
        seq.short_conv(x, w, b, kept, slots, ctx, start, a, silu=silu)
        seq.short_conv(x, w, b, kept, slots, ctx, start, o, silu=silu)
        assert torch.equal(a, o) and bool((a[T:] == 7.0).all())


@pytest.mark.parametrize("C", [1536, 4104])
@pytest.mark.parametrize("taps", [1, 2, 3, 4])
@pytest.mark.parametrize("lens", [[1, 1, 1, 1, 1, 700, 1, 2, 3, 701], [300, 1, 1, 2, 301, 0, 900], [1, 2] * 400 + [500], [1] * 9 + [0, 1500, 0, 1], [1] * 1400 + [9]])
def test_short_conv_of_prompts_among_decodes(C, taps, lens):
    """Two tokens a workgroup (all lists but the last, which has fewer than two tokens to a sequence): sequences that share one, those shorter
    than the taps, kept rows read from either of its tokens, sequences without a slot: the bits of the kernel for rows that are not of whole
    pieces."""
    T, S = sum(lens), len(lens)
    two = T * C >= 1 << 21 and T >= 2 * S   # the launcher's rule
    assert two == (lens[0:10] != [1] * 10)
    g = torch.Generator().manual_seed(C + taps + S)
    x = torch.randn(T, C + 8, generator=g).bfloat16().cuda()[:, 8:]
    w, b, kept = (torch.randn(s, generator=g).cuda() for s in ((taps, C), (C,), (S, taps - 1, C)))
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    slots = i32([-1 if s % 7 == 4 else S - 1 - s for s in range(S)])
    ctx, start = i32([n + (13 if s % 4 else 0) for s, n in enumerate(lens)]), i32([sum(lens[:s]) for s in range(S + 1)])
    a, o = torch.full((T, C), 7.0, dtype=torch.bfloat16, device="cuda"), torch.full((T, C + 1), 7.0, dtype=torch.bfloat16, device="cuda")[:, 1:]
    seq.short_conv(x, w, b, kept, slots, ctx, start, a, silu=True)
    seq.short_conv(x, w, b, kept, slots, ctx, start, o, silu=True)
    assert torch.equal(a, o)


@pytest.mark.parametrize("mode", ["gated", "head", "bonus"])
@pytest.mark.parametrize("D,V", [(128, 128), (72, 24), (64, 64), (24, 40)])
@pytest.mark.parametrize("n", [129, 144, 145, 176, 191, 192, 255, 300])
def test_linear_attention_chunks(mode, D, V, n):
    """Portions whose last chunk of 64 ends at and around each 16 tokens, fp32, a state before them, against the recurrence in 64 bits. An
    output is sums of D and of 64 terms, rounded some (D + 64) times by 2^-24 at most."""
    g = torch.Generator().manual_seed(n + D)
    H, d = 2, "cuda"
    q, k, v, z = (torch.randn(n, H * w, generator=g).to(d) for w in (D, D, V, D))
    state = torch.randn(1, H, D, V, generator=g).to(d)
    bonus = torch.randn(H, D, generator=g).to(d) if mode == "bonus" else None
    fade = torch.tensor([0.5, 0.97], device=d) if mode == "head" else None
    if mode == "head":
        a, z = fade.double()[None, :, None].expand(n, H, D), None
    elif mode == "bonus":
        z = z - 2.0
        a = torch.exp(-torch.exp(z.double())).view(n, H, D)
    else:
        a = torch.exp(torch.nn.functional.logsigmoid(z.double()) / 4.0).view(n, H, D)
    S, want = state[0].double(), torch.empty(n, H, V, dtype=torch.float64, device=d)
    for t in range(n):
        kv = k[t].double().view(H, D, 1) * v[t].double().view(H, 1, V)
        new = a[t][:, :, None] * S + kv
        read = S + bonus.double()[:, :, None] * kv if mode == "bonus" else new
        want[t], S = (read * q[t].double().view(H, D, 1)).sum(1), new
    want = want / torch.sqrt((want * want).mean(-1, keepdim=True) + 1e-6)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=d)  # noqa: E731
    out, gate = torch.empty(n, H * V, device=d), torch.full((n, H * V), 40.0, device=d)
    seq.linear_attn(q, k, v, gate, z, fade, 4.0, 1.0, False, None, False, False, state, i32([0]), i32([n + 7]), i32([0, n]), out, 1e-6,
                    decay_exp=mode == "bonus", bonus=bonus)
    for got, exact in ((out.view(n, H, V), want), (state[0], S)):
        assert ((got.double() - exact).norm() / exact.norm()).item() < (D + 64) * 2.0 ** -24


@pytest.mark.parametrize("bonus", [False, True])
@pytest.mark.parametrize("D,V", [(128, 128), (64, 64), (24, 64)])
def test_linear_attention_weights_keys_token_by_token(D, V, bonus):
    """What a token of the first chunk of 64 reads of each key: the key times the decays after it, one token at a time in fp32, then times the
    query, whatever the tokens' distance. One channel is used, token j's value is 1 in column j, and eps is 2^60: nothing else rounds."""
    n, fade, d = 200, torch.tensor([0.97], dtype=torch.float32), min(D - 1, 37)
    g = torch.Generator().manual_seed(D + V)
    q, k = torch.zeros(n, D), torch.zeros(n, D)
    q[:, d], k[:, d] = torch.randn(n, generator=g), torch.randn(n, generator=g)
    v = torch.zeros(n, V)
    v[torch.arange(64), torch.arange(64)] = 1.0
    u = torch.randn(1, D, generator=g)
    want = torch.zeros(64, 64)
    for j in range(64):
        x = k[j, d]
        want[j, j] = q[j, d] * x
        if bonus:
            want[j, j] = (q[j, d] * u[0, d]) * x
        for i in range(j + 1, 64):
            if bonus:
                want[i, j] = q[i, d] * x
            x = x * fade[0]
            if not bonus:
                want[i, j] = q[i, d] * x
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    out, state = torch.empty(n, V, device="cuda"), torch.zeros(1, 1, D, V, device="cuda")
    seq.linear_attn(q.cuda(), k.cuda(), v.cuda(), torch.full((n, V), 40.0, device="cuda"), None, fade.cuda(), 1.0, 1.0, False, None, False, False,
                    state, i32([0]), i32([n]), i32([0, n]), out, 2.0 ** 60, bonus=u.cuda() if bonus else None)
    assert torch.equal(out[:64, :64].cpu() * 2.0 ** 30, want)
