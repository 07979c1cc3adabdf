"""The medium-row GEMMs (17 .. 64 rows) at the edges of their images of x: three m-tiles at once and two, K that ends within a 64-k tile, K slices and
whole tiles, a folded norm and a residual in place."""
import pytest
import torch

from vgate import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [17, 32, 33, 40, 48, 49, 64])
@pytest.mark.parametrize("N,K", [(4608, 992), (8192, 1024), (6464, 1664), (4608, 1696), (4096, 2016), (1536, 4128), (512, 2336), (1536, 1536)])
def test_rows_of_a_mixed_step(M, N, K):
    torch.manual_seed(M + N + K)
    rand = lambda *s: torch.randn(*s, device="cuda")  # noqa: E731
    w, x, gamma = (rand(N, K) * K ** -0.5).bfloat16(), rand(M, K + 8).bfloat16()[:, :K], (torch.rand(K, device="cuda") + 0.5).bfloat16()
    res = rand(M, N).bfloat16()
    # fp32 sums of K products of size ~ K^-1/2 in another order, bf16 once before and once after the residual
    close = lambda got, want: bool(((got.float() - want).abs() <= 2.0 ** -7 * want.abs() + 16.0 * K * 2.0 ** -24 + 2.0 ** -7).all())  # noqa: E731
    want = x.float() @ w.float().t()
    out = res.clone()
    ops.linear(x, ops.Linear(w), out=out, residual=out)
    assert close(out, want + res.float())
    nl = ops.Linear(w.clone(), kind="silu")
    assert nl.fold_norm(gamma)
    xn = x.float() * torch.rsqrt((x.float() ** 2).mean(-1, keepdim=True) + 1e-6)
    y = xn @ (w.float() * gamma.float()).bfloat16().float().t()
    for forced in (None, dict(path=2, waves=8), dict(path=2, waves=4)):
        got = ops.linear(x, nl, norm=(gamma, 1e-6), **(forced or {}))
        assert close(got, torch.nn.functional.silu(y[:, : N // 2]) * y[:, N // 2:])


@pytest.mark.parametrize("M", [17, 32, 41, 64])
@pytest.mark.parametrize("N,K", [(512, 32), (512, 96), (544, 480), (5376, 224), (8512, 160), (8256, 544), (1296, 1312), (12352, 416), (20992, 96), (528, 2016)])
def test_images_of_few_and_uneven_waves(M, N, K):
    """One to eight waves stage an image of one to 32 tiles, the last of them whole or half: by halves of tiles dealt out to the waves, and
    (two to a 16-row tile) by a piece of every tile each."""
    torch.manual_seed(M + N + K)
    w, x = (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16(), torch.randn(M, K + 8, device="cuda").bfloat16()
    x[:, K:] = float("nan")   # (nothing past K counts)
    lin, want = ops.Linear(w), x[:, :K].float() @ w.float().t()
    for forced in (None, dict(path=2, waves=8), dict(path=2, waves=1), dict(path=2, waves=2), dict(path=2, waves=4)):
        got = ops.linear(x[:, :K], lin, out_f32=True, **(forced or {}))
        assert ((got - want).abs() <= 8.0 * K * 2.0 ** -24 + 1e-6).all(), forced


@pytest.mark.parametrize("M", [17, 25, 33, 64])
@pytest.mark.parametrize("N,K", [(8192, 1024), (8256, 2560), (12352, 2112), (32000, 1536), (28672, 2176), (25600, 576)])
def test_many_columns_of_a_mixed_step(M, N, K):
    """Four-wave tiles of 64 and 128 columns: LM heads whose rows come from anywhere in x, and pairs with a norm folded in."""
    torch.manual_seed(M + N + K)
    w, gamma = (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16(), (torch.rand(K, device="cuda") + 0.5).bfloat16()
    x = torch.randn(300, K + 8, device="cuda").bfloat16()[:, :K]
    rows = torch.randint(0, 300, (M,), device="cuda", dtype=torch.int32)
    rows[0], rows[-1] = 299, 0
    y = x[rows.long()].float()
    yn = y * torch.rsqrt((y ** 2).mean(-1, keepdim=True) + 1e-6)
    head = ops.Linear(w.clone())
    out = torch.full((M + 1, N + 8), 7.0, device="cuda")
    ops.linear(x, head, out=out[:M, :N], out_f32=True, row_idx=rows)
    assert ((out[:M, :N] - y @ w.float().t()).abs() <= 8.0 * K * 2.0 ** -24 + 1e-6).all()
    assert bool((out[M] == 7).all() and (out[:, N:] == 7).all())
    assert head.fold_norm(gamma)
    wg = (w.float() * gamma.float()).bfloat16().float()
    got = ops.linear(x, head, out_f32=True, row_idx=rows, norm=(gamma, 1e-6))
    assert ((got - yn @ wg.t()).abs() <= 32.0 * K * 2.0 ** -24 + 1e-5).all()
    pair = ops.Linear(w.clone(), kind="silu")
    assert pair.fold_norm(gamma)
    got, want = ops.linear(x[:M], pair, norm=(gamma, 1e-6)), x[:M].float()
    want = (want * torch.rsqrt((want ** 2).mean(-1, keepdim=True) + 1e-6)) @ wg.t()
    want = torch.nn.functional.silu(want[:, : N // 2]) * want[:, N // 2:]
    assert ((got.float() - want).abs() <= 2.0 ** -7 * want.abs() + 2.0 ** -7).all()


@pytest.mark.parametrize("M", [17, 48])
@pytest.mark.parametrize("N,K", [(32768, 256), (62208, 512), (62336, 512), (65536, 256), (65536, 320), (65600, 512), (98304, 512)])
def test_heads_of_short_k_behind_a_norm(M, N, K):
    """Blocks of 128 columns that fill whole rounds of CUs, and nearly, on either side of the lines to four-wave tiles."""
    test_many_columns_of_a_mixed_step(M, N, K)


@pytest.mark.parametrize("stride", [17_300_000, (1 << 25) + 8])
@pytest.mark.parametrize("M", [17, 64])
def test_rows_far_apart(M, stride):
    """Rows of x that span more than 2 GiB, of which 32-bit offsets (the larger stride) and buffer descriptors (both) see only a part."""
    gap = stride if M == 64 else 4 * stride
    K = 4128
    x = torch.empty((M - 1) * gap + K, device="cuda", dtype=torch.bfloat16).as_strided((M, K), (gap, 1))
    x.copy_(torch.randn(M, K, device="cuda"))
    assert x.stride(0) * (M - 1) * 2 > 1 << 31
    rows = torch.randperm(M, device="cuda").int()
    for N, k in ((1536, 1536), (4608, 992), (512, 4128), (8192, 1024)):
        torch.manual_seed(M + N)
        w = (torch.randn(N, k, device="cuda") * k ** -0.5).bfloat16()
        lin, xs = ops.Linear(w), x[:, :k]
        want = xs.float() @ w.float().t()
        for forced in (None, dict(path=2, waves=8), dict(path=2, waves=4)):
            got = ops.linear(xs, lin, **(forced or {}))
            assert ((got.float() - want).abs() <= 2.0 ** -8 * want.abs() + 8.0 * k * 2.0 ** -24 + 1e-6).all(), (N, forced)
        got = ops.linear(xs, lin, out_f32=True, row_idx=rows)
        assert ((got - want[rows.long()]).abs() <= 8.0 * k * 2.0 ** -24 + 1e-6).all(), N


@pytest.mark.parametrize("M", [8, 40, 80])
def test_head_of_more_than_2_gib(M):
    """An LM head whose last columns lie past 2 GiB, of gathered rows, and of rows in place also where stream-K is asked for."""
    N, K = 131072, 8320
    assert N * K * 2 > 1 << 31
    torch.manual_seed(M)
    w = torch.empty(N, K, device="cuda", dtype=torch.bfloat16).normal_(0.0, K ** -0.5)
    lin = ops.Linear(w)
    x = torch.randn(300, K, device="cuda").bfloat16()
    rows = torch.randint(0, 300, (M,), device="cuda", dtype=torch.int32)
    out = ops.linear(x, lin, out_f32=True, row_idx=rows)
    plain = ops.linear(x[:M], lin, out_f32=True, path=3 if M <= 16 else 0)
    for cols in (slice(0, 256), slice(N - 4096, N)):
        for got, rs in ((out, rows.long()), (plain, slice(0, M))):
            want = x[rs].float() @ w[cols].float().t()
            assert ((got[:, cols] - want).abs() <= 8.0 * K * 2.0 ** -24 + 1e-6).all(), cols
