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
