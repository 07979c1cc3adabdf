"""Half tiles of the decode GEMMs (8 columns over all of K per workgroup, up to 8 rows) against fp32 products: rows, waves with fewer k-quads than
others, strides, bias and residual, and the sums of squares of 8 columns that they hand to the next projection's norm."""
import pytest
import torch

from vgate import ops

pytestmark = pytest.mark.gpu


def _rand(*s):
    return torch.randn(*s, device="cuda")


def _close(out, want, K):
    # fp32 sums of K products of size ~ K^-1/2 in another order, rounded to bf16 before and after the residual
    assert ((out.float() - want).abs() <= 2.0 ** -7 * want.abs() + 8.0 * K * 2.0 ** -24 + 2.0 ** -7).all()


def _close_pair(out, want):
    # one rounding to bf16 of a pair whose halves are off by some 2^-24 K^1/2 each, at most 5 of the other and its slope
    assert ((out.float() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all()


@pytest.mark.parametrize("M", [1, 2, 4, 5, 8])
@pytest.mark.parametrize("N,K", [(16, 128), (48, 384), (512, 2176), (1536, 1536), (2048, 6144), (1024, 6272), (256, 10240), (2048, 8960)])
def test_half_tiles(M, N, K):
    torch.manual_seed(M + N + K)
    w, bias = (_rand(N, K) * K ** -0.5).bfloat16(), _rand(N).bfloat16()
    lin, lb = ops.Linear(w), ops.Linear(w, bias=bias)
    x, res = _rand(M, K + 64).bfloat16()[:, 32:K + 32], _rand(M, N + 8).bfloat16()[:, :N]
    want = x.float() @ w.float().t()
    whole = torch.full((M + 1, N + 8), 7.0, device="cuda", dtype=torch.bfloat16)
    ops.linear(x, lin, out=whole[:M, :N], residual=res)
    _close(whole[:M, :N], want + res.float(), K)
    assert bool((whole[M] == 7).all() and (whole[:, N:] == 7).all())
    _close(ops.linear(x, lb), want + bias.float(), K)


@pytest.mark.parametrize("M", [1, 3, 8])
@pytest.mark.parametrize("N,K", [(256, 256), (1536, 1536), (1536, 8960), (2048, 10240)])
def test_sums_of_8_columns(M, N, K):
    """The residual projection stores the sums, three kinds of consumers take their row scale from them: the same as from the rows."""
    torch.manual_seed(M + N + K)
    assert ops.half_tiles(M, N)
    lin = ops.Linear((_rand(N, K) * K ** -0.5).bfloat16())
    x, h = _rand(M, K).bfloat16(), _rand(M, N).bfloat16()
    plain, ssp = h.clone(), torch.full((M, N // 8), float("nan"), device="cuda")
    ops.linear(x, lin, out=h, residual=h, norm_out=(None, ssp, None))
    ops.linear(x, lin, out=plain, residual=plain)
    assert torch.equal(h, plain) or not bool(((h.float() - plain.float()).abs() > 2.0 ** -6 * plain.float().abs() + 2.0 ** -7).any())
    torch.testing.assert_close(ssp, h.float().pow(2).reshape(M, N // 8, 8).sum(-1), rtol=1e-5, atol=1e-4)
    for rows, path in ((512, 0), (8192, 0), (8192, 4)):   # few tiles, many, whole tiles per CU
        w, gamma = (_rand(rows, N) * N ** -0.5).bfloat16(), (torch.rand(N, device="cuda") + 0.5).bfloat16()
        nx = ops.Linear(w.clone(), kind="silu")
        assert nx.fold_norm(gamma)
        nx.dec_path = path
        got, want = ops.linear(h, nx, prenorm=(ssp, 1e-6)), ops.linear(h, nx, norm=(gamma, 1e-6))
        assert ((got.float() - want.float()).abs() <= 2.0 ** -7 * want.float().abs() + 2.0 ** -9).all()
        sums16 = ssp.reshape(M, N // 16, 2).sum(-1).contiguous()
        old = ops.linear(h, nx, prenorm=(sums16, 1e-6))
        assert ((got.float() - old.float()).abs() <= 2.0 ** -7 * old.float().abs() + 2.0 ** -9).all()


@pytest.mark.parametrize("M", [1, 8, 9, 16])
@pytest.mark.parametrize("N,K", [(48, 128), (1024, 1280), (2064, 1024), (3072, 1536), (4096, 512), (4112, 1536), (8208, 2048), (12304, 512), (20480, 1408),
                                 (1024, 4096), (512, 10240), (20496, 512), (28672, 512), (28672, 1024), (32784, 1024)])
def test_register_stationary_choice(M, N, K):
    """Shapes on the lines of the launcher's choice of the register-stationary kernel: one to eight whole tiles per CU, more tiles than waves to
    finish them, one-tile blocks, K slices; both result types, pairs of either activation, a folded norm."""
    torch.manual_seed(M + N + K)
    w, x = (_rand(N, K) * K ** -0.5).bfloat16(), _rand(M, K).bfloat16()
    lin, want = ops.Linear(w), x.float() @ w.float().t()
    res = _rand(M, N).bfloat16()
    _close(ops.linear(x, lin, residual=res), want + res.float(), K)
    f32 = ops.linear(x, lin, out_f32=True)
    assert ((f32 - want).abs() <= 8.0 * K * 2.0 ** -24 + 1e-6).all()
    g, u = want[:, : N // 2], want[:, N // 2:]
    _close_pair(ops.linear(x, ops.Linear(w, kind="silu")), torch.nn.functional.silu(g) * u)
    gelu = ops.Linear(w, kind="silu")
    gelu.glu = (4, 0.0, 0.0)
    _close_pair(ops.linear(x, gelu), torch.nn.functional.gelu(g, approximate="tanh") * u)
    gelu.glu = (2, 0.7, 1.702)
    gc, uc = g.clamp(max=0.7), u.clamp(-0.7, 0.7)
    _close_pair(ops.linear(x, gelu), gc * torch.sigmoid(1.702 * gc) * (uc + 1))
    nl, gamma = ops.Linear(w.clone(), kind="silu"), (torch.rand(K, device="cuda") + 0.5).bfloat16()
    assert nl.fold_norm(gamma)
    xn = x.float() * torch.rsqrt((x.float() ** 2).mean(-1, keepdim=True) + 1e-6)
    y = xn @ (w.float() * gamma.float()).bfloat16().float().t()
    _close_pair(ops.linear(x, nl, norm=(gamma, 1e-6)), torch.nn.functional.silu(y[:, : N // 2]) * y[:, N // 2:])


@pytest.mark.parametrize("M", [1, 16])
@pytest.mark.parametrize("N,K", [(20480, 512), (28672, 512), (16384, 384), (8192, 128), (12304, 256), (32768, 128), (32784, 640)])
def test_int4_blocks_with_fewer_waves_than_tiles(M, N, K):
    from vgate.ops import reference as ref
    torch.manual_seed(M + N + K)
    q = torch.randint(0, 16, (N, K), dtype=torch.int32)
    scales, zeros = (torch.rand(K // 128, N) * 0.02 + 0.005).bfloat16(), torch.randint(0, 16, (K // 128, N)).float().bfloat16()
    w = ref.awq_dequant_ref(q, scales, zeros, 128).cuda()
    lin = ops.Linear(None, awq={"qint": q, "scales": scales.cuda(), "zeros": zeros.cuda(), "group": 128})
    x = _rand(M, K).bfloat16()
    got, want = ops.linear(x, lin).float(), ref.linear_ref(x, w).float()
    assert (got - want).norm() / want.norm() < 2e-2   # (as every int4 product here: bf16 scales times zero points)
    assert bool(((got - want).abs().amax(0) < 0.1 * want.abs().max()).all())


@pytest.mark.parametrize("M", [1, 4, 5, 16])
@pytest.mark.parametrize("N,K", [(64, 128), (1536, 384), (4096, 640), (4128, 640), (1024, 896), (1024, 512)])
def test_sums_of_16_columns_of_short_k(M, N, K):
    """A norm's sums handed over where no wave can ask for them ahead (K % 256), on either side of the line below which the tile blocks take them."""
    torch.manual_seed(M + N + K)
    w, gamma, h = (_rand(N, K) * K ** -0.5).bfloat16(), (torch.rand(K, device="cuda") + 0.5).bfloat16(), _rand(M, K).bfloat16()
    lin = ops.Linear(w.clone(), kind="silu")
    assert lin.fold_norm(gamma)
    ssp = h.float().pow(2).reshape(M, K // 16, 16).sum(-1).contiguous()
    xn = h.float() * torch.rsqrt((h.float() ** 2).mean(-1, keepdim=True) + 1e-6)
    y = xn @ (w.float() * gamma.float()).bfloat16().float().t()
    want = torch.nn.functional.silu(y[:, : N // 2]) * y[:, N // 2:]
    _close_pair(ops.linear(h, lin, prenorm=(ssp, 1e-6)), want)
