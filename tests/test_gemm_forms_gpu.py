"""The launcher's own choice of GEMM form (no plan, no forced tile): every form it can take, at the row counts where it
changes, with the operands a model gives it (column slices of a wider matrix, bias, residual, fp32 or bf16 results, a
SiLU pair) and without a workspace, against the product in float32."""
import pytest
import torch

from vgate import ops

pytestmark = pytest.mark.gpu

# (N, K): short and long K, narrow and wide N, one column past a whole 128- and 256-column tile
SHAPES = [(512, 512), (576, 768), (1024, 1024), (1536, 1536), (1024, 4096), (1536, 8960), (4160, 1024), (4352, 1024), (6656, 1536)]
ROWS = [17, 32, 33, 64, 65, 127, 128, 129, 300, 513, 2048]


@pytest.mark.parametrize("epi", ["bf16", "f32", "silu", "bias_residual", "no_workspace"])
@pytest.mark.parametrize("N,K", SHAPES)
def test_default_form_matches_float32(N, K, epi):
    C, dev = ops.native(), "cuda"
    g = torch.Generator(dev).manual_seed(N + K)
    w = (torch.randn(N, K, device=dev, generator=g) * K ** -0.5).bfloat16()
    perm = ops.row_permutation(N, "silu") if epi == "silu" else None
    wp = ops.pack_weight(w if perm is None else w[perm.to(dev)])
    bias = torch.randn(N, device=dev, generator=g).bfloat16() if epi == "bias_residual" else None
    for M in ROWS:
        x = torch.randn(M, K + 64, device=dev, generator=g).bfloat16()[:, 32: 32 + K]   # rows 2 (K + 64) bytes apart
        res = torch.randn(M, N, device=dev, generator=g).bfloat16() if epi == "bias_residual" else None
        cols = N // 2 if epi == "silu" else N
        out = torch.empty(M, cols, dtype=torch.float32 if epi == "f32" else torch.bfloat16, device=dev)
        ws = None if epi == "no_workspace" else ops.workspace(torch.device(dev))
        C.gemm(x, wp, N, K, out, {"f32": 1, "silu": 2}.get(epi, 0), bias=bias, res=res, ws=ws, fault=ops.fault_word(dev))
        y = x.float() @ w.float().t()
        if epi == "silu":
            gate, up = y.split(N // 2, 1)
            y = torch.nn.functional.silu(gate) * up
        if bias is not None:
            y = (y + bias.float()).bfloat16().float() + res.float()
        # fp32 sums of K products of size ~ K^-1/2: error <= K 2^-24 of their absolute sum, itself < 4 here. A bf16 result is
        # off by half an ulp, <= 2^-8 of its value; before a residual the sum is rounded to bf16 too, and sums that differ in
        # the last fp32 places may round to neighbours: one ulp, <= 2^-7 of |sum| <= |result| + |residual|.
        tol = 4.0 * K * 2.0 ** -24
        bound = torch.full_like(y, tol) if epi == "f32" else tol + 2.0 ** -8 * y.abs()
        if res is not None:
            bound = bound + 2.0 ** -7 * (y.abs() + res.float().abs())
        if epi == "silu":
            bound = bound + tol * 8.0   # (the product of the pair carries both errors, each times the other's size)
        bad = (out.float() - y).abs() > bound
        assert not bad.any(), (M, N, K, float((out.float() - y).abs().max()))


@pytest.mark.parametrize("N,K", [(3008, 2304), (3072, 2304), (4096, 4096), (4160, 2304), (8128, 2304), (8192, 2304), (8256, 2304)])
def test_lines_of_the_medium_forms(N, K):
    C, dev = ops.native(), "cuda"
    g = torch.Generator(dev).manual_seed(N + K)
    w = (torch.randn(N, K, device=dev, generator=g) * K ** -0.5).bfloat16()
    wp = ops.pack_weight(w)
    for M in (17, 24, 25, 32, 33, 64):
        x, out = torch.randn(M, K, device=dev, generator=g).bfloat16(), torch.empty(M, N, dtype=torch.bfloat16, device=dev)
        C.gemm(x, wp, N, K, out, 0, ws=ops.workspace(torch.device(dev)), fault=ops.fault_word(dev))
        y = x.float() @ w.float().t()
        assert ((out.float() - y).abs() <= 4.0 * K * 2.0 ** -24 + 2.0 ** -8 * y.abs()).all(), (M, N, K)   # (bound as above)


@pytest.mark.parametrize("N,K", [(512, 512), (1024, 1024), (1536, 1536), (1600, 2048), (2048, 1792), (4096, 1024), (4160, 2048), (1024, 4096)])
def test_folded_norm_on_the_lines(N, K):
    C, dev = ops.native(), "cuda"
    g = torch.Generator(dev).manual_seed(N + K)
    w = (torch.randn(N, K, device=dev, generator=g) * K ** -0.5).bfloat16()
    wp = ops.pack_weight(w)
    for M in (17, 20, 21, 32, 33, 64, 96, 128, 257, 512, 1024):
        x, out = (3 * torch.randn(M, K, device=dev, generator=g)).bfloat16(), torch.empty(M, N, dtype=torch.float32, device=dev)
        C.gemm(x, wp, N, K, out, 1, rownorm=True, eps=1e-6, ws=ops.workspace(torch.device(dev)), fault=ops.fault_word(dev))
        f = x.double()
        y = f @ w.double().t() * torch.rsqrt(f.pow(2).mean(1, keepdim=True) + 1e-6)
        # K fp32 products with |x| |w| sums < 4 after the norm, and a sum of K squares: each off by K 2^-24 of itself at most
        assert ((out.double() - y).abs() <= 8.0 * K * 2.0 ** -24 + K * 2.0 ** -24 * y.abs()).all(), (M, N, K)
