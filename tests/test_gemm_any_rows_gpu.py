"""The row-major GEMM's form for few rows or few tiles against fp32 products: rows around its passes and tiles, columns and K
around its pieces, batches, experts (empty ones and ones of many rows too), gathers, pairs, gates, biases, both result types."""
import pytest
import torch

from vgate.ops import seq

pytestmark = pytest.mark.gpu


def _close(out, want, K):
    # fp32 sums of K products of size ~ K^-1/2 in another order, then one rounding to the result's type
    tol = 4.0 * K * 2.0 ** -24 + (2.0 ** -8 * want.abs() if out.dtype == torch.bfloat16 else 0.0)
    assert ((out.float() - want).abs() <= 2 * tol + 1e-6).all(), float((out.float() - want).abs().max())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,K", [(8, 1024), (17, 8), (64, 264), (200, 136), (1024, 2048)])
@pytest.mark.parametrize("M", [1, 16, 17, 32, 33, 64, 65, 300, 513])
def test_plain(M, N, K, dt):
    g = torch.Generator("cuda").manual_seed(M * N + K)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    a, w, bias = rand(M, K + 8).bfloat16()[:, :K], (rand(N, K) * K ** -0.5).bfloat16(), rand(N)
    out = torch.full((M, N), float("nan"), device="cuda", dtype=dt)
    seq.gemm(a, w, out, bias=bias)
    _close(out, a.float() @ w.float().t() + bias, K)


@pytest.mark.parametrize("gate_dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M", [1, 32, 40, 130, 1100])
def test_batches_with_gates(M, gate_dt):
    B, N, K = 3, 72, 136
    g = torch.Generator("cuda").manual_seed(M)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    a, w = rand(M, B, K).bfloat16().transpose(0, 1), (rand(B, N, K) * K ** -0.5).bfloat16()
    gate = rand(M, B, N).to(gate_dt).transpose(0, 1)
    out = torch.full((M, B, N), float("nan"), device="cuda", dtype=torch.bfloat16).transpose(0, 1)
    seq.gemm(a, w, out, gate=gate)
    _close(out, torch.matmul(a.float(), w.float().transpose(1, 2)) * torch.sigmoid(gate.float()), K)


@pytest.mark.parametrize("kind", ["outputs", "rows", "rows fp32", "outputs fp32", "outputs off 16 B"])
@pytest.mark.parametrize("M,B,N,K", [(1412, 16, 128, 72), (1025, 11, 256, 512), (2047, 12, 128, 8)])
def test_long_batches_with_gates(M, B, N, K, kind):
    """Products of whole 128-column tiles that fill the chip: a gate per output (its tile through LDS), one per row, and the gates that
    the 64-row tiles keep; rows past the last whole tile, K below and past a step."""
    g = torch.Generator("cuda").manual_seed(M + K)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    a, w = rand(M, B, K).bfloat16().transpose(0, 1), (rand(B, N, K) * K ** -0.5).bfloat16()
    dt = torch.float32 if "fp32" in kind else torch.bfloat16
    if kind.startswith("rows"):
        gate = rand(M, B).to(dt).unsqueeze(-1).expand(-1, -1, N).transpose(0, 1)
    else:
        off = 1 if "off" in kind else 0
        gate = rand(M * B * N + 1).to(dt)[off: off + M * B * N].view(M, B, N).transpose(0, 1)
    out = torch.full((M, B, N), float("nan"), device="cuda", dtype=torch.bfloat16).transpose(0, 1)
    seq.gemm(a, w, out, gate=gate)
    _close(out, torch.matmul(a.float(), w.float().transpose(1, 2)) * torch.sigmoid(gate.float()), K)


@pytest.mark.parametrize("off", [0, 1, 4])
@pytest.mark.parametrize("M,N,K", [(1024, 512, 64), (1153, 516, 96), (1090, 640, 8), (1025, 518, 136), (1024, 1020, 40)])
def test_long_products_in_fp32(M, N, K, off):
    """fp32 outputs of the 128-row tiles, stored in whole pieces where rows lie on 16 B and by the value where they don't: rows and columns
    past the last whole tile, K below and past a step; what lies beside the outputs stays."""
    g = torch.Generator("cuda").manual_seed(M + N)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    a, w, bias = rand(M, K).bfloat16(), (rand(N, K) * K ** -0.5).bfloat16(), rand(N)
    whole = torch.full((M + 1, N + 8), 7.0, device="cuda")
    out = whole[:M, off: off + N]
    seq.gemm(a, w, out, bias=bias)
    _close(out, a.float() @ w.float().t() + bias, K)
    assert bool((whole[M] == 7).all() and (whole[:, :off] == 7).all() and (whole[:, off + N:] == 7).all())


@pytest.mark.parametrize("sizes", [[1, 0, 2, 17], [0, 0, 90], [16, 32, 33, 64, 65], [2] * 64, [5] * 40, [500, 3], [1] * 70])
@pytest.mark.parametrize("N,K", [(48, 72), (1024, 512)])
def test_experts(N, K, sizes):
    E, M = len(sizes), sum(sizes)
    g = torch.Generator("cuda").manual_seed(M + N)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    x, w, w2 = rand(M, K).bfloat16(), (rand(E, N, K) * K ** -0.5).bfloat16(), (rand(E, N, K) * K ** -0.5).bfloat16()
    rows = torch.randperm(M, device="cuda", generator=g).int()
    off = torch.tensor([sum(sizes[:i]) for i in range(E + 1)], dtype=torch.int32, device="cuda")
    out, pair = (torch.full((M, N), float("nan"), device="cuda", dtype=torch.bfloat16) for _ in range(2))
    seq.gemm(x, w, out, group_off=off)
    seq.gemm(x, w, pair, w2=w2, a_rows=rows, group_off=off, act=seq.ACT_SILU_MUL)
    for e in range(E):
        a, b = int(off[e]), int(off[e + 1])
        _close(out[a:b], x[a:b].float() @ w[e].float().t(), K)
        h = x[rows[a:b].long()].float()
        _close(pair[a:b], torch.nn.functional.silu(h @ w[e].float().t()) * (h @ w2[e].float().t()), 8 * K)


@pytest.mark.parametrize("M", [1024, 1151, 2049])
@pytest.mark.parametrize("N,K", [(128, 136), (256, 512)])
def test_many_products_of_many_rows(M, N, K):
    B = 16
    g = torch.Generator("cuda").manual_seed(M + N)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    a, w = rand(M, B, K).bfloat16().transpose(0, 1), (rand(B, N, K) * K ** -0.5).bfloat16()
    out = torch.full((M, B, N), float("nan"), device="cuda", dtype=torch.bfloat16).transpose(0, 1)
    seq.gemm(a, w, out)
    _close(out, torch.matmul(a.float(), w.float().transpose(1, 2)), K)


@pytest.mark.parametrize("M", [8, 9, 128, 129, 256, 513, 1023, 1024])
@pytest.mark.parametrize("N,K", [(512, 520), (512, 1032), (2048, 264), (64, 40)])
def test_lines_between_the_forms(M, N, K):
    g = torch.Generator("cuda").manual_seed(M * N + K)
    a, w = torch.randn(M, K, device="cuda", generator=g).bfloat16(), (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).bfloat16()
    out = torch.full((M, N), float("nan"), device="cuda", dtype=torch.bfloat16)
    seq.gemm(a, w, out)
    _close(out, a.float() @ w.float().t(), K)


@pytest.mark.parametrize("sizes", [[8, 0], [9, 0], [16] * 63 + [15], [16] * 64, [24] * 32, [33] * 32, [65, 3] * 15])
@pytest.mark.parametrize("N,K", [(512, 72), (1024, 520)])
def test_experts_on_the_lines(N, K, sizes):
    E, M = len(sizes), sum(sizes)
    g = torch.Generator("cuda").manual_seed(M + N)
    x, w = torch.randn(M, K, device="cuda", generator=g).bfloat16(), (torch.randn(E, N, K, device="cuda", generator=g) * K ** -0.5).bfloat16()
    off = torch.tensor([sum(sizes[:i]) for i in range(E + 1)], dtype=torch.int32, device="cuda")
    out = torch.full((M, N), float("nan"), device="cuda", dtype=torch.bfloat16)
    seq.gemm(x, w, out, group_off=off)
    for e in range(E):
        a, b = int(off[e]), int(off[e + 1])
        _close(out[a:b], x[a:b].float() @ w[e].float().t(), K)


@pytest.mark.parametrize("M", [1024, 1153])
@pytest.mark.parametrize("K", [8, 32, 40, 136, 256, 264])
def test_many_workgroups_and_short_k(M, K):
    B, N = 16, 640
    g = torch.Generator("cuda").manual_seed(M + K)
    a = torch.randn(M, B, K, device="cuda", generator=g).bfloat16().transpose(0, 1)
    w = (torch.randn(B, N, K, device="cuda", generator=g) * K ** -0.5).bfloat16()
    out = torch.full((M, B, N), float("nan"), device="cuda", dtype=torch.bfloat16).transpose(0, 1)
    seq.gemm(a, w, out)
    _close(out, torch.matmul(a.float(), w.float().transpose(1, 2).contiguous()), K)


@pytest.mark.parametrize("out", ["bf16", "odd", "gate", "row", "fp32"])
@pytest.mark.parametrize("M,N,K", [(1025, 640, 256), (1153, 520, 320), (4100, 1160, 256), (4224, 1032, 576)])
def test_stages_by_dma(M, N, K, out):
    """128-row tiles whose operands come by LDS-DMA, four stages (few tiles) and two (many): rows and columns past the last whole tile,
    strided operands, as few k stages as there are buffers and more, every way to store; what lies beside the outputs stays."""
    g = torch.Generator("cuda").manual_seed(M + N)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    N -= 3 if out == "odd" else 0
    a, w, bias = rand(M, K + 8).bfloat16()[:, :K], (rand(N, K) * K ** -0.5).bfloat16(), rand(N)
    gate = rand(M, N).bfloat16() if out == "gate" else (rand(M, 1).bfloat16().expand(M, N) if out == "row" else None)
    whole = torch.full((M + 1, N + 8), 7.0, device="cuda", dtype=torch.float32 if out == "fp32" else torch.bfloat16)
    seq.gemm(a, w, whole[:M, :N], bias=bias, gate=gate)
    want = a.float() @ w.float().t() + bias
    _close(whole[:M, :N], want if gate is None else want * torch.sigmoid(gate.float()), K)
    assert bool((whole[M] == 7).all() and (whole[:, N:] == 7).all())


@pytest.mark.parametrize("out", ["bf16", "odd", "gate", "fp32"])
@pytest.mark.parametrize("M,N,K", [(4097, 2056, 256), (4097, 2056, 512), (4100, 2056, 576), (4100, 2184, 1024), (4100, 2184, 1088)])
def test_many_tiles_of_short_k(M, N, K, out):
    """More than two 128-row tiles per CU: by way of registers up to K = 512 (1024 with gates), by LDS-DMA beyond."""
    test_stages_by_dma(M, N, K, out)


@pytest.mark.parametrize("N,K", [(2560, 320), (2184, 640), (2184, 704)])
def test_many_experts_of_short_k(N, K):
    test_experts(N, K, [70, 0, 130, 33, 1] * 7)


@pytest.mark.parametrize("sizes", [[70, 0, 46, 33, 1, 127, 40, 55] * 4, [33] * 31 + [1100], [128, 0, 129] * 7 + [2, 0, 0]])
@pytest.mark.parametrize("N,K", [(768, 320), (520, 256), (896, 576)])
def test_experts_on_a_workgroup_per_cu(N, K, sizes):
    """More workgroups than CUs, of which some 0.7 to 1.8 per CU have rows: four stages in LDS below 11/12 of the CUs, two above."""
    test_experts(N, K, sizes)


@pytest.mark.parametrize("sizes", [[300, 0, 129, 1, 600], [128] * 9 + [127, 0, 2], [700] * 6])
@pytest.mark.parametrize("N,K", [(520, 256), (1024, 320)])
def test_experts_by_dma(N, K, sizes):
    test_experts(N, K, sizes)
