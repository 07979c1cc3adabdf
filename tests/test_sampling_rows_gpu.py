"""Sampling with few and with many waves per row: the choice of a row does not depend on how many rows share the launch, which
decides how the row is split and how many waves sweep it."""
import pytest
import torch

from vgate import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [4096, 49156, 152064])
def test_rows_do_not_depend_on_the_batch(V):
    dev, B = "cuda", 130
    g = torch.Generator(dev).manual_seed(V)
    # no two logits closer than a rounding of the sums that a split changes: no candidate on the nucleus' edge at this seed
    lg = 2.0 * torch.randn(B, V, device=dev, generator=g)
    t = torch.tensor([0.0, 0.8, 1.0] * B, device=dev)[:B]
    p = torch.tensor([1.0, 0.95, 0.5, 0.9] * B, device=dev)[:B]
    k = torch.tensor([-1, -1, -1, 50, -1] * B, dtype=torch.int32, device=dev)[:B]
    seeds, offs = torch.arange(B, device=dev), torch.arange(B, device=dev) % 7

    def run(rows):
        out = torch.full((rows.numel(),), -1, dtype=torch.int32, device=dev)
        ops.sample(lg[rows].contiguous(), t[rows], p[rows], k[rows], seeds[rows], offs[rows], out=out)
        return out

    whole = run(torch.arange(B, device=dev))                      # one workgroup per row
    for n in (1, 16, 33, 128):
        rows = torch.arange(n, device=dev)
        assert torch.equal(run(rows), whole[:n]), n
    assert torch.equal(whole[::3], lg[::3].argmax(-1).int())      # temperature 0


@pytest.mark.parametrize("V,B", [(16384, 257), (49152, 300), (70000, 513), (70000, 512)])
def test_more_rows_than_workgroups(V, B):
    dev = "cuda"
    g = torch.Generator(dev).manual_seed(V + B)
    lg = 2.0 * torch.randn(B, V, device=dev, generator=g)
    t, p = torch.tensor([0.0, 0.8, 1.0] * B, device=dev)[:B], torch.tensor([1.0, 0.95, 0.5, 0.9] * B, device=dev)[:B]
    k = torch.tensor([-1, -1, -1, 50, -1] * B, dtype=torch.int32, device=dev)[:B]
    seeds, offs = torch.arange(B, device=dev), torch.arange(B, device=dev) % 7

    def run(n):
        out = torch.full((n,), -1, dtype=torch.int32, device=dev)
        ops.sample(lg[:n].contiguous(), t[:n], p[:n], k[:n], seeds[:n], offs[:n], out=out)
        return out

    whole = run(B)
    assert torch.equal(run(64), whole[:64]) and torch.equal(whole[::3], lg[::3].argmax(-1).int())


@pytest.mark.parametrize("B,V", [(1, 4096), (8, 32000), (40, 8192), (300, 4096)])
def test_extreme_logits_and_the_ring(B, V):
    """Masked logits (-inf, the type's lowest value), one of +inf and NaN beside finite ones: the token is one of the few that count. The
    ids also go to the ring's slot, with the fault word behind them only where it is set."""
    dev = "cuda"
    g = torch.Generator().manual_seed(B * V)
    lg = torch.empty(B, V)
    few = torch.randint(0, V, (B, 3), generator=g)
    for b in range(B):
        lg[b] = (-torch.inf, torch.finfo(torch.float32).min, torch.nan)[b % 3]
        lg[b, few[b]] = torch.tensor([1.0, 1.5, 0.5])
        if b % 4 == 3:
            lg[b, few[b, 0]] = torch.inf
    t = torch.tensor([0.8, 0.0, 1.0, 0.7, 0.9] * B)[:B]
    p = torch.tensor([0.9, 1.0, 0.95] * B)[:B]
    ring = torch.full((2, B + 4), -7, dtype=torch.int32, pin_memory=True)
    slot = torch.tensor([1], dtype=torch.int32, device=dev)
    fault = ops.fault_word(torch.device(dev))
    seen = []
    for word in (0, 4):
        fault.fill_(word)
        out = ops.sample(lg.to(dev), t.to(dev), p.to(dev), None, torch.arange(B, device=dev), torch.full((B,), 3, device=dev), ring=(ring, slot, 0))
        torch.cuda.synchronize()
        seen.append((out.cpu(), ring.clone()))
    fault.zero_()
    for (ids, r), tail in zip(seen, (-7, 4)):
        assert torch.equal(r[1, :B], ids) and torch.all(r[0] == -7) and r[1, B:].tolist() == [-7, -7, -7, tail]
        assert torch.equal(ids, seen[0][0])
        for b in range(B):
            assert ids[b] in few[b], (b, int(ids[b]))
            if b % 4 == 3:
                assert ids[b] == few[b, 0], b
            elif t[b] == 0.0:
                assert ids[b] == few[b][lg[b, few[b]].argmax()], b


@pytest.mark.parametrize("B", [1, 8, 200])
def test_collective_words_in_the_ring(B):
    """The three words of the own all-reduce behind the ids: a buffer that stands for its signal area, every word its own index."""
    dev = "cuda"
    area = torch.arange(1 << 16, dtype=torch.int32, device=dev)
    ring = torch.full((2, B + 4), -7, dtype=torch.int32, pin_memory=True)
    slot = torch.zeros(1, dtype=torch.int32, device=dev)
    lg = torch.randn(B, 8192, device=dev)
    for base in (0, area.data_ptr()):
        out = ops.sample(lg, torch.zeros(B, device=dev), ring=(ring, slot, base))
        torch.cuda.synchronize()
        assert torch.equal(ring[0, :B], out.cpu()) and torch.all(ring[1] == -7)
        error, ticks, calls, fault = ring[0, B:].tolist()
        assert fault == -7 and ((error, ticks, calls) == (-7, -7, -7) if base == 0 else 0 < error == ticks - 1 == calls - 2)


@pytest.mark.parametrize("T", [3.0e38, float("inf")])
@pytest.mark.parametrize("B,V", [(1, 4096), (8, 32000), (300, 4096)])
def test_infinite_temperature(B, V, T):
    """Every logit that counts weighs the same: draws come from all of the nucleus (those with fewer than top_p n, or top_k, above them),
    and the log-probability is that of one in n. Some rows have most of their logits masked."""
    dev, draws = "cuda", 24
    g = torch.Generator().manual_seed(B + V)
    lg = torch.randn(B, V, generator=g)
    lg[::3, V // 4:] = -torch.inf
    n = torch.isfinite(lg).sum(1)
    p, k = torch.tensor([0.5, 1.0, 0.9, 1.0] * B)[:B], torch.tensor([-1, -1, -1, 300] * B, dtype=torch.int32)[:B]
    most = torch.where(p < 1.0, p.double() * n, torch.where(k > 0, k, n).double())
    above = lg.argsort(dim=1, descending=True, stable=True).argsort(dim=1)
    seen = []
    for d in range(draws):
        lp = torch.empty(B, device=dev)
        ids = ops.sample(lg.to(dev), torch.full((B,), T, device=dev), p.to(dev), k.to(dev), torch.arange(B, device=dev),
                         torch.full((B,), d, device=dev), out_logprob=lp).cpu()
        assert torch.isfinite(lg[torch.arange(B), ids.long()]).all()
        torch.testing.assert_close(lp.cpu(), -n.float().log(), rtol=1e-5, atol=0.0)
        seen.append(above[torch.arange(B), ids.long()])
    seen = torch.stack(seen).double() / most   # ranks as shares of the nucleus, uniform on [0, 1)
    assert (seen < 1.0).all()
    # mean 1/2 with a deviation of (12 draws)^-1/2 = 0.06; 6 of them
    assert ((seen.mean(0) - 0.5).abs() < 6 * (12 * draws) ** -0.5).all()
