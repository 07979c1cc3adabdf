"""The residual kernels of hybrid models at widths around the columns that a thread takes, few rows and many, against the ops' CPU
forms."""
import pytest
import torch

from vgate.ops import seq

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (3, 255), (3, 256), (3, 257), (2, 513), (2, 769), (2, 1000), (2, 1025), (3, 1536), (2, 1537), (2, 2048), (2, 2049), (1024, 2049), (2, 4100)]


def _close(a, b):   # fp32 sums of up to 4100 squares in other orders: a few 1e-6 of values of size ~ 4; exp in sigmoid within 2e-7
    assert ((a.cpu() - b).abs() <= 2e-5 + 1e-5 * b.abs()).all()


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,W", SIZES)
def test_gated_residual(T, W, dt):
    g = torch.Generator().manual_seed(T + W)
    x, b1, b2 = torch.randn(T, W, generator=g), torch.randn(W, generator=g), torch.randn(W, generator=g)
    y1, y2 = torch.randn(T, W, generator=g).to(dt), torch.randn(T, W, generator=g).to(dt)
    gates = torch.randn(T, 2 * W + 3, generator=g).to(dt)       # columns of a wider row
    for args in ((y1,), (y1, gates[:, :W], b1), (y1, gates[:, :W], None, y2, gates[:, W: 2 * W], b2), (y1, None, None, y2)):
        want, got = x.clone(), x.cuda()
        seq.gated_residual(want, *args)
        seq.gated_residual(got, *(None if a is None else a.cuda() if a.dim() < 2 or a.is_contiguous() else
                                  gates.cuda()[:, a.storage_offset(): a.storage_offset() + W] for a in args))
        _close(got, want)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("planes", [0, 1, 4])
@pytest.mark.parametrize("T,W", SIZES)
def test_post_norm_add(T, W, planes, dt):
    g = torch.Generator().manual_seed(T + W)
    x, w, y1, y2 = torch.randn(T, W, generator=g), torch.randn(W, generator=g), torch.randn(T, W, generator=g).to(dt), torch.randn(T, W, generator=g).to(dt)
    hist, coef = torch.randn(4, T, W, generator=g), torch.randn(4, generator=g)

    def run(dev):
        h, act, mix = hist.clone().to(dev), torch.zeros(T, W, dtype=torch.bfloat16, device=dev), torch.zeros(T, W, device=dev)
        xd = x.clone().to(dev)
        out = h[planes - 1] if planes else xd                   # (in place without a history)
        kw = dict(hist=h, planes=planes, coef=coef[:planes].to(dev), mix=mix) if planes else {}
        seq.post_norm_add(xd, y1.to(dev), w.to(dev), 1e-6, out, 0.7, y2.to(dev), 0.3, act_out=act, **kw)
        return out.float(), mix, act.float()

    got, want = run("cuda"), run("cpu")
    _close(got[0], want[0])
    _close(got[1], want[1])
    assert ((got[2].cpu() - want[2]).abs() <= 2.0 ** -7 * want[2].abs() + 2e-5).all()   # (an ulp where rounding differs)


def _round(a, b, dt):   # an ulp where an fp32 sum in another order rounds the other way
    assert ((a.float().cpu() - b.float()).abs() <= 2e-5 + (2.0 ** -7 if dt == torch.bfloat16 else 1e-5) * b.float().abs()).all()


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,W", SIZES)
def test_norm_rows(T, W, dt):
    g = torch.Generator().manual_seed(T + W)
    wide, w = torch.randn(T, W + 5, generator=g).to(dt), torch.randn(W, generator=g)
    pick = torch.randint(0, T, (T + 2,), generator=g, dtype=torch.int32)
    for center in (False, True):
        for scalar in (False, True):
            for rows in (None, pick):
                def run(dev):
                    out = torch.zeros(len(pick) if rows is not None else T, W, dtype=dt, device=dev)
                    return seq.norm_rows(wide.to(dev)[:, 3: 3 + W], (w[:1] if scalar else w).to(dev), 1e-3, out, center=center, scalar=scalar,
                                         rows=None if rows is None else rows.to(dev))
                _round(run("cuda"), run("cpu"), dt)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,W", SIZES)
def test_rows_that_carry_the_next_norm(T, W, dt):
    """The embedding and the gated residual with the next sublayers' inputs: the bits of the row kernels that make them alone."""
    g = torch.Generator().manual_seed(T + W)
    table, prev = torch.randn(9, W, generator=g).to(dt).cuda(), torch.randint(0, 9, (T,), generator=g, dtype=torch.int32).cuda()
    ids = torch.randint(0, 9, (T,), generator=g, dtype=torch.int32)
    ids[::3] = -1 - ids[::3] % T
    ids[-1:] = 77 if T > 1 else ids[-1:]     # outside the table: zeros
    ids, w1, w2 = ids.cuda(), torch.randn(W, generator=g).cuda(), torch.randn(W, generator=g).cuda()
    x, want = torch.empty(T, W, device="cuda"), torch.empty(T, W, device="cuda")
    h, h2, n, n2 = (torch.empty(T, W, dtype=dt, device="cuda") for _ in range(4))
    seq.embed_rows(ids, table, want, prev=prev, scale=0.7)
    seq.embed_rows(ids, table, x, prev=prev, scale=0.7, h=h)
    assert torch.equal(x, want) and torch.equal(h, want.to(dt))
    for kw in (dict(), dict(center=True), dict(scalar=True), dict(h2=h2, norm2=w2)):
        first = w1[:1] if "scalar" in kw else w1
        seq.embed_rows(ids, table, x, prev=prev, scale=0.7, h=h, norm=first, eps=1e-3, **kw)
        seq.norm_rows(want, first, 1e-3, n, scalar="scalar" in kw, center="center" in kw)
        assert torch.equal(x, want) and torch.equal(h, n)
    assert torch.equal(h2, seq.norm_rows(want, w2, 1e-3, n2))
    y1, y2 = torch.randn(T, W, generator=g).to(dt).cuda(), torch.randn(T, W, generator=g).to(dt).cuda()
    gates = torch.randn(T, 2 * W + 3, generator=g).to(dt).cuda()
    args = (y1, gates[:, :W], w1, y2, gates[:, W: 2 * W], w2)
    seq.gated_residual(x, *args, norm=w1[:1], eps=1e-3, h=h)
    seq.gated_residual(want, *args)
    assert torch.equal(x, want) and torch.equal(h, seq.norm_rows(want, w1[:1], 1e-3, n, scalar=True))


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rank,n", [(16, 1), (256, 512), (513, 513), (64, 1024), (1000, 1030), (512, 2100)])
def test_latent_write_with_the_querys_norm(rank, n, dt):
    g = torch.Generator().manual_seed(rank + n)
    T, rot = 5, 6
    P = torch.randn(T, rank + rot + n + 3, generator=g).to(dt).cuda()
    w, qw = torch.randn(rank, generator=g).cuda(), torch.randn(n, generator=g).cuda()
    pos, slots = torch.arange(T, dtype=torch.int32, device="cuda"), torch.tensor([3, -1, 17, 0, -1], dtype=torch.int32, device="cuda")
    inv = seq.rope_inv_freq(rot, 50.0, "cuda")
    kv, q = P[:, 2: 2 + rank + rot], P[:, 2 + rank + rot: 2 + rank + rot + n]
    caches = [torch.full((2, 16, rank + rot), 7.0, dtype=dt, device="cuda") for _ in range(3)]
    trs = [torch.full((2, rank, 16), 7.0, dtype=dt, device="cuda") if dt == torch.bfloat16 else None for _ in range(2)]
    y, alone = torch.empty(T, n, dtype=dt, device="cuda"), torch.empty(T, n, dtype=dt, device="cuda")
    seq.latent_write(kv, w, 1e-5, pos, slots, inv, rot, caches[0], rank, cache_t=trs[0], query=(q, qw, y))
    seq.latent_write(kv, w, 1e-5, pos, slots, inv, rot, caches[1], rank, cache_t=trs[1])
    assert torch.equal(caches[0], caches[1]) and (trs[0] is None or torch.equal(trs[0], trs[1]))
    assert torch.equal(y, seq.norm_rows(q, qw, 1e-5, alone))
    host = caches[2].cpu()
    seq.latent_write(kv.cpu(), w.cpu(), 1e-5, pos.cpu(), slots.cpu(), inv.cpu(), rot, host, rank)
    _round(caches[0], host, dt)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("W", [1, 300, 2500])
def test_embedding_table_without_rows(W, dt):
    """No id names a row of it: zeros, and nothing is read."""
    table, ids = torch.empty(0, W, dtype=dt, device="cuda"), torch.tensor([0, 5, -3], dtype=torch.int32, device="cuda")
    x, h = torch.full((3, W), 7.0, device="cuda"), torch.full((3, W), 7.0, dtype=dt, device="cuda")
    seq.embed_rows(ids, table, x, h=h, norm=torch.ones(W, device="cuda"), eps=1e-3)
    assert not x.any() and not h.any()
