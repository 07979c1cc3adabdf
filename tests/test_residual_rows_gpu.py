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
