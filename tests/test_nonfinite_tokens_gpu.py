"""An infinity or a NaN in one token reaches that token and later ones of its sequence, never an earlier token or another sequence:
the recurrences that take a portion in chunks, against their own outputs on finite inputs."""
import pytest
import torch

from vgate.ops import seq

pytestmark = pytest.mark.gpu

LENS, POS = [200, 3, 70], [0, 9, 4]     # chunks of 32 and 64 tokens, whole and cut short, and a portion run token by token
H, D = 3, 64


def _linear(rows, f32, bonus):
    n, T = H * D, rows.shape[0]
    q, k, v, g = (rows[:, i * n: (i + 1) * n] for i in range(4))
    out = torch.zeros(T, n, dtype=rows.dtype, device="cuda")
    seq.linear_attn(q, k, v, g, f32[:, :n], None, 1.0, D ** -0.5, False, torch.ones(n if bonus else D, device="cuda"), False, True,
                    _state(), *_meta(), out, 1e-5, decay_exp=bonus, bonus=f32[0, :n].view(H, D).contiguous() if bonus else None,
                    norm_full=bonus)
    return out


def _delta(rows, f32):
    n, T = H * D, rows.shape[0]
    cols = [rows[:, i * n: (i + 1) * n] for i in (0, 1, 2, 3, 4)]
    out, one = torch.zeros(T, n, dtype=rows.dtype, device="cuda"), torch.ones(n, device="cuda")
    seq.delta_rule(*cols, f32[:, :n].to(rows.dtype), one, one, one, _state(), *_meta(), out, 0.6, 1e-6, 1e-6)
    return out


def _gated(rows, f32):
    n, T = H * D, rows.shape[0]
    q, k, v = (rows[:, i * n: (i + 1) * n] for i in range(3))
    out = torch.zeros(T, n, dtype=rows.dtype, device="cuda")
    seq.gated_delta(q, k, v, rows[:, 3 * n: 3 * n + H], f32[:, :n], f32[:, n: 2 * n], torch.ones(H, device="cuda"), torch.ones(D, device="cuda"),
                    f32[:4, :].repeat(1, 2)[:, : 3 * n].contiguous(), _state(), torch.zeros(len(LENS), 3, 3 * n, device="cuda"), *_meta(), out,
                    1e-6, D ** -0.5, 1e-6)
    return out


def _state():
    return torch.randn(len(LENS), H, D, D, generator=torch.Generator().manual_seed(5)).cuda()


def _meta():
    ctx = torch.tensor([p + m for p, m in zip(POS, LENS)], dtype=torch.int32, device="cuda")
    qs = torch.tensor([0] + LENS).cumsum(0).int().cuda()
    return torch.arange(len(LENS), dtype=torch.int32, device="cuda"), ctx, qs


@pytest.mark.parametrize("value", [float("nan"), float("inf")])
@pytest.mark.parametrize("column", ["key", "value"])
@pytest.mark.parametrize("op", ["linear", "bonus", "delta", "gated"])
@pytest.mark.parametrize("token", [5, 40, 130, 199, 205, 260])
def test_earlier_tokens_do_not_see_it(op, column, value, token):
    g = torch.Generator().manual_seed(token)
    T, n = 700, H * D                                             # (rows of a padded step: chunks whatever the portions)
    rows, f32 = torch.randn(T, 5 * n, generator=g).cuda(), torch.randn(T, 2 * n, generator=g).cuda()
    run = {"linear": lambda r: _linear(r, f32, False), "bonus": lambda r: _linear(r, f32, True), "delta": lambda r: _delta(r, f32),
           "gated": lambda r: _gated(r, f32)}[op]
    want = run(rows)[: sum(LENS)]
    h, d = 1, 7
    bad = rows.clone()
    bad[token, (1 if column == "key" else 2) * n + h * D + d] = value
    got = run(bad)[: sum(LENS)]
    starts = torch.tensor([0] + LENS).cumsum(0)
    s = int(torch.searchsorted(starts, token, right=True)) - 1
    clean = torch.ones(sum(LENS), H, dtype=torch.bool, device="cuda")
    clean[token: int(starts[s + 1]), h] = False                    # the head's outputs from this token on
    got, want = got.view(-1, H, D), want.view(-1, H, D)
    # sums of up to 64 fp32 products of size ~ 1 may run in another order where the chunk has such a value
    assert ((got - want).abs()[clean] <= 1e-4 * want.abs().max()).all()
    assert not torch.isfinite(got[token, h]).all()
