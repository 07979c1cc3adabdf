"""Preparing queries, keys and values for window attention (a wave per head) against the op's CPU form: head sizes around a
lane's pairs, odd ones too, both norms, both pairings, every option."""
import pytest
import torch

from vgate.ops import seq

pytestmark = pytest.mark.gpu


def _run(H, G, GV, D, V, dt, norm, rot_half, extras, device):
    g = torch.Generator().manual_seed(H * D + V)
    T, page, pages = 21, 16, 4
    rows = torch.randn(T, H * D + G * D + GV * V + 8, generator=g).to(dt).to(device)   # columns of one fused projection
    q, k, v = rows[:, : H * D], rows[:, H * D: (H + G) * D], rows[:, (H + G) * D: (H + G) * D + GV * V]
    n = {"none": (0, 0), "head": (D, D), "all": (H * D, G * D)}[norm]
    qw, kw = (1 + 0.1 * torch.randn(m, generator=g) if m else None for m in n)
    other = torch.randn(T, GV * V, generator=g).to(dt)
    scale = 1 + 0.1 * torch.rand(H, generator=g)
    slots = torch.randperm(page * pages, generator=g)[:T].int()
    slots[5] = -1                                                                        # a padding row
    pos = torch.randint(0, 3000, (T,), generator=g).int()
    rot = D - D % 2 if rot_half else (D // 2) // 2 * 2
    dev = lambda x: None if x is None else x.to(device)  # noqa: E731
    kc, vc = torch.zeros(pages, G, page, D, dtype=dt, device=device), torch.zeros(pages, GV, page, V, dtype=dt, device=device)
    out = torch.zeros(T, H * D, dtype=dt, device=device)
    vt = torch.zeros(pages, GV, V, page, dtype=dt, device=device) if dt == torch.bfloat16 and device == "cuda" else None
    freq = lambda m: seq.rope_inv_freq(m, 10000.0, device) if m >= 2 else torch.zeros(1, device=device)  # noqa: E731
    kw_args = dict(q_head_scale=dev(scale), q_temp_coef=0.2, q_temp_every=100, v_other=dev(other), lam=0.3) if extras else {}
    seq.window_write(q, k, v, dev(qw), dev(kw), 1e-6, norm == "all", dev(pos), dev(slots), freq(rot), rot,
                     freq(2 * (V // 2)) if extras and V >= 2 else None, kc, vc, out, H, G, vt=vt, rot_half=rot_half, **kw_args)
    keep = torch.arange(T) != 5                                                          # (a padding row's query means nothing)
    return out.float().cpu()[keep], kc.float().cpu(), vc.float().cpu(), None if vt is None else vt.float().cpu()


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("norm,rot_half,extras", [("none", False, True), ("head", True, False), ("head", False, True), ("all", True, True)])
@pytest.mark.parametrize("H,G,GV,D,V", [(3, 3, 3, 1, 3), (4, 2, 1, 24, 20), (8, 2, 2, 128, 128), (2, 1, 1, 130, 65), (3, 1, 1, 256, 256),
                                        (2, 2, 2, 300, 40)])
def test_matches_cpu_form(H, G, GV, D, V, norm, rot_half, extras, dt):
    got, want = (_run(H, G, GV, D, V, dt, norm, rot_half, extras, d) for d in ("cuda", "cpu"))
    # fp32: sums of up to 1024 squares in other orders and sines of the same fp32 angles, a few 1e-6 of values of size ~ 4; bf16
    # results are off by an ulp, 2^-7 of the value, where those differ across a rounding boundary
    for a, b in zip(got[:3], want[:3]):
        assert ((a - b).abs() <= (2e-5 if dt == torch.float32 else 2.0 ** -7 * b.abs() + 2e-5)).all()
    if got[3] is not None:
        assert torch.equal(got[3], got[2].transpose(2, 3))


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("H,G,GV,D", [(1, 1, 1, 8), (12, 2, 2, 128), (14, 2, 2, 128), (100, 10, 5, 128), (8, 4, 4, 300), (250, 5, 1, 24)])
def test_norm_over_the_whole_projection(H, G, GV, D, in_place, dt):
    """Heads that fit one workgroup's waves, one more, many: queries prepared beside or in their own rows."""
    def run(device):
        g = torch.Generator().manual_seed(H)
        T, page, pages = 9, 16, 2
        q, k, v = (torch.randn(T, h * D, generator=g).to(dt).to(device) for h in (H, G, GV))
        qw, kw = (1 + 0.1 * torch.randn(h * D, generator=g).to(device) for h in (H, G))
        slots, pos = torch.randperm(page * pages, generator=g)[:T].int().to(device), torch.randint(0, 3000, (T,), generator=g).int().to(device)
        kc, vc = torch.zeros(pages, G, page, D, dtype=dt, device=device), torch.zeros(pages, GV, page, D, dtype=dt, device=device)
        out = q if in_place else torch.zeros_like(q)
        seq.window_write(q, k, v, qw, kw, 1e-6, True, pos, slots, seq.rope_inv_freq(8, 10000.0, device), 8, None, kc, vc, out, H, G)
        return out.float().cpu(), kc.float().cpu(), vc.float().cpu()

    for a, b in zip(run("cuda"), run("cpu")):   # (bounds as above)
        assert ((a - b).abs() <= (2e-5 if dt == torch.float32 else 2.0 ** -7 * b.abs() + 2e-5)).all()
