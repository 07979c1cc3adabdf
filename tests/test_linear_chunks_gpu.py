"""Linear attention's forms (chunks, tokens one by one, the general one) against the op's CPU form, at the sizes where chunks,
staged tokens and tiles end and where one form hands over to the other, in every variant of decay, norm, gate and bonus."""
import pytest
import torch

from vgate.ops import seq

pytestmark = pytest.mark.gpu

VARIANTS = {   # decay, norm, rotation, bonus, silu on q / k / v, silu gate
    "channel": dict(decay="channel", norm="head"),
    "constant": dict(decay="head", norm="all", silu=True, gate_silu=False),
    "turned": dict(decay="head", norm="none", rot="half"),
    "turned pairs": dict(decay="channel", norm="head", rot="pairs", silu=True),
    "bonus": dict(decay="exp", norm="full", bonus=True),
}


def _run(H, D, V, lens, pos, dt, variant, seed, device, pad=3):
    v = VARIANTS[variant]
    g = torch.Generator().manual_seed(seed)
    n, S = sum(lens), len(lens)
    T = n + pad                                                 # with padding rows
    P = torch.randn(T, H * (2 * D + 2 * V) + 8, generator=g).to(dt).to(device)   # columns of one fused projection
    q, k = P[:, : H * D], P[:, H * D: 2 * H * D]
    val, gate = P[:, 2 * H * D: 2 * H * D + H * V], P[:, 2 * H * D + H * V: 2 * H * (D + V)]
    z = torch.randn(T, H * D, generator=g).to(device) if v["decay"] != "head" else None
    dec = (0.8 + 0.2 * torch.rand(H, generator=g)).to(device) if v["decay"] == "head" else None
    nw = {"head": V, "full": H * V, "all": H * V, "none": 0}[v["norm"]]
    nw = (1 + 0.1 * torch.randn(nw, generator=g)).to(device) if nw else None
    bonus = torch.randn(H, D, generator=g).to(device) if v.get("bonus") else None
    state = torch.randn(S + 2, H, D, V, generator=g).to(device)   # slots hold another owner's state
    slots = torch.randperm(S + 2, generator=g)[:S].int().to(device)
    ctx = torch.tensor([p + m for p, m in zip(pos, lens)], dtype=torch.int32).to(device)
    qs = torch.tensor([0] + lens, dtype=torch.int32).cumsum(0).int().to(device)
    positions = torch.cat([torch.arange(p, p + m) for p, m in zip(pos, lens)] + [torch.zeros(pad, dtype=torch.long)]).int().to(device)
    rot = 2 * (D // 2) if v.get("rot") else 0
    freq = seq.rope_inv_freq(rot, 10000.0, device) if rot else None
    out = torch.zeros(T, H * V, dtype=dt, device=device)
    seq.linear_attn(q, k, val, gate, z, dec, 4.0 if v["decay"] == "channel" else 1.0, D ** -0.5, v.get("silu", False), nw,
                    v["norm"] == "all", v.get("gate_silu", True), state, slots, ctx, qs, out, 1e-5, k_scale=0.5,
                    positions=positions, inv_freq=freq, rot_dims=rot, rot_half=v.get("rot") == "half",
                    decay_exp=v["decay"] == "exp", bonus=bonus, norm_full=v["norm"] == "full")
    return out[:n].float().cpu(), state.cpu()


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("variant", list(VARIANTS))
@pytest.mark.parametrize("H,D,V", [(2, 1, 5), (3, 32, 33), (2, 64, 16), (1, 100, 128), (9, 128, 128), (2, 130, 40)])
@pytest.mark.parametrize("lens,pos", [([1100], [0]), ([300, 65, 1, 64, 150], [0, 9, 40, 0, 2]), ([1] * 15 + [129, 150], [5] * 17),
                                      ([1] * 6 + [3, 2], [4] * 8), ([64, 65, 1], [0, 9, 40]), ([124], [2]), ([125], [0])])
def test_matches_cpu_form(H, D, V, lens, pos, variant, dt):
    out, state = _run(H, D, V, lens, pos, dt, variant, 3 * H + D + V, "cuda")
    want, state_w = _run(H, D, V, lens, pos, dt, variant, 3 * H + D + V, "cpu")
    # both sum up to 1100 fp32 products under decays < 1 in other orders (and turn by the same fp32 angles): relative error
    # of the whole below 2^-24 x 1100 < 7e-5 in the worst order, 5e-5 taken; a bf16 result rounds by 2^-8
    rel = lambda a, b: float((a - b).norm() / b.norm())  # noqa: E731
    assert rel(state, state_w) < 5e-5
    assert rel(out, want) < (5e-5 if dt == torch.float32 else 2.0 ** -8)


@pytest.mark.parametrize("variant", ["bonus", list(VARIANTS)[0]])
@pytest.mark.parametrize("lens,pos,pad", [([20], [3], 1100), ([1], [0], 1), ([65], [0], 1000), ([3, 30], [0, 2], 500)])
def test_fewer_tokens_than_rows(lens, pos, pad, variant):
    """A step's rows are padded to a size of their own: few tokens among many rows."""
    out, state = _run(3, 64, 48, lens, pos, torch.float32, variant, 11, "cuda", pad)
    want, state_w = _run(3, 64, 48, lens, pos, torch.float32, variant, 11, "cpu", pad)
    assert float((state - state_w).norm() / state_w.norm()) < 5e-5   # (as above)
    assert float((out - want).norm() / want.norm()) < 5e-5


@pytest.mark.parametrize("variant", ["bonus", "constant"])
@pytest.mark.parametrize("lens,pad", [([1] * 97, 31), ([1] * 128, 0), ([1] * 200, 56), ([1] * 63 + [65], 0), ([1] * 127 + [129], 0), ([1] * 255 + [258], 0)])
def test_many_decoded_tokens(lens, pad, variant):
    pos = [3] * len(lens)   # (none at position 0, where a token's output is one product whose rounding the norm can blow up)
    out, state = _run(2, 64, 48, lens, pos, torch.float32, variant, 7, "cuda", pad)
    want, state_w = _run(2, 64, 48, lens, pos, torch.float32, variant, 7, "cpu", pad)
    assert float((state - state_w).norm() / state_w.norm()) < 5e-5   # (as above)
    assert float((out - want).norm() / want.norm()) < 5e-5
