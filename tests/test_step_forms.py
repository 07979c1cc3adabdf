"""Which form a step of the recurrent mixers takes, by its rows (with padding) and sequences: host rules, no GPU."""
from types import SimpleNamespace

import pytest
import torch

from vgate import ops
from vgate.models import hybrid


def _plan(name, *sizes):
    return getattr(ops.native(), name)(*sizes)


@pytest.mark.parametrize("T", [12, 16, 32, 64, 96, 128])
def test_delta_rule_lone_middle_portions_take_the_scan(T):
    assert _plan("delta_rule_plan", T, 1, 8, 128)[0]


@pytest.mark.parametrize("T,S,H,D,scan,chunks", [(8, 1, 8, 128, False, False), (192, 1, 8, 128, False, True), (2048, 1, 8, 128, False, True),
                                                 (128, 2, 8, 128, True, False), (256, 4, 8, 128, True, True), (448, 4, 8, 128, False, True),
                                                 (64, 8, 8, 128, False, False), (64, 8, 4, 128, True, False), (512, 8, 4, 128, True, True),
                                                 (96, 1, 8, 64, True, False), (128, 1, 8, 64, False, True), (64, 8, 16, 64, True, False),
                                                 (64, 16, 16, 64, False, False)])
def test_delta_rule_lines(T, S, H, D, scan, chunks):
    one, _, n = _plan("delta_rule_plan", T, S, H, D)
    assert one == scan and (n > 0) == chunks


@pytest.mark.parametrize("T,S", [(1, 1), (64, 64), (96, 128), (128, 128), (256, 256), (512, 512)])
def test_decoding_steps_take_one_launch(T, S):
    scan, lim, chunks = _plan("delta_rule_plan", T, S, 8, 128)
    assert not scan and lim >= T and chunks == 0
    small, lim, chunks = _plan("linear_attn_plan", T, S, 8, 128, 128)
    assert small and lim >= T and chunks == 0


@pytest.mark.parametrize("T,S", [(128, 64), (192, 128), (256, 128)])
def test_linear_attention_nearly_decoding_steps_take_one_launch(T, S):
    assert _plan("linear_attn_plan", T, S, 8, 128, 128)[2] == 0


@pytest.mark.parametrize("T,S,H,D,V,small", [(2048, 1, 8, 64, 64, True), (2048, 1, 16, 64, 64, False), (2048, 1, 32, 64, 64, False),
                                             (512, 1, 8, 64, 64, False), (160, 1, 8, 64, 64, True), (128, 1, 8, 64, 64, False),
                                             (128, 1, 8, 128, 128, True), (2048, 1, 16, 128, 128, True), (1600, 4, 4, 64, 64, True),
                                             (1600, 4, 16, 64, 64, False), (720, 2, 8, 64, 64, False), (1024, 2, 8, 32, 32, False),
                                             (1024, 16, 32, 64, 64, True), (768, 16, 4, 128, 128, False), (256, 256, 1, 32, 32, True)])
def test_linear_attention_lines(T, S, H, D, V, small):
    assert _plan("linear_attn_plan", T, S, H, D, V)[0] == small


@pytest.mark.parametrize("name,args", [("delta_rule_plan", (8, 128)), ("linear_attn_plan", (8, 128, 128))])
def test_chunks_cover_every_way_to_share_the_rows(name, args):
    """Whole chunks of C tokens and one that is not whole for each sequence of more than `lim` tokens."""
    C = 32 if name == "delta_rule_plan" else 64
    for T in (65, 97, 128, 129, 200, 513, 2048):
        for S in (1, 2, 3, 7, 31, 100):
            one, lim, chunks = _plan(name, T, S, *args)
            if T <= lim or (name == "linear_attn_plan" and not one):
                continue
            for n in range(1, min(S, T // (lim + 1)) + 1):     # n equal portions, the last one takes the rest
                lens = [max(lim + 1, T // n // C * C + 1)] * (n - 1)
                if sum(lens) >= T:
                    lens = [lim + 1] * (n - 1)
                lens.append(T - sum(lens))
                assert sum(-(-m // C) for m in lens if m > lim) <= chunks, (T, S, lens)


@pytest.mark.parametrize("rows", [1000, 1024, 1088, 1360])
@pytest.mark.parametrize("f32", [False, True])
def test_row_major_projections_are_not_padded_past_whole_tiles_of_64(rows, f32):
    w = torch.randn(rows, 64).to(torch.float32 if f32 else torch.bfloat16)
    proj, col = hybrid._fuse_inputs(SimpleNamespace(in_rows=[("a", w)]), [], 64, "cpu", f32)
    assert proj.N == -(-rows // 64) * 64 and col == {"a": (0, rows)}
    assert torch.equal(proj.w[:rows], w) and not proj.w[rows:].any()
