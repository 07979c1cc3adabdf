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


@pytest.mark.parametrize("N,K,norm,slices", [
    (2048, 1536, True, {128: 6, 192: 4, 256: 4, 320: 4, 384: 2, 448: 2, 640: 1, 1024: 1, 2048: 1}),
    (1536, 1536, False, {128: 6, 192: 1, 256: 1, 512: 1, 768: 1, 2048: 1}),
    (17920, 1536, True, {96: 1, 128: 1, 256: 1, 448: 1, 1024: 1, 2048: 1}),
    (1536, 8960, False, {65: 8, 96: 8, 256: 8, 320: 6, 384: 6, 448: 4, 640: 4, 768: 3, 1024: 4, 1536: 3, 2048: 4})])
def test_int4_steps_keep_their_cut_of_k(N, K, norm, slices):
    """The stretches into which K is cut decide the last bits of a product, and in a model with random int4 weights those can decide a
    token: the cut of every size stays as it is, whichever kernels are added or fitted anew."""
    C, ws = ops.native(), torch.empty(65536 + (64 << 20), dtype=torch.int32)
    lin = SimpleNamespace(N=N, K=K, layout="qkv" if norm else "plain")
    plan = ops._awq_plan(lin, sorted(slices), ws)
    for M, nz in slices.items():
        code, sk = ops._awq_cut(plan[M], M, N, K, norm, True, ws)
        for group128 in (False, True):
            path, code2, sk2 = C.q4_prompt_form(M, N, K, norm, True, group128, ws, code, sk)
            # (path 6: the tile kernels of short K, a single chain; K-tiles of 64 cut into sk2 slices otherwise)
            assert (path == 6 and sk2 == 0 and nz == 1) or (path in (1, 5) and sk2 == nz), (M, path, code2, sk2)


def test_int4_forms_that_only_one_kernel_sums_alike():
    """Persistent forms of more tiles than CUs, tile kernels that sum the squares of a norm their own way, few rows of short K."""
    C, ws = ops.native(), torch.empty(65536 + (64 << 20), dtype=torch.int32)
    form = lambda *a, code, sk: C.q4_prompt_form(*a, True, ws, code, sk)  # noqa: E731
    assert C.q4_cut(2048, 28672, 4096, False, True, False, ws) == (1025, 0)
    assert form(2048, 28672, 4096, False, True, code=1025, sk=0) == (1, 1025, 0)
    assert form(300, 1536, 1536, True, True, code=0, sk=1)[0] == 6 and form(300, 1536, 1536, False, True, code=0, sk=1)[2] <= 1
    assert C.q4_cut(96, 1536, 1536, False, True, False, ws)[0] == -1 and form(96, 1536, 1536, False, True, code=-1, sk=0) == (6, 0, 0)
    assert C.q4_prompt_form(300, 1536, 1536, False, False, True, ws, 641, 2)[0] == 1   # (rows off 16 B)
    small = torch.empty(65536 + 4096, dtype=torch.int32)                                # no room for partials: one chain
    assert C.q4_prompt_form(300, 1536, 8960, False, True, True, small, *C.q4_cut(300, 1536, 8960, False, True, False, small))[2] == 1
