"""Decoded tokens of hybrid models: latent attention whose keys several workgroups share, against the CPU
form."""
import pytest
import torch

from vgate.ops import seq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rank,rot,H", [(128, 64, 8), (256, 64, 16), (512, 64, 12), (512, 64, 1), (512, 128, 16), (264, 64, 12), (200, 24, 5), (100, 64, 16), (96, 32, 3)])
@pytest.mark.parametrize("S", [1, 3, 40, 300])
def test_latent_attn_of_decoded_tokens(rank, rot, H, S):
    """Whole tiles (nothing clamped) and others, contexts from one key to some tiles per wave, one to eight workgroups per sequence. Values are
    at most 4: a softmax weight's rounding to bf16 moves a sum by 2^-9 of them, the result's by as much again."""
    g = torch.Generator().manual_seed(rank + H + S)
    E, lens = rank + rot, [1 + (i * 317 + 40 * (i % 3)) % 1100 if S < 100 else 1 + i % 70 for i in range(S)]
    pages = [-(-n // 16) for n in lens]
    cache = (torch.randn(sum(pages), 16, E, generator=g).clamp(-4, 4)).bfloat16()
    tables, at = torch.zeros(S, max(pages), dtype=torch.int32), 0
    order = torch.randperm(sum(pages), generator=g).int()
    for i, n in enumerate(pages):
        tables[i, :n] = order[at: at + n]
        at += n
    qa = torch.randn(S, H, E, generator=g).bfloat16()
    sink, start = torch.randn(H, generator=g), torch.arange(S + 1, dtype=torch.int32)
    ctx, scale = torch.tensor(lens, dtype=torch.int32), E ** -0.5
    tr = cache[:, :, :rank].transpose(1, 2).contiguous()
    for window in (seq.LATENT_FULL, 70):
        got, want = torch.empty(S, H, rank, dtype=torch.bfloat16, device="cuda"), torch.empty(S, H, rank)
        seq.latent_attn(qa.cuda(), cache.cuda(), tables.cuda(), ctx.cuda(), start.cuda(), got, scale, H, rank, rot, num_seqs=S, cache_t=tr.cuda(),
                        window=window, sink=sink.cuda())
        seq.latent_attn(qa.float(), cache.float(), tables, ctx, start, want, scale, H, rank, rot, num_seqs=S, window=window, sink=sink)
        assert ((got.float().cpu() - want).abs() <= 4 * 2.0 ** -8 + 1e-4).all()
