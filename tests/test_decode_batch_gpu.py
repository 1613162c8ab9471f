"""Decoding batches that fill the grid by themselves, through HipDecoder: every number of waves that _attn_cfg gives them against the same
sequences in small batches, where a workgroup has eight waves and long contexts are split over the grid."""
import pytest
import torch

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


@pytest.mark.parametrize("B,top,waves", [(32, 700, 8), (48, 700, 4), (136, 300, 2), (260, 200, 1), (40, 1900, 8), (136, 1100, 4), (208, 1100, 2)])
def test_batches_agree_with_small_ones(B, top, waves):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ssd_amd import weights as W
    from ssd_amd.hip import ops as H
    from ssd_amd.model import AttnMeta, HipDecoder
    from ssd_amd.model_config import ModelConfig
    bs, max_len = 64, 2048
    cfg = ModelConfig("llama", 256, 1, 16, 8, 64, 512, 512, 1e-5, 5e5, max_len, False)
    dec = HipDecoder(cfg, max_tokens=B, max_seqs=B, max_blocks=max_len // bs, block_size=bs, max_model_len=max_len, device=torch.device("cuda", 0))
    dec.load_weights(W.synthetic_weights(cfg, 0, 0.1))
    g = torch.Generator().manual_seed(B)
    ctx = [top] + torch.randint(1, top + 1, (B - 1,), generator=g).tolist()
    need = [-(-c // bs) for c in ctx]
    dec.alloc_kv(sum(need))
    dec.kv_cache.normal_()
    bt, at = torch.full((B, max_len // bs), -1, dtype=torch.int32), 0
    for b, n in enumerate(need):
        bt[b, :n] = torch.arange(at, at + n, dtype=torch.int32)
        at += n
    slots = torch.tensor([int(bt[b, (c - 1) // bs]) * bs + (c - 1) % bs for b, c in enumerate(ctx)], dtype=torch.int32)
    ids = torch.randint(0, 512, (B,), generator=g).cuda()
    pos, bt, slots, lens = (torch.tensor(ctx) - 1).cuda(), bt.cuda(), slots.cuda(), torch.tensor(ctx, dtype=torch.int32).cuda()

    def logits(a, b):
        meta = AttnMeta(H.MODE_CAUSAL, b - a, 1, slots[a:b], lens[a:b], bt[a:b].contiguous(), q_per_seq=1, ctx_hint=top)
        cfg_ = dec._attn_cfg(b - a, meta)
        dec.forward(ids[a:b], pos[a:b], b - a, meta)
        dec.compute_logits(b - a)
        return cfg_, dec.logits[:b - a].float().clone()

    plan, got = logits(0, B)
    assert plan == (1, waves)
    want = torch.cat([logits(a, min(B, a + 8))[1] for a in range(0, B, 8)])
    d = (got - want).abs()
    # one layer, rows of another order of summation: six roundings to bf16 in a row of at most 2^-9, independent -> a relative error of at most
    # 6 * 2^-9 / sqrt(3) = 0.0068 (2-norm) of the last row and so of the logits' deviation; the largest of 10^5 lies within 4.6 of those, with the
    # logits' own rounding at 4.5 deviations (2^-8 of them) 0.049
    assert float(d.max()) <= 0.05 * float(want.std()) and float(d.mean()) <= 0.01 * float(want.std()), (float(d.max()), float(d.mean()), float(want.std()))
