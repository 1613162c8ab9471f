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


def test_greedy_accept_of_many_rows_at_a_wide_head(monkeypatch):
    """24 verify rows at a head that is too wide for argmax candidates: logits rows (gemm_pf), their argmax, then accept / reject, against the oracle
    engine and against the same engine with candidates."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from oracle.runner import oracle_runner_factory
    from ssd_amd.engine.llm_engine import LLMEngine
    from ssd_amd.hip import ops as H
    from ssd_amd.model import HipDecoder
    from ssd_amd.model_config import ModelConfig
    from ssd_amd.sampling_params import SamplingParams
    from tests.util import assert_stream_matches, seq_margins
    t = ModelConfig("llama", 256, 2, 4, 2, 64, 512, 2048, 1e-5, 5e5, 1024, False)
    d = ModelConfig("llama", 256, 1, 4, 2, 64, 512, 2048, 1e-5, 5e5, 1024, False)
    prompts = [[(13 * j + 5 * i) % 2048 for j in range(20 + 9 * i)] for i in range(3)]
    kw = dict(hf_config=t, draft="d", draft_hf_config=d, speculate=True, speculate_k=7, max_num_seqs=3, max_model_len=256, max_num_batched_tokens=256,
              kvcache_block_size=16, num_kvcache_blocks=64, num_draft_kvcache_blocks=64, weights_std=0.1)
    sp = SamplingParams(temperature=0, max_new_tokens=12, ignore_eos=True)
    calls = []
    real = {n: getattr(H, n) for n in ("gemm_pf", "verify_greedy", "argmax_parts_verify")}
    for n in real:
        monkeypatch.setattr(H, n, lambda *a, n=n, **k: (calls.append(n), real[n](*a, **k))[1])
    plain, _ = LLMEngine("t", **kw).generate(prompts, sp, use_tqdm=False)
    assert "argmax_parts_verify" in calls and "verify_greedy" not in calls
    calls.clear()
    monkeypatch.setattr(HipDecoder, "AP_WIDE_HEAD_BYTES", 1 << 20)          # this head has 1 MiB, and is the only matrix of that size
    monkeypatch.setattr(HipDecoder, "PF_MIN_WEIGHT_BYTES", 1 << 20)
    monkeypatch.setattr(HipDecoder, "PF_ALWAYS_WEIGHT_BYTES", 1 << 20)
    wide, _ = LLMEngine("t", **kw).generate(prompts, sp, use_tqdm=False)
    assert "gemm_pf" in calls and "verify_greedy" in calls and "argmax_parts_verify" not in calls
    cpu = LLMEngine("t", runner_factory=oracle_runner_factory(), **kw)
    want, _ = cpu.generate(prompts, sp, use_tqdm=False)
    for i, (a, b, c) in enumerate(zip(wide, plain, want)):
        for out in (a, b):
            assert_stream_matches(out["token_ids"], c["token_ids"], seq_margins(cpu.model_runner.margin_log, i), len(prompts[i]), what=f"sequence {i}")
