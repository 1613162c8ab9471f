"""Prompts of more than 160 tokens at published layer shapes, the length from which products and attention take the forms for many rows: logits behind
them against the oracle and exact arithmetic, and greedy speculation that starts from one."""
import dataclasses
import random

import pytest
import torch

pytestmark = pytest.mark.gpu


def counted(monkeypatch, H, name):
    calls, real = [], getattr(H, name)
    monkeypatch.setattr(H, name, lambda *a, **k: (calls.append(a), real(*a, **k))[1])
    return calls


@pytest.mark.parametrize("preset", ["llama-3.2-1b", "llama-3.1-8b", "qwen3-8b"])
@pytest.mark.parametrize("lens", [[161], [45, 300, 1]])
def test_prompts_and_the_rows_behind_them(monkeypatch, preset, lens):
    """Two layers of the preset's shapes over a short vocabulary (the head sees the prompts' last rows only): the last row of every prompt, then 7 rows behind
    the first.  Criterion of the other real-shape tests: a row as close to exact arithmetic as the oracle's bf16 pipeline."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from oracle.model import Ctx, OracleModel
    from ssd_amd import weights as W
    from ssd_amd.hip import ops as H
    from ssd_amd.model import AttnMeta, HipDecoder
    from ssd_amd.model_config import PRESETS
    from tests.util import truth_forward
    cfg = dataclasses.replace(PRESETS[preset], num_layers=2, vocab_size=2048)
    full = W.synthetic_state_dict(cfg, seed=5, std=0.02)
    bs, T, M = 256, sum(lens), 7
    need = [-(-(n + M) // bs) for n in lens]
    order, tables = list(range(sum(need)))[::-1], []
    for n in need:
        tables.append(order[:n])
        order = order[n:]
    dec = HipDecoder(cfg, max_tokens=T, max_seqs=len(lens), max_blocks=4, block_size=bs, max_model_len=1024, device=torch.device("cuda", 0))
    dec.load_weights(iter(full.items()))
    dec.alloc_kv(sum(need))
    orc = OracleModel(cfg, full, sum(need), bs)
    random.seed(T)
    toks = [[random.randint(0, 2047) for _ in range(n + (M if b == 0 else 0))] for b, n in enumerate(lens)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32)
    slots = lambda b, ps: [tables[b][p // bs] * bs + p % bs for p in ps]
    bt = i32([t + [-1] * (4 - len(t)) for t in tables])
    ids = torch.tensor([t for b, n in enumerate(lens) for t in toks[b][:n]])
    pos = torch.tensor([p for n in lens for p in range(n)])
    sm = i32([s for b, n in enumerate(lens) for s in slots(b, range(n))])
    cu = torch.cat([i32([0]), i32(lens).cumsum(0).to(torch.int32)])
    big = counted(monkeypatch, H, "gemm_big")
    dec.forward(ids.cuda(), pos.cuda(), T, AttnMeta(H.MODE_CAUSAL, len(lens), max(lens), sm.cuda(), i32(lens).cuda(), bt.cuda(), cu_q=cu.cuda()))
    n = dec.compute_logits(T, gather=(cu[1:] - 1).cuda(), rows=len(lens))
    got = [dec.logits[:n].double().cpu()]
    assert len(big) == 4 * cfg.num_layers
    c = Ctx("prefill", slot_mapping=sm, cu_q=cu, cu_k=cu)
    ref = [orc.compute_logits(orc.forward(ids, pos, c)[(cu[1:] - 1).long()]).double()]
    P = lens[0]
    ids, pos, sm = torch.tensor(toks[0][P:]), torch.arange(P, P + M), i32(slots(0, range(P, P + M)))
    dec.forward(ids.cuda(), pos.cuda(), M, AttnMeta(H.MODE_CAUSAL, 1, M, sm.cuda(), i32([P + M]).cuda(), bt[:1].cuda(), q_per_seq=M))
    n = dec.compute_logits(M)
    got.append(dec.logits[:n].double().cpu())
    ref.append(orc.compute_logits(orc.forward(ids, pos, Ctx("verify", slot_mapping=sm, context_lens=i32([P + M]), block_tables=bt[:1],
                                                            cu_q=i32([0, M])))).double())
    truths = [truth_forward(cfg, full, t) for t in toks]
    truth = torch.cat([torch.stack([t[m - 1] for t, m in zip(truths, lens)]), truths[0][P:]])
    e_hip, e_ref = (torch.cat(got) - truth).abs(), (torch.cat(ref) - truth).abs()
    rms = lambda e: e.pow(2).mean(-1).sqrt()
    print(f"{preset} {lens}: |HIP - exact| rms {rms(e_hip).max():.5f} max {e_hip.max():.4f}, |oracle - exact| rms {rms(e_ref).max():.5f} max {e_ref.max():.4f}")
    assert bool((rms(e_hip) <= 1.25 * rms(e_ref) + 1e-3).all()) and float(e_hip.max()) <= 1.5 * float(e_ref.max()) + 1e-3


@pytest.mark.parametrize("lens", [[170], [300, 150]])
def test_greedy_speculation_from_long_prompts(monkeypatch, lens):
    """1B layers and vocabulary, 4 layers over 2: greedy streams against the oracle engine, near ties by its margin."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from oracle.runner import oracle_runner_factory
    from ssd_amd import weights as W
    from ssd_amd.engine.llm_engine import LLMEngine, hip_runner_factory
    from ssd_amd.hip import ops as H
    from ssd_amd.model_config import PRESETS
    from ssd_amd.sampling_params import SamplingParams
    from tests.util import assert_stream_matches, seq_margins
    tcfg = dataclasses.replace(PRESETS["llama-3.2-1b"], num_layers=4, tie_word_embeddings=False)
    dcfg = dataclasses.replace(tcfg, num_layers=2)
    recipe = {"kind": "pair", "shared": 2048, "snr": 8.0, "layer_gain": 0.05}
    wt, wd = (W.synthetic_state_dict(c, s, 0.02, recipe=recipe) for s, c in enumerate((tcfg, dcfg)))
    random.seed(2)
    prompts = [[random.randint(0, 10000) for _ in range(n)] for n in lens]
    kw = dict(hf_config=tcfg, max_num_seqs=2, max_model_len=1024, max_num_batched_tokens=1024, kvcache_block_size=256, num_kvcache_blocks=6,
              num_draft_kvcache_blocks=6, draft="d", draft_hf_config=dcfg, speculate=True, speculate_k=6)

    def factory(config, model_cfg, *, is_draft, topo, **k):
        return hip_runner_factory(config, model_cfg, is_draft=is_draft, topo=topo, weight_source=iter((wd if is_draft else wt).items()), **k)

    sp = SamplingParams(temperature=0, max_new_tokens=24, ignore_eos=True)
    cpu = LLMEngine("t", runner_factory=oracle_runner_factory(wt, wd), **kw)
    want, _ = cpu.generate(prompts, sp, use_tqdm=False)
    big = counted(monkeypatch, H, "gemm_big")
    got, _ = LLMEngine("t", runner_factory=factory, **kw).generate(prompts, sp, use_tqdm=False)
    assert sum(lens) in {a[3] for a in big}
    for i, (a, b) in enumerate(zip(got, want)):
        n = assert_stream_matches(a["token_ids"], b["token_ids"], seq_margins(cpu.model_runner.margin_log, i), len(prompts[i]), what=f"prompt {i}")
        print(f"prompt of {len(prompts[i])}: {n} of 24 tokens as the oracle's")
        assert n >= 6
