"""HipDecoder._parts_cfg (host logic, no GPU): every (splits, waves) plan it hands to ssd_gemm_parts must respect the kernel's
"<= 8 k-tiles per wave" register budget for the shapes that take the slab path: the two-slab fused-consumer plan
violated it for h = 3072 with I = 14336 and hard-failed at launch."""
import itertools

from ssd_amd.model import HipDecoder


def tiles_per_wave(N, K, fused):
    S, wv = HipDecoder._parts_cfg(N, K, fused)
    assert 1 <= S <= 16 and 1 <= wv <= 16
    return -(-(-(-(K // 32) // S)) // wv)


def test_presets_on_the_slab_path_fit_the_register_budget():
    from ssd_amd.model_config import PRESETS
    for name, cfg in PRESETS.items():
        if cfg.family == "eagle3":
            continue
        h, qn, I = cfg.hidden_size, cfg.num_heads * cfg.head_dim, cfg.intermediate_size
        g = h // 16
        if not (g < 256 or 256 < g < 512):
            continue                         # rows kernels
        fused_possible = (not cfg.qk_norm) and h // 8 <= 1024
        ok = all(tiles_per_wave(h, k, f) <= 8 for k in (qn, I) for f in ((False, True) if fused_possible else (False,)))
        # a model whose plan does not fit must fall back to the rows kernels (use_parts False), never fail at launch: the same
        # predicate HipDecoder.__init__ evaluates
        if name in ("llama-3.2-1b", "qwen3-0.6b", "qwen3-32b"):
            assert ok, name


def test_unfused_consumer_plans_fit_for_arbitrary_shapes():
    for N, K in itertools.product((1024, 2048, 3072, 5120, 6144), (1024, 2048, 4096, 8192, 14336, 25600, 28672)):
        g = N // 16
        if g < 256 or 256 < g < 512:
            t = tiles_per_wave(N, K, False)
            assert t <= 8 or K // 32 > 16 * 16 * 8, (N, K, t)


def test_wide_down_projections_leave_the_slabs_at_two_token_tiles():
    for h, I, rows in ((5120, 25600, 16), (3584, 18944, 16), (3072, 12288, 16), (3072, 8192, 32), (2048, 16384, 32), (2048, 24576, 32), (1024, 3072, 32)):
        d = HipDecoder.__new__(HipDecoder)
        d.h, d.I, d.use_parts, d.use_coll = h, I, True, False
        assert [d.parts_plan(T) for T in (1, 16, 17, 32, 33)] == [True, True, rows == 32, rows == 32, False], (h, I)


def test_kernels_of_17_to_128_rows(monkeypatch):
    """Which GEMM a chunk of m rows of an N x K matrix takes: where the measured lines lie (HipDecoder._gemm_chunk)."""
    import torch
    import ssd_amd.model as M
    took = []
    for n in ("gemm", "gemm_pf", "gemm_big"):
        monkeypatch.setattr(M.H, n, lambda *a, n=n, **k: took.append(n))
    monkeypatch.setattr(M.H, "gemm_pf_workspace_bytes", lambda *a: 0)
    d = HipDecoder.__new__(HipDecoder)
    d._ws_pf = d._ws_big = torch.zeros(1)
    rows, silu = M.H.EPI_ROWS, M.H.EPI_SILU_FRAG
    S, P, B = "gemm", "gemm_pf", "gemm_big"
    for N, K, epi, want in (                                  # m = 16, 17, 32, 33, 64, 65
            (4096, 14336, rows, (S, B, B, B, B, P)), (28672, 4096, silu, (S, S, S, B, B, P)),              # 8B down, gate_up
            (4096, 4096, rows, (S, B, B, B, B, S)), (3072, 2048, rows, (S, S, S, S, S, S)),                # 8B o, 1B qkv
            (57344, 8192, silu, (S, P, P, P, P, P)), (28672, 8192, silu, (S, S, S, P, P, P)),              # 70B gate_up, of two shards
            (14336, 8192, silu, (S, S, S, B, B, P)), (8192, 28672, rows, (S, P, P, P, P, P)),              # of four; 70B down
            (8192, 1024, rows, (S, S, S, B, B, S)), (51200, 5120, silu, (S, P, P, P, P, P)),               # 70B o of eight; 32B gate_up
            (128256, 2048, rows, (S, S, S, P, P, P)), (151936, 5120, rows, (S, P, P, P, P, P)),            # heads of 1B and 32B
            (16384, 512, rows, (S, B, B, B, B, S)), (256, 64, rows, (S, S, S, S, S, S))):
        took.clear()
        for m in (16, 17, 32, 33, 64, 65):
            d._gemm_chunk(None, K, None, N, None, m, N, epi, None)
        assert tuple(took) == want, (N, K, epi, took)


def test_peaky_recipe_scales_the_same_tokens_in_target_and_eagle_draft():
    """bench.py --workload c4e builds its EAGLE pair with the "peaky" recipe (ssd_amd/weights.py peaky_rows): the LM-head rows
    of the same few tokens -- draft-vocabulary ids pushed through the draft's d2t -- are scaled in BOTH models, everything
    else is the plain seeded N(0, std)."""
    import torch
    from ssd_amd import weights as W
    from ssd_amd.model_config import ModelConfig
    t = ModelConfig("llama", 128, 2, 4, 2, 32, 256, 512, 1e-5, 5e5, 1024, False)
    d = ModelConfig("eagle3", 64, 1, 2, 1, 32, 128, 512, 1e-5, 5e5, 1024, False, draft_vocab_size=128, d_model_target=128, eagle_taps=3)
    rec = {"kind": "peaky", "gain": 6.0, "peaks": 3, "draft_seed": 1, "draft_vocab": 128, "target_vocab": 512}
    tw, dw = dict(W.synthetic_weights(t, 0, 0.1, recipe=rec)), dict(W.synthetic_weights(d, 1, 0.1, recipe=rec))
    plain_t, plain_d = dict(W.synthetic_weights(t, 0, 0.1)), dict(W.synthetic_weights(d, 1, 0.1, recipe={"target_vocab": 512}))
    dp, tp = W.peaky_rows(rec)
    assert ((torch.arange(128) + dw["d2t"])[dp] == tp).all()                 # the SAME tokens in both vocabularies
    for w, plain, rows in ((tw, plain_t, tp), (dw, plain_d, dp)):
        ratio = w["lm_head.weight"].float().norm(dim=1) / plain["lm_head.weight"].float().norm(dim=1)
        assert torch.allclose(ratio[rows], torch.full((3,), 6.0), rtol=0.02)
        mask = torch.ones(ratio.numel(), dtype=torch.bool)
        mask[rows] = False
        assert torch.allclose(ratio[mask], torch.ones(int(mask.sum())), rtol=1e-3)
        assert all(torch.equal(w[k], plain[k]) for k in w if k != "lm_head.weight")
