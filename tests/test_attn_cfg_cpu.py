"""HipDecoder._attn_cfg (host logic, no GPU): waves per workgroup of decoding batches that fill the grid by themselves."""
import pytest

from ssd_amd.model import AttnMeta, HipDecoder


@pytest.mark.parametrize("nh,nkv,hd", [(32, 8, 128), (64, 8, 128), (32, 8, 64), (16, 8, 128), (32, 32, 128), (8, 1, 64)])
def test_waves_of_large_decoding_batches(nh, nkv, hd):
    d = HipDecoder.__new__(HipDecoder)
    d.nh, d.nkv, d.hd, d.max_splits, d.max_split_tokens, d.max_model_len = nh, nkv, hd, 16, 256, 32768
    for B in (1, 8, 32, 33, 48, 64, 128, 256):
        for q in (1, 4, 8, 24):
            tiles = -(-q * nh // nkv // 16)
            base = B * nkv * (-(-tiles // 2) if tiles > 8 else tiles)
            last = 8
            for ctx in (100, 1024, 1025, 30000):
                meta = AttnMeta(0, B, q, None, None, None, q_per_seq=q, ctx_hint=ctx)
                splits, waves = d._attn_cfg(B * q, meta)
                if base < 256 and B * q <= d.max_split_tokens:
                    continue
                assert splits == 1 and waves in (1, 2, 4, 8)
                # never more waves than are resident together, but for long contexts of batches that come close
                assert waves == 1 or base * waves * hd <= 128 * (2048 if ctx <= 1024 else 4096), (B, q, ctx, waves)
                assert waves == 8 or base > 256
                if ctx <= 1024:
                    last = waves
                else:
                    assert waves >= last                         # a longer scan never gets fewer
