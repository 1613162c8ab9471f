"""Batches of many tokens turn their values through LDS on the way to the cache (csrc/attention_window.hip): the same bytes as in portions too small for
that, at tokens and columns that no tile divides, scattered slots and tokens without one."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f32", [True, False])
@pytest.mark.parametrize("T,H,G,D,Dv,bs", [(256, 2, 2, 16, 128, 32), (257, 3, 3, 24, 100, 16), (319, 4, 4, 32, 64, 64), (448, 8, 8, 8, 33, 8), (300, 3, 3, 8, 85, 7)])
def test_values_of_a_large_batch_equal_those_of_small_portions(T, H, G, D, Dv, bs, f32):
    from ssd_amd.hip import ops
    el = torch.float32 if f32 else torch.bfloat16
    gen = torch.Generator().manual_seed(T + Dv)
    ld = (H + G) * D + G * Dv + 3
    pages = T // bs + 3
    x = torch.randn(T, ld, generator=gen).cuda()
    slots = torch.randperm(pages * bs, generator=gen)[:T].int()
    slots[[0, 65, T - 1]] = -1
    slots, pos = slots.cuda(), torch.arange(T).cuda()
    w = (1.0 + 0.3 * torch.randn(D, generator=gen)).to(el).cuda()
    freqs = torch.rand(D // 2, generator=gen).cuda()

    def store(step):
        q = torch.zeros(T, H * D, dtype=el, device="cuda")
        kc = torch.full((pages, G, bs, D), 7.0, dtype=el, device="cuda")
        vc = torch.full((pages, G, Dv, bs), 7.0, dtype=el, device="cuda")
        for a in range(0, T, step):
            n = min(step, T - a)
            ops.winattn_store_norm_rope(x[a:], ld, w, w, 1e-5, pos[a:], freqs, D, slots[a:], q[a:], kc, vc, n, H, G, D, Dv, bs, f32)
        return q, kc, vc

    for one, portions in zip(store(T), store(100)):
        assert torch.equal(one, portions)
    vc = store(T)[2]
    t = T // 2
    slot = int(slots[t])
    assert torch.equal(vc[slot // bs, :, :, slot % bs], x[t, (H + G) * D:(H + G) * D + G * Dv].view(G, Dv).to(el))
