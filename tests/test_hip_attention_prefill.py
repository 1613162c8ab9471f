"""Throughput form of causal attention (csrc/attention_prefill.hip, through ssd_attn_paged) against fp64: prompts at the edges of 16-row tiles,
128-row workgroups and 64-key tiles, behind cached prefixes, over scattered pages of the smallest and an ordinary size, unwritten slots NaN,
scores whose maximum moves far enough to be re-based."""
import pytest
import torch

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


def reference(q, K, V, scale):
    """Last q.shape[0] rows of one sequence: q [n][H][hd], K, V [N][G][hd], fp64."""
    n, H = q.shape[:2]
    N, G = K.shape[:2]
    K, V = K.repeat_interleave(H // G, 1).transpose(0, 1), V.repeat_interleave(H // G, 1).transpose(0, 1)
    s = torch.matmul(q.transpose(0, 1), K.transpose(1, 2).contiguous()) * scale
    hide = torch.arange(N, device=q.device)[None] > torch.arange(N - n, N, device=q.device)[:, None]
    return torch.matmul(torch.softmax(s.masked_fill(hide, float("-inf")), -1), V).transpose(0, 1)


@pytest.mark.parametrize("nh,nkv,hd,bs,new,old", [
    (4, 1, 64, 16, [33, 1, 129], [0, 31, 64]),            # the third crosses a workgroup; a single token beside prompts
    (8, 2, 128, 16, [161], [0]), (8, 2, 128, 256, [64, 65, 63, 200], [0, 1, 255, 256]),
    (6, 2, 64, 64, [191, 43], [63, 4200]),               # more than 64 key tiles: page ids are looked up again; 3 heads per group
    (16, 1, 128, 32, [9, 190], [500, 0])])
def test_prompts(nh, nkv, hd, bs, new, old):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ssd_amd.hip import ops as H
    g = torch.Generator().manual_seed(nh * hd + sum(new))
    rnd = lambda *s: torch.randn(*s, generator=g).to(BF).cuda()
    ctx = [a + b for a, b in zip(new, old)]
    need = [-(-c // bs) for c in ctx]
    order, at = torch.randperm(sum(need), generator=g).tolist(), 0
    kc = torch.full((sum(need), nkv, bs, hd), float("nan"), dtype=BF, device="cuda")
    vc = kc.clone()
    bt = torch.full((len(ctx), max(need)), -1, dtype=torch.int32)
    T, refs = sum(new), []
    q = rnd(T, nh, hd)
    scale, row = hd ** -0.5, 0
    for b, c in enumerate(ctx):
        pages = order[at:at + need[b]]
        at += need[b]
        bt[b, :need[b]] = torch.tensor(pages, dtype=torch.int32)
        K, V = rnd(c, nkv, hd), rnd(c, nkv, hd)
        # keys that some row looks at with scores of 30 and more, ever larger towards the end: the running reference has to follow
        for i in range(8):
            j = (i + 1) * c // 9
            K[j, 0] = (q[row + new[b] - 1, 0].float() / q[row + new[b] - 1, 0].float().norm() * hd ** 0.5 * (1.0 + 0.6 * i)).to(BF)
        for j, pg in enumerate(pages):
            part = slice(j * bs, min(c, (j + 1) * bs))
            kc[pg, :, :part.stop - part.start], vc[pg, :, :part.stop - part.start] = K[part].transpose(0, 1), V[part].transpose(0, 1)
        refs.append(reference(q[row:row + new[b]].double(), K.double(), V.double(), scale))
        row += new[b]
    ref = torch.cat(refs)
    assert T > 160 and max(new) * (nh // nkv) > 128
    cu = torch.tensor([0] + new).cumsum(0).to(torch.int32).cuda()
    rows = torch.full((T, nh * hd), 7.0, dtype=BF, device="cuda")
    frag = torch.zeros(H.frag_numel(T, nh * hd), dtype=BF, device="cuda")
    H.attn_paged(q, kc, vc, bt.cuda(), bt.shape[1], torch.tensor(ctx, dtype=torch.int32).cuda(), len(ctx), T, max(new), nh, nkv, hd, bs, scale,
                 cu_q=cu, out_rows=rows, out_frag=frag)
    # one rounding to bf16 of weighted means of N(0, 1) values; weights to 2^-17, sums and exponentials in fp32
    d = (rows.double() - ref.flatten(1)).abs()
    assert bool((d <= 2.0 ** -8 * ref.flatten(1).abs() + 2.0 ** -13).all()), float(d.max())
    back = torch.zeros(T, nh * hd, dtype=BF, device="cuda")
    H.frag_to_rows(frag, back, T, nh * hd)
    assert torch.equal(back, rows)


@pytest.mark.parametrize("waves", [0, 3, 4, 8])              # the throughput form up to three, the general one from four on
def test_waves(waves):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ssd_amd.hip import ops as H
    nh, nkv, hd, bs, new, c = 8, 1, 128, 64, 170, 1000
    g = torch.Generator().manual_seed(1)
    rnd = lambda *s: torch.randn(*s, generator=g).to(BF).cuda()
    n = -(-c // bs)
    q, K, V = rnd(new, nh, hd), rnd(n * bs, nkv, hd), rnd(n * bs, nkv, hd)
    pages = lambda t: t.view(n, bs, nkv, hd).transpose(1, 2).contiguous()
    rows = torch.full((new, nh * hd), 7.0, dtype=BF, device="cuda")
    H.attn_paged(q, pages(K), pages(V), torch.arange(n, dtype=torch.int32, device="cuda").view(1, n), n, torch.tensor([c], dtype=torch.int32).cuda(), 1,
                 new, new, nh, nkv, hd, bs, hd ** -0.5, cu_q=torch.tensor([0, new], dtype=torch.int32).cuda(), out_rows=rows, waves=waves)
    ref = reference(q.double(), K[:c].double(), V[:c].double(), hd ** -0.5).flatten(1)
    d = (rows.double() - ref).abs()
    assert bool((d <= 2.0 ** -8 * ref.abs() + 2.0 ** -13).all()), float(d.max())          # (bounds as above)


@pytest.mark.parametrize("scale,ctx,fixed", [
    (0.125, [0, 30, 200], True), (0.125, [0, 30, 200], False),       # a sequence without keys, one with fewer keys than rows
    (-0.125, [64, 70, 300], False), (0.0, [64, 64, 100], True)])      # scores that fall with the products; equal weights
def test_rows_without_keys_and_any_scale(scale, ctx, fixed):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ssd_amd.hip import ops as H
    nh, nkv, hd, bs, new = 8, 2, 64, 16, 64
    g = torch.Generator().manual_seed(sum(ctx))
    rnd = lambda *s: torch.randn(*s, generator=g).to(BF).cuda()
    need = [-(-c // bs) for c in ctx]
    kc = torch.full((sum(need), nkv, bs, hd), float("nan"), dtype=BF, device="cuda")
    vc = kc.clone()
    bt, at, refs = torch.full((len(ctx), max(need)), -1, dtype=torch.int32), 0, []
    T = new * len(ctx)
    q = 4.0 * rnd(T, nh, hd)
    for b, c in enumerate(ctx):
        bt[b, :need[b]] = torch.arange(at, at + need[b], dtype=torch.int32)
        K, V = rnd(c, nkv, hd), rnd(c, nkv, hd)
        for j in range(need[b]):
            part = slice(j * bs, min(c, (j + 1) * bs))
            kc[at + j, :, :part.stop - part.start], vc[at + j, :, :part.stop - part.start] = K[part].transpose(0, 1), V[part].transpose(0, 1)
        at += need[b]
        refs.append(reference(q[b * new:(b + 1) * new].double(), K.double(), V.double(), scale).nan_to_num(0.0))       # (no key: zeros)
    ref = torch.cat(refs).flatten(1)
    cu = None if fixed else torch.arange(0, T + 1, new, dtype=torch.int32, device="cuda")
    rows = torch.full((T, nh * hd), 7.0, dtype=BF, device="cuda")
    H.attn_paged(q, kc, vc, bt.cuda(), bt.shape[1], torch.tensor(ctx, dtype=torch.int32).cuda(), len(ctx), T, new, nh, nkv, hd, bs, scale, cu_q=cu,
                 q_per_seq=new, out_rows=rows)
    d = (rows.double() - ref).abs()
    assert bool((d <= 2.0 ** -8 * ref.abs() + 2.0 ** -13).all()), float(d.max())          # (bounds as above)
