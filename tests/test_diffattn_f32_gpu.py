"""The matrix-core form of the fp32 differential attention (csrc/attention_diff.hip): the last rows of sequences whose lengths lie at the edges of
steps (16 keys), segments (64) and rounds (512), against fp64 -- and the same bits whether a row comes alone, in a small batch, inside
a prompt portion, or with its segments over the grid."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def reference(q, K, V, gate, scale, lam, osc, eps):
    """One sequence's last rows q [n][H][2][D] over K [N][G][2][D], V [N][G][Dv] in fp64; row i sees the first N - n + i + 1 keys."""
    n, H = q.shape[:2]
    N, G = K.shape[:2]
    out = []
    for i in range(n):
        see = N - n + i + 1
        a = []
        for m in range(2):
            s = torch.einsum("hd,khd->hk", q[i, :, m], K[:see, :, m].repeat_interleave(H // G, 1)) * scale
            a.append(torch.einsum("hk,khv->hv", torch.softmax(s, -1), V[:see].repeat_interleave(H // G, 1)))
        o = a[0] - lam * a[1]
        out.append(o / torch.sqrt((o * o).mean(-1, keepdim=True) + eps) * osc * gate[i].unsqueeze(-1))
    return torch.stack(out).flatten(1)


@pytest.mark.parametrize("Hh,G,D,Dv,bs", [(16, 4, 64, 128, 64), (2, 2, 16, 16, 16), (16, 1, 48, 80, 32)])
def test_rows_alone_and_in_portions(Hh, G, D, Dv, bs):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ssd_amd.hip import ops as H
    eps, scale, lam, osc = 1e-5, D ** -0.5, 0.4, 0.75
    lens = [1, 15, 17, 63, 64, 65, 511, 512, 513, 1100]
    g = torch.Generator().manual_seed(D + Dv)
    rnd = lambda *s: torch.randn(*s, generator=g).cuda()
    nb = sum(-(-n // bs) for n in lens)
    order, at = torch.randperm(nb, generator=g).tolist(), 0
    kc = torch.full((nb, G, bs, 2 * D), float("nan"), device="cuda")
    vc = torch.full((nb, G, Dv, bs), float("nan"), device="cuda")
    for n in lens:
        pages = order[at:at + -(-n // bs)]
        at += len(pages)
        K, V = rnd(n, G, 2, D), rnd(n, G, Dv)
        for j, p in enumerate(pages):
            part = slice(j * bs, min(n, (j + 1) * bs))
            kc[p, :, :part.stop - part.start] = K[part].flatten(2).transpose(0, 1)
            vc[p, :, :, :part.stop - part.start] = V[part].permute(1, 2, 0)
        bt = torch.tensor([pages], dtype=torch.int32).cuda()
        rows = min(n, 40)
        q, gate = rnd(rows, Hh, 2, D), torch.sigmoid(rnd(rows, Hh))
        ctx = torch.tensor([n], dtype=torch.int32).cuda()

        def attend(a, b, slots=0, hint=0):
            T = b - a
            out = torch.zeros(T, Hh * Dv, device="cuda")
            ws = torch.full((G * slots * 4160,), float("nan"), device="cuda") if slots else None
            pos = torch.arange(n - rows + a, n - rows + b).cuda()
            H.diffattn_paged(q[a:b].contiguous(), kc, vc, gate[a:b].contiguous(), bt, len(pages), pos, 1, T, Hh, G, D, Dv, bs, scale, lam, osc,
                             eps, out, True, cu_q=torch.tensor([0, T], dtype=torch.int32).cuda(), context_lens=ctx, max_q=T,
                             workspace=ws, ctx_hint=hint)
            return out

        whole = attend(0, rows)
        ref = reference(q.double(), K.double(), V.double(), gate.double(), scale, lam, osc, eps)
        # sums of up to 1100 fp32 terms and a hardware exponential (2^-21 relative), then a norm that divides by the maps' difference
        torch.testing.assert_close(whole.double(), ref, rtol=1e-4, atol=1e-4)
        for i in {0, rows // 2, rows - 1}:
            assert torch.equal(attend(i, i + 1), whole[i:i + 1]), (n, i)
        assert torch.equal(attend(max(0, rows - 3), rows), whole[max(0, rows - 3):]), n
        # segments over the grid: room for all of them, for the first nine, a hint that falls short of the context
        for slots, hint in ((18, 1152), (9, 1152), (18, 640)):
            assert torch.equal(attend(rows - 1, rows, slots, hint), whole[rows - 1:]), (n, slots, hint)
