"""Large-tile GEMM of many token rows (csrc/gemm_big.hip) against fp64 products: edges of every tile shape, K remainders of a split,
strided rows, both epilogues."""
import pytest
import torch

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


@pytest.fixture(scope="module")
def H():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ssd_amd.hip import ops
    return ops


def frag(H, x):
    out = torch.zeros(H.frag_numel(*x.shape), dtype=BF, device="cuda")
    H.rows_to_frag(x.cuda().contiguous(), out, *x.shape)
    return out


def operands(M, N, K, seed):
    g = torch.Generator().manual_seed(seed)
    x, w, b = torch.randn(M, K, generator=g).to(BF), (torch.randn(N, K, generator=g) / K ** 0.5).to(BF), torch.randn(N, generator=g).to(BF)
    return x, w, b


# one rounding to bf16 (relative 2^-9 at most, 2^-8 between neighbours) after fp32 sums, whose own error (K terms, 2^-24 each, of a sum
# of absolute values about sqrt(K) times the result's size) stays far below it; against the size of the row's terms where they cancel
def check(y, ref, what):
    y = y.double().cpu()
    tol = 2.0 ** -8 * ref.abs() + 2.0 ** -12
    assert bool(((y - ref).abs() <= tol).all()), (what, float(((y - ref).abs() - tol).max()))


@pytest.mark.parametrize("shape", [-1, 0, 1, 2, 3, 4])
@pytest.mark.parametrize("M,N,K,splits", [(1, 16, 96, 1), (129, 272, 96, 1), (257, 144, 352, 3), (255, 512, 1024, 8), (64, 4112, 160, 1), (700, 128, 2080, 2)])
def test_rows(H, shape, M, N, K, splits):
    x, w, b = operands(M, N, K, M + N + K)
    ref = x.double() @ w.double().T
    ws = torch.empty(splits * M * N, dtype=torch.float32, device="cuda")
    xf, wf = frag(H, x), frag(H, w)
    for bias, ldy in ((None, N), (b, N + 12)):
        y = torch.full((M, ldy), 7.0, dtype=BF, device="cuda")
        H.gemm_big(xf, wf, y, M, N, K, ldy, bias=None if bias is None else bias.cuda(), workspace=ws, shape=shape, splits=splits)
        check(y[:, :N], ref if bias is None else ref + bias.double(), (shape, M, N, K, splits, ldy))
        assert bool((y[:, N:] == 7.0).all())


@pytest.mark.parametrize("shape", [-1, 0, 1, 2, 3, 4])
@pytest.mark.parametrize("M,I,K,splits", [(130, 96, 96, 1), (257, 160, 416, 2)])
def test_silu(H, shape, M, I, K, splits):
    x, w, _ = operands(M, 2 * I, K, M + I)
    wf = torch.zeros(2 * I * K, dtype=BF, device="cuda")
    H.rows_to_frag(w.cuda(), wf, 2 * I, K, mode=1)
    act = torch.zeros(H.frag_numel(M, I), dtype=BF, device="cuda")
    ws = torch.empty(splits * M * 2 * I, dtype=torch.float32, device="cuda")
    H.gemm_big(frag(H, x), wf, act, M, 2 * I, K, 0, epilogue=H.EPI_SILU_FRAG, workspace=ws, shape=shape, splits=splits)
    rows = torch.zeros(M, I, dtype=BF, device="cuda")
    H.frag_to_rows(act, rows, M, I)
    z = (x.double() @ w.double().T).to(torch.float32)
    g, u = z[:, :I].to(BF).double(), z[:, I:].to(BF).double()
    # the result's rounding, 2^-9 of it; a gate or up value that rounds to its neighbour moves by 2^-8 of itself (silu's slope is below 1.1)
    ref = g * torch.sigmoid(g) * u
    tol = 2.0 ** -8 * (1.5 * ref.abs() + 1.1 * (g * u).abs()) + 2.0 ** -20
    assert bool(((rows.double().cpu() - ref).abs() <= tol).all())


def test_refusals(H):
    from ssd_amd.hip.lib import SsdHipError
    x = torch.zeros(1 << 16, dtype=BF, device="cuda")
    for M, N, K, ldy in ((0, 16, 96, 16), (16, 24, 96, 24), (16, 16, 80, 16), (16, 16, 64, 16), (16, 16, 96, 8), (16, 16, 96, 18)):
        with pytest.raises(SsdHipError):
            H.gemm_big(x, x, x, M, N, K, ldy)
    with pytest.raises(SsdHipError):
        H.gemm_big(x, x, x, 16, 16, 96, 16, shape=2, splits=2)          # too few k-steps, and no workspace
