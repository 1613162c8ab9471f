"""Few-row form of the row-major GEMM (csrc/gemm_rows.hip) against fp64 products: row counts around the ring shapes (4, 8, 16), K below, at and off
the 256-byte stages and the four waves' runs, features off 16, gathered rows of uneven groups; a row's bits do not depend on the rows beside it."""
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


def operands(M, N, K, f32, E=None):
    g = torch.Generator().manual_seed(M + N + K)
    dt = torch.float32 if f32 else BF
    w = torch.randn(*([E] if E else []), N, K, generator=g) / K ** 0.5
    return torch.randn(M, K, generator=g).to(dt).cuda(), w.to(dt).cuda()


# fp32 sums of K terms of variance 1 / K: at most K roundings of 2^-24 of a partial sum below 6 in bf16 products (K <= 2^13: 2^-9 at the
# worst, a thousandth of it in practice); the fp32 mode's segments keep chains at 256 + K / 256 roundings: 2^-13
def tol(f32):
    return 2.0 ** -13 if f32 else 2.0 ** -9


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("K", [64, 96, 128, 256, 288, 1024, 2080, 3072, 7424])
def test_rows_of_every_ring_shape(H, K, f32):
    for M, N in ((1, 16), (4, 33), (5, 40), (8, 17), (9, 100), (16, 130)):
        x, w = operands(M, N, K, f32)
        y = torch.full((M, N), 7.0, device="cuda")
        H.gemm_rows(x, w, y, M, N, K, f32, 0)
        d = float((y.double() - x.double() @ w.double().T).abs().max())
        assert d <= tol(f32), (M, N, K, d)
        one = torch.zeros(1, N, device="cuda")
        H.gemm_rows(x[M - 1:], w, one, 1, N, K, f32, 0)
        assert torch.equal(one[0], y[M - 1]), (M, N, K)


@pytest.mark.parametrize("M,N,K,G", [(3, 4096, 1024, 1), (3, 4096, 1032, 1), (3, 4097, 1032, 1), (16, 4096, 2056, 1), (5, 4112, 2056, 1), (9, 2048, 4104, 2), (9, 2049, 4104, 2),
                                     (4, 40, 1000, 3), (1, 8, 14720, 1), (4, 50, 128, 3), (16, 33, 256, 2), (5, 33, 264, 2),
                                     (7, 8192, 512, 1), (7, 8193, 512, 1), (16, 8208, 264, 1)])
def test_bf16_one_four_and_eight_waves(H, M, N, K, G):
    """Both sides of the lines between them -- 512 workgroups of 16 features and K = 256 or 512, 256 workgroups and K = 1024 -- with the last run a part of
    one."""
    g = torch.Generator().manual_seed(M + N + K)
    w = (torch.randn(G, N, K, generator=g) / K ** 0.5).to(BF).cuda()
    x = torch.randn(M, G * K, generator=g).to(BF).cuda()
    y = torch.full((M, G * N), 7.0, device="cuda")
    H.gemm_rows_batched(x, w, y, M, N, K, G, G * K, K, G * N, N, False)
    one = torch.zeros(1, G * N, device="cuda")
    H.gemm_rows_batched(x[M - 1:], w, one, 1, N, K, G, G * K, K, G * N, N, False)
    assert torch.equal(one[0], y[M - 1])
    for i in range(G):
        d = float((y[:, i * N:(i + 1) * N].double() - x[:, i * K:(i + 1) * K].double() @ w[i].double().T).abs().max())
        assert d <= tol(False) * max(1.0, K / 2 ** 13), (M, N, K, i, d)


@pytest.mark.parametrize("K", [8, 24, 40, 136, 264, 1032])
def test_bf16_ends_inside_an_operand(H, K):
    """What lies behind a row's end is not part of its sum, whatever it holds."""
    for M, N in ((3, 16), (7, 31), (16, 50)):
        x, w = operands(M, N, K, False)
        xs = torch.full((M, K + 8), float("nan"), dtype=BF, device="cuda")
        xs[:, :K] = x
        y = torch.full((M, N), 7.0, device="cuda")
        H.gemm_rows_batched(xs, w, y, M, N, K, 1, K + 8, 0, N, 0, False)
        d = float((y.double() - x.double() @ w.double().T).abs().max())
        assert d <= tol(False), (M, N, K, d)


@pytest.mark.parametrize("f32,K", [(False, 320), (True, 320), (False, 2056), (True, 2080)])
def test_grouped_chunks(H, f32, K):
    """Runs of 0, 1, 4, 7 and 33 gathered rows: one, two and four row pieces, and three 16-row chunks in turn."""
    N, runs = 70, [1, 0, 4, 7, 33]
    offs = [0]
    for c in runs:
        offs.append(offs[-1] + c)
    rows = offs[-1]
    x, w = operands(rows, N, K, f32, E=len(runs))
    idx = torch.randperm(2 * rows, generator=torch.Generator().manual_seed(5))[:rows].int().cuda()
    y = torch.full((rows, N), 7.0, device="cuda")
    H.gemm_rows_grouped(x, w, y, torch.tensor(offs, dtype=torch.int32, device="cuda"), len(runs), rows, N, K, f32, row_idx=idx, idx_div=2)
    xg = x[(idx // 2).long()].double()
    ref = torch.cat([xg[offs[e]:offs[e + 1]] @ w[e].double().T for e in range(len(runs))])
    d = float((y.double() - ref).abs().max())
    assert d <= tol(f32), d
