"""The residual norm (csrc/norm.hip) over its thread classes -- 256 to 1024 threads, one or two chunks each -- and rows on both sides of the blocks of
128 that are dealt out to the XCDs: every row comes out once, in rows and fragment-major, with the residual's bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [32, 2048, 2080, 4064, 4096, 4128, 8192, 8224, 16384])
@pytest.mark.parametrize("T", [1, 127, 128, 300])
def test_rows_and_fragments(T, H):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ssd_amd.hip import ops as K
    g = torch.Generator().manual_seed(T + H)
    x, res = torch.randn(T, H, generator=g).bfloat16().cuda(), torch.randn(T, H, generator=g).bfloat16().cuda()
    w = torch.randn(H, generator=g).bfloat16().cuda()
    out, new = torch.zeros(T, H, dtype=torch.bfloat16, device="cuda"), torch.zeros(T, H, dtype=torch.bfloat16, device="cuda")
    frag = torch.zeros(K.frag_numel(T, H), dtype=torch.bfloat16, device="cuda")
    rows = torch.zeros_like(out)
    K.rmsnorm(x, w, 1e-5, T, H, res_in=res, res_out=new, out_rows=out, out_frag=frag)
    K.frag_to_rows(frag, rows, T, H)
    s = x.float() + res.float()
    assert torch.equal(new, s.bfloat16()) and torch.equal(rows, out)
    ref = s.double() / torch.sqrt((s.double() ** 2).mean(1, keepdim=True) + 1e-5) * w.double()
    # one rounding to bf16 (2^-9 of the value, 2^-8 to be at a tie's safe side); fp32 sums of at most 16384 squares are exact to 2^-13 of it
    assert bool(((out.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-6).all())
