"""ssd_sample_rows over slices of the vocabulary (csrc/stochastic.hip) against the same draw on the host: one workgroup per row, slices with remainders,
unaligned rows, greedy rows, -inf and NaN logits, several rows per temperature, rescaled tokens."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

M64 = np.uint64(0xffffffffffffffff)


def mix(z):
    with np.errstate(over="ignore"):
        z = (z + np.uint64(0x9e3779b97f4a7c15)) & M64
        z = ((z ^ (z >> np.uint64(30))) * np.uint64(0xbf58476d1ce4e5b9)) & M64
        z = ((z ^ (z >> np.uint64(27))) * np.uint64(0x94d049bb133111eb)) & M64
    return z ^ (z >> np.uint64(31))


def scores(x, T, seed, salt, row, boost, log_x):
    x = x.astype(np.float64)
    if T == 0:
        return x
    i = np.arange(len(x), dtype=np.uint64)
    h = mix(np.uint64(seed) ^ mix((np.uint64(salt) << np.uint64(40)) ^ (np.uint64(row) << np.uint64(32)) ^ i))
    u = ((h >> np.uint64(40)).astype(np.float64) + 0.5) / 16777216.0
    s = x / T - np.log(-np.log(u))
    s[boost] += log_x
    return s


@pytest.mark.parametrize("T,V,ld", [(1, 128256, 128256), (3, 8193, 8200), (2, 20011, 20011), (70, 9000, 9000), (1, 8192, 8192), (5, 37, 40), (1100, 8200, 8200), (192, 8200, 8200),
                                    (256, 20011, 20011), (257, 8200, 8208), (512, 9000, 9000), (600, 8200, 8200)])
def test_the_draw_is_the_hosts(T, V, ld):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ssd_amd.hip import ops as H
    g = torch.Generator().manual_seed(V)
    x = (torch.randn(T, ld, generator=g) * 3).to(torch.bfloat16)
    x[0, V // 2] = float("-inf")
    if T > 2:
        x[1, ::2] = float("nan")             # never chosen
        x[2] = float("-inf")
    rpt = 2 if T > 4 else 1
    temps = torch.rand(-(-T // rpt), generator=g) + 0.3
    if T > 1:
        temps[-1] = 0.0
    for boost in (None, torch.randint(0, V, (T, 3), generator=g, dtype=torch.int32)):
        out, out2 = torch.full((T,), -7, dtype=torch.int64, device="cuda"), torch.full((T,), -7, dtype=torch.int64, device="cuda")
        kw = {} if boost is None else dict(boost_idx=boost.cuda(), boost_k=3, boost_x=2.5)
        H.sample_rows(x.cuda(), ld, T, V, temps.cuda(), rpt, torch.tensor([987654321], dtype=torch.int64, device="cuda"), 5, out, out2, **kw)
        assert torch.equal(out, out2)
        for r in (range(T) if T < 100 else range(0, T, 97)):
            s = scores(x[r, :V].float().numpy(), float(temps[r // rpt]), 987654321, 5, r, [] if boost is None else boost[r].unique().tolist(),
                       math.log(2.5))
            if not np.isfinite(s[~np.isnan(s)]).any():
                continue                     # every candidate is -inf: the first index, checked below
            got = int(out[r])
            # the device's logarithms are good to 2^-21 of a Gumbel value of at most 17
            assert 0 <= got < V and s[got] >= np.nanmax(s) - 1e-4 * max(1.0, abs(np.nanmax(s))), (T, V, r, got)
        if T > 2:
            assert int(out[2]) == 0
