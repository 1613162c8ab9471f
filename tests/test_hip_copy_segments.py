"""ssd_copy_segments: a step's inputs from pinned memory and its results back, in one launch."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def H():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from ssd_amd.hip import ops
    return ops


def test_sizes_both_ways_and_rewritten_memory(H):
    """Part words of 16 bytes, empty segments first, last and in between, more chunks than a launch has threads; the host rewrites its buffers between
    launches; nothing behind a segment's words is touched."""
    sizes = [0, 1, 3, 4, 5, 0, 1025, 600_001, 7, 0]
    room = [max(n, 1) + 9 for n in sizes]
    host = [torch.zeros(r, dtype=torch.int32).pin_memory() for r in room]
    dev = [torch.zeros(r, dtype=torch.int32, device="cuda") for r in room]
    back = [torch.zeros(r, dtype=torch.int32).pin_memory() for r in room]
    there, home = H.SegmentCopies(list(zip(host, dev))), H.SegmentCopies(list(zip(dev, back)))
    for turn in range(3):
        for i, h in enumerate(host):
            h.copy_(torch.arange(h.numel(), dtype=torch.int32) * (turn + 3) + i)
            dev[i].fill_(-1)
            back[i].fill_(-2)
        for i, n in enumerate(sizes):
            there.words[i] = home.words[i] = n
        there.launch()
        home.launch()
        torch.cuda.synchronize()
        for i, n in enumerate(sizes):
            assert torch.equal(dev[i][:n].cpu(), host[i][:n]) and bool((dev[i][n:] == -1).all()), (turn, n)
            assert torch.equal(back[i][:n], host[i][:n]) and bool((back[i][n:] == -2).all()), (turn, n)


def test_refusals(H):
    from ssd_amd.hip.lib import load_library
    f = load_library().ssd_copy_segments
    a = torch.zeros(64, dtype=torch.int32, device="cuda")

    def call(src, dst, words, n):
        return f((ctypes.c_void_p * 1)(src), (ctypes.c_void_p * 1)(dst), (ctypes.c_int32 * 1)(words), n, 0)
    p = a.data_ptr()
    assert call(p, p + 128, -1, 1) < 0 and call(p, p + 128, 1 << 29, 1) < 0 and call(p, p + 128, 4, 0) < 0 and call(p, p + 128, 4, 11) < 0
    assert call(p + 4, p + 128, 4, 1) < 0 and call(p, p + 132, 4, 1) < 0 and call(0, p, 4, 1) < 0 and call(p, 0, 4, 1) < 0
    assert call(0, 0, 0, 1) == 0
