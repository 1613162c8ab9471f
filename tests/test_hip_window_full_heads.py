"""Heads of exactly 64 and 128 (csrc/attention_window.hip): the decode form's own kernels and the prompt form's, over pages that hold NaN where no key was
stored, against the statement and with the tolerances of tests/test_tumudra_ops_gpu.py."""
import pytest

from tests.test_tumudra_ops_gpu import check, store_and_attend

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("bs", [32, 64])
@pytest.mark.parametrize("window,lens,new", [(40, [150, 37, 121], [3, 2, 1]),             # decode batches, keys cut over workgroups
                                             (0, [1, 33, 64, 300], [1, 1, 1, 1]),
                                             (0, [700, 321], [700, 321]),                 # prompts: whole, and behind cached keys
                                             (0, [641, 513], [400, 512]),
                                             (530, [704, 600], [640, 600])])
def test_heads_of_exactly_64_and_128(D, bs, window, lens, new):
    case = (False, 8, 2, D, D, window, D // 2, bs, True, True)
    check(*store_and_attend(case, lens, new), False)
