"""What hvdhip_ranks_sum does before anything is launched, without a GPU."""
import pytest
import torch

from horovod_amd import DTYPE
from horovod_amd import host as H

pytestmark = pytest.mark.skipif(torch.cuda.is_available(), reason="hands host memory to the library")


class _NullStream:
    handle = None


def _copy(outs, ins, counts, dtype="float32", wire="float32", pre=1.0, pad=False):
    code = DTYPE[dtype]
    return H.ranks_sum(outs, ins, counts, 1, code, DTYPE[wire], code, pre, 1.0, _NullStream(), pad=pad)


def test_a_tensor_that_stays_as_it_is_costs_no_launch():
    """A world of one rank, in place and unscaled: there is nothing to do, and nothing fails for want of a device."""
    t = torch.ones(4096)
    p = t.data_ptr()
    assert _copy([p, 0, p + 800], [p, 0, p + 800], [100, 0, 100])
    # all that does something needs the device, which is not there
    for args in (dict(pre=0.5), dict(wire="float16"), dict(pad=True)):
        with pytest.raises(Exception):
            _copy([p], [p], [100], **args)
    with pytest.raises(Exception):
        _copy([p, p + 800], [p, p + 4000], [100, 100])
