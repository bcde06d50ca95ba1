"""What hvdhip_ranks_sum does before anything is launched, without a GPU."""
import os
import subprocess
import sys

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


OUT_OF_MEMORY = """
import ctypes, mmap, re, resource
import horovod_amd
lib = horovod_amd.lib()
n = 30 * 1000 * 1000
zeros = mmap.mmap(-1, 8 * n)  # all sizes, and no addresses
at = ctypes.addressof(ctypes.c_char.from_buffer(zeros))
p = ctypes.cast(at, ctypes.POINTER(ctypes.c_void_p))
counts = ctypes.cast(at, ctypes.POINTER(ctypes.c_int64))
held = int(re.search(r"VmSize:\\s+(\\d+)", open("/proc/self/status").read()).group(1)) << 10
resource.setrlimit(resource.RLIMIT_AS, (held + (256 << 20),) * 2)
print("code", lib.hvdhip_ranks_sum(p, p, counts, n, 1, 7, 7, 7, 1.0, 1.0, 0, None, None), flush=True)
"""


def test_want_of_host_memory_is_a_return_code():
    """The list of outputs that is sorted for the overlap check does not fit: HVDHIP_ERR_OUT_OF_MEMORY, not an
    exception that ends the process on its way through the C interface."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", OUT_OF_MEMORY], cwd=root, capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "code -3" in r.stdout, (r.returncode, r.stdout, r.stderr[-1000:])
