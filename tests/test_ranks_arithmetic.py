"""The arithmetic of the sums over ranks as the compiler makes it, without a GPU: kernels of a few lines over the
library's own device functions are compiled for gfx950, with the scale switched on at compile time so that nothing but
the source keeps its product and the addition that follows apart."""
import os
import re
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "horovod_amd", "csrc")

PROBE = """
#include "ranks.hip"
using namespace hvdhip;
template <typename T>
__global__ void scaled_sum_k(T* out, const T* a, const T* b, double pre) {
  const typename Factor<T>::type f = (typename Factor<T>::type)pre;
  Arr<T, 1> acc = to_wire<T, T, 1>(Arr<T, 1>{a[threadIdx.x]}, f, true);
  add_to<T, 1>(acc, to_wire<T, T, 1>(Arr<T, 1>{b[threadIdx.x]}, f, true));
  out[threadIdx.x] = acc.v[0];
}
template <typename T>
__global__ void sum_k(T* out, const T* a, const T* b) {
  Arr<T, 1> acc = {a[threadIdx.x]};
  add_to<T, 1>(acc, Arr<T, 1>{b[threadIdx.x]});
  out[threadIdx.x] = acc.v[0];
}
template __global__ void sum_k<int32_t>(int32_t*, const int32_t*, const int32_t*);
template __global__ void sum_k<int64_t>(int64_t*, const int64_t*, const int64_t*);
template __global__ void scaled_sum_k<float>(float*, const float*, const float*, double);
template __global__ void scaled_sum_k<double>(double*, const double*, const double*, double);
"""


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    """probe(kernel name, "asm" or "ir"): its assembly or the compiler's intermediate code."""
    if shutil.which("hipcc") is None:
        pytest.skip("hipcc is not installed")
    tmp = tmp_path_factory.mktemp("arithmetic")
    src = str(tmp / "probe.hip")
    with open(src, "w") as f:
        f.write(PROBE)
    cmd = ["hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
           "-packed-fp32-ops", "-Wno-unused-function", "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "-S",
           "--cuda-device-only", src]

    def compiled(kind):
        out = str(tmp / kind)
        r = subprocess.run(cmd + ["-o", out] + (["-emit-llvm"] if kind == "ir" else []), stdout=subprocess.PIPE,
                           stderr=subprocess.STDOUT, timeout=600)
        assert r.returncode == 0, r.stdout.decode(errors="replace")[-2000:]
        return open(out).read()

    with ThreadPoolExecutor(2) as pool:
        texts = dict(zip(("asm", "ir"), pool.map(compiled, ("asm", "ir"))))

    def body(name, kind):
        text = texts[kind]
        start = re.search(r"^(define .*@)?_Z\d+" + name + r"\w*[:(]", text, re.M).end()
        return text[start:text.index("s_endpgm" if kind == "asm" else "\n}", start)]

    return body


@pytest.mark.parametrize("bits", [32, 64])
def test_a_scaled_element_is_rounded_before_it_is_added(probe, bits):
    """Packing stores the product in the wire type; summing reads it from there.  A fused multiply-add would round
    once where that rounds twice."""
    body = probe("scaled_sum_kI" + ("f" if bits == 32 else "d"), "asm")
    assert "v_mul_f%d" % bits in body and "v_add_f%d" % bits in body, body
    assert not re.search(r"v_(fma|fmac|mad|mac)\w*_f%d" % bits, body), body


@pytest.mark.parametrize("bits", [32, 64])
def test_integer_sums_wrap(probe, bits):
    """Overflow is defined, as in reduce.hip: the compiler has no leave to assume that there is none (nsw)."""
    body = probe("sum_kI" + ("i" if bits == 32 else "l"), "ir")
    assert re.search(r"= add i%d " % bits, body) and not re.search(r"= add \w*nsw i%d " % bits, body), body
