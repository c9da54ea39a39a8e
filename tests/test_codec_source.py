"""The codec's kernels take their buffers as __restrict__ pointers: none may
point into another's array."""
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpugraph500_amd", "csrc")


def test_no_argument_points_into_the_decoders_record():
    with open(os.path.join(CSRC, "g5_codec.hip")) as f:
        src = f.read()
    kernels = re.findall(r"__global__[^{;]*?\((.*?)\)\s*\{", src, re.S)
    assert any("__restrict__ meta" in k and "__restrict__ flag" in k for k in kernels)
    # the record (d_meta) is passed whole, as `meta`, and nothing inside it is
    host = src[src.index("size_t S4Codec::bind"):]
    assert re.findall(r"d_meta\s*\+|&\s*d_meta\s*\[", host) == []
