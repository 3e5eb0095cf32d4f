"""What the k x k kernel that shares K out among its waves (csrc/ehip_convs.hip) reads of its input, walked on the host with the
kernel's own address arithmetic (csrc/ehip_convs_at.hpp): every lane of every k-step finds its cell, and where there is none -- taps
outside the image, the missing second unit of an odd count -- the lane's offset alone lies past the buffer."""
import ctypes
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "deep-learning-math-kernel-research_amd", "build", "libreads_check.so")


@pytest.mark.parametrize("nhwc", [0, 1])
@pytest.mark.parametrize("n,ic2,ih,iw,k,stride,pad", [
    (1, 1, 8, 8, 3, 1, 1), (2, 3, 11, 9, 5, 2, 2), (3, 5, 9, 7, 7, 1, 3), (1, 7, 13, 13, 3, 2, 0), (2, 2, 6, 7, 3, 1, 1), (1, 4, 5, 5, 5, 1, 2)])
def test_split_kernel_reads(nhwc, n, ic2, ih, iw, k, stride, pad):
    assert os.path.exists(LIB), "libreads_check.so is not built (python -c 'import __graft_entry__ as g; g.build()')"
    lib = ctypes.CDLL(LIB)
    lib.conv_split_check.restype = ctypes.c_longlong
    oh, ow = ((d + 2 * pad - k) // stride + 1 for d in (ih, iw))
    assert lib.conv_split_check(nhwc, n, ic2, ih, iw, oh, ow, k, stride, pad) == 0
