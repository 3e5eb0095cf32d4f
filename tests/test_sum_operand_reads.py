"""What the 1x1 kernels read for the in-place sum, walked on the host with their own arithmetic (csrc/ehip_sum_at.hpp): lanes with channels
of their own find their cell of the output, those whose channels only fill up a tile read nothing of it, nor behind it."""
import ctypes
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "deep-learning-math-kernel-research_amd", "build", "libreads_check.so")


@pytest.mark.parametrize("n,oc2,ohw,waves,tiles", [(2, 106, 75, 16, 4), (1, 1, 1, 4, 2), (3, 5, 49, 4, 1), (2, 17, 30, 4, 4), (1, 16, 12, 4, 2)])
def test_sum_operand_reads(n, oc2, ohw, waves, tiles):
    assert os.path.exists(LIB), "libreads_check.so is not built (python -c 'import __graft_entry__ as g; g.build()')"
    lib = ctypes.CDLL(LIB)
    lib.sum_operand_check.restype = ctypes.c_longlong
    assert lib.sum_operand_check(n, oc2, ohw, waves, tiles) == 0
