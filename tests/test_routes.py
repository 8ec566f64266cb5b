"""CPU: which kernels a 16-bit launch enqueues, as its host code decides it from what it knows: the operand's rows, not the groups' sizes, which
are on the GPU (tgg_debug_route_16bit).  The reference chooses by architecture and autotuning (gemm/BF16/m_grouped_gemm_TMA.py:25-52)."""
import ctypes

import pytest

from triton_grouped_gemm_amd import _native

GENERIC, EIGHT_WAVE, FOUR_WAVE, FOUR_OR_EIGHT, DEEP, WGRAD = range(6)
M_GROUPED, PADDED, MASKED, K_GROUPED = 0, 1, 2, 4


def route(mode, groups, rows, n, k, trans_b=True, aux=0, num_cu=256):
    out = ctypes.c_int32(-1)
    _native.call("tgg_debug_route_16bit", mode, groups, rows, aux, n, k, int(trans_b), num_cu, ctypes.addressof(out))
    return out.value


@pytest.mark.parametrize("trans_b", [True, False])
@pytest.mark.parametrize("groups", [257, 367, 512])
@pytest.mark.parametrize("rows", [200, 256, 300, 511])
@pytest.mark.parametrize("n, k", [(512, 768), (1536, 2048), (2816, 1032)])
def test_more_groups_than_threads(trans_b, groups, rows, n, k):
    """The four-wave kernel's group table is one thread's work beyond 256 groups, 35-45 us in front of a launch (367 groups of 256 rows, N = 512,
    K = 768: 106 us by the eight-wave kernel, whose 512 threads make it together, 171 here): only launches of long groups can carry that."""
    assert route(M_GROUPED, groups, groups * rows, n, k, trans_b) == EIGHT_WAVE
    assert route(M_GROUPED, groups, groups * 1024, n, k, trans_b) == FOUR_WAVE
