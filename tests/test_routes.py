"""CPU: which kernels a 16-bit launch enqueues, as its host code decides it from what it knows: the operand's rows, not the groups' sizes, which
are on the GPU (tgg_debug_route_16bit).  The reference chooses by architecture and autotuning (gemm/BF16/m_grouped_gemm_TMA.py:25-52)."""
import ctypes

import pytest

from tests._util import EIGHT_WAVE, FOUR_OR_EIGHT, FOUR_WAVE, M_GROUPED, MASKED, PADDED, route_16bit as route
from triton_grouped_gemm_amd import _native

@pytest.mark.parametrize("trans_b", [True, False])
@pytest.mark.parametrize("groups", [257, 367, 512])
@pytest.mark.parametrize("rows", [200, 256, 300, 511])
@pytest.mark.parametrize("n, k", [(512, 768), (1536, 2048), (2816, 1032)])
def test_more_groups_than_threads(trans_b, groups, rows, n, k):
    """The four-wave kernel's group table is one thread's work beyond 256 groups, 35-45 us in front of a launch (367 groups of 256 rows, N = 512,
    K = 768: 106 us by the eight-wave kernel, whose 512 threads make it together, 171 here): only launches of long groups can carry that."""
    assert route(M_GROUPED, groups, groups * rows, n, k, trans_b) == EIGHT_WAVE
    assert route(M_GROUPED, groups, groups * 1024, n, k, trans_b) == FOUR_WAVE


@pytest.mark.parametrize("trans_b", [True, False])
@pytest.mark.parametrize("k", [2048, 2056])  # without and with a tail
@pytest.mark.parametrize("groups, rows, n, expected", [
    (128, 128, 4096, FOUR_OR_EIGHT), (128, 199, 3072, FOUR_OR_EIGHT), (128, 256, 1536, FOUR_OR_EIGHT), (128, 511, 1408, FOUR_OR_EIGHT),
    (128, 512, 1408, FOUR_WAVE),
    (64, 312, 1416, FOUR_OR_EIGHT), (8, 1000, 4096, FOUR_OR_EIGHT),  # two rounds of likely tiles, not large
    (17, 597, 2368, EIGHT_WAVE), (32, 557, 840, EIGHT_WAVE), (8, 1462, 1024, EIGHT_WAVE),  # fewer
])
def test_the_rows_of_an_operand_do_not_say_how_many_the_groups_own(trans_b, k, groups, rows, n, expected):
    """Only launches of many long groups go to the four-wave kernel unseen: the groups may own a part of the operand's rows, and then the eight-wave
    kernel's narrower tiles can be the faster ones (17 groups, 10149 rows of which half are theirs, N = 2368, K = 2048: 72 us, and 90 by the other)."""
    assert route(M_GROUPED, groups, groups * rows, n, k, trans_b) == expected
    if trans_b:  # padded: groups of one row each are a whole block of the operand's
        assert route(PADDED, groups, groups * rows, n, k, aux=256) == expected


@pytest.mark.parametrize("k, expected", [(1536, FOUR_OR_EIGHT), (1544, EIGHT_WAVE)])
def test_masked_launches_are_decided_on_the_device(k, expected):
    assert route(MASKED, 128, 128 * 512, 4096, k, aux=512) == expected
    assert route(MASKED, 128, 128 * 4096, 4096, k, aux=4096) == expected


def _split_bytes(groups, m, n, tokens, fp8):
    need = ctypes.c_int64(-1)
    _native.call("tgg_k_grouped_split_bytes", groups, m, n, tokens, int(fp8), -1, ctypes.addressof(need))
    return need.value


@pytest.mark.parametrize("fp8", [False, True])
def test_the_size_of_the_operands_does_not_decide_whether_segments_are_cut(fp8):
    """A launch of few outputs is cut along K however many tokens there are, also where an operand has 2^31 values and more."""
    for tokens in (1 << 17, 1 << 19, 1 << 20, 1 << 21):
        assert _split_bytes(5, 2048, 256, tokens, fp8) > 0, tokens
