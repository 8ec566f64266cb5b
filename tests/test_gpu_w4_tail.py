"""The four-wave kernel's instantiation for any K and N (gemm_w4.hip, TAIL) where it can go wrong: K around its slab of 64, its pairs
of slabs and its least of 192; N around its 256 columns with B as [G, K, N].  Forced on every shape, against the shape-agnostic
kernel bit for bit (both add up 32 values of K at a time in ascending order and round once)."""
import pytest
import torch

from triton_grouped_gemm_amd import _native
from triton_grouped_gemm_amd.gemm.BF16.m_grouped_gemm_masked_TMA import m_grouped_gemm_masked
from triton_grouped_gemm_amd.gemm.BF16.m_grouped_gemm_TMA import m_grouped_gemm

pytestmark = pytest.mark.gpu


def _with(option, value, default, fn):
    _native.set_option(option, value)
    try:
        return fn()
    finally:
        _native.set_option(option, default)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("num_cu", [-1, 8, 3])
@pytest.mark.parametrize("K", [192, 200, 248, 256, 264, 312, 320, 328, 376, 384, 392, 1000])
@pytest.mark.parametrize("N, trans_b", [(520, True), (256, True), (256, False), (264, False), (504, False), (8, False), (1000, False)])
def test_any_k_and_n(dtype, num_cu, K, N, trans_b):
    dev = torch.device("cuda:0")
    sizes = [300, 0, 129, 256, 1, 511]
    gen = torch.Generator(device=dev).manual_seed(K + N)
    s = torch.tensor(sizes, dtype=torch.int32, device=dev)
    a = torch.randn(sum(sizes), K, device=dev, generator=gen).to(dtype)
    b = (torch.randn(len(sizes), *((N, K) if trans_b else (K, N)), device=dev, generator=gen) * K ** -0.5).to(dtype)
    run = lambda: m_grouped_gemm(a, b, s, trans_b, numSM=num_cu)
    assert torch.equal(_with("four_wave", 2, 1, run), _with("force_generic", 1, 0, run))


@pytest.mark.parametrize("K", [200, 264, 392])
def test_masked_with_a_tail(K):
    dev = torch.device("cuda:0")
    torch.manual_seed(K)
    s = torch.tensor([256, 0, 100, 129], dtype=torch.int32, device=dev)
    a, b = torch.randn(4 * 256, K, device=dev).bfloat16(), torch.randn(4, 520, K, device=dev).bfloat16()

    def run():
        out = torch.zeros(4 * 256, 520, device=dev, dtype=torch.bfloat16)
        m_grouped_gemm_masked(a, b, out, s, 256)
        return out
    assert torch.equal(_with("four_wave", 2, 1, run), _with("force_generic", 1, 0, run))


@pytest.mark.parametrize("trans_b", [True, False])
def test_what_lies_beyond_a_tail_is_not_added_up(trans_b):
    """NaN and infinities in the rows of other groups, the next rows of A and the other groups' weights leave no trace."""
    dev = torch.device("cuda:0")
    K, N, sizes = 264, 392, [70, 60, 50]
    a = torch.ones(sum(sizes), K, device=dev, dtype=torch.bfloat16)
    b = torch.ones(len(sizes), *((N, K) if trans_b else (K, N)), device=dev, dtype=torch.bfloat16)
    a[:70], a[130:], b[0], b[2] = float("nan"), float("inf"), float("inf"), float("nan")
    s = torch.tensor(sizes, dtype=torch.int32, device=dev)
    out = _with("four_wave", 2, 1, lambda: m_grouped_gemm(a, b, s, trans_b))
    assert bool((out[70:130] == K).all())
