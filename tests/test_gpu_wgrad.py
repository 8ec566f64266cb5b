"""The four-wave weight-gradient kernel (gemm_wgrad.hip) where it can go wrong: segments around its K step of 32 tokens, its
step pairs and its shortest tile of four steps, outputs around its 256x256 tiles, fewer and more tiles than workgroups, workgroup
counts with and without per-XCD queues.  Forced on every shape, against the eight-wave kernel bit for bit (both add
up 32 tokens at a time in ascending order and round once) and against torch's fp32 product."""
import pytest
import torch

from triton_grouped_gemm_amd import _native
from triton_grouped_gemm_amd.gemm.BF16.k_grouped_gemm_TMA import k_grouped_gemm

pytestmark = pytest.mark.gpu

EDGES = [0, 1, 31, 32, 33, 63, 64, 65, 95, 96, 97, 127, 128, 129, 159, 161, 0, 192, 193, 257]


def _run(four_wave, a, b, s, num_cu, bounds=()):
    _native.set_option("four_wave", four_wave)
    try:
        return k_grouped_gemm(a, b, s, *bounds, numSM=num_cu)
    finally:
        _native.set_option("four_wave", 1)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("num_cu", [-1, 8, 7])
@pytest.mark.parametrize("sizes, M, N", [
    (EDGES, 256, 256),           # every segment length at a single full tile
    (EDGES, 8, 520),             # one row of blocks, a ragged third column tile
    ([300, 0, 4, 1000], 264, 248),  # ragged in both directions, one column tile short of its width
    ([0, 0, 0], 512, 256),       # nothing to add up anywhere
    ([1], 1032, 776),            # one token
    ([2049], 776, 1544),         # a single long segment: more tiles than the small grids have workgroups
    ([129] * 256, 128, 136),     # as many groups as the kernel has threads
])
def test_weight_gradient_kernel_at_its_edges(dtype, num_cu, sizes, M, N):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(len(sizes) + M)
    rows = sum(sizes)
    a = torch.randn(max(rows, 1), M, device=dev, generator=gen).to(dtype)
    b = torch.randn(max(rows, 1), N, device=dev, generator=gen).to(dtype)
    s = torch.tensor(sizes, dtype=torch.int32, device=dev)
    out = _run(2, a, b, s, num_cu)
    assert torch.equal(out.view(torch.int16), _run(0, a, b, s, num_cu).view(torch.int16))
    end = torch.cumsum(s, 0).to(torch.int32)
    bounds = (end - s, end)
    assert torch.equal(out, _run(2, a, b, s, num_cu, bounds))
    eps = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11  # half an output ulp; 2 % and 2e-6 of the largest for the order of the sum
    at = 0
    for g, n in enumerate(sizes):
        ref = a[at:at + n].float().t() @ b[at:at + n].float()
        assert bool(((out[g].float() - ref).abs() <= ref.abs() * eps * 1.02 + 2e-6 * ref.abs().max()).all()), f"group {g}"
        at += n
    assert int(_native.work_queue(dev, None).abs().sum()) == 0  # handed back zeroed


def test_rows_beyond_a_segment_are_not_added_up():
    """Infinities and NaN in the tokens of the neighbouring groups, and in columns beside a ragged tile, stay where they are."""
    dev = torch.device("cuda:0")
    sizes = [40, 33, 50, 31]
    a = torch.ones(sum(sizes), 264, device=dev, dtype=torch.bfloat16)
    b = torch.ones(sum(sizes), 264, device=dev, dtype=torch.bfloat16)
    a[:40] = float("inf")
    b[40 + 33:] = float("nan")
    out = _run(2, a, b, torch.tensor(sizes, device=dev, dtype=torch.int32), -1)
    assert bool((out[1] == 33).all()) and bool(torch.isinf(out[0]).all()) and bool(torch.isnan(out[2:]).all())
