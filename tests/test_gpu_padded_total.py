"""The padded total that the contiguous entry points compare with M, as the GPU writes it to page-locked memory, against the reference's
expression (gemm/deep_gemm_ops.py:49-51: sizes as int32, each rounded up to block_m, summed)."""
import pytest
import torch

from triton_grouped_gemm_amd import _native
from triton_grouped_gemm_amd.gemm.deep_gemm_ops import m_grouped_bf16_nt_contiguous
from triton_grouped_gemm_amd.gemm.layout import round_up_to_alignment

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("block_m", [1, 128, 384])
@pytest.mark.parametrize("groups", [1, 63, 64, 65, 512])
def test_padded_total(dtype, block_m, groups):
    gen = torch.Generator().manual_seed(groups)
    sizes = torch.randint(-300, 5000, (groups,), generator=gen).to(dtype)
    if dtype == torch.int64:
        sizes[0] += 1 << 33  # taken as int32, as the reference's conversion does
    word = torch.zeros(2, dtype=torch.int64).pin_memory()
    on_gpu = sizes.cuda()
    _native.call("tgg_padded_total", on_gpu.data_ptr(), int(dtype == torch.int64), groups, block_m, word.data_ptr(), _native.stream_of(on_gpu))
    torch.cuda.synchronize()
    assert word.tolist() == [int(round_up_to_alignment(sizes.to(torch.int32), block_m).sum()), 1]


def test_no_groups():
    """The reference's check comes first: rows where there are no groups for them are a ValueError, small as the call may be."""
    dev = torch.device("cuda:0")
    a, b = torch.zeros(128, 64, dtype=torch.bfloat16, device=dev), torch.zeros(0, 128, 64, dtype=torch.bfloat16, device=dev)
    out = torch.zeros(128, 128, dtype=torch.bfloat16, device=dev)
    with pytest.raises(ValueError, match="expected M=0, got M=128"):
        m_grouped_bf16_nt_contiguous(a, b, torch.zeros(0, dtype=torch.int32, device=dev), out=out)
