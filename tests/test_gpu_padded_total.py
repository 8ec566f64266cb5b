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


def _small_call(dev, block_m=128):
    gen = torch.Generator(device=dev).manual_seed(3)
    sizes = torch.tensor([100, 0, 128, 1], dtype=torch.int32, device=dev)
    a, b = (torch.randint(-3, 4, shape, device=dev, generator=gen).bfloat16() for shape in ((3 * block_m, 64), (4, 136, 64)))
    want = torch.zeros(3 * block_m, 136, device=dev)
    for g, row, n in ((0, 0, 100), (2, block_m, 128), (3, 2 * block_m, 1)):
        want[row:row + n] = a[row:row + n].float() @ b[g].float().t()
    owned = torch.zeros(3 * block_m, dtype=torch.bool, device=dev)
    for row, n in ((0, 100), (block_m, 128), (2 * block_m, 1)):
        owned[row:row + n] = True
    return a, b, sizes, want.bfloat16(), owned


def _busy(dev):
    """Some milliseconds of work in front, so that the total's word is long in coming and the stream is waited for."""
    x = torch.ones(8192, 8192, dtype=torch.bfloat16, device=dev)
    for _ in range(12):
        x = (x @ x).clamp_(-1, 1)
    done = torch.cuda.Event()
    done.record()
    return done, x


@pytest.mark.parametrize("callers", [False, True])
def test_a_total_that_is_long_in_coming(callers):
    dev = torch.device("cuda:0")
    a, b, sizes, want, owned = _small_call(dev)
    torch.cuda.synchronize()
    for wrong in (False, True, False):
        out = torch.full_like(want, -7.0) if callers else None
        done, _ = _busy(dev)
        assert not done.query()
        if wrong:
            with pytest.raises(ValueError, match="expected M=384, got M=256"):
                m_grouped_bf16_nt_contiguous(a[:256], b, sizes, out=None if out is None else out[:256])
            assert out is None or bool((out == -7.0).all())
        else:
            out = m_grouped_bf16_nt_contiguous(a, b, sizes, out=out)
            assert done.query()  # the call has waited for the total, hence for what lay in front of it
            assert torch.equal(out[owned], want[owned])


@pytest.mark.parametrize("busy", [False, True])
def test_a_gemm_that_fails_while_the_total_is_on_its_way(busy):
    """The GEMM is refused (A is not 16-byte aligned) when the kernel that writes the total has been launched: the call raises, but not before the word has been
    written, whose memory the next calls get."""
    dev = torch.device("cuda:0")
    a, b, sizes, want, owned = _small_call(dev)
    crooked = torch.zeros(a.numel() + 8, dtype=a.dtype, device=dev)[1:a.numel() + 1].view_as(a)
    torch.cuda.synchronize()
    for _ in range(20):
        if busy:
            done, _keep = _busy(dev)
        with pytest.raises(RuntimeError, match="aligned"):
            m_grouped_bf16_nt_contiguous(crooked, b, sizes)
        if busy:
            assert done.query()
        out = m_grouped_bf16_nt_contiguous(a, b, sizes)
        assert torch.equal(out[owned], want[owned])
