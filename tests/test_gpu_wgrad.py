"""The four-wave weight-gradient kernels.  16-bit (gemm_wgrad.hip) where it can go wrong: segments around its K step of 32 tokens, its
step pairs and its shortest tile of four steps, outputs around its 256x256 tiles, fewer and more tiles than workgroups, workgroup
counts with and without per-XCD queues.  Forced on every shape, against the eight-wave kernel bit for bit (both add
up 32 tokens at a time in ascending order and round once) and against torch's fp32 product.  FP8 (fp8_w4.hip): around its slab
of 128 tokens and its shortest tile of two slabs."""
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


@pytest.mark.parametrize("queued", [True, False])
@pytest.mark.parametrize("num_cu", [-1, 64, 8])
@pytest.mark.parametrize("tokens", [31, 32, 63, 64, 95, 96])
@pytest.mark.parametrize("N", [256, 264])
def test_short_segments_by_the_default_route(queued, num_cu, tokens, N):
    """Either side of the lines between the two kernels (wgrad_supported), on launches large enough for the four-wave one."""
    dev = torch.device("cuda:0")
    G, M = 70, 1544
    sizes = [tokens + (g % 3 - 1) * 20 for g in range(G - 1)]
    sizes.append(tokens * G - sum(sizes))
    gen = torch.Generator(device=dev).manual_seed(tokens)
    a, b = (torch.randn(tokens * G, n, device=dev, generator=gen).bfloat16() for n in (M, N))
    s = torch.tensor(sizes, dtype=torch.int32, device=dev)

    def run(four_wave):
        out = torch.full((G, M, N), float("nan"), device=dev, dtype=torch.bfloat16)
        _native.set_option("four_wave", four_wave)
        try:
            _native.call("tgg_k_grouped_gemm_sizes", a.data_ptr(), b.data_ptr(), out.data_ptr(), s.data_ptr(), 0, G, M, N, tokens * G, _native.BF16,
                         num_cu, _native.work_queue(dev, None).data_ptr() if queued else 0, _native.stream_of(a))
        finally:
            _native.set_option("four_wave", 1)
        return out.view(torch.int16)
    out = run(1)
    assert torch.equal(out, run(0)) and torch.equal(out, run(2))
    assert not bool(torch.isnan(out.view(torch.bfloat16)).any())


@pytest.mark.parametrize("M, N", [(2 ** 21 - 8, 8), (2 ** 21, 8), (2 ** 22, 8), (8, 2 ** 21 - 8), (8, 2 ** 21), (8, 2 ** 22)])
def test_token_rows_that_are_too_long_for_the_touched_window(M, N):
    """256 touched token rows have to lie below 1 GiB, the offset of what is not fetched: longer ones stay with the eight-wave kernel."""
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(M + N)
    a, b = (torch.randn(40, n, device=dev, generator=gen).bfloat16() for n in (M, N))
    s = torch.tensor([33, 7], dtype=torch.int32, device=dev)
    out = _run(2, a, b, s, -1)
    assert torch.equal(out.view(torch.int16), _run(0, a, b, s, -1).view(torch.int16))
    ref = a[33:].float().t() @ b[33:].float()
    assert bool(((out[1].float() - ref).abs() <= ref.abs() * 2.0 ** -8 * 1.02 + 2e-6 * ref.abs().max()).all())


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


def _run_fp8(four_wave, x, xs, y, ys, s, num_cu):
    _native.set_option("four_wave", four_wave)
    try:
        (M, T), N, G = x.shape, y.shape[0], s.numel()
        out = torch.full((G, M, N), float("nan"), device=x.device, dtype=torch.bfloat16)
        code = {torch.float8_e4m3fn: _native.E4M3, torch.float8_e5m2: _native.E5M2}
        _native.call("tgg_k_grouped_gemm_fp8_channel_queued", x.data_ptr(), xs.data_ptr(), y.data_ptr(), ys.data_ptr(), out.data_ptr(), s.data_ptr(),
                     G, M, N, T, code[x.dtype], code[y.dtype], num_cu, _native.work_queue(x.device, None).data_ptr(), _native.stream_of(x))
        return out
    finally:
        _native.set_option("four_wave", 1)


@pytest.mark.parametrize("fx, fy", [(torch.float8_e4m3fn, torch.float8_e4m3fn), (torch.float8_e5m2, torch.float8_e4m3fn),
                                    (torch.float8_e4m3fn, torch.float8_e5m2), (torch.float8_e5m2, torch.float8_e5m2)])
@pytest.mark.parametrize("num_cu", [-1, 8, 7])
@pytest.mark.parametrize("sizes, M, N, spare", [
    ([0, 16, 112, 128, 144, 240, 256, 272, 384, 400, 0, 640], 256, 256, 0),  # every segment length at a single full tile
    ([0, 16, 112, 128, 144, 240, 256, 272, 384, 400, 0, 640], 5, 520, 48),   # five rows, a ragged third column tile, codes behind the last segment
    ([304, 0, 16, 1008], 263, 248, 0),
    ([0, 0], 300, 256, 16),
    ([2048], 776, 1544, 0),
    ([128] * 256, 40, 136, 0),
])
def test_fp8_weight_gradient_kernel_at_its_edges(fx, fy, num_cu, sizes, M, N, spare):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(len(sizes) + M)
    T = sum(sizes) + spare
    x = (torch.randn(M, T, device=dev, generator=gen) * 8).to(fx)
    y = (torch.randn(N, T, device=dev, generator=gen) * 8).to(fy)
    xs, ys = (torch.rand(len(sizes), n, device=dev, generator=gen) + 0.5 for n in (M, N))
    s = torch.tensor(sizes, dtype=torch.int32, device=dev)
    out = _run_fp8(1, x, xs, y, ys, s, num_cu)
    assert torch.equal(out.view(torch.int16), _run_fp8(0, x, xs, y, ys, s, num_cu).view(torch.int16))  # the eight-wave kernel's bits
    at = 0
    for g, n in enumerate(sizes):
        ref = (x[:, at:at + n].float() @ y[:, at:at + n].float().t()) * xs[g][:, None] * ys[g][None, :]
        # one rounding to bf16; 2e-3 of the largest for products that one multiply instruction truncates (below 2^-13 of its largest) and the sum's order
        assert bool(((out[g].float() - ref).abs() <= ref.abs() * 2.0 ** -8 * 1.02 + 2e-3 * ref.abs().max()).all()), f"group {g}"
        at += n
    assert int(_native.work_queue(dev, None).abs().sum()) == 0


def test_fp8_codes_of_other_segments_are_not_added_up():
    dev = torch.device("cuda:0")
    s = torch.tensor([48, 32, 80], dtype=torch.int32, device=dev)
    x, y = torch.ones(300, 160, device=dev), torch.ones(264, 160, device=dev)
    x[:, :48] = float("nan")
    y[:, 80:] = float("nan")
    one = lambda n: torch.ones(3, n, device=dev)
    out = _run_fp8(1, x.to(torch.float8_e4m3fn), one(300), y.to(torch.float8_e4m3fn), one(264), s, -1)
    assert bool((out[1] == 32).all()) and bool(torch.isnan(out[0]).all()) and bool(torch.isnan(out[2]).all())


@pytest.mark.parametrize("sizes, T", [([48, 40, 72], 160), ([160, 7], 160), ([96, 80], 160), ([16, 33, 111], 160)])
def test_fp8_counts_that_are_no_multiples_of_16(sizes, T):
    """Exactly one of the two enqueued kernels computes: odd counts, odd counts that the axis' end clips away or to a multiple of 16."""
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(T + sizes[0])
    x = (torch.randn(300, T, device=dev, generator=gen) * 8).to(torch.float8_e4m3fn)
    y = (torch.randn(264, T, device=dev, generator=gen) * 8).to(torch.float8_e4m3fn)
    one = lambda n: torch.ones(len(sizes), n, device=dev)
    out = _run_fp8(1, x, one(300), y, one(264), torch.tensor(sizes, dtype=torch.int32, device=dev), -1)
    at = 0
    for g, n in enumerate(sizes):
        end = min(T, at + n)
        ref = x[:, at:end].float() @ y[:, at:end].float().t()
        assert bool(((out[g].float() - ref).abs() <= ref.abs() * 2.0 ** -8 * 1.02 + 2e-3 * ref.abs().max()).all()), f"group {g}"
        at = end
