"""The four-wave kernel's instantiation for any K and N (gemm_w4.hip, TAIL) where it can go wrong: K around its slab of 64, its pairs
of slabs and its least of 192; N around its 256 columns with B as [G, K, N].  Forced on every shape, against the shape-agnostic
kernel bit for bit (both add up 32 values of K at a time in ascending order and round once).  At the end the launches that reach it, and
the plain instantiation, by the default route: alone, and enqueued together with the eight-wave kernel with sizes that choose either."""
import pytest
import torch

from tests._util import EIGHT_WAVE, FOUR_OR_EIGHT, FOUR_WAVE, M_GROUPED, MASKED, route_16bit
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


CUS = 8  # workgroups of the launches below: small ones then have the rounds of tiles of large ones


def _chosen(sizes, N):
    """What the sizes decide where both kernels are enqueued (sched_wide_tiles_chosen): True = the four-wave kernel."""
    full, half = (sum(-(-n // h) for n in sizes) for h in (256, 128))
    tiles_n = -(-N // 256)
    return full * -(-N // 128) > CUS and -(-half * tiles_n // CUS) * 3 > -(-full * tiles_n // CUS) * 4


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("trans_b, N, K", [(True, 1032, 776), (False, 1032, 1152), (False, 1024, 904), (True, 1024, 1024)])
@pytest.mark.parametrize("case, sizes, wide", [
    ("alone", [1500, 2, 1301, 1397], None),                                     # 512 rows a group and more, more than four rounds: the four-wave kernel alone
    ("small groups", [500, 513, 480, 300, 0, 700, 511, 300, 896], True),
    ("small groups", [470] + [40] * 8, False),                                  # groups that fill a fraction of the operand, in 128-row tiles
    ("small groups", [256] * 16 + [0] * 14, True),                              # 140 rows a group by the operand
    ("small groups", [100] * 30, False),
    ("few rounds", [330, 255, 180], True),                                      # at most four rounds, of a long K
    ("few rounds", [100, 0, 40], False),                                        # the same operand with few rows: narrow tiles
])
def test_the_default_route(dtype, trans_b, N, K, case, sizes, wide):
    dev = torch.device("cuda:0")
    G, rows = len(sizes), 4200
    if case == "few rounds":
        rows, K = 768 if N > 1024 else 1024, K + 1024
        assert -(-rows // 256) * -(-N // 128) <= 4 * CUS  # and gemm_w4.hip's likely tiles: 9 / 2 or 11 / 2 rows of them, two rounds of K = 2048
    assert route_16bit(M_GROUPED, G, rows, N, K, trans_b, num_cu=CUS) == (FOUR_WAVE if wide is None else FOUR_OR_EIGHT)
    if wide is not None:
        assert _chosen(sizes, N) == wide
    gen = torch.Generator(device=dev).manual_seed(K + rows)
    a = torch.randn(rows, K, device=dev, generator=gen).to(dtype)
    b = (torch.randn(G, *((N, K) if trans_b else (K, N)), device=dev, generator=gen) * K ** -0.5).to(dtype)
    s = torch.tensor(sizes, dtype=torch.int32, device=dev)

    def run():
        out = torch.full((rows, N), float("nan"), device=dev, dtype=dtype)
        _native.call("tgg_m_grouped_gemm", a.data_ptr(), b.data_ptr(), out.data_ptr(), s.data_ptr(), 0, G, rows, N, K, int(trans_b),
                     _native.BF16 if dtype == torch.bfloat16 else _native.F16, CUS, _native.stream_of(a))
        return out
    out = run()
    assert torch.equal(out.view(torch.int16), _with("four_wave", 0, 1, run).view(torch.int16))
    assert torch.equal(out.view(torch.int16), _with("force_generic", 1, 0, run).view(torch.int16))
    assert not bool(torch.isnan(out[:sum(sizes)]).any()) and bool(torch.isnan(out[sum(sizes):]).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("K", [904, 1024])  # the eight-wave kernels alone, both kernels
@pytest.mark.parametrize("masked, wide", [([512, 300, 511, 0, 400], True), ([40, 128, 0, 99, 128], False)])
def test_the_default_route_of_masked_launches(dtype, K, masked, wide):
    dev = torch.device("cuda:0")
    N, slots = 1032, 512
    assert _chosen(masked, N) == wide
    assert route_16bit(MASKED, len(masked), len(masked) * slots, N, K, aux=slots, num_cu=CUS) == (EIGHT_WAVE if K % 128 else FOUR_OR_EIGHT)
    gen = torch.Generator(device=dev).manual_seed(K)
    a = torch.randn(len(masked) * slots, K, device=dev, generator=gen).to(dtype)
    b = (torch.randn(len(masked), N, K, device=dev, generator=gen) * K ** -0.5).to(dtype)
    s = torch.tensor(masked, dtype=torch.int32, device=dev)

    def run():
        out = torch.full((len(masked) * slots, N), float("nan"), device=dev, dtype=dtype)
        _native.call("tgg_m_grouped_gemm_masked", a.data_ptr(), b.data_ptr(), out.data_ptr(), s.data_ptr(), 0, len(masked), slots, len(masked) * slots, N, K,
                     1, _native.BF16 if dtype == torch.bfloat16 else _native.F16, CUS, _native.stream_of(a))
        return out
    out = run()
    assert torch.equal(out.view(torch.int16), _with("force_generic", 1, 0, run).view(torch.int16))
    for g, n in enumerate(masked):
        block = out[g * slots:(g + 1) * slots]
        assert not bool(torch.isnan(block[:n]).any()) and bool(torch.isnan(block[n:]).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("num_cu", [8, 3, 1, 32, 64])  # full and half tiles in every order, in one workgroup; last rounds cut into half tiles
@pytest.mark.parametrize("K", [256, 320, 512])
@pytest.mark.parametrize("N, trans_b", [(520, True), (512, False), (264, False)])
@pytest.mark.parametrize("sizes", [[128, 1, 64, 65], [129, 384, 16, 200, 300, 127, 640], [256, 17, 256, 0, 385]])
def test_half_tiles(dtype, num_cu, K, N, trans_b, sizes):
    """Tiles of at most 128 rows beside full ones: 64 rows per wave row, a part of them or none."""
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(K + N)
    s = torch.tensor(sizes, dtype=torch.int32, device=dev)
    a = torch.randn(sum(sizes), K, device=dev, generator=gen).to(dtype)
    b = (torch.randn(len(sizes), *((N, K) if trans_b else (K, N)), device=dev, generator=gen) * K ** -0.5).to(dtype)
    run = lambda: m_grouped_gemm(a, b, s, trans_b, numSM=num_cu)
    assert torch.equal(_with("four_wave", 2, 1, run), _with("force_generic", 1, 0, run))


@pytest.mark.parametrize("trans_b", [True, False])
@pytest.mark.parametrize("N, K, sizes, num_cu", [
    (512, 768, [1, 1023, 256], 8),        # 1.6 rounds of likely tiles, of one group mostly
    (256, 776, [400, 0, 800], 8),         # a tail
    (264, 1032, [500, 130, 138], 8),      # N cut as well
    (256, 768, [400, 3, 797], 8),         # 0.81 of a round
    (256, 896, [256, 767, 1], 8),         # 0.69 of one
    (256, 768, [512, 0, 1, 511] * 75, -1),  # more groups than the four-wave kernel has threads
])
def test_mid_size_launches(trans_b, N, K, sizes, num_cu):
    """Launches of some size that the four-wave kernel does not get by default, by it and by the eight-wave kernels: the same bits."""
    dev = torch.device("cuda:0")
    assert route_16bit(M_GROUPED, len(sizes), sum(sizes), N, K, trans_b, num_cu=num_cu) != FOUR_WAVE
    gen = torch.Generator(device=dev).manual_seed(N + K)
    s = torch.tensor(sizes, dtype=torch.int32, device=dev)
    a = torch.randn(sum(sizes), K, device=dev, generator=gen).to(torch.bfloat16)
    b = (torch.randn(len(sizes), *((N, K) if trans_b else (K, N)), device=dev, generator=gen) * K ** -0.5).to(torch.bfloat16)
    run = lambda: _with("deep", 0, 1, lambda: m_grouped_gemm(a, b, s, trans_b, numSM=num_cu))
    want = _with("force_generic", 1, 0, run)
    assert torch.equal(run(), want) and torch.equal(_with("four_wave", 2, 1, run), want)
