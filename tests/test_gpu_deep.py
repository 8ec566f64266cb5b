"""The kernel for launches of few tiles (gemm_deep.hip) where it can go wrong: row counts around its tile heights, N and K around its
tiles and slabs, fewer and more slabs a tile than its rings hold, one tile a workgroup and many, every row layout.  Forced on every
shape, against the shape-agnostic kernel bit for bit (both add up 32 values of K at a time in ascending order and round once);
then the calls that reach it by default."""
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


def _tile(sizes, N, wgs):
    """The tile that the device chooses for these sizes (gemm_deep_kernel)."""
    r64, r128 = (sum(-(-n // h) for n in sizes) for h in (64, 128))
    c64, c128 = -(-N // 64), -(-N // 128)
    small, mid, wide = -(-r64 * c64 // wgs) * 16, -(-r64 * c128 // wgs) * 24, -(-r128 * c128 // wgs) * 32
    return "wide" if wide <= mid and wide < small else "small" if small <= mid else "mid"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("trans_b", [True, False])
@pytest.mark.parametrize("num_cu", [-1, 40, 16, 3])
@pytest.mark.parametrize("K", [8, 64, 72, 128, 320, 512, 584, 1000])  # 1 to 16 slabs
@pytest.mark.parametrize("sizes, N", [([63, 0, 64, 65, 1, 129], 136), ([300, 0, 127], 520), ([5], 8), ([128, 128], 128), ([0, 40], 200)])
def test_any_shape(dtype, trans_b, num_cu, K, sizes, N):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(K + N)
    s = torch.tensor(sizes, dtype=torch.int32, device=dev)
    a = torch.randn(sum(sizes), K, device=dev, generator=gen).to(dtype)
    b = (torch.randn(len(sizes), *((N, K) if trans_b else (K, N)), device=dev, generator=gen) * K ** -0.5).to(dtype)
    run = lambda: m_grouped_gemm(a, b, s, trans_b, numSM=num_cu)
    assert torch.equal(_with("deep", 2, 1, run), _with("force_generic", 1, 0, run))


def test_the_shapes_above_choose_every_tile():
    chosen = {_tile(s, n, w) for w in (256, 40, 16, 3) for s, n in (([63, 0, 64, 65, 1, 129], 136), ([300, 0, 127], 520), ([128, 128], 128))}
    assert chosen == {"small", "mid", "wide"}


@pytest.mark.parametrize("trans_b", [True, False])
def test_what_lies_beyond_a_group_is_not_added_up(trans_b):
    """NaN and infinities in the rows of other groups, the next rows of A and the other groups' weights leave no trace."""
    dev = torch.device("cuda:0")
    K, N, sizes = 264, 392, [70, 60, 50]
    a = torch.ones(sum(sizes), K, device=dev, dtype=torch.bfloat16)
    b = torch.ones(len(sizes), *((N, K) if trans_b else (K, N)), device=dev, dtype=torch.bfloat16)
    a[:70], a[130:], b[0], b[2] = float("nan"), float("inf"), float("inf"), float("nan")
    s = torch.tensor(sizes, dtype=torch.int32, device=dev)
    out = _with("deep", 2, 1, lambda: m_grouped_gemm(a, b, s, trans_b))
    assert bool((out[70:130] == K).all())


@pytest.mark.parametrize("trans_b", [True, False])
@pytest.mark.parametrize("sizes, rows, N, K", [([100, 3, 0, 61], 200, 264, 200), ([640, 2], 900, 1024, 520), ([1] * 250, 256, 64, 64), ([0, 0], 40, 72, 8)])
def test_the_default_route(sizes, rows, N, K, trans_b):
    """Groups that fill a part of the operand: rows that no group owns stay as they were, in every layout of the rows."""
    dev = torch.device("cuda:0")
    G = len(sizes)
    gen = torch.Generator(device=dev).manual_seed(K + rows)
    b = torch.randn(G, *((N, K) if trans_b else (K, N)), device=dev, generator=gen).bfloat16()
    s = torch.tensor(sizes, dtype=torch.int64, device=dev)
    stride = 128 * max(-(-max(sizes) // 128), 1)

    def check(total, starts, call):
        a = torch.randn(total, K, device=dev, generator=gen).bfloat16()

        def run():
            out = torch.full((total, N), float("nan"), device=dev, dtype=torch.bfloat16)
            call(a, out)
            return out.view(torch.int16)
        out = run()
        assert torch.equal(out, _with("deep", 0, 1, run)) and torch.equal(out, _with("force_generic", 1, 0, run))
        owned = torch.zeros(total, dtype=torch.bool)
        for at, n in zip(starts, sizes):
            owned[at:at + n] = True
        assert torch.equal(torch.isnan(out.view(torch.bfloat16)).all(1).cpu(), ~owned)

    packed = [sum(sizes[:g]) for g in range(G)]
    check(rows, packed, lambda a, out: _native.call("tgg_m_grouped_gemm", a.data_ptr(), b.data_ptr(), out.data_ptr(), s.data_ptr(), 1, G, rows, N, K,
                                                    int(trans_b), _native.BF16, -1, _native.stream_of(a)))
    check(G * stride, [g * stride for g in range(G)], lambda a, out: m_grouped_gemm_masked(a, b, out, s, stride, trans_b))
    if trans_b:
        padded = [sum(-(-n // 128) * 128 for n in sizes[:g]) for g in range(G)]
        total = sum(-(-n // 128) * 128 for n in sizes) or 128
        check(total, padded, lambda a, out: _native.call("tgg_m_grouped_gemm_padded", a.data_ptr(), b.data_ptr(), out.data_ptr(), s.data_ptr(), 1, G,
                                                         total, N, K, 128, _native.BF16, -1, _native.stream_of(a)))


@pytest.mark.parametrize("act, weight", [(torch.float8_e4m3fn, torch.float8_e4m3fn), (torch.float8_e5m2, torch.float8_e4m3fn), (torch.float8_e4m3fn, torch.float8_e5m2),
                                         (torch.float8_e5m2, torch.float8_e5m2)])
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("num_cu", [-1, 16, 3])
@pytest.mark.parametrize("K", [16, 128, 144, 512, 1040, 2048])  # 1 to 16 slabs
@pytest.mark.parametrize("sizes, N", [([63, 0, 64, 65, 1, 129], 136), ([300, 0, 127], 520), ([5], 8), ([0, 40], 200)])
def test_fp8_per_channel(act, weight, out_dtype, num_cu, K, sizes, N):
    """Against the eight-wave kernel bit for bit: the same multiplies in the same order along K, the same scaling."""
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(K + N)
    G, M = len(sizes), sum(sizes)
    a, b = torch.randn(M, K, device=dev, generator=gen).mul_(40).to(act), torch.randn(G, N, K, device=dev, generator=gen).mul_(40).to(weight)
    sa, sb = torch.rand(M, device=dev, generator=gen), torch.rand(G, N, device=dev, generator=gen).mul_(1e-3)
    s = torch.tensor(sizes, dtype=torch.int32, device=dev)
    code = {torch.float8_e4m3fn: _native.E4M3, torch.float8_e5m2: _native.E5M2}

    def run():
        out = torch.full((M + 3, N), float("nan"), device=dev, dtype=out_dtype)
        _native.call("tgg_m_grouped_gemm_fp8_channel", a.data_ptr(), sa.data_ptr(), b.data_ptr(), sb.data_ptr(), out.data_ptr(), s.data_ptr(), 0, G, M, N, K,
                     code[act], code[weight], _native.DTYPE_CODE[out_dtype], num_cu, _native.stream_of(a))
        return out.view(torch.int16)
    out = _with("deep", 2, 1, run)
    assert torch.equal(out, _with("deep", 0, 1, run)) and torch.equal(out, run())
    assert not bool(torch.isnan(out.view(out_dtype)[:M]).any()) and bool(torch.isnan(out.view(out_dtype)[M:]).all())
