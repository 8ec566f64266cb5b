"""K-grouped launches cut along K (kg_split.hpp) where they can go wrong: outputs around the tile, segments of no, one and many parts beside
one another, lengths that do not divide, few workgroups, fp16 and both FP8 formats.  Integer inputs whose sums fp32 holds exactly, so
that any way of adding them up gives the oracle's bits; then random ones against 64-bit sums."""
import ctypes
import gc

import pytest
import torch

from triton_grouped_gemm_amd import _native
from triton_grouped_gemm_amd.gemm.BF16.k_grouped_gemm import k_grouped_gemm
from triton_grouped_gemm_amd.gemm.FP8.k_grouped_gemm_channel_expert import matmul as fp8_k_grouped

pytestmark = pytest.mark.gpu


def _cut(groups, m, n, k_total, fp8, num_cu=-1):
    need = ctypes.c_int64()
    _native.call("tgg_k_grouped_split_bytes", groups, m, n, k_total, int(fp8), num_cu, ctypes.addressof(need))
    return need.value


def _parts(workspace, groups):
    """How many parts the device made of each group (the workspace's head)."""
    return workspace[:8 * groups].view(torch.int32).view(groups, 2)[:, 1].tolist()


SIZES = [[9001, 0, 130, 2500], [20000, 1, 63, 64], [3000] * 4, [16000], [0, 0, 40000, 7]]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("num_cu", [-1, 100])
@pytest.mark.parametrize("m, n", [(256, 256), (264, 520), (8, 1000), (384, 64)])
@pytest.mark.parametrize("sizes", SIZES)
@pytest.mark.parametrize("wide", [False, True])
def test_16_bit(dtype, num_cu, m, n, sizes, wide):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(m + n)
    G, total = len(sizes), sum(sizes)
    s = torch.tensor(sizes, dtype=torch.int64 if wide else torch.int32, device=dev)
    need = _cut(G, m, n, total, False, num_cu)
    assert need > 0
    workspace = torch.empty(need, dtype=torch.uint8, device=dev)

    def run(a, b):
        c = torch.full((G, m, n), float("nan"), device=dev, dtype=dtype)
        _native.call("tgg_k_grouped_gemm_split", a.data_ptr(), b.data_ptr(), c.data_ptr(), s.data_ptr(), int(wide), G, m, n, total,
                     _native.DTYPE_CODE[dtype], num_cu, _native.work_queue(dev).data_ptr(), workspace.data_ptr(), need, _native.stream_of(a))
        return c

    starts = [sum(sizes[:g]) for g in range(G)]
    a, b = (torch.randint(-1, 2, (total, w), device=dev, generator=gen).to(dtype) for w in (m, n))
    ref = torch.stack([a[at:at + k].double().t() @ b[at:at + k].double() for at, k in zip(starts, sizes)])
    out = run(a, b)
    assert max(_parts(workspace, G)) > 1 or max(sizes) < 9000
    assert torch.equal(out, ref.float().to(dtype))
    a, b = (torch.randn(total, w, device=dev, generator=gen).to(dtype) for w in (m, n))
    out = run(a, b)
    assert torch.equal(out, run(a, b))  # the same parts, added up in the same order
    assert torch.equal(k_grouped_gemm(a, b, s, numSM=num_cu), out)  # the entry point brings a workspace of its own
    ref = torch.stack([a[at:at + k].double().t() @ b[at:at + k].double() for at, k in zip(starts, sizes)])
    half_ulp = 2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12  # of the value: one rounding; besides fp32 sums of up to 40000 products
    assert bool(((out.double() - ref).abs() <= ref.abs() * half_ulp * 2.02 + 1e-5 * max(max(sizes), 1) ** 0.5).all())


@pytest.mark.parametrize("fa, fb", [(torch.float8_e4m3fn, torch.float8_e4m3fn), (torch.float8_e5m2, torch.float8_e4m3fn),
                                    (torch.float8_e4m3fn, torch.float8_e5m2), (torch.float8_e5m2, torch.float8_e5m2)])
@pytest.mark.parametrize("m, n", [(256, 256), (272, 528), (16, 1008)])
@pytest.mark.parametrize("sizes, runs_tuned", [([16000, 0, 128, 4112], True), ([20000 - 16, 16, 64, 128], True), ([24000, 0, 128, 4104, 8], False)])
def test_fp8(fa, fb, m, n, sizes, runs_tuned):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(m + n)
    G, total = len(sizes), sum(sizes)
    total += -total % 16
    s = torch.tensor(sizes, dtype=torch.int32, device=dev)
    x, y = (torch.randint(-1, 2, (w, total), device=dev, generator=gen).float().to(f) for w, f in ((m, fa), (n, fb)))
    xs, ys = (2.0 ** torch.randint(-2, 3, (G, w), device=dev, generator=gen).float() for w in (m, n))
    need = _cut(G, m, n, total, True)
    assert need > 0
    workspace = torch.empty(need, dtype=torch.uint8, device=dev)
    out = torch.full((G, m, n), float("nan"), device=dev, dtype=torch.bfloat16)
    code = {torch.float8_e4m3fn: _native.E4M3, torch.float8_e5m2: _native.E5M2}
    _native.call("tgg_k_grouped_gemm_fp8_channel_split", x.data_ptr(), xs.data_ptr(), y.data_ptr(), ys.data_ptr(), out.data_ptr(), s.data_ptr(), G, m, n,
                 total, code[fa], code[fb], -1, _native.work_queue(dev).data_ptr(), workspace.data_ptr(), need, _native.stream_of(x))
    assert max(_parts(workspace, G)) > 1 or not runs_tuned  # counts that are no multiples of 16 are the shape-agnostic kernel's, whole
    starts = [sum(sizes[:g]) for g in range(G)]
    ref = torch.stack([(x[:, at:at + k].double() @ y[:, at:at + k].double().t()) * xs[g][:, None].double() * ys[g][None, :].double()
                       for g, (at, k) in enumerate(zip(starts, sizes))])
    assert torch.equal(out, ref.float().bfloat16())
    assert torch.equal(out, fp8_k_grouped(x, xs.t(), y, ys.t(), s, m, n, total, G, 1 if fa == torch.float8_e4m3fn else 2, 1 if fb == torch.float8_e4m3fn else 2))


def test_what_the_bits_depend_on():
    """The sizes and the number of workgroups decide the parts, nothing else; a call with segment bounds has none."""
    dev = torch.device("cuda:0")
    a, b = torch.randn(30000, 256, device=dev).bfloat16(), torch.randn(30000, 264, device=dev).bfloat16()
    s = torch.tensor([17000, 4, 12996], dtype=torch.int32, device=dev)
    ends = s.cumsum(0).to(torch.int32)
    runs = {cus: k_grouped_gemm(a, b, s, numSM=cus) for cus in (-1, 64, 100)}
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        again = {cus: k_grouped_gemm(a, b, s.long(), numSM=cus) for cus in runs}
    torch.cuda.synchronize()
    assert all(torch.equal(runs[cus], again[cus]) for cus in runs)
    _native.set_option("kg_split", 0)
    try:
        uncut = k_grouped_gemm(a, b, s)
    finally:
        _native.set_option("kg_split", 1)
    assert all(torch.equal(k_grouped_gemm(a, b, s, ends - s, ends, numSM=cus), uncut) for cus in runs)
    assert all(not torch.equal(r, uncut) for r in runs.values())


def _planned_parts(sizes, m, n, unit, tile, part, cost, cus=256):
    """split_plan's choice in Python integers: how many parts each group is cut into."""
    up = lambda a, b: -(-a // b)
    per_group = up(m, 256) * up(n, 256)
    steps = [up(k, unit) for k in sizes]
    share = up(sum(steps) * per_group, cus)
    ranked = sorted(steps, reverse=True)
    uncut = max([share] + [(t + 1) * ranked[t * cus // per_group] for t in range(256) if t * cus // per_group < len(sizes)])
    best, chosen = None, None
    if uncut > share + cost + tile:
        for t in range(256):
            c = max(8, share * (64 + t % 64) >> (8 - t // 64))
            parts = [1 if k <= c else up(k, c) for k in steps]
            length = [k if q == 1 else up(k, q) for k, q in zip(steps, parts)]
            slots = sum(q for q in parts if q > 1)
            long = [(q, k) for q, k, x in zip(parts, steps, length) if 2 * x > c]
            n_long, sum_long = sum(q for q, _ in long), sum(k for _, k in long)
            expected = up(n_long * per_group, cus) * sum_long // n_long if n_long else 0
            expected = max(expected, share, max(length))
            expected += up(sum(parts) * per_group, cus) * tile + up(slots * per_group * part, cus) + cost
            if 0 < slots <= 2 * cus // per_group and sum(parts) <= 512 and expected + expected // 12 < uncut + up(len(sizes) * per_group, cus) * tile:
                if best is None or expected < best:
                    best, chosen = expected, parts
    return chosen or [1] * len(sizes)


@pytest.mark.parametrize("m, n, sizes", [
    (264, 264, [2560] * 200),                                   # equal ones: nothing is cut
    (256, 128, [37000] * 3 + [1500] * 61 + [49000, 49000, 1] + [6400] * 63),  # runs of equals, across the lanes of a wave
    (264, 520, [4000 + 640 * (g % 7) for g in range(90)]),
    (128, 128, [(2909 * g * g) % 9000 for g in range(130)]),    # hardly two alike
    (64, 256, [0] * 64 + [1000000] + [3000] * 190 + [400000]),  # every thread's group
    (2304, 1152, [130, 40000, 64]),
])
def test_the_plan(m, n, sizes):
    """The device's plan, which takes a group at a time from lanes' registers, runs of equals at once and divides by reciprocals, against the plan's
    definition: how many parts each group is in; and the result, exact."""
    dev = torch.device("cuda:0")
    assert torch.cuda.get_device_properties(dev).multi_processor_count == 256
    G, total = len(sizes), sum(sizes)
    gen = torch.Generator(device=dev).manual_seed(G)
    a, b = (torch.randint(-1, 2, (total, w), device=dev, generator=gen).bfloat16() for w in (m, n))
    s = torch.tensor(sizes, dtype=torch.int32, device=dev)
    need = _cut(G, m, n, total, False)
    assert need > 0
    workspace, c = torch.empty(need, dtype=torch.uint8, device=dev), torch.full((G, m, n), float("nan"), device=dev, dtype=torch.bfloat16)
    _native.call("tgg_k_grouped_gemm_split", a.data_ptr(), b.data_ptr(), c.data_ptr(), s.data_ptr(), 0, G, m, n, total, _native.BF16, -1,
                 _native.work_queue(dev).data_ptr(), workspace.data_ptr(), need, _native.stream_of(a))
    assert _parts(workspace, G) == _planned_parts(sizes, m, n, 64, 3, 20, 8)  # WgradSplitCost
    at = 0
    for g, k in enumerate(sizes):
        assert torch.equal(c[g], (a[at:at + k].float().t() @ b[at:at + k].float()).bfloat16()), g
        at += k


def test_what_is_not_cut():
    assert _cut(128, 2048, 1536, 32768, False) == 0   # many tiles, short segments
    assert _cut(4, 256, 256, 4096, False) == 0        # short segments
    assert _cut(300, 256, 256, 1 << 20, False) == 0   # more groups than the kernel's table
    assert _cut(8, 256, 256, 1 << 20, True) > 0 and _cut(8, 256, 256, (1 << 20) + 8, True) == 0


def test_a_cut_call_can_be_captured():
    dev = torch.device("cuda:0")
    a, b = torch.randn(20000, 256, device=dev).bfloat16(), torch.randn(20000, 512, device=dev).bfloat16()
    s = torch.tensor([12000, 8000], dtype=torch.int32, device=dev)
    queue = torch.zeros(_native.QUEUE_WORDS, dtype=torch.int32, device=dev)
    assert _cut(2, 256, 512, 20000, False) > 0
    want = k_grouped_gemm(a, b, s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = k_grouped_gemm(a, b, s, queue=queue)
    for sizes in ([12000, 8000], [100, 19900], [0, 20000], [12000, 8000]):
        s.copy_(torch.tensor(sizes, dtype=torch.int32))
        out.zero_()
        graph.replay()
        eager = k_grouped_gemm(a, b, s)
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
    assert torch.equal(out, want)


@pytest.mark.parametrize("path", ["native", "python", "fp8"])
def test_a_call_without_memory_for_its_workspace(path):
    """A launch that may be cut along K wants up to 128 MiB; where the allocator has no more to give it runs uncut, as it did before there was a cut."""
    dev = torch.device("cuda:0")
    G, m, n, total = 4, 256, 256, 32768
    assert _cut(G, m, n, total, path == "fp8") > 100 << 20
    gen = torch.Generator(device=dev).manual_seed(1)
    s = torch.tensor([20000, 4768, 8000, 0], dtype=torch.int32, device=dev)
    if path == "fp8":
        x, y = (torch.randn(w, total, device=dev, generator=gen).to(torch.float8_e4m3fn) for w in (m, n))
        xs, ys = (torch.rand(G, w, device=dev, generator=gen).t() for w in (m, n))
        run = lambda: fp8_k_grouped(x, xs, y, ys, s, m, n, total, G)
    else:
        a, b = (torch.randn(total, w, device=dev, generator=gen).bfloat16() for w in (m, n))
        if path == "python":  # the native call path takes plain tensors only
            s = torch.stack([s, s], 1)[:, 0]
        run = lambda: k_grouped_gemm(a, b, s)
    _native.set_option("kg_split", 0)
    try:
        uncut = run()
    finally:
        _native.set_option("kg_split", 1)
    cut = run()
    assert path == "fp8" or not torch.equal(cut, uncut)  # with room it is summed in another order (the rounding hides that for these FP8 sums)
    del cut
    torch.cuda.synchronize()
    gc.collect()
    torch.cuda.empty_cache()
    limit = (torch.cuda.memory_reserved(dev) + (16 << 20)) / torch.cuda.get_device_properties(dev).total_memory
    torch.cuda.set_per_process_memory_fraction(limit, dev)
    try:
        with pytest.raises(torch.OutOfMemoryError):
            torch.empty(100 << 20, dtype=torch.uint8, device=dev)
        out = run()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, dev)
    assert torch.equal(out, uncut)
