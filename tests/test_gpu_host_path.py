"""The native call path (csrc/host.cpp): it takes the ordinary eager call and gives what the operator and the wrapper give;
it leaves everything else -- gradients, tracing modes, operands that need conversion, invalid arguments -- to them."""
import ctypes
import re
import subprocess
import sys
import sysconfig
import threading
from pathlib import Path

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from triton_grouped_gemm_amd import _native, ops
from triton_grouped_gemm_amd.gemm.BF16.k_grouped_gemm import k_grouped_gemm
from triton_grouped_gemm_amd.gemm.BF16.m_grouped_gemm import m_grouped_gemm
from triton_grouped_gemm_amd.gemm.BF16.m_grouped_gemm_masked_TMA import m_grouped_gemm_masked
from triton_grouped_gemm_amd.gemm.FP8.m_grouped_gemm_channel_expert import gmm_fp8_act_per_channel_w_per_expert


def test_cpu_operands_are_left_to_the_wrapper():
    a, b, s = torch.zeros(8, 8, dtype=torch.bfloat16), torch.zeros(1, 8, 8, dtype=torch.bfloat16), torch.tensor([8])
    assert _native.host().m_grouped_gemm(a, b, s, True, -1) is None
    with pytest.raises(AssertionError, match="GPU"):
        m_grouped_gemm(a, b, s, True)


def test_the_operators_are_their_definitions():
    """The entry points that are operators are the operators' definitions, with what belongs to one; an implementation for
    all devices takes the native path out.  In a process of its own: registrations last."""
    code = """
import inspect, torch
from triton_grouped_gemm_amd.gemm.BF16.m_grouped_gemm import m_grouped_gemm
from triton_grouped_gemm_amd.gemm.FP8.m_grouped_gemm_channel_expert import gmm_fp8_act_per_channel_w_per_expert as fp8
a, b, s = torch.randn(8, 8), torch.randn(1, 8, 8), torch.tensor([8])
for op, args, name in ((m_grouped_gemm, (a, b, s), 'm_grouped_gemm'),
                       (fp8, (a, a[:, :1], b, b[:, 0], s), 'gmm_fp8_act_per_channel_w_per_expert')):
    assert isinstance(op, torch.library.CustomOpDef) and op.__name__ == name and op.__doc__
    assert list(inspect.signature(op).parameters)[0] == 'A' and not op.replaced
    op.register_autograd(lambda ctx, g: (g * 3, *[None] * (len(args) - 1)))
    op.register_kernel('cpu')(lambda x, *rest: x + 1)
    x = a.clone().requires_grad_(True)
    out = op(x, *args[1:])
    out.sum().backward()
    assert torch.equal(out, a + 1) and torch.equal(x.grad, torch.full_like(a, 3.0)) and not op.replaced
    assert torch.equal(torch.compile(lambda *t: op(*t) * 2, fullgraph=True, backend='eager')(*args), (a + 1) * 2)
    torch.library.opcheck(op, args, test_utils='test_schema')
    op.register_kernel(None)(lambda x, *rest: x + 2)
    assert op.replaced
print("checked")
"""
    run = subprocess.run([sys.executable, "-c", code], cwd=Path(_native.__file__).parents[1], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0 and "checked" in run.stdout, run.stderr[-2000:]


def test_the_interpreter_lock_is_taken_again_when_an_exception_passes(tmp_path):
    """The scope in which the native call path gives up the lock, as it stands in its source, left by an exception: the
    handler that makes a Python error of it needs the lock.  Nothing else in that source gives the lock up."""
    source = (Path(_native.__file__).parent / "csrc" / "host.cpp").read_text()
    assert "_ALLOW_THREADS" not in source and "PyEval_SaveThread" in source
    scope = re.search(r"class Unlocked \{.*?\n\};", source, re.S).group(0)
    (tmp_path / "probe.cpp").write_text("#include <Python.h>\n#include <stdexcept>\n" + scope + """
extern "C" int locked_after_throw() {
  try { const Unlocked unlocked; if (PyGILState_Check()) return -1; throw std::runtime_error("x"); } catch (...) {}
  const int held = PyGILState_Check();
  if (!held) PyGILState_Ensure();
  return held;
}""")
    so = tmp_path / "probe.so"
    subprocess.run(["g++", "-std=c++17", "-shared", "-fPIC", f"-I{sysconfig.get_paths()['include']}", str(tmp_path / "probe.cpp"),
                    "-o", str(so)], check=True)
    assert ctypes.PyDLL(str(so)).locked_after_throw() == 1


def _operands(dev, dtype=torch.bfloat16, trans_b=True):
    g = torch.Generator().manual_seed(3)
    sizes = torch.tensor([70, 0, 33, 97], dtype=torch.int32, device=dev)
    a = torch.randn(200, 72, generator=g).to(dtype).to(dev)
    b = torch.randn(*((4, 40, 72) if trans_b else (4, 72, 40)), generator=g).to(dtype).to(dev)
    return a, b, sizes


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("trans_b", [True, False])
@pytest.mark.parametrize("wide", [False, True])
def test_direct_call_equals_the_operator(dev, dtype, trans_b, wide):
    a, b, sizes = _operands(dev, dtype, trans_b)
    sizes = sizes.to(torch.int64) if wide else sizes
    want = torch.ops.moe.m_grouped_gemm(a, b, sizes, trans_b)
    got = _native.host().m_grouped_gemm(a, b, sizes, trans_b, -1)
    assert got is not None and got.dtype == dtype and torch.equal(got, want)
    assert torch.equal(m_grouped_gemm(A=a, B=b, size_per_group=sizes, trans_b=trans_b, numSM=8), want)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # the caller's current stream is the one that is used
        other = m_grouped_gemm(a * 2, b, sizes, trans_b)
    torch.cuda.current_stream().wait_stream(side)
    assert torch.equal(other, torch.ops.moe.m_grouped_gemm(a * 2, b, sizes, trans_b))


@pytest.mark.gpu
def test_what_is_left_to_the_operator(dev):
    a, b, sizes = _operands(dev)
    host = _native.host()
    call = lambda x=a, w=b, s=sizes, t=True: host.m_grouped_gemm(x, w, s, t, -1)
    assert call() is not None
    assert call(x=a.clone().requires_grad_(True)) is None
    with torch.no_grad():
        assert call(x=a.clone().requires_grad_(True)) is not None
    assert call(x=a[:, :64]) is None and call(x=a.t().contiguous().t()) is None and call(x=a.float()) is None
    assert call(s=sizes.cpu()) is None and call(s=sizes[:3]) is None and call(s=sizes.float()) is None and call(t=1) is None
    class Tensor2(torch.Tensor):
        pass
    assert call(x=a.as_subclass(Tensor2)) is None
    seen = []

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))
    with Watch():
        out = m_grouped_gemm(a, b, sizes, True)
    assert any("m_grouped_gemm" in f for f in seen) and torch.equal(out, call())
    from torch._subclasses.fake_tensor import FakeTensorMode
    with FakeTensorMode(allow_non_fake_inputs=False) as mode:
        fake = m_grouped_gemm(mode.from_tensor(a), mode.from_tensor(b), mode.from_tensor(sizes), True)
        assert type(fake).__name__ == "FakeTensor" and tuple(fake.shape) == (200, 40)
    with pytest.raises(AssertionError, match="K of A should be equal"):
        m_grouped_gemm(a[:, :64].contiguous(), b, sizes, True)
    with pytest.raises(TypeError):
        host.m_grouped_gemm(a, b)


@pytest.mark.gpu
def test_forward_mode_and_tracing_are_left_to_the_autograd_functions(dev):
    """A tangent or a trace must not be dropped: the autograd functions refuse the one and are recorded in the other."""
    import torch.autograd.forward_ad as fwd
    a, b, sizes = _operands(dev)
    idx = torch.randint(0, 4, (200, 2), device=dev, dtype=torch.int32)
    rows, where = ops.permute(a, idx, num_experts=4)
    probs = torch.rand(200, 2, device=dev)
    with fwd.dual_level():
        for call in (lambda: ops.gmm(fwd.make_dual(a, a), b, sizes, True), lambda: ops.gmm(a, fwd.make_dual(b, b), sizes, True),
                     lambda: ops.permute(fwd.make_dual(a, a), idx, num_experts=4),
                     lambda: ops.unpermute(rows, where, fwd.make_dual(probs, probs))):
            with pytest.raises(RuntimeError, match="jvp|forward"):
                call()
    traced = torch.jit.trace(lambda x: m_grouped_gemm(x, b, sizes, True), (a,), check_trace=False)
    assert torch.equal(traced(a * 2), m_grouped_gemm(a * 2, b, sizes, True))


@pytest.mark.gpu
def test_permute_gives_zeros_where_no_gradient_arrives(dev):
    class Stop(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            return x.sum()

        @staticmethod
        def backward(ctx, _):
            return None
    x = torch.randn(16, 8, device=dev, requires_grad=True)
    idx = torch.randint(0, 4, (16, 2), device=dev, dtype=torch.int32)
    grad, = torch.autograd.grad(Stop.apply(ops.permute(x, idx, num_experts=4)[0]), x)
    assert torch.equal(grad, torch.zeros_like(x))


@pytest.mark.gpu
def test_other_entry_points_agree_with_their_wrappers(dev):
    """Strided copies of the operands, which the native path refuses, against the same operands as they are."""
    a, b, sizes = _operands(dev)
    grad = torch.randn(200, 56, device=dev).to(torch.bfloat16)
    end = sizes.cumsum(0).int()
    assert torch.equal(k_grouped_gemm(a, grad, sizes), k_grouped_gemm(a, grad, sizes, end - sizes, end))
    lhs = torch.randn(4 * 128, 72, device=dev).to(torch.bfloat16)
    outs = [torch.zeros(4 * 128, 40, device=dev, dtype=torch.bfloat16) for _ in range(2)]
    assert m_grouped_gemm_masked(lhs, b, outs[0], sizes, 128) is None
    assert m_grouped_gemm_masked(lhs, b, outs[1], sizes, 128, 1) is None
    assert torch.equal(*outs) and outs[0].any()
    a8, b8 = torch.randn(200, 80, device=dev).to(torch.float8_e4m3fn), torch.randn(4, 48, 80, device=dev).to(torch.float8_e4m3fn)
    sa, sb = torch.rand(200, 1, device=dev), torch.rand(4, 48, device=dev)
    for out_type in (torch.float16, torch.bfloat16):
        got = gmm_fp8_act_per_channel_w_per_expert(a8, sa, b8, sb, sizes, out_type)
        assert got.dtype == out_type
        assert torch.equal(got, gmm_fp8_act_per_channel_w_per_expert(a8, sa.double(), b8, sb, sizes, out_type))
    idx = torch.randint(0, 4, (200, 2), device=dev, dtype=torch.int32)
    x = a.clone().requires_grad_(True)
    rows, where = ops.permute(x, idx, num_experts=4)
    with torch.no_grad():
        direct = ops.permute(x, idx, num_experts=4)
    assert rows.requires_grad and not direct[0].requires_grad
    assert torch.equal(rows, direct[0]) and torch.equal(where, direct[1])
    probs = torch.rand(200, 2, device=dev)
    assert torch.equal(ops.unpermute(direct[0], where, probs), ops.unpermute(rows, where, probs))
    assert torch.equal(ops.permute_map(idx, num_experts=4)[0], ops.permute_map(idx.long(), num_experts=4)[0])


@pytest.mark.gpu
@pytest.mark.parametrize("k", [128, 640, 8192])  # 1, 5 and 64 scale blocks per row
@pytest.mark.parametrize("sizes", [[64], [1, 0, 200, 128], [130] * 5])
def test_contiguous_entry_points_check_the_total_and_take_both_scale_layouts(dev, k, sizes):
    """Row-major activation scales (turned by a kernel) give the bits of K-block-major ones; sizes that do not add up to A's
    rows raise the reference's ValueError, before anything is written where the caller brings the output."""
    from triton_grouped_gemm_amd.gemm.deep_gemm_ops import m_grouped_bf16_nt_contiguous, m_grouped_fp8_nt_contiguous
    from triton_grouped_gemm_amd.quant.fp8_cast import per_block_cast_to_fp8, per_token_cast_to_fp8
    s = torch.tensor(sizes, dtype=torch.int32, device=dev)
    m, g, n = sum((v + 127) // 128 * 128 for v in sizes), len(sizes), 136
    x = torch.randn(m, k, device=dev).to(torch.bfloat16)
    w = torch.randn(g, n, k, device=dev).to(torch.bfloat16)
    rows = torch.cat([torch.arange(v, device=dev) + i for v, i in
                      zip(sizes, torch.tensor([0, *[(v + 127) // 128 * 128 for v in sizes]]).cumsum(0).tolist())])
    wq = per_block_cast_to_fp8(w)
    outs = [m_grouped_fp8_nt_contiguous(per_token_cast_to_fp8(x, scales_mn_major=mn), wq, sz)
            for mn in (True, False) for sz in (s, s.long())]
    assert all(torch.equal(o[rows], outs[0][rows]) for o in outs)
    xq = per_token_cast_to_fp8(x)
    kept = torch.zeros(m, n, dtype=torch.bfloat16, device=dev)
    assert m_grouped_fp8_nt_contiguous(xq, wq, s, out=kept) is kept and torch.equal(kept[rows], outs[0][rows])
    plain = m_grouped_bf16_nt_contiguous(x, w, s)
    assert torch.equal(m_grouped_bf16_nt_contiguous(x, w, s, out=kept)[rows], plain[rows])
    bad = s.clone()
    bad[0] += 128
    kept.fill_(7.0)
    for call in (lambda **kw: m_grouped_fp8_nt_contiguous(xq, wq, bad, **kw), lambda **kw: m_grouped_bf16_nt_contiguous(x, w, bad, **kw)):
        with pytest.raises(ValueError, match=f"expected M={m + 128}, got M={m}"):
            call()
        with pytest.raises(ValueError, match="padded expert rows"):
            call(out=kept)
    assert bool((kept == 7.0).all())


@pytest.mark.gpu
def test_one_block_of_activation_scales_with_any_stride(dev):
    """K = 128: a column of a wider scale tensor and one scale expanded over the rows give what contiguous copies give, on
    the native path (sizes on the GPU) and through the wrapper (sizes on the host)."""
    from triton_grouped_gemm_amd.gemm.deep_gemm_ops import m_grouped_fp8_nt_contiguous
    from triton_grouped_gemm_amd.quant.fp8_cast import per_block_cast_to_fp8
    g = torch.Generator().manual_seed(11)
    s = torch.tensor([128, 100, 0], dtype=torch.int32, device=dev)
    codes = torch.randn(256, 128, generator=g).to(dev).to(torch.float8_e4m3fn)
    wq = per_block_cast_to_fp8(torch.randn(3, 72, 128, generator=g).to(torch.bfloat16).to(dev))
    wide = torch.rand(256, 5, generator=g).to(dev) + 0.5
    for scale in (wide[:, 3:4], wide[7:8, :1].expand(256, 1), wide[:, 2:3].contiguous()):
        want = m_grouped_fp8_nt_contiguous((codes, scale.clone(memory_format=torch.contiguous_format)), wq, s)
        for sizes in (s, s.cpu()):
            got = m_grouped_fp8_nt_contiguous((codes, scale), wq, sizes)
            assert torch.equal(got[:228], want[:228])
    exact = codes.float()[:128] @ (wq[0][0].float() * wq[1][0, 0, 0]).t() * wide[:128, 2:3]
    assert float((want[:128].float() - exact).abs().max() / exact.abs().max()) < 2.0 ** -7


@pytest.mark.gpu
@pytest.mark.parametrize("which", range(4))
def test_fp8_gemm_refuses_the_gradient_of_every_operand(dev, which):
    """The operator has no derivative: backward through it says so, whichever operand asks for a gradient, and a call
    that records nothing is answered as before."""
    sizes = torch.tensor([5, 0, 11], dtype=torch.int32, device=dev)
    operands = [torch.randn(16, 32, device=dev).to(torch.float8_e4m3fn), torch.rand(16, 1, device=dev),
                torch.randn(3, 24, 32, device=dev).to(torch.float8_e4m3fn), torch.rand(3, 24, device=dev)]
    want = gmm_fp8_act_per_channel_w_per_expert(*operands, sizes)
    operands[which] = torch.nn.Parameter(operands[which])
    out = gmm_fp8_act_per_channel_w_per_expert(*operands, sizes)
    assert out.requires_grad and torch.equal(out, want)
    with pytest.raises(RuntimeError, match="autograd"):
        out.sum().backward()
    with torch.no_grad():
        out = gmm_fp8_act_per_channel_w_per_expert(*operands, sizes)
    assert not out.requires_grad and torch.equal(out, want)


@pytest.mark.gpu
@pytest.mark.parametrize("entry", ["gemm", "masked", "k_grouped", "fp8", "permute_map", "permute", "unpermute", "bf16_padded", "fp8_padded"])
def test_other_threads_run_while_a_call_allocates_and_launches(dev, entry):
    """A thread that waits for the interpreter lock gets it during the calls, without asking the interpreter to switch
    (the switch interval is set beyond the test's length)."""
    a, b, sizes = _operands(dev)
    a8, b8 = torch.randn(200, 80, device=dev).to(torch.float8_e4m3fn), torch.randn(4, 48, 80, device=dev).to(torch.float8_e4m3fn)
    sa, sb = torch.rand(200, 1, device=dev), torch.rand(4, 48, device=dev)
    lhs, out = torch.randn(512, 72, device=dev).to(torch.bfloat16), torch.empty(512, 40, device=dev, dtype=torch.bfloat16)
    idx = torch.randint(0, 4, (200, 2), device=dev, dtype=torch.int32)
    rows, where = ops.permute(a, idx, num_experts=4)
    probs, queue = torch.rand(200, 2, device=dev), _native.work_queue(a.device)
    x16, x8 = (torch.randn(384, 80, device=dev).to(t) for t in (torch.bfloat16, torch.float8_e4m3fn))
    w16, row_scale, block_scale = b8.to(torch.bfloat16), torch.rand(384, 1, device=dev), torch.rand(4, 1, 1, device=dev)
    host = _native.host()
    call = {"gemm": lambda: host.m_grouped_gemm(a, b, sizes, True, -1),
            "masked": lambda: host.m_grouped_gemm_masked(lhs, b, out, sizes, 128, True),
            "k_grouped": lambda: host.k_grouped_gemm(a, a, sizes, -1, queue),
            "fp8": lambda: host.m_grouped_gemm_fp8_channel(a8, sa, b8, sb, sizes, True),
            "permute_map": lambda: host.permute_map(idx, 0, 4, False), "permute": lambda: host.permute(a, idx, 0, 4),
            "unpermute": lambda: host.unpermute(rows, where, probs),
            "bf16_padded": lambda: host.m_grouped_bf16_contiguous(x16, w16, sizes, None, 128),
            "fp8_padded": lambda: host.m_grouped_fp8_contiguous(x8, row_scale, b8, block_scale, sizes, None, 128)}[entry]
    assert call() is not None
    gate, seen = threading.Lock(), []
    gate.acquire()
    waiting = threading.Thread(target=lambda: (gate.acquire(), seen.append(1)), daemon=True)
    interval = sys.getswitchinterval()
    try:
        waiting.start()
        sys.setswitchinterval(1000.0)
        gate.release()
        for _ in range(500):
            call()
            if seen:
                break
        assert seen
    finally:
        sys.setswitchinterval(interval)
        waiting.join()
    torch.cuda.synchronize()


@pytest.mark.gpu
@pytest.mark.parametrize("key", ["CUDA", "AutocastCUDA", "AutogradCUDA"])
def test_what_others_register_for_the_operators_is_what_runs(dev, key):
    a, b, sizes = _operands(dev)
    a8, b8 = torch.randn(200, 80, device=dev).to(torch.float8_e4m3fn), torch.randn(4, 48, 80, device=dev).to(torch.float8_e4m3fn)
    eight = (a8, torch.rand(200, 1, device=dev), b8, torch.rand(4, 48, device=dev), sizes)
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=key == "AutocastCUDA"):
        plain = m_grouped_gemm(a, b, sizes, True), gmm_fp8_act_per_channel_w_per_expert(*eight)
        with torch.library._scoped_library("moe", "IMPL") as moe, torch.library._scoped_library("myfp8", "IMPL") as myfp8:
            moe.impl("m_grouped_gemm", lambda x, *rest: x.new_full((2,), 7.0), key)
            myfp8.impl("gmm_fp8_act_per_channel_w_per_expert", lambda x, scale, *rest: scale.new_full((3,), 9.0), key)
            assert m_grouped_gemm(a, b, sizes, True).tolist() == [7.0] * 2 and ops.gmm(a, b, sizes, True).tolist() == [7.0] * 2
            assert gmm_fp8_act_per_channel_w_per_expert(*eight).tolist() == [9.0] * 3
        again = m_grouped_gemm(a, b, sizes, True), gmm_fp8_act_per_channel_w_per_expert(*eight)
        assert torch.equal(plain[0], again[0]) and torch.equal(plain[1], again[1])


@pytest.mark.gpu
def test_the_profiler_shows_the_operators(dev):
    a, b, sizes = _operands(dev)
    a8, b8 = torch.randn(200, 80, device=dev).to(torch.float8_e4m3fn), torch.randn(4, 48, 80, device=dev).to(torch.float8_e4m3fn)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU], record_shapes=True) as seen:
        ops.gmm(a, b, sizes, True)
        gmm_fp8_act_per_channel_w_per_expert(a8, torch.rand(200, 1, device=dev), b8, torch.rand(4, 48, device=dev), sizes)
    shapes = {e.name: e.input_shapes for e in seen.events()}
    assert shapes["moe::m_grouped_gemm"][:2] == [[200, 72], [4, 40, 72]]
    assert shapes["myfp8::gmm_fp8_act_per_channel_w_per_expert"][:2] == [[200, 80], [200, 1]]
