"""MoE permute / unpermute against the torch reference of the reference's own test
(grouped_gemm/grouped_gemm/permute_test.py): same generator of inputs (randperm expert choice per token,
normalised random probs), forward and backward of both ops.  Integer results (row_id_map, counts, moved rows) are
bit-exact; the weighted sums are compared in fp32 with half-ulp style bounds."""
import pytest
import torch

from oracle import permute_ref
from triton_grouped_gemm_amd import ops

pytestmark = pytest.mark.gpu


def _case(num_token, num_expert, hidden, topk, dtype, seed=0):
    g = torch.Generator().manual_seed(seed)
    x = torch.rand((num_token, hidden), generator=g).to(dtype)
    if num_token:
        indices = torch.stack([torch.randperm(num_expert, generator=g)[:topk] for _ in range(num_token)]).to(torch.int32)
    else:
        indices = torch.empty((0, topk), dtype=torch.int32)
    probs = torch.rand(num_token, topk, generator=g)
    probs = probs / probs.sum(dim=1, keepdim=True)
    return x, indices, probs


def _close(out, ref32, dtype, terms=1):
    eps = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -23}[dtype]
    err = (out.float().cpu() - ref32).abs()
    bound = ref32.abs() * eps * 1.02 + terms * 2.0 ** -22 * ref32.abs().max().clamp_min(1e-30)
    assert bool((err <= bound).all()), float((err - bound).max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("num_token,num_expert,hidden,topk", [
    (4096, 8, 512, 2), (1000, 64, 264, 6), (777, 256, 4096, 8), (5, 3, 8, 1), (2048, 1024, 128, 4)])
def test_forward_backward(dev, dtype, num_token, num_expert, hidden, topk):
    x, indices, probs = _case(num_token, num_expert, hidden, topk, dtype)
    # ---- reference (CPU torch; activations in fp32 for the gradient checks)
    ref_perm, order = permute_ref.permute(x, indices)
    ref_map = permute_ref.row_id_map(indices)
    # ---- permute forward
    xd = x.to(dev).requires_grad_(True)
    perm, rmap = ops.permute(xd, indices.to(dev), num_experts=num_expert)
    assert torch.equal(rmap.cpu(), ref_map)
    assert torch.equal(perm.detach().cpu(), ref_perm)  # rows are moved, not recomputed: bit-exact
    # ---- permute backward: grad of x[t] = sum over its topk copies
    gperm = torch.rand(perm.shape, generator=torch.Generator().manual_seed(1)).to(dtype)
    perm.backward(gperm.to(dev))
    ref_gx = torch.zeros(num_token, hidden).index_add_(0, order // topk, gperm.float())
    _close(xd.grad, ref_gx, dtype, topk)
    # ---- unpermute forward with probs
    pd = probs.to(dev).requires_grad_(True)
    ud_in = perm.detach().clone().requires_grad_(True)
    un = ops.unpermute(ud_in, rmap, pd)
    p32 = probs.clone().requires_grad_(True)
    u32_in = ref_perm.float().clone().requires_grad_(True)
    ref_un = permute_ref.unpermute(u32_in, order, p32, fp32=True)
    _close(un.detach(), ref_un.detach(), dtype, topk)
    # ---- unpermute backward: activation and prob gradients
    gun = torch.rand(un.shape, generator=torch.Generator().manual_seed(2)).to(dtype)
    un.backward(gun.to(dev))
    ref_un.backward(gun.float())
    _close(ud_in.grad, u32_in.grad, dtype)
    pg, rpg = pd.grad.cpu(), p32.grad
    assert torch.allclose(pg, rpg, rtol=1e-5, atol=1e-6 * float(rpg.abs().max())), float((pg - rpg).abs().max())


def test_counts_are_the_group_sizes(dev):
    _, indices, _ = _case(3000, 40, 8, 4, torch.bfloat16, seed=3)
    for cd in (torch.int32, torch.int64):
        rmap, counts = ops.permute_map(indices.to(dev), num_experts=40, counts_dtype=cd)
        assert counts.dtype == cd
        assert torch.equal(counts.cpu().long(), permute_ref.tokens_per_expert(indices, 40))
        assert sorted(rmap.cpu().tolist()) == list(range(3000 * 4))  # a permutation of all rows


def test_dropped_assignments_and_capacity(dev):
    x, indices, _ = _case(500, 16, 64, 2, torch.bfloat16, seed=4)
    indices[::7, 1] = -1  # dropped assignments
    ref_map = permute_ref.row_id_map(indices)
    rmap, counts = ops.permute_map(indices.to(dev), num_experts=16)
    assert torch.equal(rmap.cpu(), ref_map)
    assert torch.equal(counts.cpu().long(), permute_ref.tokens_per_expert(indices, 16))
    kept = int((indices >= 0).sum())
    perm, rmap2 = ops.permute(x.to(dev), indices.to(dev), num_experts=16)
    order = torch.argsort(indices.reshape(-1), stable=True)[indices.numel() - kept:]
    assert torch.equal(perm[:kept].cpu(), x.index_select(0, order // 2))
    # capacity: only the first 300 permuted rows are kept
    ref_cap = permute_ref.row_id_map(indices, 300)
    perm_c, rmap_c = ops.permute(x.to(dev), indices.to(dev), num_out_tokens=300, num_experts=16)
    assert perm_c.shape == (300, 64) and torch.equal(rmap_c.cpu(), ref_cap)
    assert torch.equal(perm_c.cpu(), x.index_select(0, order[:300] // 2))
    # unpermute skips dropped assignments
    un = ops.unpermute(perm_c, rmap_c, torch.ones(500, 2, device=dev))
    exp = torch.zeros(500, 64)
    for k in range(2):
        rows = ref_cap[k * 500:(k + 1) * 500]
        ok = rows >= 0
        exp[ok] += perm_c.cpu().float()[rows[ok].long()]
    _close(un, exp, torch.bfloat16, 2)


def test_empty_input_passes_through(dev):
    x = torch.empty((0, 64), dtype=torch.bfloat16, device=dev)
    out, rmap = ops.permute(x, torch.empty((0, 2), dtype=torch.int32, device=dev))
    assert out.numel() == 0 and rmap is None


@pytest.mark.parametrize("topk", [1, 8, 1024, 1100])
def test_empty_assignment_counts_are_zero(dev, topk):
    rmap, counts = ops.permute_map(torch.empty((0, topk), dtype=torch.int32, device=dev), num_experts=40)
    assert rmap.numel() == 0 and torch.equal(counts.cpu(), torch.zeros(40, dtype=torch.int32))


@pytest.mark.parametrize("num_token,hidden,topk", [
    (51200, 1024, 1), (51201, 1024, 1), (52000, 1016, 1), (51200, 1024, 2), (51201, 1024, 2)])
def test_rows_on_either_side_of_a_launch_of_their_own(dev, num_token, hidden, topk):
    """Sizes at which the placing launch stops to move the rows as well: by the number of choices and the rows' width."""
    g = torch.Generator(device=dev).manual_seed(num_token + hidden)
    x = torch.randint(-30000, 30000, (num_token, hidden), device=dev, dtype=torch.int16, generator=g).view(torch.bfloat16)
    idx = torch.randint(0, 16, (num_token, topk), device=dev, dtype=torch.int32, generator=g)
    idx[::13, 0] = -1
    rows, rmap = ops.permute(x, idx, num_experts=16)
    assert torch.equal(rmap, ops.permute_map(idx, num_experts=16)[0])
    flat = torch.argsort(torch.where(idx < 0, 99, idx).reshape(-1), stable=True)[:int((idx >= 0).sum())]
    assert torch.equal(rows[:flat.numel()].view(torch.int16), x.view(torch.int16)[flat // topk])
    assert torch.equal(rmap.view(topk, num_token)[flat % topk, flat // topk], torch.arange(flat.numel(), device=dev, dtype=torch.int32))


def test_unpermute_without_probs_asks_for_an_entry_per_row(dev):
    """More rows than map entries (a capacity above the token count) are refused, not read beyond the map."""
    x, indices, _ = _case(100, 8, 64, 1, torch.bfloat16)
    rows, rmap = ops.permute(x.to(dev), indices.to(dev), num_out_tokens=160, num_experts=8)
    assert rows.shape == (160, 64) and rmap.numel() == 100
    for r in (rows, rows.clone().requires_grad_(True)):
        with pytest.raises(RuntimeError, match="`row_id_map` shape mismatch! Expect 160, but got 100"):
            ops.unpermute(r, rmap)
    assert torch.equal(ops.unpermute(rows[:100].contiguous(), rmap).cpu(), x)


@pytest.mark.parametrize("num_token,hidden,topk", [
    (102400, 512, 3), (102401, 512, 3), (110000, 504, 3),  # the row width and the size from which rows are taken singly
    (50001, 1544, 4), (16001, 2640, 5), (70001, 2048, 2)])  # 4 waves a token, the last one ragged; 6; pairs
def test_unpermute_of_many_rows_equals_its_parts(dev, num_token, hidden, topk):
    """The sum of a token's rows has the same bits however many of them are in flight: a large call against calls on
    runs of its tokens, and those against fp32 torch."""
    g = torch.Generator(device=dev).manual_seed(num_token)
    rows = torch.randn(num_token * topk, hidden, device=dev, dtype=torch.bfloat16, generator=g)
    rmap = torch.randperm(num_token * topk, device=dev, generator=g).int()
    rmap[::11] = -1
    probs = torch.rand(num_token, topk, device=dev, generator=g)
    for p in (probs, torch.ones_like(probs)):
        whole = ops.unpermute(rows, rmap, p)
        for t0 in range(0, num_token, num_token // 5):
            part = slice(t0, min(num_token, t0 + num_token // 5))
            src = rmap.view(topk, num_token)[:, part].contiguous()
            assert torch.equal(whole[part], ops.unpermute(rows, src.reshape(-1), p[part].contiguous()))
        picked = torch.where((src >= 0)[..., None], rows[src.clamp_min(0).long()].float(), 0.0)
        _close(whole[part], (picked * p[part].t()[..., None]).sum(0).cpu(), torch.bfloat16, topk + 1)


@pytest.mark.parametrize("num_token,hidden", [(2 ** 24 + 5, 8), (2 ** 23 + 3, 1032)])
def test_unpermute_beyond_the_waves_of_one_launch(dev, num_token, hidden):
    """More pieces (64 chunks of a token) than the launch has waves: one a token, and three."""
    rows = torch.empty(num_token, hidden, device=dev, dtype=torch.bfloat16)
    rows.view(torch.int16).copy_((torch.arange(num_token * hidden, device=dev) % 16001).view(num_token, hidden))
    rmap = torch.arange(num_token - 1, -1, -1, device=dev, dtype=torch.int32)
    assert torch.equal(ops.unpermute(rows, rmap), rows.flip(0))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("num_token,chunks,topk", [
    (16384, 256, 3), (16385, 256, 3), (16385, 256, 8), (20001, 256, 1), (18000, 240, 2), (18000, 241, 2), (17001, 257, 5)])
def test_unpermute_backward_of_many_rows_equals_its_parts(dev, dtype, num_token, chunks, topk):
    """The gradients have the same bits on either side of the sizes that take rows singly: a large call against calls on
    runs of its tokens, and those against fp32 torch."""
    g = torch.Generator(device=dev).manual_seed(num_token + chunks)
    hidden = chunks * 16 // torch.empty(0, dtype=dtype).element_size()
    rows = torch.randn(num_token * topk, hidden, device=dev, generator=g).to(dtype).requires_grad_(True)
    grad = torch.randn(num_token, hidden, device=dev, generator=g).to(dtype)
    rmap = torch.randperm(num_token * topk, device=dev, generator=g).int()
    rmap[::7] = -1
    probs = torch.rand(num_token, topk, device=dev, generator=g).requires_grad_(True)
    whole = torch.autograd.grad(ops.unpermute(rows, rmap, probs), (rows, probs), grad)
    for t0 in range(0, num_token, num_token // 4):
        part = slice(t0, min(num_token, t0 + num_token // 4))
        src = rmap.view(topk, num_token)[:, part].contiguous()
        p = probs.detach()[part].contiguous().requires_grad_(True)
        got = torch.autograd.grad(ops.unpermute(rows, src.reshape(-1), p), (rows, p), grad[part])
        kept = src[src >= 0].long()
        assert torch.equal(got[0][kept], whole[0][kept]) and torch.equal(got[1], whole[1][part])
    scaled = (p.detach().t()[..., None] * grad[part].float())[src >= 0]
    _close(got[0][kept], scaled.cpu(), dtype)
    dots = torch.where(src >= 0, (rows.detach()[src.clamp_min(0).long()].double() * grad[part].double()).sum(-1), 0.0).t()
    # a sum of `hidden` products of normal numbers in fp32: the error grows like the square root of their number
    assert float((got[1].double() - dots).abs().max()) < 8 * 2.0 ** -24 * hidden


def test_feeds_the_grouped_gemm(dev):
    """permute -> grouped GEMM with the counts as size_per_group -> unpermute equals the dense per-token formula."""
    T, E, H, N, topk = 512, 8, 128, 64, 2
    x, indices, probs = _case(T, E, H, topk, torch.bfloat16, seed=5)
    w = (torch.randn(E, H, N, generator=torch.Generator().manual_seed(6)) * H ** -0.5).to(torch.bfloat16)
    perm, rmap = ops.permute(x.to(dev), indices.to(dev), num_experts=E)
    _, counts = ops.permute_map(indices.to(dev), num_experts=E)
    y = ops.gmm(perm, w.to(dev), counts, trans_b=False)
    out = ops.unpermute(y, rmap, probs.to(dev))
    ref = torch.zeros(T, N)
    for t in range(T):
        for k in range(topk):
            yk = (x[t].float() @ w[int(indices[t, k])].float()).to(torch.bfloat16).float()  # the GEMM's bf16 output
            ref[t] += probs[t, k] * yk
    err = (out.float().cpu() - ref).abs().max() / ref.abs().max()
    assert err <= 2.0 ** -7, float(err)


@pytest.mark.parametrize("num_token,num_expert,topk,hidden", [
    (1024, 128, 8, 40), (1025, 128, 8, 40),        # the last one-launch size and the first one behind it
    (3001, 1024, 7, 8), (9001, 5, 3, 24),          # table columns shared by no / many threads, ragged last chunk
    (33000, 1000, 8, 8), (70001, 1, 2, 8),         # a table that needs the scan launch; a single expert
    (8533, 64, 8, 2048), (8534, 64, 8, 2048),      # the last rows moved by the placing launch and the first by their own
    (8, 1024, 1100, 16), (20, 600, 500, 2056)])    # more assignments per token than one batch holds; several batches
def test_sort_paths(dev, num_token, num_expert, topk, hidden):
    """Every path of the sort at its edges: map, counts and moved rows are bit-exact, with ids drawn with repetition,
    dropped assignments and a capacity that cuts the last experts off."""
    g = torch.Generator().manual_seed(num_token)
    indices = torch.randint(-1, num_expert, (num_token, topk), generator=g, dtype=torch.int32)
    x = torch.randn(num_token, hidden, generator=g).to(torch.bfloat16)
    kept = int((indices >= 0).sum())
    for cap in (0, kept - kept // 5):
        ref_map = permute_ref.row_id_map(indices, cap)
        rmap, counts = ops.permute_map(indices.to(dev), cap, num_experts=num_expert)
        assert torch.equal(rmap.cpu(), ref_map)
        assert torch.equal(counts.cpu().long(), permute_ref.tokens_per_expert(indices, num_expert))
        perm, rmap2 = ops.permute(x.to(dev), indices.to(dev), num_out_tokens=cap, num_experts=num_expert)
        assert torch.equal(rmap2.cpu(), ref_map)
        rows = cap if cap else kept
        token_of = torch.empty(rows, dtype=torch.int64)
        live = ref_map >= 0
        token_of[ref_map[live].long()] = torch.arange(topk * num_token)[live] % num_token
        assert torch.equal(perm[:rows].cpu(), x[token_of])
