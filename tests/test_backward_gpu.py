"""Backward passes of the router, SwiGLU, MLP and expert ops and of the whole block, against autograd of the oracle
(float64 on the CPU) evaluated on the same inputs and, where a selection is involved, on the HIP path's own indices."""
import pytest
import torch

from helpers import rel_fro
from oracle import flashmoe_oracle as orc

pytestmark = pytest.mark.gpu

GRAD_FRO = {torch.float32: 2e-5, torch.bfloat16: 1.5e-2, torch.float16: 3e-3}


def gen(seed):
    return torch.Generator().manual_seed(seed)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,nk,K", [(64, 32, 16), (300, 128, 64), (17, 512, 128), (5, 8, 1),
                                    (6, 9000, 48),     # more keys than one LDS row pair holds: rows built 4096 keys at a time
                                    (8193, 24, 11), (16390, 64, 16), (12301, 25, 5)])   # two, four and three tokens to a wave
def test_router_backward(dtype, T, nk, K):
    from flash_moe.ops import flash_router_func
    from flash_moe.ops.hip.flash_router import router_topk_backward

    lp = orc.make_router_inputs(T, nk, seed=1).to(dtype)
    lp_dev = lp.cuda().requires_grad_(True)
    scores, indices = flash_router_func(lp_dev, nk, K)
    ds = torch.randn(T, K, generator=gen(2)).to(dtype)
    scores.backward(ds.cuda())
    idx = indices.cpu()
    # scatter-add restated with index_add_ in float64
    ref = torch.zeros(2, T, nk, dtype=torch.float64)
    rows = torch.arange(T).repeat_interleave(K)
    ref[0].index_put_((rows, (idx // nk).flatten()), ds.double().flatten(), accumulate=True)
    ref[1].index_put_((rows, (idx % nk).flatten()), ds.double().flatten(), accumulate=True)
    got = lp_dev.grad
    assert got.shape == (2, T, nk) and got.dtype == dtype
    tol = {torch.float32: 1e-6, torch.bfloat16: 8e-3, torch.float16: 1e-3}[dtype]
    torch.testing.assert_close(got.double().cpu(), ref, rtol=tol, atol=tol * max(1.0, float(ref.abs().max())))
    # the op-level function gives the same tensor, twice
    again = router_topk_backward(ds.cuda(), indices, nk)
    assert torch.equal(again, got) and torch.equal(router_topk_backward(ds.cuda(), indices, nk), got)
    # the gradient of an unselected key is exactly zero and the total is conserved per token and half
    torch.testing.assert_close(got.double().sum(-1).cpu(), ref.sum(-1), rtol=5 * tol, atol=5 * tol * max(1.0, float(ref.abs().max())))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("T,nk,K", [(64, 32, 16), (130, 128, 64), (9, 512, 128), (5, 8, 1),
                                    (7, 129, 64), (7, 128, 65), (7, 256, 128), (6, 257, 128), (6, 256, 129), (3, 1, 1),   # what registers hold
                                    (5, 8192, 64), (6, 20000, 96)])   # the last: rows built 4096 keys at a time
def test_route_backward(dtype, norm, T, nk, K):
    """Gate gradients -> gradient of the fp32 gate logits, against float64 autograd of log-softmax, pair sums, exp and
    renormalisation on the same ids; ids out of range carry nothing; the gradient of the returned logits is added."""
    from flash_moe.ops.hip.flash_router import route_backward

    logits = torch.randn(T, 2 * nk, generator=gen(1)) * 2.0
    if nk <= 512:
        idx = torch.stack([torch.randperm(nk * nk, generator=gen(10 + t))[:K] for t in range(T)])
    else:   # pairs that share keys (several gradients per key) and lie on both sides of every 4096-key boundary
        idx = torch.randint(0, nk, (T, K), generator=gen(10)) * nk + torch.randint(0, nk, (T, K), generator=gen(11))
        idx[:, : K // 2] = idx[:, K // 2 : 2 * (K // 2)] // nk * nk + (idx[:, : K // 2] % nk)
    if K > 2:
        idx[::3, 1] = nk * nk + 7
        idx[1::4, 2] = -1
    dg = torch.randn(T, K, generator=gen(2)).to(dtype)
    extra = (torch.randn(T, 2 * nk, generator=gen(3)) * 0.1).to(dtype)
    valid = (idx >= 0) & (idx < nk * nk)
    safe = idx.clamp(0, nk * nk - 1)
    lg = logits.double().requires_grad_(True)
    lp = torch.log_softmax(lg.view(T, 2, nk), -1)
    e = (lp[:, 0].gather(1, safe // nk) + lp[:, 1].gather(1, safe % nk)).exp() * valid
    gates = e / e.sum(-1, keepdim=True) if norm else e
    ((gates * dg.double()).sum() + (lg * extra.double()).sum()).backward()
    got = route_backward(dg.cuda(), idx.cuda(), logits.cuda(), nk, norm, extra.cuda())
    assert got.dtype == torch.float32 and got.shape == (T, 2 * nk)
    assert rel_fro(got, lg.grad) < 2e-5, rel_fro(got, lg.grad)
    without = route_backward(dg.cuda(), idx.cuda(), logits.cuda(), nk, norm)
    torch.testing.assert_close(without.cpu().double() + extra.double(), lg.grad, rtol=1e-4, atol=1e-5)
    assert torch.equal(route_backward(dg.cuda(), idx.cuda(), logits.cuda(), nk, norm, extra.cuda()), got)


@pytest.mark.parametrize("dtype,norm", [(torch.float32, False), (torch.float32, True), (torch.bfloat16, True)])
def test_block_autograd_node_equals_the_composition_of_ops(dtype, norm):
    """forward_autograd (one node, library calls only) and forward_autograd_ops (the reference's composition on the
    differentiable per-op functions) give the same outputs and gradients."""
    from test_block_gpu import build

    m, _ = build(128, 256, 1024, 8, norm, dtype, seed=4, std=0.05)
    x = torch.randn(2, 96, 128, generator=gen(5)).to(dtype).cuda()
    wy = torch.randn(2, 96, 128, generator=gen(6)).cuda()
    wl = (torch.randn(2, 192, 32, generator=gen(7)) * 0.1).cuda()
    results = []
    for fwd in (m.forward_autograd, m.forward_autograd_ops):
        m.router_norm.reset_running_stats()
        for p in m.parameters():
            p.grad = None
        xg = x.clone().requires_grad_(True)
        y, logits = fwd(xg)
        ((y.float() * wy).sum() + (logits.float() * wl).sum()).backward()
        results.append((y.detach(), logits.detach(), xg.grad, {k: v.grad.clone() for k, v in m.named_parameters()}))
    (y0, l0, gx0, gp0), (y1, l1, gx1, gp1) = results
    tol = 2e-5 if dtype == torch.float32 else 1.5e-2
    # same kernels for the logits; the gates come from the fused router here and from torch's exp there
    assert torch.equal(l0, l1) and rel_fro(y0, y1) < tol
    assert rel_fro(gx0, gx1) < tol, rel_fro(gx0, gx1)
    for k in gp0:
        assert rel_fro(gp0[k], gp1[k]) < tol, (k, rel_fro(gp0[k], gp1[k]))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("what", ["router", "prologue", "expert", "mlp", "block"])
def test_autograd_functions_by_class_equal_the_native_nodes(what, dtype):
    """The classes under the reference's names give the outputs and gradients of the ops, whose nodes are native."""
    from flash_moe.modules.flash_moe import FlashMoE, FlashMoEConfig
    from flash_moe.ops import flash_expert_func, flash_mlp_func, flash_router_func
    from flash_moe.ops.hip import flash_block as fb, flash_expert as fe, flash_mlp as fm, flash_router as fr

    T, H, I, E, K = 96, 128, 264, 1024, 8
    g = gen(3)
    m = FlashMoE(FlashMoEConfig(H, I, "silu", E, K, True)).to(device="cuda", dtype=dtype)
    wg, wu, wd, wr, ed, eu = (p.detach() for p in (m.gate_proj.weight, m.up_proj.weight, m.down_proj.weight, m.router_gate.weight,
                                                   m.down_embed.weight, m.up_embed.weight))
    x = torch.randn(T, H, generator=g).to(dtype).cuda()
    idx = torch.randint(0, E, (T, K), generator=g).cuda()
    gates = torch.rand(T, K, generator=g).to(dtype).cuda()
    logs = torch.log_softmax(torch.randn(2, T, 32, generator=g), -1).to(dtype).cuda()

    def native_block(*leaves):
        out, logits = fb.block(*leaves[:5], m.router_norm, *leaves[5:], 32, K, True, differentiable=True)
        return out, logits.transpose(0, 1).reshape(T, 64)

    leaves, by_class, native = {
        "router": ([logs], lambda t: fr.FlashRouterFunc.apply(t, 32, K), lambda t: flash_router_func(t, 32, K)),
        "prologue": ([x, wr], lambda *t: fr.RouterPrologueFunc.apply(*t, m.router_norm), lambda *t: fr.router_prologue(*t, m.router_norm)),
        "expert": ([x, ed, eu, gates], lambda a, d, u, w: fe.FlashExpertFunc.apply(a, d, u, idx, w),
                   lambda a, d, u, w: flash_expert_func(a, d, u, idx, w)),
        "mlp": ([x, wg, wu, wd], fm.FlashMLPFunc.apply, flash_mlp_func),
        "block": ([x, wg, wu, wd, wr, ed, eu],
                  lambda *t: fb.block_forward_autograd(*t[:5], m.router_norm, *t[5:], 32, K, True), native_block),
    }[what]
    results = []
    for fn in (by_class, native):
        ts = [t.clone().requires_grad_() for t in leaves]
        out = fn(*ts)
        out = [o for o in (out if isinstance(out, tuple) else (out,)) if o.requires_grad]
        torch.autograd.backward(out, [torch.randn(o.shape, generator=gen(5)).to(o.dtype).cuda() for o in out])
        results.append([o.detach() for o in out] + [t.grad for t in ts])
    # two library paths in the same types: sums in another order, the block's token gradients rounded once or three times
    for a, b in zip(*results):
        assert a.dtype == b.dtype and rel_fro(a, b.cpu()) < (1e-5 if dtype == torch.float32 else 1e-2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(7, 64), (3, 5, 256), (128, 1024)])
def test_swiglu_backward(dtype, shape):
    from flash_moe.ops.hip.flash_mlp import swiglu_backward

    a, b, dc = (torch.randn(shape, generator=gen(s)).to(dtype) for s in (1, 2, 3))
    a64, b64 = a.double().requires_grad_(True), b.double().requires_grad_(True)
    (torch.nn.functional.silu(a64) * b64).backward(dc.double())
    da, db = swiglu_backward(a.cuda(), b.cuda(), dc.cuda())
    assert da.shape == a.shape and db.dtype == dtype
    tol = {torch.float32: 2e-6, torch.bfloat16: 8e-3, torch.float16: 1e-3}[dtype]
    torch.testing.assert_close(da.double().cpu(), a64.grad, rtol=tol, atol=tol)
    torch.testing.assert_close(db.double().cpu(), b64.grad, rtol=tol, atol=tol)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,I", [(128, 256, 512), (96, 64, 192), (512, 1024, 1024)])
def test_mlp_backward(dtype, T, H, I):
    from flash_moe.ops import flash_mlp_func

    x = torch.randn(T, H, generator=gen(1)).to(dtype)
    wg, wu, wd = ((torch.randn(s, generator=gen(k)) * 0.05).to(dtype) for k, s in ((2, (I, H)), (3, (I, H)), (4, (H, I))))
    dy = torch.randn(T, H, generator=gen(5)).to(dtype)
    leaves = [t.cuda().requires_grad_(True) for t in (x, wg, wu, wd)]
    flash_mlp_func(*leaves).backward(dy.cuda())
    ref_leaves = [t.double().requires_grad_(True) for t in (x, wg, wu, wd)]
    orc.mlp_forward(*ref_leaves).backward(dy.double())
    for name, got, ref in zip(("dx", "dgate", "dup", "ddown"), leaves, ref_leaves):
        assert got.grad.dtype == dtype and got.grad.shape == ref.shape
        fro = rel_fro(got.grad, ref.grad)
        assert fro < GRAD_FRO[dtype], f"{name}: relative Frobenius error {fro:.3e}"


def expert_case(T, H, E, K, dtype, seed, duplicates=False):
    x, wd, wu, idx, g = orc.make_expert_inputs(T, H, E, K, seed=seed)
    if duplicates:
        idx[:, K // 2:] = idx[:, : K - K // 2]        # every id twice per token: contributions add
    return x.to(dtype), wd.to(dtype), wu.to(dtype), idx, g.to(dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,E,K,dup", [(64, 128, 256, 8, False), (200, 256, 64, 16, True), (33, 1024, 4096, 5, False),
                                         (16, 2048, 512, 4, False),
                                         (12, 8192, 48, 4, False), (20, 5120, 40, 3, True)])   # rows beyond one wave's registers
def test_expert_backward(dtype, T, H, E, K, dup):
    from flash_moe.ops import flash_expert_func
    from flash_moe.ops.hip.flash_expert import expert_backward

    x, wd, wu, idx, g = expert_case(T, H, E, K, dtype, seed=3, duplicates=dup)
    do = torch.randn(T, H, generator=gen(9)).to(dtype)
    leaves = [t.cuda().requires_grad_(True) for t in (x, wd, wu, g)]
    out = flash_expert_func(leaves[0], leaves[1], leaves[2], idx.cuda(), leaves[3])
    out.backward(do.cuda())
    ref_leaves = [t.double().requires_grad_(True) for t in (x, wd, wu, g)]
    orc.expert_forward(ref_leaves[0], ref_leaves[1], ref_leaves[2], idx, ref_leaves[3]).backward(do.double())
    for name, got, ref in zip(("dx", "ddown", "dup", "dgates"), leaves, ref_leaves):
        assert got.grad.dtype == dtype and got.grad.shape == ref.shape
        fro = rel_fro(got.grad, ref.grad)
        assert fro < GRAD_FRO[dtype], f"{name}: relative Frobenius error {fro:.3e}"
    # rows of experts nobody selected are exactly zero; the run is reproducible bit for bit
    unused = torch.ones(E, dtype=torch.bool)
    unused[idx.flatten()] = False
    assert (leaves[1].grad[unused.cuda()] == 0).all() and (leaves[2].grad[unused.cuda()] == 0).all()
    again = expert_backward(do.cuda(), x.cuda(), wd.cuda(), wu.cuda(), idx.cuda(), g.cuda())
    for a, b in zip(again, (leaves[0].grad, leaves[1].grad, leaves[2].grad, leaves[3].grad)):
        assert torch.equal(a, b)


def test_expert_backward_ignores_ids_out_of_range_and_handles_one_hot_expert():
    from flash_moe.ops.hip.flash_expert import expert_backward

    T, H, E, K, dtype = 96, 128, 32, 4, torch.float32
    x, wd, wu, idx, g = expert_case(T, H, E, K, dtype, seed=5)
    idx[:, 0] = 7                       # one expert takes a pair of every token: a long segment
    idx[::3, 1] = E + 5                 # invalid ids contribute nothing
    idx[1::3, 2] = -1
    do = torch.randn(T, H, generator=gen(4))
    dx, dwd, dwu, dg = expert_backward(*(t.cuda() for t in (do, x, wd, wu, idx, g)))
    valid = (idx >= 0) & (idx < E)
    ref_leaves = [t.double().requires_grad_(True) for t in (x, wd, wu, g)]
    safe = idx.clamp(0, E - 1)
    gates_masked = ref_leaves[3] * valid.double()
    orc.expert_forward(ref_leaves[0], ref_leaves[1], ref_leaves[2], safe, gates_masked).backward(do.double())
    for name, got, ref in zip(("dx", "ddown", "dup"), (dx, dwd, dwu), ref_leaves):
        assert rel_fro(got, ref.grad) < GRAD_FRO[dtype], name
    assert rel_fro(dg, ref_leaves[3].grad * valid.double()) < GRAD_FRO[dtype] and (dg.cpu()[~valid] == 0).all()


@pytest.mark.parametrize("norm", [False, True])
def test_block_backward_fp32(norm):
    """All parameter and input gradients of the block, against float64 autograd of the oracle's formulas evaluated on
    the HIP path's own selection (the selection itself carries no gradient)."""
    from test_block_gpu import build

    H, I, E, K, T = 128, 256, 1024, 8, 192
    nk = 32
    m, w = build(H, I, E, K, norm, torch.float32, seed=2, std=0.05)
    x = torch.randn(2, T // 2, H, generator=gen(3))
    xd = x.cuda().requires_grad_(True)
    y, logits = m(xd)
    wy, wl = torch.randn(y.shape, generator=gen(4)), torch.randn(logits.shape, generator=gen(5)) * 0.1
    ((y * wy.cuda()).sum() + (logits * wl.cuda()).sum()).backward()
    assert int(m.router_norm.num_batches_tracked) == 1

    with torch.no_grad():
        m.router_norm.reset_running_stats()
        _, _, indices, _ = m.route(xd.detach().view(-1, H))
    idx = indices.cpu()
    p = {k: v.detach().double().cpu().requires_grad_(True) for k, v in m.named_parameters()}
    x64 = x.double().requires_grad_(True)
    tok = x64.view(-1, H)
    q = torch.nn.functional.batch_norm(tok, None, None, training=True, eps=1e-5)
    lg = q @ p["router_gate.weight"].t()
    lp = torch.log_softmax(lg.view(T, 2, nk), -1)
    scores = lp[:, 0].gather(1, idx // nk) + lp[:, 1].gather(1, idx % nk)
    gates = scores.exp()
    if norm:
        gates = gates / gates.sum(-1, keepdim=True)
    y64 = orc.mlp_forward(tok, p["gate_proj.weight"], p["up_proj.weight"], p["down_proj.weight"]) + orc.expert_forward(
        tok, p["down_embed.weight"], p["up_embed.weight"], idx, gates)
    ((y64.view(y.shape) * wy.double()).sum() + (lg.view(T, 2, nk).transpose(0, 1) * wl.double()).sum()).backward()
    assert rel_fro(y, y64.view(y.shape)) < 2e-5
    assert rel_fro(xd.grad, x64.grad) < 2e-4, f"dx {rel_fro(xd.grad, x64.grad):.3e}"
    for k, v in m.named_parameters():
        fro = rel_fro(v.grad, p[k].grad)
        assert fro < 2e-4, f"{k}: relative Frobenius error {fro:.3e}"


def test_block_backward_bf16_runs_and_matches_the_fused_forward():
    from test_block_gpu import build

    m, _ = build(256, 512, 4096, 16, True, torch.bfloat16, seed=1)
    x = torch.randn(1, 256, 256, generator=gen(2)).to(torch.bfloat16).cuda()
    with torch.no_grad():
        y0, l0 = m(x)
    m.router_norm.reset_running_stats()
    y1, l1 = m(x.clone().requires_grad_(True))
    y1.float().square().mean().backward()
    assert rel_fro(y1, y0) < 1e-2 and rel_fro(l1, l0) < 1e-2
    for k, v in m.named_parameters():
        assert v.grad is not None and torch.isfinite(v.grad).all(), k


def test_expert_backward_c4_tables_fewer_tokens():
    """C4's tables (16384 experts of width 1024, top-64, bf16) on 256 tokens: float64 autograd of the oracle in chunks."""
    from flash_moe.ops.hip.flash_expert import expert_backward

    T, H, E, K, dtype = 256, 1024, 16384, 64, torch.bfloat16
    x, wd, wu, idx, g = expert_case(T, H, E, K, dtype, seed=11)
    do = torch.randn(T, H, generator=gen(12)).to(dtype)
    dx, dwd, dwu, dg = expert_backward(*(t.cuda() for t in (do, x, wd, wu, idx, g)))
    ref = [t.double().requires_grad_(True) for t in (x, wd, wu, g)]
    orc.expert_forward(ref[0], ref[1], ref[2], idx, ref[3], token_chunk=64).backward(do.double())
    for name, got, r in zip(("dx", "ddown", "dup", "dgates"), (dx, dwd, dwu, dg), ref):
        fro = rel_fro(got, r.grad)
        assert fro < GRAD_FRO[dtype], f"{name}: relative Frobenius error {fro:.3e}"


@pytest.mark.parametrize("E,ids", [(40000, "spread"), (300, "spread"), (3, "spread"), (5000, "warm"), (5000, "hot"), (700, "warm")])
def test_expert_backward_groups_pairs_alike_in_both_ways(E, ids):
    # 65536 pairs are grouped by two partition passes, 64512 in one launch; the last pair of every token names no expert, so both calls
    # sum the same pairs and, each in ascending pair index, to the same bits.  Segments that a pair ranks itself in, that are sorted in
    # LDS, that are sorted after a group too large for LDS was written (warm: ten experts of 6450 pairs, three of 21504), and one of half
    # of all pairs (hot).  The float64 sum over the pairs keeps both from being wrong alike
    from flash_moe.ops import flash_expert_func

    T, K, H = 1024, 64, 64
    indices = torch.randint(0, E, (T, K), generator=gen(E))
    if ids == "warm":
        indices = torch.randint(0, 10, (T, K), generator=gen(E))
    if ids == "hot":
        indices[torch.rand(T, K, generator=gen(1)) < 0.5] = 7
    indices[:, -1] = -1
    x, dout = torch.randn(T, H, generator=gen(2)).cuda(), torch.randn(T, H, generator=gen(3)).cuda()
    down, up = (torch.randn(E, H, generator=gen(4)) * 0.1).cuda(), (torch.randn(E, H, generator=gen(5)) * 0.1).cuda()
    gates = torch.rand(T, K, generator=gen(6)).cuda()

    def grads(keep):
        ws = [down.clone().requires_grad_(True), up.clone().requires_grad_(True)]
        flash_expert_func(x, *ws, indices[:, :keep].contiguous().cuda(), gates[:, :keep].contiguous()).backward(dout)
        return ws[0].grad, ws[1].grad

    whole, fewer = grads(K), grads(K - 1)
    for a, b in zip(whole, fewer):
        assert torch.equal(a, b)
    ids64, x64, d64 = indices[:, :-1], x.double().cpu(), dout.double().cpu()
    s = torch.einsum("th,tkh->tk", x64, down.double().cpu()[ids64])
    act = torch.nn.functional.silu(s) * gates[:, :-1].double().cpu()
    dup = torch.zeros(E, H, dtype=torch.float64).index_add_(0, ids64.flatten(), (act[..., None] * d64[:, None]).flatten(0, 1))
    torch.testing.assert_close(whole[1].double().cpu(), dup, rtol=1e-4, atol=1e-5 * float(dup.abs().max()))


@pytest.mark.parametrize("T,K,E", [(64, 10, (1 << 21) + 5), (1024, 64, (1 << 23) + 100)])
def test_expert_backward_groups_pairs_of_tables_beyond_the_other_ways(T, K, E):
    """More experts than one launch or the coarse groups of the partition passes can hold (few pairs, and 65536): the pairs are grouped by
    counters in memory, with segments of one pair, of some hundred (ordered in LDS) and of 8000 (met in order).  Weight gradients
    against float64 sums, zeros where no token went, the same bits twice."""
    from flash_moe import _C
    from flash_moe.ops.hip.flash_expert import expert_backward

    H = 8
    assert _C.lib().fmoe_expert_backward_workspace_bytes(T, H, E, K, _C.F32) > 8 * E        # a counter and an offset per expert
    g = torch.Generator(device="cuda").manual_seed(K)
    idx = torch.randint(0, E, (T, K), device="cuda", generator=g)
    idx[:, 1], idx[::3, 2], idx[0, 0], idx[1, 0], idx[2, 0] = 77, E - 1, 0, -1, E
    if K == 64:
        idx[:, 8:16] = E // 2
    x, dout = torch.randn(T, H, device="cuda", generator=g), torch.randn(T, H, device="cuda", generator=g)
    down, up = torch.randn(E, H, device="cuda", generator=g) * 0.1, torch.randn(E, H, device="cuda", generator=g) * 0.1
    gates = torch.rand(T, K, device="cuda", generator=g)
    args = (dout, x, down, up, idx, gates)
    got = expert_backward(*args)
    assert all(torch.equal(a, b) for a, b in zip(got, expert_backward(*args)))
    valid = (idx >= 0) & (idx < E)
    used, at = torch.unique(idx.clamp(0, E - 1), return_inverse=True)
    leaves = [t.double().cpu().requires_grad_(True) for t in (down[used], up[used])]
    orc.expert_forward(x.double().cpu(), *leaves, at.cpu(), (gates * valid).double().cpu()).backward(dout.double().cpu())
    for grad, ref in zip(got[1:3], leaves):
        assert rel_fro(grad[used], ref.grad) < GRAD_FRO[torch.float32]
        grad[used] = 0
        assert not grad.any()


@pytest.mark.parametrize("T,K,E,power,most_ms", [(16384, 512, 102400, 1, 2.1), (16384, 512, 102400, 3, 60), (16384, 129, 20000, 3, 25),
                                                 (1024, 64, 1500, 2, 2.1)])
def test_expert_backward_groups_experts_whose_pairs_exceed_lds(T, K, E, power, most_ms):
    """Coarse groups of 10000 pairs of 128 experts each; groups of 900000 and experts of 180000 pairs (ids that crowd towards expert 0);
    tiles of 8192 and of 2048 pairs.  Weight gradients against a float64 sum over the pairs, the same bits twice, and no path on which a
    workgroup sorts one short segment after the other or walks all ids for a long one (3.5 and 157 ms for the first two; 1.3 and 29
    without)."""
    from flash_moe.ops.hip.flash_expert import expert_backward

    H = 8
    g = torch.Generator(device="cuda").manual_seed(K)
    idx = (E * torch.rand(T, K, device="cuda", generator=g, dtype=torch.float64) ** power).long().clamp_(0, E - 1)
    idx[::5, 0] = E
    x, dout, down, up = (torch.randn(n, H, device="cuda", generator=g) * s for n, s in ((T, 1.0), (T, 1.0), (E, 0.1), (E, 0.1)))
    gates = torch.rand(T, K, device="cuda", generator=g)
    args = (dout, x, down, up, idx, gates)
    got = expert_backward(*args)
    start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    times = []
    for _ in range(3):
        start.record()
        again = expert_backward(*args)
        stop.record()
        torch.cuda.synchronize()
        times.append(start.elapsed_time(stop))
        assert all(torch.equal(a, b) for a, b in zip(got, again))
    print(f"\n{T} x {K} of {E}, power {power}: {min(times):.2f} ms")
    assert min(times) < most_ms, times
    ddown, dup = (torch.zeros(E, H, device="cuda", dtype=torch.float64) for _ in range(2))
    for lo in range(0, T, 2048):
        i, x64, do64, g64 = idx[lo:lo + 2048], x[lo:lo + 2048].double(), dout[lo:lo + 2048].double(), gates[lo:lo + 2048].double()
        g64 = g64 * (i < E)
        i = i.clamp(0, E - 1)
        s = (down[i].double() * x64[:, None]).sum(-1)
        sig = torch.sigmoid(s)
        ds = (up[i].double() * do64[:, None]).sum(-1) * g64 * sig * (1 + s * (1 - sig))
        ddown.index_add_(0, i.flatten(), (ds[..., None] * x64[:, None]).flatten(0, 1))
        dup.index_add_(0, i.flatten(), ((s * sig * g64)[..., None] * do64[:, None]).flatten(0, 1))
    # an fp32 sum of n products in one chain is off by up to n * 2^-24 of the sum of their magnitudes; a lost or doubled pair of an expert of
    # n pairs by 1 / n of it.  Relative to the tensors, whose norm the sums of n such products make, 1e-4 holds for the longest here
    assert rel_fro(got[1], ddown) < 1e-4 and rel_fro(got[2], dup) < 1e-4


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_expert_backward_column_slices(dtype):
    """Enough pairs (65536) for the column-slice schedule of the per-token part; some ids invalid, some doubled."""
    from flash_moe import _C
    from flash_moe.ops.hip.flash_expert import expert_backward

    T, H, E, K = 1024, 264, 4096, 64                    # 264 columns: the last slice is partial
    code = _C.dtype_code(dtype)
    lib = _C.lib()
    assert lib.fmoe_expert_backward_workspace_bytes(T, H, E, K, code) > lib.fmoe_expert_backward_workspace_bytes(T // 2, H, E, K, code) * 3
    x, wd, wu, idx, g = expert_case(T, H, E, K, dtype, seed=21)
    idx[:, 5] = idx[:, 4]
    idx[::7, 9] = E + 3
    idx[3::11, 17] = -2
    do = torch.randn(T, H, generator=gen(22)).to(dtype)
    dx, dwd, dwu, dg = expert_backward(*(t.cuda() for t in (do, x, wd, wu, idx, g)))
    valid = (idx >= 0) & (idx < E)
    ref = [t.double().requires_grad_(True) for t in (x, wd, wu, g)]
    orc.expert_forward(ref[0], ref[1], ref[2], idx.clamp(0, E - 1), ref[3] * valid.double(), token_chunk=128).backward(do.double())
    for name, got, r in zip(("dx", "ddown", "dup"), (dx, dwd, dwu), ref):
        fro = rel_fro(got, r.grad)
        assert fro < GRAD_FRO[dtype], f"{name}: relative Frobenius error {fro:.3e}"
    assert rel_fro(dg, ref[3].grad * valid.double()) < GRAD_FRO[dtype] and (dg.cpu()[~valid] == 0).all()
    again = expert_backward(*(t.cuda() for t in (do, x, wd, wu, idx, g)))
    assert all(torch.equal(a, b) for a, b in zip(again, (dx, dwd, dwu, dg)))


def test_block_backward_c4_full_size_properties():
    """Forward + backward of the README block at full size: finite, reproducible gradients for every parameter, and the
    gradient of the input agrees with a finite difference of the loss along a random direction (fp32 accumulation of
    a bf16 forward, so the bar is loose)."""
    from test_block_gpu import build

    dtype = torch.bfloat16
    m, _ = build(1024, 4096, 16384, 64, False, dtype)
    m.eval()                                     # running statistics: the loss is a fixed function of x
    x = torch.randn(1, 4096, 1024, generator=gen(0)).to(dtype).cuda()
    wy = torch.randn(1, 4096, 1024, generator=gen(1)).to(dtype).cuda()

    def run():
        for p in m.parameters():
            p.grad = None
        xg = x.clone().requires_grad_(True)
        y, _ = m(xg)
        (y.float() * wy.float()).sum().backward()
        return xg.grad, {k: v.grad.clone() for k, v in m.named_parameters()}

    gx, gp = run()
    gx2, gp2 = run()
    assert torch.equal(gx, gx2) and all(torch.equal(gp[k], gp2[k]) for k in gp)
    assert torch.isfinite(gx).all() and all(torch.isfinite(v).all() and v.abs().sum() > 0 for k, v in gp.items()
                                            if k != "router_gate.weight")
    # expert rows without a selected pair have zero gradient, the others (almost surely) not
    with torch.no_grad():
        _, _, indices, _ = m.route(x.view(-1, 1024))
    used = torch.zeros(16384, dtype=torch.bool, device="cuda")
    used[indices.flatten()] = True
    assert (gp["down_embed.weight"][~used] == 0).all() and (gp["up_embed.weight"][~used] == 0).all()
    assert (gp["up_embed.weight"][used].abs().sum(-1) > 0).all()


def test_backward_of_empty_batches():
    from flash_moe.ops.hip.flash_expert import expert_backward
    from flash_moe.ops.hip.flash_mlp import mlp_backward
    from flash_moe.ops.hip.flash_router import router_topk_backward

    H, E, K, I, nk = 64, 32, 4, 128, 8
    z = lambda *s: torch.zeros(*s, device="cuda")
    assert router_topk_backward(z(0, K), torch.zeros(0, K, dtype=torch.int64, device="cuda"), nk).shape == (2, 0, nk)
    wd, wu = torch.randn(E, H, device="cuda"), torch.randn(E, H, device="cuda")
    dx, dwd, dwu, dg = expert_backward(z(0, H), z(0, H), wd, wu, torch.zeros(0, K, dtype=torch.int64, device="cuda"), z(0, K))
    assert dx.shape == (0, H) and dg.shape == (0, K) and (dwd == 0).all() and (dwu == 0).all()
    dx, dwg, dwu2, dwd2 = mlp_backward(z(0, H), z(0, H), torch.randn(I, H, device="cuda"), torch.randn(I, H, device="cuda"),
                                       torch.randn(H, I, device="cuda"))
    assert dx.shape == (0, H) and (dwg == 0).all() and (dwu2 == 0).all() and (dwd2 == 0).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_autograd_of_an_empty_batch_gives_zero_gradients(dtype):
    """An empty batch with trainable parameters: the autograd functions return zero gradients of the right shapes."""
    from flash_moe.modules.flash_moe import FlashMoE, FlashMoEConfig
    from flash_moe.ops.hip.flash_mlp import flash_mlp_func

    H, I = 64, 128
    wg, wu, wd = (torch.randn(s, device="cuda").to(dtype).requires_grad_(True) for s in ((I, H), (I, H), (H, I)))
    x = torch.zeros(0, H, device="cuda", dtype=dtype, requires_grad=True)
    y = flash_mlp_func(x, wg, wu, wd)
    assert y.shape == (0, H)
    y.sum().backward()
    assert x.grad.shape == (0, H) and all(w.grad is not None and (w.grad == 0).all() for w in (wg, wu, wd))

    m = FlashMoE(FlashMoEConfig(H, I, "silu", 64, 4, False)).to(device="cuda", dtype=dtype).eval()
    out, logits = m(torch.zeros(1, 0, H, device="cuda", dtype=dtype))
    assert out.shape == (1, 0, H) and logits.shape == (2, 0, 8)
    (out.float().sum() + logits.float().sum()).backward()
    for name, p in m.named_parameters():
        assert p.grad is None or (p.grad == 0).all(), name


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_block_backward_with_a_key_count_that_is_not_a_multiple_of_four(dtype):
    """num_experts = 100 -> 10 keys per half: rows of the gate gradient are not whole 16-byte packets."""
    from flash_moe.modules.flash_moe import FlashMoE, FlashMoEConfig

    H, I, E, K, T = 64, 128, 100, 4, 96
    m = FlashMoE(FlashMoEConfig(H, I, "silu", E, K, True)).to(device="cuda", dtype=dtype)
    x = torch.randn(2, T // 2, H, generator=gen(3)).to(dtype).cuda()

    def grads(forward):
        for p in m.parameters():
            p.grad = None
        m.router_norm.reset_running_stats()
        xg = x.clone().requires_grad_(True)
        y, logits = forward(xg)
        (y.float().square().sum() + logits.float().sum() * 0.01).backward()
        return xg.grad, {k: v.grad.clone() for k, v in m.named_parameters()}

    gx, gp = grads(m.forward_autograd)
    gx2, gp2 = grads(m.forward_autograd_ops)
    tol = 1e-4 if dtype == torch.float32 else 3e-2
    assert torch.isfinite(gx).all() and rel_fro(gx, gx2) < tol
    for k in gp:
        assert torch.isfinite(gp[k]).all() and rel_fro(gp[k], gp2[k]) < tol, k
    assert gp["router_gate.weight"].shape == (20, H) and gp["router_gate.weight"].abs().sum() > 0


@pytest.mark.parametrize("dtype,H,nk,K", [
    (torch.bfloat16, 8, 3, 2), (torch.float32, 4, 1, 1),             # one packet to a row, padded rows of d
    (torch.float16, 776, 65, 17), (torch.bfloat16, 520, 129, 65),    # a packet more than whole waves; either kernel of the registers
    (torch.bfloat16, 1032, 256, 128), (torch.float32, 264, 256, 64),
    (torch.bfloat16, 72, 257, 4), (torch.bfloat16, 72, 256, 129),    # beyond them: gradients in fp32 and a launch of their own
])
def test_block_backward_operands_from_the_routing_gradient(dtype, H, nk, K):
    """The routing gradient's kernel writes what the prologue's products read; the composition of ops forms it on its own."""
    from flash_moe.modules.flash_moe import FlashMoE, FlashMoEConfig

    m = FlashMoE(FlashMoEConfig(H, 64, "silu", nk * nk, K, True)).to(device="cuda", dtype=dtype)
    with torch.no_grad():
        m.router_gate.weight.normal_(0.0, 2.0 / H**0.5)
        m.down_embed.weight.normal_(0.0, H**-0.5)       # scores of order 1: with the default of 1 the gradients pass 65504 in fp16
        m.up_embed.weight.normal_(0.0, H**-0.5)
    x = torch.randn(1, 70, H, generator=gen(3)).to(dtype).cuda()
    wl = (torch.randn(2, 70, nk, generator=gen(7)) * 0.1).cuda()
    results = []
    for forward in (m.forward_autograd, m.forward_autograd_ops):
        for p in m.parameters():
            p.grad = None
        m.router_norm.reset_running_stats()
        xg = x.clone().requires_grad_(True)
        y, logits = forward(xg)
        (y.float().square().sum() + (logits.float() * wl).sum()).backward()
        results.append((xg.grad, m.router_gate.weight.grad.clone()))
    # both round the same fp32 gradients to the activation dtype; the 16-bit gates that reach them differ in their last bit
    for a, b in zip(*results):
        assert torch.isfinite(a).all() and rel_fro(a, b) < {torch.float32: 1e-4, torch.bfloat16: 3e-2, torch.float16: 6e-3}[dtype]


@pytest.mark.parametrize("dtype,T,H,nk,K", [
    (torch.bfloat16, 70, 8, 3, 2), (torch.float32, 70, 4, 1, 1), (torch.float16, 300, 776, 65, 17), (torch.bfloat16, 70, 520, 129, 65),
    (torch.bfloat16, 333, 1032, 256, 128), (torch.float32, 1030, 264, 256, 64), (torch.bfloat16, 2100, 72, 256, 4),
])
def test_block_backward_rounds_the_routing_gradient_as_the_launch_of_its_own(dtype, T, H, nk, K):
    """The gate weights' gradient of the block against fmoe_route_backward and fmoe_router_prologue_backward on the block's own gate
    gradients, logits and statistics: the same operands of the same products, so the same bits."""
    from flash_moe import _C

    I, E, g = 64, nk * nk, gen(T + H)
    rand = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).to(dtype).cuda()
    x, dy, dl = rand(T, H), rand(T, H), rand(2, T, nk, std=0.1)
    w = [rand(*s, std=s[-1] ** -0.5) for s in ((I, H), (I, H), (H, I), (2 * nk, H), (E, H), (E, H))]
    rm, rv, nbt = torch.zeros(H, device="cuda", dtype=dtype), torch.ones(H, device="cuda", dtype=dtype), torch.zeros((), device="cuda", dtype=torch.int64)
    L, code, stream, p = _C.lib(), _C.dtype_code(dtype), _C.current_stream(x.device), _C.ptr
    ext = (T, H, I, nk, E, K, code)
    saved, ws, ws2 = (torch.zeros(f(*ext), device="cuda", dtype=torch.uint8)
                      for f in (L.fmoe_block_saved_bytes, L.fmoe_block_workspace_bytes, L.fmoe_block_backward_workspace_bytes))
    out, logits = torch.empty_like(x), rand(T, 2 * nk)
    _C.check(L.fmoe_block_forward_save(p(x), *map(p, w), p(rm), p(rv), p(nbt), code, 1, 0.1, 1e-5, T, H, I, E, nk, K, code, 1, p(out), p(logits),
                                       p(saved), saved.numel(), p(ws), ws.numel(), stream), "forward")
    dx, dwg, dwu, dwd, dwr, ded, deu = (torch.empty_like(t) for t in (x, *w))
    _C.check(L.fmoe_block_backward(p(dy), p(dl), p(x), *map(p, w), p(saved), 1, T, H, I, E, nk, K, code, 1, p(dx), p(dwg), p(dwu), p(dwd), p(dwr),
                                   p(ded), p(deu), p(ws2), ws2.numel(), stream), "backward")

    def at(buffer, offset, shape, dtype):
        n = torch.Size(shape).numel() * dtype.itemsize
        return buffer[offset:offset + n].view(dtype).view(shape), offset + (n + 255) // 256 * 256

    # what the forward keeps begins with the logits, the ids, the gates and the statistics, the backward's scratch with the gate gradients
    logits32, o = at(saved, 0, (T, 2 * nk), torch.float32)
    ids, o = at(saved, o, (T, K), torch.int64)
    _, o = at(saved, o, (T, K), dtype)
    stats, _ = at(saved, o, (2, H), torch.float32)
    dgates, _ = at(ws2, 0, (T, K), dtype)
    dlogits32, alone, dx_router = torch.empty(T, 2 * nk, device="cuda"), torch.empty_like(dwr), torch.empty_like(x)
    extra = dl.transpose(0, 1).reshape(T, 2 * nk).contiguous()
    _C.check(L.fmoe_route_backward(p(dgates), p(ids), p(logits32), p(extra), T, nk, K, code, 1, p(dlogits32), stream), "route")
    need = L.fmoe_router_prologue_backward_workspace_bytes(T, H, nk, code)
    ws3 = torch.empty(need, device="cuda", dtype=torch.uint8)
    _C.check(L.fmoe_router_prologue_backward(p(dlogits32), p(x), p(w[3]), p(stats), 1, T, H, nk, code, p(dx_router), p(alone), p(ws3), need, stream),
             "prologue")
    assert dlogits32.abs().sum() > 0 and torch.equal(dwr, alone)


@pytest.mark.parametrize("dtype,T,H,I", [
    (torch.bfloat16, 615, 776, 2072), (torch.float32, 383, 516, 1544),     # dx of the MLP in slices of k: added with the other gradients
    (torch.float16, 2050, 72, 136), (torch.bfloat16, 4101, 520, 264),      # more than one row to a wave, rows beyond the last block
    (torch.float32, 3, 4, 8), (torch.bfloat16, 16400, 72, 136),
])
def test_block_backward_adds_the_token_gradients(dtype, T, H, I):
    """dx of the block is the sum of the MLP's, the experts' and the router's, formed where the last of them is."""
    from flash_moe.modules.flash_moe import FlashMoE, FlashMoEConfig
    from flash_moe.ops.hip.flash_expert import expert_backward
    from flash_moe.ops.hip.flash_mlp import mlp_backward
    from flash_moe.ops.hip.flash_router import route_backward, router_prologue_backward

    m = FlashMoE(FlashMoEConfig(H, I, "silu", 100, 5, False)).to(device="cuda", dtype=dtype)
    with torch.no_grad():
        for p in m.parameters():
            p.copy_((torch.randn(p.shape, generator=gen(p.numel())) * p.shape[-1] ** -0.5).to(dtype))
    x, dy = (torch.randn(1, T, H, generator=gen(k)).to(dtype).cuda() for k in (1, 2))
    xg = x.clone().requires_grad_(True)
    y, logits = m(xg)
    y.backward(dy)
    w = [getattr(m, n).weight for n in ("gate_proj", "up_proj", "down_proj", "router_gate", "down_embed", "up_embed")]
    with torch.no_grad():
        m.router_norm.reset_running_stats()
        _, _, indices, gates, logits32 = m.route(x[0], return_logits32=True)
        x64 = x[0].double()
        stats = torch.stack((x64.mean(0), (x64.var(0, unbiased=False) + m.router_norm.eps).rsqrt())).float()
        mlp = mlp_backward(dy[0], x[0], *w[:3])
        experts = expert_backward(dy[0], x[0], w[4], w[5], indices, gates)
        router = router_prologue_backward(route_backward(experts[3], indices, logits32, 10, False), x[0], w[3], stats, True)
    expect = mlp[0].double() + experts[0].double() + router[0].double()
    # every term may be rounded to the type before the sum here, only the sum there
    assert rel_fro(xg.grad[0], expect) < {torch.float32: 1e-5, torch.bfloat16: 8e-3, torch.float16: 1e-3}[dtype]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_mlp_backward_with_saved_products_equals_recomputation(dtype):
    from flash_moe.ops.hip.flash_mlp import mlp_backward, mlp_forward, mlp_forward_saving

    T, H, I = 256, 256, 512
    x = torch.randn(T, H, generator=gen(1)).to(dtype).cuda()
    wg, wu, wd = ((torch.randn(s, generator=gen(k)) * 0.05).to(dtype).cuda() for k, s in ((2, (I, H)), (3, (I, H)), (4, (H, I))))
    dy = torch.randn(T, H, generator=gen(5)).to(dtype).cuda()
    out, saved = mlp_forward_saving(x, wg, wu, wd)
    assert torch.equal(out, mlp_forward(x, wg, wu, wd)) and saved.shape == (2, T, I)
    tol = 1e-5 if dtype == torch.float32 else 1e-2
    torch.testing.assert_close(saved[0].float(), x.float() @ wg.float().t(), rtol=tol, atol=tol)
    torch.testing.assert_close(saved[1].float(), x.float() @ wu.float().t(), rtol=tol, atol=tol)
    for a, b in zip(mlp_backward(dy, x, wg, wu, wd, saved), mlp_backward(dy, x, wg, wu, wd)):
        assert rel_fro(a, b) < (1e-6 if dtype == torch.float32 else 2e-3)


@pytest.mark.parametrize("what", ["mlp", "block"])
def test_memory_of_a_training_step(what):
    """In planes of [T, I], the largest tensors of a step: the forward keeps two (gate and up product), the backward works in three
    more (dh, da, db) beside the gradients."""
    from flash_moe.modules.flash_moe import FlashMoE, FlashMoEConfig
    from flash_moe.ops import flash_mlp_func

    T, H, I = 4096, 128, 8192
    plane = T * I * 2
    m = FlashMoE(FlashMoEConfig(H, I, "silu", 1024, 8)).to(device="cuda", dtype=torch.bfloat16)
    x = torch.randn(1, T, H, generator=gen(0)).bfloat16().cuda().requires_grad_()
    run = (lambda: m(x)[0]) if what == "block" else (lambda: flash_mlp_func(x, m.gate_proj.weight, m.up_proj.weight, m.down_proj.weight))
    run().sum().backward()                                   # gradients exist from here on: they are not counted below
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    y = run()
    kept = torch.cuda.memory_allocated() - before
    dy = torch.ones_like(y)
    torch.cuda.reset_peak_memory_stats()
    y.backward(dy)
    peak = torch.cuda.max_memory_allocated() - before
    # a quarter of a plane: tensors of the hidden and the routing width; half a plane more: new gradients and slices of k
    assert 2 * plane <= kept <= 2.25 * plane and peak <= 5.75 * plane, (kept / plane, peak / plane)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("stacked_weights", [False, True])
@pytest.mark.parametrize("stacked_grads", [False, True])
def test_mlp_backward_with_adjacent_and_separate_buffers(dtype, stacked_weights, stacked_grads):
    # fmoe_mlp_backward forms dWg and dWu as one product when dup_w starts where dgate_w ends, two otherwise; weights that
    # happen to follow each other in memory must make no difference.  Every combination against float64.
    from flash_moe import _C

    T, H, I = 320, 256, 384
    x = torch.randn(T, H, generator=gen(1)).to(dtype)
    wg, wu, wd = ((torch.randn(s, generator=gen(k)) * 0.05).to(dtype) for k, s in ((2, (I, H)), (3, (I, H)), (4, (H, I))))
    dy = torch.randn(T, H, generator=gen(5)).to(dtype)
    ref_leaves = [t.double().requires_grad_(True) for t in (x, wg, wu, wd)]
    orc.mlp_forward(*ref_leaves).backward(dy.double())

    xg, dyg, wdg = x.cuda(), dy.cuda(), wd.cuda()
    if stacked_weights:
        w2 = torch.cat([wg, wu]).cuda()
        wgg, wug = w2[:I], w2[I:]
        assert wug.data_ptr() == wgg.data_ptr() + I * H * wgg.element_size()
    else:
        w2 = torch.empty(2 * I * H + 64, device="cuda", dtype=dtype)          # a gap of 64 elements between the two
        wgg, wug = w2[:I * H].view(I, H).copy_(wg), w2[I * H + 64:].view(I, H).copy_(wu)
    if stacked_grads:
        g2 = torch.empty(2 * I, H, device="cuda", dtype=dtype)
        dwg, dwu = g2[:I], g2[I:]
    else:
        g2 = torch.empty(2 * I * H + 64, device="cuda", dtype=dtype)
        dwg, dwu = g2[:I * H].view(I, H), g2[I * H + 64:].view(I, H)
    dx, dwd = torch.empty_like(xg), torch.empty_like(wdg)
    L, code = _C.lib(), _C.dtype_code(dtype)
    ws_bytes = L.fmoe_mlp_backward_workspace_bytes(T, H, I, code)
    ws = torch.empty(ws_bytes, device="cuda", dtype=torch.uint8)
    status = L.fmoe_mlp_backward(_C.ptr(dyg), _C.ptr(xg), _C.ptr(wgg), _C.ptr(wug), _C.ptr(wdg), None, T, H, I, code, _C.ptr(dx),
                                 _C.ptr(dwg), _C.ptr(dwu), _C.ptr(dwd), _C.ptr(ws), ws_bytes, _C.current_stream(xg.device))
    _C.check(status, "fmoe_mlp_backward")
    torch.cuda.synchronize()
    for name, got, ref in zip(("dx", "dgate", "dup", "ddown"), (dx, dwg, dwu, dwd), ref_leaves):
        fro = rel_fro(got.cpu(), ref.grad)
        assert fro < GRAD_FRO[dtype], f"{name}: relative Frobenius error {fro:.3e}"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("training", [True, False])
@pytest.mark.parametrize("T,H,nk", [(256, 128, 16), (1000, 1024, 128), (65, 64, 8), (256, 128, 32), (1024, 1024, 128),
                                    (128, 64, 10), (70, 64, 6), (64, 128, 30), (40, 32, 81),
                                    # column sums of more row blocks than the last launch adds; rows of one packet, two, nine and 65
                                    (16384, 8, 3), (17000, 72, 12), (33000, 520, 5)])
def test_router_prologue_backward(dtype, training, T, H, nk):
    """Batch norm + gate product: gradients of the input and of the gate weights against float64 autograd."""
    from flash_moe.ops.hip.flash_router import router_prologue

    x = (torch.randn(T, H, generator=gen(1)) * 1.5 + 0.3).to(dtype)
    w = (torch.randn(2 * nk, H, generator=gen(2)) * 0.05).to(dtype)
    g32 = torch.randn(T, 2 * nk, generator=gen(3))
    g16 = (torch.randn(T, 2 * nk, generator=gen(4)) * 0.5).to(dtype)
    norm = torch.nn.BatchNorm1d(H, affine=False).cuda().to(dtype)
    with torch.no_grad():
        norm.running_mean.normal_(0.0, 0.2, generator=torch.Generator(device="cuda").manual_seed(5))
        norm.running_var.uniform_(0.5, 2.0, generator=torch.Generator(device="cuda").manual_seed(6))
    rm0, rv0 = norm.running_mean.clone(), norm.running_var.clone()
    norm.train(training)
    xd, wd = x.cuda().requires_grad_(True), w.cuda().requires_grad_(True)
    logits32, logits = router_prologue(xd, wd, norm)
    assert logits32.dtype == torch.float32 and logits.dtype == dtype
    ((logits32 * g32.cuda()).sum() + (logits.float() * g16.cuda().float()).sum()).backward()

    x64, w64 = x.double().requires_grad_(True), w.double().requires_grad_(True)
    q = torch.nn.functional.batch_norm(x64, rm0.double().cpu(), rv0.double().cpu(), training=training, eps=1e-5)
    ref = q @ w64.t()
    (ref * (g32.double() + g16.double())).sum().backward()
    tol = {torch.float32: 2e-5, torch.bfloat16: 1.2e-2, torch.float16: 3e-3}[dtype]
    assert rel_fro(logits32, ref) < tol
    assert rel_fro(xd.grad, x64.grad) < tol, f"dx {rel_fro(xd.grad, x64.grad):.3e}"
    assert rel_fro(wd.grad, w64.grad) < tol, f"dgate {rel_fro(wd.grad, w64.grad):.3e}"
    if training:   # a constant shift of the loss gradient along tokens cannot change dx: columns of dx sum to ~0
        assert float(xd.grad.float().sum(0).abs().max()) < 50 * tol * float(xd.grad.float().abs().max()) * T ** 0.5


def test_expert_backward_with_skewed_routing_is_exact_and_quick():
    """One expert selected by every one of 8192 tokens (a segment of 8192 pairs, as early in training or after a router
    collapse) next to ordinary experts: gradients against float64, bit-reproducible, and the call stays in the range of
    an ordinary backward (the long segment is walked once, in order)."""
    import time

    from flash_moe.ops.hip.flash_expert import expert_backward

    T, H, E, K = 8192, 1024, 4096, 8
    g = gen(31)
    x = torch.randn(T, H, generator=g).bfloat16()
    wd = (torch.randn(E, H, generator=g) * 0.05).bfloat16()
    wu = (torch.randn(E, H, generator=g) * 0.05).bfloat16()
    idx = torch.stack([torch.randperm(E - 1, generator=g)[:K] + 1 for _ in range(T)])
    idx[:, 3] = 0                                                # every token also selects expert 0
    gates = torch.softmax(torch.randn(T, K, generator=g), -1).bfloat16()
    dout = (torch.randn(T, H, generator=g) * 0.1).bfloat16()
    args = tuple(t.cuda() for t in (dout, x, wd, wu, idx, gates))
    got = expert_backward(*args)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    again = expert_backward(*args)
    torch.cuda.synchronize()
    elapsed = time.perf_counter() - t0
    assert all(torch.equal(a, b) for a, b in zip(got, again))
    assert elapsed < 0.05, f"{elapsed * 1e3:.1f} ms for a backward with one 8192-pair segment"
    # and against the same call on ids without such an expert: what it adds is its chain of 8192 additions, about 120 ns each in either
    # kernel of the weight gradients (twice that allowed)
    uniform = args[:4] + (torch.stack([torch.randperm(E - 1, generator=g)[:K] + 1 for _ in range(T)]).cuda(),) + args[5:]

    def call_us(call):
        times = []
        for _ in range(7):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            expert_backward(*call)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b) * 1e3)
        return sorted(times)[3]

    skewed, even = call_us(args), call_us(uniform)
    assert skewed - even < 2 * 0.12 * T, f"{skewed:.0f} us with a segment of {T} pairs, {even:.0f} without"
    # the hot expert's rows against float64: ddown[0] = sum_t ds_t x_t, dup[0] = sum_t silu(s_t) g_t dout_t
    x64, wd64, wu64, g64, do64 = (t.double() for t in (x, wd, wu, gates, dout))
    s = x64 @ wd64[0]
    sig = torch.sigmoid(s)
    act = s * sig
    u = do64 @ wu64[0]
    ds = u * g64[:, 3] * (sig * (1 + s * (1 - sig)))
    assert rel_fro(got[1][0], ds @ x64) < 1.5e-2
    assert rel_fro(got[2][0], (act * g64[:, 3]) @ do64) < 1.5e-2
    # an ordinary expert's rows too
    e = int(idx[5, 0])
    sel = (idx == e)
    tok, slot = sel.nonzero(as_tuple=True)
    s_e = x64[tok] @ wd64[e]
    sig_e = torch.sigmoid(s_e)
    u_e = do64[tok] @ wu64[e]
    assert rel_fro(got[2][e], (s_e * sig_e * g64[tok, slot]) @ do64[tok]) < 1.5e-2
    assert rel_fro(got[1][e], (u_e * g64[tok, slot] * (sig_e * (1 + s_e * (1 - sig_e)))) @ x64[tok]) < 1.5e-2


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,I", [
    (1, 8, 8), (9, 72, 136),                           # less than a tile on every side
    (65, 64, 1032), (127, 136, 264),                   # a row or a packet more or less than whole 64 x 64 tiles
    (48, 128, 4104),                                   # few tiles, long k: k split over workgroups (dx) and one k-tile (dW)
    (300, 264, 2056),                                  # one tile per compute unit at most: two k groups (dx)
    (1000, 2048, 1032),                                # 128 x 128 tiles with remainders
])
def test_mlp_backward_remainders_of_the_transposing_products(dtype, T, H, I):
    from flash_moe.ops.hip.flash_mlp import mlp_backward, mlp_forward_saving

    g = gen(T + I)
    x, dy = (torch.randn(T, H, generator=g).to(dtype).cuda() for _ in range(2))
    ws = [(torch.randn(s, generator=g) * 0.05).to(dtype).cuda() for s in ((I, H), (I, H), (H, I))]
    saved = mlp_forward_saving(x, *ws)[1]
    got = mlp_backward(dy, x, *ws, saved)
    leaves = [t.double().requires_grad_(True) for t in (x, *ws)]
    h = torch.nn.functional.silu(leaves[0] @ leaves[1].t()) * (leaves[0] @ leaves[2].t())
    (h @ leaves[3].t()).backward(dy.double())
    for name, a, leaf in zip(("dx", "dgate", "dup", "ddown"), got, leaves):
        assert rel_fro(a, leaf.grad) < GRAD_FRO[dtype], name
    assert all(torch.equal(a, b) for a, b in zip(got, mlp_backward(dy, x, *ws, saved)))      # bit for bit the same twice


@pytest.mark.parametrize("T,H,I", [(1, 4, 8), (65, 68, 1028), (300, 264, 2060), (383, 516, 1544), (900, 1032, 2056), (2500, 264, 2052),
                                   (1000, 520, 1032)])       # slices of 64 x 64 tiles beyond a round (dx, dWd)
def test_mlp_backward_remainders_of_the_transposing_products_fp32(T, H, I):
    test_mlp_backward_remainders_of_the_transposing_products(torch.float32, T, H, I)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,I", [
    (500, 2056, 4104),       # 128 x 128 tiles, one and two to a compute unit, and slices of k
    (600, 3080, 6152),       # dW on 256 x 256 tiles
    (2500, 264, 5000),       # dh on 256 x 256 tiles; slices for the weight gradients
    (260, 3080, 13000),      # dx on 256 x 256 tiles in slices
    (2048, 256, 8192), (512, 2048, 4096),      # nothing but whole 256 x 256 tiles: dh, dW
    (4096, 4096, 192), (4096, 4096, 328),      # dx on 256 x 256 tiles, two ranges of k: three k-tiles each, and with a tail
])
def test_mlp_backward_on_the_large_tiles_of_the_turned_products(dtype, T, H, I):
    test_mlp_backward_remainders_of_the_transposing_products(dtype, T, H, I)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,I", [
    (1, 8, 8), (63, 72, 64), (65, 136, 72), (127, 8, 1032), (1025, 1032, 2056),      # 64 x 64 tiles and their edges, one and many rounds
    (2049, 72, 1032), (4097, 264, 520),                                              # 128 x 128
    (129, 3080, 4104),                                                               # two launches
])
def test_mlp_backward_swiglu_gradient_in_the_product(dtype, T, H, I):
    """dh = dy Wd becomes da, db and h where it is formed: the gradients that hang on them, dx on da and db, dWd on h."""
    from flash_moe.ops.hip.flash_mlp import mlp_backward, mlp_forward_saving

    g = gen(T + H)
    x, dy = (torch.randn(T, H, generator=g).to(dtype).cuda() for _ in range(2))
    ws = [(torch.randn(s, generator=g) * s[-1] ** -0.5).to(dtype).cuda() for s in ((I, H), (I, H), (H, I))]
    saved = mlp_forward_saving(x, *ws)[1]
    a, b = saved.double()
    dh, sig = dy.double() @ ws[2].double(), torch.sigmoid(a)
    h, db = a * sig * b, dh * a * sig
    da = dh * b * sig * (1 + a * (1 - sig))
    for kept in (saved, None):                         # the products of the forward, or recomputed
        dx, dwg, dwu, dwd = mlp_backward(dy, x, *ws, kept)
        for name, got, ref in (("dwd", dwd, dy.double().t() @ h), ("dx", dx, da @ ws[0].double() + db @ ws[1].double()),
                               ("dwg", dwg, da.t() @ x.double()), ("dwu", dwu, db.t() @ x.double())):
            assert rel_fro(got, ref) < GRAD_FRO[dtype], (name, rel_fro(got, ref))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,I", [
    (1, 8, 8), (63, 72, 64), (65, 136, 72), (127, 8, 1032), (1025, 1032, 2056),      # 64 x 64 tiles and their edges, one and many rounds
    (2049, 72, 1032), (4097, 264, 520),                                              # 128 x 128
])
def test_mlp_backward_rounds_the_swiglu_gradient_once(dtype, T, H, I):
    """da, db and h as the products after them read them, from the scratch that begins with h and [da | db]: sums of H products in fp32 and
    one rounding, at most 2^-8 (2^-11) of a value and 1.66e-3 (2.1e-4) of many in the 2-norm, below 2^-9 (2^-12); with dh rounded on the way
    it would be 2.3e-3 (2.9e-4) of da and db."""
    from flash_moe import _C

    g = gen(T + I)
    rand = lambda *s, std=1.0: (torch.randn(*s, generator=g) * std).to(dtype).cuda()
    x, dy, saved = rand(T, H), rand(T, H), rand(2, T, I)
    wg, wu, wd = rand(I, H, std=H**-0.5), rand(I, H, std=H**-0.5), rand(H, I)
    L, code, p = _C.lib(), _C.dtype_code(dtype), _C.ptr
    need = L.fmoe_mlp_backward_saved_workspace_bytes(T, H, I, code)
    ws = torch.empty(need, device="cuda", dtype=torch.uint8)
    out = [torch.empty_like(t) for t in (dy, wg, wu, wd)]
    _C.check(L.fmoe_mlp_backward(p(dy), p(x), p(wg), p(wu), p(wd), p(saved), T, H, I, code, *map(p, out), p(ws), need, _C.current_stream(x.device)), "mlp")
    plane = T * I * 2
    h = ws[:plane].view(dtype).view(T, I)
    dab = ws[(plane + 255) // 256 * 256:][:2 * plane].view(dtype).view(T, 2 * I)
    a, b = saved.double()
    dh, sig = dy.double() @ wd.double(), torch.sigmoid(a)
    once = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for name, got, want in (("h", h, a * sig * b), ("db", dab[:, I:], dh * a * sig), ("da", dab[:, :I], dh * b * sig * (1 + a * (1 - sig)))):
        # beside it: the fp32 sums, and half a step of fp16 below its normal range
        slack = 1e-6 * want.abs().max() + 2.0 ** -25
        assert ((got.double() - want).abs() <= 1.001 * once * want.abs() + slack).all(), name
        assert T * I < 4096 or rel_fro(got, want) < once / 2, (name, rel_fro(got, want))


@pytest.mark.parametrize("dtype,T,H,I", [
    (torch.bfloat16, 513, 264, 520), (torch.float16, 2600, 264, 264),        # one launch on 64 x 64 tiles: whole; weight gradients in slices
    (torch.float16, 1000, 1800, 4104), (torch.bfloat16, 5200, 776, 264),     # on 128 x 128: dx in slices; weight gradients in slices
    (torch.bfloat16, 3000, 520, 1032),                                       # on 128 x 128, whole
    (torch.float16, 1500, 1544, 5000),                                       # on 256 x 256, dx in slices
    (torch.float32, 515, 132, 260), (torch.float32, 383, 516, 1544), (torch.float32, 2100, 136, 264),   # whole, dx, weight gradients
    (torch.float32, 3076, 1284, 3076),                                       # on 128 x 128, dx in slices
])
def test_mlp_backward_products_in_one_launch(dtype, T, H, I):
    """Sizes that take every tile shape and cut of the launch that forms dWd, dx, dWg and dWu together, none a multiple of a tile."""
    test_mlp_backward_remainders_of_the_transposing_products(dtype, T, H, I)


@pytest.mark.parametrize("stacked", [False, True])
@pytest.mark.parametrize("dtype,T,H,I", [
    (torch.bfloat16, 513, 264, 520), (torch.float16, 2600, 264, 264),        # products that would share a launch: whole; in slices of k
    (torch.bfloat16, 129, 3080, 4104), (torch.float32, 383, 516, 1544),
    (torch.bfloat16, 300, 2048, 11008),                                      # and products that would not
])
def test_mlp_backward_in_place(dtype, T, H, I, stacked):
    """dx in the place of dy and each weight's gradient in that of the weight, which only products before them read."""
    from flash_moe import _C
    from flash_moe.ops.hip.flash_mlp import mlp_backward, mlp_forward_saving

    g = gen(T + I)
    x, dy = (torch.randn(T, H, generator=g).to(dtype).cuda() for _ in range(2))
    both = (torch.randn(2, I, H, generator=g) * 0.05).to(dtype).cuda()
    wg, wu = both if stacked else (both[0].clone(), both[1].clone())
    wd = (torch.randn(H, I, generator=g) * 0.05).to(dtype).cuda()
    saved = mlp_forward_saving(x, wg, wu, wd)[1]
    want = mlp_backward(dy, x, wg, wu, wd, saved)
    L, code, stream = _C.lib(), _C.dtype_code(dtype), _C.current_stream(x.device)
    need = L.fmoe_mlp_backward_saved_workspace_bytes(T, H, I, code)
    ws = torch.empty(need, device="cuda", dtype=torch.uint8)
    others = [torch.empty_like(t) for t in (dy, wg, wu, wd)]
    for places in ((0,), (1, 2), (3,), (0, 1, 2, 3)):                        # which of dx, dWg, dWu, dWd lie on dy and the weights
        held = torch.stack((wg, wu)) if stacked else (wg.clone(), wu.clone())
        tensors = [dy.clone(), held[0], held[1], wd.clone()]
        out = [tensors[i] if i in places else others[i] for i in range(4)]
        _C.check(L.fmoe_mlp_backward(_C.ptr(tensors[0]), _C.ptr(x), *map(_C.ptr, tensors[1:]), _C.ptr(saved), T, H, I, code, *map(_C.ptr, out),
                                     _C.ptr(ws), need, stream), "in place")
        for name, a, b in zip(("dx", "dgate", "dup", "ddown"), out, want):
            # the same products, their sums cut differently: two roundings to the type apart at most; in fp32 two sums of up to n terms,
            # each off by the random walk of n roundings of 2^-24
            n = max(T, 2 * I)
            assert rel_fro(a, b) < {torch.float32: 2 * n ** 0.5 * 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype], (places, name)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,H,E,K", [
    (3, 24, 40, 4), (256, 264, 900, 5), (257, 520, 300, 33), (2049, 136, 5000, 9),      # waves per token of the row schedule
    (120, 2048, 70, 17), (64, 1032, 20000, 70),        # rows of several packets per lane; experts without pairs, spans of experts
    (1500, 1544, 700, 20),                             # x and dout beyond an L2: column chunks, the last one partial
    (200, 64, 3, 2), (700, 72, 2, 2),                  # segments of more than a round of pairs
])
def test_expert_backward_edges_of_the_waves_and_spans(dtype, T, H, E, K):
    from flash_moe.ops.hip.flash_expert import expert_backward

    g = gen(T + H)
    x, dy = (torch.randn(T, H, generator=g).to(dtype).cuda() for _ in range(2))
    wd, wu = (torch.randn(E, H, generator=g).mul(0.05).to(dtype).cuda() for _ in range(2))
    idx = torch.randint(0, E, (T, K), generator=g).cuda()
    gates = torch.softmax(torch.randn(T, K, generator=g), -1).to(dtype).cuda()
    got = expert_backward(dy, x, wd, wu, idx, gates)
    leaves = [t.double().requires_grad_(True) for t in (x, wd, wu, gates)]
    out = torch.zeros(T, H, device="cuda", dtype=torch.float64)
    for k in range(K):
        s = (leaves[0] * leaves[1][idx[:, k]]).sum(-1)
        out = out + (torch.nn.functional.silu(s) * leaves[3][:, k])[:, None] * leaves[2][idx[:, k]]
    out.backward(dy.double())
    for name, a, leaf in zip(("dx", "ddown", "dup", "dgates"), got, leaves):
        assert rel_fro(a, leaf.grad) < GRAD_FRO[dtype], name


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,E,K,first", [
    (4100, 136, 900, 9, 0), (2060, 520, 20000, 7, 0),  # rows below 1 KB; experts without pairs, several spans to a quarter
    (2050, 1544, 333, 3, 0),                           # the last chunk partial, spans of one
    (4099, 520, 3, 2, 0), (2200, 1032, 50, 5, 47),     # fewer experts than quarters; lists of very different lengths
    (4100, 264, 900, 13, 0), (3000, 520, 33000, 17, 0), (3001, 1544, 333, 17, 0),      # the first three with the pairs that they take
    (20001, 40, 5000, 3, 0),                           # rows shorter than a quarter's chunk
])
def test_expert_weight_gradients_by_quarter_waves(dtype, T, H, E, K, first):
    """Chunks of x and dout beyond an L2, with ids out of range among the pairs (they count for nothing)."""
    from flash_moe.ops.hip.flash_expert import expert_backward

    g = gen(T + H)
    x, dy = (torch.randn(T, H, generator=g).to(dtype).cuda() for _ in range(2))
    wd, wu = (torch.randn(E, H, generator=g).mul(0.05).to(dtype).cuda() for _ in range(2))
    idx = torch.randint(0, E, (T, K), generator=g).clamp_min(first).cuda()
    idx[5::97, 0] = E
    gates = torch.softmax(torch.randn(T, K, generator=g), -1).to(dtype).cuda()
    got = expert_backward(dy, x, wd, wu, idx, gates)
    valid = idx < E
    leaves = [t.double().requires_grad_(True) for t in (x, wd, wu, gates)]
    out = torch.zeros(T, H, device="cuda", dtype=torch.float64)
    for k in range(K):
        e = idx[:, k].clamp(max=E - 1)
        s = (leaves[0] * leaves[1][e]).sum(-1)
        out = out + (torch.nn.functional.silu(s) * leaves[3][:, k] * valid[:, k])[:, None] * leaves[2][e]
    out.backward(dy.double())
    for name, a, leaf in zip(("dx", "ddown", "dup", "dgates"), got, leaves):
        assert rel_fro(a, leaf.grad) < GRAD_FRO[dtype], name
    unused = torch.ones(E, dtype=torch.bool, device="cuda")
    unused[idx[valid]] = False
    assert (got[1][unused] == 0).all() and (got[2][unused] == 0).all()
    for a, b in zip(expert_backward(dy, x, wd, wu, idx, gates), got):
        assert torch.equal(a, b)
