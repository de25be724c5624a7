"""Parity of the HIP SwiGLU MLP (MFMA GEMMs, fused activation) with the CPU oracle, through the op."""
import pytest
import torch

from helpers import assert_output_close, cuda, rel_fro
from oracle import flashmoe_oracle as orc

pytestmark = pytest.mark.gpu


def make(T, H, I, dtype, seed, x_std=1.0, w_std=0.02):
    g = torch.Generator().manual_seed(seed)
    x = (torch.randn(T, H, generator=g) * x_std).to(dtype)
    wg = (torch.randn(I, H, generator=g) * w_std).to(dtype)
    wu = (torch.randn(I, H, generator=g) * w_std).to(dtype)
    wd = (torch.randn(H, I, generator=g) * w_std).to(dtype)
    return x, wg, wu, wd


def truth64(x, wg, wu, wd):
    return orc.mlp_forward(x.double(), wg.double(), wu.double(), wd.double())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,H,I", [
    (512, 256, 1024),      # C1
    (1024, 1024, 4096),    # C4 weights, fewer tokens (small-tile path)
    (4096, 1024, 4096),    # C4 (large-tile path for gate/up)
    (192, 128, 256),       # 64-row tiles (T a multiple of 64 only)
    (100, 128, 256),       # ragged T on the tiled path: the last tile row reads clamped rows, stores are bounds-checked
    (1000, 256, 512),
    (200, 72, 136),        # ragged in every dimension
    (1, 64, 64),
])
def test_mlp_matches_oracle(dtype, T, H, I):
    from flash_moe.ops import flash_mlp_func

    x, wg, wu, wd = make(T, H, I, dtype, seed=T + I)
    got = flash_mlp_func(*cuda(x, wg, wu, wd)).cpu()
    assert got.dtype == dtype and got.shape == (T, H)
    ref64 = truth64(x, wg, wu, wd)
    assert_output_close(got, ref64.to(dtype), dtype, "mlp vs float64 oracle")
    assert rel_fro(got, ref64) < {torch.float32: 2e-6, torch.bfloat16: 6e-3, torch.float16: 8e-4}[dtype]
    if T <= 1024:
        assert_output_close(got, orc.mlp_forward(x, wg, wu, wd), dtype, "mlp vs same-dtype oracle")


def test_mlp_fp32_tensors_off_the_16_byte_grid():
    # fp32 callers need not align their tensors: the tiled kernel moves 16-byte pieces, so these take the bounds-checked
    # kernel, and the result is the aligned one's up to summation order
    from flash_moe.ops import flash_mlp_func

    x, wg, wu, wd = cuda(*make(256, 256, 512, torch.float32, seed=9))

    def shifted(t):
        buf = torch.empty(t.numel() + 1, device="cuda", dtype=t.dtype)
        buf[1:].copy_(t.reshape(-1))
        v = buf[1:].view(t.shape)
        assert v.data_ptr() % 16 == 4
        return v

    aligned = flash_mlp_func(x, wg, wu, wd)
    moved = flash_mlp_func(shifted(x), shifted(wg), shifted(wu), shifted(wd))
    ref64 = truth64(*(t.cpu() for t in (x, wg, wu, wd)))
    assert rel_fro(aligned, ref64) < 2e-6 and rel_fro(moved, ref64) < 2e-6


def test_mlp_reference_test_distribution():
    # tests/test_mlp.py:95-107: seed 42, x ~ N(0,0.5), weights ~ N(0,0.1); its shape scaled down
    from flash_moe.ops import flash_mlp_func

    x, wg, wu, wd = make(1024, 512, 2048, torch.bfloat16, seed=42, x_std=0.5, w_std=0.1)
    got = flash_mlp_func(*cuda(x, wg, wu, wd)).cpu()
    assert rel_fro(got, truth64(x, wg, wu, wd)) < 6e-3


def test_mlp_leading_dims_and_residual():
    from flash_moe.ops import flash_mlp_func
    from flash_moe.ops.hip.flash_mlp import mlp_forward

    x, wg, wu, wd = cuda(*make(192, 128, 256, torch.bfloat16, seed=3))
    y2 = flash_mlp_func(x, wg, wu, wd)
    y3 = flash_mlp_func(x.view(2, 96, 128), wg, wu, wd)
    assert y3.shape == (2, 96, 128) and torch.equal(y3.view(192, 128), y2)
    res = torch.randn(192, 128, device="cuda").bfloat16()
    yr = mlp_forward(x, wg, wu, wd, residual=res)
    ref = truth64(*(t.cpu() for t in (x, wg, wu, wd))) + res.cpu().double()
    assert rel_fro(yr.cpu(), ref) < 6e-3
    assert flash_mlp_func(x[:0], wg, wu, wd).shape == (0, 128)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,H,I", [(4096, 1024, 4096), (1024, 1024, 4096), (192, 128, 256), (200, 72, 136)])
def test_mlp_residual_is_added_in_every_tile_shape_and_dtype(dtype, T, H, I):
    # the block's "experts + mlp" is the down projection's epilogue: one case per kernel the dispatch can pick (256 x 256 and
    # 128 x 128 tiles, 64-row tiles, the bounds-checked kernel).  The residual is large against the product, so a lane that
    # reads a neighbour's residual shows at once; the sum is rounded once, from the fp32 accumulator.
    from flash_moe.ops.hip.flash_mlp import mlp_forward

    x, wg, wu, wd = make(T, H, I, dtype, seed=T + H)
    res = torch.randn(T, H, generator=torch.Generator().manual_seed(5)).to(dtype)
    got = mlp_forward(*cuda(x, wg, wu, wd), residual=res.cuda()).cpu()
    ref64 = truth64(x, wg, wu, wd) + res.double()
    assert got.dtype == dtype and got.shape == (T, H)
    assert rel_fro(got, ref64) < {torch.float32: 2e-6, torch.bfloat16: 6e-3, torch.float16: 8e-4}[dtype]
    assert (got.double() - ref64).abs().max() < {torch.float32: 1e-5, torch.bfloat16: 4e-2, torch.float16: 6e-3}[dtype]


def test_mlp_linearity_full_size():
    # C4 at full size: out is linear in the down projection and in the up projection
    from flash_moe.ops import flash_mlp_func

    x, wg, wu, wd = cuda(*make(4096, 1024, 4096, torch.bfloat16, seed=0))
    y = flash_mlp_func(x, wg, wu, wd)
    assert torch.equal(flash_mlp_func(x, wg, wu, wd * 2), y * 2)
    assert torch.equal(flash_mlp_func(x, wg, wu * 0.5, wd), y * 0.5)
    assert flash_mlp_func(x, wg, wu * 0, wd).abs().max() == 0
    assert torch.equal(flash_mlp_func(x, wg, wu, wd), y)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,H,I", [
    (1, 8, 8), (17, 40, 24), (16, 520, 1032),          # 16-row tiles with k split over the waves
    (33, 264, 1000), (130, 1032, 136),                 # 32 x 32 tiles, remainders on every side
    (615, 776, 2072), (999, 1000, 2664),               # 64-row tiles
    (3001, 1160, 3080), (5000, 1336, 3560),            # 128 x 128 and 256 x 256 tiles
])
def test_mlp_remainders_of_every_tile_shape(dtype, T, H, I):
    # both products with their outputs between guard rows: nothing outside [T, N] may be written, and the gate and up
    # products kept for a backward pass match as well
    from flash_moe import _C

    x, wg, wu, wd = cuda(*make(T, H, I, dtype, seed=T + H + I))
    res = torch.randn(T, H, device="cuda").to(dtype)
    L, code, stream = _C.lib(), _C.dtype_code(dtype), _C.current_stream(x.device)

    def guarded(rows, cols):
        buf = torch.full((rows + 16, cols), 7.0, device="cuda", dtype=dtype)
        return buf, buf[8:8 + rows]

    (abuf, act), (sbuf, saved), (obuf, out) = guarded(T, I), guarded(2 * T, I), guarded(T, H)
    _C.check(L.fmoe_mlp_gate_up_save(*map(_C.ptr, (x, wg, wu)), T, H, I, code, _C.ptr(act), _C.ptr(saved), stream), "gate/up")
    _C.check(L.fmoe_mlp_down(_C.ptr(act), _C.ptr(wd), T, H, I, code, _C.ptr(res), _C.ptr(out), stream), "down")
    tol = {torch.float32: 2e-6, torch.bfloat16: 6e-3, torch.float16: 8e-4}[dtype]
    a, b = x.double() @ wg.double().t(), x.double() @ wu.double().t()
    assert rel_fro(saved[:T], a) < tol and rel_fro(saved[T:], b) < tol
    assert rel_fro(act, torch.nn.functional.silu(a) * b) < tol
    assert rel_fro(out, act.double() @ wd.double().t() + res.double()) < tol
    for buf in (abuf, sbuf, obuf):
        assert (buf[:8] == 7).all() and (buf[-8:] == 7).all()


@pytest.mark.parametrize("T,H,I", [(512, 256, 1024), (385, 516, 1028), (301, 260, 996), (1500, 36, 1060), (400, 4, 992), (393, 100, 1004)])
def test_mlp_fp32_on_gate_up_tiles_of_32_columns(T, H, I):
    """64 x 64 tiles of 32 gate and 32 up columns: whole ones, remainders in rows, columns and k, one k-tile and a k tail of one packet."""
    test_mlp_remainders_of_every_tile_shape(torch.float32, T, H, I)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,I", [
    (4096, 1024, 1536), (2000, 1928, 1480), (3900, 1000, 1544), (1100, 2960, 1608), (3001, 1000, 2664),     # 24, 24, 25, 26 and 42 k-tiles
    (2000, 1928, 1472),                                                                                   # the last before them
    (3969, 1000, 1536), (3969, 1000, 1544), (1025, 3080, 1736),    # one row in the last tiles: 24, 25 and 28 k-tiles
    (3970, 1000, 1544),                                            # and two
])
def test_mlp_down_on_tiles_whose_k_the_waves_divide(dtype, T, H, I):
    """128 x 128 tiles that one wave each multiplies a quarter of k of: whole ones and remainders in every extent, guard rows around the
    output, with a residual and without, and in place of it."""
    assert ((T + 127) // 128) * ((H + 127) // 128) <= 256          # a compute unit to each of these tiles
    test_mlp_remainders_of_every_tile_shape(dtype, T, H, I)
    from flash_moe import _C

    act, wd, res = (torch.randn(*s, device="cuda").to(dtype) for s in ((T, I), (H, I), (T, H)))
    wd *= 0.02
    L, code, stream = _C.lib(), _C.dtype_code(dtype), _C.current_stream(act.device)
    tol, product = {torch.bfloat16: 6e-3, torch.float16: 8e-4}[dtype], act.double() @ wd.double().t()
    plain, added = torch.empty_like(res), res.clone()
    _C.check(L.fmoe_mlp_down(_C.ptr(act), _C.ptr(wd), T, H, I, code, None, _C.ptr(plain), stream), "down")
    _C.check(L.fmoe_mlp_down(_C.ptr(act), _C.ptr(wd), T, H, I, code, _C.ptr(added), _C.ptr(added), stream), "down")
    assert rel_fro(plain, product) < tol and rel_fro(added, product + res.double()) < tol


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,H,I", [(47, 1032, 8200), (129, 520, 4104), (203, 1032, 12296), (300, 2056, 8008), (129, 1001, 4004)])
@pytest.mark.parametrize("with_residual", [False, True])
def test_mlp_down_with_slices_of_k(dtype, T, H, I, with_residual):
    # each tile shape with remainders in rows, columns and k; guard rows around the output and the sums; planes of a size that is no
    # multiple of four elements (fp32); and the result of the uncut product up to the order of the sums
    from flash_moe import _C

    if dtype != torch.float32 and H % 8:
        H += 8 - H % 8
        I += 8 - I % 8
    _, _, _, wd = cuda(*make(T, H, I, dtype, seed=T + I))
    act = torch.randn(T, I, device="cuda").to(dtype)
    res = torch.randn(T, H, device="cuda").to(dtype) if with_residual else None
    L, code, stream = _C.lib(), _C.dtype_code(dtype), _C.current_stream(act.device)
    need = L.fmoe_mlp_down_workspace_bytes(T, H, I, code)
    assert need > 0 and need % 256 == 0 and L.fmoe_mlp_down_workspace_bytes(4096, 4096, 1024, code) == 0
    ws = torch.full((need + 512,), 7, device="cuda", dtype=torch.uint8)
    buf = torch.full((T + 16, H), 7.0, device="cuda", dtype=dtype)
    out = buf[8:8 + T]
    args = (_C.ptr(act), _C.ptr(wd), T, H, I, code, _C.ptr(res) if res is not None else None)
    assert L.fmoe_mlp_down_ws(*args, _C.ptr(out), _C.ptr(ws), need - 1, stream) == -7
    _C.check(L.fmoe_mlp_down_ws(*args, _C.ptr(out), _C.ptr(ws[256:]), need, stream), "down")
    whole = torch.empty_like(out)
    _C.check(L.fmoe_mlp_down(*args, _C.ptr(whole), stream), "down")
    want = act.double() @ wd.double().t() + (res.double() if res is not None else 0.0)
    tol = {torch.float32: 2e-6, torch.bfloat16: 6e-3, torch.float16: 8e-4}[dtype]
    assert rel_fro(out, want) < tol and rel_fro(out, whole.cpu()) < tol
    assert (buf[:8] == 7).all() and (buf[-8:] == 7).all() and (ws[:256] == 7).all() and (ws[-256:] == 7).all()


@pytest.mark.parametrize("T,H,I", [(300, 4104, 16392), (1000, 2056, 16392)])
def test_mlp_down_with_slices_of_k_on_the_largest_tiles(T, H, I):
    test_mlp_down_with_slices_of_k(torch.bfloat16, T, H, I, True)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,N,K", [
    (8200, 2056, 8), (8200, 2056, 64), (8200, 2056, 136),        # one, one and three k-tiles: the loop takes two at a time
    (8192, 2048, 200), (8192, 2048, 256),                        # whole tiles with a k tail, and nothing but whole tiles
    (8449, 2312, 72),                                            # a last row and a last column of tiles of one and eight
])
def test_mlp_on_the_widest_tiles(dtype, T, N, K):
    """256 x 256 tiles: several to a workgroup, remainders in every extent, guard rows around every output, a residual large against
    the sums; and tensors off the 16-byte grid, which smaller tiles take.  Bound: the sums are exact in fp32 up to K roundings of 2^-24,
    so the one rounding to the type remains (2^-9 and 2^-12 relative), twice for the activation, which multiplies two of them."""
    from flash_moe import _C

    g = torch.Generator(device="cuda").manual_seed(T + N + K)
    x, wg, wu = (torch.randn(*s, device="cuda", generator=g).to(dtype) for s in ((T, K), (N, K), (N, K)))
    res = (100 * torch.randn(T, N, device="cuda", generator=g)).to(dtype)
    L, code, stream = _C.lib(), _C.dtype_code(dtype), _C.current_stream(x.device)

    def guarded(rows, shift=0):
        buf = torch.full(((rows + 16) * N + 8,), 7.0, device="cuda", dtype=dtype)
        return buf, buf[8 * N + shift:(8 + rows) * N + shift].view(rows, N)

    tol = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}[dtype]
    a, b = (torch.cat([x[i:i + 1024].double() @ w.double().t() for i in range(0, T, 1024)]) for w in (wg, wu))
    for shift in (0, 1):
        (abuf, act), (sbuf, saved), (obuf, out) = guarded(T), guarded(2 * T), guarded(T, shift)
        _C.check(L.fmoe_mlp_gate_up_save(*map(_C.ptr, (x, wg, wu)), T, K, N, code, _C.ptr(act), _C.ptr(saved), stream), "gate/up")
        _C.check(L.fmoe_mlp_down(_C.ptr(x), _C.ptr(wg), T, N, K, code, _C.ptr(res), _C.ptr(out), stream), "down")
        for got, want, times in ((saved[:T], a, 1), (saved[T:], b, 1), (act, torch.nn.functional.silu(a) * b, 2), (out, a + res.double(), 1)):
            off = (got.double() - want).abs()
            assert off.norm() < times * tol * want.norm() and (off <= 2 * times * tol * want.abs() + 1e-5 * K).all()
        for buf, rows, at in ((abuf, T, 0), (sbuf, 2 * T, 0), (obuf, T, shift)):
            assert (buf[:8 * N + at] == 7).all() and (buf[(8 + rows) * N + at:] == 7).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,H,I", [
    (337, 2056, 2664),        # more operand bytes than runs of tiles begin at, 3 tile-rows; dx in slices
    (1154, 392, 784),         # fewer: the order as it is
    (2200, 1016, 1992),       # several groups of eight tile-rows, the last not full
])
def test_mlp_where_tiles_are_no_multiple_of_the_xcds(dtype, T, H, I):
    """Every tile is formed once, forward and backward, however the XCDs share them out: a left-out tile is wrong by its whole size.
    Bound: one rounding to the type per stage (2^-9; fp32 sums of I products), three of them one after another in the longest chain."""
    from flash_moe.ops import flash_mlp_func

    x, *ws = (t.cuda().requires_grad_(True) for t in make(T, H, I, dtype, seed=T + H))
    dy = torch.randn(T, H, generator=torch.Generator().manual_seed(I)).to("cuda", dtype)
    y = flash_mlp_func(x, *ws)
    y.backward(dy)
    x64, *ws64 = (t.detach().double().requires_grad_(True) for t in (x, *ws))
    y64 = (torch.nn.functional.silu(x64 @ ws64[0].t()) * (x64 @ ws64[1].t())) @ ws64[2].t()
    y64.backward(dy.double())
    tol = 3 * 2.0 ** -9 if dtype == torch.bfloat16 else 2e-5
    for got, want in [(y.detach(), y64.detach())] + [(a.grad, b.grad) for a, b in zip((x, *ws), (x64, *ws64))]:
        off, size = got.double() - want, want.norm()
        assert off.norm() < tol * size
        rows = off.norm(dim=1)
        assert (rows < 4 * tol * size / want.shape[0] ** 0.5).all()
