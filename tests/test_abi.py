"""The C-ABI library: loads without a GPU, exports every symbol the header declares, and rejects bad
arguments with the documented status codes before touching the device."""
import ctypes
import os
import re

import pytest
import torch

from flash_moe import _C

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "flashmoe_hip.h")


def declared_functions():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(fmoe_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_expected_entry_points():
    names = declared_functions()
    for must in ("fmoe_router_topk", "fmoe_expert_forward", "fmoe_mlp_forward", "fmoe_last_error", "fmoe_abi_version"):
        assert must in names


def test_library_exports_every_declared_symbol():
    lib = _C.lib()
    for name in declared_functions():
        assert hasattr(lib, name), f"{name} declared in flashmoe_hip.h but not exported by {_C.lib_path()}"
    # and the Python binding table names exactly the declared functions
    assert sorted(_C.SIGNATURES) == declared_functions()
    assert lib.fmoe_abi_version() == _C.ABI_VERSION


def test_citations_in_header_point_at_the_reference_interface():
    text = open(HEADER).read()
    for cite in ("flash_router.py:381-382", "flash_expert.py:831-836", "flash_mlp.py:169-181", "flash_moe.py:101"):
        assert cite in text


def _buf(n=4096):
    b = ctypes.create_string_buffer(n + 256)
    addr = (ctypes.addressof(b) + 255) // 256 * 256
    return b, addr


def test_router_argument_checks():
    lib = _C.lib()
    keep, a = _buf()
    # top_k outside [0, nk]: the reference's assertion (flash_router.py:261-263)
    assert lib.fmoe_router_topk(a, 4, 8, 9, _C.F32, a, a, None, 0, None) == -3
    assert b"[0, 8]" in lib.fmoe_last_error()
    assert lib.fmoe_router_topk(a, 4, 8, -1, _C.F32, a, a, None, 0, None) == -3
    assert lib.fmoe_router_topk(a, 4, 8, 4, 7, a, a, None, 0, None) == -4          # dtype
    assert lib.fmoe_router_topk(a, -1, 8, 4, _C.F32, a, a, None, 0, None) == -2     # shape
    assert lib.fmoe_router_topk(None, 4, 8, 4, _C.F32, a, a, None, 0, None) == -1   # null
    assert lib.fmoe_router_topk(a, 4, 8192, 4097, _C.F32, a, a, None, 0, None) == -5  # top_k > 4096
    assert lib.fmoe_router_topk(a, 4, 70000, 4, _C.F32, a, a, None, 0, None) == -5    # num_keys > 65535
    # empty problems succeed without a launch
    assert lib.fmoe_router_topk(None, 0, 8, 4, _C.F32, None, None, None, 0, None) == 0
    assert lib.fmoe_router_topk(a, 4, 8, 0, _C.F32, a, a, None, 0, None) == 0
    assert lib.fmoe_last_error() == b""


def test_fused_router_argument_checks():
    lib = _C.lib()
    keep, a = _buf()
    f = lib.fmoe_router_forward
    need = lib.fmoe_router_workspace_bytes(64, 128, 16)
    assert need > 0 and need % 256 == 0
    ok_args = dict(x=a, w=a, rm=a, rv=a, nbt=a)
    call = lambda **kw: f(kw.get("x", a), a, a, a, a, _C.F32, kw.get("training", 1), 0.1, 1e-5, kw.get("T", 64), 128, 16,
                          kw.get("K", 4), kw.get("dtype", _C.BF16), 0, a, a, a, a, a, kw.get("ws", a), kw.get("wsb", need), None)
    assert call(K=17) == -3                       # top_k > num_keys
    assert call(dtype=9) == -4
    assert call(T=-1) == -2
    assert call(T=1) == -2                        # one token in training mode, as nn.BatchNorm1d
    assert b"more than 1 value per channel" in lib.fmoe_last_error()
    assert call(x=None) == -1
    assert call(wsb=need - 1) == -7
    assert call(T=0) == 0


def test_expert_argument_checks():
    lib = _C.lib()
    keep, a = _buf()
    f = lib.fmoe_expert_forward
    assert f(a, a, a, a, a, 4, 64, 16, 2, 9, a, None, 0, None) == -4
    assert f(a, a, a, a, a, 4, 0, 16, 2, _C.BF16, a, None, 0, None) == -2
    assert f(None, a, a, a, a, 4, 64, 16, 2, _C.BF16, a, None, 0, None) == -1
    assert f(a, a, a, None, a, 4, 64, 16, 2, _C.BF16, a, None, 0, None) == -1
    assert f(a, a, a, a, a, 4, 60, 16, 2, _C.BF16, a, None, 0, None) == -6          # row not 16-byte multiple
    assert f(a + 2, a, a, a, a, 4, 64, 16, 2, _C.BF16, a, None, 0, None) == -6      # misaligned pointer
    # rows too long for the row kernels take the column slices, which need their workspace; forcing rows is refused
    assert f(a, a, a, a, a, 4, 1 << 20, 16, 2, _C.BF16, a, None, 0, None) == -7
    assert lib.fmoe_expert_workspace_bytes(4, 1 << 20, 16, 2, _C.BF16) > 0
    assert lib.fmoe_expert_forward_algo(a, a, a, a, a, 4, 1 << 20, 16, 2, _C.BF16, a, None, 0, _C.EXPERT_ROWS, None) == -5
    assert f(None, None, None, None, None, 0, 64, 16, 2, _C.BF16, None, None, 0, None) == 0
    assert isinstance(lib.fmoe_expert_workspace_bytes(1024, 1024, 16384, 64, _C.BF16), int)
    # the size follows the schedule: column slices when a slice of the table fits L2 and there are enough pairs, else none
    sliced = lib.fmoe_expert_workspace_bytes(4096, 1024, 16384, 64, _C.BF16)
    assert sliced >= 4096 * 64 * (4 + 4 + 8 * 4) and sliced % 256 == 0               # 8 slices of 256 bytes
    wide = lib.fmoe_expert_workspace_bytes(4096, 1024, 32768, 64, _C.BF16)
    assert wide >= 4096 * 64 * (4 + 4 + 16 * 4) and wide % 256 == 0                   # 16 slices of 128 bytes
    # a table whose slices are too large for L2 takes the bucketed schedule: bucketing state, grouped order, band-major x,
    # 32 bands of partial scores, the per-owner lists of the sweep
    big = lib.fmoe_expert_workspace_bytes(32768, 2048, 262144, 128, _C.BF16)
    assert big >= 32768 * 128 * 4 * (4 + 32 + 2) + 32768 * 2048 * 2 and big % 256 == 0
    assert big == lib.fmoe_expert_workspace_bytes_algo(32768, 2048, 262144, 128, _C.BF16, _C.EXPERT_BUCKETS)
    assert lib.fmoe_expert_workspace_bytes_algo(32768, 2048, 262144, 128, _C.BF16, _C.EXPERT_ROWS) == 0
    assert lib.fmoe_expert_workspace_bytes(64, 1024, 16384, 8, _C.BF16) == 0            # too few pairs
    assert lib.fmoe_expert_workspace_bytes_algo(64, 1024, 16384, 8, _C.BF16, _C.EXPERT_SLICES) > 0
    assert lib.fmoe_expert_workspace_bytes_algo(4096, 1024, 16384, 64, _C.BF16, _C.EXPERT_ROWS) == 0
    assert lib.fmoe_expert_workspace_bytes_algo(4096, 1024, 16384, 64, _C.BF16, _C.EXPERT_AUTO) == sliced
    # a product-key memory has no score phase: it never takes the bucketed plan's workspace (the reference's PKM
    # benchmark shape, tests/test_pkm.py: 16384 tokens, top-2500, would ask for gigabytes of partial scores there)
    assert lib.fmoe_pkm_workspace_bytes(4096, 1024, 16384, 64, _C.BF16) == sliced
    assert lib.fmoe_pkm_workspace_bytes(32768, 2048, 262144, 128, _C.BF16) == 0
    assert lib.fmoe_pkm_workspace_bytes(16384, 1024, 1 << 20, 2500, _C.BF16) == 0 < lib.fmoe_expert_workspace_bytes(
        16384, 1024, 1 << 20, 2500, _C.BF16)
    assert lib.fmoe_pkm_workspace_bytes(0, 1024, 16, 4, _C.BF16) == 0 and lib.fmoe_pkm_workspace_bytes(4, 1024, 16, 4, 9) == 0


def test_mlp_argument_checks():
    lib = _C.lib()
    keep, a = _buf()
    f = lib.fmoe_mlp_forward
    need = lib.fmoe_mlp_workspace_bytes(8, 64, 128, _C.BF16)
    assert need >= 8 * 128 * 2 and need % 256 == 0
    assert lib.fmoe_mlp_workspace_bytes(8, 64, 128, _C.F32) >= 8 * 128 * 4
    assert f(a, a, a, a, 8, 64, 128, 5, None, a, a, need, None) == -4
    assert f(a, a, a, a, 8, 64, -1, _C.BF16, None, a, a, need, None) == -2
    assert f(a, None, a, a, 8, 64, 128, _C.BF16, None, a, a, need, None) == -1
    assert f(a, a, a, a, 8, 64, 128, _C.BF16, None, a, a, need - 1, None) == -7
    assert f(a, a, a, a, 8, 64, 128, _C.BF16, None, a, None, need, None) == -7
    assert f(a, a, a, a, 8, 60, 128, _C.BF16, None, a, a, need, None) == -6
    assert f(None, None, None, None, 0, 64, 128, _C.BF16, None, None, None, 0, None) == 0


def test_block_argument_checks():
    lib = _C.lib()
    keep, a = _buf()
    f = lib.fmoe_block_forward
    T, H, I, E, nk, K = 8, 64, 128, 1024, 32, 4
    need = lib.fmoe_block_workspace_bytes(T, H, I, nk, E, K, _C.BF16)
    parts = (lib.fmoe_router_workspace_bytes(T, H, nk) + lib.fmoe_expert_workspace_bytes(T, H, E, K, _C.BF16)
             + lib.fmoe_mlp_workspace_bytes(T, H, I, _C.BF16))
    assert need >= parts + T * 2 * nk * 4 + T * K * (4 + 8 + 2) + T * H * 2 and need % 256 == 0
    assert lib.fmoe_block_workspace_bytes(T, H, I, nk, E, K, 9) == 0

    def call(T=T, H=H, I=I, E=E, nk=nk, K=K, dtype=_C.BF16, x=a, ws=a, ws_bytes=need):
        return f(x, a, a, a, a, a, a, a, a, a, _C.F32, 1, 0.1, 1e-5, T, H, I, E, nk, K, dtype, 0, a, a, None, None,
                 ws, ws_bytes, None)

    assert call(dtype=6) == -4
    assert call(I=0) == -2
    assert call(nk=33) == -2                      # nk*nk > E
    assert call(K=33) == -3 and b"[0, 32]" in lib.fmoe_last_error()
    assert call(x=None) == -1
    assert call(H=60) == -6
    assert call(I=100) == -6
    assert call(ws_bytes=need - 1) == -7
    assert call(ws=None) == -7
    assert call(T=0, x=None, ws=None, ws_bytes=0) == 0


def test_backward_argument_checks():
    lib = _C.lib()
    keep, a = _buf()
    rb = lib.fmoe_router_topk_backward
    assert rb(a, a, 4, 8, 2, 9, a, None) == -4
    assert rb(a, a, 4, 0, 2, _C.F32, a, None) == -2
    assert rb(a, a, 4, 70000, 2, _C.F32, a, None) == -5                          # the forward op's own key limit
    assert rb(a, None, 4, 8, 2, _C.F32, a, None) == -1
    assert rb(None, None, 0, 8, 2, _C.F32, None, None) == 0
    rt = lib.fmoe_route_backward
    assert rt(a, a, a, None, 4, 8, 2, 9, 0, a, None) == -4                       # dtype
    assert rt(a, a, a, None, 4, 0, 2, _C.BF16, 0, a, None) == -2                 # num_keys
    assert rt(a, a, a, None, 4, 40000, 2, _C.BF16, 0, a, None) == -5             # the fused router's own key limit
    assert rt(a, a, None, None, 4, 8, 2, _C.BF16, 0, a, None) == -1              # logits
    assert rt(None, None, a, None, 4, 8, 2, _C.BF16, 0, a, None) == -1           # gate gradient with top_k > 0
    assert rt(None, None, None, None, 0, 8, 2, _C.BF16, 1, None, None) == 0      # empty batch
    off = lib.fmoe_router_workspace_stats_offset(64, 128, 16)
    assert 0 < off < lib.fmoe_router_workspace_bytes(64, 128, 16) and off % 256 == 0
    pneed = lib.fmoe_router_prologue_backward_workspace_bytes(64, 128, 16, _C.BF16)
    assert pneed >= 64 * 32 * 2 + 2 * 64 * 128 * 2 and pneed % 256 == 0
    pb = lib.fmoe_router_prologue_backward
    assert pb(a, a, a, a, 1, 64, 128, 16, 4, a, a, a, pneed, None) == -4
    assert pb(a, a, a, a, 1, 0, 128, 16, _C.BF16, a, a, a, pneed, None) == -2
    assert pb(a, a, a, a, 1, 64, 124, 16, _C.BF16, a, a, a, pneed, None) == -6
    assert pb(None, a, a, a, 1, 64, 128, 16, _C.BF16, a, a, a, pneed, None) == -1
    assert pb(a, a, a, a, 1, 64, 128, 16, _C.BF16, a, a, a, pneed - 1, None) == -7
    sb = lib.fmoe_swiglu_backward
    assert sb(a, a, a, 4, 64, 7, a, a, None) == -4
    assert sb(a, a, a, 4, 0, _C.BF16, a, a, None) == -2
    assert sb(a, a, a, 4, 60, _C.BF16, a, a, None) == -6
    assert sb(a, None, a, 4, 64, _C.BF16, a, a, None) == -1
    assert sb(None, None, None, 0, 64, _C.BF16, None, None, None) == 0
    need = lib.fmoe_expert_backward_workspace_bytes(8, 64, 256, 4, _C.BF16)
    # rows: two fp32 coefficients and a place in its expert's list for every pair, the lists' ends; with slices one of the
    # coefficients, the row's offset and two partial scores to a slice for every pair besides
    assert need >= 8 * 4 * (8 + 4) + 257 * 4 and need % 256 == 0
    sliced = lib.fmoe_expert_backward_workspace_bytes(4096, 1024, 16384, 64, _C.BF16)
    assert sliced >= 4096 * 64 * (8 + 4 + 4 + 4 + 2 * 8 * 4) + 16385 * 4 and sliced % 256 == 0
    eb = lib.fmoe_expert_backward

    def ecall(T=8, H=64, E=256, K=4, dtype=_C.BF16, dout=a, ws=a, ws_bytes=need):
        return eb(dout, a, a, a, a, a, T, H, E, K, dtype, a, a, a, a, ws, ws_bytes, None)

    assert ecall(dtype=3) == -4
    assert ecall(H=0) == -2
    assert ecall(H=60) == -6
    assert ecall(H=8192) == -7                     # long rows take the column-slice kernels: a larger workspace
    assert ecall(H=8192, E=1 << 19) == -5          # ... which cannot address tables of 4 GiB or more
    assert ecall(dout=None) == -1
    assert ecall(ws_bytes=need - 1) == -7
    mneed = lib.fmoe_mlp_backward_workspace_bytes(8, 64, 128, _C.BF16)
    assert mneed >= 6 * 8 * 128 * 2 and mneed % 256 == 0
    sneed = lib.fmoe_mlp_backward_saved_workspace_bytes(8, 64, 128, _C.BF16)
    assert 3 * 8 * 128 * 2 <= sneed <= mneed - 3 * 8 * 128 * 2
    mb = lib.fmoe_mlp_backward

    def mcall(T=8, H=64, I=128, dtype=_C.BF16, dy=a, ws_bytes=mneed):
        return mb(dy, a, a, a, a, None, T, H, I, dtype, a, a, a, a, a, ws_bytes, None)

    assert mcall(dtype=5) == -4
    assert mcall(T=0) == -2
    assert mcall(I=100) == -6
    assert mcall(dy=None) == -1
    assert mcall(ws_bytes=mneed - 1) == -7
    assert mb(a, a, a, a, a, a, 8, 64, 128, _C.BF16, a, a, a, a, a, sneed - 1, None) == -7      # with saved products


@pytest.mark.parametrize("T,H,E,K", [(1024, 2048, 16384, 32), (1960, 1536, 3481, 31), (521, 2048, 9000, 63), (2047, 2048, 9801, 31)])
def test_few_bf16_pairs_of_long_rows_keep_fp32_coefficients(T, H, E, K):
    """Below 2^16 pairs bf16 takes whole rows however many bytes they are, without scratch and with nothing kept for a backward pass: its
    column slices round the coefficients, fp16's and fp32's do not, and a product-key memory's are routing weights as they came."""
    lib = _C.lib()
    assert T * K < 1 << 16 and T * K * H * 2 >= 128000000
    assert lib.fmoe_expert_workspace_bytes(T, H, E, K, _C.BF16) == lib.fmoe_expert_saved_bytes(T, H, E, K, _C.BF16) == 0
    for code in (_C.F16, _C.F32):
        assert lib.fmoe_expert_workspace_bytes(T, H, E, K, code) == lib.fmoe_expert_workspace_bytes_algo(T, H, E, K, code, _C.EXPERT_SLICES)
    assert lib.fmoe_pkm_workspace_bytes(T, H, E, K, _C.BF16) > 0


@pytest.mark.parametrize("T,H,E,K,dtype,schedule", [
    # grouping by expert: rows from 2 KB on, in fp32 from 1.5 KB, a dozen pairs per expert, however many experts
    (24600, 256, 131072, 64, "BF16", "ROWS"), (25000, 640, 200000, 96, "F16", "ROWS"), (32768, 512, 102400, 64, "BF16", "ROWS"),
    (32768, 896, 102400, 64, "BF16", "ROWS"), (32768, 1024, 102400, 64, "BF16", "BUCKETS"), (32768, 1024, 102400, 64, "F16", "BUCKETS"),
    (32768, 352, 102400, 64, "F32", "ROWS"), (32768, 384, 102400, 64, "F32", "BUCKETS"), (19000, 384, 102400, 64, "F32", "ROWS"),
    # ordered lists where no slice fits: few tokens with many experts; rows of three, five and six slices; rows between lines
    (282, 384, 120943, 757, "BF16", "ORDERED"), (286, 256, 144100, 540, "F16", "ORDERED"), (2172, 384, 101688, 535, "F16", "ORDERED"),
    (1097, 736, 66109, 816, "BF16", "ORDERED"), (2107, 336, 25869, 881, "F16", "ORDERED"), (282, 384, 120943, 400, "BF16", "ROWS"),
    (3118, 640, 100000, 64, "BF16", "ROWS"), (282, 384, 120943, 99, "BF16", "ROWS"),
    # and where 400 tokens name every expert, instead of the grouping, which rounds the coefficients in bf16
    (8301, 1024, 334092, 1078, "BF16", "ORDERED"), (18039, 1792, 838895, 4030, "BF16", "ORDERED"), (8301, 1024, 334092, 830, "BF16", "BUCKETS"),
    # slices in fp32: from ten experts per token on, and for rows of 4 KB of more than 32768 experts
    (16384, 1024, 16000, 9, "F16", "ROWS"), (16384, 480, 16000, 11, "F32", "SLICES"), (16384, 960, 16000, 11, "F16", "ROWS"),
    (6348, 1216, 53917, 31, "F32", "SLICES"), (7000, 2048, 50000, 31, "BF16", "ROWS"),
])
def test_expert_schedule_at_the_lines_of_its_rule(T, H, E, K, dtype, schedule):
    lib, code = _C.lib(), getattr(_C, dtype)
    want = lib.fmoe_expert_workspace_bytes_algo(T, H, E, K, code, getattr(_C, "EXPERT_" + schedule))
    assert lib.fmoe_expert_workspace_bytes(T, H, E, K, code) == want and (want > 0) == (schedule != "ROWS")
    assert (lib.fmoe_expert_saved_bytes(T, H, E, K, code) > 0) == (schedule in ("SLICES", "ORDERED"))


@pytest.mark.parametrize("quarters,whole,dtype", [
    ((4096, 512, 256, 4), (4096, 512, 257, 4), "BF16"),                # 64 pairs to an expert
    ((20000, 128, 5000, 2), (20000, 136, 5000, 2), "BF16"), ((20000, 64, 5000, 2), (20000, 68, 5000, 2), "F32"),      # rows of 256 bytes
    ((2868, 512, 1024, 18), (2867, 512, 1024, 18), "F16"),             # chunks of x and dout that exceed an L2 by two fifths
    ((2868, 4096, 2048, 18), (2867, 4096, 2048, 18), "BF16"),          # ... of which longer rows have more
    ((4096, 512, 8192, 12), (4095, 512, 8192, 12), "BF16"),            # 48 K pairs
    ((4096, 1024, 43690, 16), (4096, 1024, 43691, 16), "BF16"),        # one and a half to an expert
])
def test_expert_weight_gradients_by_quarter_waves_at_the_lines_of_their_rule(quarters, whole, dtype):
    """Their entries are 16 bytes of scratch to a pair."""
    lib, code = _C.lib(), getattr(_C, dtype)
    more, less = (lib.fmoe_expert_backward_workspace_bytes(*c, code) for c in (quarters, whole))
    pairs = quarters[0] * quarters[3]
    assert 15 * pairs < more - less < 17 * pairs


@pytest.mark.parametrize("T,H,nk,dtype,slices", [(32768, 256, 24, "BF16", 16), (32768, 256, 24, "F32", 16), (8192, 512, 64, "BF16", 12), (4096, 256, 24, "F32", 8)])
def test_backward_products_of_few_tiles_over_many_tokens_are_cut_as_if_alone(T, H, nk, dtype, slices):
    """A launch shared with another product leaves a weight gradient at most four slices of the tokens, fp32 sums of [2 nk, H] each."""
    lib, code, elt = _C.lib(), getattr(_C, dtype), 4 if dtype == "F32" else 2
    operands = T * elt * (2 * nk + 2 * H)
    assert lib.fmoe_router_prologue_backward_workspace_bytes(T, H, nk, code) >= operands + slices * 2 * nk * H * 4
    # and one that takes the shared launch keeps to them
    assert lib.fmoe_router_prologue_backward_workspace_bytes(2048, 1024, 128, code) < 2048 * elt * (2 * 128 + 2 * 1024) + 5 * 2 * 128 * 1024 * 4


def test_expert_workspace_is_enough_for_both_forwards():
    """The forward alone and that of a training step: one size for both."""
    lib = _C.lib()
    for T, H, E, K in ((4800, 2048, 66049, 222), (16384, 2048, 102400, 256), (1024, 1024, 102400, 512), (4096, 1024, 16384, 64)):
        need = lib.fmoe_expert_workspace_bytes(T, H, E, K, _C.BF16)
        assert need >= lib.fmoe_expert_workspace_bytes_algo(T, H, E, K, _C.BF16, _C.EXPERT_AUTO)
        if K > 64:
            assert need >= lib.fmoe_expert_workspace_bytes_algo(T, H, E, K, _C.BF16, _C.EXPERT_ORDERED)


def test_backward_scratch_holds_only_what_its_schedule_writes():
    """The row schedule of the experts has no list of coefficients; the block keeps no fp32 gradients of the logits where the routing
    gradient leaves as the gate's products read it (up to 256 keys and 128 experts)."""
    lib = _C.lib()
    T, H, E, K = 2048, 256, 4096, 8
    pairs, group = T * K, lib.fmoe_expert_backward_workspace_bytes(0, H, E, K, _C.BF16)
    assert group == 0 and lib.fmoe_expert_saved_bytes(T, H, E, K, _C.BF16) == 0             # rows
    assert lib.fmoe_expert_backward_workspace_bytes(T, H, E, K, _C.BF16) < pairs * (8 + 4) + (E + 1) * 4 + 4 * 256
    few, many = (lib.fmoe_block_backward_workspace_bytes(4096, 64, 64, nk, 257 * 257, 4, _C.BF16) for nk in (256, 257))
    assert 4096 * 2 * 257 * 4 <= many - few


def test_training_keeps_two_planes_of_the_intermediate_width():
    """What a block's forward leaves for its backward grows by the gate and up products, [2, T, I], with the intermediate width."""
    lib = _C.lib()
    T, H, nk, E, K = 512, 256, 32, 1024, 16
    for code, elt in ((_C.F32, 4), (_C.BF16, 2), (_C.F16, 2)):
        narrow, wide = (lib.fmoe_block_saved_bytes(T, H, I, nk, E, K, code) for I in (1024, 4096))
        assert wide - narrow == 2 * T * (4096 - 1024) * elt


def test_python_wrappers_refuse_cpu_tensors():
    from flash_moe.ops import flash_expert_func, flash_mlp_func, flash_router_func

    with pytest.raises(RuntimeError, match="no CPU path"):
        flash_router_func(torch.zeros(2, 4, 8), 8, 2)
    with pytest.raises(RuntimeError, match="no CPU path"):
        flash_expert_func(torch.zeros(4, 8), torch.zeros(16, 8), torch.zeros(16, 8), torch.zeros(4, 2, dtype=torch.int64), torch.zeros(4, 2))
    with pytest.raises(RuntimeError, match="no CPU path"):
        flash_mlp_func(torch.zeros(4, 8), torch.zeros(16, 8), torch.zeros(16, 8), torch.zeros(8, 16))
