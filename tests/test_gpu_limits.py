"""Tensors past 2 GiB through the C-ABI: row-major weights, activations and outputs each larger than 2^31 bytes.

Every kernel addresses its operands through buffer descriptors based at the tile it works on (32-bit offsets inside
one tile), and its stores through 64-bit pointers; these cases check that no index wraps when the whole tensor is
larger than a 32-bit byte offset reaches. Each runs the plan and three more configurations from the library's
candidate list, and every element is compared with the oracle's arithmetic on the GPU tensors (torch fp32 GEMM)
within the north star's tolerance. (Packed weights are limited to 2 GiB by ojx_pack_weight; that limit is an
error-path check here.)
"""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = dict(max_rel=1e-2, mean_abs_rms=1e-3)
GIB2 = 1 << 31


def _say(*a):
    print(*a, flush=True)


def _configs(L, M, N, K, kind, seed):
    cands = L.candidates(M, N, K, kind)
    pick = np.random.default_rng(seed).choice(len(cands), size=min(3, len(cands)), replace=False)
    return [None] + [cands[int(i)] for i in pick]


def _check(O, got, want, what):
    ok, a, b = O.tolerance_ok(got, want, **TOL)
    assert ok, f"{what}: max_rel {a:.3e} mean/rms {b:.3e}"


@pytest.mark.parametrize("M,N,K,what", [
    (16, 73728, 16384, "weight"),     # W 2.25 GiB
    (300, 73728, 16384, "weight"),
    (65536, 256, 17408, "x"),         # x 2.125 GiB
    (65536, 16384, 512, "y"),         # y exactly 2^31 bytes
    (65600, 16384, 512, "y"),         # y past 2^31 bytes
])
def test_plain_past_2gib(pkg, ext, O, dev, M, N, K, what):
    L = pkg._lib
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device=dev).bfloat16()
    w = (torch.randn(N, K, generator=g, device=dev) * K ** -0.5).bfloat16()
    big = {"weight": w, "x": x}.get(what)
    assert big is None or big.numel() * 2 > GIB2
    assert what != "y" or M * N * 2 >= GIB2
    ref = O.linear_bf16(x, w)
    for cfg in _configs(L, M, N, K, 0, M):
        _say(f"case limits plain {what} M={M} N={N} K={K} cfg={cfg}")
        y = ext.mm(x, w, cfg=cfg)
        _check(O, y, ref, f"{what} cfg {cfg}")
        del y
    torch.cuda.synchronize()


def test_rows_far_apart(pkg, O, dev):
    """x rows 7 million elements apart: the 160 rows of the tile that the sizes alone plan span more than a descriptor's
    2^31 bytes, so that it may not be used here. Also as fp32 K planes."""
    lib, check = pkg._lib.lib(), pkg._lib.check
    M, N, K, ldx, S = 300, 16384, 512, 7_000_064, 2
    assert pkg._lib.tile_info(pkg._lib.plan(M, N, K, 0).tile)["bm"] * ldx * 2 > GIB2
    g = torch.Generator(device=dev).manual_seed(5)
    x = torch.empty((M - 1) * ldx + K, dtype=torch.bfloat16, device=dev).as_strided((M, K), (ldx, 1))
    x.copy_(torch.randn(M, K, generator=g, device=dev))
    w = (torch.randn(N, K, generator=g, device=dev) * K ** -0.5).bfloat16()
    y = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    parts = torch.empty(S, M, N, dtype=torch.float32, device=dev)
    ws = torch.empty(max(16, lib.ojx_workspace_bytes(M, N, K, 0, None)), dtype=torch.uint8, device=dev)
    st = torch.cuda.current_stream().cuda_stream
    _say(f"case limits strided M={M} N={N} K={K} ldx={ldx}")
    check(lib.ojx_gemm_bf16(x.data_ptr(), w.data_ptr(), y.data_ptr(), M, N, K, ldx, K, N, ws.data_ptr(), ws.numel(),
                            None, st))
    check(lib.ojx_gemm_splitk_f32(x.data_ptr(), w.data_ptr(), parts.data_ptr(), M, N, K, ldx, K, S, -1, st))
    ref = O.linear_bf16(x.contiguous(), w)
    _check(O, y, ref, "y")
    _check(O, parts.sum(0).bfloat16(), ref, "planes")


@pytest.mark.parametrize("tile", [0, 87, 104])
@pytest.mark.parametrize("M", [1, 3])
def test_absent_rows_wrap_inside_the_operand(pkg, O, dev, M, tile):
    """Row strides at which the offsets of the tile's absent rows (M .. 15 at least) wrap around 2^32 to between the rows
    that exist and, for one row, past its end: those lanes must read nothing there. One case per tile family."""
    lib, check = pkg._lib.lib(), pkg._lib.check
    N, K = 128, 512
    ldx = (1 << 28) + (1 << 19) if M > 1 else (1 << 29) - (1 << 19)   # elements: 8 rows are 2^32 bytes and 8 MiB more / less
    assert any(K * 2 <= m * ldx * 2 % (1 << 32) < ldx * 2 for m in range(M, 16))
    _say(f"case limits absent rows M={M} tile={tile} ldx={ldx}")
    g = torch.Generator(device=dev).manual_seed(6)
    x = torch.empty((M - 1) * ldx + K, dtype=torch.bfloat16, device=dev).as_strided((M, K), (ldx, 1))
    x.copy_(torch.randn(M, K, generator=g, device=dev))
    w = (torch.randn(N, K, generator=g, device=dev) * K ** -0.5).bfloat16()
    y = torch.empty(M, N, dtype=torch.bfloat16, device=dev)
    cfg = pkg._lib.cfg(tile, 1)
    check(lib.ojx_gemm_bf16(x.data_ptr(), w.data_ptr(), y.data_ptr(), M, N, K, ldx, K, N, None, 0, ctypes.byref(cfg),
                            torch.cuda.current_stream().cuda_stream))
    _check(O, y, O.linear_bf16(x.contiguous(), w), "y")


@pytest.mark.parametrize("kind", ["plain", "residual"])
def test_rows_of_millions(pkg, ext, O, dev, kind):
    """Rows of 20 million elements: 64 of them span more than a descriptor's 2^31 bytes, so that the plan takes a tile
    of 32 W rows. (fp32 sums of 2e7 terms of a unit result: random rounding of about 3e-5, below bf16's 4e-3.)"""
    M, N, K = 24, 64, 20_000_000
    _say(f"case limits long rows {kind} M={M} N={N} K={K} plan={pkg._lib.plan(M, N, K, 2 if kind == 'residual' else 0)}")
    g = torch.Generator(device=dev).manual_seed(11)
    x = torch.randn(M, K, generator=g, device=dev, dtype=torch.bfloat16)
    w = torch.randn(N, K, generator=g, device=dev, dtype=torch.bfloat16).mul_(K ** -0.5)
    ref = torch.zeros(M, N, dtype=torch.float64, device=dev)
    for k in range(0, K, 1 << 20):
        ref += (x[:, k:k + (1 << 20)].float() @ w[:, k:k + (1 << 20)].float().t()).double()
    ref = ref.bfloat16()
    if kind == "plain":
        _check(O, ext.mm(x, w), ref, "y")
        return
    res, w1 = torch.randn(M, N, generator=g, device=dev).bfloat16(), torch.ones(N, device=dev)
    h, hn = ext.mm_residual_rmsnorm(res, x, w, w1, None, 1e-6)
    rh, rhn = ext.add_rmsnorm(res, ref, w1, None, 1e-6)
    _check(O, h, rh, "h")
    _check(O, hn, rhn, "hn")


def test_residual_x_past_2gib(pkg, ext, O, dev):
    """The down projection's shape (N = 5120, K = 17408) at M = 65536: x 2.125 GiB, split-K planes past 2 GiB."""
    L = pkg._lib
    M, N, K = 65536, 5120, 17408
    g = torch.Generator(device=dev).manual_seed(7)
    x = torch.randn(M, K, generator=g, device=dev).bfloat16()
    w = (torch.randn(N, K, generator=g, device=dev) * K ** -0.5).bfloat16()
    res = torch.randn(M, N, generator=g, device=dev).bfloat16()
    w1 = (1.0 + 0.1 * torch.randn(N, generator=g, device=dev)).float()
    mask = (torch.rand(M, generator=g, device=dev) > 0.25).int()
    rh, rhn = O.residual_proj(res, x, w, w1, mask, 1e-6)
    for cfg in _configs(L, M, N, K, L.KIND_RESIDUAL, 3):
        _say(f"case limits residual M={M} N={N} K={K} cfg={cfg}")
        h, hn = ext.mm_residual_rmsnorm(res, x, w, w1, mask, 1e-6, cfg=cfg)
        _check(O, h, rh, f"h cfg {cfg}")
        _check(O, hn, rhn, f"hn cfg {cfg}")
        assert int(hn[mask == 0].count_nonzero()) == 0
        del h, hn
    torch.cuda.synchronize()


def test_packed_weight_limit(pkg, ext, dev):
    """ojx_pack_weight refuses a weight of 2 GiB or more (its layout is addressed with 32-bit offsets)."""
    _say("case limits packed weight refused")
    w = torch.empty(65536, 16384, dtype=torch.bfloat16, device=dev)  # exactly 2 GiB, contents not read
    with pytest.raises(RuntimeError, match="2 GiB"):
        ext.pack_weight(w)
