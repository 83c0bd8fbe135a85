"""The LDS-staged prefill kernels at the edges of what they take: int4 groups of 32 and 64 (four
16x16x32 MFMAs per K tile, weights decoded as e4m3(q - z)), zero points with groups of 128, a K that
ends inside a 128-wide tile, and one or two K tiles; dense and grouped, against the CPU oracle."""
import numpy as np
import pytest
import torch

import synth
from conftest import pkg
from test_gpu_dense import _row_major_gemm, assert_close_to_oracle
from test_gpu_moe import _stagewise

pytestmark = pytest.mark.gpu


def _weight(fmt, g, N, K, seed, E=None):
    """(w, s, z, e2m1, nvfp4) on the CPU, op layout."""
    if fmt == "mxfp4":
        return (*synth.mxfp4_weight(N, K, seed=seed, E=E), None, True, False)
    if fmt == "nvfp4":
        return (*synth.nvfp4_weight(N, K, seed=seed, E=E), True, True)
    return (*synth.int4_weight(N, K, g, seed=seed, asym=fmt == "asym", scale_floor=1e-4, E=E), False, False)


def _call(fmt):
    """(scale_fmt, has_zeros, wfmt) of a format, as the C ABI's planning calls take them."""
    return {"sym": (0, 0, 0), "asym": (0, 1, 0), "mxfp4": (1, 0, 1), "nvfp4": (2, 1, 1)}[fmt]


def _tile(fmt, g, M, N, K, silu=False, operand_order=False):
    """The (rows, columns) of the dense tile that a call runs on."""
    t = pkg("_abi").load().w4a8_probe_prefill_tile(M, N, K, *_call(fmt), g, int(silu), int(operand_order))
    return t >> 16, t & 0xFFFF


def _operand_order(fmt, g, M, N, K, silu=False):
    """Whether w4a8_linear takes the call's activations in operand order (it asks for the room)."""
    row_major = (M * K + 255) // 256 * 256 + (M * 4 + 255) // 256 * 256
    return pkg("_abi").load().w4a8_linear_workspace_bytes_for(M, N, K, *_call(fmt), g, int(silu), 2) > row_major


FMTS = [("sym", 32), ("asym", 32), ("sym", 64), ("asym", 64), ("asym", 128), ("asym", 256), ("mxfp4", 32), ("nvfp4", 16)]


# K: one tile, two, a tail of 32 to 96 behind one and three tiles, more tiles than the K loop unrolls;
# M and N: one row block and strip past a tile's edge, row tiles of 64, 128 and 256
@pytest.mark.parametrize("fmt,g", FMTS)
@pytest.mark.parametrize("M,N,K", [(17, 16, 128), (65, 144, 256), (130, 272, 160), (40, 1040, 480), (300, 528, 1088),
                                   (257, 4112, 896)])
def test_prefill_groups_and_k_tails(kernels, oracle, dev, fmt, g, M, N, K):
    if K % g:
        pytest.skip("group does not divide K")
    w, s, z, e2, nv = _weight(fmt, g, N, K, seed=M + N + K)
    # no x50 outlier channel: the MFMA aligns its products to the largest one and drops what falls below
    # about 2^-24 of it, so with one product 50 times the rest the distance grows 5 to 7 times (MXFP4 at
    # M=40 N=1040 K=480: 5.3e-4 against 7.5e-5, the same bits from the decode kernel), past the bar that
    # assert_close_to_oracle derives for sums of like terms
    x = synth.activations(M, K, seed=M + K)
    xq, xs = oracle.act_quant(synth.bits16(x), 0)
    ref = oracle.gemm(xq, xs, w.numpy(), s.view(torch.uint8).numpy() if nv else s.numpy(),
                      None if z is None else z.numpy(), g, e2, nv)
    tiles, sd = kernels.repack_w4(w.to(dev), weight_is_e2m1=e2), s.to(dev)
    zd = None if z is None else z.to(dev)
    out = kernels.w4a8_linear(x.to(dev), tiles, sd, zd, g, weight_is_e2m1=e2, kernel="wmma_tiled_tuned")
    rows = torch.tensor([0, M // 2, M - 1])  # the same rows in a smaller call, and beside a row of NaN
    xp = torch.cat([x[rows], torch.full((1, K), float("nan"), dtype=x.dtype)])
    part = kernels.w4a8_linear(xp.to(dev), tiles, sd, zd, g, weight_is_e2m1=e2, kernel="wmma_tiled_tuned")
    torch.cuda.synchronize()
    assert_close_to_oracle(out, ref, f"{fmt} g={g} M={M} N={N} K={K}")
    assert torch.equal(out[rows.to(dev)], part[:3]), "a row's bits depend on the rows beside it"


@pytest.mark.parametrize("fmt,g", FMTS)
@pytest.mark.parametrize("h,i,bm", [(320, 96, 64), (256, 160, 128)])
def test_moe_groups_and_k_tails(kernels, oracle, dev, fmt, g, h, i, bm):
    """Grouped tiles of 64 and 128 rows, both GEMMs with a ragged K (h = 320 and i = 96, 160)."""
    if h % g or i % g:
        g = max(d for d in (16, 32) if d <= g)
        if fmt == "asym" and g == 16:
            g = 32
    e, T = 4, 150
    w13, s13, z13, e2, nv = _weight(fmt, g, 2 * i, h, seed=h + i, E=e)
    w2, s2, z2, _, _ = _weight(fmt, g, h, i, seed=h + i + 1, E=e)
    x = synth.activations(T, h, seed=7)
    lg = synth.router_logits(T, e, seed=8)
    zz = [None if z is None else (z.view(torch.int32) if nv else z).to(dev) for z in (z13, z2)]
    res = kernels._moe_forward(x.to(dev), kernels.repack_w4(w13.to(dev), e2), s13.to(dev), zz[0],
                               kernels.repack_w4(w2.to(dev), e2), s2.to(dev), zz[1], lg.to(dev), 2, True,
                               weight_is_e2m1=e2, block_m=bm)
    torch.cuda.synchronize()
    u8 = (lambda t: t.view(torch.uint8)) if nv else (lambda t: t)
    rel1, rel2, _ = _stagewise(kernels, oracle, res, x, w13, u8(s13), z13, w2, u8(s2), z2, list(range(0, T, 5)),
                               e2m1=e2, nvfp4=nv)
    assert rel1 <= 2e-3 and rel2 <= 2e-3  # the bars of test_gpu_moe: bf16 rounding alone is 1.65e-3
    assert np.isfinite(res["out"].float().cpu().numpy()).all()


# one row past 64, 128, 192 and 256 rows, and sizes that take each dense tile shape of row-major int4 and of
# MXFP4 (NVFP4 has int4's)
@pytest.mark.parametrize("fmt,g", [("sym", 128), ("asym", 32), ("mxfp4", 32), ("nvfp4", 16)])
@pytest.mark.parametrize("M,N,int4,mxfp4", [(65, 80, (64, 64), (64, 64)), (129, 8208, (64, 128), (64, 128)),
                                            (193, 12304, (128, 128), (128, 128)), (321, 14352, (192, 128), (192, 128)),
                                            (391, 14320, (256, 128), (128, 256)), (577, 16400, (128, 128), (256, 256)),
                                            (1153, 8208, (192, 128), (192, 256))])
def test_dense_tile_shapes(kernels, oracle, dev, fmt, g, M, N, int4, mxfp4):
    """Every tile shape gives a row the same bits: the call's rows against the same rows in calls of
    seven, and those against the oracle."""
    K = 384
    assert fmt == "nvfp4" or _tile(fmt, g, M, N, K) == (mxfp4 if fmt == "mxfp4" else int4)
    w, s, z, e2, nv = _weight(fmt, g, N, K, seed=M + N)
    x = synth.activations(M, K, seed=M + 1)
    tiles, sd = kernels.repack_w4(w.to(dev), weight_is_e2m1=e2), s.to(dev)
    zd = None if z is None else z.to(dev)
    rows = torch.tensor(sorted({0, 15, 63, 64, M // 2, M - 2, M - 1}))
    out, part = (kernels.w4a8_linear(t.to(dev), tiles, sd, zd, g, weight_is_e2m1=e2, kernel="wmma_tiled_tuned")
                 for t in (x, x[rows].contiguous()))
    torch.cuda.synchronize()
    assert torch.equal(out[rows.to(dev)], part), f"{fmt} M={M} N={N}: a row's bits depend on the tile"
    xq, xs = oracle.act_quant(synth.bits16(x[rows]), 0)
    ref = oracle.gemm(xq, xs, w.numpy(), s.view(torch.uint8).numpy() if nv else s.numpy(),
                      None if z is None else z.numpy(), g, e2, nv)
    assert_close_to_oracle(part, ref, f"{fmt} M={M} N={N}")


@pytest.mark.parametrize("M,N,K,silu", [(4096, 4096, 384, False), (4090, 4080, 512, False), (4093, 4096, 640, True),
                                        (7900, 2048, 1152, True), (3841, 4096, 4224, False)])
@pytest.mark.parametrize("asym,g", [(False, 128), (True, 128), (True, 256)])
def test_wide_tile_matches_the_others(kernels, dev, M, N, K, silu, asym, g):
    """256 x 256 tiles (activations in operand order, grids that one round of them fills): 3 to 33 K
    tiles, ragged rows and strips and the silu arm, bit for bit against the row-major kernel (w4a8_gemm
    without a workspace) on the same codes."""
    if K % g:
        pytest.skip("group does not divide K")
    fmt = "asym" if asym else "sym"
    assert _operand_order(fmt, g, M, N, K, silu) and _tile(fmt, g, M, N, K, silu, True) == (256, 256)
    abi = pkg("_abi")
    lib = abi.load()
    w, s, z = synth.int4_weight(N, K, g, seed=N + K, asym=asym, scale_floor=1e-4)
    tiles, sd, zd = kernels.repack_w4(w.to(dev)), s.to(dev), None if z is None else z.to(dev)
    x = synth.activations(M, K, seed=M).to(dev)
    q, sc = kernels.act_quant(x)
    nout = N // 2 if silu else N
    out, ref = (torch.empty((M, nout), dtype=x.dtype, device=dev) for _ in range(2))
    wsb = lib.w4a8_linear_workspace_bytes(M, K)
    ws = torch.empty(wsb, dtype=torch.uint8, device=dev)
    abi.check(lib.w4a8_linear(abi.ptr(x), abi.BF16, M, K, K, abi.ptr(tiles), N, abi.ptr(sd), abi.SCALE_F16,
                              abi.ptr(zd), abi.W_INT4, g, abi.ptr(out), abi.BF16, nout, int(silu), abi.ptr(ws), wsb,
                              abi.KERNEL_PREFILL, abi.stream_of(x)), "w4a8_linear")
    abi.check(lib.w4a8_gemm(abi.ptr(q), K, abi.ptr(sc), M, abi.ptr(tiles), N, K, abi.ptr(sd), abi.SCALE_F16,
                            abi.ptr(zd), abi.W_INT4, g, abi.ptr(ref), abi.BF16, nout, int(silu), None, 0, abi.KERNEL_PREFILL,
                            abi.stream_of(x)), "w4a8_gemm")
    torch.cuda.synchronize()
    assert torch.equal(out, ref), f"max {(out.float() - ref.float()).abs().max().item():.3e}"


# zero points take it at such K through the 256 x 256 tile only, so on the wider weight
@pytest.mark.parametrize("fmt,N", [("asym", 13056), ("mxfp4", 2048)])
@pytest.mark.parametrize("M,K", [(1024, 4224), (1037, 8192), (1026, 8320), (1100, 16384), (1030, 16512)])
def test_long_rows_quantized_in_operand_order(kernels, dev, fmt, N, M, K):
    """Rows of more than 4096 elements on formats without seeds: four rows per workgroup up to 16384
    elements (one and two chunks per thread, ragged row blocks), two passes beyond on more than 1024 rows,
    bit for bit against the row-major quant and GEMM."""
    assert _operand_order(fmt, 32 if fmt == "mxfp4" else 128, M, N, K)
    abi = pkg("_abi")
    lib = abi.load()
    w, s, z, e2, _ = _weight(fmt, 128, N, K, seed=K)
    tiles, sd, zd = kernels.repack_w4(w.to(dev), e2), s.to(dev), None if z is None else z.to(dev)
    x = synth.activations(M, K, seed=M, outliers=True).to(dev)
    x[3] = 0
    q, sc = kernels.act_quant(x)
    out = kernels.w4a8_linear(x, tiles, sd, zd, 32 if e2 else 128, weight_is_e2m1=e2)
    ref = torch.empty_like(out)
    abi.check(lib.w4a8_gemm(abi.ptr(q), K, abi.ptr(sc), M, abi.ptr(tiles), N, K, abi.ptr(sd),
                            abi.SCALE_E8M0 if e2 else abi.SCALE_F16, abi.ptr(zd), abi.W_E2M1 if e2 else abi.W_INT4,
                            32 if e2 else 128, abi.ptr(ref), abi.BF16, N, 0, None, 0, abi.KERNEL_PREFILL,
                            abi.stream_of(x)), "w4a8_gemm")
    torch.cuda.synchronize()
    assert torch.equal(out, ref)


# below 1024 rows: int4 where 256 x 256 tiles fit the grid (one quant kernel each side of K = 4096),
# MXFP4 from 128 rows up to K = 32768 (three and four chunks per thread), and one row or K tile outside each
@pytest.mark.parametrize("fmt,M,N,K,takes", [
    ("sym", 448, 28672, 512, True), ("sym", 511, 24576, 4224, True), ("asym", 500, 28672, 384, True),
    ("asym", 1023, 14336, 4224, True), ("mxfp4", 127, 2048, 384, False), ("mxfp4", 128, 2048, 384, True),
    ("mxfp4", 129, 2064, 4224, True), ("mxfp4", 1023, 2048, 16384, True), ("mxfp4", 200, 2048, 16512, True),
    ("mxfp4", 130, 2032, 512, False), ("mxfp4", 1023, 2048, 24576, True), ("mxfp4", 131, 2048, 24704, True),
    ("mxfp4", 1024, 2048, 32768, True), ("mxfp4", 1025, 2048, 28672, True), ("mxfp4", 200, 2048, 32896, False)])
def test_few_rows_in_operand_order(kernels, dev, fmt, M, N, K, takes):
    w, s, z, e2, _ = _weight(fmt, 128, N, K, seed=M + K)
    g = 32 if e2 else 128
    assert _operand_order(fmt, g, M, N, K) == takes
    tiles, sd, zd = kernels.repack_w4(w.to(dev), e2), s.to(dev), None if z is None else z.to(dev)
    x = synth.activations(M, K, seed=M, outliers=True).to(dev)
    q, sc = kernels.act_quant(x)
    out = kernels.w4a8_linear(x, tiles, sd, zd, g, weight_is_e2m1=e2)
    ref = _row_major_gemm(q, sc, tiles, sd, zd, g, N, K, e2, x.dtype)
    torch.cuda.synchronize()
    assert torch.equal(out, ref)


@pytest.mark.parametrize("fmt", ["sym", "asym", "mxfp4"])
@pytest.mark.parametrize("M,K", [(1024, 384), (1900, 640)])  # grids of the 256 x 256 tile: zero points rewrite there only
def test_pair_rewrite_computes_seeds_where_they_are_read(kernels, dev, fmt, M, K):
    """The producer pair's codes rewritten in operand order: the workspace's row-sum seeds are written for
    symmetric int4 and left alone for the formats that read none; the outputs are the row-major GEMM's."""
    N, g = 16384, 32 if fmt == "mxfp4" else 128
    abi = pkg("_abi")
    lib = abi.load()
    w, s, z, e2, _ = _weight(fmt, 128, N, K, seed=M + K)
    tiles, sd, zd = kernels.repack_w4(w.to(dev), e2), s.to(dev), None if z is None else z.to(dev)
    x = synth.activations(M, K, seed=M).to(dev)
    q, sc = kernels.act_quant(x)
    wsb = lib.w4a8_gemm_workspace_bytes(M, N, K, abi.KERNEL_PREFILL)
    ws = torch.full((wsb,), 0xA5, dtype=torch.uint8, device=dev)
    out = torch.empty((M, N), dtype=x.dtype, device=dev)
    abi.check(lib.w4a8_gemm(abi.ptr(q), K, abi.ptr(sc), M, abi.ptr(tiles), N, K, abi.ptr(sd),
                            abi.SCALE_E8M0 if e2 else abi.SCALE_F16, abi.ptr(zd), abi.W_E2M1 if e2 else abi.W_INT4, g,
                            abi.ptr(out), abi.BF16, N, 0, abi.ptr(ws), wsb, abi.KERNEL_PREFILL, abi.stream_of(x)), "w4a8_gemm")
    ref = _row_major_gemm(q, sc, tiles, sd, zd, g, N, K, e2, x.dtype)
    torch.cuda.synchronize()
    assert torch.equal(out, ref)
    Mp = (M + 15) // 16 * 16
    seeds = ws[(Mp * K + 255) // 256 * 256:][:K // 128 * Mp * 4]
    assert not bool((ws[:Mp * K] == 0xA5).all()) and bool((seeds == 0xA5).all()) == (fmt != "sym")
