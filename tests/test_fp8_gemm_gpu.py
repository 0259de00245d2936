"""GPU parity of the FP8 projection GEMM and the e4m3 quantizer.

* quantizer: bit-exact against the oracle (torch's e4m3fn conversion of
  x / (amax/448)), scales bit-exact.
* GEMM, bf16 output: against the float64 product of the dequantized operands
  (``oracle.fp8_rowcol_gemm``); bar: relative L2 <= 4e-3 and max |err| <=
  1e-2 * max |ref| (bf16 output rounding is 2^-9 relative).
* GEMM, e4m3 output: every element within one e4m3 rounding step (2^-4
  relative, 2^-9 absolute near zero) of the float64 result / out_scale.
"""

import pytest
import torch

from oracle import hstu_oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _fp8():
    from hstu_amd import fp8

    return fp8


@pytest.mark.parametrize("shape,group", [((777, 512), 128), ((64, 4, 128), 128), ((33, 2048), 2048),
                                         ((5, 16), 8)])
def test_quantize_rows_bitexact(hip_lib, shape, group):
    fp8 = _fp8()
    g = torch.Generator().manual_seed(1)
    x = (torch.randn(shape, generator=g) * 3).to(torch.bfloat16)
    x.view(shape[0], -1)[0, :group] = 0  # an all-zero group
    q8, s = fp8.quantize_e4m3_rows(x.to(DEV), group)
    torch.cuda.synchronize()
    R = shape[0]
    xg = x.float().reshape(R, -1, group)
    r8, rs = orc.quantize_e4m3_rows(xg, dim=-1)
    assert torch.equal(s.cpu().reshape(rs.shape), rs), "scales differ"
    assert torch.equal(q8.cpu().view(torch.uint8).reshape(-1), r8.view(torch.uint8).reshape(-1)), "bytes differ"


def test_quantize_with_scale_bitexact(hip_lib):
    fp8 = _fp8()
    x = (torch.randn(300, 512, generator=torch.Generator().manual_seed(2)) * 5).to(torch.bfloat16)
    s = orc.quantize_e4m3_per_tensor(x.float(), margin=1.5)[1]
    out = fp8.quantize_with_scale(x.to(DEV), s.to(DEV))
    torch.cuda.synchronize()
    ref = (x.float() / s).clamp(-448, 448).to(torch.float8_e4m3fn)  # triton_fp8.py:760-781
    assert torch.equal(out.cpu().view(torch.uint8), ref.view(torch.uint8))


def _operands(M, N, K, seed=0, per_row=True, per_col=True):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn(M, K, generator=g)
    w = torch.randn(K, N, generator=g) * 0.05
    a8, sa = orc.quantize_e4m3_rows(a, dim=1) if per_row else orc.quantize_e4m3_per_tensor(a)
    w8t, sw = orc.quantize_e4m3_rows(w.t().contiguous(), dim=1) if per_col else orc.quantize_e4m3_per_tensor(w.t())
    return a8, sa.reshape(-1), w8t.contiguous(), sw.reshape(-1)


@pytest.mark.parametrize("M,N,K", [(1000, 2048, 512), (129, 512, 512), (1, 128, 128), (300, 256, 1536),
                                   (300, 1024, 256), (257, 1024, 2048)])
@pytest.mark.parametrize("scales", ["rowcol", "tensor"])
def test_gemm_bf16(hip_lib, M, N, K, scales):
    fp8 = _fp8()
    a8, sa, w8t, sw = _operands(M, N, K, per_row=scales == "rowcol", per_col=scales == "rowcol")
    bias = (torch.randn(N, generator=torch.Generator().manual_seed(3)) * 0.1).to(torch.bfloat16)
    silu = (0, min(N, 512))
    out = fp8.fp8_gemm(a8.to(DEV), sa.to(DEV), (w8t.to(DEV), sw.to(DEV)), bias=bias.to(DEV), silu_cols=silu)
    torch.cuda.synchronize()
    ref = orc.fp8_rowcol_gemm(a8, sa, w8t.t(), sw, bias=bias.float(), silu_cols=silu)
    got = out.double().cpu()
    err = orc.rel_l2(ref, got)
    mx = float((got - ref).abs().max() / ref.abs().max())
    assert err <= 4e-3 and mx <= 1e-2, f"rel L2 {err:.2e} max {mx:.2e}"


def test_gemm_residual_k1536(hip_lib):
    """The output projection: K=1536, bf16 residual add (k1536_fp8_addmm)."""
    fp8 = _fp8()
    M, N, K = 515, 512, 1536
    a8, sa, w8t, sw = _operands(M, N, K, seed=4)
    res = torch.randn(M, N, generator=torch.Generator().manual_seed(5)).to(torch.bfloat16)
    out = fp8.scaled_addmm_fp8_preq(a8.to(DEV), sa.to(DEV), (w8t.to(DEV), sw.to(DEV)), res.to(DEV))
    torch.cuda.synchronize()
    ref = orc.fp8_rowcol_gemm(a8, sa, w8t.t(), sw, residual=res.float())
    got = out.double().cpu()
    assert orc.rel_l2(ref, got) <= 4e-3
    assert float((got - ref).abs().max() / ref.abs().max()) <= 1e-2


@pytest.mark.parametrize("M", [700, 128 * 14 + 5])
def test_gemm_e4m3_out(hip_lib, M):
    """VQK projection emitting e4m3 at an output scale (scaled_mm_fp8_out_preq),
    in the few-row form (36 wide tiles) and the two-workgroup form (90).

    Bar: every element within one e4m3 half-step (2^-4 relative) of the
    float64 result / out_scale, plus 2.5e-5 * max|result| absolute.  The
    absolute term is the FP8 MFMA accumulation error: measured on this test at
    about 7e-6 * max (the same deviation appears on the bf16 output path), so
    near-zero elements can land one e4m3 step from the float64 rounding."""
    fp8 = _fp8()
    N, K = 1536, 512
    a8, sa, w8t, sw = _operands(M, N, K, seed=6, per_row=False, per_col=False)
    bias = (torch.randn(N, generator=torch.Generator().manual_seed(7)) * 0.1).to(torch.bfloat16)
    ref = orc.fp8_rowcol_gemm(a8, sa, w8t.t(), sw, bias=bias.float())
    out_scale = (ref.abs().max() / 448.0).float().reshape(1)
    out = fp8.scaled_mm_fp8_out_preq(a8.to(DEV), sa.to(DEV), (w8t.to(DEV), sw.to(DEV)), bias.to(DEV),
                                     output_scale=out_scale.to(DEV))
    torch.cuda.synchronize()
    assert out.dtype == torch.float8_e4m3fn
    got = out.cpu().double()
    want = (ref / out_scale.double()).clamp(-448, 448)
    tol = want.abs() * 2.0 ** -4 + 2.5e-5 * 448.0
    worst = float(((got - want).abs() - tol).max())
    assert worst <= 0, f"exceeds the bar by {worst:.3e}"
    # the e4m3 bytes must round-trip: no NaN encodings (saturating clamp)
    assert not torch.isnan(got).any()


def test_gemm_bf16_weight_path(hip_lib):
    """bf16 [K, N] weight quantized per column on the device, as the layer holds it."""
    fp8 = _fp8()
    M, N, K = 256, 2048, 512
    g = torch.Generator().manual_seed(8)
    x = torch.randn(M, K, generator=g).to(torch.bfloat16)
    w = (torch.randn(K, N, generator=g) * 0.05).to(torch.bfloat16)
    x8, sx = fp8.quantize_e4m3_rows(x.to(DEV))
    out = fp8.fp8_gemm(x8, sx, w.to(DEV))
    torch.cuda.synchronize()
    ref = x.double() @ w.double()
    assert orc.rel_l2(ref, out.double().cpu()) <= 6e-2  # two e4m3 quantizations (~2^-4 each, averaged)


@pytest.mark.parametrize("M", [162251, 262144])
def test_gemm_config4_full_size(hip_lib, M):
    """BASELINE config 4 at full size: X [M, 512] e4m3 per-row scales times
    W [512, 2048] e4m3 per-column scales (W stored transposed, [2048, 512]),
    bf16 out with bias and SiLU on the U slice (columns 0-511), M = T of
    config 3 and 262 144.  The whole product runs on the GPU; the float64
    oracle checks 1024 sampled rows (incl. the first and last) to the bf16
    bar of test_gemm_bf16."""
    fp8 = _fp8()
    N, K = 2048, 512
    a8, sa, w8t, sw = _operands(M, N, K, seed=11)
    bias = (torch.randn(N, generator=torch.Generator().manual_seed(12)) * 0.1).to(torch.bfloat16)
    out = fp8.fp8_gemm(a8.to(DEV), sa.to(DEV), (w8t.to(DEV), sw.to(DEV)), bias=bias.to(DEV), silu_cols=(0, 512))
    torch.cuda.synchronize()
    rows = torch.cat([torch.tensor([0, M - 1]),
                      torch.randint(1, M - 1, (1022,), generator=torch.Generator().manual_seed(13))])
    ref = orc.fp8_rowcol_gemm(a8[rows], sa[rows], w8t.t(), sw, bias=bias.float(), silu_cols=(0, 512))
    got = out[rows.to(DEV)].double().cpu()
    err = orc.rel_l2(ref, got)
    mx = float((got - ref).abs().max() / ref.abs().max())
    assert err <= 4e-3 and mx <= 1e-2, f"rel L2 {err:.2e} max {mx:.2e}"


def test_gemm_outproj_config4_full_size(hip_lib):
    """The output projection at config-4 size: [T=162 251, 1536] e4m3 times
    [1536, 512] e4m3 plus a bf16 residual, checked on 1024 sampled rows."""
    fp8 = _fp8()
    M, N, K = 162251, 512, 1536
    a8, sa, w8t, sw = _operands(M, N, K, seed=14)
    res = torch.randn(M, N, generator=torch.Generator().manual_seed(15)).to(torch.bfloat16)
    out = fp8.scaled_addmm_fp8_preq(a8.to(DEV), sa.to(DEV), (w8t.to(DEV), sw.to(DEV)), res.to(DEV))
    torch.cuda.synchronize()
    rows = torch.cat([torch.tensor([0, M - 1]),
                      torch.randint(1, M - 1, (1022,), generator=torch.Generator().manual_seed(16))])
    ref = orc.fp8_rowcol_gemm(a8[rows], sa[rows], w8t.t(), sw, residual=res[rows].float())
    got = out[rows.to(DEV)].double().cpu()
    assert orc.rel_l2(ref, got) <= 4e-3
    assert float((got - ref).abs().max() / ref.abs().max()) <= 1e-2


def test_gemm_proj512_config4_full_size(hip_lib):
    """Config 4's second shape at full size: X [262 144, 512] e4m3 (per-row
    scales) times W [512, 512] e4m3 (per-column scales) with a bf16 bias,
    bf16 out, no SiLU; 1024 sampled rows (incl. the first and last) against
    the float64 oracle, to the bar of test_gemm_bf16."""
    fp8 = _fp8()
    M, N, K = 262144, 512, 512
    a8, sa, w8t, sw = _operands(M, N, K, seed=21)
    bias = (torch.randn(N, generator=torch.Generator().manual_seed(22)) * 0.1).to(torch.bfloat16)
    out = fp8.fp8_gemm(a8.to(DEV), sa.to(DEV), (w8t.to(DEV), sw.to(DEV)), bias=bias.to(DEV))
    torch.cuda.synchronize()
    rows = torch.cat([torch.tensor([0, M - 1]),
                      torch.randint(1, M - 1, (1022,), generator=torch.Generator().manual_seed(23))])
    ref = orc.fp8_rowcol_gemm(a8[rows], sa[rows], w8t.t(), sw, bias=bias.float())
    got = out[rows.to(DEV)].double().cpu()
    assert orc.rel_l2(ref, got) <= 4e-3
    assert float((got - ref).abs().max() / ref.abs().max()) <= 1e-2


@pytest.mark.parametrize("M,N,K", [(162251, 512, 2048), (162251, 1536, 512), (257, 512, 2048)])
def test_dgrad_e5m2_full_size(hip_lib, M, N, K):
    """The FP8 backward's dgrad form (``bwd_fp8.fp8_dgrad``): e5m2 dY [M, K]
    times the e4m3 weight [N, K]^T with per-tensor scales, bf16 out, at the
    layer's shapes (the out-projection dgrad K = 2048 -> 512 and the UVQK
    dgrad K = 512 -> 1536 at config 3's T) and a ragged M; sampled rows
    against the float64 product."""
    from hstu_amd import bwd_fp8

    g = torch.Generator().manual_seed(M + N)
    dy8 = (torch.randn(M, K, generator=g) * 8).to(torch.float8_e5m2)
    w8 = (torch.randn(N, K, generator=g) * 40).clamp(-448, 448).to(torch.float8_e4m3fn)
    sg, sw = torch.tensor([0.02]), torch.tensor([0.003])
    out = bwd_fp8.fp8_dgrad(dy8.to(DEV), sg.to(DEV), w8.to(DEV), sw.to(DEV))
    torch.cuda.synchronize()
    rows = torch.cat([torch.tensor([0, M - 1]),
                      torch.randint(1, M - 1, (min(M, 1024) - 2,), generator=torch.Generator().manual_seed(3))])
    ref = (dy8[rows].double() * 0.02) @ (w8.double() * 0.003).t()
    got = out[rows.to(DEV)].double().cpu()
    assert orc.rel_l2(ref, got) <= 4e-3
    assert float((got - ref).abs().max() / ref.abs().max()) <= 1e-2


def test_gemm_k512_both_kernels(hip_lib):
    """K <= 512 runs the W-stationary kernel when the output rows allow
    16-byte segments and the tile kernel otherwise (row stride N + 4): both
    against the oracle."""
    import hstu_amd._lib as lib

    M, N, K = 777, 384, 512
    a8, sa, w8t, sw = _operands(M, N, K, seed=9)
    bias = (torch.randn(N, generator=torch.Generator().manual_seed(10)) * 0.1).to(torch.bfloat16)
    ref = orc.fp8_rowcol_gemm(a8, sa, w8t.t(), sw, bias=bias.float(), silu_cols=(0, 128))
    A, W, SA, SW, B = (t.to(DEV).contiguous() for t in (a8, w8t, sa, sw, bias))
    gemm = lib.fn("hstu_fp8_gemm_rowcol")
    for ldc in (N, N + 4):
        out = torch.zeros(M, ldc, dtype=torch.bfloat16, device=DEV)
        st = gemm(A.data_ptr(), K, W.data_ptr(), K, SA.data_ptr(), 1, SW.data_ptr(), 1, B.data_ptr(), None, 0,
                  out.data_ptr(), ldc, lib.HSTU_DTYPE_BF16, None, M, N, K, 0, 128,
                  torch.cuda.current_stream().cuda_stream)
        assert st == 0
        torch.cuda.synchronize()
        got = out[:, :N].double().cpu()
        assert orc.rel_l2(ref, got) <= 4e-3, ldc
        assert not bool(out[:, N:].any())                              # nothing written past N


@pytest.mark.parametrize("out8", [False, True])
@pytest.mark.parametrize("M,N", [(777, 512), (128 * 41 + 9, 512), (128 * 81 + 1, 256), (128 * 27 + 77, 768)])
def test_gemm_pc_kernel_bounds(hip_lib, M, N, out8):
    """The wide forms (N % 256, K % 256, 64-aligned SiLU) on a ragged M with a
    padded row stride: every valid element against the oracle, and nothing
    written past N in a row nor past row M (the stores are bounded by buffer
    resources at the tile's valid rows).  14 tiles of 128 x 256 run the few-row
    kernel, 84 and 82 at N <= 512 the producer/consumer kernel, 84 at N = 768 the
    two-workgroup kernel."""
    import hstu_amd._lib as lib

    K = 1024
    a8, sa, w8t, sw = _operands(M, N, K, seed=31)
    bias = (torch.randn(N, generator=torch.Generator().manual_seed(32)) * 0.1).to(torch.bfloat16)
    ref = orc.fp8_rowcol_gemm(a8, sa, w8t.t(), sw, bias=bias.float(), silu_cols=(64, 192))
    A, W, SA, SW, B = (t.to(DEV).contiguous() for t in (a8, w8t, sa, sw, bias))
    os_ = torch.tensor([0.05], device=DEV)
    ldc = N + 16
    out = torch.zeros(M + 200, ldc, dtype=torch.uint8 if out8 else torch.bfloat16, device=DEV)
    st = lib.fn("hstu_fp8_gemm_rowcol")(A.data_ptr(), K, W.data_ptr(), K, SA.data_ptr(), 1, SW.data_ptr(), 1,
                                        B.data_ptr(), None, 0, out.data_ptr(), ldc,
                                        lib.HSTU_DTYPE_FP8_E4M3 if out8 else lib.HSTU_DTYPE_BF16, os_.data_ptr(),
                                        M, N, K, 64, 192, torch.cuda.current_stream().cuda_stream)
    assert st == 0
    torch.cuda.synchronize()
    if out8:  # the bar of test_gemm_e4m3_out, in units of the output scale
        got = out[:M, :N].view(torch.float8_e4m3fn).double().cpu()
        want = (ref / 0.05).clamp(-448, 448)
        tol = want.abs() * 2.0 ** -4 + 2.5e-5 * float(want.abs().max())
        assert float(((got - want).abs() - tol).max()) <= 0
    else:
        got = out[:M, :N].double().cpu()
        assert orc.rel_l2(ref, got) <= 4e-3
    assert not bool(out[:, N:].any()) and not bool(out[M:].any())


@pytest.mark.parametrize("M,N,K,bias,resid,silu", [(1000, 512, 2048, False, False, False),
                                                   (333, 1536, 512, False, False, False),
                                                   (257, 2048, 512, True, False, True),
                                                   (130, 512, 1536, False, True, False)])
def test_bf16_gemm(hip_lib, M, N, K, bias, resid, silu):
    """``hstu_bf16_gemm`` (few-row form at these sizes): against the float64
    product of the same bf16 operands with the same epilogue;
    relative L2 <= 4e-3, max |err| <= 1e-2 * max |ref| (bf16 output)."""
    fp8 = _fp8()
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.randn(M, K, generator=g).to(torch.bfloat16)
    w = (torch.randn(N, K, generator=g) / K ** 0.5).to(torch.bfloat16)
    b = (0.1 * torch.randn(N, generator=g)).to(torch.bfloat16) if bias else None
    r = torch.randn(M, N, generator=g).to(torch.bfloat16) if resid else None
    cols = (N // 4, N // 2) if silu else None
    got = fp8.bf16_gemm(a.to(DEV), w.to(DEV), bias=None if b is None else b.to(DEV),
                        residual=None if r is None else r.to(DEV), silu_cols=cols)
    ref = a.double() @ w.double().t()
    if b is not None:
        ref = ref + b.double()
    if cols is not None:
        ref[:, cols[0]:cols[1]] = torch.nn.functional.silu(ref[:, cols[0]:cols[1]])
    if r is not None:
        ref = ref + r.double()
    got = got.cpu().double()
    assert orc.rel_l2(ref, got) <= 4e-3
    assert float((got - ref).abs().max() / ref.abs().max()) <= 1e-2


def test_bf16_gemm_rows_independent_of_batch(hip_lib):
    """A row's result does not depend on the other rows of the batch: rows of
    a 12 000-row product (two-workgroup form) equal the same rows computed in a
    300-row batch (few-row form)."""
    fp8 = _fp8()
    g = torch.Generator().manual_seed(9)
    a = torch.randn(12000, 2048, generator=g).to(torch.bfloat16).to(DEV)
    w = (torch.randn(512, 2048, generator=g) / 45).to(torch.bfloat16).to(DEV)
    full = fp8.bf16_gemm(a, w)
    part = fp8.bf16_gemm(a[1000:1300], w)
    torch.cuda.synchronize()
    assert torch.equal(full[1000:1300], part)


@pytest.mark.parametrize("M,N,K,resid,pad", [(1, 256, 128, True, 0), (127, 512, 192, False, 0), (129, 256, 320, True, 8),
                                             (385, 768, 128, False, 8), (200, 256, 64, False, 0),
                                             (200, 256, 128, True, 4), (128 * 128 + 1, 256, 128, True, 8),
                                             (128 * 129 + 77, 256, 192, False, 0), (128 * 128 + 65, 256, 320, True, 8),
                                             (128 * 64 + 9, 512, 256, False, 8), (128 * 43 + 127, 768, 128, False, 8),
                                             (128 * 100 + 3, 256, 192, True, 8), (128 * 128 + 1, 256, 64, False, 0)])
def test_bf16_gemm_two_workgroup_form(hip_lib, M, N, K, resid, pad):
    """The bf16 forms at their edges: two, three and more k-steps, ragged last
    row tiles, strided rows.  Up to 385 rows run the few-row form, 101 row tiles
    at N = 256 the tile kernel, the others above 128 row tiles (64 at N = 512, 43
    at N = 768) the two-workgroup form; one k-step and 8-byte aligned output rows
    (``pad`` 4) take the tile kernel.  Against the float64 product: relative L2
    <= 4e-3 (one bf16 rounding of a fp32 sum is 1.7e-3), SiLU on the second 64
    columns, columns outside the output and rows past it untouched."""
    fp8 = _fp8()
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.randn(M, K + 16, generator=g).to(torch.bfloat16)[:, 8:K + 8]
    w = (torch.randn(N, K, generator=g) / K ** 0.5).to(torch.bfloat16)
    b = (0.1 * torch.randn(N, generator=g)).to(torch.bfloat16)
    r = torch.randn(M, N, generator=g).to(torch.bfloat16) if resid else None
    past = torch.full((M + 130, N + pad + 8), 7.0, dtype=torch.bfloat16, device=DEV)
    wide = past[:M]
    ad = torch.empty(M, K + 16, dtype=torch.bfloat16, device=DEV)[:, 8:K + 8]
    ad.copy_(a)
    fp8.bf16_gemm(ad, w.to(DEV), bias=b.to(DEV), residual=None if r is None else r.to(DEV), silu_cols=(64, 128),
                  out=wide[:, :N])
    ref = a.double() @ w.double().t() + b.double()
    ref[:, 64:128] = torch.nn.functional.silu(ref[:, 64:128])
    if r is not None:
        ref = ref + r.double()
    assert orc.rel_l2(ref, wide[:, :N].cpu().double()) <= 4e-3
    assert bool((wide[:, N:] == 7.0).all()) and bool((past[M:] == 7.0).all())


@pytest.mark.parametrize("fmt,N,K,resid,out8", [("bf16", 512, 128, False, False), ("bf16", 512, 1536, True, False),
                                                ("e4m3", 512, 1536, True, False), ("e4m3", 768, 256, False, True),
                                                ("e4m3", 256, 512, True, True), ("e4m3", 2048, 512, False, False),
                                                ("e4m3", 512, 512, False, False), ("e4m3", 256, 1024, False, True),
                                                ("e5m2", 512, 2048, False, False), ("e5m2", 1536, 512, False, False)])
def test_gemm_few_row_form_same_bytes(hip_lib, fmt, N, K, resid, out8):
    """The few-row form gives the bytes of the forms that more rows take (bf16:
    the tile kernel; fp8: the two-workgroup form, at N <= 512 without a residual
    the producer/consumer form): 1, 64, 65 and 300 rows of such a product,
    computed alone, and its last ragged rows."""
    fp8 = _fp8()
    g = torch.Generator().manual_seed(N + K)
    M = 128 * (81 * 256 // N + 1) + 41
    a = torch.randn(M, K, generator=g).to(torch.bfloat16)
    w = torch.randn(N, K, generator=g) / K ** 0.5
    b = None if resid else (0.1 * torch.randn(N, generator=g)).to(torch.bfloat16).to(DEV)
    r = torch.randn(M, N, generator=g).to(torch.bfloat16).to(DEV) if resid else None
    if fmt == "bf16":
        ad, wd = a.to(DEV), w.to(torch.bfloat16).to(DEV)
        run = lambda s: fp8.bf16_gemm(ad[s], wd, bias=b, residual=None if r is None else r[s])  # noqa: E731
    elif fmt == "e5m2":
        from hstu_amd import bwd_fp8

        a8, w8 = (a * 8).to(torch.float8_e5m2).to(DEV), (w * 400).to(torch.float8_e4m3fn).to(DEV)
        sg, sw = torch.tensor([0.02], device=DEV), torch.tensor([0.003], device=DEV)
        run = lambda s: bwd_fp8.fp8_dgrad(a8[s], sg, w8, sw)  # noqa: E731
    else:
        a8, sa = fp8.quantize_e4m3_rows(a.to(DEV))
        wt = fp8.quantize_weight_e4m3(w.to(torch.bfloat16).t().contiguous().to(DEV))
        kw = dict(out_dtype=torch.float8_e4m3fn, out_scale=torch.tensor([0.01], device=DEV)) if out8 else {}
        run = lambda s: fp8.fp8_gemm(a8[s], sa.reshape(-1)[s], wt, bias=b,  # noqa: E731
                                     residual=None if r is None else r[s],
                                     silu_cols=None if out8 else (64, 192), **kw)
    full = run(slice(0, M)).view(torch.uint8)
    for s in (*(slice(200, 200 + rows) for rows in (1, 64, 65, 300)), slice(M - 50, M)):
        assert torch.equal(full[s], run(s).view(torch.uint8)), s


@pytest.mark.parametrize("N,K,resid", [(256, 128, False), (512, 2048, False), (512, 1536, True), (768, 192, True)])
@pytest.mark.parametrize("kind", ["randn", "cancel"])
def test_bf16_gemm_forms_same_bytes(hip_lib, N, K, resid, kind):
    """The three bf16 forms give a row the same bytes: a product of 128 x 128
    tiles for more than one round of the chip (two-workgroup form), its rows in
    batches of at most one round (tile kernel) and of a few tiles (few-row
    form), and all of it with 8-byte aligned output rows (tile kernel).
    ``cancel``: sums that cancel, so that the result is their rounding."""
    fp8 = _fp8()
    g = torch.Generator().manual_seed(N + K)
    M = 128 * (256 * 128 // N + 2) + 9
    a = torch.randn(M, K, generator=g).to(torch.bfloat16)
    w = (torch.randn(N, K, generator=g) / K ** 0.5).to(torch.bfloat16)
    if kind == "cancel":
        perm = torch.randperm(K // 2, generator=g)
        a[:, K // 2:] = a[:, :K // 2][:, perm]
        w[:, K // 2:] = -w[:, :K // 2][:, perm]
    a, w = a.to(DEV), w.to(DEV)
    b = None if kind == "cancel" else (0.1 * torch.randn(N, generator=g)).to(torch.bfloat16).to(DEV)
    r = torch.randn(M, N, generator=g).to(torch.bfloat16).to(DEV) if resid and kind != "cancel" else None
    run = lambda x, y, out=None: fp8.bf16_gemm(x, w, bias=b, residual=y, silu_cols=(64, 128), out=out)  # noqa: E731
    full = run(a, r).view(torch.int16)
    for step in (128 * (128 * 256 // N) - 7, 128 * (60 * 256 // N)):  # at most 256 tiles; 60 wide ones
        got = torch.cat([run(a[i:i + step], None if r is None else r[i:i + step]) for i in range(0, M, step)])
        assert torch.equal(full, got.view(torch.int16)), step
    wide = torch.empty(M, N + 4, dtype=torch.bfloat16, device=DEV)
    run(a, r, out=wide[:, :N])
    assert torch.equal(full, wide[:, :N].contiguous().view(torch.int16))
