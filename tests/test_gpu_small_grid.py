"""GEMMs of few rows or columns (the small-grid plan: tiles of 32 to 256 rows,
whole or split over k with a reduce pass) against an fp32 product."""
import ctypes

import pytest
import torch

from oracle.fp8 import dequantize_mx32, dequantize_rows, quantize_mx32
from oracle.metrics import assert_close

pytestmark = pytest.mark.gpu


def _randn(shape, dev, seed, std=1.0, dtype=torch.bfloat16):
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    return (torch.randn(shape, generator=g, device=dev) * std).to(dtype)


def _ulp(ref):
    # bf16 output: half an ulp of the largest value, and fp32 summation order
    return 2.0 ** -8 * ref.abs().max().item() + 2e-3


# Rows at the edges of the tiles (32 to 256 rows, 128 or 256 columns), one k-tile
# and an uneven number of them (65 over 10 or more ranges), partial column
# tiles, three segments split over k (action tokens) and whole.
SHAPES = [(1, 64, 128, 1), (1, 4160, 3072, 1), (32, 3072, 3072, 3), (33, 3072, 3072, 1), (64, 4160, 1536, 1),
          (65, 3072, 3072, 1), (129, 14336, 3072, 1), (193, 3072, 3072, 1), (225, 8960, 1536, 1),
          (400, 3072, 3072, 3), (780, 4160, 3072, 1), (1024, 8960, 1536, 1), (1560, 4160, 3072, 1),
          (2325, 14336, 3072, 1), (2325, 3072, 3072, 1), (1000, 1536, 8960, 1), (1300, 14336, 3072, 1),
          (1921, 3072, 3072, 1), (3001, 3072, 3072, 1), (64, 3072, 14336, 1), (50, 3072, 8968, 1), (129, 3072, 3072, 1),
          (40, 3072, 192, 1), (300, 3072, 200, 1), (512, 3072, 3072, 2)]


@pytest.mark.parametrize("M,K,N,nseg", SHAPES)
def test_bias_and_gelu(dev, M, K, N, nseg):
    from wam_ops import ops
    x = _randn((M, K), dev, 1)
    ws = [_randn((N, K), dev, 2 + i, 0.02) for i in range(nseg)]
    bs = [_randn((N,), dev, 9 + i, 0.5) for i in range(nseg)]
    outs = ops.linear(x, ws, bs)
    for i in range(nseg):
        ref = x.float() @ ws[i].float().t() + bs[i].float()
        assert_close(outs[i], ref, _ulp(ref), 0.99999, f"segment {i} of {M}x{K}x{N}")
    ref = torch.nn.functional.gelu(x.float() @ ws[0].float().t(), approximate="tanh")
    y = ops.linear(x, ws[0], None, epilogue=ops.EPI_BIAS_GELU)
    assert_close(y, ref, _ulp(ref), 0.99999, f"gelu, no bias, {M}x{K}x{N}")


@pytest.mark.parametrize("M,K,N", [(1, 4160, 3072), (33, 3072, 3072), (224, 14336, 3072), (400, 4160, 3072),
                                   (780, 14336, 3072), (300, 3072, 200), (2325, 3072, 3072), (3001, 3072, 3072)])
@pytest.mark.parametrize("fp32", [False, True])
def test_residuals(dev, M, K, N, fp32):
    from wam_ops import ops
    x, w, b = _randn((M, K), dev, 1), _randn((N, K), dev, 2, 0.02), _randn((N,), dev, 3)
    dt = torch.float32 if fp32 else torch.bfloat16
    res = _randn((M, N), dev, 4, 1.0, dt)
    lin = x.float() @ w.float().t() + b.float()
    bound = (lambda r: 1e-3) if fp32 else _ulp
    y = ops.linear(x, w, b, epilogue=ops.EPI_BIAS_RES, residual=res, out_dtype=dt)
    assert_close(y, res.float() + lin, bound(res.float() + lin), 0.99999, f"residual {M}x{K}x{N}")
    table, temb = _randn((1, 6, N), dev, 5, 0.3, torch.float32), _randn((1, M, 6, N), dev, 6, 0.3)
    ref = res.float() + lin * (table[:, 2] + temb[0, :, 2].float())
    y = ops.linear(x, w, b, epilogue=ops.EPI_BIAS_GATE_RES, residual=res, table=table, temb=temb, tokens=M,
                   gate_index=2, out_dtype=dt)
    assert_close(y, ref, bound(ref), 0.99999, f"gated residual {M}x{K}x{N}")


@pytest.mark.parametrize("M,K,N", [(1, 3072, 14336), (65, 14336, 3072), (224, 4160, 3072), (780, 14336, 3072)])
def test_fp8_weights(dev, M, K, N):
    from wam_ops import ops
    x, w, b = _randn((M, K), dev, 1), _randn((N, K), dev, 2, 0.02), _randn((N,), dev, 3)
    q, sc = ops.quantize_fp8_rows(w)
    ref = x.float() @ dequantize_rows(q.cpu(), sc.cpu()).to(dev).t() + b.float()
    assert_close(ops.linear(x, q, b, w_scale=sc), ref, _ulp(ref), 0.99999, f"fp8 weights {M}x{K}x{N}")


def test_without_and_with_a_small_workspace(dev):
    """No workspace runs one k range; one too small for the plan's ranges
    runs fewer."""
    from wam_ops import _lib
    M, K, N = 40, 8192, 3072
    x, w = _randn((M, K), dev, 1), _randn((N, K), dev, 2, 0.02)
    ref = x.float() @ w.float().t()
    h = _lib.lib()
    full = h.wam_linear_workspace_bytes(M, N, 1, K)
    assert full > 2 * M * N * 4
    ws = torch.empty(full, dtype=torch.uint8, device=dev)
    for nbytes in (0, 2 * M * N * 4, full - 1, full):
        out = torch.zeros(M, N, dtype=torch.bfloat16, device=dev)
        a = _lib.LinearArgs()
        a.a, a.lda, a.M, a.K, a.n_seg, a.seg_n, a.ldw, a.ldo = x.data_ptr(), K, M, K, 1, N, K, N
        a.w[0], a.out[0] = w.data_ptr(), out.data_ptr()
        a.workspace, a.workspace_bytes = (ws.data_ptr() if nbytes else None), nbytes
        _lib.check(h.wam_linear(ctypes.byref(a), None), "wam_linear")
        torch.cuda.synchronize()
        assert_close(out, ref, _ulp(ref), 0.99999, f"workspace of {nbytes} bytes")


# fp8 activations: 128-row tiles (up to 128 rows in one, 129 in two), 224-row
# ones (780 x 3072 x 14336), one k-tile, nine over the ranges, and whole k with
# 128-row tiles (2325); without a workspace one range, with one the plan's.
@pytest.mark.parametrize("M,K,N", [(1, 128, 256), (32, 3072, 14336), (128, 14336, 3072), (129, 14336, 3072),
                                   (225, 1152, 512), (780, 3072, 14336), (780, 14336, 3072), (2325, 14336, 3072)])
@pytest.mark.parametrize("room", [False, True])
def test_fp8_activations(dev, M, K, N, room):
    from wam_ops import _lib, ops
    x, w, b = _randn((M, K), dev, 1), _randn((N, K), dev, 2, 0.02), _randn((N,), dev, 3)
    qw, sw = ops.quantize_fp8_rows(w)
    wd = dequantize_rows(qw.cpu(), sw.cpu()).to(dev).t()
    ws = torch.empty(32 * M * N * 4 if room else 1, dtype=torch.uint8, device=dev)

    def run(q, out, epi, **kw):
        a = _lib.LinearArgs()
        a.a, a.lda, a.M, a.K, a.n_seg, a.seg_n, a.ldw, a.ldo = q.data_ptr(), K, M, K, 1, N, K, N
        a.w[0], a.out[0], a.bias[0], a.w_dtype, a.w_scale[0] = qw.data_ptr(), out.data_ptr(), b.data_ptr(), _lib.WAM_FP8, sw.data_ptr()
        a.epilogue, a.a_dtype = epi, _lib.WAM_FP8
        for k, v in kw.items():
            setattr(a, k, v)
        if room:
            a.workspace, a.workspace_bytes = ws.data_ptr(), ws.numel()
        _lib.check(_lib.lib().wam_linear(ctypes.byref(a), None), "wam_linear")
        torch.cuda.synchronize()
        return out

    q, sx = ops.quantize_fp8_rows(x)
    ref = dequantize_rows(q.cpu(), sx.cpu()).to(dev) @ wd + b.float()
    y = run(q, torch.zeros(M, N, dtype=torch.bfloat16, device=dev), ops.EPI_BIAS, a_scale=sx.data_ptr())
    assert_close(y, ref, _ulp(ref), 0.99999, f"fp8 rows, bias {M}x{K}x{N}")
    gelu = torch.nn.functional.gelu(ref, approximate="tanh")
    e = torch.zeros(M, N // 32, dtype=torch.uint8, device=dev)
    y = run(q, torch.zeros(M, N, dtype=torch.float8_e4m3fn, device=dev), ops.EPI_BIAS_GELU, a_scale=sx.data_ptr(),
            out_dtype=_lib.WAM_FP8_MX, out_block_scale=e.data_ptr())
    d = dequantize_mx32(y.cpu(), e.cpu()).to(dev)
    # half an e4m3 step (2^-4 of the value, 2^-10 of a subnormal's block scale) and fp32 summation order
    step = torch.maximum(gelu.abs() * 2.0 ** -4, torch.exp2(e.float() - 137).repeat_interleave(32, 1))
    assert ((d - gelu).abs() <= step + 2e-3).all()
    q, ex = quantize_mx32(x.float().cpu())
    ref = dequantize_mx32(q, ex).to(dev) @ wd + b.float()
    q, ex = q.to(dev), ex.to(dev)
    res = _randn((M, N), dev, 4, 1.0, torch.float32)
    table, temb = _randn((1, 6, N), dev, 5, 0.3, torch.float32), _randn((1, M, 6, N), dev, 6, 0.3)
    ref = res + ref * (table[:, 5] + temb[0, :, 5].float())
    y = run(q, torch.zeros(M, N, device=dev), ops.EPI_BIAS_GATE_RES, a_dtype=_lib.WAM_FP8_MX, a_block_scale=ex.data_ptr(),
            res=res.data_ptr(), ldr=N, res_dtype=_lib.WAM_F32, out_dtype=_lib.WAM_F32,
            gate=ops.modulation(table, temb, M), gate_index=5)
    assert_close(y, ref, 2e-3, 0.99999, f"MX gated residual {M}x{K}x{N}")
