"""GEMMs of few rows or columns (the small-grid plan: tiles of 32 to 256 rows,
whole or split over k with a reduce pass) against an fp32 product."""
import ctypes

import pytest
import torch

from oracle.fp8 import dequantize_rows
from oracle.metrics import assert_close

pytestmark = pytest.mark.gpu


def _randn(shape, dev, seed, std=1.0, dtype=torch.bfloat16):
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    return (torch.randn(shape, generator=g, device=dev) * std).to(dtype)


def _ulp(ref):
    # bf16 output: half an ulp of the largest value, and fp32 summation order
    return 2.0 ** -8 * ref.abs().max().item() + 2e-3


# Rows at the edges of the 32, 64, 128, 192, 224 and 256 row tiles, one k-tile
# and an uneven number of them (65 over 10 or more ranges), partial column
# tiles, three segments split over k (action tokens) and whole.
SHAPES = [(1, 64, 128, 1), (1, 4160, 3072, 1), (32, 3072, 3072, 3), (33, 3072, 3072, 1), (64, 4160, 1536, 1),
          (65, 3072, 3072, 1), (129, 14336, 3072, 1), (193, 3072, 3072, 1), (225, 8960, 1536, 1),
          (400, 3072, 3072, 3), (780, 4160, 3072, 1), (1024, 8960, 1536, 1), (1560, 4160, 3072, 1),
          (2325, 14336, 3072, 1), (40, 3072, 192, 1), (300, 3072, 200, 1), (512, 3072, 3072, 2)]


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
                                   (780, 14336, 3072), (300, 3072, 200)])
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
