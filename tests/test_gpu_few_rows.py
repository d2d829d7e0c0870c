"""The block's row passes over few rows (split_rows.hip): LayerNorm with a
workgroup per row, and the passes that take a split projection's partial sums,
through the block, against float64 / the oracle."""
import pytest
import torch

from oracle.block import block_forward
from oracle.metrics import assert_close

pytestmark = pytest.mark.gpu


def _randn(shape, dev, seed, std=1.0, dtype=torch.float32):
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    return (torch.randn(shape, generator=g, device=dev) * std).to(dtype)


# Column counts with one to four chunks per thread and partial ones; the last
# few-row count and the first of the wave-per-row kernel; per-token rows beyond.
@pytest.mark.parametrize("rows,D", [(1, 8), (3, 1000), (400, 1024), (401, 1032), (7, 2048), (32, 3072), (5, 4096), (900, 3072)])
@pytest.mark.parametrize("x32,t16,per_token", [(True, False, False), (False, True, True), (True, False, True)])
def test_layer_norm(dev, rows, D, x32, t16, per_token):
    from wam_ops import ops
    x = _randn((1, rows, D), dev, 1, 2.0, torch.float32 if x32 else torch.bfloat16)
    table = _randn((1, 6, D), dev, 2, 0.3)
    temb = _randn((1, rows if per_token else 1, 6, D), dev, 3, 0.3, torch.bfloat16 if t16 else torch.float32)
    xd = x.double()
    ln = (xd - xd.mean(-1, keepdim=True)) * torch.rsqrt(xd.var(-1, unbiased=False, keepdim=True) + 1e-6)
    ref = ln * (1 + (table[:, 4] + temb[:, :, 4].float()).double()) + (table[:, 3] + temb[:, :, 3].float()).double()
    # half an ulp of the largest value, and fp32 statistics
    bound = 2.0 ** -8 * ref.abs().max().item() + 1e-4
    y, q, sc = ops.ln_modulate(x, table, temb, 3, fp8=True)
    assert_close(y, ref.float(), bound, 0.9999 if D > 8 else 0.99, f"modulated LayerNorm {rows}x{D}")
    if D % 8 == 0:
        rq, rs = ops.quantize_fp8_rows(y.reshape(rows, D))
        assert torch.equal(q.reshape(rows, D).view(torch.uint8), rq.view(torch.uint8)) and torch.equal(sc, rs)
    g, b = _randn((D,), dev, 4, 0.2), _randn((D,), dev, 5, 0.2)
    ref = ln * (g + 1).double() + b.double()
    bound = 2.0 ** -8 * ref.abs().max().item() + 1e-4
    assert_close(ops.layer_norm_affine(x, g + 1, b), ref.float(), bound, 0.9999 if D > 8 else 0.99, f"affine {rows}x{D}")


# Every projection split (16 and 2 x 16 rows), some of them (2 x 65, 2 x 128
# rows of the wide block) and a width of three head pairs; without norm2 (the
# residual is not normalised there), per token and per frame.
@pytest.mark.parametrize("dim,ffn,B,grid,temb_len,norm2", [
    (3072, 14336, 2, (2, 8, 1), 2, True), (3072, 14336, 1, (1, 4, 4), 16, True), (3072, 14336, 2, (1, 8, 16), 1, True),
    (3072, 14336, 2, (1, 5, 13), 1, False), (768, 1536, 3, (1, 3, 3), 9, True), (1536, 8960, 1, (2, 3, 4), 2, True)])
def test_block_of_few_rows(dev, dim, ffn, B, grid, temb_len, norm2):
    from wam_ops import synthetic
    from wam_ops.block import TransformerBlock
    from wam_ops.native import NativeBlock
    shape = synthetic.BlockShape(dim, dim // 128, ffn, cross_attn_norm=norm2)
    params = synthetic.block_params(shape, seed=3, device=dev)
    M = grid[0] * grid[1] * grid[2]
    x, ctx, _, freqs = synthetic.block_inputs(shape, B, M, grid, context_len=40, context_batch=B, seed=4, device=dev)
    temb = _randn((B, temb_len, 6, dim), dev, 5, 0.1)
    with torch.device("meta"):
        blk = TransformerBlock(dim, ffn, dim // 128, cross_attn_norm=norm2)
    blk.load_state_dict(params, assign=True)
    with torch.no_grad():
        out = blk(x, ctx, temb, freqs)
        again = blk(x, ctx, temb, freqs)
        dbg = NativeBlock(blk)(x, ctx, temb, freqs, debug=True)
    assert torch.equal(out, again), "two calls differ"
    assert torch.equal(dbg["output"], out), "a debug call changed the block output"
    cpu = {k: v.cpu() for k, v in params.items()}
    keep = {}
    ref = block_forward(cpu, x.cpu(), ctx.cpu(), temb.cpu().repeat_interleave(M // temb_len, 1), freqs.cpu(), dim // 128,
                        1e-6, intermediates=keep)
    assert_close(out.cpu(), ref, 2e-2, 0.9999, f"block {dim} {B}x{M}")
    for name in ("self_q_linear", "self_k_linear", "self_q_norm", "self_k_norm", "self_q_rope", "self_k_rope", "self_v",
                 "residual1", "norm2", "cross_q_linear", "cross_q", "residual2", "modulated3"):
        want = keep[name].reshape(-1, keep[name].shape[-1]) if keep[name].dim() == 3 else keep[name].flatten(2).reshape(-1, dim)
        assert_close(dbg[name].cpu().float(), want, 2.0 ** -7 * want.abs().max().item() + 4e-3, 0.9999, f"{name} {dim} {B}x{M}")


def test_rope_table_batch_is_refused(dev, monkeypatch):
    """A table of neither one nor B samples, past the binding's own check: the
    row pass over partial sums refuses it as the one over rows does."""
    from wam_ops import native, synthetic
    from wam_ops.block import TransformerBlock
    shape = synthetic.BlockShape(256, 2, 512)
    with torch.device("meta"):
        blk = TransformerBlock(256, 512, 2, cross_attn_norm=True)
    blk.load_state_dict(synthetic.block_params(shape, seed=3, device=dev), assign=True)
    monkeypatch.setattr(native, "_check", lambda *a: None)
    for M in (16, 3000):
        x, ctx, temb, freqs = synthetic.block_inputs(shape, 2, M, (1, 1, M), context_len=20, context_batch=2, seed=4, device=dev)
        with torch.no_grad(), pytest.raises(RuntimeError, match="freq batch"):
            blk(x, ctx, temb, freqs[:1].expand(3, *freqs.shape[1:]))
    torch.cuda.synchronize()


def test_calls_go_to_the_current_stream(dev):
    """The handle the operators launch on is the current stream's, and a
    call's scratch outlives its work on a side stream."""
    from wam_ops import ops
    x, w = (_randn(s, dev, i, 0.1, torch.bfloat16) for i, s in enumerate(((32, 1536), (1536, 1536))))
    ref = ops.linear(x, w)
    side = torch.cuda.Stream(dev)
    side.wait_stream(torch.cuda.current_stream(dev))
    with torch.cuda.stream(side):
        assert ops.stream_handle(dev).value == side.cuda_stream
        outs = [ops.linear(x, w) for _ in range(8)]
    assert (ops.stream_handle(dev).value or 0) == torch.cuda.current_stream(dev).cuda_stream
    torch.cuda.synchronize()
    assert all(torch.equal(o, ref) for o in outs)
