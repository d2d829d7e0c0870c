"""The KV pool's bookkeeping on fragmented pools: by the stand-alone kernels at
the edges of their ranges, and by a workgroup of the block's q/k row pass (with
and without partial sums of a split projection)."""
import pytest
import torch

from oracle import kvcache as okv

pytestmark = pytest.mark.gpu


def _pool(P, free, H, seed):
    """Valid slots at random places with ids from a small range (ties), `free` of them free."""
    g = torch.Generator().manual_seed(seed)
    c = okv.new_cache(P, H, 128, 1, torch.bfloat16)
    slots = torch.randperm(P, generator=g)[:P - free]
    c["mask"][slots] = True
    c["id"][slots] = torch.randint(5, 12, (P - free,), generator=g)
    return c


def _expect(cpu, tokens, update):
    """Slots taken, history and pool state by the oracle."""
    ref = okv.clone_cache(cpu)
    kk = torch.zeros(1, tokens, ref["k"].shape[2], 128, dtype=torch.bfloat16)
    new = okv.update_cache(ref, kk, kk, is_pred=(update == 1))
    taken = set(new.tolist())
    hist = [s for s in okv.valid_slots(ref).tolist() if s not in taken]
    if update == 0:
        okv.restore_cache(ref, new)
    return ref, new.tolist(), hist


# Chunks of 64 slots; 8 and 32 slots per thread of 256 and 1024; none free,
# some evicted (two ids and a part of the third), all evicted, exactly enough.
@pytest.mark.parametrize("P", [1, 64, 65, 1025, 8192, 8193, 32768, 32769])
@pytest.mark.parametrize("take", ["evict", "all", "fits"])
def test_pool_layout_edges(dev, P, take):
    from wam_ops import ops
    free = {"evict": 0, "all": P // 2, "fits": (P + 2) // 3}[take]
    tokens = {"evict": max(P * 5 // 12, 1), "all": P, "fits": max(free, 1)}[take]
    cpu = _pool(P, free, 1, P)
    for update in (0, 1):
        ref, new, hist = _expect(cpu, tokens, update)
        gpu = {k: v.to(dev) for k, v in cpu.items()}
        h, n, info = ops.kv_layout(gpu, tokens, update)
        info = info.cpu().tolist()
        run = hist[0] if hist and hist[-1] - hist[0] + 1 == len(hist) else -1
        assert info[:3] == [len(hist), 0, run]
        assert h[:info[0]].cpu().tolist() == hist and n[:tokens].cpu().tolist() == new
        for key in ("mask", "id", "is_pred"):
            assert torch.equal(gpu[key].cpu(), ref[key]), (key, update)
    gpu = {k: v.to(dev) for k, v in cpu.items()}
    h, _, info = ops.kv_layout(gpu, 1, 0, candidate_rows=torch.zeros(3, dtype=torch.int64, device=dev))
    valid = okv.valid_slots(cpu).tolist()
    assert info.cpu().tolist()[:2] == [len(valid), 0] and h[:len(valid)].cpu().tolist() == valid
    for key in ("mask", "id", "is_pred"):
        assert torch.equal(gpu[key].cpu(), cpu[key]), key


# 16 rows leave partial sums of the split projection to the row pass, 2000 do
# not; the row pass does the bookkeeping of pools of up to 4096 slots, a launch
# of its own that of larger ones.
@pytest.mark.parametrize("M", [16, 2000])
@pytest.mark.parametrize("P", [2100, 8192, 8193])
def test_pool_layout_in_block(dev, P, M):
    from wam_ops import synthetic
    from wam_ops.block import TransformerBlock
    shape = synthetic.BlockShape(256, 2, 512)
    with torch.device("meta"):
        blk = TransformerBlock(shape.dim, shape.ffn, shape.heads, cross_attn_norm=True)
    blk.load_state_dict(synthetic.block_params(shape, seed=3, device=dev), assign=True)
    x, ctx, temb, freqs = synthetic.block_inputs(shape, 1, M, (1, 1, M), context_len=20, context_batch=1, seed=4, device=dev)
    cpu = _pool(P, M // 2, shape.heads, 7)
    for update in (0, 2):
        ref, new, _ = _expect(cpu, M, update)
        gpu = {k: v.to(dev) for k, v in cpu.items()}
        alone = {k: v.clone() for k, v in gpu.items()}
        blk.attn1.attn_caches["pos"] = gpu
        with torch.no_grad():
            out = blk(x, ctx, temb, freqs, update_cache=update)
        assert torch.isfinite(out).all()
        for key in ("mask", "id", "is_pred"):
            assert torch.equal(gpu[key].cpu(), ref[key]), (key, update)
        changed = (gpu["k"] != alone["k"]).flatten(2).any(-1)[0].nonzero().flatten().cpu().tolist()
        assert changed == ([] if update == 0 else sorted(new)), update


# More ids than one to evict, chosen by the bits of their distance: within one
# digit of 8, across its edges, in sparse digits, over all 64 bits.
@pytest.mark.parametrize("low,high,step", [(0, 256, 1), (7, 264, 1), (3, 70000, 5), (0, 2 ** 41, 2 ** 33),
                                           (-2 ** 62, 2 ** 62, 1), (-2 ** 63, 2 ** 62, 2 ** 58)])
@pytest.mark.parametrize("P", [70, 2100, 4096, 4097, 8193])
def test_eviction_over_many_ids(dev, P, low, high, step):
    """By the stand-alone kernel and by the block's row pass (up to 4096 slots)."""
    from wam_ops import ops, synthetic
    from wam_ops.block import TransformerBlock
    shape = synthetic.BlockShape(256, 2, 512)
    with torch.device("meta"):
        blk = TransformerBlock(shape.dim, shape.ffn, shape.heads, cross_attn_norm=True)
    blk.load_state_dict(synthetic.block_params(shape, seed=3, device=dev), assign=True)
    g = torch.Generator().manual_seed(P)
    cpu = _pool(P, 3, shape.heads, P)
    valid = okv.valid_slots(cpu)
    cpu["id"][valid] = torch.randint(low, high, (valid.numel(),), generator=g) // step * step
    cpu["id"][valid[valid.numel() // 2]] = high
    for tokens in (5, 60, 2000):
        if tokens > P:
            continue
        ref, new, hist = _expect(cpu, tokens, 2)
        gpu = {k: v.to(dev) for k, v in cpu.items()}
        h, n, info = ops.kv_layout(gpu, tokens, 2)
        assert info.cpu().tolist()[:2] == [len(hist), 0]
        assert h[:len(hist)].cpu().tolist() == hist and n[:tokens].cpu().tolist() == new
        rode = {k: v.to(dev) for k, v in cpu.items()}
        blk.attn1.attn_caches["pos"] = rode
        x, ctx, temb, freqs = synthetic.block_inputs(shape, 1, tokens, (1, 1, tokens), context_len=20, context_batch=1,
                                                     seed=4, device=dev)
        with torch.no_grad():
            blk(x, ctx, temb, freqs, update_cache=2)
        for key in ("mask", "id", "is_pred"):
            assert torch.equal(gpu[key].cpu(), ref[key]), (key, tokens)
            assert torch.equal(rode[key].cpu(), ref[key]), (key, tokens)


def test_eviction_of_many_ids_takes_few_passes(dev):
    """300 ids go in about the time that a few take (one pass over the pool
    per id took 50 times as long)."""
    from wam_ops import ops
    P, us = 2400, {}
    for per_id in (150, 1):
        times = []
        for _ in range(8):
            c = {"mask": torch.ones(P, dtype=torch.bool, device=dev), "id": torch.arange(P, device=dev) // per_id,
                 "is_pred": torch.zeros(P, dtype=torch.bool, device=dev)}
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            ops.kv_layout(c, 300, 2)
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b) * 1e3)
        us[per_id] = min(times)
    assert us[1] < 6 * us[150], us


def test_candidates_over_large_pools(dev):
    """The same 900 valid slots in pools whose bookkeeping rides with the row
    pass (read only: up to 8192 slots) and not."""
    from oracle.metrics import assert_close
    from wam_ops import synthetic
    from wam_ops.block import TransformerBlock
    shape = synthetic.BlockShape(256, 2, 512)
    with torch.device("meta"):
        blk = TransformerBlock(shape.dim, shape.ffn, shape.heads, cross_attn_norm=True)
    blk.load_state_dict(synthetic.block_params(shape, seed=3, device=dev), assign=True)
    x, ctx, temb, freqs = synthetic.block_inputs(shape, 3, 16, (1, 1, 16), context_len=20, context_batch=1, seed=4, device=dev)
    g = torch.Generator().manual_seed(1)
    slots = torch.randperm(4000, generator=g)[:900]
    rows = torch.tensor([1, 0, 1], device=dev)
    kv = torch.randn(2, 2, 900, shape.heads, 128, generator=g).to(torch.bfloat16)
    outs = []
    for P in (4096, 8192, 8193):
        c = okv.new_cache(P, shape.heads, 128, 2, torch.bfloat16)
        c["mask"][slots], c["id"][slots] = True, 3
        c["k"][:, slots], c["v"][:, slots] = kv[0], kv[1]
        gpu = {k: v.to(dev) for k, v in c.items()}
        blk.attn1.attn_caches["pos"] = gpu
        with torch.no_grad():
            outs.append(blk(x, ctx, temb, freqs, candidate_cache_rows=rows))
        for key in c:
            assert torch.equal(gpu[key].cpu(), c[key]), (key, P)
    for o in outs[1:]:  # (other key ranges: a bf16 rounding or two)
        assert_close(o, outs[0], 5e-2, 0.9999, "candidates over large pools")
