"""Attention with few queries per key source (attention_few.hip): 32, 64 and
128 queries per workgroup, whole and in key ranges, grouped batch rows, key
sources of every shape, against an fp32 softmax."""
import ctypes

import pytest
import torch

from oracle.metrics import assert_close

pytestmark = pytest.mark.gpu


def _randn(shape, dev, seed, std=1.0):
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    return (torch.randn(shape, generator=g, device=dev) * std).to(torch.bfloat16)


def _ref(q, k, v, ks):
    """fp32 attention of q [B, Mq, H, hd] over per-row key lists."""
    out = []
    for b in range(q.shape[0]):
        s = torch.einsum("qhd,khd->hqk", q[b].float(), ks[b][0].float()) / 128 ** 0.5
        out.append(torch.einsum("hqk,khd->qhd", torch.softmax(s, -1), ks[b][1].float()))
    return torch.stack(out)


def _pool(dev, Bp, P, H, valid, seed):
    slots = torch.zeros(P, dtype=torch.int32, device=dev)
    slots[:valid.numel()] = valid.int()
    run = int(valid[0]) if valid.numel() and int(valid[-1] - valid[0]) + 1 == valid.numel() else -1
    return dict(pool_k=_randn((Bp, P, H, 128), dev, seed), pool_v=_randn((Bp, P, H, 128), dev, seed + 1), slots=slots,
                n_hist=torch.tensor([valid.numel()], dtype=torch.int32, device=dev),
                hist_base=torch.tensor([run], dtype=torch.int32, device=dev))


# Own keys: one key, a tile, one more; 33 queries (two waves' worth of rows in
# one workgroup size up), 65 to 129 queries, a last partial workgroup, few
# queries over many keys (ranges and the merge).
@pytest.mark.parametrize("B,Mq,Mk,H", [(1, 1, 1, 1), (2, 16, 32, 24), (2, 31, 33, 24), (1, 33, 500, 24), (3, 65, 129, 12),
                                       (1, 129, 512, 24), (2, 200, 96, 12), (1, 780, 512, 24), (1, 1024, 1024, 12),
                                       (1, 16, 6017, 24), (1, 48, 3001, 24), (1, 500, 2000, 12)])
def test_own_keys(dev, B, Mq, Mk, H):
    from wam_ops import ops
    q, k, v = _randn((B, Mq, H, 128), dev, 1, 2.0), _randn((B, Mk, H, 128), dev, 2), _randn((B, Mk, H, 128), dev, 3)
    ref = _ref(q, k, v, list(zip(k, v)))
    assert_close(ops.attention(q, k, v), ref, 2e-2, 0.9999, f"own keys {B}x{Mq}x{Mk}x{H}")


# One own row for every batch row (a shared text context): the batch rows run
# as one list of queries; strided rows of a packed projection do not.
@pytest.mark.parametrize("B,Mq,Mk", [(14, 16, 512), (2, 128, 77), (7, 5, 40)])
def test_shared_own_row(dev, B, Mq, Mk):
    from wam_ops import ops
    H = 24
    packed = _randn((B, Mq, 3, H, 128), dev, 1, 2.0)
    k, v = _randn((1, Mk, H, 128), dev, 2), _randn((1, Mk, H, 128), dev, 3)
    for q in (packed[:, :, 0], packed[:, :, 0].contiguous(), packed[:, :, 0].contiguous().transpose(0, 1).contiguous()
              .transpose(0, 1)):
        ref = _ref(q, k, v, [(k[0], v[0])] * B)
        assert_close(ops.attention(q, k, v), ref, 2e-2, 0.9999, f"shared own row {B}x{Mq}x{Mk}")


# A pool: consecutive slots, a gap (listed slots), no valid slot; candidates
# of one and two pool rows in and out of order (groups of two batch rows of
# one, of two and of three rows of different pool rows).
@pytest.mark.parametrize("B,Mq,n,gap,rows", [
    (2, 16, 288, 0, None), (2, 16, 290, 7, None), (2, 100, 1000, 50, None), (2, 16, 0, 0, None),
    (14, 16, 1152, 0, [0] * 7 + [1] * 7), (14, 16, 720, 3, [0, 1] * 7), (14, 16, 100, 0, [1] * 14),
    (6, 9, 65, 1, [0, 0, 0, 0, 1, 1]), (4, 8, 33, 0, [1, 0, 0, 0]), (1, 20, 6000, 0, [1]), (7, 48, 900, 0, [0] * 7),
    (2, 16, 5000, 11, [0, 0])])
def test_pool(dev, B, Mq, n, gap, rows):
    from wam_ops import ops
    H, Bp = 24, (B if rows is None else 2)
    q, k, v = _randn((B, Mq, H, 128), dev, 1, 2.0), _randn((B, Mq, H, 128), dev, 2), _randn((B, Mq, H, 128), dev, 3)
    valid = torch.arange(n, device=dev)
    valid[n // 2:] += gap
    kw = _pool(dev, Bp, n + gap + 5, H, valid + 3, 4)
    if rows is not None:
        kw["pool_rows"] = torch.tensor(rows, dtype=torch.int64, device=dev)
    at = rows if rows is not None else range(B)
    src = [(torch.cat([kw["pool_k"][r][valid + 3], k[b]]), torch.cat([kw["pool_v"][r][valid + 3], v[b]]))
           for b, r in enumerate(at)]
    # what lies past the valid slots must not reach the result
    dead = torch.ones(n + gap + 5, dtype=torch.bool, device=dev)
    dead[valid + 3] = False
    kw["pool_k"][:, dead] = float("nan")
    kw["pool_v"][:, dead] = float("inf")
    assert_close(ops.attention(q, k, v, **kw), _ref(q, k, v, src), 2e-2, 0.9999, f"pool {B}x{Mq} over {n}")


@pytest.mark.parametrize("gap", [0, 9])
def test_pool_of_one_row(dev, gap):
    """A pool [1, P, H, hd] is contiguous whatever the stride of its first
    dimension: a transposed [P, 1, H, hd] has that of one slot."""
    from wam_ops import ops
    Mq, n, H = 16, 300, 24
    q, k, v = _randn((1, Mq, H, 128), dev, 1, 2.0), _randn((1, Mq, H, 128), dev, 2), _randn((1, Mq, H, 128), dev, 3)
    valid = torch.arange(n, device=dev)
    valid[n // 2:] += gap
    kw = _pool(dev, 1, n + 20, H, valid, 4)
    ref = _ref(q, k, v, [(torch.cat([kw["pool_k"][0, valid], k[0]]), torch.cat([kw["pool_v"][0, valid], v[0]]))])
    for x in ("pool_k", "pool_v"):
        rows = kw[x].new_empty(n + 20, 1, H, 128)
        rows[:, 0] = kw[x][0]
        kw[x] = rows.transpose(0, 1)
        assert kw[x].is_contiguous()
        assert kw[x].stride(0) == H * 128
    assert_close(ops.attention(q, k, v, **kw), ref, 2e-2, 0.9999, f"pool of one row, gap {gap}")


# One, two and four query waves, and groups: the first keys some wave sees.
@pytest.mark.parametrize("B,Mq,Mk,rows", [(1, 16, 300, None), (1, 50, 300, None), (1, 200, 300, None),
                                          (14, 16, 100, [0] * 14)])
def test_scores_of_minus_infinity(dev, B, Mq, Mk, rows):
    """Keys whose scores are -inf have no weight, whole tiles of them too."""
    from wam_ops import ops
    H, dead = 24, slice(32, 96)
    q = _randn((B, Mq, H, 128), dev, 1).abs() + 0.1
    k, v = _randn((B, Mk, H, 128), dev, 2), _randn((B, Mk, H, 128), dev, 3)
    keep = torch.ones(Mk, dtype=torch.bool, device=dev)
    keep[dead] = False
    src = [(k[b, keep], v[b, keep]) for b in range(B)]
    kw = {}
    if rows:
        kw = _pool(dev, 1, 70, H, torch.arange(70, device=dev), 4)
        kw["pool_rows"] = torch.tensor(rows, device=dev)
        src = [(torch.cat([kw["pool_k"][0], a]), torch.cat([kw["pool_v"][0], b])) for a, b in src]
    ref = _ref(q, k, v, src)
    k[:, dead] = float("-inf")
    assert_close(ops.attention(q, k, v, **kw), ref, 2e-2, 0.9999, f"scores of -inf {B}x{Mq}x{Mk}")


@pytest.mark.parametrize("scale", [0.0, -0.05])
@pytest.mark.parametrize("B,n,own", [(14, 304, 16), (1, 0, 128)])
def test_scales_not_above_zero(dev, scale, B, n, own):
    """Any scale, over whole 64-key tiles; candidates whose masks count."""
    from wam_ops import ops
    Mq, H = 16, 24
    q, k, v = _randn((B, Mq, H, 128), dev, 1), _randn((B, own, H, 128), dev, 2), _randn((B, own, H, 128), dev, 3)
    src, kw = list(zip(k, v)), {}
    if n:
        rows = [b // 7 for b in range(B)]
        kw = _pool(dev, 2, n, H, torch.arange(n, device=dev), 4)
        src = [(torch.cat([kw["pool_k"][r], a]), torch.cat([kw["pool_v"][r], b])) for r, (a, b) in zip(rows, src)]
        kw["pool_rows"] = torch.tensor(rows, device=dev)
    ref = _ref(q.float() * (scale * 128 ** 0.5), k, v, src)
    assert_close(ops.attention(q, k, v, scale=scale, **kw), ref, 2e-2, 0.9999, f"scale {scale}, {B}x{Mq}")


# Rows of two and three pool rows, in equal shares: one workgroup per row, pairs
# and ranges, threes and fours, pairs that straddle two pool rows.
@pytest.mark.parametrize("B,Bp,Mq,n", [(10, 2, 16, 1300), (8, 2, 16, 5000), (6, 2, 5, 3000), (8, 2, 5, 2500), (9, 3, 10, 700),
                                       (14, 2, 16, 400)])
def test_shares_of_pool_rows(dev, B, Bp, Mq, n):
    from wam_ops import ops
    H = 24
    q, k, v = _randn((B, Mq, H, 128), dev, 1, 2.0), _randn((B, Mq, H, 128), dev, 2), _randn((B, Mq, H, 128), dev, 3)
    kw = _pool(dev, Bp, n + 3, H, torch.arange(n, device=dev), 4)
    kw["pool_rows"] = torch.arange(B, device=dev) * Bp // B
    src = [(torch.cat([kw["pool_k"][r, :n], k[b]]), torch.cat([kw["pool_v"][r, :n], v[b]]))
           for b, r in enumerate(kw["pool_rows"].tolist())]
    assert_close(ops.attention(q, k, v, **kw), _ref(q, k, v, src), 2e-2, 0.9999, f"{B} rows of {Bp} x {Mq} over {n}")


def test_groups_do_not_straddle_pool_rows(dev):
    """Ten rows over two pool rows take little more time than seven over one
    (1.2 times; in pairs, one of which reads both pool rows, it was 2)."""
    from wam_ops import ops
    H, Mq, n = 24, 16, 1317
    us = {}
    for B, Bp in ((7, 1), (10, 2)):
        q, k, v = _randn((B, Mq, H, 128), dev, 1), _randn((B, Mq, H, 128), dev, 2), _randn((B, Mq, H, 128), dev, 3)
        kw = _pool(dev, Bp, n + 16, H, torch.arange(n, device=dev), 4)
        kw["pool_rows"] = torch.arange(B, device=dev) * Bp // B
        times = []
        for _ in range(12):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(20):
                ops.attention(q, k, v, **kw)
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b) * 50)
        us[B] = min(times)
    assert us[10] < 1.55 * us[7], us


def test_own_row_map_and_query_rms(dev):
    """kv_rows, and q_ssq's per-query factor (rows of the folded batch too)."""
    from wam_ops import ops
    B, Mq, Mk, H = 6, 12, 70, 24
    q, k, v = _randn((B, Mq, H, 128), dev, 1, 2.0), _randn((2, Mk, H, 128), dev, 2), _randn((2, Mk, H, 128), dev, 3)
    rows = torch.tensor([0, 1, 1, 0, 0, 1], device=dev)
    src = [(k[r], v[r]) for r in rows.tolist()]
    assert_close(ops.attention(q, k, v, kv_rows=rows), _ref(q, k, v, src), 2e-2, 0.9999, "own row map")
    ssq = (torch.rand(B * Mq, 12, device=dev) + 0.5) * 256
    f = torch.rsqrt(ssq.sum(1) / (H * 128) + 1e-6).view(B, Mq, 1, 1)
    ref = _ref(q.float() * f, k, v, [(k[0], v[0])] * B)
    assert_close(ops.attention(q, k[:1], v[:1], q_ssq=ssq), ref, 2e-2, 0.9999, "query RMS factor")


# Workgroups of 32 and of 64 queries.  With 48 queries the general kernel is
# the faster one once all of its own 32 ranges fit.
@pytest.mark.parametrize("Mq,Mk,block,most", [(16, 6000, 32, 8), (48, 3001, 64, 32)])
def test_workspace_sizes(dev, Mq, Mk, block, most):
    """The same call with less and less room: no workspace, one byte less than
    two ranges' partial results take, two and three ranges', one byte less
    than all eight ranges', all, and what the size query asks for.  Ranges
    that fit are used, nothing is written past them; the entry point without
    allocation computes what the whole workspace gives."""
    from wam_ops import _lib
    H = 24
    q, k, v = _randn((1, Mq, H, 128), dev, 1), _randn((1, Mk, H, 128), dev, 2), _randn((1, Mk, H, 128), dev, 3)
    ref = _ref(q, k, v, list(zip(k, v)))
    h = _lib.lib()
    need = h.wam_attention_workspace_bytes(1, Mq, H, Mk)
    # a range: per head and query of a workgroup 128 sums, a maximum and a weight
    one = H * block * 130 * 4
    assert need >= 8 * one
    outs = {}
    for nbytes, ranges in ((0, 1), (2 * one - 1, 1), (2 * one, 2), (4 * one - 1, 3), (8 * one - 1, 7), (8 * one, 8),
                           (need, most), (None, None)):
        ws = torch.full((max(need, 8 * one) + 4096,), 0xA5, dtype=torch.uint8, device=dev)
        o = torch.zeros_like(q)
        a = _lib.AttentionArgs()
        a.q, a.q_bstride, a.q_rstride = q.data_ptr(), q.stride(0), q.stride(1)
        a.o, a.o_bstride, a.o_rstride = o.data_ptr(), o.stride(0), o.stride(1)
        a.B, a.Mq, a.H, a.head_dim, a.Mk, a.kv_batch, a.scale, a.max_keys = 1, Mq, H, 128, Mk, 1, 128 ** -0.5, Mk
        a.k, a.v, a.kv_bstride, a.kv_rstride = k.data_ptr(), v.data_ptr(), k.stride(0), k.stride(1)
        if nbytes:
            a.workspace, a.workspace_bytes = ws.data_ptr(), nbytes
        f = h.wam_attention if nbytes is not None else h.wam_attention_noalloc
        _lib.check(f(ctypes.byref(a), None), "wam_attention")
        torch.cuda.synchronize()
        assert_close(o, ref, 2e-2, 0.9999, f"workspace of {nbytes} bytes")
        outs[nbytes] = o
        if nbytes is not None:
            written = (ws != 0xA5).nonzero()
            end = int(written[-1]) + 1 if written.numel() else 0
            # (between two and what fits, the plan may find fewer as fast)
            assert one < end <= ranges * one if ranges > 1 else end == 0, (nbytes, ranges, end / one)
            assert ranges in (1, 7) or end > (ranges - 1) * one, (nbytes, ranges, end / one)
    assert torch.equal(outs[need], outs[None]) and (most > 8 or torch.equal(outs[need], outs[8 * one]))


# Few keys, where the two kernels' predicted times are close: own keys only,
# and most of them in a pool.
@pytest.mark.parametrize("H", [12, 24])
@pytest.mark.parametrize("Mq", [1, 17, 33, 49, 60, 120])
def test_entry_points_agree(dev, Mq, H):
    """wam_attention with its whole workspace and the entry point without
    allocation run the same kernel: equal bits."""
    from wam_ops import _lib
    h = _lib.lib()
    for keys in (32, 64, 128, 192, 300):
        for n in (0, keys - min(Mq, keys - 1)):
            own = keys - n
            q, k, v = _randn((1, Mq, H, 128), dev, 1), _randn((1, own, H, 128), dev, 2), _randn((1, own, H, 128), dev, 3)
            kw = _pool(dev, 1, max(n, 1), H, torch.arange(n, device=dev), 4)
            outs = []
            for f in (h.wam_attention, h.wam_attention_noalloc):
                o = torch.zeros_like(q)
                a = _lib.AttentionArgs()
                a.q, a.q_bstride, a.q_rstride = q.data_ptr(), q.stride(0), q.stride(1)
                a.o, a.o_bstride, a.o_rstride = o.data_ptr(), o.stride(0), o.stride(1)
                a.B, a.Mq, a.H, a.head_dim, a.Mk, a.kv_batch, a.scale, a.max_keys = 1, Mq, H, 128, own, 1, 128 ** -0.5, keys
                a.k, a.v, a.kv_bstride, a.kv_rstride = k.data_ptr(), v.data_ptr(), k.stride(0), k.stride(1)
                if n:
                    a.pool_k, a.pool_v, a.pool_batch = kw["pool_k"].data_ptr(), kw["pool_v"].data_ptr(), 1
                    a.pool_bstride, a.pool_rstride = n * H * 128, H * 128
                    a.slots, a.n_hist_dev, a.hist_base_dev = (kw[x].data_ptr() for x in ("slots", "n_hist", "hist_base"))
                if not outs:
                    ws = torch.empty(h.wam_attention_workspace_bytes(1, Mq, H, keys) + 16, dtype=torch.uint8, device=dev)
                    a.workspace, a.workspace_bytes = ws.data_ptr(), ws.numel()
                _lib.check(f(ctypes.byref(a), None), "wam_attention")
                torch.cuda.synchronize()
                outs.append(o)
            assert torch.equal(*outs), (Mq, H, keys, n)


@pytest.mark.parametrize("B", [1, 6])  # fewer units than the pipelined kernel takes, and enough
def test_backward_keys(dev, B):
    """Own keys addressed from their last row back (a negative row stride)."""
    from wam_ops import _lib
    H, Mq, Mk = 24, 16, 200
    q, k, v = _randn((B, Mq, H, 128), dev, 1), _randn((B, Mk, H, 128), dev, 2), _randn((B, Mk, H, 128), dev, 3)
    ref, o = _ref(q, k, v, list(zip(k, v))), torch.zeros_like(q)
    a = _lib.AttentionArgs()
    a.q, a.q_bstride, a.q_rstride = q.data_ptr(), q.stride(0), q.stride(1)
    a.o, a.o_bstride, a.o_rstride = o.data_ptr(), o.stride(0), o.stride(1)
    a.B, a.Mq, a.H, a.head_dim, a.Mk, a.kv_batch, a.scale = B, Mq, H, 128, Mk, B, 128 ** -0.5
    a.k, a.v, a.kv_bstride, a.kv_rstride = k[0, -1].data_ptr(), v[0, -1].data_ptr(), k.stride(0), -k.stride(1)
    _lib.check(_lib.lib().wam_attention(ctypes.byref(a), None), "wam_attention")
    torch.cuda.synchronize()
    assert_close(o, ref, 2e-2, 0.9999, f"backward keys {B}x{Mq}x{Mk}")


def test_candidates_are_isolated(dev):
    """A candidate whose own rows hold infinities and NaN leaves the others,
    its neighbour in the same workgroup too, as they were."""
    from wam_ops import ops
    B, Mq, H, n = 14, 16, 24, 200
    q, k, v = _randn((B, Mq, H, 128), dev, 1), _randn((B, Mq, H, 128), dev, 2), _randn((B, Mq, H, 128), dev, 3)
    kw = _pool(dev, 2, n, H, torch.arange(n, device=dev), 4)
    kw["pool_rows"] = torch.tensor([0] * 7 + [1] * 7, device=dev)
    clean = ops.attention(q, k, v, **kw)
    v[4], k[4, 3], v[9, 0] = float("inf"), float("nan"), float("nan")
    out = ops.attention(q, k, v, **kw)
    keep = [b for b in range(B) if b not in (4, 9)]
    assert torch.equal(out[keep], clean[keep])
    assert not bool(torch.isfinite(out[[4, 9]].float()).any())
    # the other branch's history (rows 6 and 7 share a workgroup)
    kw["pool_v"][1] = float("inf")
    out = ops.attention(q, k, v, **kw)
    assert torch.equal(out[[0, 6]], clean[[0, 6]])
