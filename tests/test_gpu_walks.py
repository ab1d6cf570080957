"""Edges of the pipelined attention walks: blocks of several chunks, lists of one
block, tiles that skip blocks of their workgroup's union, unsplit grids, and
token strides past the gathers' 32-bit lane offsets or below zero."""

import numpy as np
import pytest
import torch

from _helpers import rand, say
from test_gpu_parity import _random_merged, check_attn_vs_oracle

pytestmark = pytest.mark.gpu

fta = pytest.importorskip("flash_topk_attn_v2")

WALK_CASES = [
    # B, N, H, D, g, b, q padding, kv padding, W, dtype
    (1, 500, 2, 64, 32, 160, (0, 12), (100, 40), 3, torch.float16),  # 3 chunks a block, the last of 32 keys
    (1, 500, 2, 128, 16, 130, (4, 8), (0, 20), 2, torch.bfloat16),  # the last chunk of 2 keys
    (1, 300, 2, 64, 16, 64, (0, 4), (0, 20), 1, torch.bfloat16),  # lists of one block: tiles skip most steps
    (1, 300, 2, 128, 16, 64, (0, 4), (0, 20), 1, torch.float16),
    (2, 1030, 16, 64, 64, 64, (60, 62), (63, 59), 6, torch.float16),  # unsplit grids (160 workgroups)
    (2, 1030, 16, 128, 48, 40, (0, 26), (0, 10), 5, torch.bfloat16),
    (1, 33, 2, 64, 33, 64, (0, 0), (31, 0), 1, torch.bfloat16),  # one block, two query tiles
]


@pytest.mark.parametrize("case", WALK_CASES, ids=lambda c: f"B{c[0]}N{c[1]}D{c[3]}g{c[4]}b{c[5]}W{c[8]}")
def test_walk_edges(case):
    B, N, H, D, g, b, qpad, kvpad, W, dt = case
    say(f"[walk] {case}")
    QM, M = (qpad[0] + N + qpad[1]) // g, (kvpad[0] + N + kvpad[1]) // b
    merged = _random_merged(B, H, QM, W, M, 11)
    q, k, v = (rand((B, N, H * D), 12 + i, dt, "cuda").requires_grad_(True) for i in range(3))
    tm = torch.from_numpy(merged).cuda()
    o, lse = fta.flash_topk_attn(q, k, v, tm, (tm >= 0).sum(-1).int(), H, g, b, None, None, kvpad, qpad)
    do = rand((B, N, H * D), 99, dt, "cuda")
    o.backward(do)
    torch.cuda.synchronize()
    check_attn_vs_oracle(q, k, v, do, o, lse, merged, H, g, b, qpad, kvpad, dt)


@pytest.mark.parametrize("D,b", [(64, 64), (128, 64), (256, 64)])
def test_wide_token_strides(D, b):
    """Rows 2^24 + 8 elements apart (gathered by 64-bit addresses), one KV block: o and the
    gradients are within one bf16 rounding step of the contiguous call."""
    N, H, g, W = 40, 1, 16, 1
    say(f"[wide strides] D{D}")
    stride = 2**24 + 8
    merged = torch.zeros(1, H, 3, W, dtype=torch.int32, device="cuda")
    narrow = [rand((1, N, H * D), 30 + i, torch.bfloat16, "cuda") for i in range(4)]
    wide = []
    for t in narrow:
        big = torch.empty((N - 1) * stride + H * D, dtype=t.dtype, device="cuda")
        w = big.as_strided(t.shape, (N * stride, stride, 1))
        wide.append(w.copy_(t))
    res = []
    for q, k, v, do in (narrow, wide):
        q, k, v = (x.detach().requires_grad_(True) for x in (q, k, v))
        o, lse = fta.flash_topk_attn(q, k, v, merged, None, H, g, b, None, None, (0, 24), (0, 8))
        res.append([o.detach(), lse, *torch.autograd.grad(o, (q, k, v), do)])
    torch.cuda.synchronize()
    for name, x, y in zip(("o", "lse", "dq", "dk", "dv"), *res):
        x, y = x.float().cpu().numpy(), y.float().cpu().numpy()
        step = np.maximum(np.abs(x), np.abs(y)) * 2.0**-7 + np.abs(x).max() * 2.0**-16
        assert (np.abs(x - y) <= step).all(), name


@pytest.mark.parametrize("D,b,N,H,Hk,step", [
    (64, 64, 1000, 2, 2, -1), (128, 64, 1000, 4, 2, -1), (256, 64, 500, 2, 2, -1), (128, 48, 500, 2, 2, -1),
    (96, 128, 700, 2, 1, -1), (64, 64, 136, 1, 1, 2**24 + 8), (128, 64, 136, 1, 1, 2**24 + 8)])
def test_token_strides(D, b, N, H, Hk, step):
    """Tokens stored last to first (negative token strides, C entry) or 2^24 + 8 elements
    apart, over several KV blocks: the kernels and the order of their sums are those of the
    contiguous call, so the results are its bits."""
    from flash_topk_attn_v2 import _lib

    g, dt = 16, torch.bfloat16
    say(f"[token strides] D{D} b{b} N{N} H{H}/{Hk} step {step}")
    qpad, kvpad = -N % g, -N % b
    QM, M = (N + qpad) // g, (N + kvpad) // b
    merged = torch.from_numpy(_random_merged(1, H, QM, 2, M, 17)).cuda()
    toks = [rand((N, h * D), 40 + i, dt, "cuda") for i, h in enumerate((H, Hk, Hk, H))]  # q, k, v, do
    L, stream = _lib.lib(), torch.cuda.current_stream().cuda_stream
    geo = (g, b, 0, qpad, 0, kvpad)

    def call(views):
        """o, lse, dq, dk, dv of tokens at (pointer, strides)"""
        o, dq = (torch.empty(N, H * D, device="cuda", dtype=dt) for _ in range(2))
        dk, dv = (torch.empty(N, Hk * D, device="cuda", dtype=dt) for _ in range(2))
        lse = torch.empty(1, H, N, device="cuda")
        so, sk = _lib.i64arr((N * H * D, D, H * D)), _lib.i64arr((N * Hk * D, D, Hk * D))
        (q, qs), (k, ks), (v, vs), (do, ds) = views
        code = _lib.dtype_code(dt)
        size = (1, H, N, D, *geo)
        ws = torch.empty(max(L.fta_sparse_attn_fwd_workspace_size(*size), L.fta_sparse_attn_bwd_workspace_size(*size)),
                         dtype=torch.uint8, device="cuda")
        shape = (1, H, Hk, N, D, merged.data_ptr(), QM, 2, *geo, D ** -0.5)
        _lib.check(L.fta_sparse_attn_fwd_gqa(q, qs, k, ks, v, vs, code, *shape, o.data_ptr(), so, lse.data_ptr(),
                                             ws.data_ptr(), ws.numel(), stream), "fwd")
        delta = (o.float() * toks[3].float()).view(N, H, D).sum(-1).T.contiguous()
        _lib.check(L.fta_sparse_attn_bwd_gqa(q, qs, k, ks, v, vs, do, ds, code, *shape, lse.data_ptr(),
                                             delta.data_ptr(), dq.data_ptr(), so, dk.data_ptr(), sk, dv.data_ptr(), sk,
                                             ws.data_ptr(), ws.numel(), stream), "bwd")
        torch.cuda.synchronize()
        return o, lse, dq, dk, dv

    want = call([(t.data_ptr(), _lib.i64arr((t.numel(), D, t.shape[1]))) for t in toks])
    keep, views = [], []
    for t in toks:
        if step < 0:
            store = t.flip(0).contiguous()
            views.append((store[-1].data_ptr(), _lib.i64arr((t.numel(), D, -t.shape[1]))))
        else:
            store = torch.empty((N - 1) * step + t.shape[1], dtype=dt, device="cuda")
            store.as_strided(t.shape, (step, 1)).copy_(t)
            views.append((store.data_ptr(), _lib.i64arr((N * step, D, step))))
        keep.append(store)
    for name, x, y in zip(("o", "lse", "dq", "dk", "dv"), want, call(views)):
        assert torch.equal(x, y), name


@pytest.mark.parametrize("D,H", [(160, 66), (256, 33)])
def test_wide_heads_leave_workspace(D, H):
    """Forwards of wide heads with more than 256 workgroups use no head placement and no
    split: nothing is computed into the workspace."""
    from flash_topk_attn_v2 import _lib

    N, g, b = 1024, 64, 64
    say(f"[workspace] D{D} H{H}")
    merged = torch.from_numpy(_random_merged(1, H, N // g, 2, N // b, 19)).cuda()
    q, k, v = (rand((1, N, H * D), 80 + i, torch.float16, "cuda") for i in range(3))
    want = fta.flash_topk_attn(q, k, v, merged, None, H, g, b)[0]
    L, st = _lib.lib(), _lib.i64arr((N * H * D, D, H * D))
    nbytes = L.fta_sparse_attn_fwd_workspace_size(1, H, N, D, g, b, 0, 0, 0, 0)
    ws = torch.full((nbytes,), 0x5A, dtype=torch.uint8, device="cuda")
    o, lse = torch.empty_like(want), torch.empty(1, H, N, device="cuda")
    _lib.check(L.fta_sparse_attn_fwd_gqa(q.data_ptr(), st, k.data_ptr(), st, v.data_ptr(), st, _lib.dtype_code(q.dtype),
                                         1, H, H, N, D, merged.data_ptr(), N // g, 2, g, b, 0, 0, 0, 0, D ** -0.5,
                                         o.data_ptr(), st, lse.data_ptr(), ws.data_ptr(), nbytes,
                                         torch.cuda.current_stream().cuda_stream), "fta_sparse_attn_fwd_gqa")
    torch.cuda.synchronize()
    assert torch.equal(o, want)
    assert bool((ws == 0x5A).all())


@pytest.mark.parametrize("W,offset", [(5, 0), (8, 0), (8, 1), (12, 2), (1, 3)])
def test_list_loads(W, offset):
    """Merged lists are read 16 bytes at a time where a row is a multiple of 4 ids on a
    16-byte boundary, 4 bytes otherwise: the same lists in any width and at any
    alignment (padded with -1, or at an odd place in a buffer) give the same bits."""
    B, H, N, D, g, b = 1, 2, 700, 64, 16, 64
    say(f"[list loads] W{W} offset {offset}")
    qpad, kvpad = (0, 4), (0, 4)
    merged = torch.from_numpy(_random_merged(B, H, 44, W, 11, 5)).cuda()
    base = torch.full((B, H, 44, 16), -1, dtype=torch.int32, device="cuda")
    base[..., :W] = merged
    buf = torch.empty(merged.numel() + offset, dtype=torch.int32, device="cuda")
    placed = buf[offset:].view(merged.shape).copy_(merged)
    assert placed.is_contiguous() and placed.data_ptr() % 16 == 4 * offset
    q, k, v, do = (rand((B, N, H * D), 50 + i, torch.bfloat16, "cuda") for i in range(4))
    res = []
    for lists in (base, placed):
        ql, kl, vl = (x.detach().requires_grad_(True) for x in (q, k, v))
        o, lse = fta.flash_topk_attn(ql, kl, vl, lists, None, H, g, b, None, None, kvpad, qpad)
        res.append([o.detach(), lse, *torch.autograd.grad(o, (ql, kl, vl), do)])
    for x, y in zip(*res):
        assert torch.equal(x, y)


@pytest.mark.parametrize("case", [
    # B, N, H, D, g, b, q padding, kv padding, W, dtype
    (1, 1030, 2, 256, 32, 64, (3, 23), (13, 45), 10, torch.bfloat16),  # 9 blocks a workgroup, 4 parts
    (1, 1000, 2, 224, 16, 64, (0, 8), (24, 0), 3, torch.float16),  # 224 columns run as 256; short lists
    (1, 1000, 2, 160, 16, 64, (0, 8), (24, 0), 3, torch.float16),  # not split at D = 160
    (1, 600, 1, 192, 48, 160, (0, 24), (0, 40), 2, torch.bfloat16),  # 4 blocks: not split
], ids=lambda c: f"N{c[1]}D{c[3]}b{c[5]}W{c[8]}")
def test_wide_head_split_forward(case):
    """Heads of more than 160 columns split the forward's walks on small grids too:
    against the same call without a workspace (unsplit), lse to 1e-5 and o to one 16-bit
    rounding step of the largest probability's weight (the parts round P against their
    own maxima), and against the oracle."""
    from flash_topk_attn_v2 import _lib

    B, N, H, D, g, b, qpad, kvpad, W, dt = case
    say(f"[wide split] {case}")
    QM, M = (qpad[0] + N + qpad[1]) // g, (kvpad[0] + N + kvpad[1]) // b
    merged = _random_merged(B, H, QM, W, M, 21)
    tm = torch.from_numpy(merged).cuda()
    q, k, v = (rand((B, N, H * D), 22 + i, dt, "cuda") for i in range(3))
    L = _lib.lib()
    splits = L.fta_sparse_attn_fwd_splits(B, H, N, D, g, b, *qpad, *kvpad)
    assert (splits > 1) == (M >= 8 and D > 160)
    o, lse = fta.flash_topk_attn(q, k, v, tm, None, H, g, b, None, None, kvpad, qpad)
    st = _lib.i64arr((N * H * D, D, H * D))
    o2, lse2 = torch.empty_like(o), torch.empty_like(lse)
    _lib.check(L.fta_sparse_attn_fwd_gqa(q.data_ptr(), st, k.data_ptr(), st, v.data_ptr(), st, _lib.dtype_code(dt), B,
                                         H, H, N, D, tm.data_ptr(), QM, W, g, b, *qpad, *kvpad, D ** -0.5,
                                         o2.data_ptr(), st, lse2.data_ptr(), None, 0,
                                         torch.cuda.current_stream().cuda_stream), "fta_sparse_attn_fwd_gqa")
    torch.cuda.synchronize()
    assert torch.equal(torch.isinf(lse), torch.isinf(lse2))
    fin = torch.isfinite(lse2)
    assert torch.allclose(lse[fin], lse2[fin], rtol=1e-5, atol=1e-5)
    # |v| <= 6 here, sum of P = 1 after division: rounding P twice differently moves o by
    # at most 2 * 2^-9 (bf16) * 6, and the two stored outputs by one step each
    assert (o.float() - o2.float()).abs().max() <= 2 * 2.0**-9 * 6 + 2 * 2.0**-8 * o2.float().abs().max()
    check_attn_vs_oracle(q, k, v, None, o, lse, merged, H, g, b, qpad, kvpad, dt)


@pytest.mark.parametrize("N,H,D,g", [(2500, 3, 64, 256), (1025, 1, 128, 1024), (700, 2, 64, 192)])
def test_wide_query_blocks(N, H, D, g):
    """The backward takes q-blocks of any size: blocks of ``g`` queries give the bits of
    the same lists repeated for blocks of 64 (few bitmap workgroups, log2 lse values in
    several chunks and in one partly filled one)."""
    from flash_topk_attn_v2.sparse_attn_bwd import sparse_attn_bwd

    b, W = 64, 4
    say(f"[wide q-blocks] N{N} H{H} D{D} g{g}")
    qpad, kvpad = -N % g, -N % b
    QM, M, q64 = (N + qpad) // g, (N + kvpad) // b, -N % 64
    lists = torch.from_numpy(_random_merged(1, H, QM, W, M, 7)).cuda()
    fine = lists.repeat_interleave(g // 64, dim=2)[:, :, :(N + q64) // 64].contiguous()
    q, k, v, do = (rand((1, N, H * D), 60 + i, torch.bfloat16, "cuda") for i in range(4))
    o, lse = fta.flash_topk_attn(q, k, v, fine, None, H, 64, b, None, None, (0, kvpad), (0, q64))
    res = [sparse_attn_bwd(q, k, v, o, do, lse, tm, H, gg, b, D ** -0.5, (0, qp), (0, kvpad))
           for tm, gg, qp in ((fine, 64, q64), (lists, g, qpad))]
    for x, y in zip(*res):
        assert torch.equal(x, y)


@pytest.mark.parametrize("H,g,b,W,short", [
    (3, 64, 64, 2, True), (3, 32, 64, 1, True), (3, 64, 128, 1, True), (3, 33, 64, 1, True), (3, 64, 64, 3, False),
    (3, 32, 64, 2, False), (12, 64, 64, 3, True), (12, 32, 64, 2, False)])  # 4 parts with 3 heads, 2 with 12
def test_wide_head_short_lists(H, g, b, W, short):
    """At D = 256 a small grid splits only walks of more than 4 chunks (6 in two parts):
    shorter ones give the bits of the call without a workspace (unsplit)."""
    from flash_topk_attn_v2 import _lib

    N, D = 1056, 256
    say(f"[short wide] H{H} g{g} b{b} W{W}")
    qpad, kvpad = -N % g, -N % b
    QM, M = (N + qpad) // g, (N + kvpad) // b
    merged = torch.from_numpy(_random_merged(1, H, QM, W, M, 29)).cuda()
    q, k, v = (rand((1, N, H * D), 84 + i, torch.bfloat16, "cuda") for i in range(3))
    L, st = _lib.lib(), _lib.i64arr((N * H * D, D, H * D))
    assert L.fta_sparse_attn_fwd_splits(1, H, N, D, g, b, 0, qpad, 0, kvpad) > 1
    o, lse = fta.flash_topk_attn(q, k, v, merged, None, H, g, b, None, None, (0, kvpad), (0, qpad))
    o2, lse2 = torch.empty_like(o), torch.empty_like(lse)
    _lib.check(L.fta_sparse_attn_fwd_gqa(q.data_ptr(), st, k.data_ptr(), st, v.data_ptr(), st, 0, 1, H, H, N, D,
                                         merged.data_ptr(), QM, W, g, b, 0, qpad, 0, kvpad, D ** -0.5, o2.data_ptr(), st,
                                         lse2.data_ptr(), None, 0, torch.cuda.current_stream().cuda_stream), "fwd")
    torch.cuda.synchronize()
    assert torch.equal(o, o2) == short
    if short:
        assert torch.equal(lse, lse2)


def _check_grads(tokens, lists, got, H, Hk, D, g, b):
    """dq, dk, dv (``got``) of one unpadded sequence against float64.  P and dS are rounded
    to 16 bits once (relative error u = 2^-9 or 2^-12) and so are o, which delta is formed
    from, and the results; every bound allows 2 u."""
    u2 = 2.0**-8 if tokens[0].dtype == torch.bfloat16 else 2.0**-11
    N, G, scale = tokens[0].shape[1], H // Hk, D ** -0.5
    q, k, v, do = (x.detach().double().cpu()[0].view(N, -1, D) for x in tokens)
    ref, tol = ([torch.zeros_like(x) for x in (q, k, v)] for _ in range(2))
    for h in range(H):
        for c in range(N // g):
            ids = [m for m in lists[0, h, c].tolist() if m >= 0]
            if not ids:
                continue
            r, s = slice(c * g, c * g + g), torch.cat([torch.arange(m * b, m * b + b) for m in ids])
            Q, K, V, O = q[r, h], k[s, h // G], v[s, h // G], do[r, h]
            P = (Q @ K.T * scale).softmax(-1)
            o64 = P @ V
            dS = P * (O @ V.T - (o64 * O).sum(-1, keepdim=True))
            dSt = u2 * dS.abs() + u2 * P * (o64 * O).abs().sum(-1, keepdim=True)  # rounded dS, delta from rounded o
            ref[0][r, h] += dS @ K * scale
            tol[0][r, h] += dSt @ K.abs() * scale
            ref[1][s, h // G] += dS.T @ Q * scale
            tol[1][s, h // G] += dSt.T @ Q.abs() * scale
            ref[2][s, h // G] += P.T @ O
            tol[2][s, h // G] += u2 * P.T @ O.abs()
    for name, x, y, t in zip(("dq", "dk", "dv"), got, ref, tol):
        x = x.double().cpu()[0].view(N, -1, D)
        assert ((x - y).abs() <= t + u2 * y.abs()).all(), name


# chunks (32 queries) that select each KV block: none, single ones at both ends, the last
# of a mask segment of 1024 and the first of the next, runs of every length up to 7
CHUNK_SETS = [[], [0], [1249], [5, 1023], [1023, 1024], [0, 1, 2], [7, 8, 1024, 1249], list(range(1021, 1028)),
              [3, 4, 5, 6, 7], list(range(30, 36)), [1024], list(range(100, 133))]


@pytest.mark.parametrize("D,H,Hk,dt", [(64, 1, 1, torch.bfloat16), (128, 1, 1, torch.float16), (256, 1, 1, torch.bfloat16),
                                       (64, 3, 1, torch.float16), (128, 4, 2, torch.bfloat16)])
def test_dkv_chunk_lists(D, H, Hk, dt):
    """dK / dV walks of 0 to 33 chunks in one and two mask segments (1250 chunks)."""
    N, g, b, W = 40000, 32, 64, 4
    say(f"[chunk lists] D{D} H{H}/{Hk}")
    QM, M = N // g, N // b
    lists = torch.full((1, H, QM, W), -1, dtype=torch.int32)
    for h in range(H):
        for i, chunks in enumerate(CHUNK_SETS):
            m = (53 * i + 17 * h) % M
            for c in chunks:
                c = min(c + 2 * h, QM - 1)
                row = lists[0, h, c]
                if m not in row.tolist():
                    row[(row >= 0).sum()] = m
    q, do = (rand((1, N, H * D), 70 + i, dt, "cuda") for i in range(2))
    k, v = (rand((1, N, Hk * D), 72 + i, dt, "cuda") for i in range(2))
    ql, kl, vl = (x.detach().requires_grad_(True) for x in (q, k, v))
    o, lse = fta.flash_topk_attn(ql, kl, vl, lists.cuda(), None, H, g, b, num_kv_heads=Hk)
    _check_grads((q, k, v, do), lists, torch.autograd.grad(o, (ql, kl, vl), do), H, Hk, D, g, b)


@pytest.mark.parametrize("N,H,Hk,D,g,W", [
    (6272, 16, 8, 64, 32, 2),  # 784 blocks, 768 run at once; bitmap rows of 7 words
    (6272, 16, 8, 64, 64, 1),  # rows of 4 words (16-byte loads)
    (4160, 16, 8, 128, 16, 1),  # 520 blocks, 512 at once; rows of 9 words
    (2176, 8, 8, 256, 64, 2),  # 272 blocks, 256 at once
    (2176, 16, 8, 256, 32, 1),
    (6272, 10, 10, 64, 32, 1),  # heads that no multiple of 8 covers: natural head order
])
def test_launch_order(N, H, Hk, D, g, W):
    """dK / dV grids just above what the chip holds at once, which are launched in the
    order of the blocks' counts with the heads placed by their work (GQA and D = 256)."""
    b, dt = 64, torch.bfloat16
    say(f"[launch order] N{N} H{H}/{Hk} D{D} g{g}")
    lists = torch.from_numpy(_random_merged(1, H, N // g, W, N // b, 23))
    lists[:, ::3] %= N // b // 2  # heads of unequal counts per block
    if W > 1:
        lists[..., 1] = torch.where(lists[..., 1] == lists[..., 0], -1, lists[..., 1])
    q, do = (rand((1, N, H * D), 90 + i, dt, "cuda") for i in range(2))
    k, v = (rand((1, N, Hk * D), 92 + i, dt, "cuda") for i in range(2))
    ql, kl, vl = (x.detach().requires_grad_(True) for x in (q, k, v))
    o, lse = fta.flash_topk_attn(ql, kl, vl, lists.cuda(), None, H, g, b, num_kv_heads=Hk)
    _check_grads((q, k, v, do), lists, torch.autograd.grad(o, (ql, kl, vl), do), H, Hk, D, g, b)
