"""Score blocks of 48 keys on the pipelined scorer, with per-block values."""

import numpy as np
import pytest
import torch

import fta_oracle as O
from _helpers import say
from test_gpu_parity import _pattern_qk

pytestmark = pytest.mark.gpu

fta = pytest.importorskip("flash_topk_attn_v2")

CASES = [
    # N, H, D, score padding, topk, threshold, pattern
    (4032, 2, 128, (0, 0), 16, 1.0, "increasing"),
    (4032, 2, 64, (0, 0), 8, 0.9, "decreasing"),
    (4032, 1, 128, (0, 0), 32, 1.0, "ties"),
    (4032, 2, 128, (0, 0), 16, 1.0, "jump"),  # the exact path inside the unrolled loop
    (4032, 1, 64, (0, 0), 24, 2.0, "cliff"),  # averages that underflow
    (4032, 2, 128, (0, 0), 16, 2.0, "step"),
    (4032, 2, 64, (0, 0), 32, 0.95, "uniform"),
    (5167, 2, 64, (40, 25), 5, 0.9, "peaked"),  # edge blocks of 8 and 23 keys
    (5167, 2, 128, (1, 16), 16, 0.9, "iid"),
    (1000, 2, 96, (47, 9), 12, 0.95, "iid"),  # a first block of one key
    (100, 2, 32, (0, 44), 3, 1.0, "iid"),  # three blocks, the last of 4 keys: rows past the sequence
    (48, 1, 128, (0, 0), 1, 1.0, "iid"),  # one block
    # one partial block (padded on one side: of a block padded on both, the oracle's valid
    # count leaves out the tail pad only, at every block size, where the kernels count both)
    (20, 1, 64, (28, 0), 2, 1.0, "iid"),
]


def _check(out, scores, thr, topk, pad):
    ref = O.topk_select(scores, thr, topk, 48, pad)
    for x, y in zip(out, ref):
        np.testing.assert_array_equal(x.cpu().numpy(), y)


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"N{c[0]}D{c[2]}k{c[4]}{c[6]}p{c[3][0]}")
def test_scores_b48(case):
    """Block scores against the float64 oracle (rtol 2e-4, as for every block size), and
    the fused top-k equal to the selection over them bit for bit."""
    N, H, D, pad, topk, thr, pattern = case
    say(f"[b48] {case}")
    q, k = _pattern_qk(N, H, D, pattern, 41, 48)
    scores = fta.flash_block_score(q, k, H, 48, pad).cpu().numpy()
    rows = np.unique(np.linspace(0, N - 1, 40).astype(int))
    ref = O.block_score(q.float().cpu().numpy(), k.float().cpu().numpy(), H, 48, pad, rows=rows)
    np.testing.assert_allclose(scores[:, :, rows], ref, rtol=2e-4, atol=1e-7)
    _check(fta.flash_topk_score(q, k, H, 48, topk, pad, thr), scores, thr, topk, pad)


@pytest.mark.parametrize("pattern,D", [("increasing", 128), ("ties", 64)])
def test_workspace_b48(pattern, D):
    """The sizes are those of the per-block values, and a workspace of that size serves
    any K token stride: the pipelined scorer (tokens in order) and the general one (tokens
    stored last to first) give the same lists.  The two halves of the stream path refuse
    48-key blocks."""
    from flash_topk_attn_v2 import _lib

    N, H, topk = 4032, 16, 2
    M = N // 48
    say(f"[b48 workspace] {pattern} D{D}")
    q, k = _pattern_qk(N, H, D, pattern, 43, 48)
    L = _lib.lib()
    al = lambda x: (x + 255) // 256 * 256  # noqa: E731
    nbytes = L.fta_topk_score_workspace_size_ex(1, H, N, D, 48, 0, 0, topk)
    assert nbytes == L.fta_topk_score_workspace_min(1, H, N, D, 48, 0, 0, topk)
    assert nbytes == al(H * M * N * 4) + 2 * al(H * N * 4)
    st = _lib.i64arr([N * H * D, D, H * D])
    back = _lib.i64arr([N * H * D, D, -H * D])
    kr = k.flip(1).contiguous()
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    want = fta.flash_topk_score(q, k, H, 48, topk)
    for kp, ks in ((k.data_ptr(), st), (kr.data_ptr() + 2 * (N - 1) * H * D, back)):
        out = [torch.full((1, H, N, topk), 7, dtype=t, device="cuda") for t in (torch.int32, torch.float32, torch.float32)]
        args = (q.data_ptr(), kp, 0, 1, H, N, D, st, ks, 48, 0, 0, D ** -0.5, topk)
        _lib.check(L.fta_topk_score(*args, 1.0, *(o.data_ptr() for o in out), ws.data_ptr(), nbytes, stream), "score")
        torch.cuda.synchronize()
        for x, y in zip(out, want):
            assert torch.equal(x, y)
        assert L.fta_topk_score_candidates(*args, ws.data_ptr(), nbytes, stream) == _lib.FTA_ERR_UNSUPPORTED
