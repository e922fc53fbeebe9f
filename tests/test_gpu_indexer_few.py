"""The two-pass top-k for few query rows over many keys (indexer_topk_few.h).

Calls with at most 256 four-row groups and 1,024 or more keys (few_worth draws
the line more closely), without a causal ratio, write their scores to a scratch
and select with one workgroup per row (and segment of 16,384 keys).  Scores are formed by the same fp32
operations and ranked by the same keys as in the one-wave-per-row kernel, so
every case compares the two for exact equality; two also go through the
oracle gate of tests/indexer_check.py.  Cases: both score kernels (below and
from 8 rows per batch), each register / sort width of the selection and their
edges, T not a multiple of a 32-key block or a tile, masks down to empty rows,
rows with more equal scores than the sort holds, and rows of several segments.
"""

from __future__ import annotations

import pytest
import torch

from streamindex_amd import _lib, chunked_indexer_topk, synth
from tests.indexer_check import check_indexer

pytestmark = pytest.mark.gpu


@pytest.fixture
def narrow(cuda_device):
    """fn() under the one-wave-per-row kernel."""
    def run(fn):
        _lib.load().si_indexer_set_topk_kernel(1)
        try:
            return fn()
        finally:
            _lib.load().si_indexer_set_topk_kernel(0)
    yield run
    _lib.load().si_indexer_set_topk_kernel(0)


def _same(run, narrow, label):
    a, b = run(), narrow(run)
    torch.cuda.synchronize()
    for x, y, name in zip(a, b, ("indices", "scores")):
        assert torch.equal(x, y), f"{label}: {name} differ from the one-wave-per-row kernel"
    return a


def _uses_scratch(B, S, T, H, D, k):
    return _lib.load().si_indexer_topk_scratch_bytes(B, S, T, H, D, k, 0) > 0


@pytest.mark.parametrize("B,S,T,H,D,k,wdt", [
    (1, 1, 1024, 64, 128, 512, torch.float32),
    (4, 1, 4096, 64, 128, 512, torch.float32),
    (3, 2, 4097, 33, 128, 513, torch.bfloat16),
    (1, 7, 16385, 64, 128, 1024, torch.float32),
    (2, 8, 16384, 64, 128, 1025, torch.float32),
    (1, 9, 8257, 128, 128, 2048, torch.float32),
    (1, 131, 3001, 16, 64, 64, torch.bfloat16),
    (1, 512, 1300, 100, 32, 1, torch.float32),
    (2, 1, 65536, 64, 128, 512, torch.float32),
    (5, 3, 2049, 40, 256, 600, torch.float32),
])
def test_matches_one_wave_per_row(narrow, B, S, T, H, D, k, wdt):
    assert _uses_scratch(B, S, T, H, D, k)
    q, ki, w = synth.indexer_inputs(B, S, H, D, T, seed=T + k, weights_dtype=wdt)
    label = f"B={B},S={S},T={T},H={H},D={D},k={k}"
    idx, sc = _same(lambda: chunked_indexer_topk(q, ki, w, k), narrow, label)
    if T == 16385 or T == 3001:
        check_indexer(q, ki, w, k, idx, sc, label=label)


@pytest.mark.parametrize("T,k", [(65537, 512), (200000, 2048)])
def test_several_segments(narrow, T, k):
    assert _uses_scratch(1, 2, T, 32, 32, k)
    q, ki, w = synth.indexer_inputs(1, 2, 32, 32, T, seed=T)
    _same(lambda: chunked_indexer_topk(q, ki, w, k), narrow, f"T={T}")


@pytest.mark.parametrize("S,T", [(2, 5000), (40, 5000), (2, 70000)])
def test_masks(narrow, S, T):
    q, ki, w = synth.indexer_inputs(1, S, 64, 128, T, seed=S)
    g = torch.Generator().manual_seed(S)
    mask = (torch.rand(1, S, T, generator=g) < 0.5).cuda()
    mask[:, 0] = False            # no legal key
    mask[:, 1] = False
    mask[:, 1, T - 100:] = True   # fewer legal keys than top_k
    idx, _ = _same(lambda: chunked_indexer_topk(q, ki, w, 512, causal_mask=mask), narrow, f"S={S},T={T}")
    assert (idx[:, 0] == -1).all()
    view = torch.empty(1, S, T, 2, dtype=torch.bool, device="cuda")[..., 0].copy_(mask)  # strided columns
    got, _ = chunked_indexer_topk(q, ki, w, 512, causal_mask=view)
    assert torch.equal(got, idx)


@pytest.mark.parametrize("T,distinct", [(16384, 1), (16384, 4), (4096, 3), (70001, 2)])
def test_ties(narrow, T, distinct):
    # more keys share a score than the sort holds: ties rank the smaller index first
    g = torch.Generator().manual_seed(distinct)
    base = torch.randn(distinct, 64, generator=g).to(torch.bfloat16)
    ki = base[torch.randint(0, distinct, (T,), generator=g)].unsqueeze(0).cuda()
    q = torch.randn(1, 2, 32, 64, generator=g).to(torch.bfloat16).cuda()
    w = torch.randn(1, 2, 32, generator=g).cuda()
    _same(lambda: chunked_indexer_topk(q, ki, w, 300), narrow, f"T={T},distinct={distinct}")


def test_plan_lines(cuda_device):
    assert not _uses_scratch(1, 1, 1023, 64, 128, 512)       # short rows
    assert not _uses_scratch(257, 1, 4096, 64, 128, 512)     # enough rows to fill the GPU
    assert not _uses_scratch(1, 1, 1 << 19, 64, 128, 2048)   # more segments than the merge holds
    assert not _uses_scratch(1, 1, 4096, 64, 128, 2049)      # head-split shapes
    assert not _uses_scratch(1, 1, 4096, 192, 128, 512)
    assert _lib.load().si_indexer_topk_scratch_bytes(1, 512, 4096, 64, 128, 512, 4) == 0


@pytest.mark.parametrize("B,S,T,H,D,k,few", [
    (256, 1, 30000, 64, 128, 512, True),     # rows, not groups, below 8 rows a batch
    (64, 7, 30000, 64, 128, 512, False),
    (256, 4, 4096, 32, 128, 512, False),
    (128, 1, 30000, 64, 256, 512, True),     # D = 256 and three or four head blocks fill the chip earlier
    (129, 1, 30000, 64, 256, 512, False),
    (1, 512, 30000, 64, 256, 512, True),
    (1, 516, 30000, 64, 256, 512, False),
    (1, 1024, 4096, 128, 128, 512, True),
    (1, 1024, 8192, 128, 128, 512, False),
    (1, 1, 1024, 32, 128, 128, False),       # short rows of few picks
    (1, 1, 2048, 32, 128, 128, True),
    (1, 1024, 2048, 64, 128, 16, False),
    (1, 1024, 4096, 64, 128, 16, True),
])
def test_plan_lines_of_rows_heads_and_picks(cuda_device, B, S, T, H, D, k, few):
    assert _uses_scratch(B, S, T, H, D, k) == few


@pytest.mark.parametrize("T,k", [(4096, 300), (16384, 512), (40000, 512)])
def test_scores_that_are_not_finite(narrow, T, k):
    # infinities and NaN among the scores, in rows of every kind of them: the order of their bits, as in the other kernel
    S, H, D = 6, 32, 64
    q, ki, w = synth.indexer_inputs(1, S, H, D, T, seed=T)
    g = torch.Generator().manual_seed(T)
    at = torch.randperm(T, generator=g)[:900]
    ki[0, at[:300].cuda(), 0] = float("inf")
    ki[0, at[300:600].cuda(), 1] = float("-inf")
    q[0, 1, :, :2] = 0.5                   # +inf and -inf scores
    q[0, 2, :, :2] = 0                     # 0 times infinity
    w[0, 3] = -w[0, 3].abs()               # -inf
    w[0, 4, 0] = float("nan")              # a row of NaN
    w[0, 5] = 0                            # zeros and NaN
    a, b = chunked_indexer_topk(q, ki, w, k), narrow(lambda: chunked_indexer_topk(q, ki, w, k))
    assert torch.equal(a[0], b[0])
    assert torch.equal(a[1].view(torch.int32), b[1].view(torch.int32))
    assert not torch.isfinite(a[1]).all()
