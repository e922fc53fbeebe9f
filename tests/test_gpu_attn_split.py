"""Sparse-attention forward with few rows: each row's columns split over
several workgroups and combined (attn_plan, sparse_attn_combine_kernel).

Every case runs split (as the Python operators do) and unsplit (without the
scratch) and compares the two, and checks one against the double oracle.  The
bound between the two: P is rounded to the operand type relative to each
split's own maximum, 2^-9 (bf16) or 2^-12 (fp16) of each term, in both, and so
is the output: 4 such roundings in the 2-norm; lse is fp32 throughout.
Cases: the smallest split row, uneven last splits, splits without a valid key,
rows without any, row lengths that end inside a split, both index types,
strided index columns, two KV tensors, several head groups, partial heads.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle as O
from streamindex_amd import _lib, synth
from streamindex_amd.sparse_attn import sparse_attn_fwd, sparse_attn_fwd_kv2
from tests.conftest import bf16_bits

pytestmark = pytest.mark.gpu


def _both(monkeypatch, fn):
    split = fn()
    with monkeypatch.context() as m:
        m.setattr(_lib, "scratch", lambda n, d: (None, 0))
        whole = fn()
    torch.cuda.synchronize()
    return split, whole


def _close(split, whole, eps, label):
    (o, lse), (o1, lse1) = split, whole
    d = (o.double() - o1.double()).norm() / o1.double().norm().clamp(min=1e-30)
    assert d <= 4 * eps, f"{label}: {d:.2e}"
    assert torch.allclose(lse, lse1, rtol=1e-5, atol=1e-5), f"{label}: lse"


def _splits(B, S, H, D, K):
    n = _lib.load().si_sparse_attn_fwd_scratch_bytes(B, S, H, D, K)
    return n // (B * S * ((H + 63) // 64) * 64 * (D * 4 + 8))


@pytest.mark.parametrize("B,S,H,D,N,K,dt,i32", [
    (16, 1, 64, 576, 4096, 1024, torch.bfloat16, False),
    (1, 1, 64, 576, 300, 2048, torch.bfloat16, True),
    (2, 3, 64, 512, 1000, 1025, torch.float16, False),
    (1, 5, 130, 256, 700, 1200, torch.bfloat16, True),
    (3, 2, 16, 128, 999, 1640, torch.float16, True),
    (1, 2, 40, 64, 500, 2385, torch.bfloat16, False),
    (1, 1, 64, 32, 500, 4000, torch.bfloat16, False),
    (1, 128, 64, 576, 2000, 4100, torch.bfloat16, True),
])
def test_split_matches_whole(cuda_device, monkeypatch, B, S, H, D, N, K, dt, i32):
    assert _splits(B, S, H, D, K) > 1
    q, kv, sink = synth.sparse_attn_inputs(B, S, H, D, N, seed=K)
    q, kv = q.to(dt), kv.to(dt)
    g = torch.Generator().manual_seed(S)
    idx = torch.randint(0, N, (B, S, K), generator=g)
    idx[torch.rand(B, S, K, generator=g) < 0.1] = -1
    idx[:, -1, K // 3:] = -1                        # splits without a valid key
    if S > 1:
        idx[:, 0] = -1                              # a row without one
    idx = (idx.to(torch.int32) if i32 else idx).cuda()
    label = f"B={B},S={S},H={H},D={D},K={K}"
    split, whole = _both(monkeypatch, lambda: sparse_attn_fwd(q, kv, sink, idx))
    _close(split, whole, 2 ** -9 if dt == torch.bfloat16 else 2 ** -12, label)
    if S > 1:
        assert (split[0][:, 0] == 0).all() and torch.equal(split[1][:, 0], sink.expand(B, H)) or \
            torch.allclose(split[1][:, 0], sink.expand(B, H), atol=1e-6)
    if dt == torch.bfloat16:
        ro, rl = O.sparse_attn_rows(bf16_bits(q[0]), bf16_bits(kv[0]), sink.cpu().numpy(), idx[0].cpu().numpy(), D ** -0.5)
        assert np.abs(split[0][0].float().cpu().numpy() - ro).max() < 2e-2
        assert np.abs(split[1][0].cpu().numpy() - rl).max() < 2e-2
    wide = torch.empty(B, S, K, 2, dtype=idx.dtype, device="cuda")[..., 0].copy_(idx)  # strided columns
    again = sparse_attn_fwd(q, kv, sink, wide)
    assert torch.equal(again[0], split[0]) and torch.equal(again[1], split[1])


@pytest.mark.parametrize("n1,n2", [(300, 200), (0, 200), (300, 0)])
def test_split_two_tensors_and_row_lengths(cuda_device, monkeypatch, n1, n2):
    B, S, H, D, K = 2, 4, 64, 576, 1300
    assert _splits(B, S, H, D, K) > 1
    q, kv, sink = synth.sparse_attn_inputs(B, S, H, D, n1 + n2, seed=3)
    g = torch.Generator().manual_seed(4)
    idx = torch.randint(-1, n1 + n2, (B, S, K), generator=g).to(torch.int32).cuda()
    row_len = torch.tensor([[0, 1, 33, 1300], [97, 1299, 640, -5]], dtype=torch.int32).cuda()
    a, b = kv[:, :n1].contiguous(), kv[:, n1:].contiguous()
    split, whole = _both(monkeypatch, lambda: sparse_attn_fwd_kv2(q, a, b, sink, idx, row_len=row_len))
    _close(split, whole, 2 ** -9, f"kv2 {n1}+{n2}")
    one = sparse_attn_fwd(q, kv, sink, idx, row_len=row_len)
    assert torch.equal(one[0], split[0]) and torch.equal(one[1], split[1])


def test_large_logits_and_no_sink(cuda_device, monkeypatch):
    # maxima far apart between splits, and an empty sink
    B, S, H, D, N, K = 1, 2, 64, 128, 2400, 2400
    q, kv, _ = synth.sparse_attn_inputs(B, S, H, D, N, seed=8)
    kv[:, :800] *= 30
    sink = torch.full((H,), -float("inf"), device="cuda")
    idx = torch.arange(N, dtype=torch.int32, device="cuda").expand(B, S, K).contiguous()
    split, whole = _both(monkeypatch, lambda: sparse_attn_fwd(q, kv, sink, idx))
    _close(split, whole, 2 ** -9, "large logits")


@pytest.mark.parametrize("S", [1, 2, 7, 300, 513, 2049])
def test_rows_per_workgroup(cuda_device, S):
    # every row count per workgroup gives the rows' own results (a row does not depend on its workgroup)
    H, D, N, K = 64, 576, 512, 64
    q, kv, sink = synth.sparse_attn_inputs(1, S, H, D, N, seed=5)
    idx = torch.randint(0, N, (1, S, K), generator=torch.Generator().manual_seed(6)).cuda()
    o, lse = sparse_attn_fwd(q, kv, sink, idx)
    rep = torch.cat([q] * 5, 1), torch.cat([idx] * 5, 1)
    o5, lse5 = sparse_attn_fwd(rep[0], kv, sink, rep[1])
    assert torch.equal(o5, torch.cat([o] * 5, 1)) and torch.equal(lse5, torch.cat([lse] * 5, 1))
