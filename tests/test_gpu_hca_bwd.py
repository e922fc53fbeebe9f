"""Backward of the HCA composition (si_hca_attn_bwd) against the general
sparse-attention backward over the same index rows.

Both round P and dS to the operand type; the general path also rounds each
(query, slot) dkv row to it before the fp32 sum, 2^-9 (bf16) of each term, so
dkv may differ by that in the 2-norm plus the final rounding, dq and dsink (the
same arithmetic over differently aligned tiles) by less: 2^-8 (bf16) and 2^-11
(fp16) bound all of them.  One case also goes through the double oracle.
Cases: windows of every alignment against the 32-key tiles (none, one key, a
tile more or less a key), no compressed entries, entries past the last legal
one, ragged sequences, several head groups and partial heads, every D, two
batches, each row-block size, and workspaces that force several chunks.
"""

from __future__ import annotations

import sys

import numpy as np
import pytest
import torch

from oracle import oracle as O
from streamindex_amd import flash_hca_forward, sparse_attn_bwd, sparse_attn_fwd, synth
from streamindex_amd import _lib, hca
from tests.conftest import bf16_bits

pytestmark = pytest.mark.gpu


def _inputs(B, S, H, D, T, dt, seed):
    q, kv, kvc, sink = synth.csa_attn_inputs(B, S, H, D, T, seed=seed, scale=0.7)
    g = torch.Generator().manual_seed(seed)
    do = (torch.randn(B, S, H, D, generator=g) * 0.5).to(dt).cuda()
    return q.to(dt), kv.to(dt), kvc.to(dt), sink, do


def _grads(q, kv, kvc, sink, do, n_win, m):
    leaves = [t.clone().requires_grad_(True) for t in (q, kv, kvc, sink)]
    o = flash_hca_forward(*leaves, n_win=n_win, m_prime=m)
    return torch.autograd.grad(o, leaves, do)


def _general(q, kv, kvc, sink, do, n_win, m):
    B, S = q.shape[:2]
    rows, row_len = hca._rows(B, S, n_win, kvc.shape[1], m, q.device)
    full = torch.cat([kv, kvc], 1)
    o, lse = sparse_attn_fwd(q, full, sink, rows, row_len=row_len)
    dq, dkv, ds = sparse_attn_bwd(q, full, sink, rows, o, lse, do, row_len=row_len)
    return dq, dkv[:, :S], dkv[:, S:], ds


def _check(got, ref, eps, label):
    for x, y, name in zip(got, ref, ("dq", "dkv", "dkv_compressed", "dsink")):
        assert x.shape == y.shape and x.dtype == y.dtype
        d = (x.double() - y.double()).norm()
        assert d <= eps * y.double().norm() + 1e-30, f"{label} {name}: {d / y.double().norm():.2e}"


@pytest.mark.parametrize("B,S,H,D,n_win,T,m,dt", [
    (1, 300, 64, 576, 128, 2, 128, torch.bfloat16),
    (1, 257, 16, 64, 1, 16, 16, torch.bfloat16),
    (2, 193, 64, 128, 31, 24, 8, torch.bfloat16),
    (1, 200, 130, 64, 33, 70, 2, torch.bfloat16),     # three head groups, two compressed groups
    (1, 130, 64, 512, 64, 33, 4, torch.float16),
    (1, 65, 40, 32, 200, 9, 7, torch.float16),        # window longer than the sequence
    (2, 96, 64, 256, 0, 96, 1, torch.bfloat16),       # compressed entries only
    (1, 150, 64, 64, 40, 0, 128, torch.bfloat16),     # window only
    (1, 90, 64, 128, 16, 50, 4, torch.bfloat16),      # entries past the last legal one
    (1, 1, 64, 576, 128, 0, 128, torch.bfloat16),
    (1, 4000, 16, 64, 128, 31, 128, torch.bfloat16),
    (1, 8200, 16, 512, 128, 64, 128, torch.bfloat16),  # blocks of 64 rows, the last one of 8
    (2, 6150, 4, 32, 128, 1000, 6, torch.float16),     # the same, one batch at a time
    (1, 330, 128, 576, 128, 2, 128, torch.bfloat16),   # blocks of 16
    (1, 77, 300, 64, 40, 9, 8, torch.float16),         # blocks of 8
])
def test_matches_general_backward(cuda_device, B, S, H, D, n_win, T, m, dt):
    assert _lib.load().si_hca_attn_bwd_workspace_bytes(B, S, H, D, n_win, T, m, 1 << 31) > 0
    x = _inputs(B, S, H, D, T, dt, S + D)
    got = _grads(*x, n_win, m)
    eps = 2 ** -8 if dt == torch.bfloat16 else 2 ** -11
    label = f"B={B},S={S},H={H},D={D},n_win={n_win},T={T},m={m}"
    _check(got, _general(*x, n_win, m), eps, label)
    again = _grads(*x, n_win, m)
    assert all(torch.equal(a, b) for a, b in zip(got, again)), f"{label}: not deterministic"


@pytest.mark.parametrize("B,S,chunks", [(1, 1000, 3), (2, 500, 4), (2, 130, 2)])
def test_chunks(cuda_device, monkeypatch, B, S, chunks):
    H, D, n_win, T, m = 64, 128, 50, 40, 12
    x = _inputs(B, S, H, D, T, torch.bfloat16, S)
    whole = _grads(*x, n_win, m)
    L = _lib.load()
    need = L.si_hca_attn_bwd_workspace_bytes(B, S, H, D, n_win, T, m, 1 << 40)
    cap = need // chunks + (B * S * 64 * 4 + S * (64 + 64 + T) * 4 + B * (S + T) * D * 4)
    assert 0 < L.si_hca_attn_bwd_workspace_bytes(B, S, H, D, n_win, T, m, cap) < need
    monkeypatch.setattr(sys.modules[sparse_attn_bwd.__module__], "BWD_WORKSPACE_CAP", cap)
    got = _grads(*x, n_win, m)
    assert torch.equal(got[0], whole[0]) and torch.equal(got[3], whole[3])
    _check(got, whole, 2 ** -8, f"chunks of B={B},S={S}")


def test_falls_back_below_one_chunk(cuda_device, monkeypatch):
    # no plan fits: the general backward runs
    x = _inputs(1, 64, 16, 64, 4, torch.bfloat16, 5)
    monkeypatch.setattr(_lib.load(), "si_hca_attn_bwd_workspace_bytes", lambda *a: -1)
    _check(_grads(*x, 16, 16), _general(*x, 16, 16), 0.0, "general")


def test_oracle(cuda_device):
    B, S, H, D, n_win, T, m = 1, 400, 64, 64, 100, 50, 8
    q, kv, kvc, sink, do = _inputs(B, S, H, D, T, torch.bfloat16, 9)
    dq, dkv, dkvc, ds = _grads(q, kv, kvc, sink, do, n_win, m)
    full = torch.cat([kv, kvc], 1)
    rows, row_len = hca._rows(B, S, n_win, T, m, q.device)
    o, lse = sparse_attn_fwd(q, full, sink, rows, row_len=row_len)
    rdq, rdkv, rds = O.sparse_attn_bwd_rows(bf16_bits(q[0]), bf16_bits(full[0]), bf16_bits(o[0]), bf16_bits(do[0]),
                                            sink.cpu().numpy(), lse[0].cpu().numpy(),
                                            rows[0].cpu().numpy().astype(np.int64), D ** -0.5)
    for x, y in ((dq[0], rdq), (dkv[0], rdkv[:S]), (dkvc[0], rdkv[S:])):
        assert np.linalg.norm(x.float().cpu().numpy() - y) <= 1e-2 * np.linalg.norm(y)
    assert np.abs(ds.cpu().numpy() - rds).max() <= 1e-3 * max(1.0, np.abs(rds).max())


@pytest.mark.parametrize("n1", [60, 99, 101, 150])
def test_kv_of_another_length(cuda_device, n1):
    # (the general backward serves these: the aligned kernels assume a kv row per query)
    B, S, H, D, T, n_win, m = 2, 100, 16, 64, 12, 24, 8
    q, _, kvc, sink, do = _inputs(B, S, H, D, T, torch.bfloat16, n1)
    kv = synth.csa_attn_inputs(B, n1, H, D, T, seed=n1, scale=0.7)[1]
    got = _grads(q, kv, kvc, sink, do, n_win, m)
    rows, row_len = hca._rows(B, S, n_win, T, m, q.device)
    full = torch.cat([kv, kvc], 1)
    o, lse = sparse_attn_fwd(q, full, sink, rows, row_len=row_len)
    dq, dkv, ds = sparse_attn_bwd(q, full, sink, rows, o, lse, do, row_len=row_len)
    _check(got, (dq, dkv[:, :n1], dkv[:, n1:], ds), 0.0, f"{n1} kv rows")


def test_single_head_with_a_long_stride(cuda_device):
    # one head of a [B, H, S, D] tensor seen as [B, S, H, D]: at S x D >= 2^24 its head stride passes the
    # kernels' 32-bit head offsets, which a single head does not use
    B, S, H, D, T, n_win, m = 1, 70, 1, 64, 4, 24, 16
    q, kv, kvc, sink, do = _inputs(B, S, H, D, T, torch.bfloat16, 3)
    long = q.as_strided(q.shape, (S * D, D, 1 << 25, 1))
    leaves = [t.detach().requires_grad_(True) for t in (long, kv, kvc, sink)]
    o = flash_hca_forward(*leaves, n_win=n_win, m_prime=m)
    got = torch.autograd.grad(o, leaves, do.as_strided(do.shape, long.stride()))
    assert all(torch.equal(x, y) for x, y in zip(got, _grads(q, kv, kvc, sink, do, n_win, m)))


def _same_spread(got, ref, eps, label):
    """Not finite in the same places, equal elsewhere."""
    for x, y, name in zip(got, ref, ("dq", "dkv", "dkv_compressed", "dsink")):
        fin = torch.isfinite(y)
        assert torch.equal(torch.isfinite(x), fin), f"{label} {name}: not finite elsewhere"
        _check((torch.where(fin, x, 0),), (torch.where(fin, y, 0),), eps, f"{label} {name}")


@pytest.mark.parametrize("D,n_win,T,m,H", [(64, 40, 20, 8, 20), (576, 128, 2, 128, 64), (32, 0, 60, 4, 16),
                                           (256, 33, 0, 1, 130)])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_non_finite_rows_stay_with_their_keys(cuda_device, D, n_win, T, m, H, value):
    # one element of one query's q, and of another's do: only the keys that these queries attend to take it up
    B, S = 2, 300
    q, kv, kvc, sink, do = _inputs(B, S, H, D, T, torch.bfloat16, D)
    q[0, 100, H - 1, 3] = value
    do[1, 250, 0, D - 1] = value
    x = (q, kv, kvc, sink, do)
    ref = _general(*x, n_win, m)
    assert all((~torch.isfinite(r)).any() and torch.isfinite(r).any() for r in ref[:1 + (n_win > 0)])
    _same_spread(_grads(*x, n_win, m), ref, 2 ** -8, f"D={D},n_win={n_win},T={T}")


@pytest.mark.parametrize("n_win,T,m", [(64, 0, 4), (32, 32, 1), (0, 32, 2)])
def test_non_finite_keys_stay_with_their_rows(cuda_device, n_win, T, m):
    # a masked slot gathers some row in its place, whose infinities times a weight of 0 must not reach dq
    B, S, H, D = 1, 300, 16, 64
    x = _inputs(B, S, H, D, T, torch.bfloat16, n_win)
    x[1][0, 0] = float("inf")
    if T:
        x[2][0, 7] = float("nan")
    got, ref = _grads(*x, n_win, m), _general(*x, n_win, m)
    for s in range(S):
        if torch.isfinite(ref[0][0, s]).all():
            assert torch.isfinite(got[0][0, s]).all(), f"dq of query {s}"
    keys = [torch.isfinite(r).all(dim=2)[0] for r in ref[1:3]]
    assert all((torch.isfinite(g).all(dim=2)[0] | ~k).all() for g, k in zip(got[1:3], keys))


@pytest.mark.parametrize("B,per,S,H,D,n_win,T,m", [(3, 2, 130, 64, 128, 50, 10, 12), (5, 1, 96, 16, 576, 128, 3, 32)])
def test_groups_of_batches(cuda_device, monkeypatch, B, per, S, H, D, n_win, T, m):
    # whole batches at a time, the last group shorter: the same sums
    x = _inputs(B, S, H, D, T, torch.bfloat16, B)
    whole = _grads(*x, n_win, m)
    L = _lib.load()
    group = L.si_hca_attn_bwd_workspace_bytes(per, S, H, D, n_win, T, m, 1 << 40)
    cap = group + B * S * 64 * 4
    assert group < L.si_hca_attn_bwd_workspace_bytes(B, S, H, D, n_win, T, m, cap) <= cap
    monkeypatch.setattr(sys.modules[sparse_attn_bwd.__module__], "BWD_WORKSPACE_CAP", cap)
    assert all(torch.equal(a, b) for a, b in zip(_grads(*x, n_win, m), whole))


def test_chunks_of_rows_at_d576(cuda_device, monkeypatch):
    # two batches of several chunks each, the last chunk's last block short
    B, S, H, D, n_win, T, m = 2, 1000, 16, 576, 128, 8, 128
    x = _inputs(B, S, H, D, T, torch.bfloat16, 7)
    whole = _grads(*x, n_win, m)
    L = _lib.load()
    one = L.si_hca_attn_bwd_workspace_bytes(1, S, H, D, n_win, T, m, 1 << 40)
    cap = one // 2 + (S + T) * D * 4
    assert 0 < L.si_hca_attn_bwd_workspace_bytes(B, S, H, D, n_win, T, m, cap) < one
    monkeypatch.setattr(sys.modules[sparse_attn_bwd.__module__], "BWD_WORKSPACE_CAP", cap)
    got = _grads(*x, n_win, m)
    assert torch.equal(got[0], whole[0]) and torch.equal(got[3], whole[3])
    _check(got, whole, 2 ** -8, "chunks at D = 576")


def test_chunks_of_64_row_blocks(cuda_device, monkeypatch):
    # two parts of a batch, blocks of 64 rows in both
    B, S, H, D, n_win, T, m = 1, 8400, 4, 512, 128, 640, 13
    x = _inputs(B, S, H, D, T, torch.bfloat16, 11)
    whole = _grads(*x, n_win, m)
    L = _lib.load()
    need = L.si_hca_attn_bwd_workspace_bytes(B, S, H, D, n_win, T, m, 1 << 40)
    got = L.si_hca_attn_bwd_workspace_bytes(B, S, H, D, n_win, T, m, need - 1)
    assert 0 < got < 0.6 * need
    monkeypatch.setattr(sys.modules[sparse_attn_bwd.__module__], "BWD_WORKSPACE_CAP", need - 1)
    part = _grads(*x, n_win, m)
    assert torch.equal(part[0], whole[0]) and torch.equal(part[3], whole[3])
    _check(part, whole, 2 ** -8, "parts of 64-row blocks")
