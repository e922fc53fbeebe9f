"""Host side of the HCA backward (no kernel is launched): which calls take
si_hca_attn_bwd, and what that entry refuses.

si_hca_attn_bwd reads and writes rows 0 .. S + T - 1 of [kv ; kv_compressed],
so it serves calls with one kv row per query only; the forward takes any number
of kv rows (indices past them are masked), and so does the general backward.
"""

from __future__ import annotations

import contextlib
import ctypes
import os

import pytest
import torch

from streamindex_amd import _lib, hca
from streamindex_amd.build import LIB_PATH


class _Refused(Exception):
    pass


@pytest.mark.parametrize("n1", [1, 7, 9, 40])
def test_other_kv_lengths_take_the_general_backward(monkeypatch, n1):
    S, H, D, T = 8, 2, 32, 3

    class Lib:
        def si_hca_attn_bwd_workspace_bytes(self, *a):
            raise _Refused

    general = []
    monkeypatch.setattr(_lib, "load", lambda: Lib())
    monkeypatch.setattr(_lib, "on_device", lambda d: contextlib.nullcontext())
    monkeypatch.setattr(hca, "_rows", lambda *a: ("rows", "row_len"))
    monkeypatch.setattr(hca, "sparse_attn_bwd", lambda *a, **k: general.append((a, k)) or (1, 2, 3))

    def call(n):
        q = torch.zeros(1, S, H, D)
        kv = torch.zeros(1, n + T, D)
        return hca._hca_attn_bwd(q, kv, torch.zeros(H), q, torch.zeros(1, S, H), q, T, None, 4, 2)

    assert call(n1) == (1, 2, 3)
    (a, k), = general
    assert a[1].shape[1] == n1 + T and a[3] == "rows" and k["row_len"] == "row_len"
    with pytest.raises(_Refused):
        call(S)


def _entry(B, S, H, D, N, n_win, T, m, hs=None):
    if not os.path.exists(LIB_PATH):
        pytest.skip("libstreamindex.so not built (run __graft_entry__.build())")
    lib = _lib.load()
    i64 = lambda *v: (ctypes.c_int64 * len(v))(*v)  # noqa: E731
    hs = D if hs is None else hs
    q4 = i64(S * H * D, H * D, hs, 1)
    fake = 0x1000  # never dereferenced: every call below fails validation
    kv = i64(N * D, D, 1)
    rc = lib.si_hca_attn_bwd(fake, q4, fake, kv, fake, fake, q4, fake, i64(S * H, H, 1), fake, q4, B, S, H, D, N, n_win, T,
                             m, 0.1, 0, fake, q4, fake, kv, fake, fake, 0, None)
    return rc, lib.si_last_error().decode()


@pytest.mark.parametrize("N", [0, 1, 66, 68, 200])
def test_entry_refuses_other_row_counts(N):
    rc, msg = _entry(1, 64, 16, 64, N, 16, 3, 16)
    assert rc == _lib.SI_ERR_INVALID and "N_kv" in msg


def test_entry_takes_one_row_per_query():
    rc, msg = _entry(1, 64, 16, 64, 67, 16, 3, 16)  # (goes on to the workspace check)
    assert rc == _lib.SI_ERR_INVALID and "workspace" in msg


def test_row_lengths_on_the_default_device():
    from streamindex_amd.csa import csa_row_len

    want = 4 + torch.clamp((torch.arange(10) + 1) // 2, max=3)
    for got in (csa_row_len(2, 10, 4, 3, 5, 2, None), csa_row_len(2, 10, 4, 3, 5, 2, "cpu"),
                hca.hca_row_len(2, 10, 4, 3, 2, None)):
        assert got.dtype == torch.int32 and torch.equal(got, want.to(torch.int32).expand(2, 10))


def test_entry_ignores_the_stride_of_a_single_head():
    rc, msg = _entry(1, 64, 1, 64, 67, 16, 3, 16, hs=1 << 25)
    assert rc == _lib.SI_ERR_INVALID and "workspace" in msg
    rc, msg = _entry(1, 64, 2, 64, 67, 16, 3, 16, hs=1 << 25)
    assert rc == _lib.SI_ERR_UNSUPPORTED and "head stride" in msg


def _bytes(*a):
    if not os.path.exists(LIB_PATH):
        pytest.skip("libstreamindex.so not built (run __graft_entry__.build())")
    return _lib.load().si_hca_attn_bwd_workspace_bytes(*a)


@pytest.mark.parametrize("B,S,per", [(2, 16384, 1), (4, 8192, 2), (8, 4096, 4), (6, 8192, 3), (5, 8192, 3)])
def test_plan_takes_whole_batches(B, S, per):
    # 64 heads, D = 576, window and ratio 128: the default cap holds `per` whole batches in equal groups
    shape = (S, 64, 576, 128, S // 128, 128)
    group = _bytes(per, *shape, 1 << 40)
    assert group <= 2 << 30 < _bytes(B, *shape, 1 << 40)
    # the plan of a group, and the rest of the batches' dsink terms
    assert _bytes(B, *shape, 2 << 30) == group + (B - per) * S * 64 * 4


def test_plan_parts_are_equal():
    shape = (1, 20000, 64, 576, 128, 156, 128)
    whole = _bytes(*shape, 1 << 40)
    part = _bytes(*shape, whole - 1)
    acc = 20156 * 576 * 4
    assert part < 0.6 * whole + acc  # two halves, not all rows but one block and a rest


@pytest.mark.parametrize("shape", [(1, 5000, 64, 128, 100, 40, 125), (7, 700, 16, 64, 33, 60, 11), (3, 4097, 130, 576, 128, 32, 128)])
def test_plan_of_its_own_size_is_itself(shape):
    whole = _bytes(*shape, 1 << 40)
    sizes = {_bytes(*shape, int(whole * f)) for f in (0.9, 0.7, 0.5, 0.3, 0.2, 0.1, 0.05)} - {-1}
    assert len(sizes) > 2
    for n in sizes:
        assert _bytes(*shape, n) == n and n < whole


def test_plan_holds_one_chunk_of_index_rows():
    # past 215,000 tokens (64 heads, D = 576) the rows of the whole sequence alone fill the default cap
    S = 262144
    n = _bytes(1, S, 64, 576, 128, S // 128, 128, 2 << 30)
    assert 0 < n <= 2 << 30 < S * (160 + S // 128) * 4


def _plan_bytes(B, S, H, D, n_win, T, RB, rows=None):
    """Workspace of all batches in row blocks of RB, or of one batch in parts of `rows` rows."""
    nb, rows = (B, S) if rows is None else (1, rows)
    HG, wt = (H + 63) // 64, (n_win + 62) // 32 if n_win else 0
    GW, ncg = (RB + n_win - 2) // 128 + 2 if n_win else 0, (T + 127) // 128
    sizes = (B * S * 64 * HG * 4, (S + T) * D * 4 if rows < S else 0, rows * (32 * wt + T) * 4, rows * 4,
             nb * rows * HG * (wt + (T + 31) // 32) * 8192, nb * ((rows + RB - 1) // RB) * (GW + ncg) * 128 * D * 4)
    return sum((n + 255) // 256 * 256 for n in sizes)


@pytest.mark.parametrize("B,S,H,D,n_win,T,RB", [
    (1, 16384, 64, 576, 128, 128, 64),
    (1, 8200, 16, 512, 128, 64, 64),
    (1, 4096, 64, 576, 128, 32, 32),
    (1, 8192, 64, 256, 128, 64, 32),    # two workgroups a CU up to D = 256
    (2, 9000, 16, 64, 128, 1000, 64),
    (1, 300, 16, 64, 128, 2, 32),       # few stages a block: 32 rows at least
    (1, 300, 64, 576, 128, 2, 32),
    (4, 256, 128, 576, 16, 16, 16),
    (1, 300, 256, 64, 128, 2, 8),
    (1, 300, 600, 64, 128, 2, 8),
])
def test_row_blocks(B, S, H, D, n_win, T, RB):
    assert _bytes(B, S, H, D, n_win, T, 128, 1 << 40) == _plan_bytes(B, S, H, D, n_win, T, RB)


def test_row_blocks_of_parts():
    # 132 blocks of 64 rows in two parts; 16,384 tokens in parts of 1,024 rows take blocks of 32
    shape = (1, 8400, 4, 512, 128, 640)
    assert _bytes(*shape, 13, _plan_bytes(*shape, 64) - 1) == _plan_bytes(*shape, 64, 66 * 64)
    shape = (1, 16384, 64, 576, 128, 128)
    assert _bytes(*shape, 128, _plan_bytes(*shape, 32, 1024)) == _plan_bytes(*shape, 32, 1024)


@pytest.mark.parametrize("rows,H,D,n_win,picks,general", [
    (20000, 64, 64, 16, 78, True), (20000, 64, 64, 64, 78, True), (20000, 64, 64, 128, 78, False),
    (20000, 64, 64, 0, 78, False), (20000, 64, 64, 1, 0, True), (20000, 64, 32, 0, 0, False),
    (8192, 64, 64, 16, 78, False), (8193, 64, 64, 16, 78, True), (4097, 128, 32, 16, 20, True),
    (20000, 32, 64, 16, 78, False), (20000, 33, 64, 16, 78, True),
    (20000, 64, 128, 16, 78, True), (20000, 64, 128, 64, 78, False), (20000, 65, 128, 16, 78, False),
    (20000, 64, 256, 16, 78, False), (60000, 64, 576, 1, 20, False),
])
def test_few_keys_a_group_take_the_general_backward(rows, H, D, n_win, picks, general):
    assert hca._general_is_faster(rows, H, D, n_win, picks) == general
