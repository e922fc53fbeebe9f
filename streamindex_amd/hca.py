"""Heavily Compressed Attention (HCA) forward on MI355X.

Mirrors ``flash_sparse/hca.py:24-95`` (``build_hca_topk_idxs``,
``flash_hca_forward``).  HCA has no indexer: a query at position ``s``
attends to its sliding window of the uncompressed KV and to every causally
legal compressed entry (``m'·(i+1) - 1 <= s``), through the same
sparse-attention kernel as CSA.  The index rows are written by one HIP kernel
(one workgroup per query row) instead of the reference's torch
arange/where/cat passes.

``use_triton`` is accepted for compatibility and selects nothing (one HIP
implementation).  The backward knows the rows' structure too: it sums dkv for
128 keys and a block of queries at a time (``si_hca_attn_bwd``) instead of
sorting (query, slot) pairs by key.
"""

from __future__ import annotations

from typing import Optional

import torch

from . import _lib
from .csa import _launch_hca, _row_len
from .sparse_attn import _aligned, _bwd_workspace, sparse_attn_bwd, sparse_attn_fwd_kv2

__all__ = ["flash_hca_forward", "build_hca_topk_idxs", "hca_row_len"]


def build_hca_topk_idxs(*, B: int, seq_len: int, n_win: int, n_compressed: int, m_prime: int,
                        device: torch.device) -> torch.Tensor:
    """``[B, S, n_win + n_compressed]`` int32 HCA index rows (``hca.py:24-51``).

    Window columns ``s-n_win+1 .. s`` (``-1`` below 0), then compressed entry
    ``i`` as ``i + seq_len`` where ``m_prime·(i+1) - 1 <= s``, else ``-1``.
    """
    if n_win < 0 or n_compressed < 0 or m_prime <= 0:
        raise ValueError(f"bad HCA shape: n_win={n_win}, n_compressed={n_compressed}, m_prime={m_prime}")
    device = torch.device(device)
    assert device.type == "cuda"
    out = torch.empty((B, seq_len, n_win + n_compressed), dtype=torch.int32, device=device)
    _launch_hca(out, B, seq_len, n_win, n_compressed, m_prime, seq_len)
    return out


def flash_hca_forward(
    q: torch.Tensor,
    kv: torch.Tensor,
    kv_compressed: torch.Tensor,
    attn_sink: torch.Tensor,
    *,
    n_win: int,
    m_prime: int = 128,
    softmax_scale: Optional[float] = None,
    use_triton: bool = True,
) -> torch.Tensor:
    """End-to-end HCA forward, prefill path, one layer (``hca.py:54-95``).

    Args:
      q: ``[B, S, n_h, d]`` bf16.  kv: ``[B, S, d]`` bf16 uncompressed KV.
      kv_compressed: ``[B, S/m_prime, d]`` bf16.  attn_sink: ``[n_h]`` fp32.
      n_win: sliding-window size.  m_prime: HCA compression ratio.
      softmax_scale: defaults to ``d ** -0.5``.
    Returns:
      ``o: [B, S, n_h, d]`` bf16.
    """
    del use_triton
    B, S, n_h, d = q.shape
    n_compressed = kv_compressed.shape[1]
    assert q.is_cuda
    return _HcaAttnFunc.apply(q, kv, kv_compressed, attn_sink, softmax_scale, n_win, m_prime)


def _rows(B: int, S: int, n_win: int, n_compressed: int, m_prime: int, device):
    return (build_hca_topk_idxs(B=B, seq_len=S, n_win=n_win, n_compressed=n_compressed, m_prime=m_prime, device=device),
            hca_row_len(B, S, n_win, n_compressed, m_prime, device))


class _HcaAttnFunc(torch.autograd.Function):
    """HCA attention; the backward rebuilds what it needs of the index rows."""

    @staticmethod
    def forward(ctx, q, kv, kv_compressed, attn_sink, softmax_scale, n_win, m_prime):
        topk_idxs, row_len = _rows(q.shape[0], q.shape[1], n_win, kv_compressed.shape[1], m_prime, q.device)
        # the rows index [kv ; kv_compressed]; the kernel reads both in place
        o, lse = sparse_attn_fwd_kv2(q, kv, kv_compressed, attn_sink, topk_idxs, softmax_scale, row_len=row_len)
        ctx.save_for_backward(q, kv, kv_compressed, attn_sink, o, lse)
        ctx.args = (softmax_scale, n_win, m_prime)
        return o

    @staticmethod
    def backward(ctx, do):
        q, kv, kv_compressed, attn_sink, o, lse = ctx.saved_tensors
        dq, dkv, dsink = _hca_attn_bwd(q, torch.cat([kv, kv_compressed], dim=1), attn_sink, o, lse, do.contiguous(),
                                       kv_compressed.shape[1], *ctx.args)
        n1 = kv.shape[1]
        return dq, dkv[:, :n1], dkv[:, n1:], dsink, None, None, None


def _general_is_faster(rows: int, H: int, D: int, n_win: int, picks: float) -> bool:
    """Whether the general backward is faster than the aligned one for ``rows`` queries (batches included) with a window
    of ``n_win`` and ``picks`` compressed entries each on average.

    A 128-key group that a query meets costs the aligned path the same whatever it holds; a pair costs the general one a
    16-bit row, little at D <= 128.  So the keys per group decide, once the launches (twice as many in the general
    path) no longer count, and not with up to 32 heads, where the general path works in steps of 64.  us a step,
    general against aligned, m = 128 unless given:
      D = 64, 20,000 queries, H = 64: n_win = 16 (42 keys a group) 950, 1,262; 64 (55) 1,152, 1,347; 128 (66) 1,426, 1,396;
        n_win = 0, m = 32 (71) 859, 852; 4,000 queries, n_win = m = 64 480, 367; H = 32, 16,384 queries, m = 64 1,321, 915
      D = 128, 20,000 queries, H = 64: n_win = 16 (42) 1,480, 1,644; 64 (55) 1,785, 1,739; n_win = 128,
        m = 500 (52) 1,589, 1,716; H = 128 10,000 queries, n_win = 64 2,069, 1,442; nothing at D = 256."""
    least = 64 if D <= 64 else 53 if D == 128 and H <= 64 else 0
    groups = (1 + (n_win - 1) / 128 if n_win else 0) + (picks / 128 + 0.5 if picks else 0)
    return H > 32 and rows * ((H + 63) // 64) > 8192 and n_win + picks < least * groups


def _hca_attn_bwd(q, kv, attn_sink, o, lse, do, n_compressed, softmax_scale, n_win, m_prime):
    """``(dq, dkv, dsink)`` for ``kv = [kv ; kv_compressed]``, by ``si_hca_attn_bwd`` where it serves the shape (one kv row
    per query), is the faster one and its workspace fits the backward's cap, else by the general backward over the index
    rows."""
    B, S, H, D = q.shape
    N_kv = kv.shape[1]
    L = _lib.load()
    with _lib.on_device(q.device):
        ws = None
        picks = min(n_compressed, S // m_prime) / 2
        if N_kv == S + n_compressed and not _general_is_faster(B * S, H, D, min(n_win, S), picks):
            ws = _bwd_workspace(
                lambda cap: L.si_hca_attn_bwd_workspace_bytes(B, S, H, D, n_win, n_compressed, m_prime, cap), None, q.device)
        if ws is None:
            topk_idxs, row_len = _rows(B, S, n_win, n_compressed, m_prime, q.device)
            return sparse_attn_bwd(q, kv, attn_sink, topk_idxs, o, lse, do, softmax_scale, row_len=row_len)
        # (the stride of a single head is not used, and contiguous() would leave it as it is)
        q, o, do = (t if _aligned(t) and (H == 1 or 0 <= t.stride(2) < 1 << 24) else t.contiguous() for t in (q, o, do))
        attn_sink = attn_sink.contiguous()
        dq, dkv = torch.empty_like(q, memory_format=torch.contiguous_format), torch.empty_like(kv)
        dsink = torch.empty((H,), dtype=torch.float32, device=q.device)
        rc = L.si_hca_attn_bwd(
            q.data_ptr(), _lib.strides(q), kv.data_ptr(), _lib.strides(kv), attn_sink.data_ptr(), o.data_ptr(),
            _lib.strides(o), lse.data_ptr(), _lib.strides(lse), do.data_ptr(), _lib.strides(do), B, S, H, D, N_kv,
            n_win, n_compressed, m_prime, float(D ** -0.5 if softmax_scale is None else softmax_scale), _lib.qkv_dtype(q),
            dq.data_ptr(), _lib.strides(dq), dkv.data_ptr(), _lib.strides(dkv), dsink.data_ptr(), ws.data_ptr(),
            ws.numel(), _lib.stream_ptr(q.device))
    _lib.check(rc)
    return dq, dkv, dsink


def hca_row_len(B: int, S: int, n_win: int, n_compressed: int, m_prime: int, device) -> torch.Tensor:
    """``[B, S]`` int32 used columns of the HCA rows: the window, then the
    ``min(n_compressed, (s+1)//m_prime)`` legal compressed entries; the rest
    of each row is ``-1``, so attention never runs those tiles."""
    return _row_len(B, S, n_win, n_compressed, m_prime, device)
