"""Varlen causal paged prefill (HIP kernel (b)) vs the float64 oracle.

Covers a fresh prefix (cached_len 0), the reference test's offset case
(tests/test_attention_backend.py:25-53: seed 17, cached_len in {0, 2},
q_len 3, 4 query / 2 KV heads), the cross-keystroke extension (2 new tokens
against a cached 128-token prefix, Qwen3-0.6B heads), multi-request varlen
batches and a 4096-token prefill checked on sampled query rows.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from aios_amd import _lib, paged
from oracle import attention as oatt
from tests.util import BF16_TOL, to_np64

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _make(q_lens, kv_lens, hq, hkv, d, pool, seed):
    g = torch.Generator().manual_seed(seed)
    total_kv = sum(kv_lens)
    perm = torch.randperm(pool, generator=g)[:total_kv].to(torch.int32)
    cu_q = torch.zeros(len(q_lens) + 1, dtype=torch.int32)
    cu_q[1:] = torch.tensor(q_lens).cumsum(0)
    cu_k = torch.zeros(len(kv_lens) + 1, dtype=torch.int32)
    cu_k[1:] = torch.tensor(kv_lens).cumsum(0)
    q = (torch.randn(sum(q_lens), hq, d, generator=g) * 0.5).to(torch.bfloat16)
    kc = (torch.randn(pool, hkv, d, generator=g) * 0.5).to(torch.bfloat16)
    vc = (torch.randn(pool, hkv, d, generator=g) * 0.5).to(torch.bfloat16)
    return q, kc, vc, perm, cu_q, cu_k


def _run(q, kc, vc, idx, cu_q, cu_k, hq, hkv, d):
    p = paged.plan("prefill", cu_q, cu_k, hq, hkv, d)
    out = paged.prefill(p, q.to(DEV), kc.to(DEV), vc.to(DEV), idx.to(DEV), cu_q.to(DEV),
                        cu_k.to(DEV))
    torch.cuda.synchronize()
    return out, p


def _oracle(q, kc, vc, idx, cu_q, cu_k, d):
    return oatt.paged_attention(to_np64(q), to_np64(kc), to_np64(vc), idx.numpy(), cu_q.numpy(),
                                cu_k.numpy(), d ** -0.5)


@pytest.mark.parametrize("q_lens,kv_lens,hq,hkv,d", [
    ([32], [32], 8, 2, 96),            # MiniMind-0.1B-shaped prefix prefill
    ([64], [64], 12, 4, 64),           # deployed 0.1B heads (G=3)
    ([128], [128], 16, 8, 128),        # Qwen3-0.6B-shaped prefix
    ([2], [130], 16, 8, 128),          # cross-keystroke extension: 2 tokens vs cached 128
    ([1], [77], 8, 2, 96),             # single-token extension
    ([3, 1, 40, 17], [3, 9, 40, 50], 8, 2, 96),  # ragged batch, mixed cached_len
    ([100, 33], [131, 33], 32, 8, 128),
    ([5], [5], 8, 8, 64),
])
def test_prefill_matches_oracle(q_lens, kv_lens, hq, hkv, d):
    args = _make(q_lens, kv_lens, hq, hkv, d, pool=max(512, 2 * sum(kv_lens)), seed=sum(kv_lens) + d)
    q, kc, vc, idx, cu_q, cu_k = args
    out, _ = _run(q, kc, vc, idx, cu_q, cu_k, hq, hkv, d)
    np.testing.assert_allclose(to_np64(out), _oracle(q, kc, vc, idx, cu_q, cu_k, d), **BF16_TOL)


@pytest.mark.parametrize("cached_len", [0, 2])
def test_reference_offset_case(cached_len):
    # Structure of tests/test_attention_backend.py:25-53 (seed 17, q_len 3,
    # Hq 4, Hkv 2) at the smallest built head_dim.
    d = 64
    g = torch.Generator().manual_seed(17)
    q_len = 3
    kv_len = cached_len + q_len
    q = torch.randn(q_len, 4, d, generator=g).to(torch.bfloat16)
    k = torch.randn(kv_len, 2, d, generator=g).to(torch.bfloat16)
    v = torch.randn(kv_len, 2, d, generator=g).to(torch.bfloat16)
    idx = torch.arange(kv_len, dtype=torch.int32)
    cu_q = torch.tensor([0, q_len], dtype=torch.int32)
    cu_k = torch.tensor([0, kv_len], dtype=torch.int32)
    out, _ = _run(q, k, v, idx, cu_q, cu_k, 4, 2, d)
    expect = oatt.attention_one(to_np64(q), to_np64(k), to_np64(v), cached_len, d ** -0.5)
    np.testing.assert_allclose(to_np64(out), expect, **BF16_TOL)


def test_first_query_row_sees_only_first_key():
    # Causal closed form: with cached_len 0, query row 0 attends to key 0 only.
    q_lens, kv_lens = [50], [50]
    q, kc, vc, idx, cu_q, cu_k = _make(q_lens, kv_lens, 8, 2, 96, 256, seed=4)
    out, _ = _run(q, kc, vc, idx, cu_q, cu_k, 8, 2, 96)
    v0 = vc[idx[0].long()].float().repeat_interleave(4, dim=0)
    torch.testing.assert_close(out[0].float().cpu(), v0, atol=1e-2, rtol=1e-2)


def test_long_prefill_sampled_rows():
    # 4096-token prefill at Qwen3-4B heads; oracle on sampled query rows.
    hq, hkv, d, n = 32, 8, 128, 4096
    q, kc, vc, idx, cu_q, cu_k = _make([n], [n], hq, hkv, d, pool=65536, seed=4096)
    out, p = _run(q, kc, vc, idx, cu_q, cu_k, hq, hkv, d)
    assert p.num_q_tiles * p.prefill_q_tile >= n
    rows = [0, 1, 31, 32, 33, 127, 1000, 2047, 4095]
    qn, kn, vn = to_np64(q), to_np64(kc[idx.long()]), to_np64(vc[idx.long()])
    got = to_np64(out)
    for i in rows:
        ref = oatt.attention_one(qn[i : i + 1], kn[: i + 1], vn[: i + 1], i, d ** -0.5)
        np.testing.assert_allclose(got[i : i + 1], ref, **BF16_TOL)


@pytest.mark.parametrize("q_lens,kv_lens,hq,hkv,d", [([512], [512], 32, 8, 128),
                                                     ([2, 300], [130, 600], 16, 8, 128),
                                                     ([200], [200], 8, 2, 96)])
def test_growing_logits_move_the_softmax_reference(q_lens, kv_lens, hq, hkv, d):
    # K rows scaled up along each request's positions (x1 to x51): a query
    # row's running max keeps growing over its causal range, so the
    # reference moves mid-stream and rescales O and the MFMA row sums.
    q, kc, vc, idx, cu_q, cu_k = _make(q_lens, kv_lens, hq, hkv, d, 4096, seed=29)
    scale = torch.ones(kc.shape[0])
    for r in range(len(kv_lens)):
        lo, hi = int(cu_k[r]), int(cu_k[r + 1])
        scale[idx[lo:hi].long()] = 1.0 + 50.0 * torch.arange(hi - lo, dtype=torch.float32) / (hi - lo)
    kc = (kc.float() * scale.view(-1, 1, 1)).to(torch.bfloat16)
    out, _ = _run(q, kc, vc, idx, cu_q, cu_k, hq, hkv, d)
    np.testing.assert_allclose(to_np64(out), _oracle(q, kc, vc, idx, cu_q, cu_k, d), **BF16_TOL)


@pytest.mark.parametrize("q_lens,kv_lens,hq,hkv,d", [
    ([1], [289], 8, 8, 64),                    # few rows: the shortest split range, one row
                                               # (up to 288 positions one workgroup is faster)
    ([8], [513], 32, 8, 128),                  # one full 32-row tile, one position over a part
    ([9], [1000], 32, 8, 128),                 # 36 rows: two row tiles, half the wavefronts each
    ([16, 1, 3], [900, 300, 40], 8, 2, 96),    # ragged few-row batch, one tile unsplit
    ([21], [2100], 12, 4, 64),                 # G = 3: 63 rows
    ([10], [700], 48, 8, 64),                  # G = 6
    ([65], [1400], 16, 8, 128),                # fuller tiles (ring path), a second short tile
    ([150, 33], [1500, 1033], 8, 2, 96),
    ([300], [1300], 12, 4, 64),
])
def test_split_kv_ranges_match_oracle(q_lens, kv_lens, hq, hkv, d):
    # Batches whose tiles' KV ranges are split over workgroups; K rows grow
    # along the positions, so the parts' softmax references differ widely.
    q, kc, vc, idx, cu_q, cu_k = _make(q_lens, kv_lens, hq, hkv, d, 4096, seed=sum(kv_lens))
    scale = torch.ones(kc.shape[0])
    for r in range(len(kv_lens)):
        lo, hi = int(cu_k[r]), int(cu_k[r + 1])
        scale[idx[lo:hi].long()] = 1.0 + 20.0 * torch.arange(hi - lo, dtype=torch.float32) / (hi - lo)
    kc = (kc.float() * scale.view(-1, 1, 1)).to(torch.bfloat16)
    out, p = _run(q, kc, vc, idx, cu_q, cu_k, hq, hkv, d)
    assert p.num_parts > 1 and p.ws_bytes > 0
    ref = _oracle(q, kc, vc, idx, cu_q, cu_k, d)
    np.testing.assert_allclose(to_np64(out), ref, **BF16_TOL)
    # a plan for longer ranges (a replayed prefill's capacity) on the same batch
    cap = cu_k.clone()
    cap[1:] += 320 * torch.arange(1, len(cap), dtype=torch.int32)
    wide = paged.plan("prefill", cu_q, cap, hq, hkv, d)
    roomy = torch.zeros(int(cap[-1]), dtype=torch.int32)
    roomy[: idx.numel()] = idx
    out = paged.prefill(wide, q.to(DEV), kc.to(DEV), vc.to(DEV), roomy.to(DEV), cu_q.to(DEV),
                        cu_k.to(DEV))
    np.testing.assert_allclose(to_np64(out), ref, **BF16_TOL)
    # a plan without room for the states keeps one workgroup per tile
    small = paged.plan("prefill", cu_q, cu_k, hq, hkv, d, workspace_bytes=1024)
    assert small.num_parts == 0 and small.ws_bytes == 0
    out = paged.prefill(small, q.to(DEV), kc.to(DEV), vc.to(DEV), idx.to(DEV), cu_q.to(DEV),
                        cu_k.to(DEV))
    np.testing.assert_allclose(to_np64(out), ref, **BF16_TOL)


@pytest.mark.parametrize("planned,q_lens,kv_lens,hq,hkv,d", [
    ([2, 2], [1, 3], [600, 600], 8, 2, 96),      # 12 rows in parts made for 8
    ([8, 8], [1, 15], [900, 700], 32, 8, 128),   # 60 rows in parts made for 32
    ([20, 20], [30, 10], [900, 1100], 8, 2, 64), # 120 rows in parts made for 80
])
def test_tiles_fuller_than_planned(planned, q_lens, kv_lens, hq, hkv, d):
    # The lengths on the device put more rows in a tile than the plan's parts
    # have room for: that tile is computed whole, as without the split.
    q, kc, vc, idx, cu_q, cu_k = _make(q_lens, kv_lens, hq, hkv, d, 4096, seed=sum(kv_lens))
    p = paged.plan("prefill", [0, planned[0], sum(planned)], cu_k, hq, hkv, d)
    assert p.num_parts > 1 and p.max_q_len < max(q_lens)
    out = paged.prefill(p, q.to(DEV), kc.to(DEV), vc.to(DEV), idx.to(DEV), cu_q.to(DEV),
                        cu_k.to(DEV))
    np.testing.assert_allclose(to_np64(out), _oracle(q, kc, vc, idx, cu_q, cu_k, d), **BF16_TOL)


def test_unaligned_workspace_runs_unsplit():
    q, kc, vc, idx, cu_q, cu_k = _make([6], [900], 8, 2, 96, 4096, seed=5)
    p = paged.plan("prefill", cu_q, cu_k, 8, 2, 96)
    assert p.num_parts > 1
    on = [t.to(DEV) for t in (q, kc, vc, idx, cu_q, cu_k)]
    ws = torch.full((p.ws_bytes + 256,), 85, dtype=torch.uint8, device=DEV)
    out = torch.empty_like(on[0])
    _lib.check(_lib.lib().aios_attn_prefill_ws(
        p, on[0].data_ptr(), on[0].stride(0), on[1].data_ptr(), on[2].data_ptr(), kc.shape[0],
        on[3].data_ptr(), on[4].data_ptr(), on[5].data_ptr(), out.data_ptr(), ws.data_ptr() + 64,
        p.ws_bytes, 96 ** -0.5, 0), "prefill")
    torch.cuda.synchronize()
    assert bool((ws == 85).all())
    np.testing.assert_allclose(to_np64(out), _oracle(q, kc, vc, idx, cu_q, cu_k, 96), **BF16_TOL)
