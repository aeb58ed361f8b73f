"""Decoder-layer kernels (aios_rmsnorm, aios_qk_norm_rope, aios_silu_mul) vs
the torch formulas of the reference layers on the same bf16 inputs."""
from __future__ import annotations

import pytest
import torch

from aios_amd import _lib
from aios_amd.layers import HipOps
from aios_amd.qwen3 import RotaryEmbedding
from tests.util import TorchOps

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _bf16(shape, seed, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(shape, generator=g, device=DEV) * scale).to(torch.bfloat16)


def _ulp_close(a, b, ulps=1):
    """bf16 results within `ulps` units in the last place (relative 2^-7 per ulp)."""
    a, b = a.float(), b.float()
    tol = ulps * 2.0 ** -7 * torch.maximum(a.abs(), b.abs()) + 1e-6
    assert bool(((a - b).abs() <= tol).all()), (a - b).abs().max().item()


@pytest.mark.parametrize("rows,hidden", [(1, 768), (8, 768), (37, 1024), (5, 2560), (3, 8192)])
def test_rmsnorm_and_fused_add(rows, hidden):
    x = _bf16((rows, hidden), rows, 2.0)
    r = _bf16((rows, hidden), rows + 1, 3.0)
    w = _bf16((hidden,), 7).abs() + 0.5
    ops, ref = HipOps(), TorchOps()
    _ulp_close(ops.rmsnorm(x, w, 1e-5), ref.rmsnorm(x, w, 1e-5))
    x1, r1 = x.clone(), r.clone()
    x2, r2 = x.clone(), r.clone()
    ops.fused_add_rmsnorm(x1, r1, w, 1e-6)
    ref.fused_add_rmsnorm(x2, r2, w, 1e-6)
    assert torch.equal(r1, r2)  # the residual sum is rounded once, as in the reference
    _ulp_close(x1, x2)


def test_rmsnorm_rejects_unsupported_width():
    with pytest.raises(ValueError, match="multiple of 8"):
        HipOps().rmsnorm(_bf16((2, 100), 1), _bf16((100,), 2), 1e-6)


@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 96), (12, 4, 64), (16, 8, 128), (32, 8, 128)])
def test_qk_norm_rope(hq, hkv, d):
    t = 19
    qkv = _bf16((t, (hq + 2 * hkv) * d), d + hq, 1.5)
    qw = _bf16((d,), 3).abs() + 0.5
    kw = _bf16((d,), 4).abs() + 0.5
    rot = RotaryEmbedding(d, 512, 1000000.0, DEV)
    pos = torch.tensor([0, 1, 2, 5, 31, 32, 100, 511] + list(range(200, 211)), dtype=torch.int32,
                       device=DEV)
    q1, k1 = HipOps().qk_norm_rope(qkv, qw, kw, rot.cos, rot.sin, pos, hq, hkv, d, 1e-6)
    q2, k2 = TorchOps().qk_norm_rope(qkv, qw, kw, rot.cos, rot.sin, pos, hq, hkv, d, 1e-6)
    # Same roundings as the torch ops; the norm's fp32 sum may differ in the
    # last bit, which can move an output by one bf16 step.
    _ulp_close(q1, q2, ulps=2)
    _ulp_close(k1, k2, ulps=2)
    # position 0 is the identity rotation: the output is the normalised head
    xn = TorchOps()._norm(qkv[:1, : hq * d].reshape(1, hq, d), qw, 1e-6)
    _ulp_close(q1[:1], xn)


@pytest.mark.parametrize("hq,hkv,d,t", [(8, 2, 96, 1), (12, 4, 64, 19), (16, 8, 128, 5),
                                        (8, 8, 64, 3), (32, 8, 128, 130),
                                        # two tokens a workgroup, then two head
                                        # groups a wavefront (one past the line, odd)
                                        (8, 2, 96, 513), (16, 8, 128, 513), (12, 4, 64, 821),
                                        (8, 2, 96, 1367)])
def test_qk_norm_rope_append_is_the_two_calls(hq, hkv, d, t):
    """The same bits as qk_norm_rope and store_cache, rows of other slots left
    alone, slots outside the pool skipped; qkv rows with a gap between them."""
    from aios_amd.kernel import store_cache

    qkv = _bf16((t, (hq + 2 * hkv) * d + 6), d + hq, 1.5)[:, : (hq + 2 * hkv) * d]
    qw, kw = _bf16((d,), 3).abs() + 0.5, _bf16((d,), 4).abs() + 0.5
    rot = RotaryEmbedding(d, 512, 1000000.0, DEV)
    pos = (torch.arange(t, device=DEV, dtype=torch.int32) * 37) % 600  # some past the table
    loc = torch.randperm(t + 9, generator=torch.Generator().manual_seed(t))[:t].to(torch.int32)
    if t > 2:
        loc[1], loc[2] = -1, t + 9
    loc = loc.to(DEV)
    kc, vc = _bf16((t + 9, hkv, d), 5), _bf16((t + 9, hkv, d), 6)
    k2, v2 = kc.clone(), vc.clone()
    q1, k1 = HipOps.qk_norm_rope(qkv, qw, kw, rot.cos, rot.sin, pos, hq, hkv, d, 1e-6)
    store_cache(kc, vc, loc, k1, qkv[:, (hq + hkv) * d:].view(t, hkv, d))
    q2 = HipOps.qk_norm_rope_append(qkv, qw, kw, rot.cos, rot.sin, pos, hq, 1e-6, k2, v2, loc)
    assert torch.equal(q1, q2) and torch.equal(kc, k2) and torch.equal(vc, v2)


@pytest.mark.parametrize("rows,inter", [(8, 2048), (32, 3072), (3, 9728)])
def test_silu_and_mul(rows, inter):
    x = _bf16((rows, 2 * inter), inter, 2.0)
    _ulp_close(HipOps().silu_and_mul(x), TorchOps().silu_and_mul(x))


@pytest.mark.parametrize("m,n,k", [(1, 1152, 768), (8, 1152, 768), (8, 768, 768), (8, 4096, 768),
                                   (8, 768, 2048), (8, 6400, 768), (24, 1024, 4096),
                                   (17, 2048, 1024), (64, 256, 9728), (33, 16, 128),
                                   # many column tiles: the streaming kernel (even and
                                   # uneven tiles per workgroup)
                                   (8, 16384, 768), (5, 20016, 768), (16, 32768, 1024),
                                   (8, 151936, 1024),
                                   # K 2048 plain (the down projection): 8-column tiles
                                   (1, 16, 2048), (16, 1024, 2048),
                                   # K 3072 plain (fixed step count)
                                   (8, 1024, 3072), (3, 2560, 3072)])
def test_linear_rows_matches_fp32_gemm(m, n, k):
    """Few-row GEMM kernel vs an fp32 matmul of the same bf16 operands: fp32
    accumulation, one bf16 rounding at the end."""
    x = _bf16((m, k), m + k, 1.0)
    w = _bf16((n, k), n, 0.05)
    y = HipOps().linear(x, w)
    ref = (x.float() @ w.float().T)
    err = (y.float() - ref).abs()
    assert bool((err <= 2.0 ** -8 * ref.abs() + 1e-3 * ref.abs().max()).all()), err.max().item()


def test_linear_rows_strided_input_and_fallback():
    x_big = _bf16((8, 2048), 5)
    x = x_big[:, :768]  # row stride 2048
    w = _bf16((1152, 768), 6, 0.05)
    torch.testing.assert_close(HipOps().linear(x, w).float(), (x.float() @ w.float().T),
                               atol=2e-2, rtol=1e-2)
    x65 = _bf16((65, 768), 7)  # more rows than the kernel takes: library GEMM
    torch.testing.assert_close(HipOps().linear(x65, w).float(), (x65.float() @ w.float().T),
                               atol=2e-2, rtol=1e-2)


@pytest.mark.parametrize("rows,k,n", [(1, 768, 1152), (8, 768, 1152), (8, 768, 6400),
                                      (24, 1024, 512), (40, 512, 256), (8, 2048, 768),
                                      (24, 768, 1152), (17, 768, 1152),
                                      # the streaming kernel (LM-head shapes)
                                      (8, 768, 16384), (1, 768, 20016), (8, 1024, 151936),
                                      (24, 1024, 151936)])
@pytest.mark.parametrize("with_residual", [True, False])
def test_add_rmsnorm_linear(rows, k, n, with_residual):
    """RMSNorm (with the residual add) folded into the projection: the same
    normalised operand as the separate kernels, the residual sum bit-exact;
    more rows or a longer K than that pays for (17, 24 at K 768 / 1024, 40 at
    K 512, K 2048) run as norm, then projection."""
    h = _bf16((rows, k), rows + k, 2.0)
    r = _bf16((rows, k), rows + k + 1, 3.0) if with_residual else None
    nw = _bf16((k,), 9).abs() + 0.5
    w = _bf16((n, k), n, 0.05)
    y, new_r = HipOps().add_rmsnorm_linear(h, r, nw, 1e-6, w)
    ref = TorchOps()
    if with_residual:
        x_ref, r_ref = ref.fused_add_rmsnorm(h.clone(), r.clone(), nw, 1e-6)
        assert torch.equal(new_r, r_ref)
    else:
        x_ref = ref.rmsnorm(h, nw, 1e-6)
        assert new_r is h
    y_ref = x_ref.float() @ w.float().T
    err = (y.float() - y_ref).abs()
    assert bool((err <= 2.0 ** -7 * y_ref.abs() + 2e-3 * y_ref.abs().max()).all()), err.max().item()


@pytest.mark.parametrize("rows,k,n", [(17, 128, 256), (32, 512, 1024), (32, 384, 48), (33, 256, 512),
                                      (48, 128, 16), (64, 256, 272), (64, 128, 8208)])
@pytest.mark.parametrize("silu", [False, True])
@pytest.mark.parametrize("with_residual", [True, False])
@pytest.mark.parametrize("folded", [True, False])
def test_norm_of_several_row_tiles(rows, k, n, silu, with_residual, folded):
    """The norm in front of two to four 16-row tiles, in the projection's launch
    (called directly: add_rmsnorm_linear takes it for some of these sizes) and
    as add_rmsnorm_linear runs it."""
    h = _bf16((rows, k), rows + k, 2.0)
    r = _bf16((rows, k), rows + k + 1, 3.0) if with_residual else None
    nw = _bf16((k,), 9).abs() + 0.5
    w = _bf16((2 * n if silu else n, k), n, 0.05)
    if folded:
        y, new_r = torch.empty(rows, n, dtype=h.dtype, device=DEV), torch.empty_like(h)
        _lib.check(_lib.lib().aios_linear_rows_ex(
            h.data_ptr(), k, w.data_ptr(), k, y.data_ptr(), n, rows, n, k,
            _lib.PROLOGUE_ADD_RMSNORM, r.data_ptr() if with_residual else None,
            k if with_residual else 0, nw.data_ptr(), 1e-6,
            new_r.data_ptr() if with_residual else None, k if with_residual else 0,
            _lib.EPILOGUE_SILU_MUL if silu else _lib.EPILOGUE_NONE, 0), "aios_linear_rows_ex")
        torch.cuda.synchronize()
    else:
        y, new_r = HipOps().add_rmsnorm_linear(h, r, nw, 1e-6, w, silu=silu)
    ref = TorchOps()
    x_ref = ref.rmsnorm(h, nw, 1e-6)
    if with_residual:
        x_ref, r_ref = ref.fused_add_rmsnorm(h.clone(), r.clone(), nw, 1e-6)
        assert torch.equal(new_r, r_ref)
    y_ref = x_ref.float() @ w.float().T
    if silu:
        y_ref = ref.silu_and_mul(y_ref.to(torch.bfloat16)).float()
    err = (y.float() - y_ref).abs()
    tol = 2.0 ** -6 if silu else 2.0 ** -7
    assert bool((err <= tol * y_ref.abs() + 4e-3 * y_ref.abs().max()).all()), err.max().item()


@pytest.mark.parametrize("rows,k,inter", [(8, 768, 2048), (3, 512, 256), (33, 256, 512),
                                          (1, 1024, 3072), (24, 768, 2048), (24, 1024, 3072)])
@pytest.mark.parametrize("with_residual", [True, False])
def test_add_rmsnorm_linear_silu_pair(rows, k, inter, with_residual):
    """Norm folded in front of the merged gate/up projection and SiLU-and-mul
    behind it: matches norm -> GEMM (bf16 store) -> silu_and_mul."""
    h = _bf16((rows, k), rows + k, 2.0)
    r = _bf16((rows, k), rows + k + 1, 3.0) if with_residual else None
    nw = _bf16((k,), 9).abs() + 0.5
    w = _bf16((2 * inter, k), inter, 0.05)
    y, _ = HipOps().add_rmsnorm_linear(h, r, nw, 1e-6, w, silu=True)
    ref = TorchOps()
    x_ref = (ref.fused_add_rmsnorm(h.clone(), r.clone(), nw, 1e-6)[0] if with_residual
             else ref.rmsnorm(h, nw, 1e-6))
    gu = (x_ref.float() @ w.float().T).to(torch.bfloat16)
    y_ref = ref.silu_and_mul(gu).float()
    err = (y.float() - y_ref).abs()
    assert bool((err <= 2.0 ** -6 * y_ref.abs() + 4e-3 * y_ref.abs().max()).all()), err.max().item()


@pytest.mark.parametrize("m,n,k", [(17, 16, 256), (24, 2560, 4096), (32, 48, 3072), (33, 2560, 9728),
                                   (48, 1024, 2560), (49, 272, 1280), (64, 20016, 2560),
                                   (64, 768, 2048), (1, 2560, 9728), (9, 6144, 2560),
                                   (16, 32, 4224), (24, 40000, 768)])
def test_streaming_rows_match_fp32_gemm(m, n, k):
    """The resident-row streaming GEMM: each count of 16-row tiles, one tile
    and many per workgroup, K split over workgroups (with a remainder of K
    steps), columns that do not divide over the workgroups.  fp32 sums, one
    bf16 rounding (2^-9 of the value) plus the sums' own error, bounded by
    k * 2^-24 of the magnitudes summed."""
    x = _bf16((m, k), m + k, 1.0)
    w = _bf16((n, k), n, 0.05)
    y = HipOps().linear(x, w).double()
    ref = x.double() @ w.double().T
    bound = 2.0 ** -8 * ref.abs() + k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert bool(((y - ref).abs() <= bound).all())


@pytest.mark.parametrize("m,n,k,silu", [
    (24, 2560, 4096, False), (24, 2560, 9728, False), (9, 2560, 9728, False), (17, 64, 1280, False),
    (64, 512, 2304, False), (40, 20016, 2304, False), (3, 48, 1280, False), (17, 64, 1280, True),
    (64, 512, 2304, True), (40, 10016, 2304, True), (3, 48, 1280, True)])
def test_infinite_weights_stay_infinite(m, n, k, silu):
    """Wavefronts and splits whose share of K is a step short of their registers
    add nothing for it: infinite weights at the end of every K step give the
    infinity of the plain product, not NaN."""
    x = _bf16((m, k), m + k, 1.0)
    x[:, 31::32] = x[:, 31::32].abs() + 0.5
    w = _bf16((2 * n if silu else n, k), n, 0.05)
    w[:5, 31::32] = float("inf")
    if silu:
        y = HipOps().add_rmsnorm_linear(x, None, torch.ones_like(x[0]), 1e-6, w, silu=True)[0]
        assert bool(y[:, :5].isinf().all()) and bool(y[:, 8:].isfinite().all())
    else:
        w[7, 31::32] = float("-inf")
        y = HipOps().linear(x, w)
        assert bool((y[:, :5] == float("inf")).all()) and bool((y[:, 7] == float("-inf")).all())
        assert bool(y[:, 8:].isfinite().all())


@pytest.mark.parametrize("rows,k,n", [(17, 768, 6144), (32, 2560, 512), (9, 2560, 4864),
                                      (24, 1280, 48), (24, 2304, 16), (40, 2560, 256),
                                      (64, 1024, 3072)])
@pytest.mark.parametrize("silu", [True, False])
@pytest.mark.parametrize("with_residual", [True, False])
def test_streaming_rows_norm_and_silu(rows, k, n, silu, with_residual):
    h = _bf16((rows, k), rows + k, 2.0)
    r = _bf16((rows, k), rows + k + 1, 3.0) if with_residual else None
    nw = _bf16((k,), 9).abs() + 0.5
    w = _bf16((2 * n if silu else n, k), n, 0.05)
    y, new_r = HipOps().add_rmsnorm_linear(h, r, nw, 1e-6, w, silu=silu)
    ref = TorchOps()
    if with_residual:
        x_ref, r_ref = ref.fused_add_rmsnorm(h.clone(), r.clone(), nw, 1e-6)
        assert torch.equal(new_r, r_ref)
    else:
        x_ref = ref.rmsnorm(h, nw, 1e-6)
        assert new_r is h
    y_ref = x_ref.float() @ w.float().T
    if silu:
        y_ref = ref.silu_and_mul(y_ref.to(torch.bfloat16)).float()
    err = (y.float() - y_ref).abs()
    tol = 2.0 ** -6 if silu else 2.0 ** -7
    assert bool((err <= tol * y_ref.abs() + 4e-3 * y_ref.abs().max()).all()), err.max().item()


def test_norm_takes_rows_it_cannot_read_in_place():
    """Wide rows with an odd offset, an odd stride or a column stride are copied
    for the separate norm, as before the norm read its inputs in place."""
    big = _bf16((8, 2 * 2560 + 24), 11, 1.0)
    r = _bf16((8, 2560), 12, 1.0)
    nw, w = _bf16((2560,), 13).abs() + 0.5, _bf16((64, 2560), 14, 0.05)
    for h in (big[:, 4:2564], big[:, ::2][:, :2560], big[:1, :2560].expand(8, 2560)):
        y, total = HipOps().add_rmsnorm_linear(h, r, nw, 1e-6, w)
        y_ref, t_ref = HipOps().add_rmsnorm_linear(h.contiguous(), r, nw, 1e-6, w)
        assert torch.equal(total, t_ref)
        torch.testing.assert_close(y.float(), y_ref.float(), atol=2e-2, rtol=2e-2)
