"""Decoder-layer ops on the gfx950 kernels (the layers the reference takes
from FlashInfer, Triton and torch: python/aios/layers/norm.py:10-40,
layers/activation.py:9-12, layers/attention.py:11-16, the q/k norm of
models/qwen3.py:65-66 and the Block-AttnRes depth mixer,
kernel/attnres.py:130-223).

``HipOps`` is the op set the decoder uses on the GPU; every call goes
through the C ABI of libaios_attn.so and fails loudly without it.
"""
from __future__ import annotations

import torch

from aios_amd import _lib
from aios_amd.core import runs_as_built


def _stream(t: torch.Tensor) -> int:
    return _lib.raw_stream(t)


def _check_gpu(*tensors: torch.Tensor) -> None:
    for t in tensors:
        if not t.is_cuda:
            raise ValueError("the kernels take GPU tensors")


def _check_rows(t: torch.Tensor, name: str) -> None:
    if t.dtype != torch.bfloat16 or not t.is_cuda or t.ndim != 2 or t.stride(1) != 1:
        raise ValueError(f"{name} must be a 2-D bfloat16 GPU tensor with contiguous rows")


def _plain_rows(t: torch.Tensor) -> bool:
    """16-byte aligned, contiguous, non-overlapping rows."""
    return (t.stride(1) == 1 and t.stride(0) >= t.shape[1] and t.stride(0) % 8 == 0
            and t.data_ptr() % 16 == 0)


def _plain_copy(t: torch.Tensor, name: str) -> torch.Tensor:
    """t, or a copy where its rows cannot be read in place."""
    if _plain_rows(t):
        if t.dtype == torch.bfloat16 and t.is_cuda:
            return t
    else:
        t = t.clone()
    _check_rows(t, name)
    return t


def _add_rmsnorm(h: torch.Tensor, residual: torch.Tensor, weight: torch.Tensor,
                 eps: float) -> tuple[torch.Tensor, torch.Tensor]:
    """(RMSNorm(h + residual) * weight, h + residual), the inputs left unchanged."""
    h, residual = _plain_copy(h, "x"), _plain_copy(residual, "residual")
    if h.shape != residual.shape:
        raise ValueError("x and residual must have the same shape")
    out, total = torch.empty_like(h), torch.empty_like(residual)
    _lib.check(_lib.lib().aios_add_rmsnorm(
        h.data_ptr(), h.stride(0), residual.data_ptr(), residual.stride(0), weight.data_ptr(),
        total.data_ptr(), total.stride(0), out.data_ptr(), out.stride(0), h.shape[0], h.shape[1],
        eps, _stream(h)), "aios_add_rmsnorm")
    return out, total


def _linear_rows(x: torch.Tensor, weight: torch.Tensor, n: int, silu: bool = False) -> torch.Tensor:
    """The few-row projection (aios_linear_rows_ws) to n columns."""
    _check_gpu(x, weight)
    rows, k = x.shape
    lib = _lib.lib()
    y = torch.empty(rows, n, dtype=x.dtype, device=x.device)
    # (a buffer of this call alone: calls may overlap on several streams)
    ws_bytes = 0 if silu else lib.aios_linear_rows_workspace(rows, n, k)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=x.device) if ws_bytes else None
    _lib.check(lib.aios_linear_rows_ws(
        x.data_ptr(), x.stride(0), weight.data_ptr(), weight.stride(0), y.data_ptr(), y.stride(0),
        rows, n, k, _lib.EPILOGUE_SILU_MUL if silu else _lib.EPILOGUE_NONE,
        ws.data_ptr() if ws is not None else None, ws_bytes, _stream(x)), "aios_linear_rows_ws")
    return y


class HipOps:
    """RMSNorm, residual-add RMSNorm, q/k RMSNorm + RoPE, SiLU-and-mul, and
    the projections (few-row GEMM kernel for decode-sized inputs, the
    library GEMM for larger ones)."""

    # The decoder may hand an appending decode batch's raw q/k projections to
    # the attention backend, which applies the q/k RMSNorm + RoPE of
    # qk_norm_rope inside the decode launch.
    rope_in_decode = True
    # ... and a prefill's K/V rows may be written to their pages by the launch
    # that normalises and rotates them (qk_norm_rope_append).
    rope_in_append = True

    @staticmethod
    def linear(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
        rows, k = x.shape
        n = weight.shape[0]
        if (rows > 64 or n % 16 or k % 128 or x.dtype != torch.bfloat16
                or weight.dtype != torch.bfloat16 or x.stride(1) != 1 or weight.stride(1) != 1
                or x.stride(0) % 8 or weight.stride(0) % 8):
            return torch.nn.functional.linear(x, weight)
        if rows == 0:
            return x.new_empty(0, n)
        return _linear_rows(x, weight, n)

    @staticmethod
    def _rows_ok(x: torch.Tensor, weight: torch.Tensor, k: int) -> bool:
        return (x.shape[0] <= 64 and weight.shape[0] % 16 == 0 and k % 128 == 0
                and x.dtype == torch.bfloat16 and weight.dtype == torch.bfloat16
                and x.stride(1) == 1 and weight.stride(1) == 1 and x.stride(0) % 8 == 0
                and weight.stride(0) % 8 == 0 and x.shape[0] > 0)

    def add_rmsnorm_linear(self, h: torch.Tensor, residual: torch.Tensor | None,
                           norm_weight: torch.Tensor, eps: float, weight: torch.Tensor,
                           silu: bool = False) -> tuple[torch.Tensor, torch.Tensor]:
        """RMSNormFused then a projection (norm.py:24-40): returns
        (linear(RMSNorm(h + residual) * w), h + residual); with no residual the
        new residual is h itself.  silu=True: weight is the merged gate/up
        matrix and the projection is followed by silu_and_mul
        (activation.py:9-12)."""
        rows, k = h.shape
        n = weight.shape[0] // 2 if silu else weight.shape[0]
        rows_ok = self._rows_ok(h, weight, k) and n % 16 == 0
        # One 16-row tile whose normalised fragments fit the registers (K / 128
        # of them, at most 8) takes the norm in the projection's launch.  More
        # tiles do while forming it in every workgroup costs less than a launch
        # (24 x 128 x 256 3.1 us against 4.8, 32 x 512 x 1024 5.0 against 5.7
        # without a residual, 5.8 against 5.3 with one; 24 x 768 x 1280, in two
        # launches, 9 against 6.7).
        frags = k // 128 * -(-rows // 16) if rows_ok else 9
        if (frags <= 8
                and (rows <= 16 or (frags + 2 * (residual is not None) + 2 * silu <= 8
                                    and frags * n <= 32768))
                and (residual is None
                     or (residual.stride(1) == 1 and residual.stride(0) % 8 == 0))):
            _check_gpu(h, weight, norm_weight, *(() if residual is None else (residual,)))
            y = torch.empty(rows, n, dtype=h.dtype, device=h.device)
            total = torch.empty_like(h) if residual is not None else h
            _lib.check(_lib.lib().aios_linear_rows_ex(
                h.data_ptr(), h.stride(0), weight.data_ptr(), weight.stride(0), y.data_ptr(),
                y.stride(0), rows, n, k, _lib.PROLOGUE_ADD_RMSNORM,
                residual.data_ptr() if residual is not None else None,
                residual.stride(0) if residual is not None else 0, norm_weight.data_ptr(), eps,
                total.data_ptr() if residual is not None else None,
                total.stride(0) if residual is not None else 0,
                _lib.EPILOGUE_SILU_MUL if silu else _lib.EPILOGUE_NONE, _stream(h)),
                "aios_linear_rows_ex")
            return y, total
        if residual is None:
            x, residual = self.rmsnorm(h, norm_weight, eps), h
        elif runs_as_built(self, _FUSED_NORM):
            x, residual = _add_rmsnorm(h, residual, norm_weight, eps)
        else:  # (a caller's own in-place norm, the inputs left unchanged)
            x, residual = self.fused_add_rmsnorm(h.clone(), residual.clone(), norm_weight, eps)
        if silu and rows_ok and k <= 2560 and runs_as_built(self, _LINEAR_SILU):
            return _linear_rows(x, weight, n, silu=True), residual
        y = self.linear(x, weight)
        return (self.silu_and_mul(y) if silu else y), residual

    @staticmethod
    def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
        _check_rows(x, "x")
        out = torch.empty_like(x)
        _lib.check(_lib.lib().aios_rmsnorm(x.data_ptr(), x.stride(0), None, 0, weight.data_ptr(),
                                           out.data_ptr(), out.stride(0), x.shape[0], x.shape[1],
                                           eps, _stream(x)), "aios_rmsnorm")
        return out

    @staticmethod
    def fused_add_rmsnorm(x: torch.Tensor, residual: torch.Tensor, weight: torch.Tensor,
                          eps: float) -> tuple[torch.Tensor, torch.Tensor]:
        """residual <- x + residual; x <- RMSNorm(residual) * weight (both in place)."""
        _check_rows(x, "x")
        _check_rows(residual, "residual")
        if x.shape != residual.shape:
            raise ValueError("x and residual must have the same shape")
        _lib.check(_lib.lib().aios_rmsnorm(x.data_ptr(), x.stride(0), residual.data_ptr(),
                                           residual.stride(0), weight.data_ptr(), x.data_ptr(),
                                           x.stride(0), x.shape[0], x.shape[1], eps, _stream(x)),
                   "aios_rmsnorm")
        return x, residual

    @staticmethod
    def qk_norm_rope(qkv: torch.Tensor, q_weight: torch.Tensor, k_weight: torch.Tensor,
                     cos: torch.Tensor, sin: torch.Tensor, positions: torch.Tensor,
                     num_qo_heads: int, num_kv_heads: int, head_dim: int,
                     eps: float) -> tuple[torch.Tensor, torch.Tensor]:
        """q, k = RoPE(RMSNorm_head(q)), RoPE(RMSNorm_head(k)) from qkv rows."""
        HipOps._check_rope(qkv, cos, sin, positions, head_dim)
        t = qkv.shape[0]
        q = torch.empty(t, num_qo_heads, head_dim, dtype=qkv.dtype, device=qkv.device)
        k = torch.empty(t, num_kv_heads, head_dim, dtype=qkv.dtype, device=qkv.device)
        _lib.check(_lib.lib().aios_qk_norm_rope(
            qkv.data_ptr(), qkv.stride(0), t, num_qo_heads, num_kv_heads, head_dim,
            q_weight.data_ptr(), k_weight.data_ptr(), cos.data_ptr(), sin.data_ptr(), cos.shape[0],
            positions.contiguous().data_ptr(), q.data_ptr(), k.data_ptr(), eps, _stream(qkv)),
            "aios_qk_norm_rope")
        return q, k

    @staticmethod
    def _check_rope(qkv: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor,
                    positions: torch.Tensor, head_dim: int) -> None:
        _check_rows(qkv, "qkv")
        if positions.dtype != torch.int32 or positions.numel() != qkv.shape[0]:
            raise ValueError("positions must be int32 with one entry per token")
        if cos.dtype != torch.float32 or cos.shape != sin.shape or cos.shape[1] != head_dim:
            raise ValueError("cos/sin tables must be float32 [positions, head_dim]")

    @staticmethod
    def qk_norm_rope_append(qkv: torch.Tensor, q_weight: torch.Tensor, k_weight: torch.Tensor,
                            cos: torch.Tensor, sin: torch.Tensor, positions: torch.Tensor,
                            num_qo_heads: int, eps: float, k_cache: torch.Tensor,
                            v_cache: torch.Tensor, out_loc: torch.Tensor) -> torch.Tensor:
        """qk_norm_rope with the rotated K rows and qkv's V rows written to
        rows out_loc of the contiguous bfloat16 [slots, Hkv, D] caches instead
        of returned (store_kv in the same launch); returns q."""
        _, num_kv_heads, head_dim = k_cache.shape
        HipOps._check_rope(qkv, cos, sin, positions, head_dim)
        t = qkv.shape[0]
        if qkv.shape[1] != (num_qo_heads + 2 * num_kv_heads) * head_dim:
            raise ValueError("qkv rows must hold the q, k and v heads")
        for c in (k_cache, v_cache):
            if c.dtype != torch.bfloat16 or c.shape != k_cache.shape or not c.is_contiguous():
                raise ValueError("KV caches must be contiguous bfloat16 tensors of one shape")
        _check_gpu(k_cache, v_cache, out_loc)
        if out_loc.dtype != torch.int32 or out_loc.numel() != t or not out_loc.is_contiguous():
            raise ValueError("out_loc must be contiguous int32 with one entry per token")
        q = torch.empty(t, num_qo_heads, head_dim, dtype=qkv.dtype, device=qkv.device)
        _lib.check(_lib.lib().aios_qk_norm_rope_append(
            qkv.data_ptr(), qkv.stride(0), t, num_qo_heads, num_kv_heads, head_dim,
            q_weight.data_ptr(), k_weight.data_ptr(), cos.data_ptr(), sin.data_ptr(), cos.shape[0],
            positions.contiguous().data_ptr(), q.data_ptr(), k_cache.data_ptr(),
            v_cache.data_ptr(), k_cache.shape[0], out_loc.data_ptr(), eps, _stream(qkv)),
            "aios_qk_norm_rope_append")
        return q

    @staticmethod
    def attnres_mix(bank: torch.Tensor, partial: torch.Tensor | None,
                    weighted_query: torch.Tensor, eps: float) -> torch.Tensor:
        """Depth mix of bank [S, N, D] (+ partial as the last source)."""
        from aios_amd.kernel import attnres_mix

        return attnres_mix(bank, partial, weighted_query, eps)

    @staticmethod
    def attnres_mix_step(bank: torch.Tensor, partial: torch.Tensor | None, delta: torch.Tensor,
                         weighted_query: torch.Tensor, eps: float,
                         partial_out: torch.Tensor) -> torch.Tensor:
        """partial_out <- partial + delta, then the mix with it as the last source."""
        from aios_amd.kernel import attnres_mix_step

        return attnres_mix_step(bank, partial, delta, weighted_query, eps, partial_out)

    @staticmethod
    def silu_and_mul(x: torch.Tensor) -> torch.Tensor:
        _check_rows(x, "x")
        inter = x.shape[1] // 2
        out = torch.empty(x.shape[0], inter, dtype=x.dtype, device=x.device)
        _lib.check(_lib.lib().aios_silu_mul(x.data_ptr(), x.stride(0), x.shape[0], inter,
                                            out.data_ptr(), out.stride(0), _stream(x)),
                   "aios_silu_mul")
        return out


# The ops that add_rmsnorm_linear's separate launches stand for, as built here.
_FUSED_NORM = (("fused_add_rmsnorm", HipOps.fused_add_rmsnorm),)
_LINEAR_SILU = (("linear", HipOps.linear), ("silu_and_mul", HipOps.silu_and_mul))
