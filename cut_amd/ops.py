"""Host-side mirror (Python) of the reference's operator interface for the
quantized-matmul path, over torch device tensors.

Same names and argument meaning as ``Operations::dequantize(raw, fmt, rows,
cols)`` (runtime/Operations.cpp:1354-1361) and ``Operations::matmul(a, packedB,
scales)`` (runtime/Operations.cpp:226-231), with the weights kept as GGUF
blocks.  torch only supplies device memory and the current stream; every call
goes through the C ABI of libcut_hip.so.  Shape errors raise, as the
reference's constructors do (MatMulOp.cpp:288-329).
"""
from __future__ import annotations

import ctypes as C

import torch

from . import lib as _l

_native = None


def _host():
    """The native host side of the operators that are launched most (csrc/host_ops.cpp): checks, outputs and the C-ABI call.
    A decode step of the two-layer test model, 15 launches one by one: 107 us in Python and ctypes, 68 with it; seven
    matmuls on the separated layout 94 -> 86 (bound by the kernels then)."""
    global _native
    if _native is None:
        _l.load()   # says how to build what is missing
        try:
            from . import _host_ops
        except ImportError as e:
            raise _l.CutHipError(f"cut_amd/_host_ops.so is missing or does not load: build it with `make -C cut_amd/csrc` ({e})") from e
        _host_ops.setup(_l.CutHipError, _l.FORMATS, _l.UNARY, _l.BINARY, _l.NormCarry, _l.RopeAppend, C)
        _native = _host_ops
    return _native


def _stream_ptr() -> int:
    # the handle alone: a Stream object around it costs 2.8 us more, on every launch
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device())


def _fmt(fmt) -> int:
    if isinstance(fmt, str):
        if fmt not in _l.FORMATS:
            raise _l.CutHipError(f"unknown quantization format {fmt!r}")
        return _l.FORMATS[fmt]
    return int(fmt)


def n_bytes(fmt, rows: int, cols: int) -> int:
    f = _fmt(fmt)
    if cols % _l.BLOCK_ELEMS[f]:
        raise _l.CutHipError(f"cols ({cols}) must be a multiple of the block size {_l.BLOCK_ELEMS[f]}")
    return rows * (cols // _l.BLOCK_ELEMS[f]) * _l.BLOCK_BYTES[f]


def _holds(t: torch.Tensor, rows: int, width: int) -> bool:
    """Whether a launch that writes rows of `width` elements, stride(0) apart, stays inside the rows of t."""
    if t.dim() < 2:
        return t.dim() == 1 and rows <= 1 and t.shape[0] >= width and (t.shape[0] <= 1 or t.stride(0) == 1)
    return t.shape[0] >= rows and t.numel() >= t.shape[0] * width and (t.numel() == 0 or t[0].is_contiguous())


def dequantize(raw: torch.Tensor, fmt, rows: int, cols: int, dtype: torch.dtype = torch.float32,
               out: torch.Tensor | None = None) -> torch.Tensor:
    """raw: 1-D uint8/int8 device tensor of GGUF blocks -> [rows, cols]."""
    return _host().dequantize(raw, fmt, rows, cols, dtype, out)


_FMT_NAMES = {_l.Q8_0: "Q8_0", _l.Q4_0: "Q4_0", _l.Q4_K: "Q4_K", _l.Q6_K: "Q6_K"}
_tuning = None


def enable_tuning(path: str | None = None) -> bool:
    """Lets matmul_gguf consult shape rules (cut_amd/tuning_data.json by default, the "hip" backend section) when it
    is called with variant = -1, no epilogue and a workspace: the reference's VariantSelector mechanism
    (MatMulOp.cpp:242-246).  Returns False, and changes nothing, if the file cannot be loaded."""
    global _tuning
    from . import variant_selector as _vs
    sel = _vs.VariantSelector()
    if not sel.load(path or _vs.DEFAULT_PATH):
        return False
    _tuning = sel
    return True


def disable_tuning() -> None:
    global _tuning
    _tuning = None


def matmul_gguf(a: torch.Tensor, w_blocks: torch.Tensor, fmt, N: int, K: int, out_dtype: torch.dtype | None = None,
                out: torch.Tensor | None = None, unary: str | None = None, binary: str | None = None,
                d: torch.Tensor | None = None, variant: int = -1, workspace: torch.Tensor | None = None,
                swiglu_pairs: bool = False) -> torch.Tensor:
    """C = A . dequant(W)^T.  a: [M, K] or [K] (fp32 or fp16); w_blocks: N rows
    of K/blk GGUF blocks as a 1-byte device tensor.  With `workspace` (a device
    byte tensor from matmul_gguf_workspace) the call goes through
    cuthip_matmul_gguf_ws, which opens variant 4 (dequantize once, dense GEMM).
    swiglu_pairs: weight rows 2i / 2i+1 are gate_i / up_i and the result is [M, N/2] = silu(gate) * up (M <= 8)."""
    if _tuning is not None and variant == -1 and unary is None and binary is None and not swiglu_pairs and workspace is not None:
        variant = _tuning.select("MatMulGguf" + _FMT_NAMES[_fmt(fmt)], [a.shape[0] if a.dim() == 2 else 1, K, N], -1)
        # a rule may name a variant this process cannot run (the vendor-GEMM variant without its library): the
        # hand-written two-pass GEMM takes its place
        if variant >= 0 and _l.load().cuthip_variant_available(_l.OP_MATMUL_GGUF, variant) != 1:
            variant = 4 if variant == 5 else -1
    return _host().matmul_gguf(a, w_blocks, fmt, N, K, out_dtype, out, unary, binary, d, variant, workspace, swiglu_pairs)


def norm_carry(sumsq_parts: torch.Tensor | None = None, eps: float = 0.0, next_norm_weight: torch.Tensor | None = None,
               next_x16: torch.Tensor | None = None, next_sumsq_parts: torch.Tensor | None = None) -> "_l.NormCarry":
    """cuthip_norm_carry_t from device tensors (float32 [K/8] / [N] / [N/8], fp16 [N] output)."""
    return _host().norm_carry(_l.NormCarry, sumsq_parts, eps, next_norm_weight, next_x16, next_sumsq_parts)


def matmul_gguf_carry(a: torch.Tensor, w_blocks: torch.Tensor, fmt, N: int, K: int, out: torch.Tensor, carry, binary: str | None = None,
                      d: torch.Tensor | None = None, swiglu_pairs: bool = False) -> torch.Tensor:
    """Batch-1 matmul taking part in a carried RMSNorm (cuthip_matmul_gguf_carry); a [K], out [N] (or [N/2])."""
    return _host().matmul_gguf_carry(a, w_blocks, fmt, N, K, out, carry, binary, d, swiglu_pairs)


def rope_append(runtime_params: torch.Tensor, cos_t: torch.Tensor, sin_t: torch.Tensor, q_out: torch.Tensor, k_cache: torch.Tensor,
                v_cache: torch.Tensor, q_dim: int, head_dim: int) -> "_l.RopeAppend":
    """cuthip_rope_append_t for matmul_gguf_pair: rotated q to q_out, rotated k and v to the cache row of the position."""
    return _host().rope_append(_l.RopeAppend, runtime_params, cos_t, sin_t, q_out, k_cache, v_cache, q_dim, head_dim)


def interleave_rope_rows(w_blocks: torch.Tensor, n_rows: int, head_dim: int) -> torch.Tensor:
    """Rows of [heads * head_dim, K] GGUF blocks re-ordered inside every head to d = 0, half, 1, half + 1, ...: the
    layout the RoPE epilogue of matmul_gguf_pair reads (a permutation of whole block rows)."""
    rb = w_blocks.numel() // n_rows
    half = head_dim // 2
    w = w_blocks.view(n_rows // head_dim, 2, half, rb)
    return w.permute(0, 2, 1, 3).reshape(-1).contiguous()


def matmul_gguf_pair(a: torch.Tensor, wa: torch.Tensor, fmt_a, Na: int, out_a: torch.Tensor | None, wb: torch.Tensor, fmt_b,
                     Nb: int, out_b: torch.Tensor | None, K: int, carry=None, rope=None) -> None:
    """out_a = a . dequant(wa)^T and out_b = a . dequant(wb)^T for one activation vector a [K], in one launch where the
    formats allow it (cuthip_matmul_gguf_pair)."""
    _host().matmul_gguf_pair(a, wa, fmt_a, Na, out_a, wb, fmt_b, Nb, out_b, K, carry, rope)


def matmul_gguf_workspace(fmt, M: int, K: int, N: int, a_dtype: torch.dtype, device) -> torch.Tensor:
    """Scratch for the two-pass prefill matmul (variant 4): N*K fp16 (+ M*K fp16 for fp32 activations)."""
    n = _l.load().cuthip_matmul_gguf_workspace_bytes(_fmt(fmt), M, K, N, _l.F16 if a_dtype == torch.float16 else _l.F32)
    return torch.empty(max(int(n), 256), dtype=torch.uint8, device=device)


# ---- operators between the matmuls of a decode step ---------------------------------------------------
def _dt(t: torch.Tensor) -> int:
    if t.dtype == torch.float16:
        return _l.F16
    if t.dtype == torch.float32:
        return _l.F32
    raise _l.CutHipError(f"activations must be float16 or float32, got {t.dtype}")


def rmsnorm(x: torch.Tensor, weight: torch.Tensor, eps: float, out: torch.Tensor | None = None,
            out_dtype: torch.dtype | None = None) -> torch.Tensor:
    """x: [rows, dim] or [dim]; weight: fp32 [dim] (RMSNormOpNode of the reference)."""
    return _host().rmsnorm(x, weight, eps, out, out_dtype)


def rope_kv_write(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, runtime_params: torch.Tensor, cos_t: torch.Tensor,
                  sin_t: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, head_dim: int,
                  q_out: torch.Tensor) -> torch.Tensor:
    """q [q_dim], k, v [kv_dim] (same dtype); caches fp16 [max_ctx, aligned_kv_dim]; runtime_params int32/uint32[2] on device."""
    if k_cache.dtype != torch.float16 or v_cache.dtype != torch.float16 or k.dtype != q.dtype or v.dtype != q.dtype:
        raise _l.CutHipError("rope_kv_write: caches must be fp16 and q, k, v of one dtype")
    _l.check(_l.load().cuthip_rope_kv_write(q.data_ptr(), k.data_ptr(), v.data_ptr(), _dt(q), runtime_params.data_ptr(),
                                            cos_t.data_ptr(), sin_t.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(),
                                            q_out.data_ptr(), _dt(q_out), q.numel(), k.numel(), head_dim, k_cache.stride(0),
                                            min(k_cache.shape[0], cos_t.shape[0]), _stream_ptr()))
    return q_out


def attn_decode_workspace(n_heads: int, head_dim: int, max_seq_len: int, device) -> torch.Tensor:
    n = _l.load().cuthip_attn_decode_workspace_bytes(n_heads, head_dim, max_seq_len)
    return torch.empty(n, dtype=torch.uint8, device=device)


def attn_decode(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, runtime_params: torch.Tensor, n_heads: int,
                n_kv_heads: int, head_dim: int, scale: float, workspace: torch.Tensor, out: torch.Tensor,
                max_seq_len: int | None = None) -> torch.Tensor:
    return _host().attn_decode(q, k_cache, v_cache, runtime_params, n_heads, n_kv_heads, head_dim, scale, workspace, out, max_seq_len)


def attn_decode_static(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, runtime_params: torch.Tensor, n_heads: int,
                       n_kv_heads: int, head_dim: int, scale: float, out: torch.Tensor,
                       max_seq_len: int | None = None) -> torch.Tensor:
    """attn_decode on the library's built-in scratch (no workspace, no allocation; shapes up to 4 MiB of partials)."""
    _l.check(_l.load().cuthip_attn_decode_static(q.data_ptr(), _dt(q), k_cache.data_ptr(), v_cache.data_ptr(),
                                                 runtime_params.data_ptr(), out.data_ptr(), _dt(out), n_heads, n_kv_heads,
                                                 head_dim, k_cache.stride(0), scale, max_seq_len or k_cache.shape[0],
                                                 _stream_ptr()))
    return out


def attn_partial_records(n_heads: int, head_dim: int, max_seq_len: int, device) -> torch.Tensor:
    """Records of attn_decode_partial: [n_heads, splits, 2 + head_dim] fp32 (max, sum, un-normalised output)."""
    splits = _l.load().cuthip_attn_partial_splits(max_seq_len)
    return torch.empty((n_heads, splits, 2 + head_dim), dtype=torch.float32, device=device)


def attn_decode_partial(q: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, runtime_params: torch.Tensor, n_heads: int,
                        n_kv_heads: int, head_dim: int, scale: float, records: torch.Tensor,
                        max_seq_len: int | None = None) -> torch.Tensor:
    """The attention up to the per-split records (cuthip_attn_decode_partial); attn_merge or matmul_gguf_attn_merge
    folds them.  records: attn_partial_records() for the same max_seq_len."""
    _l.check(_l.load().cuthip_attn_decode_partial(q.data_ptr(), _dt(q), k_cache.data_ptr(), v_cache.data_ptr(),
                                                  runtime_params.data_ptr(), n_heads, n_kv_heads, head_dim, k_cache.stride(0),
                                                  scale, max_seq_len or k_cache.shape[0], records.data_ptr(),
                                                  records.numel() * records.element_size(), _stream_ptr()))
    return records


def attn_merge(records: torch.Tensor, out: torch.Tensor) -> torch.Tensor:
    """out[h, :] from records [n_heads, splits, 2 + head_dim] (cuthip_attn_merge)."""
    if records.dtype != torch.float32 or records.dim() != 3 or not records.is_contiguous() or not out.is_contiguous():
        raise _l.CutHipError("attn_merge: records must be a contiguous float32 [heads, splits, 2 + head_dim] tensor")
    n_heads, splits, rec = records.shape
    if out.numel() != n_heads * (rec - 2):
        raise _l.CutHipError("attn_merge: out must hold heads x head_dim elements")
    _l.check(_l.load().cuthip_attn_merge(records.data_ptr(), splits, n_heads, rec - 2, out.data_ptr(), _dt(out), _stream_ptr()))
    return out


def matmul_gguf_attn_merge(records: torch.Tensor, w_blocks: torch.Tensor, fmt, N: int, out: torch.Tensor, carry=None,
                           binary: str | None = None, d: torch.Tensor | None = None) -> torch.Tensor:
    """out [N] = merge(records) . dequant(W)^T with K = heads x head_dim (cuthip_matmul_gguf_attn_merge): the merge of the
    attention splits rides in the staging of the matmul's activations."""
    f = _fmt(fmt)
    if records.dtype != torch.float32 or records.dim() != 3 or not records.is_contiguous() or not out.is_contiguous():
        raise _l.CutHipError("matmul_gguf_attn_merge: records must be a contiguous float32 [heads, splits, 2 + head_dim] tensor")
    n_heads, splits, rec = records.shape
    K = n_heads * (rec - 2)
    if w_blocks.numel() < n_bytes(f, N, K) or out.numel() != N:
        raise _l.CutHipError("matmul_gguf_attn_merge: weight tensor too small or output of the wrong size")
    epi, op, dptr = _l.EPI_NONE, 0, None
    if binary is not None:
        if d is None or d.numel() != N or d.dtype != out.dtype:
            raise _l.CutHipError("matmul_gguf_attn_merge: binary epilogue needs D with the size and dtype of C")
        epi, op, dptr = _l.EPI_BINARY, _l.BINARY[binary], d.data_ptr()
    import ctypes
    _l.check(_l.load().cuthip_matmul_gguf_attn_merge(f, w_blocks.data_ptr(), records.data_ptr(), splits, n_heads, rec - 2,
                                                     out.data_ptr(), _dt(out), N, epi, op, dptr,
                                                     ctypes.byref(carry) if carry is not None else None, _stream_ptr()))
    return out


def silu_mul(gate_up: torch.Tensor, out: torch.Tensor) -> torch.Tensor:
    return _host().silu_mul(gate_up, out)


def argmax(x: torch.Tensor, out_index: torch.Tensor) -> torch.Tensor:
    _l.check(_l.load().cuthip_argmax(x.data_ptr(), _dt(x), x.numel(), out_index.data_ptr(), _stream_ptr()))
    return out_index


def repetition_penalty(logits: torch.Tensor, factors: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
    """RepetitionPenaltyOpNode on the dense fp32 factor vector (1 for tokens that are not penalised)."""
    if logits.dtype != torch.float32 or factors.dtype != torch.float32 or logits.numel() != factors.numel():
        raise _l.CutHipError("RepetitionPenalty: logits and penaltyFactors must be fp32 tensors of the same shape")
    if out is None:
        out = torch.empty_like(logits)
    elif out.dtype != torch.float32 or not out.is_contiguous() or out.numel() < logits.numel():
        raise _l.CutHipError(f"RepetitionPenalty: out must hold {logits.numel()} contiguous fp32 elements")
    _l.check(_l.load().cuthip_repetition_penalty(logits.data_ptr(), factors.data_ptr(), out.data_ptr(), logits.numel(), _stream_ptr()))
    return out


def _pen_args(pen_tokens, pen_factors):
    if pen_tokens is None:
        return None, None, 0
    if pen_tokens.dtype != torch.int32 or pen_factors.dtype != torch.float32 or pen_tokens.numel() != pen_factors.numel():
        raise _l.CutHipError("penalised tokens are int32 ids with one fp32 factor each")
    return pen_tokens.data_ptr(), pen_factors.data_ptr(), pen_tokens.numel()


def argmax_penalized(logits: torch.Tensor, out_index: torch.Tensor, pen_tokens: torch.Tensor | None = None,
                     pen_factors: torch.Tensor | None = None) -> torch.Tensor:
    """Repetition penalty on the listed tokens (in place), then the arg-max (cuthip_argmax_penalized)."""
    pt, pf, n = _pen_args(pen_tokens, pen_factors)
    _l.check(_l.load().cuthip_argmax_penalized(logits.data_ptr(), _dt(logits), logits.numel(), pt, pf, n, out_index.data_ptr(),
                                               _stream_ptr()))
    return out_index


def lm_head_workspace(N: int, device) -> torch.Tensor:
    return torch.empty(max(int(_l.load().cuthip_matmul_gguf_argmax_workspace_bytes(N)), 8), dtype=torch.uint8, device=device)


def matmul_gguf_argmax(a: torch.Tensor, w_blocks: torch.Tensor, fmt, N: int, K: int, logits: torch.Tensor, out_index: torch.Tensor,
                       carry=None, pen_tokens: torch.Tensor | None = None, pen_factors: torch.Tensor | None = None,
                       workspace: torch.Tensor | None = None) -> torch.Tensor:
    """The output head with the sampling folded in: logits = a . dequant(W)^T, penalty on the listed tokens, arg-max."""
    return _host().matmul_gguf_argmax(a, w_blocks, fmt, N, K, logits, out_index, carry, pen_tokens, pen_factors, workspace)


def embedding_rows(w_blocks: torch.Tensor, fmt, token_ids: torch.Tensor, n_rows: int, dim: int, out: torch.Tensor) -> torch.Tensor:
    """out[i] = dequant(row token_ids[i]) of a GGUF table [n_rows, dim]; token_ids int32/uint32 on the device."""
    return _host().embedding_rows(w_blocks, fmt, token_ids, n_rows, dim, out)


def embedding_col(indices: torch.Tensor, matrix: torch.Tensor, scales: torch.Tensor | None, emb_dim: int, vocab: int,
                  out: torch.Tensor | None = None) -> torch.Tensor:
    """EmbeddingColOpNode: matrix [emb_dim, vocab_stride] column-wise, fp16 (scales None) or int8 with fp16 scales
    [emb_dim / 32, scale_stride]; returns fp32 [len(indices), emb_dim]."""
    fmt = 0 if scales is None else 1
    if matrix.dim() != 2 or matrix.dtype != (torch.float16 if fmt == 0 else torch.int8) or indices.dtype not in (torch.int32, torch.uint32):
        raise _l.CutHipError("embedding_col: matrix is 2-D fp16 (no scales) or int8 (fp16 scales), indices 32-bit integers")
    if out is None:
        out = torch.empty((indices.numel(), emb_dim), dtype=torch.float32, device=matrix.device)
    elif out.dtype != torch.float32 or not _holds(out, indices.numel(), emb_dim):
        raise _l.CutHipError(f"embedding_col: out must be fp32 and have contiguous room for {indices.numel()} rows of {emb_dim}")
    _l.check(_l.load().cuthip_embedding_col(indices.data_ptr(), matrix.data_ptr(), scales.data_ptr() if fmt else None, out.data_ptr(),
                                            indices.numel(), emb_dim, matrix.stride(0), scales.stride(0) if fmt else 0, out.stride(0),
                                            vocab, fmt, _stream_ptr()))
    return out


# ---- the reference's separated weight layout ----------------------------------------------------------
def matmul_sep(a: torch.Tensor, b: torch.Tensor, scales: torch.Tensor, N: int, q4: bool = False, affine: bool = False,
               out: torch.Tensor | None = None, unary: str | None = None, binary: str | None = None,
               d: torch.Tensor | None = None, variant: int = -1) -> torch.Tensor:
    """Operations::matmul(a, packedB, scalesB) of the reference on its own layout: a fp32 [M, K]; b int8 [K, N]
    (q4: uint8 [K, N/2], even column in the low nibble); scales fp16 [K/32, N] ([2K/32, N] when affine).
    variant: the reference's `spec` (an index of its MatMulQ8 / MatMulQ4 variant tables), -1 = by shape."""
    return _host().matmul_sep(a, b, scales, N, q4, affine, out, unary, binary, d, variant)


def matmul_dense_f16(a: torch.Tensor, w16: torch.Tensor, out_dtype: torch.dtype | None = None, out: torch.Tensor | None = None,
                     unary: str | None = None, binary: str | None = None, d: torch.Tensor | None = None,
                     workspace: torch.Tensor | None = None) -> torch.Tensor:
    """Prefill matmul on resident dequantized weights: w16 fp16 [N, K] (from dequantize(..., torch.float16)), a [M, K]
    fp16 or fp32; C = a . w16^T.  The quantized blocks stay the operand of the decode GEMV; this copy serves prefill."""
    a2 = a if a.dim() == 2 else a.reshape(1, -1)
    M, K = a2.shape
    if w16.dtype != torch.float16 or w16.dim() != 2 or w16.shape[1] != K or not w16.is_contiguous():
        raise _l.CutHipError(f"matmul_dense_f16: w16 must be a contiguous fp16 [N, {K}] tensor")
    N = w16.shape[0]
    if a2.dtype not in (torch.float32, torch.float16) or a2.stride(1) != 1:
        raise _l.CutHipError("matmul_dense_f16: a must be fp32 / fp16 with contiguous rows")
    if out is None:
        out = torch.empty((M, N), dtype=out_dtype or a2.dtype, device=a.device)
    elif not _holds(out, M, N):
        raise _l.CutHipError(f"matmul_dense_f16: out must have contiguous room for {M} rows of {N}")
    epi, op, dptr = _l.EPI_NONE, 0, None
    if unary is not None:
        epi, op = _l.EPI_UNARY, _l.UNARY[unary]
    elif binary is not None:
        if d is None or d.shape != out.shape or d.dtype != out.dtype or d.stride(0) != out.stride(0):
            raise _l.CutHipError("matmul_dense_f16: binary epilogue needs a D with the dtype, shape and stride of C")
        epi, op, dptr = _l.EPI_BINARY, _l.BINARY[binary], d.data_ptr()
    lib = _l.load()
    if workspace is None:
        workspace = torch.empty(max(lib.cuthip_matmul_dense_f16_workspace_bytes(M, K, N, _dt(a2)), 256), dtype=torch.uint8,
                                device=a.device)
    _l.check(lib.cuthip_matmul_dense_f16(w16.data_ptr(), a2.data_ptr(), _dt(a2), out.data_ptr(), _dt(out), M, K, N,
                                         a2.stride(0), out.stride(0), epi, op, dptr, workspace.data_ptr(), workspace.numel(),
                                         _stream_ptr()))
    return out


def matmul_q8_i8(a: torch.Tensor, w_blocks: torch.Tensor, N: int, K: int, out_dtype: torch.dtype | None = None,
                 out: torch.Tensor | None = None, unary: str | None = None, binary: str | None = None,
                 d: torch.Tensor | None = None, workspace: torch.Tensor | None = None) -> torch.Tensor:
    """Q8_0 weights (GGUF blocks [N][K/32]) x activations quantized to int8 per 32 elements, on the int8 matrix
    core: the arithmetic of the reference's MatMulQ8GemvDot for any M.  Opt-in: about 5e-3 from the fp32 path."""
    a2 = a if a.dim() == 2 else a.reshape(1, -1)
    M = a2.shape[0]
    if a2.shape[1] != K or a2.dtype not in (torch.float32, torch.float16) or a2.stride(1) != 1:
        raise _l.CutHipError(f"matmul_q8_i8: a must be fp32 / fp16 [M, {K}] with contiguous rows")
    if out is None:
        out = torch.empty((M, N), dtype=out_dtype or a2.dtype, device=a.device)
    elif not _holds(out, M, N):
        raise _l.CutHipError(f"matmul_q8_i8: out must have contiguous room for {M} rows of {N}")
    epi, op, dptr = _l.EPI_NONE, 0, None
    if unary is not None:
        epi, op = _l.EPI_UNARY, _l.UNARY[unary]
    elif binary is not None:
        if d is None or d.shape != out.shape or d.dtype != out.dtype or d.stride(0) != out.stride(0):
            raise _l.CutHipError("matmul_q8_i8: binary epilogue needs a D with the dtype, shape and stride of C")
        epi, op, dptr = _l.EPI_BINARY, _l.BINARY[binary], d.data_ptr()
    lib = _l.load()
    need = lib.cuthip_matmul_q8_i8_workspace_bytes(M, K)
    if workspace is None:
        workspace = torch.empty(max(need, 16), dtype=torch.uint8, device=a.device)
    _l.check(lib.cuthip_matmul_q8_i8(w_blocks.data_ptr(), a2.data_ptr(), _dt(a2), out.data_ptr(), _dt(out), M, K, N,
                                     a2.stride(0), out.stride(0), epi, op, dptr, workspace.data_ptr(), workspace.numel(),
                                     _stream_ptr()))
    return out


def prepare_sep(w_blocks: torch.Tensor, fmt, N: int, K: int, stride_b: int | None = None, scale_stride: int | None = None):
    """GGUF blocks [N rows of K/blk blocks] on the device -> (B, scales) in the reference's separated [K, N] layout:
    Q8_0 -> int8 [K, N] + fp16 [K/32, N]; Q4_0 -> nibbles uint8 [K, N/2] + fp16 [K/32, N]; Q4_K -> affine Q4, nibbles
    + fp16 [2K/32, N] (scales then minima: requantizeQ4KToAffine).  Row strides default to the reference's padding
    to multiples of 4 elements (MatMulOp.cpp:514-541)."""
    return _host().prepare_sep(w_blocks, fmt, N, K, stride_b, scale_stride)


def transpose_q4_nibble(packed: torch.Tensor, N: int, K: int) -> torch.Tensor:
    """Operations::transposeQ4(packed, N, K) of the reference: GGML-order nibbles [N, K/2] -> [K, N/2]."""
    if packed.dim() != 2 or packed.element_size() != 1 or packed.stride(1) != 1:
        raise _l.CutHipError("transpose_q4_nibble: packed must be a 2-D 1-byte tensor with contiguous rows")
    so = (N // 2 + 3) & ~3
    out = torch.zeros((K, so), dtype=torch.uint8, device=packed.device)
    _l.check(_l.load().cuthip_transpose_q4_nibble(packed.data_ptr(), out.data_ptr(), N, K, packed.stride(0), so, _stream_ptr()))
    return out


def quantize_rows_q8_0(x: torch.Tensor) -> torch.Tensor:
    """quantizeRowsQ8_0 of the reference's runner on the device: fp32 [n] -> Q8_0 blocks (uint8 [n/32 * 34])."""
    if x.dtype != torch.float32 or not x.is_contiguous():
        raise _l.CutHipError("quantize_rows_q8_0: x must be a contiguous fp32 tensor")
    n = x.numel()
    out = torch.empty(max(n // 32, 1) * 34, dtype=torch.uint8, device=x.device)
    _l.check(_l.load().cuthip_quantize_rows_q8_0(x.data_ptr(), n, out.data_ptr(), _stream_ptr()))
    return out


def matmul_gguf_pro(a: torch.Tensor, w_blocks: torch.Tensor, fmt, N: int, K: int, out: torch.Tensor, prologue: str,
                    norm_weight: torch.Tensor | None = None, eps: float = 0.0, unary: str | None = None,
                    binary: str | None = None, d: torch.Tensor | None = None) -> torch.Tensor:
    """Batch-1 matmul with the preceding operator fused into the activation staging:
    prologue "rmsnorm": a = x [K] (fp32 or fp16), norm_weight fp32 [K];  "swiglu": a = [gate | up] fp16 [2K]."""
    pro = {"rmsnorm": 1, "swiglu": 2}[prologue]
    need = K if pro == 1 else 2 * K
    if a.numel() != need or not a.is_contiguous() or out.numel() != N:
        raise _l.CutHipError(f"matmul_gguf_pro: a must hold {need} contiguous elements and out {N}")
    epi, op, dptr = _l.EPI_NONE, 0, None
    if unary is not None:
        epi, op = _l.EPI_UNARY, _l.UNARY[unary]
    elif binary is not None:
        if d is None or d.numel() != N or d.dtype != out.dtype:
            raise _l.CutHipError("matmul_gguf_pro: binary epilogue needs D like C")
        epi, op, dptr = _l.EPI_BINARY, _l.BINARY[binary], d.data_ptr()
    _l.check(_l.load().cuthip_matmul_gguf_pro(_fmt(fmt), w_blocks.data_ptr(), a.data_ptr(), _dt(a), out.data_ptr(), _dt(out), K, N,
                                              epi, op, dptr, pro, norm_weight.data_ptr() if norm_weight is not None else None,
                                              eps, _stream_ptr()))
    return out
