"""The reference's quantized sparse-transformer ops with their signatures.

Drop-in mirrors of the ``sptrans`` PyTorch extension the reference's layer
imports (end2end_eval/sparse_transformer_magicube/src/cuda/*.cpp): same
names, same positional arguments, same output dtypes and shapes, device
tensors in and out, every op running on the current stream (or ``stream``).

* ``quantization(x, bits, scale)`` / ``bquantization`` (quantization.cpp:3-20,
  quantization_kernel.cu:13-74,173-213): fp16 ``[..., L, D]`` -> int32
  ``[..., L, D * bits / 32]``, ``trunc(clamp(x * scale))``, lanes packed
  low first.
* ``sddmm_8b`` / ``sddmm_4b`` / ``bsddmm_8b`` / ``bsddmm_4b``
  (deq_sddmm.cpp:3-99, deq_sddmm_kernel.cu:447-466,565-636): packed Q
  ``[batch, m, k / (32 / bits)]`` and K ``[batch, n, ...]`` sampled at the
  shared mask -> fp16 ``[batch, nnz * V]`` (vector-major ``[slot][v]``),
  ``half(float(int32 S) / scale)``; padding slots hold 0.
* ``q_csr_softmax`` / ``q_bcsr_softmax`` (q_softmax.cpp:3-52,
  q_softmax_kernel.cu:180-271,394-479): fp16 logits -> int32 packed P of
  ``bits`` in the reference's SpMM A layouts (``mc_attn_softmax_f16``).
* ``bspmm_8b`` / ``bspmm_16b8b`` / ``bspmm_8b4b`` / ``bspmm_4b``
  (deq_spmm.cpp:5-141, deq_spmm_kernel.cu:593-876,1136-1361): packed P
  times packed V ``[batch, L, 64 * bits_rhs / 32]`` -> fp16
  ``[batch, m_vec * V, 64]``, ``half(float(int32 P V) / scale)``.

Masks are the reference's aligned vector-CSR: ``row_offsets`` 2 * m_vec
(start, end) pairs with starts on 16 slots (8-bit V) or 32 slots (4-bit V),
``column_indices`` -1 padded and not shuffled, ``row_indices`` the row order
(any permutation).  The products are exact two's-complement integers: the
reference feeds its signed quantized Q/K/V to unsigned tensor-core MMAs
(quantization_kernel.cu:65-69 against sddmm_utils/compute_utils.h:102),
which changes its results wherever a lane is negative; these ops compute the
signed products the layer means.

``row_indices`` is a permutation of the mask's vector rows: every row is written
once, and only the slots between rows are zeroed beside them.

Each product is one launch (``mc_spmm_batched_f16``): the kernel reads P as
the softmax op writes it and the mask's indices in their natural order, and
divides and rounds to fp16 as it stores.
"""
from __future__ import annotations

import contextlib

import torch

from . import _lib
from .attention import bquantization as _bquantization
from .spmm import current_stream_handle


def _ptr(t):
    return t.data_ptr() if t is not None else None


def _stream_handle(stream):
    return stream.cuda_stream if stream is not None else current_stream_handle()


def _on(stream):
    return torch.cuda.stream(stream) if stream is not None else contextlib.nullcontext()


def _i32(t, what):
    if not isinstance(t, torch.Tensor) or not t.is_cuda:
        raise ValueError(f"{what} must be a device tensor")
    if t.dtype != torch.int32:
        raise ValueError(f"{what} must be int32, not {t.dtype}")
    return t.contiguous()


def _check_v(vec_length):
    if vec_length not in (2, 4, 8):
        raise ValueError(f"vec_length must be 2, 4 or 8, not {vec_length}")


def _mask(row_indices, row_offsets, column_indices):
    ro = _i32(row_offsets, "row_offsets")
    ci = _i32(column_indices, "column_indices")
    ri = _i32(row_indices, "row_indices") if row_indices is not None else None
    if ro.numel() % 2:
        raise ValueError("row_offsets holds (start, end) pairs")
    m_vec = ro.numel() // 2
    if ri is not None and ri.numel() != m_vec:
        raise ValueError(f"row_indices has {ri.numel()} entries for {m_vec} vector rows")
    return ri, ro, ci, m_vec


# ---------------------------------------------------------------------------
# quantization.cpp
# ---------------------------------------------------------------------------

def bquantization(input_matrix: torch.Tensor, bits: int, scale: float, stream=None) -> torch.Tensor:
    """fp16 [batch, L, D] -> int32 [batch, L, D * bits / 32], trunc(clamp(x * scale))."""
    return _bquantization(input_matrix, bits, scale, stream=stream)


def quantization(input_matrix: torch.Tensor, bits: int, scale: float, stream=None) -> torch.Tensor:
    """fp16 [L, D] -> int32 [L, D * bits / 32] (quantization.cpp:3-8)."""
    return _bquantization(input_matrix, bits, scale, stream=stream)


# ---------------------------------------------------------------------------
# deq_sddmm.cpp
# ---------------------------------------------------------------------------

def _bsddmm(bits, row_indices, row_offsets, column_indices, lhs_matrix, rhs_matrix, vec_length, scale, stream,
            batched):
    _check_v(vec_length)
    ri, ro, ci, m_vec = _mask(row_indices, row_offsets, column_indices)
    lhs = _i32(lhs_matrix, "lhs_matrix")
    rhs = _i32(rhs_matrix, "rhs_matrix")
    if batched:
        if lhs.dim() != 3 or rhs.dim() != 3 or lhs.shape[0] != rhs.shape[0]:
            raise ValueError("lhs_matrix [batch, m, k/(32/bits)] and rhs_matrix [batch, n, ...] expected")
        batch = rhs.shape[0]
    else:
        if lhs.dim() != 2 or rhs.dim() != 2:
            raise ValueError("lhs_matrix [m, k/(32/bits)] and rhs_matrix [n, ...] expected")
        batch = 1
    m, k_int32 = lhs.shape[-2], lhs.shape[-1]
    n = rhs.shape[-2]
    k = k_int32 * (32 // bits)
    if rhs.shape[-1] != k_int32:
        raise ValueError("lhs_matrix and rhs_matrix must share k")
    if m != m_vec * vec_length:
        raise ValueError(f"lhs_matrix has {m} rows; the mask covers {m_vec} vector rows of {vec_length}")
    # rows are written up to a multiple of 8 slots: of a mask that ends inside
    # such a group, past its last slot
    nnz, slots = ci.numel(), -(-ci.numel() // 8) * 8
    with _on(stream):
        full = torch.empty((batch, slots * vec_length), dtype=torch.float16, device=lhs.device)
        out = full if slots == nnz else full[:, :nnz * vec_length]
        lib, st = _lib.lib(), _stream_handle(stream)
        # K in one pass and a divisor the kernel's quotient covers: it stores fp16 itself
        if k <= 512 and m_vec and 2.0 ** -60 <= abs(scale) <= 2.0 ** 60:
            _lib.check(lib.mc_sddmm_batched_f16(bits, batch, m_vec, k, n, _ptr(ri), _ptr(ro), _ptr(ci), slots,
                                                _ptr(lhs), m * k_int32 * 4, _ptr(rhs), n * k_int32 * 4, float(scale),
                                                _ptr(full), slots * vec_length, vec_length, st), f"bsddmm_{bits}b")
        else:
            acc = torch.zeros((batch, slots * vec_length), dtype=torch.int32, device=lhs.device)
            _lib.check(lib.mc_sddmm_batched(bits, _lib.MC_SIGNED, 1, batch, m_vec, k, n, _ptr(ri), _ptr(ro), _ptr(ci),
                                            _ptr(lhs), m * k_int32 * 4, _ptr(rhs), n * k_int32 * 4, _ptr(acc),
                                            slots * vec_length, vec_length, st), f"bsddmm_{bits}b")
            _lib.check(lib.mc_attn_dequant_f16(_ptr(acc), acc.numel(), float(scale), _ptr(full), st), "bsddmm dequant")
        if not batched:
            return out.view(-1)
        return out if slots == nnz else out.contiguous()


def bsddmm_8b(row_indices, row_offsets, column_indices, lhs_matrix, rhs_matrix, vec_length: int, bits: int,
              scale: float, stream=None) -> torch.Tensor:
    """Batched S = Q K^T at the mask, fp16(int32 / scale) (deq_sddmm.cpp:82-93)."""
    return _bsddmm(8, row_indices, row_offsets, column_indices, lhs_matrix, rhs_matrix, vec_length, scale, stream,
                   True)


def bsddmm_4b(row_indices, row_offsets, column_indices, lhs_matrix, rhs_matrix, vec_length: int, bits: int,
              scale: float, stream=None) -> torch.Tensor:
    """4-bit Q and K (deq_sddmm.cpp:56-67)."""
    return _bsddmm(4, row_indices, row_offsets, column_indices, lhs_matrix, rhs_matrix, vec_length, scale, stream,
                   True)


def sddmm_8b(row_indices, row_offsets, column_indices, lhs_matrix, rhs_matrix, vec_length: int, bits: int,
             scale: float, stream=None) -> torch.Tensor:
    """One matrix: lhs [m, k/4], rhs [n, k/4] -> fp16 [nnz * V] (deq_sddmm.cpp:69-80)."""
    return _bsddmm(8, row_indices, row_offsets, column_indices, lhs_matrix, rhs_matrix, vec_length, scale, stream,
                   False)


def sddmm_4b(row_indices, row_offsets, column_indices, lhs_matrix, rhs_matrix, vec_length: int, bits: int,
             scale: float, stream=None) -> torch.Tensor:
    """One matrix, 4-bit operands (deq_sddmm.cpp:43-54)."""
    return _bsddmm(4, row_indices, row_offsets, column_indices, lhs_matrix, rhs_matrix, vec_length, scale, stream,
                   False)


# ---------------------------------------------------------------------------
# q_softmax.cpp
# ---------------------------------------------------------------------------

def q_bcsr_softmax(row_indices, row_offsets, values, sqrt_dk: float, scale: float, vec_length: int, batch_size: int,
                   bits: int, stream=None) -> torch.Tensor:
    """fp16 logits [batch, nnz * V] -> int32 [batch, nnz * V * bits / 32]: P
    quantized to ``bits`` (16, 8 or 4) in the reference's layouts, zeros
    between a row's padded end and the next row (q_softmax.cpp:37-49)."""
    _check_v(vec_length)
    if bits not in (16, 8, 4):
        raise ValueError("bits must be 16, 8 or 4")
    ri = _i32(row_indices, "row_indices")
    ro = _i32(row_offsets, "row_offsets")
    if not isinstance(values, torch.Tensor) or values.dtype != torch.float16 or not values.is_cuda:
        raise ValueError("values must be a float16 device tensor")
    vals = values.contiguous()
    if batch_size < 1 or vals.numel() % batch_size:
        raise ValueError(f"{vals.numel()} values do not split into {batch_size} matrices")
    stride = vals.numel() // batch_size
    if (stride * bits) % 32:
        raise ValueError(f"{stride} values per matrix do not pack into int32 words of {bits}-bit P")
    attn_stride = stride * bits // 32
    # rows are written in whole groups of slots: of a mask that ends inside
    # one, past its last slot
    group = 32 if bits == 4 else 16
    slots = -(-stride // (group * vec_length)) * group
    full_stride = slots * vec_length * bits // 32
    with _on(stream):
        lib, st = _lib.lib(), _stream_handle(stream)
        rows = ri.numel()
        if 2 * rows == ro.numel():
            # every row is written: only the slots between rows need zeros
            attn = torch.empty((batch_size, full_stride), dtype=torch.int32, device=vals.device)
            _lib.check(lib.mc_attn_zero_gaps(batch_size, rows, _ptr(ro), slots, group, vec_length * bits, _ptr(attn),
                                             full_stride * 4, st), "q_bcsr_softmax")
        else:
            attn = torch.zeros((batch_size, full_stride), dtype=torch.int32, device=vals.device)
        _lib.check(lib.mc_attn_softmax_f16(batch_size, rows, vec_length, _ptr(ri), _ptr(ro), _ptr(vals), stride,
                                           float(sqrt_dk), float(scale), bits, _ptr(attn), full_stride * 4, st),
                   "q_bcsr_softmax")
        return attn if full_stride == attn_stride else attn[:, :attn_stride].contiguous()


def q_csr_softmax(row_indices, row_offsets, values, sqrt_dk: float, scale: float, vec_length: int, bits: int,
                  stream=None) -> torch.Tensor:
    """One matrix: fp16 [nnz * V] -> int32 [nnz * V * bits / 32] (q_softmax.cpp:12-22)."""
    return q_bcsr_softmax(row_indices, row_offsets, values, sqrt_dk, scale, vec_length, 1, bits, stream)[0]


# ---------------------------------------------------------------------------
# deq_spmm.cpp
# ---------------------------------------------------------------------------

def _check_groups(slots: int, bits_lhs: int, bits_rhs: int) -> None:
    """The product reads P and the column indices of a row's last group whole:
    32 slots with 4-bit V, else 16.  A mask that ends inside a group (and the P
    that its size asks for) would be read past its end."""
    group = 32 if bits_rhs == 4 else 16
    if slots % group:
        raise ValueError(f"{bits_lhs}-bit P with {bits_rhs}-bit V needs the mask's slots in groups of {group}, "
                         f"not {slots}")


def _bspmm(bits_lhs, bits_rhs, row_indices, row_offsets, column_indices, values, rhs_matrix, vec_length, scale,
           stream):
    _check_v(vec_length)
    ri, ro, ci, m_vec = _mask(row_indices, row_offsets, column_indices)
    vals = _i32(values, "values")
    rhs = _i32(rhs_matrix, "rhs_matrix")
    if rhs.dim() != 3:
        raise ValueError("rhs_matrix [batch, k, n * bits / 32] expected")
    batch, k, n_int32 = rhs.shape
    n = n_int32 * (32 // bits_rhs)
    if vals.numel() % batch:
        raise ValueError("values do not split into one P per matrix")
    vals = vals.view(batch, -1)
    nnz = ci.numel()
    _check_groups(nnz, bits_lhs, bits_rhs)
    need = nnz * vec_length * bits_lhs // 8
    if vals.shape[1] * 4 < need:
        raise ValueError(f"values hold {vals.shape[1] * 4} bytes per matrix; the mask needs {need}")
    with _on(stream):
        m = m_vec * vec_length
        out = torch.empty((batch, m, n), dtype=torch.float16, device=rhs.device)
        _lib.check(_lib.lib().mc_spmm_batched_f16(bits_lhs, bits_rhs, batch, m_vec, vec_length, n, k, _ptr(ri),
                                                  _ptr(ro), _ptr(ci), _ptr(vals), vals.stride(0) * 4, _ptr(rhs),
                                                  k * n_int32 * 4, float(scale), _ptr(out), m * n,
                                                  _stream_handle(stream)), f"bspmm L{bits_lhs}-R{bits_rhs}")
    return out


def bspmm_8b(row_indices, row_offsets, column_indices, values, rhs_matrix, vec_length: int, bits_lhs: int,
             bits_rhs: int, scale: float, stream=None) -> torch.Tensor:
    """8-bit P x 8-bit V -> fp16 [batch, m, 64] (deq_spmm.cpp:73-94)."""
    return _bspmm(8, 8, row_indices, row_offsets, column_indices, values, rhs_matrix, vec_length, scale, stream)


def bspmm_16b8b(row_indices, row_offsets, column_indices, values, rhs_matrix, vec_length: int, bits_lhs: int,
                bits_rhs: int, scale: float, stream=None) -> torch.Tensor:
    """16-bit P x 8-bit V (deq_spmm.cpp:119-141)."""
    return _bspmm(16, 8, row_indices, row_offsets, column_indices, values, rhs_matrix, vec_length, scale, stream)


def bspmm_8b4b(row_indices, row_offsets, column_indices, values, rhs_matrix, vec_length: int, bits_lhs: int,
               bits_rhs: int, scale: float, stream=None) -> torch.Tensor:
    """8-bit P x 4-bit V (deq_spmm.cpp:96-117)."""
    return _bspmm(8, 4, row_indices, row_offsets, column_indices, values, rhs_matrix, vec_length, scale, stream)


def bspmm_4b(row_indices, row_offsets, column_indices, values, rhs_matrix, vec_length: int, bits_lhs: int,
             bits_rhs: int, scale: float, stream=None) -> torch.Tensor:
    """4-bit P x 4-bit V (deq_spmm.cpp:50-71)."""
    return _bspmm(4, 4, row_indices, row_offsets, column_indices, values, rhs_matrix, vec_length, scale, stream)
