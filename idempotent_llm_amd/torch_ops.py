"""The C-ABI entry points as torch custom operators ("detllm_rocm::...").

The reference registers its device kernels as ``torch.library.custom_op`` with
a ``register_fake`` shape function (src/detllm/ops/int_prims.py:96-136), so
dynamo and inductor see each one as a single opaque node: its compiled layer
(model.py:434-467) and its graph capture through ``torch._dynamo.run``
(graphed.py:108) trace straight through them. The rocm backend's operators
follow the same pattern: each op below runs one extern "C" entry point of
libdetllm_hip.so on torch's current stream, and its fake implementation
returns integer tensors of the right shape, so ``NoFloatMode`` holds during
tracing too. The ops are registered for CUDA (HIP) tensors only: there is no
CPU kernel behind them. Schemas, fakes and documentation are here; the
kernels behind them are native (csrc/torch_binding.cpp), so a call allocates
its outputs and launches without going through the interpreter again.

Cache tensors use this backend's paged layout (kvcache.py: per-layer K pool
[n_pages, n_kv, 128, 128], V pool [n_pages, n_kv, 128, 128] holding V
transposed per page, a [B, width] int32 page table, a [B, width * 128] bool
validity mask).
"""

from __future__ import annotations

import threading

import torch

from . import _lib

I64 = torch.int64
NS = "detllm_rocm"


OPS = ("int_gemm", "isqrt_i64", "ilog2_i64", "greedy_pick", "embed_normq", "norm_quant",
       "residual_normq", "swiglu_quant", "merge_rowcol", "qkv_epilogue", "attn_prefill",
       "attn_decode")


def _op(schema):
    """Define one operator; the decorated function is its fake (shapes and
    integer dtypes), the result the operator itself."""
    name = schema.split("(", 1)[0]
    assert name in OPS
    torch.library.define(f"{NS}::{name}", schema[len(name):], tags=(torch.Tag.pt2_compliant_tag,))

    def wrap(fake):
        torch.library.register_fake(f"{NS}::{name}")(fake)
        op = getattr(torch.ops.detllm_rocm, name)
        op.__doc__ = fake.__doc__
        return op

    return wrap


# ------------------------------------------------------------------ GEMM

@_op("int_gemm(Tensor a, Tensor b) -> Tensor")
def int_gemm(a, b):
    """backends.int_gemm(a, b, "rocm"): a [*, M, K] int8 x b [*, K, N] int8 ->
    int32 [*, M, N] (a 2-D b is shared by every leading index). Other shapes
    raise ValueError, traced or run."""
    torch._check_value(a.dim() >= 2 and b.dim() >= 2, lambda: "int_gemm: operands of rank 2 or more")
    torch._check_value(b.dim() == 2 or a.dim() == b.dim(), lambda: "int_gemm: leading dimensions differ")
    torch._check_value(a.shape[-1] == b.shape[-2], lambda: "int_gemm: K differs")
    if b.dim() > 2:
        for m, n in zip(a.shape[:-2], b.shape[:-2]):
            torch._check_value(m == n, lambda: "int_gemm: leading dimensions differ")
    return a.new_empty(tuple(a.shape[:-1]) + (b.shape[-1],), dtype=torch.int32)


@_op("isqrt_i64(Tensor a) -> Tensor")
def isqrt_i64(a):
    """int_prims.py:96-103 (detllm::isqrt_i64): floor sqrt of int64."""
    return torch.empty_like(a, dtype=I64)


@_op("ilog2_i64(Tensor a) -> Tensor")
def ilog2_i64(a):
    """int_prims.py:106-113 (detllm::ilog2_i64): floor log2 of int64."""
    return torch.empty_like(a, dtype=I64)


@_op("greedy_pick(Tensor logits, Tensor head_m) -> Tensor")
def greedy_pick(logits, head_m):
    """IntQwen3.greedy_pick (model.py:482-490): [R, V] int32 -> [R] int64."""
    return logits.new_empty(logits.shape[0], dtype=I64)


# ------------------------------------------------------- fused row kernels

def _rows_fake(R, C, like):
    return (like.new_empty(R, C, dtype=torch.int8), like.new_empty(R, dtype=I64),
            like.new_empty(R, dtype=I64))


@_op("embed_normq(Tensor ids, Tensor e8, Tensor em, Tensor ek, Tensor? sm_m, SymInt sm_k, "
     "Tensor(a6!) err) -> (Tensor, Tensor, Tensor, Tensor, Tensor)")
def embed_normq(ids, e8, em, ek, sm_m, sm_k, err):
    """Embedding + residual_from_delta + _norm_quant (model.py:246-249,
    :187-198): ids [R] -> (h int32 [R, H], k_res, x8 int8 [R, H], xm, xk)."""
    R, H = ids.numel(), e8.shape[1]
    return (ids.new_empty(R, H, dtype=torch.int32), ids.new_empty(R, dtype=I64),
            *_rows_fake(R, H, ids))


@_op("norm_quant(Tensor h, Tensor? sm_m, SymInt sm_k) -> (Tensor, Tensor, Tensor)")
def norm_quant(h, sm_m, sm_k):
    """IntQwen3._norm_quant (model.py:187-198): h [R, C] int32 -> (x8, xm, xk)."""
    return _rows_fake(h.shape[0], h.shape[1], h)


@_op("residual_normq(Tensor P, Tensor row_m, Tensor row_k, Tensor col_m, SymInt col_k, "
     "SymInt tb, Tensor(a6!) h, Tensor(a7!) k_res, Tensor? sm_m, SymInt sm_k) "
     "-> (Tensor, Tensor, Tensor)")
def residual_normq(P, row_m, row_k, col_m, col_k, tb, h, k_res, sm_m, sm_k):
    """requant_i32_common(tb) + residual_add + _norm_quant (model.py:410-415,
    :424-427): P int32 [nsplit, R, C] partials; h [R, C], k_res [R] updated
    in place; returns the next GEMM's (x8, xm, xk)."""
    return _rows_fake(P.shape[1], P.shape[2], P)


@_op("swiglu_quant(Tensor P, Tensor xm, Tensor xk, Tensor gate_m, SymInt gate_k, Tensor up_m, "
     "SymInt up_k, Tensor ds_m, SymInt ds_k) -> (Tensor, Tensor, Tensor)")
def swiglu_quant(P, xm, xk, gate_m, gate_k, up_m, up_k, ds_m, ds_k):
    """gate/up requant_i32_common(14) + di_swiglu + quant_i8_pertoken
    (model.py:416-423): P int32 [nsplit, R, 2I] -> (y8 [R, I], ym, yk)."""
    return _rows_fake(P.shape[1], P.shape[2] // 2, P)


@_op("merge_rowcol(Tensor attn, Tensor os_m, SymInt os_k, Tensor col_m, SymInt col_k) "
     "-> (Tensor, Tensor, Tensor)")
def merge_rowcol(attn, os_m, os_k, col_m, col_k):
    """requant_i8_rowcol(attn * os_m, 1, os_k, col_m, col_k) (model.py:404-409):
    attn int64 [R, C] -> (a8, am, ak)."""
    return _rows_fake(attn.shape[0], attn.shape[1], attn)


# ------------------------------------------------------------- attention

@_op("qkv_epilogue(Tensor P, SymInt B, SymInt T, SymInt n_q, SymInt n_kv, Tensor xm, Tensor xk, "
     "Tensor positions, Tensor q_m, SymInt q_k, Tensor k_m, SymInt k_k, Tensor v_m, SymInt v_k, "
     "Tensor q_norm_m, SymInt q_norm_k, Tensor k_norm_m, SymInt k_norm_k, Tensor qs_m, "
     "SymInt qs_k, Tensor kq_m, Tensor kq_k, Tensor ks_m, Tensor ks_k, Tensor vq_m, Tensor vq_k, "
     "Tensor cos_t, Tensor sin_t, Tensor(a28!) kpool, Tensor(a29!) vpool, Tensor table, "
     "SymInt slot_base, Tensor(a32!) err) -> (Tensor, Tensor)")
def qkv_epilogue(P, B, T, n_q, n_kv, *rest):
    """_qk_head_pipeline + QK smoothing + Q quant + K/V static requant into
    the cache + score scale / DI-Exp constant (model.py:200-216, :303-358).
    P int32 [nsplit, B*T, (n_q + 2 n_kv) * 128]; returns (q8 [B, n_q, T, 128],
    tpos [B, n_q, T])."""
    return P.new_empty(B, n_q, T, 128, dtype=torch.int8), P.new_empty(B, n_q, T, dtype=I64)


@_op("attn_prefill(Tensor q8, Tensor tpos, Tensor kpool, Tensor vpool, Tensor table, "
     "Tensor valid, SymInt S_past) -> Tensor")
def attn_prefill(q8, tpos, kpool, vpool, table, valid, S_past):
    """Prefill attention (model.py:382-402): q8 [B, n_q, T, 128] over the
    cache's first S_past + T slots (causal by slot, valid-masked) -> exact
    int64 context [B, T, n_q * 128]."""
    B, n_q, T, _ = q8.shape
    return q8.new_empty(B, T, n_q * 128, dtype=I64)


@_op("attn_decode(Tensor q8, Tensor tpos, Tensor kpool, Tensor vpool, Tensor table, "
     "Tensor valid, SymInt S, Tensor(a7!) err) -> Tensor")
def attn_decode(q8, tpos, kpool, vpool, table, valid, S, err):
    """Decode attention (model.py:347-381, ops/fused_attn.py:47-142): one
    query per row, q8 [B, n_q, 128], over S slots -> int64 [B, n_q * 128]."""
    return q8.new_empty(q8.shape[0], q8.shape[1] * 128, dtype=I64)


# Loading the native binding registers the kernels. Where it cannot be loaded
# (not built, or built for another torch), the import goes on and a call of an
# operator raises, as the other entries do; a call after it has been built
# loads it.
_stand_ins = None
_loading = threading.Lock()


def _load_kernels():
    global _stand_ins
    with _loading:
        if _stand_ins is None:
            return
        _stand_ins._destroy()     # (before the kernels of the same key are registered)
        try:
            _lib.native()
        except Exception:
            _register_stand_ins()
            raise
        _stand_ins = None


def _register_stand_ins():
    global _stand_ins
    _stand_ins = torch.library.Library(NS, "IMPL")
    for name in OPS:
        def call_again(keyset, *args, _op=getattr(torch.ops.detllm_rocm, name).default, **kwargs):
            _load_kernels()
            return _op.redispatch(keyset, *args, **kwargs)
        _stand_ins.impl(name, call_again, "CUDA", with_keyset=True)


try:
    _lib.native()
except _lib.LibraryMissing:
    _register_stand_ins()
