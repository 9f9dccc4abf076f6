"""The tensor-level ops behind kernels/host.py, over libak355's C ABI through ctypes.

Each function has the name and signature of the torch op that the HuggingFace Kernels package
registers for the same C entry point (hf_export/torch_binding.cpp): outputs first, then inputs,
then scalars. So kernels/host.py, the one shape / dtype layer of every kernel_fn, runs unchanged
on either: bound to this module in-tree, bound to the package's torch ops in the export. Each op
makes the input's device current (when it is not already), launches on torch's current stream of
that device and raises AkError on a non-OK status.
"""
from __future__ import annotations

import ctypes
import functools

import torch

from .. import _lib


_code = _lib.dtype_code
_I64x3 = ctypes.c_int64 * 3

# torch.cuda.current_device() without its initialisation check (0.24 us per call -> 0.06): every caller
# has a GPU tensor in hand
_current_device = getattr(torch._C, "_cuda_getDevice", torch.cuda.current_device)


def _run(fn_name: str, ref: torch.Tensor, info, *args) -> None:
    """Call fn_name(*args, stream) on ref's device. info: a function giving the error message's
    details (None: ref's shape and dtype), called for a failed launch only, so that a good one does
    not build them."""
    idx = ref.get_device()
    if idx < 0:
        raise RuntimeError(f"{fn_name}: expected GPU tensors, got one on {ref.device} (no CPU path)")
    fn = getattr(_lib.load(), fn_name)
    if idx == _current_device():
        st = fn(*args, _lib.stream_of_index(idx))
    else:
        with torch.cuda.device(idx):
            st = fn(*args, _lib.stream_of_index(idx))
    if st != _lib.AK_OK:
        _lib.check(st, fn_name, **(dict(shape=tuple(ref.shape), dtype=ref.dtype) if info is None else info()))


def rmsnorm(y: torch.Tensor, x: torch.Tensor, weight: torch.Tensor, eps: float) -> None:
    _run("ak_rmsnorm", x, None, _code(x, "rmsnorm"), x.data_ptr(),
         weight.data_ptr(), y.data_ptr(), x.shape[0], x.shape[1], float(eps))


def rmsnorm_rsqrt(y: torch.Tensor, x: torch.Tensor, weight: torch.Tensor, eps: float) -> None:
    _run("ak_rmsnorm_rsqrt", x, None, _code(x, "rmsnorm"), x.data_ptr(),
         weight.data_ptr(), y.data_ptr(), x.shape[0], x.shape[1], float(eps))


def layernorm(y: torch.Tensor, x: torch.Tensor, weight: torch.Tensor | None, bias: torch.Tensor | None,
              eps: float) -> None:
    _run("ak_layernorm", x, None, _code(x, "layernorm"), x.data_ptr(),
         _lib.ptr(weight), _lib.ptr(bias), y.data_ptr(), x.shape[0], x.shape[1], float(eps))


def softmax(y: torch.Tensor, x: torch.Tensor) -> None:
    _run("ak_softmax", x, None, _code(x, "softmax"), x.data_ptr(),
         y.data_ptr(), x.shape[0], x.shape[1])


def rope(y: torch.Tensor, x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, rep_inner: int) -> None:
    _run("ak_rope", x, None, _code(x, "rotary_embedding"), x.data_ptr(),
         cos.data_ptr(), sin.data_ptr(), y.data_ptr(), x.shape[0], x.shape[1], cos.shape[0], int(rep_inner))


def cross_entropy(out: torch.Tensor, row_loss: torch.Tensor, logits: torch.Tensor, targets: torch.Tensor,
                  ignore_index: int) -> None:
    _run("ak_cross_entropy", logits, None,
         _code(logits, "cross_entropy"), logits.data_ptr(), targets.data_ptr(), row_loss.data_ptr(), out.data_ptr(),
         logits.shape[0], logits.shape[1], int(ignore_index))


@functools.lru_cache(maxsize=1024)
def _reduce_workspace_bytes(dtype: int, outer: int, reduce: int, inner: int) -> int:
    """Remembered per argument tuple: the slicing decision depends on the arguments alone."""
    return _lib.load().ak_reduce_workspace_bytes(dtype, outer, reduce, inner)


def _reduce(name: str, y: torch.Tensor, x: torch.Tensor, outer: int, reduce: int, inner: int) -> None:
    code = _code(x, name)
    nbytes = _reduce_workspace_bytes(code, outer, reduce, inner) if inner > 1 else 0
    if nbytes > 0:  # fp32 partial sums of row slices
        ws = torch.empty(nbytes // 4, device=x.device, dtype=torch.float32)
        _run(f"ak_{name}_ws", x, None, code, x.data_ptr(), y.data_ptr(),
             outer, reduce, inner, ws.data_ptr(), nbytes)
        return
    _run(f"ak_{name}", x, None, code, x.data_ptr(), y.data_ptr(), outer,
         reduce, inner)


def reduce_sum(y: torch.Tensor, x: torch.Tensor, outer: int, reduce: int, inner: int) -> None:
    _reduce("reduce_sum", y, x, outer, reduce, inner)


def reduce_max(y: torch.Tensor, x: torch.Tensor, outer: int, reduce: int, inner: int) -> None:
    _reduce("reduce_max", y, x, outer, reduce, inner)


def _ld(t: torch.Tensor) -> int:
    return t.stride(0) if t.shape[0] > 1 else max(t.shape[1], 1)


def gemm(c: torch.Tensor, a: torch.Tensor, b: torch.Tensor, b_trans: bool,
         workspace: torch.Tensor | None = None) -> None:
    """c [M, N] = a [M, K] @ op(b): b stored [K, N] (b_trans False) or [N, K] (True); every operand
    with a unit stride along its last dim, row strides passed through."""
    M, K = a.shape
    N = b.shape[0] if b_trans else b.shape[1]
    code = _code(a, "matmul")
    if workspace is not None and workspace.numel() > 0:
        _run("ak_gemm_ws", a, lambda: dict(M=M, N=N, K=K, b_trans=b_trans, dtype=a.dtype), code, a.data_ptr(),
             b.data_ptr(), c.data_ptr(), M, N, K, _ld(a), _ld(b), _ld(c), int(bool(b_trans)), workspace.data_ptr(),
             workspace.numel() * 4)
        return
    _run("ak_gemm", a, lambda: dict(M=M, N=N, K=K, b_trans=b_trans, dtype=a.dtype), code, a.data_ptr(), b.data_ptr(),
         c.data_ptr(), M, N, K, _ld(a), _ld(b), _ld(c), int(bool(b_trans)))


def gemm_batched(c: torch.Tensor, a: torch.Tensor, b: torch.Tensor, b_trans: bool) -> None:
    """c [Z, M, N] = a [Z, M, K] @ op(b) for each batch item z: b stored [Z, K, N] (b_trans False) or
    [Z, N, K] (True); unit stride along each last dim, any row and batch strides (0 broadcasts)."""
    Z, M, K = a.shape
    N = b.shape[1] if b_trans else b.shape[2]

    def ld(t):
        return t.stride(1) if t.shape[1] > 1 else max(t.shape[2], 1)
    _run("ak_gemm_batched", a, lambda: dict(Z=Z, M=M, N=N, K=K, b_trans=b_trans, dtype=a.dtype), _code(a, "matmul"),
         a.data_ptr(), b.data_ptr(), c.data_ptr(), Z, M, N, K, ld(a), ld(b), ld(c), a.stride(0), b.stride(0),
         c.stride(0), int(bool(b_trans)))


def gemm_bias(c: torch.Tensor, a: torch.Tensor, b: torch.Tensor, bias: torch.Tensor, b_trans: bool) -> None:
    """c = a @ op(b) + bias [N], the bias added to the fp32 accumulator (one rounding)."""
    M, K = a.shape
    N = b.shape[0] if b_trans else b.shape[1]
    _run("ak_gemm_bias", a, lambda: dict(M=M, N=N, K=K, b_trans=b_trans, dtype=a.dtype), _code(a, "gemm_bias"),
         a.data_ptr(), b.data_ptr(), bias.data_ptr(), c.data_ptr(), M, N, K, _ld(a), _ld(b), _ld(c),
         int(bool(b_trans)))


def gemm_bias_gelu(c: torch.Tensor, a: torch.Tensor, b: torch.Tensor, bias: torch.Tensor, b_trans: bool) -> None:
    """c = gelu(a @ op(b) + bias): the biased product rounded, then exact GELU, rounded again."""
    M, K = a.shape
    N = b.shape[0] if b_trans else b.shape[1]
    _run("ak_gemm_bias_gelu", a, lambda: dict(M=M, N=N, K=K, b_trans=b_trans, dtype=a.dtype),
         _code(a, "gemm_bias_gelu"), a.data_ptr(), b.data_ptr(), bias.data_ptr(), c.data_ptr(), M, N, K, _ld(a),
         _ld(b), _ld(c), int(bool(b_trans)))


def gemm_bias_residual(c: torch.Tensor, a: torch.Tensor, b: torch.Tensor, bias: torch.Tensor, r: torch.Tensor,
                       b_trans: bool) -> None:
    """c = r + (a @ op(b) + bias): the biased product rounded, then the sum (r shares c's row stride)."""
    M, K = a.shape
    N = b.shape[0] if b_trans else b.shape[1]
    _run("ak_gemm_bias_residual", a, lambda: dict(M=M, N=N, K=K, b_trans=b_trans, dtype=a.dtype),
         _code(a, "gemm_bias_residual"), a.data_ptr(), b.data_ptr(), bias.data_ptr(), r.data_ptr(), c.data_ptr(), M,
         N, K, _ld(a), _ld(b), _ld(c), int(bool(b_trans)))


def gemm_residual(c: torch.Tensor, a: torch.Tensor, b: torch.Tensor, r: torch.Tensor, b_trans: bool) -> None:
    """c = r + a @ op(b), the product rounded, then the sum (r shares c's row stride)."""
    M, K = a.shape
    N = b.shape[0] if b_trans else b.shape[1]
    _run("ak_gemm_residual", a, lambda: dict(M=M, N=N, K=K, b_trans=b_trans, dtype=a.dtype),
         _code(a, "gemm_residual"), a.data_ptr(), b.data_ptr(), r.data_ptr(), c.data_ptr(), M, N, K, _ld(a), _ld(b),
         _ld(c), int(bool(b_trans)))


def linear(c: torch.Tensor, x: torch.Tensor, w: torch.Tensor, bias: torch.Tensor | None, r: torch.Tensor | None,
           gelu: bool, M: int, N: int, K: int) -> None:
    """gemm_bias, gemm_bias_gelu, gemm_bias_residual or gemm_residual (whichever bias, r and gelu
    name) of dense x [.., K] (M rows), w [N, K], bias [N], r and c [.., N], whatever their rank."""
    name, mid = (("ak_gemm_residual", (r.data_ptr(),)) if bias is None
                 else ("ak_gemm_bias_residual", (bias.data_ptr(), r.data_ptr())) if r is not None
                 else ("ak_gemm_bias_gelu" if gelu else "ak_gemm_bias", (bias.data_ptr(),)))
    _run(name, x, lambda: dict(M=M, N=N, K=K, b_trans=True, dtype=x.dtype), _code(x, "linear"), x.data_ptr(),
         w.data_ptr(), *mid, c.data_ptr(), M, N, K, K, K, max(N, 1), 1)


def gemm_rope(c: torch.Tensor, a: torch.Tensor, b: torch.Tensor, b_trans: bool, cos: torch.Tensor, sin: torch.Tensor,
              seq_len: int, head_dim: int, rot_cols: int) -> None:
    """c = a @ op(b) with the model's rotary embedding on columns [0, rot_cols) (fp32 tables)."""
    M, K = a.shape
    N = b.shape[0] if b_trans else b.shape[1]
    _run("ak_gemm_rope", a, lambda: dict(M=M, N=N, K=K, head_dim=head_dim, rot_cols=rot_cols, dtype=a.dtype),
         _code(a, "gemm_rope"), a.data_ptr(), b.data_ptr(), c.data_ptr(), M, N, K, _ld(a), _ld(b), _ld(c),
         int(bool(b_trans)), cos.data_ptr(), sin.data_ptr(), seq_len, head_dim, rot_cols)


def rope_f32_tables(y: torch.Tensor, x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor, rows: int, head_dim: int,
                    table_rows: int, rep_inner: int, x_tok_stride: int) -> None:
    """The model's RoPE: x (rows / rep_inner tokens of rep_inner heads, token stride x_tok_stride)
    rotated by fp32 tables into dense y."""
    _run("ak_rope_f32_tables", x, None, _code(x, "rope_f32_tables"),
         x.data_ptr(), cos.data_ptr(), sin.data_ptr(), y.data_ptr(), rows, head_dim, table_rows, rep_inner,
         x_tok_stride)


@functools.lru_cache(maxsize=1024)
def gemm_workspace_bytes(dtype: int, M: int, N: int, K: int, lda: int, ldb: int, ldc: int, b_trans: bool) -> int:
    """Remembered per argument tuple: the split decision depends on the arguments alone."""
    return _lib.load().ak_gemm_workspace_bytes(dtype, M, N, K, lda, ldb, ldc, int(bool(b_trans)))


def mlp_gate_up(h: torch.Tensor, x: torch.Tensor, w_gate: torch.Tensor, w_up: torch.Tensor, activation: int) -> None:
    M, D = x.shape
    H = w_gate.shape[0]
    _run("ak_mlp_gate_up", x, lambda: dict(M=M, H=H, D=D, dtype=x.dtype), _code(x, "fused_mlp"), x.data_ptr(),
         w_gate.data_ptr(), w_up.data_ptr(), h.data_ptr(), M, H, D, int(activation))


@functools.lru_cache(maxsize=1024)
def _attn_workspace_bytes(dtype: int, B: int, Hq: int, Hkv: int, Sq: int, Sk: int, D: int, causal: bool) -> int:
    return _lib.load().ak_flash_attn_workspace_bytes(dtype, B, Hq, Hkv, Sq, Sk, D, int(causal))


def flash_attn_fwd(o: torch.Tensor, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, causal: bool,
                   sm_scale: float) -> None:
    """Q, O [B, Hq, Sq, D], K, V [B, Hkv, Sk, D], any strides with a contiguous head_dim."""
    B, Hq, Sq, D = q.shape
    Hkv, Sk = k.shape[1], k.shape[2]
    st = [_I64x3(*t.stride()[:3]) for t in (q, k, v, o)]
    code = _code(q, "flash_attention")
    # fp32 partials of key slices: only calls with few query rows per KV head have any
    nbytes = _attn_workspace_bytes(code, B, Hq, Hkv, Sq, Sk, D, bool(causal)) if Sq <= 16 else 0
    if nbytes > 0:
        ws = torch.empty(nbytes // 4, device=q.device, dtype=torch.float32)
        _run("ak_flash_attn_fwd_ws", q, lambda: dict(Q=tuple(q.shape), K=tuple(k.shape), dtype=q.dtype), code,
             q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), B, Hq, Hkv, Sq, Sk, D, st[0], st[1], st[2],
             st[3], int(bool(causal)), float(sm_scale), ws.data_ptr(), nbytes)
        return
    _run("ak_flash_attn_fwd", q, lambda: dict(Q=tuple(q.shape), K=tuple(k.shape), dtype=q.dtype), code, q.data_ptr(),
         k.data_ptr(), v.data_ptr(), o.data_ptr(), B, Hq, Hkv, Sq, Sk, D, st[0], st[1], st[2], st[3],
         int(bool(causal)), float(sm_scale))
