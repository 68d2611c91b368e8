"""The decoder's memory-bound operators on MI355X (gfx950) HIP kernels.

Drop-ins for the reference's operator functions in
``src/mega_trading/kernels/triton_ops.py``:

* ``rms_norm(hidden, weight, *, eps)``            <- ``triton_rms_norm`` (:11-15)
* ``add_rms_norm(hidden, residual, weight, *, eps)`` <- ``triton_add_rms_norm`` (:18-42)
* ``swiglu_gate(gate, up)``                       <- ``triton_swiglu_gate`` (:57-61)
* ``apply_rope(query, key, cos, sin)``            <- ``triton_apply_rope`` (:45-54)
* ``fused_linear_cross_entropy(hidden, weight, labels, *, ignore_index)``
                                                  <- ``triton_fused_linear_cross_entropy`` (:64-92)

Same argument meaning and results (fp32 arithmetic; outputs in the input
dtype; the roundings between steps as the reference performs them).  The
reference silently falls back to PyTorch for tensors it cannot handle; these
raise instead (``RuntimeError`` off the GPU or for an unsupported dtype,
``ValueError`` for shapes), so a run can never route around the kernels.

Each is a ``torch.library`` op with a fake implementation here and its GPU
kernels and backward in ``libmt_torch.so`` (``csrc/mt_torch.cpp``), launched on
the caller's current stream; the loss head's forward, which runs library GEMMs,
is Python.
"""

from __future__ import annotations

import torch

from . import _native
from .gemm_tuning import tuned_gemms

__all__ = ["rms_norm", "add_rms_norm", "rms_norm_mixed", "add_rms_norm_mixed", "swiglu_gate", "swiglu_gate_packed",
           "apply_rope", "fused_linear_cross_entropy", "topk_sample", "MAX_NORM_DIM", "MAX_SAMPLE_VOCAB"]

MAX_NORM_DIM = 4096
MAX_SAMPLE_VOCAB = 32768  # vocabulary of one topk_sample row (1024 threads x 32 values in registers)
_DT = {torch.bfloat16: _native.DTYPE_BF16, torch.float16: _native.DTYPE_FP16, torch.float32: _native.DTYPE_FP32}
_DTYPE_OF = {v: k for k, v in _DT.items()}


# ---------------------------------------------------------------------------
# public functions
# ---------------------------------------------------------------------------
def rms_norm(hidden: torch.Tensor, weight: torch.Tensor, *, eps: float) -> torch.Tensor:
    """``hidden * rsqrt(mean(hidden^2, -1) + eps) * weight`` (``triton_ops.py:11``, kernel ``:528-539``)."""
    _check_norm(hidden, weight)
    _native.ensure()
    y, _rstd = _rms_norm_fwd(hidden, weight, float(eps))
    return y


def add_rms_norm(
    hidden: torch.Tensor, residual: torch.Tensor, weight: torch.Tensor, *, eps: float
) -> tuple[torch.Tensor, torch.Tensor]:
    """``(new_residual, normed)`` with ``new_residual = hidden + residual`` and
    ``normed = RMSNorm(new_residual)`` from the unrounded sum (``triton_ops.py:18-42``)."""
    _check_norm(hidden, weight)
    if residual.shape != hidden.shape:
        raise ValueError("residual must have the same shape as hidden")
    if residual.dtype != hidden.dtype or residual.device != hidden.device:
        raise RuntimeError("residual must have the dtype and device of hidden")
    _native.ensure()
    new_res, y, _rstd = _add_rms_norm_fwd(hidden, residual, weight, float(eps))
    return new_res, y


def rms_norm_mixed(hidden: torch.Tensor, weight: torch.Tensor, *, eps: float, out_dtype: torch.dtype) -> torch.Tensor:
    """``rms_norm`` of an fp32 residual stream with the result rounded once to
    the 16-bit ``out_dtype``: what the fp32 norm followed by the next
    projection's autocast cast gives, in one pass.  ``weight`` fp32."""
    _check_norm(hidden, weight)
    _check_mixed(hidden, weight, out_dtype)
    _native.ensure()
    y, _rstd = _rms_norm_fwd_mixed(hidden, weight, float(eps), _DT[out_dtype])
    return y


def add_rms_norm_mixed(
    branch: torch.Tensor, residual: torch.Tensor, weight: torch.Tensor, *, eps: float
) -> tuple[torch.Tensor, torch.Tensor]:
    """``(new_residual, normed)``: ``new_residual = residual + branch`` in fp32
    (torch's promotion of an fp32 residual stream plus a 16-bit branch output)
    and ``normed = RMSNorm(new_residual)`` rounded once to the branch's dtype.
    ``residual`` and ``weight`` fp32, ``branch`` bf16 or fp16."""
    _check_norm(residual, weight)
    _check_mixed(residual, weight, branch.dtype)
    if branch.shape != residual.shape:
        raise ValueError("branch must have the shape of residual")
    if branch.device != residual.device:
        raise RuntimeError("branch must be on the device of residual")
    _native.ensure()
    new_res, y, _rstd = _add_rms_norm_fwd_mixed(branch, residual, weight, float(eps))
    return new_res, y


def swiglu_gate(gate: torch.Tensor, up: torch.Tensor) -> torch.Tensor:
    """``silu(gate) * up`` with silu rounded to the input dtype first (``triton_ops.py:57-61``)."""
    _check_device_dtype(gate, "gate")
    if up.shape != gate.shape:
        raise ValueError("gate and up must have the same shape")
    if up.dtype != gate.dtype or up.device != gate.device:
        raise RuntimeError("up must have the dtype and device of gate")
    _native.ensure()
    return _swiglu_fwd(gate, up)


def swiglu_gate_packed(gate_up: torch.Tensor) -> torch.Tensor:
    """``swiglu_gate(gate, up)`` on the packed [..., 2F] output of one GEMM
    against the stacked (w1; w3) weights: gate = the first F columns of each
    row, up = the last F.  Returns [..., F].  No reference counterpart (the
    reference gate takes the two products, ``triton_ops.py:57-61``); the
    arithmetic and roundings are ``swiglu_gate``'s."""
    _check_device_dtype(gate_up, "gate_up")
    if gate_up.ndim < 1 or gate_up.shape[-1] % 16:
        raise ValueError("gate_up's last dim must be 2F with F a multiple of 8")
    _native.ensure()
    return _swiglu_packed_fwd(gate_up)


def apply_rope(
    query: torch.Tensor, key: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor
) -> tuple[torch.Tensor, torch.Tensor]:
    """``(rot(query), rot(key))`` (``triton_apply_rope``, ``triton_ops.py:45-54``).

    ``query`` [B, Hq, T, D] and ``key`` [B, Hkv, T, D] (any strides), tables
    [1, 1, >= T, D/2] as ``RotaryEmbedding`` keeps them (any float dtype, read
    as fp32; rows past T are ignored).  Each interleaved pair (e, o) of row t
    becomes (e cos - o sin, e sin + o cos) in fp32 with one rounding to the
    input dtype; outputs have the inputs' layout.  The backward rotates the
    gradients by -theta (``triton_ops.py:204-214``)."""
    _check_device_dtype(query, "query")
    if key.dtype != query.dtype or key.device != query.device:
        raise RuntimeError("key must have the dtype and device of query")
    if query.ndim != 4 or key.ndim != 4:
        raise ValueError("query and key must be [B, H, T, D]")
    b, _hq, t, d = query.shape
    if key.shape[0] != b or key.shape[2] != t or key.shape[3] != d:
        raise ValueError("key must be [B, Hkv, T, D] with the B, T and D of query")
    if d % 2:
        raise ValueError("RoPE requires an even head dimension")
    c = _rope_table(cos, "cos", t, d, query.device)
    s = _rope_table(sin, "sin", t, d, query.device)
    if s.shape != c.shape:
        raise ValueError("cos and sin must have the same shape")
    _native.ensure()
    return _rope_fwd(query, key, c, s, False)


def fused_linear_cross_entropy(
    hidden: torch.Tensor, weight: torch.Tensor, labels: torch.Tensor, *, ignore_index: int = -100
) -> torch.Tensor:
    """Mean cross-entropy of ``hidden @ weight.T`` against ``labels`` without the
    [rows, vocab] logits ever existing at once (``triton_ops.py:64-92``).

    ``hidden`` [rows, H], ``weight`` [vocab, H] (``nn.Linear(bias=False).weight``),
    ``labels`` [rows] int32/int64; rows labelled ``ignore_index`` contribute
    nothing (all ignored: loss 0, zero gradients).  Rows are processed in chunks
    of at most 2 GB of logits: one GEMM for the chunk's logits, the HIP
    cross-entropy row kernel (loss and, in place, the logits gradient), then
    the two gradient GEMMs; the gradients are computed in the
    forward and scaled by the incoming gradient in the backward, as the
    reference does.  Under CUDA autocast the GEMMs run in the autocast dtype
    (what ``F.linear`` + ``F.cross_entropy`` do there); otherwise in hidden's
    dtype.  The loss is fp32.
    """
    if hidden.ndim != 2:
        raise ValueError("hidden must have shape [rows, hidden_dim]")
    if weight.ndim != 2 or weight.shape[1] != hidden.shape[1]:
        raise ValueError("weight must have shape [vocab, hidden_dim] matching hidden's last dim")
    if labels.ndim != 1 or labels.shape[0] != hidden.shape[0]:
        raise ValueError("labels must be a 1D tensor with one entry per hidden row")
    if labels.dtype not in (torch.int32, torch.int64):
        raise ValueError("labels must be an integer tensor")
    _check_device_dtype(hidden, "hidden")
    _check_device_dtype(weight, "weight")
    if torch.is_autocast_enabled("cuda"):
        compute = torch.get_autocast_dtype("cuda")
    else:
        compute = torch.promote_types(hidden.dtype, weight.dtype)
    need_grad = torch.is_grad_enabled() and (hidden.requires_grad or weight.requires_grad)
    _native.ensure()
    with torch.autocast("cuda", enabled=False):
        loss, _gh, _gw = _fused_linear_ce(
            hidden, weight, labels, int(ignore_index), _DT[compute], need_grad)
    return loss


# ---------------------------------------------------------------------------
# helpers
# ---------------------------------------------------------------------------
def _check_device_dtype(t: torch.Tensor, name: str) -> None:
    if t.device.type != "cuda" or not torch.version.hip:
        raise RuntimeError(f"{name} must be on a ROCm GPU (got device {t.device})")
    if t.dtype not in _DT:
        raise RuntimeError(f"{name} dtype {t.dtype} unsupported (bfloat16, float16 or float32)")


def _check_norm(hidden: torch.Tensor, weight: torch.Tensor) -> None:
    _check_device_dtype(hidden, "hidden")
    d = hidden.shape[-1] if hidden.ndim else 0
    if hidden.ndim < 1 or weight.ndim != 1 or weight.numel() != d:
        raise ValueError("weight must be 1-D with hidden.shape[-1] elements")
    if d % 8 or d > MAX_NORM_DIM:
        raise ValueError(f"hidden_dim {d} unsupported: a multiple of 8 up to {MAX_NORM_DIM}")
    if weight.device != hidden.device:
        raise RuntimeError("weight must be on the device of hidden")


def _check_mixed(stream: torch.Tensor, weight: torch.Tensor, act: torch.dtype) -> None:
    if stream.dtype != torch.float32 or weight.dtype != torch.float32:
        raise RuntimeError("the residual stream and the weight must be float32")
    if act not in (torch.bfloat16, torch.float16):
        raise RuntimeError(f"activation dtype {act} unsupported (bfloat16 or float16)")


def _rope_table(table: torch.Tensor, name: str, t: int, d: int, device: torch.device) -> torch.Tensor:
    """A [..., rows, D/2] table (leading dims of size 1) as fp32 [rows, D/2] with unit d stride."""
    if table.ndim < 2 or any(n != 1 for n in table.shape[:-2]) or table.shape[-1] != d // 2:
        raise ValueError(f"{name} must be [1, 1, T, D/2] with D/2 = {d // 2} (got {tuple(table.shape)})")
    if table.shape[-2] < t:
        raise ValueError(f"{name} has {table.shape[-2]} rows, fewer than the sequence length {t}")
    if table.device != device:
        raise RuntimeError(f"{name} must be on the device of query")
    flat = table.reshape(table.shape[-2], table.shape[-1]).to(torch.float32)
    if flat.stride(-1) != 1:
        flat = flat.contiguous()
    return flat


def _stream(t: torch.Tensor) -> int:
    return torch.cuda.current_stream(t.device).cuda_stream


def topk_sample(logits: torch.Tensor, noise: torch.Tensor, k: int) -> torch.Tensor:
    """One token per row of fp32 ``logits`` [rows, vocab]: keep the values >=
    the k-th largest (ties included), p = softmax over them, return [rows, 1]
    int64 = the first index of the largest p / ``noise`` (Exponential(1)
    draws, same shape) -- the draw ``torch.multinomial(probs, 1)`` makes after
    the reference's top-k mask (``model.py:141-145``), in one launch
    (``mt_topk_sample``)."""
    if not logits.is_cuda or logits.dtype != torch.float32 or logits.ndim != 2:
        raise RuntimeError("topk_sample takes fp32 [rows, vocab] GPU logits")
    if noise.shape != logits.shape or noise.dtype != torch.float32 or noise.device != logits.device:
        raise ValueError("noise must be fp32 with the logits' shape and device")
    if not 1 <= k <= logits.shape[1] or logits.shape[1] > MAX_SAMPLE_VOCAB:
        raise ValueError(f"need 1 <= k <= vocab <= {MAX_SAMPLE_VOCAB} (k={k}, vocab={logits.shape[1]})")
    _native.ensure()
    return _topk_sample(logits, noise, k)


# ---------------------------------------------------------------------------
# the ops: schemas and shapes here, GPU kernels and autograd in libmt_torch.so
# ---------------------------------------------------------------------------
_LIB = torch.library.Library("mega_trading_amd", "FRAGMENT")
_LIB.define("rms_norm_fwd(Tensor x, Tensor weight, float eps) -> (Tensor, Tensor)")  # (y, rstd fp32 [rows])
# (dx with x's shape and dtype, dweight with weight's dtype)
_LIB.define("rms_norm_bwd(Tensor x, Tensor weight, Tensor rstd, Tensor dy) -> (Tensor, Tensor)")
_LIB.define("add_rms_norm_fwd(Tensor x, Tensor residual, Tensor weight, float eps) -> (Tensor, Tensor, Tensor)")
_LIB.define("add_rms_norm_bwd(Tensor new_residual, Tensor weight, Tensor rstd, Tensor d_new_residual, Tensor dy) "
            "-> (Tensor, Tensor)")
# x fp32 -> (y in the 16-bit dtype of code act, rstd)
_LIB.define("rms_norm_fwd_mixed(Tensor x, Tensor weight, float eps, int act) -> (Tensor, Tensor)")
# x 16-bit, residual fp32 -> (new_residual fp32, y in x's dtype, rstd)
_LIB.define("add_rms_norm_fwd_mixed(Tensor x, Tensor residual, Tensor weight, float eps) -> (Tensor, Tensor, Tensor)")
# (ds fp32 [+ d_new_residual], ds rounded to act when want16 else empty, dweight fp32) for s fp32 and dy 16-bit
_LIB.define("rms_norm_bwd_mixed(Tensor s, Tensor weight, Tensor rstd, Tensor? d_new_residual, Tensor dy, int act, "
            "bool want16) -> (Tensor, Tensor, Tensor)")
_LIB.define("swiglu_fwd(Tensor gate, Tensor up) -> Tensor")
_LIB.define("swiglu_bwd(Tensor gate, Tensor up, Tensor dout) -> (Tensor, Tensor)")
_LIB.define("swiglu_packed_fwd(Tensor gate_up) -> Tensor")
_LIB.define("swiglu_packed_bwd(Tensor gate_up, Tensor dout) -> Tensor")
# query and key in one launch, outputs in the inputs' layout; inverse rotates by -theta (the backward)
_LIB.define("rope_fwd(Tensor query, Tensor key, Tensor cos, Tensor sin, bool inverse) -> (Tensor, Tensor)")
_LIB.define("topk_sample(Tensor logits, Tensor noise, SymInt k) -> Tensor")


def _like(x, dtype=None):
    return torch.empty_like(x, dtype=dtype, memory_format=torch.contiguous_format)


def _rstd_like(x):
    return x.new_empty((x.numel() // max(x.shape[-1], 1),), dtype=torch.float32)


@torch.library.register_fake("mega_trading_amd::rms_norm_fwd")
def _rms_norm_fwd_fake(x, weight, eps):
    return _like(x), _rstd_like(x)


@torch.library.register_fake("mega_trading_amd::rms_norm_bwd")
def _rms_norm_bwd_fake(x, weight, rstd, dy):
    return _like(x), torch.empty_like(weight)


@torch.library.register_fake("mega_trading_amd::add_rms_norm_fwd")
def _add_rms_norm_fwd_fake(x, residual, weight, eps):
    return _like(x), _like(x), _rstd_like(x)


@torch.library.register_fake("mega_trading_amd::add_rms_norm_bwd")
def _add_rms_norm_bwd_fake(new_residual, weight, rstd, d_new_residual, dy):
    return _like(new_residual), torch.empty_like(weight)


@torch.library.register_fake("mega_trading_amd::rms_norm_fwd_mixed")
def _rms_norm_fwd_mixed_fake(x, weight, eps, act):
    return _like(x, _DTYPE_OF[act]), _rstd_like(x)


@torch.library.register_fake("mega_trading_amd::add_rms_norm_fwd_mixed")
def _add_rms_norm_fwd_mixed_fake(x, residual, weight, eps):
    return _like(x, torch.float32), _like(x), _rstd_like(x)


@torch.library.register_fake("mega_trading_amd::rms_norm_bwd_mixed")
def _rms_norm_bwd_mixed_fake(s, weight, rstd, d_new_residual, dy, act, want16):
    return (_like(s, torch.float32), _like(s, _DTYPE_OF[act]) if want16 else s.new_empty((0,), dtype=_DTYPE_OF[act]),
            torch.empty_like(weight))


@torch.library.register_fake("mega_trading_amd::swiglu_fwd")
def _swiglu_fwd_fake(gate, up):
    return _like(gate)


@torch.library.register_fake("mega_trading_amd::swiglu_bwd")
def _swiglu_bwd_fake(gate, up, dout):
    return _like(gate), _like(gate)


@torch.library.register_fake("mega_trading_amd::swiglu_packed_fwd")
def _swiglu_packed_fwd_fake(gate_up):
    return gate_up.new_empty((*gate_up.shape[:-1], gate_up.shape[-1] // 2))


@torch.library.register_fake("mega_trading_amd::swiglu_packed_bwd")
def _swiglu_packed_bwd_fake(gate_up, dout):
    return _like(gate_up)


@torch.library.register_fake("mega_trading_amd::rope_fwd")
def _rope_fwd_fake(query, key, cos, sin, inverse):
    return torch.empty_like(query), torch.empty_like(key)


@torch.library.register_fake("mega_trading_amd::topk_sample")
def _topk_sample_fake(logits, noise, k):
    return logits.new_empty((logits.shape[0], 1), dtype=torch.int64)


# Logits bytes per chunk.  Measured at the C5 shape (32768 x 16384 bf16 logits,
# fwd + bwd): 64 MB chunks (cache-resident) 3.8 ms, 256 MB 2.7 ms, one 1 GB
# chunk 2.3 ms (the three GEMMs alone take 1.6 ms), against 4.4 ms for the eager
# F.linear + F.cross_entropy: on MI355X full-size GEMMs beat cache-resident
# chunks, and 288 GB of HBM leaves room for the whole logits tensor, so chunking
# only bounds memory for batches beyond 2 GB of logits.
_CE_CHUNK_BYTES = 2 << 30
_CE_SCALAR_ROWS = 1 << 17  # rows of one ce_count / ce_sum launch

# (loss fp32 scalar, d loss / d hidden, d loss / d weight); the gradients are empty tensors when need_grad is False
_LIB.define("fused_linear_ce(Tensor hidden, Tensor weight, Tensor labels, int ignore_index, int compute_dtype, "
            "bool need_grad) -> (Tensor, Tensor, Tensor)")
_LIB.define("ce_count(Tensor labels, int ignore_index) -> Tensor")
_LIB.define("ce_sum(Tensor loss_rows) -> Tensor")
_LIB.define("scale_pair(Tensor a, Tensor b, Tensor scale) -> (Tensor, Tensor)")


@torch.library.impl(_LIB, "fused_linear_ce", "CUDA")
def _fused_linear_ce_gpu(hidden, weight, labels, ignore_index, compute_dtype, need_grad):
    lib = _native.load()
    ct = _DTYPE_OF[compute_dtype]
    rows, h = hidden.shape
    vocab = weight.shape[0]
    # a vocab that is not a multiple of 8 (the reference tokenizer's always is
    # odd) gets zero weight rows up to the next multiple: the logits rows then
    # have a padded stride, and the row kernel ignores the pad columns and
    # writes them a zero gradient, so the pad rows contribute nothing
    vpad = (vocab + 7) // 8 * 8
    hc = hidden.to(ct).contiguous()
    if vpad == vocab:
        wc = weight.to(ct).contiguous()
    else:
        wc = torch.empty((vpad, h), device=weight.device, dtype=ct)
        wc[:vocab].copy_(weight)
        wc[vocab:].zero_()
    lab = labels.to(torch.int64).contiguous()
    scalars = 0 < rows <= _CE_SCALAR_ROWS
    # stays on the device: the kernel reads it
    n_valid = _ce_count(lab, ignore_index) if scalars else (lab != ignore_index).sum()
    loss_rows = torch.empty((rows,), device=hidden.device, dtype=torch.float32)
    chunk = max(1, min(rows, _CE_CHUNK_BYTES // (vpad * ct.itemsize)))
    gw = None
    if need_grad:
        gh = torch.empty((rows, h), device=hidden.device, dtype=ct)
        if chunk < rows or not rows:  # several chunks' products are summed in fp32
            gw = torch.zeros((vpad, h), device=hidden.device, dtype=torch.float32)
    with torch.cuda.device(hidden.device), tuned_gemms():
        stream = _stream(hidden)
        for start in range(0, rows, chunk):
            end = min(rows, start + chunk)
            logits = torch.mm(hc[start:end], wc.t())  # [chunk, vocab] in ct, fp32 accumulation
            rc = lib.mt_cross_entropy_rows(logits.data_ptr(), logits.stride(0), lab[start:end].data_ptr(), end - start,
                                           vocab, n_valid.data_ptr(), ignore_index, loss_rows[start:end].data_ptr(),
                                           1 if need_grad else 0, compute_dtype, stream)
            _native.check(rc, "mt_cross_entropy_rows")
            if need_grad:  # logits now hold d loss / d logits
                torch.mm(logits, wc, out=gh[start:end])
                part = torch.mm(logits.t(), hc[start:end])
                gw = part if gw is None else gw.add_(part)
    loss = _ce_sum(loss_rows) if scalars else loss_rows.sum()
    if not need_grad:
        return loss, hidden.new_empty((0,)), weight.new_empty((0,))
    return loss, gh.to(hidden.dtype), gw[:vocab].to(weight.dtype)


@torch.library.register_fake("mega_trading_amd::fused_linear_ce")
def _fused_linear_ce_fake(hidden, weight, labels, ignore_index, compute_dtype, need_grad):
    loss = hidden.new_empty((), dtype=torch.float32)
    if not need_grad:
        return loss, hidden.new_empty((0,)), weight.new_empty((0,))
    return loss, torch.empty_like(hidden), torch.empty_like(weight)


@torch.library.register_fake("mega_trading_amd::scale_pair")
def _scale_pair_fake(a, b, scale):
    return _like(a), _like(b)


# the ops as the functions above call them
_OPS = torch.ops.mega_trading_amd
_rms_norm_fwd = _OPS.rms_norm_fwd.default
_add_rms_norm_fwd = _OPS.add_rms_norm_fwd.default
_rms_norm_fwd_mixed = _OPS.rms_norm_fwd_mixed.default
_add_rms_norm_fwd_mixed = _OPS.add_rms_norm_fwd_mixed.default
_swiglu_fwd = _OPS.swiglu_fwd.default
_swiglu_packed_fwd = _OPS.swiglu_packed_fwd.default
_rope_fwd = _OPS.rope_fwd.default
_topk_sample = _OPS.topk_sample.default
_fused_linear_ce = _OPS.fused_linear_ce.default
_ce_count = _OPS.ce_count.default
_ce_sum = _OPS.ce_sum.default
