"""EPTQ HIP kernels as ``torch.library`` custom ops.

Drop-in for the reference's ``kernels/__init__.py:50-91``: the ops
``eptq::e8_forward`` and ``eptq::e8d4_forward`` keep their names, argument
order and meaning ``(Q, codebook, g, h, x, O_vals, O_col, O_row_ptr, bias)``
(an empty ``bias`` means no bias) and have fake implementations for
``torch.compile``.  They run the gfx950 kernels of ``libeptq_hip.so`` through
its C ABI on the current HIP stream; there is no CPU or PyTorch fallback.

Additions over the reference: fp32 tables are accepted (the kernels convert),
bf16 activations give bf16 outputs, ``*_grouped`` variants take ``S_group``
(the reference materializes an fp16 W instead, ``kernels/linear.py:97-120``),
``eptq::e8d4_dequant`` / ``eptq::e8_dequant`` produce the bit-exact fp16 W of
``dequantize_layer`` (``algorithms/eptq.py:406-471``) on the GPU, and
``eptq::e8d4_forward_multi`` runs several E8-D4 layers that share x (q|k|v,
gate|up) in one launch with a split-K workspace.  ``EPTQLinear.forward`` and
``EPTQMultiLinear.forward`` call only these registered ops, so, as in the
reference (``kernels/__init__.py:44-47``), ``torch.compile(fullgraph=True)``
sees each quantized Linear as one op with no graph break.
"""

from __future__ import annotations


import contextlib
import threading
from typing import List, Optional

import torch

from . import _lib
from ._lib import EPTQ_BF16, EPTQ_F16, EPTQ_F32, EptqError

__all__ = ["e8_forward", "e8d4_forward", "e8_forward_grouped", "e8d4_forward_grouped",
           "e8d4_forward_multi", "e8_dequant", "e8d4_dequant", "EptqError", "linear_forward",
           "linear_forward_multi", "dequant", "decode_workspace", "stream_workspace"]


def _ptr(t: Optional[torch.Tensor]):
    if t is None or t.numel() == 0:
        return None
    return t.data_ptr()


def _require(cond: bool, msg: str) -> None:
    if not cond:
        raise RuntimeError(msg)


def _raw_stream(device: torch.device) -> int:
    """The current stream of ``device`` as a raw hipStream_t (what
    ``torch.cuda.current_stream(device).cuda_stream`` is, without the Stream
    object: 0.3 against 2.8 us)."""
    return torch._C._cuda_getCurrentRawStream(device.index)


_NO_SWITCH = contextlib.nullcontext()


def _on(device: torch.device):
    """A context with ``device`` current (the library launches on the current
    device); entered without a switch where it already is."""
    return _NO_SWITCH if device.index == torch.cuda.current_device() else torch.cuda.device(device)


def _bad_operand(name: str, t, dev, dt) -> None:
    _require(t.device == dev, f"{name} must be on {dev}")
    _require(t.dtype == dt, f"{name} must be {dt}, got {t.dtype}")
    _require(t.is_contiguous(), f"{name} must be contiguous")


def _check_layer(kind, Q, codes, g, h, O_vals, O_col, O_row_ptr, S_group):
    # Run on every call: messages are formed only on failure.
    if not Q.is_cuda:
        raise RuntimeError("Q must be a CUDA (HIP) tensor")
    dev = Q.device
    if Q.dtype != torch.int16 or Q.dim() != 2 or not Q.is_contiguous():
        raise RuntimeError("Q must be a contiguous 2-D int16 tensor")
    M, N = Q.shape
    f16, i32 = torch.float16, torch.int32
    if g.device != dev or g.dtype != f16 or not g.is_contiguous():
        _bad_operand("g", g, dev, f16)
    if h.device != dev or h.dtype != f16 or not h.is_contiguous():
        _bad_operand("h", h, dev, f16)
    if O_vals.device != dev or O_vals.dtype != f16 or not O_vals.is_contiguous():
        _bad_operand("O_vals", O_vals, dev, f16)
    if O_col.device != dev or O_col.dtype != i32 or not O_col.is_contiguous():
        _bad_operand("O_col", O_col, dev, i32)
    if O_row_ptr.device != dev or O_row_ptr.dtype != i32 or not O_row_ptr.is_contiguous():
        _bad_operand("O_row_ptr", O_row_ptr, dev, i32)
    if g.numel() != 8 * M:
        raise RuntimeError(f"g must have {8 * M} elements")
    if h.numel() != N:
        raise RuntimeError(f"h must have {N} elements")
    if O_row_ptr.numel() != M + 1:
        raise RuntimeError(f"O_row_ptr must have {M + 1} elements")
    if O_vals.numel() != 8 * O_col.numel():
        raise RuntimeError("O_vals must be (nnz, 8) with nnz = len(O_col)")
    if codes.device != dev or not codes.is_contiguous():
        raise RuntimeError("codebook must be contiguous on the layer's device")
    if codes.dtype != f16 and codes.dtype != torch.float32:
        raise RuntimeError("codebook must be fp16 or fp32")
    if codes.numel() != (2048 if kind == "e8_d4" else 524280):
        raise RuntimeError(f"{kind} codebook must have {512 if kind == 'e8_d4' else 65535} rows")
    n_groups = 0
    if S_group is not None:
        if S_group.device != dev or S_group.dtype != f16 or not S_group.is_contiguous():
            raise RuntimeError("S_group must be a contiguous fp16 tensor on the layer's device")
        if S_group.dim() != 2 or S_group.shape[1] != N:
            raise RuntimeError("S_group must be (n_groups, in_features)")
        n_groups = S_group.shape[0]
    return M, N, n_groups


def linear_forward(kind: str, Q, codes, g, h, x, O_vals, O_col, O_row_ptr, bias=None,
                   S_group=None, two_pass: bool = False) -> torch.Tensor:
    """Run the fused quantized Linear on ``x`` (B, N) -> (B, 8M), dtype of x.
    ``two_pass`` (what the module's ops pass): the two-pass prefill instead of
    the fused C-ABI kernel where it is preferred (``_two_pass_into``)."""
    M, N, n_groups = _check_layer(kind, Q, codes, g, h, O_vals, O_col, O_row_ptr, S_group)
    dev, xdt = Q.device, x.dtype
    if x.device != dev:
        raise RuntimeError("x must be on the layer's device")
    if x.dim() != 2 or x.shape[1] != N:
        raise RuntimeError(f"x must be (B, {N})")
    if xdt != torch.float16 and xdt != torch.bfloat16:
        raise RuntimeError("x must be fp16 or bf16")
    if not x.is_contiguous():
        raise RuntimeError("x must be contiguous")
    if bias is not None and bias.numel() > 0:
        _require(bias.device == dev and bias.dtype == torch.float16 and bias.numel() == 8 * M
                 and bias.is_contiguous(), "bias must be a contiguous fp16 (out_features,) tensor")
    B = x.shape[0]
    y = torch.empty((B, 8 * M), dtype=xdt, device=dev)
    if B == 0:
        return y
    lib = _lib.load()
    if two_pass and B >= (TWO_PASS_MIN_TOKENS if kind == "e8_d4" else TWO_PASS_MIN_TOKENS_E8):
        arr = (_lib.EptqLayer * 1)(_layer_entry(Q, g, h, O_vals, O_col, O_row_ptr, bias, S_group, M, n_groups, 0))
        if _two_pass_into(lib, arr, codes, x, y, kind, stream_workspace(dev)):
            return y
    fn = lib.eptq_e8d4_forward if kind == "e8_d4" else lib.eptq_e8_forward
    with _on(dev):
        rc = fn(_ptr(Q), _ptr(codes), EPTQ_F32 if codes.dtype == torch.float32 else EPTQ_F16,
                _ptr(g), _ptr(h), x.data_ptr(), EPTQ_BF16 if xdt == torch.bfloat16 else EPTQ_F16,
                _ptr(O_vals), _ptr(O_col), _ptr(O_row_ptr), _ptr(bias), _ptr(S_group), n_groups,
                M, N, B, y.data_ptr(), _raw_stream(dev))
    _lib.check(rc, fn.__name__)
    return y


def decode_workspace(device) -> torch.Tensor:
    """A zero-filled workspace for ``linear_forward_multi(..., work=)`` on
    ``device`` (``eptq_e8d4_work_bytes`` bytes)."""
    with torch.cuda.device(device):
        n = int(_lib.load().eptq_e8d4_work_bytes())
    return torch.zeros(n, dtype=torch.uint8, device=device)


# One split-K workspace per (device, stream): launches on one stream run one
# after another, so modules that share their stream's workspace never overlap
# on it.  Created on first eager use, zero-filled before that stream uses it.
_STREAM_WORK: dict = {}


def stream_workspace(device) -> Optional[torch.Tensor]:
    """The decode workspace of the current stream on ``device`` (see
    ``decode_workspace``), created on first eager use.

    While the current stream is capturing a graph this returns None (the
    unsplit kernel, same results): a workspace made during a capture would
    come from that graph's private pool with its zero fill recorded, not run,
    and graphs captured on one stream may later replay concurrently on
    different streams.  A caller that wants split-K inside a captured graph
    attaches its own workspace (``EPTQLinear._work = decode_workspace(dev)``),
    which that graph's replays then must not share with concurrent work."""
    device = torch.device(device)
    if torch.cuda.is_current_stream_capturing():
        return None
    index = device.index if device.index is not None else torch.cuda.current_device()
    key = (index, torch._C._cuda_getCurrentRawStream(index))
    w = _STREAM_WORK.get(key)
    if w is None:
        w = _workspace_outside_graph_pools(device, torch.cuda.current_stream(device))
        _STREAM_WORK[key] = w
    return w


def _workspace_outside_graph_pools(device, stream) -> torch.Tensor:
    """``decode_workspace`` allocated and zero-filled by a helper thread on a
    stream of its own, then ordered before ``stream``.  The calling thread
    may be routing its allocations into a graph's private memory pool
    (torch.compile's cudagraph warm-up runs do, per thread), where a buffer
    kept alive across calls does not belong."""
    box = {}

    def run():
        try:
            with torch.cuda.device(device):
                side = torch.cuda.Stream(device)
                side.wait_stream(stream)
                with torch.cuda.stream(side):
                    box["w"] = decode_workspace(device)
                    box["ev"] = side.record_event()
        except BaseException as e:  # re-raised in the caller
            box["err"] = e

    t = threading.Thread(target=run, name="eptq-workspace")
    t.start()
    t.join()
    if "err" in box:
        raise box["err"]
    stream.wait_event(box["ev"])
    return box["w"]


# The least token counts at which the module's forwards may run the two-pass
# prefill (every weight decoded once into a transient fp16 W, then the
# W-streaming GEMM); ``eptq_two_pass_scratch_bytes`` decides.  E8 layers, whose
# fused GEMM gathers from a 1 MB table: 2.1x at 17 rows on 4096x4096, 1.5x on
# 11008x4096, 2.6x on 4096x11008.  E8-D4 with S_group or bf16 x: a Llama-2-7B
# layer at 130 rows 984 -> 278 us (bf16), 3022 -> 279 us (bf16 with S_group).
# E8-D4 otherwise: by estimated times, between 129 and 2048 rows either may win.
TWO_PASS_MIN_TOKENS_E8 = 17
TWO_PASS_MIN_TOKENS = 129


def _two_pass_into(lib, arr, codes, x, y, kind: str, work: Optional[torch.Tensor], always: bool = False) -> bool:
    """y[:, layer columns] = x · W_lᵀ + bias_l with each layer's W decoded once
    (S_group included) into a transient buffer and multiplied by the W-streaming
    GEMM (``eptq_two_pass_forward``; ``arr``: the layers as an ``EptqLayer``
    array), where that is preferred or ``always`` is set; False where not.  The
    table is the kernels' (fp16): the same table values the fused kernel
    multiplies."""
    B, N, n = x.shape[0], x.shape[1], len(arr)
    if B < (TWO_PASS_MIN_TOKENS if kind == "e8_d4" else TWO_PASS_MIN_TOKENS_E8) and not always:
        return False
    e8, xdt = int(kind != "e8_d4"), EPTQ_BF16 if x.dtype == torch.bfloat16 else EPTQ_F16
    with _on(x.device):
        nbytes = lib.eptq_two_pass_scratch_bytes(e8, n, arr, N, B, xdt, int(work is not None), int(always))
        if nbytes == 0:
            return False
        if codes.data_ptr() % 16:
            codes = codes.clone()
        scratch = torch.empty(nbytes, dtype=torch.uint8, device=x.device)
        rc = lib.eptq_two_pass_forward(
            e8, n, arr, codes.data_ptr(), EPTQ_F32 if codes.dtype == torch.float32 else EPTQ_F16, x.data_ptr(), xdt, N,
            B, y.data_ptr(), y.shape[1], scratch.data_ptr(), nbytes, _ptr(work), 0 if work is None else work.numel(),
            _raw_stream(x.device))
    _lib.check(rc, "eptq_two_pass_forward")
    return True


def _layer_entry(Q, g, h, O_vals, O_col, O_row_ptr, bias, S_group, M: int, n_groups: int, off: int):
    return _lib.EptqLayer(_ptr(Q), _ptr(g), _ptr(h), _ptr(O_vals), _ptr(O_col), _ptr(O_row_ptr), _ptr(bias),
                          _ptr(S_group), n_groups, M, off)


def linear_forward_multi(layers, codes, x, work: Optional[torch.Tensor] = None,
                         two_pass: bool = False) -> torch.Tensor:
    """E8-D4 layers sharing ``x`` (B, N) -> (B, Σ out) with the layers' outputs
    side by side, in one decode launch when the kernel takes them all.
    ``layers``: dicts with Q, g, h, O_vals, O_col, O_row_ptr and optional
    bias, S_group (the EPTQLinear buffers).  ``two_pass`` (what the
    module's op passes): the two-pass prefill (``_two_pass_into``) instead of
    the fused C-ABI launch where it is preferred.  ``work``: optional workspace from
    ``decode_workspace`` (lets batches of 3..16 split the columns of layers
    with few row tiles over several workgroups); calls sharing one must not
    overlap in time."""
    return _forward_multi([(L["Q"], L["g"], L["h"], L["O_vals"], L["O_col"], L["O_row_ptr"], L.get("bias"),
                            L.get("S_group")) for L in layers], codes, x, work, two_pass)


def _forward_multi(layers, codes, x, work, two_pass) -> torch.Tensor:
    """``linear_forward_multi`` on tuples (Q, g, h, O_vals, O_col, O_row_ptr, bias, S_group)."""
    if len(layers) == 0:
        raise RuntimeError("no layers")
    xdt = x.dtype
    if x.dim() != 2 or (xdt != torch.float16 and xdt != torch.bfloat16) or not x.is_contiguous():
        raise RuntimeError("x must be a contiguous 2-D fp16/bf16 tensor")
    B, N = x.shape
    dev = x.device
    arr = (_lib.EptqLayer * len(layers))()
    off = 0
    for i, (Q, g, h, O_vals, O_col, O_row_ptr, bias, S_group) in enumerate(layers):
        M, n2, n_groups = _check_layer("e8_d4", Q, codes, g, h, O_vals, O_col, O_row_ptr, S_group)
        if n2 != N or Q.device != dev:
            raise RuntimeError("layers must take x's in_features on x's device")
        arr[i] = _layer_entry(Q, g, h, O_vals, O_col, O_row_ptr, bias, S_group, M, n_groups, off)
        off += 8 * M
    y = torch.empty((B, off), dtype=xdt, device=dev)
    if B == 0:
        return y
    lib = _lib.load()
    if two_pass and B >= TWO_PASS_MIN_TOKENS and _two_pass_into(lib, arr, codes, x, y, "e8_d4", work):
        return y
    with _on(dev):
        rc = lib.eptq_e8d4_forward_multi(len(layers), arr, codes.data_ptr(),
                                         EPTQ_F32 if codes.dtype == torch.float32 else EPTQ_F16, x.data_ptr(),
                                         EPTQ_BF16 if xdt == torch.bfloat16 else EPTQ_F16, N, B, y.data_ptr(), off,
                                         _ptr(work), 0 if work is None else work.numel(), _raw_stream(dev))
    _lib.check(rc, "eptq_e8d4_forward_multi")
    return y


def dequant(kind: str, Q, codes, g, h, O_vals, O_col, O_row_ptr, S_group=None,
            out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Bit-exact fp16 W (8M, N) on the GPU; ``codes`` must be the fp32 table.
    ``out``: a contiguous fp16 (8M, N) tensor on Q's device to write W into."""
    M, N, n_groups = _check_layer(kind, Q, codes, g, h, O_vals, O_col, O_row_ptr, S_group)
    _require(codes.dtype == torch.float32, "dequant needs the fp32 table for bit-exact W")
    if out is None:
        W = torch.empty((8 * M, N), dtype=torch.float16, device=Q.device)
    else:
        _require(out.dtype == torch.float16 and tuple(out.shape) == (8 * M, N) and out.is_contiguous()
                 and out.device == Q.device, "out must be a contiguous fp16 (8M, N) tensor on Q's device")
        W = out
    lib = _lib.load()
    fn = lib.eptq_e8d4_dequant if kind == "e8_d4" else lib.eptq_e8_dequant
    with _on(Q.device):
        rc = fn(_ptr(Q), _ptr(codes), _ptr(g), _ptr(h), _ptr(O_vals), _ptr(O_col),
                _ptr(O_row_ptr), _ptr(S_group), n_groups, M, N, _ptr(W), _raw_stream(Q.device))
    _lib.check(rc, fn.__name__)
    return W


def f16_gemm(W: torch.Tensor, x: torch.Tensor, bias: Optional[torch.Tensor] = None) -> torch.Tensor:
    """y (T, F) = x (T, N) · Wᵀ + bias for fp16 W (F, N): the second pass of
    the two-pass prefill (``eptq_f16_gemm``).  Raises EptqError (code 2)
    where the kernel does not take the shape (F, N multiples of 64)."""
    _require(W.dtype == torch.float16 and x.dtype == torch.float16 and W.is_contiguous() and x.is_contiguous()
             and W.dim() == 2 and x.dim() == 2 and W.shape[1] == x.shape[1] and W.device == x.device,
             "W (F, N) and x (T, N) must be contiguous fp16 on one device")
    _require(bias is None or (bias.dtype == torch.float16 and bias.is_contiguous() and bias.numel() == W.shape[0]),
             "bias must be a contiguous fp16 (F,) tensor")
    F, N = int(W.shape[0]), int(W.shape[1])
    T = int(x.shape[0])
    y = torch.empty((T, F), dtype=torch.float16, device=x.device)
    with _on(x.device):
        rc = _lib.load().eptq_f16_gemm(_ptr(W), _ptr(x), _ptr(bias), F, N, T, _ptr(y), F, _raw_stream(x.device))
    _lib.check(rc, "eptq_f16_gemm")
    return y


# ---------------------------------------------------------------------------
# torch.library registration (names and signatures of kernels/__init__.py:50-91)
# ---------------------------------------------------------------------------

@torch.library.custom_op("eptq::e8_forward", mutates_args=())
def e8_forward(Q: torch.Tensor, codebook: torch.Tensor, g: torch.Tensor, h: torch.Tensor,
               x: torch.Tensor, O_vals: torch.Tensor, O_col: torch.Tensor,
               O_row_ptr: torch.Tensor, bias: torch.Tensor) -> torch.Tensor:
    return linear_forward("e8_lattice", Q, codebook, g, h, x, O_vals, O_col, O_row_ptr, bias, two_pass=True)


@e8_forward.register_fake
def _e8_forward_fake(Q, codebook, g, h, x, O_vals, O_col, O_row_ptr, bias):
    return x.new_empty(x.shape[0], Q.shape[0] * 8)


@torch.library.custom_op("eptq::e8d4_forward", mutates_args=())
def e8d4_forward(Q: torch.Tensor, codes: torch.Tensor, g: torch.Tensor, h: torch.Tensor,
                 x: torch.Tensor, O_vals: torch.Tensor, O_col: torch.Tensor,
                 O_row_ptr: torch.Tensor, bias: torch.Tensor) -> torch.Tensor:
    return linear_forward("e8_d4", Q, codes, g, h, x, O_vals, O_col, O_row_ptr, bias, two_pass=True)


@e8d4_forward.register_fake
def _e8d4_forward_fake(Q, codes, g, h, x, O_vals, O_col, O_row_ptr, bias):
    return x.new_empty(x.shape[0], Q.shape[0] * 8)


@torch.library.custom_op("eptq::e8_forward_grouped", mutates_args=())
def e8_forward_grouped(Q: torch.Tensor, codebook: torch.Tensor, g: torch.Tensor, h: torch.Tensor,
                       x: torch.Tensor, O_vals: torch.Tensor, O_col: torch.Tensor,
                       O_row_ptr: torch.Tensor, bias: torch.Tensor,
                       S_group: torch.Tensor) -> torch.Tensor:
    return linear_forward("e8_lattice", Q, codebook, g, h, x, O_vals, O_col, O_row_ptr, bias, S_group,
                          two_pass=True)


@e8_forward_grouped.register_fake
def _e8_forward_grouped_fake(Q, codebook, g, h, x, O_vals, O_col, O_row_ptr, bias, S_group):
    return x.new_empty(x.shape[0], Q.shape[0] * 8)


@torch.library.custom_op("eptq::e8d4_forward_grouped", mutates_args=())
def e8d4_forward_grouped(Q: torch.Tensor, codes: torch.Tensor, g: torch.Tensor, h: torch.Tensor,
                         x: torch.Tensor, O_vals: torch.Tensor, O_col: torch.Tensor,
                         O_row_ptr: torch.Tensor, bias: torch.Tensor,
                         S_group: torch.Tensor) -> torch.Tensor:
    return linear_forward("e8_d4", Q, codes, g, h, x, O_vals, O_col, O_row_ptr, bias, S_group, two_pass=True)


@e8d4_forward_grouped.register_fake
def _e8d4_forward_grouped_fake(Q, codes, g, h, x, O_vals, O_col, O_row_ptr, bias, S_group):
    return x.new_empty(x.shape[0], Q.shape[0] * 8)


@torch.library.custom_op("eptq::e8d4_dequant", mutates_args=())
def e8d4_dequant(Q: torch.Tensor, codes: torch.Tensor, g: torch.Tensor, h: torch.Tensor,
                 O_vals: torch.Tensor, O_col: torch.Tensor, O_row_ptr: torch.Tensor,
                 S_group: Optional[torch.Tensor] = None) -> torch.Tensor:
    return dequant("e8_d4", Q, codes, g, h, O_vals, O_col, O_row_ptr, S_group)


@e8d4_dequant.register_fake
def _e8d4_dequant_fake(Q, codes, g, h, O_vals, O_col, O_row_ptr, S_group=None):
    return Q.new_empty(Q.shape[0] * 8, Q.shape[1], dtype=torch.float16)


@torch.library.custom_op("eptq::e8_dequant", mutates_args=())
def e8_dequant(Q: torch.Tensor, codes: torch.Tensor, g: torch.Tensor, h: torch.Tensor,
               O_vals: torch.Tensor, O_col: torch.Tensor, O_row_ptr: torch.Tensor,
               S_group: Optional[torch.Tensor] = None) -> torch.Tensor:
    return dequant("e8_lattice", Q, codes, g, h, O_vals, O_col, O_row_ptr, S_group)


@e8_dequant.register_fake
def _e8_dequant_fake(Q, codes, g, h, O_vals, O_col, O_row_ptr, S_group=None):
    return Q.new_empty(Q.shape[0] * 8, Q.shape[1], dtype=torch.float16)


@torch.library.custom_op("eptq::e8d4_forward_multi", mutates_args=("work",))
def e8d4_forward_multi(Q: List[torch.Tensor], codes: torch.Tensor, g: List[torch.Tensor],
                       h: List[torch.Tensor], x: torch.Tensor, O_vals: List[torch.Tensor],
                       O_col: List[torch.Tensor], O_row_ptr: List[torch.Tensor],
                       bias: List[Optional[torch.Tensor]], S_group: List[Optional[torch.Tensor]],
                       work: Optional[torch.Tensor]) -> torch.Tensor:
    """E8-D4 layers sharing ``x`` (B, N) -> (B, Σ 8·M_l), outputs side by side
    (``linear_forward_multi``); the op ``EPTQLinear`` / ``EPTQMultiLinear``
    call for E8-D4 layers.  No counterpart in the reference, whose module
    calls ``eptq::e8d4_forward`` per projection (``kernels/linear.py:177-208``).

    ``work`` (required, may be None; a mutated argument with a default
    trips torch's in-place bookkeeping): a ``decode_workspace`` tensor
    (declared mutated: the split-K parts write their partial sums there; the
    counters return to zero), or None for the current stream's own (``stream_workspace``), which the op
    looks up when it runs, like a BLAS library's internal workspace."""
    if work is None and x.is_cuda:
        work = stream_workspace(x.device)
    n = len(Q)
    if any(len(t) < n for t in (g, h, O_vals, O_col, O_row_ptr, bias, S_group)):
        raise IndexError("list index out of range")
    return _forward_multi(list(zip(Q, g, h, O_vals, O_col, O_row_ptr, bias, S_group)), codes, x, work, True)


@e8d4_forward_multi.register_fake
def _e8d4_forward_multi_fake(Q, codes, g, h, x, O_vals, O_col, O_row_ptr, bias, S_group, work):
    n = len(Q)
    torch._check(n > 0 and all(len(t) == n for t in (g, h, O_vals, O_col, O_row_ptr, bias, S_group)),
                 lambda: "every per-layer list must have one entry per layer")
    return x.new_empty(x.shape[0], sum(q.shape[0] * 8 for q in Q))
