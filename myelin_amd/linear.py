"""Autograd boundary of the streamed-synapse LIF path (``x_t @ W`` fused ahead
of the neuron update).

Forward: one launch of ``myelin_linear_lif_fwd`` computes every step's
current tile on MFMA and runs the recurrence in the same workgroup (layers
narrower than 64 neurons use a split-K GEMM plus the recurrence kernel, see
``_lif_fwd``).

Saved state:
* ``checkpoint_size=None`` (the reference's stream Function,
  autograd.py:445-558): the pre-reset membranes ``[T, B, N]`` -- one tensor
  where the reference keeps pre-reset membranes and spikes;
* ``checkpoint_size=C`` (autograd.py:588-717) and the rate readout
  (autograd.py:753-885): chunk-start membranes every C steps only, except
  for layers of at most 32 neurons (readouts), which keep the whole trace
  as the stream path does (a few MB; their backward then recomputes
  nothing).

Backward, per span of whole chunks in reverse time: recompute the span's
pre-reset trace from its first chunk-start membrane (skipped when the trace
is saved), reverse recurrence -> G = dL/dI plus per-(b, n) bias partials,
then ``dX[t] = G_t @ W^T`` and ``dW += X_t^T G_t`` on MFMA GEMMs,
``db = sum_b`` of the bias partials.  Every reduction has a fixed order, so
gradients are run-to-run deterministic (the reference's Triton path uses
fp32 atomics, triton/lif.py:1336-1348).
"""

from __future__ import annotations

import contextlib
import math
from typing import Any

import torch

from myelin_amd import _lib


def _workspace(M, N, K, prec, device, split, ws):
    """(split-K workspace, its size in floats): ``ws``, a float32 buffer the
    caller has free on the stream (the kernel then splits K no more ways
    than it holds), else a new one of the size the kernel would use."""

    if not split:
        return None, 0
    if ws is not None:
        return ws, ws.numel()
    n_ws = _lib.load().myelin_gemm_workspace_elems(M, N, K, prec)
    return (torch.empty(n_ws, dtype=torch.float32, device=device) if n_ws > 0 else None), n_ws


def _gemm(A, B, C, M, N, K, lda, ldb, ldc, trans_a, trans_b, accumulate, prec, stream, bias=None, a_bits=False,
          split=True, ws=None, col_sum=None):
    """C (+)= op(A) op(B) (+ bias); A and B both float32 or both bfloat16, or
    (``a_bits``) A packed spike words (int32, lda in words) with B float32.
    ``split=False`` gives no workspace, so K is never split: every element is
    then one k-ordered sum that does not depend on M (the synapse currents,
    which a checkpointed backward recomputes over fewer rows and must
    reproduce bit for bit).  ``ws``: see _workspace.  ``col_sum`` = (src
    [R, Nc], dst [Nc]): also dst = src summed over rows, in the GEMM's
    split-K reduce launch when it has one (myelin_gemm_col_sum)."""

    ws, n_ws = _workspace(M, N, K, prec, C.device, split, ws)
    a_dt = _lib.DT_BITS if a_bits else _lib.DT[A.dtype]
    args = (_lib.ptr(A), a_dt, _lib.ptr(B), _lib.DT[B.dtype], _lib.ptr(bias), _lib.ptr(C), M, N, K, lda, ldb, ldc,
            int(trans_a), int(trans_b), int(accumulate), prec, _lib.ptr(ws), n_ws)
    if col_sum is None:
        _lib.call("myelin_gemm", *args, stream)
    else:
        src, dst = col_sum
        _lib.call("myelin_gemm_col_sum", *args, _lib.ptr(src), _lib.ptr(dst), src.numel() // dst.numel(),
                  dst.numel(), stream)


def _half(prec: int, F: int, N: int) -> bool:
    """bf16 synapse with operand rows the bf16 kernels can load 16 bytes at a
    time: its GEMMs then read bf16 copies of x, W and dL/dI (half the
    bytes, bit-identical results)."""

    return prec == _lib.PREC["bf16"] and F % 8 == 0 and N % 8 == 0


def _cast_bf16(t, stream):
    out = torch.empty(t.shape, dtype=torch.bfloat16, device=t.device)
    _lib.call("myelin_cast_bf16", _lib.ptr(t), _lib.ptr(out), t.numel(), stream)
    return out


def _transpose_bf16(w, stream):
    """[F, N] fp32 -> [N, F] bf16."""

    out = torch.empty((w.shape[1], w.shape[0]), dtype=torch.bfloat16, device=w.device)
    _lib.call("myelin_transpose_bf16", _lib.ptr(w), _lib.ptr(out), w.shape[0], w.shape[1], stream)
    return out


def _cast_transpose_bf16(x, w, stream):
    """(bf16 copy of x, [N, F] bf16 transpose of w [F, N]) in one launch."""

    xb = torch.empty(x.shape, dtype=torch.bfloat16, device=x.device)
    wt = torch.empty((w.shape[1], w.shape[0]), dtype=torch.bfloat16, device=w.device)
    _lib.call("myelin_cast_transpose_bf16", _lib.ptr(x), _lib.ptr(xb), x.numel(), _lib.ptr(w), _lib.ptr(wt),
              w.shape[0], w.shape[1], stream)
    return xb, wt


def _gemm_parts(A, B, parts, b_part, C, M, N, K, lda, ldb, ldc, trans_a, trans_b, accumulate, stream, bias=None,
                split=True, ws=None, col_sum=None):
    """C (+)= sum_p op(A) op(B_p) (+ bias), bf16 operands, B_p = B + p*b_part
    (elements); ``split``, ``ws`` and ``col_sum`` as in _gemm."""

    ws, n_ws = _workspace(M, N, K, _lib.PREC["bf16"], C.device, split, ws)
    args = (_lib.ptr(A), _lib.ptr(B), parts, b_part, _lib.ptr(bias), _lib.ptr(C), M, N, K, lda, ldb, ldc,
            int(trans_a), int(trans_b), int(accumulate), _lib.ptr(ws), n_ws)
    if col_sum is None:
        _lib.call("myelin_gemm_parts", *args, stream)
    else:
        src, dst = col_sum
        _lib.call("myelin_gemm_parts_col_sum", *args, _lib.ptr(src), _lib.ptr(dst), src.numel() // dst.numel(),
                  dst.numel(), stream)


# split of an fp32 synapse: tried for products of at least this many
# multiply-adds (the input check costs one host synchronisation)
_SPLIT_MIN_MACS = 1 << 32


class _LazyBf16:
    """A bf16 view of an fp32 input ``[T, ...]`` that keeps no whole bf16
    copy: indexing it with a slice of steps launches the cast of those steps
    on the current stream and returns a new bf16 tensor.  Used by the
    memory-lean policy (``checkpoint_size="memory"``), whose GEMMs then read
    one checkpoint chunk or span of bf16 input at a time."""

    dtype = torch.bfloat16

    def __init__(self, x: torch.Tensor):
        self.x = x
        self.shape = x.shape
        self.device = x.device
        self._last = (None, None)

    def __getitem__(self, steps: slice) -> torch.Tensor:
        # the last slice is kept: a backward span's recompute and its weight
        # gradient read the same steps, one after the other on one stream
        key = (steps.start, steps.stop, steps.step)
        if self._last[0] != key:
            part = self.x[steps]
            self._last = (key, _cast_bf16(part, _lib.stream(part.device)))
        return self._last[1]


# widest input of the int8 products: two digit sums joined stay in 32 bits
_DIGITS_MAX_F = 508 * 128
# narrowest where the fused kernel could run, which keeps the currents in LDS
# where the split writes and reads them.  N=4096, T=100, B=256, us fused and
# split: forward with dense spikes F=128 422 and 525, 192 551 and 562, 256 664
# and 556, its training step 914 and 1005, 1252 and 1086, 1358 and 1096;
# packed output F=96 332 and 333, 128 387 and 333, 192 500 and 361
_DIGITS_MIN_F_FUSED = 192
_DIGITS_MIN_F_PACKED = 128
# least multiply-adds of a layer whose input wants its gradient, where the
# planes are the other choice: the host's way from the flags to the backward's
# launches, 75 to 110 us, then runs beside the currents' products, and the
# planes' cover more of it.  Training step, digits and planes, us: 6400 x 1000 x
# 704 345 and 295-330, 8192 x 1024 x 1024 400 and 361-384, 16384 x 1024 x 1024
# 655 and 666, 25600 x 1024 x 1024 1012 and 1075; without the input's gradient
# 8192 x 1024 x 1024 196-247 and 245, 12800 x 1024 x 512 215-243 and 252
_DIGITS_MIN_MACS_DX = 3 << 32


def _cast_spikes(x, flags, stream, bf16=True):
    """(bits of x ``[T, B, F]`` as int32 words ``[ceil(F / 128), T, B, 4]``,
    its bf16 copy or None); flags as myelin_cast_spikes."""

    T, B, F = x.shape
    stages = -(-F // 128)
    words = torch.empty((stages, T, B, 4), dtype=torch.int32, device=x.device)
    xb = torch.empty(x.shape, dtype=torch.bfloat16, device=x.device) if bf16 else None
    _lib.call("myelin_cast_spikes", _lib.ptr(x), _lib.ptr(words), _lib.ptr(xb), T * B, F, 4 * stages,
              _lib.ptr(flags), stream)
    return words, xb


class _Digits:
    """An fp32 weight ``[F, N]`` as the four int8 digit planes and the column
    scales myelin_gemm_spikes reads (the ``wt`` of an input of words)."""

    def __init__(self, q: torch.Tensor, scale: torch.Tensor):
        self.q = q
        self.scale = scale


class _Split:
    """The fp32 synapse on the int8 or the bf16 MFMA.

    An input of zeros and ones (spikes) times W runs as four int8 products
    with the base-256 digits of W, summed without rounding and rounded once
    (``myelin_gemm_spikes``), where the digits hold W as well as an fp32
    product would (they are 31 bits of each column's largest weight; columns
    of too wide a range are turned away).  An input whose every value is a
    bf16 value runs as three bf16 products, ``x @ W = x @ W_hi + x @ W_mid +
    x @ W_lo`` with the three bf16 planes of W summing exactly to W, so every
    product is exact and only the fp32 summation rounds.  Per multiply-add the
    first costs 2/3 of the second, and that a fifth of the fp32 engine.

    Construction launches the checked copies of x (``words``, its bits, and
    ``xb`` bf16; without ``bf16`` only the words), the form of W they are
    tried with, an asynchronous copy of the check's flags to pinned host
    memory and, given ``first`` = (bias, steps, exact), the currents of the
    first steps from them (``head``, see _lif_fwd), which the GPU computes
    while the host waits; ``exact()`` and ``operands()`` wait for the flags.
    A sample of x is checked first: on the int8 products' route the launches
    behind it end at once where it shows real values.  What the check costs
    those (the launches and the host's wait; us without a check and with):
    784 -> 2048, T=50, B=256 forward 500 and 523, 1024 -> 2048, T=100, B=128
    packed 521 and 557, 784 -> 2048, T=50, B=64 packed 146 and 167; what it
    gives spikes: 501 -> 192, 518 -> 157, 146 -> 77.

    ``ints=False`` takes the bf16 products alone, and ``lean`` (the memory
    policy) implies it: no whole copy of x is kept then (``xb`` is a
    _LazyBf16), and a second copy and the digits of W beside the bf16 slices
    that its weight gradient reads anyway would be its largest buffers.
    Otherwise a layer over spikes holds, until its backward, x's bf16 copy,
    and while it runs the words, 4 (digits) or 6 (planes) bytes a weight and
    one chunk of currents, also where the fused kernel would keep those in
    LDS."""

    def __init__(self, x, w, stream, lean=False, bf16=True, ints=True, first=None):
        T, B, F = x.shape
        N = w.shape[1]
        dev = x.device
        self.x, self.w = x, w
        self.words = self.xb = self.digits = self._w3 = self.head = None
        digits = not lean and ints and F <= _DIGITS_MAX_F
        if digits:
            flags = torch.empty(2, dtype=torch.int32, device=dev)
            _lib.call("myelin_probe_spikes", _lib.ptr(x), x.numel(), _lib.ptr(flags), stream)
            self.words, self.xb = _cast_spikes(x, flags, stream, bf16=bf16)
            # a weight the digits cannot hold raises the words' flag as well
            kp = 128 * self.words.shape[0]
            q = torch.empty((-(-N // 32), 128, kp), dtype=torch.int8, device=dev)
            self.digits = _Digits(q, torch.empty(N, dtype=torch.float32, device=dev))
            _lib.call("myelin_weight_digits", _lib.ptr(w), _lib.ptr(q), _lib.ptr(self.digits.scale), F, N, kp,
                      _lib.ptr(flags), stream)
        else:
            flags = torch.zeros(2, dtype=torch.int32, device=dev)
            if lean:
                # no whole bf16 copy: check x slice by slice into one scratch
                # buffer (the flag is only ever set), and cast per chunk later
                self.xb = _LazyBf16(x)
                step = max(1, (1 << 22) // max(1, x[0].numel()))
                scratch = torch.empty((min(step, T), B, F), dtype=torch.bfloat16, device=dev)
                for t0 in range(0, T, step):
                    part = x[t0:t0 + step]
                    _lib.call("myelin_cast_bf16_checked", _lib.ptr(part), _lib.ptr(scratch), part.numel(),
                              _lib.ptr(flags), stream)
            else:
                self.xb = torch.empty(x.shape, dtype=torch.bfloat16, device=dev)
                _lib.call("myelin_cast_bf16_checked", _lib.ptr(x), _lib.ptr(self.xb), x.numel(), _lib.ptr(flags),
                          stream)
        self._host = torch.empty(2, dtype=torch.int32, pin_memory=True)
        self._host.copy_(flags, non_blocking=True)
        self._ready = torch.cuda.Event()
        self._ready.record(torch.cuda.current_stream(dev))
        self._flags = None
        if first is not None:
            b, steps, exact = first
            head = torch.empty((steps, B, N), dtype=torch.float32, device=dev)
            if digits:
                _lib.call("myelin_gemm_spikes_if", _lib.ptr(flags), _lib.ptr(self.words), T * B, _lib.ptr(q),
                          _lib.ptr(self.digits.scale), _lib.ptr(b), _lib.ptr(head), steps * B, N, kp, N, stream)
            else:
                _gemm_parts(self.xb[0:steps], self.w3, 3, N * F, head, steps * B, N, F, F, F, N, False, True, False,
                            stream, bias=b, split=not exact)
            self.head = head
        elif not digits:
            self.w3  # (formed while the host waits)

    @property
    def w3(self):
        """The three bf16 planes of W^T ``[3, N, F]``, formed when first asked for."""

        if self._w3 is None:
            F, N = self.w.shape
            self._w3 = torch.empty((3, N, F), dtype=torch.bfloat16, device=self.w.device)
            _lib.call("myelin_split_bf16x3", _lib.ptr(self.w), _lib.ptr(self._w3), F, N, 1,
                      _lib.stream(self.w.device))
        return self._w3

    def _answer(self):
        if self._flags is None:
            self._ready.synchronize()
            self._flags = tuple(self._host.tolist())
        return self._flags

    def exact(self) -> bool:
        """Every value of x is a bf16 value."""

        return self._answer()[0] == 0

    def operands(self):
        """(xs, wt, xg): the currents' operands on the engine that takes this
        input -- words and digits, bf16 and planes, or the fp32 input and
        None -- and what the weight gradient's GEMM reads (the bf16 copy if the
        input is exact in it, else x; None on digits without ``bf16``).
        ``head`` is dropped where it was computed on another engine."""

        inexact, other = self._answer()
        if inexact:
            self.head = None
            return self.x, None, self.x
        if self.digits is not None and not other:
            return self.words, self.digits, self.xb
        if self.digits is not None:
            self.head = None
        if self.xb is None:
            flags = torch.zeros(2, dtype=torch.int32, device=self.x.device)  # known to hold: not read back
            self.xb = _cast_spikes(self.x, flags, _lib.stream(self.x.device))[1]
        return self.xb, self.w3, self.xb


def _exact_split(wt) -> bool:
    """``wt`` belongs to a split of the fp32 synapse (see _lif_fwd)."""

    return isinstance(wt, _Digits) or (wt is not None and wt.ndim == 3)


def _pack_operands(x, xs, wt, xg):
    """(tensors to save, how to read them back) of a layer's operands (xs,
    wt, xg); a _LazyBf16 is saved as its fp32 input."""

    lazy = isinstance(xs, _LazyBf16)
    digits = isinstance(wt, _Digits)
    tensors = [x, x] if lazy else [xs, xg]
    return tensors + ([wt.q, wt.scale] if digits else [wt]), (lazy, digits)


def _unpack_operands(how, tensors):
    lazy, digits = how
    xs, xg = tensors[:2]
    if lazy:
        xs = xg = _LazyBf16(xs)
    return xs, _Digits(tensors[2], tensors[3]) if digits else tensors[2], xg


def _split_synapse(*args, **kwargs):
    """Start the split of ``x @ W`` (see _Split)."""

    return _Split(*args, **kwargs)


def _split_eligible(prec: int, T: int, B: int, F: int, N: int, ints: bool = True, packed: bool = False) -> bool:
    """fp32 synapse wide enough for tiles (narrower outputs stream the input
    once through the narrow kernels), of widths whose rows the bf16 loaders
    take (the weight gradient reads the bf16 copy on either route), with
    enough work to amortise the input check -- and no graph being captured
    on the current stream: the split's choice needs the input check's flags on
    the host (``_Split.operands``), a wait that capture does not allow and
    whose answer a replay could not revisit, so captured layers keep the fp32
    engine, and may differ in a sum's last bits from the same layer run
    eagerly.  ``ints``: the int8 products may be tried; ``packed``: the
    output is packed words only."""

    if prec != _lib.PREC["fp32"] or N <= 32 or F % 8 != 0 or N % 8 != 0 or T * B * F * N < _SPLIT_MIN_MACS:
        return False
    # the bf16 products alone: the shapes the fused kernel does not take
    if _fused(B, N) and not (ints and (_DIGITS_MIN_F_PACKED if packed else _DIGITS_MIN_F_FUSED) <= F <= _DIGITS_MAX_F):
        return False
    return not torch.cuda.is_current_stream_capturing()


class HipLinearFunction(torch.autograd.Function):
    """``inputs @ weight + bias`` on the MFMA GEMM (LinearSynapse, modules.py:112-133).

    Backward: ``dX = dY W^T``, ``dW = X^T dY``, ``db = sum over rows of dY``.
    """

    @staticmethod
    def forward(ctx: Any, x, w, b, prec):
        F, N = w.shape
        x2 = x.reshape(-1, F)
        M = x2.shape[0]
        out = torch.empty((M, N), dtype=x.dtype, device=x.device)
        _gemm(x2, w, out, M, N, F, F, N, N, False, False, False, prec, _lib.stream(x.device), bias=b)
        ctx.prec = prec
        ctx.has_b = b is not None
        ctx.save_for_backward(x2, w)
        ctx.in_shape = x.shape
        return out.reshape(*x.shape[:-1], N)

    @staticmethod
    def backward(ctx: Any, gy):
        x2, w = ctx.saved_tensors
        F, N = w.shape
        M = x2.shape[0]
        gy2 = gy.float().reshape(M, N).contiguous()
        dev = x2.device
        gx = gw = gb = None
        with torch.cuda.device(dev):
            stream = _lib.stream(dev)
            if ctx.needs_input_grad[0]:
                gx = torch.empty((M, F), dtype=x2.dtype, device=dev)
                _gemm(gy2, w, gx, M, F, N, N, N, F, False, True, False, ctx.prec, stream)
                gx = gx.reshape(ctx.in_shape)
            if ctx.has_b and ctx.needs_input_grad[2]:
                gb = torch.empty((N,), dtype=x2.dtype, device=dev)
            if ctx.needs_input_grad[1]:
                # db rides with dW's launches
                gw = torch.empty_like(w)
                _gemm(x2, gy2, gw, F, N, M, F, N, N, True, False, False, ctx.prec, stream,
                      col_sum=None if gb is None else (gy2, gb))
            elif gb is not None:
                _lib.call("myelin_col_sum_f32", _lib.ptr(gy2), _lib.ptr(gb), M, N, 0, stream)
        return gx, gw, gb, None


def linear(x, w, b, precision: str = "fp32"):
    """Differentiable ``x @ w + b`` for ``x [..., F]``, ``w [F, N]`` on the HIP GEMM."""

    _lib.require_device(x, "inputs")
    if x.dtype != torch.float32 or w.dtype != torch.float32:
        raise ValueError("inputs and weight must be float32 for the HIP path")
    if x.shape[-1] != w.shape[0]:
        raise ValueError("inputs.shape[-1] must match weight.shape[0]")
    with torch.cuda.device(x.device):
        return HipLinearFunction.apply(x.contiguous(), w.contiguous(), None if b is None else b.contiguous(),
                                       _lib.PREC[precision])


# currents buffer budget of the chunked path (floats)
_CURRENT_CHUNK_ELEMS = 1 << 25


def _fused_grid(B: int, N: int) -> int:
    """Workgroups of the fused kernel (its 8- or 4-row batch tiles)."""

    nt = -(-N // 64)
    return nt * -(-B // 8) if nt * -(-B // 8) >= 512 else nt * -(-B // 4)


def _fused(B: int, N: int) -> bool:
    """The forward takes the fused kernel (else GEMM chunks + recurrence)."""

    return N >= 64 and _fused_grid(B, N) >= 1024


def _span(T: int, checkpoint: int, BN: int, budget: int = _CURRENT_CHUNK_ELEMS) -> int:
    """Steps per backward span of a checkpointed layer: whole chunks, as
    many as keep a span's trace within ``budget`` floats."""

    return checkpoint * max(1, min(math.ceil(T / checkpoint), budget // (checkpoint * BN)))


# a narrow layer (<= 32 neurons) over packed spikes takes the one-launch
# currents + recurrence kernel from this batch size on: one workgroup per
# batch row, so smaller batches leave the chip idle and the GEMM + recurrence
# launches are faster
_NARROW_FUSED_MIN_B = 128

# forward chunk budget (floats) of the memory-lean policy: the forward's
# buffers are transient and never set a checkpointed step's peak, which the
# backward's span buffers do, so the forward keeps chunks large enough for
# its GEMMs to fill the chip
_LEAN_FWD_ELEMS = 1 << 24


def _budgets(lean: bool, checkpoint, B: int, N: int) -> tuple[int, int]:
    """(forward chunk, backward span) buffer budgets in floats.  Under the
    memory-lean policy (checkpoint_size="memory", whose purpose is to keep
    the chunk scratch small, checkpointing.py:13-20) a backward span is one
    checkpoint chunk and forward chunks hold 2**24 currents; otherwise both
    hold 2**25 -- fewer, larger GEMMs."""

    if lean and checkpoint is not None:
        return _LEAN_FWD_ELEMS, checkpoint * B * N
    return _CURRENT_CHUNK_ELEMS, _CURRENT_CHUNK_ELEMS


def _chunk_steps(T: int, B: int, N: int, budget: int) -> int:
    """Steps of a chunk of up to ``budget`` currents (see _lif_fwd)."""

    return max(1, min(T, budget // (B * N)))


def _lif_fwd(x, w, b, m0, t0, t1, decay, threshold, reset, slope, rule, prec, stream, *, m_final=None,
             spikes=None, pre=None, packed=None, rates=None, ckpt=None, ckpt_every=1, wt=None, exact=False,
             pre_from=None, x_bits=None, budget=_CURRENT_CHUNK_ELEMS, cur=None, head=None):
    """Synaptic currents + LIF recurrence over steps [t0, t1).

    ``x`` is fp32 with ``w [F, N]`` fp32, or bf16 (bf16 synapse) with ``wt``,
    the bf16 transposed weight ``[N, F]``; or a split's operands: bf16
    with ``wt`` its planes ``[3, N, F]``, or words (see _cast_spikes) with
    ``wt`` a _Digits.
    Fused (one launch, currents stay in LDS) when N >= 64 and the fused grid
    has >= 1024 workgroups, except on the split.
    Otherwise each workgroup would walk many chunks serially, so the steps
    are processed in chunks of up to ``budget`` currents: an MFMA GEMM (split-K
    when narrow) writes ``x_t @ W + b`` for the chunk, then the recurrence
    kernel consumes it, carrying the membrane and the spike counts across
    chunks; with several chunks, each chunk's GEMM runs on a side stream
    while the previous chunk's recurrence runs.  ``pre`` receives the steps
    from ``pre_from`` (default t0; the chunked route only) on; checkpoint
    rows count from t0.
    ``exact``: the GEMM never splits K, so a checkpointed forward and the
    backward's recompute of any chunk of it produce the same currents bit
    for bit (the fused kernel always sums that way).
    ``x_bits``: the input as packed spike words ``[T, B, ceil(F / 32)]``,
    which the chunked route's GEMM reads in place of ``x`` (fp32 synapse
    weights ``w``; the same sums bit for bit).
    ``cur``: an fp32 buffer of at least one chunk's currents for the chunked
    route to use instead of allocating its own (when the GEMMs run in turn
    on the one stream).
    ``head [steps, B, N]``: such a buffer that holds the currents of the
    first ``steps`` steps already (a _Split's).
    """

    digits = wt if isinstance(wt, _Digits) else None
    T, B = x_bits.shape[:2] if x_bits is not None else x.shape[1:3] if digits is not None else x.shape[:2]
    F = w.shape[0]
    half = x_bits is None and digits is None and x.dtype == torch.bfloat16
    parts = half and wt.ndim == 3  # exact split: wt holds the planes [3, N, F]
    N = wt.shape[-2] if half else w.shape[1]
    if digits is None and not parts and _fused(B, N):
        if pre_from not in (None, t0):
            raise ValueError("pre_from is a chunked-route option")
        outs = (_lib.ptr(b), _lib.ptr(m0), _lib.ptr(m_final), _lib.ptr(spikes), _lib.ptr(pre), _lib.ptr(packed),
                _lib.ptr(rates), _lib.ptr(ckpt), T, B, F, N, t0, t1, ckpt_every, decay, threshold, reset, slope, rule)
        if half:
            _lib.call("myelin_linear_lif_fwd_bf16", _lib.ptr(x), _lib.ptr(wt), *outs, stream)
        else:
            _lib.call("myelin_linear_lif_fwd", _lib.ptr(x), _lib.ptr(w), *outs, prec, stream)
        return
    dev = x.device
    p0 = t0 if pre_from is None else pre_from  # pre holds the steps from p0 on
    if (x_bits is not None and N <= 32 and B >= _NARROW_FUSED_MIN_B and not exact and packed is None
            and ckpt is None and p0 == t0 and (rates is None or (t0 == 0 and t1 == T))
            and rule in (_lib.RULE_THRESHOLD, _lib.RULE_SURROGATE) and _lib.load().myelin_narrow_bits_fits(F, N, prec)):
        # a narrow layer over spikes with a batch that fills the chip: the
        # currents and the recurrence in one launch (never for a layer whose
        # backward recomputes, which must repeat its forward's GEMM)
        _lib.call("myelin_linear_lif_fwd_narrow_bits", _lib.ptr(x_bits), _lib.ptr(w), _lib.ptr(b), _lib.ptr(m0),
                  _lib.ptr(m_final), _lib.ptr(spikes), _lib.ptr(pre), _lib.ptr(rates), T, B, F, N, t0, t1, decay,
                  threshold, reset, slope, rule, prec, stream)
        return
    step = _chunk_steps(t1 - t0, B, N, budget)
    cuts = {p0}
    done_to = t0  # the currents of the steps before it are in head
    if head is not None:
        cur, done_to = head, t0 + head.shape[0]
        cuts.add(done_to)
    bounds = sorted({*range(t0, t1, step), t1} | {c for c in cuts if t0 < c < t1})
    n = len(bounds) - 1
    # several chunks on the fp32 engine: each chunk's GEMM runs on the side
    # stream one chunk ahead of the recurrence, into two alternating
    # currents buffers.  The bf16 engines (and the split) fill the chip with
    # one workgroup per CU, and beside them the recurrence and the GEMM
    # slow each other down (the 1024 -> 4096 -> 20 rate network's step at
    # T=2000, B=32: 7.92-8.01 ms overlapped, 7.53 serial), so they run in
    # turn on the one stream.
    overlap = False
    if n > 1 and not half and digits is None:
        main = torch.cuda.current_stream(dev)
        side = _side_stream(dev)
        overlap = main.cuda_stream == stream and side.cuda_stream != stream
    if cur is not None and not overlap and cur.dtype == torch.float32 and cur.numel() >= step * B * N:
        curs = [cur.reshape(-1)[:step * B * N].view(step, B, N)]
    else:
        curs = [torch.empty((step, B, N), dtype=torch.float32, device=dev) for _ in range(2 if overlap else 1)]
    # the membrane carried across chunks lives in m_final (each lane reads
    # its m0 before writing, so m0 may be m_final); a single chunk needs no
    # carry buffer at all
    state = m_final
    if state is None and n > 1:
        state = torch.empty((B, N), dtype=torch.float32, device=dev)
    # spike counts carried across chunks (one chunk counts in registers)
    counts = torch.zeros((B, N), dtype=torch.float32, device=dev) if rates is not None and n > 1 else None
    if overlap:
        side.wait_stream(main)
        done = [torch.cuda.Event(), torch.cuda.Event()]  # GEMM wrote buffer i
        used = [torch.cuda.Event(), torch.cuda.Event()]  # the recurrence read buffer i

    def gemm(c0, c1, cur, s):
        rows = (c1 - c0) * B
        if x_bits is not None:
            _gemm(x_bits[c0:c1], w, cur, rows, N, F, x_bits.shape[2], N, N, False, False, False, prec, s, bias=b,
                  a_bits=True, split=not exact)
        elif digits is not None:
            _lib.call("myelin_gemm_spikes", _lib.ptr(x[:, c0:c1]), T * B, _lib.ptr(digits.q),
                      _lib.ptr(digits.scale), _lib.ptr(b), _lib.ptr(cur), rows, N, digits.q.shape[2], N, s)
        elif parts:
            _gemm_parts(x[c0:c1], wt, 3, N * F, cur, rows, N, F, F, F, N, False, True, False, s, bias=b,
                        split=not exact)
        elif half:
            _gemm(x[c0:c1], wt, cur, rows, N, F, F, F, N, False, True, False, prec, s, bias=b, split=not exact)
        else:
            _gemm(x[c0:c1], w, cur, rows, N, F, F, N, N, False, False, False, prec, s, bias=b, split=not exact)

    for c in range(n):
        c0, c1 = bounds[c], bounds[c + 1]
        i = c % len(curs)
        cur = curs[i]
        if c1 <= done_to:
            cur = head[c0 - t0:c1 - t0]
        s_ = side.cuda_stream if overlap else stream
        with torch.cuda.stream(side) if overlap else contextlib.nullcontext():
            if overlap and c >= 2:
                side.wait_event(used[i])
            if c1 > done_to:
                gemm(c0, c1, cur, s_)
            if overlap:
                done[i].record(side)
        if overlap:
            main.wait_event(done[i])
        last = c1 == t1
        with_pre = pre is not None and c0 >= p0
        _lib.call(
            "myelin_lif_currents_fwd",
            _lib.ptr(cur), _lib.ptr(m0 if c0 == t0 else state), _lib.ptr(state), _lib.ptr(spikes),
            _lib.ptr(pre) if with_pre else None, _lib.ptr(packed), _lib.ptr(rates) if last else None,
            _lib.ptr(counts), _lib.ptr(ckpt), T, B, N, c0, c1, p0 if with_pre else t0, t0, ckpt_every, decay,
            threshold, reset, slope, rule, stream,
        )
        if overlap:
            used[i].record(main)
    if overlap:
        # the main stream waited on every side GEMM; the inputs' and buffers'
        # last users include the side stream
        for t_ in (*curs, x, w, b, wt):
            if t_ is not None:
                t_.record_stream(side)


_SIDE_STREAMS: dict[tuple[int, int], torch.cuda.Stream] = {}


def _side_stream(dev: torch.device, which: int = 0) -> torch.cuda.Stream:
    """Side stream `which` of a device (default priority) for work that
    overlaps the current stream's, created once."""

    idx = dev.index if dev.index is not None else torch.cuda.current_device()
    s = _SIDE_STREAMS.get((idx, which))
    if s is None:
        s = torch.cuda.Stream(device=idx)
        _SIDE_STREAMS[(idx, which)] = s
    return s


def _keep_trace(F: int, N: int) -> bool:
    """A checkpointed layer keeps its whole pre-reset trace ``[T, B, N]``
    instead of checkpoints (as the uncheckpointed path does), so its
    backward recomputes nothing, when the trace is narrow: at most 32
    neurons and at most 1/8 of the saved input's bytes -- the readout
    layers, whose recompute GEMM would re-read the whole input to rebuild a
    few columns and whose serial recurrence over T runs on a few waves."""

    return N <= 32 and 8 * N <= F


def _attach_bits(out, words) -> None:
    """Records the bit-packed copy of a spike tensor the layer wrote, with
    the tensor's version: a consumer may read the bits instead (1 bit per
    spike instead of 32) while the tensor is unmodified."""

    out._myelin_bits = (words, out._version)


def _spike_bits(x):
    """The packed words of ``x [T, B, F]`` recorded by the layer that wrote
    it, or None when there are none or ``x`` changed since (its version
    moved on)."""

    rec = getattr(x, "_myelin_bits", None)
    if rec is None:
        return None
    words, version = rec
    T, B, F = x.shape
    if version != x._version or words.shape != (T, B, -(-F // 32)) or words.device != x.device:
        return None
    return words


def _bits_consumer(B: int, F: int, N: int, prec: int) -> bool:
    """A layer reads its input's packed twin: the chunked route with a
    narrow output (the GEMMs stream the input once per pass; the bits cut
    those reads 32-fold and sum the same products in the same order)."""

    return N <= 32 and not _fused(B, N) and not _half(prec, F, N)


class HipLinearLIFFunction(torch.autograd.Function):
    """Outputs ``(final_membrane, spikes)`` or, with ``rate=True``,
    ``(final_membrane, rates)`` where ``rates = spike_count / T``."""

    @staticmethod
    def forward(ctx: Any, x, w, b, decay, threshold, reset, sid, slope, checkpoint, rate, prec, rule, lean=False):
        T, B, F = x.shape
        N = w.shape[1]
        dev = x.device
        stream = _lib.stream(dev)
        need = any(ctx.needs_input_grad[:3])
        half = _half(prec, F, N)
        xs, wt = _cast_transpose_bf16(x, w, stream) if half else (x, None)
        bits = _spike_bits(x) if _bits_consumer(B, F, N, prec) else None
        fwd_budget, budget = _budgets(lean, checkpoint, B, N)
        xg = xs
        split = None
        ints = not lean or checkpoint is None
        if not _fused(B, N) and ctx.needs_input_grad[0] and T * B * F * N < _DIGITS_MIN_MACS_DX:
            ints = False
        if not half and bits is None and _split_eligible(prec, T, B, F, N, ints=ints):
            split = _split_synapse(x, w, stream, lean=lean and checkpoint is not None, bf16=need, ints=ints,
                                   first=(b, _chunk_steps(T, B, N, fwd_budget), need and checkpoint is not None))
        m_final = torch.empty((B, N), dtype=x.dtype, device=dev)
        out = torch.empty((B, N) if rate else (T, B, N), dtype=x.dtype, device=dev)
        # spikes: their packed twin too (N / 8 bytes per row more), for a
        # narrow layer reading them next
        words = torch.empty((T, B, -(-N // 32)), dtype=torch.int32, device=dev) if not rate else None
        if checkpoint is not None and _keep_trace(F, N):
            checkpoint = None
        pre = ckpt = None
        tail = 0
        fused = _fused(B, N)
        if need:
            if checkpoint is None:
                pre = torch.empty((T, B, N), dtype=x.dtype, device=dev)
            else:
                ckpt = torch.empty((math.ceil(T / checkpoint), B, N), dtype=x.dtype, device=dev)
                if not fused or split is not None:
                    # the backward starts with the last span, whose trace
                    # this forward computes anyway: keep it (the buffer the
                    # backward would fill) instead of recomputing it there
                    span = _span(T, checkpoint, B * N, budget)
                    tail = (math.ceil(T / span) - 1) * span
                    pre = torch.empty((T - tail, B, N), dtype=x.dtype, device=dev)
        if split is not None:
            # (asked for after the allocations: the GPU runs the split's
            # launches meanwhile)
            xs, wt, xg = split.operands()
            if fused and checkpoint is not None and not _exact_split(wt):
                pre, tail = None, 0  # the fused kernel keeps no part of the trace
        _lif_fwd(xs, w, b, None, 0, T, decay, threshold, reset, slope, rule, prec, stream, m_final=m_final,
                 spikes=None if rate else out, pre=pre, packed=words, rates=out if rate else None, ckpt=ckpt,
                 ckpt_every=checkpoint or 1, wt=wt, exact=ckpt is not None, pre_from=tail, x_bits=bits,
                 budget=fwd_budget, head=None if split is None else split.head)
        if words is not None:
            _attach_bits(out, words)
        if bits is not None:
            xs = xg = bits  # what the backward's weight GEMM reads
        ctx.set_materialize_grads(False)
        # the bf16 synapse keeps the bf16 copies of x and W^T (what its
        # GEMMs read), the split its copies of x and form of W
        if checkpoint is None:
            xs, wt = (xg, wt) if not isinstance(wt, _Digits) else (xg, None)  # nothing to recompute
        saved, how = _pack_operands(x, xs, wt, xg) if need else ((), None)
        ctx.meta = (decay, threshold, reset, sid, slope, checkpoint, rate, prec, rule, b is not None,
                    F if bits is not None else None, budget, how)
        if need:
            ctx.save_for_backward(w, b, pre, ckpt, *saved)
        return m_final, out

    @staticmethod
    def backward(ctx: Any, g_m, g_out):
        none = (None,) * 13
        if (g_m is None and g_out is None) or not any(ctx.needs_input_grad[:3]):
            return none
        decay, threshold, reset, sid, slope, checkpoint, rate, prec, rule, has_b, bits_f, budget, how = ctx.meta
        w, b, pre, ckpt, *saved = ctx.saved_tensors
        xs, wt, xg = _unpack_operands(how, saved)
        need_x, need_w, need_b = ctx.needs_input_grad[:3]
        gx, gw, gb = linear_backward(xs, w, b if has_b else None, pre, ckpt, wt, g_m, g_out, decay, threshold,
                                     reset, sid, slope, checkpoint, rate, prec, rule, need_x, need_w,
                                     need_b and has_b, bits_f=bits_f, budget=budget, xg=xg)
        return gx, gw, gb, None, None, None, None, None, None, None, None, None, None


def linear_backward(xs, w, b, pre, ckpt, wt, g_m, g_out, decay, threshold, reset, sid, slope, checkpoint, rate,
                    prec, rule, need_x=True, need_w=True, need_b=True, bits_f=None, budget=_CURRENT_CHUNK_ELEMS, xg=None):
    """Gradients (dX, dW, db) of the streamed-synapse LIF, span by span in
    reverse time: recompute the span's pre-reset trace from its first
    checkpoint (``checkpoint=None``: the saved trace ``pre`` covers all T;
    with a checkpoint, ``pre`` if given is the last span's trace, kept by
    the forward), reverse the recurrence into G = dL/dI, then ``dX = G W^T`` and
    ``dW += X^T G`` on the MFMA GEMM and ``db`` as a fixed-order column
    sum.  ``xs`` is fp32, or
    bf16 with ``wt = W^T`` bf16 for the bf16 synapse, or (``bits_f`` = F)
    the input spikes' packed words ``[T, B, ceil(F / 32)]``, or an exact
    split's operand with its ``wt`` (see _lif_fwd); ``xg`` is what dW's GEMM
    reads where that is not ``xs``; ``g_out`` is dL/dspikes ``[T, B, N]`` or, with ``rate``, dL/drates ``[B, N]``."""

    T, B = xs.shape[1:3] if isinstance(wt, _Digits) else xs.shape[:2]
    x_bits = xs if bits_f is not None else None
    F, N = w.shape
    BN = B * N
    dev = w.device
    xg = xs if xg is None else xg
    split = _exact_split(wt) or (xg.dtype == torch.bfloat16 and prec == _lib.PREC["fp32"])
    half = xs.dtype == torch.bfloat16 and not split
    parts = split and xg.dtype == torch.bfloat16  # dW: x exact in bf16, G as three planes
    with torch.cuda.device(dev):
        stream = _lib.stream(dev)
        wg = _cast_bf16(w, stream) if (half and need_x) else w
        # the reverse pass walks spans of whole checkpoint chunks, as many as
        # keep a span's trace within `budget` floats: one recompute
        # (from the span's first checkpoint, which the recurrence carries
        # through the later ones exactly as the forward did), one reverse
        # launch and one dX / dW GEMM pair per span instead of per chunk
        span = T if checkpoint is None else _span(T, checkpoint, BN, budget)
        per = 1 if checkpoint is None else span // checkpoint  # checkpoint rows per span
        want_gb = need_b and b is not None
        # one span and no membrane gradient: the reverse launch is the whole
        # pass (no adjoint buffer; it writes the bias sums itself), else the
        # zero-started buffers (the membrane adjoint unless given, the bias
        # gradient's accumulator) share one allocation: one fill launch
        whole = g_m is None and span >= T
        zeros = None
        if not whole and (g_m is None or want_gb):
            zeros = torch.zeros(((g_m is None) + want_gb, B, N), device=dev)
        gm = g_m.float().contiguous().clone() if g_m is not None else (None if whole else zeros[0])
        g_out = None if g_out is None else g_out.float().contiguous()
        g_spikes = None if rate else g_out
        g_rates = g_out if rate else None
        gx = torch.empty((T, B, F), device=dev) if need_x else None
        gw = torch.empty_like(w) if need_w else None  # the first (last-in-time) span overwrites it
        gb_acc = (torch.empty((B, N), device=dev) if whole else zeros[-1]) if want_gb else None
        gb = torch.empty((N,), device=dev) if want_gb else None
        # exact split: dW reads G as three bf16 planes [3, C, B, N] (C the
        # span's steps), written by the reverse pass itself unless dX needs
        # the fp32 G as well
        G3 = torch.empty(3 * min(span, T) * BN, dtype=torch.bfloat16, device=dev) if parts and need_w else None
        if G3 is not None and not need_x:
            G = G3
        else:
            G = torch.empty((min(span, T), B, N), dtype=torch.bfloat16 if half else torch.float32, device=dev)
        n_spans = math.ceil(T / span)
        tail = pre if checkpoint is not None else None  # the last span's trace, from the forward
        if tail is not None and tail.shape[0] != T - (n_spans - 1) * span:
            raise ValueError("the saved trace does not cover the last backward span")
        recomputes = checkpoint is not None and (tail is None or n_spans > 1)
        # GEMM recomputes on the fp32 engine run one span ahead on a side
        # stream, into two alternating trace buffers: span k-1's recompute
        # overlaps span k's reverse pass and weight GEMMs (the bf16 engines
        # and the split run in turn, as in the forward).  ready[i]: buffer i
        # holds its span's trace; free[i]: the reverse pass has read buffer i.
        overlap = checkpoint is not None and n_spans > 1 and not (half or split)
        # in turn, the trace buffer is spent once the reverse pass has read
        # it and is refilled only by the next span's recompute: it doubles
        # as the split-K workspace of the span's dX and dW GEMMs
        ws = None
        if recomputes:
            n_sc = min(span, T) * BN
            if not overlap:
                lib, r_span = _lib.load(), min(span, T) * B
                n_sc = max(n_sc, lib.myelin_gemm_workspace_elems(r_span, F, N, prec) if need_x else 0,
                           lib.myelin_gemm_workspace_elems(F, N, r_span, _lib.PREC["bf16"] if parts else prec)
                           if need_w else 0)
            ws = torch.empty(n_sc, device=dev)
            scratch = ws[:min(span, T) * BN].view(min(span, T), B, N)
            if overlap:
                ws = None
        else:
            scratch = None
        if overlap:
            main = torch.cuda.current_stream(dev)
            side = _side_stream(dev)
            bufs = [scratch, torch.empty_like(scratch)]
            ready = [torch.cuda.Event(), torch.cuda.Event()]
            free = [torch.cuda.Event(), torch.cuda.Event()]
            side.wait_stream(main)

            def recompute(j):
                i = j % 2
                with torch.cuda.stream(side):
                    if j + 2 < n_spans:
                        side.wait_event(free[i])
                    _lif_fwd(xs, w, b, ckpt[j * per], j * span, min(j * span + span, T), decay, threshold, reset,
                             slope, rule, prec, side.cuda_stream, pre=bufs[i], wt=wt, exact=True, x_bits=x_bits,
                             budget=budget)
                    ready[i].record(side)

            if tail is None:
                recompute(n_spans - 1)
        for k in range(n_spans - 1, -1, -1):
            t0 = k * span
            t1 = min(t0 + span, T)
            C = t1 - t0
            if checkpoint is None:
                pre_k = pre
            elif k == n_spans - 1 and tail is not None:
                if overlap:
                    recompute(k - 1)
                pre_k = tail
            elif overlap:
                if k > 0:
                    recompute(k - 1)
                main.wait_event(ready[k % 2])
                pre_k = bufs[k % 2]
            else:
                # the recompute's currents may use G's buffer: the reverse
                # pass writes G only after the recompute
                _lif_fwd(xs, w, b, ckpt[k * per], t0, t1, decay, threshold, reset, slope, rule, prec, stream,
                         pre=scratch, wt=wt, exact=True, x_bits=x_bits, budget=budget, cur=G)
                pre_k = scratch
            _lib.call(
                "myelin_linear_pre_bwd",
                _lib.ptr(pre_k), _lib.ptr(g_spikes[t0:t1]) if g_spikes is not None else None,
                _lib.ptr(g_rates), _lib.ptr(gm), _lib.ptr(G), _lib.DT_BF16X3 if G is G3 else _lib.DT[G.dtype],
                _lib.ptr(gb_acc),
                C, BN, T, decay, threshold, reset, slope, sid, rule, stream,
            )
            if overlap:
                free[k % 2].record(main)
            rows = C * B
            # (dW on a third stream beside dX measured slower on the readout
            # shapes: the 784 -> 2048 -> 10 bf16 training step at T=50,
            # B=256 went from 0.547 to 0.606 ms)
            if gx is not None:
                # dX[t0:t1] = G @ W^T : [rows, N] x [N, F]
                _gemm(G, wg, gx[t0:t1], rows, F, N, N, N, F, False, True, False, prec, stream, ws=ws)
            # db (the bias sums complete once the first span's reverse pass
            # has run) rides with that span's dW launches
            cs = (gb_acc, gb) if k == 0 and gb is not None else None
            if gw is not None and parts:
                if G is not G3:
                    _lib.call("myelin_split_bf16x3", _lib.ptr(G), _lib.ptr(G3), rows, N, 0, stream)
                _gemm_parts(xg[t0:t1], G3, 3, rows * N, gw, F, N, rows, F, N, N, True, False, k != n_spans - 1,
                            stream, ws=ws, col_sum=cs)
            elif gw is not None and x_bits is not None:
                _gemm(x_bits[t0:t1], G, gw, F, N, rows, x_bits.shape[2], N, N, True, False, k != n_spans - 1, prec,
                      stream, a_bits=True, ws=ws, col_sum=cs)
            elif gw is not None:
                # dW (+)= X[t0:t1]^T @ G : [F, rows] x [rows, N]
                _gemm(xg[t0:t1], G, gw, F, N, rows, F, N, N, True, False, k != n_spans - 1, prec, stream, ws=ws,
                      col_sum=cs)
        if overlap:
            # every side-stream kernel is behind a ready[] the main stream
            # waited on; the buffers' last users include the side stream
            for t in (*bufs, xs, w, ckpt, *(() if b is None else (b,)), *(() if wt is None else (wt,))):
                t.record_stream(side)
        if gb is not None and gw is None:
            _lib.call("myelin_col_sum_f32", _lib.ptr(gb_acc), _lib.ptr(gb), B, N, 0, stream)
    return gx, gw, gb


def linear_forward(x, w, b, params, surrogate_id: int, slope: float, checkpoint, rate: bool, precision: str,
                   rule: int = _lib.RULE_THRESHOLD, lean: bool = False):
    """Validate and run the fused streamed-synapse LIF (shared by the public
    entry points in myelin_amd.kernels).  ``lean``: the memory-lean policy
    (chunk and span buffers of one checkpoint chunk)."""

    if x.ndim != 3:
        raise ValueError(f"inputs must be shaped [T, B, F]; got {tuple(x.shape)}")
    if w.ndim != 2:
        raise ValueError(f"weight must be shaped [F, N]; got {tuple(w.shape)}")
    _lib.require_device(x, "inputs")
    if w.device != x.device or w.dtype != x.dtype:
        raise ValueError("weight must have the same device and dtype as inputs")
    if x.shape[2] != w.shape[0]:
        raise ValueError("inputs.shape[2] must match weight.shape[0]")
    if b is not None:
        if b.shape != (w.shape[1],):
            raise ValueError("bias must be shaped [N]")
        if b.device != x.device or b.dtype != x.dtype:
            raise ValueError("bias must have the same device and dtype as inputs")
    if x.dtype != torch.float32:
        raise ValueError(f"inputs must be float32 for the HIP path; got {x.dtype}")
    if x.shape[0] == 0:
        raise ValueError("inputs must have at least one timestep")
    if precision not in _lib.PREC:
        raise ValueError("synapse_precision must be 'fp32' or 'bf16'")
    with torch.cuda.device(x.device):
        return HipLinearLIFFunction.apply(
            x.contiguous(), w.contiguous(), None if b is None else b.contiguous(), float(params.decay),
            float(params.threshold), float(params.reset), surrogate_id, float(slope), checkpoint, rate,
            _lib.PREC[precision], rule, lean,
        )


def linear_packed_forward(x, w, b, params, checkpoint: int, precision: str):
    """Forward-only packed-spike output (no dense [T, B, N] spikes)."""

    from myelin_amd.packing import PackedSpikes, packed_last_dim_size

    if x.ndim != 3:
        raise ValueError(f"inputs must be shaped [T, B, F]; got {tuple(x.shape)}")
    _lib.require_device(x, "inputs")
    if x.shape[2] != w.shape[0]:
        raise ValueError("inputs.shape[2] must match weight.shape[0]")
    if x.dtype != torch.float32 or w.dtype != torch.float32:
        raise ValueError("inputs and weight must be float32 for the HIP path")
    x = x.contiguous()
    w = w.contiguous()
    b = None if b is None else b.contiguous()
    T, B, F = x.shape
    N = w.shape[1]
    m_final = torch.empty((B, N), device=x.device)
    words = torch.empty((T, B, packed_last_dim_size(N)), dtype=torch.int32, device=x.device)
    with torch.cuda.device(x.device):
        prec, stream = _lib.PREC[precision], _lib.stream(x.device)
        xs, wt, head = x, None, None
        if _split_eligible(prec, T, B, F, N, packed=True):
            split = _split_synapse(x, w, stream, bf16=False,
                                   first=(b, _chunk_steps(T, B, N, _CURRENT_CHUNK_ELEMS), False))
            xs, wt, _ = split.operands()
            head = split.head
        _lif_fwd(xs, w, b, None, 0, T, float(params.decay), float(params.threshold), float(params.reset), 10.0,
                 _lib.RULE_THRESHOLD, prec, stream, m_final=m_final, packed=words, ckpt_every=checkpoint, wt=wt,
                 budget=_CURRENT_CHUNK_ELEMS, head=head)
    return m_final, PackedSpikes(data=words, original_shape=(T, B, N))
