"""``Int4Linear``: drop-in for the bf16 ``nn.Linear`` layers of rollout decode.

The reference calls its decode linears as plain modules, ``module(x[..., K]) ->
[..., N]`` in the model dtype, under ``torch.no_grad()``
(``vrl/models/families/janus_pro/policy.py:673-678`` for the Llama trunk,
``policy.py:138-160`` for ``gen_head``).  These modules keep that calling
convention and route the arithmetic to the HIP library; the weights are frozen
(no gradient flows into the packed tensors).  A call whose input carries a gradient
(a train-time replay over the quantised base, e.g. under LoRA adapters) computes the same
product, at prompt sizes bit for bit that of a call without one, and multiplies the gradient
by the dequantised weight, so that it reaches the input.
"""

from __future__ import annotations

import functools
import weakref

import torch
import torch.nn.functional as F
from torch import nn
from torch.overrides import _get_current_function_mode_stack
from torch.utils._device import DeviceContext

from . import ops
from .int4_format import check_packed, pack_nibbles, quantize_minmax

# Calls with more activation rows than this (the prompt pass) are matrix products; the GEMV kernels are for
# decode.  They go through the launch that rebuilds the weight in registers (``ops.int4_gemm``) where that is the
# faster form, :func:`_launch_pays`; elsewhere, and wherever that launch does not apply, the bf16 weight is rebuilt
# (bit-exact tile, one launch) and handed to the library GEMM.
GEMM_ROWS = 32
PROMPT_ROWS = 2048
FUSED_ROWS = 4096
# Weights of fewer than PROMPT_COLUMNS outputs stay on the library's route at every row count, because their results
# are pinned bit for bit to the library's product.  That is not the faster form (64 to 384 outputs by 2048, 33 to 2048
# rows: 11.7 to 14 us against 8 to 9 for the launch), but a fraction of a layer of 100 us and more.
PROMPT_COLUMNS = 512
CUS = 256


@functools.lru_cache(maxsize=1024)   # (sizes only; a hit is 0.4 us less on every call of a prompt)
def _launch_pays(rows: int, K: int, columns: int, group_size: int, products: int = 1, fused: bool = False) -> bool:
    """Whether one ``ops.int4_gemm`` launch beats rebuilding the weight and a library product per weight.

    Both routes were timed, queued back to back on the GPU, at 33 to 8192 rows, K of 1024 to 11008, up to 22016 weight
    rows and groups of 32, 64 and 128, with a launch that took 3 to 40 % longer than today's: the lines below are on the
    safe side of it.  The library's rate is 1.2 to 1.6 times the launch's once its products are
    large; what the launch saves is the pass that writes the weight, SiLU's pass and the launches of a group.  A group
    costs as much again for each halving of the group size below 128, in the table of scales of every tile: ``k``
    is the K of equal cost.
    """
    groups = K // group_size
    k = max(K, 128 * groups)
    work = rows * columns * k
    if fused:
        # 2048 -> 2 x 5632: 44 against 52 us at 512 rows, 96 against 109 at 1792; 3072 -> 2 x 8192: 96 against 109 at
        # 1024, 165 against 155 at 1536; 4096 -> 2 x 11008: 83 against 102 at 256, 236 against 209 at 1024.  From
        # FUSED_ROWS on a short K is faster again on the whole, for SiLU's pass, where the library's time jumps with
        # the rows (K = 2048: 0.69 to 1.19 of its time at twelve sizes up to 12288 rows, 0.97 in the mean, 373 against
        # 408 us at 8192; K = 1024: 0.75 to 1.04, 0.88; K = 3072: 365 against 335 at 4096, 708 against 639 at 8192).
        return rows <= PROMPT_ROWS and work <= 48 << 30 or rows >= FUSED_ROWS and K <= 2048 and k <= 4096
    if rows > PROMPT_ROWS:
        return False
    # one round of workgroups: of the builds that split K, as far as their tables of scales fit the LDS
    tiles = lambda bm, bn: -(-rows // bm) * -(-columns // bn)
    small = any(groups <= most and tiles(bm, bn) <= CUS for bm, bn, most in ((32, 64, 448), (64, 64, 320), (64, 128, 128)))
    wide = groups <= 160 and tiles(128, 128) <= CUS
    if products > 1:
        # q|k|v of 2048 / 3072 / 4096 outputs each: 61 / 96 / 207 us against 87 / 136 / 194 at 1664 rows (the last
        # stays with the library), 26 / 64 / 84 against 63 / 93 / 120 at 512.  Beyond 80 groups only one workgroup
        # fits a CU and more than a round of them is slow (groups of 32, K = 4096: 56 against 98 us at 256 rows, one
        # round; 144 against 117 at 512).
        return work < 72 << 30 if groups <= 80 else small or wide
    # One weight: worth it while its tiles are one round up to 64 x 128 (5632 -> 2048: 38 against 46 us at 1024 rows,
    # 58 against 51 at 1152; 11008 -> 4096: 67 against 85 at 512, 110 against 94 at 768).  Beyond that with two of: one
    # round of 128 x 128 tiles, a short K, few rows (2048 -> 2048: 26 against 30 us at 2048 rows; 4096 -> 16384: 48
    # against 76 at 256; 2048 -> 16384: 48 against 54 at 512; 4096 -> 4096: 45 against 42 at 768, where only the first
    # holds).
    return small or wide + (k <= 3072) + (rows <= 512) >= 2


_PLAIN = (torch.Tensor, nn.Parameter)


def _wants_grad(x: torch.Tensor) -> bool:
    """Whether autograd records the call: the HIP launches are not recorded by themselves."""
    return torch.is_grad_enabled() and x.requires_grad


def _only_default_devices() -> bool:
    """Whether the function modes in force are default devices (``torch.set_default_device``, ``with
    torch.device(...)``): they give factory calls a device and watch nothing."""
    return all(type(mode) is DeviceContext for mode in _get_current_function_mode_stack())


def _launchable(x: torch.Tensor) -> bool:
    """Whether a prompt-sized call may leave the torch operators: nothing watches them (a trace, a dispatch mode,
    a functorch transform, forward-mode differentiation, an autocast to another type), and ``x`` is a plain
    tensor.  The general route goes through ``F.linear`` and serves all of those."""
    return type(x) in _PLAIN and x.is_cuda and not torch.jit.is_tracing() \
        and torch._C._len_torch_dispatch_stack() == 0 \
        and (torch._C._len_torch_function_stack() == 0 or _only_default_devices()) \
        and torch._C._functorch.peek_interpreter_stack() is None \
        and not torch._C._functorch.is_legacy_batchedtensor(x) \
        and torch.autograd.forward_ad._current_level < 0 \
        and (not torch.is_autocast_enabled("cuda") or torch.get_autocast_dtype("cuda") == torch.bfloat16)


_capturing = torch._C._cuda_isCurrentStreamCapturing   # (torch.cuda's own form costs twice as much)


def _version(t: torch.Tensor):
    """The tensor's in-place modification counter, or ``None`` where torch keeps none (inference tensors)."""
    try:
        return t._version
    except RuntimeError:
        return None


def _source_state(*tensors):
    """What identifies the tensors a prepacked copy was made from: a weak reference to each, its
    modification counter and, for a tensor torch keeps no counter for (an inference tensor), the address
    and shape of its data instead.  In-place writes to such a tensor go unnoticed: ``prepack_()`` again
    after editing int4 buffers that were created under ``torch.inference_mode``."""
    return tuple((weakref.ref(t), _version(t), (t.data_ptr(), tuple(t.shape))) for t in tensors)


def _versions(a: torch.Tensor, b: torch.Tensor, c: torch.Tensor):
    try:
        return a._version, b._version, c._version
    except RuntimeError:      # an inference tensor among them
        return _version(a), _version(b), _version(c)


def _source_changed(state, *tensors) -> bool:
    for t, (ref, v0, where) in zip(tensors, state):
        if ref() is not t:
            return True
        if v0 is None:
            if (t.data_ptr(), tuple(t.shape)) != where:
                return True
        elif _version(t) != v0:
            return True
    return False


def _rows(x: torch.Tensor, in_features: int) -> torch.Tensor:
    if x.dtype != torch.bfloat16:
        raise TypeError(f"Int4Linear runs in bfloat16 like the policy it replaces, got {x.dtype}")
    if x.shape[-1] != in_features:
        raise ValueError(f"last dimension {x.shape[-1]} != in_features {in_features}")
    return x if x.dim() == 2 and x.is_contiguous() else x.reshape(-1, in_features).contiguous()


class Int4Linear(nn.Module):
    """int4 weight-only linear: ``y = x . dequant(qweight, scales, qzeros)^T (+ bias)``.

    Buffers (saved in ``state_dict``): ``qweight`` int32 ``[N, K/8]``, ``scales`` bf16
    ``[N, K/G]``, ``qzeros`` int32 ``[N, ceil(K/G/8)]``, optional ``bias`` bf16 ``[N]``.
    """

    def __init__(self, in_features: int, out_features: int, group_size: int = 128,
                 bias: bool = False, device=None):
        super().__init__()
        if group_size % 8 != 0 or in_features % group_size != 0:
            raise ValueError("group_size must be a multiple of 8 that divides in_features")
        self.in_features = int(in_features)
        self.out_features = int(out_features)
        self.group_size = int(group_size)
        groups = in_features // group_size
        self.register_buffer("qweight", torch.zeros((out_features, in_features // 8),
                                                    dtype=torch.int32, device=device))
        self.register_buffer("scales", torch.ones((out_features, groups), dtype=torch.bfloat16,
                                                  device=device))
        self.register_buffer("qzeros", torch.zeros((out_features, (groups + 7) // 8),
                                                   dtype=torch.int32, device=device))
        if bias:
            self.register_buffer("bias", torch.zeros(out_features, dtype=torch.bfloat16, device=device))
        else:
            self.bias = None

    @classmethod
    def from_packed(cls, qweight, scales, qzeros, group_size: int, bias=None) -> "Int4Linear":
        N, K, _ = check_packed(qweight, scales, qzeros, group_size)
        mod = cls(K, N, group_size, bias=bias is not None, device=qweight.device)
        mod.qweight, mod.scales, mod.qzeros = qweight.contiguous(), scales.contiguous(), qzeros.contiguous()
        if bias is not None:
            mod.bias = bias.detach().to(torch.bfloat16).contiguous()
        return mod

    @classmethod
    def from_linear(cls, linear: nn.Linear, group_size: int = 128) -> "Int4Linear":
        """Quantise an ``nn.Linear`` (min/max, asymmetric, per K-group) on its own device."""
        qweight, scales, qzeros = quantize_minmax(linear.weight.data, group_size)
        return cls.from_packed(qweight, scales, qzeros, group_size,
                               None if linear.bias is None else linear.bias.data)

    @classmethod
    def from_unpacked_zeros(cls, qweight, scales, zeros_u8, group_size: int, bias=None):
        """Accepts zero-points as an unpacked ``uint8 [N, K/G]`` tensor and packs them."""
        return cls.from_packed(qweight, scales, pack_nibbles(zeros_u8.to(torch.int32)), group_size, bias)

    def prepack_(self) -> "Int4Linear":
        """Keep a prepacked copy of the weight for decode-sized calls (a second copy in HBM).

        Calls with few activation rows then go through the plan-free launch over the
        MFMA-shaped blob; larger ones, and ``torch.compile``, keep using the canonical
        buffers, which stay the module's ``state_dict``.  No-op if the shape has no prepacked form.
        """
        self._packed = None
        if self.qweight.is_cuda and ops.PrepackedWeight.supported(self.out_features, self.in_features,
                                                                  self.group_size):
            self._packed = ops.int4_prepack(self.qweight, self.scales, self.qzeros, self.group_size)
            self._packed_from = _source_state(self.qweight, self.scales, self.qzeros)
            self._direct_rows = self._packed.direct_rows()
            self._call = ops.DirectCall([self._packed])
        group = getattr(self, "_group", None)
        if group is not None:  # rebuild the group's launch over the new copies
            self.group_with(*group[1:])
        leader = getattr(self, "_leader", None)
        leader = leader() if leader is not None else None   # the module whose launch computes this one's output too
        if leader is not None and leader is not self and getattr(leader, "_group", None) is not None:
            leader.group_with(*leader._group[1:])
        return self

    def packed_is_stale(self) -> bool:
        """True when the canonical buffers were written (``load_state_dict``, an in-place edit) or
        replaced (``.to()``) after :meth:`prepack_` copied them."""
        return getattr(self, "_packed", None) is not None and \
            _source_changed(self._packed_from, self.qweight, self.scales, self.qzeros)

    def _fresh_packed(self):
        """The prepacked copy, made again first if the canonical buffers changed under it."""
        packed = self.__dict__.get("_packed")
        if packed is not None and _source_changed(self._packed_from, *self._canonical()):
            if self.qweight.is_cuda and torch.cuda.is_current_stream_capturing():
                raise RuntimeError("the int4 weight changed after prepack_(): call prepack_() again before "
                                   "recording a graph over this module")
            self.prepack_()
            packed = self._packed
        return packed

    def group_with(self, *others: "Int4Linear") -> "Int4Linear":
        """Launch ``others`` together with this module whenever it is called (q|k|v of one layer).

        Modules that are applied to the same input one after the other, as
        ``LlamaAttention`` applies ``q_proj``, ``k_proj``, ``v_proj`` to ``hidden_states``
        (reached from ``vrl/models/families/janus_pro/policy.py:673-678``): a decode-sized call
        of this module computes all of them in one plan-free launch and hands each sibling its
        result, which the sibling returns when it is called with the very same tensor object
        next.  Needs ``prepack_()`` on every member; anything else falls back to one launch each.
        Prompt-sized calls, with and without a gradient, share a launch the same way over the canonical
        buffers, where that is the faster route and every member has ``PROMPT_COLUMNS`` outputs; a caller
        that wants the leader's result alone pays for the siblings' too.
        """
        if len(others) + 1 > ops.DirectGemv.MAX_PROBLEMS:
            raise ValueError(f"at most {ops.DirectGemv.MAX_PROBLEMS} modules per group")
        if any(o.in_features != self.in_features for o in others):
            raise ValueError("grouped modules take the same input")
        self._group = (self, *others)
        for m in others:
            m._leader = weakref.ref(self)
        self._group_call = None
        if all(getattr(m, "_packed", None) is not None for m in self._group):
            self._group_call = ops.DirectCall([m._packed for m in self._group])
        return self

    def dequantize(self) -> torch.Tensor:
        """The canonical bf16 weight ``[N, K]`` (bit-exact tile), e.g. for the train-time replay."""
        return ops.int4_dequant(self.qweight, self.scales, self.qzeros, self.group_size)

    def keep_dense_(self, keep: bool = True) -> "Int4Linear":
        """Keep the dequantised bf16 weight between calls (2 bytes per weight beside the 0.56 of the int4
        buffers): prompt-sized calls and the train-time replay (``policy.py:419-424``: one forward per
        micro-batch) then multiply by the kept tensor instead of rebuilding it every call.  It is rebuilt
        when the canonical buffers were written or replaced since; ``keep=False`` drops it.  These are library
        products at every size: where a module without the copy takes the prompt launch its results differ by the
        order of fp32 sums, and by the rounding of gate and up before SiLU."""
        self._keep_dense = bool(keep)
        self._dense = None
        return self

    def _dense_weight(self, x: torch.Tensor) -> torch.Tensor:
        """The bf16 weight for a library GEMM over ``x``: the kept copy if there is one and it is current."""
        if not getattr(self, "_keep_dense", False):
            dequant = ops.dequant_eager if _launchable(x) else ops.int4_dequant
            return dequant(*self._canonical(), self.group_size)
        kept = getattr(self, "_dense", None)
        if kept is None or _source_changed(kept[0], self.qweight, self.scales, self.qzeros):
            kept = (_source_state(self.qweight, self.scales, self.qzeros),
                    ops.int4_dequant(self.qweight, self.scales, self.qzeros, self.group_size))
            self._dense = kept
        return kept[1]

    def _canonical(self):
        buffers = self._buffers   # (looked up through the module, a buffer costs three times as much)
        try:
            return buffers["qweight"], buffers["scales"], buffers["qzeros"]
        except KeyError:          # replaced by plain attributes
            return self.qweight, self.scales, self.qzeros

    def _prompt_gemm(self, x: torch.Tensor, rows: torch.Tensor):
        """A prompt-sized call as one launch, or ``None`` where the general route is the better or only one."""
        M, K, G = rows.shape[0], self.in_features, self.group_size
        if M > PROMPT_ROWS or self.out_features < PROMPT_COLUMNS or getattr(self, "_keep_dense", False) or \
                not _launchable(x):
            return None
        group = self.__dict__.get("_group")
        version = _version(x) if group is not None else None
        if version is not None:
            columns = 0
            for m in group:
                if m.group_size != G or m.out_features < PROMPT_COLUMNS or m.__dict__.get("_keep_dense", False):
                    break
                columns += m.out_features
            else:
                if _launch_pays(M, K, columns, G, len(group)):
                    weights = [m._canonical() for m in group]
                    ys = ops.int4_gemm(rows, weights, G)
                    if ys is not None:
                        # (x by weak reference: with a gradient it would keep what led to it alive)
                        call = weakref.ref(x), version, ops._stream_handle(x.device), _capturing()
                        for m, ym, weight in zip(group[1:], ys[1:], weights[1:]):
                            m.__dict__["_handed"] = (call, ym, [weakref.ref(t) for t in weight], _versions(*weight))
                        return ys[0]
        if not _launch_pays(M, K, self.out_features, G):
            return None
        ys = ops.int4_gemm(rows, [self._canonical()], G)
        return None if ys is None else ys[0]

    def _take(self, handed, x: torch.Tensor, grad: bool):
        """The handed result if it is this call's: of this very tensor, unchanged since, on this stream."""
        if len(handed) == 3:   # from a decode-sized launch
            return handed[2] if not grad and handed[0] is x and handed[1] == _version(x) else None
        (ref, version, stream, capturing), y, (qweight, scales, qzeros), versions = handed
        if ref() is not x or version != _version(x) or stream != ops._stream_handle(x.device) or \
                capturing != _capturing() or grad and not _launchable(x):
            return None
        mine = self._canonical()
        return y if mine[0] is qweight() and mine[1] is scales() and mine[2] is qzeros() and \
            versions == _versions(*mine) else None

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        rows = _rows(x, self.in_features)
        if torch.compiler.is_compiling():
            y = ops.int4_gemv(rows, self.qweight, self.scales, self.qzeros, self.group_size)
            return self._finish(y, x, rows)
        own = self.__dict__   # plain attributes: nn.Module's own lookups and assignments cost microseconds
        handed = own.get("_handed")
        if handed is not None:
            handed = own.pop("_handed", None)   # (one of two threads gets it)
            own["_handed"] = None
        group = own.get("_group")
        if group is not None:   # a new call of the leader: whatever it handed over before is void
            for m in group[1:]:
                m.__dict__["_handed"] = None
        grad = _wants_grad(x)
        y = None if handed is None else self._take(handed, x, grad)   # computed by the group leader's launch
        if grad:   # the same product as without a gradient, bit for bit, at every prompt size
            weight = self._dense_weight(x)
            if y is None and rows.shape[0] > GEMM_ROWS:
                y = self._prompt_gemm(x, rows)
            y = F.linear(rows, weight) if y is None else _Launched.apply(rows, [y], weight)
        elif y is None:  # eager decode: skip the operator dispatcher, it costs more than the kernel
            packed = self._fresh_packed()
            M = rows.shape[0]
            if packed is not None and packed.blob.device == rows.device:
                call = own.get("_group_call")
                version = _version(x) if call is not None else None
                if call is not None and M <= call.max_rows and version is not None and \
                        not any(m.packed_is_stale() for m in group[1:]):
                    # (an input without a modification counter cannot be recognised later: no hand-over)
                    ys = call(rows)
                    for m, ym in zip(group[1:], ys[1:]):
                        m.__dict__["_handed"] = (x, version, ym)
                    y = ys[0]
                elif M <= self._direct_rows:
                    y = self._call(rows)[0]
                else:
                    packed = None
            else:
                packed = None
            if packed is None and M > GEMM_ROWS:
                # prompt-sized call: the GEMV kernels would stream the weight once per 16 rows
                y = self._prompt_gemm(x, rows)
                if y is None:
                    y = F.linear(rows, self._dense_weight(x))
            elif packed is None:
                y = torch.empty((M, self.out_features), dtype=torch.bfloat16, device=rows.device)
                ops.int4_gemv_into(y, rows, self.qweight, self.scales, self.qzeros, self.group_size)
        return self._finish(y, x, rows)

    def _finish(self, y: torch.Tensor, x: torch.Tensor, rows: torch.Tensor) -> torch.Tensor:
        if self.bias is not None:
            y = y + self.bias
        return y if rows is x else y.reshape(*x.shape[:-1], self.out_features)

    def extra_repr(self) -> str:
        return (f"in_features={self.in_features}, out_features={self.out_features}, "
                f"group_size={self.group_size}, bias={self.bias is not None}")


def _silu_mul_ops(gate_up: torch.Tensor) -> torch.Tensor:
    gate, up = gate_up.chunk(2, dim=-1)
    return F.silu(gate) * up


class _Launched(torch.autograd.Function):
    """What a launch computed from ``rows`` (handed in as a list, or it would count as an input), with the gradient
    of ``rows . weight^T``: that of ``F.linear``, whose node saves the weight too."""

    @staticmethod
    def forward(ctx, rows, result, weight):
        ctx.save_for_backward(weight)
        return result[0]

    @staticmethod
    def backward(ctx, grad):
        weight, = ctx.saved_tensors
        if torch.is_autocast_enabled("cuda"):   # a backward called under it: the product's type is the forward's
            with torch.autocast("cuda", enabled=False):
                return grad @ weight, None, None
        return grad @ weight, None, None


class _SiLUMul(torch.autograd.Function):
    """``silu(gate) * up`` with its gradient as one launch each; only the product itself is saved.  ``result``: a
    list that holds the value where a launch has computed it with the product.  A backward that is itself recorded,
    or watched by a transform, goes through the torch operators."""

    @staticmethod
    def forward(ctx, gate_up, result):
        ctx.save_for_backward(gate_up)
        return result[0] if result else ops.silu_mul(gate_up)

    @staticmethod
    def backward(ctx, grad):
        gate_up, = ctx.saved_tensors
        if torch.is_grad_enabled() or gate_up.shape[-1] % 16 or not (_launchable(grad) and _launchable(gate_up)):
            recorded = torch.is_grad_enabled()
            with torch.enable_grad():
                return torch.autograd.grad(_silu_mul_ops(gate_up), gate_up, grad, create_graph=recorded)[0], None
        # (a saved-tensor hook may have made a view)
        return ops.silu_mul_backward(_aligned(gate_up), _aligned(grad)), None


def _aligned(t: torch.Tensor) -> torch.Tensor:
    """``t`` itself if it is contiguous and starts on a 16-byte boundary, a copy otherwise."""
    t = t.contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


def _silu_mul(gate_up: torch.Tensor) -> torch.Tensor:
    inter = gate_up.shape[-1] // 2
    if not _launchable(gate_up) or gate_up.dtype != torch.bfloat16 or inter < PROMPT_COLUMNS or inter % 8 != 0 \
            or not 0 < gate_up.numel() < 2 ** 31 or not gate_up.is_contiguous() or gate_up.data_ptr() % 16 != 0:
        return _silu_mul_ops(gate_up)
    return _SiLUMul.apply(gate_up, None) if _wants_grad(gate_up) else ops.silu_mul(gate_up)


class Int4GateUpSiLU(nn.Module):
    """Fused ``silu(gate_proj(x)) * up_proj(x)`` over one packed gate||up operand."""

    def __init__(self, gate: Int4Linear, up: Int4Linear):
        super().__init__()
        if (gate.in_features, gate.out_features, gate.group_size) != \
                (up.in_features, up.out_features, up.group_size):
            raise ValueError("gate_proj and up_proj must have the same shape and group size")
        if gate.bias is not None or up.bias is not None:
            raise ValueError("the fused gate/up operator takes bias-free projections")
        self.in_features = gate.in_features
        self.intermediate_size = gate.out_features
        self.group_size = gate.group_size
        self.register_buffer("qweight", torch.cat([gate.qweight, up.qweight], dim=0).contiguous())
        self.register_buffer("scales", torch.cat([gate.scales, up.scales], dim=0).contiguous())
        self.register_buffer("qzeros", torch.cat([gate.qzeros, up.qzeros], dim=0).contiguous())

    def prepack_(self) -> "Int4GateUpSiLU":
        """Keep a prepacked copy of gate||up for decode-sized calls (see ``Int4Linear.prepack_``)."""
        self._packed = None
        if self.qweight.is_cuda and self.intermediate_size % 16 == 0 and \
                ops.PrepackedWeight.supported(2 * self.intermediate_size, self.in_features, self.group_size):
            self._packed = ops.int4_prepack(self.qweight, self.scales, self.qzeros, self.group_size)
            self._packed_from = _source_state(self.qweight, self.scales, self.qzeros)
            self._direct_rows = self._packed.direct_rows(fused=True)
            self._call = ops.DirectCall([self._packed], fused=True)
        return self

    def _prompt_gemm(self, x: torch.Tensor, rows: torch.Tensor, grad: bool):
        """A prompt-sized call as one launch, or ``None`` where the general route is the better or only one."""
        M = rows.shape[0]
        if M <= GEMM_ROWS or self.intermediate_size < PROMPT_COLUMNS or getattr(self, "_keep_dense", False) or \
                not _launchable(x) or \
                not _launch_pays(M, self.in_features, 2 * self.intermediate_size, self.group_size, fused=True):
            return None
        products = [] if grad else None
        ys = ops.int4_gemm(rows, [self._canonical()], self.group_size, True, products)
        if ys is None or not grad:
            return None if ys is None else ys[0]
        return _SiLUMul.apply(_Launched.apply(rows, products, self._dense_weight(x)), ys)

    _canonical = Int4Linear._canonical
    packed_is_stale = Int4Linear.packed_is_stale
    _fresh_packed = Int4Linear._fresh_packed
    keep_dense_ = Int4Linear.keep_dense_
    _dense_weight = Int4Linear._dense_weight

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        rows = _rows(x, self.in_features)
        packed = None if torch.compiler.is_compiling() else self._fresh_packed()
        grad = _wants_grad(x) and not torch.compiler.is_compiling()
        if packed is not None and not grad and not torch.compiler.is_compiling() \
                and rows.shape[0] <= self._direct_rows and packed.blob.device == rows.device:
            y = self._call(rows)[0]
        elif not torch.compiler.is_compiling() and (launched := self._prompt_gemm(x, rows, grad)) is not None:
            y = launched
        elif (grad or rows.shape[0] > GEMM_ROWS) and not torch.compiler.is_compiling():
            y = _silu_mul(F.linear(rows, self._dense_weight(x)))   # prompt-sized call: one library GEMM
        else:
            y = ops.int4_gate_up_silu(rows, self.qweight, self.scales, self.qzeros, self.group_size)
        return y if rows is x else y.reshape(*x.shape[:-1], self.intermediate_size)


class Int4LlamaMLP(nn.Module):
    """``down_proj(silu(gate_proj(x)) * up_proj(x))`` with both halves in int4.

    Built from a Hugging Face ``LlamaMLP``-shaped module (attributes ``gate_proj``,
    ``up_proj``, ``down_proj``; SiLU activation).
    """

    def __init__(self, mlp: nn.Module, group_size: int = 128):
        super().__init__()
        act = getattr(mlp, "act_fn", None)
        if act is not None and not isinstance(act, nn.SiLU) and \
                getattr(act, "__name__", type(act).__name__).lower() not in ("silu", "siluactivation"):
            raise ValueError(f"fused MLP needs a SiLU activation, found {act!r}")
        as_int4 = lambda m: m if isinstance(m, Int4Linear) else Int4Linear.from_linear(m, group_size)
        self.gate_up = Int4GateUpSiLU(as_int4(mlp.gate_proj), as_int4(mlp.up_proj))
        self.down_proj = as_int4(mlp.down_proj)

    def prepack_(self) -> "Int4LlamaMLP":
        self.gate_up.prepack_()
        self.down_proj.prepack_()
        return self

    def keep_dense_(self, keep: bool = True) -> "Int4LlamaMLP":
        self.gate_up.keep_dense_(keep)
        self.down_proj.keep_dense_(keep)
        return self

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return self.down_proj(self.gate_up(x))
