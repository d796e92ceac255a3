"""Drop-in mixture-of-experts feed-forward network running on gfx950 kernels.

:class:`MoE` keeps the constructor, attribute names, parameter names/shapes and
``forward(seqs)`` contract of fairseq2's ``MoE``
(``src/fairseq2/models/llama4/moe.py:21-157``), so a fairseq2 decoder layer
(``models/transformer_lm/decoder_layer.py:194``) can call it unchanged and a
reference checkpoint loads with ``load_state_dict``.  The forward pass is four
device stages behind a C ABI: router + top-k, dispatch, grouped SwiGLU experts
(+ the optional shared expert) and combine.  It runs on the GPU only; there is no
torch-operator fallback.  With inputs or parameters that require a gradient the
layer runs as one ``torch.autograd.Function`` whose backward pass uses the same
library (:mod:`fairseq2_amd.autograd`).

Keyword-only extensions (defaults reproduce the reference):

``score_fn``      ``"sigmoid"`` (reference) or ``"softmax"``
``renormalize``   divide the K weights by their sum
``scale_on``      ``"input"`` (reference: scale the expert input) or ``"output"``
``router_bias``   add a learnable-free per-expert f32 bias to the router logits
``tile_m``        row granularity each expert's block is padded to
"""

from __future__ import annotations

import math
from abc import ABC, abstractmethod

import torch
import torch.nn as nn
from torch import Tensor
from torch.nn import Module, Parameter

from fairseq2_amd import _abi
from fairseq2_amd import ops as _ops  # noqa: F401  (registers torch.ops.fairseq2_amd.moe_forward)


class FeedForwardNetwork(Module, ABC):
    """Transformer feed-forward network interface (``models/transformer/ffn.py:25-39``)."""

    @abstractmethod
    def forward(self, seqs: Tensor) -> Tensor:
        """``seqs`` is ``(N, S, M)``; the result has the same shape."""


def _require_forward_only(*tensors: Tensor | None) -> None:
    if torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in tensors):
        raise RuntimeError(
            "this fairseq2_amd module is forward-only: call it under torch.no_grad() / "
            "torch.inference_mode(), or freeze the module with requires_grad_(False)"
        )


def _require_device(t: Tensor) -> None:
    if not t.is_cuda:
        raise RuntimeError(
            f"fairseq2_amd kernels run on the GPU only, got a tensor on {t.device} "
            "(there is no CPU fallback)"
        )


def _held(module: Module, name: str) -> Tensor:
    """``getattr(module, name)`` of a parameter, past ``Module.__getattr__`` (0.5 us of host time each, of
    three to nine a call) where the module holds it; one that is computed on access is not held."""
    p = module._parameters.get(name)
    return getattr(module, name) if p is None else p


def _part(module: Module, name: str) -> Module:
    """The same of a submodule."""
    m = module._modules.get(name)
    return getattr(module, name) if m is None else m


def _optional(obj, name: str):
    """``getattr(obj, name, None)``; a module that has nothing of the name takes 0.8 us to say so through an
    exception."""
    if isinstance(obj, Module):
        for held in (obj._parameters, obj._buffers, obj._modules):
            if name in held:
                return held[name]
        cls = type(obj)
        if name not in obj.__dict__ and cls.__getattr__ is Module.__getattr__ and not hasattr(cls, name):
            return None
    return getattr(obj, name, None)


class ExpertNetwork(Module, ABC):
    """Interface of an expert bank (``models/transformer/experts.py:117-154``)."""

    def __init__(self, num_experts: int, model_dim: int, inner_dim: int) -> None:
        super().__init__()
        self.num_experts = num_experts
        self.model_dim = model_dim
        self.inner_dim = inner_dim

    @abstractmethod
    def forward(self, x: Tensor) -> Tensor:
        """``x``: (num_local_experts, tokens_per_expert, dim) -> same shape."""

    @property
    def num_local_experts(self) -> int:
        return self.num_experts

    def extra_repr(self) -> str:
        return f"num_experts={self.num_experts}, model_dim={self.model_dim}, inner_dim={self.inner_dim}"


class GroupedExpertNetwork(ExpertNetwork):
    """SwiGLU experts with the expert dimension folded into dim 0 of the weights
    (``experts.py:24-87,157-213``): ``gate_proj``/``inner_proj`` are ``(E*D, F)``,
    ``output_proj`` is ``(E*F, D)``, all "in x out".  Like the reference, the
    parameters are left uninitialised; a checkpoint is expected to fill them.
    """

    def __init__(
        self,
        num_experts: int,
        model_dim: int,
        inner_dim: int,
        *,
        activation: Module | None = None,
        device: torch.device | None = None,
        dtype: torch.dtype | None = None,
    ) -> None:
        super().__init__(num_experts, model_dim, inner_dim)
        kw = dict(device=device, dtype=dtype)
        self.gate_proj = Parameter(torch.empty((num_experts * model_dim, inner_dim), **kw))
        self.inner_proj = Parameter(torch.empty((num_experts * model_dim, inner_dim), **kw))
        self.output_proj = Parameter(torch.empty((num_experts * inner_dim, model_dim), **kw))
        # Any module, as in the reference (experts.py:84-87).  The fused kernels implement the SiLU
        # gate; another activation runs between plain grouped GEMMs of the same library.
        self.activation = activation if activation is not None else nn.SiLU()
        # Opt-in (no counterpart in the reference): "mxfp8" rounds the inputs of the expert products
        # to block-scaled e4m3 so that, with e4m3 weights, they run on the fp8 matrix pipe (W8A8).
        self.act_quant: str | None = None

    @property
    def has_fused_gate(self) -> bool:
        return isinstance(_part(self, "activation"), nn.SiLU)

    # Rows go to the fp8 matrix pipe from this many per expert on (mean over all experts; the library
    # takes its bf16-pipe GEMMs for e4m3 weights from 27 on); below that the experts are a weight
    # stream, which activations of one byte would not make faster.
    _W8A8_MIN_ROWS_PER_EXPERT = 32

    def runs_w8a8(self, act_dtype: torch.dtype, rows: int) -> bool:
        """Whether :meth:`forward_rows` on ``rows`` rows takes the fp8 matrix pipe."""
        return (
            self.act_quant == "mxfp8" and self.has_fp8_weights and self.has_fused_gate
            and act_dtype == torch.bfloat16
            and rows // self.num_local_experts >= self._W8A8_MIN_ROWS_PER_EXPERT
            and _abi.w8a8_supported(self.model_dim, self.inner_dim, rows)
        )

    # ---- fp8 (e4m3) weights: derived, non-persistent buffers next to the Parameters ----------------
    # Stored as integers (codes as uint8, scales as the int32 bit patterns of their f32 values) so
    # that Module.to(dtype) / .float() / .bfloat16(), which cast every floating-point buffer, leave
    # them alone; the properties below hand out the typed views the kernels take.
    _FP8_NAMES = ("gate_q", "inner_q", "output_q", "gate_scale", "inner_scale", "output_scale")

    @property
    def has_fp8_weights(self) -> bool:
        return self._buffers.get("_gate_q_bits") is not None

    def clear_fp8_weights(self) -> None:
        """Drops the derived e4m3 buffers: the next forward uses the Parameters again."""
        for name in self._FP8_NAMES:
            if hasattr(self, f"_{name}_bits"):
                delattr(self, f"_{name}_bits")
        self.__dict__.pop("_fp8_view_cache", None)

    def _fp8_view(self, name: str) -> Tensor:
        bits = getattr(self, f"_{name}_bits")
        # the typed view is kept for as long as the buffer object stays the same (a view costs a few
        # microseconds of host time, and a decode step takes six of them per layer); Module.to(),
        # load_fp8_weights and clear_fp8_weights all install new buffer objects
        # (not while a compiler traces the call: the view is then part of the trace)
        tracing = torch.compiler.is_compiling()
        if not tracing:
            cache = self.__dict__.get("_fp8_view_cache")
            if cache is None:
                cache = self.__dict__["_fp8_view_cache"] = {}
            hit = cache.get(name)
            if hit is not None and hit[0] is bits:
                return hit[1]
        want = torch.uint8 if name.endswith("_q") else torch.int32
        if bits.dtype != want:
            raise RuntimeError(f"the fp8 buffer {name} was cast to {bits.dtype}; quantise again")
        view = bits.view(torch.float8_e4m3fn if name.endswith("_q") else torch.float32)
        if not tracing:
            cache[name] = (bits, view)
        return view

    gate_q = property(lambda self: self._fp8_view("gate_q"))
    inner_q = property(lambda self: self._fp8_view("inner_q"))
    output_q = property(lambda self: self._fp8_view("output_q"))
    gate_scale = property(lambda self: self._fp8_view("gate_scale"))
    inner_scale = property(lambda self: self._fp8_view("inner_scale"))
    output_scale = property(lambda self: self._fp8_view("output_scale"))

    def _fp8_operands(self) -> tuple[tuple[Tensor, ...], tuple[Tensor, ...]]:
        """The typed codes and scales (gate, inner, output each), looked up together: 1 us where the six
        properties take 4."""
        cache, buffers = self.__dict__.get("_fp8_view_cache"), self._buffers
        if cache is not None and len(cache) == 6 and not torch.compiler.is_compiling():
            views = [hit[1] for name, hit in cache.items() if buffers.get(f"_{name}_bits") is hit[0]]
            if len(views) == 6:
                g, i, o, gs, is_, os_ = (cache[name][1] for name in self._FP8_NAMES)
                return (g, i, o), (gs, is_, os_)
        return (self.gate_q, self.inner_q, self.output_q), (self.gate_scale, self.inner_scale, self.output_scale)

    def _load_from_state_dict(self, state_dict, prefix, *args, **kwargs):
        # new Parameters make the derived codes stale
        if any(k.startswith(prefix) for k in state_dict):
            self.clear_fp8_weights()
        super()._load_from_state_dict(state_dict, prefix, *args, **kwargs)

    def load_fp8_weights(self, gate_q, gate_scale, inner_q, inner_scale, output_q, output_scale):
        """Installs pre-quantised weights.  Codes are ``float8_e4m3fn`` in the reference orientation
        (``(E*D, F)``, ``(E*D, F)``, ``(E*F, D)``), scales are f32 per expert and output channel
        (``(E, F)``, ``(E, F)``, ``(E, D)``).  The kernel streams 1 KB tiles of 16 output channels x
        64 input features, so the codes are re-tiled once here."""
        e, d, f = self.num_local_experts, self.model_dim, self.inner_dim
        dev = self.gate_proj.device

        def codes(q, k, n):
            if q.dtype != torch.float8_e4m3fn or tuple(q.shape) != (e * k, n):
                raise ValueError(f"fp8 codes must be float8_e4m3fn of shape ({e * k}, {n})")
            return _abi.pack_fp8_weights(q.to(dev), e)

        def scale(s, n):
            if tuple(s.shape) != (e, n):
                raise ValueError(f"fp8 scales must have shape ({e}, {n})")
            return s.to(device=dev, dtype=torch.float32).contiguous()

        for name, val in zip(
            self._FP8_NAMES,
            (codes(gate_q, d, f), codes(inner_q, d, f), codes(output_q, f, d),
             scale(gate_scale, f), scale(inner_scale, f), scale(output_scale, d)),
        ):
            bits = val.view(torch.uint8) if name.endswith("_q") else val.view(torch.int32)
            self.register_buffer(f"_{name}_bits", bits, persistent=False)

    @torch.no_grad()
    def quantize_fp8_(self) -> None:
        """Quantises the current Parameters per expert and output channel:
        ``scale = max_k |W| / 448`` (e4m3 saturates at 448 and torch's cast does not clamp)."""
        e, d, f = self.num_local_experts, self.model_dim, self.inner_dim

        def q(w, k, n):
            w3 = w.detach().float().view(e, k, n)
            s = (w3.abs().amax(dim=1) / 448.0).clamp_min(torch.finfo(torch.float32).tiny)
            codes = (w3 / s[:, None, :]).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
            return codes.view(e * k, n), s

        gq, gs = q(self.gate_proj, d, f)
        uq, us = q(self.inner_proj, d, f)
        dq, ds = q(self.output_proj, f, d)
        self.load_fp8_weights(gq, gs, uq, us, dq, ds)

    def fuses_gather(self, act_dtype: torch.dtype, max_rows: int = 0) -> bool:
        """Whether :meth:`forward_rows` can read ``max_rows`` rows through a row map from the token
        matrix (no gathered copy needed)."""
        if not self.has_fused_gate:
            return False
        if self.has_fp8_weights:
            return _abi.fuses_gather(self.model_dim, self.inner_dim, act_dtype, torch.float8_e4m3fn)
        # the bf16 kernel addresses its activation matrices with 32-bit byte offsets
        if max_rows * max(self.model_dim, self.inner_dim) * 2 > 0xFFFFFFFF:
            return False
        return _abi.fuses_gather(self.model_dim, self.inner_dim, act_dtype, self.gate_proj.dtype)

    def forward_rows(
        self, xe: Tensor, counts: Tensor, offsets: Tensor, row_map: Tensor | None = None,
        rows_per_expert: int = 0, pairs: int = 0,
    ) -> Tensor:
        """Runs every expert on its block of rows of ``xe`` (rows, D); with ``row_map``, row ``r``
        is ``xe[row_map[r]]`` and ``xe`` is the token matrix.  ``rows_per_expert``: an upper bound
        on any expert's rows when the caller knows one (the number of tokens is one), else 0; up to 16
        the bf16 experts run as streams over their weights.  ``pairs``: how many rows the experts have in
        all when the caller knows it, else 0: the kernels are then chosen by it.  Inference only (the training paths are
        :meth:`forward` and the layer's)."""
        _require_forward_only(xe, self.gate_proj, self.inner_proj, self.output_proj)
        if not self.has_fused_gate:
            # experts.py:107-112 with the module's own activation between the library's GEMMs
            if self.has_fp8_weights or row_map is not None:
                raise NotImplementedError("e4m3 weights and the fused gather need the SiLU gate")
            grp = dict(counts=counts, offsets=offsets, num_experts=self.num_local_experts)
            # (in f32 with one rounding, like the fused SiLU gate; the training path does the same)
            g = _abi.grouped_gemm(xe, self.gate_proj.detach(), _abi.W_IN_OUT, **grp)
            u = _abi.grouped_gemm(xe, self.inner_proj.detach(), _abi.W_IN_OUT, **grp)
            h = (self.activation(g.float()) * u.float()).to(xe.dtype)
            return _abi.grouped_gemm(h.contiguous(), self.output_proj.detach(), _abi.W_IN_OUT, **grp)
        rows = xe.shape[0] if row_map is None else row_map.shape[0]
        if self.runs_w8a8(xe.dtype, rows):
            # the rows (the token matrix when they are read through a map) to block-scaled e4m3,
            # then both products on the fp8 matrix pipe
            xq, xs = _abi.mx_quantize(xe)
            ye, _, _ = _abi.grouped_swiglu_w8a8(
                xq, xs, counts, offsets, self.gate_q, self.inner_q, self.output_q,
                (self.gate_scale, self.inner_scale, self.output_scale), self.num_local_experts,
                row_map=row_map,
            )
            return ye
        if self.has_fp8_weights:
            ye, _ = _abi.grouped_swiglu(
                xe, counts, offsets, self.gate_q, self.inner_q, self.output_q,
                self.num_local_experts,
                scales=(self.gate_scale, self.inner_scale, self.output_scale), row_map=row_map, pairs=pairs,
            )
            return ye
        ye, _ = _abi.grouped_swiglu(
            xe, counts, offsets, self.gate_proj.detach(), self.inner_proj.detach(),
            self.output_proj.detach(), self.num_local_experts, row_map=row_map,
            rows_per_expert=rows_per_expert, pairs=pairs,
        )
        return ye

    def forward(self, x: Tensor) -> Tensor:
        """The reference's dense calling convention: every expert gets the same
        number of rows (``experts.py:201-213``)."""
        _require_device(x)
        e, n, d = x.shape
        if e != self.num_local_experts or d != self.model_dim:
            raise ValueError(f"expected ({self.num_local_experts}, *, {self.model_dim}), got {tuple(x.shape)}")
        counts, offsets = self._uniform_groups(n, x.device)
        params = (self.gate_proj, self.inner_proj, self.output_proj)
        if torch.is_grad_enabled() and any(t.requires_grad for t in (x, *params)):
            # training: the experts alone as one autograd function on the library's backward kernels
            if self.has_fp8_weights:
                raise RuntimeError("fairseq2_amd: e4m3 expert weights are an inference format")
            if not self.has_fused_gate and any(p.requires_grad for p in self.activation.parameters()):
                raise RuntimeError("fairseq2_amd: a gate activation with parameters of its own is not differentiated")
            if n == 0:
                return torch.empty_like(x)
            from fairseq2_amd.autograd import GroupedExpertsFunction

            ye = GroupedExpertsFunction.apply(
                x.reshape(e * n, d).contiguous(), counts, offsets, *params, e,
                None if self.has_fused_gate else self.activation, n if n <= 16 else 0)
            return ye.view(e, n, d)
        # (every expert has exactly n rows: a bound the library can use when it is small)
        return self.forward_rows(x.reshape(e * n, d).contiguous(), counts, offsets,
                                 **self._row_hints(n if n <= 16 else 0, e * n)).view(e, n, d)

    def _row_hints(self, rows_per_expert: int, pairs: int) -> dict[str, int]:
        """What is known of the rows, for :meth:`forward_rows` (an override of it may not take ``pairs``)."""
        hints = {"rows_per_expert": rows_per_expert} if rows_per_expert else {}
        if type(self).forward_rows is GroupedExpertNetwork.forward_rows:
            hints["pairs"] = pairs
        return hints

    def _uniform_groups(self, n: int, device: torch.device) -> tuple[Tensor, Tensor]:
        """counts / offsets of ``n`` rows for every expert, built once per (n, device) so that the
        call itself launches nothing but the expert kernels (and records cleanly into a HIP graph)."""
        cache = self.__dict__.setdefault("_uniform_cache", {})
        key = (n, str(device))
        if key not in cache:
            e = self.num_local_experts
            cache.clear()
            cache[key] = (
                torch.full((e,), n, dtype=torch.int32, device=device),
                torch.arange(e + 1, dtype=torch.int32, device=device) * n,
            )
        return cache[key]


class _Projection(Module):
    """Bias-free linear map holding an ``nn.Linear``-oriented ``weight`` (out, in),
    initialised like fairseq2's ``Linear`` (``nn/projection.py:638-640``)."""

    def __init__(self, input_dim: int, output_dim: int, device=None, dtype=None) -> None:
        super().__init__()
        self.input_dim, self.output_dim = input_dim, output_dim
        self.weight = Parameter(torch.empty((output_dim, input_dim), device=device, dtype=dtype))
        self.register_parameter("bias", None)
        self.reset_parameters()

    def reset_parameters(self) -> None:
        if not self.weight.is_meta:
            nn.init.kaiming_uniform_(self.weight, a=math.sqrt(5))

    def extra_repr(self) -> str:
        return f"input_dim={self.input_dim}, output_dim={self.output_dim}, bias=False"


class GLUFeedForwardNetwork(FeedForwardNetwork):
    """Bias-free SwiGLU network, the shared expert (``ffn.py:228-395`` with
    ``bias=False``, no dropout, no activation sparsity):
    ``output_proj(inner_proj(x) * silu(gate_proj(x)))``."""

    def __init__(
        self,
        model_dim: int,
        inner_dim: int,
        bias: bool = False,
        *,
        inner_dim_scale: float = 2 / 3,
        inner_dim_to_multiple: int = 1,
        device: torch.device | None = None,
        dtype: torch.dtype | None = None,
    ) -> None:
        super().__init__()
        if bias:
            raise NotImplementedError("the fused GLU kernels are bias-free")
        self.inner_dim_scale = inner_dim_scale
        self.inner_dim_to_multiple = inner_dim_to_multiple
        if inner_dim_scale != 1.0:
            inner_dim = int(inner_dim * inner_dim_scale)
        if inner_dim_to_multiple != 1:
            inner_dim = inner_dim_to_multiple * (
                (inner_dim + inner_dim_to_multiple - 1) // inner_dim_to_multiple
            )
        self.gate_proj = _Projection(model_dim, inner_dim, device, dtype)
        self.gate_activation = nn.SiLU()
        self.inner_proj = _Projection(model_dim, inner_dim, device, dtype)
        self.output_proj = _Projection(inner_dim, model_dim, device, dtype)

    def forward(self, seqs: Tensor) -> Tensor:
        _require_device(seqs)
        x = seqs.reshape(-1, seqs.shape[-1]).contiguous()
        params = (self.gate_proj.weight, self.inner_proj.weight, self.output_proj.weight)
        if torch.is_grad_enabled() and any(t.requires_grad for t in (seqs, *params)):
            # training: one autograd function on the library's backward kernels
            if x.shape[0] == 0:
                return torch.empty_like(seqs)
            from fairseq2_amd.autograd import DenseSwiGLUFunction

            return DenseSwiGLUFunction.apply(x, *params).view(seqs.shape)
        y = _abi.dense_swiglu(
            x, self.gate_proj.weight.detach(), self.inner_proj.weight.detach(),
            self.output_proj.weight.detach(),
        )
        return y.view(seqs.shape)

    def extra_repr(self) -> str:
        return (
            f"inner_dim_scale={self.inner_dim_scale:G}, "
            f"inner_dim_to_multiple={self.inner_dim_to_multiple}"
        )


_SCORE_FNS = {"sigmoid": _abi.SCORE_SIGMOID, "softmax": _abi.SCORE_SOFTMAX}


class MoE(FeedForwardNetwork):
    """Mixture-of-experts feed-forward network (token-choice top-k routing)."""

    router: Parameter
    top_k: int
    experts: ExpertNetwork
    shared_expert: GLUFeedForwardNetwork | None

    def __init__(
        self,
        model_dim: int,
        inner_dim: int,
        use_shared_expert: bool,
        num_experts: int,
        capacity_factor: float,
        top_k: int,
        *,
        moe_activation: Module | None = None,
        inner_dim_scale: float = 2 / 3,
        inner_dim_to_multiple: int = 1,
        auto_scale: bool = True,
        score_fn: str = "sigmoid",
        renormalize: bool = False,
        scale_on: str = "input",
        router_bias: bool = False,
        tile_m: int = 16,
        act_quant: str | None = None,
    ) -> None:
        super().__init__()
        if act_quant not in (None, "mxfp8"):
            raise ValueError(f"act_quant must be None or 'mxfp8', got {act_quant!r}")
        if score_fn not in _SCORE_FNS:
            raise ValueError(f"score_fn must be 'sigmoid' or 'softmax', got {score_fn!r}")
        if scale_on not in ("input", "output"):
            raise ValueError(f"scale_on must be 'input' or 'output', got {scale_on!r}")
        if not 1 <= num_experts <= _abi.MAX_EXPERTS:
            raise ValueError(f"num_experts must be in [1, {_abi.MAX_EXPERTS}], got {num_experts}")
        if not 1 <= top_k <= min(num_experts, _abi.MAX_TOP_K):
            raise ValueError(
                f"top_k must be in [1, min(num_experts, {_abi.MAX_TOP_K})], got {top_k}"
            )

        # Inner-dimension rule of the reference constructor (moe.py:52-65).
        self.inner_dim_scale = inner_dim_scale
        if inner_dim_scale != 1.0:
            inner_dim = int(inner_dim * inner_dim_scale)
        self.inner_dim_to_multiple = inner_dim_to_multiple
        if auto_scale:
            inner_dim = int(inner_dim / (capacity_factor + int(use_shared_expert)))
        if inner_dim_to_multiple != 1:
            inner_dim = inner_dim_to_multiple * (
                (inner_dim + inner_dim_to_multiple - 1) // inner_dim_to_multiple
            )
        if model_dim % 8 != 0 or inner_dim % 8 != 0:
            raise ValueError(
                f"model_dim ({model_dim}) and the expert inner dim ({inner_dim}) must be multiples of 8"
            )

        if use_shared_expert:
            self.shared_expert = GLUFeedForwardNetwork(
                model_dim, inner_dim, bias=False, inner_dim_scale=1.0, inner_dim_to_multiple=1
            )
        else:
            self.shared_expert = None

        self.router = Parameter(torch.empty(model_dim, num_experts))
        self.top_k = top_k
        self.experts = GroupedExpertNetwork(num_experts, model_dim, inner_dim, activation=moe_activation)
        # keyword-only extension, off by default: see GroupedExpertNetwork.act_quant
        self.experts.act_quant = act_quant

        # Kept for interface parity; tensor-parallel reduction is outside the single-GPU path.
        self.tp_gang = None

        self.score_fn = score_fn
        self.renormalize = renormalize
        self.scale_on = scale_on
        self.tile_m = tile_m
        if router_bias:
            self.register_buffer("router_bias", torch.zeros(num_experts, dtype=torch.float32))
        else:
            self.router_bias = None

    def forward(self, seqs: Tensor, *, residual: Tensor | None = None, norm=None) -> Tensor:
        """``seqs``: ``(*, dim)`` -> ``(*, dim)``, same dtype.

        Under ``torch.autocast("cuda", dtype)`` (the reference trainer wraps the model in it,
        ``trainer.py:650-656``) ``seqs`` is cast to the autocast dtype when the module's parameters
        are held in it, and the result comes back in that dtype, as the reference's matrix products
        would leave it; parameters of another dtype are not cast behind the caller's back.

        ``residual`` (keyword-only extension, same shape and dtype as ``seqs``): returns
        ``residual + layer(seqs)`` from one accumulation, i.e. the feed-forward half of a pre-norm
        decoder layer (``models/transformer_lm/decoder_layer.py:188-204``) without the separate
        addition pass.

        ``norm`` (keyword-only extension): the layer's RMS normalisation module (attributes
        ``weight`` -- a ``(dim,)`` tensor or None --, ``bias`` None, and ``eps``, as
        ``fairseq2.nn.RMSNorm`` has them, ``nn/normalization.py:166-254``).  The rows are then
        normalised inside the router kernel instead of by a pass of their own, so that
        ``layer(seqs, residual=seqs, norm=layer_norm)`` is the whole of ``_forward_ffn``
        (``decoder_layer.py:187-204``) for a pre-norm layer without dropout."""
        if torch.is_autocast_enabled("cuda"):
            seqs = self._autocast(seqs)
            if residual is not None:
                residual = self._autocast(residual)
        compiling = torch.compiler.is_compiling()
        wants_grad = torch.is_grad_enabled() and any(
            isinstance(t, Tensor) and t.requires_grad
            for t in (seqs, residual, getattr(norm, "weight", None), *self.parameters())
        )
        if wants_grad and not compiling:
            return self._differentiable(seqs, residual, norm)
        # (while a compiler traces the call, training goes through the registered operator below,
        # which carries its own autograd formula)
        x = self._checked_rows(seqs, allow_grad=wants_grad)
        norm_args = self._norm_args(norm, x, allow_grad=wants_grad)
        res = x if residual is seqs else None
        if residual is not None and residual is not seqs:
            if residual.shape != seqs.shape or residual.dtype != seqs.dtype:
                raise ValueError("residual must have the shape and dtype of seqs")
            _require_device(residual)
            if not wants_grad:
                _require_forward_only(residual)
            res = residual.reshape(-1, seqs.shape[-1]).contiguous()
        if x.shape[0] == 0:
            return torch.empty_like(seqs)
        ex, se = _part(self, "experts"), self.shared_expert
        w8a8 = type(ex) is GroupedExpertNetwork and ex.act_quant is not None and ex.runs_w8a8(
            x.dtype, x.shape[0] * self.top_k + ex.num_local_experts * (self.tile_m - 1))
        # (W8A8 inside the one call wherever the call takes it: output-side weights, not under a
        # compiler's trace, whose registered operator does not carry the option)
        w8a8_staged = w8a8 and (self.scale_on == "input" or compiling)
        if (type(ex) is GroupedExpertNetwork and ex.has_fused_gate and not w8a8_staged
                and (se is None or type(se) is GLUFeedForwardNetwork)):
            if compiling:
                return self._single_call(x, res, norm_args, act_quant=w8a8).view(seqs.shape)
            return self._single_call(x, res, norm_args, act_quant=w8a8, out_shape=seqs.shape)
        if wants_grad:
            # (only reachable inside a compiler's trace: the staged path below records no graph)
            raise RuntimeError(
                "fairseq2_amd.MoE: under torch.compile only the fused SiLU experts are differentiated; "
                "train this configuration eagerly")
        return self._stages(x, res, norm_args)[0].view(seqs.shape)

    def _differentiable(self, seqs: Tensor, residual: Tensor | None, norm) -> Tensor:
        """The training path: the layer as one ``torch.autograd.Function`` whose backward pass runs
        on the library's kernels (:mod:`fairseq2_amd.autograd`), for ``seqs``, ``residual`` and
        every parameter (the weight of ``norm`` included).  Covers the reference configuration and
        the extensions; e4m3 weights and other expert modules are forward-only."""
        ex, se = self.experts, self.shared_expert
        why = None
        if type(ex) is not GroupedExpertNetwork or (se is not None and type(se) is not GLUFeedForwardNetwork):
            why = "only GroupedExpertNetwork experts and a GLUFeedForwardNetwork shared expert are differentiated"
        elif not ex.has_fused_gate and any(p.requires_grad for p in ex.activation.parameters()):
            why = "a gate activation with parameters of its own is not differentiated"
        elif ex.has_fp8_weights:
            why = "e4m3 expert weights are an inference format"
        if why is not None:
            raise RuntimeError(
                f"fairseq2_amd.MoE: {why}; call it under torch.no_grad() / torch.inference_mode(), "
                "or freeze the inputs and the module with requires_grad_(False)")
        x = self._checked_rows(seqs, allow_grad=True)
        norm_args = self._norm_args(norm, x, allow_grad=True)
        res = None
        if residual is not None:
            if residual.shape != seqs.shape or residual.dtype != seqs.dtype:
                raise ValueError("residual must have the shape and dtype of seqs")
            _require_device(residual)
            res = residual.reshape(-1, seqs.shape[-1]).contiguous()
        if x.shape[0] == 0:
            return torch.empty_like(seqs)
        from fairseq2_amd.autograd import MoEFunction

        shared = (None, None, None)
        if se is not None:
            shared = (se.gate_proj.weight, se.inner_proj.weight, se.output_proj.weight)
        # (the module's own sizes; what the calls are given is checked again where addresses are taken)
        _abi.check_layer_arguments(
            x, self.router, self.router_bias, ex.gate_proj, ex.inner_proj, ex.output_proj, ex.num_local_experts,
            ex.inner_dim, None, None if se is None else shared)
        cfg = dict(
            num_experts=ex.num_local_experts, top_k=self.top_k, tile_m=self.tile_m,
            score_fn=_SCORE_FNS[self.score_fn], renormalize=self.renormalize,
            scale_input=self.scale_on == "input", router_bias=self.router_bias,
            activation=None if ex.has_fused_gate else ex.activation,
            norm_eps=None if norm_args is None else norm_args[1],
            # the forward pass routes as the inference path does (the same logits bit for bit)
            router_t=self._router_expert_major(),
        )
        out = MoEFunction.apply(x, res, self.router, ex.gate_proj, ex.inner_proj, ex.output_proj,
                                *shared, None if norm_args is None else norm_args[0], cfg)
        return out.view(seqs.shape)

    def _autocast(self, t: Tensor) -> Tensor:
        if t.is_cuda:
            dt = torch.get_autocast_dtype("cuda")
            if t.is_floating_point() and t.dtype != dt and self.router.dtype == dt:
                return t.to(dt)
        return t

    @staticmethod
    def _norm_args(norm, x: Tensor, allow_grad: bool = False) -> tuple[Tensor | None, float] | None:
        """(weight, eps) of an RMS normalisation module, checked against the rows ``x``."""
        if norm is None:
            return None
        if _optional(norm, "bias") is not None:
            raise ValueError("the fused normalisation is an RMS norm without bias")
        shape = tuple(getattr(norm, "normalized_shape", (x.shape[-1],)))
        if shape != (x.shape[-1],):
            raise ValueError(f"norm normalises over {shape}, expected ({x.shape[-1]},)")
        weight = _optional(norm, "weight")
        if weight is not None:
            _require_device(weight)
            if not allow_grad:
                _require_forward_only(weight)
            if weight.dtype != x.dtype or weight.shape != (x.shape[-1],):
                raise ValueError("the norm weight must be (dim,) in the dtype of seqs")
            weight = weight.contiguous()
        return weight, float(norm.eps)

    def _router_expert_major(self) -> Tensor | None:
        """The router matrix expert-major (see :func:`fairseq2_amd._abi.router_expert_major`)."""
        return _abi.router_expert_major(self.router, self)

    def _single_call(self, x: Tensor, residual: Tensor | None = None, norm=None, *,
                     act_quant: bool = False, out_shape: torch.Size | None = None) -> Tensor:
        """The layer through the library's whole-layer entry point: one call, one workspace
        allocation (same kernels and results as :meth:`_stages`)."""
        ex, se = _part(self, "experts"), self.shared_expert
        if ex.has_fp8_weights:
            weights, scales = ex._fp8_operands()
        else:
            weights = (_held(ex, "gate_proj"), _held(ex, "inner_proj"), _held(ex, "output_proj"))
            scales = None
        shared = None
        if se is not None:
            shared = tuple(_held(p, "weight") for p in (se.gate_proj, se.inner_proj, se.output_proj))
        if torch.compiler.is_compiling():
            # under torch.compile the call goes through the registered operator, which the tracer
            # can represent (it cannot look through ctypes); it is given the parameters themselves,
            # so that its autograd formula reaches them when the trace is one of a training step
            return torch.ops.fairseq2_amd.moe_forward(
                x, self.router, self.router_bias, *weights, *(scales or (None, None, None)),
                *(shared or (None, None, None)), residual, None if norm is None else norm[0],
                ex.num_local_experts, self.top_k, self.tile_m, _SCORE_FNS[self.score_fn],
                self.renormalize, self.scale_on == "input", norm is not None,
                0.0 if norm is None else norm[1],
            )
        router = _held(self, "router")
        return _abi.forward(
            x, router, self.router_bias, *weights, ex.num_local_experts, self.top_k,
            scales=scales, shared=shared, tile_m=self.tile_m, score_fn=_SCORE_FNS[self.score_fn],
            renormalize=self.renormalize, scale_input=self.scale_on == "input", residual=residual,
            norm=norm, router_t=_abi.router_expert_major(router, self), act_quant=act_quant,
            out_shape=out_shape,
        )

    @torch.no_grad()
    def _stages(self, x: Tensor, residual: Tensor | None = None, norm=None):
        ex = self.experts
        if norm is None:
            idx, w, _ = _abi.router_topk(
                x, self.router.detach(), self.router_bias, self.top_k, _SCORE_FNS[self.score_fn],
                self.renormalize, router_t=self._router_expert_major(),
            )
        else:
            # every later stage reads the normalised rows
            x, idx, w, _ = _abi.router_topk_norm(
                x, norm[0], norm[1], self.router.detach(), self.router_bias, self.top_k,
                _SCORE_FNS[self.score_fn], self.renormalize, router_t=self._router_expert_major(),
            )
        scale_input = self.scale_on == "input"
        # Unscaled rows need no copy in expert order: the first GEMM reads them from x through the
        # permutation (where the library offers that), and dispatch only computes the bookkeeping.
        fused = (
            not scale_input
            and isinstance(ex, GroupedExpertNetwork)
            and ex.fuses_gather(x.dtype, x.shape[0] * self.top_k + ex.num_local_experts * (self.tile_m - 1))
        )
        disp = _abi.dispatch(
            idx, w, x, ex.num_local_experts, self.tile_m, scale_input, gather=not fused
        )
        # a token takes an expert at most once: with up to 16 tokens no expert has more rows than that
        # (what the whole-layer call passes on as well)
        hint = {}
        if isinstance(ex, GroupedExpertNetwork):
            hint = ex._row_hints(x.shape[0] if x.shape[0] <= 16 else 0, idx.numel())
        if fused:
            ye = ex.forward_rows(x, disp.counts, disp.offsets, row_map=disp.perm, **hint)
        else:
            ye = ex.forward_rows(disp.xe, disp.counts, disp.offsets, **hint)
        base = None
        if self.shared_expert is not None:
            base = self.shared_expert(x)
        out = _abi.combine(ye, disp.inv_perm, idx, w, base, not scale_input, out=base, residual=residual)
        return out, idx, w, disp

    def forward_with_routing(self, seqs: Tensor):
        """Returns ``(out, topk_idx, topk_w, dispatched)``; the extra values are the
        routing artefacts the parity tests compare bit for bit."""
        x = self._checked_rows(seqs)
        if x.shape[0] == 0:
            return torch.empty_like(seqs), None, None, None
        out, idx, w, disp = self._stages(x)
        return out.view(seqs.shape), idx, w, disp

    def _checked_rows(self, seqs: Tensor, allow_grad: bool = False) -> Tensor:
        """Validates ``seqs`` against the module and returns it as contiguous ``(T, dim)`` rows."""
        if self.tp_gang is not None:
            raise NotImplementedError("tensor-parallel reduction is not part of the single-GPU path")
        _require_device(seqs)
        if not allow_grad and torch.is_grad_enabled():  # (walking the parameters costs host time)
            _require_forward_only(seqs, *self.parameters())
        router = _held(self, "router")
        if seqs.dtype != router.dtype:
            hint = ""
            if torch.is_autocast_enabled("cuda"):
                hint = (f" (autocast to {torch.get_autocast_dtype('cuda')} is on: hold the module's "
                        "parameters in that dtype)")
            raise TypeError(f"seqs is {seqs.dtype} but the module holds {router.dtype} parameters{hint}")
        dim = seqs.shape[-1]
        if dim != router.shape[0]:
            raise ValueError(f"last dimension of seqs is {dim}, expected {router.shape[0]}")
        return seqs.reshape(-1, dim).contiguous()

    def extra_repr(self) -> str:
        return (
            f"top_k={self.top_k}, score_fn={self.score_fn}, renormalize={self.renormalize}, "
            f"scale_on={self.scale_on}, tile_m={self.tile_m}"
        )


class GraphedForward:
    """One captured HIP graph of ``module(seqs)`` for a fixed input shape and dtype.

    The layer is six to eight short kernel launches; at decode sizes the gaps between them are a
    tenth of the step.  Everything the forward pass does is a kernel of the library writing into
    memory from torch's allocator (no fills, no reductions by torch), so the whole call records into
    a graph and replays with one submission.  ``__call__`` copies the argument into the graph's
    input buffer and returns the graph's output buffer: the result is overwritten by the next call.

    ``add_input=True`` captures ``module(seqs, residual=seqs)`` and ``norm`` is passed on as the
    module's ``norm`` argument, so that ``GraphedForward(layer.ffn, x, add_input=True,
    norm=layer.ffn_layer_norm)`` is one graph of a pre-norm decoder layer's whole feed-forward step.
    """

    def __init__(self, module: Module, example: Tensor, warmup: int = 2, *, add_input: bool = False,
                 norm=None) -> None:
        _require_device(example)
        self._module = module
        self._input = example.clone()
        kwargs = {}
        if add_input:
            kwargs["residual"] = self._input
        if norm is not None:
            kwargs["norm"] = norm
        # Eager runs first, on a side stream of default priority: one-time library set-up (kernel
        # attributes, device queries) must not happen while capturing.
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side), torch.no_grad():
            for _ in range(max(1, warmup)):
                module(self._input, **kwargs)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        self._graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self._graph), torch.no_grad():
            self._output = module(self._input, **kwargs)

    @property
    def input(self) -> Tensor:
        """The graph's input buffer (fill it in place to skip the copy in ``__call__``)."""
        return self._input

    @property
    def output(self) -> Tensor:
        return self._output

    def replay(self) -> Tensor:
        self._graph.replay()
        return self._output

    def __call__(self, seqs: Tensor) -> Tensor:
        if seqs.shape != self._input.shape or seqs.dtype != self._input.dtype:
            raise ValueError(
                f"graph was captured for {tuple(self._input.shape)} {self._input.dtype}, "
                f"got {tuple(seqs.shape)} {seqs.dtype}"
            )
        # (the library launches on the current device's stream, a replay and copy_ go to the tensors' device)
        if (seqs.device == self._input.device and seqs.device.index == torch._C._cuda_getDevice()
                and seqs.is_contiguous() and self._input.is_contiguous()):
            _abi.copy(seqs, self._input)
        else:
            self._input.copy_(seqs)
        return self.replay()

