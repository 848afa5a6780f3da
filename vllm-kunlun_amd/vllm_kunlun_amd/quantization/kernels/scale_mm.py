"""Dense W8A8 linear layer (the shared expert's gate_up and down projections, and any other
int8 Linear of a W8A8 checkpoint).

Mirror of `KunlunScaledMMLinearKernel` (reference: quantization/kernels/scale_mm.py:30-90), which
vLLM's `CompressedTensorsW8A8Int8` scheme instantiates per Linear. The reference derives from
vLLM's `CutlassInt8ScaledMMLinearKernel`; vLLM is not a dependency here, so this class carries the
few pieces of that base it relies on (the parameter names and what the base's
`process_weights_after_loading` leaves behind: the weight as the [k, n] transpose view of its
[n, k] storage, a per-channel weight scale, no input scale for dynamic quantisation).

Path taken by `apply_weights`: per-token absmax int8 quantisation and the int8 GEMM in one library call
(`kmoe_linear_i8`) on the weights re-arranged at load time into the MFMA tiles - up to a number of rows that
depends on the matrix (`_DynamicCall`) on a kernel whose waves split K, which quantises up to four rows (of very wide matrices one) itself, beyond as the
one-expert case of the tile kernel the fused MoE layer's prefill batches run on.
"""
from __future__ import annotations

from dataclasses import dataclass
from typing import Optional

import torch

from ... import _lib as L
from ... import _plan
from ..._plan import tile_int8_weights_, weight_layout


@dataclass
class Int8ScaledMMLinearLayerConfig:
    """The fields of vLLM's config of the same name that the kernel selection reads."""
    is_channelwise: bool = True
    is_static_input_scheme: bool = False
    input_symmetric: bool = True


_ROW_RANGES: dict = {}  # (device, rows) -> the {0, rows} row range of a dense GEMM's single expert, made once


def _row_range(device, rows):
    key = (device, rows)
    found = _ROW_RANGES.get(key)
    if found is None:
        if torch.cuda.is_current_stream_capturing():
            # (an upload cannot be captured; a launch of the graph's own writes the two numbers on every replay, into
            # the graph's memory, so the tensor is of no use to other calls)
            return torch.arange(0, rows + 1, rows, dtype=torch.int32, device=device) if rows else \
                torch.zeros(2, dtype=torch.int32, device=device)
        found = _ROW_RANGES[key] = torch.tensor([0, rows], dtype=torch.int32).to(device)
    return found


_NOTHING: dict = {}


class _DynamicCall:
    """Quantisation and GEMM of one Linear with dynamic symmetric activations: the argument block of kmoe_linear_i8 with
    everything but the batch filled in, kept on the layer. A call is one or two launches on a scratch buffer of the stream
    and one allocation, the output. Ordinary calls of up to split_max rows run in native code (`native`; a dense MLP of two
    such calls and SiLU-mul, of 64 rows: 24 us of host time where this method's own took 30)."""

    __slots__ = ("native", "args", "n", "k", "device", "scale", "at", "epoch", "split_max")

    def __init__(self, layer, names, w, w_max):
        L.require_device(w, w_max)
        L.require_contig(w, w_max)
        _, self.n, self.k = w.shape
        self.device = w.device
        self.scale = self._value(layer, names[1])
        self.at = (w.data_ptr(), w_max.data_ptr())
        self.epoch = _plan._layout_epoch
        layout = weight_layout(w)
        # rows that go to the kernel whose waves split K; more, and row-major weights, to the tile kernel
        self.split_max = L.lib.kmoe_linear_i8_split_rows(self.n, self.k) if layout == L.KMOE_W_TILED else 0
        g = L.LinearI8Args()
        g.w, g.w_max = self.at
        g.n, g.k, g.ld_x, g.ldy, g.w_layout = self.n, self.k, self.k, self.n, layout
        self.args = g
        self.native = (L.torch_calls.Linear(*self.at, self.n, self.k, layout, self.device.index, self.split_max)
                       if self.device.type == "cuda" and L.torch_calls is not None else None)

    @staticmethod
    def _value(layer, name):
        """getattr(layer, name, None), sooner for a Module's parameters (an engine may also put a buffer or a plain tensor
        in a parameter's place)."""
        value = layer.__dict__.get("_parameters", _NOTHING).get(name)
        return getattr(layer, name, None) if value is None else value

    def holds(self, layer, names) -> bool:
        """Whether the layer's tensors are still the ones the block was filled from, and a call of it still dynamic and
        symmetric (no input scale, no zero-point sums)."""
        w, scale = getattr(layer, "_kmoe_w_1nk", None), self._value(layer, names[1])
        return (scale is not None and scale is self.scale and w is not None and w.data_ptr() == self.at[0]
                and w.shape == (1, self.n, self.k) and scale.data_ptr() == self.at[1] and self._value(layer, names[2]) is None
                and self._value(layer, names[4]) is None and self.epoch == _plan._layout_epoch)

    def __deepcopy__(self, memo):
        return None  # (a copied layer fills a block of its own)

    def __reduce__(self):
        return type(None), ()

    def __call__(self, x: torch.Tensor) -> torch.Tensor:
        out = None if self.native is None else self.native(x)
        if out is not None:
            return out
        dt = L.act_dtype(x, "KunlunScaledMMLinearKernel")
        flat = x.dim() == 2 and x.is_contiguous()
        x2 = x if flat else x.reshape(-1, x.shape[-1]).contiguous()
        M, k = x2.shape
        n = self.n
        if k != self.k:
            raise ValueError(f"KunlunScaledMMLinearKernel: rows of {k} values for weights of {self.k}")
        if x2.device != self.device:
            raise RuntimeError(f"kmoe ops run on the GPU only; got a tensor on {x2.device}")
        out = x2.new_empty((M, n))
        if M:
            need = -(-M * k // 256) * 256 + 4 * M
            if torch._C._cuda_isCurrentStreamCapturing():
                scratch = torch.empty(need, dtype=torch.uint8, device=self.device)  # the graph's own
            else:
                scratch = _plan.WORKSPACE.get(need, self.device, L.raw_stream(self.device.index))
            g = L.LinearI8Args.from_buffer_copy(self.args)  # a copy: threads may share the block
            g.x, g.rows, g.y, g.act_dtype = x2.data_ptr(), M, out.data_ptr(), dt
            g.scratch, g.scratch_bytes = scratch.data_ptr(), need
            if M > self.split_max:
                lod = _row_range(self.device, M)
                g.lod = lod.data_ptr()
            L.check(L.lib.kmoe_linear_i8(g, L.raw_stream()))
        return out if flat else out.reshape(*x.shape[:-1], n)


class KunlunScaledMMLinearKernel:
    def __init__(self, c: Optional[Int8ScaledMMLinearLayerConfig] = None, w_q_param_name: str = "weight",
                 w_s_param_name: str = "weight_scale", i_s_param_name: str = "input_scale",
                 i_zp_param_name: str = "input_zero_point", azp_adj_param_name: str = "azp_adj"):
        self.config = c or Int8ScaledMMLinearLayerConfig()
        self.layer_param_names = (w_q_param_name, w_s_param_name, i_s_param_name, i_zp_param_name,
                                  azp_adj_param_name)

    @classmethod
    def is_supported(cls, compute_capability: Optional[int] = None) -> tuple[bool, Optional[str]]:
        """Reference: scale_mm.py:32-37 (there: any out-of-tree platform). Here: a HIP device."""
        if not torch.cuda.is_available():
            return False, "requires a HIP device."
        return True, None

    @classmethod
    def can_implement(cls, c: Int8ScaledMMLinearLayerConfig) -> tuple[bool, Optional[str]]:
        """Reference: scale_mm.py:39-41 accepts every config and fails later; this class says up
        front which schemes its kernels cover: all four (dynamic or static input scale, symmetric or
        asymmetric activations)."""
        return True, None

    def _get_layer_params(self, layer):
        return tuple(getattr(layer, name, None) for name in self.layer_param_names)

    def process_weights_after_loading(self, layer: torch.nn.Module) -> None:
        """Base-class part: the weight parameter becomes the [k, n] transpose view, the weight
        scale one f32 per output channel. Reference part (scale_mm.py:43-50): scale -> absmax
        (x 127), in place. Added here: the [n, k] storage is re-arranged into the MFMA tiles once
        (when n % 16 == 0 and k % 64 == 0) and kept on the layer for `apply_weights`."""
        w_q_name, w_s_name, i_s_name, i_zp_name, azp_adj_name = self.layer_param_names
        weight = getattr(layer, w_q_name)
        w_nk = weight.data
        if w_nk.dtype != torch.int8 or w_nk.dim() != 2:
            raise ValueError(f"{w_q_name}: expected int8 [n, k], got {w_nk.dtype} {tuple(w_nk.shape)}")
        w_nk = w_nk.contiguous()
        n, k = w_nk.shape
        w_s = getattr(layer, w_s_name)
        scale = w_s.data.to(torch.float32).reshape(-1)
        if scale.numel() == 1:  # per-tensor scale of an unfused layer -> one per channel
            scale = scale.expand(n)
        if scale.numel() != n:
            raise ValueError(f"{w_s_name}: {scale.numel()} scales for {n} output channels")
        scale = scale.contiguous().clone().reshape(n, 1)
        with torch.no_grad():
            scale.mul_(127.0)  # scale -> absmax, what the kernels take (x_pc_max / w_pc_max convention)
        # Static input scheme (base-class part, upstream vLLM's CutlassInt8ScaledMMLinearKernel, which is not in
        # this container: restated from its published source): a layer fused from several checkpoint tensors
        # (qkv, gate_up) carries one input scale - and zero point - per partition, and the kernels take ONE.
        # Symmetric: the largest scale. Asymmetric: the value range every partition covers,
        # [min_p scale_p (-128 - zp_p), max_p scale_p (127 - zp_p)], cut into 255 steps again.
        if self.config.is_static_input_scheme:
            i_s = getattr(layer, i_s_name, None)
            if i_s is None:
                raise ValueError(f"{i_s_name}: a static input scheme needs the input scale")
            s_in = i_s.data.to(torch.float32).reshape(-1)
            if self.config.input_symmetric:
                setattr(layer, i_s_name, torch.nn.Parameter(s_in.max().reshape(1), requires_grad=False))
            else:
                i_zp = getattr(layer, i_zp_name, None)
                if i_zp is None:
                    raise ValueError(f"{i_zp_name}: a static asymmetric scheme needs the input zero point")
                zps = i_zp.data.to(torch.int32).reshape(-1)
                if zps.numel() not in (1, s_in.numel()):
                    raise ValueError(f"{i_zp_name}: {zps.numel()} zero points for {s_in.numel()} input scales")
                if s_in.numel() > 1:  # (one partition: its scale and zero point are kept as they are)
                    range_max = (s_in * (127 - zps)).max()
                    range_min = (s_in * (-128 - zps)).min()
                    one_scale = (range_max - range_min) / 255.0
                    # rounded to the nearest integer: the quotient is an integer up to float error when one
                    # partition spans the whole range, and truncation would then lose one
                    one_zp = torch.round(-128 - range_min / one_scale).to(torch.int32)
                    setattr(layer, i_s_name, torch.nn.Parameter(one_scale.reshape(1), requires_grad=False))
                    setattr(layer, i_zp_name, torch.nn.Parameter(one_zp.reshape(1), requires_grad=False))
        # Asymmetric activations (base-class part): azp_adj = the sums of the weight codes over k per output channel,
        # times the input zero point for a static scheme, whose zero point then needs no term of its own at run time.
        if not self.config.input_symmetric:
            azp_adj = w_nk.sum(dim=1, dtype=torch.int32).reshape(1, n)
            if self.config.is_static_input_scheme:
                i_zp = getattr(layer, i_zp_name, None)
                if i_zp is None:
                    raise ValueError(f"{i_zp_name}: a static asymmetric scheme needs the input zero point")
                azp_adj = azp_adj * i_zp.data.to(torch.int32).reshape(1, 1)
            setattr(layer, azp_adj_name, torch.nn.Parameter(azp_adj.contiguous(), requires_grad=False))
        tile_int8_weights_(w_nk)  # in place, marks the memory; shapes that do not tile stay row-major
        layer._kmoe_w_1nk = w_nk.view(1, n, k)  # what the grouped GEMM takes
        setattr(layer, w_q_name, torch.nn.Parameter(w_nk.t(), requires_grad=False))
        setattr(layer, w_s_name, torch.nn.Parameter(scale, requires_grad=False))
        if getattr(layer, i_s_name, None) is not None and not self.config.is_static_input_scheme:
            setattr(layer, i_s_name, None)
        for name in (i_s_name, i_zp_name, azp_adj_name):
            if not hasattr(layer, name):
                setattr(layer, name, None)

    def apply_weights(self, layer: torch.nn.Module, x: torch.Tensor,
                      bias: Optional[torch.Tensor] = None) -> torch.Tensor:
        """Reference: scale_mm.py:52-90. The symmetric branch: quantise per token (dynamic) or with the
        layer's one input scale (static), multiply, rescale by x_max * w_max / 127^2, in x's dtype.
        Output [..., n]."""
        call = layer.__dict__.get("_kmoe_dynamic")
        if call is not None and bias is None and call.holds(layer, self.layer_param_names):
            return call(x)
        w_q, w_s, x_s, x_zp, azp_adj = self._get_layer_params(layer)
        if azp_adj is not None:
            return self._apply_asymmetric(layer, x, w_q, w_s, x_s, x_zp, azp_adj, bias)
        if bias is not None:
            # the reference's call (scale_mm.py:83-90): quantise, then matmul with the f32 bias
            x2 = x.reshape(-1, x.shape[-1]).contiguous()
            x_q, x_s2, _, static = torch.ops._C.scaled_int8_quant(
                x2, None if x_s is None else x_s.data.to(torch.float32).reshape(1), None, True)
            out = torch.ops._C.matmul(x_q, w_q.transpose(0, 1), x.dtype, x_pc_max=x_s2 * 127.0 if static else x_s2,
                                      w_pc_max=w_s.data, bias=bias.to(torch.float32).contiguous())
            return out.reshape(*x.shape[:-1], out.shape[-1])
        L.act_dtype(x, "KunlunScaledMMLinearKernel")
        w = getattr(layer, "_kmoe_w_1nk", None)
        if w is None:
            raise RuntimeError("KunlunScaledMMLinearKernel: process_weights_after_loading has not run on this layer")
        from ...ops import _custom_ops as ops  # registers torch.ops._C.*
        lead = x.shape[:-1]
        if x_s is None:
            layer.__dict__["_kmoe_dynamic"] = call = _DynamicCall(layer, self.layer_param_names, w, w_s)
            return call(x)
        x2 = x.reshape(-1, x.shape[-1]).contiguous()
        M, n = x2.shape[0], w.shape[1]
        out = torch.empty((M, n), dtype=x.dtype, device=x.device)
        if M:  # static: one scale for the tensor, so every row's max is scale x 127
            x_q, x_s, _, _ = torch.ops._C.scaled_int8_quant(x2, x_s.data.to(torch.float32).reshape(1), None, True)
            x_max = (x_s * 127.0).expand(M).contiguous()
            ops._gemm_i8(x_q, x_max, w, w_s.data.reshape(-1), self._row_range(x.device, M), out, n, L.KMOE_ACT_NONE, M)
        return out.reshape(*lead, n)

    def _apply_asymmetric(self, layer, x, w_q, w_s, x_s, x_zp, azp_adj, bias):
        """Reference: scale_mm.py:60-82. Codes with a zero point (per token, or the layer's static one), the int8
        product, and the zero-point correction in the epilogue; the weight scale goes back from absmax to scale
        (/ 127) as there."""
        L.act_dtype(x, "KunlunScaledMMLinearKernel")
        lead = x.shape[:-1]
        x2 = x.reshape(-1, x.shape[-1]).contiguous()
        x_q, x_s, x_zp, static = torch.ops._C.scaled_int8_quant(
            x2, None if x_s is None else x_s.data.to(torch.float32).reshape(1),
            None if x_zp is None else x_zp.data.to(torch.int32).reshape(1), False)
        out = torch.ops._C.cutlass_scaled_mm_azp(
            x_q, w_q, x_s, (w_s.data / 127.0).transpose(0, 1), x.dtype, azp_adj.data, None if static else x_zp,
            None if bias is None else bias.to(torch.float32).contiguous())
        return out.reshape(*lead, out.shape[-1])

    def _row_range(self, device, rows):
        return _row_range(device, rows)
