"""Q4_0 linear quant method: the plugin's operator surface for the GEMVs.

The reference swaps a layer's ``quant_method`` for a class whose
``apply(layer, x, bias=None)`` serves the fast path for batch-1 bf16 input
and defers to the stock method otherwise (Q6HeadMethod,
src/spark_vllm_ascend/integration/head.py:12-16,31).  This module offers the
same hook for Q4_0 linears on vLLM's LinearMethodBase contract:

  create_weights(layer, input_size_per_partition, output_partition_sizes,
                 input_size, output_size, params_dtype, **extra)
      registers ``layer.qweight``: uint8 [sum(output_partition_sizes),
      input_size_per_partition/32*18], GGUF Q4_0 blocks as stored in the file.
  process_weights_after_loading(layer)
      validates the loaded blocks; the GEMVs stream GGUF blocks directly, so
      no repack happens here unless the config asks for the batched GEMM's
      packed layout (Q4_0Config(pack_for_batch=True): pack(layer) below).
  pack(layer, gated=False)
      on request, for batched decode: adds ``layer.q4_0_packed``, the packed
      layout of the MFMA GEMM (torch_ops.q4_0_repack; gated for a merged
      gate|up layer's SwiGLU GEMM), as the reference repacks its weights for
      its own kernel (src/spark_vllm_ascend/integration/weights.py:42-54).
      The GGUF blocks stay: the one-row GEMV reads them.
  apply(layer, x, bias=None) -> [..., N] bf16
      one HIP launch: the Q4_0 GEMV for one activation row, the MFMA Q4_0
      GEMM for 2..16 rows (K % 64 == 0; over the packed weights when pack()
      made them; any other K: q4_0_gemm_rows, small matrices the GEMV per
      row).  More rows (prefill) multiply
      the bf16 weights the reference's stock path uses, as Q6HeadMethod
      defers to the stock method outside its one-row case: up to a few
      hundred rows in one launch that converts the weights as it reads them
      (q4_0_gemm_rows, where torch_ops.gemm_rows_preferred says it is the
      faster way), else, and where torch has to see the product (autograd,
      functorch transforms, autocast), dequantised on the device, then a
      library GEMM.  Bias added after.

vLLM is not installed in this image; when it is, the class derives from its
LinearMethodBase so vLLM's loaders accept it unchanged.
"""
from __future__ import annotations

import torch

from ..native import torch_ops
from .weights import row_bytes

try:
    from torch._C import _len_torch_dispatch_stack, _len_torch_function_stack
    from torch._C._functorch import maybe_current_level
    from torch.overrides import _get_current_function_mode_stack
    from torch.utils._device import DeviceContext
    _STATE_KNOWN = isinstance(torch.autograd.forward_ad._current_level, int)
except (ImportError, AttributeError):  # another torch: torch_sees() is always true
    _STATE_KNOWN = False

try:  # pragma: no cover - vLLM is absent here
    from vllm.model_executor.layers.linear import LinearMethodBase as _Base
except Exception:  # noqa: BLE001
    class _Base:  # minimal stand-in with vLLM's method names
        def create_weights(self, layer, *args, **kwargs):
            raise NotImplementedError

        def apply(self, layer, x, bias=None):
            raise NotImplementedError

        def process_weights_after_loading(self, layer):
            return None


#: activation rows one MFMA Q4_0 GEMM launch serves (the kernel's m limit)
GEMM_MAX_ROWS = 16

#: weights (n * k) from which q4_0_gemm_rows takes a call.  Not a crossover: smaller
#: matrices keep the launches that the dispatch tests fix for them (the GEMV per
#: row, dequantisation and the library), although one launch is the faster there
#: too (eager, kept and fused: 1024 x 2560 at 40 rows 28 us and 11, 512 x 2592 at
#: 3 rows 22 and 10)
GEMM_ROWS_MIN_WEIGHTS = 3_000_000

#: K up to which 2 and 3 rows of a matrix of few rows (n < 1536) are one
#: q4_0_gemm_rows launch.  Its 8 waves walk K, 0.7 us per 1024, where a GEMV splits
#: it further: 300 x 10016 at 2 rows 10.5 us, two GEMVs 10.9; 96 x 32800 27.1,
#: 20.2; at 3 rows 27.1, 29.8; 48 x 65568 49.9, 49.4; 4 rows 49.9, 65.4
FEW_ROWS_MAX_K = {2: 10240, 3: 40960}


class Q4_0Config:
    """Quantization config naming the method, as vLLM's QuantizationConfig.
    pack_for_batch=True makes every linear also hold the packed layout of
    the batched GEMM (built in process_weights_after_loading): faster
    2..16-row decode for twice the weight memory."""

    def __init__(self, pack_for_batch: bool = False):
        self.pack_for_batch = bool(pack_for_batch)

    @classmethod
    def get_name(cls) -> str:
        return "q4_0"

    @classmethod
    def get_supported_act_dtypes(cls):
        return [torch.bfloat16]

    def get_quant_method(self, layer, prefix: str = ""):
        return Q4_0LinearMethod(pack_for_batch=self.pack_for_batch)


class Q4_0LinearMethod(_Base):
    """Q4_0 weights, bf16 activations, fp32 accumulation, bf16 output."""

    def __init__(self, pack_for_batch: bool = False):
        self.pack_for_batch = bool(pack_for_batch)

    def create_weights(self, layer: torch.nn.Module, input_size_per_partition: int,
                       output_partition_sizes: list[int], input_size: int, output_size: int,
                       params_dtype: torch.dtype, **extra_weight_attrs) -> None:
        k = int(input_size_per_partition)
        n = int(sum(output_partition_sizes))
        if params_dtype not in (torch.bfloat16,):
            raise ValueError(f"Q4_0 linears take bf16 activations, got {params_dtype}")
        device = extra_weight_attrs.pop("device", None)
        qweight = torch.nn.Parameter(
            torch.empty((n, row_bytes(k)), dtype=torch.uint8, device=device), requires_grad=False)
        layer.register_parameter("qweight", qweight)
        layer.q4_0_n = n
        layer.q4_0_k = k
        layer.output_partition_sizes = list(output_partition_sizes)
        for key, val in extra_weight_attrs.items():
            setattr(qweight, key, val)

    def process_weights_after_loading(self, layer: torch.nn.Module) -> None:
        w = layer.qweight
        if w.dtype != torch.uint8 or tuple(w.shape) != (layer.q4_0_n, row_bytes(layer.q4_0_k)):
            raise ValueError(f"qweight must be uint8 {(layer.q4_0_n, row_bytes(layer.q4_0_k))}, "
                             f"got {w.dtype} {tuple(w.shape)}")
        if not w.is_contiguous():
            layer.qweight = torch.nn.Parameter(w.contiguous(), requires_grad=False)
        if self.pack_for_batch:
            self.pack(layer)

    def pack(self, layer: torch.nn.Module, gated: bool = False) -> bool:
        """Build ``layer.q4_0_packed`` for the batched GEMM (K % 256 == 0;
        gated: a merged [gate, up] layer of equal halves).  Returns whether
        the layer has one afterwards."""
        n, k = layer.q4_0_n, layer.q4_0_k
        if k % 256 != 0:
            return False
        if gated:
            sizes = layer.output_partition_sizes
            if len(sizes) != 2 or sizes[0] != sizes[1]:
                raise ValueError("a gated pack needs a merged [gate, up] layer of equal halves")
            n = sizes[0]
        layer.q4_0_packed = torch_ops.q4_0_repack(layer.qweight.reshape(-1), n, k, gated)
        return True

    def apply(self, layer: torch.nn.Module, x: torch.Tensor,
              bias: torch.Tensor | None = None) -> torch.Tensor:
        n, k = layer.q4_0_n, layer.q4_0_k
        if x.shape[-1] != k:
            raise ValueError(f"expected last dim {k}, got {x.shape[-1]}")
        if x.dtype != torch.bfloat16:
            raise ValueError(f"expected bf16 activations, got {x.dtype}")
        rows = x.reshape(-1, k).contiguous()
        m = rows.shape[0]
        w = layer.qweight
        if not w.is_contiguous():
            w = w.contiguous()
        if m == 0:
            out = torch.empty((0, n), dtype=torch.bfloat16, device=x.device)
        elif m == 1:
            out = torch_ops.q4_0_gemv(rows, w, n, k)
        elif m <= GEMM_MAX_ROWS and k % 64 == 0:
            out = torch_ops.q4_0_gemm(aligned16(rows), gemm_weight(layer), n, k)
        elif (m <= GEMM_MAX_ROWS and n * k >= GEMM_ROWS_MIN_WEIGHTS and w.data_ptr() % 4 == 0
              and (n >= 1536 or k <= FEW_ROWS_MAX_K.get(m, k))):
            # K % 64 != 0: one launch for all rows (4001 x 2592, 5 rows: 5.5 us;
            # the GEMV below is 5.8 us for each)
            out = torch_ops.q4_0_gemm_rows(aligned16(rows), w, n, k)
        elif m <= GEMM_MAX_ROWS:
            # the GEMV (any K % 32 == 0, 2-byte aligned), one launch per row
            out = torch.empty((m, n), dtype=torch.bfloat16, device=x.device)
            for i in range(m):
                torch_ops.q4_0_gemv(rows[i], w, n, k, out=out[i])
        elif (n * k >= GEMM_ROWS_MIN_WEIGHTS and w.data_ptr() % 4 == 0
              and torch_ops.gemm_rows_preferred(m, n, k) and not torch_sees(rows)):
            out = torch_ops.q4_0_gemm_rows(aligned16(rows), w, n, k)
        else:
            w_bf16 = torch_ops.q4_0_dequant_bf16(w, n, k)
            out = torch.nn.functional.linear(rows, w_bf16.view(n, k))
        if x.dim() != 2:
            out = out.reshape(*x.shape[:-1], n)
        if bias is not None:
            out = out + bias
        return out

    def apply_swiglu(self, layer: torch.nn.Module, x: torch.Tensor,
                     out: torch.Tensor | None = None) -> torch.Tensor:
        """Merged gate|up layer (two equal partitions): silu(gate) * up fused
        into the GEMV epilogue, for one activation row."""
        sizes = layer.output_partition_sizes
        if len(sizes) != 2 or sizes[0] != sizes[1]:
            raise ValueError("apply_swiglu needs a merged [gate, up] layer of equal halves")
        return torch_ops.q4_0_gemv_swiglu(x.reshape(-1), layer.qweight.reshape(-1), sizes[0],
                                          layer.q4_0_k, out=out)


def aligned16(rows: torch.Tensor) -> torch.Tensor:
    """The GEMM kernels stage activations in 16-byte chunks."""
    return rows.clone() if rows.data_ptr() % 16 else rows


def torch_sees(*tensors: torch.Tensor) -> bool:
    """Whether a product of the tensors has to be a torch operation: autograd or
    a forward-mode level records it, a functorch transform or a tensor subclass
    or mode intercepts it, or autocast chooses its type."""
    return (not _STATE_KNOWN
            or torch.is_grad_enabled() and any(t.requires_grad for t in tensors)
            or torch.is_autocast_enabled("cuda")
            or any(type(t) not in (torch.Tensor, torch.nn.Parameter) for t in tensors)
            or torch.autograd.forward_ad._current_level >= 0
            or maybe_current_level() is not None
            or _len_torch_dispatch_stack() > 0
            # a default device is a mode too, one that leaves products alone
            or _len_torch_function_stack() > 0 and not all(
                isinstance(m, DeviceContext) for m in _get_current_function_mode_stack()))


def gemm_weight(layer: torch.nn.Module, gated: bool = False):
    """The weights a batched GEMM of the layer reads: its packed form when
    pack() made one of that kind, else the GGUF blocks."""
    p = getattr(layer, "q4_0_packed", None)
    if p is not None and p.gated == gated:
        return p
    return layer.qweight.reshape(-1)


class Q4_0Linear(torch.nn.Module):
    """A bare linear layer driven by Q4_0LinearMethod (used by the decode
    model and tests in place of vLLM's parallel linear classes)."""

    def __init__(self, input_size: int, output_partition_sizes: list[int], device=None):
        super().__init__()
        self.quant_method = Q4_0LinearMethod()
        self.quant_method.create_weights(self, input_size, output_partition_sizes, input_size,
                                         sum(output_partition_sizes), torch.bfloat16,
                                         device=device)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return self.quant_method.apply(self, x)
