"""Tied LM head as a Q4_0 GEMV, plus greedy sampling on the device.

Mirrors Q6HeadMethod (src/spark_vllm_ascend/integration/head.py:12-16,31):
the head layer keeps its tied bf16 embedding weight, gains a packed
quantized buffer, and its ``quant_method`` is swapped for a method whose
``apply`` serves bf16 input of 1 to 16 rows (batched decode) with the native
kernels and defers to a plain bf16 matmul otherwise: more rows, a bias,
tensors or blocks the batched kernel cannot read (gemm_takes), or a product
that torch has to see (linear.torch_sees).  The quantized head here is Q4_0
[vocab, hidden] (the reference model's head is Q6_K), and the tied
embedding is bf16(dequantized head), the tying the reference prepares at
src/tools/deployment/prepare_head.py:27.
"""
from __future__ import annotations

import torch

from ..native import torch_ops
from .linear import GEMM_MAX_ROWS, aligned16, torch_sees
from .weights import dequantize_bf16, row_bytes


class Q4_0HeadMethod:
    def apply(self, layer: torch.nn.Module, x: torch.Tensor,
              bias: torch.Tensor | None = None) -> torch.Tensor:
        vocab, hidden = layer.weight.shape
        if x.shape == (1, hidden) and x.dtype == torch.bfloat16 and bias is None:
            return torch_ops.q4_0_gemv(x.contiguous(), layer.q4_0_head, vocab, hidden)
        if (x.dim() == 2 and 2 <= x.shape[0] <= GEMM_MAX_ROWS and x.shape[1] == hidden
                and x.dtype == torch.bfloat16 and bias is None and hidden % 64 == 0
                and gemm_pays(x.shape[0], vocab, hidden) and gemm_takes(layer, x)
                and not layer.weight.requires_grad and not torch_sees(x, layer.weight)):
            return torch_ops.q4_0_gemm(aligned16(x.contiguous()), layer.q4_0_head, vocab, hidden)
        out = torch.nn.functional.linear(x, layer.weight)
        return out if bias is None else out + bias


def gemm_pays(rows: int, vocab: int, hidden: int) -> bool:
    """Whether q4_0_gemm beats the bf16 product.  It reads a quarter of the
    bytes (151936 x 2560: 8 rows 53 us, 16 rows 102, bf16 242; 8000 x 512 3.3 and
    7.6), but above 8 rows its time grows faster with K, and a short bf16 product
    is then the faster: 1000 x 8192 at 8 rows 6.8 against 8.3, at 9 rows 9.3; 16
    rows of 32000 x 3072 32.4 against 31.6, 12 rows 29.0.
    (Hidden sizes to 8192 measured above 8 rows.)"""
    return (rows <= 8 or hidden <= 2560 or vocab >= 65536 and hidden <= 8192
            or rows <= 12 and (hidden <= 5120 or vocab >= 4000 and hidden <= 8192))


def gemm_takes(layer: torch.nn.Module, x: torch.Tensor) -> bool:
    """Whether q4_0_gemm can read x and the layer's blocks, and the bf16 product
    it stands for would take x."""
    w, blocks = layer.weight, layer.q4_0_head
    return (x.is_cuda and w.device == x.device == blocks.device and w.dtype == x.dtype
            and blocks.is_contiguous() and blocks.data_ptr() % 4 == 0)


class TiedQ4_0Head(torch.nn.Module):
    """Embedding/LM-head pair sharing one Q4_0 tensor."""

    def __init__(self, q4_0_blocks: torch.Tensor, vocab: int, hidden: int):
        super().__init__()
        if tuple(q4_0_blocks.shape) != (vocab, row_bytes(hidden)):
            raise ValueError("head blocks must be uint8 [vocab, hidden/32*18]")
        self.register_buffer("q4_0_head", q4_0_blocks.contiguous())
        self.weight = torch.nn.Parameter(dequantize_bf16(self.q4_0_head, vocab, hidden),
                                         requires_grad=False)
        self.quant_method = Q4_0HeadMethod()

    def logits(self, x: torch.Tensor) -> torch.Tensor:
        return self.quant_method.apply(self, x)

    def embed(self, ids: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
        return torch_ops.embedding(self.weight, ids, out=out)


def greedy_sample(logits: torch.Tensor, out: torch.Tensor | None = None,
                  keys: torch.Tensor | None = None) -> torch.Tensor:
    """argmax over the vocabulary (temperature 0), lowest index on ties; keys:
    torch_ops.argmax's workspace."""
    return torch_ops.argmax(logits, out=out, keys=keys)
