"""SiLU-and-multiply (HIP sd_silu_mul): SiluAndMul.forward of nanovllm/layers/activation.py:8-11 in one launch, with
the roundings of its eager operations."""
import torch

from nanovllm_amd import _lib


def silu_and_mul(x: torch.Tensor, out: torch.Tensor | None = None) -> torch.Tensor:
    """silu(gate) * up for x = [gate | up], bf16 [rows, 2 * columns] with unit column stride."""
    if x.dtype != torch.bfloat16 or x.dim() != 2 or x.shape[1] % 2 or x.stride(1) != 1:
        raise ValueError("silu_and_mul: bf16 [rows, 2 * columns] with unit column stride required")
    M, half = x.shape[0], x.shape[1] // 2
    if out is None:
        out = torch.empty(M, half, dtype=x.dtype, device=x.device)
    if out.dtype != x.dtype or out.shape != (M, half) or out.stride(1) != 1 or out.device != x.device:
        raise ValueError("silu_and_mul: out must be bf16 [rows, columns] with unit column stride on x's device")
    _lib.check(_lib.load().sd_silu_mul(x.data_ptr(), x.stride(0), M, half, out.data_ptr(), out.stride(0),
                                       _lib.stream_of(x.device)), "sd_silu_mul")
    return out
