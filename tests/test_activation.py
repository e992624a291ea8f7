"""silu_and_mul's argument checks (CPU only, no kernel launches)."""
import pytest
import torch

from nanovllm_amd import _lib
from nanovllm_amd.layers.activation import silu_and_mul


@pytest.mark.parametrize("out", [torch.empty(4, 16), torch.empty(3, 16, dtype=torch.bfloat16),
                                 torch.empty(4, 8, dtype=torch.bfloat16), torch.empty(4, 32, dtype=torch.bfloat16),
                                 torch.empty(64, dtype=torch.bfloat16), torch.empty(16, 4, dtype=torch.bfloat16).t(),
                                 torch.empty(4, 16, dtype=torch.bfloat16, device="meta")])
def test_silu_and_mul_refuses_a_wrong_out(out, monkeypatch):
    def load():
        raise AssertionError("reached the kernel")
    monkeypatch.setattr(_lib, "load", load)
    with pytest.raises(ValueError, match="silu_and_mul: out"):
        silu_and_mul(torch.zeros(4, 32, dtype=torch.bfloat16), out=out)
