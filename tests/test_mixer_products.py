"""The products that a mixer names for the tuner are the ones that its steps run (host only)."""
import pytest
import torch

from arle_amd.parts.base import Runtime
from arle_amd.parts.mlstm import MLSTMMixer


@pytest.mark.parametrize("dtype,widths", [(torch.bfloat16, [("qkvg", 512), ("qkvgif", 544), ("o", 96)]), (torch.float32, [])])
def test_the_mlstm_names_the_product_of_its_decoded_rows(dtype, widths):
    params = dict(hidden_size=96, heads=4, key_dim=32, value_dim=32, gate_cap=15.0, eps=1e-6)
    tensors = {name: torch.zeros(decl.shape, dtype=dtype) for name, decl in MLSTMMixer.declare_weights(params).items()}
    mixer = MLSTMMixer(params, tensors, Runtime(device=torch.device("cpu"), act_dtype=dtype))
    assert [(name, n) for name, n, *_ in mixer.products()] == widths
    assert all(k == (128 if name == "o" else 96) for name, _, k, *_ in mixer.products())
    if mixer.whole is not None:
        assert [p[-1] for p in mixer.products()] == [None, "norm", "norm"]
