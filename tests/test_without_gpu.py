"""Without a GPU every entry point says so in the package's own words."""
import pytest
import torch

pytestmark = pytest.mark.skipif(torch.cuda.is_available(), reason="needs a machine without a GPU")


@pytest.mark.parametrize("call", ["quantize_tensor", "dequantize_tensor", "quantize_tensor_for_all_procs", "quant_segments", "plan"])
def test_the_message(call):
    from super_gnn_amd import supergnn_ops as ops
    x, q, params = torch.zeros(4, 8), torch.zeros(4, 8, dtype=torch.uint8), torch.zeros(4, 2)
    segments = torch.tensor([0, 4], dtype=torch.int32)
    with pytest.raises(RuntimeError, match="super_gnn_amd needs a GPU"):
        if call == "quantize_tensor":
            ops.quantize_tensor(x, q, params, 8)
        elif call == "dequantize_tensor":
            ops.dequantize_tensor(q, x, params, 8)
        elif call == "quantize_tensor_for_all_procs":
            ops.quantize_tensor_for_all_procs(x, q, params, segments, 1, 8)
        elif call == "quant_segments":
            ops.quant_segments(segments, 8)
        else:
            ops.SpmmPlan(torch.tensor([0, 1]), torch.tensor([0]), 1)
