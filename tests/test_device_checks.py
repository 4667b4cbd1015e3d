"""Tensors that are not on the GPU are refused before anything is launched."""
import pytest
import torch


def _codes():
    return torch.zeros((2, 128), dtype=torch.int8), torch.ones((2, 2))


def test_engine_calls_refuse_cpu_tensors():
    from qwen35_amd.kernels import gemm
    q, s = _codes()
    out = torch.empty((2, 64), dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="must be on the GPU"):
        gemm.gemm_i8(q, s, torch.zeros((128, 64), dtype=torch.int8), torch.ones(64), out)
    with pytest.raises(ValueError, match="must be on the GPU"):
        gemm.gemm_i8(q, s, torch.zeros((64, 64), dtype=torch.uint8), torch.ones((2, 64)), out)


def test_linears_refuse_cpu_tensors():
    from qwen35_amd.kernels import linear
    with pytest.raises(ValueError, match="must be on the GPU"):
        linear.linear_w8(torch.zeros((2, 128), dtype=torch.float16), torch.zeros((128, 64), dtype=torch.int8),
                         torch.ones(64), torch.empty((2, 64), dtype=torch.float16))


@pytest.mark.gpu
def test_mixed_devices_are_refused():
    from qwen35_amd.kernels import gemm
    q, s = _codes()
    b, bs, out = torch.zeros((128, 64), dtype=torch.int8), torch.ones(64), torch.empty((2, 64), dtype=torch.bfloat16)
    for i in range(5):
        ts = [t.cuda() if j != i else t for j, t in enumerate((q, s, b, bs, out))]
        with pytest.raises(ValueError, match="must be on the GPU"):
            gemm.gemm_i8(*ts)
