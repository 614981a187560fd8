"""CPU-only checks of what the native half's callables accept and which route a size query announces: nothing here
launches a kernel."""

import pytest
import torch


@pytest.mark.parametrize("scale,zp", [(0.25, 7), (0.25, 7.0), (torch.tensor(0.25), torch.tensor(7.0)), (1, True)])
def test_lut_callables_take_any_real_scale_and_zero_point(scale, zp):
    """dimq_amd._C.linear_lut / conv2d_lut convert the scale with float() and the zero point with int(), so a float
    zero point read from a checkpoint reaches the op's own checks (here: that its tensors are on the GPU)."""
    from dimq_amd import _C
    pw, cb = torch.zeros(2, dtype=torch.uint8), torch.zeros(16)
    with pytest.raises(RuntimeError, match="linear_lut expects CUDA input"):
        _C.linear_lut(torch.zeros(1, 4), pw, cb, scale, zp, None, 1, 4)
    with pytest.raises(RuntimeError, match="conv2d_lut expects CUDA input"):
        _C.conv2d_lut(torch.zeros(1, 4, 1, 1), pw, cb, scale, zp, None, 1, 4, 1, 1, 1, 1, 0, 0, 1, 1, 1)
