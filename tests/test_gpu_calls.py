"""Argument errors of the native ops: the messages of the Python implementations they replaced."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.complex64, torch.int32, torch.bool, torch.float8_e4m3fn])
def test_unsupported_dtypes_are_named_as_torch_names_them(gpu, dt):
    from dimq_amd import ops
    x = torch.zeros(2, 4, device=gpu).to(dt)
    packed, cb = torch.zeros(4, dtype=torch.uint8, device=gpu), torch.zeros(16, device=gpu)
    with pytest.raises(RuntimeError, match=f"^unsupported dtype {dt}$"):
        ops.dimq_linear_codebook(x, packed, cb, 4, None, 2, 4)
