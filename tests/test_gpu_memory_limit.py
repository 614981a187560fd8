"""Layers whose workspace the allocator has no room for run on the kernels that need none.  The shortage comes from the
allocator's own limit (set_per_process_memory_fraction), on the host."""

import pytest
import torch
import torch.nn.functional as F

import oracle
from tests.conftest import announce, out_tol
from tests.test_gpu_general import _close, _gen, _weights

pytestmark = pytest.mark.gpu


def _short_of(need, f):
    """f() while the allocator may take 6 MiB more, too little for `need` bytes."""
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (6 << 20)) / total)
    try:
        with pytest.raises(torch.OutOfMemoryError):
            torch.empty(need, dtype=torch.uint8, device="cuda")
        y = f()
        torch.cuda.synchronize()
        return y
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)


def test_layers_without_room_for_their_workspace(gpu):
    from dimq_amd import _C, ops
    g = _gen(1)
    M, N, K = 40, 4096, 2176
    x, w4 = torch.randn(M, K, generator=g).half(), _weights(N, K, 8, False, g)
    xg, pg, cg = x.to(gpu), w4[0].to(gpu), w4[1].to(gpu)
    announce("memory limit: linear, general path")
    y = _short_of(_C.lib.dimq_linear_codebook_full_workspace_bytes(M, K, N, 8, _C.F16),
                  lambda: ops.dimq_linear_codebook(xg, pg, cg, 8, None, N, K))
    _close(y, x.double() @ w4[2].T, out_tol(torch.float16))

    packed, cb, w = _weights(N, K, 4, False, g, torch.float32)
    pg, cg = packed.to(gpu), cb.to(gpu)
    announce("memory limit: w4a4 linear, general path")
    y = _short_of(_C.lib.dimq_linear_lut_full_workspace_bytes(_C.F16, M, N, K, _C.F32),
                  lambda: ops.dimq_linear_lut(xg, pg, cg, 0.25, 3, None, N, K))
    a = torch.from_numpy(oracle.quantize_act_u4(x.float(), 0.25, 3)).double() - 3
    _close(y, 0.25 * (a @ w.T), 2e-6)

    M, N, K = 2048, 256, 4096
    x, (packed, cb, w) = torch.randn(M, K, generator=g), _weights(N, K, 4, True, g)
    xg, pg, cg = x.to(gpu), packed.to(gpu), cb.to(gpu)
    announce("memory limit: linear, pre-decoded weights")
    y = _short_of(_C.lib.dimq_linear_codebook_full_workspace_bytes(M, K, N, 4, _C.F32),
                  lambda: ops.dimq_linear_codebook(xg, pg, cg, 4, None, N, K, out_dtype=torch.float16))
    _close(y, x.double() @ w.T, out_tol(torch.float16))

    B, C, H = 4, 256, 64
    x, (packed, cb, w) = torch.randn(B, C, H, H, generator=g), _weights(16, C, 4, True, g)
    xg, pg, cg = x.to(gpu), packed.to(gpu), cb.to(gpu)
    announce("memory limit: conv, general path")
    y = _short_of(8 << 20, lambda: ops.dimq_conv2d_codebook(xg, pg, cg, 4, None, (16, C, 1, 1), 1, 0, 1, 1))
    _close(y, F.conv2d(x.double(), w.view(16, C, 1, 1)), out_tol(torch.float32))
    cg = cb[0].to(gpu)
    announce("memory limit: w4a4 conv, general path")
    y = _short_of(8 << 20, lambda: ops.dimq_conv2d_lut(xg, pg, cg, 0.25, 3, None, (16, C, 1, 1), 1, 0, 1, 1))
    w = cb[0].double()[torch.from_numpy(oracle.unpack_bits(packed, 16 * C, 4)).long()].view(16, C, 1, 1)
    a = torch.from_numpy(oracle.quantize_act_u4(x, 0.25, 3)).double().reshape(x.shape) - 3
    _close(y, F.conv2d(0.25 * a, w), 2e-6)
