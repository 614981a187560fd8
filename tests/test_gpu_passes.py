"""The general pre-laid path on inputs whose layout exceeds its workspace bound: whole images (Linear: rows) in several
passes over one workspace, the last pass shorter.

Bars: those of the path's other tests (conftest.out_tol; W4A4 2e-6 of the largest value)."""

import pytest
import torch
import torch.nn.functional as F

import oracle
from tests.conftest import announce, out_tol
from tests.test_gpu_general import _act, _close, _gen, _weights

pytestmark = pytest.mark.gpu

# (B, C, groups, OC, H, W, x dtype, out dtype, NHWC, activation, residual): two passes each, of 35, 51 and 45 images
CONV = [
    (69, 16, 16, 16, 112, 112, "float32", "float32", False, "relu", True),
    (101, 16, 16, 32, 112, 112, "float16", "float16", False, None, True),
    (89, 66, 33, 66, 56, 99, "bfloat16", "bfloat16", True, None, False),
]


@pytest.mark.parametrize("B,C,groups,OC,H,W,xdt,ydt,nhwc,act,res", CONV)
def test_conv_in_passes(gpu, B, C, groups, OC, H, W, xdt, ydt, nhwc, act, res):
    from dimq_amd import ops
    announce(f"conv passes {B}x{C}x{H}x{W} g{groups} {xdt}")
    g = _gen(B + C)
    xdt, ydt = getattr(torch, xdt), getattr(torch, ydt)
    mf = torch.channels_last if nhwc else torch.contiguous_format
    packed, cb, w = _weights(OC, C // groups * 9, 4, True, g)
    x, bias = torch.randn(B, C, H, W, generator=g).to(xdt), torch.randn(OC, generator=g)
    x[-1] *= 3.0  # the last image differs in size from the first pass's
    ref = F.conv2d(x.float(), w.view(OC, -1, 3, 3).float(), bias, 1, 1, 1, groups)
    r = torch.randn(ref.shape, generator=g).to(ydt) if res else None
    y = ops.dimq_conv2d_codebook(x.to(gpu).contiguous(memory_format=mf), packed.to(gpu), cb.to(gpu), 4, bias.to(gpu),
                                 (OC, C // groups, 3, 3), 1, 1, 1, groups, out_dtype=ydt, activation=act,
                                 residual=None if r is None else r.to(gpu).contiguous(memory_format=mf))
    _close(y, _act(ref.double(), r, act), out_tol(ydt))


def test_w4a4_conv_in_passes(gpu):
    from dimq_amd import ops
    announce("w4a4 conv passes")
    g = _gen(9)
    B, C, H, W = 90, 16, 112, 112
    packed, cb, w = _weights(C, 9, 4, False, g)
    x, bias = torch.randn(B, C, H, W, generator=g), torch.randn(C, generator=g)
    y = ops.dimq_conv2d_lut(x.to(gpu), packed.to(gpu), cb.to(gpu), 0.25, 3, bias.to(gpu), (C, 1, 3, 3), 1, 1, 1, C)
    a = torch.from_numpy(oracle.quantize_act_u4(x, 0.25, 3)).float().reshape(x.shape) - 3
    _close(y, F.conv2d(0.25 * a, w.view(C, 1, 3, 3).float(), bias, 1, 1, 1, C), 2e-6)


@pytest.mark.parametrize("xdt", [torch.float32, torch.float16])
def test_linear_in_passes(gpu, xdt):
    """K 3 pads to a 64-k stage: 2,033,600 fp32 rows (128 + 4 bytes each) fill the bound."""
    from dimq_amd import ops
    announce(f"linear passes {xdt}")
    g = _gen(3)
    M, N, K = 2_200_003, 5, 3
    packed, cb, w = _weights(N, K, 4, True, g)
    x = torch.randn(M, K, generator=g).to(xdt)
    r = torch.randn(M, N, generator=g).half()
    y = ops.dimq_linear_codebook(x.to(gpu), packed.to(gpu), cb.to(gpu), 4, None, N, K, out_dtype=torch.float32,
                                 residual=r.to(gpu), activation="relu")
    _close(y, _act(x.double() @ w.T, r, "relu"), out_tol(torch.float32))
