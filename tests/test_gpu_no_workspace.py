"""The kernels of the entry points without a workspace (what a C caller of those gets, and the ops when the allocator has
no room or an operand is off alignment): the generic tiles, the 8-bit tiles and the generic implicit GEMM with their range
guards, and the generic W4A4 tiles, through the C ABI."""

import pytest
import torch

import oracle
from tests.conftest import announce
from tests.test_gpu_general import _close, _weights
from tests.test_gpu_range import TOL, _codebook_case, _gen, _linear_no_workspace, _scaled

pytestmark = pytest.mark.gpu


def _call(f, *args):
    from dimq_amd import _C
    assert f(*args, torch.cuda.current_stream().cuda_stream) == 0, _C.lib.dimq_last_error()


@pytest.mark.parametrize("mode", ["huge", "tiny", "mixed", "one"])
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("name,M,N,K,bits", [("gemm_cb", 40, 100, 100, 2), ("gemm_cb_64x128", 130, 200, 100, 3),
                                             ("gemm_cb8", 40, 64, 256, 8), ("gemm_cb8_16", 17, 100, 100, 8),
                                             ("deep_64x128", 130, 200, 2048, 3), ("big_128x128", 2047, 2040, 2048, 2)])
def test_linear_range(gpu, name, M, N, K, bits, xdt, mode):
    announce(f"no workspace linear {name} {xdt} {mode}")
    g = _gen(M + N + K + bits)
    cb, packed = _codebook_case(N, K, bits, True, g)
    x, s = _scaled(torch.randn(M, K, generator=g), mode, g)
    x, bias = x.to(xdt), torch.randn(N, generator=g) * 0.1 * float(s.min())
    y = _linear_no_workspace(gpu, x, packed, cb, bits, bias, N, K)
    ref = oracle.linear_dequant_reference(x.float(), packed, bits, cb, N, K, bias)
    assert bool(torch.isfinite(y).all())
    assert oracle.rel_err(y, ref) <= TOL


# B, C, H, W, OC, K, stride, pad, groups, bits
CONV = [(2, 16, 10, 9, 32, 3, 1, 1, 1, 3), (2, 3, 31, 29, 16, 7, 2, 3, 1, 8), (2, 12, 9, 11, 24, 3, 1, 1, 4, 4)]


@pytest.mark.parametrize("mode", ["huge", "tiny", "one"])
@pytest.mark.parametrize("xdt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,C,H,W,OC,ks,st,pd,groups,bits", CONV)
def test_conv_range(gpu, B, C, H, W, OC, ks, st, pd, groups, bits, xdt, mode):
    from dimq_amd import _C
    announce(f"no workspace conv {C}x{H}x{W} k{ks} g{groups} b{bits} {xdt} {mode}")
    g = _gen(B + C + OC + bits)
    icg = C // groups
    cb, packed = _codebook_case(OC, icg * ks * ks, bits, True, g)
    x = _scaled(torch.randn(B, C, H, W, generator=g), mode, g)[0].to(xdt)
    ref = oracle.conv2d_dequant_reference(x.float(), packed, bits, cb, (OC, icg, ks, ks), None, st, pd, 1, groups)
    y = torch.empty(ref.shape, device=gpu)
    xg, pg, cg = x.to(gpu), packed.to(gpu), cb.to(gpu)
    _call(_C.lib.dimq_conv2d_codebook, xg.data_ptr(), _C._DT[xdt], _C.NCHW, B, C, H, W, pg.data_ptr(), pg.numel(), bits,
          None, 0, cg.data_ptr(), _C.F32, OC, 1 << bits, None, _C.F32, OC, ks, ks, st, st, pd, pd, 1, 1, groups,
          y.data_ptr(), _C.F32, _C.NCHW, 0)
    assert bool(torch.isfinite(y).all())
    assert oracle.rel_err(y, ref) <= TOL


@pytest.mark.parametrize("cdt", [torch.float16, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("xdt", [torch.float32, torch.bfloat16, torch.float64])
def test_generic_w4a4(gpu, cdt, xdt):
    """Exact codes and hi + lo codebook planes: 2e-6 of the largest value (tests/test_gpu_general.py)."""
    from dimq_amd import _C
    announce(f"no workspace w4a4 {cdt} {xdt}")
    for M, N, K in ((31, 354, 749), (70, 96, 256), (2, 155, 218)):
        g = _gen(M)
        packed, cb, w = _weights(N, K, 4, False, g, cdt)
        x, bias = torch.randn(M, K, generator=g).to(xdt), torch.randn(N, generator=g)
        y = torch.empty(M, N, device=gpu)
        xg, pg, cg, bg = x.to(gpu), packed.to(gpu), cb.to(gpu), bias.to(gpu)
        _call(_C.lib.dimq_linear_lut, xg.data_ptr(), _C._DT[xdt], M, pg.data_ptr(), pg.numel(), cg.data_ptr(),
              _C._DT[cdt], 16, 0.2371, 7, bg.data_ptr(), _C.F32, N, N, K, y.data_ptr())
        a = torch.from_numpy(oracle.quantize_act_u4(x.float(), 0.2371, 7)).double() - 7
        _close(y, 0.2371 * (a @ w.T) + bias.double(), 2e-6)
    for B, C, H, W, OC, ks, st, gr in ((2, 48, 9, 11, 96, 3, 2, 1), (2, 12, 6, 5, 10, 1, 1, 2), (1, 7, 8, 9, 5, 3, 1, 1)):
        g = _gen(C)
        packed, cb, w = _weights(OC, C // gr * ks * ks, 4, False, g, cdt)
        x, bias = torch.randn(B, C, H, W, generator=g).to(xdt), torch.randn(OC, generator=g)
        a = torch.from_numpy(oracle.quantize_act_u4(x, 0.25, 3)).double().reshape(x.shape) - 3
        ref = torch.nn.functional.conv2d(0.25 * a, w.view(OC, -1, ks, ks), bias.double(), st, ks // 2, 1, gr)
        y = torch.empty(ref.shape, device=gpu)
        xg, pg, cg, bg = x.to(gpu), packed.to(gpu), cb.to(gpu), bias.to(gpu)
        _call(_C.lib.dimq_conv2d_lut, xg.data_ptr(), _C._DT[xdt], B, C, H, W, pg.data_ptr(), pg.numel(), cg.data_ptr(),
              _C._DT[cdt], 16, 0.25, 3, bg.data_ptr(), _C.F32, OC, OC, C // gr, ks, ks, st, st, ks // 2, ks // 2, 1, 1,
              gr, y.data_ptr())
        _close(y, ref, 2e-6)
