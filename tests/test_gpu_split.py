"""Linears and channels-last convolutions whose k range is split over work-groups (few tiles, long k), against the
dequantized product in float64.

Bar: fp16 operands and fp32 sums, 2e-3 of the largest value plus the output's own rounding (conftest.out_tol, the bar
of every weight-only kernel)."""

import pytest
import torch
import torch.nn.functional as F

from tests.conftest import announce, out_tol
from tests.test_gpu_general import _act, _close, _gen, _weights

pytestmark = pytest.mark.gpu

# (M, N, K, bits, x dtype, out dtype, per_channel, activation, residual)
LINEAR = [
    (65, 100, 2048, 4, "float16", "float16", True, None, False),        # row and column tails, 32 stages
    (197, 768, 3072, 4, "float16", "bfloat16", True, None, True),
    (130, 257, 2112, 2, "bfloat16", "float32", False, "relu", False),   # 33 stages: ranges of unlike length; odd pitch
    (1000, 40, 3136, 3, "float32", "float16", True, "gelu", False),
]


@pytest.mark.parametrize("M,N,K,bits,xdt,ydt,pc,act,res", LINEAR)
def test_split_linear(gpu, M, N, K, bits, xdt, ydt, pc, act, res):
    from dimq_amd import _C, ops
    announce(f"split linear {M} {N} {K} {bits} {xdt} {ydt}")
    xdt, ydt = getattr(torch, xdt), getattr(torch, ydt)
    need = _C.lib.dimq_linear_codebook_full_workspace_bytes(M, K, N, bits, _C._DT[xdt])
    assert need >= 2 * M * N * 4
    g = _gen(M + N + K)
    packed, cb, w = _weights(N, K, bits, pc, g)
    x = torch.randn(M, K, generator=g).to(xdt)
    bias = torch.randn(N, generator=g)
    r = torch.randn(M, N, generator=g).to(ydt) if res else None
    y = ops.dimq_linear_codebook(x.to(gpu), packed.to(gpu), cb.to(gpu), bits, bias.to(gpu), N, K, out_dtype=ydt,
                                 residual=None if r is None else r.to(gpu), activation=act)
    _close(y, _act(x.double() @ w.T + bias.double(), r, act), out_tol(ydt))


# (B, C, H, W, OC, ks, stride, pad, bits, dtype, activation, residual)
CONV = [
    (1, 512, 7, 7, 512, 3, 1, 1, 2, "float16", None, False),
    (16, 512, 7, 7, 512, 3, 1, 1, 2, "bfloat16", "relu", True),
    (2, 192, 9, 11, 136, 5, 2, 2, 3, "float16", "relu", False),     # column tail, stride 2
    (1, 1024, 2, 3, 70, 3, 1, 1, 4, "bfloat16", None, True),        # every pixel beside the padding
]


def _conv(ops, x, packed, cb, bits, bias, oc, ks, stride, pad, ydt, r, act, gpu):
    cl = torch.channels_last
    packed = packed.to(gpu)
    prepared = ops.prepare_conv_weight(packed, bits, (oc, x.shape[1], ks, ks))
    return ops.dimq_conv2d_codebook(x.to(gpu).contiguous(memory_format=cl), packed, cb.to(gpu), bits,
                                    None if bias is None else bias.to(gpu), (oc, x.shape[1], ks, ks), stride, pad, 1, 1,
                                    out_dtype=ydt, prepared_weight=prepared, activation=act,
                                    residual=None if r is None else r.to(gpu).contiguous(memory_format=cl))


@pytest.mark.parametrize("B,C,H,W,OC,ks,stride,pad,bits,dt,act,res", CONV)
def test_split_conv(gpu, B, C, H, W, OC, ks, stride, pad, bits, dt, act, res):
    from dimq_amd import _C, ops
    announce(f"split conv {B} {C} {H} {W} {OC} {ks} {bits} {dt}")
    dt = getattr(torch, dt)
    g = _gen(B + C + OC)
    packed, cb, w = _weights(OC, C * ks * ks, bits, True, g)
    x = torch.randn(B, C, H, W, generator=g).to(dt)
    bias = torch.randn(OC, generator=g)
    ref = F.conv2d(x.double(), w.view(OC, C, ks, ks), bias.double(), stride, pad)
    r = torch.randn(ref.shape, generator=g).to(dt) if res else None
    code = _C._DT[dt]
    assert _C.lib.dimq_conv2d_codebook_workspace_bytes(
        code, 1, B, C, H, W, bits, 1, _C._DT[cb.dtype], OC, 1 << bits, OC, ks, ks, stride, stride, pad, pad, 1,
        1, 1, code, 1, int(res), 1 if act else 0, 0) >= 2 * ref.numel() * 4
    y = _conv(ops, x, packed, cb, bits, bias, OC, ks, stride, pad, dt, r, act, gpu)
    _close(y, _act(ref, r, act), out_tol(dt))


@pytest.mark.parametrize("where", ["tiny", "huge", "mixed", "zeros first"])
def test_split_range_guard(gpu, where):
    """Rows outside fp16's range, in whole tiles and beside ordinary ones, and k ranges that hold only zeros."""
    from dimq_amd import ops
    announce(f"split guard {where}")
    M, N, K = 150, 70, 2048
    g = _gen(K)
    packed, cb, w = _weights(N, K, 3, True, g)
    x = torch.randn(M, K, generator=g)
    x = x * {"tiny": 1e-9, "huge": 1e6}.get(where, 1.0)
    if where == "mixed":
        x[: M // 2] *= 1e6
    if where == "zeros first":
        x[:, : K // 2] = 0
    for xdt in (torch.float32, torch.bfloat16):
        y = ops.dimq_linear_codebook(x.to(xdt).to(gpu), packed.to(gpu), cb.to(gpu), 3, None, N, K,
                                     out_dtype=torch.float32)
        _close(y, x.to(xdt).double() @ w.T, 2e-3)
    C, H, W = 256, 5, 5
    packed, cb, w = _weights(70, C * 9, 3, True, g)
    xc = x.to(torch.bfloat16).reshape(-1)[: 3 * C * H * W].reshape(3, C, H, W)
    y = _conv(ops, xc, packed, cb, 3, None, 70, 3, 1, 1, torch.float32, None, None, gpu)
    _close(y, F.conv2d(xc.double(), w.view(70, C, 3, 3), None, 1, 1), 2e-3)
