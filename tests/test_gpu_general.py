"""The general pre-laid path (gemm_gen.hip): codebook Linears and Conv2ds of any size, layout, dtype and bit width
against the dequantized product in float64.

Bars: fp16 operands and fp32 sums, 2e-3 of the largest value plus the output's own rounding (conftest.out_tol, the
bar of every weight-only kernel); W4A4, whose operands are exact, 2e-6 of the largest value: fp32 sums of up to
2,304 products, each sum rounded to 2^-24."""

import pytest
import torch
import torch.nn.functional as F

import oracle
from tests.conftest import announce, out_tol

pytestmark = pytest.mark.gpu


def _gen(seed):
    return torch.Generator().manual_seed(seed)


def _weights(n, k, bits, per_channel, g, dtype=torch.float32):
    cb = (torch.randn(n if per_channel else 1, 1 << bits, generator=g) / k ** 0.5).sort(dim=1).values.to(dtype)
    idx = torch.randint(0, 1 << bits, (n, k), generator=g, dtype=torch.uint8)
    w = torch.gather(cb.double().expand(n, -1), 1, idx.long())
    return torch.from_numpy(oracle.pack_bits(idx, bits)), (cb if per_channel else cb[0]), w


def _close(y, ref, tol):
    y, ref = y.double().cpu(), ref.double()
    assert y.shape == ref.shape and bool(torch.isfinite(y).all())
    err, top = float((y - ref).abs().max()), float(ref.abs().max())
    assert err <= tol * top, (err / top, tol)


def _act(y, res, act):
    y = y if res is None else y + res.double()
    return torch.relu(y) if act == "relu" else F.gelu(y) if act == "gelu" else y


# (M, N, K, bits, x dtype, out dtype, per_channel, activation, residual)
LINEAR = [
    (17, 33, 33, 3, "float16", "float16", True, None, False),        # every size off its tile; one k stage and a bit
    (31, 70, 749, 4, "float32", "float32", False, "relu", True),     # split k, rows converted
    (64, 536, 3183, 4, "float16", "bfloat16", True, "gelu", False),  # odd K: fp16 rows copied to the padded pitch
    (65, 64, 96, 8, "float16", "float32", True, None, False),        # K off the 64-k stages: rows copied
    (65, 64, 192, 8, "float16", "float32", True, None, False),       # K % 64 == 0: rows read in place
    (130, 257, 1000, 8, "bfloat16", "bfloat16", False, None, True),
    (300, 200, 150, 2, "bfloat16", "float16", True, "relu", True),
    (4133, 1100, 91, 4, "float32", "float16", True, None, False),    # many tiles each way, odd pitch
    (33000, 40, 65, 3, "float16", "float16", True, None, True),      # one column of many tiles
]


@pytest.mark.parametrize("M,N,K,bits,xdt,ydt,pc,act,res", LINEAR)
def test_general_linear(gpu, M, N, K, bits, xdt, ydt, pc, act, res):
    from dimq_amd import ops
    announce(f"general linear {M} {N} {K} {bits} {xdt} {ydt}")
    g = _gen(M + N + K)
    xdt, ydt = getattr(torch, xdt), getattr(torch, ydt)
    packed, cb, w = _weights(N, K, bits, pc, g)
    x = torch.randn(M, K, generator=g).to(xdt)
    bias = torch.randn(N, generator=g)
    r = torch.randn(M, N, generator=g).to(ydt) if res else None
    y = ops.dimq_linear_codebook(x.to(gpu), packed.to(gpu), cb.to(gpu), bits, bias.to(gpu), N, K, out_dtype=ydt,
                                 residual=None if r is None else r.to(gpu), activation=act)
    _close(y, _act(x.double() @ w.T + bias.double(), r, act), out_tol(ydt))


# (B, C, H, W, OC, KH, KW, stride, pad, dil, groups, bits, x dtype, out dtype, NHWC, activation, residual)
CONV = [
    (1, 3, 9, 7, 8, 3, 3, 1, 1, 1, 1, 3, "float16", "float16", False, None, False),
    (2, 6, 11, 7, 4, 3, 2, (2, 1), (1, 0), (1, 2), 2, 4, "bfloat16", "float32", True, "relu", True),
    (3, 100, 13, 10, 130, 3, 3, 1, 2, 2, 1, 8, "float32", "float32", False, "relu", True),
    (5, 24, 19, 15, 64, 5, 5, 1, 2, 1, 1, 8, "float16", "float16", True, "gelu", False),   # read in place
    (4, 256, 14, 14, 96, 3, 3, 1, 1, 1, 1, 2, "float16", "float32", False, None, False),   # split k
    (2, 128, 9, 9, 72, 1, 1, 2, 0, 1, 2, 4, "float16", "bfloat16", True, None, False),     # groups, in place
    (17, 65, 60, 33, 140, 3, 3, 1, 1, 1, 1, 4, "float16", "float16", False, "relu", False),  # many tiles each way
    (40, 16, 40, 41, 8, 3, 3, 1, 1, 1, 1, 3, "bfloat16", "bfloat16", False, None, False),  # one column of many tiles
    (1, 8, 5, 5, 16, 7, 7, 1, 3, 1, 1, 4, "float32", "float16", True, None, False),        # taps mostly outside
]


@pytest.mark.parametrize("B,C,H,W,OC,KH,KW,stride,pad,dil,groups,bits,xdt,ydt,nhwc,act,res", CONV)
def test_general_conv(gpu, B, C, H, W, OC, KH, KW, stride, pad, dil, groups, bits, xdt, ydt, nhwc, act, res):
    from dimq_amd import ops
    announce(f"general conv {B} {C} {H} {W} {OC} {KH} {KW} {stride} {pad} {dil} {groups} {bits} {xdt} {ydt} {nhwc}")
    g = _gen(B + C + OC + KH)
    xdt, ydt = getattr(torch, xdt), getattr(torch, ydt)
    mf = torch.channels_last if nhwc else torch.contiguous_format
    packed, cb, w = _weights(OC, C // groups * KH * KW, bits, True, g)
    x = torch.randn(B, C, H, W, generator=g).to(xdt)
    bias = torch.randn(OC, generator=g)
    ref = F.conv2d(x.double(), w.view(OC, -1, KH, KW), bias.double(), stride, pad, dil, groups)
    r = torch.randn(ref.shape, generator=g).to(ydt) if res else None
    y = ops.dimq_conv2d_codebook(x.to(gpu).contiguous(memory_format=mf), packed.to(gpu), cb.to(gpu), bits, bias.to(gpu),
                                 (OC, C // groups, KH, KW), stride, pad, dil, groups, out_dtype=ydt,
                                 residual=None if r is None else r.to(gpu).contiguous(memory_format=mf), activation=act)
    assert y.is_contiguous(memory_format=mf)
    _close(y, _act(ref, r, act), out_tol(ydt))


@pytest.mark.parametrize("where", ["tiny", "huge", "mixed"])
@pytest.mark.parametrize("M,N,K", [(90, 70, 200), (300, 40, 75)])
@pytest.mark.parametrize("xdt", ["float32", "bfloat16"])
def test_general_range_guard(gpu, where, M, N, K, xdt):
    """Rows outside fp16's range, in whole tiles and beside ordinary ones, with and without a split k range."""
    from dimq_amd import ops
    announce(f"general guard {where} {M} {N} {K} {xdt}")
    g = _gen(M + K)
    packed, cb, w = _weights(N, K, 3, True, g)
    x = torch.randn(M, K, generator=g)
    x = x * {"tiny": 1e-9, "huge": 1e6}.get(where, 1.0)
    if where == "mixed":
        x[: M // 2] *= 1e6
    x = x.to(getattr(torch, xdt))
    y = ops.dimq_linear_codebook(x.to(gpu), packed.to(gpu), cb.to(gpu), 3, None, N, K, out_dtype=torch.float32)
    _close(y, x.double() @ w.T, 2e-3)
    xc = x[:, : K // 25 * 25].reshape(M, -1, 5, 5)
    packed, cb, w = _weights(24, xc.shape[1] * 9, 3, True, g)
    y = ops.dimq_conv2d_codebook(xc.to(gpu), packed.to(gpu), cb.to(gpu), 3, None, (24, xc.shape[1], 3, 3), 1, 1, 1, 1,
                                 out_dtype=torch.float32)
    _close(y, F.conv2d(xc.double(), w.view(24, -1, 3, 3), None, 1, 1), 2e-3)


@pytest.mark.parametrize("cdt", ["float16", "float32", "bfloat16"])
@pytest.mark.parametrize("xdt", ["float32", "float16", "float64"])
def test_general_w4a4(gpu, cdt, xdt):
    """The reference's own ops on shapes off the fast kernels: codes formed in the first launch, codebooks that are
    not fp16 as two weight planes (hi + lo)."""
    from dimq_amd import ops
    announce(f"general w4a4 {cdt} {xdt}")
    cdt, xdt = getattr(torch, cdt), getattr(torch, xdt)
    for scale, zp, (M, N, K) in ((0.2371, 7, (31, 354, 749)), (0.25, 0, (200, 65, 96)), (0.2, 8, (2, 155, 218))):
        g = _gen(M)
        packed, cb, w = _weights(N, K, 4, False, g, cdt)
        x, bias = torch.randn(M, K, generator=g).to(xdt), torch.randn(N, generator=g)
        y = ops.dimq_linear_lut(x.to(gpu), packed.to(gpu), cb.to(gpu), scale, zp, bias.to(gpu), N, K)
        a = torch.from_numpy(oracle.quantize_act_u4(x.float(), scale, zp)).double() - zp
        _close(y, scale * (a @ w.T) + bias.double(), 2e-6)
    for scale, zp, (B, C, H, W, OC, ks, st, gr) in ((0.2371, 7, (2, 48, 9, 11, 96, 3, 2, 1)), (0.25, 3, (3, 256, 7, 7, 64, 3, 1, 1)),
                                                    (0.2, 0, (2, 12, 6, 5, 10, 1, 1, 2))):
        g = _gen(C)
        packed, cb, w = _weights(OC, C // gr * ks * ks, 4, False, g, cdt)
        x, bias = torch.randn(B, C, H, W, generator=g).to(xdt), torch.randn(OC, generator=g)
        y = ops.dimq_conv2d_lut(x.to(gpu), packed.to(gpu), cb.to(gpu), scale, zp, bias.to(gpu), (OC, C // gr, ks, ks),
                                st, ks // 2, 1, gr)
        a = torch.from_numpy(oracle.quantize_act_u4(x.float(), scale, zp)).double().reshape(x.shape) - zp
        _close(y, F.conv2d(scale * a, w.view(OC, -1, ks, ks), bias.double(), st, ks // 2, 1, gr), 2e-6)


def test_general_graph_replay(gpu):
    """A captured call (three launches, workspace from the graph's pool) gives the eager result on every replay."""
    from dimq_amd import ops
    announce("general graph replay")
    g = _gen(5)
    packed, cb, _ = _weights(64, 256 * 9, 2, True, g)
    x = torch.randn(2, 256, 14, 14, generator=g).half().to(gpu)
    call = lambda: ops.dimq_conv2d_codebook(x, packed, cb, 2, None, (64, 256, 3, 3), 1, 1, 1, 1)  # noqa: E731
    packed, cb = packed.to(gpu), cb.to(gpu)
    call()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = call()
    for k in range(3):
        x.copy_(torch.randn(x.shape, generator=g).half())
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, call())
