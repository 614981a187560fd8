"""Linears of 65 to 2,047 rows on either side of the rule that picks the 128x128 tile over the 64x128 one, against the
dequantized product in float64.

Bar: fp16 operands and fp32 sums, 2e-3 of the largest value plus the output's own rounding (conftest.out_tol, the bar
of every weight-only kernel)."""

import pytest
import torch

import oracle
from tests.conftest import announce, out_tol
from tests.test_gpu_general import _act, _close, _gen, _weights

pytestmark = pytest.mark.gpu

# (M, N, K, bits, x dtype, out dtype, activation, residual): 407 tiles of 128x128 and up, then 396 and 11 * 48 (their
# last round is short), 4-bit fp16 (the other tile at any count)
LINEAR = [
    (1300, 4700, 2048, 2, "float16", "float16", None, False),
    (1281, 4609, 2112, 3, "bfloat16", "float32", "relu", False),     # row and column tails, odd pitch
    (1300, 4700, 2048, 4, "bfloat16", "bfloat16", None, True),
    (1300, 4700, 2048, 3, "float32", "float16", "gelu", False),
    (1300, 4600, 2048, 2, "float16", "float16", None, True),
    (1300, 6100, 2048, 3, "bfloat16", "bfloat16", None, False),
    (1300, 4700, 2048, 4, "float16", "float16", "relu", False),
    (1100, 8100, 2048, 2, "bfloat16", "bfloat16", None, False),      # 576 tiles: 2-bit only
    (1100, 8100, 2048, 3, "bfloat16", "bfloat16", None, False),
    (1500, 4096, 992, 4, "float16", "float16", None, False),         # K % 32 == 0: the 64x128 register-codebook tiles
    (1501, 4100, 992, 3, "float32", "bfloat16", "relu", True),
]


@pytest.mark.parametrize("M,N,K,bits,xdt,ydt,act,res", LINEAR)
def test_tile_choice_below_2048_rows(gpu, M, N, K, bits, xdt, ydt, act, res):
    from dimq_amd import ops
    announce(f"tiles {M} {N} {K} {bits} {xdt}")
    xdt, ydt = getattr(torch, xdt), getattr(torch, ydt)
    g = _gen(M + N + bits)
    packed, cb, w = _weights(N, K, bits, True, g)
    x, bias = torch.randn(M, K, generator=g).to(xdt), torch.randn(N, generator=g)
    r = torch.randn(M, N, generator=g).to(ydt) if res else None
    y = ops.dimq_linear_codebook(x.to(gpu), packed.to(gpu), cb.to(gpu), bits, bias.to(gpu), N, K, out_dtype=ydt,
                                 residual=None if r is None else r.to(gpu), activation=act)
    _close(y, _act(x.double() @ w.T + bias.double(), r, act), out_tol(ydt))


@pytest.mark.parametrize("M,N,K", [(512, 8192, 2176), (517, 8200, 2304)])
@pytest.mark.parametrize("cdt,xdt", [(torch.float32, torch.float32), (torch.bfloat16, torch.float16)])
def test_w4a4_products_that_fill_the_chip(gpu, M, N, K, cdt, xdt):
    """Codebooks that are not fp16 on the generic A4 tiles: exact codes and hi + lo planes, 2e-6 of the largest value."""
    from dimq_amd import ops
    announce(f"w4a4 tiles {M} {N} {K} {cdt} {xdt}")
    g = _gen(N)
    packed, cb, w = _weights(N, K, 4, False, g, cdt)
    x, bias = torch.randn(M, K, generator=g).to(xdt), torch.randn(N, generator=g)
    y = ops.dimq_linear_lut(x.to(gpu), packed.to(gpu), cb.to(gpu), 0.2371, 7, bias.to(gpu), N, K)
    a = torch.from_numpy(oracle.quantize_act_u4(x.float(), 0.2371, 7)).double() - 7
    _close(y, 0.2371 * (a @ w.T) + bias.double(), 2e-6)


@pytest.mark.parametrize("M,K", [(130, 768), (130, 3072), (1000, 768), (1000, 3072), (300, 2112)])
@pytest.mark.parametrize("act,xdt,ydt", [("relu", "float16", "float16"), ("gelu", "bfloat16", "float32")])
def test_epilogues_the_large_tiles_lack(gpu, M, K, act, xdt, ydt):
    """Residual and activation together: k split where the same layer without them splits it, the generic tiles where
    not; a workspace from the size query is then used by neither or by both."""
    from dimq_amd import ops
    announce(f"residual + {act} {M} {K} {xdt}")
    N = 768
    xdt, ydt = getattr(torch, xdt), getattr(torch, ydt)
    g = _gen(M + K)
    packed, cb, w = _weights(N, K, 4, True, g)
    x, bias, r = torch.randn(M, K, generator=g).to(xdt), torch.randn(N, generator=g), torch.randn(M, N, generator=g).to(ydt)
    y = ops.dimq_linear_codebook(x.to(gpu), packed.to(gpu), cb.to(gpu), 4, bias.to(gpu), N, K, out_dtype=ydt,
                                 residual=r.to(gpu), activation=act)
    _close(y, _act(x.double() @ w.T + bias.double(), r, act), out_tol(ydt))
