"""Stem conv at batches of every band height: each image's outputs are those of the batch whose bands are whole."""
import pytest
import torch

from tests.conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", ["nchw", "nhwc"])
@pytest.mark.parametrize("H,W,K,OC,out", [
    (96, 96, 7, 64, torch.float16),   # 48 rows of 48 outputs: batches of 1 to 11 halve the 8-row bands
    (61, 58, 7, 40, torch.float32),   # 31 x 29: ragged last band, no whole 8-pixel runs
    (34, 36, 3, 64, torch.bfloat16),  # 17 x 18: whole 8-pixel runs at eight and four rows only
])
def test_stem_band_heights(gpu, layout, H, W, K, OC, out):
    from dimq_amd import ops

    g = torch.Generator().manual_seed(H * W + K)
    n = OC * 3 * K * K
    packed = torch.randint(0, 256, (n,), generator=g, dtype=torch.uint8).to(gpu)
    cb = (torch.randn(OC, 256, generator=g) * 0.1).sort(dim=1).values.to(gpu)
    bias = torch.randn(OC, generator=g).to(gpu)
    x = torch.randn(260, 3, H, W, generator=g).half().to(gpu)  # over 512 whole bands

    def run(xb):
        xb = xb.to(memory_format=torch.channels_last) if layout == "nhwc" else xb.contiguous()
        return ops.dimq_conv2d_codebook(xb, packed, cb, 8, bias, (OC, 3, K, K), (2, 2), (K // 2, K // 2), (1, 1), 1,
                                        out_dtype=out)

    full = run(x)
    for b in (1, 2, 3, 7, 11, 16, 33, 60):
        announce(f"stem bands {layout} {H}x{W} k{K} batch {b}")
        assert torch.equal(run(x[:b]), full[:b]), b  # the same sums in the same order
