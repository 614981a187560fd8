"""Nearest-centre assignment: the register form (up to 8 centres) and the sorted form (16, 256) at the counts where
one gives way to the next, aligned and unaligned rows, one, two and four trips per work-group, and centres whose gaps
force the full scan; exact against torch's argmin (the first of equal distances)."""

import pytest
import torch

from tests.conftest import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [1, 4, 5, 8, 9, 16, 17, 256])
@pytest.mark.parametrize("rows,n", [(3, 4), (2, 1025), (5, 4100), (300, 1028), (257, 7), (1, 270_001)])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_nearest_centre_forms(gpu, K, rows, n, dt):
    from dimq_amd import ops
    announce(f"nearest K={K} rows={rows} n={n} {dt}")
    g = torch.Generator().manual_seed(K * n)
    cases = [torch.randn(rows, K, generator=g),
             torch.randint(-6, 7, (rows, K), generator=g).float() * 0.25,    # duplicates and exact ties
             torch.randn(rows, K, generator=g) * 1e-19,                      # squares below the normal range
             1.0 + torch.randint(0, 4, (rows, K), generator=g) * 2.0 ** -23]  # gaps of an ulp, far from most weights
    special = torch.randn(rows, K, generator=g)
    special[0, K // 2] = float("inf")
    special[-1, K - 1] = float("nan")
    for c in cases + [special]:
        w = torch.randn(rows, n, generator=g).to(dt)
        w[0, :4] = torch.tensor([float("nan"), float("inf"), -1e30, 0.125]).to(dt)
        idx, val = ops.hard_quantize(w.to(gpu), c.to(gpu), True)
        for r in range(rows):
            want = ((w[r].float()[:, None] - c[r][None, :]) ** 2).argmin(1)
            assert torch.equal(idx[r].cpu().long(), want)
            assert torch.equal(val[r].cpu().isnan(), c[r][want].isnan())
            assert torch.equal(val[r].cpu().nan_to_num(), c[r][want].to(dt).nan_to_num())
    off = torch.randn(n + 1, generator=g).to(dt).to(gpu)[1:]  # rows off the vector loads' alignment
    idx, val = ops.hard_quantize(off, cases[0][0].to(gpu), False)
    assert torch.equal(idx.cpu().long(), ((off.cpu().float()[:, None] - cases[0][0][None, :]) ** 2).argmin(1))


@pytest.mark.parametrize("K", [8, 9, 16, 17, 64])
@pytest.mark.parametrize("n", [9, 64, 65, 256, 257, 352, 353])
def test_nearest_centre_row_lengths(gpu, K, n):
    """More rows than CUs at the lengths where one element per thread gives way to four."""
    from dimq_amd import ops
    announce(f"nearest rows of {n} K={K}")
    g = torch.Generator().manual_seed(K + n)
    w, c = torch.randn(700, n, generator=g), torch.randn(700, K, generator=g)
    c[1, 3] = c[1, 0]
    w[0, :4] = torch.tensor([float("nan"), float("inf"), -1e30, 0.125])
    idx, val = ops.hard_quantize(w.to(gpu), c.to(gpu), True)
    want = ((w[:, :, None] - c[:, None, :]) ** 2).argmin(2)
    assert torch.equal(idx.cpu().long(), want)
    assert torch.equal(val.cpu(), torch.gather(c, 1, want))


@pytest.mark.parametrize("K", [8, 16, 256])
@pytest.mark.parametrize("rows,n", [(4096, 1028), (4100, 1025),   # two trips of 1,024, the second nearly empty
                                    (2100, 4100), (2100, 4099),   # four, the second work-group of a row with one
                                    (1, 5_000_003), (1, 5_000_004)])
def test_nearest_centre_several_trips(gpu, K, rows, n):
    from dimq_amd import ops
    announce(f"nearest trips K={K} rows={rows} n={n}")
    g = torch.Generator().manual_seed(K + rows + n)
    w, c = torch.randn(rows, n, generator=g).to(gpu), torch.randn(rows, K, generator=g).to(gpu)
    w[:, -1] = float("nan")  # the last element of the ragged trip: index 0
    idx, val = ops.hard_quantize(w, c, True)
    order = torch.arange(K, device=gpu, dtype=torch.int16)
    per = max(1, 4_000_000 // K // n)
    for r in range(0, rows, per):
        for k in range(0, n, 2_000_000 // K * 8):
            ws, cs = w[r:r + per, k:k + 2_000_000 // K * 8], c[r:r + per]
            d = (ws[:, :, None] - cs[:, None, :]) ** 2
            want = torch.where(d == d.amin(2, keepdim=True), order, torch.tensor(K, dtype=torch.int16, device=gpu)).amin(2)
            want[want == K] = 0  # a NaN equals nothing
            got = idx[r:r + per, k:k + ws.shape[1]]
            assert torch.equal(got.short(), want)
            assert torch.equal(val[r:r + per, k:k + ws.shape[1]], torch.gather(cs, 1, want.long()))
