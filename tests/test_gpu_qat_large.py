"""QAT kernels beyond 8,388,608 weights (8,192 work-groups of 1,024), where a work-group takes several chunks and keeps
its sums over them, and beyond 16,777,216, where the separation loss's runs of weights grow past two chunks; against the
float64 oracle, taken in pieces.  The bars are those of the smaller sizes."""

import pytest
import torch

from oracle import qat as oqat
from tests.conftest import announce
from tests.test_gpu_qat import _case, _gen, _rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,K", [(8_388_609, 4), (8_400_000, 17), (17_000_003, 4)])
def test_more_chunks_than_work_groups(gpu, n, K):
    from dimq_amd import qat
    announce(f"qat large n={n} K={K}")
    tau = 1e-3
    w, c = _case(n, K, n + K)
    up = torch.randn(n, generator=_gen(n))
    wd, cd = w.to(gpu).requires_grad_(), c.to(gpu).requires_grad_()
    y, loss = qat.soft_dequantize_weight(wd, cd, tau), qat.dimq_softmin_loss(wd, cd, tau)
    grads = [torch.autograd.grad(y, (wd, cd), up.to(gpu)), torch.autograd.grad(loss, (wd, cd))]
    total = torch.zeros((), dtype=torch.float64)
    gc = [torch.zeros(K, dtype=torch.float64) for _ in grads]
    top = [0.0, 0.0]
    worst = [0.0, 0.0]
    for lo in range(0, n, 1 << 20):
        part = slice(lo, min(n, lo + (1 << 20)))
        wo, co = w[part].clone().requires_grad_(), c.clone().requires_grad_()
        yo, lo_ = oqat.soft_dequantize(wo, co, tau), oqat.softmin_loss(wo, co, tau)
        assert _rel(y.detach()[part], yo.detach()) <= 1e-5
        total += lo_.detach()
        for i, (out, g) in enumerate(((yo, up[part].double()), (lo_, None))):
            hw, hc = torch.autograd.grad(out, (wo, co), g, retain_graph=True)
            gc[i] += hc.double()
            top[i] = max(top[i], float(hw.abs().max()))
            worst[i] = max(worst[i], float((grads[i][0][part].cpu().double() - hw.double()).abs().max()))
    assert _rel(loss.detach(), total) <= 2e-5
    for i in range(2):
        assert worst[i] <= 2e-4 * top[i]
        assert _rel(grads[i][1], gc[i]) <= 2e-4


@pytest.mark.parametrize("n", [8_388_609, 16_777_217, 17_000_003])
def test_separation_loss_of_longer_runs(gpu, n):
    from dimq_amd import qat
    announce(f"separation large n={n}")
    g = _gen(n)
    w, c = torch.randn(n, generator=g) * 0.05 + 0.3, (torch.randn(16, generator=g) * 0.01).sort().values
    cd = c.to(gpu).requires_grad_()
    loss = qat.separation_loss(w.to(gpu), cd)
    loss.backward()
    co = c.clone().requires_grad_()
    ref = oqat.separation_loss(w, co)
    ref.backward()
    assert _rel(loss.detach(), ref.detach()) <= 1e-5 and _rel(cd.grad, co.grad) <= 1e-4
