"""CPU-only: the model workloads of bench.py check and time their own model."""

import torch
from torch import nn


def test_each_model_workload_has_its_own_cpu_model():
    import bench
    x = torch.randn(2, 3, 4, 4, generator=torch.Generator().manual_seed(0))
    models = [nn.Sequential(nn.Flatten(), nn.Linear(48, out)).half() for out in (5, 7)]
    loads = [bench._model_workload(f"m{i}", "", "cpu", 1, m, x, 1.0, "fp16", torch.contiguous_format, {})
             for i, m in enumerate(models)]
    for wl, m in zip(loads, models):  # the first's CPU model must not serve the second
        y = wl["cpu_step"](2)
        assert y.shape == (2, m[1].out_features)
        assert torch.equal(y, m.float()(x))
