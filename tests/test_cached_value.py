"""The rule of ``ops.cached_value``: reuse only while every source keeps its
identity, version, storage and dtype; sources without a version counter are
never cached and cost no exception."""

import torch
from torch import nn

from boltz_lumi_amd import ops


class Counted(nn.Parameter):
    """A parameter that counts reads of its version counter."""

    reads = 0

    @property
    def _version(self):
        Counted.reads += 1
        return torch.Tensor._version.__get__(self)


def value(module, *sources):
    built = []
    got = ops.cached_value(module, "x", sources, lambda: built.append(1) or sum(float(p.detach().sum()) for p in sources))
    assert got == sum(float(p.detach().sum()) for p in sources)
    return bool(built)


def test_inference_sources_are_rebuilt_without_reading_versions():
    module, normal = nn.Module(), nn.Parameter(torch.ones(2))
    with torch.inference_mode():
        inf = Counted(torch.ones(2))
        for sources in ((inf,), (normal, inf), (inf, normal)):
            for _ in range(3):
                assert value(module, *sources)
                inf.add_(1)
    assert Counted.reads == 0


def test_a_source_replaced_by_an_inference_tensor():
    module, a, b = nn.Module(), nn.Parameter(torch.ones(2)), nn.Parameter(torch.ones(2))
    assert value(module, a, b) and not value(module, a, b)
    with torch.inference_mode():
        c = Counted(torch.ones(2))
        Counted.reads = 0
        for _ in range(3):
            assert value(module, a, c)
            c.add_(1)
        assert Counted.reads == 1  # the cached value's sources are read once, then asked first
    assert value(module, a, b) and not value(module, a, b)
    with torch.no_grad():
        a.mul_(2)
    assert value(module, a, b) and not value(module, a, b)
    a.data = a.data.clone()
    assert value(module, a, b)
