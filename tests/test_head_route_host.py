"""Which product a mixer family's vocabulary head takes: the own kernel for one or two rows of at least 4096 over a large head, a vendor product for the rest."""
import pytest
import torch

from exllamav3_amd import modules


@pytest.mark.parametrize("n,k,v,own", [(1, 4096, 32000, True), (2, 4096, 128256, True), (2, 8192, 32000, True), (3, 4096, 128256, False), (16, 8192, 128256, False),
                                       (1, 2048, 128256, False), (1, 4088, 128256, False), (1, 8192, 8192, False), (1, 6144, 256, False), (0, 4096, 32000, False)])
def test_head_takes_its_product_by_size(monkeypatch, n, k, v, own):
    taken = []
    product = lambda name: lambda x, w, bias=None: taken.append(name) or torch.zeros(x.shape[0], 1, dtype=x.dtype)
    monkeypatch.setattr(modules, "linear", product("own"))
    monkeypatch.setattr(modules.F, "linear", product("vendor"))
    zero = torch.zeros(1, dtype=torch.bfloat16)
    out = modules.head_logits(zero.expand(n, k), zero.expand(v, k))
    assert out.dtype == torch.float32 and taken == ["own" if own else "vendor"]
