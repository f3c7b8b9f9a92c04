"""Which product a mixer family's vocabulary head takes: the own kernel for few rows of widths that are multiples of 2048 and for small heads, a vendor product for the rest."""
import pytest
import torch

from exllamav3_amd import modules


@pytest.mark.parametrize("n,k,v,own", [(1, 4096, 32000, True), (4, 4096, 128256, True), (5, 4096, 128256, False), (2, 8192, 32000, True), (3, 8192, 32000, False), (16, 8192, 128256, False),
                                       (1, 2048, 128256, True), (8, 2048, 32000, True), (9, 2048, 32000, False), (1, 4088, 128256, False), (1, 1024, 32000, False), (2, 6144, 64000, True),
                                       (1, 3072, 8193, False), (16, 3072, 8192, True), (4, 5120, 8192, True), (5, 5120, 8192, False)])
def test_head_takes_its_product_by_size(monkeypatch, n, k, v, own):
    taken = []
    product = lambda name: lambda x, w, bias=None: taken.append(name) or torch.zeros(x.shape[0], 1, dtype=x.dtype)
    monkeypatch.setattr(modules, "linear", product("own"))
    monkeypatch.setattr(modules.F, "linear", product("vendor"))
    zero = torch.zeros(1, dtype=torch.bfloat16)
    out = modules.head_logits(zero.expand(n, k), zero.expand(v, k))
    assert out.dtype == torch.float32 and taken == ["own" if own else "vendor"]
