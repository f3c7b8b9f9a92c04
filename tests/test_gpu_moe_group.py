"""Grouping of routed assignments by expert and the combination behind the experts: exact against a stable sort and against moe_scatter's order."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    from exllamav3_amd import ext
    ext.init(0)
    return "cuda:0"


@pytest.mark.parametrize("T,k,E", [(1, 1, 1), (1, 8, 8), (31, 2, 8), (32, 2, 8), (513, 2, 3), (700, 2, 8), (999, 16, 129), (4100, 8, 512)])
def test_group_is_the_stable_sort_and_combine_the_ordered_sum(dev, T, k, E):
    from exllamav3_amd import ext
    gen = torch.Generator(device=dev).manual_seed(T + E)
    sel = torch.rand((T, E), device=dev, generator=gen).topk(k, dim=1).indices.contiguous() if T * E < 1 << 20 else torch.randint(0, E, (T, k), device=dev, generator=gen)
    if E > 2:
        sel[sel == 1] = 0 if k == 1 else sel[sel == 1]                     # (with one expert per token: a group without rows)
    tok, pos, rows = ext.moe_group(sel, E)
    order = torch.argsort(sel.reshape(-1), stable=True)
    assert torch.equal(tok, order // k)
    assert torch.equal(pos.reshape(-1)[order], torch.arange(T * k, dtype=torch.int32, device=dev))
    assert rows.tolist() == [0] + torch.bincount(sel.reshape(-1), minlength=E).cumsum(0).tolist()
    D = torch.randn((T * k, 132), device=dev, generator=gen)
    w = torch.rand((T, k), device=dev, generator=gen).half()
    want = torch.zeros((T, 132), device=dev)
    ext.moe_scatter(D, torch.arange(T * k, dtype=torch.int32, device=dev), tok, w.reshape(-1)[order].contiguous(), want)
    assert torch.equal(ext.moe_combine(D, pos, w), want)


def test_assignment_to_no_expert_keeps_every_place_in_range(dev):
    from exllamav3_amd import ext
    sel = torch.randint(0, 8, (300, 2), device=dev, generator=torch.Generator(device=dev).manual_seed(1))
    sel[17] = 0x7fffffff                                                   # what the router leaves for a row of NaN
    tok, pos, rows = ext.moe_group(sel, 8)
    assert rows[-1] == 598 and (pos[17] == -1).all() and tok.min() >= 0 and tok.max() < 300
    out = ext.moe_combine(torch.ones((600, 128), device=dev), pos, torch.ones((300, 2), dtype=torch.half, device=dev))
    assert out[17].isnan().all() and (out[torch.arange(300, device=dev) != 17] == 2).all()


@pytest.mark.parametrize("T", [128, 333, 700])
def test_block_on_packed_weights_matches_the_loop_over_experts(dev, T):
    """Against the per-expert loop (same routing): both hold activations in fp16 around the products, 2^-10 relative each, over sums of random signs."""
    from exllamav3_amd.moe_path import SyntheticEXL3MoE
    moe = SyntheticEXL3MoE(256, 384, experts=8, top_k=2, K=4, cb=2, device=dev, seed=5)
    moe.router[:, 3] = 0                                                   # an uneven routing
    moe.router[:, 5] *= 4
    x = torch.randn((T, 256), device=dev, generator=torch.Generator(device=dev).manual_seed(T)).half()
    got = moe.forward_prefill(x)
    moe.grouped_prefill = False
    want = moe.forward_prefill(x)
    assert (got - want).norm() / want.norm() < 2 ** -9
    row = x.clone(); row[7] = float("nan")
    moe.grouped_prefill = True
    again = moe.forward_prefill(row)
    keep = torch.arange(T, device=dev) != 7
    assert again[7].isnan().all() and torch.equal(again[keep], got[keep])


@pytest.mark.parametrize("T", [130, 1100, 2560])
def test_block_of_a_models_size_on_packed_weights(dev, T):
    """Mixtral's block over the chunks that take the packed form, against the form on rebuilt weights.  Bound: in each of the two products one side rounds the rotated rows and the other W^T, the
    activations between them are rounded on both: six errors of 2^-11 / sqrt(3) at most, 7e-4 together; no row of a token may be further off than three times that."""
    from exllamav3_amd.moe_path import SyntheticEXL3MoE
    moe = SyntheticEXL3MoE(4096, 14336, experts=8, top_k=2, K=4, cb=2, device=dev, seed=11)
    moe.router.copy_(torch.randn(moe.router.shape, device=dev, generator=torch.Generator(device=dev).manual_seed(3)) / 64)
    x = torch.randn((T, 4096), device=dev, generator=torch.Generator(device=dev).manual_seed(5)).half()
    assert moe._on_packed_weights(2 * T)
    got = moe.forward_prefill(x)
    moe.DGEMM_ROWS = 0
    want = moe.forward_prefill(x)
    assert (got - want).norm() / want.norm() < 8e-4
    assert float(((got - want).norm(dim=1) / want.norm(dim=1)).max()) < 2.4e-3
