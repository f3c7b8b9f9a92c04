"""Gated linear attention in time segments at key dimensions 64 and 128 (chunks of 16 tokens on the matrix instructions) against the float64 recurrence: segments that are no
multiple of a chunk, sequences shorter than one, value widths and ranks at their edges, decays that underflow within a chunk, a state carried in.

Bound.  Every float32 product and sum of the chunk form has factors at most one from the decays, so its error is that of a float32 dot product over the terms the recurrence has
(dimension times tokens that still weigh in): 2e-5 of the largest output, the bound of the token-by-token form."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,d,dv,tau,rank,bias,lens", [
    (2, 64, 128, 16.0, 16, 1.0, [130, 1, 37]), (1, 64, 70, 4.0, 5, 1.0, [200]), (3, 64, 8, 1.0, 1, -8.0, [19, 66]), (2, 128, 130, 16.0, 64, 1.0, [95, 64]),
    (1, 128, 256, 2.0, 16, 12.0, [81]), (2, 64, 300, 0.05, 64, 0.0, [50, 33]), (4, 64, 128, 16.0, 3, -90.0, [40])])
def test_segments_match_the_recurrence(H, d, dv, tau, rank, bias, lens, dtype):
    from exllamav3_amd import mix_ops
    gen = torch.Generator(device=DEV).manual_seed(H * 7 + d + dv)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=gen)
    N, B = sum(lens), len(lens)
    pad = rnd(N, H * d + 8).to(dtype)                                     # (a row stride of its own)
    q, k, v, lr = pad[:, :H * d], rnd(N, H * d).to(dtype) * 0.5, rnd(N, H * dv).to(dtype), rnd(N, rank).to(dtype)
    a2, a2b = (rnd(H * d, rank) * 1.5).to(dtype), rnd(H * d) + bias
    qs = d ** -0.5
    slots, pos0 = [B - i for i in range(B)], [5 if i == 1 else 0 for i in range(B)]
    z = (lr.double() @ a2.double().T + a2b.double()).view(N, H, d)
    alpha = torch.exp(torch.nn.functional.logsigmoid(z) / tau)
    start = rnd(B + 1, H, d, dv)
    mk = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    cu = [0]
    for l in lens:
        cu.append(cu[-1] + l)
    want, end, n = torch.empty((N, H, dv), dtype=torch.float64, device=DEV), [], 0
    for b, l in enumerate(lens):
        S = start[slots[b]].double() if pos0[b] else torch.zeros((H, d, dv), dtype=torch.float64, device=DEV)
        for _ in range(l):
            S = alpha[n][:, :, None] * S + k[n].double().view(H, d, 1) * v[n].double().view(H, 1, dv)
            want[n] = torch.einsum("hd,hdv->hv", q[n].double().view(H, d) * qs, S)
            n += 1
        end.append(S)
    for L in (16, 40, 48, max(lens)):
        state = start.clone()
        for b in range(B):
            if not pos0[b]:
                state[slots[b]] = float("nan")                            # a new sequence does not read its slot
        o = torch.full((N, H, dv), float("nan"), device=DEV)
        mix_ops.gla_scan(o, state, q, k, v, lr, a2, a2b, mk(cu), mk(slots), mk(pos0), tau, qs, segments=(-(-max(lens) // L), L))
        assert float((o - want).abs().max() / want.abs().max()) < 2e-5, L
        for b in range(B):
            assert float((state[slots[b]] - end[b]).abs().max() / end[b].abs().max()) < 2e-5, L
        assert torch.equal(state[0], start[0])                            # a slot of no sequence stays


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("what", ["v", "k", "q", "lr"])
def test_a_value_that_is_not_finite_stays_out_of_the_rows_before_it(what, value):
    """One such element in the middle of a chunk: rows in front of it, the other sequence and (an element of v) the other columns keep their bits; its own row is not finite."""
    from exllamav3_amd import mix_ops
    H, d, dv, rank, lens, at, col = 2, 64, 140, 4, [50, 70], 50 + 22, 133                # row 22 of the second sequence: the seventh of its second chunk
    gen = torch.Generator(device=DEV).manual_seed(3)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=gen)
    N = sum(lens)
    t = {"q": rnd(N, H * d), "k": rnd(N, H * d), "v": rnd(N, H * dv), "lr": rnd(N, rank)}
    a2, a2b = rnd(H * d, rank), rnd(H * d) + 1.0
    mk = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)

    def scan():
        state, o = torch.zeros((2, H, d, dv), device=DEV), torch.full((N, H, dv), float("nan"), device=DEV)
        mix_ops.gla_scan(o, state, t["q"], t["k"], t["v"], t["lr"], a2, a2b, mk([0, 50, 120]), mk([0, 1]), mk([0, 0]), 4.0, 0.125, segments=(2, 48))
        return o, state
    plain, _ = scan()
    assert plain.isfinite().all()
    t[what][at, {"v": dv + col, "k": 5, "q": 5, "lr": 0}[what]] = value
    o, state = scan()
    assert torch.equal(o[:at], plain[:at]) and state[0].isfinite().all()
    if what == "v":
        keep = torch.ones((H, dv), dtype=torch.bool, device=DEV)
        keep[1, col] = False
        assert torch.equal(o[:, keep], plain[:, keep])
        assert not o[at:, 1, col].isfinite().any() and not state[1, 1, :, col].isfinite().any()
    elif what == "q":
        assert torch.equal(o[at + 1:], plain[at + 1:]) and not o[at, 0].isfinite().any()
    elif what == "k" or value != value:
        assert not o[at:, 0].isfinite().any()
    else:                                                                               # (decays of an infinite input are 0 or 1)
        assert o.isfinite().all()
