"""exl3_dgemm (medium row counts): every row-tile count of both kernels, ragged last tiles, every width and codebook, split sums, several matrices, strided outputs,
the residual form, and the grouped form, against float64 arithmetic on the oracle's exact weights.

Bound.  The rotated activations and (fp16 outputs) the result are rounded once to 11 bits: relative 2-norm 2^-11 / sqrt(3) = 2.8e-4 each at most, 4e-4 together;
the fp32 accumulation adds below 1e-5."""
import numpy as np
import pytest
import torch

from oracle import exl3_oracle as orc

pytestmark = pytest.mark.gpu
TOL = 4.5e-4


def _dev():
    return torch.device("cuda:0")


def _lin(k, n, K, cb, seed):
    tr, suh, svh = orc.synth_linear(k, n, K, seed=seed, realistic=True)
    w = torch.from_numpy(orc.reconstruct(tr, K, cb).astype(np.float64)).to(_dev())
    h = torch.from_numpy(np.asarray(orc.hadamard_matrix_128(), dtype=np.float64)).to(_dev())
    h = h / h[0, 0].abs() / 128 ** 0.5
    t = [torch.from_numpy(a).to(_dev()) for a in (tr, suh, svh)]

    def exact(x):
        y = ((x.double() * t[1].double()).view(-1, k // 128, 128) @ h).view(-1, k) @ w
        return (y.view(-1, n // 128, 128) @ h).view(-1, n) * t[2].double()
    return t, exact


def _err(y, ref):
    return ((y.double() - ref).norm() / ref.norm()).item()


@pytest.mark.parametrize("m", [33, 64, 65, 80, 81, 97, 112, 113, 128, 129, 160, 161, 192, 193, 224, 225, 256, 257, 300, 513])
def test_dgemm_row_tiles(m):
    from exllamav3_amd import ext
    k, n, K = 384, 256, 4
    (tr, su, sv), exact = _lin(k, n, K, 2, 3)
    x = torch.randn((m, k), device=_dev(), generator=torch.Generator(device=_dev()).manual_seed(m)).half()
    ref = exact(x)
    for out in (torch.half, torch.float):
        for split in (0, 1, 3) if m <= 128 else (0, 1, 3, -1, -3):         # (negative: the kernel for many rows)
            y = torch.full((m, n), float("nan"), dtype=out, device=_dev())
            ext.dgemm(x, [tr], [y], [su], [sv], False, True, force_split=split)
            assert _err(y, ref) < TOL


@pytest.mark.parametrize("K", range(1, 9))
@pytest.mark.parametrize("cb", [0, 1, 2])
@pytest.mark.parametrize("m", [70, 200])
def test_dgemm_widths_codebooks(K, cb, m):
    from exllamav3_amd import ext
    k, n = 640, 128                                       # an odd number of 128-deep blocks
    (tr, su, sv), exact = _lin(k, n, K, cb, 10 * K + cb)
    x = torch.randn((m, k), device=_dev(), generator=torch.Generator(device=_dev()).manual_seed(K)).half()
    for split in (0, -1):
        y = torch.full((m, n), float("nan"), dtype=torch.half, device=_dev())
        ext.dgemm(x, [tr], [y], [su], [sv], cb == 1, cb == 2, force_split=split)
        assert _err(y, exact(x)) < TOL


@pytest.mark.parametrize("m", [40, 150, 300])
def test_dgemm_matrices_strides_residual_bias(m):
    """Three matrices of different widths into column ranges of one buffer, from a strided input, with a bias; then the same added to a residual."""
    from exllamav3_amd import ext
    k, ns, K = 512, (256, 128, 128), 3
    mats = [_lin(k, n, K, 0, 50 + i) for i, n in enumerate(ns)]
    mats[2][0][1].copy_(mats[1][0][1])                    # two matrices of equal input scales in different storage, and (below) of shared storage
    gen = torch.Generator(device=_dev()).manual_seed(m)
    wide = torch.randn((m, k + 64), device=_dev(), generator=gen).half()
    x = wide[:, 64:]
    sus = [mats[0][0][1], mats[1][0][1], mats[1][0][1]]
    bias = [torch.randn(n, device=_dev(), generator=gen).half() for n in ns]
    for acc in (False, True):
        buf = torch.randn((m, sum(ns)), device=_dev(), generator=gen).half()
        old, ys = buf.clone(), list(buf.split(ns, dim=1))
        ext.dgemm(x, [t[0] for t, _ in mats], ys, sus, [t[2] for t, _ in mats], False, False, bias, accumulate=acc)
        for (_, exact), y, o, b in zip(mats, ys, old.split(ns, dim=1), bias):
            assert _err(y, exact(x) + b.double() + (o.double() if acc else 0.0)) < TOL


def test_dgemm_refuses_bad_arguments():
    from exllamav3_amd import ext
    (tr, su, sv), _ = _lin(256, 128, 4, 2, 5)
    x = torch.zeros((40, 256), dtype=torch.half, device=_dev())
    y = torch.zeros((40, 128), dtype=torch.half, device=_dev())
    with pytest.raises(RuntimeError):
        ext.dgemm(x.float(), [tr], [y], [su], [sv], False, True)
    with pytest.raises(RuntimeError):
        ext.dgemm(x, [tr], [y[:39]], [su], [sv], False, True)
    with pytest.raises(RuntimeError):
        ext.dgemm(x[:, 4:], [tr], [y], [su], [sv], False, True)
    with pytest.raises(RuntimeError):                     # rows that do not start at multiples of 16 bytes
        ext.dgemm(torch.zeros((40, 260), dtype=torch.half, device=_dev())[:, 4:], [tr], [y], [su], [sv], False, True)


@pytest.mark.parametrize("rows", [(0, 0, 5, 5, 90, 90), (0, 100, 100, 431, 640, 700), (0, 256, 512, 1200, 1201, 1500)])
def test_dgemm_grouped(rows):
    """Groups without rows, of one row and of several row tiles; gathered input and two matrices, then silu(g) u input and fp32 output."""
    from exllamav3_amd import ext
    E, R, k, n, K = len(rows) - 1, rows[-1], 256, 384, 4
    mats = [[_lin(k, n, K, 2, 100 + 10 * i + e) for e in range(E)] for i in range(2)]
    bounds = torch.tensor(rows, dtype=torch.int32, device=_dev())
    g = torch.Generator(device=_dev()).manual_seed(R)
    x = torch.randn((R + 30, k), device=_dev(), generator=g).half()
    u = torch.randn((R + 30, k), device=_dev(), generator=g).half()
    pick = torch.randint(0, R + 30, (R,), device=_dev(), generator=g)

    def table(sets):
        flat = [t for s in sets for t, _ in s]
        return tuple(torch.tensor([t[j].data_ptr() for t in flat], dtype=torch.long, device=_dev()) for j in range(3))
    ys = [torch.full((R, n), float("nan"), dtype=torch.half, device=_dev()) for _ in range(2)]
    ext.dgemm_grouped(x, pick, bounds, table(mats), ys, R, K, False, True)
    for s, y in zip(mats, ys):
        assert _err(y, torch.cat([s[e][1](x[pick[rows[e]:rows[e + 1]]]) for e in range(E)])) < TOL
    y = torch.full((R, n), float("nan"), dtype=torch.float, device=_dev())
    ext.dgemm_grouped(x, None, bounds, table(mats[:1]), [y], R, K, False, True, act_u=u)
    a = (torch.nn.functional.silu(x.double()) * u.double()).half()
    assert _err(y, torch.cat([mats[0][e][1](a[rows[e]:rows[e + 1]]) for e in range(E)])) < TOL


@pytest.mark.parametrize("rows", [32, 33, 128, 129, 512, 513])
def test_linear_routes_meet(rows):
    """LinearEXL3.forward on both sides of every row threshold, against the same linear through the fp16 weight matrix; several matrices of one launch of the C entry."""
    from exllamav3_amd import ext
    from exllamav3_amd.linear import LinearEXL3
    k, n, K = 512, 384, 5
    (tr, su, sv), exact = _lin(k, n, K, 1, 9)
    lin = LinearEXL3(k, n, tr, su, sv, mcg=True)
    x = torch.randn((rows, k), device=_dev(), generator=torch.Generator(device=_dev()).manual_seed(rows)).half()
    ref = exact(x)
    assert _err(lin.forward(x), ref) < 6e-4               # (up to 128 rows: the scaled input and the unscaled output are rounded on the way, sqrt(4) x 2.8e-4)
    assert _err(lin.forward(x, {"no_reconstruct": True}), ref) < 6e-4
    assert _err(lin.forward(x, {"reconstruct": True}), ref) < 6e-4
    ys = [torch.empty((rows, n), dtype=torch.half, device=_dev()) for _ in range(2)]
    ext.exl3_mgemm_bcast(x, [tr, tr], ys, [su, su], [sv, sv], True, False)
    assert _err(ys[0], ref) < 6e-4 and torch.equal(ys[0], ys[1])


@pytest.mark.parametrize("rows", [40, 200])
def test_input_off_sixteen_bytes_keeps_its_route(rows):
    """An input that starts 8 bytes into a 16-byte piece is no input for exl3_dgemm; the entry point takes it as before (32-row passes)."""
    from exllamav3_amd.linear import LinearEXL3
    k, n, K = 256, 256, 4
    (tr, su, sv), exact = _lin(k, n, K, 2, 21)
    lin = LinearEXL3(k, n, tr, su, sv, mul1=True)
    x = torch.randn((rows * k + 4,), device=_dev(), generator=torch.Generator(device=_dev()).manual_seed(rows)).half()[4:].view(rows, k)
    assert x.data_ptr() % 16 == 8 and x.is_contiguous()
    assert _err(lin.forward(x, {"no_reconstruct": True}), exact(x)) < 6e-4


@pytest.mark.parametrize("host", ["trellis", "suh", "svh", "bias", "out"])
def test_dgemm_refuses_tensors_of_another_device(host):
    """A linear whose weights are still in host memory ended in an error on the fp16-weight route and does here: no host address reaches a kernel."""
    from exllamav3_amd import ext
    from exllamav3_amd.linear import LinearEXL3
    (tr, su, sv), _ = _lin(256, 128, 4, 2, 5)
    t = {"trellis": tr, "suh": su, "svh": sv, "bias": torch.zeros(128, dtype=torch.half, device=_dev())}
    x = torch.zeros((200, 256), dtype=torch.half, device=_dev())
    y = torch.zeros((200, 128), dtype=torch.half, device="cpu" if host == "out" else _dev())
    if host != "out":
        t[host] = t[host].cpu()
        with pytest.raises(RuntimeError):
            LinearEXL3(256, 128, t["trellis"], t["suh"], t["svh"], mul1=True, bias=t["bias"]).forward(x)
    with pytest.raises(RuntimeError, match="device"):
        ext.dgemm(x, [t["trellis"]], [y], [t["suh"]], [t["svh"]], False, True, [t["bias"]])


def test_grouped_calls_refuse_tensors_of_another_device():
    from exllamav3_amd import ext
    dev = _dev()
    bounds, tab = torch.tensor([0, 4], dtype=torch.int32, device=dev), tuple(torch.zeros(1, dtype=torch.long, device=dev) for _ in range(3))
    x, y, pick = torch.zeros((4, 256), dtype=torch.half, device=dev), torch.zeros((4, 128), device=dev), torch.zeros(4, dtype=torch.long, device=dev)
    for args in ((x, pick.cpu(), bounds, tab, [y]), (x, pick, bounds.cpu(), tab, [y]), (x, pick, bounds, tab[:2] + (tab[2].cpu(),), [y]), (x, pick, bounds, tab, [y.cpu()])):
        with pytest.raises(RuntimeError, match="device"):
            ext.dgemm_grouped(*args, 4, 4, False, True)
    with pytest.raises(RuntimeError, match="device"):
        ext.dgemm_grouped(x, None, bounds, tab, [y], 4, 4, False, True, act_u=x.cpu())
    D, pos, w = torch.zeros((4, 128), device=dev), torch.zeros((2, 2), dtype=torch.int32, device=dev), torch.zeros((2, 2), dtype=torch.half, device=dev)
    for args in ((D, pos.cpu(), w), (D, pos, w.cpu())):
        with pytest.raises(RuntimeError, match="device"):
            ext.moe_combine(*args)


@pytest.mark.parametrize("form", ["bfloat16", "strided", "one"])
def test_a_bias_of_another_form_keeps_its_route(form):
    """What `y += bias` takes and a kernel's pointer does not: other types, strides, one value for all columns."""
    from exllamav3_amd.linear import LinearEXL3
    k, n, K, rows = 256, 256, 4, 200
    (tr, su, sv), exact = _lin(k, n, K, 2, 23)
    gen = torch.Generator(device=_dev()).manual_seed(4)
    bias = {"bfloat16": torch.randn(n, device=_dev(), generator=gen).bfloat16(), "strided": torch.randn(2 * n, device=_dev(), generator=gen).half()[::2],
            "one": torch.randn(1, device=_dev(), generator=gen).half()}[form]
    x = torch.randn((rows, k), device=_dev(), generator=gen).half()
    y = LinearEXL3(k, n, tr, su, sv, mul1=True, bias=bias).forward(x)
    assert _err(y, exact(x) + bias.double()) < 6e-4       # (x W and the sum rounded once each)
    lin = LinearEXL3(k, n, tr, su, sv, mul1=True, bias=bias)
    q, p = LinearEXL3.forward_separate([lin, LinearEXL3(k, n, tr, su, sv, mul1=True)], x)
    assert torch.equal(q, y) and _err(p, exact(x)) < 6e-4


@pytest.mark.parametrize("k,n,rows,K,cb,packed", [
    (4096, 6144, 560, 8, 0, False), (4096, 6144, 300, 4, 2, True), (4096, 4096, 768, 8, 0, False), (4096, 14336, 512, 4, 2, True), (4096, 14336, 600, 8, 1, False),
    (14336, 4096, 1000, 4, 2, True), (2048, 512, 1000, 8, 0, True), (2048, 512, 1023, 4, 2, True), (2048, 512, 1024, 4, 2, False),
    (2048, 2048, 1023, 6, 2, False), (2048, 2048, 768, 6, 2, True), (4096, 22016, 400, 4, 2, True), (5120, 27648, 600, 4, 2, True), (4096, 28672, 1000, 8, 0, False)])
def test_route_follows_sizes_bits_and_codebook(k, n, rows, K, cb, packed):
    """The route with the fp16 weight matrix gives the bits of the forced one, the packed one does not; points where the two are at least 5 % apart, and the last row count."""
    from exllamav3_amd.linear import LinearEXL3
    gen = torch.Generator(device=_dev()).manual_seed(rows + K)
    tr = torch.randint(-32768, 32768, (k // 16, n // 16, 16 * K), dtype=torch.int16, device=_dev(), generator=gen)
    su = (torch.randint(0, 2, (k,), device=_dev(), generator=gen) * 2 - 1).half()
    sv = (0.02 * torch.rand(n, device=_dev(), generator=gen)).half()
    lin = LinearEXL3(k, n, tr, su, sv, mcg=cb == 1, mul1=cb == 2)
    x = torch.randn((rows, k), device=_dev(), generator=gen).half()
    y, other = lin.forward(x), lin.forward(x, {"reconstruct": True})
    assert _err(y, other.double()) < 9e-4                 # (both rounded as in the bounds above)
    assert torch.equal(y, other) != packed


@pytest.mark.parametrize("m", [40, 100, 144, 150, 200, 420, 700, 1000])
@pytest.mark.parametrize("K,cb", [(3, 1), (7, 2), (8, 0)])
def test_dgemm_full_size_plans(m, K, cb):
    """A model's size, where plans split k and use several row tiles: against the same product with one slice, 2e-6 of the largest float32 sums of 4096 products apart."""
    from exllamav3_amd import ext
    k, n = 4096, 1024
    gen = torch.Generator(device=_dev()).manual_seed(m + K)
    tr = torch.randint(-32768, 32768, (k // 16, n // 16, 16 * K), dtype=torch.int16, device=_dev(), generator=gen)
    su, sv = torch.ones(k, device=_dev()).half(), torch.ones(n, device=_dev()).half()
    x = torch.randn((m, k), device=_dev(), generator=gen).half()
    ys = [torch.full((m, n), float("nan"), device=_dev()) for _ in range(3)]
    for y, split in zip(ys, (0, 1, -1)):
        ext.dgemm(x, [tr], [y], [su], [sv], cb == 1, cb == 2, force_split=split)
    for y in ys[1:]:
        assert float((ys[0] - y).abs().max()) < 2e-6 * float(ys[0].abs().max()) * 4


@pytest.mark.parametrize("rows", [150, 256, 300, 500])
def test_gate_and_up_of_a_models_size(rows):
    """Both matrices of one launch with the activation behind it where the GEMM's fused epilogue ran from 256 rows on: against the two linears through rebuilt weights."""
    from exllamav3_amd import ext
    from exllamav3_amd.linear import LinearEXL3, _dgemm_ok
    k, n, K = 4096, 8192, 4
    gen = torch.Generator(device=_dev()).manual_seed(rows)

    def lin():
        tr = torch.randint(-32768, 32768, (k // 16, n // 16, 16 * K), dtype=torch.int16, device=_dev(), generator=gen)
        return LinearEXL3(k, n, tr, (torch.randint(0, 2, (k,), device=_dev(), generator=gen) * 2 - 1).half(), (0.02 * torch.rand(n, device=_dev(), generator=gen)).half(), mul1=True)
    gate, up = lin(), lin()
    x = torch.randn((rows, k), device=_dev(), generator=gen).half()
    assert _dgemm_ok(x, (gate, up), rows)
    g, u = (l.forward(x, {"reconstruct": True}).double() for l in (gate, up))
    # (gate and up: rotated rows against W^T, rounded to fp16 on both sides; the activation rounded once: five errors of 2.8e-4, and silu's slope of up to 1.1)
    assert _err(LinearEXL3.forward_gate_up_silu(gate, up, x), torch.nn.functional.silu(g) * u) < 8e-4
