"""Row kernels of the sequence mixers in both access widths: 16-byte pieces (aligned rows) and single elements, rows shorter than a piece per thread, rows longer than the
registers hold, against float64.

Bounds.  float32: sums of up to 16400 terms, 1e-5 relative 2-norm with room; bfloat16 outputs are rounded once to 8 bits (2^-9 / sqrt(3) = 1.1e-3), 2.5e-3 with the largest rows'
spread."""
import pytest
import torch

pytestmark = pytest.mark.gpu
TOL = {torch.float32: 1e-5, torch.bfloat16: 2.5e-3}
DEV = "cuda:0"


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm())


def _cols(n, width, off, dtype, gen):
    """(n, width) of a wider matrix, `off` columns in."""
    return torch.randn((n, width + off + 3 * (off != 0)), device=DEV, generator=gen).to(dtype)[:, off: off + width]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width,off", [(4, 0), (8, 0), (33, 0), (1024, 0), (1024, 16), (1024, 3), (2056, 0), (4096, 0), (8200, 0), (8201, 1), (16400, 0)])
def test_norms_and_gates(width, off, dtype):
    from exllamav3_amd import mix_ops
    gen = torch.Generator(device=DEV).manual_seed(width + off)
    n, vocab, eps = 5, 11, 1e-5
    table = torch.randn((vocab, width), device=DEV, generator=gen).to(dtype)
    tokens = torch.randint(0, vocab, (n,), device=DEV, generator=gen, dtype=torch.int32)
    w = 1 + 0.1 * torch.randn(width, device=DEV, generator=gen)
    norm = lambda v: v / (v.pow(2).mean(-1, keepdim=True) + eps).sqrt() * w.double()
    x, h = torch.empty((n, width), device=DEV), torch.empty((n, width), dtype=dtype, device=DEV)
    mix_ops.embed(x, h, table, tokens, 0.37, w, eps)
    ref = table.double()[tokens.long()] * 0.37
    assert _rel(x, ref) < 1e-6 and _rel(h, norm(ref)) < TOL[dtype]
    y, r = _cols(n, width, off, dtype, gen), _cols(n, width, off, dtype, gen)
    ref = x.double() + y.double() * torch.sigmoid(r.double())
    mix_ops.gated_residual(x, y, r, w, h, eps)
    assert _rel(x, ref) < 1e-6 and _rel(h, norm(ref)) < TOL[dtype]
    rows = torch.tensor([3, 0, 3], dtype=torch.int32, device=DEV)
    hw = torch.empty((3, width), dtype=dtype, device=DEV)
    mix_ops.rms_norm_rows(hw, x, rows, w, eps)
    assert _rel(hw, norm(x.double()[rows.long()])) < TOL[dtype]
    z, coef = _cols(n, width, off, dtype, gen) * 1.7 if off == 0 else _cols(n, width, off, dtype, gen), torch.tensor([0.5, -0.25, 0.125, 0.3], device=DEV)
    out = torch.empty((n, width), dtype=dtype, device=DEV)
    mix_ops.polynorm(out, z, coef, eps)
    want = sum(c * p / (p.pow(2).mean(-1, keepdim=True) + eps).sqrt() for c, p in zip(coef.double(), (z.double(), z.double() ** 2, z.double() ** 3))) + coef[3].double()
    assert _rel(out, want) < TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width,off", [(256, 0), (264, 0), (512, 0), (513, 0), (516, 0), (1000, 0), (1032, 0), (2048, 0), (2050, 0)])
def test_norms_and_gates_at_the_widths_where_the_waves_change(width, off, dtype):
    test_norms_and_gates(width, off, dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,width,off", [(1024, 513, 1), (1025, 513, 1), (1025, 1026, 1), (1024, 512, 0), (1025, 264, 0), (1025, 256, 0), (1024, 256, 0)])
def test_gate_and_polynorm_where_the_rows_choose_the_form(n, width, off, dtype):
    """Gated residual: rows off 16 bytes in eight waves up to 1024 rows and four beyond, short rows in single elements up to 1024 rows; polynomial norm of short rows likewise."""
    from exllamav3_amd import mix_ops
    gen = torch.Generator(device=DEV).manual_seed(n + width)
    x, w = torch.randn((n, width), device=DEV, generator=gen), 1 + 0.1 * torch.randn(width, device=DEV, generator=gen)
    y, r = _cols(n, width, off, dtype, gen), _cols(n, width, off, dtype, gen)
    h = torch.empty((n, width), dtype=dtype, device=DEV)
    coef = torch.tensor([0.5, -0.25, 0.125, 0.3], device=DEV)
    mix_ops.polynorm(h, y, coef, 1e-5)
    want = sum(c * p / (p.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt() for c, p in zip(coef.double(), (y.double(), y.double() ** 2, y.double() ** 3))) + coef[3].double()
    assert _rel(h, want) < TOL[dtype]
    ref = x.double() + y.double() * torch.sigmoid(r.double())
    mix_ops.gated_residual(x, y, r, w, h, 1e-5)
    assert _rel(x, ref) < 1e-6 and _rel(h, ref / (ref.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt() * w.double()) < TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("vdim,heads,off", [(4, 3, 0), (33, 2, 0), (64, 5, 0), (128, 32, 0), (128, 3, 2), (132, 1, 0), (256, 2, 4), (300, 2, 0)])
def test_gla_out(vdim, heads, off, dtype):
    from exllamav3_amd import mix_ops
    gen = torch.Generator(device=DEV).manual_seed(vdim + heads)
    n, eps = 7, 1e-5
    o = torch.randn((n, heads, vdim), device=DEV, generator=gen)
    w, g = 1 + 0.1 * torch.randn(vdim, device=DEV, generator=gen), _cols(n, heads * vdim, off, dtype, gen)
    out = torch.empty((n, heads * vdim), dtype=dtype, device=DEV)
    mix_ops.gla_out(out, o, w, g, eps)
    od = o.double()
    want = (od / (od.pow(2).mean(-1, keepdim=True) + eps).sqrt() * w.double()).view(n, -1) * torch.nn.functional.silu(g.double())
    assert _rel(out, want) < TOL[dtype]


@pytest.mark.parametrize("dim,vdim,H,G,window", [(64, 64, 4, 2, 1100), (64, 64, 70, 70, 90), (128, 128, 4, 1, 600), (192, 256, 2, 2, 300), (64, 128, 3, 3, 64), (64, 72, 2, 1, 300)])
def test_decode_attention_rows_of_whole_lines(dim, vdim, H, G, window):
    """bfloat16 rows read eight lanes at a time (and, with 72 value columns, one key per lane): lengths around the groups of eight rows and the chunks of 64, against float64.
    Bound: the output's rounding to 8 bits, 2^-9, over sums of exact products in float32."""
    from exllamav3_amd import mix_ops
    gen = torch.Generator(device=DEV).manual_seed(dim + vdim + window)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=gen).bfloat16()
    lens = [x for x in (1, 7, 8, 9, 63, 64, 65, window - 1, window, window + 5) if x > 0]
    n = len(lens)
    q, rk, rv = rnd(n, H * dim), rnd(n, window, G, dim), rnd(n, window, G, vdim)
    for b, l in enumerate(lens):                                          # entries nobody has written are not read
        rk[b, min(l, window):] = float("nan")
        rv[b, min(l, window):] = float("nan")
    sink = torch.randn(H, device=DEV, generator=gen)
    mk = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    out = torch.empty((n, H * vdim), dtype=torch.bfloat16, device=DEV)
    mix_ops.attn_decode(out, q, rk, rv, None, sink, mk(list(range(n))), mk(lens), H, dim ** -0.5)
    for b, l in enumerate(lens):
        c = min(l, window)
        k, v = (t[b, :c].double().repeat_interleave(H // G, dim=1) for t in (rk, rv))
        s = torch.einsum("hd,chd->hc", q[b].double().view(H, dim), k) * dim ** -0.5
        e = torch.exp(torch.cat([s, sink.double().view(H, 1)], dim=1) - torch.maximum(s.amax(1), sink.double()).view(H, 1))
        want = torch.einsum("hc,chv->hv", e[:, :c] / e.sum(1, keepdim=True), v)
        assert _rel(out[b].view(H, vdim), want) < 2.5e-3, l


@pytest.mark.parametrize("dim,vdim,H,G,window", [(64, 64, 4, 2, 1100), (128, 128, 2, 1, 1100), (64, 256, 2, 2, 1100), (64, 64, 40, 8, 300), (128, 192, 40, 8, 300)])
def test_decode_attention_rows_where_the_chunks_change(dim, vdim, H, G, window):
    """Rows are cut into chunks of 8 to 64 keys by their length: the lengths where a chunk grows, over 16 waves (few rows of a long window) and over 4.
    Bound: the output's rounding to 8 bits, 2^-9 / sqrt(3), over sums of exact products in float32."""
    from exllamav3_amd import mix_ops
    gen = torch.Generator(device=DEV).manual_seed(dim + vdim + H)
    rnd = lambda *s: torch.randn(*s, device=DEV, generator=gen).bfloat16()
    waves = 16 if H < 10 else 4
    lens = [l for g in (1, 2, 7) for l in (8 * waves * g - 1, 8 * waves * g, 8 * waves * g + 1) if l <= window]
    n = len(lens)
    q, rk, rv = rnd(n, H * dim), rnd(n, window, G, dim), rnd(n, window, G, vdim)
    for b, l in enumerate(lens):
        rk[b, l - 1] *= 4                                                 # the last key of a row counts: a lost one shows
        rk[b, l:], rv[b, l:] = float("nan"), float("nan")
    mk = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    out = torch.empty((n, H * vdim), dtype=torch.bfloat16, device=DEV)
    mix_ops.attn_decode(out, q, rk, rv, None, None, mk(list(range(n))), mk(lens), H, dim ** -0.5)
    for b, l in enumerate(lens):
        k, v = (t[b, :l].double().repeat_interleave(H // G, dim=1) for t in (rk, rv))
        p = torch.softmax(torch.einsum("hd,chd->hc", q[b].double().view(H, dim), k) * dim ** -0.5, dim=1)
        assert _rel(out[b].view(H, vdim), torch.einsum("hc,chv->hv", p, v)) < 2.5e-3, l
