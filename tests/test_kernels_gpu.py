"""Each kernel alone against its plain reference, at sizes other than the engine tests use."""

from __future__ import annotations

import math

import pytest
import torch

import plain_llama as pl
from tiny import ulps_of_row_max

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _ops():
    from nanospec_amd.kernels import ops

    return ops


def _tol(dtype):
    return dict(rtol=2e-5, atol=2e-6) if dtype == torch.float32 else dict(rtol=2e-2, atol=2e-3)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_embed(dtype):
    ops = _ops()
    table = torch.randn(301, 72, dtype=dtype, device=DEV)
    ids = torch.tensor([0, 300, 5, 5, 17], dtype=torch.int32, device=DEV)
    assert torch.equal(ops.embed(table, ids), table[ids.long()])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dim", [72, 1000, 4096])
def test_rmsnorm_plain_fused_and_gathered(dtype, dim):
    ops = _ops()
    torch.manual_seed(dim)
    n, eps = 7, 3e-6
    resid = torch.randn(n, dim, dtype=dtype, device=DEV) * 3
    x = torch.randn(n, dim, dtype=dtype, device=DEV)
    w = (1 + 0.1 * torch.randn(dim, device=DEV)).to(dtype)
    # plain
    ref = pl.rms_norm(resid.cpu(), w.cpu(), eps)
    torch.testing.assert_close(ops.rmsnorm(w, eps, resid=resid).cpu(), ref, **_tol(dtype))
    # fused sum, written back
    r2 = resid.clone()
    out = ops.rmsnorm(w, eps, resid=r2, x=x, write_resid=True)
    summed = pl.residual_add(resid.cpu(), x.cpu())
    assert torch.equal(r2.cpu(), summed)
    torch.testing.assert_close(out.cpu(), pl.rms_norm(summed, w.cpu(), eps), **_tol(dtype))
    # gathered rows, nothing written
    rows = torch.tensor([6, 0, 6, 3], dtype=torch.int32, device=DEV)
    r3 = resid.clone()
    out = ops.rmsnorm(w, eps, resid=r3, x=x, rows=rows)
    assert torch.equal(r3, resid)
    torch.testing.assert_close(out.cpu(), pl.rms_norm(summed, w.cpu(), eps)[rows.cpu().long()], **_tol(dtype))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(1, 40, 24), (5, 130, 200), (8, 1003, 4096), (3, 7, 18), (70, 65, 17), (200, 300, 128)])
def test_linear_generic(dtype, m, n, k):
    ops = _ops()
    torch.manual_seed(m * n)
    x = torch.randn(m, k, dtype=dtype, device=DEV)
    w = torch.randn(n, k, dtype=dtype, device=DEV)
    ref = x.cpu().double() @ w.cpu().double().T
    # a 32-bit sum of K products is off by a few units in the last place of the sum of their magnitudes, not of the result
    bound = 2.0 ** -20 * (x.cpu().double().abs() @ w.cpu().double().abs().T)
    out = ops.linear_generic(x, w, out_f32=True)
    assert ((out.cpu().double() - ref).abs() <= bound).all()
    out2 = ops.linear_generic(x, w)
    if dtype == torch.float32:
        assert torch.equal(out2, out)
    else:
        torch.testing.assert_close(out2.cpu().float(), ref.to(dtype).float(), **_tol(dtype))
    ref = ref.float()
    # a row's result does not depend on the rows beside it (up to 8 rows of 32-bit x run a kernel of their own, whose sums
    # are ordered differently: compare within a kernel)
    few = 1 if m <= 8 or dtype != torch.float32 else 9
    assert torch.equal(ops.linear_generic(x[:few].contiguous(), w, out_f32=True), out[:few])
    if dtype == torch.float32 and m > 8:
        one = ops.linear_generic(x[:1].contiguous(), w, out_f32=True)
        torch.testing.assert_close(one, out[:1], rtol=1e-5, atol=1e-4)


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 6, 7, 8, 9, 16, 17, 33, 515])
@pytest.mark.parametrize("n,k", [(1, 4), (7, 2052), (33, 60), (130, 64), (700, 516), (4100, 576), (4130, 100), (65, 2500),
                                 (250, 516), (8210, 252), (4100, 2048), (4099, 1024), (4099, 1028)])
def test_linear_f32_forms(m, n, k):
    """32-bit products of few and of many rows at the edges of their tiles (8 rows or columns, 16, 32, 64), of a stage of 64 k and of
    the stages that are in flight (three or eight, before and after a place in LDS is used again); rows of x and of the result with a stride of their own."""
    ops = _ops()
    torch.manual_seed(m + n + k)
    wide = torch.randn(m, k + 12, device=DEV)
    x, w, out = wide[:, 4 : 4 + k], torch.randn(n, k, device=DEV), torch.full((m, n + 3), 7.0, device=DEV)
    ref = x.cpu().double() @ w.cpu().double().T
    bound = 2.0 ** -20 * (x.cpu().double().abs() @ w.cpu().double().abs().T)  # as above
    ops.linear_generic(x, w, out=out[:, :n])
    assert ((out[:, :n].cpu().double() - ref).abs() <= bound).all()
    assert bool((out[:, n:] == 7).all())
    rows = 1 if m <= 8 else 9
    assert torch.equal(ops.linear_generic(x[:rows], w), out[:rows, :n])


@pytest.mark.parametrize("k,most", [(1024, 8.85e-8), (1028, 9.2e-8), (1536, 9.31e-8), (2048, 9.65e-8)])
def test_linear_f32_of_few_rows_is_as_exact_as_eight_waves(k, most):
    """Where four waves add up a row of a wide matrix, their sums are no further from 64 bits than those of eight (8.8e-8, 9.1e-8, 9.25e-8, 9.6e-8; chains of two lengths at K 1,536 were 9.37e-8)."""
    ops = _ops()
    far = []
    for seed in range(4):
        torch.manual_seed(seed)
        x, w = torch.randn(5, k, device=DEV), torch.randn(8192, k, device=DEV)
        ref = x.double() @ w.double().T
        far.append(float((ops.linear_generic(x, w).double() - ref).norm() / ref.norm()))
    assert sum(far) / 4 <= most


@pytest.mark.parametrize("m", [1, 8, 9, 33])
@pytest.mark.parametrize("stride", [(1 << 24) - 4, 1 << 24])
@pytest.mark.parametrize("n,k", [(130, 68), (4130, 324)])
def test_linear_f32_of_rows_far_apart(m, stride, n, k):
    """Rows that 32 bits address from a tile's first and rows that they do not: the same sums, bit by bit, as of rows side by side."""
    ops = _ops()
    torch.manual_seed(m + n)
    x, w = torch.randn(m, k, device=DEV), torch.randn(n, k, device=DEV)
    far = torch.empty((m - 1) * stride + k, device=DEV).as_strided((m, k), (stride, 1))
    far.copy_(x)
    assert torch.equal(ops.linear_generic(far, w), ops.linear_generic(x, w))


@pytest.mark.parametrize("rows", [64, 96, 112, 128])
@pytest.mark.parametrize("m,n,k,ranges", [(1, 1, 32, 1), (15, 130, 64, 2), (17, 131, 96, 3), (113, 257, 160, 1), (129, 64, 1056, 4), (300, 2060, 1024, 2)])
def test_linear_split(rows, m, n, k, ranges):
    """32-bit products through two float16 parts of each operand at the edges of the tiles (16 rows and the tile's, 16 and 128 columns), of a stage of 32 k and of
    uneven ranges; rows of x and of the result with a stride of their own."""
    ops = _ops()
    torch.manual_seed(m + n + k)
    wide = torch.randn(m, k + 12, device=DEV)
    x, w, out = wide[:, 4 : 4 + k], torch.randn(n, k, device=DEV), torch.full((m, n + 3), 7.0, device=DEV)
    ref = x.cpu().double() @ w.cpu().double().T
    # two parts stand for a float to 2^-23 at most and leave out 2^-22 of a product, the sum of a stage is rounded 12 times (three instructions, four blocks of 8 k
    # each); then a stage or range is added at a time
    bound = (2 + 2 + 4 + 12 + k / 32 + ranges) * 2.0**-24 * (x.cpu().double().abs() @ w.cpu().double().abs().T)
    ops.linear_split(x, w, rows, ranges, out=out[:, :n])
    assert ((out[:, :n].cpu().double() - ref).abs() <= bound).all()
    assert bool((out[:, n:] == 7).all())
    if k >= ops.SPLIT_MIN_K:  # where it is taken it is nearer to 64 bits than the 32-bit instruction (whose sums' roundings are fewer than the parts' at a few stages)
        far = lambda y: float((y.cpu().double() - ref).norm())
        assert far(out[:, :n]) <= far(ops.linear_generic(x, w))


@pytest.mark.parametrize("ranges", [1, 2])
def test_linear_split_beyond_the_parts(ranges):
    """Infinities, no numbers, the largest floats (whose first part would round up to infinity) and floats whose lower parts bfloat16 does not hold."""
    ops = _ops()
    torch.manual_seed(3)
    x, w = torch.randn(70, 128, device=DEV), torch.randn(140, 128, device=DEV)
    x[3, 5], x[4, 6], x[5, 7], x[6] = math.inf, -math.inf, math.nan, 0.0
    x[7], w[11, 3], w[12, 100] = 0.0, 0.0, math.inf
    x[8, 9] = x[9, 9] = 3.4028234e38  # (times a normal number: a large float, or infinity)
    x[10:20] *= 2.0**-120
    x[7, 1] = 2.0**-126 * 1.2345678
    out = ops.linear_split(x, w, 64, ranges).cpu()
    a, b = x.cpu().double(), w.cpu().double()
    ref = a @ b.T
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    over = ref.abs() > 3.4028235e38 * (1 + 2.0**-24)
    assert bool((out[over] == torch.sign(ref[over]).float() * math.inf).all())
    fine = torch.isfinite(ref) & (ref.abs() < 3.4e38)
    bound = 2.0**-17 * (a.abs().clamp(max=3.5e38) @ b.abs().clamp(max=3.5e38).T) + 128 * 2.0**-149  # one chain of 128, floored by the smallest float
    assert bool(((out.double() - ref).abs()[fine] <= bound[fine]).all())


# (positions, requests) of a batch: runs that fill 16-byte runs of a page, begin and end inside one, stand out of order, repeat a place of the pad page
KV_ORDERS = (([0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15, 16, 17, 18], [0] * 19), ([5, 6, 7, 8, 9, 3, 4, 5], [0] * 5 + [1] * 3),
             ([9, 8, 31, 30, 16, 17, 19, 20], [0, 0, 1, 1, 1, 1, 1, 1]), ([0, 0, 0, 12], [0, 0, 0, 1]), ([7], [1]))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("order", range(len(KV_ORDERS)))
@pytest.mark.parametrize("kind,H,G,D,E,page,rot,interleaved", [
    ("unit", 5, 2, 64, 64, 16, 0, False), ("unit", 3, 1, 16, 40, 4, 0, False), ("unit", 4, 4, 512, 8, 32, 0, False), ("borrow", 6, 2, 32, 32, 16, 0, False),
    ("bare", 2, 2, 128, 64, 8, 0, False), ("head", 6, 2, 64, 64, 16, 64, False), ("head", 3, 3, 128, 64, 8, 64, False), ("head", 2, 1, 64, 24, 32, 30, True),
    ("head", 5, 1, 16, 16, 6, 16, True), ("same", 4, 2, 32, 32, 16, 16, False), ("whole", 32, 8, 64, 64, 16, 64, False), ("whole", 3, 1, 64, 128, 16, 32, True),
    ("mixed", 5, 2, 32, 64, 4, 0, False), ("whole", 70, 20, 128, 64, 16, 128, False)])
def test_keys_and_values_in_pieces(dtype, order, kind, H, G, D, E, page, rot, interleaved):
    """Norm, rotation and write of keys and values in pieces of 8 bytes against the plain kernels, which take the same rows an odd number of values apart."""
    ops = _ops()
    g = torch.Generator().manual_seed(H * D + order)
    pos, req = (torch.tensor(a, dtype=torch.int32, device=DEV) for a in KV_ORDERS[order])
    n, own, same = len(pos), kind != "borrow", kind == "same"
    width = H * D + (G * (D + (0 if same else E)) if own else 0)
    make = lambda *shape: (2.0 * torch.randn(*shape, generator=g)).to(dtype).to(DEV)
    rows, bias, other = make(n, width), make(width), make(n, G * E)
    per = 1 if kind in ("head", "same") else H
    qw, kw = make(per * D), make((1 if per == 1 else G) * D)
    inv = torch.rand(max(1, rot // 2), generator=g).to(DEV)
    pages = 1 + 33 // page
    table = torch.randperm(2 * pages, generator=g).to(torch.int32).view(2, pages).to(DEV)
    mix = torch.full((1,), 0.375, dtype=dtype, device=DEV)
    got = []
    for extra in (0, 3):  # (rows of whole pieces; three columns more)
        wide = torch.full((n, width + 8 * (extra > 0) + extra), 5.0, dtype=dtype, device=DEV)
        wide[:, :width] = rows
        kc, vc = torch.zeros(2 * pages, G, page, D, dtype=dtype, device=DEV), torch.zeros(2 * pages, G, E, page, dtype=dtype, device=DEV)
        keep = torch.zeros(n, G * E, dtype=dtype, device=DEV)
        x = wide[:, : wide.shape[1] - extra] if extra else wide
        if kind in ("unit", "borrow", "bare"):
            ops.unit_kv_write(x, pos, req, table, kc, vc, H, G, D, E, None if kind == "bare" else 1e-3, own_kv=own)
        elif kind in ("head", "same"):
            ops.head_norm_rope_kv_write(x, pos, req, table, inv[: rot // 2], kc, vc, H, G, D, E, 1e-3, rot, bias=bias, q_weight=qw, k_weight=None if E == 24 else kw,
                                        value_is_key=same, interleaved=interleaved, factor=1.25)
        else:
            mixed = dict(mix=mix, v_other=other, v_keep=keep) if kind == "mixed" else {}
            ops.whole_norm_kv_write(x, pos, req, table, kc, vc, H, G, D, E, 1e-3, bias=bias, q_weight=qw, k_weight=None if E == 128 else kw, inv_freq=inv, rotary_dim=rot,
                                    interleaved=interleaved, **mixed)
        got.append((wide[:, :width], kc, vc, keep))
    # the sums of squares are in another order, and a channel is then a product of three: a few units of 2^-24 before it is rounded
    tol = dict(rtol=2.0**-19, atol=2.0**-18) if dtype == torch.float32 else dict(rtol=2.0**-7, atol=2.0**-8)
    last = {(int(r), int(p)): i for i, (r, p) in enumerate(zip(req, pos))}  # (a place that several tokens write keeps any of them)
    once = [i for (r, p), i in last.items() if sum(int(a) == r and int(b) == p for a, b in zip(req, pos)) == 1]
    # values are the same bit by bit; of two mixed values (1 - m) a + m b one product is rounded ahead of the sum, which one the compiler chooses: 2^-24 of it
    # (at most 0.625 times a number below 16), and a bfloat16 result may then round the other way
    alike = torch.equal if kind != "mixed" else lambda a, b: torch.allclose(a, b, rtol=0 if dtype == torch.float32 else 2.0**-7, atol=2.0**-20)
    assert torch.allclose(got[0][0], got[1][0], **tol) and alike(got[0][3], got[1][3])
    for i in once:
        at = int(table[req[i], pos[i] // page]), int(pos[i]) % page
        assert torch.allclose(got[0][1][at[0], :, at[1]], got[1][1][at[0], :, at[1]], **tol)
        assert alike(got[0][2][at[0], :, :, at[1]], got[1][2][at[0], :, :, at[1]])
    if order != 3 and own:
        written = sorted((int(table[r, p // page]), p % page) for r, p in last)
        blank = torch.ones(2 * pages, page, dtype=torch.bool)
        for a, b in written:
            blank[a, b] = False
        assert bool((got[0][1].cpu().transpose(1, 2)[blank] == 0).all()) and bool((got[0][2].cpu().permute(0, 3, 1, 2)[blank] == 0).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("n", [65, 255, 300, 1023, 1024, 1301])
@pytest.mark.parametrize("kind,H,G,D,E,page,rot", [("unit", 6, 2, 64, 64, 16, 0), ("unit", 40, 8, 128, 96, 16, 0), ("bare", 5, 3, 32, 40, 8, 0), ("head", 6, 2, 64, 64, 16, 32),
                                                   ("head", 40, 10, 128, 128, 32, 128), ("same", 40, 10, 64, 64, 16, 64), ("whole", 32, 8, 64, 64, 16, 64), ("whole", 64, 16, 64, 80, 4, 0)])
def test_keys_and_values_in_pieces_of_many_tokens(dtype, n, kind, H, G, D, E, page, rot):
    """The forms that prompts take (values by workgroups of their own and behind the heads, heads in several rounds, one unit or two a thread), two requests of odd lengths that begin inside a run of a page:
    against the plain kernels, every place of the pages."""
    ops = _ops()
    g = torch.Generator().manual_seed(n + H)
    first, starts = n // 3 | 1, (5, 3)
    pos = torch.cat([torch.arange(first) + starts[0], torch.arange(n - first) + starts[1]]).int().to(DEV)
    req = torch.cat([torch.zeros(first), torch.ones(n - first)]).int().to(DEV)
    width = H * D + G * (D + (0 if kind == "same" else E))
    make = lambda *shape: (2.0 * torch.randn(*shape, generator=g)).to(dtype).to(DEV)
    rows, bias = make(n, width), make(width)
    per = 1 if kind in ("head", "same") else H
    qw, kw, inv = make(per * D), make((1 if per == 1 else G) * D), torch.rand(max(1, rot // 2), generator=g).to(DEV)
    pages = 1 + (n + 8) // page
    table = torch.randperm(2 * pages, generator=g).to(torch.int32).view(2, pages).to(DEV)
    got = []
    for extra in (0, 3):  # (rows of whole pieces; three columns more)
        wide = torch.full((n, width + 8 * (extra > 0) + extra), 5.0, dtype=dtype, device=DEV)
        wide[:, :width] = rows
        kc, vc = torch.full((2 * pages, G, page, D), 3.0, dtype=dtype, device=DEV), torch.full((2 * pages, G, E, page), 3.0, dtype=dtype, device=DEV)
        x = wide[:, : wide.shape[1] - extra] if extra else wide
        if kind in ("unit", "bare"):
            ops.unit_kv_write(x, pos, req, table, kc, vc, H, G, D, E, None if kind == "bare" else 1e-3, own_kv=True)
        elif kind in ("head", "same"):
            ops.head_norm_rope_kv_write(x, pos, req, table, inv[: rot // 2], kc, vc, H, G, D, E, 1e-3, rot, bias=bias, q_weight=qw, k_weight=kw, value_is_key=kind == "same")
        else:
            ops.whole_norm_kv_write(x, pos, req, table, kc, vc, H, G, D, E, 1e-3, bias=bias, q_weight=qw, k_weight=kw, inv_freq=inv if rot else None, rotary_dim=rot)
        got.append((wide[:, :width], kc, vc))
    tol = dict(rtol=2.0**-19, atol=2.0**-18) if dtype == torch.float32 else dict(rtol=2.0**-7, atol=2.0**-8)  # (as above)
    assert torch.allclose(got[0][0], got[1][0], **tol) and torch.allclose(got[0][1], got[1][1], **tol) and torch.equal(got[0][2], got[1][2])


@pytest.mark.parametrize("spread", [12, 24])
def test_linear_split_of_wide_rows(spread):
    """Values over many powers of two within a block of x and a row of w: no more is lost than of values of one size."""
    ops = _ops()
    torch.manual_seed(spread)
    small = torch.randint(-spread, 1, (2, 300, 1024)).float().exp2().to(DEV)
    x, w = torch.randn(100, 1024, device=DEV) * small[0, :100], torch.randn(300, 1024, device=DEV) * small[1]
    a, b = x.cpu().double(), w.cpu().double()
    # as above: the second part has the float16 range to itself, and rows that it still does not hold are the 32-bit instruction's (four chains of 64 sums)
    bound = (2 + 2 + 4 + 12 + 32 + 1) * 2.0**-24 * (a.abs() @ b.abs().T)
    assert bool(((ops.linear_split(x, w, 64, 1).cpu().double() - a @ b.T).abs() <= bound).all())


@pytest.mark.parametrize("ranges", [1, 2])
@pytest.mark.parametrize("kind", ["zero w", "small w", "zero x", "small x", "even", "sparse"])
@pytest.mark.parametrize("factor", [1e4, 1e5, 1e6, 1e7, 1e8, 1e9, 1e10, 1e12, 1e30])
def test_linear_split_of_values_far_apart(factor, kind, ranges):
    """Large values that meet zeros or small ones in the other operand, so that all that counts is what is small beside them: as near to 64 bits as the 32-bit instruction."""
    ops = _ops()
    torch.manual_seed(17)
    x, w = torch.randn(100, 1024, device=DEV), torch.randn(300, 1024, device=DEV)
    if kind == "even":  # the small values all alike, one large one a block beside them
        x[:] = 0.1
    if kind == "sparse":  # one value a block beside the large one
        x.view(100, 32, 32)[:, :, 6:] = 0
        x.view(100, 32, 32)[:, :, :5] = 0
    large, other = (w, x) if kind.endswith("x") else (x, w)
    large[:, 3::32] *= factor
    other[:, 3::32] *= 0 if kind in ("zero w", "zero x", "even", "sparse") else 1 / factor
    ref = x.cpu().double() @ w.cpu().double().T
    far = lambda y: float((y.cpu().double() - ref).norm() / ref.norm())
    # (32 terms in all, hardly a rounding of the sums: a term is held to 2^-21, 2^-23 for either operand and 2^-22 for the product left out, and to a third of that in the mean)
    limit = 2.0**-21 / 3 if kind == "sparse" else 0
    y = ops.linear_split(x, w, 64, ranges)
    assert far(y) <= max(far(ops.linear_generic(x, w)), limit)
    if factor >= 1e12 and kind != "sparse":  # every row: the 32-bit instruction's sums
        assert torch.equal(y, ops.linear_generic(x, w))


@pytest.mark.parametrize("ranges", [1, 2])
@pytest.mark.parametrize("m", [4097, 4200])
def test_linear_split_in_portions(m, ranges):
    """More rows than a portion, the last one short: rows of x and of the result with a stride of their own, a row of the 32-bit instruction in either portion."""
    ops = _ops()
    torch.manual_seed(m)
    wide, w, out = torch.randn(m, 140, device=DEV), torch.randn(70, 128, device=DEV), torch.full((m, 77), 7.0, device=DEV)
    x = wide[:, 8:136]
    x[[5, 4096], 3] = math.inf
    split = ops.SplitWeight(w)
    ops.linear_split(x, w, 128, ranges, out=out[:, :70], split=split)
    parts = torch.cat([ops.linear_split(p, w, 64, ranges, split=split) for p in (x[:4096], x[4096:])])
    assert torch.equal(out[:, :70], parts) and bool((out[:, 70:] == 7).all())
    a, b, fine = x.cpu().double(), w.cpu().double(), torch.isfinite(x).all(1).cpu()
    bound = (2 + 2 + 4 + 12 + 4 + ranges) * 2.0**-24 * (a.abs() @ b.abs().T)  # (as in test_linear_split)
    assert ((parts.cpu().double() - a @ b.T).abs()[fine] <= bound[fine]).all() and torch.equal(parts[[5, 4096]], ops.linear_generic(x, w)[[5, 4096]])
    read = torch.tensor([4099], dtype=torch.int32, device=DEV)
    assert torch.equal(ops.linear_split(x, w, 128, ranges, split=split, read_rows=read)[:4099], parts[:4099])
    assert bool((ops.linear_split(x, w, 128, ranges, split=split, read_rows=read)[4099:] == 0).all())


@pytest.mark.parametrize("blocks,kept", [(0, True), (1, True), (8, True), (9, False), (65, False)])
def test_split_weight_of_values_far_apart(blocks, kept):
    """A matrix of which the parts do not hold too many rows keeps no second copy: its products stay the 32-bit instruction's."""
    from nanospec_amd.engine.arena import Arena
    from nanospec_amd.parts.linear import LinearWeight, drop_copies_of_little_use

    ops = _ops()
    torch.manual_seed(blocks)
    w, x = torch.randn(1040 - 5, 4096, device=DEV), torch.randn(600, 4096, device=DEV)
    assert ops.split_plan(600, 1035, 4096, ops.compute_units(x.device)) is not None
    w[0 : 16 * blocks : 16, ::5] *= 1e-12
    weight, other = LinearWeight(w), LinearWeight(torch.randn(1035, 4096, device=DEV))
    drop_copies_of_little_use([weight, other])
    assert (weight._split is not None) == kept and other._split is not None
    y, plain = weight(x, arena=Arena(x.device)), ops.linear_generic(x, w)
    lost = list(range(0, 16 * blocks, 16)) if kept else slice(None)
    assert torch.equal(y[:, lost], plain[:, lost])


@pytest.mark.parametrize("n", [40, 2072])
@pytest.mark.parametrize("blocks", [[0, 70, 255], [3, 64, 65, 127, 128, 191, 254], list(range(1, 256, 3)), list(range(256))])
def test_linear_split_mends_blocks_far_apart(blocks, n):
    """Rows for the 32-bit instruction in blocks that different waves of a workgroup find, one block at a time and four: all of them are its results, the others' are theirs."""
    ops = _ops()
    torch.manual_seed(n + len(blocks))
    x, w = torch.randn(4096, 128, device=DEV), torch.randn(n, 128, device=DEV)
    split = ops.SplitWeight(w)
    want = ops.linear_split(x, w, 64, 1, split=split)
    rows = torch.tensor([16 * b + b % 16 for b in blocks], device=DEV)
    x[rows, ::5] *= 1e12
    want[rows] = ops.linear_generic(x, w)[rows]
    for _ in range(3):
        assert torch.equal(ops.linear_split(x, w, 64, 1, split=split), want)


@pytest.mark.parametrize("n,k", [(4096, 1024), (2056, 2080), (130, 4128), (15360, 1056)])
def test_linear_split_is_the_same_whatever_the_rows_beside(n, k):
    """Any tile, segments by one workgroup or by one each, any rows beside and any place among them: the same results bit by bit."""
    ops = _ops()
    torch.manual_seed(n)
    x, w = torch.randn(600, k, device=DEV), torch.randn(n, k, device=DEV)
    x[7, 3] = math.inf  # (a row of the 32-bit instruction beside the others)
    split = ops.SplitWeight(w)
    want = ops.linear_split(x, w, 64, 1, split=split)
    for rows in (64, 96, 112, 128):
        for ranges in (1, ops.split_segments(n, k)):
            assert torch.equal(ops.linear_split(x, w, rows, ranges, split=split), want)
            assert torch.equal(ops.linear_split(x[5:305], w, rows, ranges, split=split), want[5:305])
    assert torch.equal(ops.linear_generic(x, w)[7], want[7])


@pytest.mark.parametrize("read", [0, 1, 16, 77, 100])
def test_linear_split_of_rows_that_nobody_reads(read):
    """Padding rows are zeros whatever lies there, and none of them is left to the 32-bit instruction; the others are as they are without them, through the part's own door too."""
    from nanospec_amd.engine.arena import Arena
    from nanospec_amd.parts.linear import product_f32

    ops = _ops()
    torch.manual_seed(read)
    x, w = torch.randn(100, 5120, device=DEV), torch.randn(4096, 5120, device=DEV)
    want = ops.linear_split(x, w, 64, 1)
    x[read:, ::3], x[read:, 1::3] = math.inf, 1e-30
    taken, count = [], torch.tensor([read], dtype=torch.int32, device=DEV)
    take = lambda shape, dtype: taken.append(torch.empty(shape, dtype=dtype, device=DEV)) or taken[-1]
    y = ops.linear_split(x, w, 64, 1, take=take, read_rows=count)
    assert torch.equal(y[:read], want[:read]) and bool((y[read:] == 0).all())
    lost = next(t for t in taken if t.dtype == torch.int32)
    assert not bool(lost[:-1].any())
    arena, split = Arena(x.device), ops.SplitWeight(w)
    assert ops.split_plan(100, 4096, 5120, ops.compute_units(x.device)) is not None
    arena.read_rows = (100, count)
    assert bool((product_f32(x, w, split, None, arena)[read:] == 0).all())
    arena.read_rows = (96, count)  # (a product of other rows)
    assert read == 100 or not bool(torch.isfinite(product_f32(x, w, split, None, arena)[read:]).all())


@pytest.mark.parametrize("keep_plain", [True, False])
def test_linear_weight_f32_of_many_rows(keep_plain):
    """A float32 matrix through the part's own door, with its second copy and (only one copy is kept) without; both as close as 32-bit sums."""
    from nanospec_amd.engine.arena import Arena
    from nanospec_amd.parts.linear import LinearWeight

    ops = _ops()
    torch.manual_seed(5)
    x, w = torch.randn(600, 2048, device=DEV), torch.randn(2064, 2048, device=DEV)
    linear = LinearWeight(w, keep_plain=keep_plain)
    assert ops.split_plan(600, 2064, 2048, ops.compute_units(x.device)) is not None and (linear._split is not None) == keep_plain
    y, ref = linear(x, arena=Arena(x.device)).double(), x.double() @ w.double().T
    assert float((y - ref).norm() / ref.norm()) <= (3e-7 if keep_plain else 6e-7)  # 1.8e-7 and 4.1e-7 measured at K 2,048


def test_second_copies_of_float32_matrices_are_given_back():
    """Those of a model's parts, wherever they are kept, until a runner has been made for it; the products then run on the 32-bit instruction."""
    from types import SimpleNamespace

    from nanospec_amd.engine.arena import Arena
    from nanospec_amd.parts.linear import GatedWeights, LinearWeight, second_copies
    from nanospec_amd.parts.model import DecoderModel

    ops = _ops()
    torch.manual_seed(9)
    w, x = torch.randn(2048, 2048, device=DEV), torch.randn(600, 2048, device=DEV)
    linear, gated, small, tiled = LinearWeight(w), GatedWeights(w[:1024].contiguous(), w[1024:].contiguous()), LinearWeight(w[:64, :512].contiguous()), LinearWeight(w, keep_plain=False)
    model = DecoderModel.__new__(DecoderModel)
    model.device, model.has_runner, model.layers, model.other = torch.device(DEV), True, [{"first": (linear, small)}, tiled], gated
    ctx = SimpleNamespace(arena=Arena(x.device), captured=False)
    before = linear(x, arena=ctx.arena)
    assert set(second_copies(model)) == {linear, gated} and not model.give_back_second_copies() and linear._split is not None
    model.has_runner = False
    assert model.give_back_second_copies() and not list(second_copies(model)) and not model.give_back_second_copies()
    after = linear(x, arena=ctx.arena)
    assert torch.equal(after, ops.linear_generic(x, w)) and not torch.equal(after, before)
    gated(ctx, x, out=torch.empty(600, 1024, device=DEV))


@pytest.mark.parametrize("shapes", [[(1,)], [(3, 5), (1,), (7,)], [(16, 128, 257), (2, 2048), (1,), (13,)], [(9,), (8 * 257,), (65, 1023), (4, 3)]])
def test_slot_tensors(shapes):
    """One slot of every tensor is cleared and nothing beside it: slots of single words, of odd numbers of values, of many blocks."""
    ops = _ops()
    kinds = (torch.float32, torch.bfloat16, torch.int32, torch.bfloat16)
    tensors = [torch.ones((5, *shape), dtype=dtype, device=DEV) for shape, dtype in zip(shapes, kinds)]
    slots = ops.SlotTensors(tensors)
    for slot in (4, 0, 2):
        slots.clear(slot)
    for t in tensors:
        assert [bool((t[i] == 0).all()) for i in range(5)] == [True, False, True, False, True] and bool((t[1::2] == 1).all())
    for bad in (-1, 5):
        with pytest.raises(ops.KernelRefused):
            slots.clear(bad)
    with pytest.raises(ops.KernelRefused):  # (no slots: nothing to clear, but a table all the same)
        ops.SlotTensors([t[:0] for t in tensors]).clear(0)


def test_many_f32_ranges():
    """Whole pieces, no fewer ranges than the blocks of 128 rows have, or nothing."""
    from nanospec_amd.kernels import ops

    for m in (129, 300, 2048):
        for n in (4, 260, 2048, 4096):
            for k in (512, 640, 1408, 2048, 2304, 5120, 8192):
                ranges = ops.many_f32_ranges(m, n, k, 256)
                assert ranges is None or (k % (128 * ranges) == 0 and k // ranges >= 256 and ops.rows_plan(n, k, m, units=256)[0] <= ranges <= 16)
    assert ops.many_f32_ranges(130, 2048, 4096, 256) == 4 and ops.many_f32_ranges(2048, 2048, 4096, 256) == 2 and ops.many_f32_ranges(300, 260, 3712, 256) is None


def test_split_plan():
    """What goes to the split kernel: whole stages, enough tiles; every plan is one that the launch takes."""
    from nanospec_amd.kernels import ops

    for m in (1, 47, 48, 65, 112, 128, 130, 777, 2048, 5000):
        for n in (1, 512, 2048, 3072, 16384, 128256):
            for k in (32, 1000, 1024, 1056, 2048, 8192):
                plan = ops.split_plan(m, n, k, 256)
                if plan is not None:
                    rows, ranges = plan
                    assert m >= 48 and m * n * k >= 2e9 and k % 32 == 0 and rows in (64, 96, 112, 128) and 1 <= ranges <= k // 32
    assert ops.split_plan(832, 16384, 2048, 256) == (128, 1) and ops.split_plan(512, 2048, 8192, 256) == (128, 4) and ops.split_plan(832, 2048, 2048, 256) == (64, 1)
    assert ops.split_plan(47, 128256, 2048, 256) is None and ops.split_plan(256, 512, 2048, 256) is None


@pytest.mark.parametrize("m", [1, 7, 16, 33, 64])
@pytest.mark.parametrize("n,k", [(48, 64), (130, 200), (1000, 4096), (257, 1064), (16, 8), (4096, 14336)])
def test_linear_tiled(m, n, k):
    """The streaming kernel on weights in the tiled layout: sizes that are no multiples of the tile, every wave count."""
    ops = _ops()
    torch.manual_seed(m + n + k)
    x = torch.randn(m, k, dtype=torch.bfloat16, device=DEV)
    w = torch.randn(n, k, dtype=torch.bfloat16, device=DEV)
    w2 = torch.randn(n, k, dtype=torch.bfloat16, device=DEV)
    wt, wt2 = ops.TiledWeight(w), ops.TiledWeight(w2)
    ref = x.cpu().float() @ w.cpu().float().T
    for waves in (2, 4, 8):
        out = ops.linear_tiled(x, wt, out_f32=True, waves=waves)
        torch.testing.assert_close(out.cpu(), ref, rtol=1e-4, atol=1e-3 * math.sqrt(k))
    assert ulps_of_row_max(ops.linear_tiled(x, wt).cpu(), ref).max() <= 1.0
    u = x.cpu().float() @ w2.cpu().float().T
    act = ops.linear_tiled(x, wt, w2=wt2)
    assert ulps_of_row_max(act.cpu(), ref * torch.sigmoid(ref) * u).max() <= 1.0
    if n >= 64:  # a slice of rows, as the stacked gate/up and q/k/v matrices are used
        part = ops.linear_tiled(x, wt.rows(16, 48), out_f32=True)
        torch.testing.assert_close(part.cpu(), ref[:, 16:48], rtol=1e-4, atol=1e-3 * math.sqrt(k))


@pytest.mark.parametrize("m", [1, 3, 8, 16])
@pytest.mark.parametrize("n,k", [(48, 64), (130, 200), (1000, 4096), (257, 1064), (14336, 512)])
def test_gated_product_in_half_tiles(m, n, k):
    """silu(x Wg^T) * (x Wu^T) with 8 rows of each matrix per workgroup: the same bits as with 16, at sizes off the tile."""
    ops = _ops()
    torch.manual_seed(m + n + k)
    x = torch.randn(m + 3, k + 8, dtype=torch.bfloat16, device=DEV)[:m, :k]
    wg, wu = (torch.randn(n, k, dtype=torch.bfloat16, device=DEV) * 0.3 for _ in range(2))
    tg, tu = ops.TiledWeight(wg), ops.TiledWeight(wu)
    g, u = x.cpu().float() @ wg.cpu().float().T, x.cpu().float() @ wu.cpu().float().T
    for waves in (2, 4, 8):
        whole = ops.linear_tiled(x, tg, w2=tu, waves=waves, halves=False)
        halves = ops.linear_tiled(x, tg, w2=tu, waves=waves, halves=True)
        assert torch.equal(whole, halves)
        assert ulps_of_row_max(halves.cpu(), g * torch.sigmoid(g) * u).max() <= 1.0


@pytest.mark.parametrize("m", [17, 33, 48, 64, 5])
@pytest.mark.parametrize("n,k", [(48, 64), (130, 200), (1000, 4096), (257, 1064), (4096, 14336)])
def test_linear_wide(m, n, k):
    """The kernel for 17 to 64 rows: x through LDS, K cut into ranges; every count of ranges, sizes off the tile."""
    ops = _ops()
    torch.manual_seed(m + n + k)
    x = torch.randn(m + 3, k + 8, dtype=torch.bfloat16, device=DEV)[:m, :k]  # a strided view of a wider buffer
    w = torch.randn(n, k, dtype=torch.bfloat16, device=DEV)
    w2 = torch.randn(n, k, dtype=torch.bfloat16, device=DEV)
    wt, wt2 = ops.TiledWeight(w), ops.TiledWeight(w2)
    ref = x.cpu().float() @ w.cpu().float().T
    k_tiles = -(-k // 128)
    for ks in sorted({1, 2, min(5, k_tiles), k_tiles, 0} - {k_tiles + 1}):
        if ks > k_tiles:
            continue
        for nt in (1, 2):
            out = ops.linear_wide(x, wt, out_f32=True, ksplit=ks, nt=nt)
            torch.testing.assert_close(out.cpu(), ref, rtol=1e-4, atol=1e-3 * math.sqrt(k))
    assert ulps_of_row_max(ops.linear_wide(x, wt).cpu(), ref).max() <= 1.0
    u = x.cpu().float() @ w2.cpu().float().T
    for nt in (1, 2):
        act = ops.linear_wide(x, wt, w2=wt2, nt=nt)
        assert ulps_of_row_max(act.cpu(), ref * torch.sigmoid(ref) * u).max() <= 1.0


@pytest.mark.parametrize("form", range(4))
@pytest.mark.parametrize("m,n,k", [(1, 4, 384), (129, 68, 384), (257, 132, 512), (300, 640, 2048), (1100, 260, 640)])
def test_linear_many(form, m, n, k):
    """Products of many rows from plain matrices: every tile at sizes off its edges (and more tiles than an XCD's patch), the shortest
    inner sizes, strided rows and results, everything that may follow the product in that tile, and the others refused; an activation has the values that its own kernel has."""
    ops = _ops()
    torch.manual_seed(m + n + k)
    x = torch.randn(m + 3, k + 8, dtype=torch.bfloat16, device=DEV)[:m, :k]
    w = torch.randn(n, k, dtype=torch.bfloat16, device=DEV)
    w2 = torch.randn(n, k, dtype=torch.bfloat16, device=DEV)
    ref, u = x.cpu().float() @ w.cpu().float().T, x.cpu().float() @ w2.cpu().float().T
    wide = torch.full((m + 1, n + 4), 7.0, dtype=torch.bfloat16, device=DEV)  # nothing beside the result is written
    out = wide[:m, :n]
    assert ulps_of_row_max(ops.linear_many(x, w, out, form).cpu(), ref).max() <= 1.0
    assert bool((wide[m] == 7).all()) and bool((wide[:, n:] == 7).all())
    plain = out.clone()
    for act in ops.ACTIVATIONS:
        if form < 3:
            assert torch.equal(ops.linear_many(x, w, out, form, act=act), ops.activation(plain.clone(), act)), act
        else:
            with pytest.raises(ops.KernelRefused):
                ops.linear_many(x, w, out, form, act=act)
    resid = torch.randn(m, n, dtype=torch.bfloat16, device=DEV) * 30
    out.copy_(resid)
    assert ulps_of_row_max(ops.linear_many(x, w, out, form, add=True).cpu(), resid.cpu().float() + ref).max() <= 1.0
    if form >= 2:
        assert ulps_of_row_max(ops.linear_many(x, w, out, form, w2=w2).cpu(), ref * torch.sigmoid(ref) * u).max() <= 1.5
    else:
        with pytest.raises(ops.KernelRefused):
            ops.linear_many(x, w, out, form, w2=w2)
    weight = (1 + 0.1 * torch.randn(n, device=DEV)).bfloat16()
    for ranges in (2, 4):
        if k % (128 * ranges) or k // ranges < 256:
            continue
        scratch = torch.empty(ranges * m * n, device=DEV)
        if form != 2:
            with pytest.raises(ops.KernelRefused):
                ops.linear_many(x, w, scratch, form, ranges=ranges)
            continue
        parts = ops.linear_many(x, w, scratch, form, ranges=ranges)
        torch.testing.assert_close(parts.ws.view(ranges, m, n).double().sum(0).cpu(), x.cpu().double() @ w.cpu().double().T, rtol=1e-5, atol=1e-5 * math.sqrt(k))
        assert ulps_of_row_max(ops.reduce_partial(parts).cpu(), ref).max() <= 1.0
        # the norm that reads them: the stream and the ranges are added in 32-bit and rounded once
        r = resid.clone()
        y = ops.rmsnorm(weight, 1e-5, resid=r, x=parts, write_resid=True)
        assert ulps_of_row_max(r.cpu(), resid.cpu().float() + ref).max() <= 0.51
        torch.testing.assert_close(y.cpu(), pl.rms_norm(r.cpu(), weight.cpu(), 1e-5), **_tol(torch.bfloat16))


@pytest.mark.parametrize("m,n,k", [(129, 4, 512), (257, 132, 640), (300, 640, 2048), (1100, 260, 4096), (200, 1024, 5120), (130, 2048, 4096)])
def test_linear_many_f32(m, n, k):
    """32-bit results of many rows: the kernel, and the part's own door to it."""
    from nanospec_amd.engine.arena import Arena
    from nanospec_amd.parts.linear import LinearWeight

    ops = _ops()
    torch.manual_seed(m + n + k)
    x = torch.randn(m + 3, k + 8, dtype=torch.bfloat16, device=DEV)[:m, :k]
    w = torch.randn(n, k, dtype=torch.bfloat16, device=DEV)
    a, b = x.cpu().double(), w.cpu().double()
    bound = k / 8 * 2.0**-24 * (a.abs() @ b.abs().T)  # a rounding of the sum for every block of 8 k
    wide = torch.full((m + 1, n), 7.0, device=DEV)
    y = ops.linear_many(x, w, wide[:m], ops.MANY_SPLIT_FORM)
    assert bool(((y.cpu().double() - a @ b.T).abs() <= bound).all()) and bool((wide[m] == 7).all())
    # through the part's own door in as many ranges of K as the blocks of 128 rows that other models run: as near to 64 bits as those (two norms of n independent
    # roundings differ by some n^(-1/2) of themselves by chance)
    far = lambda y: float((y.cpu().double() - a @ b.T).norm())
    arena, into = Arena(x.device), torch.empty(m, n, device=DEV)
    for z in (LinearWeight(w)(x, out_f32=True), LinearWeight(w)(x, out=into, out_f32=True, arena=arena)):
        assert far(z) <= (1 + 8 * (m * n) ** -0.5) * far(LinearWeight(w, keep_plain=False)(x, out_f32=True)) and bool(((z.cpu().double() - a @ b.T).abs() <= bound).all())
    with pytest.raises(ops.KernelRefused):  # (a 32-bit result does not go into a bfloat16 tensor)
        LinearWeight(w)(x, out=torch.empty(m, n, dtype=torch.bfloat16, device=DEV), out_f32=True)
    for bad in (dict(act="silu"), dict(add=True), dict(out=torch.empty(m, 2 * n, device=DEV)[:, :n]), dict(form=0)):
        with pytest.raises(ops.KernelRefused):
            ops.linear_many(**{**dict(x=x, w=w, out=y, form=ops.MANY_SPLIT_FORM), **bad})


def test_linear_many_refuses():
    ops = _ops()
    x, w, out = (torch.zeros(200, k, dtype=torch.bfloat16, device=DEV) for k in (512, 512, 200))
    for bad in (dict(x=x[:, :128], w=w[:, :128].contiguous()), dict(x=x[:, 4:260], w=w[:, :256].contiguous()), dict(out=out[:, :198], w=w[:198].contiguous()),
                dict(ranges=3), dict(add=True, act="silu"), dict(form=7), dict(x=x.float())):
        with pytest.raises(ops.KernelRefused):
            ops.linear_many(**{**dict(x=x, w=w, out=out, form=2), **bad})


@pytest.mark.parametrize("m", [17, 33, 48, 64, 5])
@pytest.mark.parametrize("n,k", [(48, 64), (130, 200), (1000, 4096), (257, 1064), (1440, 512)])
def test_linear_wide_dealt_to_the_compute_units(m, n, k):
    """The same kernel with three waves a workgroup (one matrix) and with gate and up by half tiles in workgroups of four
    or seven waves: every form adds a sum's terms in the same order, so the results are equal bit for bit."""
    ops = _ops()
    from nanospec_amd.kernels import KernelRefused

    torch.manual_seed(m + n + k + 1)
    x = torch.randn(m + 3, k + 8, dtype=torch.bfloat16, device=DEV)[:m, :k]
    w = torch.randn(n, k, dtype=torch.bfloat16, device=DEV)
    w2 = torch.randn(n, k, dtype=torch.bfloat16, device=DEV)
    wt, wt2 = ops.TiledWeight(w), ops.TiledWeight(w2)
    ref = x.cpu().float() @ w.cpu().float().T
    k_tiles = -(-k // 128)
    for ks in sorted({1, 2, min(3, k_tiles)}):
        if ks > k_tiles:
            continue
        four = ops.linear_wide(x, wt, out_f32=True, ksplit=ks, nt=1, waves=4)
        three = ops.linear_wide(x, wt, out_f32=True, ksplit=ks, nt=1, waves=3)
        torch.testing.assert_close(three.cpu(), ref, rtol=1e-4, atol=1e-3 * math.sqrt(k))
        assert torch.equal(three, four), f"{ks} ranges"
        if ks > 1:
            part = ops.linear_wide(x, wt, ksplit=ks, nt=1, waves=3, defer=True)
            assert torch.equal(ops.reduce_partial(part), ops.linear_wide(x, wt, ksplit=ks, nt=1, waves=4))
    u = x.cpu().float() @ w2.cpu().float().T
    whole = ops.linear_wide(x, wt, w2=wt2, ksplit=1, nt=1, waves=4, halves=False)
    assert ulps_of_row_max(whole.cpu(), ref * torch.sigmoid(ref) * u).max() <= 1.0
    for waves in (4, 7):
        halves = ops.linear_wide(x, wt, w2=wt2, ksplit=1, nt=1, waves=waves, halves=True)
        assert torch.equal(halves, whole), f"half tiles, {waves} waves"
    assert torch.equal(ops.linear_wide(x, wt, w2=wt2, ksplit=1, nt=1), whole)  # whichever form the plan deals
    for bad in (dict(waves=7), dict(waves=3, w2=wt2), dict(waves=7, halves=True), dict(w2=wt2, waves=4, halves=True, ksplit=2),
                dict(waves=3, nt=2), dict(waves=5)):
        with pytest.raises(KernelRefused):
            ops.linear_wide(x, wt, **{"ksplit": 1, "nt": 1, **bad})


def test_wide_plans_deal_evenly():
    """What the plans choose at the three shapes' sizes on 256 compute units: q/k/v of the 8B shape in workgroups of three
    waves over two ranges (256 workgroups where four waves over three ranges are 288), gate and up by half tiles."""
    ops = _ops()
    assert ops.wide_plan(6144, 4096, 64, units=256) == (2, 1) and ops.wide_waves(6144, 4096, 64, 2, 1, units=256) == (3, False)
    assert ops.wide_plan(4096, 4096, 64, units=256) == (4, 1) and ops.wide_waves(4096, 4096, 64, 4, 1, units=256) == (4, False)
    assert ops.wide_plan(4096, 14336, 64, units=256) == (4, 1) and ops.wide_waves(4096, 14336, 64, 4, 1, units=256) == (4, False)
    assert ops.wide_waves(14336, 4096, 64, 1, 1, gated=True, units=256) == (7, True)   # 1,792 half tiles: 7 for each of 256 units
    assert ops.wide_waves(8192, 2048, 64, 1, 1, gated=True, units=256) == (4, True)    # 1,024 half tiles: 4 for each
    assert ops.wide_waves(28672, 8192, 64, 1, 1, gated=True, units=256) == (4, False)  # 448 workgroups of whole tiles fill the GPU
    assert ops.wide_waves(14336, 4096, 100, 1, 1, units=256) == (4, False)             # more than 64 rows of one matrix: four waves
    assert ops.wide_waves(14336, 4096, 100, 1, 1, gated=True, units=256) == (7, True)  # gate and up: half tiles only
    assert ops.wide_waves(8192, 2048, 100, 1, 1, gated=True, units=256) == (4, True)
    assert ops.wide_waves(14336, 4096, 64, 2, 1, gated=True, units=256) == (4, False)  # gate and up over ranges: whole tiles


def test_linear_tiled_refuses():
    ops = _ops()
    from nanospec_amd.kernels import KernelRefused

    w = torch.randn(16, 64, dtype=torch.bfloat16, device=DEV)
    wt = ops.TiledWeight(w)
    with pytest.raises(KernelRefused):
        ops.linear_tiled(torch.randn(65, 64, dtype=torch.bfloat16, device=DEV), wt)  # too many rows
    with pytest.raises(KernelRefused):
        ops.linear_tiled(torch.randn(4, 60, dtype=torch.bfloat16, device=DEV), wt)  # inner size differs
    with pytest.raises(KernelRefused):
        ops.linear_tiled(torch.randn(4, 64, dtype=torch.float32, device=DEV), wt)
    with pytest.raises(KernelRefused):
        ops.TiledWeight(w.float())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_silu_mul(dtype):
    ops = _ops()
    gu = torch.randn(9, 2 * 88, dtype=dtype, device=DEV) * 3
    g, u = gu.cpu().float()[:, :88], gu.cpu().float()[:, 88:]
    torch.testing.assert_close(ops.silu_mul(gu).cpu().float(), (torch.nn.functional.silu(g) * u).to(dtype).float(), **_tol(dtype))


# ------------------------------------------------------------------------------------------------ cache helpers


def make_cache(pages, page, kvh, hd, dtype):
    k = torch.zeros(pages, kvh, page, hd, dtype=dtype, device=DEV)
    v = torch.zeros(pages, kvh, hd, page, dtype=dtype, device=DEV)
    return k, v


def scattered_tables(lens, page, pages, seed=0):
    """Block tables on scattered, non-contiguous pages."""
    g = torch.Generator().manual_seed(seed)
    perm = torch.randperm(pages, generator=g).tolist()
    width = max(-(-n // page) for n in lens)
    table = torch.full((len(lens), width), -1, dtype=torch.int32)
    for b, n in enumerate(lens):
        for i in range(-(-n // page)):
            table[b, i] = perm.pop()
    return table


FORMS = [(False, 1.0), (True, 0.75)]  # (pairs of channels 2j and 2j + 1 instead of j and j + d/2, a factor on cosine and sine)


def plain_rotation(x, cos, sin, interleaved=False, factor=1.0):
    """The rotation of x [T, heads, d] in the given form.  The half-split form is the plain implementation's; the
    interleaved form turns channels 2j and 2j + 1 by the same angle j, written out here pair by pair."""
    if not interleaved:
        return pl.rotate(x, cos * factor, sin * factor)
    half = x.shape[-1] // 2
    c, s = (cos[:, None, :half] * factor), (sin[:, None, :half] * factor)
    a, b = x.float()[..., 0::2], x.float()[..., 1::2]
    out = torch.empty_like(x, dtype=torch.float32)
    out[..., 0::2] = a * c - b * s
    out[..., 1::2] = b * c + a * s
    return out.to(x.dtype)


@pytest.mark.parametrize("form", FORMS, ids=["halves", "interleaved"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rot", [24, 16, 0])
def test_rope_kv_write(dtype, rot, form):
    """q rotated in place, k rotated into its page slot, v into the transposed page; against the plain rotation."""
    ops = _ops()
    torch.manual_seed(1)
    heads, kvh, hd, page = 6, 3, 24, 4
    starts, lens = [0, 5, 9], [7, 1, 3]
    n = sum(lens)
    table = scattered_tables([s + l for s, l in zip(starts, lens)], page, 16).to(DEV)
    positions = torch.tensor([s + i for s, l in zip(starts, lens) for i in range(l)], dtype=torch.int32, device=DEV)
    token_req = torch.tensor([b for b, l in enumerate(lens) for _ in range(l)], dtype=torch.int32, device=DEV)
    qkv = torch.randn(n, (heads + 2 * kvh) * hd, dtype=dtype, device=DEV)
    before = qkv.clone().cpu()
    k, v = make_cache(16, page, kvh, hd, dtype)
    inv = pl.inverse_frequencies(rot, 10000.0, None) if rot else torch.zeros(1)
    ops.rope_kv_write(qkv, positions, token_req, table, inv.to(DEV), k, v, heads, kvh, hd, rot, interleaved=form[0], factor=form[1])
    q0 = before[:, : heads * hd].view(n, heads, hd)
    k0 = before[:, heads * hd : (heads + kvh) * hd].view(n, kvh, hd)
    v0 = before[:, (heads + kvh) * hd :].view(n, kvh, hd)
    if rot:
        cos, sin = pl.rotation_tables(positions.cpu(), inv)
        q_ref = torch.cat([plain_rotation(q0[..., :rot], cos, sin, *form), q0[..., rot:]], -1)
        k_ref = torch.cat([plain_rotation(k0[..., :rot], cos, sin, *form), k0[..., rot:]], -1)
    else:
        q_ref, k_ref = q0, k0
    tol = _tol(dtype)
    torch.testing.assert_close(qkv.cpu()[:, : heads * hd].view(n, heads, hd).float(), q_ref.float(), **tol)
    assert torch.equal(qkv.cpu()[:, heads * hd :], before[:, heads * hd :])  # k and v stay as they were in the buffer
    for t in range(n):
        b, p = int(token_req[t]), int(positions[t])
        pg, off = int(table[b, p // page]), p % page
        torch.testing.assert_close(k[pg, :, off].cpu().float(), k_ref[t].float(), **tol)
        assert torch.equal(v[pg, :, :, off].cpu(), v0[t])


@pytest.mark.parametrize("form", FORMS, ids=["halves", "interleaved"])
@pytest.mark.parametrize("heads,kvh,hd,rot,page", [(6, 3, 32, 32, 4), (4, 1, 48, 16, 8), (8, 2, 128, 128, 16), (2, 2, 16, 0, 4)])
def test_qkv_product_with_fused_rotation_and_cache_write(heads, kvh, hd, rot, page, form):
    """One kernel for x @ [Wq; Wk; Wv]^T, the rotation of q and k and the write of k and v into their pages, against the
    plain product followed by the plain rotation."""
    ops = _ops()
    torch.manual_seed(hd + rot)
    hidden = 72
    starts, lens = [3, 0, 9], [5, 1, 2]
    n = sum(lens)
    table = scattered_tables([s + l for s, l in zip(starts, lens)], page, 16, seed=2).to(DEV)
    positions = torch.tensor([s + i for s, l in zip(starts, lens) for i in range(l)], dtype=torch.int32, device=DEV)
    token_req = torch.tensor([b for b, l in enumerate(lens) for _ in range(l)], dtype=torch.int32, device=DEV)
    w = (torch.randn((heads + 2 * kvh) * hd, hidden) * 0.3).to(torch.bfloat16)
    x = torch.randn(n, hidden).to(torch.bfloat16)
    wt = ops.TiledWeight(w.to(DEV), ops.qkv_rope_row_order(heads, kvh, hd, rot, form[0]))
    q_out = torch.zeros(n, (heads + 2 * kvh) * hd, dtype=torch.bfloat16, device=DEV)
    k, v = make_cache(16, page, kvh, hd, torch.bfloat16)
    inv = pl.inverse_frequencies(rot, 10000.0, None) if rot else torch.zeros(1)
    ops.linear_qkv_rope(x.to(DEV), wt, q_out, positions, token_req, table, inv.to(DEV), k, v, heads, kvh, hd, rot, interleaved=form[0],
                        factor=form[1])
    full = x.float() @ w.float().T  # 32-bit sums: the kernel rotates before it rounds
    q0 = full[:, : heads * hd].view(n, heads, hd)
    k0 = full[:, heads * hd : (heads + kvh) * hd].view(n, kvh, hd)
    v0 = full[:, (heads + kvh) * hd :].view(n, kvh, hd)
    if rot:
        cos, sin = pl.rotation_tables(positions.cpu(), inv)
        q0 = torch.cat([plain_rotation(q0[..., :rot], cos, sin, *form), q0[..., rot:]], -1)
        k0 = torch.cat([plain_rotation(k0[..., :rot], cos, sin, *form), k0[..., rot:]], -1)
    assert ulps_of_row_max(q_out[:, : heads * hd].cpu(), q0.reshape(n, -1)).max() <= 1.0
    for t in range(n):
        b, p = int(token_req[t]), int(positions[t])
        pg, off = int(table[b, p // page]), p % page
        assert ulps_of_row_max(k[pg, :, off].cpu().reshape(1, -1), k0[t].reshape(1, -1)).max() <= 1.0
        assert ulps_of_row_max(v[pg, :, :, off].cpu().reshape(1, -1), v0[t].reshape(1, -1)).max() <= 1.0


@pytest.mark.parametrize("form", FORMS, ids=["halves", "interleaved"])
@pytest.mark.parametrize("rows", [17, 40, 64, 100, 128])
@pytest.mark.parametrize("heads,kvh,hd,rot,page,hidden,ksplit", [(6, 3, 32, 32, 4, 384, 3), (4, 1, 48, 16, 8, 520, 2), (8, 2, 128, 128, 16, 1024, 4),
                                                                 (2, 2, 16, 0, 4, 256, 2)])
def test_qkv_product_in_ranges_joined_by_the_rotation_kernel(rows, heads, kvh, hd, rot, page, hidden, ksplit, form):
    """17 to 128 rows: the stacked product with K cut into ranges from the matrix tiled in the few-row kernel's row order,
    and one kernel that adds the ranges, rotates q and k and writes k and v into their pages; against the plain product
    followed by the plain rotation.  Requests of several tokens and of one, pages scattered."""
    ops = _ops()
    torch.manual_seed(hd + rot + rows)
    lens = [rows - 9, 1, 5, 1, 2] if rows > 20 else [rows - 4, 1, 3]
    starts = [3, 0, 9, 30, 1][: len(lens)]
    n = sum(lens)
    assert n == rows
    table = scattered_tables([s + l for s, l in zip(starts, lens)], page, 64, seed=2).to(DEV)
    positions = torch.tensor([s + i for s, l in zip(starts, lens) for i in range(l)], dtype=torch.int32, device=DEV)
    token_req = torch.tensor([b for b, l in enumerate(lens) for _ in range(l)], dtype=torch.int32, device=DEV)
    w = (torch.randn((heads + 2 * kvh) * hd, hidden) * 0.3).to(torch.bfloat16)
    x = torch.randn(n, hidden).to(torch.bfloat16)
    wt = ops.TiledWeight(w.to(DEV), ops.qkv_rope_row_order(heads, kvh, hd, rot, form[0]))
    q_out = torch.zeros(n, (heads + 2 * kvh) * hd, dtype=torch.bfloat16, device=DEV)
    k, v = make_cache(64, page, kvh, hd, torch.bfloat16)
    inv = pl.inverse_frequencies(rot, 10000.0, None) if rot else torch.zeros(1)
    part = ops.linear_wide(x.to(DEV), wt, ksplit=ksplit, nt=1, defer=True)
    assert isinstance(part, ops.PartialSums) and part.ksplit == ksplit
    ops.rope_kv_from_partial(part, q_out, positions, token_req, table, inv.to(DEV), k, v, heads, kvh, hd, rot, interleaved=form[0],
                             factor=form[1])
    full = x.float() @ w.float().T  # 32-bit sums: the kernel rotates before it rounds
    q0 = full[:, : heads * hd].view(n, heads, hd)
    k0 = full[:, heads * hd : (heads + kvh) * hd].view(n, kvh, hd)
    v0 = full[:, (heads + kvh) * hd :].view(n, kvh, hd)
    if rot:
        cos, sin = pl.rotation_tables(positions.cpu(), inv)
        q0 = torch.cat([plain_rotation(q0[..., :rot], cos, sin, *form), q0[..., rot:]], -1)
        k0 = torch.cat([plain_rotation(k0[..., :rot], cos, sin, *form), k0[..., rot:]], -1)
    assert ulps_of_row_max(q_out[:, : heads * hd].cpu(), q0.reshape(n, -1)).max() <= 1.0
    assert torch.count_nonzero(q_out[:, heads * hd :]) == 0  # only q goes to the attention input
    for t in range(n):
        b, p = int(token_req[t]), int(positions[t])
        pg, off = int(table[b, p // page]), p % page
        assert ulps_of_row_max(k[pg, :, off].cpu().reshape(1, -1), k0[t].reshape(1, -1)).max() <= 1.0
        assert ulps_of_row_max(v[pg, :, :, off].cpu().reshape(1, -1), v0[t].reshape(1, -1)).max() <= 1.0
    # without the cache write only q is produced
    k2, v2 = make_cache(64, page, kvh, hd, torch.bfloat16)
    before = (k2.clone(), v2.clone())
    ops.rope_kv_from_partial(part, q_out, positions, token_req, table, inv.to(DEV), k2, v2, heads, kvh, hd, rot, write_kv=False)
    assert torch.equal(k2, before[0]) and torch.equal(v2, before[1])


@pytest.mark.parametrize("m", [1, 7, 16])
@pytest.mark.parametrize("hidden,inner", [(136, 264), (4096, 1024), (64, 8)])
def test_product_that_updates_the_residual_and_feeds_the_next_norm(m, hidden, inner):
    """resid += x @ W^T with what the following RMS norm needs as by-products, and the products that take them in place of a
    normalised input, against the plain sum, the plain norm and the plain product."""
    ops = _ops()
    torch.manual_seed(m + hidden)
    eps = 1e-5
    x = torch.randn(m, inner).to(torch.bfloat16)
    w = (torch.randn(hidden, inner) / math.sqrt(inner)).to(torch.bfloat16)
    resid0 = torch.randn(m, hidden).to(torch.bfloat16)
    w_norm = (1 + 0.2 * torch.randn(hidden)).to(torch.bfloat16)
    resid = resid0.to(DEV).clone()
    pre = ops.linear_resid_norm(x.to(DEV), ops.TiledWeight(w.to(DEV)), resid, w_norm.to(DEV), eps)
    # the sum: product rounded to bfloat16, then added in 32-bit and rounded (reference: model/llama.py:204-208)
    delta = (x.float() @ w.float().T).to(torch.bfloat16)
    want = (resid0.float() + delta.float()).to(torch.bfloat16)
    err = (resid.cpu().float() - want.float()).abs() / want.float().abs().clamp_min(0.25)
    assert err.max() <= 2.0 ** -6  # a flipped rounding of the product moves the sum by at most two of its last places
    got = resid.cpu()
    assert torch.equal(pre.x.cpu(), (got.float() * w_norm.float()).to(torch.bfloat16))
    assert pre.ssq.shape == (m, -(-hidden // 16))
    torch.testing.assert_close(pre.ssq.sum(1).cpu(), (got.float() ** 2).sum(-1), rtol=1e-5, atol=1e-6)
    # consumers: the plain norm of the kernel's own sum, then the plain products
    normed = pl.rms_norm(got, w_norm, eps)
    out_n = 152
    w3 = (torch.randn(out_n, hidden) / math.sqrt(hidden)).to(torch.bfloat16)
    w4 = (torch.randn(out_n, hidden) / math.sqrt(hidden)).to(torch.bfloat16)
    ref = normed.float() @ w3.float().T
    out = ops.linear_tiled(pre, ops.TiledWeight(w3.to(DEV)))
    assert ulps_of_row_max(out.cpu(), ref).max() <= 2.0
    out32 = ops.linear_tiled(pre, ops.TiledWeight(w3.to(DEV)), out_f32=True)
    assert ulps_of_row_max(out32.cpu(), ref).max() <= 1.0
    up = normed.float() @ w4.float().T
    act = ops.linear_tiled(pre, ops.TiledWeight(w3.to(DEV)), w2=ops.TiledWeight(w4.to(DEV)))
    assert ulps_of_row_max(act.cpu(), ref * torch.sigmoid(ref) * up).max() <= 2.0
    # the kernel that shares x through LDS takes the same input: whole tiles, half tiles in workgroups of 4 and 7 waves,
    # one matrix in workgroups of 3 and 4 waves
    t3, t4 = ops.TiledWeight(w3.to(DEV)), ops.TiledWeight(w4.to(DEV))
    for waves, halves in ((4, False), (4, True), (7, True)):
        act = ops.linear_wide(pre, t3, w2=t4, ksplit=1, nt=1, waves=waves, halves=halves)
        assert ulps_of_row_max(act.cpu(), ref * torch.sigmoid(ref) * up).max() <= 2.0, (waves, halves)
    for waves in (3, 4):
        assert ulps_of_row_max(ops.linear_wide(pre, t3, ksplit=1, nt=1, waves=waves, out_f32=True).cpu(), ref).max() <= 1.0
    if hidden >= 256:
        from nanospec_amd.kernels import KernelRefused

        with pytest.raises(KernelRefused):
            ops.linear_wide(pre, t3, ksplit=2, nt=1)  # a pre-normed input goes with one range


@pytest.mark.parametrize("m", [65, 81, 100, 113, 128])
@pytest.mark.parametrize("n,k", [(48, 64), (130, 200), (1000, 4096), (4096, 2056)])
def test_linear_wide_up_to_128_rows(m, n, k):
    """65 to 128 rows: one matrix, one row tile per wave; every count of ranges, sizes off the tile; other forms refused."""
    ops = _ops()
    torch.manual_seed(m + n + k)
    x = torch.randn(m + 3, k + 8, dtype=torch.bfloat16, device=DEV)[:m, :k]
    w = torch.randn(n, k, dtype=torch.bfloat16, device=DEV)
    wt = ops.TiledWeight(w)
    ref = x.cpu().float() @ w.cpu().float().T
    k_tiles = -(-k // 128)
    for ks in sorted({1, min(2, k_tiles), min(5, k_tiles), k_tiles, 0}):
        out = ops.linear_wide(x, wt, out_f32=True, ksplit=ks, nt=0 if ks == 0 else 1)
        torch.testing.assert_close(out.cpu(), ref, rtol=1e-4, atol=1e-3 * math.sqrt(k))
    assert ulps_of_row_max(ops.linear_wide(x, wt).cpu(), ref).max() <= 1.0
    if k_tiles >= 2:
        part = ops.linear_wide(x, wt, ksplit=2, nt=1, defer=True)
        assert torch.equal(ops.reduce_partial(part), ops.linear_wide(x, wt, ksplit=2, nt=1))
    with pytest.raises(ops.KernelRefused):
        ops.linear_wide(x, wt, nt=2)
    with pytest.raises(ops.KernelRefused):
        ops.linear_wide(x, wt, w2=wt, ksplit=1, nt=1, waves=4, halves=False)  # whole tiles of two matrices: up to 64 rows
    with pytest.raises(ops.KernelRefused):
        ops.linear_wide(torch.randn(129, k, dtype=torch.bfloat16, device=DEV), wt)
    # gate and up by half tiles hold one set of sums, so they take these rows too
    w2 = torch.randn(n, k, dtype=torch.bfloat16, device=DEV)
    wt2 = ops.TiledWeight(w2)
    want = ref * torch.sigmoid(ref) * (x.cpu().float() @ w2.cpu().float().T)
    seven = ops.linear_wide(x, wt, w2=wt2, ksplit=1, nt=1, waves=7, halves=True)
    assert ulps_of_row_max(seven.cpu(), want).max() <= 1.0
    assert torch.equal(ops.linear_wide(x, wt, w2=wt2, ksplit=1, nt=1, waves=4, halves=True), seven)
    assert torch.equal(ops.linear_wide(x, wt, w2=wt2, ksplit=1, nt=1), seven)  # (the form the plan deals: one of the two)
    assert torch.equal(seven[:64], ops.linear_wide(x[:64], wt, w2=wt2, ksplit=1, nt=1, waves=4, halves=False))


@pytest.mark.parametrize("m", [129, 300, 1031])
@pytest.mark.parametrize("n,k", [(48, 64), (130, 200), (1000, 2056), (4096, 1024)])
def test_linear_rows(m, n, k):
    """Any number of rows in blocks of 128 (what a model that keeps the tiled layout only runs its prompts through): every
    count of row tiles per wave and several counts of ranges, sizes off every tile, the gated form, 32-bit results."""
    ops = _ops()
    torch.manual_seed(m + n + k)
    x = torch.randn(m + 3, k + 8, dtype=torch.bfloat16, device=DEV)[:m, :k]
    w = torch.randn(n, k, dtype=torch.bfloat16, device=DEV)
    w2 = torch.randn(n, k, dtype=torch.bfloat16, device=DEV)
    wt, wt2 = ops.TiledWeight(w), ops.TiledWeight(w2)
    ref = x.cpu().float() @ w.cpu().float().T
    k_tiles = -(-k // 128)
    for nt in (2, 4):
        for ks in sorted({1, min(3, k_tiles), 0}):
            out = ops.linear_rows(x, wt, out_f32=True, ksplit=ks, nt=nt if ks else 0)
            torch.testing.assert_close(out.cpu(), ref, rtol=1e-4, atol=1e-3 * math.sqrt(k))
    assert ulps_of_row_max(ops.linear_rows(x, wt).cpu(), ref).max() <= 1.0
    u = x.cpu().float() @ w2.cpu().float().T
    for nt in (1, 2):
        for ks in (1, min(2, k_tiles)):
            act = ops.linear_rows(x, wt, w2=wt2, ksplit=ks, nt=nt)
            assert ulps_of_row_max(act.cpu(), ref * torch.sigmoid(ref) * u).max() <= 1.0
    with pytest.raises(ops.KernelRefused):
        ops.linear_rows(x, wt, nt=1)


@pytest.mark.parametrize("m", [17, 40, 64, 97, 128])
@pytest.mark.parametrize("hidden,inner,ksplit", [(136, 1024, 4), (4096, 1024, 2), (72, 512, 3)])
def test_ranges_of_a_product_added_by_the_norm_that_reads_them(m, hidden, inner, ksplit):
    """The 17-to-64-row product leaves the ranges of K unadded; the RMS norm adds them as it reads them, with the residual
    sum and with a row gather; ``reduce_partial`` gives the same tensor as the product run whole."""
    ops = _ops()
    torch.manual_seed(m + hidden)
    eps = 1e-5
    x = torch.randn(m, inner).to(torch.bfloat16).to(DEV)
    w = (torch.randn(hidden, inner) / math.sqrt(inner)).to(torch.bfloat16).to(DEV)
    wt = ops.TiledWeight(w)
    resid0 = torch.randn(m, hidden).to(torch.bfloat16)
    w_norm = (1 + 0.2 * torch.randn(hidden)).to(torch.bfloat16)
    part = ops.linear_wide(x, wt, ksplit=ksplit, nt=1, defer=True)
    assert isinstance(part, ops.PartialSums) and part.ws.numel() >= ksplit * m * hidden
    whole = ops.linear_wide(x, wt, ksplit=ksplit, nt=1)
    assert torch.equal(ops.reduce_partial(part), whole)
    # sum + norm
    resid = resid0.to(DEV).clone()
    out = ops.rmsnorm(w_norm.to(DEV), eps, resid=resid, x=part, write_resid=True)
    resid_ref = resid0.to(DEV).clone()
    ref = ops.rmsnorm(w_norm.to(DEV), eps, resid=resid_ref, x=whole, write_resid=True)
    assert torch.equal(resid, resid_ref)
    assert ulps_of_row_max(out.cpu(), ref.cpu().float()).max() <= 1.0
    want = pl.rms_norm((resid0.float() + whole.cpu().float()).to(torch.bfloat16), w_norm, eps)
    assert ulps_of_row_max(out.cpu(), want.float()).max() <= 1.0
    # gathered rows, no residual
    rows = torch.tensor([m - 1, 0, 5], dtype=torch.int32, device=DEV)
    got = ops.rmsnorm(w_norm.to(DEV), eps, x=part, rows=rows)
    want = pl.rms_norm(whole.cpu()[rows.cpu().long()], w_norm, eps)
    assert ulps_of_row_max(got.cpu(), want.float()).max() <= 1.0


def test_qkv_product_takes_a_prenormed_input():
    ops = _ops()
    torch.manual_seed(3)
    heads, kvh, hd, rot, page, hidden, eps = 6, 2, 32, 32, 8, 96, 1e-6
    starts, lens = [3, 0, 9], [5, 1, 2]
    n = sum(lens)
    table = scattered_tables([s + l for s, l in zip(starts, lens)], page, 16, seed=2).to(DEV)
    positions = torch.tensor([s + i for s, l in zip(starts, lens) for i in range(l)], dtype=torch.int32, device=DEV)
    token_req = torch.tensor([b for b, l in enumerate(lens) for _ in range(l)], dtype=torch.int32, device=DEV)
    r = torch.randn(n, hidden).to(torch.bfloat16)
    w_norm = (1 + 0.2 * torch.randn(hidden)).to(torch.bfloat16)
    w = (torch.randn((heads + 2 * kvh) * hd, hidden) * 0.3).to(torch.bfloat16)
    wt = ops.TiledWeight(w.to(DEV), ops.qkv_rope_row_order(heads, kvh, hd, rot))
    inv = pl.inverse_frequencies(rot, 10000.0, None).to(DEV)
    ssq = torch.zeros(n, 3)
    ssq[:, 1] = (r.float() ** 2).sum(-1)  # any split into parts has the same sum
    pre = ops.PreNormed((r.float() * w_norm.float()).to(torch.bfloat16).to(DEV), ssq.to(DEV), hidden, eps)
    outs = []
    for src in (pre, pl.rms_norm(r, w_norm, eps).to(DEV)):
        q_out = torch.zeros(n, heads * hd, dtype=torch.bfloat16, device=DEV)
        k, v = make_cache(16, page, kvh, hd, torch.bfloat16)
        ops.linear_qkv_rope(src, wt, q_out, positions, token_req, table, inv, k, v, heads, kvh, hd, rot)
        outs.append((q_out.cpu(), k.cpu(), v.cpu()))
    for a, b in zip(*outs):
        assert ulps_of_row_max(a.reshape(1, -1), b.reshape(1, -1).float()).max() <= 2.0
    assert outs[0][1].abs().sum() > 0


def fill_cache(k, v, table, lens, page, kvh, hd, dtype, seed=0, scale=1.0):
    """Random keys and values for positions [0, len) of every request, written through the block table.
    -> per request (K [len, kvh, hd], V [len, kvh, hd]) on the CPU."""
    g = torch.Generator().manual_seed(seed)
    out = []
    for b, n in enumerate(lens):
        kk = (torch.randn(n, kvh, hd, generator=g) * scale).to(dtype)
        vv = torch.randn(n, kvh, hd, generator=g).to(dtype)
        for p in range(n):
            pg, off = int(table[b, p // page]), p % page
            if pg < 0:
                continue
            k[pg, :, off] = kk[p].to(DEV)
            v[pg, :, :, off] = vv[p].to(DEV)
        out.append((kk, vv))
    return out


def plain_paged_attention(q, kvs, starts, lens, heads, scale_fix=1.0, window=0):
    """Rows of q (flat over requests) attend to their request's keys 0 .. position with the plain attention."""
    outs, at = [], 0
    for (kk, vv), s, n in zip(kvs, starts, lens):
        qi = q[at : at + n]
        o = pl.causal_attention(qi.cpu(), kk[: s + n], vv[: s + n], first_query=s)
        if window:
            o = torch.stack([pl.causal_attention(qi[i : i + 1].cpu(), kk[max(0, s + i - window + 1) : s + i + 1],
                                                 vv[max(0, s + i - window + 1) : s + i + 1], first_query=min(s + i, window - 1))[0]
                             for i in range(n)])
        outs.append(o)
        at += n
    return torch.cat(outs)


CASES = {
    # the four cases of the reference's tests/test_backends.py:44-59
    "prefill": ([0], [40]),
    "decode": ([37], [1]),
    "append6": ([37], [6]),
    "mixed": ([21, 50, 0], [1, 6, 9]),
    "long": ([300, 0, 511], [1, 70, 1]),
    # more than 64 pages a request at every page size: the kernels hold 64 page ids at a time
    "beyond64pages": ([1300, 0], [1, 1100]),
    # a decode row and a late portion of a prompt nine thousand tokens in: many reloads of the page ids, long key ranges
    "far": ([9000, 8990], [1, 70]),
}


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("case", list(CASES))
@pytest.mark.parametrize("heads,kvh,hd,page", [(8, 2, 128, 16), (6, 1, 48, 4), (4, 4, 16, 8)])
def test_attention_generic(dtype, case, heads, kvh, hd, page):
    ops = _ops()
    starts, lens = CASES[case]
    torch.manual_seed(3)
    total = [s + l for s, l in zip(starts, lens)]
    pages = sum(-(-t // page) for t in total) + 3
    table = scattered_tables(total, page, pages)
    k, v = make_cache(pages, page, kvh, hd, dtype)
    kvs = fill_cache(k, v, table, total, page, kvh, hd, dtype)
    n = sum(lens)
    q = torch.randn(n, heads * hd, dtype=dtype, device=DEV)
    positions = torch.tensor([s + i for s, l in zip(starts, lens) for i in range(l)], dtype=torch.int32, device=DEV)
    token_req = torch.tensor([b for b, l in enumerate(lens) for _ in range(l)], dtype=torch.int32, device=DEV)
    out = torch.empty(n, heads * hd, dtype=dtype, device=DEV)
    ops.attention_generic(q, out, k, v, token_req, positions, table.to(DEV), heads, kvh, hd, 1 / math.sqrt(hd))
    ref = plain_paged_attention(q.view(n, heads, hd), kvs, starts, lens, heads).reshape(n, -1)
    if dtype == torch.float32:
        torch.testing.assert_close(out.cpu(), ref, rtol=1e-4, atol=1e-5)
    else:
        assert ulps_of_row_max(out.cpu(), ref).max() <= 4  # the reference's bound, tests/test_backends.py:71


@pytest.mark.parametrize("n,k", [(16, 128), (40, 72), (100, 264), (2048, 8192), (33, 8)])
def test_untile_gives_the_matrix_back(n, k):
    """The re-laid copy of a matrix written out in plain rows again (rows and k that are no multiples of the tile: the
    padding is not written, and nothing outside the matrix is)."""
    ops = _ops()
    torch.manual_seed(n + k)
    w = torch.randn(n, k, dtype=torch.bfloat16, device=DEV)
    guard = torch.full((n + 2, k), 7.0, dtype=torch.bfloat16, device=DEV)
    out = ops.untile(ops.TiledWeight(w), guard[1:-1])
    assert torch.equal(out, w)
    assert bool((guard[0] == 7).all()) and bool((guard[-1] == 7).all())
    with pytest.raises(ops.KernelRefused):
        ops.untile(ops.TiledWeight(w), torch.empty(n, k + 8, dtype=torch.bfloat16, device=DEV))
    if k > 128:  # a range of columns, into rows that are further apart than they are long
        k0, k1 = 128, k if k < 384 else 384
        wide = torch.full((n, k1 - k0 + 16), 7.0, dtype=torch.bfloat16, device=DEV)
        ops.untile(ops.TiledWeight(w), wide[:, : k1 - k0], k0, k1)
        assert torch.equal(wide[:, : k1 - k0], w[:, k0:k1]) and bool((wide[:, k1 - k0 :] == 7).all())
        with pytest.raises(ops.KernelRefused):
            ops.untile(ops.TiledWeight(w), wide[:, : k1 - k0 - 8], k0 + 8, k1)


def _run_mfma(ops, q, k, v, table, starts, lens, heads, kvh, hd, window=0, force_splits=None, qt=2, coop=False, step_keys=0,
              chunk_splits=1, short_offsets=True, spare_tiles=0):
    n = sum(lens)
    indptr = [0]
    for l in lens:
        indptr.append(indptr[-1] + l)
    out = torch.zeros(n, heads * hd, dtype=torch.bfloat16, device=DEV)
    group = heads // kvh
    tile = lambda b, t0: [b, t0, indptr[b], lens[b], starts[b] + lens[b], 0, 0, 0]
    ct = [tile(b, t0) for b, l in enumerate(lens) if l != 1 for t0 in range(0, l, 16 * qt)]
    ct += [[len(lens) - 1, 0, 0, 0, 0, 0, 0, 0]] * (spare_tiles if ct else 0)  # tiles without tokens, as a captured step's spare ones
    dt = [tile(b, 0) for b, l in enumerate(lens) if l == 1]
    for t in dt:
        t[5] = step_keys  # the keys all decode rows of the step read: from some number on the kernel reads them past the cache
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    if ct:
        cols = len(ct) * 16 * qt * heads
        ws = None
        if chunk_splits > 1:  # filled with NaN: a range that is read without having been written shows
            ws = (torch.full((cols * chunk_splits * hd,), float("nan"), device=DEV), torch.full((cols * chunk_splits * 2,), float("nan"), device=DEV))
        ops.attention_mfma(q, out, k, v, i32(ct), table.to(DEV), heads, kvh, hd, 1 / math.sqrt(hd), window=window, hp=1,
                           splits=chunk_splits, workspace=ws, qt=qt, coop=coop and qt == 2,  # coop: one set of waves per workgroup
                           short_offsets=short_offsets)
    if dt:
        hp = 1
        while hp < min(group, 16):
            hp *= 2
        splits = force_splits or 3
        cols = len(dt) * (16 // hp) * heads
        # filled with NaN: a range (an empty one, say: with more than 16 the later ones are, below 8,192 keys) that is read
        # without having been written shows
        ws = (torch.full((cols * splits * hd,), float("nan"), device=DEV), torch.full((cols * splits * 2,), float("nan"), device=DEV))
        ops.attention_mfma(q, out, k, v, i32(dt), table.to(DEV), heads, kvh, hd, 1 / math.sqrt(hd), window=window, hp=hp,
                           splits=splits, workspace=ws if splits > 1 else None, coop=coop)
    return out


@pytest.mark.parametrize("case", list(CASES))
@pytest.mark.parametrize("heads,kvh,hd,page", [(8, 2, 128, 16), (6, 1, 48, 4), (4, 4, 16, 8), (32, 8, 64, 16), (40, 2, 32, 16)])
def test_attention_mfma(case, heads, kvh, hd, page):
    ops = _ops()
    starts, lens = CASES[case]
    torch.manual_seed(4)
    total = [s + l for s, l in zip(starts, lens)]
    pages = sum(-(-t // page) for t in total) + 3
    table = scattered_tables(total, page, pages, seed=1)
    k, v = make_cache(pages, page, kvh, hd, torch.bfloat16)
    kvs = fill_cache(k, v, table, total, page, kvh, hd, torch.bfloat16, seed=2)
    n = sum(lens)
    q = torch.randn(n, heads * hd, dtype=torch.bfloat16, device=DEV)
    ref = plain_paged_attention(q.view(n, heads, hd), kvs, starts, lens, heads).reshape(n, -1)
    # the last number: ranges that the keys of a prompt portion's tiles are cut into (16: more than most tiles have blocks)
    for splits, qt, coop, step_keys, chunk_splits in ((1, 2, False, 0, 1), (3, 1, False, 0, 2), (7, 2, True, 0, 3), (33, 1, False, 2**30, 1),
                                                      (1, 1, True, 2**30, 5), (2, 2, True, 0, 16), (1, 2, True, 0, 1)):
        out = _run_mfma(ops, q, k, v, table, starts, lens, heads, kvh, hd, force_splits=splits, qt=qt, coop=coop, step_keys=step_keys,
                        chunk_splits=chunk_splits)
        u = ulps_of_row_max(out.cpu(), ref).max()
        assert u <= 4, f"{case} splits={splits} qt={qt} coop={coop} chunk_splits={chunk_splits}: {u:.2f} ulps"


# The prompt kernel for head sizes 64 and 128 brings keys and values straight into LDS, a page id per page of a block of
# 32 keys: every page size it takes (four, two, one page a block, a block inside a page), a group of three heads (a wave
# of the workgroup has no head), a group of eight (two workgroups a key/value head), and addresses of 64 bits.
@pytest.mark.parametrize("case", ["prefill", "mixed", "long", "beyond64pages", "far"])
@pytest.mark.parametrize("heads,kvh,hd,page,short_offsets", [(8, 2, 128, 8, True), (8, 2, 128, 32, True), (16, 4, 64, 64, True), (4, 1, 64, 8, False),
                                                             (6, 2, 128, 16, True), (8, 1, 128, 16, False), (4, 2, 64, 128, False)])
def test_attention_mfma_prompt_kernel_page_sizes_and_groups(case, heads, kvh, hd, page, short_offsets):
    ops = _ops()
    starts, lens = CASES[case]
    torch.manual_seed(14)
    total = [s + l for s, l in zip(starts, lens)]
    pages = sum(-(-t // page) for t in total) + 3
    table = scattered_tables(total, page, pages, seed=3)
    k, v = make_cache(pages, page, kvh, hd, torch.bfloat16)
    kvs = fill_cache(k, v, table, total, page, kvh, hd, torch.bfloat16, seed=4)
    n = sum(lens)
    q = torch.randn(n, heads * hd, dtype=torch.bfloat16, device=DEV)
    ref = plain_paged_attention(q.view(n, heads, hd), kvs, starts, lens, heads).reshape(n, -1)
    for coop, chunk_splits in ((False, 1), (True, 1), (True, 3), (False, 16)):
        out = _run_mfma(ops, q, k, v, table, starts, lens, heads, kvh, hd, qt=2, coop=coop, chunk_splits=chunk_splits, short_offsets=short_offsets,
                        spare_tiles=3 if chunk_splits in (1, 3) else 0)
        u = ulps_of_row_max(out.cpu(), ref).max()
        assert u <= 4, f"{case} coop={coop} chunk_splits={chunk_splits}: {u:.2f} ulps"


def test_attention_prompt_kernel_in_use():
    """Head sizes 64 and 128 with pages of 8 tokens or more run the 32x32 prompt kernel (it steps aside if it was ever
    compiled with scratch memory: then this fails, and says that the tests above did not run it), the other sizes
    the kernels they are made for."""
    ops = _ops()
    for hd, page in ((64, 8), (64, 16), (64, 64), (64, 128), (128, 8), (128, 16), (128, 32)):
        assert ops.attention_prompt_form(hd, page) == 32, (hd, page)
    assert ops.attention_prompt_form(32, 16) == 16 and ops.attention_prompt_form(96, 16) == 16
    assert ops.attention_prompt_form(48, 4) == 0 and ops.attention_prompt_form(144, 16) == 0


@pytest.mark.parametrize("hd,page", [(128, 16), (64, 8), (128, 32)])
@pytest.mark.parametrize("coop", [False, True])
def test_attention_prompt_dominant_key_at_block_and_ring_edges(hd, page, coop):
    """A prompt portion of 70 tokens over some hundred keys; one key is made to dominate every query that sees it, so
    their outputs must be its value.  Done for keys around the edges of the kernel's blocks of 32 keys, of its ring of
    three buffers (96 keys), of the pages, of the halves that two sets of waves take, and inside the portion itself, where
    only later tokens see the key."""
    ops = _ops()
    heads, kvh = 8, 2
    n, total, dtype = 70, 430, torch.bfloat16
    start = total - n
    pages = -(-total // page) + 2
    table = scattered_tables([total], page, pages, seed=6)
    torch.manual_seed(9)
    base = torch.randn(heads * hd, dtype=dtype, device=DEV)
    q = base.repeat(n, 1).contiguous()  # every token asks the same
    for special in (0, 1, 31, 32, 33, 63, 64, 95, 96, 97, 127, 128, 191, 192, 193, 215, 216, 287, 288, 359, 360, 361, 383, 384, 400, 428, 429):
        k, v = make_cache(pages, page, kvh, hd, dtype)
        kvs = fill_cache(k, v, table, [total], page, kvh, hd, dtype, seed=special, scale=0.05)
        pg, off = int(table[0, special // page]), special % page
        for h in range(kvh):
            k[pg, h, off] = (base.view(heads, hd)[h * (heads // kvh)] * 4).to(dtype)  # aligned with the group's first query head
        kvs[0][0][special] = k[pg, :, off].cpu()
        out = _run_mfma(ops, q, k, v, table, [start], [n], heads, kvh, hd, qt=2, coop=coop).view(n, heads, hd).float().cpu()
        ref = plain_paged_attention(q.view(n, heads, hd), kvs, [start], [n], heads).reshape(n, -1)
        assert ulps_of_row_max(out.reshape(n, -1), ref).max() <= 4, f"key {special}"
        for h in range(kvh):
            want = kvs[0][1][special, h].float()
            for t in range(n):
                if start + t >= special:
                    assert torch.allclose(out[t, h * (heads // kvh)], want, atol=0.05), f"key {special}, token {t}: output is not its value"


@pytest.mark.parametrize("kernel", ["generic", "mfma"])
def test_attention_far_key_and_page_edges(kernel):
    """One key among hundreds is made to dominate: its score stands out, so the output must be its value.
    Done for a key at every offset around page edges, so that a wrong page or slot shows."""
    ops = _ops()
    heads, kvh, hd, page = 4, 2, 32, 8
    total, dtype = 333, torch.bfloat16
    pages = -(-total // page) + 2
    table = scattered_tables([total], page, pages, seed=5)
    for special in (0, 7, 8, 9, 15, 16, 255, 256, 320, 331, 332):
        k, v = make_cache(pages, page, kvh, hd, dtype)
        kvs = fill_cache(k, v, table, [total], page, kvh, hd, dtype, seed=special, scale=0.05)
        q = torch.randn(1, heads * hd, dtype=dtype, device=DEV)
        pg, off = int(table[0, special // page]), special % page
        for h in range(kvh):
            k[pg, h, off] = (q.view(heads, hd)[h * (heads // kvh)] * 4).to(dtype)  # aligned with the group's first query head
        starts, lens = [total - 1], [1]
        if kernel == "mfma":
            out = _run_mfma(ops, q, k, v, table, starts, lens, heads, kvh, hd)
        else:
            out = torch.empty_like(q)
            ops.attention_generic(q, out, k, v, torch.zeros(1, dtype=torch.int32, device=DEV),
                                  torch.tensor([total - 1], dtype=torch.int32, device=DEV), table.to(DEV), heads, kvh, hd, 1 / math.sqrt(hd))
        for h in range(kvh):
            got = out.view(heads, hd)[h * (heads // kvh)].float().cpu()
            want = kvs[0][1][special, h].float()
            assert torch.allclose(got, want, atol=0.05), f"key {special}: output is not its value"


@pytest.mark.parametrize("kernel", ["generic", "mfma"])
@pytest.mark.parametrize("window", [5, 16, 40])
@pytest.mark.parametrize("hd,page", [(32, 8), (128, 16), (64, 8)])  # (the prompt kernels: one for head sizes 64 and 128, one for the others)
def test_attention_window(kernel, window, hd, page):
    ops = _ops()
    heads, kvh = 4, 2
    starts, lens = [50, 0, 100], [1, 45, 20]
    dtype = torch.bfloat16
    total = [s + l for s, l in zip(starts, lens)]
    pages = sum(-(-t // page) for t in total) + 2
    table = scattered_tables(total, page, pages, seed=7)
    k, v = make_cache(pages, page, kvh, hd, dtype)
    kvs = fill_cache(k, v, table, total, page, kvh, hd, dtype, seed=8)
    # pages wholly before every query's window are released: the kernel must not touch them
    for b, (s, l) in enumerate(zip(starts, lens)):
        first_needed = max(0, s - window + 1) // page
        table[b, :first_needed] = -1
    n = sum(lens)
    q = torch.randn(n, heads * hd, dtype=dtype, device=DEV)
    ref = plain_paged_attention(q.view(n, heads, hd), kvs, starts, lens, heads, window=window).reshape(n, -1)
    if kernel == "mfma":
        out = _run_mfma(ops, q, k, v, table, starts, lens, heads, kvh, hd, window=window)
        cut = _run_mfma(ops, q, k, v, table, starts, lens, heads, kvh, hd, window=window, chunk_splits=3)
        assert ulps_of_row_max(cut.cpu(), ref).max() <= 4
        cut = _run_mfma(ops, q, k, v, table, starts, lens, heads, kvh, hd, window=window, chunk_splits=2, coop=True)
        assert ulps_of_row_max(cut.cpu(), ref).max() <= 4
    else:
        positions = torch.tensor([s + i for s, l in zip(starts, lens) for i in range(l)], dtype=torch.int32, device=DEV)
        token_req = torch.tensor([b for b, l in enumerate(lens) for _ in range(l)], dtype=torch.int32, device=DEV)
        out = torch.empty(n, heads * hd, dtype=dtype, device=DEV)
        ops.attention_generic(q, out, k, v, token_req, positions, table.to(DEV), heads, kvh, hd, 1 / math.sqrt(hd), window=window)
    assert ulps_of_row_max(out.cpu(), ref).max() <= 4


def test_sample_greedy_and_temperature():
    ops = _ops()
    torch.manual_seed(0)
    rows, vocab = 6, 1003
    z = torch.randn(rows, vocab, device=DEV) * 3
    z[2, 100] = z[2, 900] = z[2].max() + 1  # a tie: the lowest index wins
    T = torch.tensor([0.0, 0.8, 0.0, 1.0, 0.7, 1.3], device=DEV)
    u = torch.tensor([0.3, 0.9, 0.5, 0.0, 0.5, 0.9999], device=DEV)
    tok, lp, slp = ops.unpack_sample(ops.sample(z, T, u))
    zc = z.cpu()
    for r in range(rows):
        t = float(T[r])
        if t == 0:
            assert int(tok[r]) == int(zc[r].argmax()) or r == 2
            assert float(slp[r]) == 0.0
        else:
            ref = pl.draw_token(pl.processed_logprobs(zc[r], t, 0, 1.0), float(u[r]))
            assert abs(int(tok[r]) - ref) <= 1, (r, int(tok[r]), ref)  # the cumulative sums round differently
            assert abs(float(slp[r]) - float(pl.processed_logprobs(zc[r], t, 0, 1.0)[int(tok[r])])) < 1e-4
        assert abs(float(lp[r]) - float(torch.log_softmax(zc[r], -1)[int(tok[r])])) < 1e-4
    assert int(tok[2]) == 100


@pytest.mark.parametrize("vocab", [33, 257, 4100, 128256])
def test_sample_draws_at_other_vocabulary_sizes(vocab):
    """The inverse CDF is found in two cuts of the vocabulary and a walk: sizes below one cut, off every multiple, and
    the 8B shape's; uniform numbers at both ends; the draw must be the plain implementation's or its neighbour among the
    tokens that carry weight (the cumulative sums round differently)."""
    ops = _ops()
    torch.manual_seed(vocab)
    rows = 12
    z = torch.randn(rows, vocab, device=DEV) * 4
    z[3, : vocab // 2] = -math.inf  # weightless tokens are never drawn
    z[1, vocab - vocab // 3 :] = -math.inf  # ... nor when u * total rounds up to the total and the last token is taken
    T = torch.tensor([0.5, 0.8, 1.0, 1.0, 0.7, 1.3, 0.9, 1.1, 0.6, 1.0, 2.0, 0.0], device=DEV)
    u = torch.tensor([0.0, 0.9999999, 0.5, 0.001, 0.25, 0.75, 0.1, 0.9, 0.33, 0.66, 0.999, 0.5], device=DEV)
    tok, lp, slp = ops.unpack_sample(ops.sample(z, T, u))
    zc = z.cpu()
    for r in range(rows):
        t = float(T[r])
        if t == 0:
            assert int(tok[r]) == int(zc[r].argmax())
            continue
        ref_lp = pl.processed_logprobs(zc[r], t, 0, 1.0)
        ref = pl.draw_token(ref_lp, float(u[r]))
        got = int(tok[r])
        assert ref_lp[got] > -math.inf
        cdf = torch.cumsum(torch.exp(ref_lp.double()), 0)
        assert abs(float(cdf[got]) - float(cdf[ref])) < 1e-4, (r, got, ref)  # no more than rounding apart in the CDF
        assert abs(float(slp[r]) - float(ref_lp[got])) < 2e-4
        assert abs(float(lp[r]) - float(torch.log_softmax(zc[r], -1)[got])) < 2e-4


@pytest.mark.parametrize("vocab,spread", [(500, 2.0), (40000, 4.0), (40000, 0.05), (128256, 3.0)])
def test_sample_top_k_top_p(vocab, spread):
    """Small rows; rows whose kept tokens lie within a margin of the maximum (found among the tokens gathered in LDS);
    nearly flat rows, where more tokens lie within every margin than LDS holds or the cut lies below the margin."""
    ops = _ops()
    torch.manual_seed(1)
    z = torch.randn(4, vocab, device=DEV) * spread
    T = torch.tensor([0.7, 1.0, 1.0, 0.9], device=DEV)
    k = torch.tensor([5, 0, 3, 0], dtype=torch.int32, device=DEV)
    p = torch.tensor([1.0, 0.8, 0.5, 0.2], device=DEV)
    for uu in (0.01, 0.37, 0.62, 0.999):
        u = torch.full((4,), uu, device=DEV)
        tok, lp, slp = ops.unpack_sample(ops.sample(z, T, u, top_k=k, top_p=p))
        for r in range(4):
            ref_lp = pl.processed_logprobs(z[r].cpu(), float(T[r]), int(k[r]), float(p[r]))
            ref = pl.draw_token(ref_lp, uu)
            got = int(tok[r])
            if spread >= 1:
                assert ref_lp[got] > -math.inf, "a token outside the kept set was drawn"
                assert got == ref, (r, uu, got, ref)
                assert abs(float(slp[r]) - float(ref_lp[ref])) < 1e-4
            else:  # thousands of nearly equal tokens: the border of the kept set and the sums are a matter of rounding
                cdf = torch.cumsum(torch.exp(ref_lp.double()), 0)
                assert abs(float(cdf[got]) - float(cdf[ref])) < 2e-3, (r, uu, got, ref)
                assert abs(float(slp[r]) - float(ref_lp[ref])) < 1e-2


# ------------------------------------------------------------------------------------------------ the largest sizes


def _big(n, k, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(n, k, dtype=torch.float32, device=DEV, generator=g) * 0.05).to(torch.bfloat16)


@pytest.mark.parametrize("n,k", [(8192, 28672), (28672, 8192)])
def test_products_at_the_largest_feed_forward_sizes(n, k):
    """The hand-written products at an inner size and at an output width of 28,672 (the Llama-3.1-70B feed-forward): the
    streaming kernel at 1, 8 and 16 rows, the 17-to-128-row kernel at 64 and 128 rows with K in its planned ranges, the
    many-row kernel at 300 rows, the gated forms, and the product that ends in the residual stream and feeds the next
    norm; each against the 32-bit product of the same bfloat16 values."""
    ops = _ops()
    w, w2 = _big(n, k, 1), _big(n, k, 2)
    wt, wt2 = ops.TiledWeight(w), ops.TiledWeight(w2)
    wf, w2f = w.cpu().float(), w2.cpu().float()
    x_all = (torch.randn(300, k, dtype=torch.float32, device=DEV, generator=torch.Generator(device=DEV).manual_seed(3))).to(torch.bfloat16)
    ref_all = x_all.cpu().float() @ wf.T
    for m in (1, 8, 16):
        x, ref = x_all[:m], ref_all[:m]
        assert ulps_of_row_max(ops.linear_tiled(x, wt).cpu(), ref).max() <= 1.0, m
        u = x.cpu().float() @ w2f.T
        assert ulps_of_row_max(ops.linear_tiled(x, wt, w2=wt2).cpu(), ref * torch.sigmoid(ref) * u).max() <= 1.0, m
    for m in (64, 128):
        x, ref = x_all[:m], ref_all[:m]
        ksplit, nt = ops.wide_plan(n, k, m)
        out = ops.linear_wide(x, wt, ksplit=ksplit, nt=nt)
        assert ulps_of_row_max(out.cpu(), ref).max() <= 1.0, (m, ksplit, nt)
        part = ops.linear_wide(x, wt, ksplit=max(2, ksplit), nt=1, defer=True)
        assert ulps_of_row_max(ops.reduce_partial(part).cpu(), ref).max() <= 1.0, m
    u = x_all[:64].cpu().float() @ w2f.T
    act = ops.linear_wide(x_all[:64], wt, w2=wt2, ksplit=1, nt=1)
    assert ulps_of_row_max(act.cpu(), ref_all[:64] * torch.sigmoid(ref_all[:64]) * u).max() <= 1.0
    assert ulps_of_row_max(ops.linear_rows(x_all, wt).cpu(), ref_all).max() <= 1.0
    u = x_all.cpu().float() @ w2f.T
    assert ulps_of_row_max(ops.linear_rows(x_all, wt, w2=wt2, ksplit=1, nt=2).cpu(), ref_all * torch.sigmoid(ref_all) * u).max() <= 1.0
    # resid += x W^T with the next norm's inputs as by-products, 8 rows
    m = 8
    resid = (torch.randn(m, n, device=DEV) * 2).to(torch.bfloat16)
    w_next = (1 + 0.1 * torch.randn(n, device=DEV)).to(torch.bfloat16)
    before = resid.clone()
    pre = ops.linear_resid_norm(x_all[:m], wt, resid, w_next, 1e-5)
    want = (before.cpu().float() + ref_all[:m].to(torch.bfloat16).float()).to(torch.bfloat16)
    assert ulps_of_row_max(resid.cpu(), want.float()).max() <= 1.0
    torch.testing.assert_close(pre.ssq.sum(-1).cpu(), (resid.cpu().float() ** 2).sum(-1), rtol=1e-4, atol=0)
    assert torch.equal(pre.x.cpu(), (resid.cpu().float() * w_next.cpu().float()).to(torch.bfloat16))
    # a matrix copied back into plain rows, whole and in slices of its inner size
    plain = torch.empty_like(w)
    assert torch.equal(ops.untile(wt, plain), w)
    piece = torch.empty((n, 7168 if k > 8192 else 2048), dtype=torch.bfloat16, device=DEV)
    width = piece.shape[1]
    assert torch.equal(ops.untile(wt, piece, width, 2 * width), w[:, width : 2 * width])


F32_OPTIONS = {
    "plain": {},
    "window": dict(window=70),
    "chunk": dict(chunk=96),
    "cap_sink": dict(cap=2.0, sink=True),
    "slope_learned_sink": dict(slope_exp=8.0, sink_logits=True),
}


@pytest.mark.parametrize("option", list(F32_OPTIONS))
@pytest.mark.parametrize("case", ["append6", "mixed", "long", "beyond64pages"])
@pytest.mark.parametrize("heads,kvh,hd,page", [(8, 2, 128, 16), (6, 1, 48, 4), (3, 3, 16, 8), (32, 8, 64, 16), (40, 2, 32, 64)])
def test_attention_f32(case, option, heads, kvh, hd, page):
    """The 32-bit matrix-core kernels against the plain kernel: tiles and single tokens, whole and cut into ranges, every option, and
    pages that a window has let go.  Both sum 32-bit products in orders of their own: a few units in the last place of a row's scale."""
    ops = _ops()
    starts, lens = CASES[case]
    torch.manual_seed(11)
    total = [s + l for s, l in zip(starts, lens)]
    pages = sum(-(-t // page) for t in total) + 3
    table = scattered_tables(total, page, pages, seed=4)
    opt = dict(F32_OPTIONS[option])
    if opt.get("window"):
        for b, s in enumerate(starts):
            table[b, : max(0, s - opt["window"] + 1) // page] = -1
    k, v = make_cache(pages, page, kvh, hd, torch.float32)
    k.normal_(), v.normal_()
    if opt.get("sink_logits"):
        opt["sink_logits"] = torch.randn(heads, device=DEV)
    n = sum(lens)
    wide = torch.randn(n, heads * hd + 8, device=DEV)
    q = wide[:, : heads * hd]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    positions, token_req = i32([s + i for s, l in zip(starts, lens) for i in range(l)]), i32([b for b, l in enumerate(lens) for _ in range(l)])
    scale = 1 / math.sqrt(hd)
    want = torch.empty(n, heads * hd, device=DEV)
    ops.attention_generic(q, want, k, v, token_req, positions, table.to(DEV), heads, kvh, hd, scale, **opt)
    first = [sum(lens[:b]) for b in range(len(lens))]
    ct = [(b, t, first[b], l, total[b], 0, 0, 0) for b, l in enumerate(lens) if l > 1 for t in range(0, l, 32)] + [(0, 0, 0, 0, 0, 0, 0, 0)]
    dt = [(b, 0, first[b], 1, total[b], 0, 0, 0) for b, l in enumerate(lens) if l == 1] + [(0, 0, 0, 0, 0, 0, 0, 0)]
    longest = max(total)
    span = opt.get("window") or opt.get("chunk") or longest
    outs = []
    for splits, range_keys in ((1, -(-longest // 16) * 16), (3, 128), (16, 48)):
        out = torch.full((n, heads * hd), 7.0, device=DEV)
        for tiles, rows in ((ct, False), (dt, True)):
            s = -(-min(span, longest) // range_keys) + 1 if rows else splits
            cols = len(tiles) * (1 if rows else 32) * heads
            ws = tuple(torch.full((cols * s * m,), float("nan"), device=DEV) for m in (hd, 2)) if s > 1 else None
            if s <= ops.F32_ATTENTION_MAX_RANGES:
                ops.attention_f32(q, out, k, v, i32(tiles), table.to(DEV), heads, kvh, hd, scale, rows=rows, splits=s, range_keys=range_keys if rows else 0,
                                  workspace=ws, **opt)
        outs.append(out)
        # 1,300 weights of a row, each off by a few 2^-24 of its score's scale, and their sum
        torch.testing.assert_close(out, want, rtol=2e-5, atol=2e-5)
    rows = torch.tensor([i for b, l in enumerate(lens) if l > 1 for i in range(first[b], first[b] + l)], device=DEV)
    # a row by itself in its tile, beside what its tile holds here: the same sums
    b = next(b for b, l in enumerate(lens) if l > 1)
    last = [(b, lens[b] - 1, first[b], lens[b], total[b], 0, 0, 0)]
    alone = torch.full((n, heads * hd), 7.0, device=DEV)
    ops.attention_f32(q, alone, k, v, i32(last), table.to(DEV), heads, kvh, hd, scale, rows=False, **opt)
    assert torch.equal(alone[first[b] + lens[b] - 1], outs[0][first[b] + lens[b] - 1])
    assert rows.numel() and bool((alone[: first[b] + lens[b] - 1] == 7).all())


@pytest.mark.parametrize("window", [0, 300])
@pytest.mark.parametrize("heads,kvh,hd", [(8, 2, 64), (4, 4, 128)])
def test_attention_f32_does_not_depend_on_the_batch(heads, kvh, hd, window):
    """32-bit attention of a portion and of a single token, alone and beside others that change the launch (more tiles, longer rows, a
    table of many more keys): the same bits.  The last portion has so many keys that its ranges grow."""
    from types import SimpleNamespace

    import numpy as np

    from nanospec_amd.engine.context import BatchFacts
    from nanospec_amd.parts.attention import TilePlan, f32_attention

    torch.manual_seed(hd + window)
    page, kept = 16, {"portion": (3000, 40), "single": (700, 1), "long": (9900, 70), "far": (8600, 1)}
    q = {name: torch.randn(l, heads * hd, device=DEV) for name, (_, l) in kept.items()}
    pages = {name: -(-(s + l) // page) for name, (s, l) in kept.items()}
    k, v = torch.randn(1400, kvh, page, hd, device=DEV), torch.randn(1400, kvh, hd, page, device=DEV)
    first_page = dict(zip(kept, np.cumsum([0, *pages.values()])))

    def run(names, others, capacity=None):
        reqs = [(*kept[n], first_page[n], q[n]) for n in names] + [(s, l, 0, torch.randn(l, heads * hd, device=DEV)) for s, l in others]
        lens, starts = [r[1] for r in reqs], [r[0] for r in reqs]
        total = [s + l for s, l in zip(starts, lens)]
        i32 = lambda x: np.asarray(x, dtype=np.int32)
        plan, indptr = TilePlan(), np.concatenate(([0], np.cumsum(lens))).astype(np.int32)
        shape = plan.shape(lens)
        region = np.zeros(plan.ints(shape), dtype=np.int32)
        plan.fill(region, shape, BatchFacts(sum(lens), len(lens), i32(lens), i32(starts), indptr, i32(total), len(lens), 1))
        table = torch.zeros(len(reqs), -(-max(total) // page), dtype=torch.int32)
        for b, r in enumerate(reqs):
            m = -(-total[b] // page)
            table[b, :m] = torch.arange(r[2], r[2] + m) % 1400
        dev = torch.from_numpy(region).to(DEV)
        ctx = SimpleNamespace(plans={TilePlan.key: (dev, shape)}, arena=SimpleNamespace(take=lambda sh, dt: torch.full(sh, float("nan"), dtype=dt, device=DEV)),
                              token_ids=dev, max_kv_len=capacity or max(total), max_chunk_kv=capacity or max([t for t, l in zip(total, lens) if l > 1], default=0))
        x = torch.cat([r[3] for r in reqs])
        out = f32_attention(ctx, x, torch.empty_like(x), SimpleNamespace(k=k, v=v), table.to(DEV), heads, kvh, hd, hd ** -0.5, window=window)
        assert torch.isfinite(out).all()
        return {n: out[indptr[i] : indptr[i + 1]] for i, n in enumerate(names)}

    alone = {n: run([n], [])[n] for n in kept}
    for others, capacity in (([], None), ([(0, 900)], None), ([(20, 1), (12000, 1)], None), ([(5000, 33), (0, 2000), (300, 1)], None), ([(7, 3)], 32768)):
        got = run(list(kept), others, capacity)
        for n in kept:
            assert torch.equal(got[n], alone[n]), (n, others, capacity)


def test_attention_f32_keeps_infinities_to_the_rows_that_see_them():
    """A value that is infinite or no number belongs to the tokens at its position and behind; the others' results are what they
    would be without it.  The same for keys, and for what earlier owners left in a page behind the last key."""
    ops = _ops()
    torch.manual_seed(5)
    heads, kvh, hd, page, n = 4, 2, 32, 16, 50
    table = torch.arange(4, dtype=torch.int32, device=DEV).view(1, 4)
    q = torch.randn(n, heads * hd, device=DEV)
    tiles = torch.tensor([(0, t, 0, n, n, 0, 0, 0) for t in range(0, n, 32)], dtype=torch.int32, device=DEV)
    k, v = (torch.randn(4, kvh, page, hd, device=DEV), torch.randn(4, kvh, hd, page, device=DEV))
    k[3, :, 2:], v[3, :, :, 2:] = float("nan"), float("nan")  # positions 50 to 63 are nobody's
    run = lambda: ops.attention_f32(q, torch.zeros(n, heads * hd, device=DEV), k, v, tiles, table, heads, kvh, hd, 0.2, rows=False)
    clean = run()
    assert torch.isfinite(clean).all()
    for bad in (float("inf"), float("nan")):
        for what, cache in (("v", v[2, :, 3, 5]), ("k", k[2, :, 5, 3])):  # position 37
            kept = cache.clone()
            cache.fill_(bad)
            out = run()
            cache.copy_(kept)
            torch.testing.assert_close(out[:37], clean[:37], rtol=1e-5, atol=1e-6)
            if what == "v" or bad != bad:  # (an infinite key may make a score of minus infinity: a weight of zero)
                assert not torch.isfinite(out[37:]).all(dim=1).any()
    one = torch.tensor([(0, 0, 0, 1, n, 0, 0, 0)], dtype=torch.int32, device=DEV)
    out = ops.attention_f32(q[:1], torch.zeros(1, heads * hd, device=DEV), k, v, one, table, heads, kvh, hd, 0.2, rows=True, range_keys=64)
    assert torch.isfinite(out).all()


@pytest.mark.parametrize("routing", ["spread", "one expert", "identity"])
@pytest.mark.parametrize("n,experts,top,width,ff,gated", [(8, 8, 4, 64, 24, True), (16, 32, 4, 136, 40, False), (33, 32, 4, 72, 136, True), (40, 5, 2, 264, 16, True),
                                                          (130, 3, 1, 64, 264, False), (517, 70, 3, 128, 72, True), (64, 256, 8, 64, 16, True), (65, 256, 8, 64, 16, True),
                                                          (80, 256, 8, 64, 136, False), (80, 256, 8, 64, 16, False), (400, 6, 2, 136, 136, True),
                                                          (450, 3, 1, 72, 264, False), (150, 4, 2, 520, 264, True), (400, 6, 2, 328, 264, True),
                                                          (400, 3, 2, 1320, 648, True), (450, 3, 1, 648, 1320, False), (300, 7, 2, 712, 328, True),
                                                          (300, 7, 2, 328, 712, False)])
def test_moe_expert_groups(routing, n, experts, top, width, ff, gated):
    """The sorted experts' products, streamed and tiled: tiles of 1 to 16 and to 128 rows in both forms, experts with more rows than a tile and with
    none, several tiles of an expert over more blocks of channels than they take together, pairs without an expert, sizes that end inside
    a tile and inside a piece of K, before and after a place in LDS is used again."""
    ops = _ops()
    g = torch.Generator().manual_seed(n + experts)
    rnd = lambda *shape: torch.randn(*shape, generator=g)
    h = rnd(n, width).bfloat16()
    gate, up, down = ((rnd(experts, *s) * s[1] ** -0.5).bfloat16() for s in ((ff, width), (ff, width), (width, ff)))
    sel = torch.stack([torch.randperm(experts + 1, generator=g)[:top] for _ in range(n)]).to(torch.int32)
    if routing == "one expert":
        sel[:, 0] = experts - 1
    if routing != "identity":
        sel = sel % experts  # (the same expert twice in a token is two pairs)
    wt = torch.rand(n, top, generator=g)
    take = lambda shape, dtype: torch.full(shape, 7, dtype=dtype, device=DEV) if dtype == torch.int32 else torch.full(shape, float("nan"), dtype=dtype, device=DEV)
    dev = lambda t: t.to(DEV) if t is not None else None
    out = ops.moe_experts(dev(h), dev(gate) if gated else None, dev(up), dev(down), dev(sel), dev(wt), 7.0 if gated else 0.0, 1.702 if gated else 0.0, take,
                          1.0 if gated else 0.0, *(() if gated else ("relu2",))).cpu()
    for t in range(n):
        for k in range(top):
            e = int(sel[t, k])
            if e >= experts:
                continue
            x = h[t].double()
            u = (up[e].double() @ x).float().bfloat16().double()
            if gated:
                a = (gate[e].double() @ x).float().bfloat16().double().clamp(max=7.0)
                act = a * torch.sigmoid(1.702 * a) * (u.clamp(-7.0, 7.0) + 1.0)
            else:
                act = u.clamp(min=0.0) ** 2
            act = act.float().bfloat16().double()
            want = float(wt[t, k]) * (down[e].double() @ act)
            # an inner channel's sum may round to the next bfloat16 (2^-8 of it at most), and so may the activation made of it
            bound = float(wt[t, k]) * 2.0 ** -6 * (down[e].double().abs() @ act.abs()) + 1e-5
            assert ((out[t, k].double() - want).abs() <= bound).all(), (t, k, e)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,rows,width", [(9, 31, 16), (16, 32, 48), (17, 33, 80), (33, 65, 2048), (40, 7, 20)])
def test_moe_router_of_many_tokens(n, rows, width, dtype):
    """Logits where a tile of 16 tokens or of 32 rows ends, pieces of K that four waves cannot share evenly, a width of no whole pieces."""
    ops = _ops()
    g = torch.Generator().manual_seed(n)
    h, router, bias = (torch.randn(*s, generator=g) for s in ((n, width + 4), (rows, width), (rows,)))
    h = h.to(dtype)[:, :width]
    z, sel, wt = torch.full((n, rows), float("nan"), device=DEV), torch.zeros(n, 2, dtype=torch.int32, device=DEV), torch.zeros(n, 2, device=DEV)
    wide = torch.zeros(n, width + 4, dtype=dtype, device=DEV)
    wide[:, :width] = h.to(DEV)
    ops.moe_route(wide[:, :width], router.to(DEV), bias.to(DEV), 2, sel, wt, logits=z)
    want = h.double() @ router.double().T + bias.double()
    # a 32-bit sum of `width` products and a bias: at most width + 1 roundings of 2^-24 of the sum of the magnitudes
    bound = (width + 1) * 2.0 ** -24 * (h.double().abs() @ router.double().abs().T + bias.double().abs())
    assert ((z.cpu().double() - want).abs() <= bound).all()
    assert torch.equal(sel.cpu().long(), z.cpu().topk(2).indices)


@pytest.mark.parametrize("rows", [1, 16, 17, 33, 64])
def test_moe_router_by_one_or_two_sets_of_rows(rows):
    """A workgroup takes 16 rows of the router while the units have one workgroup each and 32 beyond: a token's logits are the same bits either way."""
    ops = _ops()
    torch.manual_seed(rows)
    h, router = torch.randn(4100, 96, device=DEV).bfloat16(), torch.randn(rows, 96, device=DEV)
    def logits(n):
        z, sel, wt = torch.full((n, rows), 7.0, device=DEV), torch.empty((n, 1), dtype=torch.int32, device=DEV), torch.empty((n, 1), device=DEV)
        ops.moe_route(h[:n], router, None, 1, sel, wt, logits=z)
        return z
    many = logits(4100)  # 257 workgroups and more
    for n in (17, 800, 4096):
        assert torch.equal(logits(n), many[:n]), n
    ref = h.cpu().double() @ router.cpu().double().T
    assert float((many.cpu().double() - ref).norm() / ref.norm()) <= 2.0**-22


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,rows,width", [(64, 33, 2048), (300, 16, 4096), (40, 64, 512), (500, 64, 64)])
def test_moe_router_of_many_tokens_is_as_exact_as_the_plain_kernel(n, rows, width, dtype):
    """The logits decide which experts run: on the matrix instruction they are no further from 64 bits (2-norm over thousands of
    logits) than the plain kernel's, which takes the same rows where they lie off their 16-byte places."""
    ops = _ops()
    g = torch.Generator().manual_seed(width)
    h, router = torch.randn(n, width, generator=g).to(dtype), torch.randn(rows, width, generator=g) * 0.02
    want = h.double() @ router.double().T
    err = []
    for off in (0, 1):
        wide = torch.zeros(n, width + 4, dtype=dtype, device=DEV)
        wide[:, off : off + width] = h.to(DEV)
        z, sel, wt = torch.full((n, rows), float("nan"), device=DEV), torch.zeros(n, 2, dtype=torch.int32, device=DEV), torch.zeros(n, 2, device=DEV)
        ops.moe_route(wide[:, off : off + width], router.to(DEV), None, 2, sel, wt, logits=z)
        err.append(float((z.cpu().double() - want).norm() / want.norm()))
    assert err[0] <= err[1], err


@pytest.mark.parametrize("experts,groups,keep,best", [(1, 1, 1, 1), (31, 1, 1, 2), (63, 9, 4, 2), (64, 1, 1, 1), (64, 32, 7, 2), (64, 64, 9, 2), (64, 8, 1, 2), (65, 13, 3, 1), (130, 5, 2, 2)])
@pytest.mark.parametrize("n", [1, 6, 4099])
def test_moe_choice_among_a_wave_of_experts_and_more(experts, groups, keep, best, n):
    """The choice by lanes (up to 64 experts, where that is the faster one) and by turns: many equal scores, scores that are no numbers, the smallest and largest groups."""
    ops = _ops()
    g = torch.Generator().manual_seed(experts + groups + n)
    # a router of unit vectors: the logits are the input's columns, whole numbers (no two different pairs of their scores add up alike)
    h = torch.randint(0, 4, (n, experts), generator=g).float()
    per = experts // groups
    top = min(4, keep * per)
    corr = torch.zeros(experts)
    corr[experts // 2] = float("nan")  # counts as the lowest score
    sel, wt = torch.zeros(n, top, dtype=torch.int32, device=DEV), torch.zeros(n, top, device=DEV)
    ops.moe_route(h.to(DEV), torch.eye(experts, device=DEV), None, top, sel, wt, score="sigmoid", correction=corr.to(DEV), groups=groups, keep=keep,
                  group_best=best)
    s = torch.sigmoid(h)
    by = (s + corr).nan_to_num(nan=float("-inf"))
    for t in range(n) if n < 100 else (0, 1, n - 2, n - 1):
        row = by[t].tolist()
        tops = [sorted(row[i * per : (i + 1) * per], reverse=True)[: min(best, per)] for i in range(groups)]
        order = sorted(range(groups), key=lambda i: (-sum(tops[i]), i))[:keep]
        want = sorted((e for e in range(experts) if e // per in order), key=lambda e: (-row[e], e))[:top]
        assert sel[t].tolist() == want
        torch.testing.assert_close(wt[t].cpu(), s[t, want], rtol=1e-6, atol=0)


@pytest.mark.parametrize("n,experts,ff", [(24, 8, 264), (200, 8, 264), (700, 4, 136), (700, 4, 384)])
def test_moe_results_at_any_address(n, experts, ff):
    """A result that begins a float behind a 16-byte boundary: streamed, in the smaller tiles (700 rows of 136 channels, no whole stages, among them) and in the larger ones."""
    ops = _ops()
    g = torch.Generator(device=DEV).manual_seed(n)
    rnd = lambda *shape: torch.randn(*shape, generator=g, device=DEV).bfloat16()
    width, top = 136, 1
    h, gate, up, down = rnd(n, width), rnd(experts, ff, width), rnd(experts, ff, width), rnd(experts, width, ff)
    sel, wt = torch.randint(0, experts, (n, top), generator=g, device=DEV, dtype=torch.int32), torch.rand(n, top, generator=g, device=DEV)
    got = []
    for first in (0, 1):
        out = torch.full((first + n * top * width + 3,), 7.0, device=DEV)
        ints, act = torch.zeros(8 * (n + experts), dtype=torch.int32, device=DEV), torch.zeros(n * top, ff, dtype=torch.bfloat16, device=DEV)
        ops.moe_expert_groups(h, gate, up, down, sel, wt, 7.0, 1.702, ints, act, out[first : first + n * top * width].view(n, top, width))
        assert bool((out[:first] == 7).all()) and bool((out[first + n * top * width :] == 7).all())
        got.append(out[first : first + n * top * width])
    assert torch.equal(*got)


def test_moe_tiles_of_more_blocks_than_a_row_of_the_launch():
    """One expert of more channels than 8 x 65,536 workgroups of 64 take: the launch's second dimension."""
    ops = _ops()
    ff, width, n = (1 << 25) + 4104, 8, 3
    g = torch.Generator(device=DEV).manual_seed(5)
    rnd = lambda *shape: torch.randint(-2, 3, shape, generator=g, device=DEV, dtype=torch.int8).bfloat16()
    h, gate, up, down = rnd(n, width), rnd(1, ff, width), rnd(1, ff, width), torch.zeros(1, width, ff, dtype=torch.bfloat16, device=DEV)
    sel, wt = torch.zeros(n, 1, dtype=torch.int32, device=DEV), torch.ones(n, 1, device=DEV)
    act = torch.full((n, ff), float("nan"), dtype=torch.bfloat16, device=DEV)
    ints, out = torch.zeros(64, dtype=torch.int32, device=DEV), torch.full((n, 1, width), float("nan"), device=DEV)
    ops.moe_expert_groups(h, gate, up, down, sel, wt, float("inf"), 1.0, ints, act, out, shift=0.0)
    assert bool((out == 0).all())
    perm = ints[:n].long()  # (the places that the pairs got)
    for i in range(n):
        x = h[perm[i]].float()
        for at in range(0, ff, 1 << 20):
            a, b = gate[0, at : at + (1 << 20)].float() @ x, up[0, at : at + (1 << 20)].float() @ x  # whole numbers, exact
            torch.testing.assert_close(act[i, at : at + (1 << 20)].float(), a * torch.sigmoid(a) * b, rtol=2.0 ** -7, atol=1e-6)  # (one rounding to bfloat16)


@pytest.mark.parametrize("score", ["softmax", "sigmoid", "softmax_all"])
@pytest.mark.parametrize("infinite", ["lowest", "both"])
@pytest.mark.parametrize("experts,groups,keep,best,top", [(8, 1, 1, 1, 3), (8, 4, 2, 2, 3), (64, 32, 7, 2, 8), (64, 8, 1, 2, 2), (64, 1, 1, 2, 12), (64, 1, 1, 1, 1), (66, 1, 1, 1, 4), (130, 65, 9, 2, 8), (130, 5, 2, 2, 6)])
def test_moe_choice_among_scores_that_are_not_finite(score, infinite, experts, groups, keep, best, top):
    """Both forms of the choice, every score: infinite logits, corrections that are infinite or no number, groups whose two best add up to no number
    (they count as the lowest, like experts' scores that are none)."""
    ops = _ops()
    g = torch.Generator().manual_seed(experts + groups)
    n, per, inf = 6, experts // groups, float("inf")
    h = torch.randint(0, 4, (n, experts), generator=g).float()  # the logits: the router is of unit vectors
    bias, corr = torch.zeros(experts), torch.zeros(experts)
    bias[1::5] = -inf
    if infinite == "both" and score != "softmax_all":  # (an infinite logit leaves no number among a soft-max's scores)
        bias[2::7] = inf
    corr[experts // 2] = float("nan")
    if infinite == "both":
        corr[0], corr[1], corr[experts - 1] = inf, -inf, -inf
    corr = None if score == "softmax" else corr
    sel, wt = torch.zeros(n, top, dtype=torch.int32, device=DEV), torch.zeros(n, top, device=DEV)
    ops.moe_route(h.to(DEV), torch.eye(experts, device=DEV), bias.to(DEV), top, sel, wt, score=score, correction=None if corr is None else corr.to(DEV),
                  groups=groups, keep=keep, group_best=best)
    lowest = lambda v: v if v == v else -inf
    for t in range(n):
        z = h[t] + bias
        w = {"softmax": z, "sigmoid": torch.sigmoid(z), "softmax_all": torch.softmax(z, 0)}[score]
        row = [lowest(v) for v in (w if corr is None else w + corr).tolist()]
        tops = [sorted(row[i * per : (i + 1) * per], reverse=True)[: min(best, per)] for i in range(groups)]
        order = sorted(range(groups), key=lambda i: (-lowest(sum(tops[i])), i))[:keep]
        want = sorted((e for e in range(experts) if e // per in order), key=lambda e: (-row[e], e))[:top]
        assert sel[t].tolist() == want
        chosen = torch.softmax(z[want], 0) if score == "softmax" else w[want] / (w[want].sum() if score == "softmax_all" else 1.0)
        torch.testing.assert_close(wt[t].cpu(), chosen, rtol=1e-5, atol=0, equal_nan=True)  # (exponentials of 32 bits and a sum of up to 12)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,top,width", [(1, 1, 4), (3, 4, 1020), (5, 2, 1028), (2, 3, 2050)])
def test_moe_combine(n, top, width, dtype):
    """The experts' parts added up: rows that end inside a workgroup's 1,024 columns, the input in a part's place, a gated base or none."""
    ops = _ops()
    g = torch.Generator().manual_seed(width)
    parts, base, gate, h, wt = (torch.randn(*s, generator=g) for s in ((n, top, width), (n, width), (n, 3), (n, width), (n, top)))
    base, h = base.to(dtype), h.to(dtype)
    sel = torch.randint(0, 6, (n, top), generator=g, dtype=torch.int32)
    d = lambda t: t.to(DEV)
    for with_base, with_gate, identity in ((True, False, False), (True, True, True), (False, False, True)):
        out = torch.full((n, width), float("nan"), dtype=dtype, device=DEV)
        ops.moe_combine(d(parts), d(base) if with_base else None, out, d(gate)[:, 1] if with_gate else None, (d(sel), d(wt), d(h), 4) if identity else None)
        terms = parts.double()
        if identity:
            terms = torch.where((sel >= 4)[:, :, None], wt.double()[:, :, None] * h.double()[:, None], terms)
        if with_base:
            b = base.double() * (torch.sigmoid(gate[:, 1:2].double()) if with_gate else 1.0)
            terms = torch.cat([terms, b[:, None]], 1)
        # a rounding of 2^-24 of the magnitudes for every term and a few for the sigmoid, then one to the output's type
        bound = terms.abs().sum(1) * ((top + 6) * 2.0 ** -24 + (2.0 ** -8 if dtype == torch.bfloat16 else 0.0))
        assert ((out.cpu().double() - terms.sum(1)).abs() <= bound).all(), (with_base, with_gate, identity)


@pytest.mark.parametrize("scratch", [0, 64 << 20], ids=["piecewise", "whole"])
@pytest.mark.parametrize("H,G,D,E,lens", [(2, 1, 64, 16, [32]), (2, 2, 128, 48, [33, 1, 0, 47, 31, 100]), (8, 4, 64, 32, [5, 64, 49]), (3, 3, 128, 16, [1, 257])])
def test_delta_rule_by_chunks(monkeypatch, H, G, D, E, lens, scratch):
    """Prompt portions sixteen tokens at a time against the recurrence in 64 bits: last chunks of one and of fifteen tokens, requests that
    are too short for it among them, decays of zero and of one, the records of all chunks at once and of one at a time."""
    ops = _ops()
    monkeypatch.setattr(ops, "DELTA_CHUNK_SCRATCH", scratch)
    monkeypatch.setattr(ops, "DELTA_CHUNK_MIN", 32)
    gen = torch.Generator().manual_seed(D + len(lens))
    n, B, C = sum(lens), len(lens), 2 * G * D + H * E
    rnd = lambda *shape: torch.randn(*shape, generator=gen)
    unit = lambda t: t / t.norm(dim=-1, keepdim=True)
    q, k, v = unit(rnd(n, G, D)) * D ** -0.5, unit(rnd(n, G, D)), rnd(n, H, E)
    g, beta, S0 = torch.rand(n, H, D, generator=gen) ** 0.2, torch.rand(n, H, generator=gen), rnd(B + 1, H * D * E) * 0.2
    g[:, :, 0], g[:, :, 1], g[7::16, :, 2] = 0.0, 1.0, 0.0
    state = S0.clone().to(DEV)
    slots = torch.arange(B, 0, -1, dtype=torch.int32)
    indptr = torch.tensor([0, *lens]).cumsum(0).to(torch.int32)
    qkv = torch.cat([q.flatten(1), k.flatten(1), v.flatten(1)], 1).to(DEV)
    out = torch.full((n, H * E), float("nan"), device=DEV)
    take = lambda shape, dtype: torch.full(shape, float("nan"), dtype=dtype, device=DEV)
    ops.delta_scan(qkv, g.flatten(1).to(DEV).contiguous(), beta.to(DEV), state, indptr.to(DEV), slots.to(DEV), H, G, D, E, out=out, take=take)
    wide = lambda t: t.double().repeat_interleave(H // G, 0)
    got, after = out.cpu().double().view(n, H, E), state.cpu().double()
    for b in range(B):
        S, top = S0[slots[b]].double().view(H, D, E), 1.0
        for t in range(int(indptr[b]), int(indptr[b + 1])):
            S = S * g[t].double()[:, :, None]
            u = beta[t].double()[:, None] * (v[t].double() - (wide(k[t])[:, :, None] * S).sum(1))
            S = S + wide(k[t])[:, :, None] * u[:, None]
            top = max(top, float(S.norm(dim=1).max()), float(v[t].norm(dim=1).max()))
            want = (wide(q[t])[:, :, None] * S).sum(1)
            # a step rounds sums of D + 16 terms and hands its error on undamped at most: 2^-24 of the largest column a term and a step
            steps = t - int(indptr[b]) + 1
            assert ((got[t] - want).abs().max() <= (D + 16 + steps) * 2.0 ** -24 * top * D ** -0.5 * 4), (b, t)
        torch.testing.assert_close(after[slots[b]], S.flatten(), rtol=0, atol=(D + 16 + lens[b]) * 2.0 ** -24 * top)
    assert torch.equal(after[0], S0[0].double())


def test_delta_rule_by_chunks_keeps_infinities_to_later_tokens(monkeypatch):
    """An infinity or NaN at one token, in any of its inputs or in all of them, reaches neither the tokens before it nor other requests, as
    token by token."""
    ops = _ops()
    monkeypatch.setattr(ops, "DELTA_CHUNK_MIN", 32)
    gen = torch.Generator().manual_seed(3)
    D, E, n, C = 64, 16, 80, 2 * 64 + 16
    qkv, g, beta = torch.randn(n, C, generator=gen) * 0.1, torch.rand(n, D, generator=gen) ** 0.2, torch.rand(n, 1, generator=gen)
    indptr, slots = torch.tensor([0, 40, 80], dtype=torch.int32, device=DEV), torch.tensor([0, 1], dtype=torch.int32, device=DEV)
    take = lambda shape, dtype: torch.empty(shape, dtype=dtype, device=DEV)

    def run(x, gg, bb=beta):
        out = torch.empty(n, E, device=DEV)
        return ops.delta_scan(x.to(DEV), gg.to(DEV), bb.to(DEV), torch.zeros(2, D * E, device=DEV), indptr, slots, 1, 1, D, E, out=out, take=take).cpu()

    clean = run(qkv, g)
    assert torch.isfinite(clean).all()
    for bad in (float("inf"), float("nan")):
        for column in (3, D + 3, 2 * D + 3):  # of q, k and v
            x = qkv.clone()
            x[21, column] = bad
            out = run(x, g)
            others = torch.arange(n) != 21 if column < D else (torch.arange(n) < 21) | (torch.arange(n) >= 40)
            torch.testing.assert_close(out[others], clean[others], rtol=1e-5, atol=1e-6)
            assert not torch.isfinite(out[21]).all()
        others = (torch.arange(n) < 21) | (torch.arange(n) >= 40)
        for what in ("beta", "g", "all"):  # (a token whose row of the stream is not finite has no number anywhere)
            x, gg, bb = qkv.clone(), g.clone(), beta.clone()
            if what in ("beta", "all"):
                bb[21] = bad
            if what in ("g", "all"):
                gg[21, 3 if what == "g" else slice(None)] = bad
            if what == "all":
                x[21] = bad
            out = run(x, gg, bb)
            torch.testing.assert_close(out[others], clean[others], rtol=1e-5, atol=1e-6)
            assert not torch.isfinite(out[21]).all()


@pytest.mark.parametrize("D,lens,longest,chunks", [(64, [63, 63], 63, False), (64, [63, 64], 64, True), (128, [40, 40], 40, False), (64, [64] * 128, 64, False),
                                                  (128, [64] * 16, 64, True), (64, [40, 90], None, True)])
def test_recurrences_by_chunks_where_a_request_is_long_enough(D, lens, longest, chunks):
    """Chunks are launched where a request has the tokens that they are worth, told by the step's longest request; many requests with
    small heads stay token by token."""
    ops = _ops()
    gen = torch.Generator().manual_seed(D)
    H, E, n, B = 2, 16, sum(lens), len(lens)
    indptr, slots = torch.tensor([0, *lens]).cumsum(0).to(torch.int32).to(DEV), torch.arange(B, dtype=torch.int32, device=DEV)
    taken = []

    def take(shape, dtype):
        taken.append(shape)
        return torch.empty(shape, dtype=dtype, device=DEV)

    def scans(**kw):
        qkv, g, beta = torch.randn(n, 2 * H * D + H * E, generator=gen) * 0.1, torch.rand(n, H * D, generator=gen), torch.rand(n, H, generator=gen)
        ops.delta_scan(qkv.to(DEV), g.to(DEV), beta.to(DEV), torch.zeros(B, H * D * E, device=DEV), indptr, slots, H, H, D, E,
                       out=torch.empty(n, H * E, device=DEV), take=take, **kw)
        yield bool(taken)
        taken.clear()
        at = (0, H * D, 2 * H * D, 2 * H * D + H * E, 2 * H * D + H * E + H)
        proj = torch.randn(n, -(-(at[4] + H) // 8) * 8, generator=gen).to(DEV)
        ops.memory_scan(proj, at, None, None, torch.zeros(B, ops.memory_state_floats(H, D, E), device=DEV), indptr, slots, H, D, E, 15.0, D ** -0.5,
                        torch.empty(n, H * E, device=DEV), torch.empty(n, H, device=DEV), take=take, **kw)
        yield bool(taken)

    delta, memory = scans(longest=longest, portions=None if longest is None else B)
    assert delta == chunks and memory == (chunks or B == 128)  # (the memory's chunks are ahead at 128 requests of two heads)


def test_matrix_memory_by_chunks_keeps_infinities_to_later_tokens(monkeypatch):
    """An infinity or NaN at one token, in any of its inputs, reaches neither the tokens before it nor other requests."""
    ops = _ops()
    monkeypatch.setattr(ops, "MEMORY_CHUNK_MIN", 48)
    gen = torch.Generator().manual_seed(4)
    D, E, n = 64, 16, 120
    proj = torch.randn(n, 152, generator=gen)
    at = (0, D, 2 * D, 2 * D + E, 2 * D + E + 1)
    indptr, slots = torch.tensor([0, 60, 120], dtype=torch.int32, device=DEV), torch.tensor([0, 1], dtype=torch.int32, device=DEV)
    take = lambda shape, dtype: torch.empty(shape, dtype=dtype, device=DEV)

    def run(x):
        out, den = torch.empty(n, E, device=DEV), torch.empty(n, 1, device=DEV)
        state = torch.zeros(2, ops.memory_state_floats(1, D, E), device=DEV)
        ops.memory_scan(x.to(DEV), at, None, None, state, indptr, slots, 1, D, E, 15.0, D ** -0.5, out, den, take=take)
        return torch.cat([out, den], 1).cpu()

    clean = run(proj)
    assert torch.isfinite(clean).all()
    for bad in (float("inf"), float("nan")):
        for column in (3, at[1] + 3, at[2] + 3) + ((at[3], at[4]) if bad != bad else ()):  # (the gates' logs are capped: an infinity is the cap)
            x = proj.clone()
            x[21, column] = bad
            out = run(x)
            others = torch.arange(n) != 21 if column < D else (torch.arange(n) < 21) | (torch.arange(n) >= 60)
            torch.testing.assert_close(out[others], clean[others], rtol=1e-5, atol=1e-6)
            assert not torch.isfinite(out[21]).all()


@pytest.mark.parametrize("scratch", [0, 64 << 20], ids=["piecewise", "whole"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,D,E,lens", [(2, 64, 16, [48]), (1, 128, 48, [49, 1, 0, 63, 47, 130]), (3, 128, 32, [5, 1100])])
def test_matrix_memory_by_chunks(monkeypatch, H, D, E, lens, dtype, scratch):
    """Prompt portions sixteen tokens at a time against the recurrence in 64 bits: last chunks of one and of fifteen tokens, requests that are
    too short for it among them, more tokens than the gates' kernel takes at once, the records of all chunks at once and of one at a time."""
    ops = _ops()
    monkeypatch.setattr(ops, "MEMORY_CHUNK_SCRATCH", scratch)
    monkeypatch.setattr(ops, "MEMORY_CHUNK_MIN", 48)
    gen = torch.Generator().manual_seed(D + len(lens))
    n, B = sum(lens), len(lens)
    at = (0, H * D, 2 * H * D, 2 * H * D + H * E, 2 * H * D + H * E + H)
    proj = torch.randn(n, -(-(at[4] + H) // 8) * 8, generator=gen).to(dtype)
    bias_i, bias_f = torch.randn(H, generator=gen), torch.randn(H, generator=gen) * 3
    words = ops.memory_state_floats(H, D, E)
    S0 = torch.zeros(B + 1, words)
    S0[:, : H * E * D] = torch.randn(B + 1, H * E * D, generator=gen) * 0.2
    state, slots = S0.clone().to(DEV), torch.arange(B, 0, -1, dtype=torch.int32)
    indptr = torch.tensor([0, *lens]).cumsum(0).to(torch.int32)
    out, den = torch.full((n, H * E), float("nan"), device=DEV), torch.full((n, H), float("nan"), device=DEV)
    take = lambda shape, dt: torch.full(shape, float("nan"), dtype=dt, device=DEV)
    run = lambda a, b, st, **kw: ops.memory_scan(proj[a:b].to(DEV), at, bias_i.to(DEV), bias_f.to(DEV), st, *kw.pop("who"), H, D, E, 15.0, D ** -0.5, out[a:b],
                                                 den[a:b], **kw)
    run(0, n, state, who=(indptr.to(DEV), slots.to(DEV)), take=take)
    got, gden = out.cpu().double().view(n, H, E), den.cpu().double()
    x = proj.double()
    gi = 15 * torch.tanh((x[:, at[3] : at[3] + H] + bias_i.double()) / 15)
    gf = torch.nn.functional.logsigmoid(15 * torch.tanh((x[:, at[4] : at[4] + H] + bias_f.double()) / 15))
    for b in range(B):
        S, N, m = S0[slots[b], : H * E * D].double().view(H, E, D), torch.zeros(H, D).double(), torch.zeros(H).double()
        size, nsize = S.abs(), N.abs()  # the same with magnitudes: what roundings are relative to
        for t in range(int(indptr[b]), int(indptr[b + 1])):
            q, k, v = x[t, : H * D].view(H, D) * D ** -0.5, x[t, at[1] : at[1] + H * D].view(H, D), x[t, at[2] : at[2] + H * E].view(H, E)
            new = torch.maximum(gf[t] + m, gi[t])
            a, c, m = torch.exp(gf[t] + m - new)[:, None], torch.exp(gi[t] - new)[:, None], new
            S, size = a[:, :, None] * S + (c * v)[:, :, None] * k[:, None], a[:, :, None] * size + (c * v).abs()[:, :, None] * k.abs()[:, None]
            N, nsize = a * N + c * k, a * nsize + c * k.abs()
            # sums of D terms, at most two roundings a token that the state has passed, exponents of up to 30 and their logs' roundings
            bound = (D + 128 + 2 * (t - int(indptr[b]))) * 2.0 ** -24
            assert ((got[t] - (S * q[:, None]).sum(2)).abs() <= bound * (size * q.abs()[:, None]).sum(2) + 1e-30).all(), (b, t)
            want = torch.maximum((N * q).sum(1).abs(), torch.exp(-m)) + 1e-6
            assert ((gden[t] - want).abs() <= bound * ((nsize * q.abs()).sum(1) + want)).all(), (b, t)
    # a token more, on what the chunks left in the slots: the token form finds S, n and every copy of m
    kept, live = state.clone(), [b for b in range(B) if lens[b]]
    rows = torch.tensor([int(indptr[b + 1]) - 1 for b in live])
    more = proj[rows].contiguous().to(DEV)
    o1, d1 = torch.empty(len(live), H * E, device=DEV), torch.empty(len(live), H, device=DEV)
    who = (torch.arange(len(live) + 1, dtype=torch.int32, device=DEV), slots[live].to(DEV))
    ops.memory_scan(more, at, bias_i.to(DEV), bias_f.to(DEV), kept, *who, H, D, E, 15.0, D ** -0.5, o1, d1)
    plain, o2, d2 = S0.clone().to(DEV), torch.empty_like(o1), torch.empty_like(d1)
    run(0, n, plain, who=(indptr.to(DEV), slots.to(DEV)))
    ops.memory_scan(more, at, bias_i.to(DEV), bias_f.to(DEV), plain, *who, H, D, E, 15.0, D ** -0.5, o2, d2)
    # (both forms differ from 64 bits by less than the bound above, whose factor is at most 2 (D + 128 + 2 n) 2^-24 of the magnitudes)
    scale = 2 * (D + 128 + 2 * n) * 2.0 ** -24
    assert (o1 - o2).abs().max() <= scale * D * o2.abs().max() and (d1 - d2).abs().max() <= scale * D * d2.abs().max()
    assert torch.equal(state[0].cpu(), S0[0])


@pytest.mark.parametrize("gates", [False, True])
@pytest.mark.parametrize("starts,lens,window", [([0], [200], 0), ([0, 70, 0], [1, 129, 40], 0), ([300, 0, 1000], [64, 33, 140], 100), ([0, 5], [577, 2], 64)])
@pytest.mark.parametrize("heads,dim,rot,value,latent,page", [(3, 64, 32, 64, 192, 16), (2, 128, 64, 128, 64, 8), (8, 64, 32, 64, 512, 64)])
def test_latent_prompt(heads, dim, rot, value, latent, page, starts, lens, window, gates):
    """Prompt portions over keys and values made from latents, against the same in 64 bits: tiles that are not full, portions that end
    inside a block of keys, blocks that a window cuts, pages that it has let go, a single token among the portions, both pairings."""
    from nanospec_amd.parts.attention import TilePlan
    from nanospec_amd.engine.context import BatchFacts
    import numpy as np

    ops = _ops()
    g = torch.Generator().manual_seed(heads + sum(lens))
    rnd = lambda *shape: torch.randn(*shape, generator=g).bfloat16()
    total = [s + l for s, l in zip(starts, lens)]
    pages = sum(-(-t // page) for t in total) + 3
    table = scattered_tables(total, page, pages, seed=6)
    if window:
        for b, s in enumerate(starts):
            table[b, : max(0, s - window + 1) // page] = -1
    n, C = sum(lens), latent
    cache = torch.full((pages, 1, page, C + rot), float("nan")).bfloat16()
    lat = [rnd(t, C + rot) for t in total]
    for b, t in enumerate(total):
        for p in range(t):
            if table[b, p // page] >= 0:
                cache[table[b, p // page], 0, p % page] = lat[b][p]
    q, uk, uv = rnd(n, heads * (dim + rot)), (rnd(heads * dim, C).float() * C ** -0.5).bfloat16(), (rnd(heads * value, C).float() * C ** -0.5).bfloat16()
    inv = 10000.0 ** (-torch.arange(0, rot, 2).float() / rot)
    sink = torch.randn(heads, generator=g) if gates else None
    gate = torch.rand(n, heads, generator=g) if gates else None
    zgate = rnd(n, heads * value + 8)[:, : heads * value] if gates else None
    indptr = np.concatenate(([0], np.cumsum(lens))).astype(np.int32)
    i32 = lambda x: np.asarray(x, dtype=np.int32)
    plan = TilePlan()
    tc, td = plan.shape(lens)
    region = np.zeros(plan.ints((tc + 1, td)), dtype=np.int32)  # one tile more than the batch needs
    plan.fill(region, (tc + 1, td), BatchFacts(n, len(lens), i32(lens), i32(starts), indptr, i32(total), len(lens), 1))
    tiles = torch.from_numpy(region[: 8 * (tc + 1)].reshape(-1, 8)).to(DEV)
    blocks = -(-max(total) // 128) * 2
    portions = min(tc + 1, len(lens) + 1)
    scale, dev = (dim + rot) ** -0.5, lambda t: t.to(DEV) if t is not None else None
    for interleaved in (False, True):
        out = torch.full((n, heads * value), 7.0, dtype=torch.bfloat16, device=DEV)
        scratch = torch.full((portions * blocks * ops.latent_prompt_block(torch.bfloat16, heads, dim, rot, value, C),), float("nan"), dtype=torch.bfloat16, device=DEV)
        zg = dev(zgate)
        ops.latent_prompt(dev(q), dev(cache), dev(uk), dev(uv), scratch, tiles, table.to(DEV), dev(inv), 1.0, heads, dim, rot, value, C, portions, blocks, scale, out,
                          window=window, interleaved=interleaved, gate=dev(gate), channel_gate=zg, sink_logits=dev(sink))
        out = out.cpu()
        turn = lambda x, pos: _turned(x, pos, inv.double(), interleaved)
        for b, (s, l, t) in enumerate(zip(starts, lens, total)):
            r0 = int(indptr[b])
            if l == 1:
                assert bool((out[r0] == 7).all())
                continue
            c = lat[b][:, :C].double()
            k_rot = lat[b][:, C:].double()
            pos = torch.arange(s, t)
            seen = (torch.arange(t)[None] <= pos[:, None]) & ((torch.arange(t)[None] > pos[:, None] - window) if window else torch.ones(l, t, dtype=torch.bool))
            for h in range(heads):
                qh = q[r0 : r0 + l, h * (dim + rot) : (h + 1) * (dim + rot)].double()
                kh = torch.cat([(c @ uk[h * dim : (h + 1) * dim].double().T).bfloat16().double(), k_rot], 1)
                vh = (c @ uv[h * value : (h + 1) * value].double().T).bfloat16().double()
                qt = torch.cat([qh[:, :dim], turn(qh[:, dim:], pos).bfloat16().double()], 1)
                sc = (qt @ kh.T * scale).masked_fill(~seen, float("-inf"))
                if sink is not None:
                    sc = torch.cat([sc, sink[h].double().expand(l, 1)], 1)
                pr = torch.softmax(sc, 1)[:, :t]
                want = pr @ vh
                mag = pr @ vh.abs()
                if gates:
                    f = gate[r0 : r0 + l, h, None].double() * torch.sigmoid(zgate[r0 : r0 + l, h * value : (h + 1) * value].double())
                    want, mag = want * f, mag * f
                got = out[r0 : r0 + l, h * value : (h + 1) * value].double()
                # weights and result rounded to bfloat16 (2^-9 each), keys and values whose sums another order rounds to the other side (2^-8)
                assert ((got - want).abs() <= 2.0 ** -6 * mag + 2.0 ** -8 * want.abs() + 1e-6).all(), (b, h, interleaved)


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("window", [0, 70])
def test_latent_prompt_keeps_infinities_to_the_rows_that_see_them(window, bad):
    """A latent that is infinite or no number belongs to the tokens that see its position; the others' results are what they would be
    without it, also where they share a block of keys with it."""
    from nanospec_amd.parts.attention import TilePlan
    from nanospec_amd.engine.context import BatchFacts
    import numpy as np

    ops = _ops()
    heads, dim, rot, value, C, page, start, n, at = 2, 64, 32, 64, 64, 16, 20, 150, 90
    g = torch.Generator().manual_seed(8)
    rnd = lambda *shape: torch.randn(*shape, generator=g).bfloat16().to(DEV)
    total = start + n
    pages = -(-total // page)
    cache, q = rnd(pages, 1, page, C + rot), rnd(n, heads * (dim + rot))
    uk, uv = rnd(heads * dim, C) * C ** -0.5, rnd(heads * value, C) * C ** -0.5
    inv = (10000.0 ** (-torch.arange(0, rot, 2).float() / rot)).to(DEV)
    i32 = lambda x: np.asarray(x, dtype=np.int32)
    plan = TilePlan()
    shape = plan.shape([n])
    region = np.zeros(plan.ints(shape), dtype=np.int32)
    plan.fill(region, shape, BatchFacts(n, 1, i32([n]), i32([start]), i32([0, n]), i32([total]), 1, 1))
    tiles, table = torch.from_numpy(region.reshape(-1, 8)).to(DEV), torch.arange(pages, dtype=torch.int32, device=DEV)[None].contiguous()
    blocks = -(-total // 128) * 2

    def run():
        scratch = torch.zeros(blocks * ops.latent_prompt_block(torch.bfloat16, heads, dim, rot, value, C), dtype=torch.bfloat16, device=DEV)
        out = torch.zeros(n, heads * value, dtype=torch.bfloat16, device=DEV)
        return ops.latent_prompt(q, cache, uk, uv, scratch, tiles, table, inv, 1.0, heads, dim, rot, value, C, 1, blocks, 0.1, out, window=window).float()

    clean = run()
    assert torch.isfinite(clean).all()
    cache[at // page, 0, at % page, 5] = bad
    out = run()
    pos = torch.arange(start, total, device=DEV)
    sees = (pos >= at) & (pos - at < window if window else torch.ones_like(pos, dtype=torch.bool))
    # (the sums run in another order: the result may round to the next bfloat16)
    torch.testing.assert_close(out[~sees], clean[~sees], rtol=2.0 ** -7, atol=2.0 ** -12)
    assert not torch.isfinite(out[sees]).all(dim=1).any()


def _turned(x, pos, inv, interleaved):
    half = len(inv)
    ang = (pos[:, None].float() * inv.float()[None]).double()
    c, s = ang.cos(), ang.sin()
    a, b = (x[:, 0::2], x[:, 1::2]) if interleaved else (x[:, :half], x[:, half:])
    u, v = a * c - b * s, b * c + a * s
    return torch.stack([u, v], -1).flatten(-2) if interleaved else torch.cat([u, v], -1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("experts,extra,top,groups,keep,width", [(32, 0, 4, 1, 1, 2048), (32, 0, 4, 8, 4, 2048), (31, 1, 3, 1, 1, 260), (8, 0, 8, 2, 2, 8192), (5, 0, 1, 1, 1, 4), (28, 4, 4, 4, 2, 1032)])
def test_moe_route_of_few_tokens_in_one_launch(dtype, experts, extra, top, groups, keep, width):
    """A small router's logits and choice for up to 8 tokens are one kernel, a workgroup a token: the same bits as in two launches
    (which a router of 33 rows takes, here the same one with rows that belong to no expert below it), however many tokens the step holds."""
    ops = _ops()
    torch.manual_seed(experts + width)
    h = torch.randn(8, width, device=DEV).to(dtype)
    router = torch.randn(33, width, device=DEV) * 0.1
    bias = torch.randn(33, device=DEV) if not extra else None

    def route(n, rows=experts + extra):
        sel, wt = torch.full((n, top), -1, dtype=torch.int32, device=DEV), torch.zeros(n, top, device=DEV)
        z = torch.zeros(n, rows, device=DEV)
        ops.moe_route(h[:n], router[:rows], None if bias is None else bias[:rows], top, sel, wt, logits=z, groups=groups, keep=keep, extra=rows - experts)
        return sel, wt, z[:, : experts + extra]

    got = route(8)
    want = h.double() @ router[: experts + extra].double().T + (0 if bias is None else bias[: experts + extra].double())
    torch.testing.assert_close(got[2].double(), want, rtol=1e-5, atol=1e-5 * math.sqrt(width))
    for n in (1, 3, 8):
        for a, b, c in zip(route(n), got, route(n, 33)):
            assert torch.equal(a, b[:n]) and torch.equal(a, c)


def _check_experts(out, h, gate, up, down, sel, wt, limit, alpha, shift, activation):
    """``out`` [tokens, top, width] against 64 bits.  An inner channel's sum may round to the next bfloat16 (2^-8 of it at most), and so may the
    activation made of it."""
    x = h.double()
    for e in range(up.shape[0]):
        t, k = (sel == e).nonzero(as_tuple=True)
        if not len(t):
            continue
        u = (x[t] @ up[e].double().T).bfloat16().double()
        if gate is not None:
            a = (x[t] @ gate[e].double().T).bfloat16().double().clamp(max=limit)
            act = a * torch.sigmoid(alpha * a) * (u.clamp(-limit, limit) + shift)
        else:
            act = {"relu2": lambda v: v.clamp(min=0) ** 2, "silu": lambda v: v * torch.sigmoid(v),
                   "gelu_tanh": lambda v: v * torch.sigmoid(2 * 0.7978845608028654 * (v + 0.044715 * v**3))}[activation](u)
        act = act.bfloat16().double()
        share = wt[t, k].double()[:, None]
        want, bound = share * (act @ down[e].double().T), share * 2.0**-6 * (act.abs() @ down[e].double().abs().T) + 1e-5
        assert bool(((out[t, k].double() - want).abs() <= bound).all()), e


def _experts_call(n, width, ff, experts, sel, gated, activation, seed):
    ops = _ops()
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *shape: torch.randn(*shape, generator=g, device=DEV)
    h = rnd(n, width).bfloat16()
    gate, up, down = ((rnd(experts, *s) * s[1] ** -0.5).bfloat16() for s in ((ff, width), (ff, width), (width, ff)))
    gate = gate if gated else None
    top = sel.shape[1]
    sel, wt = sel.to(DEV).int().contiguous(), torch.rand(n, top, generator=g, device=DEV)
    tiles = int(ops.build.core().ns_moe_group_tiles(n * top, experts))
    ints = torch.full((n * top + 3 * tiles + 64,), 77, dtype=torch.int32, device=DEV)
    act, out = torch.full((n * top, ff), float("nan"), dtype=torch.bfloat16, device=DEV), torch.full((n, top, width), float("nan"), device=DEV)
    ops.moe_expert_groups(h, gate, up, down, sel, wt, 7.0, 1.702, ints[: n * top + 3 * tiles], act, out, shift=1.0, activation=activation)
    assert bool((ints[-64:] == 77).all())
    _check_experts(out, h, gate, up, down, sel, wt, 7.0, 1.702, 1.0, activation)


@pytest.mark.parametrize("activation", ["relu2", "silu", "gelu_tanh"])
@pytest.mark.parametrize("n,width,ff,experts", [(400, 256, 384, 3), (40, 256, 384, 3), (9, 256, 384, 3), (400, 264, 136, 3)])
def test_experts_without_gates_apply_each_activation(n, width, ff, experts, activation):
    """In the larger tiles, the smaller ones, streamed, and where the inner size is in no whole pairs of stages."""
    sel = torch.randint(0, experts, (n, 1), generator=torch.Generator().manual_seed(n))
    _experts_call(n, width, ff, experts, sel, False, activation, n)


@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("width,ff", [(320, 576), (704, 320), (448, 2880), (264, 1448), (192, 72)])
@pytest.mark.parametrize("n", [40, 250, 400])
def test_experts_of_an_odd_number_of_stages_and_of_no_whole_ones(n, width, ff, gated):
    """Inner sizes of an odd number of stages of 64 (five at least) and of no whole stages, each in halves and wholes of the smaller tiles and in the larger
    ones (13, 83 and 133 rows an expert)."""
    _experts_call(n, width, ff, 3, torch.randint(0, 3, (n, 1), generator=torch.Generator().manual_seed(n)), gated, None if gated else "silu", n)


@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("width,ff", [(384, 640), (256, 328), (512, 256)])
@pytest.mark.parametrize("rows", [(64, 65, 128, 129, 300, 0), (64, 65, 128, 129, 300, 0, 0, 0), (1, 0, 126, 257)], ids=["larger", "smaller", "few"])
def test_experts_of_so_many_rows(rows, width, ff, gated):
    """Exactly so many rows an expert: a half tile and a row more, a whole one and a row more, several tiles.  114 an expert on average take the larger tiles, 86 and 96 the
    smaller ones, inner sizes in whole pairs of stages (but for down's with 328 channels), blocks of channels whole and cut."""
    sel = torch.cat([torch.full((r,), e) for e, r in enumerate(rows)])[torch.randperm(sum(rows), generator=torch.Generator().manual_seed(ff))]
    _experts_call(sum(rows), width, ff, len(rows), sel[:, None], gated, None if gated else "silu", ff)


@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("n,width,ff,experts,top", [(1, 256, 256, 2, 2), (65, 256, 264, 2, 1), (129, 384, 520, 3, 2), (300, 264, 136, 5, 2), (40, 2048, 1024, 16, 2), (64, 1024, 2048, 8, 2)])
def test_expert_groups_at_the_edges_of_their_tiles(n, width, ff, experts, top, gated):
    """Experts' tiles, streamed and smaller, at inner sizes in whole pairs of stages and not, with several experts a token, an expert without rows."""
    ops = _ops()
    torch.manual_seed(n + ff)
    h = torch.randn(n, width, dtype=torch.bfloat16, device=DEV)
    mk = lambda a, b: (torch.randn(experts, a, b, device=DEV) * b**-0.5).bfloat16()
    wg, wu, wd = mk(ff, width) if gated else None, mk(ff, width), mk(width, ff)
    sel = torch.rand(n, experts, device=DEV).mul_(torch.arange(experts, device=DEV) != experts - 1).topk(top, -1).indices.int() if experts > top else \
        torch.arange(top, device=DEV).int().repeat(n, 1)
    wt = torch.rand(n, top, device=DEV)
    tiles = int(ops.build.core().ns_moe_group_tiles(n * top, experts))
    ints = torch.full((n * top + 3 * tiles + 64,), 77, dtype=torch.int32, device=DEV)
    out = torch.full((n, top, width), float("nan"), device=DEV)
    ops.moe_expert_groups(h, wg, wu, wd, sel.contiguous(), wt, 7.0, 1.702, ints[: n * top + 3 * tiles], torch.empty(n * top, ff, dtype=torch.bfloat16, device=DEV), out, shift=1.0,
                          activation=None if gated else "silu")
    assert bool((ints[-64:] == 77).all())
    x = h.double().cpu()
    for t in range(0, n, max(1, n // 16)):
        for k in range(top):
            e = int(sel[t, k])
            u = (wu[e].double().cpu() @ x[t]).bfloat16().double()
            if gated:
                g = (wg[e].double().cpu() @ x[t]).bfloat16().double().clamp(max=7.0)
                a = g * torch.sigmoid(1.702 * g) * (u.clamp(-7.0, 7.0) + 1.0)
            else:
                a = u * torch.sigmoid(u)
            y = float(wt[t, k]) * (wd[e].double().cpu() @ a.bfloat16().double())
            # the roundings of act to 8 bits, where a sum in another order falls to the other side: some of ff of them
            err = float((out[t, k].double().cpu() - y).norm() / y.norm())
            assert err < 2**-8, (t, k, err)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,width", [(1, 8), (3, 2056), (70, 4096), (5, 36), (4, 77), (1000, 8), (300, 64), (70, 2560), (66000, 72)])
def test_scaled_sum_and_clipped_glu_in_pieces_and_alone(dtype, n, width):
    """Rows in whole pieces of 16 bytes and rows that are not, results at the edges of a workgroup, what is no number where it was in a sum."""
    ops = _ops()
    torch.manual_seed(n + width)
    a, b = (torch.randn(n, width, device=DEV).mul_(3).to(dtype) for _ in range(2))
    u, v = (torch.randn(width, device=DEV).to(dtype) for _ in range(2))
    a[0, 0], b[0, width - 1], a[n - 1, width - 1] = float("nan"), float("inf"), float("-inf")
    eps = 2**-8 if dtype == torch.bfloat16 else 2**-22
    for bias, bias_b in ((None, None), (u, None), (u, v)):
        ref = 0.75 * (a.double() + (0 if bias is None else bias.double())) - 1.5 * (b.double() + (0 if bias_b is None else bias_b.double()))
        got = ops.scaled_sum(a, b, 0.75, -1.5, torch.empty_like(a), bias=bias, bias_b=bias_b)
        torch.testing.assert_close(got.double(), ref, rtol=eps, atol=1e-5, equal_nan=True)
    a, b = a.nan_to_num(1.0, -30.0, 30.0), b.nan_to_num(1.0, 30.0, -30.0)
    g, up = a.double().clamp(max=7.0), b.double().clamp(-7.0, 7.0)
    got = ops.clipped_glu(torch.cat([a, b], 1), 7.0, 1.702, torch.empty_like(a), shift=1.0)
    torch.testing.assert_close(got.double(), g * torch.sigmoid(1.702 * g) * (up + 1.0), rtol=2 * eps, atol=1e-6)


def _finite_bf16():
    z = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    z = z[torch.isfinite(z)]
    return torch.cat([z, torch.zeros(-len(z) % 64, dtype=torch.bfloat16)]).view(-1, 64).contiguous()


def _within_half_a_step(got, ref, floor):
    """bfloat16 results within half a step of 64 bits (2^-8 of the value: 8 bits) and a hair of the 32-bit value; results below ``floor`` no larger than
    the true one and of its sign."""
    near = (got - ref).abs() <= ref.abs() * (2**-8 + 2**-19) + 2.0**-134  # (half of the smallest bfloat16)
    return bool((near | ((ref.abs() < floor) & (got.abs() <= ref.abs()) & (got * ref >= 0))).all())


def test_silu_at_the_ends_of_its_range():
    """Every finite bfloat16 value against 64 bits, in each kernel that divides by 1 + exp(-z) with nothing else behind it: down to where the
    divisor is out of range (z = -88.7, a result of 2^-121), and zero from there on, not something that grows."""
    ops = _ops()
    z = _finite_bf16()
    d = z.double()
    ref = torch.where(d < -700, torch.zeros_like(d), d / (1 + torch.exp(-d.clamp(min=-700))))
    g, one, zero = z.to(DEV), torch.ones_like(z, device=DEV), torch.zeros_like(z, device=DEV)
    bias = torch.zeros(128, dtype=torch.bfloat16, device=DEV)
    for name, got in (("activation", ops.activation(g.clone(), "silu")), ("silu_mul", ops.silu_mul(torch.cat([g, one], 1))),
                      ("silu_mul_bias", ops.silu_mul_bias(torch.cat([g, one], 1), bias)),
                      ("clipped_glu", ops.clipped_glu(torch.cat([g, zero], 1), float("inf"), 1.0, torch.empty_like(g), shift=1.0))):
        got = got.cpu().double()
        assert _within_half_a_step(got, ref, 2.0**-121), name
        assert bool((got[d < -89] == 0).all()), name
    ends = torch.tensor([[float("inf"), float("nan")] * 32], dtype=torch.bfloat16, device=DEV)
    out = ops.activation(ends, "silu")
    assert bool(torch.isinf(out[0, 0])) and float(out[0, 0]) > 0 and bool(torch.isnan(out[0, 1]))


def test_gelu_at_the_ends_of_its_range():
    """Every finite bfloat16 value against 64 bits: down to where the exponential is out of range (a result of some 2^-123), and exact at the ends."""
    ops = _ops()
    z = _finite_bf16()
    d = z.double()
    u = 0.7978845608028654 * (d + 0.044715 * d**3)
    ref = torch.where(u < -350, torch.zeros_like(d), d / (1 + torch.exp(-2 * u.clamp(min=-350))))
    assert _within_half_a_step(ops.activation(z.to(DEV).clone(), "gelu_tanh").cpu().double(), ref, 2.0**-121)
    ends = torch.tensor([[float("inf"), float("nan")] * 32], dtype=torch.bfloat16, device=DEV)
    out = ops.activation(ends, "gelu_tanh")
    assert bool(torch.isinf(out[0, 0])) and float(out[0, 0]) > 0 and bool(torch.isnan(out[0, 1]))


@pytest.mark.parametrize("deviation", [0.01, 0.1, 0.3, 1.2, 4.0])
def test_gelu_is_as_near_as_its_formula(deviation):
    """32-bit GELU against 64 bits: no further off in the 2-norm than 0.5 z (1 + tanh(u)) taken in 32 bits, for small z as for large ones."""
    ops = _ops()
    torch.manual_seed(3)
    z = torch.randn(1 << 20, device=DEV) * deviation
    d = z.double()
    ref = d / (1 + torch.exp(-2 * 0.7978845608028654 * (d + 0.044715 * d**3)))
    formula = 0.5 * z * (1 + torch.tanh(0.7978845608028654 * (z + 0.044715 * z * z * z)))
    off = lambda t: float((t.double() - ref).norm() / ref.norm())
    assert off(ops.activation(z.clone(), "gelu_tanh")) <= off(formula)
