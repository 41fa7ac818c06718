"""How products of few rows are dealt to the compute units (``ops.wide_plan``, ``ops.wide_waves``, ``ops.rows_plan``):
plain arithmetic on sizes, so it runs without a GPU when the number of compute units is given."""
import pytest
import torch

from nanospec_amd.kernels import ops

UNITS = 256  # an MI355X


def busiest(tiles: int, per_group: int, ksplit: int, units: int = UNITS) -> int:
    """Row tiles times ranges' share that the busiest unit streams when groups of tiles go round the units in turn."""
    groups = -(-tiles // per_group) * ksplit
    return -(-groups // units) * per_group


@pytest.mark.parametrize("n,k", [(6144, 4096), (4096, 4096), (4096, 14336), (3072, 2048), (2048, 2048), (2048, 8192), (10240, 8192), (200, 264)])
def test_one_matrix_takes_the_form_that_leaves_the_busiest_unit_least(n, k):
    ksplit, nt = ops.wide_plan(n, k, 64, units=UNITS)
    waves, halves = ops.wide_waves(n, k, 64, ksplit, nt, units=UNITS)
    assert not halves and waves in (3, 4) and 1 <= ksplit <= 16 and ksplit <= max(1, -(-k // 128) // 4)
    if nt == 1:
        k_tiles = -(-k // 128)
        cost = lambda w: busiest(-(-n // 16), w, ksplit) * -(-k_tiles // ksplit)
        assert cost(waves) == min(cost(3), cost(4))
        assert waves == 4 or cost(3) < cost(4)  # three waves only where they gain


def test_the_shapes_of_the_benchmark():
    assert ops.wide_plan(6144, 4096, 64, units=UNITS) == (2, 1) and ops.wide_waves(6144, 4096, 64, 2, 1, units=UNITS) == (3, False)
    assert ops.wide_plan(4096, 14336, 64, units=UNITS) == (4, 1) and ops.wide_waves(4096, 14336, 64, 4, 1, units=UNITS) == (4, False)
    # gate and up: 1,792 half tiles are 7 for each of 256 units; 1,024 are 4 for each; 448 workgroups of whole tiles fill the GPU
    assert ops.wide_waves(14336, 4096, 64, 1, 1, gated=True, units=UNITS) == (7, True)
    assert ops.wide_waves(8192, 2048, 64, 1, 1, gated=True, units=UNITS) == (4, True)
    assert ops.wide_waves(28672, 8192, 64, 1, 1, gated=True, units=UNITS) == (4, False)


def test_what_each_form_is_kept_for():
    assert ops.wide_waves(14336, 4096, 100, 1, 1, units=UNITS) == (4, False)             # more than 64 rows of one matrix
    assert ops.wide_waves(14336, 4096, 100, 1, 1, gated=True, units=UNITS) == (7, True)  # ... of gate and up: half tiles only
    assert ops.wide_waves(14336, 4096, 64, 2, 1, gated=True, units=UNITS) == (4, False)  # gate and up over ranges: whole tiles
    assert ops.wide_waves(128256, 4096, 64, 1, 2, units=UNITS) == (4, False)             # two tiles a wave
    # another GPU: 304 units are dealt 1,792 half tiles as 6 each in workgroups of ... the forms at hand, whichever is least
    waves, halves = ops.wide_waves(14336, 4096, 64, 1, 1, gated=True, units=304)
    assert (waves, halves) in ((4, False), (7, True), (4, True))


def test_many_rows_in_blocks():
    ksplit, nt = ops.rows_plan(8192, 8192, 2048, units=UNITS)
    assert nt == 4 and ksplit == 1  # 32 groups of row tiles times 16 blocks of rows fill the GPU without cutting K
    ksplit, nt = ops.rows_plan(4096, 14336, 130, gated=False, units=UNITS)
    assert nt == 4 and ksplit >= 2


def test_many_rows_take_the_smallest_tile_that_fits_the_units_once():
    plan = lambda *a, **k: ops.many_plan(*a, UNITS, **k)
    assert plan(512, 2048, 2048) == (0, 1) and plan(512, 3072, 2048) == (1, 1) and plan(2048, 2048, 8192) == (2, 1) and plan(2048, 4096, 14336) == (3, 1)
    assert plan(2048, 6144, 2048) is None and plan(1024, 6144, 2048) is None  # more tiles than units
    assert plan(384, 16384, 2048) is None and plan(512, 16384, 2048) == (3, 1)  # a quarter of the tiles' rows beyond the last
    assert plan(768, 4096, 2048) == (2, 1) and plan(768, 4096, 8192) is None   # a quarter of the units without a tile, and a long K
    assert plan(512, 16384, 2048, gated=True) == (3, 1) and plan(160, 16384, 2048, gated=True) == (2, 1) and plan(2048, 28672, 4096, gated=True) is None
    # ranges of K only for readers that add them up, no more of them than fill the units, each of whole pairs of stages
    assert plan(512, 2048, 8192, may_split=True) == (2, 4) and plan(800, 2048, 8192, may_split=True) == (2, 2) and plan(512, 2048, 2048, may_split=True) == (0, 1)
    assert plan(800, 2048, 4096 + 256, may_split=True) == (2, 2)  # (512 rows, half of the units: 30.5 us, in whole tiles 26.4 and 27.5 in the library)
    # and only where they fill enough of them
    assert plan(129, 16, 8192, may_split=True) is None and plan(129, 68, 4096, may_split=True) is None and plan(256, 1024, 8192, may_split=True) is None
    assert plan(200, 1024, 4096, may_split=True) is None and plan(200, 2048, 4096, may_split=True) == (2, 4) and plan(200, 2048, 8192, may_split=True) == (2, 4) and plan(512, 2048, 4352, may_split=True) == (0, 1)
    assert plan(384, 4096, 4096, may_split=True) == (2, 2) and plan(200, 4480, 4096, may_split=True) is None and plan(384, 4096, 8192, may_split=True) == (2, 2)
    # too few tiles for the units: the more the longer K is
    assert plan(200, 64, 1024) == (0, 1) and plan(200, 64, 2048) is None and plan(1024, 512, 2048) == (0, 1) and plan(1024, 512, 4096) is None
    assert plan(2048, 512, 4096) == (0, 1) and plan(2048, 512, 6144) == (0, 1) and plan(1600, 512, 6144) is None and plan(512, 2560, 4096) is None and plan(384, 8192, 4608) == (2, 1) and plan(384, 8192, 5120) is None
    assert plan(1531, 256, 2048) == (0, 1) and plan(1531, 2048, 4096) == (2, 1)  # (level alone, ahead beside other work and on the host)
    assert plan(160, 1024, 2048, gated=True) is None and plan(256, 4096, 1024, gated=True) == (2, 1) and plan(384, 16384, 8192, gated=True) == (3, 1)
    for m, n, k in ((128, 2048, 2048), (512, 2048, 2048 + 64), (512, 2050, 2048), (512, 2048, 128)):
        assert plan(m, n, k) is None
    for m in (129, 300, 512, 1000, 1531, 2048):
        for n in (68, 2048, 4096, 16384):
            form_ranges = plan(m, n, 4096, may_split=True)
            if form_ranges is not None and form_ranges[1] > 1:
                assert form_ranges[0] == ops.MANY_SPLIT_FORM and form_ranges[1] <= ops.many_ranges(m, n, UNITS)


def expands(lens, kv, sizes, window=0, captured=False):
    """What ``LatentAttention._expands`` says of a step of these requests: (portions, blocks of 64 keys)."""
    from types import SimpleNamespace

    import torch

    from nanospec_amd.parts.attention import TILES, TilePlan
    from nanospec_amd.parts.latent import LatentAttention

    H, D, R, E, C = sizes
    shape = TILES.shape(lens)
    part = object.__new__(LatentAttention)
    part.spec, part._block = SimpleNamespace(heads=H, head_dim=D, rot_dim=R, value_dim=E, kv_rank=C, window=window), H * 64 * (D + R + E)
    ctx = SimpleNamespace(plans={TilePlan.key: (torch.zeros(TILES.ints(shape), dtype=torch.int32), shape)}, n_reqs=len(lens), captured=captured,
                          max_chunk_kv=max(k for k, n in zip(kv, lens) if n > 1) if any(n > 1 for n in lens) else 0)
    return part._expands(ctx, sum(lens), SimpleNamespace(k=torch.zeros(1, 1, 16, C + R)))


def test_where_latent_portions_have_keys_and_values_made():
    """By the portions' tokens, the keys they find, how far the wide form is behind at these sizes, and whether it has to be formed for
    single tokens all the same."""
    wide, middle, near = (32, 64, 32, 64, 512), (16, 128, 64, 128, 512), (8, 64, 32, 64, 128)
    assert expands([127], [127], wide) == (0, 0) and expands([128], [128], wide) == (1, 2) and expands([128], [2028], wide) == (1, 32)
    assert expands([128], [2049], wide) == (0, 0)
    assert expands([60] * 4, [60] * 4, wide) == (0, 0) and expands([64] * 4, [64] * 4, wide) == (4, 2)
    # a latent of 128: few tiles and many keys stay with the wide form, which cuts the keys
    assert expands([512], [7512], near) == (0, 0) and expands([128], [640], near) == (1, 10) and expands([2048], [10048], near) == (1, 158)
    # beside single tokens
    assert expands([64, 64, 64, 64, 1], [64, 64, 64, 64, 9], wide) == (4, 2)
    assert expands([64, 64, 64, 64], [64] * 4, middle) == (4, 2) and expands([64, 64, 64, 64, 1], [64, 64, 64, 64, 9], middle) == (0, 0)
    assert expands([128, 1], [128, 9], near) == (0, 0) and expands([300, 1], [300, 9], near) == (1, 6)
    # a captured step knows its tokens and the keys that its tables can name
    assert expands([512, 1], [1024, 9], wide, captured=True) == (1, 16)


@pytest.mark.parametrize("lens,unused,spare", [([40, 1, 2, 65], 0, 0), ([40, 1], 3, 4), ([1, 1, 33], 1, 1), ([1], 4, 3)])
def test_tiles_number_the_portions_that_bring_tokens(lens, unused, spare):
    """The tile list of a batch whose fixed shape has room for more portions and more tiles: a portion's tiles carry its number, the p-th
    tile's last int is portion p's first tile, and nothing is said of portions without tokens."""
    import numpy as np

    from nanospec_amd.engine.context import BatchFacts
    from nanospec_amd.parts.attention import TILES

    all_lens = lens + [0] * unused + [7]  # (the last request is the stand-in that owns the padding)
    i32 = lambda x: np.asarray(x, dtype=np.int32)
    shape = TILES.shape(lens)
    shape = (shape[0] + spare, shape[1])
    starts = [10 * b for b in range(len(lens))] + [0] * (unused + 1)
    indptr = i32(np.concatenate(([0], np.cumsum(all_lens))))
    out = np.full(TILES.ints(shape), -5, dtype=np.int32)
    TILES.fill(out, shape, BatchFacts(sum(all_lens), len(all_lens), i32(all_lens), i32(starts), indptr, i32(starts) + i32(all_lens), len(all_lens) - 1, 1))
    tiles = out[: 8 * shape[0]].reshape(-1, 8)
    many = [b for b, n in enumerate(lens) if n > 1]
    at = 0
    for p, b in enumerate(many):
        assert tiles[p, 7] == at
        for t0 in range(0, lens[b], 32):
            assert tuple(tiles[at, :7]) == (b, t0, indptr[b], lens[b], starts[b] + lens[b], 0, p)
            at += 1
    assert (tiles[at:, 1:7] == 0).all() and (tiles[len(many) :, 7] == -1).all()


def test_captured_steps_laid_out_for_long_portions():
    """Kernels for portions of 64 tokens and more are in a captured step unless hardly any portion that it takes is so long."""
    from nanospec_amd.engine.runner import MIXED_MAX_TOKENS, ModelRunner, _StepGraph

    runner = object.__new__(ModelRunner)
    for rows in (0, 1, 8, 48):
        for n in range(2, MIXED_MAX_TOKENS + 1):
            shape = runner._graph_shape([1] * rows + [n], 1)
            longest = _StepGraph.longest(shape[1])
            assert shape[1] - 12 <= longest <= shape[1]
            if shape[1] <= 64:  # a prompt of 40 tokens, alone
                assert longest < 64
            if n >= 77:
                assert longest >= 64
    assert _StepGraph.longest(0) == 1


def test_recurrences_leave_out_the_padding_behind_portions():
    """A captured step's stand-in request owns the tokens behind the portions; padding rows of one token are rows like others."""
    import torch

    from nanospec_amd.engine.context import BatchLayout, StepContext

    layout = BatchLayout(70, 5, 2, 1, 4)
    make = lambda **kw: StepContext(layout, torch.arange(layout.total, dtype=torch.int32), None, 0, 64, **kw)
    for kw, left_out in ((dict(captured=True), 1), (dict(captured=True, single_tokens=True), 0), (dict(), 0)):
        ctx = make(**kw)
        indptr, slots = ctx.spans
        assert torch.equal(indptr, ctx.qo_indptr[: 6 - left_out]) and torch.equal(slots, ctx.state_slots[: 5 - left_out])


def test_products_are_told_the_rows_that_are_read():
    """The arena of a captured step with portions knows the stand-in's first row; of any other step that uses it, nothing."""
    import torch

    from nanospec_amd.engine.arena import Arena
    from nanospec_amd.engine.context import BatchLayout, StepContext

    layout, arena = BatchLayout(70, 5, 2, 1, 4), Arena("cpu")
    for kw in (dict(captured=True), dict(captured=True, single_tokens=True), dict()):
        ctx = StepContext(layout, torch.arange(layout.total, dtype=torch.int32), arena, 0, 64, **kw)
        if kw == dict(captured=True):
            assert arena.read_rows[0] == 70 and torch.equal(arena.read_rows[1], ctx.qo_indptr[4:5])
        else:
            assert arena.read_rows is None


def test_chunks_of_the_delta_rule_beside_single_tokens():
    """Single tokens whose states take as long as a short portion's chain keep that portion token by token."""
    least = lambda portions, heads, dim, singles: ops.delta_chunk_min(portions, heads, dim, dim, singles)
    assert [least(1, 16, 128, n) for n in (0, 16, 31, 32, 64, 127, 128)] == [64, 64, 64, 96, 96, 96, 192]
    assert [least(1, 32, 128, n) for n in (8, 16, 32, 64)] == [64, 96, 96, 192]
    assert [least(1, 16, 64, n) for n in (0, 64, 127, 128)] == [64, 64, 64, 96]
    assert least(4, 16, 64, 64) == 64 and least(8, 16, 64, 0) == 96 and least(16, 16, 64, 0) == 0x7FFFFFFF


def _operands(form, device="cpu", m=160, n=256, k=512):
    """bfloat16 x [m, k] and w [n, k] of small whole numbers, in whole pieces and rows behind one another but for what ``form`` names."""
    base = torch.arange((n + m) * (k + 16), device=device).remainder(13).sub(6).bfloat16()
    x, w = base[: m * k].view(m, k), base[m * k : (m + n) * k].view(n, k)
    return {"whole": (x, w), "x of one row": (x[:1].expand(m, k), w), "x overlapping": (base.as_strided((m, k), (k // 2, 1)), w),
            "w in wider rows": (x, base.as_strided((n, k), (k + 8, 1))), "w by columns": (x, base[: n * k].view(k, n).t()),
            "w off its pieces": (x, base[4 : 4 + n * k].view(n, k)), "x off its pieces": (base[4 : 4 + m * k].view(m, k), w)}[form]


FORMS = ("x of one row", "x overlapping", "w in wider rows", "w by columns", "w off its pieces", "x off its pieces")


def test_what_the_product_of_many_rows_takes():
    """Rows that overlap or repeat and matrices that do not lie in plain rows of whole pieces are not the own kernel's."""
    from unittest import mock

    with mock.patch.object(torch.Tensor, "is_cuda", True):
        assert ops.many_takes(*_operands("whole"))
        for form in FORMS:
            assert not ops.many_takes(*_operands(form)), form
    assert not ops.many_takes(*_operands("whole"))
    out = torch.zeros(160, 264, dtype=torch.bfloat16)
    assert ops.many_writes(out, 160, 264) and ops.many_writes(out[:, :256], 160, 256)
    assert not ops.many_writes(out, 160, 256) and not ops.many_writes(out[:, 1:257], 160, 256) and not ops.many_writes(out[:, :256].t(), 256, 160)


@pytest.mark.gpu
@pytest.mark.parametrize("act", [None, "silu"])
@pytest.mark.parametrize("form", ("whole",) + FORMS)
def test_operands_of_any_layout_have_their_product(form, act):
    """At a size that the own kernel is chosen for, whichever takes them.  Every sum is a whole number of at most 36 * 512, so the result is rounded once."""
    from nanospec_amd.parts.linear import LinearWeight

    x, w = _operands(form, "cuda")
    assert ops.many_plan(*x.shape[:1], *w.shape, UNITS) is not None
    want = (x.cpu().double() @ w.cpu().double().T).bfloat16().cuda()
    got = LinearWeight(w, tiled=False)(x, act=act)
    assert torch.equal(got, want if act is None else ops.activation(want, act))


def test_a_product_of_many_rows_on_the_cpu():
    """A matrix kept in plain rows alone needs none of the kernels: its product is the library's wherever it lies."""
    from nanospec_amd.parts.linear import LinearWeight

    x, w = _operands("whole")
    assert torch.equal(LinearWeight(w, tiled=False)(x), (x.double() @ w.double().T).bfloat16())


@pytest.mark.gpu
@pytest.mark.parametrize("of", ["x", "w"])
def test_a_product_of_many_rows_has_its_gradient(of):
    """Whole numbers: the gradients of the results' sum are column sums, exact in 32-bit and rounded once (by at most half a step, 2^-9)."""
    from nanospec_amd.parts.linear import LinearWeight

    x, w = (t.clone() for t in _operands("whole", "cuda"))
    (x if of == "x" else w).requires_grad_()
    LinearWeight(w, tiled=False)(x).sum().backward()
    got, want = (x.grad, w.detach().double().sum(0).expand_as(x)) if of == "x" else (w.grad, x.detach().double().sum(0).expand_as(w))
    torch.testing.assert_close(got.double(), want, rtol=2**-8, atol=0)
    with torch.no_grad():
        assert ops.many_takes(x, w)
