"""The GEMM of prompts (ops/hip/tile_gemm.hip) and the rules that choose it."""
import pytest
import torch

FORMS = [(8, 8), (6, 8), (8, 6), (6, 6), (8, 4), (4, 4), (2, 4), (2, 8)]
STAGES = [2, 2, 2, 3, 3, 4, 6, 4]       # the fewest of a part
PLAIN, PARTS, GLU = 0, 1, 2


def _built(form, end):
    """Tiles of 64 rows are for gate/up only."""
    wm, wn = FORMS[form]
    return wn % 4 == 0 if end == GLU else wm > 2


def _operands(m, n, k):
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(m * 1000003 + n + k)
    x = torch.randn(m, k, device=dev, generator=gen).bfloat16()
    w = (torch.randn(n, k, device=dev, generator=gen) / k ** 0.5).bfloat16()
    full = x.double() @ w.double().t().contiguous()
    # f32 sums of bf16 products: k roundings of 2^-24 of the magnitudes' sums
    sums = (x.double().abs() @ w.double().abs().t().contiguous()) * k * 2 ** -24
    return x, w, full, sums


def _near(got, end, full, sums):
    if end == PARTS:
        return ((got.double().sum(0) - full).abs() <= sums).all()
    if end == PLAIN:        # and half an ulp of the result
        return ((got.double() - full).abs() <= full.abs() * 2 ** -8 + sums).all()
    f = full.shape[1] // 2
    g, u = full[:, :f], full[:, f:]
    want = torch.nn.functional.silu(g) * u
    # |silu'| < 1.1; the exponential and the division to a few 2^-23
    bound = want.abs() * (2 ** -8 + 2 ** -20) + \
        1.1 * sums[:, :f] * u.abs() + (g.abs() + 1) * sums[:, f:]
    return ((got.double() - want).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("form", range(len(FORMS)))
@pytest.mark.parametrize("m,n,k", [
    (1, 64, 256), (127, 320, 320), (129, 1088, 1024), (255, 192, 640),
    (257, 2176, 832), (300, 576, 1088), (769, 1600, 256)])
def test_forms(form, m, n, k):
    """Every tile: rows and columns short of a tile and past one, few and odd
    numbers of stages, parts of unequal length, several tiles a workgroup."""
    from rbg_amd import ops
    x, w, full, sums = _operands(m, n, k)
    for end in (PLAIN, PARTS, GLU):
        if not _built(form, end) or k // 64 < STAGES[form]:
            continue
        for parts in (1, 2, 3) if end == PARTS else (1,):
            if k // 64 // parts < max(4, STAGES[form]):
                continue
            got = ops._hip.tile_form(x, w, end, form, parts, -1, 0)
            assert _near(got, end, full, sums), (end, parts)


@pytest.mark.gpu
@pytest.mark.parametrize("end", [PLAIN, GLU])
def test_second_form_for_the_rest(end):
    from rbg_amd import ops
    x, w, full, sums = _operands(500, 2048, 512)
    for form, rest, to in ((0, 4, 512), (0, 5, 768), (4, 0, 256)):
        got = ops._hip.tile_form(x, w, end, form, 1, rest, to)
        assert _near(got, end, full, sums)


@pytest.mark.gpu
def test_many_tiles_a_workgroup():
    """More tiles than workgroups, of a few stages each: loads run several
    tiles ahead."""
    from rbg_amd import ops
    operands = {k: _operands(2100, 9280, k) for k in (256, 384)}
    for form in range(len(FORMS)):
        x, w, full, sums = operands[384 if STAGES[form] > 4 else 256]
        for end in (PLAIN, GLU):
            if not _built(form, end):
                continue
            got = ops._hip.tile_form(x, w, end, form, 1, -1, 0)
            assert _near(got, end, full, sums), (form, end)


@pytest.mark.gpu
@pytest.mark.parametrize("form", [f for f in range(len(FORMS))
                                  if _built(f, GLU)])
def test_silu_of_very_negative_gates(form):
    """Sigmoids below the smallest normal f32 are not lost, as a large up value
    makes their product with it an ordinary number; an exponential above f32's
    range gives 0.  The gates are exact: 2^-8 for the result's rounding, and
    |g| 2^-22 for the exponential's argument."""
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    gates = torch.tensor([0., -1., -60., -87., -87.5, -88., -88.5, -100.],
                         device=dev)
    m, k, up = 70, 512, 2. ** 100
    x = torch.ones(m, k, dtype=torch.bfloat16, device=dev)
    w = torch.full((128, k), up / k, device=dev)
    w[:64] = (gates / k).repeat(8)[:, None]
    got = ops._hip.tile_form(x, w.bfloat16(), GLU, form, 1, -1, 0).double()
    g = gates.double()
    want = (g / (1 + (-g).exp()) * up).masked_fill(g < -88.7, 0).repeat(8)
    assert ((got - want).abs() <= want.abs() * (2 ** -8 + 100 * 2 ** -22)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [
    (65, 2048, 12288), (128, 4096, 12288), (129, 2048, 3584),
    (65, 2048, 4096), (97, 5120, 3584), (128, 3072, 8192), (70, 12288, 4096),
    (112, 12544, 5120), (66, 14336, 4608),
    (256, 6144, 4096), (257, 2048, 5120), (999, 3136, 5120),
    (1000, 6144, 4096), (1500, 14336, 3584), (2048, 4096, 8192)])
def test_parts_route(m, n, k):
    from rbg_amd import ops
    assert ops._tile(m, n, k)
    x, w, full, sums = _operands(m, n, k)
    got = ops.linear_parts(x, w)
    assert _near(got, PARTS if got.dim() == 3 else PLAIN, full, sums)
    # rows further apart than they are long
    wide = torch.cat([x, x], dim=1)
    assert torch.equal(ops.linear_parts(wide[:, :k], w), got)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [
    (5, 16448, 2048), (33, 26624, 2048), (33, 65536, 6144), (64, 32832, 2048),
    (16, 18432, 4160), (63, 36864, 4096),
    (64, 16448, 2112), (33, 32768, 2112), (5, 32832, 2112), (33, 36864, 4160),
    (64, 57408, 2112), (17, 65536, 8192),
    (65, 24576, 1024), (128, 28672, 1088), (129, 8192, 2048),
    (256, 18432, 2048), (385, 28672, 1024), (1000, 11264, 2048),
    (2048, 28672, 1024)])
def test_swiglu_route(m, n, k):
    """In tiles, but for what the decode GEMM is asked for first: few rows of k that is
    a multiple of 2048, below 65536 columns or 8192 k."""
    from rbg_amd import ops
    assert ops._tile_glu(m, n, k)
    first = m <= 64 and k % 2048 == 0 and n * k < 2 ** 29
    assert ops.block_routes(m, (n, k), (n, k), True)[0] == (3 if first else 4)
    x, w, full, sums = _operands(m, n, k)
    assert _near(ops.linear_swiglu(x, w), GLU, full, sums)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(65, 24576, 1024), (128, 24640, 2048),
                                   (100, 32768, 1088), (129, 49152, 1024),
                                   (256, 49216, 1024)])
def test_f32_route(m, n, k):
    from rbg_amd import ops
    assert ops._tile_f32(m, n, k)
    x, w, full, sums = _operands(m, n, k)
    got = ops.linear_f32(x, w)
    assert got.dtype == torch.float32 and got.shape == (m, n)
    assert ((got.double() - full).abs() <= sums).all()
    assert not ops._tile_f32(64, n, k) and not ops._tile_f32(257, n, k)


@pytest.mark.gpu
def test_refuses_what_it_cannot_take():
    from rbg_amd import ops
    dev = torch.device("cuda:0")
    x = torch.randn(300, 512, device=dev).bfloat16()
    w = torch.randn(256, 512, device=dev).bfloat16()
    for bad in ((x[:, :500].contiguous(), w[:, :500].contiguous()),
                (x, w[:250].contiguous()), (x[:, ::2], w[:, :256]),
                (x.float(), w.float())):
        for f in (ops._hip.tile_swiglu, ops._hip.tile_parts):
            with pytest.raises(RuntimeError):
                f(*bad)
    with pytest.raises(RuntimeError):       # parts of too few stages
        ops._hip.tile_form(x, w, PARTS, 5, 4, -1, 0)
    for form in range(len(FORMS)):          # forms that are not built
        for end in (PLAIN, PARTS, GLU):
            if not _built(form, end):
                with pytest.raises(RuntimeError):
                    ops._hip.tile_form(x, w, end, form, 1, -1, 0)


def test_rules_hand_over_what_it_takes():
    from rbg_amd.ops import _tile, _tile_glu
    taken = [0, 0]
    for n in (64, 1024, 2048, 4096, 6144, 8192, 8200, 10240, 14336, 16384,
              28672, 57344):
        for k in (256, 1000, 2048, 3584, 4096, 5120, 12288, 25600):
            for rows in (0, 1, 64, 65, 128, 129, 256, 257, 999, 1000, 4096,
                         4097, 8192):
                for i, rule in enumerate((_tile, _tile_glu)):
                    if rule(rows, n, k):
                        assert rows > (64, 4)[i]
                        assert n % 64 == 0 and k % 64 == 0
                        assert k >= 256
                        taken[i] += 1
    assert min(taken) > 50


@pytest.mark.parametrize("shape", [(64,), (3, 64), (2, 3, 64), (0, 64)])
def test_norm_swiglu_of_any_rows(shape):
    """Rows in any number of dimensions, as the norm and the product take them; within
    2^-6 of the values' scale, as both and silu round to bf16."""
    from rbg_amd import ops
    gen = torch.Generator().manual_seed(len(shape))
    src, res = (torch.randn(shape, generator=gen).bfloat16() for _ in "sr")
    nw = torch.randn(64, generator=gen).bfloat16()
    w = (torch.randn(96, 64, generator=gen) / 8).bfloat16()
    total = src.double() + res.double()
    h = total * (total.square().mean(-1, keepdim=True) + 1e-5).rsqrt() * nw.double()
    gate, up = (h @ w.double().t()).chunk(2, -1)
    got, new = ops.norm_swiglu(src, res.clone(), nw, 1e-5, w)
    assert got.shape == (*shape[:-1], 48) and new.shape == shape
    bound = 2 ** -6 * (gate.abs() + 1) * (up.abs() + 1)
    want = torch.nn.functional.silu(gate) * up
    assert ((got.double() - want).abs() <= bound).all()


def test_rules_of_f32_and_few_rows_hand_over_what_is_taken():
    """Sizes that the tiles, and the decode GEMM with silu, refuse go elsewhere."""
    from rbg_amd.ops import _glu, _tile_f32, _tile_few, _tile_fits
    taken = [0, 0]
    for n in (64, 4096, 4128, 16448, 24576, 24608, 49152, 65536, 128256, 131072):
        for k in (64, 512, 768, 1000, 1088, 2048, 2112, 2304, 5120, 8192, 8256,
                  16384):
            for rows in (0, 1, 4, 5, 16, 17, 33, 64, 65, 128, 129, 256, 257):
                if _tile_f32(rows, n, k):
                    assert 64 < rows <= 256 and n % 64 == 0 and k % 64 == 0
                    assert k >= 512 and _tile_fits(rows, n, k)
                    taken[0] += 1
                if _glu(rows, n, k):
                    assert 1 <= rows <= 64 and n % 64 == 0 and k % 256 == 0
                    taken[1] += 1
                if _tile_few(rows, n, k):
                    assert 4 < rows <= 64 and k >= 1024
    assert min(taken) > 30


def test_gate_up_of_few_rows_goes_where_the_rules_say():
    """The decode GEMM is asked first, and leaves the tiles k that is no multiple of 256
    and one size of those that are."""
    from rbg_amd.ops import _glu, _own_routes, _tile_few
    left = set()
    for n in range(16448, 131073, 1216):
        for k in (2048, 2112, 2304, 4096, 4160, 6144, 7232, 7296, 8192, 8256):
            for rows in (4, 5, 32, 33, 64, 65):
                route = _own_routes(rows, (n, k), (n, k), True)[0]
                assert (route == 3) == _glu(rows, n, k)
                if rows <= 64:
                    assert (route == 4) == (_tile_few(rows, n, k) and
                                            not _glu(rows, n, k))
                    if route == 4:
                        left.add(k % 256)
                        assert n <= (98304 if k <= 7232 or rows <= 32 else 57344)
    assert left == {7296 % 256, 64}
    assert _own_routes(48, (65536, 8192), (65536, 8192), True)[0] == 4
    assert all(_glu(rows, n, 8192) for rows in (5, 64) for n in (32768, 65472))


@pytest.mark.parametrize("rows,n,k,taken", [
    (48, 33152, 4096, False), (32, 33152, 4096, True), (48, 36864, 4096, True),
    (5, 50304, 5120, False), (16, 50304, 5120, True), (16, 50304, 7168, False),
    (5, 54272, 5120, True), (64, 66048, 3584, False), (56, 66048, 2560, True),
    (48, 102400, 7168, False), (56, 102400, 7168, True), (64, 13696, 1024, False),
    (24, 22016, 7168, False), (16, 22016, 7168, True)])
def test_decode_gemm_between_rounds(rows, n, k, taken):
    """Widths a little above whole rounds of workgroups, which are the library's, and
    their neighbours."""
    from rbg_amd import ops
    assert ops._skinny(rows, n, k) == taken


@pytest.mark.parametrize("rows,n,k,taken", [
    (128, 34048, 1536, False), (128, 41984, 1536, True), (128, 34048, 2048, True),
    (128, 50304, 3584, False), (128, 50304, 2048, True), (128, 49152, 3584, True),
    (128, 66048, 4096, False), (72, 66048, 4096, True), (80, 102400, 2560, False),
    (72, 102400, 2560, True), (128, 102400, 8192, False), (128, 128256, 8192, True)])
def test_f32_tiles_between_rounds(rows, n, k, taken):
    from rbg_amd import ops
    assert ops._tile_f32(rows, n, k) == taken


@pytest.mark.parametrize("rows,n,k,fewer", [
    (130, 65536, 65536, (130, 65536, 65024)),
    (129, 131072, 32768, (129, 131072, 32512)),
    (200, 14336, 289280, (200, 14336, 289216)),
    (4096, 2048, 1677824, (4096, 2048, 1677696)),
    (2 ** 24, 8192, 1024, (2 ** 24 - 1, 8192, 1024)),
    (2 ** 24 - 1, 16384, 1024, (2 ** 23, 16384, 1024))])
def test_rules_leave_what_it_refuses(rows, n, k, fewer):
    """Beyond its 32-bit offsets and numbers of tiles a product stays with the
    library, on both ways to it; a little below it is taken."""
    from rbg_amd import ops
    assert not ops._tile(rows, n, k) and not ops._tile_glu(rows, n, k)
    for glu in (False, True):
        assert not {2, 4} & set(ops.block_routes(rows, (n, k), (n, k), glu))
    assert ops._tile(*fewer) or ops._tile_glu(*fewer)


def test_switched_off_everything_is_the_librarys(monkeypatch):
    """Also after the same sizes were asked for with the switch on."""
    from rbg_amd import ops

    class Rows(torch.Tensor):
        is_cuda = True
    for rows, n, k in ((300, 16384, 2048), (2048, 4096, 14336), (64, 4096, 4096)):
        x, w = (torch.zeros(1, dtype=torch.bfloat16).expand(m, k)
                .as_subclass(Rows) for m in (rows, n))
        monkeypatch.setattr(ops, "_plain", lambda *a: True)
        monkeypatch.setattr(ops, "SKINNY_GEMM", 1)
        rules = ops._tile, ops._tile_glu
        assert any(ops._takes_tile(x, w, r) for r in rules) or \
            ops._takes_skinny(x, w, parts=True)
        assert any(ops.block_routes(rows, (n, k), (n, k), True))
        monkeypatch.setattr(ops, "SKINNY_GEMM", 0)
        assert not any(ops._takes_tile(x, w, r) for r in rules)
        assert not ops._takes_skinny(x, w, parts=True)
        assert not any(ops.block_routes(rows, (n, k), (n, k), True))


def test_wide_matrices_are_taken_with_any_k():
    """65 to 128 rows: no window between the sizes of common models."""
    from rbg_amd.ops import _tile
    for rows in (65, 96, 97, 128):
        for n in (12288, 13312, 14336):
            assert all(_tile(rows, n, k) for k in range(3584, 12289, 64))


def test_few_rows_of_gate_up_by_bounds():
    """Beyond a round's tiles but for a few, what is taken of some k and rows is
    taken of longer k and more rows; what tiles of 128 columns would need more than
    a round of is left."""
    from rbg_amd.ops import _tile_few
    for n in range(53312, 65537, 64):
        taken = [[_tile_few(rows, n, k) for k in (2048, 4096, 6144, 8192)]
                 for rows in (5, 32, 33, 64)]
        assert all(row == sorted(row) for row in taken)
        assert all(list(col) == sorted(col) for col in zip(*taken))
        assert taken[0][3] and taken[2][2]
    for n in (26688, 28672, 32768):
        assert not any(_tile_few(rows, n, k) for rows in range(5, 65)
                       for k in (2048, 4096, 6144, 8192))


# form, fewest stages of a part, whether with silu too: (7, 8), (5, 8), (5, 4), (3, 4),
# (4, 2) times 32 rows and rows of W
MORE_FORMS = [(8, 2, True), (9, 3, True), (10, 4, True), (11, 5, True),
              (12, 6, False)]


@pytest.mark.gpu
@pytest.mark.parametrize("form,stages,silu", MORE_FORMS)
@pytest.mark.parametrize("m,n,k", [
    (1, 64, 384), (95, 320, 448), (97, 192, 1024), (161, 1088, 832),
    (223, 576, 640), (225, 2176, 832), (449, 1600, 384)])
def test_more_forms(form, stages, silu, m, n, k):
    """As test_forms, around the rows of these tiles; parts of unequal length."""
    from rbg_amd import ops
    x, w, full, sums = _operands(m, n, k)
    for end in (PLAIN, PARTS, GLU) if silu else (PLAIN, PARTS):
        for parts in (1, 2, 3) if end == PARTS else (1,):
            if k // 64 // parts < stages:
                continue
            got = ops._hip.tile_form(x, w, end, form, parts, -1, 0)
            assert _near(got, end, full, sums), (end, parts)
    if not silu:
        with pytest.raises(RuntimeError):
            ops._hip.tile_form(x, w, GLU, form, 1, -1, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [
    (65, 1024, 2112), (113, 1984, 6144), (200, 16384, 1024), (257, 3904, 2048),
    (300, 6144, 4096), (700, 2048, 4096), (5000, 1024, 1024)])
def test_parts_route_of_other_sizes(m, n, k):
    """What the rule took up later; short k of many rows in bf16."""
    from rbg_amd import ops
    assert ops._tile(m, n, k)
    x, w, full, sums = _operands(m, n, k)
    got = ops.linear_parts(x, w)
    assert got.dim() == 2 or m <= 256 or k >= 5120
    assert _near(got, PARTS if got.dim() == 3 else PLAIN, full, sums)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [
    (65, 2048, 1536), (100, 11264, 2048), (70, 26624, 8192), (65, 57344, 8192),
    (321, 36864, 5120), (700, 4096, 4096), (2100, 2048, 1088)])
def test_swiglu_route_of_other_sizes(m, n, k):
    from rbg_amd import ops
    assert ops._tile_glu(m, n, k)
    assert ops.block_routes(m, (n, k), (n, k), True)[0] == 4
    x, w, full, sums = _operands(m, n, k)
    assert _near(ops.linear_swiglu(x, w), GLU, full, sums)


def test_rules_by_the_result():
    """Sums only for a norm that takes them; by the rows where the rules say so."""
    from rbg_amd.ops import _tile, _tile_glu
    for n in (1024, 2048, 6144, 16384):
        for k in (1024, 2048, 4096, 5120):
            taken = [_tile(rows, n, k) for rows in range(257, 2000, 13)]
            assert taken == sorted(taken) and taken[-1]
    assert not any(_tile(300, n, 8192) for n in (960, 16448, 28672))
    assert not _tile(200, 2048, 1536) and _tile(200, 2048, 1600)
    assert _tile(200, 2048, 2112) and not _tile(200, 2048, 2048)
    assert not _tile_glu(320, 36864, 5120) and not _tile_glu(384, 24576, 5120)
    assert not _tile_glu(300, 4096, 8192) and _tile_glu(2100, 4096, 8192)


@pytest.mark.parametrize("rows,n,k", [
    (163, 13312, 3584), (191, 14336, 4096), (257, 10880, 5376), (300, 13824, 5120),
    (313, 12288, 5120), (450, 9216, 5120), (600, 7168, 5120), (786, 6464, 16896),
    (797, 6528, 13824), (800, 5120, 5120), (800, 6144, 5120), (1050, 4096, 4992),
    (1112, 4608, 5504)])
def test_sums_of_these_are_not_rounded(rows, n, k):
    """A reader that adds up gets these products in f32 parts."""
    from rbg_amd import ops
    if ops._hip is None:
        pytest.skip("extension not built")
    assert ops._tile(rows, n, k) and ops._hip.tile_split(rows, n, k) > 1


def _in_f32_all_along(rows, n, k):
    """Sizes of more than 64 rows whose gate and up silu has always had unrounded."""
    if n < 8192 or k > n or k < 1024 or k % 64 or n % 64 or rows <= 64:
        return False
    if rows <= 128:
        return 24576 <= n <= 32768
    if k >= 3584 and n <= (16384 if rows <= 256 else 12288) and rows < 1000:
        return False
    return rows <= 256 or rows > 384 or n <= 16384


def test_gate_up_is_not_rounded_before_silu():
    """They go to the tiles with silu, or where the parts that linear_parts makes are
    sooner, to those."""
    from rbg_amd import ops
    if ops._hip is None:
        pytest.skip("extension not built")
    seen = [0, 0]
    for n in (*range(8192, 16385, 320), *range(16448, 65537, 2048), 24576, 28672,
              51200, 57344):
        for k in (*range(1024, 6000, 192), *range(6144, 20000, 1024), 8704):
            for rows in (65, 80, 99, 128, 129, 160, 200, 256, 257, 300, 384, 385,
                         450, 490, 512, 513, 600, 999, 1000, 2048):
                if _in_f32_all_along(rows, n, k) and ops._tile_fits(rows, n, k):
                    fused = ops._tile_glu(rows, n, k)
                    seen[fused] += 1
                    assert fused or (ops._route(rows, n, k, True) == 2 and
                                     ops._hip.tile_split(rows, n, k) > 1), \
                        (rows, n, k)
    assert min(seen) > 1000


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [
    (65, 24576, 4096), (99, 24576, 4096), (200, 22528, 5120), (155, 38912, 2112),
    (600, 12800, 8192), (210, 8192, 3008), (440, 14080, 9728), (330, 14336, 4608)])
def test_swiglu_by_unrounded_gates(m, n, k):
    from rbg_amd import ops
    assert ops.block_routes(m, (n, k), (n, k), True)[0] == (2 if m == 440 else 4)
    x, w, full, sums = _operands(m, n, k)
    assert _near(ops.linear_swiglu(x, w), GLU, full, sums)


@pytest.mark.parametrize("n,k,rows,taken", [
    (6144, 4096, (257, 270, 288), False), (6144, 4096, (256, 289, 300, 320), True),
    (6144, 2304, (264,), False), (6144, 4736, (270,), True), (5376, 4096, (270,), True),
    (6464, 4096, (270,), True), (10240, 4096, (257, 288), False),
    (10240, 4096, (289, 512), True), (4096, 4096, (321, 384), False),
    (4096, 4096, (320, 385), True), (3840, 4160, (365,), True),
    (12288, 4096, (321, 384), False), (12288, 4096, (320, 385), True),
    (3584, 4096, (513, 576), False), (9728, 4608, (513, 576), False),
    (9728, 4608, (512, 577), True)])
def test_whole_products_that_the_library_ends_sooner(n, k, rows, taken):
    """Of more than 256 rows and a k that is not split."""
    from rbg_amd import ops
    assert all(ops._tile(m, n, k) == taken for m in rows)


@pytest.mark.gpu
@pytest.mark.parametrize("form,stages,silu", MORE_FORMS)
def test_more_forms_for_the_rest(form, stages, silu):
    """Beginning at a column between, and before another form's columns."""
    from rbg_amd import ops
    x, w, full, sums = _operands(500, 2048, 512)
    for end in (PLAIN, GLU) if silu else (PLAIN,):
        for first, rest, to in ((0, form, 256), (0, form, 768), (form, 5, 512)):
            got = ops._hip.tile_form(x, w, end, first, 1, rest, to)
            assert _near(got, end, full, sums), (end, first, rest, to)


@pytest.mark.gpu
@pytest.mark.parametrize("form,stages,silu", MORE_FORMS)
def test_more_forms_many_tiles_a_workgroup(form, stages, silu):
    """As test_many_tiles_a_workgroup, with the fewest stages that they take, and sums
    of one part and of several."""
    from rbg_amd import ops
    x, w, full, sums = _operands(2100, 9280, 64 * max(stages, 4))
    for end in (PLAIN, PARTS, GLU) if silu else (PLAIN, PARTS):
        got = ops._hip.tile_form(x, w, end, form, 1, -1, 0)
        assert _near(got, end, full, sums), end
    x, w, full, sums = _operands(2100, 2112, 64 * stages * 4)
    got = ops._hip.tile_form(x, w, PARTS, form, 4, -1, 0)
    assert _near(got, PARTS, full, sums)


@pytest.mark.gpu
@pytest.mark.parametrize("form", [f for f, _, silu in MORE_FORMS if silu])
def test_more_forms_of_very_negative_gates(form):
    test_silu_of_very_negative_gates(form)
