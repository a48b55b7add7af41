"""Pure-function pins for the decode launch policies: hipGraph batch
bucketing and the XCD-filling split-KV heuristic.  Both are graph-safety
contracts — they must depend only on (padded batch, config), never on
per-step tensor values — and the split policy encodes a measured optimum
(~1024 workgroups fills 256 CUs / 8 XCDs; profiles/decode_breakdown.md
r59 sweep), so a regression here silently costs decode bandwidth."""
import pytest

from rbg_amd.engine.model_runner import GRAPH_BATCH_SIZES
from rbg_amd.ops import pick_decode_splits


def test_graph_buckets_cover_and_round_up():
    # monotone ascending, 1..256: every batch <= 256 has a bucket >= it
    assert list(GRAPH_BATCH_SIZES) == sorted(set(GRAPH_BATCH_SIZES))
    assert GRAPH_BATCH_SIZES[0] == 1 and GRAPH_BATCH_SIZES[-1] == 256

    def bucket(n):
        for b in GRAPH_BATCH_SIZES:
            if n <= b:
                return b
        return GRAPH_BATCH_SIZES[-1]

    for n in range(1, 257):
        assert bucket(n) >= n
        assert bucket(n) in GRAPH_BATCH_SIZES
    assert bucket(300) == 256          # oversize clamps to the last bucket
    assert bucket(128) == 128          # exact sizes map to themselves


def test_split_policy_targets_chip_fill():
    kv_heads, ctx = 8, 2048
    # measured optima from the r59 sweep (v4 packs 2 seqs/WG):
    # B128 -> 1024 base WGs at splits=2; B64 -> splits=4
    assert pick_decode_splits(128, kv_heads, ctx, variant=4) == 2
    assert pick_decode_splits(64, kv_heads, ctx, variant=4) == 4
    # a huge batch already fills the chip: no split-KV overhead
    assert pick_decode_splits(512, kv_heads, ctx, variant=4) == 1
    # splits never exceed what the context can feed (>= one page pair
    # per split) nor the hard cap of 16
    assert pick_decode_splits(1, kv_heads, 64, variant=4) <= 2
    for bs in (1, 2, 7, 64, 128, 256):
        s = pick_decode_splits(bs, kv_heads, ctx, variant=4)
        assert 1 <= s <= 16


def test_split_policy_is_batch_deterministic():
    """Graph safety: same (batch, config) -> same splits, always."""
    a = [pick_decode_splits(b, 8, 4096, variant=4) for b in range(1, 129)]
    b = [pick_decode_splits(b, 8, 4096, variant=4) for b in range(1, 129)]
    assert a == b


def test_prefill_plan_covers_every_row():
    """Every block of rows once, whatever the order."""
    import torch

    from rbg_amd import ops
    cu, cu_k = [0, 5, 5, 300, 301], [0, 105, 110, 405, 1406]
    for heads, kvh in ((32, 8), (6, 2), (8, 8)):
        tokens = 128 // (heads // kvh)
        plan = ops.prefill_plan(cu, cu_k, heads, kvh, "cpu")
        got = sorted(map(tuple, torch.cat(
            [plan.blocks, plan.lens[:, None]], 1).tolist()))
        want = sorted(
            (cu[b], i, cu_k[b], cu_k[b + 1] - cu_k[b] - cu[b + 1] + cu[b],
             cu_k[b + 1] - cu_k[b])
            for b in range(4)
            for i in range(-(-(cu[b + 1] - cu[b]) // tokens)))
        assert got == want


@pytest.mark.parametrize("kvh", [1, 3, 4, 8, 40])
def test_cut_prefill_covers_every_tile(kvh):
    """Of a block that is cut every tile of keys once, its parts in order and
    numbered in a row; few enough for a bounded workspace; some blocks are cut
    and some whole."""
    import random

    from rbg_amd import ops
    rng = random.Random(kvh)
    cut = 0
    for _ in range(200):
        n = rng.randint(1, 12)
        rows = [int(2 ** rng.uniform(0, 11)) for _ in range(n)]
        pasts = [rng.choice([0, -min(3, r - 1), int(2 ** rng.uniform(0, 14))])
                 for r in rows]
        cu, cu_k = [0], [0]
        for r, p in zip(rows, pasts):
            cu.append(cu[-1] + r)
            cu_k.append(cu_k[-1] + r + p)
        group = rng.choice([1, 3, 4, 8, 128])
        plan = ops.prefill_plan(cu, cu_k, kvh * group, kvh, "cpu")
        if plan.items is None:
            continue
        cut += 1
        assert plan.parts * kvh <= 768          # 64 KB of sums each
        pieces = {}
        for b, begin, end, part in sorted(plan.items.tolist()):
            pieces.setdefault(b, []).append((begin, end, part))
        joins = {b: list(range(first, first + count))
                 for b, first, count in plan.joins.tolist()}
        assert sorted(sum(joins.values(), [])) == list(range(plan.parts))
        for b, ((_, nth, _, past), keys) in enumerate(
                zip(plan.blocks.tolist(), plan.lens.tolist())):
            need = min(past + (nth + 1) * (128 // group), keys)
            ends = [0] + [p[1] for p in pieces[b]]
            assert ends[-1] == max(-(-need // 64), 0)
            assert [p[0] for p in pieces[b]] == ends[:-1]
            assert [p[2] for p in pieces[b]] == joins.get(b, [-1])
    assert cut > 5


def test_default_parts_are_bounded():
    """Of the default form: no more for a longer table than fill the chip, and
    so a bounded workspace; about as many for one sequence more."""
    for kvh in (1, 2, 4, 8, 16):
        for bs in GRAPH_BATCH_SIZES + (49,):
            counts = [pick_decode_splits(bs, kvh, c, variant=7)
                      for c in (64, 2048, 8192, 40960, 131072, 1 << 20)]
            assert counts == sorted(counts) and counts[0] == 1
            assert counts[-1] <= 32
            # a head's sums are 128 floats; groups of 8
            assert counts[-1] * bs * kvh * 8 * 512 <= 32 << 20
    for cap in (8192, 40960, 131072):
        counts = [pick_decode_splits(b, 8, cap, variant=7)
                  for b in range(1, 257)]
        assert all(b >= a / 2 and a >= b / 2
                   for a, b in zip(counts, counts[1:]))


def test_parts_of_other_pages():
    """Only pages of 16 have the form whose parts many pairs gain by."""
    for cap in (8192, 131072):
        for bs in (64, 128, 256):
            assert pick_decode_splits(bs, 8, cap, variant=7, page_size=32) == \
                pick_decode_splits(bs, 8, cap, variant=4)
        for bs in (1, 8, 48):
            assert pick_decode_splits(bs, 8, cap, variant=7, page_size=32) == \
                pick_decode_splits(bs, 8, cap, variant=7)


def test_silu_in_the_product_fits_its_kernel():
    """What the rule hands to the decode GEMM with silu is what it takes."""
    from rbg_amd.ops import _glu
    taken = 0
    for n in (32, 64, 96, 1024, 4096, 10240, 12288, 12320, 14336, 18432, 51200):
        for k in (256, 512, 1000, 2048, 2560, 4096, 8192):
            for rows in (0, 1, 2, 4, 5, 16, 17, 32, 33, 64, 65):
                glu = _glu(rows, n, k)
                assert not glu or 1 <= rows <= 64
                assert not glu or n % 64 == 0 and k % 512 == 0
                taken += glu
    assert taken > 100


def test_decode_products_fit_their_kernels():
    """What the rules hand to the decode GEMM is what it takes, and a reader of
    parts gets them wherever a sum is worth its launch."""
    from rbg_amd.ops import _skinny
    sizes = (32, 64, 96, 1000, 1024, 2048, 4096, 5120, 10240, 10272, 12288,
             12320, 14336, 16384, 24576, 32768, 40960, 51200, 128256)
    taken = 0
    for n in sizes:
        for k in (256, 512, 1000, 2048, 2560, 4096, 8192, 12288, 25600):
            for rows in (0, 1, 2, 4, 5, 16, 17, 32, 33, 64, 65, 128, 129, 192,
                         256, 257):
                own = _skinny(rows, n, k)
                assert not own or 1 <= rows <= 256
                assert not own or n % 32 == 0 and k % 512 == 0
                if own and n <= 10240 and k > 2048 and rows <= 128:
                    assert _skinny(rows, n, k, parts=True)
                taken += own
    assert taken > 500
