"""Host-side planning rules that exist twice: the C++ runtime's (checked by
tests/native/geometry_contract_test.cpp) and their Python mirror in tatara_amd.stack,
which bench.py and the stub stack use.  The same figures are pinned here, so the two
cannot drift apart unnoticed."""
import pytest

from tatara_amd import stack as S


@pytest.mark.parametrize("visible,split,live", [
    ([32768] * 4, 1024, 256),                    # the headline wave
    ([32768], 256, 256),
    ([100000], 800, 250),
    ([16384] * 4, 512, 256),
    ([1], 128, 2),
    ([262144] * 16, 32768, 256),
    ([100000] * 4, 3136, 256),
    ([32768] * 3, 800, 246),                     # 768 keys would be 258 workgroups
    ([32768, 30000, 24576, 8192], 768, 252),     # config 3's ragged lanes
    ([65536, 50001, 40001, 30001, 20001, 10001, 5001, 1001], 1792, 254),
    ([], 128, 0),
])
def test_split_keys_rule_matches_the_runtime(visible, split, live):
    assert S.choose_split_keys(visible) == split
    assert S.split_workgroups(visible, split) == live
    assert split % 32 == 0 and split >= 128
    assert live <= 256


def test_split_keys_rule_never_oversubscribes():
    """Whatever the depths, the workgroups that hold keys fit the compute units (the
    measured cost of one too many is a third of the walk), and one notch finer would not."""
    import random
    rng = random.Random(0x5EED)
    for _ in range(300):
        lanes = rng.randint(1, 16)
        visible = [rng.randint(257, 262144) for _ in range(lanes)]
        for units in (256, 304, 64):
            split = S.choose_split_keys(visible, units)
            assert S.split_workgroups(visible, split) <= units
            if split > 128:
                share = -(-2 * sum(visible) // units)
                assert split - 32 < share or S.split_workgroups(visible, split - 32) > units


@pytest.mark.parametrize("rows,units,splits,scratch", [
    (2048, 256, 2, 512 + 128 * 2 * 270336), (1024, 256, 4, 256 + 64 * 4 * 270336),
    (512, 256, 8, 256 + 32 * 8 * 270336), (256, 256, 8, 256 + 16 * 8 * 270336),
    (13, 256, 8, 256 + 2 * 8 * 270336), (4096, 256, 1, 0), (16384, 256, 1, 0),
    (2048, 304, 2, 512 + 128 * 2 * 270336), (2048, 128, 1, 0), (2049, 256, 1, 0), (0, 256, 1, 0)])
def test_flash_prefill_sharing_plan(rows, units, splits, scratch):
    """tt_flash_prefill_splits: as many workgroups per position tile (32 rows x 2 kv heads) as fit
    the compute units, between one and eight; tt_flash_prefill_scratch_bytes: a 4-byte arrival
    count per tile and kv head, padded to 256 bytes, and 270,336 bytes per sharer - 32 f32x4 of O
    and one of {reference, row sum} for each of 512 lanes."""
    from tatara_amd import backend as B
    assert B.flash_prefill_splits(rows, 32768, units) == splits
    assert B.flash_prefill_splits(rows, 480, units) == 1     # a longest walk under 16 key tiles
    assert B.flash_prefill_splits(rows, 481, units) == splits
    assert B.flash_prefill_scratch_bytes(rows, splits) == scratch
    assert B.flash_prefill_scratch_bytes(rows, 1) == 0


# (tile, rows, in_dim, out_dim) of the dense_bf16 blocks that tests/test_gpu_stack.py runs: every tile
# with fewer units of 64 columns than its ring holds, as many and more (256 x 256 is not taken for two
# units or less), at remainders of rows and outputs and at output rows that are not 8-byte aligned.  None of
# them is launched as another shape that fills the rounds better; those have cases of their own below.
DENSE_TILE_CASES = [(tile, rows, in_dim, out_dim) for tile, rows, out_dim in [
    ("256x256", 3073, 4095), ("128x128", 641, 6141), ("128x128-deep", 129, 12350), ("128x64", 65, 12350),
    ("64x64", 33, 9213), ("32x64", 17, 61)]
    for in_dim in (64, 128, 192, 256) if tile != "256x256" or in_dim > 128] + [
    ("256x256", 1021, 2048, 12349), ("128x128", 2049, 192, 12352), ("256x256", 7937, 4096, 2046),
    ("128x128", 500, 2048, 9213), ("128x128", 500, 2048, 9216), ("128x128-deep", 2047, 4096, 2045),
    ("128x64", 777, 4096, 2046), ("128x64", 100, 2048, 12352), ("64x64", 129, 256, 9216),
    ("64x64", 129, 2048, 9213), ("32x64", 66, 2048, 515), ("32x64", 100, 64, 4096)]


def tile_shape(tile):
    return tuple(int(side) for side in tile.removesuffix("-deep").split("x"))


@pytest.mark.parametrize("tile,rows,in_dim,out_dim", DENSE_TILE_CASES, ids=lambda v: str(v))
def test_block_tile_of_the_cases(tile, rows, in_dim, out_dim):
    """The rule still gives the cases the tiles they are there for, and launches them: a change of
    its figures that left a tile without a case fails here."""
    from tatara_amd import backend as B
    assert B.block_product_tile(rows, in_dim, out_dim, 256) == tile
    assert B.block_product_shape(rows, in_dim, out_dim, 256) == tile_shape(tile)


# Rows of the 4-bit blocks that tests/test_gpu_q4_project.py holds to 64-bit sums, and the way each goes by family.
Q4_SHAPES = {"gdn": (2048, 12352), "attn": (2048, 9216), "out": (4096, 2048)}
Q4_WIDE_RANGE_ROWS = [17, 63, 65, 129, 511, 8193]
Q4_SHORT_ROWS = [32, 33, 64, 66, 96, 97, 128, 130, 200, 385, 420]
Q4_UNFOLDED_ROWS = [350, 777, 1057, 2047, 4500, 5450]


def test_every_block_tile_has_cases():
    """What is launched, of bf16 and of f16 operands: every tile and every height of the rows that are multiplied
    with weights unpacked in the product.  (The f16 32 x 64 is launched for slices of a queue with little
    workspace only, and tested there.)"""
    from tatara_amd import backend as B
    assert {case[0] for case in DENSE_TILE_CASES} == set(B.BLOCK_TILES)
    assert {case[0] for case in REFINED_TILE_CASES} == {tile_shape(tile) for tile in B.REFINED_TILES}
    taken = {name: {B.q4_block_tile(rows, *shape, 256)
                    for rows in Q4_WIDE_RANGE_ROWS + Q4_SHORT_ROWS + Q4_UNFOLDED_ROWS}
             for name, shape in Q4_SHAPES.items()}
    short = {"short-32", "short-64", "short-96"}
    assert taken["gdn"] >= short | {"short-128"} and taken["attn"] >= short | {"short-128"}
    assert {tile for tile in taken["out"] if tile.startswith("short")} == short
    assert set.union(*taken.values()) - short - {"short-128"} == set(B.BLOCK_TILES + B.REFINED_TILES) - {"32x64"}


@pytest.mark.parametrize("rows,in_dim,out_dim,tile", [
    (16384, 2048, 9216, "256x256"), (16384, 2048, 12352, "256x256"), (8192, 4096, 2048, "256x256"),
    (5500, 4096, 2048, "256x256"),      # 176 tiles: idle compute units make the others faster
    (4050, 2048, 12352, "128x128"), (5450, 2176, 9216, "128x128"),   # just over three rounds of 256 x 256
    (3000, 2176, 12352, "256x256"), (10300, 4096, 2048, "128x128"),
    (4102, 4096, 2048, "256x256"),
    (4096, 2048, 9216, "128x128"), (2048, 2048, 9216, "128x128"), (2048, 4096, 2048, "128x128-deep"),
    (100, 2048, 12352, "128x64"), (300, 4096, 2048, "64x64"), (100, 4096, 2048, "32x64")])
def test_block_tile_where_it_was_measured(rows, in_dim, out_dim, tile):
    """The fastest of the six tiles at sizes where all of them were timed on 256 compute units (some of
    which are launched as a shape that fills the rounds better still); and a tile for any number of
    compute units."""
    from tatara_amd import backend as B
    assert B.block_product_tile(rows, in_dim, out_dim, 256) == tile
    for units in (0, 1, 64, 304):
        assert B.block_product_tile(rows, in_dim, out_dim, units) in B.BLOCK_TILES


# (shape, rows, in_dim, out_dim) of the dense_bf16 blocks that tests/test_gpu_stack.py runs on the tiles
# that fill the rounds better: one and two rounds, remainders of rows and outputs, an odd number of
# units, output rows that are not 8-byte aligned.
REFINED_TILE_CASES = [
    ((256, 288), 2048, 2048, 9216), ((256, 288), 2047, 1088, 9213),
    ((224, 256), 1000, 1024, 12349), ((224, 256), 2049, 2048, 12352), ((224, 256), 3000, 2048, 9214),
    ((160, 256), 777, 1088, 12350), ((160, 256), 790, 2048, 11000), ((160, 256), 1590, 1024, 12352)]


@pytest.mark.parametrize("shape,rows,in_dim,out_dim", REFINED_TILE_CASES, ids=lambda v: str(v))
def test_refined_shape_of_the_cases(shape, rows, in_dim, out_dim):
    from tatara_amd import backend as B
    assert B.block_product_shape(rows, in_dim, out_dim, 256) == shape
    for units in (0, 1, 64, 304):
        assert B.block_product_shape(rows, in_dim, out_dim, units)[0] in (32, 64, 128, 160, 224, 256)


@pytest.mark.parametrize("rows,in_dim,out_dim,shape", [
    (16384, 2048, 12352, (256, 256)), (100, 2048, 12352, (128, 64)), (2048, 4096, 2048, (128, 128)),
    (640, 960, 12352, (128, 128)),       # under 1024 columns the six tiles only
    # a shorter estimate of 224 x 256 that did not hold: one round over a long K, few columns
    (5150, 4096, 2048, (256, 256)), (2401, 5120, 4294, (256, 256)), (6000, 4096, 2048, (256, 256)),
    (1647, 1152, 7237, (128, 128)), (2095, 1088, 5501, (128, 128)),
])
def test_shape_is_the_basic_tile_where_no_other_fills_better(rows, in_dim, out_dim, shape):
    from tatara_amd import backend as B
    assert B.block_product_shape(rows, in_dim, out_dim, 256) == shape


# ((whole rounds, last round) in runs, rows, in_dim, out_dim): one round of a lower band, one of tiles in order of
# the workgroups, of whole bands, rounds of which the last one goes by number and in runs.
DEALT_CASES = [
    ((True, True), 777, 1088, 12350), ((False, False), 776, 256, 1119), ((True, False), 1000, 64, 4096),
    ((True, False), 20000, 64, 900), ((True, True), 300, 256, 12349)]


@pytest.mark.parametrize("runs,rows,in_dim,out_dim", DEALT_CASES + [
    # measured either way: narrow and short products were up to 9 % slower in runs, wide and low ones up to 25 % without
    ((True, True), 777, 2048, 12352), ((True, True), 1000, 2048, 9216), ((True, True), 300, 2048, 12352),
    ((True, True), 2500, 2048, 9216), ((False, False), 3380, 960, 1083), ((False, False), 11448, 640, 533),
    ((False, False), 7210, 3392, 756), ((False, False), 4431, 3776, 104), ((False, False), 17, 3648, 17),
    ((True, True), 956, 2304, 572), ((True, True), 331, 64, 8988), ((False, False), 3144, 1408, 1189)],
    ids=lambda v: str(v))
def test_rounds_dealt_in_runs(runs, rows, in_dim, out_dim):
    from tatara_amd import backend as B
    assert B.block_product_runs(rows, in_dim, out_dim, 256) == runs
    for units in (0, 1, 64, 304):
        assert isinstance(B.block_product_runs(rows, in_dim, out_dim, units), tuple)


@pytest.mark.parametrize("family,rows,tile", [
    ("gdn", 17, "short-32"), ("gdn", 64, "short-64"), ("gdn", 96, "short-96"), ("gdn", 256, "short-128"),
    ("gdn", 384, "short-64"), ("gdn", 385, "128x128"), ("gdn", 448, "128x128"), ("gdn", 777, "160x256"),
    ("attn", 320, "short-64"), ("attn", 400, "short-64"), ("attn", 480, "short-96"), ("attn", 512, "short-64"),
    ("attn", 513, "128x128"), ("attn", 2048, "256x288"), ("out", 128, "short-32"), ("out", 256, "short-64"),
    ("out", 384, "short-96"), ("out", 385, "64x64"), ("out", 8193, "256x256"), ("out", 5450, "224x256")])
def test_q4_block_route_where_it_was_measured(family, rows, tile):
    """4-bit blocks: weights unpacked in the product where that was faster on 256 compute units (GDN
    projections up to 384 rows, attention projections up to 512, where 321 to 384 take as long either way,
    output projections up to 384), and a tile for any number of compute units."""
    from tatara_amd import backend as B
    assert B.q4_block_tile(rows, *Q4_SHAPES[family], 256) == tile
    for units in (0, 1, 64, 304):
        assert isinstance(B.q4_block_tile(rows, *Q4_SHAPES[family], units), str)
