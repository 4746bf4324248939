"""Affine 4-bit projections either side of the attention family on the GPU, through
the C ABI, against the CPU checker (itself bit-equal to the reference's
q4_dot_reference).

Decode operators (`*_project`, `*_project_ms{,_v2}`, `gdn_outproj{,_ms,_ms_v2}`) keep the
reference's sequence of operations, so every bf16 output must be the checker's bit
pattern.  The block operators (`*_blk`) are held to the path's bar (max-abs 2e-2,
mean-abs 2e-3) with a 2-step allowance on large values: their sums run in another
order."""
import numpy as np
import pytest

import oracle_lib as ol
from gpu_util import check_bf16, gpu, run
from test_host_rules import Q4_SHORT_ROWS, Q4_UNFOLDED_ROWS, Q4_WIDE_RANGE_ROWS

pytestmark = pytest.mark.gpu
o = ol.oracle

ATTN = {"name": "attn_project", "segments": [8192, 512, 512], "k": 2048, "out": 10, "threads": 128}
GDN = {"name": "gdn_project", "segments": [8192, 4096, 32, 32], "k": 2048, "out": 13, "threads": 128}
OUT = {"name": "gdn_outproj", "segments": [2048], "k": 4096, "out": 4, "threads": 64}


def _matrix(seed, rows, k):
    rng = np.random.default_rng(seed)
    words = rng.integers(0, 2 ** 32, rows * k // 8, dtype=np.uint64).astype(np.uint32)
    scales = ol.f32_to_bf16(rng.uniform(0.002, 0.01, rows * k // 64).astype(np.float32))
    biases = ol.f32_to_bf16((-7.5 * ol.bf16_to_f32(scales) +
                             rng.normal(0.0, 1e-3, scales.size)).astype(np.float32))
    return words, scales, biases


def _family(dev, family, seed):
    host, device = [], {}
    for index, rows in enumerate(family["segments"]):
        w, s, b = _matrix(seed + index, rows, family["k"])
        host.append((w, s, b))
        slot = 1 + 3 * index
        device[slot], device[slot + 1], device[slot + 2] = (dev.buffer_from(w), dev.buffer_from(s),
                                                            dev.buffer_from(b))
    return host, device


def _groups(family):
    per = family["threads"] // 32
    return (sum(family["segments"]) + per - 1) // per


def _expected(family, host, x, rows, out_stride=None):
    total = sum(family["segments"])
    stride = out_stride or total
    want = np.zeros(rows * stride, np.uint16)
    first = 0
    for (w, s, b), n in zip(host, family["segments"]):
        o.tto_q4_project(x, family["k"], rows, w, s, b, family["k"], n, want[first:], stride, 8)
        first += n
    return want


@pytest.mark.parametrize("family", [ATTN, GDN, OUT], ids=lambda f: f["name"])
def test_single_row_projection_bit_for_bit(family):
    print(f"[case] {family['name']} one row", flush=True)
    B, dev, queue, lib = gpu()
    host, bindings = _family(dev, family, 0x9000)
    x = ol.gaussian_bf16(0x9100, family["k"], 0.0, 1.0)
    total = sum(family["segments"])
    out = dev.create_buffer(total * 2)
    bindings[0] = dev.buffer_from(x)
    bindings[family["out"]] = out
    ms = run(lambda cb: cb.encode(lib.pipeline(family["name"]), bindings, {}, (_groups(family), 1, 1),
                                  (family["threads"], 1, 1)))
    assert np.array_equal(out.read(np.uint16), _expected(family, host, x, 1))
    print(f"[time] {family['name']}: {ms * 1e3:.1f} us", flush=True)


@pytest.mark.parametrize("rows,tile", [(1, 16), (3, 1), (3, 2), (16, 16), (13, 5)])
@pytest.mark.parametrize("family,suffix", [(ATTN, "_ms"), (ATTN, "_ms_v2"), (GDN, "_ms"),
                                           (GDN, "_ms_v2"), (OUT, "_ms"), (OUT, "_ms_v2")],
                         ids=["attn", "attn_v2", "gdn", "gdn_v2", "out", "out_v2"])
def test_wave_projection_bit_for_bit(family, suffix, rows, tile):
    name = family["name"] + suffix
    print(f"[case] {name} rows={rows} tile={tile}", flush=True)
    B, dev, queue, lib = gpu()
    host, bindings = _family(dev, family, 0x9200)
    x = ol.gaussian_bf16(0x9300 + rows, rows * family["k"], 0.0, 1.0)
    total = sum(family["segments"])
    strided = family is OUT
    stride = total + 64 if strided else total
    out = dev.buffer_from(np.full(rows * stride, 0x7FC0, np.uint16))
    bindings[0] = dev.buffer_from(x)
    bindings[family["out"]] = out
    slot = family["out"] + 1
    constants = {slot: rows, slot + 1: stride, slot + 2: tile} if strided else {slot: rows, slot + 1: tile}
    tiles = (rows + tile - 1) // tile
    ms = run(lambda cb: cb.encode(lib.pipeline(name), bindings, constants, (_groups(family), tiles, 1),
                                  (family["threads"], 1, 1)))
    got = out.read(np.uint16).reshape(rows, stride)
    want = _expected(family, host, x, rows, stride).reshape(rows, stride)
    assert np.array_equal(got[:, :total], want[:, :total])
    assert np.all(got[:, total:] == 0x7FC0)
    print(f"[time] {name} rows={rows} tile={tile}: {ms * 1e3:.1f} us", flush=True)


def test_wave_projection_of_every_small_bf16_input_bit_for_bit():
    """attn_project_ms on inputs that run through every bf16 bit pattern below 2^30 in
    magnitude (the subnormals among them), ordered by magnitude so that a row of 2048 holds
    neighbouring binades: what the reference's model does with subnormal inputs, products
    and sums (q4_dot_reference), bit for bit."""
    print("[case] attn_project_ms over every bf16 input below 2^30", flush=True)
    B, dev, queue, lib = gpu()
    family = ATTN
    host, bindings = _family(dev, family, 0x9800)
    patterns = np.arange(65536, dtype=np.uint32).astype(np.uint16)
    small = patterns[(patterns & 0x7FFF) < 0x4E80]
    small = small[np.argsort(small & 0x7FFF, kind="stable")]
    rows = 16
    x = np.resize(small, rows * family["k"])            # 32768 values: the 32768 smallest magnitudes
    assert x.size <= small.size
    total = sum(family["segments"])
    out = dev.create_buffer(rows * total * 2)
    bindings[0] = dev.buffer_from(x)
    bindings[family["out"]] = out
    slot = family["out"] + 1
    run(lambda cb: cb.encode(lib.pipeline("attn_project_ms"), bindings, {slot: rows, slot + 1: 16},
                             (_groups(family), 1, 1), (family["threads"], 1, 1)))
    got = out.read(np.uint16)
    want = _expected(family, host, x, rows)
    differ = np.flatnonzero(got != want)
    assert differ.size == 0, (f"{differ.size} of {got.size} outputs differ, first: row "
                              f"{differ[0] // total} got {got[differ[0]]:#06x} want {want[differ[0]]:#06x}")


@pytest.mark.parametrize("rows", [1, 2, 4, 13, 16])
@pytest.mark.parametrize("family", [ATTN, GDN, OUT], ids=lambda f: f["name"])
def test_wave_projection_on_the_matrix_unit(family, rows):
    """The _mfma_ms forms (no reference counterpart): the bindings and grids of the _ms forms,
    sums in another order - held to the path's bar, with the share of bit-identical outputs
    printed."""
    name = family["name"] + "_mfma_ms"
    print(f"[case] {name} rows={rows}", flush=True)
    B, dev, queue, lib = gpu()
    host, bindings = _family(dev, family, 0x9800)
    x = ol.gaussian_bf16(0x9900 + rows, rows * family["k"], 0.0, 1.0)
    total = sum(family["segments"])
    strided = family is OUT
    stride = total + 64 if strided else total
    out = dev.buffer_from(np.full(rows * stride, 0x7FC0, np.uint16))
    bindings[0] = dev.buffer_from(x)
    bindings[family["out"]] = out
    slot = family["out"] + 1
    constants = {slot: rows, slot + 1: stride, slot + 2: 16} if strided else {slot: rows, slot + 1: 16}
    ms = run(lambda cb: cb.encode(lib.pipeline(name), bindings, constants, (_groups(family), 1, 1),
                                  (family["threads"], 1, 1)))
    got = out.read(np.uint16).reshape(rows, stride)
    want = _expected(family, host, x, rows, stride).reshape(rows, stride)
    check_bf16(got[:, :total], want[:, :total], name, ulps=2)
    assert np.all(got[:, total:] == 0x7FC0)
    print(f"[time] {name} rows={rows}: {ms * 1e3:.1f} us", flush=True)


@pytest.mark.parametrize("family,name", [(ATTN, "attn_project_blk"), (GDN, "gdn_project_blk"),
                                         (OUT, "outproj_blk")], ids=["attn", "gdn", "out"])
@pytest.mark.parametrize("rows", [1, 37, 130])
def test_block_projection(family, name, rows):
    print(f"[case] {name} rows={rows}", flush=True)
    B, dev, queue, lib = gpu()
    host, bindings = _family(dev, family, 0x9400)
    x = ol.gaussian_bf16(0x9500 + rows, rows * family["k"], 0.0, 1.0)
    total = sum(family["segments"])
    out = dev.create_buffer(rows * total * 2)
    bindings[0] = dev.buffer_from(x)
    bindings[family["out"]] = out
    slot = family["out"] + 1
    constants = {slot: rows, slot + 1: family["k"]} if family is OUT else {slot: rows}
    ms = run(lambda cb: cb.encode(lib.pipeline(name), bindings, constants, (_groups(family), 1, 1),
                                  (family["threads"], 1, 1)))
    check_bf16(out.read(np.uint16), _expected(family, host, x, rows), name, ulps=2)
    print(f"[time] {name} rows={rows}: {ms * 1e3:.1f} us", flush=True)


@pytest.mark.parametrize("family,name", [(ATTN, "attn_project_blk"), (GDN, "gdn_project_blk"),
                                         (OUT, "outproj_blk")], ids=["attn", "gdn", "out"])
@pytest.mark.parametrize("rows", [256, 257, 700, 2048, 16384])
def test_block_projection_over_several_row_tiles(family, name, rows):
    """Blocks that span more than one tile of rows, up to the 16384 rows the benchmark times,
    among them the reference's 2048-row block, whose last round of tiles is partly filled (as that
    of most sizes here is): every output row is produced, and a sample of rows - the first and last of the block, the rows either
    side of each tile boundary sampled, a few inside - is held to the checker."""
    print(f"[case] {name} rows={rows} (sampled rows)", flush=True)
    B, dev, queue, lib = gpu()
    host, bindings = _family(dev, family, 0x9600)
    k = family["k"]
    x = ol.gaussian_bf16(0x9700 + rows, rows * k, 0.0, 1.0)
    total = sum(family["segments"])
    out = dev.buffer_from(np.full(rows * total, 0x7FC0, np.uint16))      # NaN until written
    bindings[0] = dev.buffer_from(x)
    bindings[family["out"]] = out
    slot = family["out"] + 1
    constants = {slot: rows, slot + 1: k} if family is OUT else {slot: rows}
    run(lambda cb: cb.encode(lib.pipeline(name), bindings, constants, (_groups(family), 1, 1),
                             (family["threads"], 1, 1)))
    got = out.read(np.uint16).reshape(rows, total)
    assert not np.any((got & 0x7FFF) > 0x7F80), "an output row was left unwritten"
    sample = {0, rows - 1, rows // 2, rows // 3}
    for edge in range(256, rows, 256 if rows <= 1024 else 4096):
        sample.update({edge - 1, edge})
    sample = sorted(r for r in sample if 0 <= r < rows)
    xs = np.ascontiguousarray(x.reshape(rows, k)[sample]).reshape(-1)
    want = _expected(family, host, xs, len(sample)).reshape(len(sample), total)
    check_bf16(got[sample], want, f"{name} rows {sample[:4]}..{sample[-1]}", ulps=2)


@pytest.mark.parametrize("family,name", [(ATTN, "attn_project_blk"), (GDN, "gdn_project_blk"),
                                         (OUT, "outproj_blk")], ids=["attn", "gdn", "out"])
@pytest.mark.parametrize("rows", Q4_WIDE_RANGE_ROWS)
def test_block_projection_against_64_bit_sums_over_the_whole_range(family, name, rows):
    """Rows either side of the tile heights a block is launched with, and of the 8192 rows the
    out-projection takes at a time, over inputs and weights of all magnitudes: rows of 2^-100 to
    2^100 with a value 2^12 times the others in every 64 columns, a row of zeros, matrices whose
    groups differ by 2^8 and whose rows by 2^40.  The terms that are summed are exact in fp32 to
    2^-24 of their group's largest, so an output may differ from the 64-bit sum by half a bf16
    step (2^-9, doubled to 2^-8 at a binade's lower end) and 2^-20 of the sum of magnitudes."""
    print(f"[case] {name} rows={rows} whole range", flush=True)
    B, dev, queue, lib = gpu()
    rng = np.random.default_rng(rows)
    k, total = family["k"], sum(family["segments"])
    x = rng.standard_normal((rows, k), dtype=np.float32)
    x[:, ::64] *= 4096.0
    x = ol.f32_to_bf16((x * np.exp2(rng.integers(-100, 60, (rows, 1))).astype(np.float32)).reshape(-1))
    x = x.reshape(rows, k)
    x[rows // 2] = 0
    bindings, host = {0: dev.buffer_from(x.reshape(-1))}, []
    for index, n in enumerate(family["segments"]):
        words = rng.integers(0, 2 ** 32, n * k // 8, dtype=np.uint64).astype(np.uint32)
        scale = rng.uniform(0.5, 1.0, (n, k // 64)) * np.exp2(rng.integers(-8, 1, (n, k // 64)))
        scale *= np.exp2(rng.integers(-40, 1, (n, 1)))
        scales = ol.f32_to_bf16(scale.astype(np.float32).reshape(-1))
        biases = ol.f32_to_bf16((scale * rng.uniform(-8.0, 0.5, scale.shape)).astype(np.float32).reshape(-1))
        slot = 1 + 3 * index
        bindings.update({slot: dev.buffer_from(words), slot + 1: dev.buffer_from(scales),
                         slot + 2: dev.buffer_from(biases)})
        host.append((words, scales, biases))
    out = dev.buffer_from(np.full(rows * total, 0x7FC0, np.uint16))      # NaN until written
    bindings[family["out"]] = out
    slot = family["out"] + 1
    constants = {slot: rows, slot + 1: k} if family is OUT else {slot: rows}
    run(lambda cb: cb.encode(lib.pipeline(name), bindings, constants, (_groups(family), 1, 1),
                             (family["threads"], 1, 1)))
    got = ol.bf16_to_f32(out.read(np.uint16)).reshape(rows, total).astype(np.float64)
    assert np.isfinite(got).all()
    sample = sorted({0, 15, 16, rows // 2, rows - 2, rows - 1} | {r for r in (63, 64, 127, 128, 8191)
                                                                  if r < rows})
    xs = ol.bf16_to_f32(x[sample].reshape(-1)).reshape(len(sample), k).astype(np.float64)
    first = 0
    for words, scales, biases in host:
        n = len(words) * 8 // k
        nibbles = (words[:, None] >> (4 * np.arange(8, dtype=np.uint32))[None, :]) & 15
        widened = [np.repeat(ol.bf16_to_f32(v).reshape(n, k // 64), 64, axis=1).astype(np.float64)
                   for v in (scales, biases)]
        weights = widened[0] * nibbles.reshape(n, k) + widened[1]
        want, magnitudes = xs @ weights.T, np.abs(xs) @ np.abs(weights).T
        error = np.abs(got[sample, first:first + n] - want)
        bar = np.abs(want) * 2.0 ** -8 + magnitudes * 2.0 ** -20 + 2.0 ** -126
        assert (error <= bar).all(), np.argwhere(error > bar)[:4]
        first += n


@pytest.mark.parametrize("family,name", [(ATTN, "attn_project_blk"), (GDN, "gdn_project_blk"),
                                         (OUT, "outproj_blk")], ids=["attn", "gdn", "out"])
@pytest.mark.parametrize("rows", Q4_SHORT_ROWS)
def test_block_projection_with_the_weights_unpacked_in_the_product(family, name, rows):
    """Either side of the row tiles of 32, 64, 96 and (but for the output projection) 128 that short blocks
    are multiplied in, one and several of them, and past the last rows that the GDN and the output projection
    take so, against the 64-bit sums and with the bound above."""
    B = gpu()[0]
    tile = B.q4_block_tile(rows, family["k"], sum(family["segments"]), gpu()[1].compute_units)
    assert tile.startswith("short") == (rows <= 384 or family is ATTN), tile
    test_block_projection_against_64_bit_sums_over_the_whole_range(family, name, rows)


@pytest.mark.parametrize("family,name", [(ATTN, "attn_project_blk"), (GDN, "gdn_project_blk"),
                                         (OUT, "outproj_blk")], ids=["attn", "gdn", "out"])
@pytest.mark.parametrize("rows", Q4_UNFOLDED_ROWS)
def test_block_projection_on_the_tiles_that_fill_the_rounds(family, name, rows):
    """Rows that take 256 x 288, 224 x 256, 160 x 256 and the tiles beside them over unfolded weights (see
    tests/test_host_rules.py), with remainders, against the 64-bit sums and with the bound above."""
    test_block_projection_against_64_bit_sums_over_the_whole_range(family, name, rows)


@pytest.mark.parametrize("family,name", [(ATTN, "attn_project_blk"), (GDN, "gdn_project_blk"),
                                         (OUT, "outproj_blk")], ids=["attn", "gdn", "out"])
@pytest.mark.parametrize("rows", [17, 100, 600])
def test_block_projection_keeps_scales_far_below_the_largest_of_their_row(family, name, rows):
    """Every output row has a group of scale 1 whose inputs are zero, and scales of 129 to 255 times 2^-35
    beside it: with the largest of 8 |scale| brought below 2^15 each of those is a whole number of f16's
    smallest subnormals, with one bit less room the odd ones are not.  Inputs are small whole numbers
    and the biases take the nibbles' offset of 8 out, so that every sum is exact and the result correctly
    rounded, by either route of a block (17 and 100 rows unpack the weights in the product, 600 do not)."""
    print(f"[case] {name} rows={rows} scales far below their row's largest", flush=True)
    B, dev, queue, lib = gpu()
    rng = np.random.default_rng(0xB0 + rows)
    k, total = family["k"], sum(family["segments"])
    x = rng.integers(-2, 3, (rows, k)) * (rng.random((rows, k)) < 0.05)
    x[:, :64] = 0
    bindings, want = {0: dev.buffer_from(ol.f32_to_bf16(x.astype(np.float32).reshape(-1)))}, []
    for index, n in enumerate(family["segments"]):
        words = rng.integers(0, 2 ** 32, n * k // 8, dtype=np.uint64).astype(np.uint32)
        units = rng.integers(64, 128, n) * 2 + 1
        scale = np.repeat(units[:, None] * 2.0 ** -35, k // 64, axis=1)
        scale[:, 0] = 1.0
        slot = 1 + 3 * index
        bindings.update({slot: dev.buffer_from(words),
                         slot + 1: dev.buffer_from(ol.f32_to_bf16(scale.astype(np.float32).reshape(-1))),
                         slot + 2: dev.buffer_from(ol.f32_to_bf16((-8.0 * scale).astype(np.float32).reshape(-1)))})
        nibbles = ((words[:, None] >> (4 * np.arange(8, dtype=np.uint32))[None, :]) & 15).reshape(n, k)
        sums = x.astype(np.float64) @ (nibbles.astype(np.float64) - 8.0).T * units
        assert np.abs(sums).max() < 2 ** 24
        want.append((sums * 2.0 ** -35).astype(np.float32))
    out = dev.buffer_from(np.full(rows * total, 0x7FC0, np.uint16))      # NaN until written
    bindings[family["out"]] = out
    slot = family["out"] + 1
    constants = {slot: rows, slot + 1: k} if family is OUT else {slot: rows}
    run(lambda cb: cb.encode(lib.pipeline(name), bindings, constants, (_groups(family), 1, 1),
                             (family["threads"], 1, 1)))
    got = ol.bf16_to_f32(out.read(np.uint16))
    want = ol.bf16_to_f32(ol.f32_to_bf16(np.concatenate(want, axis=1).reshape(-1)))
    assert np.count_nonzero(want) > want.size // 2
    assert np.array_equal(got, want), f"{np.mean(got != want):.4f} of the outputs differ"


@pytest.mark.parametrize("family,name", [(ATTN, "attn_project_blk"), (GDN, "gdn_project_blk"),
                                         (OUT, "outproj_blk")], ids=["attn", "gdn", "out"])
@pytest.mark.parametrize("rows", [17, 300, 1500])
def test_block_projection_in_queues_of_less_workspace(family, name, rows):
    """A queue that could not have its whole workspace takes the operands through in slices of output
    rows and of input rows (8 MiB: 768 outputs and rows at a time at the hidden width, 256 at
    the attention width): the same sums, bit for bit.  One without workspace evaluates the rows in
    the reference's order: the oracle's bits."""
    B, dev, _, lib = gpu()
    # the output projection's slices of 256 rows and outputs: where unfolded weights take the 32 x 64 tile
    assert B.block_product_tile(256, 4352, 256, dev.compute_units) == "32x64"
    assert B.block_product_shape(256, 4352, 256, dev.compute_units) == (32, 64)
    host, bindings = _family(dev, family, 0xA800)
    k, total = family["k"], sum(family["segments"])
    x = ol.gaussian_bf16(0xA900 + rows, rows * k, 0.0, 1.0)
    bindings[0] = dev.buffer_from(x)
    slot = family["out"] + 1
    constants = {slot: rows, slot + 1: k} if family is OUT else {slot: rows}
    got = {}
    for workspace in (None, 60 << 20, 20 << 20, 8 << 20, 1 << 20, 0):
        print(f"[case] {name} rows={rows} workspace={workspace}", flush=True)
        queue = dev.create_queue(workspace)
        out = dev.buffer_from(np.full(rows * total, 0x7FC0, np.uint16))
        cb = queue.create_command_buffer()
        cb.begin_compute_pass()
        cb.encode(lib.pipeline(name), {**bindings, family["out"]: out}, constants, (_groups(family), 1, 1),
                  (family["threads"], 1, 1))
        cb.end_compute_pass()
        ms = cb.commit().wait()
        got[workspace] = out.read(np.uint16).reshape(rows, total)
        print(f"[time] {ms * 1e3:.1f} us", flush=True)
    for workspace in (60 << 20, 20 << 20, 8 << 20):
        assert np.array_equal(got[workspace], got[None]), workspace
    assert np.array_equal(got[0], got[1 << 20])
    sample = sorted({0, 15, 16, rows // 2, rows - 1})
    want = _expected(family, host, np.ascontiguousarray(x.reshape(rows, k)[sample]).reshape(-1), len(sample))
    assert np.array_equal(got[0][sample].reshape(-1), want)


def _cancelling_matrix(rng, rows, k):
    """Matrices whose second half of K undoes the first: columns k / 2 on hold, permuted, 16 minus the
    nibbles (1 .. 15) of the first, one scale to a row, biases of -7.5 scales and then -8.5 (scales of
    three bits, so that both are bf16 numbers).  With x repeated by the same permutation every exact
    result is zero, so that what a projection returns is the error of its fp32 sums, which rounding
    an ordinary result to bf16 hides."""
    order = rng.permutation(k // 2)
    half = rng.integers(1, 16, (rows, k // 2), dtype=np.uint32)
    nibbles = np.concatenate([half, 16 - half[:, order]], axis=1).reshape(rows, k // 8, 8)
    words = np.bitwise_or.reduce(nibbles << (4 * np.arange(8, dtype=np.uint32)), axis=2).astype(np.uint32)
    scales = np.repeat(rng.choice([0.5, 0.625, 0.75, 0.875], (rows, 1)), k // 64, axis=1)
    biases = scales * np.where(np.arange(k // 64) < k // 128, -7.5, -8.5)
    return (order, words.reshape(-1),
            *(ol.f32_to_bf16(v.astype(np.float32).reshape(-1)) for v in (scales, biases)))


@pytest.mark.parametrize("family,name", [(ATTN, "attn_project"), (GDN, "gdn_project"), (OUT, "outproj")],
                         ids=["attn", "gdn", "out"])
@pytest.mark.parametrize("rows", [2, 4, 5, 8, 9, 12, 13, 16])
def test_short_block_sums_are_no_further_from_exact_than_the_reference_order(family, name, rows):
    """`*_mfma_blk` (2..16 rows on the matrix unit, one instantiation for every four rows) against
    the `_blk` form, which keeps the reference's order: where the exact result is zero, the rms of
    what is left of the fp32 sums is no larger.  (Measured 4.1e-6 against 6.5e-6 over 2048 columns and
    5.7e-6 against 11.5e-6 over 4096; 4096 outputs or more are a sample that puts an rms within about
    1 %.)"""
    print(f"[case] {name}_mfma_blk rows={rows} fp32 sums", flush=True)
    B, dev, queue, lib = gpu()
    rng = np.random.default_rng(0xA500 + rows)
    k, total = family["k"], sum(family["segments"])
    order, words, scales, biases = _cancelling_matrix(rng, total, k)
    x = rng.standard_normal((rows, k // 2), dtype=np.float32)
    x = ol.f32_to_bf16(np.concatenate([x, x[:, order]], axis=1).reshape(-1))
    bindings, first = {0: dev.buffer_from(x)}, 0
    for index, n in enumerate(family["segments"]):
        for part, (values, per) in enumerate(((words, k // 8), (scales, k // 64), (biases, k // 64))):
            bindings[1 + 3 * index + part] = dev.buffer_from(values[first * per:(first + n) * per])
        first += n
    got = {}
    for suffix in ("_blk", "_mfma_blk"):
        out = dev.buffer_from(np.full(rows * total, 0x7FC0, np.uint16))
        bindings[family["out"]] = out
        slot = family["out"] + 1
        constants = {slot: rows, slot + 1: k} if family is OUT else {slot: rows}
        run(lambda cb: cb.encode(lib.pipeline(name + suffix), bindings, constants, (_groups(family), 1, 1),
                                 (family["threads"], 1, 1)))
        left = ol.bf16_to_f32(out.read(np.uint16)).astype(np.float64)
        assert np.isfinite(left).all()
        got[suffix] = np.sqrt(np.mean(left ** 2))
    print(f"[parity] {name} rows {rows}: rms left of zero, reference's order {got['_blk']:.3e}, "
          f"matrix unit {got['_mfma_blk']:.3e}", flush=True)
    assert got["_mfma_blk"] <= got["_blk"]


@pytest.mark.parametrize("family,name", [(ATTN, "attn_project"), (GDN, "gdn_project"), (OUT, "outproj")],
                         ids=["attn", "gdn", "out"])
@pytest.mark.parametrize("rows", [1, 4, 7, 12, 16])
def test_short_block_projection_on_the_matrix_unit(family, name, rows):
    print(f"[case] {name}_mfma_blk rows={rows}", flush=True)
    B, dev, queue, lib = gpu()
    host, bindings = _family(dev, family, 0xA600)
    k, total = family["k"], sum(family["segments"])
    x = ol.gaussian_bf16(0xA700 + rows, rows * k, 0.0, 1.0)
    out = dev.buffer_from(np.full(rows * total, 0x7FC0, np.uint16))
    bindings.update({0: dev.buffer_from(x), family["out"]: out})
    slot = family["out"] + 1
    constants = {slot: rows, slot + 1: k} if family is OUT else {slot: rows}
    run(lambda cb: cb.encode(lib.pipeline(name + "_mfma_blk"), bindings, constants, (_groups(family), 1, 1),
                             (family["threads"], 1, 1)))
    check_bf16(out.read(np.uint16), _expected(family, host, x, rows), name + "_mfma_blk", ulps=2)
    with pytest.raises(B.BackendError) as e:
        run(lambda cb: cb.encode(lib.pipeline(name + "_mfma_blk"), bindings, {**constants, slot: 17},
                                 (_groups(family), 1, 1), (family["threads"], 1, 1)))
    assert e.value.status == 15


@pytest.mark.parametrize("rows", [2, 4, 13, 16])
@pytest.mark.parametrize("family", [ATTN, GDN], ids=lambda f: f["name"])
def test_wave_projection_with_the_norm_in_its_prologue(family, rows):
    """`*_project_rms_mfma_ms` (no reference counterpart) on rows that have not been normed
    against `rms_only_ms` followed by `*_project_mfma_ms`: the same bits, and the norm the
    fused form applies is the checker's."""
    name = family["name"]
    print(f"[case] {name}_rms_mfma_ms rows={rows}", flush=True)
    B, dev, queue, lib = gpu()
    host, bindings = _family(dev, family, 0x9A00)
    x = ol.gaussian_bf16(0x9B00 + rows, rows * 2048, 0.0, 1.5)
    weight = ol.gaussian_bf16(0x9C00, 2048, 1.0, 0.25)
    total = sum(family["segments"])
    b_x, b_w = dev.buffer_from(x), dev.buffer_from(weight)
    b_normed = dev.create_buffer(rows * 2048 * 2)
    two_step = dev.buffer_from(np.full(rows * total, 0x7FC0, np.uint16))
    fused = dev.buffer_from(np.full(rows * total, 0x7FC0, np.uint16))
    out, slot = family["out"], family["out"] + 1
    grid = (_groups(family), 1, 1)

    def rec(cb):
        cb.encode(lib.pipeline("rms_only_ms"), {0: b_x, 1: b_w, 2: b_normed}, {3: 2048, 4: 2048},
                  (1, rows), (512,))
        cb.barrier()
        cb.encode(lib.pipeline(name + "_mfma_ms"), {**bindings, 0: b_normed, out: two_step},
                  {slot: rows, slot + 1: 16}, grid, (family["threads"], 1, 1))
        cb.encode(lib.pipeline(name + "_rms_mfma_ms"), {**bindings, 0: b_x, out: fused, out + 3: b_w},
                  {slot: rows, slot + 1: 16}, grid, (family["threads"], 1, 1))
    run(rec)
    normed = np.zeros(rows * 2048, np.uint16)
    o.tto_rms_only(x, weight, rows, 2048, normed)
    assert np.array_equal(b_normed.read(np.uint16), normed)
    assert np.array_equal(fused.read(np.uint16), two_step.read(np.uint16))
    check_bf16(fused.read(np.uint16), _expected(family, host, normed, rows), name + "_rms_mfma_ms", ulps=2)


@pytest.mark.parametrize("in_place", [False, True], ids=["apart", "in-place"])
@pytest.mark.parametrize("rows", [2, 4, 16])
def test_wave_out_projection_with_the_residual_in_its_epilogue(rows, in_place):
    """`gdn_outproj_residual_mfma_ms` (no reference counterpart) against `gdn_outproj_mfma_ms`
    followed by the residual sum of `residual_rms_ms`: the same bits, with the output in a
    buffer of its own and in the residual buffer itself."""
    print(f"[case] gdn_outproj_residual_mfma_ms rows={rows} in_place={in_place}", flush=True)
    B, dev, queue, lib = gpu()
    host, bindings = _family(dev, OUT, 0x9D00)
    mixed = ol.gaussian_bf16(0x9E00 + rows, rows * 4096, 0.0, 1.0)
    x = ol.gaussian_bf16(0x9F00 + rows, rows * 2048, 0.0, 1.0)
    weight = ol.gaussian_bf16(0xA000, 2048, 1.0, 0.25)
    b_mixed, b_x, b_w = dev.buffer_from(mixed), dev.buffer_from(x), dev.buffer_from(weight)
    b_delta = dev.create_buffer(rows * 2048 * 2)
    b_sum, b_normed = dev.create_buffer(rows * 2048 * 2), dev.create_buffer(rows * 2048 * 2)
    b_fused = dev.buffer_from(x) if in_place else dev.create_buffer(rows * 2048 * 2)
    b_before = b_fused if in_place else b_x

    def rec(cb):
        cb.encode(lib.pipeline("gdn_outproj_mfma_ms"), {**bindings, 0: b_mixed, 4: b_delta},
                  {5: rows, 6: 2048, 7: 16}, (1024, 1, 1), (64, 1, 1))
        cb.barrier()
        cb.encode(lib.pipeline("residual_rms_ms"), {0: b_x, 1: b_delta, 2: b_sum, 3: b_w, 4: b_normed},
                  {5: 2048, 6: 2048, 7: 2048}, (1, rows), (512,))
        cb.encode(lib.pipeline("gdn_outproj_residual_mfma_ms"),
                  {**bindings, 0: b_mixed, 4: b_fused, 8: b_before}, {5: rows, 6: 2048, 7: 16},
                  (1024, 1, 1), (64, 1, 1))
    run(rec)
    assert np.array_equal(b_fused.read(np.uint16), b_sum.read(np.uint16))
    delta = ol.bf16_to_f32(b_delta.read(np.uint16))
    want = ol.f32_to_bf16(ol.bf16_to_f32(x) + delta)
    assert np.array_equal(b_fused.read(np.uint16), want)


def test_projection_validation():
    B, dev, queue, lib = gpu()
    host, bindings = _family(dev, ATTN, 0x9600)
    bindings[0] = dev.create_buffer(16 * 2048 * 2)
    bindings[10] = dev.create_buffer(16 * 9216 * 2)
    cb = queue.create_command_buffer()
    cb.begin_compute_pass()
    ms = lib.pipeline("attn_project_ms")
    cases = [
        (bindings, {11: 17, 12: 16}, (2304, 2, 1), 15),     # more rows than a wave holds
        (bindings, {11: 16, 12: 17}, (2304, 1, 1), 15),     # tile beyond the batch maximum
        (bindings, {11: 16, 12: 4}, (2304, 3, 1), 15),      # tiles do not cover the rows
        (bindings, {11: 16, 12: 4}, (2303, 4, 1), 15),      # groups do not cover the output rows
        ({**bindings, 4: dev.create_buffer(512 * 256 * 4 - 4)}, {11: 4, 12: 4}, (2304, 1, 1), 10),
        ({**bindings, 10: dev.create_buffer(4 * 9216 * 2 - 2)}, {11: 4, 12: 4}, (2304, 1, 1), 10),
        ({**bindings, 0: dev.create_buffer(4 * 2048 * 2 - 2)}, {11: 4, 12: 4}, (2304, 1, 1), 10),
    ]
    for buffers, constants, grid, status in cases:
        with pytest.raises(B.BackendError) as e:
            cb.encode(ms, buffers, constants, grid, (128, 1, 1))
        assert e.value.status == status, (constants, grid)
    host, out_bindings = _family(dev, OUT, 0x9700)
    out_bindings[0] = dev.create_buffer(4 * 4096 * 2)
    out_bindings[4] = dev.create_buffer(4 * 2048 * 2)
    with pytest.raises(B.BackendError) as e:   # output stride below the hidden width
        cb.encode(lib.pipeline("gdn_outproj_ms"), out_bindings, {5: 4, 6: 2047, 7: 4}, (1024, 1, 1),
                  (64, 1, 1))
    assert e.value.status == 8
    with pytest.raises(B.BackendError) as e:   # input width not a multiple of 512
        cb.encode(lib.pipeline("outproj_blk"), out_bindings, {5: 4, 6: 4000}, (1024, 1, 1), (64, 1, 1))
    assert e.value.status == 15
    # the block form moves 16-byte pieces: an input bound 2 bytes off is refused when encoded
    blk_bindings = dict(bindings)
    blk_bindings[0] = (dev.create_buffer(64 * 2048 * 2 + 16), 2)
    blk_bindings[10] = dev.create_buffer(64 * 9216 * 2)
    with pytest.raises(B.BackendError) as e:
        cb.encode(lib.pipeline("attn_project_blk"), blk_bindings, {11: 64}, (2304, 1, 1), (128, 1, 1))
    assert e.value.status == 10
    assert cb.command_count == 0
