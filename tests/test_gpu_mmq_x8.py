"""The prefill GEMM of the formats with an fp16 scale per 32 weights on 32 x 128 wavefront tiles (kernels/mmq_x8.h, taken by
rein_matmul_ws), at the edges of its tiles, groups and ranges, against the CPU oracle and beside the tile of mmq_gemm.h."""
import numpy as np
import pytest

import reinstinct_amd as rein
from oracle import orc
from reinstinct_amd import hip, quant, runtime
from reinstinct_amd._lib import init, set_option
from tests.helpers import assert_close_f32

pytestmark = pytest.mark.gpu
FORMATS = [rein.Q8_0, rein.Q4_0, rein.IQ4_XS, rein.IQ3_S]
OPTIONS = ("REIN_MMQXH", "REIN_MMQXH_SPLIT", "REIN_MMQXH_GROUPS")


@pytest.fixture(autouse=True)
def _options():
    init()
    hip.set_device(0)
    yield
    for name in OPTIONS:
        set_option(name, None)


def blocks(fmt, in_dim, out_dim, seed):
    rng = np.random.default_rng(seed)
    if fmt == rein.IQ3_S:                            # no quantizer: random block bytes with scales near 0.02
        raw = rng.integers(0, 256, (out_dim * in_dim // 256, 110), dtype=np.uint8)
        raw[:, :2] = rng.uniform(1e-3, 2e-3, raw.shape[0]).astype(np.float16)[:, None].view(np.uint8)
        return raw.reshape(-1)
    return quant.quantize_weights(fmt, rng.standard_normal((out_dim, in_dim)).astype(np.float32) * 0.02)


def matmul(fmt, packed, x, out_dim, mode, split=None, groups=None):
    rows, in_dim = x.shape
    for name, v in zip(OPTIONS, (mode, split, groups)):
        set_option(name, None if v is None else str(v))
    size = runtime.matmul_scratch_bytes(fmt, in_dim, rows)
    dw, dx, scratch = hip.DeviceBuf.from_host(packed), hip.DeviceBuf.from_host(x), hip.DeviceBuf(size)
    guard = 64                                        # words behind the output that must stay as they are
    dy = hip.DeviceBuf.from_host(np.full(rows * out_dim + guard, 12345.0, np.float32))
    print(f"fmt {fmt} rows {rows} in {in_dim} out {out_dim} mode {mode} split {split} groups {groups}", flush=True)
    runtime.matmul_ws(fmt, dw, dx, dy, in_dim, out_dim, rows, scratch, size)
    hip.synchronize()
    y = dy.to_host(np.float32)
    assert (y[rows * out_dim:] == 12345.0).all()
    return y[:rows * out_dim].reshape(rows, out_dim)


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("rows, in_dim, out_dim, split, groups", [
    (9, 256, 5, None, None),             # one token tile, one superblock, a row block almost empty, scalar stores
    (33, 768, 130, 3, 2),                # groups of one tile, a range per superblock
    (64, 1024, 200, 2, 1),               # padded weight rows (32 sub-blocks): 16-bit transfers of the scales
    (90, 768, 127, None, None),
    (128, 2048, 264, 1, 1),              # four tiles; padded
    (129, 1280, 128, 2, 2),              # groups of three and two tiles
    (300, 2304, 257, 4, None),           # uneven ranges of nine superblocks
    (520, 256, 16384, None, 5),          # 640 units: a whole round and a tail, groups of four and three
])
def test_against_the_oracle(fmt, rows, in_dim, out_dim, split, groups):
    packed = quant.repack_for_matvec(fmt, blocks(fmt, in_dim, out_dim, rows), in_dim, out_dim)
    x = np.random.default_rng(in_dim).standard_normal((rows, in_dim)).astype(np.float32)
    x[0] *= 1e-20
    x[rows // 2] = 0.0
    x[rows - 1] *= 1e20
    got = matmul(fmt, packed, x, out_dim, 2, split, groups)
    want = orc.matvec_q8(fmt, packed, in_dim, out_dim, orc.quantize_q8(x), rows)
    scale = np.abs(x).max(axis=1, keepdims=True) + (np.abs(x).max(axis=1, keepdims=True) == 0)
    assert_close_f32(got / scale, want / scale, what=f"fmt {fmt}")


@pytest.mark.parametrize("fmt", FORMATS)
def test_the_bits_of_the_other_tile(fmt):
    """unsplit, the same products and sums in the same order as the 32- and 64-token tiles of mmq_gemm.h, whatever the groups"""
    rows, in_dim, out_dim = 97, 1536, 200
    packed = quant.repack_for_matvec(fmt, blocks(fmt, in_dim, out_dim, 1), in_dim, out_dim)
    x = np.random.default_rng(2).standard_normal((rows, in_dim)).astype(np.float32)
    dw, xq, dy = hip.DeviceBuf.from_host(packed), hip.DeviceBuf.from_host(orc.quantize_q8(x)), hip.DeviceBuf(rows * out_dim * 4)
    runtime.mmq_xq8(fmt, dw, xq, dy, in_dim, out_dim, rows)
    hip.synchronize()
    want = dy.to_host(np.uint32).reshape(rows, out_dim)
    for groups in (1, 2, 4):
        assert np.array_equal(matmul(fmt, packed, x, out_dim, 2, 1, groups).view(np.uint32), want)


def test_largest_dots():
    """every product of a block 127 * -128 and 127 * 127: the sums on the bits of 1.5 * 2^23 at their ends"""
    rows, in_dim, out_dim = 40, 512, 64
    raw = np.zeros((out_dim, in_dim // 32, 34), np.uint8)
    raw[:, :, :2] = np.array([1.0], np.float16).view(np.uint8)
    raw[:, :, 2:] = np.where(np.arange(out_dim) % 2, 127, -128).astype(np.int8).view(np.uint8)[:, None, None]
    packed = quant.repack_for_matvec(rein.Q8_0, raw.reshape(-1), in_dim, out_dim)
    x = np.where(np.arange(rows) % 3, 127.0, -127.0).astype(np.float32)[:, None] * np.ones(in_dim, np.float32)
    want = x[:, :1] * np.where(np.arange(out_dim) % 2, 127.0, -128.0)[None, :] * in_dim
    assert np.array_equal(matmul(rein.Q8_0, packed, x, out_dim, 2), want.astype(np.float32))


@pytest.mark.parametrize("fmt", [rein.Q8_0, rein.IQ4_XS])
@pytest.mark.parametrize("rows, in_dim, skip", [(33, 256, 0), (129, 1280, 0), (77, 768, 1)])          # skip: x not 16-byte aligned
def test_the_scratch_holds_the_quantized_rows(fmt, rows, in_dim, skip):
    out_dim = 96
    x = np.random.default_rng(rows).standard_normal((rows, in_dim)).astype(np.float32)
    x[rows // 2] = 0.0
    set_option("REIN_MMQXH", "2")
    size = runtime.matmul_scratch_bytes(fmt, in_dim, rows)
    dw = hip.DeviceBuf.from_host(quant.repack_for_matvec(fmt, blocks(fmt, in_dim, out_dim, 1), in_dim, out_dim))
    dx = hip.DeviceBuf.from_host(np.concatenate([np.zeros(skip, np.float32), x.reshape(-1)]))
    scratch, dy = hip.DeviceBuf.from_host(np.full(size, 0xA5, np.uint8)), hip.DeviceBuf(rows * out_dim * 4)
    runtime.matmul_ws(fmt, dw, dx.ptr + 4 * skip, dy, in_dim, out_dim, rows, scratch, size)
    hip.synchronize()
    want = orc.quantize_q8(x)
    got = scratch.to_host(np.uint8)
    assert np.array_equal(got[:want.size], want)
    assert (got[want.size:(want.size + 255) // 256 * 256] == 0xA5).all()          # up to the image nothing is touched


def test_smaller_scratch_and_capture():
    """a scratch without the room runs the launches of rein_mmq_xq8_ws, bit for bit; a captured call replays to the eager bits"""
    fmt, rows, in_dim, out_dim = rein.Q8_0, 200, 4096, 640
    packed = quant.repack_for_matvec(fmt, blocks(fmt, in_dim, out_dim, 5), in_dim, out_dim)
    x = np.random.default_rng(6).standard_normal((rows, in_dim)).astype(np.float32)
    size = runtime.matmul_scratch_bytes(fmt, in_dim, rows)
    dw, dx, scratch, dy = hip.DeviceBuf.from_host(packed), hip.DeviceBuf.from_host(x), hip.DeviceBuf(size), hip.DeviceBuf(rows * out_dim * 4)

    def call(n, stream=None):
        runtime.matmul_ws(fmt, dw, dx, dy, in_dim, out_dim, rows, scratch, n, stream)

    call(size)
    hip.synchronize()
    eager = dy.to_host(np.uint32)
    small = (rows * in_dim // 32 * 40 + 255) // 256 * 256 + 4096             # less than the activation image
    call(small)
    hip.synchronize()
    without = dy.to_host(np.uint32)
    set_option("REIN_MMQXH", "0")
    call(small)
    hip.synchronize()
    assert np.array_equal(without, dy.to_host(np.uint32))
    set_option("REIN_MMQXH", None)
    stream = hip.Stream()
    stream.begin_capture()
    call(size, stream)
    graph = stream.end_capture().instantiate()
    for _ in range(3):
        runtime.quantize_q8(dx, scratch, in_dim, rows)          # the program's own work on the same scratch between replays
        hip.synchronize()
        graph.launch(stream)
        stream.synchronize()
        assert np.array_equal(dy.to_host(np.uint32), eager)


@pytest.mark.parametrize("split", [1, 2])
def test_infinities_and_nan_stay_where_they_are(split):
    """rows of x with an infinity or a NaN and weight rows with such a scale: non-finite where the other tile is, every other result
    the bits of a product without them"""
    fmt, rows, in_dim, out_dim = rein.Q8_0, 97, 1024, 200
    rng = np.random.default_rng(fmt)
    x = rng.standard_normal((rows, in_dim)).astype(np.float32)
    w = blocks(fmt, in_dim, out_dim, 7).reshape(out_dim, -1, 34)
    bad_x, bad_w = x.copy(), w.copy()
    for r, v in {3: np.inf, 40: np.nan, 64: -np.inf, 96: np.inf}.items():
        bad_x[r, (11 * r) % in_dim] = v
    for r, v in {0: np.nan, 77: np.inf, 130: -np.inf, 199: np.nan}.items():
        bad_w[r, r % 4, :2] = np.array([v], np.float16).view(np.uint8)

    def product(w, x, mode):
        return matmul(fmt, quant.repack_for_matvec(fmt, np.ascontiguousarray(w).reshape(-1), in_dim, out_dim), x, out_dim, mode, split)

    clean, got, tile = product(w, x, 2), product(bad_w, bad_x, 2), product(bad_w, bad_x, 0)
    assert np.array_equal(np.isfinite(got), np.isfinite(tile))
    assert not np.isfinite(got[[3, 64, 96]]).any() and not np.isfinite(got[:, [0, 77, 130, 199]]).any()
    rest = np.ix_(np.setdiff1d(np.arange(rows), [3, 40, 64, 96]), np.setdiff1d(np.arange(out_dim), [0, 77, 130, 199]))
    assert np.array_equal(got[rest].view(np.uint32), clean[rest].view(np.uint32))
