"""The Q4_K / Q5_K / Q6_K prefill GEMM with exact block dots on the fp16 instruction (kernels/mmq_exact16.h, taken by rein_matmul_ws),
at the edges of its tiles, against the CPU oracle, and its distance from 64-bit sums beside the int8 tile's."""
import numpy as np
import pytest

import reinstinct_amd as rein
from oracle import orc
from reinstinct_amd import hip, quant, runtime
from reinstinct_amd._lib import init, set_option
from tests.helpers import assert_close_f32

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _options():
    init()
    hip.set_device(0)
    yield
    for name in ("REIN_MMQXH", "REIN_MMQXH_SPLIT"):
        set_option(name, None)


def matmul(fmt, packed, x, out_dim, mode, split=None):
    rows, in_dim = x.shape
    set_option("REIN_MMQXH", str(mode))
    set_option("REIN_MMQXH_SPLIT", split and str(split))
    size = runtime.matmul_scratch_bytes(fmt, in_dim, rows)
    dw, dx, scratch = hip.DeviceBuf.from_host(packed), hip.DeviceBuf.from_host(x), hip.DeviceBuf(size)
    guard = 64                                        # words behind the output that must stay as they are
    dy = hip.DeviceBuf.from_host(np.full(rows * out_dim + guard, 12345.0, np.float32))
    print(f"fmt {fmt} rows {rows} in {in_dim} out {out_dim} mode {mode} split {split}", flush=True)
    runtime.matmul_ws(fmt, dw, dx, dy, in_dim, out_dim, rows, scratch, size)
    hip.synchronize()
    y = dy.to_host(np.float32)
    assert (y[rows * out_dim:] == 12345.0).all()
    return y[:rows * out_dim].reshape(rows, out_dim)


def weights(fmt, in_dim, out_dim, seed):
    w = np.random.default_rng(seed).standard_normal((out_dim, in_dim)).astype(np.float32) * 0.02
    return quant.repack_for_matvec(fmt, quant.quantize_weights(fmt, w), in_dim, out_dim)


@pytest.mark.parametrize("fmt", [rein.Q4_K, rein.Q5_K, rein.Q6_K])
@pytest.mark.parametrize("rows, in_dim, out_dim, split", [
    (33, 256, 5, None),          # two token tiles, one superblock, a row block almost empty, scalar stores
    (128, 512, 128, None),       # one whole unit; padded weight rows (16 sub-blocks)
    (64, 1024, 200, 2),
    (90, 768, 130, 3),           # a range per superblock
    (128, 2048, 264, 1),
    (129, 1280, 127, 2),         # groups of three and two tiles
    (300, 2304, 257, 4),         # uneven ranges of nine superblocks
    (777, 512, 96, None),
])
def test_against_the_oracle(fmt, rows, in_dim, out_dim, split):
    packed = weights(fmt, in_dim, out_dim, rows)
    x = np.random.default_rng(in_dim).standard_normal((rows, in_dim)).astype(np.float32)
    x[0] *= 1e-20
    x[rows // 2] = 0.0
    x[rows - 1] *= 1e20
    got = matmul(fmt, packed, x, out_dim, 2, split)
    want = orc.matvec_q8(fmt, packed, in_dim, out_dim, orc.quantize_q8(x), rows)
    scale = np.abs(x).max(axis=1, keepdims=True) + (np.abs(x).max(axis=1, keepdims=True) == 0)
    assert_close_f32(got / scale, want / scale, what=f"fmt {fmt}")


@pytest.mark.parametrize("fmt", [rein.Q4_K, rein.Q5_K, rein.Q6_K])
@pytest.mark.parametrize("rows, in_dim, out_dim, split", [
    (9, 256, 1, None),           # scales come word by word: fewer than sixteen scale words behind them
    (40, 256, 15, None),
    (33, 256, 16, None),         # and by sixteen bytes, up to the last scale word
    (64, 1280, 3, 2),
    (20, 1024, 129, None),       # rows of the slab padded to an odd number of sub-blocks: odd rows start between two dwords
    (45, 2048, 257, 3),          # ranges of an odd and an even number of superblocks
    (64, 2304, 100, 4),
    (96, 768, 130, 1),
])
def test_groups_of_one_and_two_tiles(fmt, rows, in_dim, out_dim, split):
    packed = weights(fmt, in_dim, out_dim, rows)
    x = np.random.default_rng(out_dim).standard_normal((rows, in_dim)).astype(np.float32)
    assert_close_f32(matmul(fmt, packed, x, out_dim, 3, split), orc.matvec_q8(fmt, packed, in_dim, out_dim, orc.quantize_q8(x), rows), what=f"fmt {fmt}")


@pytest.mark.parametrize("fmt", [rein.Q4_K, rein.Q6_K])
@pytest.mark.parametrize("rows, in_dim, skip", [(33, 256, 0), (129, 1280, 0), (77, 768, 1)])          # skip: x not 16-byte aligned
def test_the_scratch_holds_the_quantized_rows(fmt, rows, in_dim, skip):
    """the first part of the scratch is what rein_quantize_q8 writes, here as on every other launch of rein_matmul_ws: a caller that
    quantizes with one projection may run the next one on it"""
    out_dim = 96
    x = np.random.default_rng(rows).standard_normal((rows, in_dim)).astype(np.float32)
    x[rows // 2] = 0.0
    set_option("REIN_MMQXH", "2")
    size = runtime.matmul_scratch_bytes(fmt, in_dim, rows)
    dw, dx = hip.DeviceBuf.from_host(weights(fmt, in_dim, out_dim, 1)), hip.DeviceBuf.from_host(np.concatenate([np.zeros(skip, np.float32), x.reshape(-1)]))
    scratch, dy = hip.DeviceBuf.from_host(np.full(size, 0xA5, np.uint8)), hip.DeviceBuf(rows * out_dim * 4)
    runtime.matmul_ws(fmt, dw, dx.ptr + 4 * skip, dy, in_dim, out_dim, rows, scratch, size)
    hip.synchronize()
    want = orc.quantize_q8(x)
    got = scratch.to_host(np.uint8)
    assert np.array_equal(got[:want.size], want)
    behind = (want.size + 255) // 256 * 256               # up to the image nothing is touched
    assert (got[want.size:behind] == 0xA5).all()


@pytest.mark.parametrize("fmt", [rein.Q4_K, rein.Q5_K, rein.Q6_K])
def test_no_further_from_64_bits_than_the_int8_tile(fmt):
    rows, in_dim, out_dim = 160, 4352, 256
    w = quant.quantize_weights(fmt, np.random.default_rng(1).standard_normal((out_dim, in_dim)).astype(np.float32) * 0.02)
    packed = quant.repack_for_matvec(fmt, w, in_dim, out_dim)
    x = np.random.default_rng(2).standard_normal((rows, in_dim)).astype(np.float32)
    q = orc.quantize_q8(x).reshape(-1, 40)
    xd = (q[:, 8:].view(np.int8) * q[:, :4].copy().view(np.float32).astype(np.float64)).reshape(rows, in_dim)
    if fmt == rein.Q6_K:
        exact = xd @ orc.dequantize_to_f32(fmt, w, out_dim * in_dim).astype(np.float64).reshape(out_dim, in_dim).T
    else:                                            # the minimum term goes with the blocks' xsum, not with their quants
        blocks = w.reshape(out_dim * in_dim // 256, -1)
        no_min, only_min = blocks.copy(), blocks.copy()
        no_min[:, 2:4] = 0
        only_min[:, 16:] = 0
        part = [orc.dequantize_to_f32(fmt, b.reshape(-1), out_dim * in_dim).astype(np.float64).reshape(out_dim, in_dim) for b in (no_min, only_min)]
        xsum = q[:, 4:8].copy().view(np.float32).astype(np.float64).reshape(rows, in_dim // 32)
        exact = xd @ part[0].T + xsum @ part[1][:, ::32].T
    err = [np.linalg.norm(matmul(fmt, packed, x, out_dim, mode) - exact) / np.linalg.norm(exact) for mode in (2, 0)]
    print("relative error: exact dots", err[0], "int8 tile", err[1], flush=True)
    assert err[0] <= 1.05 * err[1]


def test_all_scales_and_quants_are_exact():
    """every scale byte of Q6_K, -128 and 127 among them, against every quant: integers through and through"""
    in_dim, out_dim, rows = 256, 256, 65
    rng = np.random.default_rng(3)
    blocks = np.zeros((out_dim, 210), np.uint8)
    blocks[:, :192] = rng.integers(0, 256, (out_dim, 192))
    blocks[:, 192:208] = (np.arange(out_dim)[:, None] + 16 * np.arange(16)[None, :]).astype(np.uint8)
    blocks[:, 208:] = np.array([1.0], np.float16).view(np.uint8)
    packed = quant.repack_for_matvec(rein.Q6_K, blocks.reshape(-1), in_dim, out_dim)
    x = rng.integers(-15, 16, (rows, in_dim)).astype(np.float32)
    x.reshape(rows, -1, 32)[:, :, 0] = 127.0         # activation scale 1
    got = matmul(rein.Q6_K, packed, x, out_dim, 2)
    w = orc.dequantize_to_f32(rein.Q6_K, blocks.reshape(-1), in_dim * out_dim).reshape(out_dim, in_dim).astype(np.int64)
    want = x.astype(np.int64) @ w.T
    exact = np.abs(want) < 1 << 22
    assert exact.mean() > 0.5
    assert (got.astype(np.int64) == want)[exact].all()


def test_smaller_scratch_and_capture():
    """a scratch without the room runs the launches of rein_mmq_xq8_ws, bit for bit; a captured call replays to the eager bits"""
    fmt, rows, in_dim, out_dim = rein.Q6_K, 200, 4096, 640
    packed = weights(fmt, in_dim, out_dim, 5)
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
    assert np.array_equal(without, dy.to_host(np.uint32)) and not np.array_equal(without, eager)
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


D_AT = {rein.Q4_K: (144, 0), rein.Q5_K: (176, 0), rein.Q6_K: (210, 208)}        # bytes of a block, where d lies


@pytest.mark.parametrize("fmt", list(D_AT))
@pytest.mark.parametrize("split", [1, 2])
def test_infinities_and_nan_stay_where_they_are(fmt, split):
    """rows of x with an infinity or a NaN and weight rows with such a scale: non-finite where the int8 tile is, every other result
    the bits of a product without them"""
    rows, in_dim, out_dim = 97, 1024, 200
    rng = np.random.default_rng(fmt)
    x = rng.standard_normal((rows, in_dim)).astype(np.float32)
    blocks = quant.quantize_weights(fmt, rng.standard_normal((out_dim, in_dim)).astype(np.float32) * 0.02).reshape(out_dim, -1, D_AT[fmt][0])
    at = D_AT[fmt][1]
    bad_x, bad_w = x.copy(), blocks.copy()
    for r, v in {3: np.inf, 40: np.nan, 64: -np.inf, 96: np.inf}.items():
        bad_x[r, (11 * r) % in_dim] = v
    for r, v in {0: np.nan, 77: np.inf, 130: -np.inf, 199: np.nan}.items():
        bad_w[r, r % 4, at:at + 2] = np.array([v], np.float16).view(np.uint8)

    def product(w, x, mode):
        return matmul(fmt, quant.repack_for_matvec(fmt, np.ascontiguousarray(w).reshape(-1), in_dim, out_dim), x, out_dim, mode, split)

    clean, got, tile = product(blocks, x, 2), product(bad_w, bad_x, 2), product(bad_w, bad_x, 0)
    assert np.array_equal(np.isfinite(got), np.isfinite(tile))
    assert not np.isfinite(got[[3, 64, 96]]).any() and not np.isfinite(got[:, [0, 77, 130, 199]]).any()
    rest = np.ix_(np.setdiff1d(np.arange(rows), [3, 40, 64, 96]), np.setdiff1d(np.arange(out_dim), [0, 77, 130, 199]))
    assert np.array_equal(got[rest].view(np.uint32), clean[rest].view(np.uint32))
    nan_row = got[40][np.isfinite(got[40])]
    assert_close_f32(nan_row, tile[40][np.isfinite(got[40])], what="row with a NaN")


@pytest.mark.parametrize("fmt, rows, out_dim", [
    (rein.Q4_K, 520, 16384),                          # five groups of 17 tiles: bands of three and two; 512 of 640 units whole, the last row block in part
    (rein.Q6_K, 1100, 7424),                          # nine groups of 35 tiles: three bands of three; 56 row blocks and eight units of the next
    (rein.Q5_K, 1030, 8192),                          # 576 units, the last tile almost empty
])
def test_every_unit_of_a_banded_round_once(fmt, rows, out_dim):
    in_dim = 256
    packed = weights(fmt, in_dim, out_dim, rows)
    x = np.random.default_rng(rows).standard_normal((rows, in_dim)).astype(np.float32)
    got = matmul(fmt, packed, x, out_dim, 2)
    assert_close_f32(got, orc.matvec_q8(fmt, packed, in_dim, out_dim, orc.quantize_q8(x), rows), what=f"fmt {fmt}")


@pytest.mark.parametrize("fmt, mode, rows, in_dim, out_dim", [
    (rein.Q6_K, 3, 33, 768, 513),                     # few operations: groups of one and two tiles to 128 rows, above groups of four
    (rein.Q6_K, 3, 128, 768, 520),
    (rein.Q6_K, 2, 129, 768, 1030),
    (rein.Q4_K, 3, 33, 1024, 513),                    # below four million weights
    (rein.Q4_K, 3, 33, 1024, 4095),                   # 64 pieces of 128 x 32
    (rein.Q4_K, 3, 65, 4096, 2560),                   # 60
    (rein.Q4_K, 3, 128, 2048, 4096),                  # 128
    (rein.Q5_K, 3, 33, 768, 4000),                    # 64
    (rein.Q5_K, 3, 97, 1024, 6001),                   # 188
    (rein.Q5_K, 2, 128, 2560, 5200),                  # 164
    (rein.Q6_K, 3, 40, 2048, 512),                    # narrow matrices
    (rein.Q4_K, 3, 33, 1024, 1),
    (rein.Q5_K, 3, 65, 17408, 640),                   # less than a twentieth of the contraction
])
def test_the_rule_takes_the_tiles_and_the_scratch_holds_their_plan(fmt, mode, rows, in_dim, out_dim):
    packed = weights(fmt, in_dim, out_dim, rows)
    x = np.random.default_rng(rows).standard_normal((rows, in_dim)).astype(np.float32)
    got = matmul(fmt, packed, x, out_dim, 1)
    assert np.array_equal(got.view(np.uint32), matmul(fmt, packed, x, out_dim, mode).view(np.uint32))
    assert_close_f32(got, orc.matvec_q8(fmt, packed, in_dim, out_dim, orc.quantize_q8(x), rows), what=f"fmt {fmt}")
