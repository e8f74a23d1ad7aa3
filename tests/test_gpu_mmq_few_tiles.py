"""The exact-dot fp16 GEMM in groups of one and two token tiles (rein_xf_*, kernels/mmq_exact16.h): the edges of its groups, ranges and
rounds against the oracle and beside the groups of four, and the activations in the scratch."""
import numpy as np
import pytest

import reinstinct_amd as rein
from oracle import orc
from reinstinct_amd import hip, quant, runtime
from reinstinct_amd._lib import init, set_option
from tests.helpers import assert_close_f32

pytestmark = pytest.mark.gpu
OPTIONS = ("REIN_MMQXH", "REIN_MMQXH_SPLIT", "REIN_MMQXH_GROUPS")


@pytest.fixture(autouse=True)
def _options():
    init()
    hip.set_device(0)
    yield
    for name in OPTIONS:
        set_option(name, None)


def weights(fmt, in_dim, out_dim, seed):
    w = np.random.default_rng(seed).standard_normal((out_dim, in_dim)).astype(np.float32) * 0.02
    return quant.repack_for_matvec(fmt, quant.quantize_weights(fmt, w), in_dim, out_dim)


def matmul(fmt, packed, x, out_dim, mode, split=None, groups=None):
    rows, in_dim = x.shape
    for name, v in zip(OPTIONS, (mode, split, groups)):
        set_option(name, None if v is None else str(v))
    size = runtime.matmul_scratch_bytes(fmt, in_dim, rows)
    dw, dx, scratch = hip.DeviceBuf.from_host(packed), hip.DeviceBuf.from_host(x), hip.DeviceBuf(size)
    guard = 64
    dy = hip.DeviceBuf.from_host(np.full(rows * out_dim + guard, 12345.0, np.float32))
    print(f"fmt {fmt} rows {rows} in {in_dim} out {out_dim} mode {mode} split {split} groups {groups}", flush=True)
    runtime.matmul_ws(fmt, dw, dx, dy, in_dim, out_dim, rows, scratch, size)
    hip.synchronize()
    y = dy.to_host(np.float32)
    assert (y[rows * out_dim:] == 12345.0).all()
    return y[:rows * out_dim].reshape(rows, out_dim), scratch.to_host(np.uint8)


@pytest.mark.parametrize("fmt", [rein.Q4_K, rein.Q5_K, rein.Q6_K])
@pytest.mark.parametrize("rows, in_dim, out_dim, split, groups", [
    (9, 256, 5, None, None),             # one tile, one superblock, a row block almost empty, scalar stores
    (32, 1024, 200, 4, None),            # padded weight rows; a range per superblock
    (33, 768, 130, 3, 1),                # a group of two tiles
    (33, 768, 130, 2, 2),                # two groups of one
    (129, 2304, 257, 4, 3),              # groups of two, two and one, uneven ranges of nine superblocks
    (64, 256, 49408, None, 2),           # 772 units: a whole round of 768 and a tail
    (96, 512, 33024, 2, 3),              # 774 units, the first that is cut in the middle of a row block
])
def test_against_the_oracle(fmt, rows, in_dim, out_dim, split, groups):
    packed = weights(fmt, in_dim, out_dim, rows)
    x = np.random.default_rng(in_dim).standard_normal((rows, in_dim)).astype(np.float32)
    x[0] *= 1e-20
    x[rows // 2] = 0.0
    x[rows - 1] *= 1e20
    got, scratch = matmul(fmt, packed, x, out_dim, 3, split, groups)
    xq = orc.quantize_q8(x)
    assert np.array_equal(scratch[:xq.size], xq)      # where every launch of rein_matmul_ws leaves them
    want = orc.matvec_q8(fmt, packed, in_dim, out_dim, xq, rows)
    scale = np.abs(x).max(axis=1, keepdims=True) + (np.abs(x).max(axis=1, keepdims=True) == 0)
    assert_close_f32(got / scale, want / scale, what=f"fmt {fmt}")


@pytest.mark.parametrize("fmt", [rein.Q4_K, rein.Q5_K, rein.Q6_K])
def test_the_bits_of_the_larger_groups(fmt):
    """the same products and sums whatever the groups, given the same ranges; infinities and NaN where they are there"""
    rows, in_dim, out_dim = 100, 1536, 200
    packed = weights(fmt, in_dim, out_dim, 1)
    x = np.random.default_rng(2).standard_normal((rows, in_dim)).astype(np.float32)
    for r, v in {3: np.inf, 40: np.nan, 99: -np.inf}.items():
        x[r, 11 * r] = v
    want = matmul(fmt, packed, x, out_dim, 2, 2)[0]
    finite = np.isfinite(want)
    assert not finite[[3, 99]].any() and finite.sum() > rows * out_dim * 0.9
    for groups in (2, 4):
        got = matmul(fmt, packed, x, out_dim, 3, 2, groups)[0]
        assert np.array_equal(np.isfinite(got), finite) and np.array_equal(got[finite], want[finite])


def test_capture():
    fmt, rows, in_dim, out_dim = rein.Q5_K, 45, 4096, 1280
    x = np.random.default_rng(6).standard_normal((rows, in_dim)).astype(np.float32)
    size = runtime.matmul_scratch_bytes(fmt, in_dim, rows)
    dw, dx, scratch, dy = hip.DeviceBuf.from_host(weights(fmt, in_dim, out_dim, 5)), hip.DeviceBuf.from_host(x), hip.DeviceBuf(size), hip.DeviceBuf(rows * out_dim * 4)

    def call(stream=None):
        runtime.matmul_ws(fmt, dw, dx, dy, in_dim, out_dim, rows, scratch, size, stream)

    call()
    hip.synchronize()
    eager = dy.to_host(np.uint32)
    stream = hip.Stream()
    stream.begin_capture()
    call(stream)
    graph = stream.end_capture().instantiate()
    for _ in range(3):
        runtime.quantize_q8(dx, scratch, in_dim, rows)          # the program's own work on the same scratch between replays
        hip.synchronize()
        graph.launch(stream)
        stream.synchronize()
        assert np.array_equal(dy.to_host(np.uint32), eager)
