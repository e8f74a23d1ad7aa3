"""The on-disk matvec with its activations in LDS (rein_mvd_<fmt>) where it can go wrong: rows of less than a trip, of a trip and a
part, more rows than one pass of the grid with a remainder, and shapes that take the kernels without LDS (a contraction that does not
fit; few rows of Q6_K and Q8_0)."""
import numpy as np
import pytest

import reinstinct_amd as rein
from reinstinct_amd import hip, runtime
from reinstinct_amd._lib import init
from oracle import orc
from helpers import assert_close_f32, dev, random_raw_weights

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    init()
    hip.set_device(0)
    yield
    hip.synchronize()


@pytest.mark.parametrize("fmt", [rein.Q4_K, rein.Q5_K, rein.Q6_K, rein.Q8_0])
@pytest.mark.parametrize("in_dim,out_dim", [(256, 1), (1280, 6), (256, 2049), (1280, 2054), (1024, 16389), (2304, 8195), (131072, 3)])
def test_ondisk_lds_matvec(fmt, in_dim, out_dim):
    raw = random_raw_weights(fmt, in_dim, out_dim, seed=fmt + out_dim)
    x = np.random.default_rng(in_dim).standard_normal((1, in_dim)).astype(np.float32)
    xq = orc.quantize_q8(x)
    dy = dev(np.full(out_dim + 8, np.nan, np.float32))
    runtime.matvec_ondisk_xq8(fmt, dev(raw), dev(xq), dy, in_dim, out_dim)
    hip.synchronize()
    got = dy.to_host(np.float32)
    assert np.all(np.isnan(got[out_dim:]))
    want = orc.matvec_q8(fmt, orc.repack_for_matvec(fmt, raw, in_dim, out_dim), in_dim, out_dim, xq, 1)[0]
    assert_close_f32(got[:out_dim], want, what=f"on-disk fmt {fmt} {in_dim} -> {out_dim}")


@pytest.mark.parametrize("in_dim,out_dim", [(64, 5), (64, 2053), (320, 8200)])
def test_ondisk_q8_0_pairs_of_blocks(in_dim, out_dim):
    raw = random_raw_weights(rein.Q8_0, in_dim, out_dim, seed=in_dim)
    xq = orc.quantize_q8(np.random.default_rng(7).standard_normal((1, in_dim)).astype(np.float32))
    dy = dev(np.full(out_dim, np.nan, np.float32))
    runtime.matvec_ondisk_xq8(rein.Q8_0, dev(raw), dev(xq), dy, in_dim, out_dim)
    hip.synchronize()
    want = orc.matvec_q8(rein.Q8_0, orc.repack_for_matvec(rein.Q8_0, raw, in_dim, out_dim), in_dim, out_dim, xq, 1)[0]
    assert_close_f32(dy.to_host(np.float32), want, what="Q8_0 pairs")


# in_dim / 32 padded to whole 256: (256 + pad) / 8 bytes of quants and 4, 8 or 12 of scales and sums for each, in 160 KiB of LDS
LARGEST = {rein.Q4_K: 124672, rein.Q5_K: 124672, rein.Q6_K: 109056, rein.Q8_0: 137728}


@pytest.mark.parametrize("fmt", list(LARGEST))
@pytest.mark.parametrize("more", [0, 256])
def test_the_longest_contraction_that_fits_the_lds(fmt, more):
    """and the next one, which does not; three rows over and over, so that few rows are computed by the oracle"""
    in_dim, out_dim, few = LARGEST[fmt] + more, 2052, 3
    raw = random_raw_weights(fmt, in_dim, few, seed=fmt + more)
    xq = orc.quantize_q8(np.random.default_rng(fmt).standard_normal((1, in_dim)).astype(np.float32))
    dy = dev(np.full(out_dim, np.nan, np.float32))
    runtime.matvec_ondisk_xq8(fmt, dev(np.tile(raw, out_dim // few)), dev(xq), dy, in_dim, out_dim)
    hip.synchronize()
    want = orc.matvec_q8(fmt, orc.repack_for_matvec(fmt, raw, in_dim, few), in_dim, few, xq, 1)[0]
    assert_close_f32(dy.to_host(np.float32), np.tile(want, out_dim // few), what=f"fmt {fmt} {in_dim}")


BLOCK = {rein.Q4_K: (144, 0), rein.Q5_K: (176, 0), rein.Q6_K: (210, 208), rein.Q8_0: (34, 0)}        # bytes, where d lies


@pytest.mark.parametrize("fmt", list(BLOCK))
def test_infinite_and_nan_scales_stay_in_their_row(fmt):
    in_dim, out_dim = 1280, 2311
    raw = random_raw_weights(fmt, in_dim, out_dim, seed=fmt)
    size, at = BLOCK[fmt]
    rows = raw.reshape(out_dim, -1, size)
    bad = {0: np.nan, 5: np.inf, 1024: -np.inf, out_dim - 1: np.nan}
    for r, v in bad.items():
        rows[r, r % rows.shape[1], at:at + 2] = np.array([v], np.float16).view(np.uint8)
    xq = orc.quantize_q8(np.random.default_rng(fmt).standard_normal((1, in_dim)).astype(np.float32))
    dy = dev(np.zeros(out_dim, np.float32))
    runtime.matvec_ondisk_xq8(fmt, dev(raw), dev(xq), dy, in_dim, out_dim)
    hip.synchronize()
    got = dy.to_host(np.float32)
    assert set(np.flatnonzero(~np.isfinite(got))) == set(bad)
    want = orc.matvec_q8(fmt, orc.repack_for_matvec(fmt, raw, in_dim, out_dim), in_dim, out_dim, xq, 1)[0]
    fine = np.isfinite(got)
    assert_close_f32(got[fine], want[fine], what=f"fmt {fmt}")


@pytest.mark.parametrize("fmt", list(BLOCK))
@pytest.mark.parametrize("special", [np.inf, -np.inf, np.nan])
def test_infinite_and_nan_activations_reach_every_row(fmt, special):
    """an activation block whose scale (infinity) or sum (NaN) is not a number: as in the matvec over the repacked rows"""
    in_dim, out_dim = 1280, 2100
    raw = random_raw_weights(fmt, in_dim, out_dim, seed=fmt)
    x = np.random.default_rng(fmt).standard_normal(in_dim).astype(np.float32)
    x[700] = special
    dq, dy, dz = hip.DeviceBuf(in_dim // 32 * 40), dev(np.zeros(out_dim, np.float32)), dev(np.zeros(out_dim, np.float32))
    runtime.quantize_q8(dev(x), dq, in_dim)
    runtime.matvec_ondisk_xq8(fmt, dev(raw), dq, dy, in_dim, out_dim)
    runtime.matvec_xq8(fmt, dev(orc.repack_for_matvec(fmt, raw, in_dim, out_dim)), dq, dz, in_dim, out_dim)
    hip.synchronize()
    got, other = dy.to_host(np.float32), dz.to_host(np.float32)
    assert np.array_equal(np.isfinite(got), np.isfinite(other))
    assert np.isinf(special) <= (not np.isfinite(got).any())
    fine = np.isfinite(got)
    assert_close_f32(got[fine], other[fine], what=f"fmt {fmt}")
