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
