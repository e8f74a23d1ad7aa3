"""The few-row kernels in the builds that differ in how they load the weights, on both sides of the sizes where one follows the
other, with a remainder of rows; one matrix and several in one launch; every build against the others, bit for bit."""
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


# plain, nontemporal (1-2 rows; mixed from 3 or 5 rows), mixed, padded rows
@pytest.mark.parametrize("fmt,in_dim,out_dim", [(rein.Q4_K, 1280, 1031), (rein.Q5_K, 2560, 3701), (rein.Q6_K, 3072, 6151),
                                                (rein.Q4_K, 5120, 10247), (rein.Q8_0, 4096, 6149), (rein.Q8_0, 1536, 17411)])
def test_loads(fmt, in_dim, out_dim):
    raw = random_raw_weights(fmt, in_dim, out_dim, seed=fmt + out_dim)
    w = orc.repack_for_matvec(fmt, raw, in_dim, out_dim)
    dw = dev(w)
    xq = orc.quantize_q8(np.random.default_rng(in_dim).standard_normal((8, in_dim)).astype(np.float32))
    dx = dev(xq)
    want = orc.matvec_q8(fmt, w, in_dim, out_dim, xq, 8).reshape(8, out_dim)
    for rows in (1, 2, 3, 4, 5, 8):
        dy = dev(np.full(rows * out_dim + 8, np.nan, np.float32))
        runtime.mmq_xq8(fmt, dw, dx, dy, in_dim, out_dim, rows)
        hip.synchronize()
        got = dy.to_host(np.float32)
        assert np.all(np.isnan(got[rows * out_dim:]))
        assert_close_f32(got[:rows * out_dim].reshape(rows, out_dim), want[:rows], what=f"fmt {fmt} {in_dim} -> {out_dim}, {rows} rows")


@pytest.mark.parametrize("outs", [(1031, 260), (6144, 1031), (17411, 12001)])
@pytest.mark.parametrize("rows", [1, 2])
def test_loads_of_several_matrices(outs, rows):
    in_dim, fmts = 2560, (rein.Q4_K, rein.Q6_K)
    xq = orc.quantize_q8(np.random.default_rng(5).standard_normal((rows, in_dim)).astype(np.float32))
    ws = [orc.repack_for_matvec(f, random_raw_weights(f, in_dim, n, seed=n), in_dim, n) for f, n in zip(fmts, outs)]
    dws = [dev(w) for w in ws]
    ys = [dev(np.full(rows * n, np.nan, np.float32)) for n in outs]
    runtime.matvec_multi_xq8(list(fmts), dws, ys, list(outs), dev(xq), in_dim, rows)
    hip.synchronize()
    for f, n, w, y in zip(fmts, outs, ws, ys):
        assert_close_f32(y.to_host(np.float32).reshape(rows, n), orc.matvec_q8(f, w, in_dim, n, xq, rows).reshape(rows, n), what=f"fmt {f} -> {n}")


FAMILIES = {                                        # options that keep every row count on one family
    "rein_mv_": {"REIN_MV_LDS": 0, "REIN_QUAD_LDS": 0, "REIN_SKINNY_FROM": 99, "REIN_QUAD_FROM": 99},
    "rein_mvl_": {"REIN_MV_LDS": 1},
    "rein_mvql_": {"REIN_QUAD_LDS": 1},
}


@pytest.mark.parametrize("family, rows", [("rein_mv_", (1, 2, 4)), ("rein_mvl_", (2, 4)), ("rein_mvql_", (4, 8, 16))])
@pytest.mark.parametrize("fmt", [rein.Q4_0, rein.Q4_K, rein.Q5_K, rein.Q6_K, rein.Q8_0, rein.IQ4_XS, rein.IQ3_S])
def test_every_build_gives_the_same_bits(family, rows, fmt, options):
    in_dim, out_dim = 1536, 1031
    w = orc.repack_for_matvec(fmt, random_raw_weights(fmt, in_dim, out_dim, seed=fmt), in_dim, out_dim)
    dw, dx = dev(w), dev(orc.quantize_q8(np.random.default_rng(fmt).standard_normal((16, in_dim)).astype(np.float32)))
    for name, value in FAMILIES[family].items():
        options.set(name, value)
    for n in rows:
        seen = {}
        for build in (0, 1, 2):
            options.set("REIN_MV_LOADS", build)
            kernel = runtime.matvec_kernel_name(fmt, in_dim, out_dim, n)
            assert kernel.startswith(family)
            dy = dev(np.full(n * out_dim, np.nan, np.float32))
            runtime.mmq_xq8(fmt, dw, dx, dy, in_dim, out_dim, n)
            hip.synchronize()
            seen[kernel] = dy.to_host(np.uint32)
        assert len(seen) == (3 if n <= 4 else 2)
        first = next(iter(seen.values()))
        assert not np.isnan(first.view(np.float32)).any()
        assert all(np.array_equal(v, first) for v in seen.values())


@pytest.mark.parametrize("rows", [1, 2, 4])
def test_every_build_of_the_multi_matrix_launch_gives_the_same_bits(rows, options):
    in_dim, outs, fmts = 1536, (517, 130, 65), (rein.Q5_K, rein.Q6_K, rein.Q8_0)
    dx = dev(orc.quantize_q8(np.random.default_rng(3).standard_normal((rows, in_dim)).astype(np.float32)))
    dws = [dev(orc.repack_for_matvec(f, random_raw_weights(f, in_dim, n, seed=n), in_dim, n)) for f, n in zip(fmts, outs)]
    got = []
    for build in (0, 1, 2):
        options.set("REIN_MV_LOADS", build)
        ys = [dev(np.full(rows * n, np.nan, np.float32)) for n in outs]
        runtime.matvec_multi_xq8(list(fmts), dws, ys, list(outs), dx, in_dim, rows)
        hip.synchronize()
        got.append(np.concatenate([y.to_host(np.uint32) for y in ys]))
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
    assert not np.isnan(got[0].view(np.float32)).any()
