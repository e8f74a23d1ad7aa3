"""CPU-side tests of the product's host code: the C ABI loads and exports every
symbol include/rein.h declares, the src/quant mirror reproduces the oracle's
repack byte for byte, the synthetic quantizers emit valid blocks, the dispatch
thresholds and the error model.  No compute call is made (no GPU here)."""
import ctypes as C
import os
import re

import numpy as np
import pytest

import reinstinct_amd as rein
from reinstinct_amd import _lib, quant, runtime
from oracle import orc
from helpers import random_raw_weights, rel_l2

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ALL = [rein.Q4_0, rein.Q8_0, rein.Q4_K, rein.Q5_K, rein.Q6_K, rein.IQ4_XS]


def test_header_symbols_all_exported_and_typed():
    text = open(os.path.join(ROOT, "include", "rein.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    declared = set(re.findall(r"\b(rein_[a-z0-9_]+)\s*\(", text))
    declared -= {"rein_moe_shape"}
    assert len(declared) > 55
    lib = _lib.load()
    for name in sorted(declared):
        assert hasattr(lib, name), f"{name} declared in rein.h but not exported by librein.so"
    assert declared == set(_lib.SIGNATURES), declared ^ set(_lib.SIGNATURES)


def test_format_ids_match_reference_enum():  # src/gguf/types.rs:16-35
    assert (rein.Q4_0, rein.Q8_0, rein.Q4_K, rein.Q5_K, rein.Q6_K, rein.IQ4_XS) == (2, 8, 12, 13, 14, 23)
    for fmt in ALL:
        assert quant.block_size(fmt) == orc.block_size(fmt)
        assert quant.bytes_per_block(fmt) == orc.bytes_per_block(fmt)
    assert quant.block_size(99) == 0


@pytest.mark.parametrize("fmt", ALL)
@pytest.mark.parametrize("in_dim,out_dim", [(256, 1), (512, 3), (768, 5), (2048, 4), (5120, 2)])
def test_repack_matches_oracle_bytes(fmt, in_dim, out_dim):
    raw = random_raw_weights(fmt, in_dim, out_dim, seed=fmt * 7 + in_dim)
    got = quant.repack_for_matvec(fmt, raw, in_dim, out_dim)
    want = orc.repack_for_matvec(fmt, raw, in_dim, out_dim)
    assert quant.repacked_len(fmt, in_dim, out_dim) == want.size
    assert quant.repacked_n_sub_padded(in_dim) == orc.repacked_n_sub_padded(in_dim)
    assert np.array_equal(got, want)


def test_repack_threaded_path_matches_oracle():
    fmt, in_dim, out_dim = rein.Q5_K, 4096, 1100       # above the threading threshold, ragged split
    raw = random_raw_weights(fmt, in_dim, out_dim, seed=3)
    assert np.array_equal(quant.repack_for_matvec(fmt, raw, in_dim, out_dim),
                          orc.repack_for_matvec(fmt, raw, in_dim, out_dim))


def test_repack_small_blocks_odd_counts():
    for fmt in (rein.Q4_0, rein.Q8_0):
        for in_dim in (32, 96, 128, 160):
            raw = random_raw_weights(fmt, in_dim, 3, seed=in_dim)
            assert np.array_equal(quant.repack_for_matvec(fmt, raw, in_dim, 3),
                                  orc.repack_for_matvec(fmt, raw, in_dim, 3))


def test_repack_errors():
    raw = np.zeros(144, np.uint8)
    with pytest.raises(rein.ReinError) as e:
        quant.repack_for_matvec(rein.Q4_K, raw, 200, 1)        # the reference asserts (q4_k.rs:127)
    assert e.value.code == -3 and "multiple of 256" in str(e.value)
    with pytest.raises(rein.ReinError) as e:
        quant.repack_for_matvec(99, raw, 256, 1)
    assert e.value.code == -2


@pytest.mark.parametrize("fmt,tol", [(rein.Q8_0, 6e-3), (rein.Q6_K, 2e-2), (rein.Q5_K, 4e-2), (rein.Q4_K, 8e-2),
                                     (rein.Q4_0, 1.2e-1), (rein.IQ4_XS, 1.2e-1)])
def test_quantize_weights_valid_and_close(fmt, tol):
    rng = np.random.default_rng(fmt)
    w = (rng.standard_normal((16, 1024)) * 0.02).astype(np.float32)
    raw = quant.quantize_weights(fmt, w)
    assert raw.size == w.size // quant.block_size(fmt) * quant.bytes_per_block(fmt)
    deq = orc.dequantize_to_f32(fmt, raw, w.size).reshape(w.shape)
    assert np.all(np.isfinite(deq))
    assert rel_l2(deq, w) < tol
    # all-zero input stays zero and finite
    z = quant.quantize_weights(fmt, np.zeros(512, np.float32))
    assert np.all(orc.dequantize_to_f32(fmt, z, 512) == 0)


def test_quantize_weights_q8_0_matches_reference_quantizer():
    w = (np.random.default_rng(0).standard_normal(4096) * 0.02).astype(np.float32)
    assert np.array_equal(quant.quantize_weights(rein.Q8_0, w), orc.q8_0_quantize_from_f32(w))


def test_matmul_dispatch_thresholds():
    # 1 row -> matvec; 2..8 -> weight-streaming batched matvec (the reference
    # switches to its narrow MMQ at 5, prefill.rs:358,383); above -> MMQ.
    # Row counts are the reference's own sweep (prefill.rs:579-682).
    want = {1: "matvec", 4: "batched_matvec", 5: "batched_matvec", 8: "batched_matvec",
            15: "mmq", 16: "mmq", 20: "mmq"}
    for fmt in ALL:
        for n, path in want.items():
            assert runtime.matmul_path(fmt, n) == path
    with pytest.raises(rein.ReinError):
        runtime.matmul_path(99, 1)
    with pytest.raises(rein.ReinError):
        runtime.matmul_path(rein.Q4_K, 0)


def test_mmq_tile_plan():
    # 64-token tiles per row block of the MMQ launch: never more than fit, none where the
    # grid is resident at once (up to three 32-token workgroups per CU), all of them once
    # the grid is large, and a mix
    # with 32-token fillers in between (512 x 17408: 2176 small workgroups on 256 CUs)
    for fmt in ALL:
        for out_dim, p_rows in [(200, 70), (5120, 96), (17408, 128), (17408, 512), (5120, 2048), (151936, 4096)]:
            n64 = runtime.mmq_tile_plan(fmt, 5120, out_dim, p_rows)
            assert 0 <= n64 <= p_rows // 64
    assert runtime.mmq_tile_plan(rein.Q8_0, 5120, 200, 70) == 0
    assert runtime.mmq_tile_plan(rein.Q8_0, 5120, 5120, 128) == 0           # two 32-token workgroups per CU at most
    # three per CU resident: the 64-token kernel where its tile is cheap enough (Q8_0), else the 32-token one
    assert runtime.mmq_tile_plan(rein.Q8_0, 5120, 17408, 128) == 2
    assert runtime.mmq_tile_plan(rein.Q4_K, 5120, 17408, 128) == 0
    assert 1 <= runtime.mmq_tile_plan(rein.Q8_0, 5120, 17408, 512) <= 8
    assert runtime.mmq_tile_plan(rein.Q8_0, 5120, 17408, 2048) == 32
    assert runtime.mmq_tile_plan(rein.Q8_0, 5120, 151936, 4096) == 64
    # the price of a 64-token tile is per format: Q4_K's 32-token kernel is the leaner one unless the rows of
    # the slab are padded (a power-of-two sub-block count)
    assert runtime.mmq_tile_plan(rein.Q4_K, 5120, 151936, 4096) == 0
    assert runtime.mmq_tile_plan(rein.Q4_K, 8192, 151936, 4096) == 64
    assert runtime.mmq_tile_plan(rein.Q4_K, 5120, 34816, 256) == 0
    assert runtime.mmq_tile_plan(rein.Q8_0, 5120, 34816, 256) >= 1
    assert runtime.mmq_tile_plan(rein.Q4_K, 5120, 17408, 512) == runtime.mmq_tile_plan(rein.Q4_K, 5120, 17408, 512)
    with pytest.raises(rein.ReinError):
        runtime.mmq_tile_plan(99, 128, 128, 128)
    with pytest.raises(rein.ReinError):
        runtime.mmq_tile_plan(rein.Q4_K, 128, 0, 128)
    with pytest.raises(rein.ReinError):
        runtime.mmq_tile_plan(rein.Q4_K, 0, 128, 128)


def test_compute_calls_fail_loudly_without_runtime():
    lib = _lib.load()
    if lib.rein_is_loaded():
        pytest.skip("a GPU runtime is loaded in this process")
    rc = lib.rein_matvec_xq8(rein.Q4_K, 16, 16, 16, 256, 8, None)
    assert rc == -1 and b"no CPU fallback" in lib.rein_last_error()
    # argument errors are reported before anything touches the device
    assert lib.rein_matvec_xq8(rein.Q4_K, 16, 16, 16, 200, 8, None) == -3
    assert lib.rein_matvec_xq8(99, 16, 16, 16, 256, 8, None) == -2
    assert lib.rein_matvec_xq8(rein.Q4_K, 8, 16, 16, 256, 8, None) == -4 and b"16-byte aligned" in lib.rein_last_error()
    assert lib.rein_matvec_batched_xq8(rein.Q4_K, 16, 16, 16, 256, 8, 9, None) == -6
    assert lib.rein_quantize_q8(16, 16, 48, 1, None) == -3
    assert lib.rein_moe_grouped_gemm(rein.Q4_0, 16, 16, 16, 16, 1, 16, 16, 256, 8, 1, None) == -2
    assert lib.rein_moe_grouped_swiglu_q8(rein.Q4_0, 16, 16, 16, 16, 16, 1, 16, 16, 256, 32, 1, None) == -2
    assert lib.rein_moe_grouped_swiglu_q8(rein.Q8_0, 16, 16, 16, 16, 16, 1, 16, 16, 256, 40, 1, None) == -3   # ff not whole blocks


def test_moe_workspace_layout():
    sh = runtime.moe_shape(512, 2048, 128, 8, 768, rein.Q4_K, rein.Q6_K)
    n = runtime.moe_workspace_bytes(sh)
    ne = 512 * 8
    # ids, weights, perm, inverse perm; count, cursor; two offset arrays; quantized x; gathered x;
    # gate and up outputs; quantized intermediate; sorted down outputs (combined in place)
    need = ne * 4 * 4 + 128 * 4 * 2 + 129 * 4 * 2 + 512 * 64 * 40 + ne * 64 * 40 + ne * 768 * 4 * 2 + ne * 24 * 40 \
        + ne * 2048 * 4
    assert need <= n <= need + 14 * 256
    assert runtime.moe_gemm_bn() == 32


def test_options_table():
    # rein_set_option / rein_get_option / rein_reset_options: the library's launch switches live in one table
    # that the environment seeds once; names are enumerable, unknown names and malformed values are refused
    from reinstinct_amd import _lib
    lib = _lib.load()
    names = [lib.rein_option_name(i).decode() for i in range(lib.rein_option_count())]
    assert len(names) == len(set(names)) >= 20 and all(n.startswith("REIN_") for n in names)
    assert lib.rein_option_name(-1) is None and lib.rein_option_name(len(names)) is None
    _lib.reset_options()
    for n in names:
        assert _lib.get_option(n) is None
    _lib.set_option("REIN_MMQ6_FROM", 17)
    assert _lib.get_option("REIN_MMQ6_FROM") == 17
    # the table, not the environment, is what the entry points read: a later change of the environment is not seen
    import os
    os.environ["REIN_MMQ6_FROM"] = "999"
    try:
        assert _lib.get_option("REIN_MMQ6_FROM") == 17
        # 17 rows now have an fp6 workspace form; back to the default threshold they have none
        assert lib.rein_mmq_workspace_min_bytes(12, 512, 20) > 0
        _lib.set_option("REIN_MMQ6_FROM", None)
        assert _lib.get_option("REIN_MMQ6_FROM") is None
        assert lib.rein_mmq_workspace_min_bytes(12, 512, 20) == 0
    finally:
        os.environ.pop("REIN_MMQ6_FROM", None)
    _lib.set_option("REIN_MV_ROWS", "4")
    _lib.reset_options()
    assert _lib.get_option("REIN_MV_ROWS") is None
    for bad_name in ("REIN_NO_SUCH_OPTION", ""):
        with pytest.raises(_lib.ReinError) as err:
            _lib.set_option(bad_name, 1)
        assert err.value.code == -8
    for bad_value in ("-1", "abc", "12x", "4294967296"):
        with pytest.raises(_lib.ReinError) as err:
            _lib.set_option("REIN_MV_ROWS", bad_value)
        assert err.value.code == -3
    assert _lib.get_option("REIN_MV_ROWS") is None


def test_mmq_form_ws_follows_the_launch_rules():
    # rein_mmq_form_ws: host logic only -- which of the four launches rein_mmq_xq8_ws takes for a shape and a
    # workspace size (0 plain int8, 1 fp6 one token group per workgroup, 2 fp6 split-tail, 3 int8 split-tail)
    _lib.reset_options()
    Q4_K, Q6_K, Q8_0 = rein.Q4_K, rein.Q6_K, rein.Q8_0

    def form(fmt, k, n, m, bytes_=None):
        full = runtime.mmq_workspace_bytes(fmt, k, m)
        return runtime.mmq_form_ws(fmt, k, n, m, full if bytes_ is None else bytes_)

    # units = 128-row blocks x 4-tile token groups on 512 resident slots
    assert form(Q4_K, 5120, 17408, 512) == 2        # 544 units: one round + 32 that split eight ways
    assert form(Q4_K, 5120, 17408, 1024) == 2       # two rounds + 64 that split four ways
    assert form(Q4_K, 5120, 17408, 2048) == 1       # four rounds: the mixed launch
    assert form(Q4_K, 8192, 8192, 1024) == 1        # 512 units: no tail
    assert form(Q4_K, 8192, 28672, 256) == 2        # 448 units, no round, unsplit: from 341 units split-tail
    assert form(Q4_K, 8192, 10240, 512) == 1        # 320 units: 1.25 per CU, the mixed launch's narrower groups
    assert form(Q4_K, 5120, 17408, 256) in (0, 3)   # 272 units: too few for an unsplit fp6 launch
    assert form(Q4_K, 8192, 28672, 128) == 2        # from 128 rows when the GEMM is large and the tail splits
    assert form(Q4_K, 8192, 28672, 127) in (0, 3)   # below 128 rows never
    assert form(Q4_K, 4096, 4096, 128) in (0, 3)    # 2 M N K below 2.8e10
    assert form(Q4_K, 3584, 18944, 320) in (0, 3)   # ragged last token group (10 tiles in three groups), not even
    assert form(Q4_K, 5120, 17408, 1984) == 1       # ragged, but five and more 128-token workgroups per CU
    # the image alone admits the mixed launch only; less than the image is the caller's error, not a form
    image = runtime.mmq_workspace_min_bytes(Q4_K, 5120, 512)
    assert 0 < image < runtime.mmq_workspace_bytes(Q4_K, 5120, 512)
    assert form(Q4_K, 5120, 17408, 512, image) in (0, 1)
    assert form(Q4_K, 5120, 17408, 512, 0) == 0
    # int8 split-tail with 64-token units: behind one or two rounds when the tail has a CU per workgroup
    assert form(Q6_K, 17408, 5120, 1024) == 3       # 640 units: one round + 128, two ranges each
    assert form(Q6_K, 5120, 17408, 512) == 3        # 1088 units: two rounds + 64
    assert form(Q6_K, 5120, 17408, 1024) == 0       # four rounds
    assert form(Q6_K, 3584, 18944, 768) == 3        # 1776 units: three rounds + 240
    assert form(Q6_K, 8192, 10240, 640) == 0        # one round + 288 units: more than half the slots
    assert form(Q8_0, 5120, 17408, 1024) == 3       # Q8_0 keeps the form up to six rounds
    assert form(Q8_0, 5120, 17408, 2048) == 0       # eight rounds
    assert form(Q6_K, 17408, 5120, 64) == 3         # 40 units on 256 CUs
    assert form(Q6_K, 17408, 5120, 64, 0) == 0
    # every answer is a form, and the fp6 forms belong to Q4_K with whole superblocks from 128 rows
    rng = np.random.default_rng(5)
    for _ in range(3000):
        fmt = [Q4_K, Q6_K, Q8_0, rein.Q5_K, rein.Q4_0, rein.IQ4_XS, rein.IQ3_S][rng.integers(7)]
        k = int(rng.integers(1, 120)) * (32 if fmt in (Q8_0, rein.Q4_0) else 256)
        n, m = int(rng.integers(1, 40000)), int(rng.integers(1, 3000))
        got = form(fmt, k, n, m)
        assert got in (0, 1, 2, 3)
        if got in (1, 2):
            assert fmt == Q4_K and k % 256 == 0 and m >= 128 and 2.0 * m * n * k >= 2.8e10
        assert form(fmt, k, n, m, 0) == 0


def test_matvec_kernel_name_follows_the_dispatch_rules():
    # rein_matvec_kernel_name: host logic only -- which kernel 1..32 activation rows launch for a shape, by the rules
    # beside use_mvl / use_mvql / use_quad in rein_api.cpp and the option table
    import reinstinct_amd as rein
    from reinstinct_amd import _lib
    _lib.reset_options()
    name = runtime.matvec_kernel_name
    # one row: dot4, rows per wavefront by the width
    assert name(rein.Q4_K, 5120, 5120, 1) == "rein_mv_q4k_r2_b1"
    assert name(rein.Q4_K, 5120, 34816, 1) == "rein_mv_q4k_r4_b1_m"
    # two rows: LDS-staged dot4 at long contractions and, for Q4_K, against many rows; dot4 otherwise
    assert name(rein.Q4_K, 17408, 5120, 2) == "rein_mvl_q4k_r1_b2_m"
    assert name(rein.Q4_K, 5120, 34816, 2) == "rein_mvl_q4k_r2_b2_m"
    assert name(rein.Q6_K, 5120, 34816, 2) == "rein_mv_q6k_r2_b2_m"
    assert name(rein.Q8_0, 5120, 34816, 2) == "rein_mvl_q8_0_r2_b2_m"
    assert name(rein.Q8_0, 5120, 7168, 2) == "rein_mv_q8_0_r2_b2_m"
    assert name(rein.Q4_K, 5120, 5120, 2) == "rein_mv_q4k_r2_b2"
    # three to four rows: the sliced 4x4x4 kernel on narrow matrices (not Q8_0), LDS-staged dot4 for Q8_0 and mid sizes
    assert name(rein.Q4_K, 5120, 5120, 4) == "rein_mvql_q4k_t4_m"
    assert name(rein.Q8_0, 5120, 5120, 3) == "rein_mvl_q8_0_r1_b4_m"
    assert name(rein.Q4_K, 4096, 4096, 4) == "rein_mvl_q4k_r1_b4"
    assert name(rein.Q4_K, 5120, 34816, 4) == "rein_mvql_q4k_t4_m"
    assert name(rein.Q6_K, 5120, 34816, 4) == "rein_mvql_q6k_t4_m"
    assert name(rein.IQ4_XS, 5120, 34816, 4) == "rein_mvq_iq4xs_t4"           # the 4x4x4 kernel without LDS
    assert name(rein.Q4_K, 2048, 1536, 4) == "rein_mv_q4k_r1_b4_p"            # small matrices stay on dot4
    # five to eight rows
    assert name(rein.Q4_K, 17408, 5120, 8) == "rein_mvql_q4k_t8_m"
    assert name(rein.Q4_K, 5120, 34816, 8) == "rein_mmqs_q4k_v4"
    assert name(rein.Q6_K, 5120, 34816, 8) == "rein_mvql_q6k_t8_m"
    # nine and more rows arrive through rein_mmq_xq8
    assert name(rein.Q6_K, 5120, 5120, 12) == "rein_mvql_q6k_t16_m"
    assert name(rein.Q4_K, 5120, 5120, 12) == "rein_mmqs_q4k_v8"
    assert name(rein.Q4_K, 4096, 14336, 12) == "rein_mvql_q4k_t16_m"            # a contraction that is a multiple of 4096
    assert name(rein.Q4_K, 5120, 13824, 12) == "rein_mmqs_q4k_v8"
    assert name(rein.Q8_0, 13824, 5120, 16) == "rein_mvql_q8_0_t16_m"           # long contraction against at most 6144 rows
    assert name(rein.Q4_K, 5120, 5120, 32) == "rein_mvql_q4k_t32w"            # the build for sixteen wavefronts
    assert name(rein.Q6_K, 5120, 5120, 32) == "rein_mvql_q6k_t32"             # Q6_K: the build for eight
    assert name(rein.Q4_K, 5120, 34816, 32) == ""                             # token tiles
    assert name(rein.Q4_K, 5120, 5120, 33) == ""
    # options pin a family
    try:
        _lib.set_option("REIN_QUAD_LDS", 0)
        assert name(rein.Q4_K, 5120, 5120, 4) == "rein_mvl_q4k_r1_b4_m"
        assert name(rein.Q4_K, 17408, 5120, 8) == "rein_mmqs_q4k_v4"
        _lib.set_option("REIN_MV_LDS", 0)
        assert name(rein.Q4_K, 5120, 5120, 4) == "rein_mmqs_q4k_v2"
        _lib.set_option("REIN_SKINNY_FROM", 99)
        _lib.set_option("REIN_QUAD_FROM", 99)
        assert name(rein.Q4_K, 5120, 5120, 4) == "rein_mv_q4k_r2_b4_m"
        _lib.set_option("REIN_QUAD_FROM", 1)
        assert name(rein.Q4_K, 5120, 5120, 4) == "rein_mvq_q4k_t4"
    finally:
        _lib.reset_options()
    with pytest.raises(_lib.ReinError):
        name(rein.Q4_K, 5120, 0, 1)
    with pytest.raises(_lib.ReinError):
        name(99, 5120, 5120, 1)


def test_matvec_multi_checks_its_tables_on_the_host():
    """rein_matvec_multi_xq8 refuses bad tables before anything reaches a device"""
    from reinstinct_amd import runtime
    from reinstinct_amd._lib import ReinError
    ok = dict(fmts=[rein.Q4_K, rein.Q6_K], ws=[4096, 8192], ys=[4096, 8192], out_dims=[8, 8], xq=4096, in_dim=256)
    bad = [dict(fmts=[], ws=[], ys=[], out_dims=[]),                                   # no matrix
           dict(fmts=[rein.Q4_K] * 5, ws=[4096] * 5, ys=[4096] * 5, out_dims=[8] * 5),  # more than four
           dict(fmts=[rein.Q4_K, 99]),                                                 # unknown format
           dict(fmts=[rein.Q4_K, rein.Q5_1]),                                          # an expert-only format
           dict(ws=[4096, 0]), dict(ys=[0, 4096]), dict(ws=[4096, 4100]),              # NULL and misaligned pointers
           dict(out_dims=[8, 0]), dict(in_dim=200), dict(xq=0), dict(n_rows=0), dict(n_rows=5)]
    for change in bad:
        a = dict(dict(ok, n_rows=1), **change)
        with pytest.raises(ReinError):
            runtime.matvec_multi_xq8(a["fmts"], a["ws"], a["ys"], a["out_dims"], a["xq"], a["in_dim"], a["n_rows"])
