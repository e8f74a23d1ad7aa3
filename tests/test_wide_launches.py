"""The GEMMs of rein_matmul_ws on 32 x 128 wavefront tiles: what the size query costs and holds, and which kernels are launched (CPU:
tests/launches.py records the launches)."""
import random
import statistics
import time

import pytest

import reinstinct_amd as rein
from launches import P, record
from reinstinct_amd import runtime

INT8 = {rein.Q8_0: "q8_0", rein.Q4_0: "q4_0", rein.IQ4_XS: "iq4xs", rein.IQ3_S: "iq3s"}
K_QUANTS = {rein.Q4_K: "q4k", rein.Q5_K: "q5k", rein.Q6_K: "q6k"}


@pytest.mark.parametrize("fmt", [rein.Q8_0, rein.Q5_K, rein.Q6_K])
def test_the_size_query_prices_no_plans(fmt):
    """a program whose prompts differ in length asks before each of them"""
    took = []
    for rows in range(101, 1101, 10):
        start = time.perf_counter()
        runtime.matmul_scratch_bytes(fmt, 5120, rows)
        took.append(time.perf_counter() - start)
    assert statistics.median(took) < 30e-6


@pytest.mark.parametrize("mode, tags", [(2, {f: "x8_" + t for f, t in INT8.items()}), (3, {f: "xf_" + t for f, t in K_QUANTS.items()})])
def test_a_scratch_of_the_size_asked_for_holds_every_plan(mode, tags, tmp_path):
    """whatever the number of weight rows: a launch that did not fit would quietly be another one"""
    rng = random.Random(mode)
    shapes = [(f, k, rows) for f in tags for k, rows in
              [(256, 9), (512, 33), (768, 4097), (1024, 64), (2048, 400), (4096, 128), (17408, 45), (5120, 65535),
               *((256 * rng.randint(1, 72), rng.randint(9, 3000)) for _ in range(8))]]
    pin = [("option", ["REIN_MMQXH", mode])]
    sizes = record(pin + [("matmul_scratch_bytes", list(s)) for s in shapes], tmp_path)[1:]
    calls = [("matmul_ws", [f, P, P, P, k, n, rows, P, size["value"]]) for (f, k, rows), size in zip(shapes, sizes)
             for n in (1, 640, 5120, 17408, *(rng.randint(1, 80000) for _ in range(16)))]
    for call, done in zip(calls, record(pin + calls, tmp_path)[1:]):
        names = [r[0] for r in done["launches"]]
        tag = tags[call[1][0]]
        assert names[:2] == [f"rein_{tag[:3]}quantize", "rein_" + tag] and names[2:] in ([], [f"rein_{tag[:3]}sum"]), call


def wide(done):
    return any(r[0].startswith(("rein_x8_", "rein_xf_", "rein_xh_")) for r in done["launches"])


def taken(cases, tmp_path):
    sizes = record([("matmul_scratch_bytes", [f, k, rows]) for f, k, _, rows, _ in cases], tmp_path)
    done = record([("matmul_ws", [f, P, P, P, k, n, rows, P, size["value"]]) for (f, k, n, rows, _), size in zip(cases, sizes)], tmp_path)
    for case, d in zip(cases, done):
        kernels = [r[0] for r in d["launches"]]
        assert wide(d) == bool(case[-1]), (case, kernels)
        assert not wide(d) or f"rein_{case[-1]}" in kernels, (case, kernels)


def test_where_the_int8_gemm_is_taken(tmp_path):
    q8, q4, i4, i3 = rein.Q8_0, rein.Q4_0, rein.IQ4_XS, rein.IQ3_S
    taken([(q8, 512, 4096, 64, 0), (q8, 512, 32, 33, 0), (i3, 256, 151936, 512, 0), (q4, 512, 65536, 2048, 0),          # short contractions
           (q8, 768, 8192, 32, "x8_q8_0"), (q8, 768, 8320, 32, 0), (i4, 1024, 2048, 128, "x8_iq4xs"), (i4, 1024, 2048, 129, 0),          # 64 pieces and 65
           (q4, 1280, 32768, 128, 0), (q4, 1280, 32768, 129, "x8_q4_0"), (q4, 768, 65536, 512, 0),          # 1024 pieces and 1280
           (i3, 2048, 8192, 128, "x8_iq3s"), (i3, 2048, 8192, 129, 0), (q8, 2048, 8192, 256, 0), (q8, 2048, 8192, 257, "x8_q8_0"),
           (q8, 1536, 32, 17, "x8_q8_0"), (i4, 2304, 8192, 256, "x8_iq4xs"), (q8, 5120, 17408, 2048, "x8_q8_0"),
           (q8, 3072, 1024, 9, "x8_q8_0"), (q8, 2816, 256, 16, 0), (q4, 5120, 1536, 16, 0), (q8, 8192, 2048, 9, "x8_q8_0"), (q8, 8192, 2080, 9, 0),
           (i4, 11008, 3584, 12, "x8_iq4xs"), (q4, 5120, 14336, 9, 0), (q4, 5120, 16384, 9, "x8_q4_0"), (i3, 6144, 12288, 16, "x8_iq3s"),
           (q8, 6144, 12288, 16, 0), (q4, 5120, 18464, 16, 0)], tmp_path)


def test_where_the_small_groups_are_taken(tmp_path):
    q4, q5, q6 = rein.Q4_K, rein.Q5_K, rein.Q6_K
    taken([(q6, 256, 32768, 17, 0), (q6, 512, 16384, 32, "xf_q6k"), (q6, 8192, 8192, 9, 0), (q6, 11008, 8192, 9, "xf_q6k"), (q6, 6144, 10240, 16, "xf_q6k"), (q6, 8192, 18464, 16, 0), (q6, 2048, 1024, 32, 0),
           (q4, 768, 8192, 32, 0), (q4, 1024, 8192, 32, "xf_q4k"), (q5, 1024, 8224, 17, 0), (q4, 1280, 12288, 24, "xf_q4k"), (q4, 4096, 12320, 24, 0),
           (q5, 9984, 12288, 32, "xf_q5k"), (q5, 10240, 5152, 32, 0), (q5, 17408, 5120, 17, "xf_q5k"), (q4, 14336, 10240, 24, 0),
           (q5, 768, 32768, 33, 0), (q5, 1024, 32768, 64, "xf_q5k"), (q5, 2816, 32800, 64, 0), (q5, 3072, 32800, 64, "xf_q5k"), (q5, 2816, 49184, 33, "xf_q5k"),
           (q5, 256, 151936, 64, 0),
           (q4, 11008, 8192, 9, 0), (q4, 11008, 6144, 9, "xf_q4k"), (q4, 10752, 8224, 16, "xf_q4k"), (q4, 8192, 14336, 12, 0), (q4, 6144, 16384, 9, 0),
           (q4, 5120, 17408, 9, "xf_q4k"), (q5, 6144, 18432, 16, "xf_q5k"), (q5, 11008, 8192, 9, 0), (q5, 17408, 5120, 12, 0)], tmp_path)


def test_narrow_matrices_of_the_k_quants(tmp_path):
    """33 to 128 rows: the small groups down to one row of weights"""
    tags = {f: "xf_" + t for f, t in K_QUANTS.items()}
    taken([(f, k, n, rows, tags[f]) for f in tags for k, n, rows in [(1024, 1, 33), (2048, 512, 40), (2048, 513, 40), (2048, 512, 64), (1280, 96, 128), (3072, 32, 33 if f == rein.Q6_K else 65)]] +
          [(rein.Q5_K, 17408, n, 65, "xf_q5k") for n in (32, 512, 513, 640, 832)] + [(rein.Q4_K, 768, 512, 40, 0), (rein.Q5_K, 512, 512, 40, 0), (rein.Q6_K, 512, 512, 40, 0)] +
          # Q4_K by pieces of 128 x 32: 64, 128 and 256
          [(rein.Q4_K, k, n, rows, tags[rein.Q4_K] if yes else 0) for k, n, rows, yes in
           [(1280, 4096, 64, 1), (1280, 4224, 64, 0), (1536, 8192, 64, 1), (1536, 8320, 64, 0), (2304, 8320, 64, 0), (2560, 16384, 64, 1), (2560, 16512, 64, 0),
            (1792, 2048, 128, 1), (1792, 2176, 128, 0), (2048, 4096, 128, 1), (2048, 4224, 128, 0), (3840, 4096, 128, 1), (4096, 2688, 95, 1), (4096, 2816, 95, 0)]], tmp_path)


def test_where_the_exact_dot_gemm_of_q5_k_is_taken(tmp_path):
    q5, kernel = rein.Q5_K, "xh_q5k"
    taken([(q5, 1536, 4064, 1024, 0), (q5, 1536, 4096, 1024, kernel), (q5, 2816, 3072, 1024, 0), (q5, 3072, 512, 1024, kernel), (q5, 2816, 18944, 1023, 0),
           (q5, 3072, 17408, 160, 0), (q5, 3072, 17408, 161, kernel), (q5, 4096, 17408, 160, kernel), (q5, 17408, 832, 65, "xf_q5k"), (q5, 17408, 1024, 65, kernel),
           (q5, 17408, 640, 101, kernel), (q5, 8192, 640, 100, kernel)], tmp_path)


def test_the_sum_has_workgroups_for_the_tiles_there_are(tmp_path):
    for fmt, k, n, rows in [(rein.Q5_K, 17408, 5120, 45), (rein.Q8_0, 17408, 5120, 20), (rein.Q6_K, 17408, 5120, 777), (rein.Q8_0, 5120, 17408, 300)]:
        size = runtime.matmul_scratch_bytes(fmt, k, rows)
        (image, *_), (gemm, *_), (total, grid, *_) = record([("matmul_ws", [fmt, P, P, P, k, n, rows, P, size])], tmp_path)[0]["launches"]
        assert total.endswith("_sum") and grid[1] % 4 == 0 and grid[1] // 4 <= min(4 if gemm[6] != "f" else 2, (rows + 31) // 32), (gemm, grid)
