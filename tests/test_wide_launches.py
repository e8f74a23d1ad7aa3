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
