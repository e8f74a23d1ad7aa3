"""Which kernels the entry points launch (CPU: tests/launches.py records the launches instead of making them)."""
import random
import re

import reinstinct_amd as rein
from reinstinct_amd._lib import HSACO_PATH
from launches import P, record

DENSE = (rein.Q4_0, rein.Q4_K, rein.Q5_K, rein.Q6_K, rein.Q8_0, rein.IQ4_XS, rein.IQ3_S)


def test_the_reported_name_is_the_kernel_that_is_launched(tmp_path):
    """rein_matvec_kernel_name against the launch of the same product: sizes on both sides of every line between the builds that
    differ in their loads (6.5, 14, 25 and 28 MB), each family pinned, every format and row count"""
    rng = random.Random(5)
    shapes = [(1280, 1024), (2560, 3712), (3072, 6144), (5120, 5120), (5120, 10240), (4096, 14336), (1536, 17408), (17408, 5120), (5120, 34816)]
    shapes += [(256 * rng.randint(1, 72), rng.randint(1, 20000)) for _ in range(12)]
    calls = []
    for pin in ([], [("REIN_QUAD_LDS", 0)], [("REIN_QUAD_LDS", 0), ("REIN_MV_LDS", 0)], [("REIN_SKINNY_FROM", 99), ("REIN_QUAD_FROM", 99)],
                [("REIN_QUAD_FROM", 3)], [("REIN_QUAD_LDS", 1), ("REIN_QUAD_WIDE32", 0)], [("REIN_MV_LDS", 1)]):
        calls += [("option", [n, v]) for n, v in pin]
        for fmt in DENSE:
            for k, n in shapes:
                for rows in (1, 2, 3, 4, 5, 8, 12, 16, 24, 32):
                    calls += [("matvec_kernel_name", [fmt, k, n, rows]), ("mmq_xq8", [fmt, P, P, P, k, n, rows])]
        calls += [("option", [n, None]) for n, _ in pin]
    done = record(calls, tmp_path)
    builds = set()
    for i, (name, args) in enumerate(calls):
        if name != "matvec_kernel_name":
            continue
        told, launched = done[i]["value"], [r[0] for r in done[i + 1]["launches"]]
        assert len(launched) == 1, (args, launched)
        if told:
            assert launched == [told], args
            builds.add(told.split("_")[-1])
        else:
            assert args[3] > 8 and launched[0].startswith("rein_mmq_"), args
    assert {"m", "p", "b1", "t4", "t32", "t32w", "v4"} <= builds


def test_every_few_row_kernel_of_the_code_object_can_be_launched(tmp_path):
    """no build of the decode matvecs is compiled for nothing: products of every size class, with each choice pinned in turn,
    reach every rein_mv* symbol"""
    code = open(HSACO_PATH, "rb").read()
    there = {m.decode() for m in re.findall(rb"\0(rein_mv[a-z0-9_]+)\.kd(?=\0)", code)}
    shapes = [(1024, 1024), (2560, 3712), (4096, 3072), (5120, 5120), (5120, 8192), (4096, 14336), (5120, 34816)]
    calls = []
    for pin in ([], [("REIN_QUAD_LDS", 1)], [("REIN_QUAD_LDS", 1), ("REIN_QUAD_WIDE32", 0)], [("REIN_QUAD_LDS", 1), ("REIN_QUAD_WIDE32", 1)],
                [("REIN_QUAD_FROM", 1)], *([("REIN_MV_LDS", 1), ("REIN_MV_ROWS", r)] for r in (1, 2, 4)),
                *([("REIN_MV_LDS", 0), ("REIN_QUAD_LDS", 0), ("REIN_SKINNY_FROM", 99), ("REIN_QUAD_FROM", 99), ("REIN_MV_ROWS", r)] for r in (1, 2, 4))):
        calls += [("option", [n, v]) for n, v in pin]
        for k, n in shapes:
            for rows in (1, 2, 3, 8, 16, 32):
                calls += [("mmq_xq8", [fmt, P, P, P, k, n, rows]) for fmt in DENSE]
                if rows <= 4:
                    calls.append(("matvec_multi_xq8", [[rein.Q4_K, rein.Q6_K], [P, P], [P, P], [n, 8], P, k, rows]))
        calls += [("option", [n, None]) for n, _ in pin]
    calls += [("matvec_ondisk_xq8", [fmt, P, P, P, 2048, 8192]) for fmt in (rein.Q4_K, rein.Q5_K, rein.Q6_K, rein.Q8_0)]
    reached = {r[0] for d in record(calls, tmp_path) for r in d["launches"]}
    assert len(there) > 100
    assert there - reached == set()
