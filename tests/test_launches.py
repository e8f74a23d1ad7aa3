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


def xh(done):
    return [r[0] for r in done["launches"] if r[0].startswith("rein_xh_")]


def test_exact_dot_gemm_needs_no_more_scratch_than_its_plan(tmp_path):
    """rein_matmul_ws: a scratch of the size the query gives runs the exact-dot GEMM for every number of weight rows; one that holds
    the shape's own image and partial tiles does too; one that does not runs the other launches"""
    rng = random.Random(9)
    shapes = [(fmt, k, rows) for fmt in (rein.Q4_K, rein.Q5_K, rein.Q6_K) for k, rows in
              [(256, 33), (512, 4097), (768, 200), (4096, 128), (17408, 777), (5120, 65535), *((256 * rng.randint(1, 72), rng.randint(33, 3000)) for _ in range(6))]]
    sizes = record([("option", ["REIN_MMQXH", 2])] + [("matmul_scratch_bytes", list(s)) for s in shapes], tmp_path)[1:]
    calls = [("option", ["REIN_MMQXH", 2])]
    for (fmt, k, rows), size in zip(shapes, sizes):
        for n in [1, 640, 5120, 17408, *(rng.randint(1, 40000) for _ in range(20))]:
            calls.append(("matmul_ws", [fmt, P, P, P, k, n, rows, P, size["value"]]))
    for call, done in zip(calls[1:], record(calls, tmp_path)[1:]):
        assert xh(done)[:1] == ["rein_xh_quantize"], call
    # 200 rows against 4096 -> 640: ten units of sixteen superblocks in sixteen ranges at most
    fmt, k, n, rows = rein.Q6_K, 4096, 640, 200
    front = (rows * k // 32 * 40 + 255) // 256 * 256
    image = k // 64 * 7 * 4352
    call = [fmt, P, P, P, k, n, rows, P]
    calls = [("option", ["REIN_MMQXH_SPLIT", 1]), ("matmul_ws", call + [front + image]), ("option", ["REIN_MMQXH_SPLIT", None]),
             ("matmul_ws", call + [front + image + 160 * 65536]), ("matmul_ws", call + [front + image - 1]), ("matmul_ws", call + [front + image])]
    _, unsplit, _, split, none, least = record(calls, tmp_path)
    assert xh(unsplit) == ["rein_xh_quantize", "rein_xh_q6k"]
    assert xh(split) == ["rein_xh_quantize", "rein_xh_q6k", "rein_xh_sum"]
    assert xh(none) == [] and xh(least) == [] and none["launches"]
    # the int8 tile's split-tail launch switched off does not switch this one off
    off = record([("option", ["REIN_MMQ_SK", 0]), *(("matmul_ws", [f] + call[1:] + [front + image + (64 << 20)]) for f in (rein.Q5_K, rein.Q6_K)),
                  ("option", ["REIN_MMQXH", 2]), ("matmul_ws", [rein.Q5_K] + call[1:] + [front + image + (64 << 20)])], tmp_path)
    assert [bool(xh(d)) for d in off[1:3] + off[4:]] == [False, True, True]          # (Q5_K below 384 rows only where it is asked for)


def test_exact_dot_gemm_and_the_scratch_query_without_partial_tiles(tmp_path):
    """a contraction of one superblock is never split: the query asks for no more than the other launches want"""
    from reinstinct_amd import runtime
    for fmt in (rein.Q5_K, rein.Q6_K):
        assert runtime.matmul_scratch_bytes(fmt, 256, 64) <= (64 * 8 * 40 + 255) // 256 * 256 + (16 << 20)


def test_narrow_on_disk_matrices_keep_the_kernel_of_64_lanes(tmp_path):
    """Q8_0, and Q6_K where the last 2048 weights of a row fill it, up to a workgroup of eight rows per CU"""
    shapes = [(rein.Q6_K, 2048, 1024, 0), (rein.Q6_K, 2048, 2048, 0), (rein.Q6_K, 2048, 2049, 1), (rein.Q6_K, 1024, 256, 1), (rein.Q6_K, 3072, 2048, 1),
              (rein.Q6_K, 1280, 64, 0), (rein.Q8_0, 1024, 2048, 0), (rein.Q8_0, 5120, 512, 0), (rein.Q8_0, 5120, 2049, 1), (rein.Q4_K, 2048, 32, 1),
              (rein.Q5_K, 4096, 1024, 1), (rein.Q8_0, 5152, 4096, 0), (rein.Q4_K, 131072, 4096, 0), (rein.Q6_K, 2048, 151936, 1)]
    done = record([("matvec_ondisk_xq8", [f, P, P, P, k, n]) for f, k, n, _ in shapes], tmp_path)
    for (f, k, n, lds), d in zip(shapes, done):
        (kernel, *_), = d["launches"]
        assert kernel.startswith("rein_mvd_" if lds else "matvec_q"), (f, k, n, kernel)


def test_form_of_the_expert_ffn(tmp_path):
    """rein_moe_ffn: the decode launches while little is read twice, then every touched expert once, then the pipeline"""
    q4, q6, q8 = rein.Q4_K, rein.Q6_K, rein.Q8_0
    few, decode, tiles = "rein_moe_few_gate_up", "gate_up_swiglu_q8", "rein_mmq_"
    # tokens, hidden, experts, used, width, formats
    cases = [((1, 2048, 4, 4, 768, q4, q6), decode), ((1, 2048, 8, 8, 768, q4, q6), decode), ((2, 2048, 4, 2, 768, q4, q6), decode),
             ((4, 2048, 8, 2, 768, q4, q6), decode), ((8, 2048, 8, 2, 768, q4, q6), few), ((1, 4096, 8, 8, 1536, q4, q6), decode),
             ((3, 4096, 32, 8, 1536, q4, q6), decode), ((4, 4096, 32, 8, 1536, q4, q6), few), ((10, 2048, 128, 8, 768, q4, q6), decode),
             ((16, 2048, 128, 8, 768, q4, q6), few), ((12, 2048, 128, 8, 768, q8, q8), decode), ((20, 2048, 128, 8, 768, q8, q8), few),
             ((48, 2048, 128, 8, 768, q4, q6), few), ((96, 2048, 128, 8, 768, q4, q6), tiles)]
    for (shape, form), d in zip(cases, record([("moe_ffn", list(s)) for s, _ in cases], tmp_path)):
        kernels = [r[0] for r in d["launches"]]
        assert any(form in k for k in kernels), (shape, kernels)
        assert form == few or not any(few in k for k in kernels), (shape, kernels)


def test_where_the_exact_dot_gemm_is_taken(tmp_path):
    cases = [(rein.Q6_K, 256, 20000, 33, 1), (rein.Q6_K, 256, 4096, 33, 0), (rein.Q6_K, 1024, 4096, 64, 1), (rein.Q6_K, 5120, 17408, 32, 0),
             (rein.Q4_K, 2816, 8192, 64, 0), (rein.Q4_K, 3072, 8192, 64, 1), (rein.Q4_K, 3584, 18944, 65, 0), (rein.Q4_K, 3584, 18944, 512, 0),
             (rein.Q4_K, 4096, 4096, 95, 0), (rein.Q4_K, 4096, 4096, 96, 1), (rein.Q4_K, 3840, 4096, 2048, 0),
             (rein.Q5_K, 4096, 4096, 383, 0), (rein.Q5_K, 4096, 4096, 384, 1), (rein.Q5_K, 3584, 3584, 512, 0), (rein.Q5_K, 3584, 18944, 512, 1),
             (rein.Q5_K, 2816, 18944, 512, 0), (rein.Q8_0, 5120, 17408, 512, 0)]
    sizes = record([("matmul_scratch_bytes", [f, k, rows]) for f, k, _, rows, _ in cases], tmp_path)
    done = record([("matmul_ws", [f, P, P, P, k, n, rows, P, size["value"]]) for (f, k, n, rows, _), size in zip(cases, sizes)], tmp_path)
    for case, d in zip(cases, done):
        assert bool(xh(d)) == bool(case[-1]), case


def test_which_products_of_several_matrices_stage_their_activations_in_lds(tmp_path):
    q4, q5, q6, q8, i4 = rein.Q4_K, rein.Q5_K, rein.Q6_K, rein.Q8_0, rein.IQ4_XS
    dot4, matrix, plain = "rein_mvl_multi_", "rein_mvql_multi_t4_m", "rein_mv_multi_"
    cases = [(([q5, q5, q6], 4096, [4096, 1024, 1024], 4), dot4), (([q4, q4, q6], 4096, [4096, 4096, 4096], 4), plain),
             (([q8, q8], 2048, [8192, 8192], 3), dot4), (([q4, q4], 2048, [8192, 8192], 3), plain), (([q4, q4], 3072, [8192, 8192], 3), dot4),
             (([i4, i4], 3072, [8192, 8192], 3), plain), (([q4, q4, q6], 5120, [5120, 1024, 1024], 2), dot4), (([q6, q6], 5120, [17408, 17408], 2), plain),
             (([q6, q6], 8192, [24576, 24576], 2), dot4), (([q4, q4], 5120, [17408, 17408], 1), plain), (([q5, q5], 4096, [14336, 14336], 4), matrix),
             (([q4, q6], 8192, [8192, 8192], 3), matrix), (([q4, q4, q4], 5120, [17408, 17408, 17408], 4), "rein_mvql_q4k_t4_m"),
             (([q4, q6], 5120, [8192, 12288], 3), "rein_mvql_q4k_t4_m"), (([i4, i4], 5120, [17408, 17408], 4), "rein_mvq_iq4xs_t4")]
    calls = [("matvec_multi_xq8", [f, [P] * len(f), [P] * len(f), outs, P, k, rows]) for (f, k, outs, rows), _ in cases]
    for (case, kernel), d in zip(cases, record(calls, tmp_path)):
        names = [r[0] for r in d["launches"]]
        assert names[0].startswith(kernel), (case, names)
        assert len(names) == (1 if "multi" in kernel else len(case[0])), (case, names)
    # a pinned choice of the other forms keeps them
    pins = [("REIN_MV_LDS", 0, 0), ("REIN_MV_ROWS", 2, 0), ("REIN_MV_WPB", 4, 0), ("REIN_QUAD_LDS", 0, 10), ("REIN_MV_LOADS", 0, 10)]
    for name, value, at in pins:
        _, d, _ = record([("option", [name, value]), calls[at], ("option", [name, None])], tmp_path)
        assert not d["launches"][0][0].startswith(cases[at][1]), (name, d["launches"])


def test_which_products_of_three_to_eight_rows_take_the_4x4x4_kernel_with_the_rows_in_lds(tmp_path):
    q4, q5, q6, q8, i4, i3 = rein.Q4_K, rein.Q5_K, rein.Q6_K, rein.Q8_0, rein.IQ4_XS, rein.IQ3_S
    cases = [(q4, 1024, 4096, 3, 1), (q4, 1024, 4064, 3, 0), (q4, 2560, 6496, 4, 1), (q4, 2816, 5120, 4, 0), (q5, 2048, 4608, 3, 1), (q6, 1280, 5120, 3, 1),
             (q6, 1536, 5120, 3, 0), (q8, 2048, 4608, 4, 1), (q8, 2048, 4608, 3, 0), (i4, 1536, 4096, 4, 1), (i4, 1536, 4096, 3, 0), (q8, 7168, 7168, 3, 1),
             (q8, 8192, 8192, 4, 0), (q8, 8192, 10240, 4, 1), (q8, 5120, 5120, 4, 0), (i4, 5120, 16384, 3, 1), (i4, 5120, 16416, 3, 0), (i3, 2048, 8192, 4, 1),
             (q4, 2048, 8192, 4, 0), (q4, 1024, 4096, 2, 0), (q5, 2304, 1664, 5, 1), (q5, 2048, 1536, 8, 0), (q8, 1024, 1536, 6, 1), (q4, 1024, 1504, 7, 0),
             (q4, 4096, 28672, 5, 1), (q4, 4096, 28640, 5, 0), (q4, 2304, 30720, 8, 0), (q4, 6144, 30720, 8, 0), (q8, 8192, 20512, 8, 1), (q8, 7168, 24576, 5, 0)]
    calls = [("mmq_xq8", [f, P, P, P, k, n, rows]) for f, k, n, rows, _ in cases]
    for case, d in zip(cases, record(calls, tmp_path)):
        assert d["launches"][0][0].startswith("rein_mvql_") == bool(case[-1]), (case, d["launches"])
