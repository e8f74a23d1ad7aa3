"""Which kernels the products of two to eight activation rows launch, on both sides of each line (CPU: tests/launches.py records the
launches)."""
import reinstinct_amd as rein
from launches import P, record

Q4, Q4_0, Q5, Q6, Q8, I4, I3 = rein.Q4_K, rein.Q4_0, rein.Q5_K, rein.Q6_K, rein.Q8_0, rein.IQ4_XS, rein.IQ3_S


def quad_lds(cases, tmp_path):
    """(format, in_dim, out_dim, rows, taken): the 4x4x4 kernel with the rows in LDS"""
    calls = [("mmq_xq8", [f, P, P, P, k, n, rows]) for f, k, n, rows, _ in cases]
    for case, d in zip(cases, record(calls, tmp_path)):
        assert d["launches"][0][0].startswith("rein_mvql_") == bool(case[-1]), (case, d["launches"])


def test_five_to_eight_rows_against_many(tmp_path):
    quad_lds([(Q4, 512, 151936, 8, 0), (Q8, 512, 65536, 5, 0), (Q8, 1024, 151936, 8, 1), (Q4, 1024, 40960, 6, 1), (Q4, 1024, 40992, 6, 0), (I3, 1536, 36864, 5, 0),
              (Q8, 1536, 36864, 5, 0), (Q4_0, 2048, 151936, 5, 1), (Q8, 2560, 28672, 8, 1), (Q4, 2560, 32768, 5, 0), (Q4, 2560, 32800, 5, 1), (Q4_0, 3584, 65536, 8, 0),
              (I3, 4096, 65536, 7, 1), (Q8, 4608, 151936, 5, 1), (Q8, 5120, 34816, 8, 0), (Q8, 8192, 28672, 6, 1), (Q8, 8448, 28672, 6, 0), (Q5, 512, 151936, 8, 1)], tmp_path)


def test_five_to_eight_rows_of_q5_k_against_a_thousand(tmp_path):
    quad_lds([(Q5, 3584, 1024, 5, 0), (Q5, 4096, 864, 8, 0), (Q5, 4608, 832, 5, 1), (Q5, 3584, 1088, 6, 1), (Q5, 5120, 1024, 5, 1), (Q4, 4096, 1024, 5, 1),
              (Q6, 3584, 1024, 5, 1)], tmp_path)


def test_three_and_four_rows_of_q5_k_and_q8_0(tmp_path):
    quad_lds([(Q5, 2048, 5088, 3, 1), (Q5, 2048, 5120, 3, 0), (Q5, 1536, 7168, 4, 0), (Q5, 1536, 6144, 4, 1), (Q5, 2560, 4608, 3, 0), (Q5, 1024, 8192, 3, 1),
              (Q4, 2048, 7168, 4, 1), (Q8, 3072, 7168, 3, 0), (Q8, 3328, 8192, 4, 0), (Q8, 3584, 7168, 3, 1), (Q8, 3072, 8224, 4, 1), (Q8, 256, 22464, 4, 0), (Q8, 512, 10240, 4, 1),
              (I3, 2304, 8192, 3, 1), (I3, 2304, 8224, 3, 1), (Q4, 2304, 8192, 3, 0)], tmp_path)


def test_several_matrices_with_the_activations_in_lds(tmp_path):
    cases = [([Q4, Q4, Q6], 256, [256, 128, 128], 3, 0), ([Q8, Q8], 256, [256, 256], 4, 0), ([Q4, Q4, Q6], 512, [512, 128, 128], 3, 1),
             ([Q4_0] * 3, 3072, [3072, 768, 768], 2, 0), ([I3] * 3, 4096, [4096, 512, 512], 2, 0), ([I4, I4, Q5], 3584, [3584, 448, 448], 2, 0),
             ([Q8] * 3, 4096, [4096, 1024, 1024], 2, 0), ([Q8] * 3, 5120, [4096, 1024, 1024], 2, 1), ([Q4_0] * 3, 5120, [4096, 512, 513], 2, 1), ([Q4, Q4, Q6], 4096, [4096, 1024, 1024], 2, 1),
             ([Q8] * 3, 3072, [3072, 512, 512], 2, 1), ([I4, I4], 8192, [12288, 12288], 2, 1), ([I4, I4], 8192, [12288, 12320], 2, 0),
             ([Q4_0, Q4_0], 8192, [24576, 24576], 2, 1)]
    calls = [("matvec_multi_xq8", [f, [P] * len(f), [P] * len(f), outs, P, k, rows]) for f, k, outs, rows, _ in cases]
    for case, d in zip(cases, record(calls, tmp_path)):
        (kernel, *_), = d["launches"]
        assert kernel.startswith("rein_mvl_multi_" if case[-1] else "rein_mv_multi_"), (case, kernel)


def test_two_matrices_in_one_launch_of_the_4x4x4_kernel(tmp_path):
    """(Q8_0 from a contraction of 8192: one workgroup to a CU, of as many wavefronts as its LDS holds)"""
    cases = [([Q8, Q8], 8448, [8200, 8200], 1), ([Q8, Q8], 12288, [12288, 12288], 1), ([Q8, Q8], 22528, [8200, 8200], 1), ([Q8, Q8], 8192, [8200, 8200], 0),
             ([Q4, Q4], 5120, [17408, 17408], 1)]
    calls = [("matvec_multi_xq8", [f, [P] * 2, [P] * 2, outs, P, k, 4]) for f, k, outs, _ in cases]
    for case, d in zip(cases, record(calls, tmp_path)):
        assert len(d["launches"]) == (1 if case[-1] else 2), case
        if case[-1]:
            (kernel, grid, block, lds), = d["launches"]
            assert kernel == "rein_mvql_multi_t4_m" and grid[0] <= 256 and lds <= 160 << 10, (case, d["launches"])


def test_the_gpu_cases_of_several_matrices_launch_what_they_name(tmp_path):
    from test_gpu_matvec_multi_lds import DOT4, MATRIX
    for pin, cases, kernel in ((("REIN_MV_LDS", "1"), [c + (r, None) for c in DOT4 for r in (2, 3, 4)], "rein_mvl_multi_"), (None, MATRIX, "rein_mvql_multi_t4_m")):
        for fmts, k, outs, rows, quad in cases:
            pins = [("option", list(p)) for p in (pin, quad and ("REIN_QUAD_LDS", quad)) if p]
            done = record(pins + [("matvec_multi_xq8", [fmts, [P] * len(fmts), [P] * len(fmts), outs, P, k, rows])], tmp_path)[-1]
            (name, *_), = done["launches"]
            assert name.startswith(kernel), (fmts, k, outs, rows, name)
