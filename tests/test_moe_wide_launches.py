"""rein_moe_ffn on the wide tiles, without a GPU (tests/launches.py records the launches): what workspace it has, and where it is taken."""
import random

import pytest

import reinstinct_amd as rein
from launches import record
from reinstinct_amd import runtime

FORMATS = (rein.Q4_K, rein.Q5_K, rein.Q6_K, rein.Q8_0)


def kernels(calls, tmp_path):
    return [[r[0] for r in d["launches"]] for d in record(calls, tmp_path)]


def wide(names):
    return any("_swiglu" in n and "_xg" in n for n in names)


def pipeline_bytes(n_tok, hidden, n_expert, n_used, ff, gu=0, dn=0):
    """the pipeline of 32-token tiles: routing, lists of the sort, BlockQ8 rows of the tokens and the entries, gate, up, their rows, down"""
    ne = n_tok * n_used
    parts = [4 * ne, 4 * ne, 4 * n_expert, 4 * n_expert, 4 * ne, 4 * ne, 4 * n_expert + 4, 4 * n_expert + 4, n_tok * hidden // 32 * 40,
             ne * hidden // 32 * 40, 4 * ne * ff, 4 * ne * ff, ne * ff // 32 * 40, 4 * ne * hidden]
    return sum((p + 255) // 256 * 256 for p in parts)


@pytest.mark.parametrize("option", [None, "REIN_MOE_WIDE"])
def test_the_workspace_is_that_of_the_pipeline(option, options):
    """what a call may take instead of the pipeline lives inside the pipeline's own room, so no option changes the size"""
    if option:
        options.set(option, "1")
    rng = random.Random(3)
    shapes = [(1, 2048, 128, 8, 768), (16, 2048, 128, 8, 768), (48, 2048, 128, 8, 768), (32, 4096, 256, 8, 1536), (512, 2048, 128, 8, 768), (1, 256, 1, 1, 256)]
    shapes += [(int(2 ** rng.uniform(0, 12)), 256 * rng.randint(1, 16), e, rng.randint(1, min(8, e)), 256 * rng.randint(1, 8)) for e in (2, 8, 60, 128, 300) for _ in range(40)]
    for s in shapes:
        gu, dn = rng.choice(FORMATS), rng.choice(FORMATS)
        assert runtime.moe_workspace_bytes(runtime.moe_shape(*s, gu, dn)) == pipeline_bytes(*s), (s, gu, dn)


def test_wide_tiles_that_have_no_room_are_not_taken(tmp_path):
    """one entry of an expert would be charged a whole tile: however it is asked for, the workspace does not hold that"""
    q4, q6, q8 = rein.Q4_K, rein.Q6_K, rein.Q8_0
    pins = [("option", [n, v]) for n, v in (("REIN_MOE_FEW", 0), ("REIN_MOE_CHAIN", 0), ("REIN_MOE_WIDE", 1))]
    cases = [((48, 2048, 128, 8, 768, q4, q6), 0), ((96, 2048, 128, 8, 768, q8, q8), 0), ((256, 2048, 128, 8, 768, q8, q8), 1), ((272, 2048, 128, 8, 768, q4, q6), 0),
             ((512, 2048, 128, 8, 768, q4, q6), 1), ((512, 4096, 128, 8, 256, q4, q4), 1), ((1, 256, 1, 1, 256, q4, q6), 0)]
    for (shape, want), names in zip(cases, kernels(pins + [("moe_ffn", list(s)) for s, _ in cases], tmp_path)[len(pins):]):
        assert wide(names) == bool(want), (shape, names)


def test_a_pinned_pipeline_has_one_form(tmp_path):
    """REIN_MOE_CHAIN and the options of the 32-token tiles keep them at every number of tokens; only REIN_MOE_WIDE = 1 is asked for by name"""
    calls = [("moe_ffn", [n, 2048, 128, 8, 768, rein.Q4_K, rein.Q6_K]) for n in (1, 48, 479, 480, 2048)]
    for pins, want in ([], [0, 0, 0, 1, 1]), ([("REIN_MOE_CHAIN", 0)], [0] * 5), ([("REIN_MOE_FUSED", 1)], [0] * 5), ([("REIN_GROUPED_STRIDED", 1)], [0] * 5), \
            ([("REIN_MOE_WIDE", 0)], [0] * 5), ([("REIN_MOE_CHAIN", 0), ("REIN_MOE_WIDE", 1)], [0, 0, 1, 1, 1]):
        done = kernels([("option", list(p)) for p in pins] + calls, tmp_path)[len(pins):]
        assert [wide(names) for names in done] == [bool(w) for w in want], pins
        if pins == [("REIN_MOE_CHAIN", 0)]:
            assert all("rein_mmq_q4k_grouped_swiglu_q8" in names and "rein_mmq_q6k_grouped_t32" in names for names in done)


def test_where_the_wide_tiles_are_taken(tmp_path):
    """both sides of every line: entries per expert by formats, units of the gate + up launch, superblocks of the down projection"""
    q4, q5, q6, q8 = FORMATS
    k2, k4, tiles = ("rein_mmq_{}_xg2_swiglu", "rein_mmq_{}_xg2_rows"), ("rein_mmq_{}_xg4_swiglu", "rein_mmq_{}_xg4_rows"), None
    # tokens, hidden, experts, used, width, formats
    cases = [((480, 2048, 128, 8, 768, q4, q6), ("q4k", k2, "q6k", k2)), ((479, 2048, 128, 8, 768, q4, q6), tiles),           # 30 entries per expert
             ((480, 1024, 128, 8, 768, q5, q4), ("q5k", k2, "q4k", k2)), ((480, 1024, 128, 8, 768, q6, q8), ("q6k", k2, "q8_0", k4)),
             ((576, 2048, 128, 8, 768, q4, q5), ("q4k", k2, "q5k", k2)), ((575, 2048, 128, 8, 768, q4, q5), tiles),           # 36 with a Q5_K down
             ((576, 2048, 128, 8, 512, q4, q6), ("q4k", k2, "q6k", k2)), ((575, 2048, 128, 8, 512, q4, q6), tiles),           # and with two superblocks to it
             ((672, 2048, 128, 8, 512, q4, q5), ("q4k", k2, "q5k", k2)), ((671, 2048, 128, 8, 512, q4, q5), tiles),           # 42 with both
             ((2048, 2048, 128, 8, 256, q4, q6), tiles), ((2048, 2048, 128, 8, 256, q8, q8), tiles),                          # one superblock
             ((288, 2048, 32, 4, 768, q4, q6), ("q4k", k2, "q6k", k2)), ((287, 2048, 32, 4, 768, q4, q6), tiles),             # 384 units: 36
             ((480, 2048, 64, 4, 512, q4, q6), tiles), ((384, 2048, 43, 4, 768, q4, q6), ("q4k", k2, "q6k", k2)), ((323, 2048, 43, 4, 768, q4, q6), ("q4k", k2, "q6k", k2)),
             ((322, 2048, 43, 4, 768, q4, q6), tiles), ((384, 2048, 42, 4, 768, q4, q6), ("q4k", k2, "q6k", k2)), ((377, 2048, 42, 4, 768, q4, q6), tiles),          # 516 units and 504
             ((72, 256, 8, 4, 2560, q4, q6), ("q4k", k2, "q6k", k2)), ((71, 256, 8, 4, 2560, q4, q6), tiles),                 # 320 units
             ((128, 256, 8, 4, 2304, q4, q6), tiles), ((129, 256, 8, 4, 2304, q4, q6), ("q4k", k2, "q6k", k2)),               # 288, and twice as many
             ((288, 2048, 128, 8, 768, q8, q8), ("q8_0", k4, "q8_0", k4)), ((287, 2048, 128, 8, 768, q8, q8), tiles),         # 18 of Q8_0
             ((288, 2048, 128, 8, 768, q8, q5), ("q8_0", k4, "q5k", k2)), ((288, 2048, 128, 8, 512, q8, q6), ("q8_0", k4, "q6k", k2)),
             ((512, 2080, 128, 8, 768, q8, q8), tiles), ((512, 2048, 128, 8, 800, q8, q8), tiles)]                            # contractions of whole superblocks
    for (shape, want), names in zip(cases, kernels([("moe_ffn", list(s)) for s, _ in cases], tmp_path)):
        if want is tiles:
            assert any("_grouped_swiglu_q8" in n for n in names) and not wide(names), (shape, names)
        else:
            gu, (first, _), dn, (_, second) = want
            assert first.format(gu) in names and second.format(dn) in names, (shape, names)
