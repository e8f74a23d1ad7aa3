"""rein_moe_ffn on the wide tiles (kernels/moe_wide.h) against the CPU chain: experts of no, one, 31 to 33, 63 to 65 and more entries, groups of two
(K-quants) and of four tiles (Q8_0), every pair of image kinds, rows of the slab with and without padding (a power of two of sub-blocks), superblocks in odd and even
number, the one-launch and the four-launch sort, ids that leave experts out."""
import numpy as np
import pytest

import reinstinct_amd as rein
from reinstinct_amd import hip, quant, runtime
from reinstinct_amd._lib import init
from helpers import assert_close_f32, dev, rel_l2
from oracle import orc
from test_gpu_moe_few import slab

pytestmark = pytest.mark.gpu

# entries of the experts of a routing in which every token picks one expert
COUNTS = [0, 1, 31, 32, 33, 63, 64, 65, 127, 129, 5, 0]
GUARD = 1 << 17


@pytest.fixture(scope="module", autouse=True)
def gpu():
    init()
    hip.set_device(0)
    yield
    hip.synchronize()


def ffn(gu, dn, hidden, ff, x, logits, n_used, weights, scale, fill=None):
    """fill: every byte of the workspace, and of GUARD more that have to stay as they are"""
    n_tok, n_expert = logits.shape
    sh = runtime.moe_shape(n_tok, hidden, n_expert, n_used, ff, gu, dn)
    size, out = runtime.moe_workspace_bytes(sh), dev(np.full(n_tok * hidden, np.nan, np.float32))
    ws = hip.DeviceBuf(size) if fill is None else dev(np.full(size + GUARD, fill, np.uint8))
    runtime.moe_ffn(sh, dev(x), dev(logits), *[dev(w) for w in weights], dev(scale), ws, out)
    hip.synchronize()
    assert fill is None or (ws.to_host(np.uint8, GUARD, size) == fill).all(), "written behind the workspace"
    return out.to_host(np.float32).reshape(n_tok, hidden)


def reference(gu, dn, hidden, ff, x, logits, n_used, weights, scale):
    n_tok, n_expert = logits.shape
    ids, wts = orc.moe_topk(logits, n_used)
    perm, eoff, _ = orc.moe_sort(ids, n_expert, 32)
    gin = orc.moe_gather_xq(orc.quantize_q8(x), perm, hidden // 32, n_used)
    bg, bd = orc.repacked_len(gu, hidden, ff), orc.repacked_len(dn, ff, hidden)
    eg, eu = (orc.grouped_gemm(gu, w, bg, eoff, gin, hidden, ff) for w in weights[:2])
    gout = orc.grouped_gemm(dn, weights[2], bd, eoff, orc.quantize_q8(orc.swiglu_mul(eg, eu)), ff, hidden)
    return orc.moe_combine(orc.moe_scatter_rows(gout, perm, hidden).reshape(n_tok, n_used, hidden), ids, wts, scale)


def check(got, want, what):
    # The intermediate is quantized again after SwiGLU: fp32 noise in gate / up can move a quant by one step, 1/127 of its block's largest value.
    # With 256 columns and a largest value of 5 times their rms that is 5 / 127 / 16 = 0.0025 of a token's row in the norm: 5e-4 over all is
    # such a step in one row of 25 (seen: 1.6e-4).
    assert not np.isnan(got).any(), what
    assert rel_l2(got, want) < 5e-4, what
    assert_close_f32(got, want, rel=2e-2, abs_=2e-3, what=what)


def one_each(rng):
    choice = rng.permutation(np.repeat(np.arange(len(COUNTS)), COUNTS))
    logits = rng.standard_normal((len(choice), len(COUNTS))).astype(np.float32)
    logits[np.arange(len(choice)), choice] += 20.0
    return logits


@pytest.mark.parametrize("gu,dn,hidden,ff", [(rein.Q4_K, rein.Q6_K, 1024, 768), (rein.Q6_K, rein.Q4_K, 768, 256), (rein.Q5_K, rein.Q5_K, 256, 1024),
                                             (rein.Q8_0, rein.Q5_K, 512, 256), (rein.Q4_K, rein.Q8_0, 1280, 512), (rein.Q8_0, rein.Q8_0, 256, 768)])
def test_experts_of_every_number_of_tiles(gu, dn, hidden, ff, options):
    rng = np.random.default_rng(hidden + ff)
    logits = one_each(rng)
    x = rng.standard_normal((len(logits), hidden)).astype(np.float32)
    weights = [slab(f, k, n, len(COUNTS), s) for f, k, n, s in ((gu, hidden, ff, 1), (gu, hidden, ff, 2), (dn, ff, hidden, 3))]
    scale = rng.uniform(0.5, 1.5, len(COUNTS)).astype(np.float32)
    want = reference(gu, dn, hidden, ff, x, logits, 1, weights, scale)
    options.set("REIN_MOE_FEW", "0")
    options.set("REIN_MOE_CHAIN", "0")
    options.set("REIN_MOE_WIDE", "1")
    got = ffn(gu, dn, hidden, ff, x, logits, 1, weights, scale)
    check(got, want, "wide tiles")
    options.set("REIN_MOE_SORT_SPLIT", "1")
    options.set("REIN_TOPK_WAVE", "0")
    assert np.array_equal(ffn(gu, dn, hidden, ff, x, logits, 1, weights, scale).view(np.uint32), got.view(np.uint32))


# more experts than the one-wavefront router and a scan of 64 hold (at 150 tokens the workspace has no room for the wide tiles)
@pytest.mark.parametrize("n_expert,n_used,n_tok", [(300, 3, 150), (70, 4, 150), (300, 3, 1800), (70, 4, 400)])
def test_many_experts(n_expert, n_used, n_tok, options):
    gu, dn, hidden, ff = rein.Q4_K, rein.Q6_K, 512, 256
    rng = np.random.default_rng(n_expert)
    logits, x = rng.standard_normal((n_tok, n_expert)).astype(np.float32), rng.standard_normal((n_tok, hidden)).astype(np.float32)
    logits[:, 1] += 2.0                                                         # an expert of many tiles
    weights = [slab(f, k, n, n_expert, s) for f, k, n, s in ((gu, hidden, ff, 1), (gu, hidden, ff, 2), (dn, ff, hidden, 3))]
    scale = np.ones(n_expert, np.float32)
    options.set("REIN_MOE_FEW", "0")
    options.set("REIN_MOE_CHAIN", "0")
    options.set("REIN_MOE_WIDE", "1")
    check(ffn(gu, dn, hidden, ff, x, logits, n_used, weights, scale), reference(gu, dn, hidden, ff, x, logits, n_used, weights, scale), "many experts")


@pytest.mark.parametrize("n_tok,n_used", [(64, 5), (200, 2)])
def test_the_default_choice_equals_the_pinned_one(n_tok, n_used, options):
    # 40 and 50 entries per expert of 8: ff 2560 makes 320 units, where the wide tiles are the default from 36 on
    gu, dn, hidden, ff = rein.Q4_K, rein.Q6_K, 256, 2560
    rng = np.random.default_rng(n_tok)
    logits, x = rng.standard_normal((n_tok, 8)).astype(np.float32), rng.standard_normal((n_tok, hidden)).astype(np.float32)
    weights = [slab(f, k, n, 8, s) for f, k, n, s in ((gu, hidden, ff, 1), (gu, hidden, ff, 2), (dn, ff, hidden, 3))]
    scale = np.ones(8, np.float32)
    default = ffn(gu, dn, hidden, ff, x, logits, n_used, weights, scale)
    options.set("REIN_MOE_WIDE", "1")
    assert np.array_equal(ffn(gu, dn, hidden, ff, x, logits, n_used, weights, scale).view(np.uint32), default.view(np.uint32))
    check(default, reference(gu, dn, hidden, ff, x, logits, n_used, weights, scale), "default")


def test_on_the_pinned_pipeline_a_token_has_the_same_bits_in_every_call(options):
    gu, dn, hidden, ff = rein.Q4_K, rein.Q6_K, 256, 2560
    rng = np.random.default_rng(7)
    logits, x = rng.standard_normal((64, 8)).astype(np.float32), rng.standard_normal((64, hidden)).astype(np.float32)
    weights = [slab(f, k, n, 8, s) for f, k, n, s in ((gu, hidden, ff, 1), (gu, hidden, ff, 2), (dn, ff, hidden, 3))]
    scale = np.ones(8, np.float32)
    options.set("REIN_MOE_CHAIN", "0")
    together = ffn(gu, dn, hidden, ff, x, logits, 5, weights, scale)               # 40 entries per expert
    for some in (slice(0, 1), slice(20, 33)):
        assert np.array_equal(ffn(gu, dn, hidden, ff, x[some], logits[some], 5, weights, scale).view(np.uint32), together[some].view(np.uint32))


PAIRS = [(rein.Q4_K, rein.Q6_K, 512, 768), (rein.Q6_K, rein.Q4_K, 768, 512), (rein.Q5_K, rein.Q5_K, 512, 512), (rein.Q8_0, rein.Q5_K, 512, 512),
         (rein.Q4_K, rein.Q8_0, 768, 512), (rein.Q8_0, rein.Q8_0, 512, 768)]


def pinned(options, n_expert, gu, dn, hidden, ff, seed):
    """the wide tiles wherever they have room, x and logits of a routing in which every token picks one expert, weights, scales"""
    for name, value in (("REIN_MOE_FEW", "0"), ("REIN_MOE_CHAIN", "0"), ("REIN_MOE_WIDE", "1")):
        options.set(name, value)
    rng = np.random.default_rng(seed)
    logits = one_each(rng)
    weights = [slab(f, k, n, n_expert, s) for f, k, n, s in ((gu, hidden, ff, 1), (gu, hidden, ff, 2), (dn, ff, hidden, 3))]
    return rng.standard_normal((len(logits), hidden)).astype(np.float32), logits, weights, rng.uniform(0.5, 1.5, n_expert).astype(np.float32)


@pytest.mark.parametrize("gu,dn,hidden,ff", PAIRS)
@pytest.mark.parametrize("split", ["0", "1"])
def test_what_the_workspace_holds_before_reaches_no_result(gu, dn, hidden, ff, split, options):
    """places of a tile that no entry belongs to are never written: their columns of the product, whatever they are, stay their own"""
    x, logits, weights, scale = pinned(options, len(COUNTS), gu, dn, hidden, ff, 11)
    options.set("REIN_MOE_SORT_SPLIT", split)
    clean = ffn(gu, dn, hidden, ff, x, logits, 1, weights, scale, 0)
    assert not np.isnan(clean).any()
    for fill in (0xFF, 0x7C):                        # NaN in fp32, fp16 and bf16; an fp16 infinity's upper byte
        assert np.array_equal(ffn(gu, dn, hidden, ff, x, logits, 1, weights, scale, fill).view(np.uint32), clean.view(np.uint32)), fill


D_AT = {rein.Q4_K: (144, 0), rein.Q5_K: (176, 0), rein.Q6_K: (210, 208), rein.Q8_0: (34, 0)}        # bytes of a block, where d lies


@pytest.mark.parametrize("gu,dn,hidden,ff", PAIRS)
def test_infinities_and_nan_stay_where_they_are(gu, dn, hidden, ff, options):
    """tokens with an infinity or a NaN, an expert's rows of the down projection with such a scale: non-finite where the 32-token tiles are, every
    other result the bits of a call without them"""
    x, logits, weights, scale = pinned(options, len(COUNTS), gu, dn, hidden, ff, 12)
    n_tok, expert = len(x), 9                        # 129 entries: two full groups of two tiles, one of four, and one more
    down = quant.quantize_weights(dn, (np.random.default_rng(13).standard_normal((hidden, ff)) * 0.02).astype(np.float32)).reshape(hidden, -1, D_AT[dn][0])
    bad_down, bad_x = down.copy(), x.copy()
    for r, v in {0: np.nan, 77: np.inf, hidden - 1: -np.inf}.items():
        bad_down[r, r % down.shape[1], D_AT[dn][1]:D_AT[dn][1] + 2] = np.array([v], np.float16).view(np.uint8)
    bad = {3: np.inf, 40: np.nan, 64: -np.inf, n_tok - 1: np.inf}
    for t, v in bad.items():
        bad_x[t, (11 * t) % hidden] = v

    def call(blocks, x):
        slabs = weights[2].reshape(len(COUNTS), -1).copy()
        slabs[expert] = quant.repack_for_matvec(dn, np.ascontiguousarray(blocks).reshape(-1), ff, hidden)
        return ffn(gu, dn, hidden, ff, x, logits, 1, [*weights[:2], slabs.reshape(-1)], scale)

    clean, got = call(down, x), call(bad_down, bad_x)
    options.set("REIN_MOE_WIDE", "0")
    assert np.array_equal(np.isfinite(got), np.isfinite(call(bad_down, bad_x)))
    hit = logits.argmax(1) == expert
    assert hit.sum() == COUNTS[expert] and not np.isfinite(got[np.ix_(hit, [0, 77, hidden - 1])]).any()
    same = np.ones(got.shape, bool)
    same[list(bad)] = False
    same[np.ix_(hit, [0, 77, hidden - 1])] = False
    assert np.array_equal(got[same].view(np.uint32), clean[same].view(np.uint32))


@pytest.mark.parametrize("split", ["0", "1"])
def test_a_captured_call_replays(split, options):
    """the launches recorded once, other inputs in the same buffers and the program's own call on the same workspace between the replays"""
    gu, dn, hidden, ff = PAIRS[0]
    x, logits, weights, scale = pinned(options, len(COUNTS), gu, dn, hidden, ff, 14)
    options.set("REIN_MOE_SORT_SPLIT", split)
    n_tok = len(x)
    sh = runtime.moe_shape(n_tok, hidden, len(COUNTS), 1, ff, gu, dn)
    dx, dl, dw, ds = dev(x), dev(logits), [dev(w) for w in weights], dev(scale)
    ws, out, other = hip.DeviceBuf(runtime.moe_workspace_bytes(sh)), dev(np.zeros(n_tok * hidden, np.float32)), dev(np.zeros(n_tok * hidden, np.float32))
    stream = hip.Stream()
    stream.begin_capture()
    runtime.moe_ffn(sh, dx, dl, *dw, ds, ws, out, stream)
    graph = stream.end_capture().instantiate()
    for replay in range(3):
        dx.copy_from_host(np.roll(x, replay, 0))
        dl.copy_from_host(np.roll(logits, 5 * replay, 0))
        runtime.moe_ffn(sh, dx, dl, *dw, ds, ws, other)
        hip.synchronize()
        graph.launch(stream)
        stream.synchronize()
        assert np.array_equal(out.to_host(np.uint32), other.to_host(np.uint32)), replay
