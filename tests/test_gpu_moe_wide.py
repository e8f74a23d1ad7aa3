"""rein_moe_ffn on the wide tiles (kernels/moe_wide.h) against the CPU chain: experts of no, one, 31 to 33, 63 to 65 and more entries, groups of two
(K-quants) and of four tiles (Q8_0), every pair of image kinds, rows of the slab with and without padding (a power of two of sub-blocks), superblocks in odd and even
number, the one-launch and the four-launch sort, ids that leave experts out."""
import numpy as np
import pytest

import reinstinct_amd as rein
from reinstinct_amd import hip, runtime
from reinstinct_amd._lib import init
from helpers import assert_close_f32, dev, rel_l2
from oracle import orc
from test_gpu_moe_few import slab

pytestmark = pytest.mark.gpu

# entries of the experts of a routing in which every token picks one expert
COUNTS = [0, 1, 31, 32, 33, 63, 64, 65, 127, 129, 5, 0]


@pytest.fixture(scope="module", autouse=True)
def gpu():
    init()
    hip.set_device(0)
    yield
    hip.synchronize()


def ffn(gu, dn, hidden, ff, x, logits, n_used, weights, scale):
    n_tok, n_expert = logits.shape
    sh = runtime.moe_shape(n_tok, hidden, n_expert, n_used, ff, gu, dn)
    ws, out = hip.DeviceBuf(runtime.moe_workspace_bytes(sh)), dev(np.full(n_tok * hidden, np.nan, np.float32))
    runtime.moe_ffn(sh, dev(x), dev(logits), *[dev(w) for w in weights], dev(scale), ws, out)
    hip.synchronize()
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
    # the intermediate is quantized again after SwiGLU: fp32 noise in gate / up can move a quant by one step
    assert not np.isnan(got).any(), what
    assert rel_l2(got, want) < 2e-3, what
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
    # 40 and 50 entries per expert of 8: ff 2560 makes 320 units, where the wide tiles are the default from 30 on
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
