"""rein_moe_ffn with every touched expert read once (kernels/moe_few.hip): widths of the lane groups with and without idle lanes, one to more
than eight entries of an expert, experts without any, ragged runs of rows -- against the CPU chain."""
import numpy as np
import pytest

import reinstinct_amd as rein
from reinstinct_amd import hip, quant, runtime
from reinstinct_amd._lib import init
from oracle import orc
from helpers import assert_close_f32, dev, rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    init()
    hip.set_device(0)
    yield
    hip.synchronize()


def slab(fmt, in_dim, out_dim, n_expert, seed):
    if fmt == rein.Q5_1:                # no quantizer: random codes, tame fp16 d and m
        g = np.random.default_rng(seed)
        raw = g.integers(0, 256, (n_expert * out_dim * in_dim // 32, 24), dtype=np.uint8)
        raw[:, 0:2] = g.uniform(0.0005, 0.001, raw.shape[0]).astype(np.float16).view(np.uint8).reshape(-1, 2)
        raw[:, 2:4] = g.uniform(-0.02, -0.01, raw.shape[0]).astype(np.float16).view(np.uint8).reshape(-1, 2)
        per = out_dim * in_dim // 32
        return np.concatenate([quant.repack_for_matvec(fmt, raw[e * per:(e + 1) * per].reshape(-1), in_dim, out_dim) for e in range(n_expert)])
    w = (np.random.default_rng(seed).standard_normal((n_expert, out_dim, in_dim)) * 0.02).astype(np.float32)
    return np.concatenate([quant.repack_for_matvec(fmt, quant.quantize_weights(fmt, w[e]), in_dim, out_dim) for e in range(n_expert)])


@pytest.mark.parametrize("gu,dn", [(rein.Q4_K, rein.Q6_K), (rein.Q6_K, rein.Q4_K), (rein.Q5_K, rein.Q8_0), (rein.Q8_0, rein.Q5_K), (rein.Q5_1, rein.Q5_1)])
@pytest.mark.parametrize("n_tok,n_expert,n_used,hidden,ff,skew", [
    (1, 8, 2, 1024, 256, 0), (9, 16, 4, 512, 768, 0), (21, 7, 3, 1280, 512, 0), (40, 12, 2, 2304, 1024, 0),
    (70, 9, 2, 256, 256, 6.0)])          # skew: nearly every token picks the same experts, more than eight batches of them
def test_few_tokens_per_expert(gu, dn, n_tok, n_expert, n_used, hidden, ff, skew, options):
    options.set("REIN_MOE_FEW", "1")
    rng = np.random.default_rng(n_tok + hidden)
    x = rng.standard_normal((n_tok, hidden)).astype(np.float32)
    logits = rng.standard_normal((n_tok, n_expert)).astype(np.float32)
    logits[:, :2] += np.float32(skew)
    gate, up, down = slab(gu, hidden, ff, n_expert, 1), slab(gu, hidden, ff, n_expert, 2), slab(dn, ff, hidden, n_expert, 3)
    scale = rng.uniform(0.5, 1.5, n_expert).astype(np.float32)
    sh = runtime.moe_shape(n_tok, hidden, n_expert, n_used, ff, gu, dn)
    ws = hip.DeviceBuf(runtime.moe_workspace_bytes(sh))
    d_out = dev(np.full(n_tok * hidden, np.nan, np.float32))
    runtime.moe_ffn(sh, dev(x), dev(logits), dev(gate), dev(up), dev(down), dev(scale), ws, d_out)
    hip.synchronize()
    got = d_out.to_host(np.float32).reshape(n_tok, hidden)
    ids, wts = orc.moe_topk(logits, n_used)
    perm, eoff, _ = orc.moe_sort(ids, n_expert, 32)
    gin = orc.moe_gather_xq(orc.quantize_q8(x), perm, hidden // 32, n_used)
    bg, bd = orc.repacked_len(gu, hidden, ff), orc.repacked_len(dn, ff, hidden)
    eg = orc.grouped_gemm(gu, gate, bg, eoff, gin, hidden, ff)
    eu = orc.grouped_gemm(gu, up, bg, eoff, gin, hidden, ff)
    gout = orc.grouped_gemm(dn, down, bd, eoff, orc.quantize_q8(orc.swiglu_mul(eg, eu)), ff, hidden)
    want = orc.moe_combine(orc.moe_scatter_rows(gout, perm, hidden).reshape(n_tok, n_used, hidden), ids, wts, scale)
    # the intermediate is re-quantized after SwiGLU: fp32 noise in gate / up can move a quant by one step
    assert rel_l2(got, want) < 2e-3
    assert_close_f32(got, want, rel=2e-2, abs_=2e-3, what="moe_ffn, touched experts once")


@pytest.mark.parametrize("gu,dn", [(rein.Q4_K, rein.Q6_K), (rein.Q6_K, rein.Q5_K), (rein.Q8_0, rein.Q8_0)])
@pytest.mark.parametrize("hidden, ff", [(1024, 256), (1280, 512)])          # without and with lanes past the contraction
def test_infinities_and_nan_stay_where_they_are(gu, dn, hidden, ff, options):
    """tokens with an infinity or a NaN, and an expert with such a scale in one row of its down projection: non-finite where the
    pipeline is, every other result the bits of a call without them"""
    n_tok, n_expert, n_used = 30, 6, 2
    rng = np.random.default_rng(hidden)
    x = rng.standard_normal((n_tok, hidden)).astype(np.float32)
    logits = rng.standard_normal((n_tok, n_expert)).astype(np.float32)
    gate, up = slab(gu, hidden, ff, n_expert, 1), slab(gu, hidden, ff, n_expert, 2)
    blocks = quant.quantize_weights(dn, (rng.standard_normal((n_expert, hidden, ff)) * 0.02).astype(np.float32)).reshape(n_expert, hidden, -1)
    size, at = {rein.Q5_K: (176, 0), rein.Q6_K: (210, 208), rein.Q8_0: (34, 0)}[dn]
    bad_x, bad = x.copy(), blocks.copy()
    for t, v in {2: np.inf, 17: np.nan, 29: -np.inf}.items():
        bad_x[t, 9 * t] = v
    row, expert = 77, 4
    bad[expert, row, at:at + 2] = np.array([np.inf], np.float16).view(np.uint8)
    scale = np.ones(n_expert, np.float32)
    sh = runtime.moe_shape(n_tok, hidden, n_expert, n_used, ff, gu, dn)
    ws = hip.DeviceBuf(runtime.moe_workspace_bytes(sh))

    def ffn(x, down, few):
        options.set("REIN_MOE_FEW", few)
        down = np.concatenate([quant.repack_for_matvec(dn, down[e].reshape(-1), ff, hidden) for e in range(n_expert)])
        d_out = dev(np.full(n_tok * hidden, 12345.0, np.float32))
        runtime.moe_ffn(sh, dev(x), dev(logits), dev(gate), dev(up), dev(down), dev(scale), ws, d_out)
        hip.synchronize()
        return d_out.to_host(np.float32).reshape(n_tok, hidden)

    clean, got, other = ffn(x, blocks, 1), ffn(bad_x, bad, 1), ffn(bad_x, bad, 0)
    assert np.array_equal(np.isfinite(got), np.isfinite(other))
    # gate and up of these tokens are NaN, whose blocks of the intermediate have quants of 0 and a NaN for their sum: only formats with
    # minimums read the sum (the pipeline the same)
    assert np.isfinite(got[[2, 29]]).any() != (dn == rein.Q5_K)
    ids, _ = orc.moe_topk(logits, n_used)
    there = (ids.reshape(n_tok, n_used) == expert).any(axis=1)
    assert there.any() and not np.isfinite(got[there, row]).any()
    rest = np.ix_(np.setdiff1d(np.arange(n_tok), [2, 17, 29]), np.setdiff1d(np.arange(hidden), [row]))
    assert np.array_equal(got[rest].view(np.uint32), clean[rest].view(np.uint32))
