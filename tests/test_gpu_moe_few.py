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
