"""kernels/moe_few.hip: a batch of one or two entries goes on dot4, three to eight on the 4x4x4 matrix instruction, and an entry's result is
the same bits whichever it is in: the router's order puts a token's entry into any batch."""
import numpy as np
import pytest

import reinstinct_amd as rein
from reinstinct_amd import hip, runtime
from reinstinct_amd._lib import init
from helpers import dev
from test_gpu_moe_few import slab

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    init()
    hip.set_device(0)
    yield
    hip.synchronize()


@pytest.mark.parametrize("gu,dn", [(rein.Q4_K, rein.Q6_K), (rein.Q6_K, rein.Q8_0), (rein.Q5_K, rein.Q5_K), (rein.Q8_0, rein.Q4_K), (rein.Q5_1, rein.Q5_1)])
@pytest.mark.parametrize("hidden,ff", [(1024, 256), (2304, 768), (512, 1280)])         # 16, 8 and 4 lanes to a row, with and without idle ones
def test_a_token_alone_and_among_others(gu, dn, hidden, ff, options):
    options.set("REIN_MOE_FEW", "1")
    n_expert, n_used = 3, 2
    rng = np.random.default_rng(hidden + ff)
    x = rng.standard_normal((11, hidden)).astype(np.float32)
    logits = np.tile(np.array([3.0, 1.0, 2.0], np.float32), (11, 1))            # every token picks the experts 0 and 2
    weights = [dev(slab(f, k, n, n_expert, s)) for f, k, n, s in ((gu, hidden, ff, 1), (gu, hidden, ff, 2), (dn, ff, hidden, 3))]
    scale = dev(np.ones(n_expert, np.float32))

    def ffn(tokens):
        sh = runtime.moe_shape(len(tokens), hidden, n_expert, n_used, ff, gu, dn)
        out = dev(np.full(len(tokens) * hidden, np.nan, np.float32))
        ws = hip.DeviceBuf(runtime.moe_workspace_bytes(sh))
        runtime.moe_ffn(sh, dev(x[tokens]), dev(logits[tokens]), *weights, scale, ws, out)
        hip.synchronize()
        return out.to_host(np.uint32).reshape(len(tokens), hidden)

    alone = np.concatenate([ffn([t]) for t in range(11)])
    assert np.isfinite(alone.view(np.float32)).all()
    for n in (2, 3, 4, 5, 8, 9, 11):                # 9 and 11: a second batch of one and of three
        assert np.array_equal(ffn(list(range(n))), alone[:n]), n
