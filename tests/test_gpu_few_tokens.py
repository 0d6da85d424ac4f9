"""The fused decode kernel at 2 to 4 tokens (tickets taken from the stripes' counters, a selection
per token) against the same tokens one at a time, with calls of different sizes on one context."""
import numpy as np
import pytest

import k3moe

pytestmark = pytest.mark.gpu


# one round of tickets and many, widths ragged in the 512-column quads and 1024-column chunks; the
# last one's routed down tickets are sliced at 2 tokens (1536 of them whole) and whole at 3 (2304)
@pytest.mark.parametrize("hidden,inter,experts,topk", [(256, 64, 8, 2), (1184, 544, 48, 6),
                                                       (3072, 1056, 96, 8)])
def test_few_tokens_match_single_tokens(gpu, hidden, inter, experts, topk):
    shape = k3moe.Shape("few", hidden, experts, topk, inter, n_shared=1, routed_scale=2.5,
                        x_bf16=False, scale_lo=-8, scale_hi=-6)
    layer = k3moe.SynthLayer(shape, seed=51, layout="tiled")
    x = layer.tokens(4)
    L = layer.dev_tiled
    ctx = k3moe.Ctx(L, max_tokens=4)
    dx, dout = k3moe.DevBuf.from_array(x), k3moe.DevBuf(4 * hidden * 4)
    didx, dwt = k3moe.DevBuf(4 * topk * 4), k3moe.DevBuf(4 * topk * 4)

    def run(t0, T):
        print(f"case: fused decode {hidden} x {inter}, {experts} experts, tokens {t0}..{t0 + T - 1}",
              flush=True)
        ctx.moe(L, dx.ptr + t0 * hidden * 4, T, dout.ptr, didx.ptr, dwt.ptr)
        ctx.sync()
        return (dout.download(np.float32, T * hidden).reshape(T, hidden),
                didx.download(np.int32, T * topk).reshape(T, topk),
                dwt.download(np.float32, T * topk).reshape(T, topk))

    one = [run(t, 1) for t in range(4)]
    for t0, T in ((0, 4), (1, 3), (2, 2), (0, 3), (0, 2), (0, 4)):
        out, idx, wt = run(t0, T)
        for t in range(T):
            o, i, w = (v[0] for v in one[t0 + t])
            assert np.array_equal(idx[t], i)
            # a weight's float logit may be the engine's neighbour
            np.testing.assert_allclose(wt[t], w, rtol=1e-6, atol=0)
            # fp32 sums in another order: 2^-24 sqrt(terms) twice over
            assert np.linalg.norm(out[t] - o) <= 2e-6 * np.linalg.norm(o)
    ctx.destroy()
