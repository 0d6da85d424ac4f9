"""The sliced matrix-core logits at the edges of their tiles (16 experts x 32 tokens, the second 16
tokens left out when there are none) and slices, against the engine's routing bit for bit."""
import numpy as np
import pytest

import k3moe
import oracle as O

pytestmark = pytest.mark.gpu


# experts and widths of one slice and many, slices with no step left, several workgroups a tile
@pytest.mark.parametrize("E,d,k", [(16, 64, 2), (48, 192, 4), (400, 1088, 8), (896, 2048, 16)])
def test_router_few_tokens(gpu, E, d, k):
    W = np.ascontiguousarray(k3moe.host_normal(E * d, 21, 501, 0, 0.05).reshape(E, d))
    bias = k3moe.host_normal(E, 21, 502, 0, 0.01)
    x = np.ascontiguousarray(k3moe.host_normal(49 * d, 21, 503, 0, 1.0).reshape(49, d))
    L = k3moe.K3gLayer()
    L.hidden, L.n_experts, L.topk, L.inter, L.latent = d, E, k, 128, d
    L.renorm, L.routed_scale = 1, 2.5
    dW, db, dx = (k3moe.DevBuf.from_array(a) for a in (W, bias, x))
    L.gate, L.bias = dW.ptr, db.ptr
    ctx = k3moe.Ctx(L, max_tokens=49)
    didx, dwt = k3moe.DevBuf(49 * k * 4), k3moe.DevBuf(49 * k * 4)
    want = [O.oracle().router(v, W, bias, E, k, 1, 2.5) for v in x]
    for T in (4, 15, 16, 17, 32, 33, 48, 49):
        print(f"case: router E={E} k={k} d={d}, {T} tokens", flush=True)
        ctx.router(L, dx.ptr, T, didx.ptr, dwt.ptr)
        ctx.sync()
        idx = didx.download(np.int32, T * k).reshape(T, k)
        wt = dwt.download(np.float32, T * k).reshape(T, k)
        for t in range(T):
            assert np.array_equal(idx[t], want[t][0]), (T, t)
            # a weight's float logit may be the engine's neighbour: one ulp of it, two of expf
            np.testing.assert_allclose(wt[t], want[t][1], rtol=1e-6, atol=0)
    ctx.destroy()
