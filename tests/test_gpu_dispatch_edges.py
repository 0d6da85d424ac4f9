"""The one-pair-a-thread dispatch at the edges of its waves and of its range, against a stable
sort."""
import numpy as np
import pytest

import k3moe

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [1, 63, 64, 65, 1023, 1024, 1025])
@pytest.mark.parametrize("E,hot", [(1, False), (300, True), (1024, False)])
def test_dispatch_edges(gpu, P, E, hot):
    """hot: nine pairs of ten on the last expert; one slot in seven is dropped."""
    print(f"case: k3g_dispatch {P} pairs over {E} experts", flush=True)
    rng = np.random.default_rng(P + E)
    idx = rng.integers(0, E, P).astype(np.int32)
    if hot:
        idx[rng.random(P) < 0.9] = E - 1
    idx[rng.random(P) < 1 / 7] = -1
    L = k3moe.K3gLayer()
    L.hidden = L.latent = L.inter = 128
    L.n_experts, L.topk = E, 1
    ctx = k3moe.Ctx(L, max_tokens=P)
    didx = k3moe.DevBuf.from_array(idx)
    dperm, doff = k3moe.DevBuf(P * 4), k3moe.DevBuf((E + 1) * 4)
    ctx.dispatch(didx.ptr, P, 1, E, dperm.ptr, doff.ptr)
    ctx.sync()
    keep = np.flatnonzero(idx >= 0)
    perm = keep[np.argsort(idx[keep], kind="stable")]
    off = np.concatenate([[0], np.cumsum(np.bincount(idx[keep], minlength=E))])
    assert np.array_equal(doff.download(np.int32, E + 1), off)
    assert np.array_equal(dperm.download(np.int32, P)[:perm.size], perm)
    ctx.destroy()
