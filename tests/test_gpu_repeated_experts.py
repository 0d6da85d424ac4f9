"""Tokens that have an expert more than once: a token with fewer than topk selectable experts (its
scores NaN, or a bias of -inf) has expert 0 in every slot left over, as in the engine, so one
expert can have more pairs than the call has tokens. The other tokens' outputs through k3g_moe
against the same tokens called without them, on a context that holds an earlier call's rows."""
import numpy as np
import pytest

import k3moe

pytestmark = pytest.mark.gpu


class _Moe:
    def __init__(self, experts, topk, x_bf16, max_tokens):
        shape = k3moe.Shape("repeat", 512, experts, topk, 256, n_shared=1, routed_scale=2.5,
                            x_bf16=x_bf16, scale_lo=-8, scale_hi=-6)
        self.layer = k3moe.SynthLayer(shape, seed=61, layout="tiled")
        self.L, self.k, self.d = self.layer.dev_tiled, topk, 512
        self.ctx = k3moe.Ctx(self.L, max_tokens=max_tokens)

    def __call__(self, x):
        T = x.shape[0]
        dx = k3moe.DevBuf.from_array(np.ascontiguousarray(x, np.float32))
        dout, didx = k3moe.DevBuf(T * self.d * 4), k3moe.DevBuf(T * self.k * 4)
        dwt = k3moe.DevBuf(T * self.k * 4)
        self.ctx.moe(self.L, dx.ptr, T, dout.ptr, didx.ptr, dwt.ptr)
        self.ctx.sync()
        return (dout.download(np.float32, T * self.d).reshape(T, self.d),
                didx.download(np.int32, T * self.k).reshape(T, self.k))


def _same(got, want):
    """The same sums over the same rows: the weights' float logits may be neighbours."""
    for g, w in zip(got, want):
        assert np.linalg.norm(g - w) <= 2e-6 * np.linalg.norm(w)


# tokens of NaN ahead of the valid ones: more than 64 pairs of expert 0, the valid ones last
@pytest.mark.parametrize("T,nan,experts,topk", [(9, 8, 16, 8), (64, 16, 16, 4), (64, 8, 40, 8),
                                                (33, 12, 24, 6)])
def test_nan_tokens_leave_the_others_alone(gpu, T, nan, experts, topk):
    print(f"case: moe of {T} tokens, the first {nan} of them NaN, top-{topk} of {experts}", flush=True)
    m = _Moe(experts, topk, False, T)
    x = m.layer.tokens(T)
    m(1e3 * x[::-1])
    want, iw = m(np.concatenate([x[nan:]] * 64)[:max(5, T - nan)])
    m(1e3 * x[::-1])
    x[:nan] = np.nan
    got, ig = m(x)
    assert (ig[:nan] == 0).all() and np.isnan(got[:nan]).all()
    assert (ig[nan:] == 0).any(), "no valid token with expert 0"
    assert np.array_equal(ig[nan:], iw[:T - nan])
    _same(got[nan:], want[:T - nan])
    m.ctx.destroy()


# finite tokens, all but topk - 1 experts' bias -inf: expert 0 twice a token
@pytest.mark.parametrize("x_bf16", [False, True])
@pytest.mark.parametrize("T,experts,topk", [(64, 16, 8), (40, 24, 4), (64, 8, 2)])
def test_one_selectable_expert_short(gpu, T, experts, topk, x_bf16):
    print(f"case: moe of {T} tokens, {topk - 1} of {experts} experts selectable for top-{topk}, "
          f"bf16 x {x_bf16}", flush=True)
    m = _Moe(experts, topk, x_bf16, T)
    bias = np.full(experts, -np.inf, np.float32)
    bias[:topk - 1] = m.layer.bias[:topk - 1]
    m.layer.d_bias.upload(bias)
    x = m.layer.tokens(T)
    m(1e3 * x[::-1])
    got, idx = m(x)
    assert ((idx == 0).sum(axis=1) == 2).all()
    for t in range(0, T, 8):             # 16 pairs of expert 0 at a time
        want, iw = m(x[t:t + 8])
        assert np.array_equal(idx[t:t + 8], iw)
        _same(got[t:t + 8], want)
    m.ctx.destroy()
