"""The routed experts' grouped GEMMs (FP6 pieces on the FP4 x FP6 matrix cores; bf16 gate/up where
every x is a bf16 value) at the edges of their tiles, through k3g_grouped_gemm_bf16, against the
expert products in float64 on the exactly dequantised weights."""
import ctypes as C

import numpy as np
import pytest

import k3moe
import oracle as O

pytestmark = pytest.mark.gpu

# Four E2M3 pieces: each leaves at most 1/16 of its block's largest value (a spacing of 0.5 where
# the scale puts that value in [4, 8)), so 2^-16 of it in all at worst, 2^-20 in the mean. Over
# gate, up and down the worst case is 3 * 2^-16 * sqrt(32) of a row that one value dominates; the
# mean case is 3e-6. fp32 accumulation of 2^10 products adds below 1e-6.
REL = 1e-5


def _expert(layer, e):
    """One expert's w1, w3, w2 as float64."""
    s, g = layer.shape, layer.geo
    d, i = s.hidden, s.inter
    run = layer.expert_host(e)
    return [O.oracle().dequant(run[po:po + r * c // 2], run[so:so + r * (c // 32)], r, c // 2)
            .reshape(r, c).astype(np.float64)
            for po, so, r, c in ((g.p1_off, g.s1_off, i, d), (g.p3_off, g.s3_off, i, d),
                                 (g.p2_off, g.s2_off, d, i))]


def _dequant(layer):
    return [_expert(layer, e) for e in range(layer.shape.n_experts)]


def _rows(layer, x, idx, offset=0, trace=None):
    """contrib [T][k][d] (NaN where the call leaves a row alone); x at offset floats."""
    T, k = idx.shape
    d = layer.shape.hidden
    L = layer.dev_tiled
    ctx = k3moe.Ctx(L, max_tokens=T)
    dx = k3moe.DevBuf((x.size + offset) * 4)
    dx.upload(x.astype(np.float32), 4 * offset)
    didx = k3moe.DevBuf.from_array(idx.astype(np.int32))
    dc = k3moe.DevBuf.from_array(np.full(T * k * d, np.nan, np.float32))
    if trace is not None:
        k3moe.lib().k3g_ctx_set_trace(ctx.ptr, C.c_void_p(trace.ptr))
    ctx.experts("bf16", L, dx.ptr + 4 * offset, T, didx.ptr, dc.ptr)
    ctx.sync()
    out = dc.download(np.float32, T * k * d).reshape(T, k, d)
    ctx.destroy()
    return out


def _want(w, x, e):
    g, u = w[e][0] @ x, w[e][1] @ x
    with np.errstate(over="ignore"):
        return w[e][2] @ (g / (1.0 + np.exp(-g)) * u)


# pairs per expert at the edges of the 16-column blocks, of the 64-pair items and of the 128-pair
# tiles; widths whole, ragged in the 128-column steps and the 512-column quads, below one step
@pytest.mark.parametrize("hidden,inter", [(512, 256), (544, 416), (1184, 96), (96, 736)])
@pytest.mark.parametrize("bf16", [False, True])
def test_tile_edges(gpu, hidden, inter, bf16):
    counts = [1, 15, 16, 17, 33, 48, 49, 64, 65, 127, 128, 129, 200]
    print(f"case: grouped experts hidden={hidden} inter={inter} bf16 x={bf16}, {counts} pairs",
          flush=True)
    shape = k3moe.Shape("edge", hidden, len(counts), 2, inter, n_shared=0, x_bf16=bf16,
                        scale_lo=-8, scale_hi=-6)
    layer = k3moe.SynthLayer(shape, seed=31, layout="both")
    pairs = np.concatenate([np.full(n, e) for e, n in enumerate(counts)])
    pairs = np.random.default_rng(1).permutation(pairs)
    if pairs.size % 2:
        pairs = np.append(pairs, -1)
    idx = pairs.reshape(-1, 2)
    x = layer.tokens(idx.shape[0])
    got = _rows(layer, x, idx)
    w = _dequant(layer)
    num = den = 0.0
    for t in range(idx.shape[0]):
        for j in range(2):
            if idx[t, j] < 0:
                assert np.isnan(got[t, j]).all()
                continue
            want = _want(w, x[t].astype(np.float64), idx[t, j])
            num += np.sum((got[t, j] - want) ** 2)
            den += np.sum(want ** 2)
    rel = np.sqrt(num / den)
    print(f"  rel-L2 {rel:.2e}", flush=True)
    assert rel <= REL


def test_many_tiles_take_the_tall_workgroups(gpu):
    """Enough column tiles for the 512-row workgroups of gate/up and of down, 3 and 4 column blocks,
    an odd number of feature tiles, the last one ragged; and the workgroups' records: one of every
    column tile and feature tile (128 features of gate/up, 512 rows of down)."""
    E, hidden, inter = 300, 1760, 864
    print(f"case: grouped experts, {E} experts x 40 and 60 pairs, hidden {hidden} inter {inter}", flush=True)
    nf, nr = -(-inter // 128), -(-hidden // 256)
    assert nf % 2 and nr % 2 and E * ((nf + 1) // 2) >= 1024 and E * ((nr + 1) // 2) >= 1024
    shape = k3moe.Shape("tall", hidden, E, 1, inter, n_shared=0, x_bf16=False, scale_lo=-8, scale_hi=-6)
    layer = k3moe.SynthLayer(shape, seed=32, layout="both")
    idx = np.random.default_rng(2).permutation(
        np.concatenate([np.full(40 + 20 * (e % 2), e) for e in range(E)])).reshape(-1, 1)
    T = idx.shape[0]
    x = layer.tokens(T)
    places = 32 * -(-(-(-T // 128) + E) // 32)
    n0, n1 = places * nf, places * -(-hidden // 512)
    trace = k3moe.DevBuf.from_array(np.zeros(4 * (n0 + n1), np.uint64))
    got = _rows(layer, x, idx, trace=trace)
    for t in range(0, T, 97):
        want = _want({idx[t, 0]: _expert(layer, idx[t, 0])}, x[t].astype(np.float64), idx[t, 0])
        assert np.linalg.norm(got[t, 0] - want) <= REL * np.linalg.norm(want)
    rec = trace.download(np.uint64, 4 * (n0 + n1)).reshape(-1, 4)
    for part, n in ((rec[:n0], nf), (rec[n0:], -(-hidden // 512))):
        part = part[part[:, 1] != 0]
        assert (part[:, 0] != 0).all() and (part[:, 0] <= part[:, 1]).all()
        assert sorted(part[:, 2].tolist()) == [t << 32 | f for t in range(E) for f in range(n)]


def test_not_finite_and_unaligned_x(gpu):
    """A token with an infinity or a NaN gives NaN rows and no other token's; x at an address
    that is not a multiple of 16 bytes gives the same bits."""
    print("case: grouped experts, tokens with inf and NaN, x at 4 bytes past 16", flush=True)
    shape = k3moe.Shape("nan", 544, 4, 2, 416, n_shared=0, x_bf16=False, scale_lo=-8, scale_hi=-6)
    layer = k3moe.SynthLayer(shape, seed=33, layout="both")
    idx = np.random.default_rng(3).integers(0, 4, (40, 2))
    x = layer.tokens(40)
    clean = _rows(layer, x, idx)
    assert np.isfinite(clean).all()
    assert np.array_equal(_rows(layer, x, idx, offset=1).view(np.uint32), clean.view(np.uint32))
    x[7, 100], x[8, 3], x[30, 543] = np.inf, np.nan, -np.inf
    got = _rows(layer, x, idx)
    bad = [7, 8, 30]
    assert np.isnan(got[bad]).all()
    keep = [t for t in range(40) if t not in bad]
    assert np.array_equal(got[keep].view(np.uint32), clean[keep].view(np.uint32))
