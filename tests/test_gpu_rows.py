"""The routed experts of checkpoint-layout MXFP4 weights (eight FP6 pieces on the FP4 x FP6 matrix
cores) at the edges of their tiles, through k3g_expert_gemv, against the expert products in float64
on the exactly dequantised weights."""
import ctypes as C

import numpy as np
import pytest

import k3moe
import oracle as O

pytestmark = pytest.mark.gpu

# Eight E2M3 pieces leave at most 2^-32 of a block's largest value (1/16 each); the
# products accumulate in fp32, K / 128 sums a column: 6e-8 sqrt(K / 128) of the largest partial
# sum, below 3e-7 of the result at K <= 1200, over gate, up and down.
REL = 1e-6



class _Layer:
    """A layer whose expert table points at copies of the experts' codes and scales at `at` bytes
    past an aligned address (codes, scales), with scale bytes 255 (a block of zeros) and 0 among
    them if `ends`."""

    def __init__(self, hidden, inter, n_experts, seed, at=(0, 0), ends=True):
        shape = k3moe.Shape("rows", hidden, n_experts, 2, inter, n_shared=0, x_bf16=False,
                            scale_lo=-8, scale_hi=-6)
        self.synth = k3moe.SynthLayer(shape, seed=seed, layout="engine")
        g, self.w, self.keep = self.synth.geo, [], []
        tab = (k3moe.K3ExpertQ * n_experts)()
        for e in range(n_experts):
            run, ptr, w = self.synth.expert_host(e), [], []
            for p, s, r, c in ((g.p1_off, g.s1_off, inter, hidden),
                               (g.p3_off, g.s3_off, inter, hidden),
                               (g.p2_off, g.s2_off, hidden, inter)):
                codes, scales = run[p:p + r * c // 2], run[s:s + r * (c // 32)]
                if ends:
                    scales[5::97], scales[7::89] = 255, 0
                w.append(O.oracle().dequant(codes, scales, r, c // 2).reshape(r, c)
                         .astype(np.float64))
                for v, o in ((codes, at[0]), (scales, at[1])):
                    b = k3moe.DevBuf(v.size + o)
                    b.upload(v, o)
                    self.keep.append(b)
                    ptr.append(b.ptr + o)
            tab[e] = k3moe.K3ExpertQ(*ptr)
            self.w.append(w)
        self.table = k3moe.DevBuf.from_array(np.frombuffer(bytes(tab), np.uint8))
        self.L = self.synth.dev
        self.L.experts = self.table.ptr

    def h(self, x, e):
        g, u = self.w[e][0] @ x, self.w[e][1] @ x
        with np.errstate(over="ignore"):
            return g / (1.0 + np.exp(-g)) * u

    def contrib(self, x, idx):
        (T, k), d = idx.shape, self.L.hidden
        ctx = k3moe.Ctx(self.L, max_tokens=T)
        dx = k3moe.DevBuf.from_array(x.astype(np.float32))
        didx = k3moe.DevBuf.from_array(idx.astype(np.int32))
        dc = k3moe.DevBuf.from_array(np.full(T * k * d, np.nan, np.float32))
        ctx.experts("gemv", self.L, dx.ptr, T, didx.ptr, dc.ptr)
        ctx.sync()
        out = dc.download(np.float32, T * k * d).reshape(T, k, d)
        ctx.destroy()
        return out


# widths whole, ragged in the 128-column steps and the 256- and 512-column intervals, below one
# step; pairs per expert at the edges of the passes of 8 and of their groups of 2
@pytest.mark.parametrize("hidden,inter,at", [
    (1024, 256, (0, 0)), (1184, 544, (0, 1)), (544, 96, (8, 3)), (288, 800, (4, 2)),
    (32, 32, (0, 0))])
def test_tile_edges(gpu, hidden, inter, at):
    counts = [1, 2, 3, 4, 5, 7, 8, 9, 17]
    print(f"case: expert rows hidden={hidden} inter={inter}, {counts} pairs, {at} past aligned",
          flush=True)
    m = _Layer(hidden, inter, len(counts), 41, at)
    idx = np.random.default_rng(1).permutation(
        np.concatenate([np.full(n, e) for e, n in enumerate(counts)])).reshape(-1, 2)
    x = m.synth.tokens(idx.shape[0])
    got = m.contrib(x, idx)
    want = np.array([[m.w[e][2] @ m.h(x[t].astype(np.float64), e) for e in idx[t]]
                     for t in range(idx.shape[0])])
    rel = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(f"  rel-L2 {rel:.2e}", flush=True)
    assert rel <= REL


def test_not_finite(gpu):
    """Infinities and NaN give what the products in fp32 give, and no other pair's rows change:
    an h that overflows leaves the sign of its weight, or NaN where that is zero."""
    print("case: expert rows, tokens with NaN and with one h past fp32", flush=True)
    # (without the scale bytes 255 and 0: the conversion makes 2^-127 of both, subnormal weights)
    m = _Layer(544, 96, 3, 42, ends=False)
    idx = np.array([[0, 1], [1, 2], [2, 0], [1, 0]], np.int32)
    x = m.synth.tokens(4)
    clean = m.contrib(x, idx)
    assert np.isfinite(clean).all()
    x[0, 9] = np.nan
    x[2] *= np.float32(1e15)
    top = np.sort(np.abs(m.h(x[2].astype(np.float64), 2)))[-2:]
    x[2] *= np.float32(np.sqrt(np.finfo(np.float32).max / np.sqrt(top[0] * top[1])))
    got = m.contrib(x, idx)
    assert np.isnan(got[0]).all()
    with np.errstate(over="ignore", invalid="ignore"):
        h = m.h(x[2].astype(np.float64), 2).astype(np.float32)
        assert np.isinf(h).sum() == 1
        want = m.w[2][2] @ h.astype(np.float64)
    assert np.isinf(want).any() and np.isnan(want).any()
    assert np.array_equal(got[2, 0], want.astype(np.float32), equal_nan=True)
    assert np.array_equal(got[[1, 3]].view(np.uint32), clean[[1, 3]].view(np.uint32))


# each count of rows per wave (16 .. 1 by the number of row tiles and tokens), rows that do not
# fill the last wave, widths below and past a wave's 1024 columns
@pytest.mark.parametrize("T", [1, 4, 5])
@pytest.mark.parametrize("rows,K", [(37, 16), (2051, 1040), (4097, 48), (8195, 32), (16390, 16),
                                    (32780, 16)])
def test_dense_rows_per_wave(gpu, T, rows, K):
    """bf16 products by row, alone and as silu(a) b, against float64: K fp32 multiply-adds."""
    print(f"case: k3k_dense bf16 {rows} x {K}, {T} tokens", flush=True)
    rng = np.random.default_rng(rows + K)
    a, b = (rng.standard_normal((rows, K)).astype(np.float32).view(np.uint32) >> 16
            for _ in range(2))
    x = rng.standard_normal((T, K)).astype(np.float32)
    fa, fb = ((v << 16).astype(np.uint32).view(np.float32).astype(np.float64) for v in (a, b))
    da, db = (k3moe.DevBuf.from_array(v.astype(np.uint16)) for v in (a, b))
    dx, dy = k3moe.DevBuf.from_array(x), k3moe.DevBuf(T * rows * 4)
    fn = k3moe.lib().k3k_dense
    fn.argtypes = [C.c_int, C.c_void_p, C.c_void_p, C.c_int, C.c_int, C.c_void_p, C.c_int, C.c_int,
                   C.c_void_p, C.c_int, C.c_float, C.c_float, C.c_void_p]
    g, u = x @ fa.T, x @ fb.T
    for wb, want in ((None, g), (db.ptr, g / (1.0 + np.exp(-g)) * u)):
        assert fn(2, da.ptr, wb, rows, K, dx.ptr, K, T, dy.ptr, rows, k3moe.SWIGLU_CAP,
                  k3moe.SWIGLU_CAP, None) == 0
        k3moe.sync()
        got = dy.download(np.float32, T * rows).reshape(T, rows)
        assert np.linalg.norm(got - want) <= 1e-6 * np.linalg.norm(want)
