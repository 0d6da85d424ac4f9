"""Activations with values far below their block's largest (32 columns): some values of every block
are large and meet weights of zero, so that the products are those of the others alone. The expert
products through the device API against float64 on the exactly dequantised weights."""
import numpy as np
import pytest

import k3moe
import oracle as O

pytestmark = pytest.mark.gpu

E = 3


def _zero_columns(codes, rows, cols, at):
    """The nibbles of columns at, at + 32, .. of packed E2M1 codes set to zero."""
    v = codes.reshape(rows, cols // 2)
    v[:, at // 2::16] &= 0x0F if at % 2 else 0xF0


class _Layer:
    """Experts whose gate and up take nothing from columns 32 b + c, c in `big`, and whose down takes
    nothing from features 32 b + 6; those features' up rows are `big_h` (a power of two) times as
    large."""

    def __init__(self, hidden, inter, seed, tiled, big_h=1, big=(5,)):
        shape = k3moe.Shape("outlier", hidden, E, 2, inter, n_shared=0, x_bf16=False, scale_lo=-8,
                            scale_hi=-6)
        self.synth = k3moe.SynthLayer(shape, seed=seed, layout="tiled" if tiled else "engine")
        g, self.w, self.keep = self.synth.geo, [], []
        tab = (k3moe.K3ExpertQ * E)()
        for e in range(E):
            run, ptr, w = self.synth.expert_host(e), [], []
            for m, p, s, r, c in ((1, g.p1_off, g.s1_off, inter, hidden),
                                  (3, g.p3_off, g.s3_off, inter, hidden),
                                  (2, g.p2_off, g.s2_off, hidden, inter)):
                codes, scales = run[p:p + r * c // 2].copy(), run[s:s + r * (c // 32)].copy()
                for at in (6,) if m == 2 else big:
                    _zero_columns(codes, r, c, at)
                if m == 3:
                    scales.reshape(r, c // 32)[6::32] += int(np.log2(big_h))
                w.append(O.oracle().dequant(codes, scales, r, c // 2).reshape(r, c)
                         .astype(np.float64))
                assert not any(w[-1][:, at::32].any() for at in ((6,) if m == 2 else big))
                if tiled:
                    codes, scales = k3moe.tile_mxfp4_host(codes, scales, r, c), None
                for v in (codes, scales):
                    if v is not None:
                        self.keep.append(k3moe.DevBuf.from_array(v))
                    ptr.append(self.keep[-1].ptr if v is not None else None)
            tab[e] = k3moe.K3ExpertQ(*ptr)
            self.w.append(w)
        self.table = k3moe.DevBuf.from_array(np.frombuffer(bytes(tab), np.uint8))
        self.L = self.synth.dev
        self.L.experts = self.table.ptr
        self.kind, self.big = "bf16" if tiled else "gemv", big

    def want(self, x, e):
        g, u = self.w[e][0] @ x, self.w[e][1] @ x
        return self.w[e][2] @ (g / (1.0 + np.exp(-g)) * u)

    def error(self, x, idx, ctx):
        """rel-L2 of the contrib rows"""
        (T, k), d = idx.shape, self.L.hidden
        dx, didx = k3moe.DevBuf.from_array(x), k3moe.DevBuf.from_array(idx.astype(np.int32))
        dc = k3moe.DevBuf.from_array(np.full(T * k * d, np.nan, np.float32))
        ctx.experts(self.kind, self.L, dx.ptr, T, didx.ptr, dc.ptr)
        ctx.sync()
        got = dc.download(np.float32, T * k * d).reshape(T, k, d)
        want = np.array([[self.want(x[t].astype(np.float64), e) for e in idx[t]] for t in range(T)])
        return np.linalg.norm(got - want) / np.linalg.norm(want)


# pairs per expert in one, two, three and four column blocks; widths of whole and ragged 128-column
# steps; every row or one in five with the large values
_SIZES = [(512, 256, 20), (544, 416, 45), (1184, 160, 70), (96, 736, 110)]


def _inputs(m, pairs, scale, every, seed=3):
    T = pairs * E // 2
    idx = np.random.default_rng(seed).permutation(np.repeat(np.arange(E), pairs)[:2 * T]).reshape(T, 2)
    x = m.synth.tokens(T)
    for c in m.big:
        x[::every, c::32] *= np.float32(scale)
    return x, idx


# Four FP6 pieces leave 3e-7 of a block's largest value on each of its values, 8e-5 and 3e-4 of them
# here; two bf16 pieces 2.5e-6 of each. gate, up and down together: three times that.
@pytest.mark.parametrize("hidden,inter,pairs", _SIZES)
@pytest.mark.parametrize("scale,every,big", [(256, 1, 1), (1000, 1, 1), (1000, 5, 1), (1e5, 1, 1),
                                             (300, 1, 4), (300, 1, 16), (3000, 1, 24)])
def test_grouped_x(gpu, hidden, inter, pairs, scale, every, big):
    big = tuple(sorted((5 + 13 * i) % 32 for i in range(big)))
    print(f"case: grouped experts {hidden} x {inter}, {pairs} pairs each, x {scale} times as large in "
          f"columns {big} of 32, every {every}th token", flush=True)
    m = _Layer(hidden, inter, 71, True, big=big)
    x, idx = _inputs(m, pairs, scale, every)
    ctx = k3moe.Ctx(m.L, max_tokens=x.shape[0])
    rel = m.error(x, idx, ctx)
    for c in big:                         # ordinary blocks on the same context
        x[:, c::32] = 0
    plain = m.error(x, idx, ctx)
    ctx.destroy()
    print(f"  rel-L2 {rel:.2e}, without {plain:.2e}", flush=True)
    assert rel <= 7.5e-6 and plain <= 7.5e-6


# Where gates are large, half of h's values are next to nothing: four pieces, for the products are
# those of the others (as for ordinary h).
@pytest.mark.parametrize("hidden,inter,pairs", _SIZES)
def test_grouped_h_of_large_gates(gpu, hidden, inter, pairs):
    print(f"case: grouped experts {hidden} x {inter}, {pairs} pairs each, x 64 times as large", flush=True)
    m = _Layer(hidden, inter, 74, True)
    x, idx = _inputs(m, pairs, 1, 1)
    x *= np.float32(64)
    ctx = k3moe.Ctx(m.L, max_tokens=x.shape[0])
    rel = m.error(x, idx, ctx)
    ctx.destroy()
    print(f"  rel-L2 {rel:.2e}", flush=True)
    assert rel <= 1e-5


# h had been a bf16 piece and an MXFP8 remainder: 4e-5 of each value
@pytest.mark.parametrize("hidden,inter,pairs", _SIZES)
@pytest.mark.parametrize("big_h", [512, 8192])
@pytest.mark.parametrize("bf16", [False, True])
def test_grouped_h(gpu, hidden, inter, pairs, big_h, bf16):
    print(f"case: grouped experts {hidden} x {inter}, {pairs} pairs each, h {big_h} times as large in "
          f"one feature of 32, bf16 x {bf16}", flush=True)
    m = _Layer(hidden, inter, 72, True, big_h)
    x, idx = _inputs(m, pairs, 1, 1)
    if bf16:
        x = (x.view(np.uint32) & np.uint32(0xffff0000)).view(np.float32)
    ctx = k3moe.Ctx(m.L, max_tokens=x.shape[0])
    rel = m.error(x, idx, ctx)
    ctx.destroy()
    print(f"  rel-L2 {rel:.2e}", flush=True)
    assert rel <= 4e-5


# checkpoint-layout experts: fp32's 24 bits of each value, K / 128 sums (1e-6 as for ordinary values)
@pytest.mark.parametrize("hidden,inter,pairs", [(512, 256, 2), (544, 416, 9), (1184, 160, 6)])
@pytest.mark.parametrize("scale,big_h", [(1000, 1), (1e5, 1), (1e9, 1), (1, 4096), (1, 2**40)])
def test_rows(gpu, hidden, inter, pairs, scale, big_h):
    print(f"case: expert rows {hidden} x {inter}, {pairs} pairs each, one column of 32 {scale} and one "
          f"feature {big_h} times as large", flush=True)
    m = _Layer(hidden, inter, 73, False, big_h)
    x, idx = _inputs(m, pairs, scale, 1)
    ctx = k3moe.Ctx(m.L, max_tokens=x.shape[0])
    rel = m.error(x, idx, ctx)
    ctx.destroy()
    print(f"  rel-L2 {rel:.2e}", flush=True)
    assert rel <= 1e-6
