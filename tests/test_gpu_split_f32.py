"""GPU: the f32 convolutions that run on the bf16 matrix cores (three bf16 pieces per value, six
piece products, csrc/split.h) against 64-bit sums, at the edges of their tiles, on values that are not
finite, at both ends of f32's range, and the fused blocks against the single layers.

Worst case: the matrix core rounds its f32 accumulator once per 8 products; the full-size accumulator
takes 16 of the K products per 4 such roundings, its partner twice as many of sums 2^-7 as large, the
dropped products are 2^-24 of a product, and bias, final sum and store add three roundings; a 1x1 layer
adds the two accumulators every 32 products. Every rounding is at most 2^-23 (it may truncate) of a
partial sum, itself at most S = |b| + sum |x w|, so |err| <= (K / 4 * (1 + 2^-6) + 4.5 + [1x1] (K / 32 +
1)) * 2^-23 * S.

That bound grows past the third pieces' part of a result, so that of random products (rms_bound) is held
too: roundings to nearest are at most 2^-24 of a partial sum and independent, so that the rms of err / S2,
S2^2 = b^2 + sum (x w)^2, stays below (sqrt(K / 7) + 2) * 2^-24: K / 4 + K / 32 roundings of partial sums
of half the mean square, and the rest. A missing piece product leaves 2.7e-6 at least, whatever K is
(tests/test_split_bounds.py)."""

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from zenjpegai_amd import _lib, model, nn, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = nn.Engine(0, "f32")
    yield e
    e.close()


def rms_bound(k):
    return ((k / 7) ** 0.5 + 2) * 2.0 ** -24


def _layer(eng, kind, cin, cout, groups, seed):
    if kind in ("t3", "t4"):  # stride 2, padding 1
        k = int(kind[1])
        w = synth.normal(seed, f"split/w{kind}{cin}{cout}", (cin, cout, k, k), 1.0)
        b = synth.normal(seed, f"split/b{cout}", (cout,), 1.0)

        def ref_t(x, w, b):
            t = [torch.from_numpy(a).double() for a in (x[None], w, b)]
            return F.conv_transpose2d(*t, 2, 1, 4 - k)[0].numpy()

        return w, b, lambda w, b: nn.ConvTransposeLayer(nn.ConvTranspose2d(cin, cout, k, 2, 1, 4 - k, w, b), eng), ref_t
    k, stride = {"1x1": (1, 1), "3x3": (3, 1), "s2": (3, 2), "2x2": (2, 1)}[kind]
    w = synth.normal(seed, f"split/w{kind}{cin}{cout}", (cout, cin // groups, k, k), 1.0)
    b = synth.normal(seed, f"split/b{cout}", (cout,), 1.0)
    pad, ext = {"1x1": ((0, 0), (0, 0, 0, 0)), "2x2": ((0, 0), (0, 0, 1, 1))}.get(kind, ((1, 1), (0, 0, 0, 0)))

    def ref(x, w, b):
        x = torch.from_numpy(x).double()[None]
        x = F.pad(x, {"1x1": (0, 0, 0, 0), "2x2": (0, 1, 0, 1)}.get(kind, (1, 1, 1, 1)))
        return F.conv2d(x, torch.from_numpy(w).double(), torch.from_numpy(b).double(), stride, 0, 1, groups)[0].numpy()

    return w, b, lambda w, b: nn.ConvLayer(nn.Conv2d(cin, cout, (k, k), stride, pad, groups, w, b), eng, extra_pad=ext), ref


# (kind, cin, cout, groups, h, w): every tile shape, channel counts off 16 and 64, one-row and
# one-column maps, sizes around the 16-column and 4- / 8- / 16-row tiles.
CASES = [("3x3", 4, 4, 1, 1, 1), ("3x3", 20, 24, 1, 9, 17), ("3x3", 160, 160, 1, 13, 19), ("3x3", 48, 40, 1, 130, 66),
         ("3x3", 64, 128, 1, 90, 97), ("3x3", 32, 128, 1, 177, 190), ("3x3", 16, 192, 1, 200, 210),
         ("3x3", 16, 128, 1, 260, 250), ("3x3", 64, 64, 4, 33, 31), ("3x3", 64, 64, 4, 150, 161),
         ("3x3", 128, 128, 4, 15, 16), ("3x3", 128, 128, 4, 150, 161), ("s2", 20, 16, 1, 1, 7), ("s2", 64, 64, 1, 35, 33),
         ("s2", 24, 32, 1, 66, 64), ("s2", 64, 64, 1, 175, 177), ("s2", 16, 128, 1, 255, 257), ("s2", 16, 128, 1, 440, 431),
         ("s2", 16, 192, 1, 440, 431), ("s2", 16, 16, 1, 500, 431), ("s2", 20, 12, 1, 450, 515),
         ("2x2", 160, 256, 1, 4, 6), ("2x2", 20, 12, 1, 17, 15), ("2x2", 64, 128, 1, 128, 127),
         ("2x2", 16, 16, 1, 210, 201), ("2x2", 20, 12, 1, 300, 130),
         ("2x2", 16, 192, 1, 150, 161), ("1x1", 4, 4, 1, 1, 1), ("1x1", 20, 24, 1, 9, 7), ("1x1", 48, 16, 1, 33, 64),
         ("1x1", 160, 160, 1, 8, 15), ("1x1", 128, 64, 1, 128, 127), ("1x1", 96, 128, 1, 150, 130),
         ("1x1", 32, 256, 1, 171, 190), ("1x1", 16, 12, 1, 240, 251), ("1x1", 12, 36, 1, 301, 260),
         ("1x1", 8, 200, 1, 130, 129), ("t3", 20, 12, 1, 1, 1), ("t3", 36, 64, 1, 17, 15), ("t3", 32, 96, 1, 90, 97),
         ("t3", 16, 128, 1, 130, 33), ("t4", 20, 24, 1, 3, 5), ("t4", 48, 64, 1, 31, 34), ("t4", 16, 160, 1, 70, 65),
         ("t4", 16, 128, 1, 135, 100)]


@pytest.mark.parametrize("kind,cin,cout,groups,h,w", CASES)
def test_error_against_64_bits(eng, kind, cin, cout, groups, h, w):
    wt, b, make, ref = _layer(eng, kind, cin, cout, groups, 31)
    x = synth.normal(32, f"split/x{cin}{h}", (cin, h, w), 1.0)
    y = make(wt, b).forward(eng, nn.BTensor.from_planar(eng, x)).to_planar()
    want, size = ref(x, wt, b), ref(np.abs(x), np.abs(wt), np.abs(b))
    assert y.shape == want.shape
    kk = cin * 4 if kind[0] == "t" else wt[0].size  # at most 2 x 2 taps reach an output
    bound = (kk / 4 * (1 + 2.0 ** -6) + 4.5 + (kk / 32 + 1 if kind == "1x1" else 0)) * 2.0 ** -23 * size
    assert np.all(np.abs(y - want) <= bound), float(np.max(np.abs(y - want) / bound))
    if y.size >= 1000:
        rms = float(np.sqrt(np.mean((y - want) ** 2 / ref(x * x, wt * wt, b * b))))
        assert rms <= rms_bound(kk), (rms, rms_bound(kk))


@pytest.mark.parametrize("kind", ["1x1", "3x3", "s2", "2x2", "t3", "t4"])
def test_values_that_are_not_finite(eng, kind):
    """Infinities and NaN in the input or the weights reach the outputs that f32 arithmetic sends
    them to, and only those."""
    wt, b, make, ref = _layer(eng, kind, 32, 16, 1, 33)
    if kind[0] == "t":
        wt = np.ascontiguousarray(wt.transpose(1, 0, 2, 3))  # outputs first, as the others, for the edits below
    wt[3, 5] = 0.0  # 0 * inf is NaN
    x = synth.normal(34, "split/nf", (32, 24, 40), 1.0)
    for ch, r, c, v in ((0, 2, 3, np.inf), (5, 7, 20, -np.inf), (9, 12, 33, np.nan), (31, 23, 39, np.inf), (5, 18, 8, np.inf), (6, 18, 9, -np.inf)):
        x[ch, r, c] = v
    for w in (wt, np.where(np.arange(16)[:, None, None, None] == 7, np.float32(np.inf), wt)):
        w = np.ascontiguousarray(w.transpose(1, 0, 2, 3) if kind[0] == "t" else w)
        y = make(w, b).forward(eng, nn.BTensor.from_planar(eng, x)).to_planar()
        want = ref(x, w, b)
        np.testing.assert_array_equal(np.isnan(y), np.isnan(want))
        inf = np.isinf(want)
        np.testing.assert_array_equal(y[inf], want[inf])
        fin = np.isfinite(want)
        assert np.isfinite(y[fin]).all() and np.allclose(y[fin], want[fin], rtol=1e-4, atol=1e-3)


@pytest.fixture(scope="module")
def eng_igemm():
    e = nn.Engine(0, "f32", flags=_lib.CTX_IGEMM_CONV1X1)
    yield e
    e.close()


# (kind, cin, cout, channel, columns between values): single chunks, whole and odd pairs of chunks, wide and
# narrow tiles, the transposed layers phase by phase and (at 1280 columns) merged.
ONE_CHANNEL = [("1x1", 4, 64, 2, 4), ("1x1", 32, 64, 21, 4), ("1x1", 48, 16, 40, 4), ("1x1", 160, 160, 70, 4),
               ("3x3", 4, 128, 1, 4), ("3x3", 64, 64, 50, 4), ("s2", 20, 128, 17, 4), ("2x2", 36, 64, 33, 4),
               ("t3", 20, 64, 7, 4), ("t3", 32, 128, 30, 32), ("t4", 32, 32, 11, 4)]
N_VALUES = 40


def _products(e, kind, cin, cout, ch, step, xv, wv):
    """wv[o] * xv[i] as the layer computes them, [o][i]: the input is zero but for channel ch of every
    step-th column, the weights but for the tap of that channel on the output's own position."""
    x = np.zeros((cin, 1, step * len(xv)), np.float32)
    x[ch, 0, ::step] = xv
    if kind[0] == "t":
        k = int(kind[1])
        w = np.zeros((cin, cout, k, k), np.float32)
        w[ch, :, 1, 1] = wv
        layer = nn.ConvTransposeLayer(nn.ConvTranspose2d(cin, cout, k, 2, 1, 4 - k, w, np.zeros(cout, np.float32)), e)
        scale = 2
    else:
        k, stride = {"1x1": (1, 1), "3x3": (3, 1), "s2": (3, 2), "2x2": (2, 1)}[kind]
        pad, ext = {"1x1": ((0, 0), (0, 0, 0, 0)), "2x2": ((0, 0), (0, 0, 1, 1))}.get(kind, ((1, 1), (0, 0, 0, 0)))
        w = np.zeros((cout, cin, k, k), np.float32)
        w[:, ch, (k - 1) // 2, (k - 1) // 2] = wv
        layer = nn.ConvLayer(nn.Conv2d(cin, cout, (k, k), stride, pad, 1, w, np.zeros(cout, np.float32)), e, extra_pad=ext)
        scale = 1 / stride
    y = layer.forward(e, nn.BTensor.from_planar(e, x)).to_planar()
    return y[:, 0, ::int(step * scale)][:, :len(xv)]


def _cycle(values, n):
    return np.resize(np.asarray(values, np.float32), n)


F32 = np.finfo(np.float32)
# Around 0x7f7f7fff, the largest f32 that rounds to a finite bf16, and up to f32's own largest.
TOP = np.array([0x7f7f7fff, 0x7f7f8000, 0x7f7f8001, 0x7f7fffff, 0x7f7fffa5, 0x7f7e1234, 0x7f7f6f43, 0x7f6fffff],
               np.uint32).view(np.float32)


@pytest.mark.parametrize("kind,cin,cout,ch,step", ONE_CHANNEL)
@pytest.mark.parametrize("weights", [False, True])
def test_the_largest_finite_values(eng, eng_igemm, kind, cin, cout, ch, step, weights):
    """Finite values above bf16's largest are three pieces like any other: times zero and the powers of
    two up to one every bit is there, times other values the six products' 2^-22."""
    top, other = np.concatenate([TOP, -TOP]), [0.0, 1.0, -1.0, 0.5, -2.0 ** -20, 2.0 ** -100, 0.3, -0.7123456]
    xv, wv = (_cycle(other, N_VALUES), _cycle(top, cout)) if weights else (_cycle(top, N_VALUES), _cycle(other, cout))
    want = wv[:, None] * xv
    exact = np.frexp(np.abs(wv[:, None] if not weights else xv[None]))[0] * np.ones_like(want)
    exact = (exact == 0.5) | (exact == 0)
    for e in (eng, eng_igemm) if kind == "1x1" else (eng,):
        y = _products(e, kind, cin, cout, ch, step, xv, wv)
        np.testing.assert_array_equal(y[exact], want[exact])
        np.testing.assert_allclose(y[~exact], want[~exact], rtol=2.0 ** -22)


@pytest.mark.parametrize("kind,cin,cout,ch,step", ONE_CHANNEL)
def test_single_values_that_are_not_finite(eng, eng_igemm, kind, cin, cout, ch, step):
    """Every pairing of infinities, NaN, zeros, values of one, two and three pieces and the largest ones,
    one product an output: what f32 gives, infinity times infinity among it."""
    v = [np.inf, -np.inf, np.nan, 0.0, 1.0, -1.0 - 2.0 ** -9, 0.3, F32.max, -F32.max, 1e-30]
    xv, wv = _cycle(v, N_VALUES), _cycle(np.repeat(v, 2), cout)
    with np.errstate(all="ignore"):
        want = wv[:, None] * xv
    for e in (eng, eng_igemm) if kind == "1x1" else (eng,):
        y = _products(e, kind, cin, cout, ch, step, xv, wv)
        fin = np.isfinite(want)
        np.testing.assert_array_equal(y[~fin], want[~fin])
        np.testing.assert_allclose(y[fin], want[fin], rtol=2.0 ** -22)


@pytest.mark.parametrize("kind,cin,cout,ch,step", ONE_CHANNEL)
@pytest.mark.parametrize("igemm", [False, True])
def test_products_that_overflow(eng, eng_igemm, kind, cin, cout, ch, step, igemm):
    """A finite product past f32's largest is infinite, of its own sign, although its small piece
    products may have overflowed to the other one."""
    n = N_VALUES
    xv = synth.uniform(35, "split/ovx", (n,), 1.0, 2.0) * _cycle([-1e30, 1e30], n)
    wv = synth.uniform(36, f"split/ovw{cout}", (cout,), 1.0, 2.0) * _cycle([-1e30, 1e30, 1e30], cout)
    with np.errstate(over="ignore"):
        want = wv[:, None] * xv
    assert np.isinf(want).all()
    np.testing.assert_array_equal(_products(eng_igemm if igemm else eng, kind, cin, cout, ch, step, xv, wv), want)


@pytest.mark.parametrize("op,comp", [("sop", "y"), ("hop", "y"), ("hop", "uv")])
def test_fused_blocks_split_large_values_as_the_single_layers_do(op, comp):
    """Every fifth gate value of the feed-forward halves and channel inside the ResAUs past the size from
    which a p0 is cut off (taken back by the next weights): waves of the fused kernels then split both
    kinds, to the same bits as the layers by themselves."""
    p = {k: np.array(v) for k, v in synth.random_params(op, comp, seed=41, gain=0.5).items()}
    big = np.float32(2.0 ** 18)
    n = 0
    for k in p:
        if k.endswith("ffn.dwconv.weight"):
            hid = p[k].shape[0] // 2
            p[k][hid::5] *= big
            p[k.replace("dwconv", "project_out")][:, ::5] /= big
            n += 1
        elif k.endswith(".conv2.weight") and k.replace("conv2", "conv") in p and p[k].shape[2] == 1:
            p[k.replace("conv2", "conv")][::5] *= big
            p[k][:, ::5] /= big
            n += 1
    assert n >= 2, n
    lh, lw = 7, 9
    y, uv = synth.latent(41, "big/y", 160, lh, lw), synth.latent(41, "big/uv", 96, lh, lw)
    outs = []
    for flags in (0, _lib.CTX_UNFUSED_BLOCKS):
        e = nn.Engine(0, "f32", flags=flags)
        yt = nn.BTensor.from_planar(e, y)
        if comp == "y":
            outs.append(model.SynthesisPrimary.load(p, op, e).forward(e, yt, 16 * lh, 16 * lw))
        else:
            net = model.SynthesisSecondary.load(p, op, e)
            outs.append(net.forward(e, yt, nn.BTensor.from_planar(e, uv), 16 * lh, 16 * lw))
        e.close()
    assert np.isfinite(outs[0]).all() and len(np.unique(outs[0])) > 1000
    np.testing.assert_array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))


@pytest.mark.parametrize("kind,cin,cout,ch,step", ONE_CHANNEL)
@pytest.mark.parametrize("weights", [False, True])
def test_the_smallest_values(eng, kind, cin, cout, ch, step, weights):
    """Below 2^-110 the pieces run out of bf16's exponents: what is left of an operand is within 2^-134 (half
    of the smallest bf16) of it, and the rest as for any other product."""
    n = N_VALUES
    tiny = synth.uniform(37, "split/tiny", (n,), 1.0, 2.0) * (2.0 ** -np.linspace(100, 149, n)).astype(np.float32)
    tiny, other = np.concatenate([tiny[::2], -tiny[1::2]]).astype(np.float32), [1.0, -0.3, 2.0 ** 60, 1.2345e37, 0.0]
    xv, wv = (_cycle(other, n), _cycle(tiny, cout)) if weights else (tiny, _cycle(other, cout))
    want = wv[:, None].astype(np.float64) * xv
    left = np.abs(_cycle(other, n)[None] if weights else _cycle(other, cout)[:, None]) * 2.0 ** -134
    y = _products(eng, kind, cin, cout, ch, step, xv, wv)
    bound = left * (1 + 2.0 ** -7) + 2.0 ** -22 * np.abs(want) + 2.0 ** -149
    assert np.all(np.abs(y - want) <= bound), float(np.max(np.abs(y - want) / bound))
