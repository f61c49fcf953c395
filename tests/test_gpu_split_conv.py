"""Convolutions as GEMMs over channel-major activations read in place (k_gemm_x3.hip): transposed
convolutions by taps, strided ones by windows. Every fp32 operand is three bf16 parts, six partial
products are kept.

Bound per element, from the arithmetic, for K products (see test_gpu_split_gemm.py) and at most 8 more
sums of a split K's parts: |y - ref| <= (K / 7 + 12) 2^-24 S, S = sum |a||b| + |bias|.
"""
import numpy as np
import pytest

from metalaudio_amd import nn
from oracle import layers as oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return nn.AudioDevice(0)


def run(dev, layer, *xs):
    s = nn.Stream(dev)
    ts = [nn.Tensor.from_numpy(dev, x) for x in xs]
    out = layer(ts[0], s) if len(ts) == 1 else layer.forward_alloc(*ts, s)
    s.sync(20000)
    return out.to_numpy().astype(np.float64)


def within(y, ref, S, K):
    return np.all(np.abs(y - ref) <= (K / 7 + 12) * 2.0 ** -24 * S)


def weights(r, *shape):
    return (r.standard_normal(shape) * 0.05).astype(np.float32)


# channels (one, partial stages, several stages), outputs, kernel, stride, padding, length, batch:
# 1, 2 and 4 taps; rows of every alignment; lengths below a chunk's window, at tile edges and beyond
TRANSPOSED = [(3, 5, 8, 4, 2, 4, 1), (16, 24, 8, 4, 2, 5, 3), (33, 20, 8, 4, 0, 63, 2),
              (48, 33, 8, 4, 2, 64, 1), (50, 40, 8, 4, 2, 127, 2), (96, 48, 8, 4, 2, 1025, 1),
              (40, 24, 4, 4, 0, 130, 2), (33, 17, 4, 4, 0, 67, 2), (20, 12, 8, 2, 3, 66, 2),
              (7, 9, 16, 4, 6, 259, 1), (384, 192, 8, 4, 2, 86, 1), (64, 48, 8, 4, 2, 9001, 2),
              (128, 40, 8, 4, 2, 301, 1), (250, 31, 8, 4, 2, 67, 2), (256, 17, 4, 4, 0, 130, 1)]


@pytest.mark.parametrize("Cin,Cout,K,s,p,L,B", TRANSPOSED)
def test_taps_error_bound(dev, Cin, Cout, K, s, p, L, B):
    print(f"taps {Cin}->{Cout} k{K} s{s} p{p} L{L} B{B}", flush=True)
    r = np.random.default_rng(Cin * L + K)
    x = r.standard_normal((B, Cin, L)).astype(np.float32)
    w, b = weights(r, Cin, Cout, K), weights(r, Cout)
    layer = nn.ConvTranspose1D(dev, Cin, Cout, K, s, p)
    layer.load_weights(w, b)
    y = run(dev, layer, x)
    ref = oracle.conv_transpose1d(x, w, b, s, p)
    S = oracle.conv_transpose1d(np.abs(x), np.abs(w), np.abs(b), s, p)
    assert within(y, ref, S, K // s * Cin)


@pytest.mark.parametrize("C1,L", [(20, 203), (8, 64), (40, 1000)])
def test_taps_across_the_concatenation(dev, C1, L):
    """Stages whose channels come from both inputs give what stages of one input give, bit for bit."""
    print(f"taps concat {C1} L{L}", flush=True)
    r = np.random.default_rng(C1)
    x = r.standard_normal((2, 48, L)).astype(np.float32)
    args = weights(r, 48, 32, 8), weights(r, 32), np.ones(32, np.float32), np.zeros(32, np.float32)
    ys = []
    for c in (C1, 32):
        block = nn.UNetDecoderBlock(dev, c, 48 - c, 32)
        block.load_weights(*args)
        ys.append(run(dev, block, np.ascontiguousarray(x[:, :c]), np.ascontiguousarray(x[:, c:])))
    np.testing.assert_array_equal(ys[0], ys[1])


def test_taps_not_finite(dev):
    """Infinities reach the outputs under them and no others: not the next channel's row, whose first
    samples lie beside this one's last."""
    print("taps not finite", flush=True)
    r = np.random.default_rng(8)
    Cin, Cout, L = 32, 24, 203
    x = r.standard_normal((1, Cin, L)).astype(np.float32)
    x[0, 4, L - 1] = np.inf
    x[0, 9, 100] = -np.inf
    x[0, 20, 0] = np.nan
    w = r.integers(1, 4, (Cin, Cout, 8)).astype(np.float32)
    layer = nn.ConvTranspose1D(dev, Cin, Cout, 8, 4, 2, use_bias=False)
    layer.load_weights(w)
    y = run(dev, layer, x)
    with np.errstate(invalid="ignore"):
        touched = oracle.conv_transpose1d((~np.isfinite(x)).astype(np.float32), w, None, 4, 2) > 0
    assert np.array_equal(np.isfinite(y), ~touched)
    assert np.all(y[0, :, 399:405] == -np.inf) and np.all(y[0, :, -1] == np.inf)
    assert np.all(np.isnan(y[0, :, 0]))
    x0 = np.where(np.isfinite(x), x, 0)
    ref = oracle.conv_transpose1d(x0, w, None, 4, 2)
    S = oracle.conv_transpose1d(np.abs(x0), w, None, 4, 2)
    # blocks that are computed again in fp32 round once per product
    assert np.all((np.abs(y - ref) <= (2 * Cin + 11) * 2.0 ** -24 * S)[~touched])


# channels, outputs, padding, its mode, length, batch: one stage and more, windows that end at and
# past the signal, row pitches of every alignment, outputs at the edges of the 64..128-wide tiles
STRIDED = [(4, 32, 2, "explicit", 8, 1), (8, 33, 2, "reflect", 21, 2), (12, 96, 2, "reflect", 255, 2),
           (48, 96, 2, "reflect", 1026, 1), (48, 130, 0, "explicit", 516, 2),
           (96, 192, 3, "explicit", 1023, 1), (20, 64, 1, "reflect", 20005, 2)]


@pytest.mark.parametrize("Cin,Cout,p,mode,L,B", STRIDED)
def test_windows_error_bound(dev, Cin, Cout, p, mode, L, B):
    print(f"windows {Cin}->{Cout} p{p} {mode} L{L} B{B}", flush=True)
    r = np.random.default_rng(Cin * L)
    x = r.standard_normal((B, Cin, L)).astype(np.float32)
    w, b = weights(r, Cout, Cin, 8), weights(r, Cout)
    layer = nn.Conv1D(dev, Cin, Cout, 8, 4, p, padding_mode=mode)
    layer.load_weights(w, b)
    y = run(dev, layer, x)
    om = "reflect" if mode == "reflect" else "zeros"
    ref = oracle.conv1d(x, w, b, 4, p, mode=om)
    S = oracle.conv1d(np.abs(x), np.abs(w), np.abs(b), 4, p, mode=om)
    assert within(y, ref, S, 8 * Cin)


def test_windows_not_finite(dev):
    print("windows not finite", flush=True)
    r = np.random.default_rng(9)
    Cin, Cout, L = 16, 48, 518
    x = r.standard_normal((1, Cin, L)).astype(np.float32)
    x[0, 3, L - 1], x[0, 7, 200], x[0, 11, 0] = np.inf, -np.inf, np.nan
    w = r.integers(1, 4, (Cout, Cin, 8)).astype(np.float32)
    layer = nn.Conv1D(dev, Cin, Cout, 8, 4, 2, use_bias=False)
    layer.load_weights(w)
    y = run(dev, layer, x)
    touched = oracle.conv1d((~np.isfinite(x)).astype(np.float32), w, None, 4, 2) > 0
    assert np.array_equal(np.isfinite(y), ~touched)
    assert np.all(np.isnan(y[0, :, 0])) and np.all(y[0, :, 50] == -np.inf)
    x0 = np.where(np.isfinite(x), x, 0)
    ref = oracle.conv1d(x0, w, None, 4, 2)
    S = oracle.conv1d(np.abs(x0), w, None, 4, 2)
    assert np.all((np.abs(y - ref) <= (8 * Cin + 11) * 2.0 ** -24 * S)[~touched])


def test_long_signals(dev):
    """Few channels and 2^25 samples or more, beyond what the transposed form addresses: a Conv1D against
    64 bits at the ends, at every power of two and in between, and an encoder level of a periodic
    signal against a short one, from which its statistics differ by the two edges only."""
    L = 2 ** 25 + 5
    print(f"windows, long signals L{L}", flush=True)
    r = np.random.default_rng(25)
    period = r.standard_normal((8, 4096)).astype(np.float32)
    x = np.tile(period, (1, L // 4096 + 1))[:, :L].copy()
    w, b = weights(r, 32, 8, 8), weights(r, 32)
    layer = nn.Conv1D(dev, 8, 32, 8, 4, 2)
    layer.load_weights(w, b)
    y = run(dev, layer, x[None])[0]
    lo = (L + 4 - 8) // 4 + 1
    assert y.shape == (32, lo)
    pos = np.unique(np.concatenate([np.arange(3), lo - 1 - np.arange(3), 2 ** np.arange(2, 23),
                                    r.integers(0, lo, 2000)]))
    idx = 4 * pos[:, None] - 2 + np.arange(8)
    win = np.where((idx >= 0) & (idx < L), x[:, np.clip(idx, 0, L - 1)], 0).astype(np.float64)
    ref = np.einsum("ocj,cnj->on", w.astype(np.float64), win) + b[:, None]
    S = np.einsum("ocj,cnj->on", np.abs(w).astype(np.float64), np.abs(win)) + np.abs(b)[:, None]
    assert within(y[:, pos], ref, S, 64)
    del y

    block = nn.UNetEncoderBlock(dev, 4, 32, 8, 4, 1, rewrite=True)
    block.load_weights(weights(r, 32, 4, 8), b, 1 + weights(r, 32), weights(r, 32),
                       weights(r, 64, 32, 1), weights(r, 64))
    outs = []
    for n in (2 ** 20, 2 ** 25):
        s = nn.Stream(dev)
        out = block(nn.Tensor.from_numpy(dev, np.ascontiguousarray(x[None, :4, :n])), s)
        s.sync(20000)
        outs.append(out.to_numpy()[0][:, 4096:8192])
    # the mean and variance move by at most 8 of 2^18 columns' share
    np.testing.assert_allclose(outs[1], outs[0], rtol=0, atol=2e-4 * np.abs(outs[0]).max())


@pytest.mark.parametrize("H,W", [(8192, 4096), (5793, 5793)])
def test_large_planes_stay_on_the_matrix_cores(dev, H, W):
    """2-D transposed convolutions of 2^25 positions and more: rows of whole 16-byte chunks and odd ones."""
    print(f"taps, large plane {H}x{W}", flush=True)
    r = np.random.default_rng(H)
    x = np.tile(r.standard_normal((1, 4, 1, W)).astype(np.float32), (1, 1, H, 1))
    x *= np.exp2(np.arange(H) % 7).astype(np.float32)[:, None]
    w, b = weights(r, 4, 3, 1, 1), weights(r, 3)
    layer = nn.ConvTranspose2D(dev, 4, 3, 1)
    layer.load_weights(w, b)
    dev.set_kernel_timing(True)
    dev.reset_kernel_timing()
    y = run(dev, layer, x)
    launches = dev.kernel_timing("convt2d_f32_mfma")[0]
    dev.set_kernel_timing(False)
    assert launches == 1
    for rows in (slice(0, 4), slice(H // 2, H // 2 + 4), slice(H - 4, H)):
        xr = x[0, :, rows].astype(np.float64)
        ref = np.einsum("io,ihw->ohw", w[:, :, 0, 0].astype(np.float64), xr) + b[:, None, None]
        S = np.einsum("io,ihw->ohw", np.abs(w[:, :, 0, 0]).astype(np.float64), np.abs(xr))
        S += np.abs(b)[:, None, None]
        assert within(y[0][:, rows], ref, S, 4)


def test_one_product_per_output(dev):
    """Windows and taps that meet a single sample: as test_gpu_split_gemm.py's rows with one element."""
    print("windows, taps: one product", flush=True)
    r = np.random.default_rng(15)
    C = 16
    x = np.zeros((1, C, 16384), np.float32)
    n = np.arange(0, 16384, 8)
    x[0, n // 8 % C, n] = np.exp2(r.uniform(0, 1, n.size))
    mantissas = lambda *shape: np.exp2(r.uniform(0, 1, shape)).astype(np.float32)
    w = mantissas(48, C, 8)
    conv = nn.Conv1D(dev, C, 48, 8, 4, 0, use_bias=False)
    conv.load_weights(w)
    v = mantissas(C, 24, 8)
    convt = nn.ConvTranspose1D(dev, C, 24, 8, 4, 2, use_bias=False)
    convt.load_weights(v)
    for y, ref in ((run(dev, conv, x), oracle.conv1d(x, w, None, 4, 0)),
                   (run(dev, convt, x), oracle.conv_transpose1d(x, v, None, 4, 2))):
        assert np.all(np.abs(y - ref) <= 2.1 * 2.0 ** -24 * np.abs(ref))


@pytest.mark.parametrize("split", ["2", "5"])
def test_forced_split_leaves_plain_convolutions(dev, monkeypatch, split):
    """MNN_ENC_CONV_SPLIT forces the encoders' K split; a plain Conv1D, which has none, still runs."""
    print(f"windows, forced split {split}", flush=True)
    monkeypatch.setenv("MNN_ENC_CONV_SPLIT", split)
    test_windows_error_bound(dev, 20, 64, 1, "reflect", 2005, 2)
    test_windows_error_bound(dev, 48, 96, 2, "reflect", 1026, 1)
