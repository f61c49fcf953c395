"""The fp32 GEMM whose products run on the bf16 matrix cores (k_gemm_x3.hip), through Linear: every
fp32 operand is three bf16 parts, six partial products are kept.

Bound per element, from the arithmetic, in units of 2^-24 S, S = sum |a||b| + |bias|: the dropped
products m*l + l*m + l*l are at most (2 * 2^-8 * 2^-17 + 2^-34) |a b|, 1.001 units; the K / 16
accumulations of h*h round to 2 units each (a matrix instruction: at most an ulp of the partial sum, at
most 1.01 S), the 5 K / 16 of the smaller products to 2^-7 of that; adding the two sums and the bias,
one each. |y - ref| <= (K / 8 + 5 K / 1024 + 3.1) 1.01 units, below K / 7 + 4.
"""
import numpy as np
import pytest

from metalaudio_amd import nn

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    return nn.AudioDevice(0)


def run(dev, x, w, b, act="none"):
    layer = nn.Linear(dev, w.shape[1], w.shape[0], activation=act)
    layer.load_weights(w, b)
    s = nn.Stream(dev)
    out = layer(nn.Tensor.from_numpy(dev, x), s)
    s.sync(20000)
    return out.to_numpy()


# rows x outputs x depth: one row, edges of the 64- and 128-row tiles, outputs that are no multiple
# of 4 (unaligned epilogue), one stage, odd and even stage counts, enough tiles for each tile shape
SHAPES = [(1, 4, 32), (63, 33, 64), (65, 132, 96), (129, 64, 160), (67, 1536, 384),
          (1000, 130, 512), (5376, 384, 224), (10752, 384, 96), (4100, 1030, 64)]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_parts_gemm_error_bound(dev, M, N, K):
    print(f"split gemm {M}x{N}x{K}", flush=True)
    r = np.random.default_rng(M + N + K)
    x = r.standard_normal((M, K)).astype(np.float32)
    w = (r.standard_normal((N, K)) * 0.05).astype(np.float32)
    b = r.standard_normal(N).astype(np.float32)
    y = run(dev, x, w, b).astype(np.float64)
    ref = x.astype(np.float64) @ w.astype(np.float64).T + b
    S = np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T + np.abs(b)
    assert np.all(np.abs(y - ref) <= (K / 7 + 4) * 2.0 ** -24 * S)


# two teams of waves with half of K each: 4 + 4 stages (the fewest), 6 + 6, 24 + 24; one output, tile edges
TEAMS = [(1, 1, 256), (64, 64, 256), (65, 33, 512), (67, 1536, 384), (130, 100, 1536), (1000, 384, 384)]


@pytest.mark.parametrize("M,N,K", TEAMS)
def test_two_teams_error_bound(dev, M, N, K):
    """As above: half the chain each, and one more addition."""
    test_parts_gemm_error_bound(dev, M, N, K)


def test_two_teams_not_finite(dev):
    """An infinity in one team's half of K, opposite ones in both, NaN: as fp32 products give them."""
    print("split gemm teams not finite", flush=True)
    r = np.random.default_rng(16)
    M, N, K = 70, 40, 256
    x = r.standard_normal((M, K)).astype(np.float32)
    w = r.integers(1, 4, (N, K)).astype(np.float32)
    x[3, 5], x[10, 250], x[40, 128] = np.inf, -np.inf, np.nan
    x[66, 7], x[66, 200] = np.inf, -np.inf
    y = run(dev, x, w, np.zeros(N, np.float32))
    assert np.all(y[3] == np.inf) and np.all(y[10] == -np.inf)
    assert np.all(np.isnan(y[[40, 66]]))
    fine = [i for i in range(M) if i not in (3, 10, 40, 66)]
    ref = x[fine].astype(np.float64) @ w.astype(np.float64).T
    S = np.abs(x[fine]).astype(np.float64) @ w.astype(np.float64).T
    assert np.all(np.abs(y[fine] - ref) <= (K + 3) * 2.0 ** -24 * S)


def test_parts_keep_every_bit(dev):
    """Against unit weights each output is one operand: its three parts must sum to it exactly, small
    elements beside large ones included (here 2^-90 .. 2^90 in one row)."""
    print("split gemm exact parts", flush=True)
    r = np.random.default_rng(5)
    K = 64
    x = np.ldexp(r.standard_normal((70, K)), r.integers(-90, 91, (70, K))).astype(np.float32)
    y = run(dev, x, np.eye(K, dtype=np.float32), np.zeros(K, np.float32))
    np.testing.assert_array_equal(y, x)


def test_not_finite_comes_out_as_from_fp32(dev):
    """Infinities, NaN, values that bf16 would round to infinity and sums that overflow give what fp32
    products give; rows without them are untouched."""
    print("split gemm not finite", flush=True)
    r = np.random.default_rng(6)
    M, N, K = 130, 68, 64
    x = r.standard_normal((M, K)).astype(np.float32)
    w = r.integers(1, 4, (N, K)).astype(np.float32)  # positive, few bits: no inf - inf, no 0 * inf
    x[3, 5], x[70, 60], x[71, 2] = np.inf, -np.inf, np.nan
    x[9] = 0.0
    x[9, 7] = np.float32(3.4e38)   # rounds to infinity in bf16
    x[100] = 3e38                  # the sum overflows
    w[:, 7] = 1.0
    y = run(dev, x, w, np.zeros(N, np.float32))
    assert np.all(y[3] == np.inf) and np.all(y[70] == -np.inf) and np.all(np.isnan(y[71]))
    assert np.all(y[9] == np.float32(3.4e38)) and np.all(y[100] == np.inf)
    fine = [i for i in range(M) if i not in (3, 70, 71, 9, 100)]
    ref = x[fine].astype(np.float64) @ w.astype(np.float64).T
    S = np.abs(x[fine]).astype(np.float64) @ w.astype(np.float64).T
    # the fp32 products of a recomputed block round once per k
    assert np.all(np.abs(y[fine] - ref) <= (K + 3) * 2.0 ** -24 * S)


def test_reloaded_weights_take_effect(dev):
    print("split gemm reload", flush=True)
    layer = nn.Linear(dev, 64, 64, use_bias=False)
    x = nn.Tensor.from_numpy(dev, np.eye(64, dtype=np.float32))
    s = nn.Stream(dev)
    for k in (1.0, 2.5):
        layer.load_weights(np.full((64, 64), k, np.float32))
        out = layer(x, s)
        s.sync(20000)
        assert np.all(out.to_numpy() == np.float32(k))


def test_folded_weight_that_overflows(dev):
    """Loaded weights are finite, but one times its LayerNorm's scale need not be: an infinite product of the
    fold stays one through the three parts, and what it reaches is infinite, not NaN."""
    print("split gemm infinite folded weight", flush=True)
    r = np.random.default_rng(12)
    E, F, S, k, h = 64, 96, 70, 5, 40
    t = nn.TransformerLayer(dev, E, 1, F)
    w1 = r.standard_normal((F, E)).astype(np.float32)
    w1[:, k] = 0
    w1[h, k] = 1e25
    scale = np.ones(E, np.float32)
    scale[k] = 1e25
    w2 = r.standard_normal((E, F)).astype(np.float32)
    w2[:, h] = 1
    t.load_state({"attn.out_proj.weight": np.zeros((E, E), np.float32), "norm2.weight": scale,
                  "linear1.weight": w1, "linear2.weight": w2})
    x = -r.uniform(1, 2, (S, E)).astype(np.float32)
    x[:, k] = r.uniform(1, 2, S)
    s = nn.Stream(dev)
    out = t(nn.Tensor.from_numpy(dev, x), s)
    s.sync(20000)
    y = out.to_numpy()
    assert np.all(y == np.inf)


def test_one_product_per_output(dev):
    """Rows with a single element, where nothing hides in the accumulations' allowance: the dropped products
    are 1.001 units (up to 2^-22.5 were one operand truncated), the last sum is one, and the sums of the
    small products, 2^-7 of the output, round to 2 * 2^-7 each."""
    print("split gemm one product", flush=True)
    r = np.random.default_rng(14)
    M, N, K = 2048, 512, 32
    x = np.zeros((M, K), np.float32)
    x[np.arange(M), np.arange(M) % K] = np.exp2(r.uniform(0, 1, M))
    w = (np.exp2(r.uniform(0, 1, (N, K))) * r.choice([-1, 1], (N, K))).astype(np.float32)
    y = run(dev, x, w, np.zeros(N, np.float32)).astype(np.float64)
    ref = x.astype(np.float64) @ w.astype(np.float64).T
    assert np.all(np.abs(y - ref) <= 2.1 * 2.0 ** -24 * np.abs(ref))


@pytest.mark.parametrize("K", [64, 256])  # one team of waves, two
def test_tiny_operands(dev, K):
    """Rows of values whose low parts lie below bf16's range keep fp32's accuracy beside ordinary rows;
    blocks that are computed again in fp32 round once per k (and to 2^-149)."""
    print(f"split gemm tiny operands K{K}", flush=True)
    r = np.random.default_rng(17 + K)
    M, N = 130, 68
    x = r.standard_normal((M, K)).astype(np.float32)
    x[5] = np.ldexp(x[5], -124)
    x[64:80] = np.ldexp(x[64:80], -118)
    x[90] = 0
    w = (16 * r.standard_normal((N, K))).astype(np.float32)
    y = run(dev, x, w, np.zeros(N, np.float32)).astype(np.float64)
    ref = x.astype(np.float64) @ w.astype(np.float64).T
    S = np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T
    assert np.all(np.abs(y - ref) <= (K + 3) * (2.0 ** -24 * S + 2.0 ** -149))


def test_first_pass_folds_in_one_launch(dev):
    """A transformer layer's first pass writes each folded weight split, with no second launch over a plain
    copy; reloaded weights are folded again, once."""
    print("split gemm first pass", flush=True)
    t = nn.TransformerLayer(dev, 64, 1, 96)
    x = nn.Tensor.from_numpy(dev, np.random.default_rng(2).standard_normal((70, 64)).astype(np.float32))
    s = nn.Stream(dev)
    for folds in (2, 0, 1):  # new, again, one weight reloaded
        if folds == 1:
            t.load_state({"linear1.weight": np.ones((96, 64), np.float32)})
        dev.set_kernel_timing(True)
        dev.reset_kernel_timing()
        t(x, s)
        s.sync(20000)
        counts = dev.kernel_timing("ln_fold")[0], dev.kernel_timing("x3_planes")[0]
        dev.set_kernel_timing(False)
        assert counts == (folds, 0)
