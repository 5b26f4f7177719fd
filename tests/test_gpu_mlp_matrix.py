"""The pruner network's matrix-core kernels against the FP64 oracle at the
edges of their 32-sample tiles and launches, and on values a split into bf16
parts could lose: tiny, huge and infinite inputs, weights that are not finite."""

import numpy as np
import pytest

from gpu_inscy_amd import _lib, pruner
from oracle import oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    _lib.lib()


def weights(seed):
    rng = np.random.default_rng(seed)
    return pruner.bf16_round(pruner.init_params(seed) + rng.normal(0, 0.01, _lib.MLP_PARAMS).astype(np.float32))


# one sample, a tile, one more, a block of four tiles, one more, more than the
# 512 blocks hold at once; sums of at most 129 float32 terms per unit
@pytest.mark.parametrize("N", [1, 32, 33, 128, 129, 65537])
def test_scores_at_tile_edges(N):
    print("scores", N, flush=True)
    P = weights(5)
    X = np.random.default_rng(N).random((N, _lib.MLP_INPUTS), dtype=np.float32)
    prob = pruner.Trainer(P).forward(X).cpu().numpy().astype(np.float64)
    np.testing.assert_allclose(prob, 1.0 / (1.0 + np.exp(-O.mlp_forward(P, X))), rtol=0, atol=2e-5)


@pytest.mark.parametrize("N,nblocks", [(1, 1), (32, 1), (33, 2), (65, 2), (4096, 128), (4129, 128)])
def test_gradient_at_tile_edges(N, nblocks):
    print("gradient", N, nblocks, flush=True)
    P = weights(6)
    rng = np.random.default_rng(N)
    X = rng.random((N, _lib.MLP_INPUTS), dtype=np.float32)
    Y = (rng.random(N) < 0.3).astype(np.float32)
    W = rng.uniform(0.5, 2.0, N).astype(np.float32)
    dev = lambda a: torch.from_numpy(a).cuda()
    g = pruner.Trainer(P, nblocks=nblocks).gradient(dev(X), dev(Y), dev(W), 1.0 / N).cpu().numpy().astype(np.float64)
    ref, loss = O.mlp_grad(P, X, Y, W, 1.0 / N)
    assert abs(g[-1] - loss) <= 1e-5 * max(1.0, abs(loss))
    assert np.linalg.norm(g[:-1] - ref) <= 2e-5 * np.linalg.norm(ref)


def _fp64(P, X):
    """The network in float64 with the kernels' ReLU: max(x, 0), 0 for NaN."""
    H, I = _lib.MLP_HIDDEN, _lib.MLP_INPUTS
    cut = np.cumsum([0, H * I, H, H * H, H, H, 1])
    W1, b1, W2, b2, w3, b3 = (P.astype(np.float64)[a:b] for a, b in zip(cut[:-1], cut[1:]))
    with np.errstate(all="ignore"):
        h = np.fmax((X.astype(np.float64)[:, None, :] * W1.reshape(H, I)).sum(-1) + b1, 0.0)
        h = np.fmax((h[:, None, :] * W2.reshape(H, H)).sum(-1) + b2, 0.0)
        return 1.0 / (1.0 + np.exp(-((h * w3).sum(-1) + b3)))


# inputs of 1e-30 and 1e6 beside ordinary ones keep every bit in the split
# (1e6 scales the sums, and with them the float32 error of the logit: 64 + 128
# terms of up to 1e6 at 2^-24 each, judged where the logit is not saturated);
# an infinite input or weight behaves as in a float32 sum
@pytest.mark.parametrize("case", ["tiny", "huge", "infinite input", "nan input", "infinite weight"])
def test_scores_of_extreme_values(case):
    print("extreme", case, flush=True)
    P = weights(7)
    rng = np.random.default_rng(8)
    X = rng.random((40, _lib.MLP_INPUTS), dtype=np.float32)
    tol = 2e-5
    if case == "tiny":
        X *= rng.choice([1e-30, 1e-20, 1.0], X.shape).astype(np.float32)
    elif case == "huge":
        X[::3, 5] = 1e6
        P = P.copy()
        P[np.arange(_lib.MLP_HIDDEN) * _lib.MLP_INPUTS + 5] *= np.float32(2.0 ** -20)
    elif case == "infinite input":
        X[3, 7] = np.inf
        X[35, 0] = -np.inf
    elif case == "nan input":
        X[1::4, 2] = np.nan
    else:
        P = P.copy()
        P[5] = np.inf
    prob = pruner.Trainer(P).forward(X).cpu().numpy().astype(np.float64)
    ref = _fp64(P, X)
    assert np.array_equal(np.isnan(prob), np.isnan(ref))
    ok = ~np.isnan(ref)
    np.testing.assert_allclose(prob[ok], ref[ok], rtol=0, atol=tol)
