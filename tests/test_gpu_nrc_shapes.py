"""The cache's kernels where their shapes end: inference by single blocks of
16 samples and by staged tiles of 64 (from 131,073 samples on), training over
ragged tiles and over more tiles than workgroups, and directions far from
unit length or along an axis.  A sample's arithmetic is the same in both
inference kernels, so their outputs are compared bit for bit, and the
hash-grid inputs with binary32 sums in the definition's order; the oracle
comparisons and their bounds are those of the cache's other tests."""
import numpy as np
import pytest

from oracle import nrc as N

from test_gpu_nrc import features, test_gradient_matches_oracle as gradient_matches_oracle, weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [131073, 131072 + 64 * 256 * 16 + 17])
def test_staged_inference_equals_single_blocks(engine, n):
    engine.nrc_set_weights(weights(11))
    f = features(n, 13)
    staged = engine.nrc_infer(f)
    for lo, count in ((0, 1), (0, 15), (0, 16), (1, 17), (n - 131072, 131072)):
        one = engine.nrc_infer(np.ascontiguousarray(f[lo:lo + count]))
        assert np.array_equal(one.view(np.uint32), staged[lo:lo + count].view(np.uint32)), (lo, count)


@pytest.mark.parametrize("n", [4099, 131073])
def test_grid_inputs_round_as_defined(engine, n):
    """A network of unit matrices hands its bf16 inputs through, three at a
    time: the trilinear sums, one rounding per product and per addition."""
    w = np.zeros(N.N_PARAMS, np.float32)
    w[:16384] = np.tile(np.eye(64, dtype=np.float32).ravel(), 4)
    w[N.N_MLP:] = np.random.default_rng(15).random(N.N_TABLE)
    f = features(n, 16)
    tab = w[N.N_MLP:].reshape(N.LEVELS, N.ROWS, N.LFEAT)
    want = np.zeros((n, 2 * N.LEVELS), np.float32)
    for level in range(N.LEVELS):
        rows, wts = N.grid_corners(level, f[:, :3])
        for k in range(8):
            want[:, 2 * level:2 * level + 2] += wts[:, k:k + 1].astype(np.float32) * tab[level][rows[:, k]]
    want = N.bf16(want).astype(np.float32)
    for first in range(0, 16, 3):
        dims = range(first, min(first + 3, 16))
        w[16384:N.N_MLP] = 0
        for c, d in enumerate(dims):
            w[16384 + 64 * c + d] = 1
        engine.nrc_set_weights(w)
        got = engine.nrc_infer(f)[:, :len(dims)]
        assert np.array_equal(got.view(np.uint32), np.ascontiguousarray(want[:, dims]).view(np.uint32)), first


def test_directions_along_the_axes(engine):
    """Octahedral coordinates of 0, 1/2 and 1, where half of a one-blob
    Gaussian is cut off."""
    w = weights(11)
    engine.nrc_set_weights(w)
    f = features(600, 17)
    f[:, 3:6] = np.concatenate([np.eye(3), -np.eye(3)])[np.arange(600) % 6]
    got = engine.nrc_infer(f).astype(np.float64)
    ref, _ = N.forward(w, f)
    err = np.abs(got - ref) / np.sqrt(np.mean(ref ** 2))
    assert np.median(err) < 2e-3 and np.quantile(err, 0.99) < 2e-2, (np.median(err), np.quantile(err, 0.99))


@pytest.mark.parametrize("scale", [2.0 ** -60, 2.0 ** -30, 2.0 ** 30, 2.0 ** 60, 0.0])
def test_direction_length_does_not_matter(engine, scale):
    w = weights(11)
    engine.nrc_set_weights(w)
    f = features(1000, 14)
    f[:, 3:6] *= np.float32(scale)
    got = engine.nrc_infer(f).astype(np.float64)
    ref, _ = N.forward(w, f)
    err = np.abs(got - ref) / np.sqrt(np.mean(ref ** 2))
    assert np.median(err) < 2e-3 and np.quantile(err, 0.99) < 2e-2, (np.median(err), np.quantile(err, 0.99))


@pytest.mark.parametrize("n", [1, 65, 4097, 512 * 64 + 1])
def test_gradient_of_ragged_tiles(engine, n):
    gradient_matches_oracle(engine, n)
