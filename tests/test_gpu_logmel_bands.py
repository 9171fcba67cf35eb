"""GPU parity of the log-mel transform at band counts off its usual ones, and for
samples whose power is not finite."""
import numpy as np
import pytest

from vokra_amd import hip

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = hip.HipContext(0)
    yield c
    c.close()


@pytest.mark.parametrize("n_mels", [1, 7, 201, 1024])
def test_log_mel_band_counts(ctx, oracle, n_mels):
    """Wide bands, and so many that some hold no bin (their floor)."""
    g = np.random.default_rng(n_mels)
    x = (0.1 * g.standard_normal(50000)).astype(np.float32)
    assert np.abs(ctx.log_mel(x, n_mels) - oracle.log_mel(x, n_mels)).max() <= 1e-4


@pytest.mark.parametrize("n_mels", [1, 80, 128])
@pytest.mark.parametrize("sample", [1e25, 3e38, np.inf, -np.inf, np.nan])
def test_log_mel_wild_samples(ctx, oracle, n_mels, sample):
    """A sample whose frames' powers overflow or are not numbers: the reference sums
    every bin of a band, so those frames fall to the floor and the rest of the clip
    keeps its own maximum."""
    g = np.random.default_rng(n_mels)
    x = (0.1 * g.standard_normal(50000)).astype(np.float32)
    x[20011] = sample
    got, want = ctx.log_mel(x, n_mels), oracle.log_mel(x, n_mels)
    assert np.isfinite(want).all() and np.abs(got - want).max() <= 1e-4
