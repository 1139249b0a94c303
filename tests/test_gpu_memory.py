"""Large results copied to the host in pieces by several threads, and device blocks that are
used again from call to call (ytm_memory.hip), against numpy."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ytm_amd = pytest.importorskip("ytm_amd")
from ytm_amd import Binarizer, MultiClassTM  # noqa: E402

MB = 1 << 20


def binned(n, seed):
    """n values through a one-level binarizer, and what numpy gives: 4 n bytes of output."""
    x = np.random.default_rng(seed).integers(0, 256, (1, n)).astype(np.uint8)
    b = Binarizer(1).fit  # thresholds given: no percentile pass
    obj = b.__self__
    b(x, thresholds=[100.0], min_val=0, max_val=255)
    return obj.transform(x).reshape(-1), (x.reshape(-1) >= 100).astype(np.uint32)


@pytest.mark.parametrize("n", [MB - 1, MB, MB + 1, 2 * MB - 64, 2 * MB + 3, 9 * MB + 77, 1, 20 * MB])
def test_copies_of_every_length(n):
    got, want = binned(n, n)
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("n", [104857, 104858, 300001])
def test_class_sums_of_every_length(n):
    """Class sums below 4 MiB come back through one pinned buffer, from there on in pieces."""
    tm = MultiClassTM(40, 50, 5.0, (100, 1, 1), 10, seed=3)
    rng = np.random.default_rng(n)
    L = tm.number_of_literals
    ta = np.where(rng.random((40, L)) < 3 / L, 200, 60).astype(np.uint32)
    w = rng.integers(-50, 51, (40, 10)).astype(np.float32)
    tm.load_state_dict({"state": {"ta_state": ta, "clause_weights": w, "min_y": None, "max_y": None,
                                  "patch_weights": np.zeros((40, 1), np.int32)}})
    bits = rng.integers(0, 2, (n, 100), dtype=np.uint8)
    lits = np.concatenate([bits, 1 - bits], 1).astype(np.float32)
    miss = (1 - lits) @ (ta > 128).T.astype(np.float32)
    fire = (miss == 0) & (ta > 128).any(1)
    np.testing.assert_array_equal(tm.score(tm.encode(bits.astype(np.uint32)), is_X_encoded=True),
                                  (fire.astype(np.float64) @ w).astype(np.float32))


def test_threads_and_reused_blocks():
    """Calls of several threads at once, each with its own results, over blocks that earlier
    calls of other sizes leave behind."""
    def one(i):
        got, want = binned((1 + i % 5) * MB + i, i)
        return np.array_equal(got, want)

    with ThreadPoolExecutor(4) as pool:
        assert all(pool.map(one, range(16)))


def test_state_after_models_of_other_sizes():
    """A new model's state does not depend on what an earlier one left in its blocks."""
    def states(seed):
        tm = MultiClassTM(300, 15, 3.9, (1200, 1, 1), 3, seed=seed)
        X = np.random.default_rng(1).integers(0, 2, (400, 1200)).astype(np.uint32)
        enc, y = tm.encode(X), np.arange(400, dtype=np.uint32) % 3
        tm.fit(enc, y, is_X_encoded=True)
        out = tm.get_ta_state(), tm.get_weights(), tm.score(enc, is_X_encoded=True)
        tm.release()
        return out

    first = states(5)
    states(6)
    for a, b in zip(first, states(5)):
        np.testing.assert_array_equal(a, b)
