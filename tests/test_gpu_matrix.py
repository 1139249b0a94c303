"""Scoring on the matrix cores (ytm_matrix.hip) against the oracle: every number of literal
steps and of patch tiles per wave, the edges of the tiles of 32 patches, clauses and samples,
samples whose negated literals are not complements, and weights of one to five digits.  Class
sums are whole numbers: compared bit for bit."""
import numpy as np
import pytest

from oracle import oracle as orc

pytestmark = pytest.mark.gpu

ytm_amd = pytest.importorskip("ytm_amd")
from ytm_amd import MultiClassTM  # noqa: E402


def pair(clauses, dim, classes, rng, weight=50, **kw):
    """The GPU model and the oracle with one random state: clauses of no, few and many literals,
    some with a literal and its negation."""
    tm = MultiClassTM(clauses, 50, 5.0, dim, classes, seed=7, **kw)
    ref = orc.OracleTM(clauses, 50, 5.0, dim, classes, seed=7, **kw)
    C, L = tm.number_of_clauses, tm.number_of_literals
    p = np.choose(rng.integers(0, 10, C), [0.0] + [2.0 / L] * 6 + [5.0 / L] * 2 + [0.3])
    inc = rng.random((C, L)) < p[:, None]
    ta = np.where(inc, 200, 60).astype(np.uint32)
    w = rng.integers(-weight, weight + 1, (C, classes)).astype(np.float32)
    tm.load_state_dict({"state": {"ta_state": ta, "clause_weights": w, "min_y": None, "max_y": None,
                                  "patch_weights": np.zeros((C, tm.number_of_patches), np.int32)}})
    ref.ta[...] = ta.reshape(ref.ta.shape)
    ref.w[...] = w.reshape(ref.w.shape)
    return tm, ref


def check(tm, ref, enc, path=5):
    data = tm._device_data(enc)
    want = ref.score(enc)
    np.testing.assert_array_equal(tm.score_device(data), want)
    np.testing.assert_array_equal(tm.score_device(data), want)  # the kept operands
    assert tm.stats()["score_path"] == path
    return want


def image(rng, n, dim):
    return (rng.random((n, dim[0] * dim[1] * dim[2])) < 0.6).astype(np.uint32)


@pytest.mark.parametrize("dim,patch,clauses,n", [
    ((3, 2, 1), (2, 2), 1, 1),         # 2 patches, 1 step, one clause and sample
    ((7, 6, 1), (2, 3), 33, 70),       # 24 patches: samples share a wave
    ((9, 7, 1), (2, 3), 64, 33),       # 40 patches: tiles of one sample in two waves
    ((6, 9, 9), (3, 2), 31, 5),        # 32 patches: a whole tile
    ((13, 12, 10), (3, 4), 300, 9),    # 2 literal steps
    ((20, 20, 1), (10, 12), 290, 6),   # 99 patches
    ((28, 28, 1), (10, 10), 500, 7),   # 361 patches, 3 steps
    ((12, 12, 24), (3, 3), 270, 40),   # 4 steps
    ((32, 32, 24), (3, 3), 2600, 3),   # 900 patches, 5 steps: one sample fills the waves
    ((40, 33, 24), (3, 3), 100, 2),    # 1178 patches: a sample in two rounds
    ((10, 10, 33), (3, 3), 130, 21),   # 6 steps
    ((9, 8, 47), (3, 3), 65, 20),      # 7 steps
    ((9, 8, 54), (3, 3), 65, 20),      # 8 steps
    ((9, 8, 62), (3, 3), 65, 20),      # 9 steps
])
def test_steps_and_tiles(dim, patch, clauses, n):
    rng = np.random.default_rng(3)
    tm, ref = pair(clauses, dim, 3, rng, patch_dim=patch)
    want = check(tm, ref, tm.encode(image(rng, n, dim)))
    assert clauses < 30 or np.unique(want).size > 1


@pytest.mark.parametrize("dim,patch,negated", [
    ((12, 12, 2), (4, 4), False),    # no negations: all literals, 1 step
    ((28, 28, 1), (10, 10), True),   # 272 literals without complements: 5 steps
    ((14, 14, 24), (3, 3), True),    # 476: 8 steps
    ((9, 8, 62), (3, 3), True),      # beyond 9 steps: the literal lists
])
def test_all_literals(dim, patch, negated):
    """Samples whose negated literals are not the complements of the positive ones (encoded
    elsewhere), beside the same model's scores of framework-encoded samples."""
    rng = np.random.default_rng(4)
    tm, ref = pair(200, dim, 4, rng, patch_dim=patch, append_negated=negated)
    enc = tm.encode(image(rng, 12, dim))
    odd = enc & rng.integers(0, 2**32, enc.shape, dtype=np.uint32) | enc & rng.integers(0, 2**32, enc.shape,
                                                                                       dtype=np.uint32)
    check(tm, ref, enc)
    check(tm, ref, odd, path=5 if tm.number_of_literals <= 9 * 64 else 4)
    check(tm, ref, enc)


@pytest.mark.parametrize("classes,weight", [(2, 1), (10, 127), (10, 128), (17, 32639), (11, 40000), (33, 8355711),
                                            (7, 9000000), (40, 2**30), (5, 2**31 - 256), (70, 300)])
def test_weight_digits(classes, weight):
    """Weights of every number of base-256 digits, at their largest, over one and several column
    groups; the sums of few firing clauses stay exact in float32 or round once, as the
    oracle's do."""
    rng = np.random.default_rng(5)
    dim, patch = (9, 9, 2), (4, 4)
    tm, ref = pair(150, dim, classes, rng, weight=weight, patch_dim=patch)
    w = tm.get_weights()
    w[::3] = np.where(w[::3] < 0, -weight, weight)
    state = tm.get_state_dict()
    state["clause_weights"] = w.reshape(-1)
    tm.load_state_dict({"state": state})
    ref.w[...] = w.reshape(ref.w.shape)
    check(tm, ref, tm.encode(image(rng, 37, dim)))


def test_operands_follow_the_model():
    """Kept operands are made again after a fit, new weights and new states."""
    rng = np.random.default_rng(6)
    dim = (10, 10, 1)
    tm, ref = pair(60, dim, 3, rng, patch_dim=(4, 4))
    X = image(rng, 50, dim)
    enc, y = tm.encode(X), rng.integers(0, 3, 50).astype(np.uint32)
    check(tm, ref, enc)
    ref.load_state(ref.ta, ref.w, np.zeros((60, tm.number_of_patches), np.int32), 0)
    tm.fit(enc, y, is_X_encoded=True)
    ref.fit_encoded(enc, ref.encode_y_multiclass(y))
    check(tm, ref, enc)
    state = tm.get_state_dict()
    state["clause_weights"] = -state["clause_weights"]
    tm.load_state_dict({"state": state})
    ref.w[...] = -ref.w
    check(tm, ref, enc)


@pytest.mark.parametrize("bits,clauses,n", [
    (600, 70, 1),      # one sample
    (33, 40, 31),      # 2 steps, a tile less one
    (32, 33, 33),      # 1 step made 2, a tile and one
    (200, 2000, 65),   # few samples: a block per tile
    (784, 300, 7000),  # many samples: 256 by 256 tiles, a partial one in each direction
    (100, 8200, 257),  # 257 clause tiles
    (2111, 257, 8193),
    (513, 40, 40001),  # one clause tile beyond the first of a block
])
def test_one_patch(bits, clauses, n):
    rng = np.random.default_rng(8)
    tm, ref = pair(clauses, (bits, 1, 1), 5, rng)
    enc = tm.encode(image(rng, n, (bits, 1, 1)))
    want = check(tm, ref, enc)
    assert np.unique(want).size > 1
    odd = enc & rng.integers(0, 2**32, enc.shape, dtype=np.uint32)  # negations are not complements
    check(tm, ref, odd)
    check(tm, ref, enc)


@pytest.mark.parametrize("dim,patch,clauses,n,room,odd", [
    ((784, 1, 1), None, 2000, 2500, 1056 * 1088 + 256, 0),     # 1056 rows a pass, the last of 388 by single tiles
    ((784, 1, 1), None, 2000, 2500, 1056 * 1088 + 256, 1500),  # one sample of the second pass without complements
    ((784, 1, 1), None, 2000, 2500, 1056 * 1088 + 256, 2400),  # one of the last
    ((784, 1, 1), None, 60, 70, 0, 0),                         # 32 a pass: the first makes the operands
    ((9, 8, 2), (3, 3), 60, 100, 32 * 16 + 256, 0),            # several patches, a last pass of 4
])
def test_several_passes(monkeypatch, dim, patch, clauses, n, room, odd):
    """Rows of more samples than a pass has room for."""
    monkeypatch.setenv("YTM_SCORE_PASS", str(room))
    rng = np.random.default_rng(10)
    tm, ref = pair(clauses, dim, 5, rng, **({"patch_dim": patch} if patch else {}))
    enc = tm.encode(image(rng, n, dim))
    if odd:
        enc = enc.copy()
        enc[odd] &= rng.integers(0, 2**32, enc[odd].shape, dtype=np.uint32)
    want = check(tm, ref, enc)
    assert np.unique(want).size > 1


@pytest.mark.parametrize("bits,clauses,n,negated", [(90, 64, 300, False), (1000, 33, 70000, False),
                                                    (10000, 40, 7000, True), (10000, 7000, 300, True)])
def test_one_patch_without_allocation(bits, clauses, n, negated):
    """The allocation-free scorer: operands and samples in the scratch, in one pass and several,
    and the literal lists where the operands exceed it (7000 clauses of 20000 literals)."""
    from test_zz_no_alloc import score_both

    rng = np.random.default_rng(9)
    tm, ref = pair(clauses, (bits, 1, 1), 4, rng, append_negated=negated)
    enc = tm.encode(image(rng, n, (bits, 1, 1)))
    got, noalloc = score_both(tm, tm._device_data(enc), 4)
    assert tm.stats()["score_path"] == (3 if clauses == 7000 else 5)
    np.testing.assert_array_equal(got, noalloc)
    np.testing.assert_array_equal(got[:200], ref.score(enc[:200]))


def test_literal_lists_of_wide_patches(monkeypatch):
    """Patches of more literals than the product's registers hold keep the literal-list scorer:
    blocks over every clause of a sample and over chunks of 4096 clauses."""
    rng = np.random.default_rng(7)
    dim = (16, 16, 64)
    tm, ref = pair(4200, dim, 3, rng, patch_dim=(3, 3))
    enc = tm.encode(image(rng, 5, dim))
    for least in ("1", "1000000"):
        monkeypatch.setenv("YTM_SCORE_WHOLE_MIN", least)
        check(tm, ref, enc, path=4)


@pytest.mark.parametrize("dim,clauses,wgs,opts", [
    ((33, 3, 1), 33, "2", {}),                            # 31 patches, 1 step, 16 or 17 clauses a workgroup
    ((34, 3, 4), 64, "2", {}),                            # 32 patches, 2 steps, 32 clauses
    ((35, 3, 11), 66, "2", dict(append_negated=False)),   # 33 patches, binary literals, 33 clauses
    ((34, 34, 20), 97, "1", {}),                          # 1024 patches, 4 steps, one workgroup of 97
    ((47, 47, 1), 130, "1", {}),                          # 2025 patches: 64 words of them
    ((5, 4, 53), 96, "1", {}),                            # 6 patches, 8 steps
])
@pytest.mark.parametrize("env", [{}, {"YTM_TRAIN_THREADS": "256"}, {"YTM_JIT": "0"}])
def test_training_on_several_patches(monkeypatch, dim, clauses, wgs, opts, env):
    """The training kernel of clause state in global memory with its evaluation as a product:
    edges of the tiles of patches and clauses, of the literal steps and of the workgroup's waves,
    dropped clauses, and samples whose negated literals are not complements (the list walks),
    against the oracle, bit for bit."""
    monkeypatch.setenv("YTM_TRAIN_GLOBAL", "1")
    monkeypatch.setenv("YTM_TRAIN_MMA", "1")
    monkeypatch.setenv("YTM_TRAIN_WGS", wgs)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    print(f"[training] {dim} {clauses} {wgs} {opts} {env}", flush=True)
    rng = np.random.default_rng(dim[2])
    kw = dict(patch_dim=(3, 3), **opts)
    tm, ref = pair(clauses, dim, 3, rng, **kw)
    n = 6
    X = (rng.random((n, int(np.prod(dim)))) < 0.4).astype(np.uint32)
    y = rng.integers(0, 3, n)
    enc = tm.encode(X)
    odd = enc.copy()
    odd[:, 0, 0] ^= np.uint32(4)
    encY = ref.encode_y_multiclass(y)
    drops = np.random.default_rng(7)  # the model's numpy generator
    for data, p, inject in ((enc, 0.0, False), (enc, 0.3, False), (odd, 0.0, False), (enc, 0.0, True)):
        kw, kr = {}, {}
        if inject:
            kw["random_stream"] = kr["inject"] = rng.random(tm.random_stream_size(n)).astype(np.float32)
        if p:
            kw["clause_drop_p"] = p
            kr["drop"] = (drops.random(ref.C) <= p).astype(np.uint32)
        tm.fit(data, y, is_X_encoded=True, **kw)
        upd = ref.fit_encoded(data, encY, **kr)
        st = tm.stats()
        assert st["train_kind"] == 2 and st["last_fit_updates"] == upd
        assert st["train_product"] == (data is enc or not tm.append_negated)
        np.testing.assert_array_equal(tm.get_ta_state().reshape(ref.ta.shape), ref.ta)
        np.testing.assert_array_equal(tm.get_weights().reshape(ref.w.shape), ref.w)
        np.testing.assert_array_equal(tm.get_patch_weights().reshape(ref.pw.shape), ref.pw)


@pytest.mark.parametrize("clauses,wgs,jit,product", [(21, "1", "1", 0), (22, "1", "1", 1), (43, "2", "1", 1), (42, "2", "1", 0),
                                                     (99, "1", "0", 0), (100, "1", "0", 1)])
def test_training_product_from_enough_clauses(monkeypatch, clauses, wgs, jit, product):
    """Fewer than 22 clauses a workgroup (100 with the built-in kernel) train on literal lists."""
    monkeypatch.setenv("YTM_TRAIN_GLOBAL", "1")
    monkeypatch.setenv("YTM_TRAIN_WGS", wgs)
    monkeypatch.setenv("YTM_JIT", jit)
    rng = np.random.default_rng(2)
    tm, ref = pair(clauses, (9, 8, 2), 3, rng, patch_dim=(3, 3))
    y = rng.integers(0, 3, 8)
    enc = tm.encode(image(rng, 8, (9, 8, 2)))
    tm.fit(enc, y, is_X_encoded=True)
    ref.fit_encoded(enc, ref.encode_y_multiclass(y))
    assert tm.stats()["train_kind"] == 2 and tm.stats()["train_product"] == product
    np.testing.assert_array_equal(tm.get_ta_state().reshape(ref.ta.shape), ref.ta)
    np.testing.assert_array_equal(tm.get_weights().reshape(ref.w.shape), ref.w)


@pytest.mark.parametrize("clauses,wgs", [(130, "1"), (160, "2")])
def test_first_sample_of_a_launch_counts_includes(monkeypatch, clauses, wgs):
    """Injected fits of one sample each, so that every sample is the first of its launch: its
    include counts, on both sides of max_included_literals over more clauses than a workgroup
    has waves, decide between Type Ia and Ib feedback."""
    monkeypatch.setenv("YTM_TRAIN_GLOBAL", "1")
    monkeypatch.setenv("YTM_TRAIN_WGS", wgs)
    print(f"[first sample] {clauses} {wgs}", flush=True)
    rng = np.random.default_rng(12)
    dim = (12, 12, 2)
    tm, ref = pair(clauses, dim, 3, rng, patch_dim=(3, 3), max_included_literals=3)
    counts = (ref.ta > 128).sum(-1)
    assert (counts > 3).sum() > 20 and ((counts > 0) & (counts <= 3)).sum() > 20
    X = image(rng, 8, dim)
    y = rng.integers(0, 3, 8)
    enc, encY = tm.encode(X), ref.encode_y_multiclass(y)
    for e in range(8):
        draws = rng.random(tm.random_stream_size(1)).astype(np.float32)
        tm.fit(enc[e:e + 1], y[e:e + 1], is_X_encoded=True, random_stream=draws)
        upd = ref.fit_encoded(enc[e:e + 1], encY[e:e + 1], inject=draws)
        st = tm.stats()
        assert st["train_kind"] == 2 and st["train_product"] == 1 and st["last_fit_updates"] == upd
        np.testing.assert_array_equal(tm.get_ta_state().reshape(ref.ta.shape), ref.ta)
        np.testing.assert_array_equal(tm.get_weights().reshape(ref.w.shape), ref.w)
        np.testing.assert_array_equal(tm.get_patch_weights().reshape(ref.pw.shape), ref.pw)
