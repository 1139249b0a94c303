"""libytm's host code on a HIP runtime of host memory (fake_hip.c), in a child process, since the
runtime stands in for the real one.

Error exits: every HIP call that an entry point makes fails in turn.  The entry point then
reports an error, leaves no work behind on its stream (its blocks go back to the pool, which
hands them on without waiting), and loses no memory.

Memory: which device blocks are kept between calls, and when they are given back."""
import ctypes
import os
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

HERE = Path(__file__).resolve().parent
CALLS = ["hipMalloc", "hipHostMalloc", "hipMemcpyAsync", "hipMemcpy", "hipMemsetAsync", "hipStreamSynchronize",
         "hipEventRecord", "hipEventSynchronize", "hipEventElapsedTime", "hipLaunchKernel",
         "hipLaunchCooperativeKernel", "hipGetDevice", "hipGetSymbolAddress", "hipStreamCreateWithFlags",
         "hipEventCreate", "hipGetDevicePropertiesR0600", "hipOccupancyMaxActiveBlocksPerMultiprocessor"]


@pytest.fixture(scope="session")
def fake_hip(tmp_path_factory):
    out = tmp_path_factory.mktemp("fake") / "libfakehip.so"
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-pthread", "-w", "-I/opt/rocm/include", "-o", str(out),
                    str(HERE / "fake_hip.c")], check=True)
    return out


def child(fake, what):
    env = dict(os.environ, YTM_JIT="0", PYTHONPATH=os.pathsep.join([str(HERE.parent), str(HERE)]))
    r = subprocess.run([sys.executable, "-u", __file__, str(fake), what], env=env, capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, f"{what}: {r.returncode}\n{r.stdout[-3000:]}\n{r.stderr[-3000:]}"


ENTRIES = ["create", "encode", "encode_binarized", "dataset", "dataset_targets", "fit", "fit_inject", "fit_banks",
           "fit_patches", "score", "score_long", "score_again", "score_few", "score_patches", "score_lists", "noalloc",
           "noalloc_patches", "transform", "transform_patches", "get_state", "set_state", "binarize", "collapse"]


@pytest.mark.parametrize("entry", ENTRIES)
def test_every_call_failing(fake_hip, entry):
    child(fake_hip, entry)


@pytest.mark.parametrize("what", ["oldest_leave_first", "given_back_with_the_last_model", "models_in_turn", "allocations_unlocked", "staging_per_device",
                                  "new_models_first_score", "room_for_operands"])
def test_blocks(fake_hip, what):
    child(fake_hip, what)


# ------------------------------------------------------------------------------ the child
def entry(name, lib, L):
    """(prepare() -> handles, call(handles) -> status, free(handles)) of one entry point."""
    VP = ctypes.c_void_p

    def model(clauses=40, classes=3, dim=(20, 1, 1), patch=None, coalesced=1):
        patch = patch or dim[:2]
        half = patch[0] * patch[1] * dim[2] + dim[0] - patch[0] + dim[1] - patch[1]
        p = L.YtmParams(clauses=clauses, classes=classes, dim0=dim[0], dim1=dim[1], dim2=dim[2], patch_dim0=patch[0],
                        patch_dim1=patch[1], number_of_ta_states=256, max_included_literals=2 * half,
                        append_negated=1, encode_loc=1, coalesced=coalesced, negative_polarity=1, thresh=10, s_inv=0.2,
                        q_prob=1.0, seed=1)
        return p

    def create(p):
        m = VP()
        return lib.ytm_create(ctypes.byref(p), ctypes.byref(m)), m

    def rows(m, n):
        g = (ctypes.c_int64 * 4)()
        assert lib.ytm_geometry(m, g) == 0
        return np.zeros((n, g[2], g[1]), np.uint32)

    keep = []

    def with_model(p, body):
        def prepare():
            rc, m = create(p)
            assert rc == 0
            return [m]

        return prepare, lambda h: body(h[0]), lambda h: lib.ytm_destroy(h[0])

    def with_data(p, n, body, targets=False, first=lambda m, d: 0):
        def prepare():
            rc, m = create(p)
            assert rc == 0
            d, X, Y = VP(), rows(m, n), np.zeros((n, p.classes), np.int32)
            assert lib.ytm_dataset_create(m, X.ctypes.data, Y.ctypes.data if targets else None, n, ctypes.byref(d)) == 0
            assert first(m, d) == 0
            return [m, d]

        def free(h):
            lib.ytm_dataset_destroy(h[1])
            lib.ytm_destroy(h[0])

        return prepare, lambda h: body(h[0], h[1]), free

    def score(m, d, n, classes=3):
        out = np.empty((n, classes), np.float32)
        return lib.ytm_score_dataset(m, d, out.ctypes.data)

    def noalloc(m, d, n, classes=3):
        out = np.empty((n, classes), np.float32)
        keep.append(out)
        return lib.ytm_score_dataset_noalloc(m, d, out.ctypes.data)

    flat, patches = model(), model(dim=(8, 8, 1), patch=(3, 3))
    wide = model(clauses=400, dim=(800, 1, 1))
    long = model(clauses=4000, dim=(4000, 1, 1))  # the samples are looked at before their first score
    lists = model(dim=(8, 8, 80), patch=(3, 3))  # more literals than the product takes

    def created(h):
        rc, m = create(flat)
        h.append(m)
        return rc

    def dataset(m, targets):
        d, X, Y = VP(), rows(m, 9), np.zeros((9, 3), np.int32)
        rc = lib.ytm_dataset_create(m, X.ctypes.data, Y.ctypes.data if targets else None, 9, ctypes.byref(d))
        if rc == 0:
            lib.ytm_dataset_destroy(d)
        return rc

    def fit(m, p, inject=False):
        X, Y = rows(m, 5), np.zeros((5, 3), np.int32)
        g = (ctypes.c_int64 * 4)()
        lib.ytm_geometry(m, g)
        C, K = p.clauses, p.classes
        draws = np.zeros(5 * (C * g[2] + 2 * C * K + C * K * g[0]), np.float32) if inject else None
        return lib.ytm_fit(m, X.ctypes.data, Y.ctypes.data, 5, None, draws.ctypes.data if inject else None)

    def encode(m):
        X = np.zeros((1 << 16, 20), np.uint32)  # 8 MB of words: the staged copy too
        out = np.empty((1 << 16, 1, 2), np.uint32)
        keep[:] = [X, out]
        return lib.ytm_encode(m, X.ctypes.data, X.shape[0], out.ctypes.data)

    def encode_binarized(m):
        X, t, out = np.zeros((9, 10), np.uint8), np.zeros(2, np.float64), np.empty((9, 1, 2), np.uint32)
        return lib.ytm_encode_binarized(m, X.ctypes.data, 0, 9, t.ctypes.data, 0, 2, 0, 0, out.ctypes.data)

    def transform(m, clauses):
        X = rows(m, 4)
        out = np.empty((4, clauses, X.shape[1]), np.uint32)
        return lib.ytm_transform(m, X.ctypes.data, 4, 1, out.ctypes.data)

    def state(m, set_it):
        ta, w, pw = np.zeros((40, 40), np.uint32), np.zeros((40, 3), np.float32), np.zeros(40, np.int32)
        names = [(lib.ytm_set_ta_state, lib.ytm_get_ta_state), (lib.ytm_set_weights, lib.ytm_get_weights),
                 (lib.ytm_set_patch_weights, lib.ytm_get_patch_weights)]
        for (setter, getter), a in zip(names, (ta, w, pw)):
            rc = (setter if set_it else getter)(m, a.ctypes.data)
            if rc:
                return rc
        return 0

    def binarize():
        X, t, out = np.zeros(1 << 21, np.uint8), np.zeros(1, np.float64), np.empty(1 << 21, np.uint32)
        return lib.ytm_binarize(X.ctypes.data, 0, X.size, t.ctypes.data, 0, 1, 0, 0, out.ctypes.data)

    def collapse():
        B, out = np.zeros((50, 4), np.uint32), np.empty(50, np.int64)
        return lib.ytm_collapse_bins(B.ctypes.data, 50, 4, 0, 0, out.ctypes.data)

    def alone(f):
        return lambda: [], lambda h: f(), lambda h: None

    banks = model(clauses=39, coalesced=0)
    return {
        "create": lambda: (lambda: [], created, lambda h: lib.ytm_destroy(h[0])),
        "encode": lambda: with_model(flat, encode),
        "encode_binarized": lambda: with_model(flat, encode_binarized),
        "dataset": lambda: with_model(patches, lambda m: dataset(m, False)),
        "dataset_targets": lambda: with_model(patches, lambda m: dataset(m, True)),
        "fit": lambda: with_model(flat, lambda m: fit(m, flat)),
        "fit_inject": lambda: with_model(patches, lambda m: fit(m, patches, True)),
        "fit_banks": lambda: with_model(banks, lambda m: fit(m, banks)),
        "fit_patches": lambda: with_model(patches, lambda m: fit(m, patches)),
        "score": lambda: with_data(wide, 20000, lambda m, d: score(m, d, 20000)),
        "score_long": lambda: with_data(long, 10000, lambda m, d: score(m, d, 10000)),
        "score_again": lambda: with_data(wide, 3, lambda m, d: score(m, d, 3), first=lambda m, d: score(m, d, 3)),
        "score_few": lambda: with_data(wide, 3, lambda m, d: score(m, d, 3)),
        "score_patches": lambda: with_data(patches, 9, lambda m, d: score(m, d, 9)),
        "score_lists": lambda: with_data(lists, 9, lambda m, d: score(m, d, 9)),
        "noalloc": lambda: with_data(wide, 20000, lambda m, d: noalloc(m, d, 20000)),
        "noalloc_patches": lambda: with_data(patches, 9, lambda m, d: noalloc(m, d, 9)),
        "transform": lambda: with_model(wide, lambda m: transform(m, 400)),
        "transform_patches": lambda: with_model(patches, lambda m: transform(m, 40)),
        "get_state": lambda: with_model(flat, lambda m: state(m, False)),
        "set_state": lambda: with_model(flat, lambda m: state(m, True)),
        "binarize": lambda: alone(binarize),
        "collapse": lambda: alone(collapse),
    }[name]()


def binarize(lib, n):
    """A call with blocks of n and 4 n bytes."""
    X, t, out = np.zeros(n, np.uint8), np.zeros(1, np.float64), np.empty(n, np.uint32)
    assert lib.ytm_binarize(X.ctypes.data, 0, n, t.ctypes.data, 0, 1, 0, 0, out.ctypes.data) == 0


def small_model(lib, L):
    p = L.YtmParams(clauses=40, classes=3, dim0=20, dim1=1, dim2=1, patch_dim0=20, patch_dim1=1, number_of_ta_states=256,
                    max_included_literals=40, append_negated=1, encode_loc=1, coalesced=1, negative_polarity=1,
                    thresh=10, s_inv=0.2, q_prob=1.0, seed=1)
    m = ctypes.c_void_p()
    assert lib.ytm_create(ctypes.byref(p), ctypes.byref(m)) == 0
    return m


MALLOC, FREE, HOST_MALLOC, HOST_FREE, LARGE = range(5)
MB = 1 << 20


def oldest_leave_first(fake, lib, L):
    """Blocks of sizes that no call asks for any more make room for those that calls use."""
    m = small_model(lib, L)
    binarize(lib, 203 * MB)  # blocks of 204 and 812 MB, just below what is kept
    binarize(lib, 3 * MB)
    before = fake.fake_calls(MALLOC)
    for _ in range(5):
        binarize(lib, 3 * MB)
    assert fake.fake_calls(MALLOC) == before, "the blocks of the latest calls were not kept"
    assert fake.fake_live(0) < 1100 * MB, fake.fake_live(0)
    lib.ytm_destroy(m)


def given_back_with_the_last_model(fake, lib, L):
    """Without a model, 256 MiB stay idle at most; with one, more.  ytm_shutdown leaves nothing."""
    binarize(lib, 100 * MB)
    assert fake.fake_live(0) < 257 * MB, "blocks kept without a model"
    a, b = small_model(lib, L), small_model(lib, L)
    binarize(lib, 100 * MB)
    lib.ytm_destroy(a)
    assert fake.fake_live(0) > 500 * MB, "blocks given back although a model lives"
    lib.ytm_destroy(b)
    assert fake.fake_live(0) < 257 * MB, fake.fake_live(0)
    assert lib.ytm_shutdown() == 0
    assert fake.fake_live(0) == fake.fake_live(-1) == 0


def models_in_turn(fake, lib, L):
    """A model after another one has ended finds its blocks and its pinned ones there."""
    def one():
        m = small_model(lib, L)
        X, out = np.zeros((5, 1, 2), np.uint32), np.empty((5, 3), np.float32)
        assert lib.ytm_score(m, X.ctypes.data, 5, out.ctypes.data) == 0
        binarize(lib, 3 * MB)
        lib.ytm_destroy(m)
        return fake.fake_calls(MALLOC) + fake.fake_calls(HOST_MALLOC)

    first = one()
    assert one() == first


def allocations_unlocked(fake, lib, L):
    """A long hipMalloc of one thread keeps no other thread from blocks that are idle."""
    import threading
    import time

    m = small_model(lib, L)
    binarize(lib, 1000)
    fake.fake_delay_malloc(1000)
    t = threading.Thread(target=binarize, args=(lib, 5 * MB))
    t.start()
    time.sleep(0.3)
    start = time.perf_counter()
    binarize(lib, 1000)
    took = time.perf_counter() - start
    t.join()
    fake.fake_delay_malloc(0)
    lib.ytm_destroy(m)
    assert took < 0.4, took


def staging_per_device(fake, lib, L):
    """Large copies from two devices in turn make each device's pinned buffers once."""
    models = []
    for d in (0, 1):
        assert fake.hipSetDevice(d) == 0
        models.append(small_model(lib, L))
    for _ in range(3):
        for d in (0, 1):
            assert fake.hipSetDevice(d) == 0
            binarize(lib, 3 * MB)
    assert fake.fake_calls(HOST_MALLOC) == 2, fake.fake_calls(HOST_MALLOC)
    for m in models:
        lib.ytm_destroy(m)
    assert fake.fake_calls(HOST_FREE) == 0
    assert lib.ytm_shutdown() == 0
    assert fake.fake_live(-1) == fake.fake_live(0) == fake.fake_live(1) == 0


def new_models_first_score(fake, lib, L):
    """While a model lives, another one's first score finds its pinned and its large buffers there."""
    def score(m, n, bits):
        X, out = np.zeros((n, 1, (2 * bits + 31) // 32), np.uint32), np.empty((n, 3), np.float32)
        before = fake.fake_calls(LARGE) + fake.fake_calls(HOST_MALLOC)
        assert lib.ytm_score(m, X.ctypes.data, n, out.ctypes.data) == 0
        return fake.fake_calls(LARGE) + fake.fake_calls(HOST_MALLOC) - before

    def model(bits):
        p = L.YtmParams(clauses=600, classes=3, dim0=bits, dim1=1, dim2=1, patch_dim0=bits, patch_dim1=1,
                        number_of_ta_states=256, max_included_literals=2 * bits, append_negated=1, encode_loc=1,
                        coalesced=1, negative_polarity=1, thresh=10, s_inv=0.2, q_prob=1.0, seed=1)
        m = ctypes.c_void_p()
        assert lib.ytm_create(ctypes.byref(p), ctypes.byref(m)) == 0
        return m

    for bits, n in ((784, 1), (784, 10000), (5000, 3), (40, 2000)):
        first, second = model(bits), model(bits)
        score(first, n, bits)
        assert score(second, n, bits) == 0, (bits, n)
        lib.ytm_destroy(second)
        lib.ytm_destroy(first)


def room_for_operands(fake, lib, L):
    """A model of 180 MB of states: created where little more than these fits, without the room of
    its scores' operands; and one of 1.1 GB of states holds no such room."""
    def model(clauses):
        p = L.YtmParams(clauses=clauses, classes=3, dim0=10000, dim1=1, dim2=1, patch_dim0=10000, patch_dim1=1,
                        number_of_ta_states=256, max_included_literals=20000, append_negated=1, encode_loc=1,
                        coalesced=1, negative_polarity=1, thresh=10, s_inv=0.2, q_prob=1.0, seed=1)
        m = ctypes.c_void_p()
        return lib.ytm_create(ctypes.byref(p), ctypes.byref(m)), m

    for clauses, most, least in ((8000, 185 * MB, None), (8000, 0, 250 * MB), (50000, 0, None)):
        planes = clauses * 9 * 625 * 4
        fake.fake_limit(most)
        rc, m = model(clauses)
        fake.fake_limit(0)
        assert rc == 0, (clauses, most)
        held = fake.fake_live(0)
        assert held > least if least else held < planes + 30 * MB, (clauses, most, held)
        lib.ytm_destroy(m)


def every_call_failing(name, fake, lib, L):
    prepare, call, free = entry(name, lib, L)
    wrong = []
    for fn in CALLS:
        for after in range(200):
            h = prepare()
            fake.fake_fail(fn.encode(), after, 2 if fn in ("hipMalloc", "hipHostMalloc") else 1)  # tried again
            rc = call(h)
            reached = fake.fake_failed()
            fake.fake_fail(b"", -1, 0)
            where = f"{name}: call {after} of {fn} failing"
            copied = name in ("encode", "binarize") and fn in ("hipHostMalloc", "hipStreamCreateWithFlags", "hipGetDevice")
            if reached and rc != L.YTM_EHIP and not (copied and rc == 0):  # without the staged copy: the runtime's
                wrong.append(f"{where}: status {rc}")
            if not reached and rc != 0:
                wrong.append(f"{where}: not reached, status {rc}")
            if fake.fake_busy():
                wrong.append(f"{where}: returned with work under way")
            free(h)
            assert lib.ytm_shutdown() == 0
            if fake.fake_live(0) or fake.fake_live(-1):
                wrong.append(f"{where}: {fake.fake_live(0)} bytes of device and {fake.fake_live(-1)} of pinned memory lost")
                print("\n".join(wrong))
                sys.exit(1)
            if not reached:
                break
    print("\n".join(wrong))
    sys.exit(1 if wrong else 0)


if __name__ == "__main__":
    fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
    fake.fake_live.restype = ctypes.c_size_t
    fake.fake_calls.restype = ctypes.c_long
    fake.fake_limit.argtypes = [ctypes.c_size_t]
    from ytm_amd import _lib

    if sys.argv[2] in ENTRIES:
        every_call_failing(sys.argv[2], fake, _lib.lib, _lib)
    else:
        globals()[sys.argv[2]](fake, _lib.lib, _lib)
