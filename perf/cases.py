"""Workloads for timing ytm_amd through its public entry points.

The listed cases are what a user of the framework has it do, over the range of sizes of the
benchmark configurations (workloads.py) and below them: training on flat, image and text
data, with coalesced clauses and with one clause bank per class, from host arrays and from
data kept on the GPU; scoring and prediction from a single sample up to a whole test set;
and encoding raw images.  draw() gives more cases over the same ranges.

Training starts from a new model, as a program's first epoch does, and every pass is one more
epoch over the same samples.  Scoring uses a model state made here to look like a trained one
(clauses of literals that hold in some patch of a class, as many as trained clauses hold), so
that its class sums can be worked out without the framework.
"""
import math

import numpy as np
import torch

from ytm_amd import MultiClassTM, ThermometerBinarizer

HALF = 128  # an automaton above half of its 256 states includes its literal


# ------------------------------------------------------------------------------- the cases
def listed():
    flat = dict(data="digits", size=28, levels=1, patch=28)
    conv = dict(data="digits", size=28, levels=1, patch=10)
    colour = dict(data="images", size=32, levels=8, patch=3)
    text = dict(data="text", size=10000, levels=1, patch=10000)
    m_flat = dict(clauses=2000, classes=10, T=50, s=10.0, banks=False)
    m_conv = dict(clauses=8000, classes=10, T=10000, s=5.0, banks=False)
    m_colour = dict(clauses=20000, classes=10, T=15000, s=10.0, banks=False)
    m_text = dict(clauses=10000, classes=2, T=8000, s=2.0, banks=False)
    return [
        # the smallest training in use: a dozen bits, ten clauses, 40% label noise, from host
        # arrays; every sample's chain of evaluation and feedback counts
        dict(name="fit_xor", op="fit", data="xor", size=12, levels=1, patch=12, n=5000, clauses=10, classes=2, T=15,
             s=3.9, banks=False),
        # an epoch over 60000 binary 28x28 images seen whole, the data kept on the GPU
        dict(name="fit_digits", op="fit_device", n=60000, **flat, **m_flat),
        # the convolutional model on the same images in 10x10 patches, from encoded host arrays
        # (the samples are copied in on every call)
        dict(name="fit_conv", op="fit", n=8000, **conv, **m_conv),
        # colour images of 24 bits a pixel in 3x3 patches, the largest clause count
        dict(name="fit_images", op="fit_device", n=4000, **colour, **m_colour),
        # bags of words over 10000 words: the longest literal rows and the largest state
        dict(name="fit_text", op="fit_device", n=12000, **text, **m_text),
        # one bank of clauses per class (coalesced=False), the original multi-class machine
        dict(name="fit_banks", op="fit_device", n=3000, **flat, **dict(m_flat, clauses=200, banks=True)),
        # one image at a time from raw bits: encode, score, decide -- a server's latency
        dict(name="predict_one", op="predict", n=1, **flat, **m_flat),
        # a test set of encoded host arrays
        dict(name="predict_digits", op="predict_encoded", n=10000, **flat, **m_flat),
        # class sums of a test set kept on the GPU, many patches
        dict(name="score_conv", op="score_device", n=10000, **conv, **m_conv),
        # the same for colour images, the most patches, literals and clauses
        dict(name="score_images", op="score_device", n=2000, **colour, **m_colour),
        # the same for bags of words, clauses of hundreds of literals
        dict(name="score_text", op="score_device", n=10000, **text, **m_text),
        # 8-bit colour images to literal words, levels and patches in one pass
        dict(name="encode_images", op="encode", n=2000, **colour, **m_colour),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    op = rng.choice(["fit", "fit_device", "fit_device", "banks", "predict", "predict_encoded", "score_device",
                     "score_device", "encode"])
    banks = op == "banks"
    op = "fit_device" if banks else op
    data = "images" if op == "encode" else rng.choice(["digits", "conv", "images", "text"])
    fit = op.startswith("fit")
    if data == "text":
        size = log(600, 10000)
        c = dict(data="text", size=size, levels=1, patch=size, clauses=log(100, 10000), classes=rng.randint(2, 6),
                 s=round(rng.uniform(1.5, 6.0), 1), n=log(200, 4000) if fit else log(1, 10000))
    elif data == "images":
        c = dict(data="images", size=rng.randint(12, 32), levels=rng.randint(1, 8), patch=rng.randint(2, 5),
                 clauses=log(200, 20000), classes=rng.randint(2, 12), s=round(rng.uniform(3.0, 12.0), 1),
                 n=log(100, 2000) if fit else log(1, 2000))
    elif data == "conv":
        size = rng.randint(10, 28)
        c = dict(data="digits", size=size, levels=1, patch=rng.randint(3, min(12, size - 1)), clauses=log(50, 8000),
                 classes=rng.randint(2, 12), s=round(rng.uniform(3.0, 12.0), 1),
                 n=log(200, 4000) if fit else log(1, 5000))
    else:
        size = rng.randint(4, 28)
        c = dict(data="digits", size=size, levels=1, patch=size, clauses=log(10, 2000), classes=rng.randint(2, 12),
                 s=round(rng.uniform(2.0, 12.0), 1), n=log(500, 30000) if fit else log(1, 10000))
    c["T"] = log(max(4, c["clauses"] // 40), max(8, c["clauses"]))
    if banks:  # clauses are then per class
        c["clauses"] = max(4, min(c["clauses"] // c["classes"], 400))
        c["n"] = min(c["n"], 2000)
    c.update(op=op, banks=banks)
    if fit and rng.random() < 0.25:
        c["max_literals"] = rng.choice([8, 16, 32])
    if fit and rng.random() < 0.25:
        c["drop"] = 0.1
    return c


# ------------------------------------------------------------------------------ geometry
def dims(case):
    """dim and patch_dim of the model."""
    if case["data"] in ("xor", "text"):
        return (case["size"], 1, 1), (case["size"], 1)
    z = case["levels"] * (3 if case["data"] == "images" else 1)
    return (case["size"], case["size"], z), (case["patch"], case["patch"])


def geometry(case):
    """Clauses, literals, literal words and patches of the model, input values per sample."""
    (w, h, z), (pw, ph) = dims(case)
    half = pw * ph * z + (w - pw) + (h - ph)
    banks = case["classes"] if case["banks"] else 1
    return banks * case["clauses"], 2 * half, (2 * half + 31) // 32, (w - pw + 1) * (h - ph + 1), w * h * z


# ------------------------------------------------------------------------------ the data
def generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def smooth(shape, width, g):
    """Smooth random fields in [0, 1] over the last two axes."""
    f = torch.randn(shape, generator=g, device="cuda")
    r = 3 * width
    k = torch.exp(-0.5 * (torch.arange(-r, r + 1, device="cuda") / width) ** 2)
    k = k / k.sum()
    n = f.shape[-1]
    f = f.reshape(-1, 1, n, n)
    f = torch.nn.functional.conv2d(f, k.view(1, 1, 1, -1), padding=(0, r))
    f = torch.nn.functional.conv2d(f, k.view(1, 1, -1, 1), padding=(r, 0)).reshape(shape)
    lo, hi = f.amin((-2, -1), keepdim=True), f.amax((-2, -1), keepdim=True)
    return (f - lo) / (hi - lo)


def samples(case, seed):
    """Samples on the GPU and their classes: bits (n, values) uint8, or 8-bit images."""
    g, n, K, size = generator(seed), case["n"], case["classes"], case["size"]
    if case["data"] == "xor":
        X = torch.randint(0, 2, (n, size), generator=g, device="cuda", dtype=torch.uint8)
        flip = torch.rand(n, generator=g, device="cuda") < 0.4
        return X, (X[:, 0] ^ X[:, 1] ^ flip).long()
    if case["data"] == "digits":
        p = 0.02 + 0.93 * smooth((K, size, size), max(1, size // 9), g).reshape(K, -1)
        y = torch.randint(0, K, (n,), generator=g, device="cuda")
        return (torch.rand((n, size * size), generator=g, device="cuda") < p[y]).to(torch.uint8), y
    if case["data"] == "images":
        mean = 255.0 * smooth((K, 3, size, size), max(1, size // 8), g).permute(0, 2, 3, 1)
        y = torch.randint(0, K, (n,), generator=g, device="cuda")
        noise = torch.randn((n, size, size, 3), generator=g, device="cuda")
        return (mean[y] + 32.0 * noise).clamp_(0, 255).to(torch.uint8), y
    base = torch.arange(1, size + 1, device="cuda", dtype=torch.float64) ** -1.1
    perm, own = torch.randperm(size, generator=g, device="cuda"), max(1, size // 50)
    y = torch.randint(0, K, (n,), generator=g, device="cuda")
    X = torch.zeros((n, size), dtype=torch.uint8, device="cuda")
    for k in range(K):
        p = base.clone()
        p[perm[own * k:own * (k + 1)]] *= 3.0
        rows = (y == k).nonzero()[:, 0]
        u = torch.rand((rows.numel(), 150), generator=g, device="cuda", dtype=torch.float64)
        words = torch.searchsorted(torch.cumsum(p / p.sum(), 0), u).clamp_(max=size - 1)
        X[rows[:, None], words] = 1
    return X, y


def bits_of(case, X):
    """The binary input values (n, values) of the samples."""
    if case["data"] != "images":
        return X
    t = torch.arange(1, case["levels"] + 1, device="cuda", dtype=torch.float64) * 255 / (case["levels"] + 1)
    return (X.double()[..., None] >= t).to(torch.uint8).reshape(X.shape[0], -1)


def literals(case, bits):
    """The literals (n, patches, literals) of binary input values, uint8."""
    (w, h, z), (pw, ph) = dims(case)
    n, ny, nx = bits.shape[0], h - ph + 1, w - pw + 1
    v = bits.reshape(n, h, w * z).unfold(1, ph, 1).unfold(2, pw * z, z)  # (n, ny, nx, ph, pw * z)
    pos = torch.empty((n, ny, nx, (ny - 1) + (nx - 1) + ph * pw * z), dtype=torch.uint8, device=bits.device)
    py, px = torch.arange(ny, device=bits.device), torch.arange(nx, device=bits.device)
    pos[..., :ny - 1] = (py[None, :-1] < py[:, None])[:, None]
    pos[..., ny - 1:ny + nx - 2] = (px[None, :-1] < px[:, None])[None]
    pos[..., ny + nx - 2:] = v.reshape(n, ny, nx, -1)
    pos = pos.reshape(n, ny * nx, -1)
    return torch.cat([pos, 1 - pos], 2)


def host_bits(bits):
    return bits.to(torch.int32).cpu().numpy().view(np.uint32)


def encoded(case, tm, X):
    """The samples as the framework encodes them, on the host."""
    if case["data"] == "images":
        return tm.encode_binarized(X.cpu().numpy(), ThermometerBinarizer(case["levels"]))
    return np.concatenate([tm.encode(host_bits(b)) for b in X.split(4000)])


def trained_state(case, seed):
    """A state as training leaves it: includes (clauses, literals), bool, and weights (clauses,
    classes), float32, on the GPU.

    A clause takes literals that are true in one patch of one of a few samples (other ones of
    the same classes), mostly those that hold in most samples of its class; how many, as
    clauses trained on such data hold."""
    C, L, _, P, _ = geometry(case)
    K = case["classes"]
    X, cls = samples(dict(case, n=24 * K), seed)
    lits = literals(case, bits_of(case, X))
    g = generator(seed + 1)
    hold = torch.stack([lits[cls == k].float().mean(0) if bool((cls == k).any()) else lits.float().mean(0)
                        for k in range(K)])  # (K, P, L)
    of = torch.randint(0, 24 * K, (C,), generator=g, device="cuda")
    at = torch.randint(0, P, (C,), generator=g, device="cuda")
    z = torch.randn(C, generator=g, device="cuda")
    if case["data"] == "text":
        count, spread = (0.015 * L + 0.004 * L * z).clamp(L / 1500, 0.034 * L), 0.06
    elif case["data"] == "images":
        count, spread = (0.12 * L * torch.exp(0.7 * z)).clamp(2, 0.42 * L), 0.15
    elif P > 1:
        count, spread = (0.095 * L + 0.026 * L * z).clamp(2, 0.16 * L), 0.3
    else:
        count, spread = (4.2 + 1.3 * z).clamp(1, 10), 0.35
    count = count.round().long()
    most = int(count.max())
    inc = torch.zeros((C, L), dtype=torch.bool, device="cuda")
    for c in range(0, C, 2000):
        o, p, n = of[c:c + 2000], at[c:c + 2000], count[c:c + 2000]
        score = hold[cls[o], p] + spread * torch.randn((o.numel(), L), generator=g, device="cuda")
        score[lits[o, p] == 0] = -1e9
        top = score.topk(min(most, L), 1).indices
        keep = torch.arange(top.shape[1], device="cuda")[None] < n[:, None]
        inc[c:c + 2000].scatter_(1, top, keep & (score.gather(1, top) > -1e8))
    mag = torch.randint(0, 60, (C, K), generator=g, device="cuda").float()
    sign = torch.full((C, K), -1.0, device="cuda")
    sign[torch.arange(C, device="cuda"), cls[of]] = 1.0
    return inc, (mag * sign).float()


# ------------------------------------------------------------------------------- the runs
def model(case, seed):
    dim, patch = dims(case)
    opt = {"max_included_literals": case["max_literals"]} if "max_literals" in case else {}
    return MultiClassTM(case["clauses"], case["T"], case["s"], dim, case["classes"], patch_dim=patch,
                        coalesced=not case["banks"], seed=seed, **opt)


def prepare(case, seed):
    X, y = samples(case, seed)
    tm = model(case, seed)
    st = {"op": case["op"], "tm": tm, "drop": case.get("drop", 0.0)}
    labels = y.to(torch.int32).cpu().numpy().view(np.uint32)
    if case["op"] == "encode":
        st["X"], st["binarizer"] = X.cpu().numpy(), ThermometerBinarizer(case["levels"])
        return st
    if case["op"].startswith("fit"):
        tm.load_kernels()
        st["X"], st["y"] = encoded(case, tm, X), labels
        if case["op"] == "fit_device":
            st["data"] = tm.device_data(st.pop("X"), st["y"], is_X_encoded=True)
        return st
    inc, w = trained_state(case, seed)
    g = generator(seed + 2)
    ta = torch.randint(0, HALF + 1, inc.shape, generator=g, device="cuda", dtype=torch.int32)
    ta = torch.where(inc, 2 * HALF - ta.clamp_(max=HALF - 1), ta)
    C, _, _, P, _ = geometry(case)
    tm.load_state_dict({"state": {"ta_state": ta.cpu().numpy().view(np.uint32), "clause_weights": w.cpu().numpy(),
                                  "patch_weights": np.zeros(C * P, np.int32), "min_y": None, "max_y": None}})
    if case["op"] == "predict":
        st["X"] = host_bits(bits_of(case, X))
    elif case["op"] == "predict_encoded":
        st["X"] = encoded(case, tm, X)
    else:
        st["data"] = tm.device_data(encoded(case, tm, X), is_X_encoded=True)
    return st


def run(state):
    tm, op = state["tm"], state["op"]
    if op == "encode":
        return tm.encode_binarized(state["X"], state["binarizer"])
    if op == "predict":
        return tm.predict(state["X"])
    if op == "predict_encoded":
        return tm.predict(state["X"], is_X_encoded=True)
    if op == "score_device":
        return tm.score_device(state["data"])
    if op == "fit":
        tm.fit(state["X"], state["y"], is_X_encoded=True, clause_drop_p=state["drop"])
    else:
        tm.fit_device(state["data"], clause_drop_p=state["drop"])
    return {"ta_state": tm.get_ta_state().view(np.int32), "weights": tm.get_weights(),
            "patch_weights": tm.get_patch_weights()}


def work(case):
    """Bytes: samples and targets read once, the model's state (2 bytes an automaton, 4 a
    weight) read once and, in training, written once, results written once.  Operations: two
    (AND, OR) for each literal word of each clause on each patch of each sample, which is what
    evaluating the clauses without leaving any out comes to."""
    C, L, W, P, F = geometry(case)
    n, K = case["n"], case["classes"]
    x = 4 * n * P * W
    state = 2 * C * L + 4 * C * K
    ops = 2 * n * C * P * W
    if case["op"] == "encode":
        return {"bytes": n * F // case["levels"] + x, "flops": 0}
    if case["op"].startswith("fit"):
        return {"bytes": x + 4 * n * K + 2 * state + 4 * C * P, "flops": ops}
    return {"bytes": (4 * n * F if case["op"] == "predict" else x) + state + 4 * n * K, "flops": ops}


def tolerance(case):
    # Everything here is a whole number: literal words, automaton states, integer-valued
    # weights and their sums (well below 2^24), the same for every order of summation.
    return "exact"


def exact(case, seed):
    """Class sums from the clauses' definition: a clause votes when some patch has all of its
    literals.  Trained states follow the framework's own random stream, which nothing outside
    it gives; encoded words are whole numbers, compared as they are."""
    if case["op"] == "encode" or case["op"].startswith("fit"):
        return None
    X, y = samples(case, seed)
    inc, w = trained_state(case, seed)
    need = inc.float().t().contiguous()
    votes = w.double()
    votes[~inc.any(1)] = 0.0
    C, L, _, P, _ = geometry(case)
    out = []
    for part in bits_of(case, X).split(max(1, 400_000_000 // (P * max(C, L)))):
        miss = (1 - literals(case, part)).float().reshape(-1, L) @ need  # literals of a clause not in a patch
        fire = (miss.reshape(part.shape[0], P, C) == 0).any(1)
        out.append(fire.double() @ votes)
    sums = torch.cat(out).cpu().numpy()
    return [None, sums] if case["op"].startswith("predict") else sums
