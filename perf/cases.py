"""Performance cases: the calls that users of this package make, from a single short path to gigabytes of signatures.

Four kinds of call ("op"):

  sig     signatures of a batch of paths (feature extraction, scoring)
  train   signatures and the gradient with respect to the paths (a layer of a network), through autograd
  logsig  the same for log signatures (Lyndon coordinates), tables prepared beforehand as a program does once
  stream  running signatures extended by one increment and joined with the signatures of the next block, with the
          gradients of all inputs (online features of a recurrent model)

listed() holds fixed cases, draw() makes more of the same ranges.
"""
import math

import torch

import pysiglib_amd as P

DTYPES = {"f32": torch.float32, "f64": torch.float64}


def _case(name, op, dtype, batch, length, dim, degree, time_aug=False, lead_lag=False, points=False, method=1):
    c = dict(op=op, dtype=dtype, batch=batch, length=length, dim=dim, degree=degree, time_aug=time_aug, lead_lag=lead_lag,
             points=points, method=method)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one short path as it arrives, scored online: nothing but latency
        _case("one_short_path_f32", "sig", "f32", 1, 64, 3, 4),
        # a few short paths in double precision, forward and backward: latency of a whole training step
        _case("few_paths_train_f64", "train", "f64", 4, 32, 4, 5),
        # an ordinary training batch of narrow time series
        _case("batch_train_f32", "train", "f32", 128, 256, 4, 6),
        # the quick-start shape of the package in double precision
        _case("quick_start_train_f64", "train", "f64", 32, 1000, 10, 5, points=True),
        # features of simulated Brownian paths, fairly deep, single precision
        _case("brownian_features_f32", "sig", "f32", 128, 1024, 5, 7),
        # long paths of three channels to a high degree in double precision: the largest amount of arithmetic
        _case("high_degree_f64", "sig", "f64", 64, 4096, 3, 12),
        # lead-lag and time augmentation, a training batch
        _case("augmented_train_f32", "train", "f32", 256, 500, 8, 4, time_aug=True, lead_lag=True),
        # many short wide paths at degree 2 (covariance-like features of embeddings)
        _case("wide_degree2_train_f32", "train", "f32", 2048, 256, 64, 2),
        # ten channels to degree 6
        _case("ten_channels_train_f32", "train", "f32", 64, 200, 10, 6),
        # sixty-four channels to degree 4: few paths, a million times sixteen coefficients each
        _case("wide_degree4_train_f32", "train", "f32", 16, 200, 64, 4),
        # log-signature layer, odd sizes throughout
        _case("log_signature_train_f32", "logsig", "f32", 257, 99, 7, 5),
        # running signatures of a large batch of streams: bound by memory
        _case("stream_update_f64", "stream", "f64", 1024, 2, 10, 5),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        op = rng.choice(("sig", "sig", "train", "train", "train", "logsig", "stream"))
        dtype = rng.choice(("f32", "f32", "f64"))
        batch, length = _log_int(rng, 1, 4096), _log_int(rng, 16, 8192)
        dim, degree = _log_int(rng, 2, 96), rng.randint(2, 12)
        time_aug = op in ("sig", "train") and rng.random() < 0.25
        lead_lag = op in ("sig", "train") and dim <= 16 and rng.random() < 0.25
        c = _case(None, op, dtype, batch, 2 if op == "stream" else length, dim, degree, time_aug, lead_lag,
                  points=dtype == "f64" and op == "train" and rng.random() < 0.25, method=rng.choice((1, 2)))
        if op == "logsig" and _coefs(c) > 60000:        # the tables of the Lyndon words are prepared in seconds at most
            continue
        w = work(c)
        if _channels(c) ** degree <= 20000000 and w["bytes"] <= 6e9 and w["flops"] <= 2e11:
            return c


def _channels(c):
    return (2 * c["dim"] if c["lead_lag"] else c["dim"]) + (1 if c["time_aug"] else 0)


def _coefs(c):
    return sum(_channels(c) ** k for k in range(1, c["degree"] + 1))


def _paths(c, gen):
    dtype, shape = DTYPES[c["dtype"]], (c["batch"], c["length"], c["dim"])
    if c["points"]:             # independent points
        return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float64).to(dtype)
    inc = torch.randn(shape, generator=gen, device="cuda", dtype=torch.float64) / math.sqrt(c["length"])
    return inc.cumsum(1).to(dtype)      # a random walk over about one unit, as after normalisation


def prepare(case, seed):
    c = dict(case)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    dtype, d, n = DTYPES[c["dtype"]], _channels(c), _coefs(c)
    if c["op"] == "stream":
        walks = dict(c, length=24, points=False)
        sigs = [_rows(_signature(_paths(walks, gen), c["degree"])).to(dtype) for _ in range(2)]
        state = {"sig": sigs[0].requires_grad_(True), "block": sigs[1].requires_grad_(True),
                 "increment": (torch.randn((c["batch"], d), generator=gen, device="cuda", dtype=dtype) * 0.2).requires_grad_(True)}
    else:
        state = {"path": _paths(c, gen)}
        if c["op"] != "sig":
            state["path"].requires_grad_(True)
        if c["op"] == "logsig":
            P.prepare_log_sig(d, c["degree"], c["method"])
            n = P.log_sig_length(d, c["degree"])
    if c["op"] != "sig":
        state["grad"] = torch.randn((c["batch"], n), generator=gen, device="cuda", dtype=dtype)
    state["case"] = c
    return state


def run(state):
    c = state["case"]
    if c["op"] == "sig":
        return P.sig(state["path"], c["degree"], time_aug=c["time_aug"], lead_lag=c["lead_lag"])
    if c["op"] == "train":
        out = P.torch_api.sig(state["path"], c["degree"], time_aug=c["time_aug"], lead_lag=c["lead_lag"])
        return [out.detach(), *torch.autograd.grad(out, state["path"], state["grad"])]
    if c["op"] == "logsig":
        out = P.torch_api.log_sig(state["path"], c["degree"], method=c["method"])
        return [out.detach(), *torch.autograd.grad(out, state["path"], state["grad"])]
    joined = P.torch_api.sig_join(state["sig"], state["increment"], c["dim"], c["degree"])
    out = P.torch_api.sig_combine(joined, state["block"], c["dim"], c["degree"])
    inputs = (state["sig"], state["increment"], state["block"])
    return [out.detach(), *torch.autograd.grad(out, inputs, state["grad"])]


def _horner(d, moving, degree):
    """Flops of one Horner step: level t is reached through levels 1 .. t-1, one multiply-add per value; `moving` of the
    d letters can be non-zero in a step."""
    return sum(2 * d ** (k - 1) * (moving if k > 1 else d) for t in range(1, degree + 1) for k in range(1, t + 1))


def work(case):
    c = case
    d, n, size = _channels(c), _coefs(c), 4 if c["dtype"] == "f32" else 8
    rows, path = c["batch"] * n * size, c["batch"] * c["length"] * c["dim"] * size
    if c["op"] == "stream":
        # Chen products: a coefficient of level t sums over its t - 1 inner splits; three of them (the forward and the
        # gradients of both factors), and three Horner passes for the increment
        chen = 2 * c["batch"] * sum((t - 1) * d ** t for t in range(1, c["degree"] + 1))
        step = c["batch"] * _horner(d, d, c["degree"])
        # read: two signatures and the gradient; written: the result and two gradients
        return {"bytes": 6 * rows + 2 * c["batch"] * d * size, "flops": 3 * chen + 3 * step}
    steps = ((2 * c["length"] - 1) if c["lead_lag"] else c["length"]) - 1
    moving = c["dim"] + (1 if c["time_aug"] else 0)
    forward = c["batch"] * steps * _horner(d, moving, c["degree"])
    if c["op"] == "sig":
        return {"bytes": path + rows, "flops": forward}
    # reverse step: the state up to level N - 1 is taken back (one Horner step), and every product of the step passes
    # gradients to both of its factors
    backward = c["batch"] * steps * (2 * _horner(d, moving, c["degree"]) + _horner(d, moving, c["degree"] - 1))
    if c["op"] == "train":
        return {"bytes": 2 * path + 2 * rows, "flops": forward + backward}
    # the tensor logarithm: degree - 1 Chen products, gradients of both factors on the way back
    log = 2 * c["batch"] * (c["degree"] - 1) * sum((t - 1) * d ** t for t in range(1, c["degree"] + 1))
    small = c["batch"] * P.log_sig_length(d, c["degree"]) * size
    return {"bytes": 2 * path + 2 * small, "flops": forward + backward + 3 * log}


# Relative error (2-norm) and largest single error of single precision that correct code shows: four times what the calls
# differ by from the same calls in double precision, over the listed and a hundred drawn cases.  Signatures differ by up to
# 1.2e-6 / 2.1e-4, with gradients among the outputs by up to 1.1e-5 / 4.9e-4 (their reverse sweep recovers every earlier
# state from the final one), running signatures by 1.0e-6 / 8.2e-5, log signatures, sums of terms that cancel, by up to
# 3.6e-5 / 2.4e-3.
_SINGLE = {"sig": (5e-6, 1e-3), "train": (5e-5, 2e-3), "stream": (5e-6, 4e-4), "logsig": (1.5e-4, 1e-2)}


def tolerance(case):
    rel, most = _SINGLE[case["op"]]
    unit = 1.0 if case["dtype"] == "f32" else 2.0 ** -29        # double precision: by the ratio of the two roundings
    return {"rel": rel * unit, "max": most * unit}


# ---- the same in 64 bits, with plain torch ----
# A signature is a list of its levels, level k of shape (rows, d ** k); the leading 1 is left out.

def _augmented(path, time_aug, lead_lag):
    if lead_lag:        # lag and lead channels, the lead moves first
        twice = path.repeat_interleave(2, 1)
        path = torch.cat((twice[:, :-1], twice[:, 1:]), 2)
    if time_aug:
        time = torch.linspace(0.0, 1.0, path.shape[1], dtype=path.dtype, device=path.device)
        path = torch.cat((path, time.expand(path.shape[0], -1).unsqueeze(2)), 2)
    return path


def _outer(a, b):
    return (a.unsqueeze(2) * b.unsqueeze(1)).reshape(a.shape[0], -1)


def _times(a, b, unit=1.0):
    """Truncated tensor product; with unit 0 of the two without their leading 1."""
    out = []
    for t in range(len(a)):
        v = (a[t] + b[t]) if unit else torch.zeros_like(a[t])
        for k in range(t):
            v = v + _outer(a[k], b[t - 1 - k])
        out.append(v)
    return out


def _extended(levels, z):
    """levels times exp(z), by Horner's rule."""
    out = list(levels)
    for t in range(len(levels), 0, -1):
        v = z / t
        for k in range(1, t):
            v = _outer(levels[k - 1] + v, z / (t - k))
        out[t - 1] = levels[t - 1] + v
    return out


def _rows(levels):
    return torch.cat(levels, 1)


def _pieces(z, degree):
    """Increments (rows, steps, d) cut in time into pieces that are swept beside each other: (rows * pieces, steps, d)."""
    rows, steps, d = z.shape
    size = 8.0 * rows * sum(d ** k for k in range(1, degree + 1))
    pieces = 1
    while pieces < 64 and steps >= 32 * pieces and size * 2 * pieces <= 3e7:
        pieces *= 2
    each = -(-steps // pieces)
    z = torch.nn.functional.pad(z, (0, 0, 0, pieces * each - steps))
    return z.reshape(rows * pieces, each, d), pieces


def _joined(levels, pieces):
    while pieces > 1:
        halves = [v.reshape(-1, 2, v.shape[1]) for v in levels]
        levels, pieces = _times([v[:, 0] for v in halves], [v[:, 1] for v in halves]), pieces // 2
    return levels


def _signature(path, degree, time_aug=False, lead_lag=False, grad_of=None):
    """Levels of the signature, or with grad_of(levels) -> scalar: (levels, gradient with respect to the path)."""
    path = path.detach().double()
    if grad_of is not None:
        path.requires_grad_(True)
    with torch.set_grad_enabled(grad_of is not None):
        points = _augmented(path, time_aug, lead_lag)
        cut, pieces = _pieces(points[:, 1:] - points[:, :-1], degree)
    z, d = cut.detach(), cut.shape[2]
    state = [torch.zeros((z.shape[0], d ** k), dtype=torch.float64, device=z.device) for k in range(1, degree + 1)]
    stride = max(1, math.isqrt(z.shape[1]))
    kept = []               # the state before every `stride` steps, from which the gradient sweeps them again
    for s in range(z.shape[1]):
        if grad_of is not None and s % stride == 0:
            kept.append(state)
        state = _extended(state, z[:, s])
    if grad_of is None:
        return _joined(state, pieces)
    ends = [v.requires_grad_(True) for v in state]
    with torch.enable_grad():
        whole = _joined(ends, pieces)
        back = torch.autograd.grad(grad_of(whole), ends)
    dz = torch.zeros_like(z)
    for n in range(len(kept) - 1, -1, -1):
        part = z[:, n * stride:(n + 1) * stride].clone().requires_grad_(True)
        first = [v.detach().requires_grad_(True) for v in kept.pop()]
        with torch.enable_grad():
            v = first
            for s in range(part.shape[1]):
                v = _extended(v, part[:, s])
        got = torch.autograd.grad(v, [part, *first], back)
        dz[:, n * stride:(n + 1) * stride] = got[0]
        back = got[1:]
    return [v.detach() for v in whole], torch.autograd.grad(cut, path, dz)[0]


def _logarithm(levels):
    out, power = list(levels), levels
    for k in range(2, len(levels) + 1):
        power = _times(power, levels, 0.0)
        out = [a + b * ((-1) ** (k + 1) / k) for a, b in zip(out, power)]
    return out


def _lyndon_words(d, degree):
    """By length, then in alphabetical order (Duval's successor rule)."""
    found, w = [[] for _ in range(degree)], [-1]
    while w:
        w[-1] += 1
        found[len(w) - 1].append(tuple(w))
        w = [w[i % len(w)] for i in range(degree)]
        while w and w[-1] == d - 1:
            w.pop()
    return found


def _index(word, d):
    n = 0
    for letter in word:
        n = n * d + letter
    return n


def _coordinates(d, degree, method):
    """Functions of the levels of a tensor logarithm: its coefficients at the Lyndon words, or its coordinates in the basis
    of their brackets [u, v], v the longest proper suffix that is a Lyndon word."""
    found, brackets, parts = _lyndon_words(d, degree), {}, []
    for words in found:
        at = torch.tensor([_index(w, d) for w in words], device="cuda")
        matrix = None
        if method == 2:
            matrix = torch.eye(len(words), dtype=torch.float64)
            position = {w: i for i, w in enumerate(words)}
            for j, w in enumerate(words):
                if len(w) == 1:
                    brackets[w] = {w: 1.0}
                    continue
                cut = next(i for i in range(1, len(w)) if w[i:] in brackets)
                terms = {}
                for a, x in brackets[w[:cut]].items():
                    for b, y in brackets[w[cut:]].items():
                        terms[a + b] = terms.get(a + b, 0.0) + x * y
                        terms[b + a] = terms.get(b + a, 0.0) - x * y
                brackets[w] = terms
                for a, x in terms.items():
                    if a in position:
                        matrix[position[a], j] = x
            matrix = matrix.cuda()
        parts.append((at, matrix))

    def read(levels):
        out = []
        for v, (at, matrix) in zip(levels, parts):
            v = v[:, at]
            out.append(v if matrix is None else torch.linalg.solve_triangular(matrix, v.T, upper=False).T)
        return _rows(out)
    return read


def exact(case, seed):
    c, degree, d = case, case["degree"], _channels(case)
    steps = (2 * c["length"] - 1) if c["lead_lag"] else c["length"]
    # sweeps in launches: the forward sweep, and for the gradient a second one and the way back of each
    launches = degree * (degree + 1) * 1.5 * (1 if c["op"] == "sig" else 5)
    if c["op"] != "stream" and steps * launches * 6e-6 > 18 and c["batch"] * _coefs(c) > 50000:
        return None
    if c["op"] == "logsig" and c["method"] == 2 and sum(map(len, _lyndon_words(d, degree))) > 6000:
        return None
    state = prepare(case, seed)
    rows = max(1, int(1e9 // (8 * _coefs(c) * (1 if c["op"] == "sig" else degree))))     # paths at a time
    read = _coordinates(d, degree, c["method"]) if c["op"] == "logsig" else None
    out = []
    for n in range(0, c["batch"], rows):
        part = slice(n, n + rows)
        if c["op"] == "stream":
            x, z, y = (state[k].detach()[part].double().requires_grad_(True) for k in ("sig", "increment", "block"))
            with torch.enable_grad():
                levels = [v.split([d ** k for k in range(1, degree + 1)], 1) for v in (x, y)]
                whole = _rows(_times(_extended(levels[0], z), levels[1]))
            out.append([whole.detach(), *torch.autograd.grad(whole, (x, z, y), state["grad"][part].double())])
            continue
        path, options = state["path"][part], (degree, c["time_aug"], c["lead_lag"])
        if c["op"] == "sig":
            out.append([_rows(_signature(path, *options))])
            continue
        grad = state["grad"][part].double()
        last = (lambda v: read(_logarithm(v))) if read else _rows
        levels, dpath = _signature(path, *options, grad_of=lambda v: (last(v) * grad).sum())
        out.append([last(levels), dpath])
    out = [torch.cat(v) for v in zip(*out)]
    return out[0] if c["op"] == "sig" else out
