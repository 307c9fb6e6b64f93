"""Performance cases of the circulant attention entry points on one GPU.

A case is a dict of plain values:

  op        "attention": y = circulant_mh_attention(...) without the matrix
            A (materialize=False), the fused kernels;
            "dense": the same call returning (y, A) (materialize=True, the
            default of the API), A a Circulant;
            "adjacency": A = circulant_mh_adjacency(sim, x, x, ...), then
            A ⨷ z and the transposed A ⨷ z (a graph formed once and applied);
            "compose": C = A + scale(m, B), then C ⨷ x, on two Circulants the
            program already holds
  sim       "dot" or "distance"
  n1, n2    spatial size, fastest first; n2 = 0 is a one-dimensional signal
  window    the window's odd side
  channels  channels of the signal over all heads (complex ones for complex)
  heads, batch
  complex   ComplexF32 signals instead of Float32
  last      channels-last tensors ("attention" only)
  train     the gradients of q, k, v are formed as well

listed() are the cases that are timed every time; draw() gives further ones of
the same ranges.  exact() restates the results in 64-bit torch operations: one
roll of the signal per window offset, none of the package's code.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "circulantattention.jl_amd"))

import circulant_attention as ca  # noqa: E402


def _case(op, sim, n1, n2, window, channels, heads, batch, *, complex=False, last=False,
          train=False, name=None):
    c = {"op": op, "sim": sim, "n1": n1, "n2": n2, "window": window, "channels": channels,
         "heads": heads, "batch": batch, "complex": complex, "last": last, "train": train}
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # a single small patch in a serving loop: latency and launches
        _case("attention", "dot", 24, 20, 15, 32, 2, 1, name="patch_infer"),
        # denoising-size image, 64 channels in one head, the documented
        # quick-start's size, without A
        _case("attention", "dot", 128, 96, 15, 64, 1, 2, name="image_infer_head64"),
        # training step of multi-head attention on square images
        _case("attention", "dot", 256, 256, 15, 64, 4, 4, train=True, name="image_train_heads4"),
        # complex-valued images (as of MRI), two heads
        _case("attention", "dot", 320, 320, 11, 32, 2, 2, complex=True, train=True,
              name="complex_train"),
        # a large image with a wide window and the distance similarity
        _case("attention", "distance", 512, 512, 31, 32, 1, 1, train=True, name="wide_window_train"),
        # a long one-dimensional signal
        _case("attention", "distance", 262144, 0, 63, 32, 1, 2, train=True, name="line_train"),
        # feature maps of a convolutional model (channels-last), odd sizes, a
        # window and a head width between the common ones
        _case("attention", "dot", 131, 101, 9, 96, 2, 2, last=True, train=True,
              name="ragged_last_train"),
        # the quick-start call: y and A
        _case("dense", "dot", 128, 96, 15, 64, 1, 2, name="dense_infer"),
        # training through the matrix-returning call, complex, two heads
        _case("dense", "dot", 320, 320, 11, 32, 2, 2, complex=True, train=True,
              name="dense_complex_train"),
        # the same, distance similarity on a small odd image
        _case("dense", "distance", 97, 75, 7, 64, 4, 1, train=True, name="dense_ragged_train"),
        # a non-local graph formed from features and applied to codes
        _case("adjacency", "distance", 200, 120, 23, 32, 1, 1, name="graph_wide"),
        # two attention maps combined and applied
        _case("compose", "dot", 320, 320, 11, 32, 2, 2, complex=True, name="compose_complex"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(c):
    P, K = c["n1"] * max(1, c["n2"]), c["window"] ** (2 if c["n2"] else 1)
    real = c["channels"] * (2 if c["complex"] else 1)
    dense = c["op"] in ("dense", "adjacency", "compose")
    return P * K * c["batch"] * (real * (3 if c["train"] else 1) + (60 * c["heads"] if dense else 0))


def draw(rng):
    """Images of 16 to 512 pixels a side (64 to 262144 along a line), windows
    of 3 to 31 (7 to 63 on a line), 8 to 64 real components per head, at most
    the largest listed case's work."""
    most = max(_cost(c) for c in listed())
    while True:
        op = rng.choice(["attention"] * 5 + ["dense"] * 3 + ["adjacency", "compose"])
        line = op == "attention" and rng.random() < 0.25
        if line:
            n1, n2 = _log_int(rng, 256, 262144), 0
            window = rng.choice([7, 15, 31, 63])
        else:
            n1, n2 = _log_int(rng, 16, 512), _log_int(rng, 16, 512)
            window = rng.choice([3, 5, 7, 9, 11, 13, 15, 15, 17, 23, 31])
        cplx = rng.random() < 0.25
        per = rng.choice([8, 16, 16, 24, 32, 32, 48, 64])
        heads = rng.choice([1, 2, 4])
        c = _case(op, rng.choice(["dot", "distance"]), n1, n2, window,
                  per * heads // (2 if cplx else 1), heads, rng.choice([1, 2, 3, 4]),
                  complex=cplx, last=op == "attention" and rng.random() < 0.3,
                  train=op in ("attention", "dense") and rng.random() < 0.6)
        nnz = n1 * max(1, n2) * window ** (2 if n2 else 1) * heads * c["batch"]
        if window <= n1 and (n2 == 0 or window <= n2) and _cost(c) <= most and (
                op == "attention" or nnz <= 60_000_000):
            return c


# ---------------------------------------------------------------------------
# inputs and the call
# ---------------------------------------------------------------------------
_TENSORS = {"attention": 4, "dense": 4, "adjacency": 3, "compose": 1}


def _signal_shape(c):
    sp = (c["n2"], c["n1"]) if c["n2"] else (c["n1"],)
    return (c["batch"], *sp, c["channels"]) if c["last"] else (c["batch"], c["channels"], *sp)


def _inputs(c, seed):
    """N(0,1) features (complex: unit variance); "adjacency", whose similarity
    is not scaled, has features of unit expected norm per head, as a learned
    embedding's; for "compose" also the two attention maps (softmaxed N(0,1)
    scores) and their weight m."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    dt = torch.complex64 if c["complex"] else torch.float32
    xs = [torch.randn(_signal_shape(c), device="cuda", dtype=dt, generator=g)
          for _ in range(_TENSORS[c["op"]])]
    if c["op"] == "adjacency":
        xs[0] *= (c["channels"] // c["heads"]) ** -0.5
    if c["op"] != "compose":
        return xs
    P, K = c["n1"] * max(1, c["n2"]), c["window"] ** (2 if c["n2"] else 1)
    maps = [torch.randn((c["batch"], c["heads"], P, K), device="cuda", generator=g).softmax(-1)
            for _ in range(2)]
    m = torch.randn((c["batch"], c["heads"], 1, 1), device="cuda", generator=g)
    return xs + maps + [m]


def prepare(case, seed):
    c = case
    xs = _inputs(c, seed)
    sim = ca.DotSimilarity() if c["sim"] == "dot" else ca.DistanceSimilarity()
    s = {"case": c, "sim": sim}
    if c["op"] in ("attention", "dense"):
        s["q"], s["k"], s["v"], s["dy"] = xs
        for t in xs[:3]:
            t.requires_grad_(c["train"])
    elif c["op"] == "adjacency":
        s["x"], s["z1"], s["z2"] = xs
    else:
        spatial = (c["n1"], c["n2"]) if c["n2"] else (c["n1"],)
        s["x"], s["m"] = xs[0], xs[3]
        s["A"], s["B"] = (ca.Circulant(t, c["window"], spatial) for t in xs[1:3])
    return s


def run(state):
    s, c = state, state["case"]
    if c["op"] in ("attention", "dense"):
        kw = {"materialize": c["op"] == "dense", "honor_simfun": True}
        if c["last"]:
            kw["channels_last"] = True
        args = (s["sim"], s["q"], s["k"], s["v"], c["window"], c["heads"])
        if not c["train"]:
            with torch.no_grad():
                y, A = ca.circulant_mh_attention(*args, **kw)
            return (y,) if A is None else (y, A.nzval)
        y, A = ca.circulant_mh_attention(*args, **kw)
        grads = torch.autograd.grad(y, (s["q"], s["k"], s["v"]), s["dy"])
        return (y.detach(), *grads) if A is None else (y.detach(), A.nzval.detach(), *grads)
    with torch.no_grad():
        if c["op"] == "adjacency":
            A = ca.circulant_mh_adjacency(s["sim"], s["x"], s["x"], c["window"], c["heads"])
            return (A.nzval, ca.Otimes(A, s["z1"]),
                    ca.circulant_mh_transposed_attention(A, s["z2"]))
        C = s["A"] + ca.scale(s["m"], s["B"])
        return C.nzval, ca.Otimes(C, s["x"])


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    c = case
    P, K = c["n1"] * max(1, c["n2"]), c["window"] ** (2 if c["n2"] else 1)
    real = c["channels"] * (2 if c["complex"] else 1)
    T = 4 * P * real * c["batch"]                       # one signal
    N = 4 * P * K * c["heads"] * c["batch"]             # one matrix's values
    U = 2 * P * K * real * c["batch"]                   # one window contraction
    if c["op"] == "adjacency":
        return {"bytes": 5 * T + N, "flops": 3 * U}
    if c["op"] == "compose":
        return {"bytes": 2 * T + 3 * N, "flops": U + N // 2}
    nA = N if c["op"] == "dense" else 0
    if c["train"]:
        return {"bytes": 8 * T + nA, "flops": 6 * U}
    return {"bytes": 4 * T + nA, "flops": 2 * U}


def tolerance(case):
    """Four times the largest error seen against exact() over the ranges: the
    fused backward forms the probabilities again from a rounded log-sum-exp,
    and products of 16-bit halves add to that; the matrix-forming path sums
    plain 32-bit products."""
    if case["op"] == "attention":
        return {"rel": 1.2e-5, "max": 1e-4}
    return {"rel": 3e-6, "max": 4e-5}


# ---------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------
def _offsets(c):
    """(u1, u2) of every window offset, u1 fastest."""
    p = c["window"] // 2
    r2 = range(-p, p + 1) if c["n2"] else (0,)
    return [(u1, u2) for u2 in r2 for u1 in range(-p, p + 1)]


def _at(x, u):
    """x at the pixel u away, circularly (the last axis is n1's)."""
    return torch.roll(x, (-u[0], -u[1]), (-1, -2)) if u[1] else torch.roll(x, -u[0], -1)


def _from(x, u):
    return _at(x, (-u[0], -u[1]))


def _order(c):
    """Slot order: along each axis a row's window columns ascend, so near the
    border they start at the wrapped ones; (n, window) offset indices."""
    p = c["window"] // 2
    out = []
    for n in (c["n1"], c["n2"]) if c["n2"] else (c["n1"],):
        cols = (torch.arange(n, device="cuda")[:, None] + torch.arange(-p, p + 1, device="cuda")) % n
        out.append(cols.argsort(dim=1, stable=True))
    return out


def _to_slots(c, a):
    """(units, offsets, *spatial) -> (batch, heads, P, slots)."""
    w = c["window"]
    o = _order(c)
    nu = a.shape[0]
    if c["n2"]:
        a = a.reshape(nu, w, w, c["n2"], c["n1"]).permute(0, 3, 4, 1, 2)
        a = a.gather(3, o[1][None, :, None, :, None].expand(nu, -1, c["n1"], -1, w))
        a = a.gather(4, o[0][None, None, :, None, :].expand(nu, c["n2"], -1, w, -1))
    else:
        a = a.permute(0, 2, 1).gather(2, o[0][None].expand(nu, -1, -1))
    return a.reshape(c["batch"], c["heads"], -1, w ** len(o))


def _to_offsets(c, a):
    """The inverse of _to_slots."""
    w = c["window"]
    o = [t.argsort(dim=1) for t in _order(c)]
    nu = c["batch"] * c["heads"]
    if c["n2"]:
        a = a.reshape(nu, c["n2"], c["n1"], w, w)
        a = a.gather(3, o[1][None, :, None, :, None].expand(nu, -1, c["n1"], -1, w))
        a = a.gather(4, o[0][None, None, :, None, :].expand(nu, c["n2"], -1, w, -1))
        return a.permute(0, 3, 4, 1, 2).reshape(nu, w * w, c["n2"], c["n1"])
    return a.reshape(nu, c["n1"], w).gather(2, o[0][None].expand(nu, -1, -1)).permute(0, 2, 1)


def _units(c, x):
    """A signal in 64 bits as (batch * heads, channels per head, *spatial)."""
    x = x.detach().to(torch.complex128 if c["complex"] else torch.float64)
    if c["last"]:
        x = x.movedim(-1, 1)
    return x.reshape(c["batch"] * c["heads"], c["channels"] // c["heads"], *x.shape[2:]).contiguous()


def _signal(c, x):
    x = x.reshape(c["batch"], c["channels"], *x.shape[2:])
    return x.movedim(1, -1).contiguous() if c["last"] else x


def _scores(c, q, k, scale):
    out = []
    for u in _offsets(c):
        ku = _at(k, u)
        s = (q * ku.conj()).real.sum(1) if c["sim"] == "dot" else -0.5 * (q - ku).abs().square().sum(1)
        out.append(scale * s)
    return torch.stack(out, 1)


def _apply(c, A, x):
    y = torch.zeros_like(x)
    for i, u in enumerate(_offsets(c)):
        y += A[:, i, None] * _at(x, u)
    return y


def exact(case, seed):
    c = case
    xs = _inputs(c, seed)
    if c["op"] == "compose":
        x, A, B, m = _units(c, xs[0]), xs[1].double(), xs[2].double(), xs[3].double()
        C = A + m * B
        return C, _signal(c, _apply(c, _to_offsets(c, C), x))
    if c["op"] == "adjacency":
        x, z1, z2 = (_units(c, t) for t in xs)
        A = _scores(c, x, x, 1.0).softmax(1)
        yt = torch.zeros_like(z2)
        for i, u in enumerate(_offsets(c)):
            yt += _from(A[:, i, None] * z2, u)
        return _to_slots(c, A), _signal(c, _apply(c, A, z1)), _signal(c, yt)
    q, k, v, dy = (_units(c, t) for t in xs)
    scale = 1.0 / math.sqrt(q.shape[1])
    A = _scores(c, q, k, scale).softmax(1)
    out = [_signal(c, _apply(c, A, v))]
    if c["op"] == "dense":
        out.append(_to_slots(c, A))
    if c["train"]:
        offs = _offsets(c)
        dA = torch.stack([(dy * _at(v, u).conj()).real.sum(1) for u in offs], 1)
        dS = scale * A * (dA - (A * dA).sum(1, keepdim=True))
        del dA
        dq, dk, dv = torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
        for i, u in enumerate(offs):
            d = dS[:, i, None]
            if c["sim"] == "dot":
                dq += d * _at(k, u)
                dk += _from(d * q, u)
            else:
                t = d * (_at(k, u) - q)
                dq += t
                dk -= _from(t, u)
            dv += _from(A[:, i, None] * dy, u)
        out += [_signal(c, t) for t in (dq, dk, dv)]
    return tuple(out)
