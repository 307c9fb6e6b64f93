"""Streamed kernels (csrc/fused_stream_impl.h) against the float64 oracle: the
sizes where they can go wrong.

Component counts that fill no whole group of 16 (the last group then overlaps
the one before, or repeats a component), windows between and past those of the
compile-time-window kernels, images narrower than the window and than a tile,
odd sizes, every layout, and images large enough for each workgroup shape; each
case names the shape that it is there for, and the library is asked which it
takes.  The bar is the repository's (1e-5 forward, 1e-4 gradients, max-norm
relative).  Further tests: channels far smaller than their neighbours, each
held to its own size; magnitudes from 1e-7 to 1e4; one pixel of one tensor
extreme or not finite, which must not disturb a pixel whose window it is not in;
and the error's 2-norm over small and wide windows against a bound derived from
the roundings."""
import ctypes

import numpy as np
import pytest

from conftest import rel_err
from large_scores import abs_err, flash_bounds
from test_gpu_parity import _attention_case, dev, host, seeded, shape_of
from test_gpu_parity import ca  # noqa: F401

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import oracle as O  # noqa: E402
from test_gpu_magnitudes import MAGS, _across_magnitudes  # noqa: E402


def routes(dims, ws, C, B, nh, kind, cplx, last=False):
    """Workgroup shapes (10 H + W wavefronts; 0, 1: other kernels) of the forward
    and the two backward passes."""
    from circulant_attention import _lib as L
    n1, n2 = dims if len(dims) == 2 else (dims[0], 1)
    f = L.lib.circatt_route_fused
    f.argtypes = [ctypes.c_int] * 9 + [ctypes.c_int64, ctypes.c_int]
    return tuple(f(m, kind, 2 if cplx else 1, len(dims), n1, n2, ws, C // nh, nh, nh * B, last) for m in range(3))


# (spatial, ws, C, B, nheads, kind, complex)
CASES = [
    ((37, 21), 9, 48, 1, 1, 0, False), ((16, 8), 9, 24, 2, 1, 1, False),
    ((33, 9), 13, 34, 1, 2, 0, False),      # 17 components: one past a group
    ((20, 17), 9, 33, 1, 1, 1, False),      # 33, planar real, odd
    ((15, 31), 17, 40, 1, 1, 0, False), ((12, 10), 17, 64, 1, 1, 1, False),  # ws > n
    ((5, 3), 9, 48, 1, 1, 0, False), ((1, 40), 9, 64, 1, 1, 0, False),
    ((40, 36), 23, 8, 1, 1, 1, False), ((45, 40), 21, 5, 1, 1, 0, False),
    ((19, 22), 31, 32, 1, 1, 1, False), ((24, 20), 17, 64, 2, 2, 0, False),
    ((29, 18), 7, 56, 1, 1, 0, False), ((29, 18), 5, 64, 1, 1, 1, False),
    ((22, 19), 9, 12, 1, 1, 0, True), ((22, 19), 11, 25, 1, 1, 1, True),
    ((26, 21), 13, 64, 1, 2, 0, True),
    ((700,), 31, 48, 1, 1, 0, False), ((130,), 63, 8, 2, 1, 1, False), ((129,), 63, 20, 1, 1, 0, True),
    ((20,), 31, 64, 1, 1, 1, False),        # ws > n, one dimension
    ((300,), 31, 17, 1, 1, 0, False),
    ((31, 26), 3, 24, 1, 1, 0, False), ((100, 90), 7, 5, 2, 1, 1, False),  # the smallest windows
]
# (..., workgroup shapes of the three passes)
SHAPE_CASES = [
    ((150, 130), 9, 32, 2, 2, 0, False, (42, 42, 42)), ((20000,), 31, 17, 1, 1, 1, False, (42, 42, 42)),
    ((200, 190), 9, 32, 1, 1, 0, False, (82, 82, 82)), ((200, 190), 21, 16, 1, 1, 0, False, (82, 82, 82)),
    ((272, 260), 9, 16, 2, 1, 1, False, (82, 82, 82)), ((200, 190), 17, 8, 1, 1, 0, True, (82, 82, 82)),
    ((193, 190), 23, 32, 1, 1, 0, False, (82, 82, 82)), ((200, 187), 23, 16, 1, 1, 1, True, (82, 82, 82)),
    ((256, 250), 15, 32, 1, 1, 0, False, (82, 82, 82)),  # window 15: past the Float32 tiles' one round
    ((250, 245), 15, 16, 1, 1, 0, True, (82, 82, 82)), ((40, 36), 15, 8, 1, 1, 0, False, (0, 22, 22)),
    ((40, 30), 31, 64, 1, 1, 1, False, (32, 32, 32)), ((500,), 63, 64, 1, 1, 0, False, (42, 42, 32)),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{'x'.join(map(str, c[0]))}-ws{c[1]}-C{c[2]}-B{c[3]}-h{c[4]}-"
                                                     f"{'dist' if c[5] else 'dot'}-{'c32' if c[6] else 'f32'}")
def test_stream_against_oracle(ca, cuda, case):  # noqa: F811
    dims, ws, C, B, nh, kind, cplx = case
    assert min(routes(*case)) >= 22
    _attention_case(ca, cuda, dims, ws, C, B, nh, 700 + C + ws, cplx, kind, materialize=False)


@pytest.mark.parametrize("case", SHAPE_CASES, ids=lambda c: f"{'x'.join(map(str, c[0]))}-ws{c[1]}-C{c[2]}-{c[7]}")
def test_stream_shapes_against_oracle(ca, cuda, case):  # noqa: F811
    dims, ws, C, B, nh, kind, cplx, shapes = case
    assert routes(*case[:7]) == shapes
    _attention_case(ca, cuda, dims, ws, C, B, nh, 700 + C + ws, cplx, kind, materialize=False)


@pytest.mark.parametrize("case", [((36, 30), 23, 16, 1, 1), ((33, 29), 9, 48, 1, 1), ((700,), 31, 64, 1, 1)],
                         ids=lambda c: f"{'x'.join(map(str, c[0]))}-ws{c[1]}-C{c[2]}")
@pytest.mark.parametrize("which", ["v_dy", "q_k", "all"])
@pytest.mark.parametrize("mag", MAGS)
@pytest.mark.parametrize("kind", [0, 1])
def test_stream_across_magnitudes(ca, cuda, case, which, mag, kind):  # noqa: F811
    assert min(routes(*case, kind, False)) >= 22
    _across_magnitudes(ca, cuda, case, which, mag, False, kind, 300)


@pytest.mark.parametrize("dims,ws,C,nh,kind,cplx", [((37, 21), 9, 96, 2, 0, False), ((26, 18), 13, 80, 2, 1, False),
                                                   ((30, 25), 17, 24, 2, 0, True), ((260,), 31, 20, 1, 1, False),
                                                   ((150, 140), 23, 32, 1, 0, False)])  # (workgroups of 16)
def test_stream_channels_last(ca, cuda, dims, ws, C, nh, kind, cplx):  # noqa: F811
    """The layouts carry the same values through the same arithmetic."""
    sim = ca.DistanceSimilarity() if kind else ca.DotSimilarity()
    assert min(routes(dims, ws, C, 2, nh, kind, cplx, True)) >= (82 if dims[0] == 150 else 22)
    xs = [dev(seeded(40 + i, shape_of(dims, C, 2), cplx), cuda) for i in range(4)]
    out = []
    for last in (False, True):
        t = [(x.movedim(1, -1).contiguous() if last else x).clone().requires_grad_(i < 3) for i, x in enumerate(xs)]
        y, _ = ca.circulant_mh_attention(sim, *t[:3], ws, nh, materialize=False, honor_simfun=True,
                                         channels_last=last)
        g = torch.autograd.grad(y, t[:3], t[3])
        out.append([z.movedim(-1, 1) if last else z for z in (y.detach(), *g)])
    for a, b in zip(*out):
        assert torch.equal(a, b.contiguous())


def distance_from(shape, at):
    """Circular distance (the larger axis) of every pixel from one."""
    out = np.zeros(shape, int)
    for d, (n, c) in enumerate(zip(shape, at)):
        i = np.abs(np.arange(n) - c)
        out = np.maximum(out, np.minimum(i, n - i).reshape([-1 if e == d else 1 for e in range(len(shape))]))
    return out


@pytest.mark.parametrize("dims,ws,C,kind", [((40, 37), 9, 64, 0), ((50, 49), 23, 8, 0), ((40, 37), 9, 48, 1),
                                           ((50, 49), 23, 32, 1), ((300,), 31, 64, 0), ((300,), 63, 24, 1)])
@pytest.mark.parametrize("which", range(4), ids=["q", "k", "v", "dy"])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf"), -3.4028234e38, 1e30, 1e6, 3e2])
@pytest.mark.parametrize("first", [True, False], ids=["first", "inside"])
def test_stream_extreme_pixel(ca, cuda, dims, ws, C, kind, which, value, first):  # noqa: F811
    """One pixel of one tensor holds an extreme value in every component: the
    first of a tile (Distance centres on the tile's pixels) or one inside it.
    An output that it does not enter, most of them in tiles that hold it, keeps
    to the usual bar against the oracle (y and dq: at a distance beyond p; dk and
    dv: beyond p for q and dy, beyond 2 p for k and v, whose every query's row
    changes).  The others meet the large-score bar where the value is finite and
    no row's scores all grow with it beyond some 10^3 (a row's log-sum-exp is
    kept in Float32)."""
    sim = ca.DistanceSimilarity() if kind else ca.DotSimilarity()
    assert min(routes(dims, ws, C, 1, 1, kind, False)) >= 22
    shape = shape_of(dims, C, 1)
    at = tuple(n // 32 * 16 + (0 if first else 5) for n in reversed(dims))
    xs = [seeded(60 + i, shape) for i in range(4)]
    plain = [x.copy() for x in xs]
    plain[which][(0, slice(None), *at)] = 0.5
    xs[which][(0, slice(None), *at)] = np.float32(value)
    t = [dev(x, cuda).requires_grad_(i < 3) for i, x in enumerate(xs)]
    y, _ = ca.circulant_mh_attention(sim, *t[:3], ws, 1, materialize=False, honor_simfun=True)
    got = [host(z) for z in (y, *torch.autograd.grad(y, t[:3], t[3]))]
    ref = [O.attention_fwd(kind, *plain[:3], ws, 1)[0], *O.attention_bwd(kind, *plain, ws, 1)]
    dist, p = distance_from(shape[2:], at), ws // 2
    for i, (a, b) in enumerate(zip(got, ref)):
        far = dist > (2 * p if i >= 2 and which in (1, 2) else p)
        assert far.any() and (i >= 2 or (far & (dist <= p + 4)).any())
        assert rel_err(a[0][:, far], b[0][:, far]) < (1e-5 if i == 0 else 1e-4)
    if abs(value) <= 1e6 and (which != 0 or (kind == 0 and value == 3e2)):
        ref = [O.attention_fwd(kind, *xs[:3], ws, 1)[0], *O.attention_bwd(kind, *xs, ws, 1)]
        for a, b, bar in zip(got, ref, flash_bounds(kind, *(x.astype(np.float32) for x in xs), ws, 1, ref)):
            assert abs_err(a, b) <= bar


@pytest.mark.parametrize("dims,ws,C,kind", [((400, 390), 9, 32, 0), ((60000,), 31, 48, 1)])
def test_stream_nan_in_several_items(ca, cuda, dims, ws, C, kind):  # noqa: F811
    """Workgroups of two and more items each, the second pass over some of them:
    NaN in v at scattered pixels."""
    sim = ca.DistanceSimilarity() if kind else ca.DotSimilarity()
    shape = shape_of(dims, C, 1)
    xs = [seeded(70 + i, shape) for i in range(4)]
    spots = np.random.default_rng(7).integers(0, shape[2:], (40, len(dims)))
    t = [dev(x, cuda) for x in xs]
    dist = np.full(shape[2:], 1 << 20)
    for at in spots:
        t[2][(0, slice(None), *map(int, at))] = float("nan")
        dist = np.minimum(dist, distance_from(shape[2:], at))
    t = [x.requires_grad_(i < 3) for i, x in enumerate(t)]
    y, _ = ca.circulant_mh_attention(sim, *t[:3], ws, 1, materialize=False, honor_simfun=True)
    got = [host(z) for z in (y, *torch.autograd.grad(y, t[:3], t[3]))]
    ref = [O.attention_fwd(kind, *xs[:3], ws, 1)[0], *O.attention_bwd(kind, *xs, ws, 1)]
    p = ws // 2
    for i, (a, b) in enumerate(zip(got, ref)):
        far = dist > (2 * p if i >= 2 else p)
        assert rel_err(a[0][:, far], b[0][:, far]) < (1e-5 if i == 0 else 1e-4)
        assert np.isnan(a[0][:, dist == 0]).all() if i < 2 else True


@pytest.mark.parametrize("dims,ws,C", [((60, 50), 9, 48), ((60, 50), 31, 32), ((60, 50), 15, 64), ((2000,), 31, 64)])
def test_stream_error_rms(ca, cuda, dims, ws, C):  # noqa: F811
    """Relative 2-norm errors against 64 bits.  A row's probabilities carry the
    rounding of its log-sum-exp (half an ulp of a number in [4, 8), 2.4e-7 at
    most, 1.4e-7 rms), their own scores' (a few ulps of numbers up to 8 in
    base-2 units) and the products' (what the thirds leave out and their sums,
    2^-24 to 2^-23): 6e-7 bounds their sum."""
    xs = [seeded(80 + i, shape_of(dims, C, 1)) for i in range(4)]
    t = [dev(x, cuda).requires_grad_(i < 3) for i, x in enumerate(xs)]
    y, _ = ca.circulant_mh_attention(ca.DotSimilarity(), *t[:3], ws, 1, materialize=False)
    got = [y, *torch.autograd.grad(y, t[:3], t[3])]
    ref = [O.attention_fwd(O.DOT, *xs[:3], ws, 1)[0], *O.attention_bwd(O.DOT, *xs, ws, 1)]
    for a, b in zip(got, ref):
        a = host(a)
        assert np.linalg.norm(a - b) < 6e-7 * np.linalg.norm(b)


def channel_errors(out, ref):
    """Largest error of each channel over the channel's largest value."""
    e, r = (np.abs(z).max(axis=(0, *range(2, z.ndim))) for z in (out - ref, ref))
    return e / r


# heads of 8 to 64 real components, 1D and 2D, of each workgroup shape; every
# fourth channel of one tensor scaled
@pytest.mark.parametrize("dims,ws,C,nh,kind,cplx", [
    ((37, 29), 9, 64, 1, 0, False), ((33, 26), 15, 48, 1, 1, False), ((40, 36), 23, 32, 1, 0, False),
    ((40, 36), 21, 8, 1, 1, False), ((30, 25), 13, 32, 2, 0, True), ((400,), 31, 64, 1, 0, False)])
@pytest.mark.parametrize("which", ["q", "k", "v", "dy"])
@pytest.mark.parametrize("scale", [1e-3, 1e-6, 1e-8])
def test_stream_small_channels(ca, cuda, dims, ws, C, nh, kind, cplx, which, scale):  # noqa: F811
    """A channel far smaller than its neighbours keeps its own precision: the
    repository's bar holds for every channel of every output, whatever the
    others' size.  (Distance with channels of k scaled: dq = sum dS (k - q), whose
    second term vanishes but for its rounding, is held to its largest channel.)"""
    xs = [seeded(90 + i, shape_of(dims, C, 1), cplx) for i in range(4)]
    i = "qkvdy".index(which) if which != "dy" else 3
    xs[i][:, ::4] *= scale
    xs[i] = xs[i].astype(np.complex64 if cplx else np.float32).astype(xs[i].dtype)
    t = [dev(x, cuda).requires_grad_(j < 3) for j, x in enumerate(xs)]
    sim = ca.DistanceSimilarity() if kind else ca.DotSimilarity()
    y, _ = ca.circulant_mh_attention(sim, *t[:3], ws, nh, materialize=False, honor_simfun=True)
    got = [y, *torch.autograd.grad(y, t[:3], t[3])]
    ref = [O.attention_fwd(kind, *xs[:3], ws, nh)[0], *O.attention_bwd(kind, *xs, ws, nh)]
    for name, bar, a, b in zip("y dq dk dv".split(), (1e-5, 1e-4, 1e-4, 1e-4), got, ref):
        if (kind, which, name) == (1, "k", "dq"):
            assert rel_err(host(a), b) < bar
        else:
            assert channel_errors(host(a), b).max() < bar, name


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("size", [1e2, 1e4])
def test_stream_unbalanced_channels(ca, cuda, kind, size):  # noqa: F811
    """Some channels of q large and of k small by the same factor (Distance:
    both small): scores of the usual size from operands of very unequal ones."""
    dims, ws, C = (38, 30), 15, 64
    xs = [seeded(95 + i, shape_of(dims, C, 1)) for i in range(4)]
    xs[0][:, :8] *= 1 / size if kind else size
    xs[1][:, :8] *= 1 / size
    xs = [x.astype(np.float32).astype(np.float64) for x in xs]
    t = [dev(x, cuda).requires_grad_(j < 3) for j, x in enumerate(xs)]
    sim = ca.DistanceSimilarity() if kind else ca.DotSimilarity()
    y, _ = ca.circulant_mh_attention(sim, *t[:3], ws, 1, materialize=False, honor_simfun=True)
    got = [y, *torch.autograd.grad(y, t[:3], t[3])]
    ref = [O.attention_fwd(kind, *xs[:3], ws, 1)[0], *O.attention_bwd(kind, *xs, ws, 1)]
    # the rounding of y's own sums, as over equal channels (Float32 products: 2e-7)
    assert channel_errors(host(got[0]), ref[0]).max() < 2e-6
    for a, b in zip(got[1:], ref[1:]):
        assert channel_errors(host(a), b).max() < 1e-4


@pytest.mark.parametrize("which", [2, 3], ids=["v", "dy"])
@pytest.mark.parametrize("scale", [1e-36, 1e-30, 1e20])
@pytest.mark.parametrize("dims,ws,C,kind", [((33, 29), 9, 48, 0), ((40, 36), 23, 16, 1)])
def test_stream_ends_of_the_range(ca, cuda, dims, ws, C, kind, which, scale):  # noqa: F811
    """v or dy near the ends of Float32's range: the thirds of the smallest
    values would be subnormal without the staged tensors' power of two."""
    xs = [seeded(97 + i, shape_of(dims, C, 1)) for i in range(4)]
    xs[which] = (xs[which] * scale).astype(np.float32).astype(np.float64)
    t = [dev(x, cuda).requires_grad_(j < 3) for j, x in enumerate(xs)]
    sim = ca.DistanceSimilarity() if kind else ca.DotSimilarity()
    y, _ = ca.circulant_mh_attention(sim, *t[:3], ws, 1, materialize=False, honor_simfun=True)
    got = [y, *torch.autograd.grad(y, t[:3], t[3])]
    ref = [O.attention_fwd(kind, *xs[:3], ws, 1)[0], *O.attention_bwd(kind, *xs, ws, 1)]
    for bar, a, b in zip((1e-5, 1e-4, 1e-4, 1e-4), got, ref):
        assert rel_err(host(a), b) < bar
