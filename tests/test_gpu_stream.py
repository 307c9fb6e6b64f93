"""Streamed split-half kernels (csrc/fused_stream_impl.h) against the float64
oracle: the sizes where they can go wrong.

Component counts that fill no whole group of 16 (the last group then overlaps
the one before, or repeats a component), windows between and past those of the
other split-half kernels, images narrower than the window and than a tile, odd
sizes, every layout, and images large enough for each of the three workgroup
shapes.  The bar is the repository's (1e-5 forward, 1e-4 gradients, max-norm
relative).  A second test puts one extreme pixel into one tensor: values that a
common power-of-two scale cannot carry beside ordinary ones must not disturb
the pixels whose windows do not reach it, and a third holds the backward's
error over small and wide windows to a bound derived from its roundings."""
import numpy as np
import pytest

from conftest import rel_err
from test_gpu_parity import _attention_case, dev, host, seeded, shape_of
from test_gpu_parity import ca  # noqa: F401

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import oracle as O  # noqa: E402

# (spatial, ws, C, B, nheads, kind, complex)
CASES = [
    ((37, 21), 9, 48, 1, 1, 0, False), ((16, 8), 9, 24, 2, 1, 1, False),
    ((33, 9), 13, 34, 1, 2, 0, False),      # 17 components: one past a group
    ((20, 17), 9, 33, 1, 1, 1, False),      # 33, planar real, odd
    ((15, 31), 17, 40, 1, 1, 0, False), ((12, 10), 17, 64, 1, 1, 1, False),  # ws > n
    ((5, 3), 9, 48, 1, 1, 0, False), ((1, 40), 9, 64, 1, 1, 0, False),
    ((40, 36), 23, 8, 1, 1, 1, False), ((45, 40), 21, 5, 1, 1, 0, False),
    ((19, 22), 31, 32, 1, 1, 1, False), ((24, 20), 15, 64, 2, 2, 0, False),
    ((29, 18), 7, 56, 1, 1, 0, False), ((29, 18), 5, 64, 1, 1, 1, False),
    ((22, 19), 9, 12, 1, 1, 0, True), ((22, 19), 11, 25, 1, 1, 1, True),
    ((26, 21), 13, 64, 1, 2, 0, True),
    ((700,), 31, 48, 1, 1, 0, False), ((130,), 63, 8, 2, 1, 1, False), ((129,), 63, 40, 1, 1, 0, True),
    ((20,), 31, 64, 1, 1, 1, False),        # ws > n, one dimension
    ((300,), 31, 17, 1, 1, 0, False),
    ((150, 130), 9, 32, 2, 2, 0, False),    # workgroups of 8 wavefronts
    ((272, 260), 9, 16, 2, 1, 1, False),    # of 16
    ((230, 220), 15, 32, 1, 1, 0, False),   # window 15: images past those of the Float32 tiles
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{'x'.join(map(str, c[0]))}-ws{c[1]}-C{c[2]}-B{c[3]}-h{c[4]}-"
                                                     f"{'dist' if c[5] else 'dot'}-{'c32' if c[6] else 'f32'}")
def test_stream_against_oracle(ca, cuda, case):  # noqa: F811
    dims, ws, C, B, nh, kind, cplx = case
    _attention_case(ca, cuda, dims, ws, C, B, nh, 700 + C + ws, cplx, kind, materialize=False)


@pytest.mark.parametrize("dims,ws,C,nh,kind,cplx", [((37, 21), 9, 96, 2, 0, False), ((26, 18), 13, 80, 2, 1, False),
                                                   ((30, 25), 17, 24, 2, 0, True), ((260,), 31, 20, 1, 1, False)])
def test_stream_channels_last(ca, cuda, dims, ws, C, nh, kind, cplx):  # noqa: F811
    """The layouts carry the same values through the same arithmetic."""
    sim = ca.DistanceSimilarity() if kind else ca.DotSimilarity()
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


@pytest.mark.parametrize("dims,ws,C,kind", [((40, 37), 9, 64, 0), ((45, 37), 23, 8, 0), ((40, 37), 9, 48, 1),
                                           ((300,), 31, 64, 0)])
@pytest.mark.parametrize("which", range(4), ids=["q", "k", "v", "dy"])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf"), -3.4028234e38, 1e30, 1e6])
def test_stream_extreme_pixel(ca, cuda, dims, ws, C, kind, which, value):  # noqa: F811
    """One pixel of one tensor holds an extreme value in every component: the
    outputs of pixels farther than two windows from it (y: its own window; dk
    and dv: a window of queries that each see a window) are those of the same
    inputs with an ordinary value there."""
    sim = ca.DistanceSimilarity() if kind else ca.DotSimilarity()
    shape = shape_of(dims, C, 1)
    xs = [dev(seeded(60 + i, shape), cuda) for i in range(4)]
    at = tuple(n // 2 for n in reversed(dims))
    res = []
    for v in (0.5, value):
        t = [x.clone() for x in xs]
        t[which][(0, slice(None), *at)] = v
        t = [x.requires_grad_(i < 3) for i, x in enumerate(t)]
        y, _ = ca.circulant_mh_attention(sim, *t[:3], ws, 1, materialize=False, honor_simfun=True)
        res.append([y.detach(), *torch.autograd.grad(y, t[:3], t[3])])
    far = torch.zeros(shape[2:], dtype=torch.bool, device=cuda)
    for d, (n, c) in enumerate(zip(shape[2:], at)):
        i = (torch.arange(n, device=cuda) - c).abs()
        view = [1] * len(at)
        view[d] = n
        far |= (torch.minimum(i, n - i) > ws + 4).reshape(view)  # (4: a block's masked pixels)
    for a, b in zip(*res):
        a, b = a[0][:, far], b[0][:, far]
        assert torch.isfinite(b).all()
        # (other scales and the plain products round differently)
        assert rel_err(host(b), host(a)) < 2e-5


@pytest.mark.parametrize("dims,ws,C", [((60, 50), 9, 48), ((60, 50), 31, 32), ((60, 50), 15, 64), ((2000,), 31, 64)])
def test_stream_error_rms(ca, cuda, dims, ws, C):  # noqa: F811
    """Relative 2-norm errors against 64 bits.  A row's probabilities carry the
    rounding of its log-sum-exp (half an ulp of a number in [4, 8), 2.4e-7 at
    most, 1.4e-7 rms), their own scores' (a few ulps of numbers up to 8 in
    base-2 units) and the halves' (2^-24 to 2^-23): 6e-7 bounds their sum."""
    xs = [seeded(80 + i, shape_of(dims, C, 1)) for i in range(4)]
    t = [dev(x, cuda).requires_grad_(i < 3) for i, x in enumerate(xs)]
    y, _ = ca.circulant_mh_attention(ca.DotSimilarity(), *t[:3], ws, 1, materialize=False)
    got = [y, *torch.autograd.grad(y, t[:3], t[3])]
    ref = [O.attention_fwd(O.DOT, *xs[:3], ws, 1)[0], *O.attention_bwd(O.DOT, *xs, ws, 1)]
    for a, b in zip(got, ref):
        a = host(a)
        assert np.linalg.norm(a - b) < 6e-7 * np.linalg.norm(b)
