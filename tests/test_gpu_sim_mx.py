"""Similarity from scores held in registers (csrc/sim_mx.hip) against the
float64 oracle, at the sizes where it can go wrong: every count of block rows
and column strips, component counts around the groups of 4 and of 16, images as
narrow as the window and the halo (and just below, where another kernel runs),
sizes that fill no whole tile, odd widths (16-byte loads that straddle the
circular wrap), several units.

A dot product of n components is accumulated in float32 in any order: its error
is at most (n + 4) 2^-24 sum |x| |y|; a squared difference rounds three times
and its sum has positive terms: (n + 8) 2^-24 of the value.  A component that is
not finite may reach its own pixel's slots only."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import oracle as O  # noqa: E402

# (spatial, ws, C, nb, complex)
CASES = [
    ((21, 25), 17, 16, 2, False), ((25, 21), 17, 33, 1, False), ((41, 37), 17, 3, 1, False), ((17, 17), 17, 8, 1, False),
    ((37, 41), 19, 18, 1, False), ((47, 46), 21, 7, 1, False), ((60, 52), 23, 40, 1, False), ((50, 49), 25, 16, 1, False),
    ((54, 46), 27, 4, 1, False), ((49, 52), 29, 8, 1, False), ((49, 50), 31, 16, 1, False), ((58, 55), 33, 20, 1, False),
    ((31, 31), 31, 8, 1, False),
    ((30, 27), 17, 1, 2, True), ((45, 41), 17, 17, 1, True), ((36, 41), 21, 8, 1, True), ((52, 46), 23, 3, 1, True), ((52, 55), 31, 10, 1, True),
    # enough workgroups for two query blocks of a wavefront (Distance)
    ((101, 90), 19, 4, 9, False), ((60, 67), 23, 5, 9, False), ((61, 57), 27, 4, 10, False),
    ((58, 60), 33, 2, 10, False), ((90, 101), 21, 2, 9, True),
]


def case_id(c):
    return f"{'x'.join(map(str, c[0]))}-ws{c[1]}-C{c[2]}-nb{c[3]}-{'c32' if c[4] else 'f32'}"


def draw(case):
    dims, ws, C, nb, cplx = case
    rng = np.random.default_rng(300 + ws + C)

    def image():
        z = rng.standard_normal((nb, C, int(np.prod(dims)), 2 if cplx else 1)).astype(np.float32)
        return z.view(np.complex64)[..., 0] if cplx else z[..., 0]
    return image(), image()


def similarity(cuda, kind, x, y, dims, ws, scale):
    from circulant_attention import _functions as F
    from circulant_attention import _lib as L
    nsp, n1, n2 = F.geometry(dims)
    xd, yd = torch.from_numpy(x).to(cuda), torch.from_numpy(y).to(cuda)
    nz = torch.full((x.shape[0], n1 * n2 * ws * ws), float("nan"), device=cuda)
    L.check(L.lib.circatt_similarity(kind, F.dtype_code(xd), nsp, n1, n2, ws, x.shape[1], x.shape[0], scale,
                                     F.ptr(xd), F.ptr(yd), F.ptr(nz), F.stream_ptr(cuda)))
    return nz.cpu().numpy()


@pytest.mark.parametrize("kind", [0, 1], ids=["dot", "dist"])
@pytest.mark.parametrize("case", CASES, ids=case_id)
def test_similarity_against_oracle(cuda, case, kind):
    dims, ws, C, nb, cplx = case
    x, y = draw(case)
    n = C * (2 if cplx else 1)
    ref = O.similarity(kind, x, y, dims, ws, 0.25)
    if kind:
        bound = (n + 8) * 2.0 ** -24 * np.abs(ref)
    else:
        ax, ay = (np.abs(z.view(np.float32)) if cplx else np.abs(z) for z in (x, y))
        ax, ay = (z.reshape(nb, C, -1, n // C).view(np.complex64)[..., 0] if cplx else z for z in (ax, ay))
        bound = (n + 4) * 2.0 ** -24 * O.similarity(0, ax, ay, dims, ws, 0.25)
    out = similarity(cuda, kind, x, y, dims, ws, 0.25)
    assert (np.abs(out - ref) <= bound + 1e-30).all()


@pytest.mark.parametrize("kind", [0, 1], ids=["dot", "dist"])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("case", [((37, 41), 17, 18, 1, False), ((47, 46), 23, 5, 1, False), ((37, 41), 17, 9, 1, True)],
                         ids=case_id)
def test_values_that_are_not_finite(cuda, case, value, kind):
    dims, ws, _, _, cplx = case
    x, y = draw(case)
    clean = similarity(cuda, kind, x, y, dims, ws, 1.0)
    at = x.shape[2] // 3
    y[:, -1, at] = value
    out = similarity(cuda, kind, x, y, dims, ws, 1.0)
    with np.errstate(invalid="ignore"):
        ref = O.similarity(kind, x, y, dims, ws, 1.0)
    meets = np.isin(O.pattern(dims, ws, 1)[1], at + 1)
    assert np.array_equal(out[~meets], clean[~meets])
    assert np.array_equal(np.isnan(out), np.isnan(ref))
    assert np.array_equal(out[np.isinf(ref)], ref[np.isinf(ref)].astype(np.float32))
