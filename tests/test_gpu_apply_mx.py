"""Matrix-core products A x, A' x and the similarity pullback's pair
(csrc/apply_mx.hip) against the float64 oracle, at the sizes where they can go
wrong: component counts around the groups of 16, windows from 7 to past 31,
images as narrow as the window and the halo (and just below, where another
kernel runs), sizes that fill no whole tile, odd widths (16-byte loads that
straddle the circular wrap), x in several chunks, several units and passes.

An output is a sum of K products (the pullback's correction: as many again),
accumulated in float32 in any order: its error is at most
(K + 8) 2^-24 sum |A| |x|, which the oracle forms from the magnitudes.  A
second test puts NaN and infinities into one pixel of x or one row of A: the
outputs that they do not enter keep to the same bound."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import oracle as O  # noqa: E402

# (spatial, ws, C, nb, complex)
CASES = [
    ((37, 41), 17, 32, 1, False), ((41, 37), 17, 16, 2, False), ((31, 33), 31, 17, 1, False),
    ((39, 31), 31, 5, 1, False), ((33, 50), 33, 48, 1, False), ((47, 46), 23, 33, 1, False),
    ((60, 52), 23, 64, 1, False), ((70, 64), 19, 70, 2, False), ((52, 49), 45, 8, 1, False),
    ((40, 44), 21, 8, 1, True), ((45, 41), 17, 9, 1, True), ((64, 62), 31, 25, 1, True),
    ((50, 47), 19, 40, 1, True), ((160, 150), 17, 8, 4, False),
    ((40, 23), 7, 16, 2, False), ((23, 22), 9, 3, 1, False), ((16, 13), 13, 8, 1, True), ((30, 27), 15, 16, 1, False),
    ((700,), 15, 32, 2, False), ((129,), 63, 40, 1, False), ((200,), 31, 9, 1, True), ((79,), 63, 16, 1, False),
    ((5000,), 127, 70, 1, False), ((140000,), 15, 8, 2, False),
    # 256 to 511 tiles of 8 wavefronts, none of 4 (their chunks reach past the image)
    ((195, 43), 27, 8, 4, False), ((512, 31), 17, 32, 2, False), ((145, 29), 19, 8, 8, True),
]


def case_id(c):
    return f"{'x'.join(map(str, c[0]))}-ws{c[1]}-C{c[2]}-nb{c[3]}-{'c32' if c[4] else 'f32'}"


def draw(case):
    dims, ws, C, nb, cplx = case
    rng = np.random.default_rng(900 + ws + C)
    P, K = int(np.prod(dims)), ws ** len(dims)

    def image():
        z = rng.standard_normal((nb, C, P, 2 if cplx else 1)).astype(np.float32)
        return z.view(np.complex64)[..., 0] if cplx else z[..., 0]
    return rng.standard_normal((nb, P * K)).astype(np.float32), image(), image(), P, K


def mags(z):
    """|re|, |im| side by side, so that one product bounds both parts."""
    return np.abs(z.real) + 1j * np.abs(z.imag) if np.iscomplexobj(z) else np.abs(z)


def check(out, ref, bound, ok=None):
    out, ref, bound = (np.ascontiguousarray(z) for z in (out.astype(ref.dtype), ref, bound))
    if np.iscomplexobj(ref):
        out, ref, bound = (z.view(np.float64) for z in (out, ref, bound))
        ok = None if ok is None else np.repeat(ok, 2, axis=-1)
    bad = ~(np.abs(out - ref) <= bound + 1e-30)
    assert not (bad if ok is None else bad & ok).any()


@pytest.mark.parametrize("case", CASES, ids=case_id)
def test_products_against_oracle(cuda, case):
    from circulant_attention import _functions as F
    from circulant_attention import _lib as L
    dims, ws, C, nb, cplx = case
    A, x, y, P, K = draw(case)
    dt = np.complex128 if cplx else np.float64
    u = (K + 8) * 2.0 ** -24
    Ad, xd, yd = (torch.from_numpy(z).to(cuda) for z in (A, x, y))
    fwd, bwd = (O.apply(A, x, dims, ws, tr).astype(dt) for tr in (False, True))
    bf, bb = (O.apply(np.abs(A), mags(x), dims, ws, tr).astype(dt) * u for tr in (False, True))
    check(F.apply_raw(Ad, xd, dims, ws, False).cpu().numpy(), fwd, bf)
    check(F.apply_raw(Ad, xd, dims, ws, True).cpu().numpy(), bwd, bb)
    fy, by = O.apply(A, y, dims, ws).astype(dt), O.apply(np.abs(A), mags(y), dims, ws).astype(dt) * u
    rs, cs = O.rowsum(A, P, K)[:, None], O.colsum(A, dims, ws)[:, None]
    ra, ca = O.rowsum(np.abs(A), P, K)[:, None], O.colsum(np.abs(A), dims, ws)[:, None]
    nsp, n1, n2 = F.geometry(dims)
    for kind, dx, bx, dy, by_ in ((0, fy, by, bwd, bb),
                                  (1, fy - rs * x, by + u * ra * mags(x), bwd - cs * y, bb + u * ca * mags(y))):
        gx, gy = torch.empty_like(xd), torch.empty_like(yd)
        L.check(L.lib.circatt_similarity_bwd(kind, F.dtype_code(xd), nsp, n1, n2, ws, C, nb, 0.5, F.ptr(Ad),
                                             F.ptr(xd), F.ptr(yd), F.ptr(gx), F.ptr(gy), F.stream_ptr(cuda)))
        check(gx.cpu().numpy(), 0.5 * dx, bx)
        check(gy.cpu().numpy(), 0.5 * dy, by_)


@pytest.mark.parametrize("case", [((37, 41), 17, 20, 1, False), ((33, 30), 9, 7, 1, False), ((200,), 31, 9, 1, True)],
                         ids=case_id)
@pytest.mark.parametrize("value", [float("nan"), float("inf"), float("-inf")])
@pytest.mark.parametrize("which", ["x", "A"])
def test_values_outside_a_window_do_not_enter(cuda, case, value, which):
    from circulant_attention import _functions as F
    dims, ws, C, nb, cplx = case
    A, x, _, P, K = draw(case)
    dt = np.complex128 if cplx else np.float64
    touched = np.zeros_like(A), np.zeros((nb, 1, P))
    at = P // 3
    if which == "x":
        x[:, :, at] = value
        touched[0][:], touched[1][:, :, at] = 1, 1
    else:
        A[:, at * K:(at + 1) * K] = value
        touched[0][:, at * K:(at + 1) * K], touched[1][:] = 1, 1
    out0 = [F.apply_raw(*(torch.from_numpy(z).to(cuda) for z in (A, x)), dims, ws, tr).cpu().numpy()
            for tr in (False, True)]
    A, x = np.where(touched[0] * (which == "A") > 0, 0, A), np.where(touched[1] * (which == "x") > 0, 0, x)
    for tr in (False, True):
        ok = O.apply(touched[0], touched[1], dims, ws, tr) == 0
        assert ok.any() and not ok.all()
        ref = O.apply(A, x, dims, ws, tr).astype(dt)
        bound = O.apply(np.abs(A), mags(x), dims, ws, tr).astype(dt) * (K + 8) * 2.0 ** -24
        with np.errstate(invalid="ignore"):
            check(out0[tr], ref, bound, np.broadcast_to(ok, ref.shape))
        assert not np.isfinite(out0[tr][np.broadcast_to(~ok, ref.shape)]).all()
