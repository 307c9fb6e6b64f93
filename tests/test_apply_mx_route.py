"""CPU check of the matrix-core products' rule and plan (csrc/apply_mx.hip):
every call that the rule takes has a plan, for one product (A x, A' x, a
pullback with one output) and for two (a pullback with both).  The plan tries
tiles of 8 wavefronts and, where those are few, of 4, whose shorter columns
leave LDS for wider chunks and may reach further past the halo than the image
is wide."""
import ctypes
import itertools

import pytest


@pytest.fixture(scope="module")
def route():
    from circulant_attention import _lib
    f = _lib.lib.circatt_route_apply_mx
    f.restype = ctypes.c_int
    f.argtypes = [ctypes.c_int] * 6 + [ctypes.c_int64, ctypes.c_int]
    return f


@pytest.mark.parametrize("n1,n2,ws,C,ncomp,nb", [
    (195, 43, 27, 8, 1, 4), (512, 40, 31, 16, 1, 2), (512, 31, 17, 32, 1, 2), (400, 39, 31, 8, 1, 4),
    (512, 24, 17, 32, 1, 4), (145, 29, 19, 16, 2, 8)])
@pytest.mark.parametrize("products", [1, 2])
def test_narrow_images_have_a_plan(route, n1, n2, ws, C, ncomp, nb, products):
    # (256 to 511 tiles of 8 wavefronts, and no chunk that fits for 4)
    assert route(2, n1, n2, ws, C, ncomp, nb, products) > 0


@pytest.mark.parametrize("ws", [7, 9, 11, 15, 17, 19, 23, 27, 31, 33, 45])
def test_every_call_taken_has_a_plan(route, ws):
    sizes = sorted({n for n in (ws, ws + 1, ws + 5, ws + 12, 64, 97, 145, 200, 320, 512) if n >= ws})
    taken = 0
    for n1, n2, C, ncomp, nb, products in itertools.product(sizes, sizes, (1, 8, 16, 17, 32, 48, 64, 70), (1, 2),
                                                            (1, 2, 3, 4, 8, 16), (1, 2)):
        r = route(2, n1, n2, ws, C, ncomp, nb, products)
        assert r >= 0, (n1, n2, C, ncomp, nb, products)
        taken += r > 0
    assert taken


@pytest.mark.parametrize("ws", [15, 31, 63, 127, 511])
def test_every_line_taken_has_a_plan(route, ws):
    taken = 0
    for n, C, ncomp, nb, products in itertools.product(
            (ws, ws + 1, ws + 30, ws + 130, 700, 5000, 65537, 262144), (1, 8, 17, 32, 64, 70), (1, 2), (1, 2, 5, 64),
            (1, 2)):
        r = route(1, n, 1, ws, C, ncomp, nb, products)
        assert r >= 0, (n, C, ncomp, nb, products)
        taken += r > 0
    assert taken


@pytest.mark.parametrize("n1,n2,ws,C,nb,products,taken", [
    # both sides of the lines in matrix values (75, 120 and 170 million), in pixels and in
    # components
    (256, 254, 29, 32, 1, 1, True), (256, 254, 29, 32, 2, 2, False), (256, 254, 31, 64, 4, 1, False),
    (256, 254, 21, 32, 4, 1, True), (256, 254, 23, 32, 4, 1, False), (256, 254, 25, 64, 4, 2, True),
    (256, 254, 33, 32, 4, 1, True), (128, 126, 7, 16, 1, 1, True), (128, 126, 7, 16, 1, 2, True),
    (128, 126, 9, 16, 1, 2, True), (128, 126, 9, 17, 1, 1, False), (200, 180, 9, 16, 1, 1, False),
    (40, 40, 5, 8, 1, 1, False)])
def test_lines_of_the_rule(route, n1, n2, ws, C, nb, products, taken):
    assert (route(2, n1, n2, ws, C, 1, nb, products) > 0) == taken
