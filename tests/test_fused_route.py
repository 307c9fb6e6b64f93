"""CPU check of the fused dispatch (csrc/fused.hip, dispatch() of
csrc/fused_stream_impl.h) for 256 CUs: both sides of each line of its rules, as
the library answers without a launch.  1: compile-time windows; 10 H + W: the
streamed kernels' workgroups of H x W wavefronts; 0: the general kernels."""
import ctypes

import pytest


@pytest.fixture(scope="module")
def route():
    from circulant_attention import _lib
    f = _lib.lib.circatt_route_fused
    f.restype = ctypes.c_int
    f.argtypes = [ctypes.c_int] * 9 + [ctypes.c_int64, ctypes.c_int]
    return lambda n1, n2, ws, dh, units=1, kind=0, ncomp=1, heads=1, last=0: tuple(
        f(m, kind, ncomp, 2 if n2 else 1, n1, n2 or 1, ws, dh, heads, units, last) for m in range(3))


@pytest.mark.parametrize("kw,want", [
    # compile-time windows, and their counts of components
    (dict(n1=256, n2=256, ws=15, dh=16, units=16), (1, 1, 1)), (dict(n1=320, n2=320, ws=11, dh=16, ncomp=2), (1, 1, 1)),
    (dict(n1=262144, n2=0, ws=63, dh=32), (1, 1, 1)), (dict(n1=64, n2=64, ws=9, dh=16), (22, 22, 22)),
    # window 15 at 32: 0.7 (complex 0.9) 16x16 tiles a CU
    (dict(n1=208, n2=208, ws=15, dh=32), (1, 1, 1)), (dict(n1=224, n2=224, ws=15, dh=32), (82, 82, 82)),
    (dict(n1=224, n2=224, ws=15, dh=16, ncomp=2), (1, 1, 1)), (dict(n1=256, n2=240, ws=15, dh=16, ncomp=2), (82, 82, 82)),
    # window 15 to 16 components, forward: two 8x8 tiles a CU
    (dict(n1=128, n2=127, ws=15, dh=8, units=2), (0, 42, 42)), (dict(n1=128, n2=127, ws=15, dh=8, units=3), (82, 82, 82)),
    (dict(n1=128, n2=127, ws=13, dh=8), (22, 22, 22)),
    # 2 x 2 wavefronts to half a round of 4 x 2, 8 x 2 where they save rounds
    (dict(n1=128, n2=128, ws=17, dh=32), (22, 22, 22)), (dict(n1=128, n2=136, ws=17, dh=32), (42, 42, 42)),
    (dict(n1=256, n2=128, ws=17, dh=32), (42, 42, 42)), (dict(n1=272, n2=128, ws=17, dh=32), (82, 82, 82)),
    (dict(n1=256, n2=264, ws=17, dh=32), (42, 42, 42)),
    # (504 tiles of 16x8, but 264 of 32x8)
    (dict(n1=327, n2=94, ws=23, dh=8, units=2), (42, 42, 42)), (dict(n1=272, n2=128, ws=17, dh=48), (42, 42, 42)),
    # LDS: 64 components from some window on by 3 x 2, past 33 not at all
    (dict(n1=512, n2=512, ws=23, dh=64), (42, 42, 42)), (dict(n1=512, n2=512, ws=31, dh=64), (32, 32, 32)),
    (dict(n1=512, n2=512, ws=35, dh=64), (0, 0, 0)), (dict(n1=512, n2=512, ws=77, dh=32, kind=1), (42, 42, 42)),
    (dict(n1=512, n2=512, ws=81, dh=32, kind=1), (0, 0, 0)),
    # more components; channels-last heads of no multiple of 4
    (dict(n1=64, n2=64, ws=9, dh=65), (0, 0, 0)), (dict(n1=64, n2=64, ws=9, dh=24, last=1), (22, 22, 22)),
    (dict(n1=64, n2=64, ws=9, dh=25, last=1), (0, 0, 0))])
def test_lines_of_the_rules(route, kw, want):
    assert route(**kw) == want
