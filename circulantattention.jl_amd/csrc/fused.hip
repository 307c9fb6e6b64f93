// Host planning and dispatch of the windowed-tile MFMA kernels (kernels in
// fused_impl.h, one translation unit per mode in fused_<mode>.hip).
#include "fused2d_impl.h"
#include "fused2h_impl.h"
#include "fused_impl.h"
#include "fused_stream_impl.h"
#include "fused_wide_impl.h"

namespace circatt {

// ---------------------------------------------------------------------------
// host planning and dispatch
// ---------------------------------------------------------------------------
namespace {

using Plan = FusedPlan;

int device_cus() {
    static int cus[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (cus[dev] == 0) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            n <= 0)
            n = 256;
        cus[dev] = n;
    }
    return cus[dev];
}

Plan make_plan(FusedMode mode, const FusedProblem &pr) {
    Plan pl{};
    FArgs &a = pl.a;
    a.q = pr.q; a.k = pr.k; a.v = pr.v; a.y = pr.y; a.dy = pr.dy; a.lse = pr.lse;
    a.yout = pr.yout; a.lse_out = pr.lse_out; a.dq = pr.dq; a.dk = pr.dk; a.dv = pr.dv;
    a.dbuf = pr.dbuf; a.nz = pr.nz;
    a.g = pr.g;
    a.dh = pr.dh;
    a.ncomp = pr.ncomp;
    a.ncr = pr.dh * pr.ncomp;
    a.unit_stride = pr.g.P * pr.dh * pr.ncomp;
    a.cl = pr.cl;
    a.nheads = pr.nheads;
    a.ncrall = pr.nheads * pr.dh * pr.ncomp;
    a.scale = pr.scale;
    a.c2 = pr.scale * kLog2e;
    pl.nc = a.ncr <= 16 ? 16 : a.ncr <= 32 ? 32 : a.ncr <= 64 ? 64 : 0;
    if (pl.nc == 0) return pl;
    const bool dist = pr.kind == 1;
    const int ntensor = mode == MODE_SIM ? 1 : 2;
    const int nscalar = mode == MODE_BWDKV ? 2 : (dist ? 1 : 0);
    const int ppt = pl.nc * ntensor <= 32 ? 2 : 1;
    // (Distance: nc floats after the halo hold the item's centre)
    a.hg = plan_halo(pr.g.nsp, pr.g.p, pl.nc, ntensor, nscalar, ppt, dist ? pl.nc : 0);
    if (!a.hg.ok) return pl;
    if (pr.g.nsp == 2) {
        a.tiles_h = (pr.g.n1 + 7) / 8;
        a.tiles_w = (pr.g.n2 + 7) / 8;
    } else {
        a.tiles_h = (pr.g.n1 + 63) / 64;
        a.tiles_w = 1;
    }
    pl.lds_bytes = (size_t)a.hg.lds_floats * sizeof(float);
    const int64_t nitems = (int64_t)a.tiles_h * a.tiles_w * pr.nunits;
    if (nitems <= 0 || nitems > INT32_MAX / 2) return pl;
    a.nitems = (int)nitems;
    a.per_xcd = (int)((nitems + 7) / 8);
    // persistent grid: a multiple of 8 workgroups (one run per XCD), at most
    // one workgroup per item of each XCD run
    const int wg_per_cu = (int)std::max<size_t>(1, std::min<size_t>(2, kLdsMax / pl.lds_bytes));
    int64_t grid = (int64_t)device_cus() * wg_per_cu;
    grid = std::min<int64_t>(grid, 8LL * a.per_xcd);
    grid = std::max<int64_t>(8, grid / 8 * 8);
    pl.grid = dim3((unsigned)grid);
    pl.ok = true;
    return pl;
}

// Channel-chunked kernels (fused_wide_impl.h) for heads wider than 64 real
// components.
struct WidePlan {
    FArgs a;
    size_t lds_bytes;
    dim3 grid;
    bool ok;
};

WidePlan make_wide_plan(FusedMode mode, const FusedProblem &pr) {
    WidePlan wp{};
    if (mode == MODE_SIM) return wp;
    const bool dist = pr.kind == 1;
    const int ntensor = mode == MODE_FWD ? 1 : 2;
    const int nscal = mode == MODE_BWDKV ? 2 : (dist ? 1 : 0);
    const wide::Plan w = wide::plan(pr.g.nsp, pr.g.p, ntensor, nscal);
    if (!w.ok) return wp;
    FArgs &a = wp.a;
    a.q = pr.q; a.k = pr.k; a.v = pr.v; a.y = pr.y; a.dy = pr.dy; a.lse = pr.lse;
    a.yout = pr.yout; a.lse_out = pr.lse_out; a.dq = pr.dq; a.dk = pr.dk; a.dv = pr.dv;
    a.dbuf = pr.dbuf;
    a.g = pr.g;
    a.hg = w.hg;
    a.dh = pr.dh;
    a.ncomp = pr.ncomp;
    a.ncr = pr.dh * pr.ncomp;
    a.unit_stride = pr.g.P * pr.dh * pr.ncomp;
    a.cl = pr.cl;
    a.nheads = pr.nheads;
    a.ncrall = pr.nheads * pr.dh * pr.ncomp;
    a.scale = pr.scale;
    a.c2 = pr.scale * kLog2e;
    a.rb = w.rb;
    a.cr = w.cr;
    a.nst = w.nst;
    a.ncc = (a.ncr + wide::CC - 1) / wide::CC;
    a.noc = (a.ncr + wide::OC - 1) / wide::OC;
    if (pr.g.nsp == 2) {
        a.tiles_h = (pr.g.n1 + 7) / 8;
        a.tiles_w = (pr.g.n2 + 7) / 8;
    } else {
        a.tiles_h = (pr.g.n1 + 63) / 64;
        a.tiles_w = 1;
    }
    const int64_t nitems = (int64_t)a.tiles_h * a.tiles_w * pr.nunits;
    if (nitems <= 0 || nitems > INT32_MAX / 2) return wp;
    a.nitems = (int)nitems;
    a.per_xcd = (int)((nitems + 7) / 8);
    int64_t grid = (int64_t)device_cus() * 2;
    grid = std::min<int64_t>(grid, 8LL * a.per_xcd);
    grid = std::max<int64_t>(8, grid / 8 * 8);
    wp.grid = dim3((unsigned)grid);
    wp.lds_bytes = (size_t)w.lds_floats * sizeof(float);
    wp.ok = true;
    return wp;
}

}  // namespace

bool fused_supported(FusedMode mode, const FusedProblem &pr) {
    Plan pl = make_plan(mode, pr);
    return pl.ok || make_wide_plan(mode, pr).ok;
}

// tiles of n x n pixels (runs of n n in one dimension) of all units
int64_t tiles_of(const FusedProblem &pr, int n) {
    const int64_t t = pr.g.nsp == 1 ? (pr.g.n1 + n * n - 1) / (n * n)
                                    : (int64_t)((pr.g.n1 + n - 1) / n) * ((pr.g.n2 + n - 1) / n);
    return t * pr.nunits;
}

// Whether the compile-time-window kernels (fused2d_impl.h, fused2h_impl.h) take a
// shape.
bool takes_f2d(FusedMode mode, const FusedProblem &pr) {
    const int ncr = pr.dh * pr.ncomp;
    if (mode == MODE_SIM || pr.nunits > INT32_MAX) return false;
    const bool split = math_mode() == CIRCATT_MATH_SPLIT_F16;
    // one-dimensional signals: the split-half kernels of the windows they
    // instantiate (no Float32 matrix-core counterpart)
    if (pr.g.nsp == 1)
        return split && f2h::supported1(pr.g.p, ncr) && pr.g.P * ncr * 4 < (int64_t)INT32_MAX;
    if (!f2d::supported(pr.g.nsp, pr.g.p, ncr, pr.g.P)) return false;
    // Window 15 at 32 real components: the streamed kernels (launch_stream), whose
    // errors in the gradients are a quarter of the Float32 tiles' (2.1e-7 against
    // 8.4e-7), from about where their 32x8 tiles and the 16x16 ones fill the CUs once,
    // a little later for complex components, whose planar loads are half as wide.  us,
    // forward / backward, Float32 tiles -> streamed, Dot, Distance: 208x208 (169 tiles of
    // 16x16) 38/102 -> 38/99, 41/108 -> 46/126; 224x224 (196) 49/131 -> 39/102, 53/141 ->
    // 47/129; 256x254 57/146 -> 40/113, 61/154 -> 48/145; 272x256 59/161 -> 68/184, 64/173 ->
    // 85/218; 320x320 87/236 -> 73/192, 91/250 -> 89/244; 4 x 256x254 221/567 -> 149/401,
    // 232/602 -> 178/496; complex: 208x208 34/96 -> 46/115, 37/104 -> 55/141; 240x240 (225)
    // 45/126 -> 47/120, 49/135 -> 56/146; 320x320 77/219 -> 87/221, 84/234 -> 104/273; 4 x
    // 256x254 173/489 -> 168/441, 188/523 -> 201/532.
    return !(split && ncr == 32 && pr.g.p == 7 &&
             10 * tiles_of(pr, 16) >= (pr.ncomp == 2 ? 9 : 7) * device_cus());
}

hipError_t launch_f2d(FusedMode mode, const FusedProblem &pr, hipStream_t s) {
    const int ncr = pr.dh * pr.ncomp;
    const bool one = pr.g.nsp == 1;
    f2d::Args a{};
    a.q = pr.q; a.k = pr.k; a.v = pr.v; a.y = pr.y; a.dy = pr.dy; a.lse = pr.lse;
    a.yout = pr.yout; a.lse_out = pr.lse_out; a.dq = pr.dq; a.dk = pr.dk; a.dv = pr.dv;
    a.dbuf = pr.dbuf;
    a.n1 = pr.g.n1;
    a.n2 = pr.g.n2;
    a.P = (int)pr.g.P;
    a.unit_stride = (int)(pr.g.P * ncr);
    a.cl = pr.cl;
    a.nheads = pr.nheads;
    a.ncrall = pr.nheads * ncr;
    a.scale = pr.scale;
    a.c2 = pr.scale * kLog2e;
    a.nunits = (int)pr.nunits;
    const int nt = ncr / 16;
    const bool cplx = pr.ncomp == 2, dist = pr.kind == 1;
    const int cus = device_cus();
    if (one) {
        if (nt == 1) {
            if (mode == MODE_FWD) return launch_f1h_fwd(pr.g.p, cplx, dist, a, cus, s);
            if (mode == MODE_BWDQ) return launch_f1h_bwdq(pr.g.p, cplx, dist, a, cus, s);
            return launch_f1h_bwdkv(pr.g.p, cplx, dist, a, cus, s);
        }
        if (mode == MODE_FWD) return launch_f1h2_fwd(pr.g.p, cplx, dist, a, cus, s);
        if (mode == MODE_BWDQ) return launch_f1h2_bwdq(pr.g.p, cplx, dist, a, cus, s);
        return launch_f1h2_bwdkv(pr.g.p, cplx, dist, a, cus, s);
    }
    if (nt == 1 && math_mode() == CIRCATT_MATH_SPLIT_F16) {
        hipError_t e = hipErrorNotSupported;
        if (mode == MODE_FWD) e = launch_f2h_fwd(pr.g.p, cplx, dist, a, cus, s);
        if (mode == MODE_BWDQ) e = launch_f2h_bwdq(pr.g.p, cplx, dist, a, cus, s);
        if (mode == MODE_BWDKV) e = launch_f2h_bwdkv(pr.g.p, cplx, dist, a, cus, s);
        if (e != hipErrorNotSupported) return e;
    }
    if (nt == 2 && math_mode() == CIRCATT_MATH_SPLIT_F16) {
        hipError_t e = hipErrorNotSupported;
        if (mode == MODE_FWD) e = launch_f2h2_fwd(pr.g.p, cplx, dist, a, cus, s);
        if (mode == MODE_BWDQ) e = launch_f2h2_bwdq(pr.g.p, cplx, dist, a, cus, s);
        if (mode == MODE_BWDKV) e = launch_f2h2_bwdkv(pr.g.p, cplx, dist, a, cus, s);
        if (e != hipErrorNotSupported) return e;
    }
    switch (mode) {
    case MODE_FWD: return launch_f2d_fwd(pr.g.p, nt, cplx, dist, a, cus, s);
    case MODE_BWDQ: return launch_f2d_bwdq(pr.g.p, nt, cplx, dist, a, cus, s);
    case MODE_BWDKV: return launch_f2d_bwdkv(pr.g.p, nt, cplx, dist, a, cus, s);
    default: return hipErrorNotSupported;
    }
}

// Streamed kernels (fused_stream_impl.h): any window, up to 64 real
// components per head; hipErrorNotSupported otherwise.  Buffer offsets are 32
// bits, and channels-last components are loaded four at a time.
hipError_t launch_stream(FusedMode mode, const FusedProblem &pr, hipStream_t s, int *route = nullptr) {
    const int ncr = pr.dh * pr.ncomp;
    const int64_t all = (int64_t)pr.nheads * ncr;
    if (mode == MODE_SIM || math_mode() != CIRCATT_MATH_SPLIT_F16 || ncr > 64 || pr.nunits > INT32_MAX ||
        pr.g.p < 1 || pr.g.P * (pr.cl ? all : ncr) * 4 >= (int64_t)fst::kMaxBytes || (pr.cl && ncr % 4 != 0))
        return hipErrorNotSupported;
    const int nt = (ncr + 15) / 16;
    // Any window and component count but one case of the forward: window 15 to 16
    // components, which is compiled into the Float32 kernel, on up to two of its 8x8
    // tiles a CU.  us, Float32 -> here, Dot / Distance, 8 components: 128x127 15 -> 19 /
    // 16 -> 23, 2 units 20 -> 20 / 20 -> 24, 3 units 28 -> 26 / 30 -> 31, 256x254 34 -> 28 /
    // 36 -> 33; 4 complex ones: 2 units 19 -> 24 / 21 -> 28, 3 units 28 -> 31 / 30 -> 35.
    // The backward is the more precise here (8 components, ws 13: 2.3e-7 of 2-norm error
    // in dq against 3.5e-7) and 0.66 to 1.4 times the Float32 kernels' time there.  Other
    // small images, both passes, 128x127, 8 components: ws 3 34 -> 30 / 36 -> 34, ws 7 37 ->
    // 39 / 40 -> 41, ws 9 46 -> 34 / 53 -> 38, ws 11 52 -> 52 / 57 -> 60, ws 13 54 -> 53 /
    // 59 -> 60, ws 17 87 -> 62 / 96 -> 74; 12 complex ones, ws 7 50 -> 58 / 55 -> 68, ws 9
    // 78 -> 59 / 84 -> 69; three units of that size, ws 7 67 -> 55 / 71 -> 68, ws 13 106 ->
    // 69 / 116 -> 87.
    if (mode == MODE_FWD && nt == 1 && pr.g.nsp == 2 && pr.g.ws == 15 && tiles_of(pr, 8) <= 2 * device_cus())
        return hipErrorNotSupported;
    fst::Args a{};
    a.q = pr.q; a.k = pr.k; a.v = pr.v; a.y = pr.y; a.dy = pr.dy; a.lse = pr.lse;
    a.yout = pr.yout; a.lse_out = pr.lse_out; a.dq = pr.dq; a.dk = pr.dk; a.dv = pr.dv;
    a.dbuf = pr.dbuf;
    a.n1 = pr.g.n1;
    a.n2 = pr.g.n2;
    a.P = (int)pr.g.P;
    a.ncr = ncr;
    a.ncrall = (int)all;
    a.lay = pr.cl ? fst::LAST : pr.ncomp == 2 ? fst::PLANAR_C : fst::PLANAR;
    a.nheads = pr.nheads;
    a.unit_stride = (int)(pr.g.P * ncr);
    a.scale = pr.scale;
    a.c2 = pr.scale * kLog2e;
    a.p = pr.g.p;
    a.route = route;
    a.pe = 1;
    while (a.pe < 10 && (1 << (a.pe + 1)) < pr.g.K) ++a.pe;
    const bool one = pr.g.nsp == 1, dist = pr.kind == 1;
    const int nu = (int)pr.nunits, cus = device_cus();
#define CIRCATT_FST_MODE(M)                                        \
    switch (nt) {                                                  \
    case 1: return launch_fst_##M##_1(one, dist, a, nu, cus, s);     \
    case 2: return launch_fst_##M##_2(one, dist, a, nu, cus, s);     \
    case 3: return launch_fst_##M##_3(one, dist, a, nu, cus, s);     \
    default: return launch_fst_##M##_4(one, dist, a, nu, cus, s);    \
    }
    if (mode == MODE_FWD) CIRCATT_FST_MODE(fwd)
    if (mode == MODE_BWDQ) CIRCATT_FST_MODE(bwdq)
    CIRCATT_FST_MODE(bwdkv)
#undef CIRCATT_FST_MODE
}

hipError_t launch_fused(FusedMode mode, const FusedProblem &pr, hipStream_t s) {
    if (mode != MODE_SIM) {
        hipError_t e = takes_f2d(mode, pr) ? launch_f2d(mode, pr, s) : hipErrorNotSupported;
        if (e == hipErrorNotSupported) e = launch_stream(mode, pr, s);
        if (e != hipErrorNotSupported) return e;
    }
    Plan pl = make_plan(mode, pr);
    if (!pl.ok) {
        const WidePlan wp = make_wide_plan(mode, pr);
        if (!wp.ok) return hipErrorNotSupported;
        return launch_wide(mode, pr.g.nsp, pr.kind == 1, wp.a, wp.lds_bytes, wp.grid, s);
    }
    const bool dist = pr.kind == 1;
    switch (mode) {
    case MODE_FWD: return launch_fused_fwd(pl, pr.g.nsp, dist, s);
    case MODE_SIM: return launch_fused_sim(pl, pr.g.nsp, dist, s);
    case MODE_BWDQ: return launch_fused_bwdq(pl, pr.g.nsp, dist, s);
    case MODE_BWDKV: return launch_fused_bwdkv(pl, pr.g.nsp, dist, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace circatt

// The kernel that a fused call takes, without a launch: 1 for the compile-time
// windows, 10 H + W for the streamed kernels' workgroups of H x W wavefronts, 0 for
// the general kernels.  For the tests; no part of the C ABI.
extern "C" int circatt_route_fused(int mode, int kind, int ncomp, int nsp, int n1, int n2, int ws, int dh, int nheads,
                                   int64_t nunits, int channels_last) {
    circatt::FusedProblem pr{};
    pr.g = circatt::make_geom(nsp, n1, n2, ws);
    pr.kind = kind;
    pr.ncomp = ncomp;
    pr.dh = dh;
    pr.nunits = nunits;
    pr.nheads = nheads;
    pr.cl = channels_last;
    pr.scale = 1.f;
    const circatt::FusedMode m = mode == 0 ? circatt::MODE_FWD : mode == 1 ? circatt::MODE_BWDQ : circatt::MODE_BWDKV;
    if (circatt::takes_f2d(m, pr)) return 1;
    int route = 0;
    circatt::launch_stream(m, pr, nullptr, &route);
    return route;
}
