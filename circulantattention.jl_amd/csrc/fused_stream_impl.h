// Streamed split-half kernels: fused circulant attention for windows of any
// width and heads of up to 64 real components, one- and two-dimensional.
//
// Arithmetic.  As in fused2h_impl.h every Float32 operand x is carried as two
// halves, x = hi + lo with hi = f16(x), lo = f16(x - hi), and a product a.b is
// taken as hi.hi + lo.hi + hi.lo on v_mfma_f32_16x16x32_f16 with Float32
// accumulation: 48 cycles for a 16x16 block over 32 components, where
// v_mfma_f32_16x16x4f32 takes 256.
//
// Decomposition.  fused2h_impl.h keeps an item's whole halo in LDS and unrolls
// the walk over its window, which fits a few (window, components) pairs.  Here
// the halo passes through LDS in chunks of 4 pixel columns, all rows of the
// tile's halo at a time, and the window is a run-time value, so any window
// fits.  A wavefront holds 4x4 register pixels (16x1 in one dimension) and
// walks the 4x4 (16x1) LDS blocks of a chunk that its windows meet, two blocks
// at a time.  4x4 blocks on 4x4 pixels waste the least for a general window
// (9 blocks for ws 9 and 25 for ws 15 or 17, where 8x2 pixels and 2x8 blocks
// take 16, 22 and 36), and keep every wavefront's blocks aligned to chunks of
// 4 columns.  A workgroup is NWH x NWW wavefronts over a (4 NWH) x (4 NWW)
// tile, tall rather than square: the wavefronts of a tall tile are active in
// nearly all of its chunks.  The next chunk's (or item's) global loads are
// issued into registers before the current chunk's walk.
//
// LDS layout.  A slot holds a pixel of both staged tensors,
// [t0: 64 NT bytes | t1: 64 NT bytes | 32 bytes of pad], each tensor its
// 32-component groups as [32 hi | 32 lo] halves and a last odd group of 16 as
// [16 hi | 16 lo].  gfx950 serves a ds_read_b128 in groups of 16 lanes that
// are not consecutive, {0-3, 12-15, 20-27}, {4-11, 16-19, 28-31} and the same
// plus 32, and ds_read_b64_tr_b16 in two groups of 32 (measured: pairs of
// lanes on one bank, all others on one address).  With a slot stride of
// 8 NT + 2 units of 16 bytes and CR = 4 mod 8 slots per column every row read
// and every transposing read of a block is free of bank conflicts under those
// groups.
//
// What bounds it.  The walk's issue of matrix-core and vector instructions,
// which add up on a SIMD (a 16x16 block of 32 components: 6 MFMA at 16 cycles
// in the forward and some 100 cycles of exponentials, splits and sums), is half
// of the time; the rest is the staging that the walks of one workgroup do not
// overlap: its loads (the texture path, 14 cycles per 256 bytes), its splits
// and two barriers per chunk.  Larger tiles stage less per pixel: the shape is
// the largest that the image fills.  Measured against the Float32 run-time
// window kernels of fused_impl.h (forward / query- / key-centric pass, us):
// 512x512, 32 components, Distance, ws 31: 751 / 952 / 1136 -> 300 / 410 / 580;
// 131x101, 48 components, 2 heads, B = 2, ws 9: 179 / 262 / 314 -> 33 / 38 / 45;
// 128x96, 64 components, B = 2, ws 15, forward: 102 -> 40; a line of 30011, 64
// components, B = 4, ws 31: 135 / 354 / 490 -> 38 / 48 / 56; 150x170, 8
// components, B = 4, ws 9: 51 / 58 / 74 -> 32 / 37 / 46.
//
// Range.  Staged tensors carry one power-of-two shift for the item so far (the
// accumulators follow its changes), register operands one for the wavefront, as the f16 halves would lose Float32's range.  Values
// that a common shift cannot carry (infinities, NaN, outliers and masks of
// extreme magnitude beside ordinary pixels) send the wavefront's pixels to
// plain_item, which forms them from Float32 products one pixel at a time.
#pragma once
#include "fused2h_impl.h"

// keeps the compiler from hoisting the next block's LDS reads (and their
// registers) into the current one
#define FST_FENCE() __builtin_amdgcn_sched_barrier(0)

namespace circatt {
namespace fst {

using f2d::f4;
using f2d::gmax;
using f2d::gsum;
using f2d::kLn2;
using f2d::kLog2e;
using f2h::cat;
using f2h::h2;
using f2h::h4;
using f2h::h8;
using f2h::ldtr;
using f2h::mfmah;
using f2h::split2;
using f2h::split4;
typedef float f2 __attribute__((ext_vector_type(2)));
// vectors at any Float32 address
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f2u __attribute__((ext_vector_type(2), aligned(4)));

enum { FWD = 0, BWDQ = 1, BWDKV = 2 };
// Byte offset past every buffer (buffers are shorter than kMaxBytes): loads
// from there give 0
constexpr float kLog2eLo = 1.925963033500e-8f;  // log2(e) - kLog2e
constexpr int kOut = 0x7fffff00, kMaxBytes = 0x7ffffe00;
enum { PLANAR = 0, PLANAR_C = 1, LAST = 2 };  // layouts of the signals

struct Args {
    const float *q, *k, *v, *y, *dy, *lse;
    float *yout, *lse_out, *dq, *dk, *dv, *dbuf;
    int n1, n2, P;          // image, pixels
    int ncr, ncrall;        // real components per head, per pixel (all heads)
    int lay, nheads;
    int unit_stride;        // floats per unit (planar)
    float scale, c2;        // similarity scale, scale * log2(e)
    int p;                  // half window
    int pe;                 // exponent PE of the backward's probabilities
    int fine;               // products include lo.lo (small windows, below)
    int nk;                 // LDS blocks per wavefront along a dimension
    int hr, cr;             // staged rows, LDS column stride (slots)
    int cbc, nchunk;        // block columns per chunk, chunks per item (1, 1 in 1D)
    int npx, wt;            // staged pixels per chunk, wave tasks per chunk
    int os;                 // byte offset of the per-slot scalars
    int om;                 // byte offset of the window masks
    int ox;                 // byte offset of the exchange words
    int tiles_h, tiles_w, nitems, per_xcd;
    FastDiv div_tiles, div_th, div_nh, div_hr;
};

template <int NT>
constexpr int slot_bytes() { return 128 * NT + 32; }
// byte offset in a tensor's part of a slot of the hi halves of components
// 16 h .. 16 h + 15, and from them to the lo halves
template <int NT>
constexpr int hi_off(int h) { return 128 * (h >> 1) + ((NT & 1) && h == NT - 1 ? 0 : 32 * (h & 1)); }
template <int NT>
constexpr int lo_step(int h) { return (NT & 1) && h == NT - 1 ? 32 : 64; }

// exchange words, (item << 9) | value: largest exponents of what the item has
// staged so far (tensor 0, centred; tensor 1), 255 - the smallest non-zero
// exponent of either tensor, the largest exponent of tensor 0 before centring
// (Distance) and of the staged D (key-centric pass)
enum { XE0 = 0, XE1 = 1, XM0 = 2, XM1 = 3, XR0 = 4, XD = 5, NXW = 8 };

// One pass over a wavefront's register pixels in Float32, the reference's
// formulas as they stand: lane c holds component c, one pixel and one window
// offset at a time.
template <bool DIST, int MODE, bool ONE>
__device__ __forceinline__ void plain_item(const Args &a, int64_t uoff, int64_t soff, int row0, int col0) {
    const int lane = threadIdx.x & 63;
    const bool on = lane < a.ncr;
    auto at = [&](const float *t, int pix) {
        const int o = a.lay == LAST     ? pix * a.ncrall + lane
                      : a.lay == PLANAR ? pix + a.P * lane
                                        : 2 * pix + 2 * a.P * (lane >> 1) + (lane & 1);
        return on ? t[uoff + o] : 0.f;
    };
    auto put = [&](float *t, int pix, float x) {
        const int o = a.lay == LAST     ? pix * a.ncrall + lane
                      : a.lay == PLANAR ? pix + a.P * lane
                                        : 2 * pix + 2 * a.P * (lane >> 1) + (lane & 1);
        if (on) t[uoff + o] = x;
    };
    auto wsum = [](float x) {
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) x += __shfl_xor(x, d);
        return x;
    };
    auto score = [&](float x, float y) {
        const float d = x - y;
        return DIST ? -0.5f * wsum(d * d) : wsum(x * y);
    };
    const int p2 = ONE ? 0 : a.p;
    for (int i = 0; i < 16; ++i) {
        const int r = row0 + (ONE ? i : i & 3), c = col0 + (ONE ? 0 : i >> 2);
        if (r >= a.n1 || c >= a.n2) continue;
        const int pix = r + a.n1 * c;
        const float x0 = at(MODE == BWDKV ? a.k : a.q, pix);
        const float xs = DIST ? x0 : x0 * a.scale;  // (scaled first: no overflow the tiled kernels do not have)
        float x1 = 0.f, D = 0.f, L = 0.f;
        if constexpr (MODE == BWDQ) {
            x1 = at(a.dy, pix);
            D = wsum(x1 * at(a.y, pix));
            L = a.lse[soff + pix];
        }
        if constexpr (MODE == BWDKV) x1 = at(a.v, pix);
        float m = -INFINITY, l = 0.f, o0 = 0.f, o1 = 0.f;
        for (int d2 = -p2; d2 <= p2; ++d2)
            for (int d1 = -a.p; d1 <= a.p; ++d1) {
                const int op = pmod(r + d1, a.n1) + a.n1 * (ONE ? 0 : pmod(c + d2, a.n2));
                const float y0 = at(MODE == BWDKV ? a.q : a.k, op);
                const float y1 = at(MODE == BWDKV ? a.dy : a.v, op);
                const float s = (DIST ? a.scale : 1.f) * score(xs, y0);
                if constexpr (MODE == FWD) {
                    if (s == -INFINITY) continue;
                    if (!(s <= m)) {
                        const float f = m == -INFINITY ? 0.f : expf(m - s);
                        l *= f;
                        o0 *= f;
                        m = s;
                    }
                    const float e = expf(s - m);
                    l += e;
                    o0 += e * y1;
                } else {
                    if constexpr (MODE == BWDKV) {
                        L = a.lse[soff + op];
                        D = a.dbuf[soff + op];
                    }
                    const float e = expf(s - L);
                    const float ds = e * (wsum(x1 * y1) - D);
                    o0 += ds * (DIST ? y0 - x0 : y0);
                    if constexpr (MODE == BWDKV) o1 += e * y1;
                }
            }
        if constexpr (MODE == FWD) {
            put(a.yout, pix, o0 / l);
            if (lane == 0) a.lse_out[soff + pix] = m + logf(l);
        } else {
            put(MODE == BWDQ ? a.dq : a.dk, pix, a.scale * o0);
            if constexpr (MODE == BWDKV) put(a.dv, pix, o1);
            if constexpr (MODE == BWDQ)
                if (lane == 0) a.dbuf[soff + pix] = D;
        }
    }
}

// largest magnitude, NaN if any value is (v_maximum3_f32), and its biased
// exponent (255 for infinities and NaN)
template <int N>
__device__ __forceinline__ float maxabs(const float (&x)[N], float m = 0.f) {
#pragma unroll
    for (int i = 0; i < N; i += 2)
        m = __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, __builtin_fabsf(x[i])),
                                          __builtin_fabsf(x[i + 1]));
    return m;
}
__device__ __forceinline__ unsigned bexp(float m) { return (__float_as_uint(m) >> 23) & 255u; }
// maximum over the wave, in an SGPR
__device__ __forceinline__ unsigned wave_max(unsigned u) {
    return __builtin_amdgcn_readlane(f2h::wave_umax63(u), 63);
}

// NT: 16-component groups per pixel; T: wave tasks per wavefront and chunk;
// CL: channels-last signals (planar: real or complex, a run-time choice of
// scalar strides)
template <int NT, int NWH, int NWW, int T, int EU, bool DIST, int MODE, bool ONE, bool CL>
__global__ __launch_bounds__(64 * NWH * NWW, EU) void kernel_stream(Args a) {
    constexpr int NW = NWH * NWW;
    constexpr int SB = slot_bytes<NT>();
    constexpr int T1 = 64 * NT;             // tensor 1's part of a slot
    constexpr int NG = (NT + 1) / 2;        // 32-component groups (the last may be a 16)
    constexpr bool ODD = NT & 1;
    constexpr int NTP = NT == 1 ? 1 : NT == 2 ? 2 : 4;  // lanes per staged pixel
    constexpr int PXW = 64 / NTP;           // staged pixels per wave task
    constexpr int RB = ONE ? 16 : 4;        // rows of a block
    constexpr bool KV = MODE == BWDKV;
    // Backward: probabilities are formed as pt = 2^PE p / rho (below), large
    // enough for their halves, and dS' = 2^-DE pt (dP' - D').  The staged
    // tensor 1 and its register partner stay under 2^3, so
    // |dS'| < 2^(PE + 1 - DE) * 2 * 16 NT * 2^6 <= 2^15.
    constexpr int DSE = NT == 1 ? 3 : NT == 2 ? 2 : 1;  // PE - DE
    const int PE = a.pe;
    const float DEf = __builtin_amdgcn_ldexpf(1.f, DSE - PE);
    constexpr unsigned HI1 = MODE == FWD ? 131u : 129u;
    char *const lds = reinterpret_cast<char *>(circatt_lds2);
    unsigned *const xw = reinterpret_cast<unsigned *>(lds + a.ox);
    float *const sc0 = reinterpret_cast<float *>(lds + a.os);
    float *const sc1 = sc0 + (ONE ? 1 : 4 * a.cbc) * a.cr;

    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wh = wv % NWH, ww = wv / NWH;
    const int j = lane & 15, g = lane >> 4;
    const int jr = ONE ? j : j & 3, jc = ONE ? 0 : j >> 2;

    // score rows: element j of a block, halves 8 g .. 8 g + 7 of a 32-half run
    const char *const pA = lds + (RB * wh + jr + a.cr * jc) * SB + 16 * g;
    // apply rows by transposing reads: lane j of group g addresses components
    // 4 (j & 3) .. + 3 of element 4 g + (j >> 2): row j >> 2 of column g, or
    // row 4 g + (j >> 2) in one dimension
    const char *const pR =
        lds + (RB * wh + (j >> 2) + (ONE ? 4 * g : a.cr * g)) * SB + 8 * (j & 3);
    // scalars of elements 4 g .. 4 g + 3 (adjacent rows)
    const float *const pS0 = sc0 + RB * wh + (ONE ? 4 * g : a.cr * g);
    const float *const pS1 = sc1 + RB * wh + (ONE ? 4 * g : a.cr * g);

    // Window masks: 0 or -inf for the four elements of a lane's accumulator, per
    // block along the rows, read from a table in LDS and added to the score
    // products' initial accumulators: four full-rate adds and no branch, where
    // lane masks in SGPRs take four half-rate selects and 30 SGPRs.  The row
    // past the last block masks everything (the second block of an odd tail).
    // In 2D the mask along the columns is one value per lane and chunk.
    constexpr int MROW = ONE ? 64 : 4;  // entries per block
    f4 *const mtab = reinterpret_cast<f4 *>(lds + a.om);
    const f4 *const pM = mtab + (ONE ? lane : jr);
    auto inwin = [&](int u) { return u >= 0 && u <= 2 * a.p ? 0.f : -INFINITY; };
    for (int i = threadIdx.x; i < MROW * (a.nk + 1); i += 64 * NW) {
        const int b = i / MROW, e = i % MROW;
        f4 x;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            x[r] = b == a.nk ? -INFINITY : inwin(RB * b + (ONE ? 4 * (e >> 4) : 0) + r - (ONE ? e & 15 : e));
        mtab[i] = x;
    }

    // Components.  Group h covers components 16 h .. 16 h + 15; the last one
    // the head's last 16 (so that every load is in bounds), of which those
    // that earlier groups hold count as 0 on the register side.  A head of
    // fewer than 16 repeats its last component.
    const int last0 = max(a.ncr - 16, 0), lastlo = 16 * NT - max(a.ncr, 16), lasthi = min(a.ncr, 16);
    auto comp_of = [&](int h, int c) { return (h == NT - 1 ? last0 : 16 * h) + c; };
    auto comp_ok = [&](int h, int c) { return h < NT - 1 || (c >= lastlo && c < lasthi); };
    const bool full = a.ncr == 16 * NT;
    // Products of groups of 32 leave out lo.lo, some 2^-24 of a product: less
    // than Float32 sums round over a large window, more than they round over
    // a small one, where it is formed as well
    const bool fine = a.fine != 0;
    const int pm = a.lay == PLANAR_C ? 2 : 1;  // floats between pixels (planar)
    // float offset of component c0 + c from c0's, c0 even (planar)
    const int p1 = a.lay == PLANAR_C ? 1 : a.P;
    auto coff = [&](int c) { return (c >> 1) * 2 * a.P + (c & 1 ? p1 : 0); };

    // ---- staging: wave task wt = wv + NW i stages PXW pixels of tensor
    // wt & 1, one group of 16 components per lane ----
    float pv[T][16], pl[T], pd[T];
    const int th = NT == 1 ? 0 : min(lane / PXW, NT - 1);  // the lane's group
    int srow[T], scol[T];                                  // its pixel in the chunk
    bool sok[T];
#pragma unroll
    for (int i = 0; i < T; ++i) {
        const int px = ((wv + NW * i) >> 1) * PXW + (lane & (PXW - 1));
        const int pc = min(px, a.npx - 1);
        scol[i] = ONE ? 0 : fdiv(pc, a.div_hr);
        srow[i] = pc - scol[i] * a.hr;
        sok[i] = px < a.npx && (NT != 3 || lane < 48);
    }
    const bool bigh = a.n1 >= a.hr + a.p, bigw = a.n2 >= 4 * a.cbc * a.nchunk + a.p;

    auto decode = [&](int item, int &unit, int &h0, int &w0) {
        unit = fdiv(item, a.div_tiles);
        const int tile = item - unit * (a.tiles_h * a.tiles_w);
        const int tw = fdiv(tile, a.div_th);
        h0 = (tile - tw * a.tiles_h) * (RB * NWH);
        w0 = tw * (ONE ? 1 : 4 * NWW);
    };
    auto unit_off = [&](int unit) {
        if constexpr (CL) {
            const int b = fdiv(unit, a.div_nh);
            return (int64_t)b * a.P * a.ncrall + (int64_t)(unit - b * a.nheads) * a.ncr;
        }
        return (int64_t)unit * a.unit_stride;
    };
    // bytes from the unit's first element to the end of its data
    auto unit_len = [&](int unit) {
        if constexpr (CL) {
            const int hd = unit - fdiv(unit, a.div_nh) * a.nheads;
            return (a.P * a.ncrall - hd * a.ncr) * 4;
        }
        return a.unit_stride * 4;
    };

    // (straight-line code: a branch around a load makes the compiler copy the
    // staged registers where the paths meet, after waiting for them)
    auto load_stage = [&](int unit, int h0, int w0, int ch) __attribute__((always_inline)) {
        const int64_t uoff = unit_off(unit), soff = (int64_t)unit * a.P;
        const int len = unit_len(unit);
        // (formed here each time: 16 multiples kept in registers over the
        // walks would spill)
        int pb = a.P * 4, pb1 = a.lay == PLANAR_C ? 4 : a.P * 4;
        asm volatile("" : "+s"(pb), "+s"(pb1));
#pragma unroll
        for (int i = 0; i < T; ++i) {
            const int wt = wv + NW * i;
            const bool t1 = wt & 1;
            const float *const base = t1 ? (KV ? a.dy : a.v) : (KV ? a.q : a.k);
            const auto rs = f2d::rsrc(base + uoff, len);
            int gh = h0 - a.p + srow[i], gw = ONE ? 0 : w0 - a.p + 4 * a.cbc * ch + scol[i];
            if (bigh) {
                gh += gh < 0 ? a.n1 : 0;
                gh -= gh >= a.n1 ? a.n1 : 0;
            } else {
                gh = pmod(gh, a.n1);
            }
            if constexpr (!ONE) {
                if (bigw) {
                    gw += gw < 0 ? a.n2 : 0;
                    gw -= gw >= a.n2 ? a.n2 : 0;
                } else {
                    gw = pmod(gw, a.n2);
                }
            }
            const int gp = gh + a.n1 * gw;
            const bool on = wt < a.wt;  // (an idle task loads nothing)
            const int c0 = comp_of(th, 0);
            if constexpr (CL) {
                const int vo = on ? (gp * a.ncrall + c0) * 4 : kOut;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const f4 x = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(
                                                            rs, vo, 16 * (NT == 1 ? min(c, lasthi / 4 - 1) : c), 0));
#pragma unroll
                    for (int e = 0; e < 4; ++e) pv[i][4 * c + e] = x[e];
                }
            } else {
                const int vo = on ? (pm * gp + coff(c0)) * 4 : kOut;
#pragma unroll
                for (int c = 0; c < 16; ++c) {
                    const int c_ = NT == 1 ? min(c, lasthi - 1) : c;
                    pv[i][c] = f2d::bload(rs, vo, (c_ >> 1) * 2 * pb + (c_ & 1 ? pb1 : 0));
                }
            }
            if constexpr (KV) {
                pl[i] = f2d::bload(f2d::rsrc(a.lse + soff, a.P * 4), on ? gp * 4 : kOut, 0);
                pd[i] = f2d::bload(f2d::rsrc(a.dbuf + soff, a.P * 4), on ? gp * 4 : kOut, 0);
            }
        }
    };
    // register operands: 32-component group G (lane holds components 8 g ..
    // 8 g + 7 of it) or the last 16 of an odd NT (8 (g & 1) .. + 7)
    auto h_of = [&](int G) { return ODD && G == NG - 1 ? NT - 1 : 2 * G + (g >> 1); };
    auto load8 = [&](const float *t, int64_t uoff, int len, int pix, int G, float (&x)[8])
                     __attribute__((always_inline)) {
        const auto rs = f2d::rsrc(t + uoff, len);
        const int h = h_of(G), c8 = 8 * (g & 1), c0 = comp_of(h, c8);
        if constexpr (CL) {
#pragma unroll
            for (int c = 0; c < 8; c += 4) {
                const f4 z = __builtin_bit_cast(
                    f4, __builtin_amdgcn_raw_buffer_load_b128(
                            rs, comp_ok(h, c8 + c) ? (pix * a.ncrall + c0 + c) * 4 : kOut, 0, 0));
#pragma unroll
                for (int e = 0; e < 4; ++e) x[c + e] = z[e];
            }
        } else {
#pragma unroll
            for (int c = 0; c < 8; ++c)
                x[c] = f2d::bload(rs, comp_ok(h, c8 + c) ? (pm * pix + coff(c0) + coff(c)) * 4 : kOut, 0);
        }
    };
    auto load1 = [&](const float *t, int64_t uoff, int len, int pix, int h, int c) {
        const int k_ = comp_of(h, c);
        const int o = CL ? pix * a.ncrall + k_ : pm * pix + coff(k_);
        return f2d::bload(f2d::rsrc(t + uoff, len), comp_ok(h, c) ? o * 4 : kOut, 0);
    };

    auto item_of = [&](int n) {
        const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, nslot = gridDim.x >> 3;
        const int it = xcd * a.per_xcd + slot + n * nslot;
        return it < min(a.nitems, (xcd + 1) * a.per_xcd) ? it : a.nitems;
    };
    int k = 0;
    int item = item_of(0);
    if (item >= a.nitems) return;
    if (threadIdx.x < NXW) xw[threadIdx.x] = 0u;
    int unit, h0, w0;
    decode(item, unit, h0, w0);
    load_stage(unit, h0, w0, 0);
    // Distance: lane 16 h + c holds component (h, c) of k at the tile's first pixel
    const int mh = min(lane >> 4, NT - 1);
    float nmu = 0.f;
    if constexpr (DIST) nmu = load1(a.k, unit_off(unit), unit_len(unit), h0 + a.n1 * w0, mh, lane & 15);
    __syncthreads();  // exchange words cleared

    while (true) {
        const int64_t uoff = unit_off(unit), soff = (int64_t)unit * a.P;
        const int len = unit_len(unit);
        const int rh = h0 + RB * wh + jr, rw = w0 + (ONE ? 0 : 4 * ww + jc);
        const bool rvalid = rh < a.n1 && rw < a.n2;
        const int rpix = rvalid ? rh + a.n1 * rw : 0;
        const unsigned key = (unsigned)k << 9;
        const float cmu = nmu;

        // the wavefront's register operands as halves
        h8 r0h[NG], r0l[NG], r1h[NG], r1l[NG];
        bool plain = false;
        unsigned bq = 0u;
        int sp = 0, sd = 0;
        float rlse = 0.f, rowD = 0.f, sq = 0.f, m = 0.f, rrho = 1.f, ninit = 0.f, fsd = 1.f, kb = 0.f;
        // backward: p = 2^s / 2^lse2 is formed as pt = 2^(s + PE - I)
        // with lse2 = I + f, I whole: p = 2^-PE rho pt, rho = 2^-f in (1/2, 1].  The
        // whole number adds no rounding to the scores, pt is large enough for
        // its halves where p is not, and rho multiplies the row's results
        // (query-centric pass) or its staged dy and D (key-centric pass).
        auto row_split = [&](float lse, float &ipart, float &rho) {
            ipart = floorf(lse * kLog2e);
            rho = __builtin_amdgcn_exp2f(-__builtin_fmaf(lse, kLog2eLo, __builtin_fmaf(lse, kLog2e, -ipart)));
        };
        {
            float x0[NG][8], x1[NG][8], x2[NG][8];
            // register operands: q (k in the key-centric pass) and, in the
            // backward, dy (v); forward: the query's own k
#pragma unroll
            for (int G = 0; G < NG; ++G) {
                load8(KV ? a.k : a.q, uoff, len, rpix, G, x0[G]);
                load8(KV ? a.v : MODE == FWD ? a.k : a.dy, uoff, len, rpix, G, x1[G]);
                if constexpr (MODE == BWDQ) load8(a.y, uoff, len, rpix, G, x2[G]);
            }
            if constexpr (MODE == BWDQ) rlse = f2d::bload(f2d::rsrc(a.lse + soff, a.P * 4), rpix * 4, 0);
            if constexpr (DIST) {
#pragma unroll
                for (int G = 0; G < NG; ++G)
#pragma unroll
                    for (int c = 0; c < 8; ++c) {
                        const float mu = __shfl(cmu, 16 * h_of(G) + 8 * (g & 1) + c);
                        x0[G][c] -= mu;
                        if constexpr (MODE == FWD) x1[G][c] -= mu;
                    }
            }
            // |q - mu|^2 (k in the key-centric pass); forward: reference score m,
            // the query's own pixel as key (always in its window, so l >= 1)
            float mr0 = 0.f, mr1 = 0.f;
#pragma unroll
            for (int G = 0; G < NG; ++G) {
                float s2 = 0.f, dot = 0.f;
#pragma unroll
                for (int c = 0; c < 8; ++c) {
                    if constexpr (DIST) s2 += x0[G][c] * x0[G][c];
                    if constexpr (MODE == FWD) dot += DIST ? x1[G][c] * (x0[G][c] - 0.5f * x1[G][c]) : x0[G][c] * x1[G][c];
                }
                mr0 = maxabs(x0[G], mr0);
                if constexpr (MODE != FWD) mr1 = maxabs(x1[G], mr1);
                const bool twice = ODD && G == NG - 1 && g >= 2;
                sq += twice ? 0.f : s2;
                m += twice ? 0.f : dot;
            }
            if constexpr (DIST) sq = gsum(sq);
            if constexpr (MODE == FWD) m = gsum(m) * a.c2;
            // q' = q c2 2^sp with one shift for the wavefront (0 for magnitudes in
            // [2^-2, 2^5)); a non-finite register operand goes the plain way
            bq = wave_max(bexp(mr0 * a.c2));
            plain |= bq == 255u;
            sp = bq == 0u ? 0 : max(-100, min(100, f2h::shift_of(bq)));
            auto rsplit = [&](const float (&x)[8], float sc, h8 &hi, h8 &lo) { f2h::reg_split(x, sc, hi, lo); };
#pragma unroll
            for (int G = 0; G < NG; ++G) rsplit(x0[G], __builtin_amdgcn_ldexpf(a.c2, sp), r0h[G], r0l[G]);
            // sd: shift of the register dy (per pixel) or v (one for the wavefront)
            if constexpr (MODE == BWDQ) {
                float dd = 0.f;
#pragma unroll
                for (int G = 0; G < NG; ++G) {
                    float d = 0.f;
#pragma unroll
                    for (int c = 0; c < 8; ++c) d += x1[G][c] * x2[G][c];
                    dd += ODD && G == NG - 1 && g >= 2 ? 0.f : d;  // (held twice)
                }
                rowD = gsum(dd);
                const unsigned b = bexp(gmax(mr1));
                plain |= __builtin_amdgcn_ballot_w64(bexp(mr1) == 255u || !(fabsf(rowD) < INFINITY) || !(fabsf(rlse) < INFINITY)) != 0;
                sd = b == 0u ? 0 : max(-100, min(100, 129 - (int)b));
#pragma unroll
                for (int G = 0; G < NG; ++G) rsplit(x1[G], __builtin_amdgcn_ldexpf(1.f, sd), r1h[G], r1l[G]);
            }
            if constexpr (KV) {
                const unsigned b = wave_max(bexp(mr1));
                plain |= b == 255u;
                sd = b == 0u ? 0 : max(-100, min(100, 129 - (int)b));
#pragma unroll
                for (int G = 0; G < NG; ++G) rsplit(x1[G], __builtin_amdgcn_ldexpf(1.f, sd), r1h[G], r1l[G]);
            }
            if constexpr (MODE == BWDQ) {
                float I;
                row_split(rlse, I, rrho);
                ninit = PE - I - (DIST ? 0.5f * a.c2 * sq : 0.f);
            }
            fsd = KV ? __builtin_amdgcn_ldexpf(1.f, sd) : 1.f;
            kb = KV && DIST ? -0.5f * a.c2 * sq : 0.f;
        }
        f4 acc0[NT], acc1[NT];
#pragma unroll
        for (int h = 0; h < NT; ++h) acc0[h] = acc1[h] = f4{0.f, 0.f, 0.f, 0.f};
        float lsum = 0.f, corr = 0.f;
        int s0 = 0, s1 = 0;
        int xunit = unit, xh0 = h0, xw0 = w0;
        const int nitem = item_of(k + 1);
        const bool has_next = nitem < a.nitems;

        for (int ch = 0; ch < a.nchunk; ++ch) {
            // largest and smallest exponents of what this chunk stages.  The
            // ballots settle the ordinary case; a wave whose values lie
            // outside it reduces them
            bool skew = false;
#pragma unroll
            for (int i = 0; i < T; ++i) {
                const int wt = wv + NW * i;
                if (wt >= a.wt) continue;
                const bool t1 = wt & 1;
                unsigned eraw = 0u;
                FST_FENCE();
                if constexpr (DIST) {
                    if (!t1) {
                        eraw = bexp(maxabs(pv[i]));
#pragma unroll
                        for (int c = 0; c < 16; ++c) pv[i][c] -= __shfl(cmu, 16 * th + c);
                        if (!full) {
#pragma unroll
                            for (int c = 0; c < 16; ++c) pv[i][c] = comp_ok(th, c) ? pv[i][c] : 0.f;
                        }
                    }
                }
                if constexpr (KV) {
                    bool bad = !(fabsf(pl[i]) < INFINITY);
                    if (t1) {
                        float I, rho;
                        row_split(pl[i], I, rho);
                        bad |= !(fabsf(pd[i]) < INFINITY);
                        pd[i] *= rho;
                        const unsigned ed = wave_max(bexp(pd[i]));
                        if (lane == 0)
                            __hip_atomic_fetch_max(xw + XD, key | ed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
#pragma unroll
                        for (int c = 0; c < 16; ++c) pv[i][c] *= rho;
                    }
                    skew |= __builtin_amdgcn_ballot_w64(bad) != 0;
                }
                const unsigned e = bexp(maxabs(pv[i]));
                if constexpr (!DIST) eraw = e;
                if (t1) eraw = e;
                const unsigned top = t1 ? HI1 : 131u;
                const bool odd = __builtin_amdgcn_ballot_w64(e > top || eraw > 138u || (eraw != 0u && eraw < 122u)) != 0 ||
                                 __builtin_amdgcn_ballot_w64(e >= 125u) == 0;
                unsigned em = 128u, el = 0u, er = 0u;
                if (odd) {
                    em = wave_max(e);
                    er = wave_max(eraw);
                    el = wave_max(eraw == 0u ? 0u : 255u - eraw);
                }
                if (lane == 0) {
                    __hip_atomic_fetch_max(xw + (t1 ? XE1 : XE0), key | em, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_WORKGROUP);
                    if (odd) {
                        __hip_atomic_fetch_max(xw + (t1 ? XM1 : XM0), key | el, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_WORKGROUP);
                        if (DIST && !t1)
                            __hip_atomic_fetch_max(xw + XR0, key | er, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_WORKGROUP);
                    }
                }
            }
            if constexpr (KV) {
                if (skew && lane == 0)
                    __hip_atomic_fetch_max(xw + XE1, key | 255u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
            __syncthreads();  // the previous chunk's LDS reads are done; maxima in
            auto word = [&](int w) __attribute__((always_inline)) {
                const unsigned x = __builtin_amdgcn_readfirstlane(xw[w]);
                return (x & ~511u) == key ? x & 511u : 0u;
            };
            const unsigned b0 = word(XE0), b1 = word(XE1);
            const unsigned l0 = word(XM0), l1 = word(XM1);
            const unsigned br0 = DIST ? max(b0, word(XR0)) : b0;
            // spread of the pixels' magnitudes (0: not over 2^9), in powers of two
            const int d0 = l0 ? (int)(br0 + l0) - 255 : 0, d1 = l1 ? (int)(b1 + l1) - 255 : 0;
            // A small pixel beside large ones keeps 2^(25 + 2) of its spread
            // with the largest magnitude at [4, 8), and 2^(25 + 12) at
            // [2^12, 2^13), where spread pixels are taken if the products'
            // bounds allow it (all but the backward's tensor 1, whose products
            // become halves again).  What no shift carries goes the plain way:
            // non-finite values and greater spreads, least where scores are large.
            plain |= br0 == 255u || b1 == 255u || d0 > 20 || d1 > (MODE == FWD ? 20 : 14);
            plain |= d0 > 14 && (int)(b0 + bq) - 252 > 12;
            auto shift = [](unsigned b, unsigned hi, bool wide) {
                if (b == 0u || (!wide && b >= 125u && b <= hi)) return 0;
                return max(-100, min(100, (wide ? 139 : 129) - (int)b));
            };
            const int n0 = shift(b0, 131u, d0 > 7), n1s = shift(b1, HI1, MODE == FWD && d1 > 7);
            // the accumulators follow the shifts
            if (ch > 0 && (n0 != s0 || n1s != s1)) {
                const int e1 = n1s - s1, e0 = MODE == FWD ? e1 : e1 + n0 - s0;
#pragma unroll
                for (int h = 0; h < NT; ++h)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        acc0[h][r] = __builtin_amdgcn_ldexpf(acc0[h][r], e0);
                        if constexpr (KV) acc1[h][r] = __builtin_amdgcn_ldexpf(acc1[h][r], e1);
                    }
                if constexpr (DIST && MODE != FWD) corr = __builtin_amdgcn_ldexpf(corr, e1);
            }
            s0 = n0;
            s1 = n1s;

            // split and store
#pragma unroll
            for (int i = 0; i < T; ++i) {
                const int wt = wv + NW * i;
                if (wt >= a.wt) continue;
                const bool t1 = wt & 1;
                const int sh = t1 ? s1 : s0;
                FST_FENCE();
                float q2 = 0.f;
                if constexpr (DIST) {
                    if (!t1) {
#pragma unroll
                        for (int c = 0; c < 16; ++c) q2 += pv[i][c] * pv[i][c];
                        if constexpr (NTP == 2) q2 += __shfl_xor(q2, 32);
                        if constexpr (NTP == 4) {
                            if (NT == 3 && lane >= 48) q2 = 0.f;
                            q2 = gsum(q2);
                        }
                    }
                }
                if (sh != 0) {
#pragma unroll
                    for (int c = 0; c < 16; ++c) pv[i][c] = __builtin_amdgcn_ldexpf(pv[i][c], sh);
                }
                h2 hi[8], lo[8];
#pragma unroll
                for (int c = 0; c < 8; ++c) split2(pv[i][2 * c], pv[i][2 * c + 1], hi[c], lo[c]);
                const int slot = srow[i] + a.cr * scol[i];
                const bool last16 = ODD && th == NT - 1;
                char *const sp_ = lds + slot * SB + (t1 ? T1 : 0) + 128 * (th >> 1) + (last16 ? 0 : 32 * (th & 1));
                char *const sl_ = sp_ + (last16 ? 32 : 64);
                if (sok[i]) {
#pragma unroll
                    for (int c = 0; c < 8; c += 4) {
                        *reinterpret_cast<f4 *>(sp_ + 4 * c) =
                            f4{__builtin_bit_cast(float, hi[c]), __builtin_bit_cast(float, hi[c + 1]),
                               __builtin_bit_cast(float, hi[c + 2]), __builtin_bit_cast(float, hi[c + 3])};
                        *reinterpret_cast<f4 *>(sl_ + 4 * c) =
                            f4{__builtin_bit_cast(float, lo[c]), __builtin_bit_cast(float, lo[c + 1]),
                               __builtin_bit_cast(float, lo[c + 2]), __builtin_bit_cast(float, lo[c + 3])};
                    }
                    if (th == 0) {
                        const int si = srow[i] + a.cr * scol[i];
                        if constexpr (KV) {
                            if (t1) {
                                sc1[si] = -__builtin_amdgcn_ldexpf(pd[i], s1);
                            } else {
                                float I, rho;
                                row_split(pl[i], I, rho);
                                sc0[si] = PE - I - (DIST ? 0.5f * a.c2 * q2 : 0.f);
                            }
                        } else if constexpr (DIST) {
                            if (!t1) sc0[si] = -0.5f * a.c2 * q2;
                        }
                    }
                }
            }
            // D sums over windows that reach past the staged pixels: it is held
            // to the bound that |dP'| has by its operands
            if constexpr (MODE != FWD) {
                const int ed = KV ? (int)word(XD) : (int)wave_max(bexp(rowD));
                const int es = KV ? ed + s1 + sd : (int)wave_max(bexp(__builtin_amdgcn_ldexpf(rowD, sd + s1)));
                plain |= ed != 0 && es - 126 > 10 + (NT > 2 ? 2 : NT - 1);
            }
            __syncthreads();  // chunk staged

            const bool lastch = ch + 1 == a.nchunk;
            if (lastch && has_next) decode(nitem, xunit, xh0, xw0);
            load_stage(xunit, xh0, xw0, lastch ? 0 : ch + 1);
            if constexpr (DIST)
                nmu = load1(a.k, unit_off(xunit), unit_len(xunit), xh0 + a.n1 * xw0, mh, lane & 15);

            const int eu = sp + s0;
            const float nD = MODE == BWDQ ? -__builtin_amdgcn_ldexpf(rowD, sd + s1) : 0.f;

            // score-type product of a block's 16 pixels with the register
            // pixels over all components
            auto score = [&](const char *A, const h8 (&rhi)[NG], const h8 (&rlo)[NG], f4 x) __attribute__((always_inline)) {
#pragma unroll
                for (int G = 0; G < NG; ++G) {
                    const h8 hi = *reinterpret_cast<const h8 *>(A + 128 * G);
                    if (ODD && G == NG - 1) {
                        x = mfmah(hi, rhi[G], x);
                        x = mfmah(hi, rlo[G], x);
                    } else {
                        const h8 lo = *reinterpret_cast<const h8 *>(A + 128 * G + 64);
                        if (fine) x = mfmah(lo, rlo[G], x);
                        x = mfmah(lo, rhi[G], x);
                        x = mfmah(hi, rlo[G], x);
                        x = mfmah(hi, rhi[G], x);
                    }
                }
                return x;
            };
            auto apply = [&](const char *R0, const char *R1, h8 ph, h8 pl_, f4 (&acc)[NT]) __attribute__((always_inline)) {
#pragma unroll
                for (int h = 0; h < NT; ++h) {
                    const h8 vh = cat(ldtr(R0 + hi_off<NT>(h)), ldtr(R1 + hi_off<NT>(h)));
                    const h8 vl = cat(ldtr(R0 + hi_off<NT>(h) + lo_step<NT>(h)),
                                      ldtr(R1 + hi_off<NT>(h) + lo_step<NT>(h)));
                    if (NT == 1 || fine) acc[h] = mfmah(vl, pl_, acc[h]);
                    acc[h] = mfmah(vl, ph, acc[h]);
                    acc[h] = mfmah(vh, pl_, acc[h]);
                    acc[h] = mfmah(vh, ph, acc[h]);
                }
            };
            // EX: scores unscaled by 2^-eu after the product (and, in the
            // backward, held to pt <= 2^(PE + 1))
            auto walk = [&](auto EX, int bc, int cc) __attribute__((always_inline)) {
                constexpr bool ex = decltype(EX)::value;
                const float cw = ONE ? 0.f : inwin(4 * bc + g - jc);
                const int co = ONE ? 0 : 4 * cc * a.cr;  // slots before the block column
#pragma clang loop unroll(disable)
                for (int b = 0; b < a.nk; b += 2) {
                    FST_FENCE();
                    const bool two = b + 1 < a.nk;
                    const int o0 = (co + b * RB) * SB, o1 = two ? o0 + RB * SB : o0;
                    const char *const A0 = pA + o0, *const A1 = pA + o1;
                    const char *const R0 = pR + o0, *const R1 = pR + o1;
                    float p[2][4];
                    f4 x[2];
                    if constexpr (MODE == FWD) {
#pragma unroll
                        for (int u = 0; u < 2; ++u) {
                            const float c = cw - m;
                            f4 in = pM[MROW * (b + u)] + f4{c, c, c, c};
                            if constexpr (DIST) in = in + *reinterpret_cast<const f4 *>(pS0 + co + RB * (u && two ? b + 1 : b));
                            if constexpr (ex) {
                                const f4 z = score(u ? A1 : A0, r0h, r0l, f4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                                for (int r = 0; r < 4; ++r) x[u][r] = __builtin_amdgcn_ldexpf(z[r], -eu) + in[r];
                            } else {
                                x[u] = score(u ? A1 : A0, r0h, r0l, in);
                            }
                        }
                        auto probs = [&]() {
#pragma unroll
                            for (int u = 0; u < 2; ++u)
#pragma unroll
                                for (int r = 0; r < 4; ++r) p[u][r] = __builtin_amdgcn_exp2f(x[u][r]);
                            return ((p[0][0] + p[0][1]) + (p[0][2] + p[0][3])) +
                                   ((p[1][0] + p[1][1]) + (p[1][2] + p[1][3]));
                        };
                        float ps = probs();
                        if (__builtin_amdgcn_ballot_w64(!(ps <= 256.f)) != 0) {
                            // a score more than 8 above m: m becomes the
                            // pair's maximum where that is larger
                            float mx = 0.f;
#pragma unroll
                            for (int u = 0; u < 2; ++u)
#pragma unroll
                                for (int r = 0; r < 4; ++r) mx = fmaxf(mx, x[u][r]);
                            mx = gmax(mx);
                            const float f = __builtin_amdgcn_exp2f(-mx);
                            m += mx;
                            lsum *= f;
#pragma unroll
                            for (int h = 0; h < NT; ++h) acc0[h] = acc0[h] * f4{f, f, f, f};
#pragma unroll
                            for (int u = 0; u < 2; ++u) x[u] = x[u] - f4{mx, mx, mx, mx};
                            ps = probs();
                        }
                        lsum += ps;
                        h4 h0_, l0_, h1_, l1_;
                        split4(p[0], h0_, l0_);
                        split4(p[1], h1_, l1_);
                        apply(R0 + T1, R1 + T1, cat(h0_, h1_), cat(l0_, l1_), acc0);
                    } else {
                        float ds[2][4];
#pragma unroll
                        for (int u = 0; u < 2; ++u) {
                            const int bb = u && two ? b + 1 : b;
                            const float c = cw + (KV ? kb : ninit);
                            f4 in = pM[MROW * (b + u)], dp;
                            if constexpr (KV || DIST) in = in + *reinterpret_cast<const f4 *>(pS0 + co + RB * bb);
                            if constexpr (!KV || DIST || !ONE) in = in + f4{c, c, c, c};
                            if constexpr (KV)
                                dp = *reinterpret_cast<const f4 *>(pS1 + co + RB * bb) * f4{fsd, fsd, fsd, fsd};
                            else
                                dp = f4{nD, nD, nD, nD};
                            if constexpr (ex) {
                                const f4 z = score(u ? A1 : A0, r0h, r0l, f4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                                for (int r = 0; r < 4; ++r)
                                    x[u][r] = fminf(__builtin_amdgcn_ldexpf(z[r], -eu) + in[r], (float)(PE + 1));
                            } else {
                                x[u] = score(u ? A1 : A0, r0h, r0l, in);
                            }
                            dp = score((u ? A1 : A0) + T1, r1h, r1l, dp);
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                p[u][r] = __builtin_amdgcn_exp2f(x[u][r]);
                                ds[u][r] = p[u][r] * (dp[r] * DEf);
                            }
                            if constexpr (DIST) corr += (ds[u][0] + ds[u][1]) + (ds[u][2] + ds[u][3]);
                        }
                        h4 h0_, l0_, h1_, l1_;
                        split4(ds[0], h0_, l0_);
                        split4(ds[1], h1_, l1_);
                        apply(R0, R1, cat(h0_, h1_), cat(l0_, l1_), acc0);
                        if constexpr (KV) {
                            split4(p[0], h0_, l0_);
                            split4(p[1], h1_, l1_);
                            apply(R0 + T1, R1 + T1, cat(h0_, h1_), cat(l0_, l1_), acc1);
                        }
                    }
                }
            };
            const bool ex = eu != 0 || (int)(b0 + bq) - 252 > 17;
            for (int cc = 0; cc < (ONE ? 1 : a.cbc); ++cc) {
                const int bc = ONE ? 0 : ch * a.cbc + cc - ww;
                if (bc < 0 || bc >= (ONE ? 1 : a.nk)) continue;
                if (ex)
                    walk(std::true_type{}, bc, cc);
                else
                    walk(std::false_type{}, bc, cc);
            }
        }

        // ---- results ----
        auto put4 = [&](float *t, int h, const float (&x)[4]) {
            const int c = comp_of(h, 4 * g);
            float *const o = t + uoff;
            if constexpr (CL) {
                if (comp_ok(h, 4 * g)) *reinterpret_cast<f4u *>(o + (int64_t)rpix * a.ncrall + c) = f4u{x[0], x[1], x[2], x[3]};
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (comp_ok(h, 4 * g + r)) o[pm * rpix + coff(c) + coff(r)] = x[r];
            }
        };
        if (plain) {
            plain_item<DIST, MODE, ONE>(a, uoff, soff, h0 + RB * wh, w0 + (ONE ? 0 : 4 * ww));
        } else if constexpr (MODE == FWD) {
            const float l = gsum(lsum);
            float inv = __builtin_amdgcn_rcpf(l);
            inv = __builtin_fmaf(__builtin_fmaf(-l, inv, 1.f), inv, inv);
            if (rvalid) {
#pragma unroll
                for (int h = 0; h < NT; ++h) {
                    float x[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) x[r] = __builtin_amdgcn_ldexpf(acc0[h][r] * inv, -s1);
                    put4(a.yout, h, x);
                }
                if (g == 0) a.lse_out[soff + rpix] = lse_of(m, l, DIST ? 0.5f * sq * a.scale : 0.f);
            }
        } else {
            const float cs = DIST ? gsum(corr) : 0.f;
#pragma unroll
            for (int h = 0; h < NT; ++h) {
                float xk[4], xv[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float v = __builtin_amdgcn_ldexpf(acc0[h][r], -(sd + s1 + s0) - DSE);
                    if constexpr (DIST) {
                        const float reg = load1(KV ? a.k : a.q, uoff, len, rpix, h, 4 * g + r) -
                                          __shfl(cmu, 16 * h + 4 * g + r);
                        v -= __builtin_amdgcn_ldexpf(cs, -(sd + s1) - DSE) * reg;
                    }
                    xk[r] = v * a.scale * rrho;
                    if constexpr (KV) xv[r] = __builtin_amdgcn_ldexpf(acc1[h][r], -s1 - PE);
                }
                if (rvalid) {
                    put4(KV ? a.dk : a.dq, h, xk);
                    if constexpr (KV) put4(a.dv, h, xv);
                }
            }
            if constexpr (MODE == BWDQ)
                if (rvalid && g == 0) a.dbuf[soff + rpix] = rowD;
        }
        if (!has_next) break;
        ++k;
        unit = xunit;
        h0 = xh0;
        w0 = xw0;
    }
}

// Launch shape of a problem; ok = false where it does not fit
struct Shape {
    int nk, hr, cr, cbc, nchunk, npx, wt, os, om, ox, bytes;
    bool ok;
};
template <int NT, int NWH, int NWW, int T, bool DIST, int MODE, bool ONE>
inline Shape shape_of(int p, int cap = (int)f2d::kLdsCap) {
    constexpr int RB = ONE ? 16 : 4, NW = NWH * NWW, NSC = MODE == BWDKV ? 2 : (DIST ? 1 : 0);
    constexpr int PXW = NT == 1 ? 64 : NT == 2 ? 32 : 16;
    constexpr int WH = ONE ? NW : NWH, WW = ONE ? 1 : NWW;
    Shape s{};
    s.nk = 1 + (2 * p + RB - 1) / RB;
    s.hr = RB * (WH + s.nk - 1);
    s.cr = s.hr + ((4 - s.hr % 8) + 8) % 8;
    // the widest chunk of whole block columns that LDS and the wave tasks hold
    const int ncol = ONE ? 1 : WW + s.nk - 1;
    for (s.cbc = ncol; s.cbc >= 1; --s.cbc) {
        const int nc = ONE ? 1 : 4 * s.cbc;
        s.nchunk = (ncol + s.cbc - 1) / s.cbc;
        if (s.cbc > 1 && (ncol + s.cbc - 2) / (s.cbc - 1) == s.nchunk) continue;  // (no fewer chunks than a narrower one)
        s.npx = s.hr * nc;
        s.wt = 2 * ((s.npx + PXW - 1) / PXW);
        s.os = s.cr * nc * slot_bytes<NT>();
        s.om = s.os + NSC * s.cr * nc * 4;
        s.ox = s.om + (ONE ? 64 : 4) * 16 * (s.nk + 1);
        s.bytes = s.ox + NXW * 4;
        if (s.wt <= NW * T && s.bytes <= cap) break;
    }
    s.ok = s.cbc >= 1;
    return s;
}

template <int NT, int NWH, int NWW, int T, int EU, bool DIST, int MODE, bool ONE, bool CL>
hipError_t launch_shape(const Args &a0, const Shape &sh, int nunits, int cus, hipStream_t s) {
    constexpr int WH = ONE ? NWH * NWW : NWH, WW = ONE ? 1 : NWW;
    auto kern = kernel_stream<NT, WH, WW, T, EU, DIST, MODE, ONE, CL>;
    static const hipError_t attr = hipFuncSetAttribute(
        reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)f2d::kLdsCap);
    if (attr != hipSuccess) return attr;
    Args a = a0;
    a.nk = sh.nk; a.hr = sh.hr; a.cr = sh.cr; a.cbc = sh.cbc; a.nchunk = sh.nchunk;
    a.npx = sh.npx; a.wt = sh.wt; a.os = sh.os; a.om = sh.om; a.ox = sh.ox;
    a.tiles_h = (a.n1 + (ONE ? 16 : 4) * WH - 1) / ((ONE ? 16 : 4) * WH);
    a.tiles_w = ONE ? 1 : (a.n2 + 4 * WW - 1) / (4 * WW);
    const int64_t nitems = (int64_t)a.tiles_h * a.tiles_w * nunits;
    if (nitems <= 0 || nitems > (1 << 22)) return hipErrorNotSupported;
    a.nitems = (int)nitems;
    a.per_xcd = (int)((nitems + 7) / 8);
    a.div_tiles = make_fastdiv((uint32_t)(a.tiles_h * a.tiles_w));
    a.div_th = make_fastdiv((uint32_t)a.tiles_h);
    a.div_nh = make_fastdiv((uint32_t)a.nheads);
    a.div_hr = make_fastdiv((uint32_t)a.hr);
    const int per_cu = std::max(1, std::min(4 * EU / (WH * WW), (int)f2d::kLdsCap / sh.bytes));
    int64_t grid = std::min<int64_t>((int64_t)cus * per_cu, 8LL * a.per_xcd);
    grid = std::max<int64_t>(8, grid / 8 * 8);
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(64 * WH * WW), sh.bytes, s, a);
    return hipGetLastError();
}

template <int NT, int MODE, bool DIST, bool ONE, bool CL>
hipError_t dispatch(const Args &a, int nunits, int cus, hipStream_t s) {
    const Shape m = shape_of<NT, 4, 2, 3, DIST, MODE, ONE>(a.p);
    // (two workgroups of 4 wavefronts per CU where half of LDS holds a chunk)
    Shape c = shape_of<NT, 2, 2, 3, DIST, MODE, ONE>(a.p, (int)f2d::kLdsCap / 2);
    if (!c.ok) c = shape_of<NT, 2, 2, 3, DIST, MODE, ONE>(a.p);
    const int64_t px = (int64_t)(ONE ? (a.n1 + 127) / 128 : ((a.n1 + 15) / 16) * ((a.n2 + 7) / 8)) * nunits;
    if constexpr (NT == 1 || (NT == 2 && MODE != BWDKV)) {
        const Shape b = shape_of<NT, 8, 2, 1, DIST, MODE, ONE>(a.p);
        if (!ONE && b.ok && px >= 4LL * cus)
            return launch_shape<NT, 8, 2, 1, 4, DIST, MODE, ONE, CL>(a, b, nunits, cus, s);
    }
    if (m.ok && (px >= cus / 2 || !c.ok)) return launch_shape<NT, 4, 2, 3, 2, DIST, MODE, ONE, CL>(a, m, nunits, cus, s);
    if (c.ok) return launch_shape<NT, 2, 2, 3, 2, DIST, MODE, ONE, CL>(a, c, nunits, cus, s);
    return hipErrorNotSupported;
}
template <int NT, int MODE>
hipError_t dispatch(bool one, bool dist, const Args &a, int nunits, int cus, hipStream_t s) {
#define CIRCATT_FST_CL(D, O)                                                  \
    return a.lay == LAST ? dispatch<NT, MODE, D, O, true>(a, nunits, cus, s)   \
                         : dispatch<NT, MODE, D, O, false>(a, nunits, cus, s);
    if (one) {
        if (dist) CIRCATT_FST_CL(true, true)
        CIRCATT_FST_CL(false, true)
    }
    if (dist) CIRCATT_FST_CL(true, false)
    CIRCATT_FST_CL(false, false)
#undef CIRCATT_FST_CL
}

}  // namespace fst

// one translation unit per mode and group count (fused_stream_*.hip)
#define CIRCATT_FST_DECL(M) \
    hipError_t launch_fst_##M##_1(bool one, bool dist, const fst::Args &a, int nunits, int cus, hipStream_t s); \
    hipError_t launch_fst_##M##_2(bool one, bool dist, const fst::Args &a, int nunits, int cus, hipStream_t s); \
    hipError_t launch_fst_##M##_3(bool one, bool dist, const fst::Args &a, int nunits, int cus, hipStream_t s); \
    hipError_t launch_fst_##M##_4(bool one, bool dist, const fst::Args &a, int nunits, int cus, hipStream_t s);
CIRCATT_FST_DECL(fwd)
CIRCATT_FST_DECL(bwdq)
CIRCATT_FST_DECL(bwdkv)
#undef CIRCATT_FST_DECL
#define CIRCATT_FST_DEF(M, MODE, NT)                                                                       \
    hipError_t launch_fst_##M##_##NT(bool one, bool dist, const fst::Args &a, int nunits, int cus, hipStream_t s) { \
        return fst::dispatch<NT, MODE>(one, dist, a, nunits, cus, s);                                      \
    }

}  // namespace circatt
