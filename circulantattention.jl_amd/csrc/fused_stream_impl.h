// Streamed kernels: fused circulant attention for windows of any width and
// heads of up to 64 real components, one- and two-dimensional.
//
// Arithmetic.  Every Float32 operand x is carried as three bf16 thirds,
// x = a + b + c with a = bf16(x), b the next 8 bits of x - a, c the rest: the
// sum is exact, as 8 bits each make Float32's 24 and bf16 has its exponents.  A
// product is taken as the six partial products down to 2^-16 of it on
// v_mfma_f32_16x16x32_bf16 with Float32 accumulation; those left out (b.c, c.b,
// c.c) come to 2^-23 of it at most, 2^-26 as a rule, of either sign.  96 cycles for a 16x16 block
// over 32 components, where v_mfma_f32_16x16x4f32 takes 256.  Two f16 halves
// (fused2h_impl.h) take 48, but hold an operand to 2^-25 of the largest one that
// shares its power-of-two scale: a component a thousandth of its neighbours'
// size would come out with five digits, one of 10^-8 as 0.  Thirds need no scale
// and treat every component, pixel and magnitude alike.
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
// [t0: 96 NT bytes | t1: 96 NT bytes | 32 bytes of pad], each tensor its
// 32-component groups as [32 a | 32 b | 32 c] thirds and a last odd group of 16 as
// [16 a | 16 b | 16 c].  gfx950 serves a ds_read_b128 in groups of 16 lanes that
// are not consecutive, {0-3, 12-15, 20-27}, {4-11, 16-19, 28-31} and the same
// plus 32, and ds_read_b64_tr_b16 in two groups of 32 (measured: pairs of
// lanes on one bank, all others on one address).  With a slot stride of
// 12 NT + 2 units of 16 bytes (2 mod 4) and CR = 4 mod 8 slots per column every row
// read and every transposing read of a block falls on distinct banks under those
// groups (tests/test_stream_model.py).
//
// What bounds it.  On large images the issue of vector and matrix-core
// instructions, which add up on a SIMD: 512x512, 32 components, Distance, ws 31,
// forward 0.57 of the time vector and 0.30 matrix-core, query-centric 0.54 and 0.35,
// key-centric 0.54 and 0.37.  Images of one round of workgroups are bound by one
// workgroup's own chain of staging, barriers and walk (0.36 and 0.2 at 2 x 131x101).
// Some kernels spill registers: none of the forward's; the query-centric ones of 16
// wavefronts with planar Distance 11; the key-centric ones of 16 wavefronts 5 to 41, and
// of 48 and 64 components with Distance, or on the 3 x 2 tile, 2 to 49 (512x512 as above
// writes 47 MB for 35 and 115 for 67).  Larger tiles stage less per pixel: see the rule
// at dispatch.  Against the Float32 run-time-window kernels of fused_impl.h (forward /
// query- / key-centric pass, us): 512x512 as above 720 / 911 / 1113 -> 386 / 490 / 623;
// 131x101, 48 components, 2 heads, B = 2, ws 9: 178 / 263 / 314 -> 36 / 43 / 53; 128x96, 64
// components, B = 2, ws 15: 104 / 127 / 145 -> 50 / 57 / 70; a line of 30011, 64 components,
// B = 4, ws 31: 130 / 357 / 493 -> 41 / 48 / 57; 150x170, 8 components, B = 4, ws 9: 49 / 56 /
// 71 -> 29 / 31 / 41.  (Halves took 311 / 396 / 568 in the first, 33 / 38 / 46 in the second.)
//
// Precision.  Relative 2-norm errors against 64 bits on N(0,1) data, y / dq / dk / dv
// in units of 1e-7, Float32 kernels -> these: 512x512 as above 8.2 / 11.6 / 10.6 / 9.6 ->
// 3.7 / 5.7 / 5.3 / 4.7; 131x101 2.7 / 3.5 / 3.4 / 3.3 -> 1.6 / 2.2 / 2.2 / 2.0; 8 components,
// ws 3 0.95 / 1.8 / 1.7 / 1.5 -> 0.87 / 1.6 / 1.5 / 1.3, ws 21 3.2 / 4.6 / 4.3 / 4.2 ->
// 1.9 / 2.8 / 2.6 / 2.4; smaller at every window and component count measured.  Half of
// that comes from forming the smaller partial products from 0 and adding them once
// (into the running sum, 256x254, 32 components, ws 31: 5.2 / 5.5 / 5.3 / 5.3 -> 2.5 / 3.0 /
// 3.0 / 2.8, for 1 to 4% of the time).
//
// Range.  Staged tensors carry a factor 2^24 and the register partner of a dP
// product a power of two per pixel, so that the thirds of small values stay
// normal: magnitudes from 2^-126 to 2^100 are carried exactly.  Anything that is
// not finite on the way (infinities, NaN, masks near the type's lowest value)
// leaves a result that is not finite; the wavefront's pixels are then formed by
// plain_item from Float32 products and their own windows alone.
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
typedef unsigned u4 __attribute__((ext_vector_type(4)));
typedef unsigned u2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
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
    int nk;                 // LDS blocks per wavefront along a dimension
    int hr, cr;             // staged rows, LDS column stride (slots)
    int cbc, nchunk;        // block columns per chunk, chunks per item (1, 1 in 1D)
    int npx, wt;            // staged pixels per chunk, wave tasks per chunk
    int os;                 // byte offset of the per-slot scalars
    int om;                 // byte offset of the window masks
    int oc;                 // byte offset of the Distance centre
    int tiles_h, tiles_w, nitems, per_xcd;
    FastDiv div_tiles, div_th, div_nh, div_hr;
    int *route;             // host only: the shape is written here and nothing launched
};

template <int NT>
constexpr int slot_bytes() { return 192 * NT + 32; }
// byte offset in a tensor's part of a slot of the first thirds of components
// 16 h .. 16 h + 15, and from them to the next thirds
template <int NT>
constexpr int third_off(int h) { return 192 * (h >> 1) + ((NT & 1) && h == NT - 1 ? 0 : 32 * (h & 1)); }
template <int NT>
constexpr int third_step(int h) { return (NT & 1) && h == NT - 1 ? 32 : 64; }

__device__ __forceinline__ f4 mfmab(u4 a, u4 b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), c, 0, 0, 0);
}
// the thirds of two values as packed pairs.  The first is rounded (by one packed
// conversion), so that the rest, and with it what the products leave out, has
// either sign; the others are cut off, which is exact for the last.
__device__ __forceinline__ void split3(float x0, float x1, unsigned &a, unsigned &b, unsigned &c) {
    constexpr unsigned top = 0xffff0000u, sel = 0x07060302u;  // upper halves of two words
    a = __builtin_bit_cast(unsigned, __builtin_convertvector((f2{x0, x1}), bf2));
    const float r0 = x0 - __uint_as_float(a << 16), r1 = x1 - __uint_as_float(a & top);
    b = __builtin_amdgcn_perm(__float_as_uint(r1), __float_as_uint(r0), sel);
    const float s0 = r0 - __uint_as_float(__float_as_uint(r0) & top), s1 = r1 - __uint_as_float(__float_as_uint(r1) & top);
    c = __builtin_amdgcn_perm(__float_as_uint(s1), __float_as_uint(s0), sel);
}
template <int N>
__device__ __forceinline__ void split3(const float (&x)[8], u4 &a, u4 &b, u4 &c) {
    static_assert(N == 8);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        unsigned u, v, w;
        split3(x[2 * i], x[2 * i + 1], u, v, w);
        a[i] = u;
        b[i] = v;
        c[i] = w;
    }
}
// transposing LDS reads of four components in two blocks
__device__ __forceinline__ u4 ldtr2(const char *p0, const char *p1) {
    const u2 x = __builtin_bit_cast(u2, f2h::ldtr(p0)), y = __builtin_bit_cast(u2, f2h::ldtr(p1));
    return u4{x[0], x[1], y[0], y[1]};
}

// Powers of two: of the staged tensors, and of dP' and D' beside the register
// operand's own (below)
constexpr int kUp = 24, kUpP = 12;

// One pass over a wavefront's register pixels in Float32, the reference's
// formulas as they stand: lane j + 16 g holds 4 NT components of pixel j, all
// lanes one window offset at a time.  Slow, and for values that are not finite
// alone: with one in every tile 512x512, 32 components, Distance, ws 31 takes 16.5 / 16.6 /
// 18.3 ms a pass instead of 0.39 / 0.50 / 0.77 (one pixel at a time, a component a
// lane: 54 / 55 / 103 ms), 131x101, 48 components, 4 units, ws 9 0.41 ms instead of 0.04; the
// loads, each 16 runs of 4 pixels, bound it.
template <int NT, bool DIST, int MODE, bool ONE>
__device__ __forceinline__ void plain_item(const Args &a, int64_t uoff, int64_t soff, int row0, int col0) {
    constexpr int N = 4 * NT;
    const int j = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4;
    const int r = row0 + (ONE ? j : j & 3), c = col0 + (ONE ? 0 : j >> 2);
    const bool valid = r < a.n1 && c < a.n2;
    const int pix = valid ? r + a.n1 * c : 0;
    auto off = [&](int px, int i) {
        const int k = N * g + i;
        return a.lay == LAST ? px * a.ncrall + k : a.lay == PLANAR ? px + a.P * k : 2 * px + 2 * a.P * (k >> 1) + (k & 1);
    };
    auto load = [&](const float *t, int px, float (&x)[N]) {
#pragma unroll
        for (int i = 0; i < N; ++i) x[i] = N * g + i < a.ncr ? t[uoff + off(px, i)] : 0.f;
    };
    auto put = [&](float *t, const float (&x)[N], float f) {
#pragma unroll
        for (int i = 0; i < N; ++i)
            if (valid && N * g + i < a.ncr) t[uoff + off(pix, i)] = f * x[i];
    };
    auto dot = [&](const float (&x)[N], const float (&y)[N]) {
        float d = 0.f;
#pragma unroll
        for (int i = 0; i < N; ++i) d += x[i] * y[i];
        return gsum(d);
    };
    float x0[N], x1[N], o0[N], o1[N];
    load(MODE == BWDKV ? a.k : a.q, pix, x0);
    float m = -INFINITY, l = 0.f, D = 0.f, L = 0.f;
    if constexpr (MODE == BWDQ) {
        load(a.y, pix, o0);
        load(a.dy, pix, x1);
        D = dot(x1, o0);
        L = a.lse[soff + pix];
    }
    if constexpr (MODE == BWDKV) load(a.v, pix, x1);
#pragma unroll
    for (int i = 0; i < N; ++i) o0[i] = o1[i] = 0.f;
    const int p2 = ONE ? 0 : a.p, first = pmod(r - a.p, a.n1);
    int c2 = ONE ? 0 : pmod(c - p2, a.n2);
    for (int d2 = 0; d2 <= 2 * p2; ++d2, c2 = c2 + 1 == a.n2 ? 0 : c2 + 1)
        for (int d1 = 0, r2 = first; d1 <= 2 * a.p; ++d1, r2 = r2 + 1 == a.n1 ? 0 : r2 + 1) {
            const int op = r2 + a.n1 * c2;
            float y0[N], y1[N];
            load(MODE == BWDKV ? a.q : a.k, op, y0);
            load(MODE == BWDKV ? a.dy : a.v, op, y1);
            float s = 0.f;
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const float d = x0[i] - y0[i];
                // (scaled before the product: no overflow the tiled kernels do not have)
                s += DIST ? d * d : x0[i] * a.scale * y0[i];
            }
            s = gsum(s) * (DIST ? -0.5f * a.scale : 1.f);
            if constexpr (MODE == FWD) {
                const bool up = !(s <= m), on = s != -INFINITY;
                const float f = !up ? 1.f : m == -INFINITY ? 0.f : expf(m - s);
                if (up) m = s;
                const float e = on ? expf(s - m) : 0.f;
                l = l * f + e;
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    if (up) o0[i] = f == 0.f ? 0.f : o0[i] * f;
                    if (on) o0[i] += e * y1[i];
                }
            } else {
                if constexpr (MODE == BWDKV) {
                    L = a.lse[soff + op];
                    D = a.dbuf[soff + op];
                }
                const float e = expf(__builtin_elementwise_minimum(s - L, 0.f));
                const float ds = e * (dot(x1, y1) - D);
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    o0[i] += ds * (DIST ? y0[i] - x0[i] : y0[i]);
                    if constexpr (MODE == BWDKV) o1[i] += e * y1[i];
                }
            }
        }
    if constexpr (MODE == FWD) {
        put(a.yout, o0, 1.f / l);
        if (valid && g == 0) a.lse_out[soff + pix] = m + logf(l);
    } else {
        put(MODE == BWDQ ? a.dq : a.dk, o0, a.scale);
        if constexpr (MODE == BWDKV) put(a.dv, o1, 1.f);
        if constexpr (MODE == BWDQ)
            if (valid && g == 0) a.dbuf[soff + pix] = D;
    }
}

// largest magnitude and its biased exponent
template <int N>
__device__ __forceinline__ float maxabs(const float (&x)[N], float m = 0.f) {
#pragma unroll
    for (int i = 0; i < N; i += 2)
        m = __builtin_elementwise_maximum(__builtin_elementwise_maximum(m, __builtin_fabsf(x[i])),
                                          __builtin_fabsf(x[i + 1]));
    return m;
}
__device__ __forceinline__ unsigned bexp(float m) { return (__float_as_uint(m) >> 23) & 255u; }
// NT: 16-component groups per pixel; T: wave tasks per wavefront and chunk;
// CL: channels-last signals (planar: real or complex, a run-time choice of
// scalar strides)
template <int NT, int NWH, int NWW, int T, int EU, bool DIST, int MODE, bool ONE, bool CL>
__global__ __launch_bounds__(64 * NWH * NWW, EU) void kernel_stream(Args a) {
    constexpr int NW = NWH * NWW;
    constexpr int SB = slot_bytes<NT>();
    constexpr int T1 = 96 * NT;             // tensor 1's part of a slot
    constexpr int NG = (NT + 1) / 2;        // 32-component groups (the last may be a 16)
    constexpr bool ODD = NT & 1;
    constexpr int NTP = NT == 1 ? 1 : NT == 2 ? 2 : 4;  // lanes per staged pixel
    constexpr int PXW = 64 / NTP;           // staged pixels per wave task
    constexpr int RB = ONE ? 16 : 4;        // rows of a block
    constexpr bool KV = MODE == BWDKV;
    // Loads of the next chunk after the walk instead of before it: the backward
    // passes of 16 wavefronts (128 registers each) would spill 25 to 80 registers
    // around them (512x512, 32 components, Distance, ws 31, query- / key-centric pass
    // 480 / 740 -> 461 / 579 us; without Distance 416 / 574 -> 416 / 536; the forward's fit)
    constexpr bool LATE = MODE != FWD && EU == 4;
    char *const lds = reinterpret_cast<char *>(circatt_lds2);
    float *const cen = reinterpret_cast<float *>(lds + a.oc);
    float *const sc0 = reinterpret_cast<float *>(lds + a.os);
    float *const sc1 = sc0 + (ONE ? 1 : 4 * a.cbc) * a.cr;

    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wh = wv % NWH, ww = wv / NWH;
    const int j = lane & 15, g = lane >> 4;
    const int jr = ONE ? j : j & 3, jc = ONE ? 0 : j >> 2;

    // score rows: element j of a block, thirds 8 g .. 8 g + 7 of a run of 32
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
    bool redo = false;
    int item = item_of(0);
    if (item >= a.nitems) return;
    int unit, h0, w0;
    decode(item, unit, h0, w0);
    load_stage(unit, h0, w0, 0);
    // Distance: lane 16 h + c holds component (h, c) of the item's centre, the
    // median of k at the tile's first, middle and last pixel (one outlying
    // pixel, of whose size the expanded differences would be, does not move it)
    const int mh = min(lane >> 4, NT - 1);
    float nmu = 0.f;
    auto load_centre = [&](int unit, int h0, int w0) {
        constexpr int TH = RB * NWH, TW = ONE ? 1 : 4 * NWW;
        const int hm = min(h0 + TH / 2, a.n1 - 1), wm = ONE ? 0 : min(w0 + TW / 2, a.n2 - 1);
        const int hl = min(h0 + TH - 1, a.n1 - 1), wl = ONE ? 0 : min(w0 + TW - 1, a.n2 - 1);
        auto at = [&](int h, int w) { return load1(a.k, unit_off(unit), unit_len(unit), h + a.n1 * w, mh, lane & 15); };
        return __builtin_amdgcn_fmed3f(at(h0, w0), at(hm, wm), at(hl, wl));
    };
    if constexpr (DIST) nmu = load_centre(unit, h0, w0);

    while (true) {
        const int64_t uoff = unit_off(unit), soff = (int64_t)unit * a.P;
        const int len = unit_len(unit);
        const int rh = h0 + RB * wh + jr, rw = w0 + (ONE ? 0 : 4 * ww + jc);
        const bool rvalid = rh < a.n1 && rw < a.n2;
        const int rpix = rvalid ? rh + a.n1 * rw : 0;
        const float cmu = nmu;

        // the wavefront's register operands as thirds (the last odd group of 16,
        // which a lane holds twice over: a, b, and a in the lower and c in the
        // upper half of the lane groups)
        u4 r0[NG][3], r1[NG][3];
        int sd = 0;
        float rlse = 0.f, rowD = 0.f, sq = 0.f, m = 0.f, rrho = 1.f, ninit = 0.f, fsd = 1.f, kb = 0.f;
        // backward: p = 2^s / 2^lse2 is formed as pt = 2^(s - I + PE) with lse2 = I + f,
        // I whole: p = 2^-PE rho pt, rho = 2^-f in (1/2, 1].  The whole number adds no
        // rounding to the scores, PE (some log2 of the window's slots) keeps the
        // exponents near 0, where their rounding is least, and rho multiplies the
        // row's results (query-centric pass) or its staged dy and D (key-centric
        // pass).
        auto row_split = [&](float lse, float &ipart, float &rho) {
            ipart = floorf(lse * kLog2e);
            // (the rest of a log-sum-exp of 2^23 and more is its rounding alone)
            const float f = __builtin_fmaf(lse, kLog2eLo, __builtin_fmaf(lse, kLog2e, -ipart));
            rho = __builtin_amdgcn_exp2f(-__builtin_amdgcn_fmed3f(f, -1.f, 2.f));
        };
        auto rsplit = [&](const float (&x)[NG][8], u4 (&r)[NG][3]) {
#pragma unroll
            for (int G = 0; G < NG; ++G) {
                split3<8>(x[G], r[G][0], r[G][1], r[G][2]);
                if (ODD && G == NG - 1) r[G][2] = g < 2 ? r[G][0] : r[G][2];
            }
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
            float mr1 = 0.f;
#pragma unroll
            for (int G = 0; G < NG; ++G) {
                float s2 = 0.f, dot = 0.f;
#pragma unroll
                for (int c = 0; c < 8; ++c) {
                    if constexpr (DIST) s2 += x0[G][c] * x0[G][c];
                    if constexpr (MODE == FWD) dot += DIST ? x1[G][c] * (x0[G][c] - 0.5f * x1[G][c]) : x0[G][c] * x1[G][c];
                }
                if constexpr (MODE != FWD) mr1 = maxabs(x1[G], mr1);
                const bool twice = ODD && G == NG - 1 && g >= 2;
                sq += twice ? 0.f : s2;
                m += twice ? 0.f : dot;
            }
            if constexpr (DIST) sq = gsum(sq);
            if constexpr (MODE == FWD) m = gsum(m) * a.c2;
            // q' = q c2 2^-24
            const float c2s = __builtin_amdgcn_ldexpf(a.c2, -kUp);
#pragma unroll
            for (int G = 0; G < NG; ++G)
#pragma unroll
                for (int c = 0; c < 8; ++c) x0[G][c] *= c2s;
            rsplit(x0, r0);
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
            }
            // sd: the power of two that brings the pixel's dy (v) into [4, 8)
            if constexpr (MODE != FWD) {
                sd = max(-126, min(114, 129 - (int)bexp(gmax(mr1))));
#pragma unroll
                for (int G = 0; G < NG; ++G)
#pragma unroll
                    for (int c = 0; c < 8; ++c) x1[G][c] = __builtin_amdgcn_ldexpf(x1[G][c], sd + kUpP - kUp);
                rsplit(x1, r1);
            }
            if constexpr (MODE == BWDQ) {
                float I;
                row_split(rlse, I, rrho);
                ninit = a.pe - I - (DIST ? 0.5f * a.c2 * sq : 0.f);
            }
            fsd = KV ? __builtin_amdgcn_ldexpf(1.f, sd + kUpP) : 1.f;
            kb = KV && DIST ? -0.5f * a.c2 * sq : 0.f;
        }
        f4 acc0[NT], acc1[NT];
#pragma unroll
        for (int h = 0; h < NT; ++h) acc0[h] = acc1[h] = f4{0.f, 0.f, 0.f, 0.f};
        float lsum = 0.f, corr = 0.f;
        int xunit = unit, xh0 = h0, xw0 = w0;
        const int nitem = item_of(k + 1);
        const bool has_next = nitem < a.nitems;

        for (int ch = 0; ch < a.nchunk; ++ch) {
            if constexpr (DIST)
                if (ch == 0 && wv == 0) cen[lane] = cmu;
            __syncthreads();  // the previous chunk's LDS reads are done; the centre is in
            // centre, scale, split and store
#pragma unroll
            for (int i = 0; i < T; ++i) {
                const int wt = wv + NW * i;
                if (wt >= a.wt) continue;
                const bool t1 = wt & 1;
                FST_FENCE();
                float up = __builtin_amdgcn_ldexpf(1.f, kUp), sv = 0.f;
                if constexpr (DIST) {
                    if (!t1) {
                        float q2 = 0.f;
#pragma unroll
                        for (int c = 0; c < 16; c += 4) {
                            const f4 mu = *reinterpret_cast<const f4 *>(cen + 16 * th + c);
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                float &x = pv[i][c + e];
                                x -= mu[e];
                                if (!full) x = comp_ok(th, c + e) ? x : 0.f;
                                q2 += x * x;
                            }
                        }
                        if constexpr (NTP == 2) q2 += __shfl_xor(q2, 32);
                        if constexpr (NTP == 4) {
                            if (NT == 3 && lane >= 48) q2 = 0.f;
                            q2 = gsum(q2);
                        }
                        sv = -0.5f * a.c2 * q2;
                    }
                }
                if constexpr (KV) {
                    float I, rho;
                    row_split(pl[i], I, rho);
                    if (t1) {
                        sv = -pd[i] * rho;
                        up *= rho;
                    } else {
                        sv += a.pe - I;
                    }
                }
                u4 st[6];
#pragma unroll
                for (int c = 0; c < 8; ++c) {
                    unsigned x, y, z;
                    split3(pv[i][2 * c] * up, pv[i][2 * c + 1] * up, x, y, z);
                    st[c >> 2][c & 3] = x;
                    st[2 + (c >> 2)][c & 3] = y;
                    st[4 + (c >> 2)][c & 3] = z;
                }
                const int slot = srow[i] + a.cr * scol[i];
                const bool last16 = ODD && th == NT - 1;
                char *const sp_ = lds + slot * SB + (t1 ? T1 : 0) + 192 * (th >> 1) + (last16 ? 0 : 32 * (th & 1));
                if (sok[i]) {
#pragma unroll
                    for (int c = 0; c < 6; ++c)
                        *reinterpret_cast<u4 *>(sp_ + (c >> 1) * (last16 ? 32 : 64) + 16 * (c & 1)) = st[c];
                    if (th == 0) {
                        if (KV && t1) sc1[slot] = sv;
                        if ((KV || DIST) && !t1) sc0[slot] = sv;
                    }
                }
            }
            __syncthreads();  // chunk staged

            const bool lastch = ch + 1 == a.nchunk;
            if (lastch && has_next) decode(nitem, xunit, xh0, xw0);
            if constexpr (!LATE) load_stage(xunit, xh0, xw0, lastch ? 0 : ch + 1);
            if constexpr (DIST)
                nmu = load_centre(xunit, xh0, xw0);

            const float ptop = (float)(a.pe + 1);
            const float nD = MODE == BWDQ ? -__builtin_amdgcn_ldexpf(rowD, sd + kUpP) : 0.f;

            // score-type product of a block's 16 pixels with the register
            // pixels over all components: the smaller partial products from 0,
            // then x0 is added and the largest, so that the sum is rounded at
            // its full size once for x0 and once for every 32 components
            auto score = [&](const char *A, const u4 (&r)[NG][3], f4 x0) __attribute__((always_inline)) {
                f4 x = f4{0.f, 0.f, 0.f, 0.f};
                u4 t[NG];
#pragma unroll
                for (int G = 0; G < NG; ++G) {
                    const char *const B = A + 192 * G;
                    t[G] = *reinterpret_cast<const u4 *>(B);
                    if (ODD && G == NG - 1) {
                        // runs of 32: [c | a] on (a, c), [a | b] on (b, b) and (a, a)
                        const u4 ca = *reinterpret_cast<const u4 *>(B + (g < 2 ? 64 : -32));
                        x = mfmab(ca, r[G][2], x);
                        x = mfmab(t[G], r[G][1], x);
                    } else {
                        const u4 c = *reinterpret_cast<const u4 *>(B + 128);
                        const u4 b = *reinterpret_cast<const u4 *>(B + 64);
                        x = mfmab(c, r[G][0], x);
                        x = mfmab(t[G], r[G][2], x);
                        x = mfmab(b, r[G][1], x);
                        x = mfmab(b, r[G][0], x);
                        x = mfmab(t[G], r[G][1], x);
                    }
                }
                x = x + x0;
#pragma unroll
                for (int G = 0; G < NG; ++G) x = mfmab(t[G], r[G][0], x);
                return x;
            };
            // sums of a block pair's pixels, weighted: the smaller partial products
            // from 0 again, so that the sum is rounded at its full size twice
            auto apply = [&](const char *R0, const char *R1, const float (&w)[2][4], f4 (&acc)[NT]) __attribute__((always_inline)) {
                u4 wa, wb, wc;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    unsigned x, y, z;
                    split3(w[i >> 1][2 * (i & 1)], w[i >> 1][2 * (i & 1) + 1], x, y, z);
                    wa[i] = x;
                    wb[i] = y;
                    wc[i] = z;
                }
#pragma unroll
                for (int h = 0; h < NT; ++h) {
                    FST_FENCE();
                    const int o = third_off<NT>(h), d = third_step<NT>(h);
                    const u4 c = ldtr2(R0 + o + 2 * d, R1 + o + 2 * d), b = ldtr2(R0 + o + d, R1 + o + d),
                             a_ = ldtr2(R0 + o, R1 + o);
                    f4 t = mfmab(c, wa, f4{0.f, 0.f, 0.f, 0.f});
                    t = mfmab(a_, wc, t);
                    t = mfmab(b, wb, t);
                    t = mfmab(b, wa, t);
                    t = mfmab(a_, wb, t);
                    acc[h] = mfmab(a_, wa, acc[h] + t);
                }
            };
            auto walk = [&](int bc, int cc) __attribute__((always_inline)) {
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
                    if constexpr (MODE == FWD) {
                        // scores less c0 (masked: -inf)
                        f4 x[2];
                        auto scores = [&](float c0) __attribute__((always_inline)) {
#pragma unroll
                            for (int u = 0; u < 2; ++u) {
                                const float c = cw - c0;
                                f4 in = pM[MROW * (b + u)] + f4{c, c, c, c};
                                if constexpr (DIST)
                                    in = in + *reinterpret_cast<const f4 *>(pS0 + co + RB * (u && two ? b + 1 : b));
                                FST_FENCE();
                                x[u] = score(u ? A1 : A0, r0, in);
                            }
                        };
                        auto probs = [&]() __attribute__((always_inline)) {
#pragma unroll
                            for (int u = 0; u < 2; ++u)
#pragma unroll
                                for (int r = 0; r < 4; ++r) p[u][r] = __builtin_amdgcn_exp2f(x[u][r]);
                            return ((p[0][0] + p[0][1]) + (p[0][2] + p[0][3])) +
                                   ((p[1][0] + p[1][1]) + (p[1][2] + p[1][3]));
                        };
                        scores(m);
                        float ps = probs();
                        if (__builtin_amdgcn_ballot_w64(!(ps <= 256.f)) != 0) {
                            // a score more than 8 above m: m becomes the pair's
                            // maximum where that is larger.  The scores are formed
                            // again without m, of whose rounding they would
                            // otherwise keep a part if it lay far below them.
                            scores(0.f);
                            float mx = m;
#pragma unroll
                            for (int u = 0; u < 2; ++u)
#pragma unroll
                                for (int r = 0; r < 4; ++r) mx = fmaxf(mx, x[u][r]);
                            mx = gmax(mx);
                            const float f = __builtin_amdgcn_exp2f(m - mx);
                            m = mx;
                            lsum *= f;
#pragma unroll
                            for (int h = 0; h < NT; ++h) acc0[h] = acc0[h] * f4{f, f, f, f};
#pragma unroll
                            for (int u = 0; u < 2; ++u) x[u] = x[u] - f4{mx, mx, mx, mx};
                            ps = probs();
                        }
                        lsum += ps;
                        apply(R0 + T1, R1 + T1, p, acc0);
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
                            FST_FENCE();
                            const f4 x = score(u ? A1 : A0, r0, in);
                            dp = score((u ? A1 : A0) + T1, r1, dp);
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                // (p <= 1: the rounding of very large scores, 2^20 and
                                // more, would carry some far past it; NaN stays)
                                p[u][r] = __builtin_amdgcn_exp2f(__builtin_elementwise_minimum(x[r], ptop));
                                ds[u][r] = p[u][r] * dp[r];
                            }
                            if constexpr (DIST) corr += (ds[u][0] + ds[u][1]) + (ds[u][2] + ds[u][3]);
                        }
                        apply(R0, R1, ds, acc0);
                        if constexpr (KV) apply(R0 + T1, R1 + T1, p, acc1);
                    }
                }
            };
            for (int cc = 0; cc < (ONE ? 1 : a.cbc); ++cc) {
                const int bc = ONE ? 0 : ch * a.cbc + cc - ww;
                if (bc < 0 || bc >= (ONE ? 1 : a.nk)) continue;
                walk(bc, cc);
            }
            if constexpr (LATE) load_stage(xunit, xh0, xw0, lastch ? 0 : ch + 1);
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
        // a result that is not finite (values outside the pixel's window, or the
        // powers of two, may have made it so): NaN marks the wavefront's pixels for
        // the second pass below
        float top = MODE == FWD ? 0.f : fabsf(rlse);
        bool bad = false;
#pragma unroll
        for (int h = 0; h < NT; ++h)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                bad |= !(fabsf(acc0[h][r]) < INFINITY);
                if constexpr (KV) bad |= !(fabsf(acc1[h][r]) < INFINITY);
            }
        const float l = MODE == FWD ? gsum(lsum) : 1.f;
        const float cs = DIST && MODE != FWD ? gsum(corr) : 0.f;
        bad |= !(top < INFINITY) || !(l > 0.f && l < INFINITY) || !(fabsf(m) < INFINITY) || !(fabsf(cs) < INFINITY);
        const bool again = __builtin_amdgcn_ballot_w64(bad && rvalid) != 0;
        redo |= again;
        if constexpr (MODE == FWD) {
            float inv = __builtin_amdgcn_rcpf(l);
            inv = again ? NAN : __builtin_fmaf(__builtin_fmaf(-l, inv, 1.f), inv, inv);
            if (rvalid) {
#pragma unroll
                for (int h = 0; h < NT; ++h) {
                    float x[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) x[r] = __builtin_amdgcn_ldexpf(acc0[h][r] * inv, -kUp);
                    put4(a.yout, h, x);
                }
                if (g == 0) a.lse_out[soff + rpix] = lse_of(m, l, DIST ? 0.5f * sq * a.scale : 0.f);
            }
        } else {
            const float f = again ? NAN : a.scale * rrho;
#pragma unroll
            for (int h = 0; h < NT; ++h) {
                float xk[4], xv[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float v = __builtin_amdgcn_ldexpf(acc0[h][r], -(sd + kUpP + kUp) - a.pe);
                    if constexpr (DIST) {
                        const float reg = load1(KV ? a.k : a.q, uoff, len, rpix, h, 4 * g + r) -
                                          __shfl(cmu, 16 * h + 4 * g + r);
                        v -= __builtin_amdgcn_ldexpf(cs, -(sd + kUpP) - a.pe) * reg;
                    }
                    xk[r] = v * f;
                    if constexpr (KV) xv[r] = __builtin_amdgcn_ldexpf(acc1[h][r], -kUp - a.pe);
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
    if (!redo) return;
    // second pass, over the wavefront's marked pixels (here, where the first
    // pass's registers are free)
    for (int n = 0; n <= k; ++n) {
        decode(item_of(n), unit, h0, w0);
        const int64_t uoff = unit_off(unit);
        const int rh = h0 + RB * wh + jr, rw = w0 + (ONE ? 0 : 4 * ww + jc);
        // (component 0, read by the lane that wrote it)
        bool again = false;
        if (g == 0 && rh < a.n1 && rw < a.n2) {
            const int pix = rh + a.n1 * rw;
            const float x = (MODE == FWD ? a.yout : MODE == BWDQ ? a.dq : a.dk)[uoff + (CL ? pix * a.ncrall : pm * pix)];
            again = x != x;
        }
        if (__builtin_amdgcn_ballot_w64(again) != 0)
            plain_item<NT, DIST, MODE, ONE>(a, uoff, (int64_t)unit * a.P, h0 + RB * wh, w0 + (ONE ? 0 : 4 * ww));
    }
}

// Launch shape of a problem; ok = false where it does not fit
struct Shape {
    int nk, hr, cr, cbc, nchunk, npx, wt, os, om, oc, bytes;
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
        s.oc = s.om + (ONE ? 64 : 4) * 16 * (s.nk + 1);
        s.bytes = s.oc + (DIST ? 256 : 0);
        if (s.wt <= NW * T && s.bytes <= cap) break;
    }
    s.ok = s.cbc >= 1;
    return s;
}

template <int NT, int NWH, int NWW, int T, int EU, bool DIST, int MODE, bool ONE, bool CL>
hipError_t launch_shape(const Args &a0, const Shape &sh, int nunits, int cus, hipStream_t s) {
    constexpr int WH = ONE ? NWH * NWW : NWH, WW = ONE ? 1 : NWW;
    Args a = a0;
    a.nk = sh.nk; a.hr = sh.hr; a.cr = sh.cr; a.cbc = sh.cbc; a.nchunk = sh.nchunk;
    a.npx = sh.npx; a.wt = sh.wt; a.os = sh.os; a.om = sh.om; a.oc = sh.oc;
    a.tiles_h = (a.n1 + (ONE ? 16 : 4) * WH - 1) / ((ONE ? 16 : 4) * WH);
    a.tiles_w = ONE ? 1 : (a.n2 + 4 * WW - 1) / (4 * WW);
    const int64_t nitems = (int64_t)a.tiles_h * a.tiles_w * nunits;
    if (nitems <= 0 || nitems > (1 << 22)) return hipErrorNotSupported;
    if (a.route) {
        *a.route = 10 * NWH + NWW;
        return hipSuccess;
    }
    auto kern = kernel_stream<NT, WH, WW, T, EU, DIST, MODE, ONE, CL>;
    static const hipError_t attr = hipFuncSetAttribute(
        reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)f2d::kLdsCap);
    if (attr != hipSuccess) return attr;
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
    // Tiles of 4 x 2 wavefronts; workgroups of these are one a CU in most cases.
    // us, forward / query- / key-centric pass, at the crossings (256 CUs):
    //   tiles    shape                      2 x 2          4 x 2         8 x 2
    //   96       32 components, ws 9        14/15/19       15/17/21      20/22/28
    //            64, ws 15                  40/44/54       44/50/63
    //   144      32, ws 9                   16/19/23       15/17/22      20/22/28
    //            64, ws 15                  70/79/96       44/52/64
    //   256      32, ws 17                  30/35/44       25/30/38      34/39/51
    //   288      32, ws 9                   24/28/34       26/31/39      21/24/30
    //            32, ws 31, Distance        134/150/183    146/167/205   93/115/142
    //   512      16, ws 9                   21/23/28       20/23/28      16/18/23
    //            32, ws 17                  55/66/84       46/55/69      38/45/59
    //            32, ws 31, Distance        161/184/227    146/169/209   94/121/154
    //   544      32, ws 17                  69/82/103      64/78/98      68/79/104
    //            32, ws 31, Distance        206/229/279    213/247/306   182/225/283
    //   768      32, ws 17                  80/95/121      66/78/99      69/79/105
    //   1200     32, ws 9                   56/66/80       59/69/86      57/67/85
    //   1536     32, ws 17                  154/184/235    125/152/194   102/120/158
    //            32, ws 31, Distance        463/529/654    438/502/618   270/344/436
    const int64_t tiles = (int64_t)(ONE ? (a.n1 + 127) / 128 : ((a.n1 + 15) / 16) * ((a.n2 + 7) / 8)) * nunits;
    if constexpr (NT <= 2 && !ONE) {
        // twice the tile where that saves rounds of workgroups: a round of these
        // takes some one and a half times as long
        const Shape b = shape_of<NT, 8, 2, 1, DIST, MODE, ONE>(a.p);
        const int64_t tall = (int64_t)((a.n1 + 31) / 32) * ((a.n2 + 7) / 8) * nunits;
        const int64_t r8 = (tall + cus - 1) / cus, r4 = (tiles + cus - 1) / cus;
        if (b.ok && 3 * r8 < 2 * r4)
            return launch_shape<NT, 8, 2, 1, 4, DIST, MODE, ONE, CL>(a, b, nunits, cus, s);
    }
    const Shape m = shape_of<NT, 4, 2, 3, DIST, MODE, ONE>(a.p);
    // half the tile up to half a round, two workgroups a CU where half of LDS
    // holds a chunk
    Shape c = shape_of<NT, 2, 2, 3, DIST, MODE, ONE>(a.p, (int)f2d::kLdsCap / 2);
    if (!c.ok) c = shape_of<NT, 2, 2, 3, DIST, MODE, ONE>(a.p);
    if (m.ok && (tiles > cus / 2 || !c.ok))
        return launch_shape<NT, 4, 2, 3, 2, DIST, MODE, ONE, CL>(a, m, nunits, cus, s);
    if (c.ok) return launch_shape<NT, 2, 2, 3, 2, DIST, MODE, ONE, CL>(a, c, nunits, cus, s);
    if constexpr (NT == 4) {
        // (the widest windows, whose chunks of the taller tile do not fit LDS)
        const Shape w = shape_of<NT, 3, 2, 4, DIST, MODE, ONE>(a.p);
        if (w.ok) return launch_shape<NT, 3, 2, 4, 2, DIST, MODE, ONE, CL>(a, w, nunits, cus, s);
    }
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
