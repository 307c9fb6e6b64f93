// Products A ⊗ x and Aᵀ ⊗ x of a Circulant's values on the Float32 matrix
// cores, and the similarity pullback's two products in one grid.
//
// A wavefront holds 4x4 output pixels (16x1 in one dimension) and walks the
// 4x4 (16x1) blocks of pixels that their windows meet.  One
// v_mfma_f32_16x16x4f32 contracts four pixels of a block: operand A is x
// (16 components of 4 pixels, from LDS), operand B the matrix values (16
// output pixels by 4 pixels), its result 16 components of the 16 outputs.
// The lane that holds output pixel j and group g takes the four elements of
// block column g (rows r = 0 .. 3), so in the forward product its values are
// four adjacent slots of row j, one 16-byte load straight from memory into the
// operand, and in the transposed one four 4-byte loads a row of A apart, of
// which four lanes share a run of four.  Where a reference row's slot order is
// rotated (output pixels, or source pixels of the transposed product, within p
// of the image's border) each element is loaded from its own slot.
//
// x passes through LDS in planes, one per channel, [column][row] (complex:
// [column][row][part]) floats, by 16-byte LDS-DMA loads, in chunks of whole
// block columns where it does not fit; a lane's operand of four steps is one
// 16-byte read of four rows.  With a plane of 8 mod 16 floats and a column of an
// odd number of 16-byte units those reads are free of bank
// conflicts (gfx950 serves ds_read_b128 in the lane groups {0-3, 12-15, 20-27},
// {4-11, 16-19, 28-31} and the same plus 32).
//
// What bounds it: the matrix values' way through the texture path (each lane
// its own 16 bytes, some 40 cycles an instruction) and the wait for it.  A 200x120
// image, window 23, 32 components: A x 230 -> 53 us, A' x 282 -> 65 us (51 MB of
// values, 10 us at the rate of a large copy) in 1.5 wavefronts a SIMD, the
// texture path's data side 0.52 of the time busy, its addresses 0.3, the matrix
// cores 0.16 (128 cycles for a block and 16 components), and 73 / 88 MB read from
// memory.  Workgroups are not persistent: two fit a CU, and one stages while the
// other walks.
//
// Values outside a window count as 0 but meet x in the product, so a result
// that is not a number is formed again from its own window alone.
#include <algorithm>

#include "buffer_dma.h"
#include "circatt_common.h"
#include "circatt_kernels.h"

extern __shared__ __attribute__((aligned(16))) float circatt_ldsx[];

namespace circatt {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
using dma::dma16;
using dma::dma_rsrc;
using dma::i4v;
using dma::kMaxBytes;
using dma::kOut;
using dma::rsrc;
using dma::wrap;
// Matrix values are fetched in bursts of kBurst blocks, a burst ahead of the
// products: the blocks of a burst lie in the same cache lines (a window row is
// a third of a line at ws 11), which loads spread over the walk would fetch
// from L2 once for each block (320x320, ws 11, 32 components of 4 units: 200 us
// with one load per block, 176 us in bursts).
constexpr int kBurst = 4;

struct MxArgs {
    const float *nz, *x, *z;
    float *y;
    int n1, n2, P, ws, p, K, nk;
    int ncr, pm, npass;          // real components per unit, floats between pixels, passes of 16 NT
    float scale;
    int corr;                    // subtract sums(A) .* z
    int hr, cr, pl, cbc, nchunk, npx, ow;  // ow: float offset of the weights
    int tiles_h, tiles_w, nitems, per_xcd;
    FastDiv div_pass, div_tiles, div_th, div_cr;
};

__device__ __forceinline__ float gsum(float v) {
    v += __shfl_xor(v, 16);
    return v + __shfl_xor(v, 32);
}

// offset of component k from component 0 (floats)
__device__ __forceinline__ int coff(const MxArgs &a, int k) {
    return a.pm == 2 ? 2 * a.P * (k >> 1) + (k & 1) : a.P * k;
}

// the products of one wavefront's pixels from their own windows alone: lane c
// holds component c0 + c, one pixel at a time
template <bool TRANS, bool ONE>
__device__ __forceinline__ void plain_pixels(const MxArgs &a, const float *nz, int64_t xo, int row0, int col0, int c0,
                                             int nc) {
    const int lane = threadIdx.x & 63, p2 = ONE ? 0 : a.p;
    const bool on = lane < nc;
    const int co = coff(a, c0 + (on ? lane : 0));
    for (int i = 0; i < 16; ++i) {
        const int r = row0 + (ONE ? i : i & 3), c = col0 + (ONE ? 0 : i >> 2);
        if (r >= a.n1 || c >= a.n2) continue;
        const int pix = r + a.n1 * c;
        float acc = 0.f, sum = 0.f;
        for (int d2 = -p2; d2 <= p2; ++d2)
            for (int d1 = -a.p; d1 <= a.p; ++d1) {
                const int r2 = pmod(r + d1, a.n1), c2 = ONE ? 0 : pmod(c + d2, a.n2);
                // row pix at offset d, or row (pix + d) at offset -d
                const int sr = TRANS ? r2 : r, sc = TRANS ? c2 : c, e1 = TRANS ? -d1 : d1, e2 = TRANS ? -d2 : d2;
                const int m1 = offset_to_slot(e1, slot_shift(sr + 1, a.n1, a.p), a.ws, a.p);
                const int m2 = ONE ? 0 : offset_to_slot(e2, slot_shift(sc + 1, a.n2, a.p), a.ws, a.p);
                const float w = nz[(int64_t)(sr + a.n1 * sc) * a.K + m2 * a.ws + m1];
                if (on) acc = __builtin_fmaf(w, a.x[xo + a.pm * (r2 + a.n1 * c2) + co], acc);
                sum += w;
            }
        if (on) {
            const int64_t o = xo + a.pm * pix + co;
            if (a.corr) acc -= sum * a.z[o];
            a.y[o] = a.scale * acc;
        }
    }
}

// INNER: no row of A that the wavefront reads has a rotated slot order (nor,
// transposed, lies past a circular wrap).  Two bodies rather than a branch in
// the walk: where the paths of a branch around a load meet, the compiler waits
// for it.  Their barriers match.
template <int NT, int NWH, int NWW, bool TRANS, bool ONE, bool CPLX, bool INNER>
__device__ __forceinline__ void mx_walk(const MxArgs &a, int item) {
    constexpr int NW = NWH * NWW, RB = ONE ? 16 : 4;
    constexpr int PF = CPLX ? 2 : 1;             // floats of a pixel in a plane
    constexpr int NPL = CPLX ? 8 * NT : 16 * NT;  // planes: channels
    float *const lds = circatt_ldsx;
    typedef __attribute__((address_space(3))) const char *lcp;
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)reinterpret_cast<uintptr_t>((lcp)(char *)lds));
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wh = wv % NWH, ww = wv / NWH;
    const int j = lane & 15, g = lane >> 4;
    const int jr = ONE ? j : j & 3, jc = ONE ? 0 : j >> 2;

    const int upass = fdiv(item, a.div_tiles);
    const int tile = item - upass * (a.tiles_h * a.tiles_w);
    const int unit = fdiv(upass, a.div_pass), c0 = (upass - unit * a.npass) * 16 * NT;
    const int tw = fdiv(tile, a.div_th);
    const int h0 = (tile - tw * a.tiles_h) * RB * NWH, w0 = ONE ? 0 : tw * 4 * NWW;
    const int nc = min(16 * NT, a.ncr - c0);
    const int64_t xo = (int64_t)unit * a.P * a.ncr;
    const float *const nz = a.nz + (int64_t)unit * a.P * a.K;
    const auto rn = rsrc(nz, a.P * a.K * 4);
    const i4v rx = dma_rsrc(a.x + xo, a.P * a.ncr * 4);
    const auto rxb = rsrc(a.x + xo, a.P * a.ncr * 4);

    const int hw = h0 + RB * wh, wc = w0 + (ONE ? 0 : 4 * ww);  // the wavefront's first pixel
    const int rh = hw + jr, rw = wc + jc;
    const bool rvalid = rh < a.n1 && rw < a.n2;
    const int rpix = rvalid ? rh + a.n1 * rw : 0;
    // slot shifts of the output pixel's row (forward, near the border)
    const int s1 = slot_shift(rh + 1, a.n1, a.p), s2 = ONE ? 0 : slot_shift(rw + 1, a.n2, a.p);
    // lane part of the element index of a block's first element (inner)
    const int lbase = TRANS ? ((hw - a.p + (ONE ? 4 * g : 0)) + a.n1 * (ONE ? 0 : wc - a.p + g)) * a.K +
                                  (ONE ? 0 : (jc + 2 * a.p - g) * a.ws) + jr + 2 * a.p - (ONE ? 4 * g : 0)
                            : rpix * a.K + (ONE ? 4 * g : (g - jc) * a.ws) - jr;

    // four matrix values of block (br, bc) for this lane; 0 unless on
    auto fetch = [&](int br, int bc, bool on) __attribute__((always_inline)) {
        f4 v;
        if constexpr (INNER && !TRANS) {
            const int o = lbase + RB * br + 4 * bc * a.ws;
            v = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rn, on ? o * 4 : kOut, 0, 0));
        } else if constexpr (INNER) {
            const int o = on ? (lbase + RB * br * (a.K - 1) + 4 * bc * (a.n1 * a.K - a.ws)) * 4 : kOut;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                v[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rn, (int)((unsigned)o + 4u * r * (a.K - 1)), 0, 0));
        } else {
            const int u2 = ONE ? 0 : 4 * bc + g - jc;
            const int q2 = ONE ? 0 : wrap(wc - a.p + 4 * bc + g, a.n2);  // source pixel's column
            const int m2 = ONE ? 0
                               : wrap(TRANS ? 2 * a.p - u2 + slot_shift(q2 + 1, a.n2, a.p) : u2 + s2, a.ws);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int R = RB * br + (ONE ? 4 * g : 0) + r, u1 = R - jr;
                const bool in = on && u1 >= 0 && u1 <= 2 * a.p && u2 >= 0 && (ONE || u2 <= 2 * a.p);
                int o;
                if constexpr (TRANS) {
                    const int q1 = wrap(hw - a.p + R, a.n1);
                    o = (q1 + a.n1 * q2) * a.K + m2 * a.ws + wrap(2 * a.p - u1 + slot_shift(q1 + 1, a.n1, a.p), a.ws);
                } else {
                    o = rpix * a.K + m2 * a.ws + wrap(u1 + s1, a.ws);
                }
                v[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rn, in ? o * 4 : kOut, 0, 0));
            }
        }
        return v;
    };

    constexpr int NA = NT == 1 ? 2 : 1;  // (two accumulators keep one component group's products independent)
    f4 acc[NA][NT];
#pragma unroll
    for (int i = 0; i < NA; ++i)
#pragma unroll
        for (int h = 0; h < NT; ++h) acc[i][h] = f4{0.f, 0.f, 0.f, 0.f};
    float sum = 0.f;

    f4 va[kBurst], vb[kBurst];
    // Weights of a lane's four elements: 1 in the window, 0 outside, per block
    // row and (2D) per block column.  A loaded value is multiplied by both
    // (full-rate products; a select under a branch would make the compiler wait
    // for the load there).
    constexpr int WROW = ONE ? 64 : 4;
    f4 *const wtab = reinterpret_cast<f4 *>(lds + a.ow);
    const f4 *const wrow = wtab + (ONE ? lane : jr);
    float *const ctab = lds + a.ow + 4 * WROW * a.nk;
    const float *const wcol = ctab + jc + 4 * g;
    auto win = [&](int u) { return u >= 0 && u <= 2 * a.p ? 1.f : 0.f; };
    for (int i = threadIdx.x; i < WROW * a.nk; i += 64 * NW) {
        const int b = i / WROW, e = i % WROW;
        f4 w;
#pragma unroll
        for (int r = 0; r < 4; ++r) w[r] = win(RB * b + (ONE ? 4 * (e >> 4) : 0) + r - (ONE ? e & 15 : e));
        wtab[i] = w;
    }
    if constexpr (!ONE)
        for (int i = threadIdx.x; i < 16 * a.nk; i += 64 * NW) ctab[i] = win(4 * (i >> 4) + ((i & 15) >> 2) - (i & 3));
    // planes of a lane: component 16 h + j (real); complex channels 16 h' + j
    // give their real and imaginary parts to groups 2 h' and 2 h' + 1, and an
    // odd last group takes 8 channels, both parts side by side
    constexpr int NPAIR = CPLX ? NT / 2 : 0;
    const float *const px = lds + (RB * wh + (ONE ? 4 * g : a.cr * g)) * PF;
    auto comp = [&](int h, int i) {  // component (from c0) of row i of group h
        if (!CPLX) return 16 * h + i;
        return h < 2 * NPAIR ? 2 * (16 * (h >> 1) + i) + (h & 1) : 32 * NPAIR + i;
    };

    for (int ch = 0; ch < a.nchunk; ++ch) {
        if (ch > 0) __syncthreads();  // the previous chunk's reads are done
        {
            // task: 64 16-byte pieces (4 pixels of a column, or 2 complex
            // ones) of 4 planes
            const int npc = a.npx * PF / 4, ntile = (npc + 63) >> 6;
            const int cfirst = c0 / PF, clast = a.ncr / PF - 1;
            for (int t = wv; t < ntile * (NPL / 4); t += NW) {
                const int ti = t / (NPL / 4), cg = t - ti * (NPL / 4);
                const int pc = ti * 64 + lane, px_ = pc * (4 / PF);
                if (pc < npc) {
                    const int col = ONE ? 0 : fdiv(px_, a.div_cr), row = px_ - col * a.cr;
                    const int gr = wrap(h0 - a.p + row, a.n1);
                    const int gc = ONE ? 0 : wrap(w0 - a.p + 4 * a.cbc * ch + col, a.n2);
                    const int vo = (gr + a.n1 * gc) * PF * 4;
                    // pieces that straddle the circular wrap: pixel by pixel
                    const bool cross = gr + 4 / PF > a.n1;
                    if (!cross) {
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            dma16(rx, lds0 + ((4 * cg + i) * a.pl + ti * 256) * 4, vo,
                                  min(cfirst + 4 * cg + i, clast) * a.P * PF * 4);
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int so = min(cfirst + 4 * cg + i, clast) * a.P * PF * 4;
                            f4 v;
#pragma unroll
                            for (int q = 0; q < 4; ++q) {
                                const int r2 = gr + q / PF, o = (wrap(r2, a.n1) - gr) * PF + q % PF;
                                v[q] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rxb, vo + 4 * o + so, 0, 0));
                            }
                            *reinterpret_cast<f4 *>(lds + (4 * cg + i) * a.pl + 4 * pc) = v;
                        }
                    }
                }
            }
        }
        // this chunk's blocks: block columns b0 .. b1 - 1, all block rows; the
        // first values are in flight over the staging
        const int b0 = ONE ? 0 : max(ch * a.cbc - ww, 0), b1 = ONE ? 1 : min((ch + 1) * a.cbc - ww, a.nk);
        int n = b1 > b0 ? (b1 - b0) * a.nk : 0;
        int br = 0, bc = b0, fr = 0, fc = b0;  // the block at hand, the next to fetch
        auto ahead = [&]() __attribute__((always_inline)) {
            const f4 v = fetch(fr, fc, fc < b1);
            const bool wrap = fr + 1 == a.nk;
            fr = wrap ? 0 : fr + 1;
            fc += wrap ? 1 : 0;
            return v;
        };
        auto burst = [&](f4 (&v)[kBurst]) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < kBurst; ++i) v[i] = ahead();
        };
        burst(va);
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();  // chunk staged
        auto products = [&](const f4 (&vs)[kBurst]) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < kBurst; ++i) {
                // (weights 0 outside the window)
                const float wc_ = ONE ? 1.f : wcol[16 * bc];
                const f4 v = vs[i] * wrow[WROW * br] * f4{wc_, wc_, wc_, wc_};
                sum += (v[0] + v[1]) + (v[2] + v[3]);
                const float *const xb = px + (RB * br + (ONE ? 0 : 4 * (bc + ww - ch * a.cbc) * a.cr)) * PF;
                f4 xv[NT];
                if constexpr (!CPLX) {
#pragma unroll
                    for (int h = 0; h < NT; ++h) xv[h] = *reinterpret_cast<const f4 *>(xb + (16 * h + j) * a.pl);
                } else {
#pragma unroll
                    for (int h = 0; h < NPAIR; ++h) {
                        const float *const q = xb + (16 * h + j) * a.pl;
                        const f4 lo = *reinterpret_cast<const f4 *>(q), hi = *reinterpret_cast<const f4 *>(q + 4);
                        xv[2 * h] = f4{lo[0], lo[2], hi[0], hi[2]};
                        xv[2 * h + 1] = f4{lo[1], lo[3], hi[1], hi[3]};
                    }
                    if constexpr (NT & 1) {
                        const float *const q = xb + (16 * NPAIR + (j >> 1)) * a.pl + (j & 1);
                        xv[NT - 1] = f4{q[0], q[2], q[4], q[6]};
                    }
                }
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int h = 0; h < NT; ++h)
                        acc[NA == 2 ? r & 1 : 0][h] =
                            __builtin_amdgcn_mfma_f32_16x16x4f32(xv[h][r], v[r], acc[NA == 2 ? r & 1 : 0][h], 0, 0, 0);
                const bool wrap = br + 1 == a.nk;
                br = wrap ? 0 : br + 1;
                bc += wrap ? 1 : 0;
                if (--n == 0) break;
            }
        };
        while (n > 0) {
            burst(vb);
            products(va);
            if (n == 0) break;
            burst(va);
            products(vb);
        }
    }
    if constexpr (NA == 2) acc[0][0] = acc[0][0] + acc[1][0];
    sum = gsum(sum);
    bool nan = false;
#pragma unroll
    for (int h = 0; h < NT; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r) nan |= !(acc[0][h][r] == acc[0][h][r]);
    if (__builtin_amdgcn_ballot_w64(nan) != 0) {
        plain_pixels<TRANS, ONE>(a, nz, xo, hw, wc, c0, nc);
        return;
    }
    if (rvalid) {
#pragma unroll
        for (int h = 0; h < NT; ++h)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int c = comp(h, 4 * g + r);
                if (c < nc) {
                    const int64_t o = xo + a.pm * rpix + coff(a, c0 + c);
                    float v = acc[0][h][r];
                    if (a.corr) v -= sum * a.z[o];
                    a.y[o] = a.scale * v;
                }
            }
    }
}

template <int NT, int NWH, int NWW, bool TRANS, bool ONE, bool CPLX>
__device__ __forceinline__ void mx_item(const MxArgs &a, int item) {
    constexpr int RB = ONE ? 16 : 4;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int upass = fdiv(item, a.div_tiles), tile = item - upass * (a.tiles_h * a.tiles_w);
    const int tw = fdiv(tile, a.div_th);
    const int hw = (tile - tw * a.tiles_h) * RB * NWH + RB * (wv % NWH), wc = ONE ? 0 : tw * 4 * NWW + 4 * (wv / NWH);
    const int e = TRANS ? 2 * a.p : a.p;
    if (hw >= e && hw + (RB - 1) < a.n1 - e && (ONE || (wc >= e && wc + 3 < a.n2 - e)))
        mx_walk<NT, NWH, NWW, TRANS, ONE, CPLX, true>(a, item);
    else
        mx_walk<NT, NWH, NWW, TRANS, ONE, CPLX, false>(a, item);
}

template <int NT, int NWH, int NWW, bool TRANS, bool ONE, bool CPLX>
__global__ __launch_bounds__(64 * NWH * NWW, 4) void apply_mx_kernel(MxArgs a) {
    const int item = (blockIdx.x & 7) * a.per_xcd + (blockIdx.x >> 3);
    if ((blockIdx.x >> 3) >= a.per_xcd || item >= a.nitems) return;
    mx_item<NT, NWH, NWW, TRANS, ONE, CPLX>(a, item);
}
// both products of the pullback: a tile's forward and transposed item follow
// each other on one XCD, so that the second finds the rows of A in its L2
template <int NT, int NWH, int NWW, bool ONE, bool CPLX>
__global__ __launch_bounds__(64 * NWH * NWW, 4) void apply_mx_pair_kernel(MxArgs f, MxArgs t) {
    const int slot = blockIdx.x >> 3;
    const int item = (blockIdx.x & 7) * f.per_xcd + (slot >> 1);
    if ((slot >> 1) >= f.per_xcd || item >= f.nitems) return;
    if (slot & 1)
        mx_item<NT, NWH, NWW, true, ONE, CPLX>(t, item);
    else
        mx_item<NT, NWH, NWW, false, ONE, CPLX>(f, item);
}

struct MxShape {
    int nk, hr, cr, pl, cbc, nchunk, npx, ow, bytes;
    bool ok;
};
MxShape mx_shape(bool one, bool cplx, int p, int nt, int nwh, int nww, int cap) {
    MxShape s{};
    const int rb = one ? 16 : 4;
    s.nk = 1 + (2 * p + rb - 1) / rb;
    s.hr = rb * (nwh + s.nk - 1);
    // (real: 4 mod 8 rows, complex: 2 mod 4, an odd number of 16-byte units)
    s.cr = cplx ? s.hr + ((2 - s.hr % 4) + 4) % 4 : s.hr + ((4 - s.hr % 8) + 8) % 8;
    const int ncol = one ? 1 : nww + s.nk - 1;
    for (s.cbc = ncol; s.cbc >= 1; --s.cbc) {
        s.nchunk = (ncol + s.cbc - 1) / s.cbc;
        s.npx = one ? s.cr : 4 * s.cbc * s.cr;
        const int f = s.npx * (cplx ? 2 : 1);
        s.pl = f + ((8 - f % 16) + 16) % 16;
        s.ow = (cplx ? 8 : 16) * nt * s.pl;
        s.bytes = (s.ow + (one ? 256 : 32) * s.nk) * 4;
        if (s.bytes <= cap) break;
    }
    s.ok = s.cbc >= 1;
    return s;
}

constexpr int kLds = 160 * 1024;

// Geometry of a launch.  Tiles of 8 wavefronts (16x8 pixels, 128 in one
// dimension) of which two fit a CU, or of 4 (8x8, 64) where the image is
// too small to give every CU one of those.
struct MxPlan {
    MxArgs a;
    MxShape s;
    bool big, one;
    int nt;
    bool ok;
};
MxPlan mx_plan(const Geom &g, int C, int ncomp, int64_t nb, int products) {
    MxPlan pl{};
    pl.one = g.nsp == 1;
    // (a window larger than the image, which meets pixels twice, is left to the others)
    if (g.p < 1 || g.n1 < g.ws || (!pl.one && g.n2 < g.ws) || (int64_t)C * ncomp >= 1 << 28 ||
        g.P * g.K * 4 >= kMaxBytes || (int64_t)g.P * C * ncomp * 4 >= kMaxBytes || g.n1 > (1 << 24) ||
        g.n2 > (1 << 24))
        return pl;
    const int ncr = C * ncomp;
    pl.nt = ncr > 48 ? 4 : (ncr + 15) / 16;
    MxArgs &a = pl.a;
    a.n1 = g.n1;
    a.n2 = g.n2;
    a.P = (int)g.P;
    a.ws = g.ws;
    a.p = g.p;
    a.K = g.K;
    a.ncr = ncr;
    a.pm = ncomp;
    a.npass = (ncr + 16 * pl.nt - 1) / (16 * pl.nt);
    const int rb = pl.one ? 16 : 4;
    for (int big = 1; big >= 0; --big) {
        const int nwh = pl.one ? (big ? 8 : 4) : (big ? 4 : 2), nww = pl.one ? 1 : 2;
        MxShape sh{};
        // (two workgroups a CU, or one: room for three gives smaller chunks, 200x120
        // at ws 23: 61 / 71 us, two 54 / 65, one 68 / 87)
        for (int per = 2; per >= 1; --per) {
            sh = mx_shape(pl.one, ncomp == 2, g.p, pl.nt, nwh, nww, kLds / per);
            if (sh.ok) break;
        }
        // (halos that wrap once at most: the smaller tiles' wider chunks may
        // reach further past a narrow image than the larger tiles' do)
        if (!sh.ok || g.n1 < sh.cr - g.p || (!pl.one && g.n2 < 4 * sh.cbc * sh.nchunk - g.p)) continue;
        const int th = (g.n1 + rb * nwh - 1) / (rb * nwh), tw = pl.one ? 1 : (g.n2 + 4 * nww - 1) / (4 * nww);
        const int64_t n = (int64_t)th * tw * a.npass * nb;
        if (n * products > (1 << 27)) continue;
        pl.s = sh;
        pl.big = big;
        a.tiles_h = th;
        a.tiles_w = tw;
        a.nitems = (int)n;
        if (!big || n * products >= 512) break;
    }
    if (!pl.s.ok) return pl;
    a.nk = pl.s.nk;
    a.hr = pl.s.hr;
    a.cr = pl.s.cr;
    a.pl = pl.s.pl;
    a.cbc = pl.s.cbc;
    a.nchunk = pl.s.nchunk;
    a.npx = pl.s.npx;
    a.ow = pl.s.ow;
    a.per_xcd = (a.nitems + 7) / 8;
    a.div_pass = make_fastdiv((uint32_t)a.npass);
    a.div_tiles = make_fastdiv((uint32_t)(a.tiles_h * a.tiles_w));
    a.div_th = make_fastdiv((uint32_t)a.tiles_h);
    a.div_cr = make_fastdiv((uint32_t)a.cr);
    pl.ok = true;
    return pl;
}

template <typename Kern>
hipError_t lds_attr(Kern kern) {
    return hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
}

template <int NT, int NWH, int NWW, bool ONE, bool CPLX>
hipError_t launch_one(bool trans, const MxPlan &pl, hipStream_t s) {
    const dim3 grid(8u * (unsigned)pl.a.per_xcd), block(64 * NWH * NWW);
    if (trans) {
        auto kern = apply_mx_kernel<NT, NWH, NWW, true, ONE, CPLX>;
        static const hipError_t e = lds_attr(kern);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(kern, grid, block, pl.s.bytes, s, pl.a);
    } else {
        auto kern = apply_mx_kernel<NT, NWH, NWW, false, ONE, CPLX>;
        static const hipError_t e = lds_attr(kern);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(kern, grid, block, pl.s.bytes, s, pl.a);
    }
    return hipGetLastError();
}
template <int NT, int NWH, int NWW, bool ONE, bool CPLX>
hipError_t launch_two(const MxPlan &pl, const MxArgs &f, const MxArgs &t, hipStream_t s) {
    auto kern = apply_mx_pair_kernel<NT, NWH, NWW, ONE, CPLX>;
    static const hipError_t e = lds_attr(kern);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3(16u * (unsigned)pl.a.per_xcd), dim3(64 * NWH * NWW), pl.s.bytes, s, f, t);
    return hipGetLastError();
}

}  // namespace

// Where these kernels run; elsewhere the row, band and wide kernels do.
// Measured both ways (us, others -> these: A x / A' x / the pullback's pair):
//  - windows past 15.  The band kernels (to 31) leave the chip idle on few pixels,
//    some 9 us a window column however few, and pass once over each row of A,
//    where these fetch its lines some three times: 2.0 to 3.7 us for a million
//    values, rising with the window, against 3.2 (ws 17) falling to 1.8 (ws 31),
//    twice that for more than 32 components.  200x120, 32 components, ws 17 179/222/224 ->
//    30/38/63, ws 31 295/361/359 -> 105/106/175; 4 x 256x254, 32 components, ws 21 (115 M
//    values) 301/332/584 -> 297/277/486, ws 23 (138 M) 325/359/629 against 384/365/657,
//    ws 31 444/475/870 against 757/646/1206, 64 components, ws 25 (163 M) 612/709/1264 ->
//    511/514/904, ws 31 766/840/1569 against 914/869/1606; 2 units, ws 25, 32 components
//    (81 M) 251/304/358 -> 244/216/367, ws 29 (109 M) 284/346/429 against 398/253/544, ws 31
//    (125 M) 305/366/459 against 473/319/664; 8 x 200x120, ws 23 (102 M) 338/405/657 ->
//    312/295/515.
//  - windows 7 to 15 with few components and pixels, where the row kernels
//    leave matrix cores or CUs idle: 128x126, 16 components, ws 7 13/13/14 ->
//    11/12/15, ws 13 27/29/32 -> 14/17/21; 2 units, ws 7 14/15/15 -> 13/15/20 (the pair
//    slower there, its sums the more precise: 2.5e-7 of 2-norm error in a step at
//    97x75, 4 units, against 2.7e-7), ws 9 19/19/20 -> 11/15/20, ws 11 23/25/26 -> 17/20/27; with 24 components ws 11
//    17/18/25 against 16/19/23, 2 units 17/19/26 against 21/23/33; 256x254, 16
//    components, ws 9 19/20/26 against 15/20/35, ws 11 24/26/33 against 24/27/47.
//  - lines from ws 15 on: 65536, ws 15, 32 components 19/24/52 -> 9/10/18; 8 x
//    65536, ws 63, 64 components 169/184/363 -> 116/126/275; under that 8
//    components of 8 x 65536 at ws 7 take 22/23/58 against 29/32/72.
bool apply_mx_supported(const Geom &g, int C, int ncomp, int64_t nb, int products) {
    const int64_t px = g.P * nb, values = px * g.K, ncr = (int64_t)C * ncomp;
    if (g.nsp == 1) {
        if (g.ws < 15) return false;
    } else if (g.ws <= 15) {
        if (g.ws < 7 || ncr > 16 || px > (1 << 15)) return false;
    } else if (g.ws <= 31) {
        if (values > (g.ws > 25 ? 75000000 : ncr > 32 ? 170000000 : 120000000)) return false;
    }
    return mx_plan(g, C, ncomp, nb, products).ok;
}

#define CIRCATT_MX_SH(F, NT, CPLX, ...)                                                                      \
    return pl.one ? (pl.big ? F<NT, 8, 1, true, CPLX>(__VA_ARGS__) : F<NT, 4, 1, true, CPLX>(__VA_ARGS__))    \
                  : (pl.big ? F<NT, 4, 2, false, CPLX>(__VA_ARGS__) : F<NT, 2, 2, false, CPLX>(__VA_ARGS__));
#define CIRCATT_MX_NT(F, ...)                                                                             \
    if (pl.a.pm == 2) {                                                                                    \
        switch (pl.nt) {                                                                                   \
        case 1: CIRCATT_MX_SH(F, 1, true, __VA_ARGS__)                                                     \
        case 2: CIRCATT_MX_SH(F, 2, true, __VA_ARGS__)                                                     \
        case 3: CIRCATT_MX_SH(F, 3, true, __VA_ARGS__)                                                     \
        default: CIRCATT_MX_SH(F, 4, true, __VA_ARGS__)                                                    \
        }                                                                                                  \
    }                                                                                                      \
    switch (pl.nt) {                                                                                       \
    case 1: CIRCATT_MX_SH(F, 1, false, __VA_ARGS__)                                                        \
    case 2: CIRCATT_MX_SH(F, 2, false, __VA_ARGS__)                                                        \
    case 3: CIRCATT_MX_SH(F, 3, false, __VA_ARGS__)                                                        \
    default: CIRCATT_MX_SH(F, 4, false, __VA_ARGS__)                                                       \
    }

hipError_t launch_apply_mx(bool trans, bool corr, int ncomp, const Geom &g, int C, int64_t nb, float scale,
                           const float *nz, const float *x, const float *z, float *y, hipStream_t s) {
    MxPlan pl = mx_plan(g, C, ncomp, nb, 1);
    if (!pl.ok) return hipErrorNotSupported;
    pl.a.nz = nz;
    pl.a.x = x;
    pl.a.z = z;
    pl.a.y = y;
    pl.a.scale = scale;
    pl.a.corr = corr;
    CIRCATT_MX_NT(launch_one, trans, pl, s)
}

hipError_t launch_apply_mx_pair(bool corr, int ncomp, const Geom &g, int C, int64_t nb, float scale, const float *nz,
                                const float *x, const float *y, float *dx, float *dy, hipStream_t s) {
    // dx = A ⊗ y (- rowsum(A) .* x), dy = Aᵀ ⊗ x (- colsum(A) .* y)
    MxPlan pl = mx_plan(g, C, ncomp, nb, 2);
    if (!pl.ok) return hipErrorNotSupported;
    MxArgs f = pl.a;
    f.nz = nz;
    f.scale = scale;
    f.corr = corr;
    MxArgs t = f;
    f.x = y;
    f.z = x;
    f.y = dx;
    t.x = x;
    t.z = y;
    t.y = dy;
    CIRCATT_MX_NT(launch_two, pl, f, t, s)
}

}  // namespace circatt

// The tiles that a call's products take (1: of 8 wavefronts, 2: of 4; 0: another
// kernel's call), without a launch; -1 if the rule above sends the call here and
// the plan refuses it.  For the host tests; no part of the C ABI.
extern "C" int circatt_route_apply_mx(int nsp, int n1, int n2, int ws, int C, int ncomp, int64_t nb, int products) {
    const circatt::Geom g = circatt::make_geom(nsp, n1, n2, ws);
    if (!circatt::apply_mx_supported(g, C, ncomp, nb, products)) return 0;
    const circatt::MxPlan pl = circatt::mx_plan(g, C, ncomp, nb, products);
    return !pl.ok ? -1 : pl.big ? 1 : 2;
}
