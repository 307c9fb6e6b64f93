// Similarity of a pixel with the pixels of its 2D window, windows 17 to 33:
// nzVal(slot, pixel) = scale Re<x(pixel), y(pixel + offset)>, or
// -scale |x - y|^2 / 2 from the differences.
//
// A wavefront holds 4x4 query pixels and NK x CB blocks of 4x4 key pixels (all
// block rows of the window, CB of its block columns): 4 scores per lane and
// block, 16 queries by 16 keys.  Dot products are formed by
// v_mfma_f32_16x16x4f32, four components a step; differences by vector
// instructions, of which a lane takes the four rows of one key column.  The
// components pass through LDS in planes of 16 at a time, so any number of them
// keeps its scores in registers.  A row of nzVal is then put together in LDS
// and stored in 16-byte pieces (a lane's four scores stored as they lie would
// take the texture path 40 cycles for each 16 bytes a lane).
//
// What bounds it: issue.  Distance at 200x120, window 23, 32 components: vector
// instructions 0.82 of the time, LDS 0.42 (a 16-byte read for 8 vector instructions,
// or 16 where a wavefront takes two query blocks), stores at 0.7 TB/s.  200x120, window 23, 32 components: 171 -> 48 us,
// Distance 213 -> 73 us (51 MB of scores, 10 us at the rate of a large copy).
#include <algorithm>

#include "buffer_dma.h"
#include "circatt_common.h"
#include "circatt_kernels.h"

extern __shared__ __attribute__((aligned(16))) float circatt_ldss[];

namespace circatt {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef f4 f4u __attribute__((aligned(4)));
using dma::dma16;
using dma::dma_rsrc;
using dma::i4v;
using dma::kMaxBytes;
using dma::kOut;
using dma::rsrc;
using dma::wrap;
constexpr int kLds = 160 * 1024;
constexpr int kNW = 2;               // wavefronts along each dimension of a workgroup
constexpr int kW = kNW * kNW;

struct SimArgs {
    const float *x, *y;  // queries, keys
    float *nz;
    int n1, n2, P, ws, p, K;
    int ncr;             // real components per unit
    float scale;
    int cr, pl, npx;     // floats... of a plane: pixels per column, floats, pixels
    int seg, region;     // floats of a query's scores and of a wavefront's in LDS
    int tiles_h, tiles_w, nstrip, nitems, per_xcd;
    FastDiv div_tiles, div_th, div_strip, div_cr;
};

__device__ __forceinline__ float load(__amdgpu_buffer_rsrc_t r, int o) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, o, 0, 0));
}
// Block columns of a wavefront: a window to 17 whole, wider ones in strips whose
// scores leave registers and LDS for 3 or 4 wavefronts per SIMD.
constexpr int strip_of(int nk) { return nk <= 5 ? nk : nk == 6 ? 3 : 2; }
// The queries of a block whose rows are put together at a time: in strips half,
// since their region of LDS, not the planes, would bound the workgroups of a CU
// (4 x 256x254, dot, 32 components, ws 21 319 -> 252 us, ws 31 650 -> 575; but whole
// windows, ws 17, 162 -> 189, and two query blocks, Distance, ws 31, 954 -> 1110,
// where registers bound them already).
constexpr int parts_of(int nk, int qh) { return nk >= 6 && qh == 1 ? 2 : 1; }

template <int NK, int CB, int QH, bool DIST, bool CPLX>
__global__ __launch_bounds__(64 * kW, 2) void sim_mx_kernel(SimArgs a) {
    const int item = (blockIdx.x & 7) * a.per_xcd + (blockIdx.x >> 3);
    if ((blockIdx.x >> 3) >= a.per_xcd || item >= a.nitems) return;
    constexpr int PF = CPLX ? 2 : 1;  // floats of a pixel in a plane
    constexpr int NPL = 16 / PF;      // planes (channels) at a time
    float *const lds = circatt_ldss;
    typedef __attribute__((address_space(3))) const char *lcp;
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)reinterpret_cast<uintptr_t>((lcp)(char *)lds));
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wh = wv % kNW, ww = wv / kNW;
    const int j = lane & 15, g = lane >> 4;
    const int jr = j & 3, jc = j >> 2;

    const int it = fdiv(item, a.div_strip), strip = item - it * a.nstrip;
    const int unit = fdiv(it, a.div_tiles), tile = it - unit * (a.tiles_h * a.tiles_w);
    const int tw = fdiv(tile, a.div_th);
    const int h0 = (tile - tw * a.tiles_h) * 4 * QH * kNW, w0 = tw * 4 * kNW;
    const int b0 = strip * CB;  // first block column
    const int64_t xo = (int64_t)unit * a.P * a.ncr;
    const i4v ry = dma_rsrc(a.y + xo, a.P * a.ncr * 4);
    const auto ryb = rsrc(a.y + xo, a.P * a.ncr * 4);
    const auto rxb = rsrc(a.x + xo, a.P * a.ncr * 4);

    const int hw = h0 + 4 * QH * wh, wc = w0 + 4 * ww;  // the wavefront's first pixel
    const int rh = hw + jr, rw = wc + jc;               // the lane's query, of the first block
    int rpix[QH];
#pragma unroll
    for (int b = 0; b < QH; ++b) rpix[b] = rh + 4 * b < a.n1 && rw < a.n2 ? rh + 4 * b + a.n1 * rw : 0;
    // byte offset of component k of the query, past the buffer from ncr on
    auto qoff = [&](int b, int k) {
        return k < a.ncr ? ((CPLX ? 2 * a.P * (k >> 1) + (k & 1) : a.P * k) + PF * rpix[b]) * 4 : kOut;
    };

    f4 acc[QH][NK * CB];
#pragma unroll
    for (int b = 0; b < QH; ++b)
#pragma unroll
        for (int i = 0; i < NK * CB; ++i) acc[b][i] = f4{0.f, 0.f, 0.f, 0.f};

    for (int c0 = 0; c0 < a.ncr; c0 += 16) {
        if (c0 > 0) __syncthreads();  // the previous components' reads are done
        {
            // task: 64 16-byte pieces (4 pixels of a column, or 2 complex
            // ones) of 4 planes
            const int npc = a.npx * PF / 4, ntile = (npc + 63) >> 6;
            const int cfirst = c0 / PF, clast = a.ncr / PF - 1;
            for (int t = wv; t < ntile * (NPL / 4); t += kW) {
                const int ti = t / (NPL / 4), cg = t - ti * (NPL / 4);
                const int pc = ti * 64 + lane, px_ = pc * (4 / PF);
                if (pc < npc && cfirst + 4 * cg <= clast) {
                    const int col = fdiv(px_, a.div_cr), row = px_ - col * a.cr;
                    const int gr = wrap(h0 - a.p + row, a.n1);
                    const int gc = wrap(w0 - a.p + 4 * b0 + col, a.n2);
                    const int vo = (gr + a.n1 * gc) * PF * 4;
                    // pieces that straddle the circular wrap: pixel by pixel
                    const bool cross = gr + 4 / PF > a.n1;
                    if (!cross) {
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            dma16(ry, lds0 + ((4 * cg + i) * a.pl + ti * 256) * 4, vo,
                                  min(cfirst + 4 * cg + i, clast) * a.P * PF * 4);
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const int so = min(cfirst + 4 * cg + i, clast) * a.P * PF * 4;
                            f4 v;
#pragma unroll
                            for (int q = 0; q < 4; ++q) {
                                const int r2 = gr + q / PF, o = (wrap(r2, a.n1) - gr) * PF + q % PF;
                                v[q] = load(ryb, vo + 4 * o + so);
                            }
                            *reinterpret_cast<f4 *>(lds + (4 * cg + i) * a.pl + 4 * pc) = v;
                        }
                    }
                }
            }
        }
        const int nc = min(16, a.ncr - c0);
        float q[QH];
#pragma unroll
        for (int b = 0; b < QH; ++b) q[b] = load(rxb, qoff(b, c0 + (DIST ? 0 : g)));
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();  // planes staged
        if constexpr (DIST) {
            // key rows 0 .. 3 of block column bc's column g
            const float *const kb = lds + (4 * QH * wh + a.cr * (4 * ww + g)) * PF;
            for (int k = 0; k < nc; k += PF) {
                float qn[QH], qi[QH];
#pragma unroll
                for (int b = 0; b < QH; ++b) {
                    qn[b] = load(rxb, qoff(b, c0 + min(k + PF, nc - 1)));
                    if constexpr (CPLX) qi[b] = load(rxb, qoff(b, c0 + k + 1));
                }
                const float *const kp = kb + k / PF * a.pl;
#pragma unroll
                for (int bc = 0; bc < CB; ++bc)
#pragma unroll
                    for (int br = 0; br < NK + QH - 1; ++br) {
                        const float *const kq = kp + 4 * bc * a.cr * PF + 4 * br * PF;
                        const f4 lo = *reinterpret_cast<const f4 *>(kq);
                        f4 re = lo, im;
                        if constexpr (CPLX) {
                            const f4 hi = *reinterpret_cast<const f4 *>(kq + 4);
                            re = f4{lo[0], lo[2], hi[0], hi[2]};
                            im = f4{lo[1], lo[3], hi[1], hi[3]};
                        }
#pragma unroll
                        for (int b = 0; b < QH; ++b) {  // (query block b meets its block row br - b)
                            if (br - b < 0 || br - b >= NK) continue;
                            f4 &s = acc[b][bc * NK + br - b];
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                const float d = q[b] - re[r];
                                s[r] = __builtin_fmaf(d, d, s[r]);
                                if constexpr (CPLX) {
                                    const float e = qi[b] - im[r];
                                    s[r] = __builtin_fmaf(e, e, s[r]);
                                }
                            }
                        }
                    }
#pragma unroll
                for (int b = 0; b < QH; ++b) q[b] = qn[b];
            }
        } else {
            // key (row j & 3, column j >> 2) of a block, component 4 s + g
            const float *const kb = lds + (4 * wh + jr + a.cr * (4 * ww + jc)) * PF + (CPLX ? (g >> 1) * a.pl + (g & 1) : g * a.pl);
            auto step = [&](int s, bool part) __attribute__((always_inline)) {
                const float *const kp = kb + (4 / PF) * s * a.pl;
#pragma unroll
                for (int bc = 0; bc < CB; ++bc)
#pragma unroll
                    for (int br = 0; br < NK; ++br) {
                        float kv = kp[4 * bc * a.cr * PF + 4 * br * PF];
                        if (part && 4 * s + g >= nc) kv = 0.f;
                        acc[0][bc * NK + br] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv, q[0], acc[0][bc * NK + br], 0, 0, 0);
                    }
            };
            const int full = nc >> 2;
            for (int s = 0; s < full; ++s) {
                const float qn = load(rxb, qoff(0, c0 + 4 * (s + 1) + g));
                step(s, false);
                q[0] = qn;
            }
            if (nc & 3) step(full, true);
        }
    }
    __syncthreads();  // the last reads are done: the wavefronts' regions overlay the planes

    // A query's scores of this strip, [window column from u0][slot of the
    // first dimension], then the slots' runs in memory: the window's columns
    // u0 .. are slots (u0 + s2) mod ws .. of the second dimension, in order up
    // to the wrap.
    float *const out = lds + wv * a.region;
    const float sc = DIST ? -0.5f * a.scale : a.scale;
    float *const nz = a.nz + (int64_t)unit * a.P * a.K;
    auto copy = [&](const float *src, float *dst, int n) __attribute__((always_inline)) {
        for (int e = 4 * lane; e < n; e += 256) {
            if (e + 3 < n) {
                *reinterpret_cast<f4u *>(dst + e) = *reinterpret_cast<const f4u *>(src + e);
            } else {
                for (int i = e; i < n; ++i) dst[i] = src[i];
            }
        }
    };
    // (LDS operations of a wavefront are in order)
    constexpr int NH = parts_of(NK, QH), QR = 16 / NH;
#pragma unroll
    for (int b = 0; b < QH; ++b) {
        const int s1 = slot_shift(min(rh + 4 * b, a.n1 - 1) + 1, a.n1, a.p);  // (rows past the image: any slots)
        const int uj = max(4 * b0 - jc, 0);
        int col[CB];
#pragma unroll
        for (int bc = 0; bc < CB; ++bc) {
            const int u2 = 4 * (b0 + bc) + g - jc;
            col[bc] = u2 >= 0 && u2 <= 2 * a.p ? j % QR * a.seg + (u2 - uj) * a.ws : 1 << 24;
        }
        const int dump = QR * a.seg;
        const int nr = min(4, a.n1 - hw - 4 * b);  // rows of the image
        for (int h = 0; h < NH; ++h) {
            if (j / QR == h) {
#pragma unroll
                for (int br = 0; br < NK; ++br)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int u1 = 4 * br + r - jr;
                        const int m1 = u1 >= 0 && u1 <= 2 * a.p ? wrap(u1 + s1, a.ws) : 1 << 24;
#pragma unroll
                        for (int bc = 0; bc < CB; ++bc) out[min(col[bc] + m1, dump)] = acc[b][bc * NK + br][r] * sc;
                    }
            }
            for (int c = QR / 4 * h; c < QR / 4 * (h + 1); ++c) {
                if (wc + c >= a.n2 || nr <= 0) break;
                float *const row = nz + (int64_t)(hw + 4 * b + a.n1 * (wc + c)) * a.K;
                const int s2 = slot_shift(wc + c + 1, a.n2, a.p);
                const int u0 = max(4 * b0 - c, 0), u1 = min(4 * (b0 + CB) - c, a.ws);  // window columns [u0, u1)
                if (u1 <= u0) continue;
                const int m0 = wrap(u0 + s2, a.ws), n0 = min(u1 - u0, a.ws - m0), n1 = u1 - u0 - n0;
                const float *const from = out + 4 * (c % (QR / 4)) * a.seg;
                if (a.seg == a.K && n1 == 0) {  // whole rows, one after the other
                    copy(from, row, nr * a.K);
                } else {
                    for (int r = 0; r < nr; ++r) {
                        copy(from + r * a.seg, row + r * a.K + m0 * a.ws, n0 * a.ws);
                        if (n1 > 0) copy(from + r * a.seg + n0 * a.ws, row + r * a.K, n1 * a.ws);
                    }
                }
            }
        }
    }
}

struct SimPlan {
    SimArgs a;
    int nk, qh, bytes;
    bool ok;
};
// qh: query blocks of a wavefront, one above the other (differences: two share
// the LDS reads of all but two of their block rows)
SimPlan sim_plan(int qh, const Geom &g, int C, int ncomp, int64_t nb) {
    SimPlan pl{};
    pl.qh = qh;
    if (g.nsp != 2 || g.p < 1 || g.ws > 33 || g.n1 < g.ws || g.n2 < g.ws || (int64_t)C * ncomp >= 1 << 28 ||
        g.P * g.K * 4 >= kMaxBytes || (int64_t)g.P * C * ncomp * 4 >= kMaxBytes)
        return pl;
    SimArgs &a = pl.a;
    a.n1 = g.n1;
    a.n2 = g.n2;
    a.P = (int)g.P;
    a.ws = g.ws;
    a.p = g.p;
    a.K = g.K;
    a.ncr = C * ncomp;
    pl.nk = 1 + (2 * g.p + 3) / 4;
    const int cb = strip_of(pl.nk);
    a.nstrip = (pl.nk + cb - 1) / cb;
    // 4 mod 8 pixels a column, planes 16 mod 32 pixels apart: the 4x4 pixels of
    // four planes fall on 64 banks
    const int hr = 4 * (qh * kNW + pl.nk - 1);
    a.cr = hr + (4 - hr % 8 + 8) % 8;
    const int ncol = 4 * (kNW + cb - 1);
    a.npx = a.cr * ncol;
    a.pl = (a.npx + (16 - a.npx % 32 + 32) % 32) * ncomp;
    // (halos that wrap once at most)
    if (g.n1 < a.cr - g.p || g.n2 < 4 * (kNW - 1 + a.nstrip * cb) - g.p) return pl;
    a.seg = cb == pl.nk ? a.K : std::min(4 * cb, g.ws) * g.ws;
    a.region = (16 / parts_of(pl.nk, qh) * a.seg + 1 + 3) / 4 * 4;
    pl.bytes = std::max(16 / ncomp * a.pl, kW * a.region) * 4;
    if (pl.bytes > kLds) return pl;
    a.tiles_h = (g.n1 + 4 * qh * kNW - 1) / (4 * qh * kNW);
    a.tiles_w = (g.n2 + 4 * kNW - 1) / (4 * kNW);
    const int64_t n = (int64_t)a.tiles_h * a.tiles_w * a.nstrip * nb;
    if (n > 1 << 27) return pl;
    a.nitems = (int)n;
    a.per_xcd = (a.nitems + 7) / 8;
    a.div_tiles = make_fastdiv((uint32_t)(a.tiles_h * a.tiles_w));
    a.div_th = make_fastdiv((uint32_t)a.tiles_h);
    a.div_strip = make_fastdiv((uint32_t)a.nstrip);
    a.div_cr = make_fastdiv((uint32_t)a.cr);
    pl.ok = true;
    return pl;
}

// Two query blocks from windows of 19 on, where that leaves two rounds of
// workgroups or more (us, one block, its rows put together whole, -> two;
// Distance, 32 components: 4 x 256x254, ws 21 503 -> 415, ws 31 1232 -> 954, with 64
// components 2180 -> 1620; 2 x 128x126, ws 31, 1280 workgroups of two, 171 -> 154,
// ws 25, 1024, 90 -> 91 (78 in halves); 200x120, ws 23, 780, 73 -> 103; at ws 17 whole
// windows no longer fit: 282 -> 292).
SimPlan sim_best(bool dist, const Geom &g, int C, int ncomp, int64_t nb) {
    if (dist && g.ws >= 19) {
        const SimPlan pl = sim_plan(2, g, C, ncomp, nb);
        if (pl.ok && pl.a.nitems >= 1200) return pl;
    }
    return sim_plan(1, g, C, ncomp, nb);
}

template <int NK, int QH, bool DIST, bool CPLX>
hipError_t launch_nk(const SimPlan &pl, hipStream_t s) {
    auto kern = sim_mx_kernel<NK, strip_of(NK), QH, DIST, CPLX>;
    static const hipError_t e =
        hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3(8u * (unsigned)pl.a.per_xcd), dim3(64 * kW), pl.bytes, s, pl.a);
    return hipGetLastError();
}
template <bool DIST, bool CPLX>
hipError_t launch_kind(const SimPlan &pl, hipStream_t s) {
    constexpr int Q = DIST ? 2 : 1;
    switch (pl.nk) {
    case 5: return launch_nk<5, 1, DIST, CPLX>(pl, s);
    case 6: return pl.qh == 1 ? launch_nk<6, 1, DIST, CPLX>(pl, s) : launch_nk<6, Q, DIST, CPLX>(pl, s);
    case 7: return pl.qh == 1 ? launch_nk<7, 1, DIST, CPLX>(pl, s) : launch_nk<7, Q, DIST, CPLX>(pl, s);
    case 8: return pl.qh == 1 ? launch_nk<8, 1, DIST, CPLX>(pl, s) : launch_nk<8, Q, DIST, CPLX>(pl, s);
    case 9: return pl.qh == 1 ? launch_nk<9, 1, DIST, CPLX>(pl, s) : launch_nk<9, Q, DIST, CPLX>(pl, s);
    }
    return hipErrorNotSupported;
}

}  // namespace

// Where this kernel runs; elsewhere the row kernel (windows to 15, which it
// matches for dot products at most: 4 x 320x320, ws 11, 32 components 138 us
// against 145) and the sub-row kernel (lines, wider windows).  Measured both ways
// (us, sub-row kernel -> this one, dot / Distance): 68x60, ws 17, 32 components
// 119/154 -> 18/36; 200x120, ws 23, 171/213 -> 48/73; 4 x 256x254, ws 17, 434/480 ->
// 159/282, ws 31 1294/1338 -> 575/954, 64 components 1488/1670 -> 844/1627.  Past
// 64 components the differences of windows 27 to 31 on large images stay: 4 x 256x254,
// ws 31, 72 components 1781 against 1806, 96 2164 against 2293; 2 units, ws 27, 72
// components 727 against 717, 96 860 against 900, ws 31 916 against 918 and 1068 against
// 1160; one unit (65024 pixels), ws 31, 72 689 -> 476; ws 33, 2 units, 72 components
// 1169 -> 920.
bool sim_mx_supported(bool dist, const Geom &g, int C, int ncomp, int64_t nb) {
    if (g.ws <= 15 || (dist && g.ws > 25 && g.ws < 33 && (int64_t)C * ncomp > 64 && g.P * nb > 100000)) return false;
    return sim_best(dist, g, C, ncomp, nb).ok;
}

hipError_t launch_sim_mx(bool dist, int ncomp, const Geom &g, int C, int64_t nb, float scale, const float *x,
                         const float *y, float *nz, hipStream_t s) {
    SimPlan pl = sim_best(dist, g, C, ncomp, nb);
    if (!pl.ok) return hipErrorNotSupported;
    pl.a.x = x;
    pl.a.y = y;
    pl.a.nz = nz;
    pl.a.scale = scale;
    if (ncomp == 2) return dist ? launch_kind<true, true>(pl, s) : launch_kind<false, true>(pl, s);
    return dist ? launch_kind<true, false>(pl, s) : launch_kind<false, false>(pl, s);
}

}  // namespace circatt
