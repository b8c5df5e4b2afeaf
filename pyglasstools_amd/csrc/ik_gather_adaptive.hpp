// ik_gather_adaptive.hpp -- field gather with the adaptive bond integral.
// Included by ik_gather_adaptive.hip.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "ik_bonds.hpp"
#include "ik_device.hpp"
#include "ik_geom.hpp"
#include "ik_launch.hpp"

namespace pgt {

// A wavefront takes P = 64 / lpp consecutive grid points of the Morton order
// (adaptive_points), lpp lanes per point, so that even a grid of a thousand
// points fills the GPU.  Each particle inside a point's ball adds its kinetic
// term, and each of its bonds the pair term with the bond integral
//   int_0^1 Delta(|x - (r_i + s r_ij)|^2) ds
// by QAG (qag_start, qag_refine), the integrand normalised as the reference
// integrates it (CoarseGrainFunction.h:42-45), so the tolerance tests see the
// same values.
//
// 1. The lanes of a point walk the cells around it side by side; the bonds of
//    the particles found go to a list shared by the wavefront.
// 2. When the list is full, and at the end: every listed integral gets the
//    15-point rule on its whole segment, one integral per lane.  Most are
//    done with that (a segment inside the ball is a polynomial for the Octic
//    kernel).
// 3. The others are listed in turn and bisected, one per lane, so that the
//    lanes of a wavefront bisect side by side; 32 or fewer of them by two
//    lanes each, one per half.
//
// What bounds it is the longest chain of bisections (about 20 for the Octic
// kernel at 1e-10, two 15-point rules each), so a lane must never wait for
// another's: dealing the integrals to lanes while walking the cells let one
// lane of a point integrate at a time, and a frame of 1,024 points (Octic,
// 1e-10) took 2,210 us; it takes 58 us.
//
// The kernel shape is chosen at run time (cg), the bond list is the FP64
// layout of BondLayout.  Terms are added to the points' FP64 sums in LDS in a
// fixed order.  GWS false: the interval table of each integral in private
// memory and LDS (kQagMax intervals), an integral that needs more sets
// *capped; GWS true: in the global workspace ws, wcap intervals per lane (the
// caller's limit), lane-interleaved.
struct AdaptCaps {
    static constexpr int MAXI = 512;  // listed integrals
};

template <int D, int OD, bool VIR, bool ELA, bool GWS>
__global__ __launch_bounds__(64) void k_gather_adaptive(Geom g, int n, int G, const double *__restrict__ grid,
                                                        const int *__restrict__ perm, int cg, AdaptQ Q,
                                                        double cgnorm, const int *__restrict__ cstart,
                                                        const double *__restrict__ spos,
                                                        const double *__restrict__ skin, int cap,
                                                        const int *__restrict__ bcount,
                                                        const double *__restrict__ bonds, GatherOut out,
                                                        int *__restrict__ capped, double *__restrict__ ws, int wcap,
                                                        int lpp)
{
    constexpr int MAXI = AdaptCaps::MAXI;
    constexpr int PS = (D == 2) ? 2 : 4;
    constexpr int KN = OD * (OD + 1) / 2;
    constexpr bool PAIRS = VIR || ELA;
    constexpr int KT = ((VIR ? KN : 0) + (ELA ? KN : 0)) | 1;
    using LY = BondLayout<D, OD, ELA, double>;
    constexpr int ES = LY::ES;
    __shared__ double s_x[64][3];         // the points
    __shared__ double s_acc[64][KT];      // their pair sums
    __shared__ int s_p[MAXI];             // listed integrals: particle,
    __shared__ unsigned s_pj[MAXI];       // point << 16 | bond
    __shared__ unsigned short s_hard[MAXI];  // those to bisect
    __shared__ double s_e[GWS ? 1 : kQagLds][64];

    const int f = blockIdx.y;
    const int lane = threadIdx.x;
    const int np = 64 / lpp;              // points of this wavefront (lpp a power of two)
    const int own = lane / lpp, sub = lane - own * lpp;
    const int t = xcd_tile(blockIdx.x, gridDim.x) * np + own;
    const bool live = t < G;
    const bool KIN = skin != nullptr;
    const double *sp = spos + (size_t)f * n * PS;
    const int *st = cstart + (size_t)f * (g.ncell + 1);
    const int *bc = bcount + (size_t)f * n;
    const double *bd = bonds + (size_t)f * n * (size_t)cap * ES;
    const double *sk = KIN ? skin + (size_t)f * n * KN : nullptr;

    const int gp = live ? perm[t] : 0;
    double x[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int a = 0; a < D; ++a) x[a] = grid[(size_t)gp * 3 + a];
    if (sub == 0)
#pragma unroll
        for (int a = 0; a < 3; ++a) s_x[own][a] = x[a];
#pragma unroll
    for (int k = 0; k < KT; ++k) s_acc[lane][k] = 0.0;
    double ak[KN];
#pragma unroll
    for (int k = 0; k < KN; ++k) ak[k] = 0.0;
    unsigned long long nball = 0, ncontrib = 0;
    bool hit_cap = false;

    using WS = typename std::conditional<GWS, QagGlobal, QagLds>::type;
    WS wsp;
    if constexpr (GWS) {
        wsp.p = ws + ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * 64 + lane;
        wsp.stride = (size_t)gridDim.x * gridDim.y * 64;
        wsp.n = wcap;
    } else {
        wsp.el = &s_e[0][lane];
    }

    // ---- integrate the first ni listed bonds --------------------------------
    auto flush = [&](int ni) {
        __syncthreads();
        // the segment of listed bond k: t(s) = A + s (B + s C)
        auto segment = [&](int k, double &A, double &B, double &C, const double *&e, int &pt) {
            const int p = s_p[k];
            const unsigned pj = s_pj[k];
            pt = (int)(pj >> 16);
            e = bd + ((size_t)p * cap + (pj & 0xffffu)) * ES;
            A = B = C = 0.0;
#pragma unroll
            for (int a = 0; a < D; ++a) {
                const double r = minimg(sp[(size_t)p * PS + a] - s_x[pt][a], g.L[a], g.pinvL[a]) * g.inv_rc;
                A = fma(r, r, A);
                B = fma(2.0 * r, e[a], B);
                C = fma(e[a], e[a], C);
            }
        };
        auto add = [&](int pt, const double *e, double w) {
            double v[KT];
            int q = 0;
            if constexpr (VIR) {
                const double c = w * e[LY::OC], c0 = c * e[0], c1 = c * e[1];
                v[q++] = c0 * e[0];
                v[q++] = c1 * e[1];
                if constexpr (OD == 2) {
                    v[q++] = c0 * e[1];
                } else {
                    v[q++] = c * e[2] * e[2];
                    v[q++] = c0 * e[1];
                    v[q++] = c0 * e[2];
                    v[q++] = c1 * e[2];
                }
            }
            if constexpr (ELA)
#pragma unroll
                for (int m = 0; m < KN; ++m) v[q++] = w * e[LY::OE + m];
#pragma unroll
            for (int m = 0; m < (VIR ? KN : 0) + (ELA ? KN : 0); ++m)
                __hip_atomic_fetch_add(&s_acc[pt][m], v[m], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        };
        int nh = 0;
        for (int k0 = 0; k0 < ni; k0 += 64) {
            const int k = k0 + lane;
            bool hard = false;
            if (k < ni) {
                double A, B, C;
                const double *e;
                int pt;
                segment(k, A, B, C, e, pt);
                auto obj = [&](double sv) { return cgnorm * shape_rt(cg, fma(sv, fma(sv, C, B), A)); };
                const QagStart s = qag_start(obj, Q);
                hard = !s.done;
                if (s.done) add(pt, e, s.result / cgnorm);
            }
            const unsigned long long bm = __builtin_amdgcn_ballot_w64(hard);
            if (hard)
                s_hard[nh + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(bm >> 32),
                                                           __builtin_amdgcn_mbcnt_lo((unsigned)bm, 0u))] =
                    (unsigned short)k;
            nh += __popcll(bm);
        }
        __syncthreads();
        auto bisect = [&](int k, bool add_it, auto pair) {
            double A, B, C;
            const double *e;
            int pt;
            segment(s_hard[k], A, B, C, e, pt);
            auto obj = [&](double sv) { return cgnorm * shape_rt(cg, fma(sv, fma(sv, C, B), A)); };
            const QagStart s = qag_start(obj, Q);
            const double w = qag_refine<decltype(pair)::value>(obj, Q, s, hit_cap, wsp);
            if (add_it) add(pt, e, w / cgnorm);
        };
        int k0 = 0;
        for (; nh - k0 > 32; k0 += 64)
            if (k0 + lane < nh) bisect(k0 + lane, true, std::false_type());
        if (k0 + (lane >> 1) < nh) bisect(k0 + (lane >> 1), !(lane & 1), std::true_type());
        __syncthreads();
    };

    // ---- walk the cells, the lanes of a point side by side -------------------
    {
        const int cx = cell_coord(g, 0, x[0]), cy = cell_coord(g, 1, x[1]), cz = cell_coord(g, 2, x[2]);
        int rows[kMaxRows];
        const int nrows = neighbour_rows(g, cy, cz, rows);  // as many in every lane
        int r = -1, c0 = 0, len0 = 0, len = 0, b0 = 0, b1 = 0;
        // the step's candidate of this lane and its bonds, listed up to `base`
        int p = 0, nb = 0, before = 0, total = 0, base = 0;
        for (bool more = true; more;) {
            int ni = 0;  // listed integrals (the same in every lane)
            for (;;) {
                if (base < total) {
                    if (base == 0 && ni > 0 && ni + total > MAXI) break;  // a step is not split over two lists
                    const int first = ni + before - base;
                    for (int j = max(0, -first); j < nb && first + j < MAXI; ++j) {
                        s_p[first + j] = p;
                        s_pj[first + j] = (unsigned)own << 16 | (unsigned)j;
                    }
                    const int placed = min(total - base, MAXI - ni);
                    ni += placed;
                    base += placed;  // more bonds than a list holds: the rest in the next
                    if (base < total) break;
                }
                c0 += lpp;
                while (r < nrows && __builtin_amdgcn_ballot_w64(c0 < len) == 0ull) {
                    ++r;
                    c0 = 0;
                    if (r < nrows) {  // the row as one run of candidates
                        int rb[2], re[2];
                        const int nr = row_ranges(g, st, rows[r], cx, rb, re);
                        b0 = rb[0];
                        len0 = re[0] - rb[0];
                        b1 = nr > 1 ? rb[1] : 0;
                        len = live ? len0 + (nr > 1 ? re[1] - rb[1] : 0) : 0;
                    }
                }
                more = r < nrows;
                if (!more) break;
                const int c = c0 + sub;
                nb = 0;
                if (c < len) {
                    p = c < len0 ? b0 + c : b1 + (c - len0);
                    double asq = 0.0;
#pragma unroll
                    for (int a = 0; a < D; ++a) {
                        const double d = minimg(sp[(size_t)p * PS + a] - x[a], g.L[a], g.pinvL[a]);
                        asq = a == 0 ? d * d : fma(d, d, asq);
                    }
                    if (asq < g.rc2) {
                        ++nball;
                        if (KIN) {
                            const double w = shape_rt(cg, asq * g.inv_rc2);
#pragma unroll
                            for (int k = 0; k < KN; ++k) ak[k] = fma(w, sk[(size_t)p * KN + k], ak[k]);
                        }
                        if constexpr (PAIRS) nb = min(bc[p], cap);
                    }
                }
                if constexpr (PAIRS) {
                    ncontrib += (unsigned long long)nb;
                    int v = nb;
#pragma unroll
                    for (int off = 1; off < 64; off <<= 1) {
                        const int u = __shfl_up(v, off, 64);
                        if (lane >= off) v += u;
                    }
                    total = __builtin_amdgcn_readlane(v, 63);
                    before = v - nb;
                    base = 0;
                }
            }
            if constexpr (PAIRS)
                if (ni > 0) flush(ni);
        }
    }
    __syncthreads();

    // the point's lanes: a fixed butterfly over the lpp lanes of the group
    if (KIN)
        for (int m = 1; m < lpp; m <<= 1)
#pragma unroll
            for (int k = 0; k < KN; ++k) ak[k] += __shfl_xor(ak[k], m, 64);
    if (live && sub == 0) {
        const size_t ob = ((size_t)f * G + gp) * OD * OD;
        auto store = [&](double *dst, const double *acc, double scale) {
            for (int aa = 0; aa < OD; ++aa) dst[ob + aa + OD * aa] = acc[aa] * scale;
            if (OD == 2) {
                dst[ob + 1] = acc[2] * scale;
                dst[ob + 2] = acc[2] * scale;
            } else {
                dst[ob + 1] = dst[ob + 3] = acc[3] * scale;
                dst[ob + 2] = dst[ob + 6] = acc[4] * scale;
                dst[ob + 5] = dst[ob + 7] = acc[5] * scale;
            }
        };
        if (VIR) store(out.vir, s_acc[own], 1.0);
        if (ELA) store(out.ela, s_acc[own] + (VIR ? KN : 0), 1.0);
        if (KIN) store(out.kin, ak, cgnorm);
    }
    if (hit_cap) atomicOr(capped, 1);
    nball = wave_sum(nball);
    ncontrib = wave_sum(ncontrib);
    if (lane == 0) {
        const size_t w = (size_t)blockIdx.y * gridDim.x + blockIdx.x;
        out.wave_counts[2 * w] = nball;
        out.wave_counts[2 * w + 1] = ncontrib;
    }
}

}  // namespace pgt
