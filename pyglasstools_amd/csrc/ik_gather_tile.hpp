// ik_gather_tile.hpp -- the item-balanced field gather ("tile" gather) of
// the IK stress-field engine.  Included by ik_gather_launch.hpp.
//
// A workgroup is one wavefront and takes a tile: up to 64 neighbouring grid
// points (a block of the grid's Morton order).  Work items are the (grid
// point, particle) pairs with the particle inside the point's ball; an item
// integrates the particle's bonds for the point.
//
// 1. Window: the particles within r_cg of the tile's bounding box, read from
//    the rows of cells that cover it, one particle per lane, into a list in
//    LDS.
// 2. Masks: a lane holds one window particle and tests it against every point
//    of the tile (FP64, |a|^2 < r_cg^2; the points are broadcast from LDS),
//    which gives the particle's mask of points.
// 3. Items: the particles are ordered by bond count, largest first, and their
//    items written to a list in that order, a particle's items side by side.
// 4. Integration: lane l takes items l, l + 64, ...: the 64 items of a step
//    have nearly equal bond counts, so the bond loop wastes few lanes
//    whatever the spread of the counts, and neighbouring lanes mostly share
//    their particle, so that a load of bond entries touches the entries of
//    about nine particles instead of 64.  A lane sums its item in registers
//    and adds it to the point's FP64 accumulators in LDS.
//
// The wavefront runs alone in its workgroup and every step is in a fixed
// order, so the sums are the same from run to run.
//
// Why particles, not points, are spread over the lanes in the scan: scattered
// loads pace this kernel (a CU's L1 takes about one lane's 16 bytes a cycle
// when the lanes' lines differ).  With a point per lane, each lane walked its
// own cells and every item fetched its particle from memory: 216 loads a
// wavefront on the 2D N = 65,536 job with a 256^2 grid.  Here a window
// particle is loaded once per tile, and an item's entries are shared by its
// neighbours.  Measured against that scan (one launch): 100 such frames
// 1.68 -> 1.38 ms, 3D N = 131,072 with a 64^3 grid, FP32 form, 20 frames
// 4.30 -> 3.72 ms, 3D FP64 with the kinetic field, N = 20,011, 5 frames
// 0.43 -> 0.37 ms, a sweep of eight systems whose grids are up to 2.4 r_cg / 2
// apart 0.80 -> 0.65 ms.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "ik_bonds.hpp"
#include "ik_device.hpp"
#include "ik_gather.hpp"
#include "ik_geom.hpp"
#include "ik_launch.hpp"
#include "ik_sweep.hpp"

namespace pgt {

// Capacities of the tile gather.
struct TileCaps {
    static constexpr int BLK = kTileThreads;  // one wavefront
    static constexpr int TP = kTilePoints;    // most grid points of a tile
    static constexpr int MAXW = 128;          // window particles listed at a time
    static constexpr int MAXI = 1024;         // items listed at a time
    static constexpr int SBITS = 8;           // item word: window slot | point << SBITS
    static constexpr int MAXNB = 255;         // bond count of a particle (one byte); more: overflow
    static_assert(TP == 64 && BLK == 64, "one wavefront, masks of 64 points");
    static_assert(MAXW <= (1 << SBITS) && MAXW % 64 == 0, "window slots of an item word");
};

template <typename T>
__device__ __forceinline__ T wave_max(T v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = max(v, __shfl_xor(v, off, 64));
    return v;
}

template <typename T>
__device__ __forceinline__ T wave_min(T v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v = min(v, __shfl_xor(v, off, 64));
    return v;
}

// Wavefronts per SIMD the compiler sizes registers for: four for the 2D forms
// without elastic terms (a few registers spilled at most) and for the 3D FP32
// virial form (126 registers, no spill; 131 and three waves unbounded, with
// the gather 7% slower on the 3D N = 131,072 job), which hides more memory
// latency; the others are left to the compiler (two or three: the 3D FP64
// virial form would spill 88 bytes a lane at four).
template <int D, bool ELA, bool KIN, typename ER>
struct TileWaves {
    static constexpr bool F32 = std::is_same<ER, float>::value;
    static constexpr int value = ((D == 2 && !ELA) || (D == 3 && F32 && !ELA && !KIN)) ? 4 : 1;
};

// Cells of one axis that hold every particle within r of [lo, hi]: w0 (in
// [0, nc)) and wn cells from it, taken periodically; the whole axis when
// they would reach around it.  The margin covers the rounding of the cell
// coordinates, and bounds that are not finite give the whole axis.
__device__ __forceinline__ void axis_cells(const Geom &g, int a, double lo, double hi, double r, int &w0, int &wn)
{
    const int nc = g.nc[a];
    w0 = 0;
    wn = nc;
    if (nc == 1) return;
    const double m = r + 1e-10 * (fabs(lo) + fabs(hi) + g.L[a]);
    const double f0 = floor((lo - m - g.lo[a]) / g.cs[a]), f1 = floor((hi + m - g.lo[a]) / g.cs[a]);
    if (!(f1 - f0 + 1.0 < (double)nc)) return;
    const int k = (int)(f0 - (double)nc * floor(f0 / (double)nc));
    w0 = k < 0 ? 0 : (k >= nc ? nc - 1 : k);
    wn = (int)(f1 - f0) + 1;
}

// The body works on one frame's arrays (cell starts st, sorted positions
// sp, kinetic terms sk, bond counts bc, entries bd; out's field pointers at
// the frame's first value) for the cnt points from t0 on of the Morton order
// perm (cnt <= 0: none), and stores its counts at out.wave_counts[2 wi ..].
template <int D, int OD, int CG, int NQ, bool VIR, bool ELA, bool KIN, typename ER>
__device__ __forceinline__ void gather_tile_body(const Geom &g, int n, const double *__restrict__ grid,
                                                 const int *__restrict__ perm, const GLRule &R,
                                                 const double *__restrict__ gld, double cgnorm,
                                                 const int *__restrict__ st, const double *__restrict__ sp,
                                                 const double *__restrict__ sk, int cap,
                                                 const int *__restrict__ bc, const ER *__restrict__ bd,
                                                 const GatherOut &out, size_t wi, int t0, int cnt,
                                                 int *__restrict__ overflow)
{
    using CP = TileCaps;
    using LY = BondLayout<D, OD, ELA, ER>;
    constexpr int MAXW = CP::MAXW, MAXI = CP::MAXI, SBITS = CP::SBITS;
    constexpr int PS = (D == 2) ? 2 : 4;
    constexpr int KN = OD * (OD + 1) / 2;
    constexpr bool PAIRS = VIR || ELA;
    constexpr int KV = (VIR ? KN : 0) + (ELA ? KN : 0);  // pair accumulators per point
    constexpr int KT = KV + (KIN ? KN : 0);             // all accumulators per point
    constexpr int KTA = KT | 1;  // accumulator stride: odd, so 64 points fall on distinct LDS banks
    constexpr int KNA = KIN ? KN : 1;
    constexpr int ES = LY::ES;    // values per entry
    constexpr int GRP = LY::GRP;  // entries per read group
    constexpr int GV = LY::GV;    // values per read group

    __shared__ double s_pt[64][PS];              // the tile's points (NaN beyond them)
    __shared__ double s_acc[64][KTA];            // their accumulators
    __shared__ double s_wp[MAXW][D];             // window: positions,
    __shared__ int s_wid[MAXW];                  // particles,
    __shared__ unsigned long long s_wm[MAXW];    // point masks,
    __shared__ unsigned char s_wnb[MAXW];        // bond counts,
    __shared__ unsigned short s_wof[MAXW];       // first items
    __shared__ unsigned short s_item[MAXI];      // items in order
    __shared__ int s_bucket[64];                 // items per bond count, then their offsets
    __shared__ int s_seg[64], s_segb[64];        // segments of cells: first candidate, first particle

    const int l = threadIdx.x;
    if (cnt <= 0) {
        if (l == 0) {
            out.wave_counts[2 * wi] = 0;
            out.wave_counts[2 * wi + 1] = 0;
        }
        return;
    }
    const bool live = l < cnt;
    const int gp = perm[t0 + (live ? l : 0)];
    double xg[D];
#pragma unroll
    for (int a = 0; a < D; ++a) xg[a] = grid[(size_t)gp * 3 + a];
#pragma unroll
    for (int a = 0; a < D; ++a) s_pt[l][a] = live ? xg[a] : __builtin_nan("");
#pragma unroll
    for (int k = 0; k < KTA; ++k) s_acc[l][k] = 0.0;

    // bounding box of the points: centre xc, half lengths xh.  When the box
    // and its ball fit in less than a period (near), a particle has one image
    // that can be inside any of the balls, the one nearest to xc.
    double xc[D], xh[D];
    int w0[3] = {0, 0, 0}, wn[3] = {1, 1, 1};
    bool near = true;
#pragma unroll
    for (int a = 0; a < D; ++a) {
        const double lo = wave_min(xg[a]), hi = wave_max(xg[a]);
        axis_cells(g, a, lo, hi, g.rc, w0[a], wn[a]);
        w0[a] = __builtin_amdgcn_readfirstlane(w0[a]);
        wn[a] = __builtin_amdgcn_readfirstlane(wn[a]);
        xc[a] = 0.5 * (lo + hi);
        xh[a] = 0.5 * (hi - lo);
        near = near && (g.pinvL[a] == 0.0 || 2.0 * (xh[a] + g.rc) < 0.999 * g.L[a]);
    }

    unsigned long long nball = 0;     // items, per lane
    unsigned long long ncontrib = 0;  // bond counts of the items, per lane
    bool over = false;                // an item's bond count exceeds MAXNB
    const double s2 = 2.0 * g.inv_rc;

    // ---- integrate items 0 .. ni - 1 of the list --------------------------
    auto integrate = [&](int ni) {
        // the next item's first bond entries and kinetic term are loaded
        // before the current one is integrated
        auto fetch = [&](int k, int &slot, int &ip, int &nb, double (&kk)[KNA], ER (&E)[GV]) {
            const bool valid = k < ni;
            const unsigned it = s_item[valid ? k : 0];
            slot = (int)(it & ((1u << SBITS) - 1u));
            ip = (int)(it >> SBITS);
            const int p = s_wid[slot];
            nb = (PAIRS && valid) ? (int)s_wnb[slot] : 0;
            if constexpr (KIN)
#pragma unroll
                for (int q = 0; q < KN; ++q) kk[q] = sk[(size_t)p * KN + q];
            if constexpr (PAIRS)
                if (nb > 0) load_entry<ER, GV>(bd + (size_t)p * cap * ES, E);
        };
        int slot, ip, nb;
        double kk[KNA];
        ER E0[GV];
        fetch(l, slot, ip, nb, kk, E0);
        for (int k0 = 0; k0 < ni; k0 += 64) {
            const int k = k0 + l;
            int nslot, nip, nnb;
            double nkk[KNA];
            ER nE0[GV];
            fetch(k + 64, nslot, nip, nnb, nkk, nE0);
            if (k < ni) {
                double a[3];
                a[0] = minimg(s_wp[slot][0] - s_pt[ip][0], g.L[0], g.pinvL[0]);
                a[1] = minimg(s_wp[slot][1] - s_pt[ip][1], g.L[1], g.pinvL[1]);
                a[2] = 0.0;
                if constexpr (D == 3) a[2] = minimg(s_wp[slot][D - 1] - s_pt[ip][D - 1], g.L[2], g.pinvL[2]);
                const double A = (a[0] * a[0] + a[1] * a[1] + a[2] * a[2]) * g.inv_rc2;
                double acc[KTA];
#pragma unroll
                for (int q = 0; q < KTA; ++q) acc[q] = 0.0;
                if constexpr (KIN) {
                    const double wk = shape<CG, double>(A);
#pragma unroll
                    for (int q = 0; q < KN; ++q) acc[KV + q] = wk * kk[q];
                }
                if constexpr (PAIRS) {
                    ER ta[3];
                    ta[0] = (ER)(a[0] * s2);
                    ta[1] = (ER)(a[1] * s2);
                    ta[2] = (ER)(a[2] * s2);
                    const ER Aj = (ER)A;
                    auto one = [&](const ER (&Gv)[GV], auto O) {
                        constexpr int o = decltype(O)::value;
                        const ER *e = Gv + o;
                        ER C = e[0] * e[0];
                        C = fma(e[1], e[1], C);
                        if (D == 3) C = fma(e[2], e[2], C);
                        ER B = ta[0] * e[0] + ta[1] * e[1];
                        if (D == 3) B = fma(ta[2], e[2], B);
                        const ER wq = bond_quad<CG, NQ, ER>(R, gld, R.n, Aj, B, C);
                        if constexpr (VIR) {
                            const ER c = wq * e[LY::OC];
                            const ER cb0 = c * e[0], cb1 = c * e[1];
                            if constexpr (std::is_same<ER, double>::value) {
                                acc[0] = fma(cb0, e[0], acc[0]);
                                acc[1] = fma(cb1, e[1], acc[1]);
                                if constexpr (OD == 2) {
                                    acc[2] = fma(cb0, e[1], acc[2]);
                                } else {
                                    const ER cb2 = c * e[2];
                                    acc[2] = fma(cb2, e[2], acc[2]);
                                    acc[3] = fma(cb0, e[1], acc[3]);
                                    acc[4] = fma(cb0, e[2], acc[4]);
                                    acc[5] = fma(cb1, e[2], acc[5]);
                                }
                            } else if constexpr (OD == 2) {
                                // FP32 entries, 2D: products in FP32, sums
                                // in FP64 (the registers of the 3D form
                                // below would spill here)
                                acc[0] += (double)(cb0 * e[0]);
                                acc[1] += (double)(cb1 * e[1]);
                                acc[2] += (double)(cb0 * e[1]);
                            } else {
                                // FP32 entries, 3D: c' w and b' widened, the
                                // products and sums in FP64
                                const double cd = (double)c, d0 = (double)e[0], d1 = (double)e[1];
                                const double d2 = (double)e[2];
                                const double q0 = cd * d0, q1 = cd * d1, q2 = cd * d2;
                                acc[0] = fma(q0, d0, acc[0]);
                                acc[1] = fma(q1, d1, acc[1]);
                                acc[2] = fma(q2, d2, acc[2]);
                                acc[3] = fma(q0, d1, acc[3]);
                                acc[4] = fma(q0, d2, acc[4]);
                                acc[5] = fma(q1, d2, acc[5]);
                            }
                        }
                        if constexpr (ELA) {
                            constexpr int EO = VIR ? KN : 0;
#pragma unroll
                            for (int q = 0; q < KN; ++q) {
                                if constexpr (std::is_same<ER, double>::value)
                                    acc[EO + q] = fma(wq, e[LY::OE + q], acc[EO + q]);
                                else acc[EO + q] += (double)(wq * e[LY::OE + q]);
                            }
                        }
                    };
                    auto group = [&](const ER (&Gv)[GV], int kk2) {
                        one(Gv, std::integral_constant<int, 0>());
                        if constexpr (GRP >= 2)
                            if (GRP * kk2 + 1 < nb) one(Gv, std::integral_constant<int, ES>());
                        if constexpr (GRP >= 3)
                            if (GRP * kk2 + 2 < nb) one(Gv, std::integral_constant<int, 2 * ES>());
                        if constexpr (GRP >= 4)
                            if (GRP * kk2 + 3 < nb) one(Gv, std::integral_constant<int, 3 * ES>());
                    };
                    const ER *ptr = bd + (size_t)s_wid[slot] * cap * ES;
                    const int ng = (nb + GRP - 1) / GRP;
                    ER E1[GV];
                    int kk2 = 0;
                    for (; kk2 + 1 < ng; kk2 += 2) {
                        load_entry<ER, GV>(ptr + (size_t)(kk2 + 1) * GV, E1);
                        group(E0, kk2);
                        if (kk2 + 2 < ng) load_entry<ER, GV>(ptr + (size_t)(kk2 + 2) * GV, E0);
                        group(E1, kk2 + 1);
                    }
                    if (kk2 < ng) group(E0, kk2);
                }
#pragma unroll
                for (int q = 0; q < KT; ++q)
                    __hip_atomic_fetch_add(&s_acc[ip][q], acc[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
            }
            slot = nslot;
            ip = nip;
            nb = nnb;
            if constexpr (KIN)
#pragma unroll
                for (int q = 0; q < KN; ++q) kk[q] = nkk[q];
            if constexpr (PAIRS)
#pragma unroll
                for (int q = 0; q < GV; ++q) E0[q] = nE0[q];
        }
        __syncthreads();
    };

    // ---- the items of window particles 0 .. nw - 1 --------------------------
    auto process = [&](int nw) {
        s_bucket[l] = 0;
        __syncthreads();
        for (int r = 0; r < nw; r += 64) {
            const int slot = r + l;
            const bool valid = slot < nw;
            const int ws = valid ? slot : 0;
            int nbc = 0;
            if constexpr (PAIRS) nbc = min(bc[s_wid[ws]], cap);
            double x[D];
#pragma unroll
            for (int a = 0; a < D; ++a) x[a] = s_wp[ws][a];
            bool shift = !near;
#pragma unroll
            for (int a = 0; a < D; ++a) shift = shift || !(rint((x[a] - xc[a]) * g.pinvL[a]) == 0.0);
            // bit j of the mask: the particle is in point j's ball.  Bits
            // enter at the low end (m = 2 m + bit, one add with carry).
            unsigned m[2] = {0u, 0u};
            auto test = [&](auto image) {
                constexpr bool IMAGE = decltype(image)::value;
#pragma unroll
                for (int h = 1; h >= 0; --h) {
                    if (32 * h >= cnt) continue;
                    unsigned mm = 0u;
#pragma unroll 4
                    for (int j = 31; j >= 0; --j) {
                        double d[3] = {0.0, 0.0, 0.0};
#pragma unroll
                        for (int a = 0; a < D; ++a) {
                            d[a] = x[a] - s_pt[32 * h + j][a];
                            if constexpr (IMAGE) d[a] = minimg(d[a], g.L[a], g.pinvL[a]);
                        }
                        const bool in = d[0] * d[0] + d[1] * d[1] + d[2] * d[2] < g.rc2;
                        mm = mm + mm + (in ? 1u : 0u);
                    }
                    m[h] = mm;
                }
            };
            // no lane's particle needs another image: the plain difference is
            // the minimum image of every pair that can be inside a ball
            if (__builtin_amdgcn_ballot_w64(shift) == 0ull) test(std::false_type());
            else test(std::true_type());
            if (!valid) m[0] = m[1] = 0u;
            const int pc = __popc(m[0]) + __popc(m[1]);
            if (nbc > CP::MAXNB && pc > 0) over = true;
            const int nb = min(nbc, CP::MAXNB);
            nball += (unsigned long long)pc;
            ncontrib += (unsigned long long)pc * (unsigned long long)nb;
            if (valid) {
                s_wnb[slot] = (unsigned char)nb;
                s_wm[slot] = (unsigned long long)m[1] << 32 | m[0];
                atomicAdd(&s_bucket[63 - min(nb, 63)], pc);
            }
        }
        __syncthreads();
        int total;
        {
            const int c = s_bucket[l];
            int v = c;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const int u = __shfl_up(v, off, 64);
                if (l >= off) v += u;
            }
            total = __builtin_amdgcn_readlane(v, 63);
            __syncthreads();
            s_bucket[l] = v - c;  // first item of the bond count
        }
        __syncthreads();
        for (int base = 0; base < total; base += MAXI) {
            for (int r = 0; r < nw; r += 64) {
                const int slot = r + l;
                if (slot < nw) {
                    const unsigned long long mk = s_wm[slot];
                    unsigned m0 = (unsigned)mk, m1 = (unsigned)(mk >> 32);
                    int k;
                    if (base == 0) {
                        // an LDS atomic; the lanes of one instruction are
                        // served in a fixed order
                        k = atomicAdd(&s_bucket[63 - min((int)s_wnb[slot], 63)], __popc(m0) + __popc(m1));
                        s_wof[slot] = (unsigned short)k;
                    } else {
                        k = s_wof[slot] - base;
                    }
                    while (m0 | m1) {
                        const bool low = m0 != 0u;
                        const unsigned mm = low ? m0 : m1;
                        const int j = __ffs(mm) - 1 + (low ? 0 : 32);
                        const unsigned rest = mm & (mm - 1u);
                        m0 = low ? rest : 0u;
                        m1 = low ? m1 : rest;
                        if ((unsigned)k < (unsigned)MAXI) s_item[k] = (unsigned short)(slot | (j << SBITS));
                        ++k;
                    }
                }
            }
            __syncthreads();
            integrate(min(total - base, MAXI));
        }
    };

    // ---- window: candidates of the cell rows, in segments of one row --------
    const int nx = g.nc[0], ny = g.nc[1], nz = g.nc[2];
    const int parts = w0[0] + wn[0] > nx ? 2 : 1;  // a row that wraps is two segments
    const int nseg = wn[1] * wn[2] * parts;
    const double rr = g.rc2 * (1.0 + 1e-9);
    int nw = 0;
    for (int s0 = 0; s0 < nseg; s0 += 64) {
        int b = 0, len = 0;
        if (s0 + l < nseg) {
            const int r = (s0 + l) / parts, part = (s0 + l) - r * parts;
            const int iz = r / wn[1], iy = r - iz * wn[1];
            const int z = w0[2] + iz < nz ? w0[2] + iz : w0[2] + iz - nz;
            const int y = w0[1] + iy < ny ? w0[1] + iy : w0[1] + iy - ny;
            const int row = (z * ny + y) * nx;
            b = st[part ? row : row + w0[0]];
            len = st[part ? row + w0[0] + wn[0] - nx : row + min(w0[0] + wn[0], nx)] - b;
        }
        int v = len;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int u = __shfl_up(v, off, 64);
            if (l >= off) v += u;
        }
        const int total = __builtin_amdgcn_readlane(v, 63);
        __syncthreads();
        s_seg[l] = v - len;
        s_segb[l] = b;
        __syncthreads();
        const int ns = min(nseg - s0, 64);
        for (int c0 = 0; c0 < total; c0 += 64) {
            const int c = min(c0 + l, total - 1);
            // the last segment that starts at or before candidate c
            int lo = 0;
#pragma unroll
            for (int h = 32; h > 0; h >>= 1)
                if (lo + h < ns && s_seg[lo + h] <= c) lo += h;
            const int id = s_segb[lo] + c - s_seg[lo];
            double x[D], d2 = 0.0;
#pragma unroll
            for (int a = 0; a < D; ++a) x[a] = sp[(size_t)id * PS + a];
#pragma unroll
            for (int a = 0; a < D; ++a) {
                const double d = fmax(fabs(minimg(x[a] - xc[a], g.L[a], g.pinvL[a])) - xh[a], 0.0);
                d2 = fma(d, d, d2);
            }
            // not near: any image may matter, so every candidate is kept
            const bool in = c0 + l < total && (!near || d2 < rr);
            const unsigned long long bm = __builtin_amdgcn_ballot_w64(in);
            const int k = __popcll(bm);
            if (nw + k > MAXW) {
                __syncthreads();
                process(nw);
                nw = 0;
            }
            if (in) {
                const int w = nw + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(bm >> 32),
                                                                  __builtin_amdgcn_mbcnt_lo((unsigned)bm, 0u));
                s_wid[w] = id;
#pragma unroll
                for (int a = 0; a < D; ++a) s_wp[w][a] = x[a];
            }
            nw += k;
        }
    }
    __syncthreads();
    if (nw > 0) process(nw);
    __syncthreads();

    if (live) {
        const size_t ob = (size_t)gp * OD * OD;
        double av[KN], ae[KN], ak[KN];
#pragma unroll
        for (int k = 0; k < KN; ++k) {
            av[k] = VIR ? s_acc[l][k] : 0.0;
            ae[k] = ELA ? s_acc[l][(VIR ? KN : 0) + k] : 0.0;
            ak[k] = KIN ? s_acc[l][KV + k] : 0.0;
        }
        auto store = [&](double *dst, const double *acc, double scale) {
            for (int a = 0; a < OD; ++a) dst[ob + a + OD * a] = acc[a] * scale;
            if constexpr (OD == 2) {
                dst[ob + 1] = acc[2] * scale;
                dst[ob + 2] = acc[2] * scale;
            } else {
                dst[ob + 1] = dst[ob + 3] = acc[3] * scale;
                dst[ob + 2] = dst[ob + 6] = acc[4] * scale;
                dst[ob + 5] = dst[ob + 7] = acc[5] * scale;
            }
        };
        if (VIR) store(out.vir, av, 1.0);
        if (ELA) store(out.ela, ae, 1.0);
        if (KIN) store(out.kin, ak, cgnorm);
    }
    nball = wave_sum(nball);
    ncontrib = wave_sum(ncontrib);
    if (l == 0) {
        out.wave_counts[2 * wi] = nball;
        out.wave_counts[2 * wi + 1] = ncontrib;
    }
    if (over) atomicOr(overflow, 2);
}

// The points of workgroup b of a frame: tile b / (64 / tp), its tp points
// from b mod (64 / tp) times tp on (tp 64: the whole tile).  tiles[k] is
// where tile k starts in the Morton order.
__device__ __forceinline__ void tile_points(const int *__restrict__ tiles, int b, int tp, int &t0, int &cnt)
{
    const int sub = kTilePoints / tp, k = b / sub;
    t0 = tiles[k] + (b - k * sub) * tp;
    cnt = min(tiles[k + 1] - t0, tp);
}

// One frame per y row; block x takes the points of tile_points(xcd_tile(x,
// gridDim.x)), so each XCD works through a contiguous eighth of the frame's
// points.
template <int D, int OD, int CG, int NQ, bool VIR, bool ELA, bool KIN, typename ER>
__global__ __launch_bounds__(64, (TileWaves<D, ELA, KIN, ER>::value)) void k_gather_tile(
    Geom g, int n, int G, const double *__restrict__ grid, const int *__restrict__ perm,
    const int *__restrict__ tiles, int tp, GLRule R, const double *__restrict__ gld, double cgnorm,
    const int *__restrict__ cstart, const double *__restrict__ spos, const double *__restrict__ skin, int cap,
    const int *__restrict__ bcount, const ER *__restrict__ bonds, GatherOut out, int *__restrict__ overflow)
{
    constexpr int PS = (D == 2) ? 2 : 4;
    constexpr int KN = OD * (OD + 1) / 2;
    constexpr int ES = BondLayout<D, OD, ELA, ER>::ES;
    const int f = blockIdx.y;
    const size_t fo = (size_t)f * n, oo = (size_t)f * G * OD * OD;
    GatherOut of = out;
    if (VIR) of.vir = out.vir + oo;
    if (ELA) of.ela = out.ela + oo;
    if (KIN) of.kin = out.kin + oo;
    int t0, cnt;
    tile_points(tiles, xcd_tile(blockIdx.x, gridDim.x), tp, t0, cnt);
    gather_tile_body<D, OD, CG, NQ, VIR, ELA, KIN, ER>(
        g, n, grid, perm, R, gld, cgnorm, cstart + (size_t)f * (g.ncell + 1), spos + fo * PS,
        KIN ? skin + fo * KN : nullptr, cap, bcount + fo, bonds + fo * (size_t)cap * ES, of,
        (size_t)blockIdx.y * gridDim.x + blockIdx.x, t0, cnt, overflow);
}

// The sweep's field gather (2D or 3D, virial and/or kinetic): each
// workgroup finds its system, frame and tile in the sweep's table
// (ik_sweep.hpp).  Padding workgroups store zero counts for their slot, so
// k_reduce_stats can read every slot.  Three waves per SIMD: the system's
// geometry and pointers come from the table and stay in registers (a kernel
// argument would be reloaded instead), which at the single-system kernel's
// four waves spills 24 bytes a lane in the 2D FP64 form; with the room of
// three there is no spill, and the eight-system 2D sweep's gather takes
// 5.87 ms against 5.89 at four.
constexpr int kSweepGatherWaves = 3;

template <int D, int OD, bool VIR, bool KIN, typename ER>
__global__ __launch_bounds__(64, kSweepGatherWaves) void k_sweep_gather(
    const SweepSys *__restrict__ T, int ns, GLRule R, const int *__restrict__ cstart,
    const double *__restrict__ spos, const double *__restrict__ skin, int cap, const int *__restrict__ bcount,
    const ER *__restrict__ bonds, unsigned long long *__restrict__ wave_counts,
    int *__restrict__ overflow)
{
    constexpr int PS = (D == 2) ? 2 : 4;
    constexpr int KN = OD * (OD + 1) / 2;
    constexpr int ES = BondLayout<D, OD, false, ER>::ES;
    const SweepSys &S = T[sweep_system(T, ns, SW_GATHER, blockIdx.x)];
    int f, b;
    if (!sweep_frame_tile(S, SW_GATHER, blockIdx.x, f, b)) {
        if (threadIdx.x == 0) {
            wave_counts[2 * (size_t)blockIdx.x] = 0;
            wave_counts[2 * (size_t)blockIdx.x + 1] = 0;
        }
        return;
    }
    const Geom &g = S.g;
    const int n = S.n, G = S.G;
    const size_t fo = (size_t)S.p0 + (size_t)f * n, oo = (size_t)f * G * OD * OD;
    GatherOut of{};
    of.vir = VIR ? S.vir + oo : nullptr;
    of.kin = KIN ? S.kin + oo : nullptr;
    of.wave_counts = wave_counts;
    int t0, cnt;
    tile_points(S.tiles, b, S.tp, t0, cnt);
    gather_tile_body<D, OD, 0, 5, VIR, false, KIN, ER>(
        g, n, S.grid, S.perm, R, nullptr, S.cgnorm, cstart + (size_t)S.c0 + (size_t)f * (g.ncell + 1),
        spos + fo * PS, KIN ? skin + fo * KN : nullptr, cap, VIR ? bcount + fo : nullptr,
        VIR ? bonds + fo * (size_t)cap * ES : nullptr, of, blockIdx.x, t0, cnt, overflow);
}

}  // namespace pgt
