// ik_gather_tile.hpp -- the item-balanced field gather ("tile" gather) of
// the IK stress-field engine.  Included by ik_gather_launch.hpp.
//
// A workgroup is one wavefront and takes a tile of the grid (a block of 8 x 8
// or 4 x 4 x 4 of its sites, 64 slots, see TileRec) or a part of one.  Work
// items are the (grid point, particle) pairs with the particle inside the
// point's ball; an item integrates the particle's bonds for the point.
//
// 1. Window: the particles within r_cg of the points' bounding box, read from
//    the rows of cells that cover it, one particle per lane, into a list in
//    LDS.
// 2. Masks: a lane holds one window particle and tests it against every point
//    (FP64, |a|^2 < r_cg^2), which gives the particle's mask of points.  Where
//    the tile's points are the product of their axes' coordinates (any
//    regular grid), the squares of the differences along x are shared by a
//    column of points, and those along x and y in 3D: 3 operations a pair
//    and the axes' instead of 7 (2D) or 9 (3D).
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
// order, so the sums are the same from run to run.  They are also the same
// whatever part of a tile a workgroup takes, which depends on how many tiles a
// launch has: the window is listed in the order, and in the batches, that the
// tile's unit gives (the part that the particles' density asks for, whatever
// the launch), so a point's particles lie in the same batches in the same
// order, and a smaller part only leaves out those too far from its own points.
// Up to four batches go through steps 2 to 4 as one list, each ordered by
// itself.  Parts scan their unit's cells for it: gather of one frame, their
// own windows alone, a step of 64 candidates at a time / this: 2D N = 2,000, 32^2
// grid 12 / 15 us, N = 65,536, 256^2 26 / 29; 3D N = 4,000, 12^3 25 / 32, N = 20,011,
// 37^3 89 / 98; whole tiles, whose scan is the same, are no slower (3D FP32 form,
// 20 frames of N = 131,072, 3,150 / 3,120).  The boxes lie in LDS rather than in
// registers that the item loop would spill, and four steps' candidates are
// found and loaded together: a step waited for the six reads of its segment's
// search and for one load, one after the other (one step at a time / four: the
// 3D frames 41 / 32 and 106 / 98, 20 frames of N = 20,011, 30^3 616 / 588; 2D N = 8,192,
// open box, 40 frames 217 / 169).  A list of several batches has each batch's
// bond counts from the largest down, so its steps are less even: what a dear
// rule pays most for (3D, Mollifier kernel, 10 nodes, N = 8,000, 20^3, one frame
// 105 / 141).
//
// Why particles, not points, are spread over the lanes in the scan: scattered
// loads pace this kernel (a CU's L1 takes about one lane's 16 bytes a cycle
// when the lanes' lines differ).  With a point per lane, each lane walked its
// own cells and every item fetched its particle from memory: 216 loads a
// wavefront on the 2D N = 65,536 job with a 256^2 grid, 5,814 VALU
// instructions.  Here a window particle is loaded once per tile, and an
// item's entries are shared by its neighbours: 125 loads, 4,724 VALU
// instructions (5,360 before the product tiles' masks, fewer operations of the
// 5-node rule and the two register sets of the item loop).  Measured (one launch, point
// per lane / particle per lane / with those three): 100 such frames 1.68 /
// 1.38 / 1.17 ms; 3D N = 131,072 with a 64^3 grid, FP32 form, 20 frames 4.30 /
// 3.72 / 3.23 ms; 3D FP64 with the kinetic field, N = 20,011, 5 frames 0.43 /
// 0.37 / 0.34 ms; 2D FP32 form, N = 30,011, 117^2 grid, 33 frames 0.152 /
// 0.132 / 0.107 ms; a sweep of eight systems whose grid points are up to 2.4
// apart (r_cg = 2) 0.80 / 0.65 / 0.58 ms.  VALU issue is now 73% of the time.
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

// Capacities of the tile gather.  LDS in the 2D virial + kinetic form: 9.9 KB,
// 16 wavefronts per CU, the four per SIMD that its registers allow.
struct TileCaps {
    static constexpr int BLK = kTileThreads;  // one wavefront
    static constexpr int TP = kTilePoints;    // most grid points of a tile
    static constexpr int MAXW = 128;          // window particles listed at a time
    static constexpr int MAXI = 1024;         // items listed at a time
    static constexpr int NBATCH = 4;          // most batches of a list
    static constexpr int NKEY = 32;           // classes of bond counts (count_class)
    static constexpr int SBITS = 8;           // item word: window slot | point << SBITS
    static constexpr int MAXNB = 255;         // bond count of a particle (one byte); more: overflow
    static_assert(TP == 64 && BLK == 64, "one wavefront, masks of 64 points");
    static_assert(MAXW <= (1 << SBITS) && MAXW % 64 == 0, "window slots of an item word");
};

// The class that orders particles by bond count (at most MAXNB): the count
// itself up to 16, then four classes to each doubling.
__device__ __forceinline__ int count_class(int nb)
{
    const int e = 31 - __clz(nb | 1);
    return nb < 16 ? nb : 4 * e + ((nb >> (e - 2)) & 3);
}

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
// latency; three for the 3D FP64 virial + kinetic form (184 registers and two
// waves unbounded, 36 bytes a lane spilled: N = 20,011, 37^3 grid, 5 frames, the
// job 455 -> 446 us; N = 19,459, 18^3, 19 frames 454 -> 443; Rect, 5 nodes, 641 ->
// 555) but for the Mollifier kernel, which would spill 144 (10 nodes 1,969 ->
// 2,014 us); in 2D that kernel is as fast at three as at four; the others are left
// to the compiler (one to three: the 3D FP64 virial form would spill 88 bytes a
// lane at four).
template <int D, int CG, bool ELA, bool KIN, typename ER>
struct TileWaves {
    static constexpr bool F32 = std::is_same<ER, float>::value;
    static constexpr bool four = (D == 2 && !ELA) || (D == 3 && F32 && !ELA && !KIN);
    static constexpr bool three = D == 3 && CG != 2 && !F32 && !ELA && KIN;
    static constexpr int value = four ? 4 : three ? 3 : 1;
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

// A value that is the same in every lane, in scalar registers.
__device__ __forceinline__ double uniform(double v)
{
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)u);
    const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(u >> 32));
    return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}

// The body works on one frame's arrays (cell starts st, sorted positions
// sp, kinetic terms sk, bond counts bc, entries bd; out's field pointers at
// the frame's first value) for slots j0 .. j0 + tp - 1 of tile record tr (tp:
// 64, 32, 16 or 4, j0 a multiple of it), whose grid points are tperm[0 .. 63],
// and stores its counts at out.wave_counts[2 wi ..].  unit, at least tp, of the
// same sizes: the slots whose window sets the order of the sums.  LT: FP32
// terms rounded as the lane gather of two points a lane rounds them, so that an
// engine whose gather was not chosen may take either.
template <int D, int OD, int CG, int NQ, bool VIR, bool ELA, bool KIN, typename ER, bool LT = false>
__device__ __forceinline__ void gather_tile_body(const Geom &g, const double *__restrict__ grid,
                                                 const TileRec &tr, const int *__restrict__ tperm, int j0, int tp,
                                                 int unit, const GLRule &R, const double *__restrict__ gld,
                                                 double cgnorm,
                                                 const int *__restrict__ st, const double *__restrict__ sp,
                                                 const double *__restrict__ sk, int cap,
                                                 const int *__restrict__ bc, const ER *__restrict__ bd,
                                                 const GatherOut &out, size_t wi, int *__restrict__ overflow)
{
    using CP = TileCaps;
    using LY = BondLayout<D, OD, ELA, ER>;
    constexpr int MAXW = CP::MAXW, MAXI = CP::MAXI, SBITS = CP::SBITS;
    constexpr int NR = MAXW / 64;  // window particles per lane
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

    __shared__ double s_pt[64][D];               // the points
    __shared__ double s_box[2][2 * D];           // centre and half lengths of the unit's box, and of theirs
    __shared__ double s_acc[64][KTA];            // their accumulators
    __shared__ double s_wp[MAXW][D];             // window: positions,
    __shared__ int s_wid[MAXW];                  // particles,
    __shared__ unsigned char s_wnb[MAXW];        // their batches, then bond counts,
    __shared__ unsigned short s_wof[MAXW];       // first items
    // items per batch and class of bond counts, then their offsets: two
    // 16-bit counters a word (a list has at most MAXW TP of them)
    constexpr int NBATCH = CP::NBATCH, NKEY = CP::NKEY;
    __shared__ unsigned s_bucket[64];
    static_assert(NBATCH * NKEY == 128 && MAXW * CP::TP <= 65535, "two counters a lane");
    // items in order, and one past the list for those of another piece;
    // while the window is filled, the segments' first candidates and particles
    __shared__ union {
        unsigned short item[MAXI + 2];
        struct {
            int first[64], particle[64];
        } seg;
    } s_u;

    const int l = threadIdx.x;
    const int gp = tperm[l];
    const bool live = gp >= 0 && l >= j0 && l < j0 + tp;
    const unsigned long long points = __builtin_amdgcn_ballot_w64(live);
    if (points == 0ull) {
        if (l == 0) {
            out.wave_counts[2 * wi] = 0;
            out.wave_counts[2 * wi + 1] = 0;
        }
        return;
    }
    const bool product = tr.product != 0;

    // bounding box of the unit's points: centre xc, half lengths xh.  When the
    // box and its ball fit in less than a period (near), a particle has one
    // image that can be inside any of the balls, the one nearest to xc.
    const bool part = tp < unit;
    int w0[3] = {0, 0, 0}, wn[3] = {1, 1, 1};
    bool near = true;
    {
        const int u0 = j0 & ~(unit - 1);
        const bool ulive = gp >= 0 && l >= u0 && l < u0 + unit;
        double xg[D];
#pragma unroll
        for (int a = 0; a < D; ++a) {
            xg[a] = ulive ? grid[(size_t)gp * 3 + a] : 0.0;
            s_pt[l][a] = live ? xg[a] : __builtin_nan("");
        }
#pragma unroll
        for (int k = 0; k < KTA; ++k) s_acc[l][k] = 0.0;
        // box of slots b .. b + nb - 1; in: whether the lane holds one of their points
        auto box = [&](int b, int nb, bool in, double (&lo)[D], double (&hi)[D]) {
            if (product) {
                // over the axes' coordinates (lines without points are NaN,
                // which the minimum and the maximum pass over)
#pragma unroll
                for (int a = 0; a < D; ++a) lo[a] = __builtin_huge_val(), hi[a] = -__builtin_huge_val();
                const int q0 = b >> 4, q1 = (b + nb - 1) >> 4;
                for (int q = q0; q <= q1; ++q) {
                    const double *ax = tr.ax[q];
                    // a row of four points (nb 4) has one y and one z
                    const int r = nb == 4 ? (b >> 2) & 3 : -1;
#pragma unroll
                    for (int k = 0; k < 8; ++k) {
                        const int a = k < 4 ? 0 : ((D == 2 || k < 6) ? 1 : D - 1);
                        if (r >= 0 && k >= 4 && (D == 2 ? k - 4 != r : a == 1 ? k - 4 != (r & 1) : k - 6 != r >> 1))
                            continue;
                        lo[a] = fmin(lo[a], ax[k]);
                        hi[a] = fmax(hi[a], ax[k]);
                    }
                }
            } else {
                const int first = __ffsll((unsigned long long)__builtin_amdgcn_ballot_w64(in)) - 1;
#pragma unroll
                for (int a = 0; a < D; ++a) {
                    const double f = __shfl(xg[a], first, 64);  // (with every lane active)
                    const double v = in ? xg[a] : f;
                    lo[a] = wave_min(v);
                    hi[a] = wave_max(v);
                }
            }
        };
        double lo[D], hi[D];
        box(u0, unit, ulive, lo, hi);
#pragma unroll
        for (int a = 0; a < D; ++a) {
            axis_cells(g, a, lo[a], hi[a], g.rc, w0[a], wn[a]);
            w0[a] = __builtin_amdgcn_readfirstlane(w0[a]);
            wn[a] = __builtin_amdgcn_readfirstlane(wn[a]);
            const double xh = 0.5 * (hi[a] - lo[a]);
            s_box[0][a] = 0.5 * (lo[a] + hi[a]);
            s_box[0][D + a] = xh;
            near = near && (g.pinvL[a] == 0.0 || 2.0 * (xh + g.rc) < 0.999 * g.L[a]);
        }
        near = __builtin_amdgcn_ballot_w64(near) != 0ull;  // the same in every lane: a scalar
        if (part && near) {
            box(j0, tp, live, lo, hi);
#pragma unroll
            for (int a = 0; a < D; ++a) {
                s_box[1][a] = 0.5 * (lo[a] + hi[a]);
                s_box[1][D + a] = 0.5 * (hi[a] - lo[a]);
            }
        }
    }

    // whether a window particle's image nearest to xc is not the particle
    // itself (or may not be): pairs then take the minimum image, which is the
    // plain difference otherwise
    bool images = !near;
    auto nearest = [&](double v, int a) { return fma(-g.L[a], rint((v - s_box[0][a]) * g.pinvL[a]), v); };

    unsigned long long nball = 0;     // items (the same in every lane)
    unsigned long long ncontrib = 0;  // bond counts of the items, per lane
    bool over = false;                // an item's bond count exceeds MAXNB
    const double s2 = 2.0 * g.inv_rc;

    // ---- integrate items 0 .. ni - 1 of the list --------------------------
    auto integrate = [&](int ni) {
        // the next item's first bond entries and kinetic term are loaded
        // before the current one is integrated
        auto fetch = [&](int k, int &slot, int &ip, int &nb, double (&kk)[KNA], ER (&E)[GV]) {
            const bool valid = k < ni;
            const unsigned it = s_u.item[valid ? k : 0];
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
        auto item = [&](int slot, int ip, int nb, const double (&kk)[KNA], ER (&E0)[GV]) {
                double a[3];
                a[0] = s_wp[slot][0] - s_pt[ip][0];
                a[1] = s_wp[slot][1] - s_pt[ip][1];
                a[2] = 0.0;
                if constexpr (D == 3) a[2] = s_wp[slot][D - 1] - s_pt[ip][D - 1];
                if (images) {
#pragma unroll
                    for (int q = 0; q < D; ++q) a[q] = minimg(a[q], g.L[q], g.pinvL[q]);
                }
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
                    // site: 0 and 1, the loop's even and odd groups; 2, the
                    // last of an odd number of groups
                    auto one = [&](const ER (&Gv)[GV], auto O, auto site) {
                        constexpr int o = decltype(O)::value;
                        const ER *e = Gv + o;
                        ER C = e[0] * e[0];
                        C = fma(e[1], e[1], C);
                        if (D == 3) C = fma(e[2], e[2], C);
                        // Written as fused operations, so that the FP32
                        // form's rounding does not hang on how the compiler
                        // contracts each copy: results of earlier builds
                        // repeat bit for bit with y's product rounded first
                        // in the odd groups and in 3D without elastic terms,
                        // x's elsewhere.  The lane gather's virial forms have
                        // y's rounded first, but for the last of an odd number
                        // of groups in 3D without elastic terms.
                        constexpr int S = decltype(site)::value;
                        constexpr bool YF = LT ? D == 2 || ELA || S != 2 : (D == 3 && !ELA) || S == 1;
                        ER B;
                        if constexpr (YF) B = fma(ta[0], e[0], ta[1] * e[1]);
                        else B = fma(ta[1], e[1], ta[0] * e[0]);
                        if constexpr (D == 3) B = fma(ta[2], e[2], B);
                        ER wq;
                        if constexpr (CG == 0 && NQ == 5 && std::is_same<ER, double>::value) wq = bond_octic5(R, Aj, B, C);
                        else wq = bond_quad<CG, NQ, ER>(R, gld, R.n, Aj, B, C);
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
                    auto group = [&](const ER (&Gv)[GV], int kk2, auto site) {
                        one(Gv, std::integral_constant<int, 0>(), site);
                        if constexpr (GRP >= 2)
                            if (GRP * kk2 + 1 < nb) one(Gv, std::integral_constant<int, ES>(), site);
                        if constexpr (GRP >= 3)
                            if (GRP * kk2 + 2 < nb) one(Gv, std::integral_constant<int, 2 * ES>(), site);
                        if constexpr (GRP >= 4)
                            if (GRP * kk2 + 3 < nb) one(Gv, std::integral_constant<int, 3 * ES>(), site);
                    };
                    const ER *ptr = bd + (size_t)s_wid[slot] * cap * ES;
                    const int ng = (nb + GRP - 1) / GRP;
                    ER E1[GV];
                    int kk2 = 0;
                    for (; kk2 + 1 < ng; kk2 += 2) {
                        load_entry<ER, GV>(ptr + (size_t)(kk2 + 1) * GV, E1);
                        group(E0, kk2, std::integral_constant<int, 0>());
                        if (kk2 + 2 < ng) load_entry<ER, GV>(ptr + (size_t)(kk2 + 2) * GV, E0);
                        group(E1, kk2 + 1, std::integral_constant<int, 1>());
                    }
                    if (kk2 < ng) group(E0, kk2, std::integral_constant<int, 2>());
                }
#pragma unroll
                for (int q = 0; q < KT; ++q)
                    __hip_atomic_fetch_add(&s_acc[ip][q], acc[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        };
        // two sets of registers in turn, so that nothing is copied between steps
        int slot, ip, nb, nslot, nip, nnb;
        double kk[KNA], nkk[KNA];
        ER E0[GV], nE0[GV];
        fetch(l, slot, ip, nb, kk, E0);
        for (int k0 = 0; k0 < ni; k0 += 128) {
            fetch(k0 + 64 + l, nslot, nip, nnb, nkk, nE0);
            if (k0 + l < ni) item(slot, ip, nb, kk, E0);
            if (k0 + 64 >= ni) break;
            fetch(k0 + 128 + l, slot, ip, nb, kk, E0);
            if (k0 + 64 + l < ni) item(nslot, nip, nnb, nkk, nE0);
        }
        __syncthreads();
    };

    // m = 2 m + (d2 < r_cg^2) for a d2 that is a number: the sign of the
    // difference, which rounding keeps, moved in by one instruction (a compare
    // and the selects of its result would be three)
    auto push = [&](unsigned &m, double d2) {
        m = __builtin_amdgcn_alignbit(m, (unsigned)((unsigned long long)__double_as_longlong(d2 - g.rc2) >> 32), 31);
    };
    // Mask of the points whose balls hold x: bit j for slot j (bits enter at
    // the low end, the last slot first).  Slots without a point are masked
    // off: their coordinates are NaN.
    auto point_mask = [&](const double (&x)[D], unsigned (&m)[2]) {
        m[0] = m[1] = 0u;
        if (near && product) {
            for (int q = (j0 + tp - 1) >> 4; q >= j0 >> 4; --q) {
                const double *ax = tr.ax[q];
                double dx2[4], d1[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const double d = x[0] - ax[k];
                    dx2[k] = d * d;
                    d1[k] = D == 2 || k < 2 ? x[1] - ax[4 + k] : x[D - 1] - ax[4 + k];  // 3D: 2 along y, 2 along z
                }
                unsigned mm = (q & 2) ? m[1] : m[0];
                if constexpr (D == 2) {
#pragma unroll
                    for (int r = 15; r >= 0; --r) push(mm, fma(d1[r >> 2], d1[r >> 2], dx2[r & 3]));
                } else {
                    double dxy2[8];
#pragma unroll
                    for (int k = 0; k < 8; ++k) dxy2[k] = fma(d1[k >> 2], d1[k >> 2], dx2[k & 3]);
#pragma unroll
                    for (int r = 15; r >= 0; --r) push(mm, fma(d1[2 + (r >> 3)], d1[2 + (r >> 3)], dxy2[r & 7]));
                }
                if (tp < 32) mm <<= (q & 1) * 16;
                if (q & 2) m[1] = mm;
                else m[0] = mm;
            }
        } else {
#pragma unroll
            for (int h = 1; h >= 0; --h) {
                unsigned mm = 0u;
                if ((unsigned)(points >> (32 * h)) != 0u) {
#pragma unroll 4
                    for (int j = 31; j >= 0; --j) {
                        double d[3] = {0.0, 0.0, 0.0};
#pragma unroll
                        for (int a = 0; a < D; ++a) d[a] = x[a] - s_pt[32 * h + j][a];
                        if (!near) {
#pragma unroll
                            for (int a = 0; a < D; ++a) d[a] = minimg(d[a], g.L[a], g.pinvL[a]);
                        }
                        const bool in = fma(d[2], d[2], fma(d[1], d[1], d[0] * d[0])) < g.rc2;
                        mm = mm + mm + (in ? 1u : 0u);
                    }
                }
                m[h] = mm;
            }
        }
        m[0] &= (unsigned)points;
        m[1] &= (unsigned)(points >> 32);
    };

    // ---- the items of window particles 0 .. nw - 1 --------------------------
    auto process = [&](int nw) {
        s_bucket[l] = 0u;
        __syncthreads();
        unsigned m[NR][2];
        int nbs[NR];
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const int slot = r * 64 + l;
            m[r][0] = m[r][1] = 0u;
            nbs[r] = 0;
            if (r * 64 >= nw) continue;
            const bool valid = slot < nw;
            const int ws = valid ? slot : 0;
            int nbc = 0;
            if constexpr (PAIRS) nbc = min(bc[s_wid[ws]], cap);
            double x[D];
#pragma unroll
            for (int a = 0; a < D; ++a) x[a] = s_wp[ws][a];
            if (images && near) {
#pragma unroll
                for (int a = 0; a < D; ++a) x[a] = nearest(x[a], a);
            }
            point_mask(x, m[r]);
            if (!valid) m[r][0] = m[r][1] = 0u;
            const int pc = __popc(m[r][0]) + __popc(m[r][1]);
            if (nbc > CP::MAXNB && pc > 0) over = true;
            const int nb = min(nbc, CP::MAXNB);
            ncontrib += (unsigned long long)pc * (unsigned long long)nb;
            nbs[r] = (int)s_wnb[ws] * NKEY + NKEY - 1 - count_class(nb);
            if (valid) {
                s_wnb[slot] = (unsigned char)nb;
                atomicAdd(&s_bucket[nbs[r] >> 1], (unsigned)pc << (nbs[r] & 1) * 16);
            }
        }
        __syncthreads();
        int total;
        {
            const unsigned c = s_bucket[l];
            const int mine = (int)(c & 0xffffu) + (int)(c >> 16);
            int v = mine;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const int u = __shfl_up(v, off, 64);
                if (l >= off) v += u;
            }
            total = __builtin_amdgcn_readlane(v, 63);
            nball += (unsigned long long)total;
            __syncthreads();
            v -= mine;  // first items
            s_bucket[l] = (unsigned)v | ((unsigned)v + (c & 0xffffu)) << 16;
        }
        __syncthreads();
        for (int base = 0; base < total; base += MAXI) {
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const int slot = r * 64 + l;
                if (r * 64 >= nw) continue;
                int k = 0;
                if (base == 0) {
                    // an LDS atomic; the lanes of one instruction are served
                    // in a fixed order
                    if (slot < nw) {
                        const int sh = (nbs[r] & 1) * 16;
                        const unsigned pc = (unsigned)(__popc(m[r][0]) + __popc(m[r][1]));
                        k = (int)(atomicAdd(&s_bucket[nbs[r] >> 1], pc << sh) >> sh & 0xffffu);
                        s_wof[slot] = (unsigned short)k;
                    }
                } else {
                    // a further piece of a long list: the masks again, rather
                    // than registers held through the integration
                    double x[D];
#pragma unroll
                    for (int a = 0; a < D; ++a) x[a] = s_wp[slot < nw ? slot : 0][a];
                    if (images && near) {
#pragma unroll
                        for (int a = 0; a < D; ++a) x[a] = nearest(x[a], a);
                    }
                    point_mask(x, m[r]);
                    if (slot < nw) k = s_wof[slot] - base;
                    else m[r][0] = m[r][1] = 0u;
                }
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    unsigned mm = m[r][h];
                    const int word = slot | (32 * h) << SBITS;
                    if (total <= MAXI) {
                        unsigned short *q = s_u.item + k;
                        k += __popc(mm);
                        for (; mm; mm &= mm - 1u) *q++ = (unsigned short)(word + (__builtin_ctz(mm) << SBITS));
                    } else {
                        // items of other pieces go to the slot past the list
                        for (; mm; mm &= mm - 1u, ++k)
                            s_u.item[min((unsigned)k, (unsigned)MAXI)] =
                                (unsigned short)(word + (__builtin_ctz(mm) << SBITS));
                    }
                }
            }
            __syncthreads();
            integrate(min(total - base, MAXI));
        }
    };

    // ---- window: candidates of the cell rows, in segments of one row --------
    const int nx = g.nc[0], ny = g.nc[1], nz = g.nc[2];
    const int wrap = w0[0] + wn[0] > nx ? 1 : 0;  // a row that wraps is two segments
    const int nseg = (wn[1] * wn[2]) << wrap;
    const double rr = g.rc2 * (1.0 + 1e-9);
    int s0 = 0, c0 = 0;  // the next candidate: c0 of the segments from s0 on
    bool more = true;
    while (more) {
        int nw = 0, nu = 0;              // particles listed, and those of the unit's window in this batch
        int bs = s0, bc0 = c0, bw = 0;  // where the batch began: its first candidate and place
        int nbatch = 0;
        bool full = false;
        for (more = false; s0 < nseg && !full;) {
            int b = 0, len = 0;
            if (s0 + l < nseg) {
                const int r = (s0 + l) >> wrap, part = (s0 + l) & wrap;
                const int iz = D == 2 ? 0 : r / wn[1], iy = r - iz * wn[1];
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
            const int ns = min(nseg - s0, 64);
            __syncthreads();
            s_u.seg.first[l] = v - len;
            s_u.seg.particle[l] = b;
            __syncthreads();
            while (c0 < total && !full) {
                constexpr int NC = 4;  // steps whose candidates are found and loaded together
                int ids[NC], lo[NC];
                double xs[NC][D];
#pragma unroll
                for (int q = 0; q < NC; ++q) lo[q] = 0;
                // the last segment that starts at or before each candidate
                for (int h = ns > 8 ? 32 : 4; h > 0; h >>= 1) {
                    int f[NC];
#pragma unroll
                    for (int q = 0; q < NC; ++q) f[q] = s_u.seg.first[min(lo[q] + h, 63)];
#pragma unroll
                    for (int q = 0; q < NC; ++q)
                        if (lo[q] + h < ns && f[q] <= min(c0 + 64 * q + l, total - 1)) lo[q] += h;
                }
#pragma unroll
                for (int q = 0; q < NC; ++q)
                    ids[q] = s_u.seg.particle[lo[q]] + min(c0 + 64 * q + l, total - 1) - s_u.seg.first[lo[q]];
#pragma unroll
                for (int q = 0; q < NC; ++q)
#pragma unroll
                    for (int a = 0; a < D; ++a) xs[q][a] = sp[(size_t)ids[q] * PS + a];
#pragma unroll
                for (int q = 0; q < NC; ++q) {
                    if (c0 >= total) break;
                    const int id = ids[q];
                    double x[D], d2 = 0.0, p2 = 0.0;
#pragma unroll
                    for (int a = 0; a < D; ++a) x[a] = xs[q][a];
                    bool shift = false;
                    if (near) {
#pragma unroll
                        for (int a = 0; a < D; ++a) {
                            const double y = nearest(x[a], a);
                            shift = shift || y != x[a];
                            const double d = fabs(y - s_box[0][a]) - s_box[0][D + a];
                            d2 = fma(d > 0.0 ? d : d - d, d > 0.0 ? d : d - d, d2);
                            if (part) {
                                const double e = fabs(y - s_box[1][a]) - s_box[1][D + a];
                                p2 = fma(e > 0.0 ? e : e - e, e > 0.0 ? e : e - e, p2);
                            }
                        }
                    }
                    // not near: any image may matter, so every candidate is kept
                    const bool inu = c0 + l < total && d2 < rr, in = inu && p2 < rr;
                    const int ku = __popcll(__builtin_amdgcn_ballot_w64(inu));
                    const unsigned long long bm = __builtin_amdgcn_ballot_w64(in);
                    const int k = __popcll(bm);
                    if (nu + ku > MAXW) {  // these candidates begin the next batch
                        full = ++nbatch == NBATCH || !part;
                        if (full) break;
                        nu = 0;
                        bs = s0;
                        bc0 = c0;
                        bw = nw;
                    }
                    full = nw + k > MAXW;
                    if (full) {  // the batch with the next list
                        s0 = bs;
                        c0 = bc0;
                        nw = bw;
                        break;
                    }
                    images = images || __builtin_amdgcn_ballot_w64(in && shift) != 0ull;
                    if (in) {
                        const int w = nw + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(bm >> 32),
                                                                          __builtin_amdgcn_mbcnt_lo((unsigned)bm, 0u));
                        s_wid[w] = id;
                        s_wnb[w] = (unsigned char)nbatch;
#pragma unroll
                        for (int a = 0; a < D; ++a) s_wp[w][a] = x[a];
                    }
                    nw += k;
                    nu += ku;
                    c0 += 64;
                }
            }
            if (full) {
                more = true;
            } else {
                c0 = 0;
                s0 += 64;
            }
        }
        __syncthreads();
        if (nw > 0) process(nw);
        __syncthreads();
    }

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
    ncontrib = wave_sum(ncontrib);
    if (l == 0) {
        out.wave_counts[2 * wi] = nball;
        out.wave_counts[2 * wi + 1] = ncontrib;
    }
    if (over) atomicOr(overflow, 2);
}

// One frame per y row; block x takes part b mod (64 / tp) of tile b / (64 /
// tp), b = xcd_tile(x, gridDim.x), so each XCD works through a contiguous
// eighth of the frame's tiles.
template <int D, int OD, int CG, int NQ, bool VIR, bool ELA, bool KIN, typename ER, bool LT = false>
__global__ __launch_bounds__(64, (TileWaves<D, CG, ELA, KIN, ER>::value)) void k_gather_tile(
    Geom g, int n, int G, const double *__restrict__ grid, const TileRec *__restrict__ tiles,
    const int *__restrict__ tperm, int tp, int unit, GLRule R, const double *__restrict__ gld, double cgnorm,
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
    const int b = xcd_tile(blockIdx.x, gridDim.x), sub = kTilePoints / tp, k = b / sub;
    gather_tile_body<D, OD, CG, NQ, VIR, ELA, KIN, ER, LT>(
        g, grid, tiles[k], tperm + (size_t)k * kTilePoints, (b - k * sub) * tp, tp, unit, R, gld, cgnorm,
        cstart + (size_t)f * (g.ncell + 1), spos + fo * PS, KIN ? skin + fo * KN : nullptr, cap, bcount + fo,
        bonds + fo * (size_t)cap * ES, of, (size_t)blockIdx.y * gridDim.x + blockIdx.x, overflow);
}

// The sweep's field gather (2D or 3D, virial and/or kinetic): each
// workgroup finds its system, frame and tile in the sweep's table
// (ik_sweep.hpp).  Padding workgroups store zero counts for their slot, so
// k_reduce_stats can read every slot.  Four waves per SIMD in 2D: the system's
// geometry and pointers come from the table and stay in registers (a kernel
// argument would be reloaded instead), so the forms with both fields spill 28
// to 36 bytes a lane, and are the faster for the fourth wave: the eight-system
// sweep's job 1,246 us at three, 1,188 at four; with 125 frames a system, gather
// 4.15 -> 3.85 ms FP64, 3.62 -> 3.22 FP32 form.  3D: three, as the single-system
// kernel.
constexpr int sweep_gather_waves(int D) { return D == 2 ? 4 : 3; }

template <int D, int OD, bool VIR, bool KIN, typename ER>
__global__ __launch_bounds__(64, sweep_gather_waves(D)) void k_sweep_gather(
    const SweepSys *__restrict__ T, int ns, const TileRec *__restrict__ tiles, const int *__restrict__ tperm,
    GLRule R, const int *__restrict__ cstart, const double *__restrict__ spos, const double *__restrict__ skin, int cap, const int *__restrict__ bcount,
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
    const int sub = kTilePoints / S.tp, q = b / sub, k = S.tile0 + q;
    gather_tile_body<D, OD, 0, 5, VIR, false, KIN, ER>(
        g, S.grid, tiles[k], tperm + (size_t)k * kTilePoints, (b - q * sub) * S.tp, S.tp, S.unit, R, nullptr, S.cgnorm,
        cstart + (size_t)S.c0 + (size_t)f * (g.ncell + 1), spos + fo * PS, KIN ? skin + fo * KN : nullptr, cap,
        VIR ? bcount + fo : nullptr, VIR ? bonds + fo * (size_t)cap * ES : nullptr, of, blockIdx.x, overflow);
}

}  // namespace pgt
