// ik_bonds.hpp -- bond-list kernel of the IK stress-field engine.
// Included by ik_kernels.hpp.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "ik_device.hpp"
#include "ik_geom.hpp"

namespace pgt {

// Entries of particle p (cell-sorted index) sit at bonds[(f*n + p)*cap*ES ...],
// one per neighbour j within max_rcut with a nonzero pair force (or, with the
// elastic field, a nonzero force at r_ij + u_ij).  N_cg is the kernel
// normalisation and w the quadrature sum of the unnormalised kernel shape.
//
// FP64 (ER = double), ES = D + 1 (+ KN) values, no padding:
//   [0, D)     b' = r_ij / rc                   (scaled bond vector)
//   [D]        c' = 0.5 * N_cg * (F/r) * rc^2   (virial: T += c' w b' (x) b')
//   [D+1, ..)  elastic: 0.5 * N_cg * (F1_a (u+r)_b - F_a r_b), packed symmetric
// The gather reads entries two at a time (a group of 2*ES doubles, a whole
// number of 16-byte pieces, 16-byte aligned since cap is even) and
// recomputes |b'|^2 itself: the memory path of a CU returns about one
// scattered 16-byte piece per lane per cycle, so bytes per bond set the
// gather's speed.
//
// FP32 (ER = float), the same fields unpadded (a 2D virial entry is 12
// bytes, a 3D one 16), read in groups of 4, 2 or 1 entries (the fewest that
// make a whole number of 16-byte pieces).
template <int D, int OD, bool ELA, typename ER>
struct BondLayout {
    static constexpr int KN = OD * (OD + 1) / 2;
    static constexpr bool F64 = std::is_same<ER, double>::value;
    static constexpr int OC = D;           // offset of c'
    static constexpr int OE = OC + 1;      // offset of the elastic terms
    static constexpr int RAW = OE + (ELA ? KN : 0);
    static constexpr int PER16 = 16 / (int)sizeof(ER);
    static constexpr int ES = RAW;
    // entries per read group (FP64 always pairs)
    static constexpr int GRP = F64 ? 2 : (RAW % PER16 == 0 ? 1 : ((2 * RAW) % PER16 == 0 ? 2 : 4));
    static constexpr int GV = GRP * ES;  // values per group, a multiple of PER16
    static_assert(GV % PER16 == 0, "a read group is a whole number of 16-byte pieces");
};

// One wavefront per 64 (small jobs: 16) consecutive cell-sorted particles, one
// particle per lane.
//
// The particles sit in one or a few runs of cells of one row each (pieces),
// and a lane's candidates in the rows within reach of its own.  For every
// piece and neighbouring row the wavefront takes the particles of the piece's
// cells widened by the reach (a segment; cells past the ends of a row are
// those of its other end) and copies them to LDS, kBondWin at a time; a
// lane's candidates of a row are a stretch of the segment.  Pairs take the
// minimum image only where a segment holds one (the box's edges); elsewhere
// it is the plain difference.  Read from memory instead, each lane's
// candidates are scattered loads: a CU takes about one lane's 16 bytes a
// cycle of them, which was 69% of this kernel's time on the 2D N = 65,536
// job.  Measured, from memory / from LDS with a compare and a listing per
// candidate / this (one launch): that job, 100 frames 753 / 505 / 462 us; 2D
// FP32 form, N = 30,011, 33 frames 119 / 81 / 73 us; 3D N = 131,072, FP32 form,
// 20 frames 1,259 / 866 / 758 us; 3D FP64, N = 20,011, 5 frames 126 / 82 / 73 us.
// VALU issue is at 75%: 1,700 instructions a wavefront in 2D, half of them in
// pass 2 (three FP64 divisions a pair).
//
// Pass 1 lists a lane's candidates within max_rcut and (without elastic
// terms) within a bound of their own pair cutoff, about 4 of 37 in 2D and 7 of
// 226 in 3D.  Pass 2 evaluates the pair forces.  The listed pairs of the
// wavefront are dealt to its lanes evenly, whoever listed them: a lane by lane
// loop would run as long as the longest list, about twice the mean.  A
// listed pair whose force is zero after all (the bound is loose by the FP32
// form's rounding) and elastic terms (whose lists hold many such pairs) take
// that loop, since an entry's slot then depends on the forces before it.
// Entries keep the candidate order (cells in a fixed order, input order
// inside a cell).  In 3D the kernel stores each particle's bond count in its
// FP32 record.
//
// The body works on one frame's arrays (sorted cell keys kf, cell starts st,
// sorted positions sp, diameters sd, displacements sdp, counts bc, entries
// bd, FP32 records rf) for the particles of block pb, and stores the
// wavefront's largest count at *wmax.  pw: particles per block.
constexpr int kBondBlock = 64;  // lanes, and at most as many particles, of a block
constexpr int kBondWin = 256;   // candidates in LDS
// Wavefronts per SIMD the registers are held to: four in 2D without elastic
// terms (a few registers over otherwise, three wavefronts; 588 -> 538 us on
// the 2D N = 65,536 job when this was set), left to the compiler elsewhere (the 3D forms
// would spill 110 bytes a lane, and their LDS lets 13 wavefronts onto a CU).
constexpr int bond_waves(int D, bool ELA) { return D == 2 && !ELA ? 4 : 1; }

// Where the particles of cell c of a row start, in the frame's sorted order
// continued past the row's ends by its other end (st: the row's cell starts,
// nx cells of count particles; c from -nx to 2 nx).
__device__ __forceinline__ int row_start(const int *__restrict__ st, int nx, int count, int c)
{
    const int w = c < 0 ? 1 : (c > nx ? -1 : 0);
    return st[c + w * nx] - w * count;
}

template <int D, int OD, bool VIR, bool ELA, typename ER>
__device__ __forceinline__ void bonds_body(const Geom &g, int n, const PotParams &P, double cgnorm,
                                           const int *__restrict__ kf, const int *__restrict__ st,
                                           const double *__restrict__ sp, const double *__restrict__ sd,
                                           const double *__restrict__ sdp, int cap, int *__restrict__ bc,
                                           ER *__restrict__ bd, int *__restrict__ wmax, float4 *__restrict__ rf, int pb, int pw)
{
    constexpr int PS = (D == 2) ? 2 : 4;
    using LY = BondLayout<D, OD, ELA, ER>;
    constexpr int ES = LY::ES;
    // listed candidates per lane; more are listed by another scan
    constexpr int MAXC = ELA ? (D == 2 ? 24 : 40) : 16;
    constexpr int MAXP = 512;  // listed pairs dealt at a time
    constexpr int NB = 4;      // candidates per step of pass 1
    constexpr int NROW = 3;    // rows whose ranges are loaded together
    static_assert(kBondWin <= 256, "list entries are bytes");
    __shared__ double s_x[kBondWin + NB][D];  // candidates: positions,
    __shared__ double s_d[kBondWin + NB];     // diameters (the last step of a scan may read past the window),
    __shared__ int s_id[ELA ? kBondWin : 1];  // sorted indices
    __shared__ unsigned char lq[MAXC][64];    // each lane's list
    // segments: first candidate, sorted index of the first particle (as
    // row_start continues it) less that, the row's first particle, its count
    // and its first cell
    __shared__ int s_sf[64], s_of[64], s_rs[64], s_rc[64], s_rb[64];
    __shared__ int s_slot[64];  // a lane's next entry less its first pair's number
    __shared__ union {
        struct {
            int lo[64], hi[64], row[64];  // pieces: first and last cell, row
        } piece;
        unsigned short pair[MAXP];  // listed pairs: lane | candidate << 6
    } s_u;

    const int lane = threadIdx.x;
    const int p0 = pb * pw, pn = min(pw, n - p0);
    // lanes past the end shadow the last particle without writing, so the
    // whole wavefront takes part in the staging and in the maximum at the end
    const bool live = lane < pn;
    const int p = p0 + min(lane, pn - 1);
    double xi[D];
#pragma unroll
    for (int a = 0; a < D; ++a) xi[a] = sp[(size_t)p * PS + a];
    const double di = sd[p];
    const double h = 0.5 * cgnorm, hc = h * g.rc2;
    int cnt = 0;

    // whether pairs take the minimum image: on an axis of one cell under
    // periodic boundaries, and with segments across the box's edges
    bool one_cell = false, img = false;
#pragma unroll
    for (int a = 0; a < D; ++a) one_cell = one_cell || (g.nc[a] == 1 && g.periodic[a]);

    ER *const bd0 = bd + (size_t)p0 * (size_t)cap * ES;  // the block's entries

    // force of particle p0 + i (position x, diameter d) and candidate q; writes
    // the entry to slot k of the particle's list and returns true unless it is zero
    auto bond = [&](int i, const double *x, double d, int q, int k, bool write) {
        const double dj = s_d[q];
        double b[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int a = 0; a < D; ++a) {
            b[a] = s_x[q][a] - x[a];
            if (img) {
                asm volatile("");  // a branch: most blocks have none of these
                b[a] = minimg(b[a], g.L[a], g.pinvL[a]);
            }
        }
        const double rsq = fma(b[2], b[2], fma(b[1], b[1], b[0] * b[0]));
        // false for numbers that are none, which the list may hold (force_divr
        // ends with the same test of the pair's own cutoff)
        if (!(rsq < g.mr2)) return false;
        double f0, f1 = 0.0;
        double ur[3] = {0, 0, 0};
        if constexpr (std::is_same<ER, double>::value) f0 = force_divr<double>(P, rsq, d, dj);
        else f0 = (double)force_divr<float>(P, (float)rsq, (float)d, (float)dj);
        if constexpr (ELA) {
            for (int a = 0; a < 3; ++a) ur[a] = sdp[(size_t)s_id[q] * 3 + a] - sdp[(size_t)(p0 + i) * 3 + a] + b[a];
            const double ursq = ur[0] * ur[0] + ur[1] * ur[1] + ur[2] * ur[2];
            if constexpr (std::is_same<ER, double>::value) f1 = force_divr<double>(P, ursq, d, dj);
            else f1 = (double)force_divr<float>(P, (float)ursq, (float)d, (float)dj);
        }
        if (f0 == 0.0 && f1 == 0.0) return false;
        // entries beyond the capacity are counted, not written
        if (write && k < cap) {
            ER ev[ES];
#pragma unroll
            for (int a = 0; a < D; ++a) ev[a] = (ER)(b[a] * g.inv_rc);
            ev[LY::OC] = VIR ? (ER)(hc * f0) : (ER)0;
            if constexpr (ELA) {
                ER *t = ev + LY::OE;
                auto T = [&](int a, int c) { return h * (f1 * ur[a] * ur[c] - f0 * b[a] * b[c]); };
                for (int a = 0; a < OD; ++a) t[a] = (ER)T(a, a);
                if (OD == 2) t[2] = (ER)T(0, 1);
                else { t[3] = (ER)T(0, 1); t[4] = (ER)T(0, 2); t[5] = (ER)T(1, 2); }
            }
            ER *e = bd0 + (unsigned)((i * cap + k) * ES);
            if constexpr (ES % LY::PER16 == 0) {
                using V = typename std::conditional<std::is_same<ER, double>::value, double2, float4>::type;
                V t[ES / LY::PER16];
                __builtin_memcpy(t, ev, sizeof(ev));
#pragma unroll
                for (int q16 = 0; q16 < ES / LY::PER16; ++q16) reinterpret_cast<V *>(e)[q16] = t[q16];
            } else {
#pragma unroll
                for (int a = 0; a < ES; ++a) e[a] = ev[a];
            }
        }
        return true;
    };

    // pass 2 over the m candidates each lane listed
    auto forces = [&](int m) {
        bool alone = ELA;  // lane by lane
        if constexpr (!ELA) {
            int v = live ? m : 0;
            const int mine = v;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const int u = __shfl_up(v, off, 64);
                if (lane >= off) v += u;
            }
            const int total = __builtin_amdgcn_readlane(v, 63), first = v - mine;
            alone = total > MAXP;
            if (!alone) {
                s_slot[lane] = cnt - first;
                for (int k = 0; k < mine; ++k) s_u.pair[first + k] = (unsigned short)(lane | lq[k][lane] << 6);
                __syncthreads();
                bool zero = false;
                for (int k0 = 0; k0 < total; k0 += 64) {
                    const int k = k0 + lane;
                    const int w = s_u.pair[min(k, total - 1)], i = w & 63;
                    double x[D];  // the particle's own data, from the lane that holds it
#pragma unroll
                    for (int a = 0; a < D; ++a) x[a] = __shfl(xi[a], i, 64);
                    const double d = __shfl(di, i, 64);
                    if (k < total && !bond(i, x, d, w >> 6, k + s_slot[i], true)) zero = true;
                }
                alone = __builtin_amdgcn_ballot_w64(zero) != 0ull;
                if (!alone) cnt += mine;
                __syncthreads();
            }
        }
        if (alone)
            for (int k = 0; k < m; ++k)
                if (bond(p - p0, xi, di, lq[k][lane], cnt, live)) ++cnt;
    };

    // pass 1 over candidates b .. e - 1 (self: the particle itself): m counts
    // those within reach, of which numbers skip .. skip + MAXC - 1 are listed.
    // Up to 32 candidates set the bits of a mask, each by the sign of a
    // difference (one instruction moves it in; a compare and a listing under
    // it, which some lane of 64 nearly always takes, would be eight), the last
    // candidate first; then a lane lists its few.
    auto scan = [&](int b, int e, int self, int skip, int &m, auto image) {
        for (; b < e; b += 32) {
            const int len = min(e - b, 32);
            unsigned mask = 0u;
            for (int j = (len - 1) & ~(NB - 1); j >= 0; j -= NB) {
                double c[NB][D], dj[NB];
#pragma unroll
                for (int u = 0; u < NB; ++u) {
#pragma unroll
                    for (int a = 0; a < D; ++a) c[u][a] = s_x[b + j + u][a];
                    dj[u] = s_d[b + j + u];
                }
#pragma unroll
                for (int u = NB - 1; u >= 0; --u) {
                    double b2 = 0.0;
#pragma unroll
                    for (int a = 0; a < D; ++a) {
                        double d = c[u][a] - xi[a];
                        if constexpr (decltype(image)::value) d = minimg(d, g.L[a], g.pinvL[a]);
                        b2 = a == 0 ? d * d : fma(d, d, b2);
                    }
                    double r2 = g.mr2;
                    if constexpr (!ELA) {
                        const double s = (di + dj[u]) * fma(P.leps, fabs(di - dj[u]), P.lim);
                        r2 = fmin(s * s, r2);
                    }
                    mask = __builtin_amdgcn_alignbit(
                        mask, (unsigned)((unsigned long long)__double_as_longlong(b2 - r2) >> 32), 31);
                }
            }
            mask &= ~0u >> (32 - len);
            if ((unsigned)(self - b) < 32u) mask &= ~(1u << (self - b));
            for (; mask; mask &= mask - 1u, ++m)
                if ((unsigned)(m - skip) < (unsigned)MAXC) lq[m - skip][lane] = (unsigned char)(b + __builtin_ctz(mask));
        }
    };

    // the lane's cell, and the pieces: runs of lanes of one row
    const int nx = g.nc[0], ny = g.nc[1], nz = g.nc[2], R = g.reach;
    const int key = kf[p];
    const int row = (int)(((double)key + 0.5) * g.inv_nc[0]);  // (exact: a cell's half is far from rounding)
    const int cx = key - row * nx;
    const int prow = __shfl_up(row, 1, 64);
    const unsigned long long starts = __builtin_amdgcn_ballot_w64(lane == 0 || row != prow);
    const int npiece = __popcll(starts);
    const int piece = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(starts >> 32),
                                                     __builtin_amdgcn_mbcnt_lo((unsigned)starts, 0u)) +
                      (int)((starts >> lane) & 1ull) - 1;
    const int ry = ny == 1 ? 1 : 2 * R + 1, rz = nz == 1 ? 1 : 2 * R + 1, nrow = ry * rz;
    const int own = (nz == 1 ? 0 : R) * ry + (ny == 1 ? 0 : R);  // the row of the lane's own cell
    const float inv_npiece = __builtin_amdgcn_rcpf((float)npiece), inv_ry = __builtin_amdgcn_rcpf((float)ry);
    // a lane's candidates of a row: cells lx .. hx - 1, relative to its own
    const int lx = nx == 1 ? -cx : -R, hx = nx == 1 ? 1 - cx : R + 1;

    // rows in blocks of at most 64 segments: segment (row - r0) npiece + piece
    const int block = min(nrow, 64 / npiece);
    for (int r0 = 0; r0 < nrow; r0 += block) {
        const int nr = min(block, nrow - r0), nseg = nr * npiece;
        if ((starts >> lane) & 1ull) {
            s_u.piece.lo[piece] = cx;
            s_u.piece.row[piece] = row;
        }
        if (lane == 63 || ((starts >> ((lane + 1) & 63)) & 1ull)) s_u.piece.hi[piece] = cx;
        __syncthreads();
        int len = 0, begin = 0;
        {
            // quotients of integers below 2^7, half a step from the next
            const int sg = min(lane, nseg - 1);
            const int rr = (int)(((float)sg + 0.5f) * inv_npiece), q = sg - rr * npiece, r = r0 + rr;
            const int dz = D == 2 ? 0 : (int)(((float)r + 0.5f) * inv_ry), dy = r - dz * ry;
            const int pr = s_u.piece.row[q];
            const int cz = D == 2 ? 0 : (int)(((double)pr + 0.5) * g.inv_nc[1]), cy = pr - cz * ny;
            int z = 0, y = 0, k = 0;
            if (nz > 1) {
                z = cz + dz - R;
                k |= z < 0 || z >= nz;
                z = z < 0 ? z + nz : (z >= nz ? z - nz : z);
            }
            if (ny > 1) {
                y = cy + dy - R;
                k |= y < 0 || y >= ny;
                y = y < 0 ? y + ny : (y >= ny ? y - ny : y);
            }
            const int rb = (z * ny + y) * nx;
            const int first = st[rb], count = st[rb + nx] - first;
            const int lo = nx == 1 ? 0 : s_u.piece.lo[q] - R, hi = nx == 1 ? 1 : s_u.piece.hi[q] + R + 1;
            begin = row_start(st + rb, nx, count, lo);
            if (lane < nseg) len = row_start(st + rb, nx, count, hi) - begin;
            img = one_cell || __builtin_amdgcn_ballot_w64(k || lo < 0 || hi > nx) != 0ull;
            s_rs[lane] = first;
            s_rc[lane] = count;
            s_rb[lane] = rb;
        }
        int v = len;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int u = __shfl_up(v, off, 64);
            if (lane >= off) v += u;
        }
        const int total = __builtin_amdgcn_readlane(v, 63);
        s_sf[lane] = v - len;
        s_of[lane] = begin - (v - len);
        __syncthreads();
        // windows of whole rows, or part of one that is longer than a window
        for (int ra = 0, c0 = 0; ra < nr;) {
            auto row_end = [&](int r) {
                return r + 1 < nr ? __builtin_amdgcn_readfirstlane(s_sf[(r + 1) * npiece]) : total;
            };
            int rb = ra, c1 = c0;
            for (int e; rb < nr && (e = row_end(rb)) - c0 <= kBondWin; ++rb) c1 = e;
            const bool part = rb == ra;
            if (part) {
                rb = ra + 1;
                c1 = c0 + kBondWin;
            }
            // the window's particles and the ranges of its first rows are in
            // flight together: what this kernel waits for is one load after
            // another, not their number
            constexpr int NL = kBondWin / 64;
            double wx[NL][D], wd[NL];
            int wid[NL];
#pragma unroll
            for (int u = 0; u < NL; ++u) {
                if (64 * u >= c1 - c0) continue;
                const int c = min(c0 + 64 * u + lane, c1 - 1);
                int s = 0;  // the last segment that starts at or before candidate c
                for (int step = nseg > 4 ? 32 : 2; step > 0; step >>= 1)
                    if (s + step < nseg && s_sf[s + step] <= c) s += step;
                const int first = s_rs[s], count = s_rc[s];
                int id = s_of[s] + c;
                id = id < first ? id + count : (id >= first + count ? id - count : id);
#pragma unroll
                for (int a = 0; a < D; ++a) wx[u][a] = sp[(size_t)id * PS + a];
                wd[u] = sd[id];
                wid[u] = id;
            }
            int rbeg[NROW], rend[NROW];
            auto ranges = [&](int r) {  // of rows r .. r + NROW - 1
#pragma unroll
                for (int u = 0; u < NROW; ++u) {
                    const int s = min(r + u, rb - 1) * npiece + piece;
                    const int to = -s_of[s] - c0;  // sorted index to candidate in LDS
                    const int *rst = st + s_rb[s];
                    rbeg[u] = max(to + row_start(rst, nx, s_rc[s], cx + lx), 0);
                    rend[u] = min(to + row_start(rst, nx, s_rc[s], cx + hx), c1 - c0);
                }
            };
            ranges(ra);
#pragma unroll
            for (int u = 0; u < NL; ++u) {
                const int k = 64 * u + lane;
                if (k >= c1 - c0) continue;
#pragma unroll
                for (int a = 0; a < D; ++a) s_x[k][a] = wx[u][a];
                s_d[k] = wd[u];
                if (ELA) s_id[k] = wid[u];
            }
            __syncthreads();
            for (int skip = 0;; skip += MAXC) {
                int m = 0;
                for (int r = ra; r < rb; r += NROW) {
                    if (r > ra || skip > 0) ranges(r);
#pragma unroll
                    for (int u = 0; u < NROW; ++u) {
                        if (r + u >= rb) break;
                        const int self = r0 + r + u == own ? p - s_of[(r + u) * npiece + piece] - c0 : -1;
                        if (img) scan(rbeg[u], rend[u], self, skip, m, std::true_type());
                        else scan(rbeg[u], rend[u], self, skip, m, std::false_type());
                    }
                }
                forces(min(max(m - skip, 0), MAXC));
                if (__builtin_amdgcn_ballot_w64(m > skip + MAXC) == 0ull) break;
            }
            __syncthreads();
            c0 = c1;
            ra = part && c1 < row_end(ra) ? ra : rb;
        }
    }

    if (live) {
        bc[p] = cnt;
        // 3D: the bond count completes the particle's FP32 record (the
        // candidate scans read only its position words)
        if (D == 3) reinterpret_cast<int *>(rf + p)[3] = cnt;
    }
    int mc = live ? cnt : 0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mc = max(mc, __shfl_xor(mc, off, 64));
    // the largest count of the wavefront, stored per wavefront in launch
    // order (k_reduce_stats takes the maximum)
    if (lane == 0) *wmax = mc;
}

// One frame per y row; block x takes the particles of block
// xcd_tile(x, gridDim.x), so each XCD works through a contiguous eighth of
// the frame.
template <int D, int OD, bool VIR, bool ELA, typename ER>
__global__ __launch_bounds__(kBondBlock, bond_waves(D, ELA)) void k_bonds(Geom g, int n, int pw, PotParams P, double cgnorm,
                                               const int *__restrict__ keys, const int *__restrict__ cstart, const double *__restrict__ spos,
                                               const double *__restrict__ sdiam, const double *__restrict__ sdisp,
                                               int cap, int *__restrict__ bcount, ER *__restrict__ bonds,
                                               int *__restrict__ wave_max, float4 *__restrict__ rec)
{
    constexpr int PS = (D == 2) ? 2 : 4;
    constexpr int ES = BondLayout<D, OD, ELA, ER>::ES;
    const int f = blockIdx.y;
    const size_t fo = (size_t)f * n;
    bonds_body<D, OD, VIR, ELA, ER>(
        g, n, P, cgnorm, keys + fo, cstart + (size_t)f * (g.ncell + 1), spos + fo * PS, sdiam + fo,
        ELA ? sdisp + fo * 3 : nullptr, cap, bcount + fo, bonds + fo * (size_t)cap * ES,
        wave_max + (size_t)blockIdx.y * gridDim.x + blockIdx.x, D == 3 ? rec + fo : nullptr,
        xcd_tile(blockIdx.x, gridDim.x), pw);
}

}  // namespace pgt
