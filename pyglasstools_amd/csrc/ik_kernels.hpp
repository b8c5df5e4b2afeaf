// ik_kernels.hpp -- cell-list, bond-list and surrogate kernels of the IK
// stress-field engine (gfx950).  Included once, by ik_engine.hip; the field
// gathers live in their own translation units (ik_gather_*.hip).
//
//   cell list   k_sort_hist -> k_sort_scan -> k_sort_scatter (per digit), or k_sort_small;
//               k_sort_finish
//   bond list   k_bonds   (ik_bonds.hpp)
//   fields      k_gather  (ik_gather.hpp); with the adaptive bond integral
//               k_gather_adaptive (ik_gather_adaptive.hpp)
//
// All per-frame arrays are stacked along blockIdx.y (one frame per y index).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "ik_device.hpp"
#include "ik_geom.hpp"

namespace pgt {

// ------------------------------------------------------------------------
// cell list: a stable LSD radix sort of (cell, input index) per frame.
// Every pass keeps the input order among equal digits, so particles end up
// in cell order and, inside a cell, in input order: the cell-sorted arrays
// do not depend on scheduling.  No global atomics are used.
// ------------------------------------------------------------------------
constexpr int kSortBlock = 256;                     // threads per workgroup
constexpr int kSortRows = 4;                        // rows of kSortBlock items per chunk
constexpr int kSortChunk = kSortBlock * kSortRows;  // items per chunk (one workgroup)
constexpr int kSortMaxRadix = 256;                  // digits of at most 8 bits

__device__ __forceinline__ int cell_of(const Geom &g, const double *p)
{
    const int cx = cell_coord(g, 0, p[0]), cy = cell_coord(g, 1, p[1]), cz = cell_coord(g, 2, p[2]);
    return (cz * g.nc[1] + cy) * g.nc[0] + cx;
}

// Count the digit (key >> shift) & (radix - 1) over chunk ch of one frame
// into hf[digit * nchunk + ch] (hf: the frame's histogram).  With FIRST the
// keys are the particles' cells, computed here from the frame's input
// positions and stored in kf.
template <bool FIRST>
__device__ __forceinline__ void sort_hist_body(const Geom &g, int n, int ch, int nchunk, int shift, int radix,
                                               const double *__restrict__ pos, int *__restrict__ kf,
                                               int *__restrict__ hf)
{
    __shared__ int h[kSortMaxRadix];
    const int t = threadIdx.x;
    h[t] = 0;
    __syncthreads();
    const int base = ch * kSortChunk;
    for (int r = 0; r < kSortRows; ++r) {
        const int i = base + r * kSortBlock + t;
        if (i >= n) break;
        int k;
        if constexpr (FIRST) {
            k = cell_of(g, pos + (size_t)i * 3);
            kf[i] = k;
        } else {
            k = kf[i];
        }
        atomicAdd(&h[(k >> shift) & (radix - 1)], 1);
    }
    __syncthreads();
    if (t < radix) hf[(size_t)t * nchunk + ch] = h[t];
}

// A job's first launch zeroes its counters on the way (maxcount null: not the
// first launch of a job).
__device__ __forceinline__ void clear_counts(int *maxcount, unsigned long long *stats)
{
    if (maxcount && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < 2) {
        maxcount[threadIdx.x] = 0;
        stats[threadIdx.x] = 0;
    }
}

// One frame per y row (frames dealt to XCDs whole), one chunk per workgroup:
// hist[f][digit][chunk].
template <bool FIRST>
__global__ __launch_bounds__(kSortBlock) void k_sort_hist(Geom g, int n, int nf, int shift, int radix,
                                                          const double *__restrict__ pos, int *__restrict__ keys,
                                                          int *__restrict__ hist, int *__restrict__ maxcount,
                                                          unsigned long long *__restrict__ stats)
{
    if constexpr (FIRST) clear_counts(maxcount, stats);
    int f, ch;
    if (!frame_block(nf, f, ch)) return;
    sort_hist_body<FIRST>(g, n, ch, gridDim.x, shift, radix, pos + (size_t)f * n * 3, keys + (size_t)f * n,
                          hist + (size_t)f * radix * gridDim.x);
}

// In-place exclusive scan of the len ints at a, by one 1024-thread
// workgroup: a frame's hist[digit][chunk] becomes the first output slot of
// that digit's items of that chunk.  8,192 at a time, eight consecutive ones a
// thread in two loads; each thread walking its 1,024th of the whole array an
// int at a time waited for every one of its loads (one launch, before
// / after: 100 frames of 8,192 13.4 / 5.1 us, a sweep's 128 of up to 24,576
// 42 / 7.9, 20 of 16,384 26 / 4.9).
__device__ __forceinline__ void scan_body(int len, int *__restrict__ a)
{
    constexpr int PER = 8, NW = 1024 / 64;
    __shared__ int s_wave[2][NW];
    const int t = threadIdx.x, w = t >> 6;
    int base = 0;
    for (int t0 = 0, turn = 0; t0 < len; t0 += 1024 * PER, turn ^= 1) {
        const int k = t0 + t * PER;
        int x[PER];
        if (k + PER <= len) {
            __builtin_memcpy(x, a + k, sizeof(x));
        } else {
#pragma unroll
            for (int q = 0; q < PER; ++q) x[q] = k + q < len ? a[k + q] : 0;
        }
        int sum = 0;
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int v = x[q];
            x[q] = sum;
            sum += v;
        }
        int v = sum;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int u = __shfl_up(v, off, 64);
            if ((t & 63) >= off) v += u;
        }
        if ((t & 63) == 63) s_wave[turn][w] = v;
        __syncthreads();  // (the other turn's sums are read before this one's next barrier)
        int first = base + v - sum;
#pragma unroll
        for (int q = 0; q < NW; ++q) {
            const int c = s_wave[turn][q];
            if (q < w) first += c;
            base += c;
        }
#pragma unroll
        for (int q = 0; q < PER; ++q) x[q] += first;
        if (k + PER <= len) {
            __builtin_memcpy(a + k, x, sizeof(x));
        } else {
#pragma unroll
            for (int q = 0; q < PER; ++q)
                if (k + q < len) a[k + q] = x[q];
        }
    }
}

// One workgroup per frame (blockIdx.x), len ints each.
__global__ __launch_bounds__(1024) void k_sort_scan(int len, int *__restrict__ hist)
{
    scan_body(len, hist + (size_t)blockIdx.x * len);
}

// Move the items of one chunk to their slots for this digit.  A chunk's items
// lie in rows of kSortBlock; an item's slot is the chunk's offset for its
// digit, plus the items of that digit in earlier rows, in earlier wavefronts
// of its row, and in lower lanes of its wavefront (found with one ballot per
// digit bit).  The chunk is put in order in LDS first, so that neighbouring
// lanes store to neighbouring slots: stored from their input order, 64 lanes'
// items went to as many lines, one lane a cycle.  One launch on 100 frames of
// 65,536: 57 -> 24 us, the eight-system sweep's 46 and 36 -> 26 and 21.  With
// FIRST the value is the input index.
template <bool FIRST>
__device__ __forceinline__ void sort_scatter_body(int n, int ch, int nchunk, int shift, int radix,
                                                  const int *__restrict__ kin, const int *__restrict__ vin,
                                                  const int *__restrict__ hf, int *__restrict__ kout,
                                                  int *__restrict__ vout)
{
    constexpr int NW = kSortBlock / 64, NE = kSortRows * NW;
    static_assert(kSortBlock == kSortMaxRadix, "a thread per digit");
    __shared__ unsigned short wc[NE][kSortMaxRadix];  // digit counts of each row's wavefronts, then their first places
    __shared__ int s_key[kSortChunk], s_val[kSortChunk];  // the chunk in order
    __shared__ int s_off[kSortMaxRadix];                  // a digit's first slot less its first place
    __shared__ int s_wave[NW];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const unsigned long long below = lane ? (~0ull >> (64 - lane)) : 0ull;  // lanes under this one
    const int base = ch * kSortChunk, items = min(kSortChunk, n - base);
    int key[kSortRows], val[kSortRows], rank[kSortRows];
#pragma unroll
    for (int r = 0; r < kSortRows; ++r) {
        const int i = base + min(r * kSortBlock + t, items - 1);
        key[r] = kin[i];
        val[r] = FIRST ? i : vin[i];
    }
    const int first = t < radix ? hf[(size_t)t * nchunk + ch] : 0;
#pragma unroll
    for (int e = 0; e < NE; ++e) wc[e][t] = 0;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortRows; ++r) {
        const bool valid = r * kSortBlock + t < items;
        const int d = (key[r] >> shift) & (radix - 1);
        unsigned long long peers = __ballot(valid);
        for (int b = 1; b < radix; b <<= 1) {
            const bool bit = d & b;
            const unsigned long long m = __ballot(bit);
            peers &= bit ? m : ~m;
        }
        rank[r] = __popcll(peers & below);
        if (valid && rank[r] == 0) wc[r * NW + w][d] = (unsigned short)__popcll(peers);
    }
    __syncthreads();
    // thread t: the places of digit t
    int c[NE], sum = 0;
#pragma unroll
    for (int e = 0; e < NE; ++e) {
        c[e] = wc[e][t];
        sum += c[e];
    }
    int place = sum;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int u = __shfl_up(place, off, 64);
        if (lane >= off) place += u;
    }
    if (lane == 63) s_wave[w] = place;
    __syncthreads();
    place -= sum;
#pragma unroll
    for (int q = 0; q < NW; ++q)
        if (q < w) place += s_wave[q];
    s_off[t] = first - place;
#pragma unroll
    for (int e = 0; e < NE; ++e) {
        wc[e][t] = (unsigned short)place;
        place += c[e];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortRows; ++r) {
        if (r * kSortBlock + t >= items) continue;
        const int k = wc[r * NW + w][(key[r] >> shift) & (radix - 1)] + rank[r];
        s_key[k] = key[r];
        s_val[k] = val[r];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortRows; ++r) {
        const int k = r * kSortBlock + t;
        if (k >= items) continue;
        const int kk = s_key[k];
        const int slot = s_off[(kk >> shift) & (radix - 1)] + k;
        kout[slot] = kk;
        vout[slot] = s_val[k];
    }
}

template <bool FIRST>
__global__ __launch_bounds__(kSortBlock) void k_sort_scatter(int n, int nf, int shift, int radix,
                                                             const int *__restrict__ kin, const int *__restrict__ vin,
                                                             const int *__restrict__ hist, int *__restrict__ kout,
                                                             int *__restrict__ vout)
{
    int f, ch;
    if (!frame_block(nf, f, ch)) return;
    const size_t fo = (size_t)f * n;
    sort_scatter_body<FIRST>(n, ch, gridDim.x, shift, radix, kin + fo, vin + fo, hist + (size_t)f * radix * gridDim.x,
                             kout + fo, vout + fo);
}

// Write sorted slot k of a frame's particle arrays from its input particle
// fi.  Positions are wrapped into the box along periodic axes (x - L floor((x -
// lo) / L): unchanged, bit for bit, inside the box), so a particle sits where
// its cell says.  In 3D with bonds it also writes the particle's FP32 record
// (x, y, z; the bond kernel adds the count) for the lane gather's FP32
// pre-test.
template <int D, int OD>
__device__ __forceinline__ void sorted_particle(const Geom &g, int k, size_t fi, const double *__restrict__ pos,
                                                const double *__restrict__ diam, const double *__restrict__ mass,
                                                const double *__restrict__ vel, const double *__restrict__ disp,
                                                double *__restrict__ spos, double *__restrict__ sdiam,
                                                double *__restrict__ skin, double *__restrict__ sdisp,
                                                float4 *__restrict__ rec)
{
    constexpr int PS = (D == 2) ? 2 : 4;
    constexpr int KN = OD * (OD + 1) / 2;
    // Every load first.  The rows of the inputs lie anywhere in the frame: four
    // lines a particle, one lane's at a time, bound this kernel (274 us for 100
    // frames of 65,536; its bytes alone take 156).  Streaming the inputs and
    // scattering the sorted arrays instead wrote partly filled lines (900 MB
    // for 320): 321 us; reading the frame once in order before: 294.
    const double p[3] = {pos[fi * 3], pos[fi * 3 + 1], D == 3 ? pos[fi * 3 + 2] : 0.0};
    const double d = diam[fi];
    double m = 1.0, v[3] = {0.0, 0.0, 0.0}, u[3] = {0.0, 0.0, 0.0};
    if (skin && mass) m = mass[fi];
    if (skin && vel) {
#pragma unroll
        for (int a = 0; a < OD; ++a) v[a] = vel[fi * 3 + a];
    }
    if (sdisp && disp) {
#pragma unroll
        for (int a = 0; a < 3; ++a) u[a] = disp[fi * 3 + a];
    }
    double *sp = spos + (size_t)k * PS;
    auto wrap = [&](int a) {
        return g.periodic[a] ? p[a] - g.L[a] * floor((p[a] - g.lo[a]) * g.invL[a]) : p[a];
    };
    sp[0] = wrap(0);
    sp[1] = wrap(1);
    if (D == 3) { sp[2] = wrap(2); sp[3] = 0.0; }
    if (D == 3 && rec) rec[k] = make_float4((float)sp[0], (float)sp[1], (float)sp[2], 0.0f);
    sdiam[k] = d;
    if (skin) {
        double *kk = skin + (size_t)k * KN;
        // symmetric packing: diagonal, then (0,1) [, (0,2), (1,2)]
        for (int a = 0; a < OD; ++a) kk[a] = m * v[a] * v[a];
        if (OD == 2) kk[2] = m * v[0] * v[1];
        else { kk[3] = m * v[0] * v[1]; kk[4] = m * v[0] * v[2]; kk[5] = m * v[1] * v[2]; }
    }
    if (sdisp)
        for (int a = 0; a < 3; ++a) sdisp[(size_t)k * 3 + a] = u[a];
}

// Write the cell-sorted particle arrays (slot k takes input particle
// vals[k]) and the cell starts: cstart[c] = first slot of cell c, and
// cstart[ncell] = n (keys are sorted, so slot k writes the starts of the
// cells after its predecessor's up to its own).
template <int D, int OD>
__device__ __forceinline__ void sort_finish_body(const Geom &g, int n, int k, int ncell, const int *__restrict__ keys,
                                                 const int *__restrict__ vals, const double *__restrict__ pos,
                                                 const double *__restrict__ diam, const double *__restrict__ mass,
                                                 const double *__restrict__ vel, const double *__restrict__ disp,
                                                 int *__restrict__ st, double *__restrict__ spos,
                                                 double *__restrict__ sdiam, double *__restrict__ skin,
                                                 double *__restrict__ sdisp, float4 *__restrict__ rec)
{
    if (k >= n) return;
    const int c = keys[k], i = vals[k], cb = keys[max(k - 1, 0)];
    const int cp = k == 0 ? -1 : cb;
    sorted_particle<D, OD>(g, k, (size_t)i, pos, diam, mass, vel, disp, spos, sdiam, skin, sdisp, rec);
    for (int q = cp + 1; q <= c; ++q) st[q] = k;
    if (k == n - 1)
        for (int q = c + 1; q <= ncell; ++q) st[q] = n;
}

template <int D, int OD>
__global__ __launch_bounds__(256) void k_sort_finish(Geom g, int n, int nf, int ncell, const int *__restrict__ keys,
                                                     const int *__restrict__ vals, const double *__restrict__ pos,
                                                     const double *__restrict__ diam, const double *__restrict__ mass,
                                                     const double *__restrict__ vel, const double *__restrict__ disp,
                                                     int *__restrict__ cstart, double *__restrict__ spos,
                                                     double *__restrict__ sdiam, double *__restrict__ skin,
                                                     double *__restrict__ sdisp, float4 *__restrict__ rec)
{
    constexpr int PS = (D == 2) ? 2 : 4;
    constexpr int KN = OD * (OD + 1) / 2;
    int f, bx;
    if (!frame_block(nf, f, bx)) return;
    const size_t fo = (size_t)f * n;
    sort_finish_body<D, OD>(g, n, bx * blockDim.x + threadIdx.x, ncell, keys + fo, vals + fo, pos + fo * 3,
                            diam + fo, mass ? mass + fo : nullptr, vel ? vel + fo * 3 : nullptr,
                            disp ? disp + fo * 3 : nullptr, cstart + (size_t)f * (ncell + 1), spos + fo * PS,
                            sdiam + fo, skin ? skin + fo * KN : nullptr, sdisp ? sdisp + fo * 3 : nullptr,
                            rec ? rec + fo : nullptr);
}

// ------------------------------------------------------------------------
// cell list of small frames: one workgroup per frame, counts and order in LDS
// ------------------------------------------------------------------------
// A counting sort by cell: cell sizes by LDS atomics, their scan, then every
// particle takes a slot of its cell in whatever order the atomics give, and
// finally counts the particles of its cell with a lower input index, which is
// its place: the radix sort's keys and values from one launch instead of six.
// Those launches, a few microseconds each whatever their size, were a third
// of a small frame's time on the GPU: N = 2,000 6 us against 20 in six kernels
// (and their gaps), N = 4,000 10 us; a driver call on them 147 -> 125 and 194 ->
// 173 us.  The counting is quadratic in a cell's particles (open boxes have
// cells as long as the box), so a frame with more than kSmallCrowd in one is
// put in order by a radix sort in LDS instead, which takes up to 25 us longer
// whatever the cells: sort of an open box of N = 8,192 (one cell) 3,080 us by
// counting, 18 by this, 15 to 24 by the radix launches; N = 2,000 201 / 11 / 15 to 20;
// a cluster of N = 8,192 in a periodic box, about 60 in a cell, 48 / 47 / 48 to 65, 90
// 54 / 45 / 54, 200 80 / 51 / 55, all in one 811 / 52 / 59.  With clear0 and clear1 not
// null the first workgroup also zeroes the job's counters.
constexpr int kSmallBlock = 1024;
constexpr int kSmallParticles = 8192;  // most particles of a frame, eight per thread
constexpr int kSmallCells = 8192;      // most cells (32 KB of LDS each for cells and particles)
constexpr int kSmallCrowd = 40;        // most particles of a cell that are counted one against another
constexpr int kSmallRow = 130;         // counts of a digit, 128 and two that put the digits on other LDS banks

__global__ __launch_bounds__(kSmallBlock) void k_sort_small(Geom g, int n, int ncell, const double *__restrict__ pos,
                                                            int *__restrict__ keys, int *__restrict__ vals,
                                                            int *__restrict__ clear0,
                                                            unsigned long long *__restrict__ clear1)
{
    constexpr int PER = kSmallParticles / kSmallBlock, CPT = kSmallCells / kSmallBlock;
    __shared__ int s_cell[128 * kSmallRow / 2];  // counts, then each cell's next slot
    unsigned short *const s_count = reinterpret_cast<unsigned short *>(s_cell);  // crowded frames
    static_assert(128 * kSmallRow / 2 >= kSmallCells, "a slot per cell");
    __shared__ int s_order[kSmallParticles];
    __shared__ int s_wave[kSmallBlock / 64], s_most[kSmallBlock / 64];
    const int t = threadIdx.x, f = blockIdx.x;
    const size_t fo = (size_t)f * n;
    pos += fo * 3;
    keys += fo;
    vals += fo;
    if (f == 0 && t < 2 && clear0) {
        clear0[t] = 0;
        clear1[t] = 0ull;
    }
    double x[PER][3];  // the frame's positions, in flight together
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        if (u * kSmallBlock >= n) continue;
        const double *p = pos + (size_t)min(u * kSmallBlock + t, n - 1) * 3;
#pragma unroll
        for (int a = 0; a < 3; ++a) x[u][a] = p[a];
    }
    for (int c = t; c < ncell; c += kSmallBlock) s_cell[c] = 0;
    __syncthreads();
    int key[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        key[u] = -1;
        if (u * kSmallBlock + t < n) {
            key[u] = cell_of(g, x[u]);
            atomicAdd(&s_cell[key[u]], 1);
        }
    }
    __syncthreads();
    // exclusive scan of the counts, `per` consecutive cells per thread
    const int per = (ncell + kSmallBlock - 1) / kSmallBlock;
    int own[CPT], sum = 0, most = 0;
#pragma unroll
    for (int q = 0; q < CPT; ++q) {
        own[q] = q < per && t * per + q < ncell ? s_cell[t * per + q] : 0;
        sum += own[q];
        most = max(most, own[q]);
    }
    int v = sum;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int w = __shfl_up(v, off, 64);
        if ((t & 63) >= off) v += w;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) most = max(most, __shfl_xor(most, off, 64));
    if ((t & 63) == 63) {
        s_wave[t >> 6] = v;
        s_most[t >> 6] = most;
    }
    __syncthreads();
    int run = v - sum;
#pragma unroll
    for (int w = 0; w < kSmallBlock / 64; ++w) {
        run += w < (t >> 6) ? s_wave[w] : 0;
        most = max(most, s_most[w]);
    }
#pragma unroll
    for (int q = 0; q < CPT; ++q) {
        if (q < per && t * per + q < ncell) s_cell[t * per + q] = run;
        run += own[q];
    }
    if (most > kSmallCrowd) {
        // a radix sort of cell << 13 | input index in LDS, digits of 7 bits
        constexpr int NW = kSmallBlock / 64, NE = PER * NW, ND = 128;  // chunks of 64 items, digits
        static_assert(NE == 128 && ND * NE == 16 * kSmallBlock && kSmallParticles == 1 << 13, "16 counts a thread");
        const unsigned long long below = (t & 63) ? (~0ull >> (64 - (t & 63))) : 0ull;  // lanes under this one
#pragma unroll
        for (int u = 0; u < PER; ++u)
            if (key[u] >= 0) s_order[u * kSmallBlock + t] = key[u] << 13 | (u * kSmallBlock + t);
        for (int shift = 13; (ncell - 1) >> (shift - 13); shift += 7) {
            __syncthreads();
            int item[PER], rank[PER];
#pragma unroll
            for (int u = 0; u < PER; ++u) item[u] = s_order[min(u * kSmallBlock + t, n - 1)];
            for (int q = t; q < ND * kSmallRow / 2; q += kSmallBlock) s_cell[q] = 0;
            __syncthreads();
#pragma unroll
            for (int u = 0; u < PER; ++u) {
                if (u * kSmallBlock >= n) continue;
                const bool valid = u * kSmallBlock + t < n;
                const int d = item[u] >> shift & (ND - 1);
                unsigned long long peers = __builtin_amdgcn_ballot_w64(valid);
#pragma unroll
                for (int b = 1; b < ND; b <<= 1) {
                    const unsigned long long m = __builtin_amdgcn_ballot_w64((d & b) != 0);
                    peers &= (d & b) ? m : ~m;
                }
                rank[u] = __popcll(peers & below);
                if (valid && rank[u] == 0)
                    s_count[d * kSmallRow + u * NW + (t >> 6)] = (unsigned short)__popcll(peers);
            }
            __syncthreads();
            // the first places: an exclusive scan, a digit's chunks by 8 threads
            unsigned short *const c = s_count + (t >> 3) * kSmallRow + (t & 7) * 16;
            int x[16], all = 0;
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                x[q] = all;
                all += c[q];
            }
            int w = all;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const int o = __shfl_up(w, off, 64);
                if ((t & 63) >= off) w += o;
            }
            if ((t & 63) == 63) s_wave[t >> 6] = w;
            __syncthreads();
            w -= all;
#pragma unroll
            for (int q = 0; q < NW; ++q) w += q < (t >> 6) ? s_wave[q] : 0;
#pragma unroll
            for (int q = 0; q < 16; ++q) c[q] = (unsigned short)(w + x[q]);
            __syncthreads();
#pragma unroll
            for (int u = 0; u < PER; ++u)
                if (u * kSmallBlock + t < n)
                    s_order[s_count[(item[u] >> shift & (ND - 1)) * kSmallRow + u * NW + (t >> 6)] + rank[u]] = item[u];
        }
        __syncthreads();
        for (int k = t; k < n; k += kSmallBlock) {
            keys[k] = s_order[k] >> 13;
            vals[k] = s_order[k] & (kSmallParticles - 1);
        }
        return;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PER; ++u)
        if (key[u] >= 0) s_order[atomicAdd(&s_cell[key[u]], 1)] = u * kSmallBlock + t;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        if (key[u] < 0) continue;
        const int i = u * kSmallBlock + t;
        const int begin = key[u] ? s_cell[key[u] - 1] : 0, end = s_cell[key[u]];
        int k = begin;
        for (int q = begin; q < end; ++q) k += s_order[q] < i ? 1 : 0;
        keys[k] = key[u];
        vals[k] = i;
    }
}

// Clears that a captured HIP graph can hold (a memset node is avoided there).
template <typename T>
__global__ void k_fill(T *__restrict__ p, T v, size_t n)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Up to five arrays of doubles copied by one launch between device memory and
// pinned host memory, which a kernel reads and writes over PCIe like its own:
// for the arrays of a small frame the copy engines' start and hand-over cost
// several times the transfer (pgt_ik_set_particles, pgt_ik_compute).
struct CopySegs {
    const double *src[5];
    double *dst[5];
    int n[5];
};

__device__ __forceinline__ void copy_segs(const CopySegs &c, int tid, int stride)
{
#pragma unroll
    for (int k = 0; k < 5; ++k)
        for (int i = tid; i < c.n[k]; i += stride) c.dst[k][i] = c.src[k][i];
}

__global__ __launch_bounds__(256) void k_copy_segs(CopySegs c)
{
    copy_segs(c, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x);
}

// Fold the per-wavefront statistics of one batch into the job totals: sums
// of (balls, contributions) into stats[0..1], the largest bond count into
// maxcount[0].  The first nrb workgroups reduce a stretch of the per-wavefront
// arrays each and add their result with one atomic per total (a few hundred
// atomics per batch, against one per wavefront of the batch's kernels before);
// the rest copy the segments of `out`.  host_counts (nrb = 1 only): pinned
// host memory that takes the job's counters, maxcount[0..1] in the first word
// and the two totals after it, so that a job ends with its last kernel and one
// synchronisation, without copies of a few bytes behind it.
__global__ __launch_bounds__(1024) void k_reduce_stats(int nrb, int nw, const unsigned long long *__restrict__ wave_counts,
                                                       int nm, const int *__restrict__ wave_max,
                                                       unsigned long long *__restrict__ stats, int *__restrict__ maxcount,
                                                       unsigned long long *__restrict__ host_counts, CopySegs out)
{
    if ((int)blockIdx.x >= nrb) {
        copy_segs(out, (blockIdx.x - nrb) * blockDim.x + threadIdx.x, (gridDim.x - nrb) * blockDim.x);
        return;
    }
    __shared__ unsigned long long s0[16], s1[16];
    __shared__ int sm[16];
    unsigned long long a = 0, b = 0;
    int m = 0;
    const int stride = nrb * blockDim.x;
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < nw; k += stride) {
        a += wave_counts[2 * k];
        b += wave_counts[2 * k + 1];
    }
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < nm; k += stride) m = max(m, wave_max[k]);
    a = wave_sum(a);
    b = wave_sum(b);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = max(m, __shfl_xor(m, off, 64));
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        s0[w] = a;
        s1[w] = b;
        sm[w] = m;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const int nwv = blockDim.x >> 6;
        for (int k = 1; k < nwv; ++k) {
            a += s0[k];
            b += s1[k];
            m = max(m, sm[k]);
        }
        if (host_counts) {  // the only workgroup: no other adds beside it
            a += stats[0];
            b += stats[1];
            m = max(m, maxcount[0]);
            stats[0] = a;
            stats[1] = b;
            maxcount[0] = m;
            host_counts[0] = (unsigned long long)(unsigned)m | ((unsigned long long)(unsigned)maxcount[1] << 32);
            host_counts[1] = a;
            host_counts[2] = b;
        } else {
            if (a) atomicAdd(&stats[0], a);
            if (b) atomicAdd(&stats[1], b);
            if (m) atomicMax(maxcount, m);
        }
    }
}

}  // namespace pgt

#include "ik_bonds.hpp"
#include "ik_surrogate.hpp"
