// pairlist.hip -- cell grid and half pair list on gfx950.
//
// Reproduces the pair set of Ensemble::set_pairlist/update_pairlist
// (src/Ensemble.cpp:454-525) and CellManager (src/utils/CellManager.h:82-203,
// src/utils/CellManager.cpp:43-314): the same cell grid, the same atom->cell
// arithmetic with clamping, the same 13-cell forward stencil, the same FP64
// distance predicate r^2 < (cutoff+cutBuff)^2 evaluated without contraction,
// and the same row order (in-cell successors, then stencil cells in order,
// atoms in index order).  Rows are stored ELL-style: row i at nb[i*stride].
//
// Rows are written owned-first: the reference's row i fills row i from the
// front, in its order; the same pairs seen from their other atom fill it from
// the back, so every atom's row holds all its partners and the pair kernels
// need no atomics.  Cell grid: one pass per step assigns atoms to cells, scans
// the counts and compacts each cell's atoms in index order; the pairs are then
// tested once per pair of cells and each atom's row made from the hits (see
// k_list_hits, k_list_rows).  Without cells, one wavefront per atom tests all atoms.
#include <algorithm>
#include <climits>

#include "smd_internal.h"

namespace smd {

// The 13 forward shifts in CellManager::build_cell_neighbor order
// (src/utils/CellManager.h:161-186).
__constant__ int c_stencil[13][3] = {
    {0, 0, -1}, {1, 0, -1}, {1, 0, 0},  {1, 0, 1},  {-1, 1, -1},
    {0, 1, -1}, {1, 1, -1}, {-1, 1, 0}, {0, 1, 0},  {1, 1, 0},
    {-1, 1, 1}, {0, 1, 1},  {1, 1, 1}};

struct CellGrid {
    int n[3];
    int nxy, ncell;
    double origin[3];
    double rlen[3];
};

__device__ __forceinline__ int cell_coord(double v, int n) {
    // (Int)(delta*rLen) then clamp (CellManager.h:97-119); v is finite for
    // every in-range coordinate, NaN lands in the last cell.
    if (!(v < (double)n)) return n - 1;
    if (v < 0.0) return 0;
    int x = (int)v;
    return x >= n ? n - 1 : x;
}

// Rebuild preamble of the MD step (LFIntegrator::run :306-341): count the
// update, zero the displacements and shift each molecule so its centre lies
// in the box.
struct RebuildPrep {
    int on;
    double* com;
    double* disp;
    double* scalars;   // [2] list updates
};

// Atom -> cell (CellManager::find_cell, src/utils/CellManager.h:97-119) and the
// per-cell counts, aggregated in LDS when the grid fits there.  One thread
// per molecule, so the MD step's molecule rewrap runs in the same pass.
template <bool LDS_HIST>
__global__ __launch_bounds__(128) void k_cell_assign(int nmol, const int32_t* __restrict__ mol_start, double* pos,
                                                      CellGrid g, Box box, RebuildPrep pr,
                                                      int32_t* __restrict__ cell_of, int32_t* __restrict__ cnt,
                                                      const int* gate) {
    if (gate && !*gate) return;
    extern __shared__ int32_t hist[];
    if constexpr (LDS_HIST) {
        for (int k = threadIdx.x; k < g.ncell; k += blockDim.x) hist[k] = 0;
        __syncthreads();
    }
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m < nmol) {
        const int s = mol_start[m], e = mol_start[m + 1];
        if (pr.on) {
            if (m == 0) pr.scalars[2] += 1.0;
            for (int i = s; i < e; ++i) pr.disp[3 * i] = pr.disp[3 * i + 1] = pr.disp[3 * i + 2] = 0.0;
            const double c0x = pr.com[3 * m], c0y = pr.com[3 * m + 1], c0z = pr.com[3 * m + 2];
            double cx = c0x, cy = c0y, cz = c0z;
            pbc(cx, cy, cz, box);
            const double dx = cx - c0x, dy = cy - c0y, dz = cz - c0z;
            pr.com[3 * m] = cx; pr.com[3 * m + 1] = cy; pr.com[3 * m + 2] = cz;
            for (int i = s; i < e; ++i) { pos[3 * i] += dx; pos[3 * i + 1] += dy; pos[3 * i + 2] += dz; }
        }
        for (int i = s; i < e; ++i) {
            const double dx = pos[3 * i] - g.origin[0];
            const double dy = pos[3 * i + 1] - g.origin[1];
            const double dz = pos[3 * i + 2] - g.origin[2];
            const int x = cell_coord(dx * g.rlen[0], g.n[0]);
            const int y = cell_coord(dy * g.rlen[1], g.n[1]);
            const int z = cell_coord(dz * g.rlen[2], g.n[2]);
            const int c = z * g.nxy + y * g.n[0] + x;
            cell_of[i] = c;
            if constexpr (LDS_HIST) atomicAdd(&hist[c], 1);
            else atomicAdd(&cnt[c], 1);
        }
    }
    if constexpr (LDS_HIST) {
        __syncthreads();
        for (int k = threadIdx.x; k < g.ncell; k += blockDim.x)
            if (hist[k]) atomicAdd(&cnt[k], hist[k]);
    }
}

// One block per cell: its start (the sum of the counts of lower cells) and
// its atoms compacted in index order (set_atom appends in atom order,
// CellManager.cpp:145-170); it stops once the cell is full.  The counts are
// cleared later, by k_list_hits.  A host's build also gets the largest cell
// past the `held` atoms of the hit bits.
constexpr int FILL_THREADS = 1024;
constexpr int FILL_WAVES = FILL_THREADS / WAVE;

__global__ __launch_bounds__(FILL_THREADS) void k_cell_fill(int n, int ncell, const int32_t* __restrict__ cell_of,
                                                            const int32_t* __restrict__ cnt,
                                                            int32_t* __restrict__ start, int32_t* __restrict__ atoms,
                                                            int held, unsigned* largest, const int* gate) {
    if (gate && !*gate) return;
    __shared__ int32_t wsum[FILL_WAVES];
    const int c = blockIdx.x;
    if (c >= ncell) return;
    const int lane = threadIdx.x % WAVE, w = threadIdx.x / WAVE;
    int32_t part = 0;
    for (int k = threadIdx.x; k < c; k += blockDim.x) part += cnt[k];
    part = wave_sum(part);
    if (lane == 0) wsum[w] = part;
    __syncthreads();
    int base = 0;
#pragma unroll
    for (int k = 0; k < FILL_WAVES; ++k) base += wsum[k];
    const int end = base + cnt[c];
    __syncthreads();
    if (threadIdx.x == 0) {
        start[c] = base;
        if (c == ncell - 1) start[ncell] = end;
        if (largest && end - base > held) atomicMax(largest, (unsigned)(end - base));
    }
    const uint64_t below = (1ull << lane) - 1ull;
    for (int a0 = 0; a0 < n && base < end; a0 += FILL_THREADS) {
        const int a = a0 + threadIdx.x;
        const bool hit = (a < n) && (cell_of[a] == c);
        const uint64_t m = __ballot(hit);
        if (lane == 0) wsum[w] = __popcll(m);
        __syncthreads();
        int off = 0, tot = 0;
#pragma unroll
        for (int k = 0; k < FILL_WAVES; ++k) {
            off += k < w ? wsum[k] : 0;
            tot += wsum[k];
        }
        if (hit && base + off + __popcll(m & below) < end) atoms[base + off + __popcll(m & below)] = a;
        base += tot;
        __syncthreads();
    }
}

struct ListArgs {
    int n;
    const double* pos;
    const int32_t* excl_off;
    const int32_t* excl;
    double rlist2;
    Box box;
    int32_t* nb;
    int32_t* nb_cnt;
    int32_t* nb_own;
    int32_t stride;
    unsigned* status;
    uint64_t* mask;    // [27][mask_words][n] hit bits of the cell-pair pass, by cell-order slot
    int mask_words;
};

struct Excl {
    int cnt;
    int lo, hi;        // smallest and largest excluded index
    int ids[8];
    const int32_t* rest;
};

__device__ __forceinline__ bool excluded(const Excl& e, int j) {
    // Ensemble::exclusion_check (src/Ensemble.h:294-305); the first eight
    // entries are compared without a loop so they stay in registers
    if (j < e.lo || j > e.hi) return false;
    bool hit = false;
#pragma unroll
    for (int k = 0; k < 8; ++k) hit = hit || (e.ids[k] == j);
    if (!hit && e.cnt > 8)
        for (int k = 8; k < e.cnt; ++k)
            if (e.rest[k] == j) return true;
    return hit;
}

// Test 64 candidates (one per lane) and append the hits to row i in lane
// order.  Pairs the reference's half list holds in row i ("owned") fill the
// row from the front, in the reference's order; the others fill it from the
// back.
__device__ __forceinline__ void test_and_append(const ListArgs& a, int i, double px, double py, double pz,
                                                const Excl& ex, bool valid, int j, bool owned, bool use_pbc,
                                                int& count, int& n_owned) {
    const int lane = threadIdx.x % WAVE;
    bool hit = false;
    if (valid && !excluded(ex, j)) {
        double dx = a.pos[3 * j] - px;
        double dy = a.pos[3 * j + 1] - py;
        double dz = a.pos[3 * j + 2] - pz;
        if (use_pbc) pbc(dx, dy, dz, a.box);
        hit = len2_exact(dx, dy, dz) < a.rlist2;
    }
    const uint64_t below = (1ull << lane) - 1ull;
    const uint64_t mo = __ballot(hit && owned), mn = __ballot(hit && !owned);
    const int n_non = count - n_owned;
    if (hit) {
        // the two segments meet only on overflow, which the count reports
        const int slot = owned ? n_owned + __popcll(mo & below) : a.stride - 1 - (n_non + __popcll(mn & below));
        if (slot >= 0 && slot < a.stride && (owned ? slot < a.stride - n_non : slot >= n_owned))
            a.nb[(int64_t)i * a.stride + slot] = j;
    }
    count += __popcll(mo) + __popcll(mn);
    n_owned += __popcll(mo);
}

__device__ __forceinline__ Excl load_excl(const ListArgs& a, int i) {
    Excl e;
    const int o = a.excl_off[i];
    e.cnt = a.excl_off[i + 1] - o;
    e.rest = a.excl + o;
#pragma unroll
    for (int k = 0; k < 8; ++k) e.ids[k] = (k < e.cnt) ? e.rest[k] : -1;
    e.lo = INT_MAX;
    e.hi = -1;
    for (int k = 0; k < e.cnt; ++k) {
        e.lo = min(e.lo, (int)e.rest[k]);
        e.hi = max(e.hi, (int)e.rest[k]);
    }
    return e;
}

// ---- cell-pair list build ----------------------------------------------------
//
// Cell c is paired with its neighbour s: s = 0 the cell itself (no PBC,
// CellManager.cpp:257-279), s = 1..13 the forward stencil (the reference's row
// of the atom in c), s = 14..26 the backward stencil (the same pairs seen from
// the other atom).  k_list_hits tests every pair of atoms once and records
// both atoms' hits as bits; k_list_rows, a wave per atom, turns an atom's bits
// into its row.

constexpr int LB_THREADS = 256;
constexpr int LB_WAVES = LB_THREADS / WAVE;

// Neighbour s of cell c, around the box.
__device__ __forceinline__ int neighbour_cell(const CellGrid& g, int c, int s) {
    if (s == 0) return c;
    const int sgn = s <= 13 ? 1 : -1;
    const int k = s <= 13 ? s - 1 : s - 14;
    const int cz = c / g.nxy, cy = (c % g.nxy) / g.n[0], cx = c % g.n[0];
    int xx = cx + sgn * c_stencil[k][0], yy = cy + sgn * c_stencil[k][1], zz = cz + sgn * c_stencil[k][2];
    if (xx >= g.n[0]) xx = 0; else if (xx < 0) xx = g.n[0] - 1;
    if (yy >= g.n[1]) yy = 0; else if (yy < 0) yy = g.n[1] - 1;
    if (zz >= g.n[2]) zz = 0; else if (zz < 0) zz = g.n[2] - 1;
    return zz * g.nxy + yy * g.n[0] + xx;
}

// The reference's distance test of a pair vector.  In the cell itself
// (SELF) it takes no PBC; for a neighbour, apply_pbc's loop makes at most one
// step of L when |d| < 1.5 L (NEAR), which d - L rint(d / L) makes too, in
// the same single operation.  The two may differ for |d| next to L/2 only,
// where neither result is inside a list radius of at most L/3 (a grid has at
// least three cells per axis).  Every operation is odd in d, so the test
// gives the same answer from either atom.
template <bool SELF, bool NEAR>
__device__ __forceinline__ bool list_hit(const ListArgs& a, double dx, double dy, double dz) {
    if constexpr (!SELF) {
        if constexpr (NEAR) pbc_near(dx, dy, dz, a.box);
        else pbc(dx, dy, dz, a.box);
    }
    return len2_exact(dx, dy, dz) < a.rlist2;
}

// One wave's tile: 64 atoms of cell c, one per lane, against nb (up to 64)
// atoms of the neighbour in LDS (whose rows past nb repeat an atom).  Returns
// the lane's hits as bits; back gets, in lane b, the hits of candidate b over
// the 64 atoms (the ballot of the same test), so the backward stencil costs
// no tests of its own.
template <bool SELF, bool NEAR>
__device__ __forceinline__ uint64_t hit_tile(const ListArgs& a, const double (*sj)[3], int nb, double px, double py,
                                             double pz, bool act, uint64_t& back) {
    uint32_t word[2] = {0u, 0u}, blo = 0, bhi = 0;
    const int lane = threadIdx.x % WAVE;
#pragma unroll
    for (int half = 0; half < 2; ++half)
        // four candidates at a time, so that their chains overlap
        for (int b = 32 * half; b < 32 * half + 32 && b < nb; b += 4) {
            bool hit[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                hit[u] = list_hit<SELF, NEAR>(a, sj[b + u][0] - px, sj[b + u][1] - py, sj[b + u][2] - pz) && act;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                word[half] |= hit[u] ? 1u << ((b + u) & 31) : 0u;
                const uint64_t m = __ballot(hit[u]);
                const bool mine = lane == b + u;
                blo = mine ? (uint32_t)m : blo;
                bhi = mine ? (uint32_t)(m >> 32) : bhi;
            }
        }
    back = ((uint64_t)bhi << 32) | blo;
    const uint64_t all = ((uint64_t)word[1] << 32) | word[0];
    return nb < WAVE ? all & ((1ull << nb) - 1ull) : all;
}

// Hits of all pairs of cell blockIdx.x and its neighbour blockIdx.y (0..13),
// in tiles of 64 x 64 atoms, a wave each; word (s, t) of an atom holds its
// hits among atoms 64 t.. of neighbour s.  Exclusions and the atom itself are
// left in; k_list_rows takes them out.  Bound by the FP64 test, about 25
// instructions a pair: 42 us for 4,096 waters in 64 cells (17.4 million
// pairs), 18 for 1,021 in 27; testing each pair from both atoms, a block per
// neighbour, took 63 and 46.
__global__ __launch_bounds__(LB_THREADS) void k_list_hits(ListArgs a, CellGrid g, const int32_t* __restrict__ start,
                                                          const int32_t* __restrict__ catoms,
                                                          int32_t* __restrict__ slot, int32_t* cell_cnt,
                                                          const int* gate) {
    if (gate && !*gate) return;
    __shared__ double sj[LB_WAVES][WAVE][3];
    const int c = blockIdx.x, s = blockIdx.y;
    // the cell counts were last read by k_cell_fill: clear them for the next build
    if (c == 0 && s == 0 && blockIdx.z == 0)
        for (int k = threadIdx.x; k < g.ncell; k += blockDim.x) cell_cnt[k] = 0;
    const int nc = neighbour_cell(g, c, s);
    const int ib = start[c], ie = start[c + 1];
    const int jb = start[nc], je = start[nc + 1];
    const int ti_n = (ie - ib + WAVE - 1) / WAVE, tj_n = (je - jb + WAVE - 1) / WAVE;
    const int lane = threadIdx.x % WAVE, w = threadIdx.x / WAVE;
    const size_t n = a.n;
    for (int t = blockIdx.z * LB_WAVES + w; t < ti_n * tj_n; t += gridDim.z * LB_WAVES) {
        const int ti = t / tj_n, tj = t % tj_n;
        // the places of the cell's atoms, for k_list_rows
        if (s == 0 && ti == tj && ib + ti * WAVE + lane < ie) slot[catoms[ib + ti * WAVE + lane]] = ib + ti * WAVE + lane;
        if ((s == 0 && tj < ti) || (ti >= a.mask_words && tj >= a.mask_words)) continue;
        // the wave's time is one candidate's times the candidates': the
        // larger side takes the lanes
        const int ki = ib + ti * WAVE, kj = jb + tj * WAVE;
        const bool swap = min(WAVE, ie - ki) < min(WAVE, je - kj);
        const int kl = swap ? kj : ki, kl_end = swap ? je : ie, tl = swap ? tj : ti, sl = s == 0 ? 0 : swap ? s + 13 : s;
        const int kc = swap ? ki : kj, kc_end = swap ? ie : je, tc = swap ? ti : tj, sc = s == 0 ? 0 : swap ? s : s + 13;
        const bool act = kl + lane < kl_end;
        const int i = catoms[act ? kl + lane : kl], j = catoms[min(kc + lane, kc_end - 1)];
        const double px = a.pos[3 * i], py = a.pos[3 * i + 1], pz = a.pos[3 * i + 2];
        // |x| < 3/4 L on every axis keeps each pair's |d| under 1.5 L
        bool near = fabs(px) < 0.75 * a.box.L[0] && fabs(py) < 0.75 * a.box.L[1] && fabs(pz) < 0.75 * a.box.L[2];
        wave_lds_order();   // the tile before this one has been read
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const double x = a.pos[3 * j + d];
            sj[w][lane][d] = x;
            near = near && fabs(x) < 0.75 * a.box.L[d];
        }
        wave_lds_order();
        const int nb = min(WAVE, kc_end - kc);
        uint64_t back = 0, word;
        if (s == 0) word = hit_tile<true, true>(a, sj[w], nb, px, py, pz, act, back);
        else if (__all(near)) word = hit_tile<false, true>(a, sj[w], nb, px, py, pz, act, back);
        else word = hit_tile<false, false>(a, sj[w], nb, px, py, pz, act, back);
        if (act && tc < a.mask_words) a.mask[((size_t)sl * a.mask_words + tc) * n + kl + lane] = word;
        if ((s > 0 || ti != tj) && lane < nb && tl < a.mask_words)
            a.mask[((size_t)sc * a.mask_words + tl) * n + kc + lane] = back;
    }
}

// Row of each atom, in cell order, from its hit bits, a wave per atom: lanes
// take the neighbours' candidates in stencil order (ten for the own cell, of
// which most atoms are hits, two for each of the others), so a scan over the
// lanes' counts gives every lane the slots of its hits.  Owned hits (same
// cell j > i, forward cells) fill the row from the front, the others from the
// back; both segments are in the reference's order.  Words of atoms past the
// mask (a neighbour of more than 64 mask_words atoms) are tested here.
// The places are put in order in LDS, so that the row leaves in whole cache
// lines: 42 us at 4,096 waters (430 partners a row), 20 at 1,021; a lane per
// atom and neighbour, each storing to its own row, took 52 and 36 and a pass
// for the slots before it.
// A row longer than the stride is cut to it and filled: owned atoms to its
// end, the others in the slots the owned leave.  In the MD step the pair
// kernels walk the row, up to the stride, before the host reads the status.
// A row past ROW_LDS is stored in place; only a cut one tests each slot (20,000
// atoms, long rows: 603 us, with the test in all of them 729).
constexpr int LR_THREADS = 1024;
constexpr int ROW_LDS = 1024;   // longest row put in order in LDS
__global__ __launch_bounds__(LR_THREADS) void k_list_rows(ListArgs a, CellGrid g, const int32_t* __restrict__ start,
                                                          const int32_t* __restrict__ catoms,
                                                          const int32_t* __restrict__ cell_of,
                                                          const int32_t* __restrict__ slot, const int* gate) {
    if (gate && !*gate) return;
    constexpr int SELF_LANES = 10, WORDS = 4, EXCL = 4;
    static_assert(SELF_LANES % 2 == 0 && SELF_LANES + 52 <= WAVE, "lanes of 27 neighbours");
    __shared__ int32_t ranked[LR_THREADS / WAVE][ROW_LDS];
    const int lane = threadIdx.x % WAVE;
    const int k = blockIdx.x * (LR_THREADS / WAVE) + __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    if (k >= a.n) return;
    const int s = lane < SELF_LANES ? 0 : 1 + (lane - SELF_LANES) / 2;
    const int q = s == 0 ? lane : lane & 1, Q = s == 0 ? SELF_LANES : 2;
    const size_t n = a.n;
    const int i = catoms[k], c = cell_of[i];
    int jb = 0, je = 0, h0 = 0, h1 = 0;
    if (s <= 26) {
        const int nc = neighbour_cell(g, c, s);
        jb = start[nc];
        je = start[nc + 1];
        const int nh = (je - jb + 31) / 32;
        h0 = q * nh / Q;
        h1 = (q + 1) * nh / Q;
    }
    const int e0 = a.excl_off[i], ne = a.excl_off[i + 1] - e0;
    int out[EXCL];   // the first excluded atoms' places
#pragma unroll
    for (int e = 0; e < EXCL; ++e) out[e] = e < ne ? slot[a.excl[e0 + e]] : -1;
    const uint32_t* mask = reinterpret_cast<const uint32_t*>(a.mask + (size_t)s * a.mask_words * n + k);
    // the lane's hits among candidates 32 h.. of its neighbour
    auto hits = [&](int h) {
        uint32_t word = 0;
        const int base = jb + 32 * h;
        if (h < 2 * a.mask_words) {
            word = mask[2 * n * (h >> 1) + (h & 1)];
        } else {
            for (int b = 0; b < 32 && base + b < je; ++b) {
                const int j = catoms[base + b];
                const double dx = a.pos[3 * j] - a.pos[3 * i], dy = a.pos[3 * j + 1] - a.pos[3 * i + 1],
                             dz = a.pos[3 * j + 2] - a.pos[3 * i + 2];
                const bool hit = s == 0 ? list_hit<true, false>(a, dx, dy, dz) : list_hit<false, false>(a, dx, dy, dz);
                word |= hit ? 1u << b : 0u;
            }
        }
        if (s == 0 && (unsigned)(k - base) < 32u) word &= ~(1u << (k - base));
#pragma unroll
        for (int e = 0; e < EXCL; ++e)
            if ((unsigned)(out[e] - base) < 32u) word &= ~(1u << (out[e] - base));
        for (int e = EXCL; e < ne; ++e) {
            const int at = slot[a.excl[e0 + e]] - base;
            if ((unsigned)at < 32u) word &= ~(1u << at);
        }
        return word;
    };
    // which of them row i owns: forward cells, and in its own cell the atoms
    // after it (a cell's atoms are in index order)
    auto owned = [&](int h) {
        if (s > 0) return s <= 13 ? ~0u : 0u;
        const int at = k - (jb + 32 * h);
        return at < 0 ? ~0u : at >= 31 ? 0u : ~0u << (at + 1);
    };
    uint32_t words[WORDS];   // the lane's first words, their loads issued together
    int own = 0, non = 0;
#pragma unroll
    for (int u = 0; u < WORDS; ++u) words[u] = h0 + u < h1 ? hits(h0 + u) : 0u;
#pragma unroll
    for (int u = 0; u < WORDS; ++u) {
        own += __popc(words[u] & owned(h0 + u));
        non += __popc(words[u] & ~owned(h0 + u));
    }
    for (int h = h0 + WORDS; h < h1; ++h) {
        const uint32_t word = hits(h), mine = owned(h);
        own += __popc(word & mine);
        non += __popc(word & ~mine);
    }
    int own_at = own, non_at = non;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
        const int x = __shfl_up(own_at, o), y = __shfl_up(non_at, o);
        own_at += lane >= o ? x : 0;
        non_at += lane >= o ? y : 0;
    }
    const int own_all = __shfl(own_at, WAVE - 1), all = own_all + __shfl(non_at, WAVE - 1);
    own_at -= own;
    non_at -= non;
    if (lane == 0) {
        a.nb_cnt[i] = all;
        a.nb_own[i] = own_all;
        if (all > a.stride) atomicOr(a.status, ST_LIST_OVERFLOW);
    }
    int32_t* row = a.nb + (int64_t)i * a.stride;
    int32_t* order = ranked[threadIdx.x / WAVE];
    // the lane's hits, `put` getting each one's rank (owned ones first) and place
    auto place = [&](auto put) {
        auto bits_of = [&](int h, uint32_t bits) {
            const uint32_t mine = owned(h);
            while (bits) {
                const int b = __ffs(bits) - 1;
                bits &= bits - 1u;
                put(mine >> b & 1u ? own_at++ : own_all + non_at++, jb + 32 * h + b);
            }
        };
#pragma unroll
        for (int u = 0; u < WORDS; ++u) bits_of(h0 + u, words[u]);
        for (int h = h0 + WORDS; h < h1; ++h) bits_of(h, hits(h));
    };
    auto slot_of = [&](int t) { return t < own_all ? t : a.stride - 1 - (t - own_all); };
    if (all > a.stride) {
        place([&](int t, int at) {
            const int to = slot_of(t);
            if (t < own_all ? to < a.stride : to >= own_all) row[to] = catoms[at];
        });
        return;
    }
    if (all > ROW_LDS) {
        place([&](int t, int at) { row[slot_of(t)] = catoms[at]; });
        return;
    }
    place([&](int t, int at) { order[t] = at; });
    wave_lds_order();
    for (int t = lane; t < all; t += WAVE) row[slot_of(t)] = catoms[order[t]];
}

// Ensemble::build_pairlist (src/Ensemble.cpp:492-525): all j != i with the
// min-image predicate; the reference's row i holds the j > i.
__global__ __launch_bounds__(256) void k_pairs_brute(ListArgs a, const int* gate) {
    if (gate && !*gate) return;
    const int i = blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
    if (i >= a.n) return;
    const int lane = threadIdx.x % WAVE;
    const double px = a.pos[3 * i], py = a.pos[3 * i + 1], pz = a.pos[3 * i + 2];
    const Excl ex = load_excl(a, i);
    int count = 0, n_owned = 0;
    for (int j0 = 0; j0 < a.n; j0 += WAVE) {
        const int j = j0 + lane;
        test_and_append(a, i, px, py, pz, ex, j < a.n && j != i, j, j > i, true, count, n_owned);
    }
    if (lane == 0) {
        a.nb_cnt[i] = count;
        a.nb_own[i] = n_owned;
        if (count > a.stride) atomicOr(a.status, ST_LIST_OVERFLOW);
    }
}

// ---------------------------------------------------------------------------

static bool cell_setup(double len, const double L[3], int n[3], double rlen[3]) {
    // CellManager::set_cellManager (src/utils/CellManager.cpp:43-84)
    if ((len <= 0) || (len > L[0] / 3.0) || (len > L[1] / 3.0) || (len > L[2] / 3.0)) return false;
    for (int d = 0; d < 3; ++d) {
        n[d] = (int)(L[d] / len);
        const double cl = L[d] / n[d];
        rlen[d] = 1.0 / cl;
    }
    return true;
}

int pairlist_alloc(Ctx* c, int32_t stride) {
    if (stride <= c->stride && c->d_nb) return SMD_OK;
    if (c->d_nb) (void)hipFree(c->d_nb);
    drop_step_graphs(c);
    c->d_nb = nullptr;
    const size_t bytes = (size_t)c->n * (size_t)stride * sizeof(int32_t);
    if (hipMalloc(&c->d_nb, bytes ? bytes : 4) != hipSuccess) {
        c->stride = 0;
        return fail(c, SMD_ENOMEM, "pair list allocation of %zu bytes failed", bytes);
    }
    c->stride = stride;
    return SMD_OK;
}

// The molecule rewrap alone, for the brute-force list of the MD step.
__global__ __launch_bounds__(256) void k_rebuild_prep(int nmol, const int32_t* __restrict__ mol_start, double* pos,
                                                      Box box, RebuildPrep pr, const int* gate) {
    if (gate && !*gate) return;
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= nmol) return;
    const int s = mol_start[m], e = mol_start[m + 1];
    if (m == 0) pr.scalars[2] += 1.0;
    for (int i = s; i < e; ++i) pr.disp[3 * i] = pr.disp[3 * i + 1] = pr.disp[3 * i + 2] = 0.0;
    const double c0x = pr.com[3 * m], c0y = pr.com[3 * m + 1], c0z = pr.com[3 * m + 2];
    double cx = c0x, cy = c0y, cz = c0z;
    pbc(cx, cy, cz, box);
    const double dx = cx - c0x, dy = cy - c0y, dz = cz - c0z;
    pr.com[3 * m] = cx; pr.com[3 * m + 1] = cy; pr.com[3 * m + 2] = cz;
    for (int i = s; i < e; ++i) { pos[3 * i] += dx; pos[3 * i + 1] += dy; pos[3 * i + 2] += dz; }
}

static int launch_list(Ctx* c, const int* gate, bool md_prep) {
    RebuildPrep pr{};
    pr.on = md_prep ? 1 : 0;
    pr.com = c->d_com;
    pr.disp = c->d_disp;
    pr.scalars = c->d_scalars;
    ListArgs a;
    a.n = c->n;
    a.pos = c->d_pos;
    a.excl_off = c->d_excl_off;
    a.excl = c->d_excl;
    double pc = c->list_cutoff + c->list_buff;   // pairCutOff (src/Ensemble.cpp:456-457)
    pc *= pc;
    a.rlist2 = pc;
    a.box = c->box;
    a.nb = c->d_nb;
    a.nb_cnt = c->d_nb_cnt;
    a.nb_own = c->d_nb_own;
    a.stride = c->stride;
    a.status = c->d_status;
    a.mask = c->d_list_mask;
    a.mask_words = c->list_mask_words;
    const int waves_per_block = 4;
    const dim3 grid((c->n + waves_per_block - 1) / waves_per_block);
    ProfScope ps(c, "pairlist");
    if (c->list_cells) {
        CellGrid g;
        for (int d = 0; d < 3; ++d) {
            g.n[d] = c->ncell[d];
            g.rlen[d] = c->cell_rlen[d];
            g.origin[d] = -c->box.L[d] / 2.0;   // origin0 (CellManager.cpp:74)
        }
        g.nxy = g.n[0] * g.n[1];
        g.ncell = g.nxy * g.n[2];
        const int nc = g.ncell;
        const dim3 ga((c->nmol + 127) / 128);
        if (nc <= 8192)
            hipLaunchKernelGGL((k_cell_assign<true>), ga, dim3(128), sizeof(int32_t) * nc, c->stream, c->nmol,
                               c->d_mol_start, c->d_pos, g, c->box, pr, c->d_cell_of, c->d_cell_cnt, gate);
        else
            hipLaunchKernelGGL((k_cell_assign<false>), ga, dim3(128), 0, c->stream, c->nmol, c->d_mol_start, c->d_pos,
                               g, c->box, pr, c->d_cell_of, c->d_cell_cnt, gate);
        if (c->list_fork) SMD_HIP(c, hipEventRecord(c->list_fork, c->stream));   // positions are final here
        hipLaunchKernelGGL(k_cell_fill, dim3(nc), dim3(FILL_THREADS), 0, c->stream, c->n, nc, c->d_cell_of,
                           c->d_cell_cnt, c->d_cell_start, c->d_cell_atoms, WAVE * c->list_mask_words,
                           gate ? nullptr : c->d_status + 1, gate);
        // tiles of a cell pair beyond four go to further blocks; a dilute grid
        // has less than an atom a cell
        const int tiles = std::max(1, (c->n / nc + WAVE - 1) / WAVE);
        const dim3 gl(nc, 14, std::min(8, (tiles * tiles + LB_WAVES - 1) / LB_WAVES));
        hipLaunchKernelGGL(k_list_hits, gl, dim3(LB_THREADS), 0, c->stream, a, g, c->d_cell_start, c->d_cell_atoms,
                           c->d_cell_slot, c->d_cell_cnt, gate);
        constexpr int per = LR_THREADS / WAVE;
        hipLaunchKernelGGL(k_list_rows, dim3((c->n + per - 1) / per), dim3(LR_THREADS), 0, c->stream, a, g,
                           c->d_cell_start, c->d_cell_atoms, c->d_cell_of, c->d_cell_slot, gate);
    } else {
        if (md_prep)
            hipLaunchKernelGGL(k_rebuild_prep, dim3((c->nmol + 255) / 256), dim3(256), 0, c->stream, c->nmol,
                               c->d_mol_start, c->d_pos, c->box, pr, gate);
        if (c->list_fork) SMD_HIP(c, hipEventRecord(c->list_fork, c->stream));
        hipLaunchKernelGGL(k_pairs_brute, grid, dim3(WAVE * waves_per_block), 0, c->stream, a, gate);
    }
    SMD_HIP(c, hipGetLastError());
    return SMD_OK;
}

// Hit bits for the largest cell a build found, and a quarter more for the
// rebuilds inside a step.  Slabs and droplets fill cells far beyond the mean,
// and k_list_rows tests what the bits do not hold one lane per word.  Calls
// of 16,000 waters in an eighth of their box, radius 1.3 nm, 1,370 -> 420 us;
// 4,096 in a 27th, 446 -> 167.  A list row holds about five atoms for each of a cell's,
// so the bits stay well below the list's own size.  Without the memory the
// smaller mask stays.
static void mask_grow(Ctx* c, int largest) {
    const int words = (largest + largest / 4 + WAVE - 1) / WAVE;
    uint64_t* mask = nullptr;
    if (hipMalloc(&mask, sizeof(uint64_t) * 27 * (size_t)c->n * words) != hipSuccess) {
        (void)hipGetLastError();
        return;
    }
    (void)hipFree(c->d_list_mask);
    c->d_list_mask = mask;
    c->list_mask_words = words;
    drop_step_graphs(c);
}

// Builds the list.  With on_device_flag the kernels are gated on d_flag[0]
// and begin with the MD step's rebuild preamble (used inside the MD step,
// where the Verlet trigger is evaluated on the device); the grid must then
// already be configured.
int pairlist_build(Ctx* c, double cutoff, double cut_buff, int use_cells, bool on_device_flag) {
    if (on_device_flag) return launch_list(c, c->d_flag, true);
    if (!c->box_set) return fail(c, SMD_ESTATE, "box not set");
    c->list_cutoff = cutoff;
    c->list_buff = cut_buff;
    const double len = cutoff + cut_buff;   // cellLen (src/Ensemble.cpp:462)
    int n[3];
    double rl[3];
    c->list_cells = use_cells && cell_setup(len, c->box.L, n, rl);
    if (c->list_cells) {
        for (int d = 0; d < 3; ++d) { c->ncell[d] = n[d]; c->cell_rlen[d] = rl[d]; }
        const int nc = n[0] * n[1] * n[2];
        if (nc + 1 > c->cell_alloc) {
            if (c->d_cell_cnt) (void)hipFree(c->d_cell_cnt);
            if (c->d_cell_start) (void)hipFree(c->d_cell_start);
            SMD_HIP(c, hipMalloc(&c->d_cell_cnt, sizeof(int32_t) * (nc + 1)));
            SMD_HIP(c, hipMalloc(&c->d_cell_start, sizeof(int32_t) * (nc + 1)));
            // k_list_hits clears the counts after each use; they start at zero
            // (hipMemset returns before it is done, and this stream does not
            // wait for the null stream)
            SMD_HIP(c, hipMemsetAsync(c->d_cell_cnt, 0, sizeof(int32_t) * (nc + 1), c->stream));
            c->cell_alloc = nc + 1;
        }
        // hit bits for neighbour cells of up to twice the mean occupancy
        const int words = (2 * c->n / nc + 63) / 64 + 1;
        if (words > c->list_mask_words) {
            if (c->d_list_mask) (void)hipFree(c->d_list_mask);
            c->d_list_mask = nullptr;
            c->list_mask_words = 0;
            drop_step_graphs(c);
            const size_t bytes = sizeof(uint64_t) * 27 * (size_t)c->n * words;
            if (hipMalloc(&c->d_list_mask, bytes) != hipSuccess)
                return fail(c, SMD_ENOMEM, "pair-list mask allocation of %zu bytes failed", bytes);
            c->list_mask_words = words;
        }
    }
    // Row capacity: user value, else estimate from the density and grow on
    // overflow (the list is rebuilt until it fits).
    int32_t stride = c->want_stride;
    if (stride <= 0) {
        const double vol = c->box.L[0] * c->box.L[1] * c->box.L[2];
        const double rho = c->n / vol;
        const double half = rho * 4.0 / 3.0 * PI * len * len * len;   // full row
        stride = (int32_t)(2.5 * half) + 64;
        stride = (stride + 63) / 64 * 64;
        if (stride > c->n) stride = ((c->n + 63) / 64) * 64;
        if (stride < 64) stride = 64;
        if (c->stride > stride) stride = c->stride;
    }
    for (int attempt = 0; attempt < 6; ++attempt) {
        int rc = pairlist_alloc(c, stride);
        if (rc) return rc;
        SMD_HIP(c, hipMemsetAsync(c->d_status, 0, 2 * sizeof(unsigned), c->stream));
        rc = launch_list(c, nullptr, false);
        if (rc) return rc;
        unsigned st[2] = {0, 0};
        SMD_HIP(c, hipMemcpyAsync(st, c->d_status, sizeof st, hipMemcpyDeviceToHost, c->stream));
        SMD_HIP(c, hipStreamSynchronize(c->stream));
        if (c->list_cells && st[1] > (unsigned)(WAVE * c->list_mask_words)) mask_grow(c, (int)st[1]);
        if (!(st[0] & ST_LIST_OVERFLOW)) {
            c->list_valid = true;
            return SMD_OK;
        }
        if (c->want_stride > 0) return fail(c, SMD_ECAPACITY, "pair list row capacity %d exceeded", stride);
        // grow to the observed maximum
        std::vector<int32_t> cnt(c->n);
        SMD_HIP(c, hipMemcpy(cnt.data(), c->d_nb_cnt, sizeof(int32_t) * c->n, hipMemcpyDeviceToHost));
        int32_t mx = 0;
        for (int32_t v : cnt) mx = v > mx ? v : mx;
        stride = ((int32_t)(mx * 1.25) + 64 + 63) / 64 * 64;
    }
    return fail(c, SMD_ECAPACITY, "pair list did not fit after resizing");
}

}  // namespace smd

using namespace smd;

extern "C" int smd_build_pairlist(smd_ctx* c, double cutoff, double cut_buff, int use_cells) {
    if (!c) return SMD_EINVAL;
    if (!(cutoff > 0) || !(cut_buff >= 0)) return fail(c, SMD_EINVAL, "bad cutoff/buffer");
    return pairlist_build(c, cutoff, cut_buff, use_cells, false);
}

extern "C" int smd_set_pairlist_capacity(smd_ctx* c, int32_t row_capacity) {
    if (!c || row_capacity < 0) return SMD_EINVAL;
    c->want_stride = row_capacity;
    return SMD_OK;
}

extern "C" int smd_pairlist_info(smd_ctx* c, int64_t* n_pairs, int32_t* max_row, int32_t* used_cells) {
    if (!c) return SMD_EINVAL;
    if (!c->list_valid) return fail(c, SMD_ESTATE, "no pair list");
    std::vector<int32_t> cnt(c->n), own(c->n);
    SMD_HIP(c, hipStreamSynchronize(c->stream));
    SMD_HIP(c, hipMemcpy(cnt.data(), c->d_nb_cnt, sizeof(int32_t) * c->n, hipMemcpyDeviceToHost));
    SMD_HIP(c, hipMemcpy(own.data(), c->d_nb_own, sizeof(int32_t) * c->n, hipMemcpyDeviceToHost));
    int64_t tot = 0;
    int32_t mx = 0;
    for (int i = 0; i < c->n; ++i) { tot += own[i]; mx = cnt[i] > mx ? cnt[i] : mx; }
    if (n_pairs) *n_pairs = tot;
    if (max_row) *max_row = mx;
    if (used_cells) *used_cells = c->list_cells ? 1 : 0;
    return SMD_OK;
}

// The reference's half list is the front segment of each device row.
extern "C" int smd_get_pairlist(smd_ctx* c, int32_t* offsets, int32_t* nb, int64_t cap) {
    if (!c || !offsets) return SMD_EINVAL;
    if (!c->list_valid) return fail(c, SMD_ESTATE, "no pair list");
    std::vector<int32_t> cnt(c->n), own(c->n);
    SMD_HIP(c, hipStreamSynchronize(c->stream));
    SMD_HIP(c, hipMemcpy(cnt.data(), c->d_nb_cnt, sizeof(int32_t) * c->n, hipMemcpyDeviceToHost));
    SMD_HIP(c, hipMemcpy(own.data(), c->d_nb_own, sizeof(int32_t) * c->n, hipMemcpyDeviceToHost));
    offsets[0] = 0;
    for (int i = 0; i < c->n; ++i) {
        if (cnt[i] > c->stride) return fail(c, SMD_ECAPACITY, "row %d overflowed", i);
        offsets[i + 1] = offsets[i] + own[i];
    }
    if (offsets[c->n] > cap) return fail(c, SMD_ECAPACITY, "need %d entries, cap %lld", offsets[c->n], (long long)cap);
    if (!nb) return SMD_OK;
    std::vector<int32_t> rows((size_t)c->n * c->stride);
    SMD_HIP(c, hipMemcpy(rows.data(), c->d_nb, rows.size() * sizeof(int32_t), hipMemcpyDeviceToHost));
    for (int i = 0; i < c->n; ++i) {
        const int32_t* r = rows.data() + (size_t)i * c->stride;
        std::copy(r, r + own[i], nb + offsets[i]);
    }
    return SMD_OK;
}
