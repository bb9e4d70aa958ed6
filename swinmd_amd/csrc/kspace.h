// kspace.h -- reciprocal space of point charges as matrix products.
//
// exp(i k.r) = X^nx Y^ny Z^nz with X = exp(i 2 pi x / Lx), ... (for a sheared
// cell x is the coordinate along the tilted lattice).  The k set is kept as
// rows (nx, ny), each holding nz = -m..m, and +nz and -nz share everything but
// a sign: with c_n + i s_n = Z^n and a + i b = q X^nx Y^ny,
//
//   structure factors   sum_i {a, b}(row, i) {c_n, s_n}(i)
//   forces              T(row, i) = sum_n U(row, n) c_n(i) + V(row, n) s_n(i),
//                       force on i = sum_rows Im(a + i b)(T, T') (nx, ny, nz)
//
// are products of a 16-row tile with 16 columns over the inner index (atoms,
// or the 2 n1 functions c_n, s_n), which the matrix cores take: FP64
// (v_mfma_f64_16x16x4) in the FP64 form, FP32 (v_mfma_f32_16x16x4) with FP64
// totals every 64 atoms in the mixed form.  Powers come from an FP64
// recurrence in both.  Work per (row, atom): 2 multiply-adds per k for the
// factors, 4 for the forces, the padding of the sphere's rows to n1 included
// about twice that; a walk along nz with a rotation per k takes 8 and more
// vector instructions per k, and k times the latency.
#pragma once

#include <type_traits>

#include "smd_internal.h"

namespace smd {

constexpr int KS_TILE = 64;       // atoms per LDS table
constexpr int KS_MAXW = 8;        // waves of a block, at most
constexpr int KS_THREADS = KS_MAXW * WAVE;
// Waves per SIMD the force pass is compiled for: FP32 fits four without
// spilling (two blocks of eight per CU), FP64 three.
template <typename R> constexpr int KS_FORCE_OCC = sizeof(R) == 8 ? 3 : 4;
constexpr int KS_ROWS = 16;       // rows of a matrix tile
constexpr int KS_VT = 2;          // tiles per wave of the structure-factor pass
constexpr int KS_MAXSTEP = 8;     // inner steps held in registers by the force pass
// LDS of the tables: two blocks to a CU with the force pass's partials beside them
// (12 KiB more), which together are what one launch may ask for at most.
constexpr size_t KS_TABLE_LDS = 65536, KS_CU_LDS = 163840;
static_assert(2 * (KS_TABLE_LDS + (size_t)KS_MAXW * KS_TILE * 3 * sizeof(double)) <= KS_CU_LDS, "k-space LDS");

template <typename R> struct KsMat;
template <> struct KsMat<double> {
    typedef double acc __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ acc mul(double a, double b, acc c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    // row of register r of the product in this lane; the column is lane % 16
    static __device__ __forceinline__ int row(int lane, int r) { return 4 * r + lane / 16; }
};
template <> struct KsMat<float> {
    typedef float acc __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ acc mul(float a, float b, acc c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lane, int r) { return 4 * (lane / 16) + r; }
};

template <typename R> struct alignas(2 * sizeof(R)) KsC { R re, im; };

// Table stride: a wave reads 16 powers of 4 neighbouring atoms.  Sixteen-byte
// entries are read 16 lanes at a time, which an odd stride puts on distinct
// banks; eight-byte ones 32 at a time, 16 powers of 2 atoms, which 2 mod 32
// does.
template <typename R>
__host__ __device__ constexpr int ks_stride() { return KS_TILE + (sizeof(R) == 8 ? 1 : 2); }

// Waves of a block for `units` tiles, `per` of them per wave at a time, so
// that no wave has one more than the others where that can be avoided.
inline int ks_waves(int units, int per, int most, int least) {
    const int passes = (units + most * per - 1) / (most * per);
    const int w = (units + passes * per - 1) / (passes * per);
    return w < least ? least : w;
}
template <typename R>
__device__ __forceinline__ KsC<R> ks_mul(KsC<R> a, KsC<R> b) {
    return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}

struct KsRows {
    int nrows, n1;       // rows; nz = 0..n1-1 and their negatives
    int nx1, ny1;        // powers of X (0..nx1-1) and of Y (0..ny1-1, conjugated for ny < 0)
    int ts;              // table stride (ks_stride of the pass's precision)
    const int* xy;       // [nrows] nx << 16 | (ny & 0xffff)
    __host__ __device__ int tiles() const { return (nrows + KS_ROWS - 1) / KS_ROWS; }
    __host__ __device__ int powers() const { return nx1 + ny1 + n1; }
    __host__ __device__ int steps() const { return (2 * n1 + 3) / 4; }   // of four functions
    __host__ __device__ int col_groups() const { return (n1 + 15) / 16; }
    __host__ __device__ bool half() const { return n1 <= 8; }   // c_n and s_n fit in 16 columns
    __host__ __device__ size_t table_entries() const { return (size_t)powers() * ts; }
    // per-row coefficients of the force pass: [tile][4][4 steps][16]
    __host__ __device__ size_t coef_entries() const { return (size_t)tiles() * 4 * steps() * 4 * KS_ROWS; }
};
__host__ __device__ inline int ks_nx(int v) { return v >> 16; }
__host__ __device__ inline int ks_ny(int v) { return (int)(short)(v & 0xffff); }

// Powers 0..cnt-1 of (c1, s1) into column u of a table, times f.
template <typename R>
__device__ __forceinline__ void ks_powers(KsC<R>* tab, int ts, int u, int cnt, double c1, double s1, double f) {
    double er = f, ei = 0.0;
    tab[u] = {(R)er, (R)ei};
    for (int k = 1; k < cnt; ++k) {
        const double nr = er * c1 - ei * s1, ni = er * s1 + ei * c1;
        er = nr; ei = ni;
        tab[(size_t)k * ts + u] = {(R)er, (R)ei};
    }
}

// Tables (with several weights also their values) of a structure-factor pass
// that a block fills together, so that their loads and phases overlap: as many
// as fit in KS_TABLE_LDS, or with several weights in twice that, one block to
// a CU being what its accumulators leave room for; at most KS_TABLES.
constexpr int KS_TABLES = 4;
template <typename R>
__host__ __device__ inline size_t ks_table_bytes(const KsRows& kr, int nw) {
    return kr.table_entries() * 2 * sizeof(R) + (nw > 1 ? (size_t)nw * KS_TILE * sizeof(R) : 0);
}
template <typename R>
__host__ __device__ inline int ks_tables(const KsRows& kr, int nw, int chunk_tiles) {
    const int fit = (int)((nw > 1 ? 2 : 1) * KS_TABLE_LDS / ks_table_bytes<R>(kr, nw));
    const int m = fit < KS_TABLES ? fit : KS_TABLES;
    return m < 1 ? 1 : (m < chunk_tiles ? m : chunk_tiles);
}

// Tables of atoms t0.. up to i1: a wave per (table, axis or weights), lane u
// filling column u.  Columns past i1 have charge 0.
template <typename R, int NW, typename At>
__device__ __forceinline__ void ks_fill(const KsRows& kr, const At& at, int t0, int i1, int nt, KsC<R>* tabs) {
    constexpr int TASKS = NW > 1 ? 4 : 3;
    const size_t te = ks_table_bytes<R>(kr, NW) / sizeof(KsC<R>);   // a table, then its weights
    const int lane = threadIdx.x % WAVE, w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    for (int task = w; task < nt * TASKS; task += blockDim.x / WAVE) {
        const int tb = task / TASKS, fp = task % TASKS;
        const int ia = t0 + tb * KS_TILE + lane;
        const bool live = ia < i1;
        KsC<R>* tab = tabs + tb * te;
        if (fp < 3) {
            double2 p = make_double2(1.0, 0.0);
            double f = 1.0;
            if (live) p = at.phase(ia, fp);
            if (fp == 0) f = live ? at.charge(ia) : 0.0;
            const int base = fp == 0 ? 0 : (fp == 1 ? kr.nx1 : kr.nx1 + kr.ny1);
            ks_powers<R>(tab + (size_t)base * kr.ts, kr.ts, lane, fp == 0 ? kr.nx1 : (fp == 1 ? kr.ny1 : kr.n1), p.x, p.y,
                         f);
        } else {
            double d[3] = {0.0, 0.0, 0.0};
            if (live) at.offset(ia, d);
            R* q = reinterpret_cast<R*>(tab + kr.table_entries()) + lane;
            q[0] = R(1);
            q[KS_TILE] = (R)d[0];
            q[2 * KS_TILE] = (R)d[1];
            q[3 * KS_TILE] = (R)d[2];
            q[4 * KS_TILE] = (R)(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
        }
    }
}

// This lane's place in a unit of the structure factors, 16 rows by 16 n.
template <typename R>
struct KsUnit {
    int ox, oy, oz;
    R sy;
    __device__ __forceinline__ KsUnit(const KsRows& kr, int tile, int cg, int cols = 16) {
        const int lane = threadIdx.x % WAVE;
        const int v = kr.xy[min(tile * KS_ROWS + lane % 16, kr.nrows - 1)];
        ox = ks_nx(v) * kr.ts;
        oy = (kr.nx1 + abs(ks_ny(v))) * kr.ts;
        oz = (kr.nx1 + kr.ny1 + min(lane % cols + 16 * cg, kr.n1 - 1)) * kr.ts;
        sy = ks_ny(v) < 0 ? R(-1) : R(1);
    }
    __device__ __forceinline__ KsC<R> row(const KsC<R>* tab, int u) const {
        KsC<R> y = tab[oy + u];
        y.im *= sy;
        return ks_mul(tab[ox + u], y);
    }
};

// Sums of the four products {a, b} {c_n, s_n} of one unit and weight: FP64
// products add up in their accumulators, FP32 ones enter FP64 sums after every
// table.
// HALF (KsRows::half): c_n and s_n share the 16 columns, so two products do.
// compute_long, mixed, |n|^2 <= 49: 96,000 atoms 140 -> 113 us, 12,288 57 -> 52.
template <typename R, bool HALF = false>
struct KsAcc {
    static constexpr bool SPLIT = sizeof(R) == 4;
    static constexpr int NP = HALF ? 2 : 4;
    typename KsMat<R>::acc acc[NP];
    double tot[SPLIT ? NP : 1][SPLIT ? 4 : 1];
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                acc[p][r] = R(0);
                if constexpr (SPLIT) tot[p][r] = 0.0;
            }
    }
    __device__ __forceinline__ void add(R er, R ei, KsC<R> z) {
        typedef KsMat<R> M;
        if constexpr (HALF) {
            const R f = threadIdx.x % 16 < 8 ? z.re : z.im;
            acc[0] = M::mul(er, f, acc[0]);
            acc[1] = M::mul(ei, f, acc[1]);
        } else {
            acc[0] = M::mul(er, z.re, acc[0]);
            acc[1] = M::mul(er, z.im, acc[1]);
            acc[2] = M::mul(ei, z.re, acc[2]);
            acc[3] = M::mul(ei, z.im, acc[3]);
        }
    }
    __device__ __forceinline__ void table_end() {
        if constexpr (SPLIT) {
#pragma unroll
            for (int p = 0; p < NP; ++p)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    tot[p][r] += (double)acc[p][r];
                    acc[p][r] = R(0);
                }
        }
    }
    // out[((row nw + w) 4 + p) n1 + n]
    __device__ __forceinline__ void store(const KsRows& kr, double* __restrict__ out, int nw, int tile, int cg, int w) const {
        const int lane = threadIdx.x % WAVE, n = HALF ? lane % 8 : lane % 16 + 16 * cg;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = tile * KS_ROWS + KsMat<R>::row(lane, r);
            if (n < kr.n1 && row < kr.nrows)
#pragma unroll
                for (int p = 0; p < NP; ++p) {
                    const int product = HALF ? 2 * p + lane / 8 % 2 : p;
                    double* o = out + ((size_t)(row * nw + w) * 4 + product) * kr.n1 + n;
                    if constexpr (SPLIT) *o = tot[p][r];
                    else *o = acc[p][r];
                }
        }
    }
};

// Structure factors of atoms [i0, i1), by one block with `nt` tables:
// out[(row 4 + p) n1 + n] is the sum over the atoms of a c_n, a s_n, b c_n,
// b s_n (p = 0..3).  The block takes the (group of 16 n, vpw tiles per wave)
// sets g0, g0 + gs, ... (vpw at most KS_VT).  At gives an atom's phase per axis
// and its charge.  Tables that hold the whole chunk stay for all of the
// block's sets.
template <typename R, typename At>
__device__ __forceinline__ void ks_sfac(const KsRows& kr, const At& at, int i0, int i1, int g0, int gs, int vpw, int nt,
                                        void* lds, double* __restrict__ out) {
    const size_t te = ks_table_bytes<R>(kr, 1) / sizeof(KsC<R>);
    KsC<R>* const tabs = static_cast<KsC<R>*>(lds);
    const int lane = threadIdx.x % WAVE, w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int nw = blockDim.x / WAVE, groups = (kr.tiles() + nw * vpw - 1) / (nw * vpw);
    bool filled = false;
    const bool stay = i1 - i0 <= nt * KS_TILE;
    for (int g = g0; g < groups * kr.col_groups(); g += gs) {
        const int cg = g / groups, tile0 = g % groups * nw * vpw + w;
        const bool on0 = tile0 < kr.tiles(), on1 = vpw > 1 && tile0 + nw < kr.tiles();
        const KsUnit<R> unit[KS_VT] = {{kr, on0 ? tile0 : 0, cg}, {kr, on1 ? tile0 + nw : 0, cg}};
        KsAcc<R> sum[KS_VT];
#pragma unroll
        for (int t = 0; t < KS_VT; ++t) sum[t].clear();
        for (int t0 = i0; t0 < i1; t0 += KS_TILE) {
            const int tb = (t0 - i0) / KS_TILE % nt;
            if (tb == 0 && !filled) {
                __syncthreads();
                ks_fill<R, 1>(kr, at, t0, i1, nt, tabs);
                __syncthreads();
                filled = stay;
            }
            const KsC<R>* tab = tabs + tb * te;
            // One or both tiles per pass over the table, without a branch
            // inside, so the reads of later steps are issued ahead of the
            // products; columns past i1 add zeros.
            auto products = [&](auto tiles) {
#pragma unroll 4
                for (int k = 0; k < KS_TILE / 4; ++k) {
                    const int u = 4 * k + lane / 16;
                    const KsC<R> z = tab[unit[0].oz + u];
#pragma unroll
                    for (int t = 0; t < decltype(tiles)::value; ++t) {
                        const KsC<R> e = unit[t].row(tab, u);
                        sum[t].add(e.re, e.im, z);
                    }
                }
            };
            if (on1) products(std::integral_constant<int, 2>{});   // wave-uniform
            else if (on0) products(std::integral_constant<int, 1>{});
#pragma unroll
            for (int t = 0; t < KS_VT; ++t) sum[t].table_end();
        }
        if (on0) sum[0].store(kr, out, 1, tile0, cg, 0);
        if (on1) sum[1].store(kr, out, 1, tile0 + nw, cg, 0);
    }
}

// The same with the weights 1, d_i and |d_i|^2 (d = r - R_mol, from At's
// offset): out[((row 5 + w) 4 + p) n1 + n].  A block of `split` h waves takes
// the h units (tile, group of 16 n) of set g, a wave the unit v % h with a
// share of the weights: split 2, the first three or the other two, so that a
// row's values are formed once for its weights, a SIMD holds a wave of each
// kind and the chunk's atoms pass through the tables once; split 5, one each.
constexpr int KS_WEIGHTS = 5;
template <typename R, bool HALF, typename At>
__device__ __forceinline__ void ks_sfac_weights(const KsRows& kr, const At& at, int i0, int i1, int g, int split, int nt,
                                                void* lds, double* __restrict__ out) {
    const size_t te = ks_table_bytes<R>(kr, KS_WEIGHTS) / sizeof(KsC<R>);
    KsC<R>* const tabs = static_cast<KsC<R>*>(lds);
    const int lane = threadIdx.x % WAVE, w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int h = blockDim.x / WAVE / split, id = g * h + w % h, part = w / h;
    const int w0 = split == 2 ? 3 * part : part, nw = split == 2 ? 3 - part : 1;
    const int tile = id % kr.tiles(), cg = id / kr.tiles();
    const bool on = cg < kr.col_groups();
    const KsUnit<R> unit(kr, tile, on ? cg : 0, HALF ? 8 : 16);
    KsAcc<R, HALF> sum[3];
#pragma unroll
    for (int t = 0; t < 3; ++t) sum[t].clear();
    for (int t0 = i0; t0 < i1; t0 += KS_TILE) {
        const int tb = (t0 - i0) / KS_TILE % nt;
        if (tb == 0) {
            __syncthreads();
            ks_fill<R, KS_WEIGHTS>(kr, at, t0, i1, nt, tabs);
            __syncthreads();
        }
        const KsC<R>* tab = tabs + tb * te;
        const R* wts = reinterpret_cast<const R*>(tab + kr.table_entries()) + w0 * KS_TILE;
        auto products = [&](auto weights) {
#pragma unroll 2
            for (int k = 0; k < KS_TILE / 4; ++k) {
                const int u = 4 * k + lane / 16;
                const KsC<R> z = tab[unit.oz + u], e = unit.row(tab, u);
#pragma unroll
                for (int t = 0; t < decltype(weights)::value; ++t) {
                    const R f = wts[t * KS_TILE + u];
                    sum[t].add(e.re * f, e.im * f, z);
                }
            }
        };
        if (on && nw == 3) products(std::integral_constant<int, 3>{});   // wave-uniform
        else if (on && nw == 2) products(std::integral_constant<int, 2>{});
        else if (on) products(std::integral_constant<int, 1>{});
#pragma unroll
        for (int t = 0; t < 3; ++t) sum[t].table_end();
    }
    if (on)
#pragma unroll
        for (int t = 0; t < 3; ++t)
            if (t < nw) sum[t].store(kr, out, KS_WEIGHTS, tile, cg, w0 + t);
}
// Its sets for nt tables of atoms: of at most four units, the same number in
// all of them but the last; or where there is one unit, or units and tables
// together make at most two blocks to a CU, a unit each with a wave per weight
// (3,000 atoms, 1,535 k in FP64: compute_long 56 us, 59 with four units).
struct KsSets { int count, units, split; };
inline KsSets ks_weight_sets(const KsRows& kr, int nt) {
    const int u = kr.tiles() * kr.col_groups(), sets = (u + KS_MAXW / 2 - 1) / (KS_MAXW / 2);
    if (u == 1 || u * nt <= 512) return {u, 1, KS_WEIGHTS};
    return {sets, (u + sets - 1) / sets, 2};
}

// The force pass's coefficients of one (row, n) from G+ = (bC, bS) of +nz and
// G- of -nz (0 where the set has no such k): functions 2n (c_n) and 2n + 1
// (s_n) of the four outputs Re T, Im T, Re T', Im T'.
template <typename R>
__device__ __forceinline__ void ks_coef(const KsRows& kr, R* __restrict__ coef, int row, int n, double cp, double sp,
                                        double cm, double sm) {
    // conj(G+) + conj(G-) and i (conj(G+) - conj(G-))
    const double ur = cp + cm, ui = -(sp + sm), vr = sp - sm, vi = cp - cm;
    const int kp = 4 * kr.steps();
    R* w = coef + ((size_t)(row / KS_ROWS) * 4 * kp + 2 * n) * KS_ROWS + row % KS_ROWS;
    const size_t o = (size_t)kp * KS_ROWS;
    const double f = (double)n;
    w[0] = (R)ur;                 w[KS_ROWS] = (R)vr;
    w[o] = (R)ui;                 w[o + KS_ROWS] = (R)vi;
    w[2 * o] = (R)(f * vi);       w[2 * o + KS_ROWS] = (R)(-f * ui);
    w[3 * o] = (R)(-f * vr);      w[3 * o + KS_ROWS] = (R)(f * ur);
}
// Zeros for the functions past 2 n1 and, in rows past the last, all of them.
template <typename R>
__device__ __forceinline__ void ks_coef_pad(const KsRows& kr, R* __restrict__ coef, int row, int tid, int nt) {
    const int kp = 4 * kr.steps(), from = row < kr.nrows ? 2 * kr.n1 : 0;
    for (int t = tid; t < 4 * (kp - from); t += nt) {
        const int o = t / (kp - from), k = from + t % (kp - from);
        coef[(((size_t)(row / KS_ROWS) * 4 + o) * kp + k) * KS_ROWS + row % KS_ROWS] = R(0);
    }
}

// The table, then the waves' partial forces.
template <typename R>
__host__ __device__ inline size_t ks_force_table(const KsRows& kr) { return (kr.table_entries() * 2 * sizeof(R) + 15) / 16 * 16; }
template <typename R>
inline size_t ks_force_lds(const KsRows& kr, int waves) {
    return ks_force_table<R>(kr) + (size_t)waves * KS_TILE * 3 * sizeof(double);
}

// Waves of the force pass for so many blocks: the tiles in turn, or where
// tiles and blocks are few, each tile's four groups of 16 atoms over two or
// four waves (ks_force_split).  In FP64 over four only, up to a block for half
// the CUs: beside the pair kernel its waves take what that kernel has (a step
// of 4,096 waters with |n|^2 <= 27, three tiles over two waves 113 us, else
// 104; 1,500, 90 and 86; mixed 86, 88).
__host__ __device__ inline int ks_force_split(int tiles, int waves) {
    return 4 * tiles <= waves ? 4 : (2 * tiles <= waves ? 2 : 1);
}
inline int ks_force_waves(const KsRows& kr, int blocks, bool mixed) {
    const int t = kr.tiles(), most = ks_force_split(t, KS_MAXW);
    const int split = (mixed ? blocks <= 256 : blocks <= 128 && most == 4) ? most : 1;
    return split == 1 ? ks_waves(t, 1, KS_MAXW, 3) : (split * t < 3 ? 3 : split * t);
}

// sum_k (bC sin(k.r) - bS cos(k.r)) (nx, ny, nz) of atoms [i0, i0 + 64), by
// one block of three waves or more: thread t < 192 returns atom i0 + t / 3,
// component t % 3.  A wave holds a tile's coefficients in registers, all KS
// inner steps of them, or with KS = 0 (more than KS_MAXSTEP) KS_MAXSTEP at a
// time for two groups of atoms, in FP64 half of that for one.  SPLIT: the launch may have split
// the tiles' atoms over waves.
template <typename R, int KS, bool SPLIT, typename At>
__device__ __forceinline__ double ks_force(const KsRows& kr, const At& at, const R* __restrict__ coef, int i0, int i1,
                                           void* lds) {
    typedef KsMat<R> M;
    KsC<R>* tab = static_cast<KsC<R>*>(lds);
    const int lane = threadIdx.x % WAVE, w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int fu = threadIdx.x % KS_TILE, fp = threadIdx.x / KS_TILE, nw = blockDim.x / WAVE;
    if (fp < 3) {
        const int ia = min(i0 + fu, i1 - 1);   // idle columns repeat the last atom; nothing reads them
        const double2 p = at.phase(ia, fp);
        const int base = fp == 0 ? 0 : (fp == 1 ? kr.nx1 : kr.nx1 + kr.ny1);
        ks_powers<R>(tab + (size_t)base * kr.ts, kr.ts, fu, fp == 0 ? kr.nx1 : (fp == 1 ? kr.ny1 : kr.n1), p.x,
                     p.y, 1.0);
    }
    __syncthreads();
    const KsC<R>* tz = tab + (size_t)(kr.nx1 + kr.ny1) * kr.ts;
    const int steps = KS ? KS : kr.steps(), kp = 4 * steps;
    const int split = SPLIT ? ks_force_split(kr.tiles(), nw) : 1, tw = w / split, ntw = nw / split;
    const int a0 = SPLIT ? w % split * (4 / split) : 0, a1 = SPLIT ? a0 + 4 / split : 4;
    // functions 4 s + lane / 16: part (lane / 16) & 1 of power 2 s + lane / 32
    const R* tzp = reinterpret_cast<const R*>(tz) + ((lane / 16) & 1);
    double* part = reinterpret_cast<double*>(static_cast<char*>(lds) + ks_force_table<R>(kr)) + (size_t)w * KS_TILE * 3;
    for (int tile = tw; tile < kr.tiles(); tile += ntw) {
        const R* cw = coef + (size_t)tile * 4 * kp * KS_ROWS + lane;   // function lane / 16 of a step, row lane % 16
        int ox[4], oy[4];
        R sy[4];
        double nx[4], ny[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int v = kr.xy[min(tile * KS_ROWS + M::row(lane, r), kr.nrows - 1)];
            ox[r] = ks_nx(v) * kr.ts;
            oy[r] = (kr.nx1 + abs(ks_ny(v))) * kr.ts;
            sy[r] = ks_ny(v) < 0 ? R(-1) : R(1);
            nx[r] = (double)ks_nx(v);
            ny[r] = (double)ks_ny(v);
        }
        // the tile's share of the forces on atoms 16 a.. from its T
        auto add = [&](int a, const typename M::acc (&T)[4]) {
            const int u = 16 * a + lane % 16;
            double g[3] = {0.0, 0.0, 0.0};
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                KsC<R> y = tab[oy[r] + u];
                y.im *= sy[r];
                const KsC<R> e = ks_mul(tab[ox[r] + u], y);
                const double val = (double)(e.im * T[0][r] + e.re * T[1][r]);
                g[0] = fma(val, nx[r], g[0]);
                g[1] = fma(val, ny[r], g[1]);
                g[2] += (double)(e.im * T[2][r] + e.re * T[3][r]);
            }
            // the four lanes of an atom hold different rows of the tile
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                g[d] += __shfl_xor(g[d], 16, WAVE);
                g[d] += __shfl_xor(g[d], 32, WAVE);
            }
            if (lane < 16) {
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    double* o = part + 3 * u + d;
                    *o = tile == tw ? g[d] : *o + g[d];
                }
            }
        };
        auto function = [&](int s, int a) {
            return tzp[2 * (min(2 * s + lane / 32, kr.n1 - 1) * kr.ts + 16 * a + lane % 16)];   // within KS_TABLE_LDS
        };
        if constexpr (KS > 0) {
            R A[4][KS];
#pragma unroll
            for (int o = 0; o < 4; ++o)
#pragma unroll
                for (int s = 0; s < KS; ++s) A[o][s] = cw[((size_t)o * kp + 4 * s) * KS_ROWS];
            auto group = [&](int a) {
                typename M::acc T[4] = {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
                for (int s = 0; s < KS; ++s) {
                    const R bz = function(s, a);
#pragma unroll
                    for (int o = 0; o < 4; ++o) T[o] = M::mul(A[o][s], bz, T[o]);
                }
                add(a, T);
            };
            if (split == 1)   // all four, a loop of known length
                for (int a = 0; a < 4; ++a) group(a);
            else
                for (int a = a0; a < a1; ++a) group(a);
        } else {
            // FP64 holds half the steps for a group at a time, which leaves room
            // for another wave (300 waters in a box of 1:1:12, 1:1:6 with 500:
            // a step 93 -> 87 us, 85 -> 82)
            constexpr int GROUPS = sizeof(R) == 8 ? 1 : 2, HELD = KS_MAXSTEP * GROUPS / 2;
            for (int a = a0; a < a1; a += GROUPS) {
                typename M::acc T[GROUPS][4] = {};
                for (int s0 = 0; s0 < steps; s0 += HELD) {
                    R A[4][HELD];   // steps past the last: coefficients read again, times no function
#pragma unroll
                    for (int o = 0; o < 4; ++o)
#pragma unroll
                        for (int s = 0; s < HELD; ++s)
                            A[o][s] = cw[((size_t)o * kp + 4 * min(s0 + s, steps - 1)) * KS_ROWS];
#pragma unroll
                    for (int s = 0; s < HELD; ++s) {
                        const bool in = s0 + s < steps;
                        if (GROUPS == 1 && !in) break;
#pragma unroll
                        for (int u = 0; u < GROUPS; ++u) {
                            // a group past the wave's last repeats it and is not added
                            const R bz = in ? function(s0 + s, SPLIT ? min(a + u, a1 - 1) : a + u) : R(0);
#pragma unroll
                            for (int o = 0; o < 4; ++o) T[u][o] = M::mul(A[o][s], bz, T[u][o]);
                        }
                    }
                }
#pragma unroll
                for (int u = 0; u < GROUPS; ++u)
                    if (!SPLIT || a + u < a1) add(a + u, T[u]);
            }
        }
    }
    __syncthreads();
    double f = 0.0;
    if (threadIdx.x < 3 * KS_TILE) {
        const int a = (int)threadIdx.x / 3 / 16, aw = a / (4 / split);   // the waves of this atom's group
        for (int v = 0; v < min(ntw, kr.tiles()); ++v)
            f += part[(ptrdiff_t)(v * split + aw - w) * KS_TILE * 3 + threadIdx.x];
    }
    return f;
}

}  // namespace smd
