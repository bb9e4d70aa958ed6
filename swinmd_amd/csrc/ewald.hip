// ewald.hip -- point-charge Ewald pieces other than the real-space pair loop.
//
//   set_up / ctor             src/forces/EwaldForce.cpp:21-89, :198-257  (host)
//   intraMolCorrect           :709-813   one thread per molecule
//   surfDipoleCorrect         :816-937   two passes over atoms
//   reciprocal_term           :529-698   structure factors, then forces
//
// Reciprocal space: kspace.h.  Three launches:
//   k_recip_sfac: structure factors of an atom chunk, phases exp(i 2 pi r_p /
//     L_p) evaluated on the way and kept for the forces.  With Lustig terms
//     also the sums weighted by d = r - R_mol and |d|^2; in FP64 those take
//     k_recip_phase and k_recip_walk, on the vector units.
//   k_recip_reduce: partials summed over chunks in a fixed order, then per k:
//     energy, volume derivatives and virial (:596-607) and the force pass's
//     coefficients; the reference's per-atom Lustig sums of the force loop
//     (:609-658) are sums over atoms of products with the per-k sums, so they
//     are formed here per k.
//   k_recip_force: forces of 64 atoms per block.  Without Lustig sums (the MD
//     steps, which report no second derivative) it also forms the first
//     derivative's molecular part, sum_k sum_i f_ik (k.d_i) = sum_i F_i . d_i,
//     so the d-weighted structure factors are not needed there.
// Every sum is taken in a fixed order: results do not depend on scheduling.
#include <algorithm>
#include <cstdlib>
#include <mutex>

#include "kspace.h"
#include "smd_internal.h"

namespace smd {

constexpr int SF_CHUNKS = 256; // blocks of the structure-factor passes, at most: one per CU
constexpr int GK = 8;          // k of a run: consecutive nz within one (nx, ny) row
constexpr int WALK_SUMS = 10;  // per-k sums of k_recip_walk
constexpr int WALK_WAVES = 8;  // its waves per block: the same runs, different atoms

// The structure factors with Lustig terms: as products (mixed, and FP64 where
// blocks are few) in chunks of whole tiles, sets.count blocks each; or in FP64
// by k_recip_walk in chunks of 32 atoms and more, a block per 64 runs each.
// At most `most` chunks, and a block per CU.
struct LustigPlan {
    bool walk;
    KsSets sets;
    int per, chunks;
    size_t part;   // doubles of a chunk's partials
};
static LustigPlan lustig_plan(const KsRows& kr, int n, int K, int runs, int most, bool mixed) {
    const int nt = (n + KS_TILE - 1) / KS_TILE;
    LustigPlan p;
    p.sets = ks_weight_sets(kr, nt);
    p.walk = !mixed && p.sets.split == 2 && (!kr.half() || kr.tiles() * nt > 3072);
    if (p.walk) {
        const int c = std::max(1, std::min(most, SF_CHUNKS / ((runs + WAVE - 1) / WAVE)));
        p.per = std::max(32, (n + c - 1) / c);
        p.part = (size_t)K * WALK_SUMS;
    } else {
        const int c = std::max(1, std::min({nt, most, SF_CHUNKS / p.sets.count}));
        p.per = (nt + c - 1) / c * KS_TILE;
        p.part = (size_t)kr.nrows * KS_WEIGHTS * 4 * kr.n1;
    }
    p.chunks = (n + p.per - 1) / p.per;
    return p;
}

// d_e1 holds the phases [n][3] (complex) and then, 32-byte aligned, the
// per-atom (q, d) of k_recip_walk.
static size_t e1_am_offset(int n) { return (6 * (size_t)n + 3) & ~(size_t)3; }

// ---- host setup -----------------------------------------------------------

int ewald_setup(Ctx* c, const smd_ewald_params* p) {
    if (!c->box_set) return fail(c, SMD_ESTATE, "box not set");
    if (!(p->alpha > 0) || !(p->real_cut > 0) || !(p->kcut > 0)) return fail(c, SMD_EINVAL, "bad Ewald parameters");
    c->ew = *p;
    const double kCut2 = p->kcut * p->kcut;
    const double alpha2 = p->alpha * p->alpha;
    const double alphaR4 = 1.0 / (4.0 * alpha2);
    int nmax[3];
    for (int d = 0; d < 3; ++d) nmax[d] = (int)(p->kcut * c->box.L[d] / (2 * PI));
    const double vx = 2.0 * PI / c->box.L[0], vy = 2.0 * PI / c->box.L[1], vz = 2.0 * PI / c->box.L[2];
    std::vector<int32_t> kn;
    std::vector<double> ek;
    for (int nx = 0; nx <= nmax[0]; nx++) {
        const double kx = nx * vx;
        for (int ny = (nx == 0 ? 0 : -nmax[1]); ny <= nmax[1]; ny++) {
            const double ky = ny * vy;
            for (int nz = ((nx == 0 && ny == 0) ? 1 : -nmax[2]); nz <= nmax[2]; nz++) {
                const double kz = nz * vz;
                const double k2 = kx * kx + ky * ky + kz * kz;
                if (k2 < kCut2) {
                    ek.push_back(exp(-k2 * alphaR4) / k2);
                    kn.push_back(nx); kn.push_back(ny); kn.push_back(nz);
                }
            }
        }
    }
    const int K = (int)ek.size();
    if (K == 0) return fail(c, SMD_EINVAL, "no k-vectors below kcut");
    for (int d = 0; d < 3; ++d) c->nmax[d] = nmax[d];
    auto realloc = [&](auto*& ptr, size_t bytes) -> int {
        if (ptr) (void)hipFree(ptr);
        ptr = nullptr;
        if (hipMalloc(&ptr, bytes) != hipSuccess) return fail(c, SMD_ENOMEM, "Ewald allocation of %zu bytes", bytes);
        return SMD_OK;
    };
    // rows (nx, ny) of the set, in its order, and per (row, |nz|) the factor
    // exp(-k^2 / 4 alpha^2) / k^2, 0 where the set has no such k
    KsRows kr{};
    kr.n1 = nmax[2] + 1;
    kr.nx1 = nmax[0] + 1;
    kr.ny1 = nmax[1] + 1;
    // runs of at most GK consecutive nz in a row, stored as (first k, count,
    // nx << 16 | (ny & 0xffff), nz of the first k); the rows' first k
    std::vector<int32_t> xy, rowk;
    std::vector<double> rexp;
    std::vector<int4> runs;
    for (int k = 0; k < K; ++k) {
        const int v = (kn[3 * k] << 16) | (kn[3 * k + 1] & 0xffff);
        const bool same = !xy.empty() && xy.back() == v;
        if (same && kn[3 * k + 2] == kn[3 * k - 1] + 1 && runs.back().y < GK) ++runs.back().y;
        else runs.push_back(make_int4(k, 1, v, kn[3 * k + 2]));
        if (!same) {
            xy.push_back(v);
            rowk.push_back(k);
            rexp.resize(rexp.size() + kr.n1, 0.0);
        }
        rexp[rexp.size() - kr.n1 + std::abs(kn[3 * k + 2])] = ek[k];
    }
    rowk.push_back(K);
    kr.nrows = (int)xy.size();
    const int ng = (int)runs.size();
    // The sets this path takes: the powers and weights of 64 atoms, and 16
    // bytes per k and per run of eight, within 64 KiB.
    const size_t ne = (size_t)nmax[0] + nmax[1] + nmax[2] + 3;
    if (ne * ks_stride<double>() * 16 + 5 * KS_TILE * 8 > KS_TABLE_LDS || (size_t)(K + ng) * 16 > KS_TABLE_LDS)
        return fail(c, SMD_ENOTSUP, "reciprocal space too large for the LDS-resident passes (%d k-vectors, nmax %d %d %d)",
                    K, nmax[0], nmax[1], nmax[2]);
    int rc;
    if ((rc = realloc(c->d_kxy, sizeof(int32_t) * xy.size()))) return rc;
    if ((rc = realloc(c->d_expk, sizeof(double) * rexp.size()))) return rc;
    if ((rc = realloc(c->d_kf, sizeof(double) * kr.coef_entries()))) return rc;
    const int nt = (c->n + KS_TILE - 1) / KS_TILE;
    c->sfac_chunks = std::max(1, std::min(nt, SF_CHUNKS));
    // the largest of the forms' partials: one weight, or with Lustig terms
    size_t part = (size_t)kr.nrows * 4 * kr.n1 * c->sfac_chunks;
    for (bool mixed : {false, true}) {
        const LustigPlan p = lustig_plan(kr, c->n, K, ng, SF_CHUNKS, mixed);
        part = std::max(part, p.part * p.chunks);
    }
    if ((rc = realloc(c->d_sfac_part, sizeof(double) * part))) return rc;
    if ((rc = realloc(c->d_e1, sizeof(double) * (e1_am_offset(c->n) + 4 * (size_t)c->n)))) return rc;
    if ((rc = realloc(c->d_kruns, sizeof(int4) * runs.size()))) return rc;
    if ((rc = realloc(c->d_rowk, sizeof(int32_t) * rowk.size()))) return rc;
    SMD_HIP(c, hipMemcpy(c->d_kruns, runs.data(), sizeof(int4) * runs.size(), hipMemcpyHostToDevice));
    SMD_HIP(c, hipMemcpy(c->d_rowk, rowk.data(), sizeof(int32_t) * rowk.size(), hipMemcpyHostToDevice));
    SMD_HIP(c, hipMemcpy(c->d_kxy, xy.data(), sizeof(int32_t) * xy.size(), hipMemcpyHostToDevice));
    SMD_HIP(c, hipMemcpy(c->d_expk, rexp.data(), sizeof(double) * rexp.size(), hipMemcpyHostToDevice));
    c->n_krows = kr.nrows;
    c->n_kruns = ng;
    c->K = K;
    // self and charged-system energies (ctor :69-79)
    double qSum = 0.0, q2Sum = 0.0;
    for (int i = 0; i < c->n; ++i) { qSum += c->h_q[i]; q2Sum += c->h_q[i] * c->h_q[i]; }
    const double volume = c->box.L[0] * c->box.L[1] * c->box.L[2];
    c->self_energy = -q2Sum * p->alpha / SQRT_PI;
    c->charged_energy = 0.0;
    if (fabs(qSum) > 1.0e-5) c->charged_energy = -PI * qSum * qSum / (2.0 * volume * alpha2);
    c->ewald_ready = true;
    return SMD_OK;
}

// ---- intramolecular correction ---------------------------------------------

struct IntraArgs {
    int nmol;
    Box box;
    const int32_t* mol_start;
    const double* pos;
    const double* q;
    const int32_t* excl_off;
    const int32_t* excl;
    double* force;
    double* terms;
    Red red;
    double alpha, alpha2, alpha2PI, volume;
    int use_constraint;
};

__global__ __launch_bounds__(256) void k_ewald_intra(IntraArgs a) {
    // EwaldForce::intraMolCorrect (src/forces/EwaldForce.cpp:709-813)
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    double v[4] = {0.0, 0.0, 0.0, 0.0};   // sum qij erf/r, U_i, molderiv, mol2ndDeriv
    if (m < a.nmol) {
        const int s = a.mol_start[m], e = a.mol_start[m + 1];
        const double vol2 = a.volume * a.volume;
        for (int i = s; i < e; ++i) {
            const double qi = a.q[i];
            const double rix = a.pos[3 * i], riy = a.pos[3 * i + 1], riz = a.pos[3 * i + 2];
            for (int j = i + 1; j < e; ++j) {
                bool ex = false;
                for (int k = a.excl_off[i]; k < a.excl_off[i + 1]; ++k) ex = ex || (a.excl[k] == j);
                if (!ex) continue;
                double dx = a.pos[3 * j] - rix, dy = a.pos[3 * j + 1] - riy, dz = a.pos[3 * j + 2] - riz;
                pbc(dx, dy, dz, a.box);
                const double r2 = dx * dx + dy * dy + dz * dz;
                const double r = sqrt(r2);
                const double qij = qi * a.q[j];
                const double er = erf(a.alpha * r) / r;
                const double ex2 = exp(-a.alpha2 * r2);
                v[0] += qij * er;
                v[1] += a.alpha2PI * qij * ex2;
                if (!a.use_constraint) {
                    const double dudr = er - a.alpha2PI * ex2;
                    v[2] += qij * dudr / (3.0 * a.volume);
                    v[3] += (-2.0 * qij * dudr + qij * (-2.0 * dudr + 2.0 * a.alpha2PI * a.alpha2 * ex2 * r2)) / (9.0 * vol2);
                    const double s2 = qij * dudr / r2;
                    // atoms of one molecule belong to this thread only
                    a.force[3 * i] += s2 * dx; a.force[3 * i + 1] += s2 * dy; a.force[3 * i + 2] += s2 * dz;
                    a.force[3 * j] -= s2 * dx; a.force[3 * j + 1] -= s2 * dy; a.force[3 * j + 2] -= s2 * dz;
                }
            }
        }
    }
    block_part<4>(v, a.red, RS_EW_INTRA);
}

int ewald_intra(Ctx* c, int lustig) {
    (void)lustig;
    IntraArgs a;
    a.nmol = c->nmol;
    a.box = c->box;
    a.mol_start = c->d_mol_start;
    a.pos = c->d_pos;
    a.q = c->d_q;
    a.excl_off = c->d_excl_off;
    a.excl = c->d_excl;
    a.force = c->d_force;
    a.terms = c->d_terms;
    a.red = c->red;
    a.alpha = c->ew.alpha;
    a.alpha2 = a.alpha * a.alpha;
    a.alpha2PI = 2.0 * a.alpha / SQRT_PI;
    a.volume = c->box.L[0] * c->box.L[1] * c->box.L[2];
    a.use_constraint = c->ew.use_constraint;
    ProfScope ps(c, "ewald_intra");
    hipLaunchKernelGGL(k_ewald_intra, dim3((c->nmol + 255) / 256), dim3(256), 0, c->stream, a);
    SMD_HIP(c, hipGetLastError());
    return red_finish(c, RS_EW_INTRA, (c->nmol + 255) / 256, 4, c->d_terms + T_IN_E);
}

// ---- surface dipole ---------------------------------------------------------

// The dipole sums feed every atom's force: block partials added in block
// order by a finisher launch, so the forces do not depend on scheduling.
__global__ __launch_bounds__(256) void k_surf_sums(int n, const double* __restrict__ pos, const double* __restrict__ q,
                                                   const int32_t* __restrict__ mol, const double* __restrict__ com,
                                                   double* part) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    double v[6] = {0, 0, 0, 0, 0, 0};
    if (i < n) {
        const double qi = q[i];
        const int m = mol[i];
        for (int d = 0; d < 3; ++d) { v[d] = qi * pos[3 * i + d]; v[3 + d] = qi * com[3 * m + d]; }
    }
    block_store<6>(v, part, gridDim.x);
}

__global__ __launch_bounds__(256) void k_surf_force(int n, const double* __restrict__ pos, const double* __restrict__ q,
                                                    double* __restrict__ force, double* terms, double coeff,
                                                    Red red) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const double qx = coeff * terms[T_SU_QR], qy = coeff * terms[T_SU_QR + 1], qz = coeff * terms[T_SU_QR + 2];
    double v[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    if (i < n) {
        const double qi = q[i];
        const double tx = -qi * qx, ty = -qi * qy, tz = -qi * qz;
        const double rx = pos[3 * i], ry = pos[3 * i + 1], rz = pos[3 * i + 2];
        const double s = 2.0 * qi;
        force[3 * i] -= s * qx; force[3 * i + 1] -= s * qy; force[3 * i + 2] -= s * qz;
        v[0] = tx * rx; v[1] = ty * rx; v[2] = tz * rx;
        v[3] = tx * ry; v[4] = ty * ry; v[5] = tz * ry;
        v[6] = tx * rz; v[7] = ty * rz; v[8] = tz * rz;
    }
    block_part<9>(v, red, RS_EW_SURF);
}

int ewald_surface(Ctx* c) {
    const double volume = c->box.L[0] * c->box.L[1] * c->box.L[2];
    const double coeff = 2.0 * PI * (1.0 / volume) / 3.0;
    const dim3 g((c->n + 255) / 256);
    hipLaunchKernelGGL(k_surf_sums, g, dim3(256), 0, c->stream, c->n, c->d_pos, c->d_q, c->d_mol, c->d_com,
                       c->part_su);
    int rc = rows_finish(c, c->stream, c->part_su, (int)g.x, (int)g.x, 6, c->d_terms + T_SU_QR);
    if (rc) return rc;
    hipLaunchKernelGGL(k_surf_force, g, dim3(256), 0, c->stream, c->n, c->d_pos, c->d_q, c->d_force, c->d_terms, coeff,
                       c->red);
    SMD_HIP(c, hipGetLastError());
    return red_finish(c, RS_EW_SURF, g.x, 9, c->d_terms + T_SU_VIR);
}

// ---- reciprocal space ---------------------------------------------------------

struct RecipArgs {
    int n, K, chunks, per;     // atoms per chunk, a multiple of KS_TILE
    int vpw;                   // tiles per wave of the structure factors at a time
    KsSets sets;               // with Lustig terms
    int nper;                  // n of a row per block of k_recip_reduce
    int ng;                    // runs
    const int4* runs;
    const int32_t* rowk;       // [nrows + 1] first k of each row
    double4* am;               // [n] (q, d) per atom, d = r - R_mol
    KsRows kr;
    double vk[3];              // 2 pi / L per axis
    const double* pos;
    const double* q;
    const int32_t* mol;
    const double* com;
    const double* expk;        // [nrows][n1]
    double* part;              // [chunk][nrows][weights][4][n1], of k_recip_walk [chunk][K][WALK_SUMS]
    void* kf;                  // force-pass coefficients, R
    double2* e1;               // [n][3] exp(i 2 pi r_p / L_p) per atom
    double* force;
    int store;                 // 1: the force pass stores (separate array), 0: adds
    Red red;
    double alphaR4, pi4V, pi8V;
};

struct RecipAtoms {
    const RecipArgs& a;
    bool keep;                 // this block's phases go to e1 for the force pass
    __device__ __forceinline__ double2 phase(int i, int p) const {
        double s, c;
        sincos(a.vk[p] * a.pos[3 * i + p], &s, &c);
        const double2 e = make_double2(c, s);
        if (keep) a.e1[3 * i + p] = e;
        return e;
    }
    __device__ __forceinline__ double charge(int i) const { return a.q[i]; }
    __device__ __forceinline__ void offset(int i, double (&d)[3]) const {
        const int m = a.mol[i];
#pragma unroll
        for (int k = 0; k < 3; ++k) d[k] = a.pos[3 * i + k] - a.com[3 * m + k];
    }
};

struct RecipPhases {
    const double2* e1;
    __device__ __forceinline__ double2 phase(int i, int p) const { return e1[3 * i + p]; }
};

// Few atoms wait for the table fill (loads, sincos, powers: about 6 us with
// the launch), many for the matrix cores.  64 atoms a block until 256 blocks
// are reached.  The three kernels alone, mixed, 12,288 atoms, 1,535 k: factors
// 10.0, sums 8.9, forces 9.5 us; a walk along nz on the vector units took
// 3.8 (phases) + 23.0, 6.2 and 20.9.  3,063 atoms in FP64: 11, 7.3, 11.9
// against 3.0 + 17.4, 6.0 and 23.7; 48,000 atoms beside the pair kernel: the
// step 383 -> 316 us.
template <typename R, int NW, bool HALF>
__global__ __launch_bounds__(KS_THREADS) void k_recip_sfac(RecipArgs a) {
    extern __shared__ double lds[];
    const int i0 = blockIdx.x * a.per, i1 = min(a.n, i0 + a.per);
    const RecipAtoms at{a, blockIdx.y == 0};
    const int nt = ks_tables<R>(a.kr, NW, a.per / KS_TILE);
    double* part = a.part + (size_t)blockIdx.x * a.kr.nrows * NW * 4 * a.kr.n1;
    if constexpr (NW > 1) ks_sfac_weights<R, HALF>(a.kr, at, i0, i1, blockIdx.y, a.sets.split, nt, lds, part);
    else ks_sfac<R>(a.kr, at, i0, i1, blockIdx.y, gridDim.y, a.vpw, nt, lds, part);
}

// FP64 with Lustig terms, many atoms: the matrix cores multiply FP64 at the
// vector units' rate on this card, and five weights of 16-row tiles padded to
// 16 functions are two to three times the arithmetic of a walk over the set
// itself.  48,000 atoms, 1,535 k 93 us and the phases 6 (as products 83 to 98);
// few atoms wait for latencies, which the products spread over more blocks:
// 648 atoms, 1,535 k 13 + 2.5 us (10.5).  Long axes pad most: 2,048 waters in a
// 1:1:2 box, 78 us a call (86).  Where c_n and s_n share the columns
// the padding is half, and the products hold longer (lustig_plan).  A call of
// compute_long with |n|^2 <= 49 at 24,576, 48,000 and 96,000 atoms: walk 72, 95
// and 141 us, products 70, 99 and 154; <= 27: 61, 71 and 94 against 58, 70, 97.
__global__ __launch_bounds__(256) void k_recip_phase(RecipArgs a) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    const RecipAtoms at{a, true};
    if (k < a.n) {
        double d[3];
        at.offset(k, d);
        a.am[k] = make_double4(a.q[k], d[0], d[1], d[2]);
    }
    if (k < 3 * a.n) at.phase(k / 3, k % 3);
}

// A block of WALK_WAVES waves owns 64 runs (one per lane) and a chunk of
// atoms.  Per 64-atom table a lane starts its run at q X^nx Y^ny Z^nz0 and
// walks along nz, each term the one before times Z.  Per k: 0 q sin, 1 q cos,
// 2-4 q cos d, 5-7 q sin d, 8 q cos |d|^2, 9 q sin |d|^2 (reciprocal_term
// :568-594 and the moments its force loop needs).  The waves split a table's
// atoms and are added in LDS, in order.
__global__ __launch_bounds__(WALK_WAVES * WAVE) void k_recip_walk(RecipArgs a) {
    extern __shared__ double lds[];
    static_assert(WALK_WAVES * WAVE >= 4 * KS_TILE, "one fill task per thread");
    KsC<double>* tab = reinterpret_cast<KsC<double>*>(lds);
    const int ts = a.kr.ts, ey0 = a.kr.nx1, ez0 = ey0 + a.kr.ny1;
    double* misc = reinterpret_cast<double*>(tab + a.kr.table_entries());   // [5][KS_TILE]: q, d, |d|^2
    const int lane = threadIdx.x % WAVE, w = threadIdx.x / WAVE;
    const int g = blockIdx.x * WAVE + lane;
    const int i0 = blockIdx.y * a.per, i1 = min(a.n, i0 + a.per);
    const int4 run = g < a.ng ? a.runs[g] : make_int4(0, 0, 0, 0);
    const int nx = ks_nx(run.z), ny = ks_ny(run.z);
    const int ox = nx * ts, oy = (ey0 + abs(ny)) * ts, oz = (ez0 + abs(run.w)) * ts;
    const double sy = ny < 0 ? -1.0 : 1.0, sz = run.w < 0 ? -1.0 : 1.0;
    double acc[GK][WALK_SUMS];
#pragma unroll
    for (int t = 0; t < GK; ++t)
#pragma unroll
        for (int u = 0; u < WALK_SUMS; ++u) acc[t][u] = 0.0;
    // thread fu + KS_TILE fp writes atom fu's powers along axis fp (fp < 3) or
    // its moments; its inputs for the next table are loaded before the current
    // one is walked
    const int fu = threadIdx.x % KS_TILE, fp = threadIdx.x / KS_TILE;
    double2 pe = make_double2(1.0, 0.0);
    double4 pm = make_double4(0.0, 0.0, 0.0, 0.0);
    auto fetch = [&](int t0) {
        const int ia = t0 + fu;
        if (fp < 3 && ia < i1) pe = a.e1[3 * ia + fp];
        else if (fp == 3 && ia < i1) pm = a.am[ia];
    };
    fetch(i0);
    for (int t0 = i0; t0 < i1; t0 += KS_TILE) {
        const int na = min(KS_TILE, i1 - t0);
        __syncthreads();
        if (fp < 3 && fu < na) {
            const int base = fp == 0 ? 0 : (fp == 1 ? ey0 : ez0);
            ks_powers<double>(tab + (size_t)base * ts, ts, fu, fp == 0 ? a.kr.nx1 : (fp == 1 ? a.kr.ny1 : a.kr.n1), pe.x,
                              pe.y, 1.0);
        } else if (fp == 3 && fu < na) {
            misc[fu] = pm.x;
            misc[KS_TILE + fu] = pm.y;
            misc[2 * KS_TILE + fu] = pm.z;
            misc[3 * KS_TILE + fu] = pm.w;
            misc[4 * KS_TILE + fu] = pm.y * pm.y + pm.z * pm.z + pm.w * pm.w;
        }
        __syncthreads();
        fetch(t0 + KS_TILE);
        if (g < a.ng)
            for (int u = w; u < na; u += WALK_WAVES) {
                KsC<double> Y = tab[oy + u], Z = tab[oz + u];
                Y.im *= sy;
                Z.im *= sz;
                KsC<double> e = ks_mul(ks_mul(tab[ox + u], Y), Z);
                const double q = misc[u];
                e.re *= q;
                e.im *= q;
                // Z itself; without one (n1 = 1) a run has one k
                const KsC<double> z1 = tab[(ez0 + min(1, a.kr.n1 - 1)) * ts + u];
                const double dx = misc[KS_TILE + u], dy = misc[2 * KS_TILE + u], dz = misc[3 * KS_TILE + u];
                const double d2 = misc[4 * KS_TILE + u];
                // all GK sums are formed (uniform control flow); those past
                // the run's count are never stored
#pragma unroll
                for (int t = 0; t < GK; ++t) {
                    acc[t][0] += e.im;
                    acc[t][1] += e.re;
                    acc[t][2] += e.re * dx; acc[t][3] += e.re * dy; acc[t][4] += e.re * dz;
                    acc[t][5] += e.im * dx; acc[t][6] += e.im * dy; acc[t][7] += e.im * dz;
                    acc[t][8] += e.re * d2; acc[t][9] += e.im * d2;
                    e = ks_mul(e, z1);
                }
            }
    }
    double* red = lds;   // [(WALK_WAVES - 1) * WAVE][WALK_SUMS]
#pragma unroll
    for (int t = 0; t < GK; ++t) {
        __syncthreads();
        if (w > 0)
#pragma unroll
            for (int u = 0; u < WALK_SUMS; ++u) red[((w - 1) * WAVE + lane) * WALK_SUMS + u] = acc[t][u];
        __syncthreads();
        if (w == 0 && t < run.y) {
            double* p = a.part + ((size_t)blockIdx.y * a.K + run.x + t) * WALK_SUMS;
#pragma unroll
            for (int u = 0; u < WALK_SUMS; ++u) {
                double s = acc[t][u];
                for (int v = 0; v < WALK_WAVES - 1; ++v) s += red[(v * WAVE + lane) * WALK_SUMS + u];
                p[u] = s;
            }
        }
    }
}

// One block per row and nper n (and per padding row of the last tile, which only
// clears its coefficients).  The waves sum an equal share of the chunks each,
// in order, and their shares are added in order; then a thread takes the row's
// k with nz = +-n.  Bound by the latency of the chunk loads, so a block is as
// many waves as there are shares of a dozen chunks.
// NW 0: the sums of k_recip_walk.
template <typename R, int NW>
__global__ __launch_bounds__(1024) void k_recip_reduce(RecipArgs a) {
    extern __shared__ double lds[];
    constexpr bool WALK = NW == 0, LUSTIG = NW != 1;
    const int row = blockIdx.y, n0 = blockIdx.x * a.nper, blocks = gridDim.x * gridDim.y;
    const int lane = threadIdx.x % WAVE, qt = threadIdx.x / WAVE;
    R* kf = static_cast<R*>(a.kf);
    if (n0 == 0) ks_coef_pad<R>(a.kr, kf, row, threadIdx.x, blockDim.x);
    double o[3 + 9 + 4] = {0};   // energy, longDeriv, long2ndDeriv, virial[9], Ff, Ffk2, d2UV1, d2UrR
    if (row < a.kr.nrows) {
        const int nn = min(a.nper, a.kr.n1 - n0);   // this block's n, at most 58: the set's limit on nmax
        const int k0 = WALK ? a.rowk[row] : 0, count = WALK ? a.rowk[row + 1] - k0 : 0;
        // the walk's row runs over nz = -m..m, the first over 1..m
        const int m = a.kr.xy[row] == 0 ? count : (count - 1) / 2, zero = a.kr.xy[row] == 0 ? -1 : m;   // k of nz = 0
        // values of +n and of -n (walk) or of all weights and products
        const int nv = WALK ? 2 * nn * WALK_SUMS : NW * 4 * nn;
        auto place = [&](int v) -> int64_t {
            if constexpr (WALK) {
                const int n = n0 + v / (2 * WALK_SUMS), neg = v / WALK_SUMS & 1, k = zero + (neg ? -n : n);
                return n <= m && k >= 0 ? (int64_t)(k0 + k) * WALK_SUMS + v % WALK_SUMS : -1;
            } else {
                if (nn == a.kr.n1) return (int64_t)row * nv + v;
                return ((int64_t)row * NW * 4 + v / nn) * a.kr.n1 + n0 + v % nn;
            }
        };
        // wave qt: share qt / vw of the chunks, values qt % vw of vw
        const int nw = blockDim.x / WAVE, vw = NW == 1 ? 1 : min((nv + WAVE - 1) / WAVE, nw), nq = nw / vw, q = qt / vw;
        const int c0 = (a.chunks * q) / nq, c1 = (a.chunks * (q + 1)) / nq;
        const size_t stride = WALK ? (size_t)a.K * WALK_SUMS : (size_t)a.kr.nrows * NW * 4 * a.kr.n1;
        for (int v = (qt % vw) * WAVE + lane; v < nv && q < nq; v += vw * WAVE) {
            const int64_t at = place(v);
            double s = 0.0;
            if (at >= 0) {
                const double* p = a.part + at;
#pragma unroll 8
                for (int ch = c0; ch < c1; ++ch) s += p[(size_t)ch * stride];
            }
            lds[q * nv + v] = s;
        }
        __syncthreads();
        for (int v = threadIdx.x; v < nv; v += blockDim.x) {
            double s = lds[v];
            for (int u = 1; u < nq; ++u) s += lds[u * nv + v];
            lds[v] = s;
        }
        __syncthreads();
        const int n = n0 + threadIdx.x;
        if (threadIdx.x < nn) {
            const int v = a.kr.xy[row];
            const int nx = ks_nx(v), ny = ks_ny(v);
            const double ek = a.expk[(size_t)row * a.kr.n1 + n];
            const double kx = nx * a.vk[0], ky = ny * a.vk[1];
            double sum[WALK ? 1 : NW][4];
            if constexpr (!WALK) {
#pragma unroll
                for (int w = 0; w < NW; ++w)
#pragma unroll
                    for (int p = 0; p < 4; ++p) sum[w][p] = lds[(w * 4 + p) * nn + threadIdx.x];
            }
            const double b = a.pi8V * ek;
            double G[2][2] = {{0.0, 0.0}, {0.0, 0.0}};
            // +nz, and -nz where the half space has it
            const int signs = ek == 0.0 ? 0 : (n == 0 || (nx == 0 && ny == 0) ? 1 : 2);
            for (int s = 0; s < signs; ++s) {
                const double sg = s ? -1.0 : 1.0;
                const double kz = sg * n * a.vk[2];
                const double k2 = kx * kx + ky * ky + kz * kz;
                const double* sk = lds + (2 * threadIdx.x + s) * WALK_SUMS;   // of the walk
                double cosSum, sinSum, cd[4], sd[4];   // and with the weights d, |d|^2
                if constexpr (WALK) {
                    sinSum = sk[0];
                    cosSum = sk[1];
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        cd[w] = sk[w < 3 ? 2 + w : 8];
                        sd[w] = sk[w < 3 ? 5 + w : 9];
                    }
                } else {
                    cosSum = sum[0][0] - sg * sum[0][3];
                    sinSum = sum[0][2] + sg * sum[0][1];
#pragma unroll
                    for (int w = 0; w < NW - 1; ++w) {
                        cd[w] = sum[w + 1][0] - sg * sum[w + 1][3];
                        sd[w] = sum[w + 1][2] + sg * sum[w + 1][1];
                    }
                }
                const double te = a.pi4V * ek * (sinSum * sinSum + cosSum * cosSum);
                const double coeff = 2.0 * (a.alphaR4 + 1.0 / k2);
                const double kk = (te * kx) * kx + (te * ky) * ky + (te * kz) * kz;
                o[0] += te;
                o[1] += -te + kk * 2.0 * a.alphaR4;
                const double t7 = ((7.0 * te * kx) * kx + (7.0 * te * ky) * ky + (7.0 * te * kz) * kz) * 2.0 * a.alphaR4;
                const double dd = kk * 2.0 * a.alphaR4;
                const double t2 = ((dd * kx) * kx + (dd * ky) * ky + (dd * kz) * kz) * 2.0 * a.alphaR4;
                o[2] += 4.0 * te - t7 + t2;
                o[3 + 0] += te - te * coeff * kx * kx;
                o[3 + 4] += te - te * coeff * ky * ky;
                o[3 + 8] += te - te * coeff * kz * kz;
                o[3 + 1] += -te * coeff * kx * ky;
                o[3 + 2] += -te * coeff * kx * kz;
                o[3 + 5] += -te * coeff * ky * kz;
                if constexpr (LUSTIG) {
                    // sum_i val_i (k.d_i) with val_i = b (q_i sin_i C - q_i cos_i S)
                    const double kSD = kx * sd[0] + ky * sd[1] + kz * sd[2];
                    const double kCD = kx * cd[0] + ky * cd[1] + kz * cd[2];
                    const double ff = b * (cosSum * kSD - sinSum * kCD);
                    o[12] += ff;
                    o[13] += ff * (4.0 * a.alphaR4 * k2);
                    const double bkk = (b * kx) * kx + (b * ky) * ky + (b * kz) * kz;
                    o[14] += bkk * (cosSum * cd[3] + sinSum * sd[3]);
                    o[15] += bkk * ((cd[0] * cd[0] + cd[1] * cd[1] + cd[2] * cd[2]) +
                                    (sd[0] * sd[0] + sd[1] * sd[1] + sd[2] * sd[2]));
                }
                G[s][0] = b * cosSum;
                G[s][1] = b * sinSum;
            }
            ks_coef<R>(a.kr, kf, row, n, G[0][0], G[0][1], G[1][0], G[1][1]);
        }
        o[3 + 3] = o[3 + 1];
        o[3 + 6] = o[3 + 2];
        o[3 + 7] = o[3 + 5];
    }
    // the sums are in the first wave; the rest of the block has none
    if (threadIdx.x < WAVE && blocks <= a.red.cap) {
        double* part = red_part(a.red, RS_RECIP) + blockIdx.y * gridDim.x + blockIdx.x;
#pragma unroll
        for (int k = 0; k < (LUSTIG ? 16 : 12); ++k) {
            const double t = wave_sum(o[k]);
            if (threadIdx.x == 0) part[(size_t)k * a.red.cap] = t;
        }
    }
}

// Force on atom i, sum_k (b C q sin - b S q cos) k (:609-658).  FF: also the
// block's sum of F . d (T_RC_FF).
template <typename R, int KS, bool FF, bool SPLIT>
__global__ __launch_bounds__(KS_THREADS, KS_FORCE_OCC<R>) void k_recip_force(RecipArgs a) {
    extern __shared__ double lds[];
    const int i0 = blockIdx.x * KS_TILE;
    const RecipPhases at{a.e1};
    const double g = ks_force<R, KS, SPLIT>(a.kr, at, static_cast<const R*>(a.kf), i0, a.n, lds);
    const int i = i0 + (int)threadIdx.x / 3, d = threadIdx.x % 3;
    double ff[1] = {0.0};
    if (threadIdx.x < 3 * KS_TILE && i < a.n) {
        const double f = a.q[i] * g * a.vk[d];
        if (a.store) a.force[3 * i + d] = f;
        else a.force[3 * i + d] += f;
        if constexpr (FF) ff[0] = f * (a.pos[3 * i + d] - a.com[3 * a.mol[i] + d]);
    }
    if constexpr (FF) {
        __syncthreads();
        block_part<1>(ff, a.red, RS_RECIP_FF);
    }
}

template <typename R, bool FF, bool SPLIT>
static void launch_recip_force(hipStream_t s, const RecipArgs& a, int waves) {
    const dim3 g((a.n + KS_TILE - 1) / KS_TILE), b(waves * WAVE);
    const size_t lds = ks_force_lds<R>(a.kr, waves);
    switch (a.kr.steps()) {
        case 1: hipLaunchKernelGGL((k_recip_force<R, 1, FF, SPLIT>), g, b, lds, s, a); break;
        case 2: hipLaunchKernelGGL((k_recip_force<R, 2, FF, SPLIT>), g, b, lds, s, a); break;
        case 3: hipLaunchKernelGGL((k_recip_force<R, 3, FF, SPLIT>), g, b, lds, s, a); break;
        case 4: hipLaunchKernelGGL((k_recip_force<R, 4, FF, SPLIT>), g, b, lds, s, a); break;
        case 5: hipLaunchKernelGGL((k_recip_force<R, 5, FF, SPLIT>), g, b, lds, s, a); break;
        case 6: hipLaunchKernelGGL((k_recip_force<R, 6, FF, SPLIT>), g, b, lds, s, a); break;
        case 7: hipLaunchKernelGGL((k_recip_force<R, 7, FF, SPLIT>), g, b, lds, s, a); break;
        case 8: hipLaunchKernelGGL((k_recip_force<R, 8, FF, SPLIT>), g, b, lds, s, a); break;
        default: hipLaunchKernelGGL((k_recip_force<R, 0, FF, SPLIT>), g, b, lds, s, a); break;
    }
}
template <typename R, bool FF>
static void launch_recip_force(hipStream_t s, const RecipArgs& a) {
    const int waves = ks_force_waves(a.kr, (a.n + KS_TILE - 1) / KS_TILE, sizeof(R) == 4);
    if (ks_force_split(a.kr.tiles(), waves) > 1) launch_recip_force<R, FF, true>(s, a, waves);
    else launch_recip_force<R, FF, false>(s, a, waves);
}

static dim3 recip_reduce_grid(const RecipArgs& a) {
    return dim3((a.kr.n1 + a.nper - 1) / a.nper, a.kr.tiles() * KS_ROWS);
}

// NW 0: by k_recip_walk.
template <typename R, int NW>
static void launch_recip_sums(hipStream_t s, const RecipArgs& a, unsigned passes) {
    if (passes & RECIP_SFAC) {
        if constexpr (NW == 0) {
            hipLaunchKernelGGL(k_recip_phase, dim3((3 * a.n + 255) / 256), dim3(256), 0, s, a);
            const size_t lds = std::max(ks_table_bytes<double>(a.kr, KS_WEIGHTS),
                                        (size_t)(WALK_WAVES - 1) * WAVE * WALK_SUMS * sizeof(double));
            hipLaunchKernelGGL(k_recip_walk, dim3((a.ng + WAVE - 1) / WAVE, a.chunks), dim3(WALK_WAVES * WAVE), lds, s, a);
        } else {
            int waves, gy;
            if constexpr (NW > 1) {
                waves = a.sets.split * a.sets.units;
                gy = a.sets.count;
            } else {
                // A chunk's tiles go side by side over blocks only where the
                // chunks alone leave CUs idle, since each block fills its own
                // table.
                waves = ks_waves(a.kr.tiles(), a.vpw, KS_MAXW, 3);
                const int sets = (a.kr.tiles() + waves * a.vpw - 1) / (waves * a.vpw) * a.kr.col_groups();
                gy = std::min(sets, std::max(1, 256 / a.chunks));
                gy = (sets + (sets + gy - 1) / gy - 1) / ((sets + gy - 1) / gy);   // no block with one set more
            }
            const size_t lds = ks_table_bytes<R>(a.kr, NW) * ks_tables<R>(a.kr, NW, a.per / KS_TILE);
            const dim3 g(a.chunks, gy), b(waves * WAVE);
            if (NW > 1 && a.kr.half()) hipLaunchKernelGGL((k_recip_sfac<R, NW, (NW > 1)>), g, b, lds, s, a);
            else hipLaunchKernelGGL((k_recip_sfac<R, NW, false>), g, b, lds, s, a);
        }
    }
    if (passes & RECIP_REDUCE) {
        // a share of the chunks for every dozen, as far as 16 waves hold all of a
        // row's sums per share: the loads of one wave follow each other, the
        // epilogue waits for all
        const int nn = std::min(a.nper, a.kr.n1), nv = NW == 0 ? 2 * nn * WALK_SUMS : NW * 4 * nn;
        const int vw = NW == 1 ? 1 : std::min(16, (nv + WAVE - 1) / WAVE);
        const int nq = std::max(1, std::min(16 / vw, (a.chunks + 11) / 12)), waves = std::max(4, vw * nq);
        const size_t lds = sizeof(double) * std::max(waves * std::max(WAVE, NW == 1 ? nv : 0), nv);
        hipLaunchKernelGGL((k_recip_reduce<R, NW>), recip_reduce_grid(a), dim3(waves * WAVE), lds, s, a);
    }
}

// Scratch of the reciprocal-space passes: the force pass's coefficients, the
// chunks' partials, per-atom phases.
struct RecipScratch { double* kf; double* part; double* e1; int chunks; };

static int ewald_recip_with(Ctx* c, int prec, int lustig, unsigned passes, const RecipScratch& sc);

int ewald_recip(Ctx* c, int prec, int lustig, unsigned passes) {
    return ewald_recip_with(c, prec, lustig, passes, RecipScratch{c->d_kf, c->d_sfac_part, c->d_e1, lustig ? SF_CHUNKS : c->sfac_chunks});
}

// ---- the allocation-free form's scratch -------------------------------------
// One static device array per GPU holds the reciprocal-space scratch of
// smd_ewald_compute_long_static.  In host code `scratch` is only a host-side
// stand-in: its device address, one per GPU, comes from hipGetSymbolAddress
// with that GPU current (static_scratch_init, called by smd_ctx_create) and is
// the only form ever passed to a kernel or a copy.
constexpr size_t STATIC_SCRATCH_DOUBLES = SMD_STATIC_SCRATCH_BYTES / sizeof(double);
static __device__ __align__(256) double scratch[STATIC_SCRATCH_DOUBLES];

constexpr int MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static double* g_scratch_ptr[MAX_DEVICES] = {};

int static_scratch_init(Ctx* c) {
    if (c->device < 0 || c->device >= MAX_DEVICES) return fail(c, SMD_EINVAL, "device %d out of range", c->device);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[c->device]) {
        void* ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) return hip_fail(c, e, "hipGetSymbolAddress(scratch)");
        g_scratch_ptr[c->device] = static_cast<double*>(ptr);
    }
    c->static_scratch = g_scratch_ptr[c->device];
    return SMD_OK;
}

static int ewald_recip_with(Ctx* c, int prec, int lustig, unsigned passes, const RecipScratch& sc) {
    if (!c->ewald_ready) return fail(c, SMD_ESTATE, "Ewald not set up");
    RecipArgs a;
    a.n = c->n;
    a.K = c->K;
    a.kr.nrows = c->n_krows;
    a.kr.nx1 = c->nmax[0] + 1;
    a.kr.ny1 = c->nmax[1] + 1;
    a.kr.n1 = c->nmax[2] + 1;
    a.kr.ts = prec == SMD_PREC_MIXED ? ks_stride<float>() : ks_stride<double>();
    a.kr.xy = c->d_kxy;
    a.ng = c->n_kruns;
    a.runs = c->d_kruns;
    a.rowk = c->d_rowk;
    const bool mixed = prec == SMD_PREC_MIXED;
    bool walk = false;
    if (lustig) {
        const LustigPlan p = lustig_plan(a.kr, c->n, c->K, c->n_kruns, sc.chunks, mixed);
        walk = p.walk;
        a.sets = p.sets;
        a.per = p.per;
    } else {   // whole tiles per chunk
        const int nt = (c->n + KS_TILE - 1) / KS_TILE;
        a.per = (nt + sc.chunks - 1) / sc.chunks * KS_TILE;
    }
    a.chunks = (c->n + a.per - 1) / a.per;
    a.vpw = a.chunks < 128 ? 1 : KS_VT;   // one tile per wave while blocks are few
    a.nper = a.kr.tiles() * KS_ROWS * a.kr.col_groups() <= c->red.cap ? 16 : a.kr.n1;
    for (int d = 0; d < 3; ++d) a.vk[d] = 2.0 * PI / c->box.L[d];
    a.pos = c->d_pos;
    a.q = c->d_q;
    a.mol = c->d_mol;
    a.com = c->d_com;
    a.expk = c->d_expk;
    a.part = sc.part;
    a.kf = sc.kf;
    a.e1 = reinterpret_cast<double2*>(sc.e1);
    a.am = reinterpret_cast<double4*>(sc.e1 + e1_am_offset(c->n));
    a.store = c->recip_store ? 1 : 0;
    a.force = c->recip_store ? c->d_frecip : c->d_force;
    a.red = c->red;
    a.alphaR4 = 1.0 / (4.0 * (c->ew.alpha * c->ew.alpha));
    const double volume = c->box.L[0] * c->box.L[1] * c->box.L[2];
    a.pi4V = 4.0 * PI * (1.0 / volume);
    a.pi8V = 2.0 * a.pi4V;
    for (unsigned pass : {(unsigned)RECIP_SFAC, (unsigned)RECIP_REDUCE}) {
        if (!(passes & pass)) continue;
        ProfScope ps(c, pass == RECIP_SFAC ? "recip_sfac" : "recip_reduce");
        if (mixed) {
            if (lustig) launch_recip_sums<float, KS_WEIGHTS>(c->stream, a, pass);
            else launch_recip_sums<float, 1>(c->stream, a, pass);
        } else {
            if (walk) launch_recip_sums<double, 0>(c->stream, a, pass);
            else if (lustig) launch_recip_sums<double, KS_WEIGHTS>(c->stream, a, pass);
            else launch_recip_sums<double, 1>(c->stream, a, pass);
        }
        SMD_HIP(c, hipGetLastError());
        if (pass == RECIP_REDUCE) {
            const dim3 g = recip_reduce_grid(a);
            const int rc = red_finish(c, RS_RECIP, (int)(g.x * g.y), lustig ? 16 : 12, c->d_terms + T_RC_E);
            if (rc) return rc;
        }
    }
    if (passes & RECIP_FORCE) {
        ProfScope ps(c, "recip_force");
        if (mixed) {
            if (lustig) launch_recip_force<float, false>(c->stream, a);
            else launch_recip_force<float, true>(c->stream, a);
        } else {
            if (lustig) launch_recip_force<double, false>(c->stream, a);
            else launch_recip_force<double, true>(c->stream, a);
        }
        SMD_HIP(c, hipGetLastError());
        if (!lustig) return red_finish(c, RS_RECIP_FF, (a.n + KS_TILE - 1) / KS_TILE, 1, c->d_terms + T_RC_FF);
    }
    return SMD_OK;
}

}  // namespace smd

using namespace smd;

extern "C" int smd_ewald_setup(smd_ctx* c, const smd_ewald_params* p, int32_t* n_kvec) {
    if (!c || !p) return SMD_EINVAL;
    int rc = ewald_setup(c, p);
    if (rc) return rc;
    if (n_kvec) *n_kvec = c->K;
    return SMD_OK;
}

static int fetch_forces_into(smd_ctx* c, double* f_accum) {
    std::vector<double> f(3 * (size_t)c->n);
    SMD_HIP(c, hipMemcpyAsync(f.data(), c->d_force, f.size() * sizeof(double), hipMemcpyDeviceToHost, c->stream));
    SMD_HIP(c, hipStreamSynchronize(c->stream));
    for (size_t k = 0; k < f.size(); ++k) f_accum[k] += f[k];
    return SMD_OK;
}

extern "C" int smd_ewald_compute(smd_ctx* c, int prec, double* f_accum, smd_ewald_out* out) {
    // EwaldForce::compute (src/forces/EwaldForce.cpp:128-176)
    if (!c || !out) return SMD_EINVAL;
    if (!c->ewald_ready) return fail(c, SMD_ESTATE, "Ewald not set up");
    if (!c->list_valid) return fail(c, SMD_ESTATE, "no pair list");
    if (f_accum) SMD_HIP(c, hipMemsetAsync(c->d_force, 0, sizeof(double) * 3 * c->n, c->stream));
    SMD_HIP(c, hipMemsetAsync(c->d_terms, 0, sizeof(double) * T_COUNT, c->stream));
    int rc = ewald_real(c, prec, 1);
    if (!rc) rc = ewald_intra(c, 1);
    if (!rc && c->ew.surface) rc = ewald_surface(c);
    if (rc) return rc;
    double t[T_COUNT];
    if ((rc = read_terms(c, t))) return rc;
    *out = smd_ewald_out{};
    out->real_energy = t[T_EW_E];
    out->real_deriv = t[T_EW_D1];
    out->real_deriv2 = t[T_EW_D2];
    out->self_energy = c->self_energy;
    out->charged_energy = c->charged_energy;
    out->intra_energy = -t[T_IN_E];
    out->intra_vir_correct = -t[T_IN_U];
    out->mol_deriv = t[T_IN_D1];
    out->mol_deriv2 = t[T_IN_D2];
    for (int k = 0; k < 9; ++k) out->virial[k] = t[T_EW_VIR + k];
    if (c->ew.surface) {
        // surfDipoleCorrect energy and derivatives (:854-864)
        const double volume = c->box.L[0] * c->box.L[1] * c->box.L[2];
        const double vr = 1.0 / volume;
        const double coeff = 2.0 * PI * vr / 3.0;
        const double* qr = t + T_SU_QR;
        const double* qR = t + T_SU_QRR;
        const double rr = qr[0] * qr[0] + qr[1] * qr[1] + qr[2] * qr[2];
        const double rR = qr[0] * qR[0] + qr[1] * qR[1] + qr[2] * qR[2];
        const double RR = qR[0] * qR[0] + qR[1] * qR[1] + qR[2] * qR[2];
        out->surf_energy = coeff * rr;
        if (c->ew.use_constraint) {
            out->surf_deriv = -coeff * vr * rr + 2.0 * coeff * vr * rR / 3.0;
            out->surf_deriv2 = 2.0 * coeff * vr * vr * rr - 16.0 * coeff * vr * vr * rR / 9.0 + 2.0 * coeff * vr * vr * RR / 9.0;
        } else {
            out->surf_deriv = -coeff * vr * rr / 3.0;
            out->surf_deriv2 = 4.0 * coeff * vr * vr * rr / 9.0;
        }
        for (int k = 0; k < 9; ++k) out->virial[k] += t[T_SU_VIR + k];
    }
    if (f_accum) return fetch_forces_into(c, f_accum);
    return SMD_OK;
}

static int recip_long_out(smd_ctx* c, smd_ewald_long_out* out);

extern "C" int smd_ewald_compute_long(smd_ctx* c, int prec, double* f_accum, smd_ewald_long_out* out) {
    // EwaldForce::compute_long (src/forces/EwaldForce.cpp:178-196)
    if (!c || !out) return SMD_EINVAL;
    if (!c->ewald_ready) return fail(c, SMD_ESTATE, "Ewald not set up");
    if (f_accum) SMD_HIP(c, hipMemsetAsync(c->d_force, 0, sizeof(double) * 3 * c->n, c->stream));
    SMD_HIP(c, hipMemsetAsync(c->d_terms, 0, sizeof(double) * T_COUNT, c->stream));
    int rc = ewald_recip(c, prec, 1);
    if (rc) return rc;
    if ((rc = recip_long_out(c, out))) return rc;
    if (f_accum) return fetch_forces_into(c, f_accum);
    return SMD_OK;
}

// Clears the term accumulators with a kernel rather than a memset node.
__global__ __launch_bounds__(256) void k_clear_terms(double* t, int n) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) t[i] = 0.0;
}

// The same passes with their scratch in the static array: no device
// allocation.  Every atom's phases and moments, the per-k coefficients and
// the (chunk, k) partials are written before they are read in each call, so
// nothing in the array needs clearing; the term accumulators (context state)
// are cleared by a fill kernel on the context stream.
extern "C" int smd_ewald_compute_long_static(smd_ctx* c, int prec, smd_ewald_long_out* out) {
    if (!c || !out) return SMD_EINVAL;
    if (!c->ewald_ready) return fail(c, SMD_ESTATE, "Ewald not set up");
    if (prec != SMD_PREC_FP64 && prec != SMD_PREC_MIXED) return fail(c, SMD_EINVAL, "bad precision %d", prec);
    if (!c->static_scratch) return fail(c, SMD_ESTATE, "static scratch not resolved for device %d", c->device);
    auto up = [](size_t v) { return (v + 31) / 32 * 32; };   // 256-byte segments
    // The documented room: 80 bytes per atom, 16 per k and 80 per (k, chunk),
    // with a chunk per 64 k-runs and CU but at least 32 atoms in each.  What
    // it admits leaves the passes, whose coefficients and mixed partials take
    // more, chunks enough.
    const int gt = (c->n_kruns + WAVE - 1) / WAVE;
    const int quota = std::max(1, 256 / gt);
    const int per = std::max(32, (c->n + quota - 1) / quota);
    const size_t need = up(((6 * (size_t)c->n + 3) & ~(size_t)3) + 4 * (size_t)c->n) + up(2 * (size_t)c->K) +
                        up((size_t)10 * c->K * ((c->n + per - 1) / per));
    const size_t n_e1 = up(e1_am_offset(c->n) + 4 * (size_t)c->n);
    KsRows kr{};
    kr.nrows = c->n_krows;
    kr.n1 = c->nmax[2] + 1;
    const size_t n_kf = up(kr.coef_entries());
    // as many chunks as the rest of the array holds
    const size_t rest = n_e1 + n_kf < STATIC_SCRATCH_DOUBLES ? STATIC_SCRATCH_DOUBLES - n_e1 - n_kf : 0;
    const size_t part = lustig_plan(kr, c->n, c->K, c->n_kruns, SF_CHUNKS, prec == SMD_PREC_MIXED).part;
    const int chunks = (int)std::min<size_t>(SF_CHUNKS, rest / part);
    if (need > STATIC_SCRATCH_DOUBLES || chunks < 1)
        return fail(c, SMD_ECAPACITY,
                    "static scratch holds %zu bytes; %d atoms and %d k-vectors need %zu (use smd_ewald_compute_long)",
                    (size_t)SMD_STATIC_SCRATCH_BYTES, c->n, c->K, need * sizeof(double));
    const RecipScratch sc{c->static_scratch + n_e1, c->static_scratch + n_e1 + n_kf, c->static_scratch, chunks};
    hipLaunchKernelGGL(k_clear_terms, dim3(1), dim3(256), 0, c->stream, c->d_terms, (int)T_COUNT);
    SMD_HIP(c, hipGetLastError());
    int rc = ewald_recip_with(c, prec, 1, RECIP_ALL, sc);
    if (rc) return rc;
    return recip_long_out(c, out);
}

// compute_long's outputs from the term accumulators (reads them back).
static int recip_long_out(smd_ctx* c, smd_ewald_long_out* out) {
    int rc;
    double t[T_COUNT];
    if ((rc = read_terms(c, t))) return rc;
    out->energy = t[T_RC_E];
    out->deriv = t[T_RC_D1];
    out->deriv2 = t[T_RC_D2];
    if (c->ew.use_constraint) {   // :671-676
        out->deriv += t[T_RC_FF];
        out->deriv2 += -6.0 * t[T_RC_FF] + t[T_RC_FFK2] - t[T_RC_D2UV1] + t[T_RC_D2URR];
    }
    for (int k = 0; k < 9; ++k) out->virial[k] = t[T_RC_VIR + k];
    return SMD_OK;
}
