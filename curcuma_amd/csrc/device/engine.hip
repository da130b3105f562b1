// GFN-FF energy + gradient on one MI355X (gfx950): FP64 path and mixed path,
// single molecules and batches of independent molecules.
//
// One evaluation is a fixed sequence of kernels on two streams (launch_eval):
//   second stream: the reduced EEQ matrix (k_eeq_reduced / k_eeq_reduced_batch),
//     for single molecules the solver's preconditioner (k_bjacobi_setup), for
//     batches the per-molecule factorisation (k_lstep_tiles, k_bstep_diag64,
//     k_bstep_tiles or the per-molecule forms); solvation (k_solv_*); of a
//     batch also the hydrogen bonds, behind the factorisation;
//   evaluation stream:
//   k_start             coordinates, flags, bounding boxes
//   k_cn / k_cn_mol     CN (6 Bohr), log cap, dlogdcn, D4 weights, EEQ rhs, CN neighbour lists
//   k_terms             bonded term lists (per-atom gradient slots), D4 half contraction, reduced rhs
//   k_hb_roles/k_hb_full  hydrogen bonds
//   k_slot_gather       per-atom sum of the slots (and of a molecule's hydrogen bonds)
//   -- join --
//   EEQ solve           k_eeq_pcg_one / _res / k_eeq_pcg or k_chol_* + k_trsv_* (single), k_bsolve_subst (batches)
//   k_charges           charges from the reduced solution, self energy, qtmp
//   k_pairs_sym         Coulomb + D4 dispersion + repulsion, each pair once (64 x 64 tiles)
//   k_pairs_sym_reduce  fixed-order sum of the tile partials (no atomics), corrections of the
//                       repulsion over the topological neighbourhood, dE/dCN totals
//   k_finish            CN chain rule + gradient assembly, fixed-order energy reductions
// Reference semantics: see oracle/gfnff_oracle.c (same formulas, same cut-offs).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <mutex>
#include <numeric>
#include <string>
#include <vector>

#include "engine.hpp"

namespace gfnff {

namespace {

#define HIP_OK(x)                                                   \
    do {                                                            \
        hipError_t e_ = (x);                                        \
        if (e_ != hipSuccess) {                                     \
            msg = std::string(#x) + ": " + hipGetErrorString(e_);   \
            return kErrDevice;                                      \
        }                                                           \
    } while (0)

constexpr int NB = 64;          // Cholesky block size
#define MFMA_F32_ROW_FROM_REG false  // FP32 16x16x4 result layout (see MfmaT)
constexpr int MAXNB_CN = 128;   // CN neighbour list capacity per atom
constexpr int TILE = 256;       // pair kernel tile / workgroup size

constexpr double KN = -7.5;
// CN count 0.5 (1 + erf(v)); for v <= -6, erf(v) rounds to -1 and the count
// is 0 (the branch skips erf for the many list members beyond the covalent
// distance; also the hydrogen-bond coordination count of X-H bonds)
__device__ inline double cn_count(double v) {
    double c = 0.0;
    if (v > -6.0) c = 0.5 * (1.0 + erf(v));
    return c;
}
constexpr double CNMAX = 4.4;
constexpr double SQRTPI_TRUNC = 1.77245385091;   // constant used by the reference's dCN
constexpr double TSQRT2PI = 0.797884560802866;
constexpr double TSQRT2PI_SELF = 0.797884560802865;

// FLAG_LU: the dense fallback has solved what FLAG_CHOL reports (never leaves an evaluation)
enum Flag { FLAG_CHOL = 1, FLAG_CNOVF = 2, FLAG_SOLVE = 4, FLAG_LU = 32 };
__host__ __device__ inline int final_flags(int f) { return f & FLAG_LU ? f & ~(FLAG_LU | FLAG_CHOL | FLAG_SOLVE) : f; }

// ---------------------------------------------------------------------------
// small helpers
// ---------------------------------------------------------------------------
__device__ inline double3 ld3(const double* x, int i) { return make_double3(x[3 * i], x[3 * i + 1], x[3 * i + 2]); }
__device__ inline double sq(double v) { return v * v; }
__device__ inline double cube(double v) { return v * v * v; }
__device__ inline double3 operator-(double3 a, double3 b) { return make_double3(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ inline double3 operator+(double3 a, double3 b) { return make_double3(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ inline double3 operator*(double s, double3 a) { return make_double3(s * a.x, s * a.y, s * a.z); }
__device__ inline double dot(double3 a, double3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ inline double3 cross(double3 a, double3 b) {
    return make_double3(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}
__device__ inline double nrm(double3 a) { return sqrt(dot(a, a)); }
__device__ inline void st3(double* s, int slot, double3 v) {
    s[3 * slot] = v.x;
    s[3 * slot + 1] = v.y;
    s[3 * slot + 2] = v.z;
}

// ---------------------------------------------------------------------------
// K1: CN, log cap, dlogdcn, D4 weights, EEQ right-hand side, neighbour list
// cn_calculator.cpp:367-428; gfnff_method.cpp:5880-5930; d4param_generator.cpp:1079-1213,1692-1768
// ---------------------------------------------------------------------------
// One wavefront per atom i (four atoms per workgroup share the LDS j tiles).
// Lanes test 64 partners j at a time; __ballot and a prefix popcount give the
// position of every hit, so each neighbour list is ascending in j with the
// strict d^2 < 36 compare of the reference's builder (cn_calculator.cpp:
// 367-428).  The raw CN is summed per lane and combined by a fixed butterfly.
__device__ void cn_atom_finish(int i, double raw, int cnt, const int* __restrict__ elem, const int* __restrict__ nref,
                               const double* __restrict__ refcn, const double* __restrict__ chi_base,
                               const double* __restrict__ cnf, double* __restrict__ cn, double* __restrict__ dlog,
                               double* __restrict__ gw, double* __restrict__ dgw, double* __restrict__ rhs,
                               int* __restrict__ nbn, int* __restrict__ flags);

// Head of an evaluation, one launch: the coordinates into the engine's buffer,
// the status flags and the arrival counter of the energy reduction (k_finish)
// cleared, and for a single molecule (bb != nullptr) the exact bounding boxes
// of the 256-atom tiles of the atom order (k_cn's partner tiles):
// bb[6 t] = (min x, min y, min z, max x, max y, max z).
__global__ __launch_bounds__(256) void k_start(int n, const double* __restrict__ xin, double* __restrict__ x,
                                               int* __restrict__ flags, int* __restrict__ arrived,
                                               double* __restrict__ bb) {
    __shared__ double red[6][256];
    const int t = blockIdx.x, tid = threadIdx.x, e = t * 256 + tid;
    if (e == 0) {
        flags[0] = 0;
        arrived[0] = 0;
    }
    if (e < 3 * n) x[e] = xin[e];
    if (!bb || t * 256 >= n) return;  // uniform over the workgroup
    const double3 p = ld3(xin, min(e, n - 1));
    red[0][tid] = p.x;
    red[1][tid] = p.y;
    red[2][tid] = p.z;
    red[3][tid] = p.x;
    red[4][tid] = p.y;
    red[5][tid] = p.z;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (tid < w) {
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                red[d][tid] = fmin(red[d][tid], red[d][tid + w]);
                red[3 + d][tid] = fmax(red[3 + d][tid], red[3 + d][tid + w]);
            }
        }
        __syncthreads();
    }
    if (tid < 6) bb[6 * t + tid] = red[tid][0];
}

__global__ __launch_bounds__(256) void k_cn(int n, const double* __restrict__ x, const double* __restrict__ rcov,
                                            const int* __restrict__ elem, const int* __restrict__ nref,
                                            const double* __restrict__ refcn, const double* __restrict__ chi_base,
                                            const double* __restrict__ cnf, double* __restrict__ cn,
                                            double* __restrict__ dlog, double* __restrict__ gw,
                                            double* __restrict__ dgw, double* __restrict__ rhs,
                                            int* __restrict__ nbn, int* __restrict__ nbl, int* __restrict__ flags,
                                            const int* __restrict__ mol_of, const int* __restrict__ mol_off,
                                            const double* __restrict__ tbox) {
    __shared__ double sx[256], sy[256], sz[256], sr[256];
    const int lane = threadIdx.x & 63;
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6);
    const bool act = i < n;
    double3 xi = act ? ld3(x, i) : make_double3(0, 0, 0);
    double ri = act ? rcov[i] : 0.0;
    double raw = 0.0;
    int cnt = 0;
    // partner range: all atoms, or in a batch the molecules of this block's atoms
    int jlo = 0, jhi = n, mlo = 0, mhi = n;
    if (mol_of) {
        const int first = blockIdx.x * 4, last = min(n, first + 4) - 1;
        jlo = mol_off[mol_of[first]];
        jhi = mol_off[mol_of[last] + 1];
        if (act) {
            mlo = mol_off[mol_of[i]];
            mhi = mol_off[mol_of[i] + 1];
        }
    }
    for (int t0 = jlo; t0 < jhi; t0 += 256) {
        // single molecule: skip a partner tile whose bounding box (tbox, the
        // 256-atom tiles of the atom order) is beyond the cut-off for all four
        // atoms; the margin covers the rounding of both distance tests
        bool near = true;
        if (!mol_of) {
            const double* bx = tbox + 6 * (t0 >> 8);
            const double ex = fmax(0.0, fmax(bx[0] - xi.x, xi.x - bx[3]));
            const double ey = fmax(0.0, fmax(bx[1] - xi.y, xi.y - bx[4]));
            const double ez = fmax(0.0, fmax(bx[2] - xi.z, xi.z - bx[5]));
            near = act && ex * ex + ey * ey + ez * ez <= 36.0 * (1.0 + 1e-9);
        }
        if (!__syncthreads_or(near)) continue;
        int jl = t0 + threadIdx.x;
        if (jl < jhi) {
            sx[threadIdx.x] = x[3 * jl];
            sy[threadIdx.x] = x[3 * jl + 1];
            sz[threadIdx.x] = x[3 * jl + 2];
            sr[threadIdx.x] = rcov[jl];
        }
        __syncthreads();
        const int m = min(256, jhi - t0);
        for (int s0 = 0; s0 < m; s0 += 64) {
            const int jj = s0 + lane, j = t0 + jj;
            bool hit = false;
            double contrib = 0.0;
            if (act && jj < m && j != i && j >= mlo && j < mhi) {
                double dx = xi.x - sx[jj], dy = xi.y - sy[jj], dz = xi.z - sz[jj];
                // unfused products and sums: the list membership test matches
                // the reference's ((dx*dx + dy*dy) + dz*dz) < 36 bit for bit
                double d2 = __dadd_rn(__dadd_rn(__dmul_rn(dx, dx), __dmul_rn(dy, dy)), __dmul_rn(dz, dz));
                if (d2 < 36.0) {
                    hit = true;
                    double r = sqrt(d2);
                    double rij = ri + sr[jj];
                    contrib = cn_count(KN * (r - rij) / rij);
                }
            }
            const unsigned long long mask = __ballot(hit);
            if (hit) {
                int pos = cnt + __popcll(mask & ((1ull << lane) - 1ull));
                if (pos < MAXNB_CN) nbl[(size_t)i * MAXNB_CN + pos] = j;
                raw += contrib;
            }
            cnt += __popcll(mask);
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) raw += __shfl_xor(raw, off);
    if (!act || lane != 0) return;
    cn_atom_finish(i, raw, cnt, elem, nref, refcn, chi_base, cnf, cn, dlog, gw, dgw, rhs, nbn, flags);
}

// Per-atom part of the CN kernels once the neighbour scan is done: list
// length, log-capped CN and its derivative, D4 weights, EEQ right-hand side.
__device__ void cn_atom_finish(int i, double raw, int cnt, const int* __restrict__ elem, const int* __restrict__ nref,
                               const double* __restrict__ refcn, const double* __restrict__ chi_base,
                               const double* __restrict__ cnf, double* __restrict__ cn, double* __restrict__ dlog,
                               double* __restrict__ gw, double* __restrict__ dgw, double* __restrict__ rhs,
                               int* __restrict__ nbn, int* __restrict__ flags) {
    if (cnt > MAXNB_CN) atomicOr(flags, FLAG_CNOVF);
    nbn[i] = min(cnt, MAXNB_CN);
    double c = log(1.0 + exp(CNMAX)) - log(1.0 + exp(CNMAX - raw));
    cn[i] = c;
    dlog[i] = exp(CNMAX) / (exp(CNMAX) + exp(raw));
    int e = elem[i], nr = nref[e];
    double ex[7], dex[7], norm = 0.0, dnorm = 0.0;
#pragma unroll
    for (int r = 0; r < 7; ++r) {
        ex[r] = 0.0;
        dex[r] = 0.0;
        if (r < nr) {
            double df = c - refcn[e * 7 + r];
            ex[r] = exp(-4.0 * df * df);
            dex[r] = -8.0 * df * ex[r];
            norm += ex[r];
            dnorm += dex[r];
        }
    }
#pragma unroll
    for (int r = 0; r < 7; ++r) {
        double g = 0.0, dg = 0.0;
        if (norm > 1e-10) {
            if (r < nr) {
                g = ex[r] / norm;
                dg = (dex[r] * norm - ex[r] * dnorm) / (norm * norm);
            }
        } else if (r == 0 && nr > 0) {
            g = 1.0;
        }
        gw[(size_t)i * 7 + r] = g;
        dgw[(size_t)i * 7 + r] = dg;
    }
    rhs[i] = chi_base[i] + cnf[i] * sqrt(c);
}

// CN for a batch of molecules of at most CNMOL_MAX atoms each: one
// workgroup per molecule stages the molecule's coordinates and radii once;
// wave w scans atoms w, w + 4, ... against every atom of the molecule with
// the ballot-ordered list construction of k_cn (ascending partners) and
// leaves the raw CN and list length in LDS; the per-atom epilogue (log cap,
// D4 weights, EEQ right-hand side) then runs one thread per atom.  The LDS
// arrays are sized at launch for the batch's largest molecule (cap atoms,
// 44 bytes each), so that workgroups of small-molecule batches share a CU
// many at a time and hide the latency of each wavefront's scan.
constexpr int CNMOL_MAX = 1024;
constexpr int CNMOL_LDS_BYTES = 5 * 8 + 4;  // per atom of the cap
__global__ __launch_bounds__(256, 6) void k_cn_mol(int cap, const int* __restrict__ mol_off, const double* __restrict__ x,
                                                const double* __restrict__ rcov, const int* __restrict__ elem,
                                                const int* __restrict__ nref, const double* __restrict__ refcn,
                                                const double* __restrict__ chi_base, const double* __restrict__ cnf,
                                                double* __restrict__ cn, double* __restrict__ dlog,
                                                double* __restrict__ gw, double* __restrict__ dgw,
                                                double* __restrict__ rhs, int* __restrict__ nbn,
                                                int* __restrict__ nbl, int* __restrict__ flags) {
    extern __shared__ double cnm_lds[];
    double *sx = cnm_lds, *sy = sx + cap, *sz = sy + cap, *sr = sz + cap, *sraw = sr + cap;
    int* scnt = (int*)(sraw + cap);
    const int m = blockIdx.x, a0 = mol_off[m], nm = mol_off[m + 1] - a0;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    for (int k = tid; k < nm; k += 256) {
        sx[k] = x[3 * (a0 + k)];
        sy[k] = x[3 * (a0 + k) + 1];
        sz[k] = x[3 * (a0 + k) + 2];
        sr[k] = rcov[a0 + k];
    }
    __syncthreads();
    for (int ii = w; ii < nm; ii += 4) {
        const int i = a0 + ii;
        const double xix = sx[ii], xiy = sy[ii], xiz = sz[ii], ri = sr[ii];
        double raw = 0.0;
        int cnt = 0;
        for (int s0 = 0; s0 < nm; s0 += 64) {
            const int jj = s0 + lane;
            bool hit = false;
            double contrib = 0.0;
            if (jj < nm && jj != ii) {
                const double dx = xix - sx[jj], dy = xiy - sy[jj], dz = xiz - sz[jj];
                // unfused products and sums, as in k_cn
                const double d2 = __dadd_rn(__dadd_rn(__dmul_rn(dx, dx), __dmul_rn(dy, dy)), __dmul_rn(dz, dz));
                if (d2 < 36.0) {
                    hit = true;
                    const double r = sqrt(d2);
                    const double rij = ri + sr[jj];
                    contrib = cn_count(KN * (r - rij) / rij);
                }
            }
            const unsigned long long mask = __ballot(hit);
            if (hit) {
                const int pos = cnt + __popcll(mask & ((1ull << lane) - 1ull));
                if (pos < MAXNB_CN) nbl[(size_t)i * MAXNB_CN + pos] = a0 + jj;
                raw += contrib;
            }
            cnt += __popcll(mask);
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) raw += __shfl_xor(raw, off);
        if (lane == 0) {  // scan results; the per-atom epilogue runs below, one thread per atom
            sraw[ii] = raw;
            scnt[ii] = cnt;
        }
    }
    __syncthreads();
    for (int k = tid; k < nm; k += 256)
        cn_atom_finish(a0 + k, sraw[k], scnt[k], elem, nref, refcn, chi_base, cnf, cn, dlog, gw, dgw, rhs, nbn, flags);
}

// ---------------------------------------------------------------------------
// K2: reduced EEQ matrix.  Per fragment f with atoms a_1 < ... < a_m, the
// charges are q = qp + N p with qp = Q_f/m and columns e_a - e_last, so
//   Ared(a,b) = A(ia,ib) - A(ia,lb) - A(la,ib) + A(la,lb)
// with A the Coulomb matrix of eeq_solver.cpp:3571-3650.  Lower triangle of
// the padded (np x np) matrix; the padding is the identity.
// ---------------------------------------------------------------------------
// 1/sqrt(v) in FP64: the hardware estimate refined by two Newton steps
// (within about one ulp; each step doubles the correct bits)
__device__ inline double rsqrt_nr2(double v) {
    double y = __builtin_amdgcn_rsq(v);
    const double h = 0.5 * v;
    y = y * fma(-h * y, y, 1.5);
    y = y * fma(-h * y, y, 1.5);
    return y;
}

// 1/sqrt(v) and 1/v from the hardware estimate y (relative error e, about
// 2^-23) by one step of third order, which leaves e^3: with h = 1 - v y^2,
// 1/sqrt(v) = y (1 + h / 2 + 3 h^2 / 8 + ..), and with h = 1 - v y,
// 1/v = y (1 + h + h^2 + ..).  Five and three operations behind the estimate,
// against about 14 of a division and 20 of a square root.  Within about one
// unit in the last place; v has to be finite, normal and, with its reciprocal,
// in range: 0 and infinity give NaN.
__device__ inline double rsqrt_c(double v) {
    const double y = __builtin_amdgcn_rsq(v);
    const double h = fma(-v * y, y, 1.0);
    return fma(y * h, fma(h, 0.375, 0.5), y);
}
__device__ inline double rcp_c(double v) {
    const double y = __builtin_amdgcn_rcp(v);
    const double h = fma(-v, y, 1.0);
    return fma(y, fma(h, h, h), y);
}

// A(i, j) = erf(g r) / r with g = 1 / sqrt(alp_i + alp_j), evaluated as
// erf(g r2 / r) / r from one reciprocal square root of r2 (no divide or
// square root sequence on the dependency chain).  For g r >= 6, erfc(g r) <
// 2.2e-17 lies below half an ulp of 1 and erf(g r) is 1: the branch is
// uniform over a wavefront of far-apart atoms and skips the erf evaluation.
__device__ inline double eeq_a_r2(double r2, double ai, double aj) {
    const double rinv = rsqrt_nr2(r2);
    const double g = rsqrt_nr2(ai + aj);
    const double v = g * (r2 * rinv);
    double ef = 1.0;
    if (v < 6.0) ef = erf(v);
    return ef * rinv;
}

// erf(v) and exp(-v^2) for v >= 0 (screened Coulomb pair term and its
// derivative).  From v = 9 (FP64) or v = 5 (FP32) on, erf(v) rounds to 1 and
// the derivative's (2 / sqrt(pi)) v exp(-v^2) lies below the type's
// resolution relative to erf(v), so both are skipped.
__device__ inline void erf_exp(double v, double& ef, double& eg) {
    ef = 1.0;
    eg = 0.0;
    if (v < 9.0) {
        ef = erf(v);
        eg = exp(-v * v);
    }
}
__device__ inline void erf_exp(float v, float& ef, float& eg) {
    ef = 1.0f;
    eg = 0.0f;
    if (v < 5.0f) {
        ef = erff(v);
        eg = __expf(-v * v);
    }
}

__device__ inline double eeq_a(int i, int j, const double* __restrict__ x, const double* __restrict__ alp,
                               const double* __restrict__ diag) {
    if (i == j) return diag[i];
    double3 d = ld3(x, i) - ld3(x, j);
    return eeq_a_r2(dot(d, d), alp[i], alp[j]);
}

__global__ __launch_bounds__(256) void k_eeq_diag(int n, const double* __restrict__ gam,
                                                  const double* __restrict__ alp, double* __restrict__ diag) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) diag[i] = gam[i] + TSQRT2PI / sqrt(alp[i]);
}

// Reduced variables of one fragment are consecutive and share the last atom
// la, so a 64-block of variables touches few distinct last atoms (32 for
// water, 1 for one large molecule).  Per tile, the A entries that involve a
// last atom, A(ia, lb), A(la, ib) and A(la, lb), are evaluated once per
// distinct last atom into LDS (ul: the block's distinct last atoms, lidx: a
// variable's index among them), and every element then needs one fresh
// A(ia, ib).  The sum is formed in the same order as the direct form, so R is
// bit-identical; tiles with more than RED_UMAX distinct last atoms use the
// direct four-term form.
constexpr int RED_UMAX = 32;
// eeq_a for two distinct atoms from staged positions and alphas (the same
// operations as eeq_a, so the same bits)
__device__ inline double eeq_a_v(double3 pi, double ai, double3 pj, double aj) {
    double3 d = pi - pj;
    return eeq_a_r2(dot(d, d), ai, aj);
}
struct RedSm {
    union {
        struct {
            double Aiu[NB][RED_UMAX + 1], Aui[RED_UMAX][NB + 1], Auu[RED_UMAX][RED_UMAX + 1];
        } c;
        double Tl[NB][NB + 1];  // the transposed tile, after the caches are no longer read
    };
    double3 rp[NB], cp[NB], urp[RED_UMAX], ucp[RED_UMAX];
    double ra_[NB], ca_[NB], ura[RED_UMAX], uca[RED_UMAX];
    int sia[NB], sib[NB], slr[NB], slc[NB], sur[RED_UMAX], suc[RED_UMAX];
};
constexpr int RED_T = 512;  // threads per tile of k_eeq_reduced
__global__ __launch_bounds__(RED_T) void k_eeq_reduced(int nr, int np, const int* __restrict__ ra,
                                                     const int* __restrict__ rl, const int* __restrict__ lidx,
                                                     const int* __restrict__ ul, const int* __restrict__ nul,
                                                     const double* __restrict__ x, const double* __restrict__ alp,
                                                     const double* __restrict__ diag, double* __restrict__ A,
                                                     int full) {
    // one 64x64 lower tile per workgroup of RED_T threads; grid enumerates
    // tiles (bi >= bj).  full == 0: lower triangle of the row-major np x np
    // matrix (Cholesky).  full == 1: also the mirrored upper tile.  full == 2:
    // packed symmetric storage for the iterative solver, tile t at A + t 64^2
    // (row-major), diagonal tiles completed from their lower triangle
    __shared__ RedSm sm;
    int t = blockIdx.x;
    int bi = (int)((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
    while ((bi + 1) * (bi + 2) / 2 <= t) ++bi;
    while (bi * (bi + 1) / 2 > t) --bi;
    int bj = t - bi * (bi + 1) / 2;
    const int tid = threadIdx.x;
    const int nur = nul[bi], nuc = nul[bj];
    const bool ded = nur <= RED_UMAX && nuc <= RED_UMAX;
    if (tid < NB) {
        const int r = bi * NB + tid, c = bj * NB + tid;
        const int ia = (r < nr) ? ra[r] : -1, ib = (c < nr) ? ra[c] : -1;
        sm.sia[tid] = ia;
        sm.slr[tid] = (r < nr) ? lidx[r] : 0;
        sm.sib[tid] = ib;
        sm.slc[tid] = (c < nr) ? lidx[c] : 0;
        sm.rp[tid] = ld3(x, max(ia, 0));
        sm.ra_[tid] = alp[max(ia, 0)];
        sm.cp[tid] = ld3(x, max(ib, 0));
        sm.ca_[tid] = alp[max(ib, 0)];
    } else if (ded && tid < NB + RED_UMAX) {
        const int u = tid - NB;
        if (u < nur) {
            const int a = ul[bi * NB + u];
            sm.sur[u] = a;
            sm.urp[u] = ld3(x, a);
            sm.ura[u] = alp[a];
        }
        if (u < nuc) {
            const int a = ul[bj * NB + u];
            sm.suc[u] = a;
            sm.ucp[u] = ld3(x, a);
            sm.uca[u] = alp[a];
        }
    }
    __syncthreads();
    if (ded) {
        for (int e = tid; e < NB * nuc; e += RED_T) {
            const int r = e / nuc, u = e - r * nuc;
            sm.c.Aiu[r][u] = (sm.sia[r] >= 0) ? eeq_a_v(sm.rp[r], sm.ra_[r], sm.ucp[u], sm.uca[u]) : 0.0;
        }
        for (int e = tid; e < nur * NB; e += RED_T) {
            const int u = e / NB, c = e - u * NB;
            sm.c.Aui[u][c] = (sm.sib[c] >= 0) ? eeq_a_v(sm.urp[u], sm.ura[u], sm.cp[c], sm.ca_[c]) : 0.0;
        }
        for (int e = tid; e < nur * nuc; e += RED_T) {
            const int u = e / nuc, w = e - u * nuc;
            sm.c.Auu[u][w] = (sm.sur[u] == sm.suc[w]) ? diag[sm.sur[u]]
                                                      : eeq_a_v(sm.urp[u], sm.ura[u], sm.ucp[w], sm.uca[w]);
        }
        __syncthreads();
    }
    // thread tid owns column cc = tid % 64 of rows rr = tid / 64 + (RED_T / 64) u
    constexpr int PER = NB * NB / RED_T, RS = RED_T / 64;
    const int cc = tid & 63, c = bj * NB + cc;
    double vals[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int rr = (tid >> 6) + RS * u, r = bi * NB + rr;
        double v = 0.0;
        if (c <= r) {
            if (r >= nr || c >= nr) {
                v = (r == c) ? 1.0 : 0.0;
            } else if (ded) {
                const int ia = sm.sia[rr], ib = sm.sib[cc];
                const double a1 = (ia == ib) ? diag[ia] : eeq_a_v(sm.rp[rr], sm.ra_[rr], sm.cp[cc], sm.ca_[cc]);
                v = a1 - sm.c.Aiu[rr][sm.slc[cc]] - sm.c.Aui[sm.slr[rr]][cc] + sm.c.Auu[sm.slr[rr]][sm.slc[cc]];
            } else {
                int ia = ra[r], la = rl[r], ib = ra[c], lb = rl[c];
                v = eeq_a(ia, ib, x, alp, diag) - eeq_a(ia, lb, x, alp, diag) - eeq_a(la, ib, x, alp, diag) +
                    eeq_a(la, lb, x, alp, diag);
            }
            if (full == 2)
                A[(size_t)t * NB * NB + rr * NB + cc] = v;
            else
                A[(size_t)r * np + c] = v;
        }
        vals[u] = v;
    }
    if (!full || (full == 2 && bi != bj)) return;
    __syncthreads();  // the caches are no longer read: Tl reuses their memory
#pragma unroll
    for (int u = 0; u < PER; ++u) sm.Tl[(tid >> 6) + RS * u][cc] = vals[u];
    __syncthreads();
    // upper counterpart: A(bj*64 + i, bi*64 + j) = T(j, i), row-contiguous stores
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int i = (tid >> 6) + RS * u, j = cc;
        if (bi == bj && j <= i) continue;
        if (full == 2)
            A[(size_t)t * NB * NB + i * NB + j] = sm.Tl[j][i];
        else
            A[(size_t)(bj * NB + i) * np + bi * NB + j] = sm.Tl[j][i];
    }
}

// reduced right-hand side: b(a) = (x - A qp)(ia) - (x - A qp)(la)
__global__ __launch_bounds__(256) void k_eeq_rhs_qp(int n, const double* __restrict__ x,
                                                    const double* __restrict__ alp, const double* __restrict__ diag,
                                                    const double* __restrict__ qp, const double* __restrict__ rhs,
                                                    double* __restrict__ r, const int* __restrict__ mol_of,
                                                    const int* __restrict__ mol_off) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double s = 0.0;
    const int j0 = mol_of ? mol_off[mol_of[i]] : 0, j1 = mol_of ? mol_off[mol_of[i] + 1] : n;
    for (int j = j0; j < j1; ++j)
        if (qp[j] != 0.0) s += eeq_a(i, j, x, alp, diag) * qp[j];
    r[i] = rhs[i] - s;
}

__device__ __forceinline__ void rhs_reduce_entry(int a, int nr, int np, const int* __restrict__ ra,
                                                 const int* __restrict__ rl, const double* __restrict__ r,
                                                 double* __restrict__ b) {
    if (a >= np) return;
    b[a] = (a < nr && ra[a] >= 0) ? r[ra[a]] - r[rl[a]] : 0.0;  // ra < 0: padding of a batched block
}

// ---------------------------------------------------------------------------
// K3: blocked Cholesky, right-looking, lower, row-major with leading dim np.
// ---------------------------------------------------------------------------
// 1 / sqrt(d) from the hardware estimate refined by Newton steps
// (v_rsq_f64 ~23 bits: two steps reach double precision; f32: one step)
__device__ __forceinline__ double rsqrt_nr(double d) {
    double y = __builtin_amdgcn_rsq(d);
    y = y * (1.5 - 0.5 * d * y * y);
    return y * (1.5 - 0.5 * d * y * y);
}
__device__ __forceinline__ float rsqrt_nr(float d) {
    const float y = __builtin_amdgcn_rsqf(d);
    return y * (1.5f - 0.5f * d * y * y);
}

// Factorisation L L^T of one NB x NB diagonal block and the inverse of L by
// one workgroup of 256 threads, in steps of four columns, with the working
// matrix resident in LDS.  Thread (t, q) = (tid / 4, tid % 4) owns the
// entries (t, 4u + q).  Step b (columns k = 4b .. 4b + 3):
//  1. every thread reads the 4 x 4 pivot block and factors it redundantly
//     (four reciprocal square roots), reads its row's four entries and solves
//     them against the pivot factor: L(t, k .. k + 3);
//  2. the rows below the block store their L(t, k + q) (only their own quad
//     read those entries); barrier; the pivot rows store theirs;
//  3. every thread updates its entries A(t, j) -= sum_m L(t, k + m) L(j, k + m),
//     k + 3 < j <= t, reading the published columns; barrier.
// Two barriers per four columns (32 for the block), a rolled step loop (no
// register arrays, compact code).  The inverse X = L^{-1} is formed four
// rows at a time: thread (c, q) keeps X(4u + q, c) in registers; for rows
// 4b .. 4b + 3 the four partial sums L(r, :4b) X(:4b, c) are taken together
// (independent chains), combined over the quad by shuffles, and the 4 x 4
// lower-triangular system with the pivot factor is solved (no barrier).
// The block routine operates on caller-provided LDS so that one workgroup can
// also factor a whole small matrix (batched path); `col` is not used.
template <typename T>
__device__ __forceinline__ void chol_diag_block(int np, int k0, T* __restrict__ A, T* __restrict__ Linv, int* __restrict__ flags,
                                T (*sL)[NB + 1], T (*col)[NB], T* rdiag, bool write_L = true) {
    const int tid = threadIdx.x;
    const int t = tid >> 2, q = tid & 3, qb = tid & ~3 & 63;  // qb: lane of the quad's q = 0
    _Pragma("unroll") for (int u_ = 0, e = tid; u_ < NB * NB / 256; ++u_, e += 256) sL[e / NB][e % NB] = A[(size_t)(k0 + e / NB) * np + k0 + e % NB];
    __syncthreads();
    // the working matrix stays in LDS: thread (t, q) owns the entries (t, 4u + q)
    int bad = 0;
#pragma unroll 1
    for (int b = 0; b < NB / 4; ++b) {
        const int k = 4 * b;
        // pivot factor (lower 4 x 4), redundantly in every thread
        T p[4][4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int jj = 0; jj <= i; ++jj) p[i][jj] = sL[k + i][k + jj];
        T l[4][4] = {}, il[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int jj = 0; jj < i; ++jj) {
                T s = p[i][jj];
#pragma unroll
                for (int m = 0; m < jj; ++m) s -= l[i][m] * l[jj][m];
                l[i][jj] = s * il[jj];
            }
            T d = p[i][i];
#pragma unroll
            for (int m = 0; m < i; ++m) d -= l[i][m] * l[i][m];
            if (!(d > T(0))) {
                bad = 1;
                d = T(1);
            }
            il[i] = rsqrt_nr(d);
            l[i][i] = d * il[i];
        }
        // this row's L(t, k .. k + 3): solved against the pivot factor below the block,
        // the pivot factor's row inside it
        T y[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            T sv = sL[t][k + m];
#pragma unroll
            for (int jj = 0; jj < m; ++jj) sv -= l[m][jj] * y[jj];
            y[m] = sv * il[m];
        }
        const bool piv_row = t >= k && t < k + 4;
        if (piv_row) {
            const int i = t - k;  // static register indices: select among the pivot factor's rows
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const T lm = (i == 0) ? l[0][m] : (i == 1) ? l[1][m] : (i == 2) ? l[2][m] : l[3][m];
                y[m] = (m <= i) ? lm : T(0);
            }
        }
        // rows below the pivot block publish now (only their own quad read these entries);
        // the pivot rows after the barrier, once every thread has read the pivot block
        if (t >= k + 4) sL[t][k + q] = y[q];
        __syncthreads();
        if (piv_row) sL[t][k + q] = y[q];
        // A(t, j) -= sum_m L(t, k + m) L(j, k + m) for this thread's columns j > k + 3
        if (t >= k + 4) {
            for (int j = k + 4 + q; j <= t; j += 4)
                sL[t][j] -= y[0] * sL[j][k] + y[1] * sL[j][k + 1] + y[2] * sL[j][k + 2] + y[3] * sL[j][k + 3];
        }
        __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < NB / 4; ++u)
        if (4 * u + q > t) sL[t][4 * u + q] = T(0);  // the factor's upper triangle
    __syncthreads();
    if (q == 0) rdiag[t] = T(1) / sL[t][t];
    if (write_L) {
        _Pragma("unroll") for (int u_ = 0, e = tid; u_ < NB * NB / 256; ++u_, e += 256) {
            int r = e / NB, c = e % NB;
            if (c <= r) A[(size_t)(k0 + r) * np + k0 + c] = sL[r][c];
        }
    }
    __syncthreads();
    const int c = t;
    T xr[NB / 4];
#pragma unroll
    for (int u = 0; u < NB / 4; ++u) xr[u] = T(0);
#pragma unroll
    for (int b = 0; b < NB / 4; ++b) {
        const int r = 4 * b;
        T part[4] = {T(0), T(0), T(0), T(0)};
#pragma unroll
        for (int u = 0; u < b; ++u)
#pragma unroll
            for (int m = 0; m < 4; ++m) part[m] += sL[r + m][4 * u + q] * xr[u];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            part[m] += __shfl_xor(part[m], 1);
            part[m] += __shfl_xor(part[m], 2);
        }
        T x[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            T s = ((r + m == c) ? T(1) : T(0)) - part[m];
#pragma unroll
            for (int jj = 0; jj < m; ++jj) s -= sL[r + m][r + jj] * x[jj];
            x[m] = s * rdiag[r + m];
        }
        xr[b] = x[q];
        __builtin_amdgcn_sched_barrier(0);
    }
    T* Li = Linv + (size_t)(k0 / NB) * NB * NB;
#pragma unroll
    for (int u = 0; u < NB / 4; ++u) Li[(4 * u + q) * NB + c] = xr[u];
    if (bad && tid == 0) atomicOr(flags, FLAG_CHOL);
}

template <typename T>
__global__ __launch_bounds__(256, 3) void k_chol_diag(int np, int k0, T* __restrict__ A, T* __restrict__ Linv,
                                                   int* __restrict__ flags) {
    __shared__ T sL[NB][NB + 1];
    __shared__ T col[2][NB];
    __shared__ T rdiag[NB];
    chol_diag_block<T>(np, k0, A, Linv, flags, sL, col, rdiag);
}

// panel: rows below the diagonal block, L(i, k-block) = A(i, k-block) * Linv^T
// panel tile: rows r0 .. r0 + 63 of the column block k0, L = A Linv_k^T
template <typename T>
__device__ __forceinline__ void chol_panel_tile(int np, int k0, int r0, T* __restrict__ A, const T* __restrict__ Linv,
                                T (*S)[NB + 1], T (*W)[NB + 1]) {
    int tid = threadIdx.x;
    const T* Li = Linv + (size_t)(k0 / NB) * NB * NB;
    _Pragma("unroll") for (int u_ = 0, e = tid; u_ < NB * NB / 256; ++u_, e += 256) {
        int r = e / NB, c = e % NB;
        S[r][c] = A[(size_t)(r0 + r) * np + k0 + c];
        W[r][c] = Li[e];
    }
    __syncthreads();
    // out(r, c) = sum_p S(r, p) * W(c, p), p <= c
    int tr = tid / 16, tc = tid % 16;
    T acc[4][4] = {};
    for (int p = 0; p < NB; ++p) {
        T a[4], b[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            a[u] = S[tr * 4 + u][p];
            b[u] = W[tc * 4 + u][p];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[u][v] += a[u] * b[v];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) A[(size_t)(r0 + tr * 4 + u) * np + k0 + tc * 4 + v] = acc[u][v];
}

template <typename T>
__global__ __launch_bounds__(256) void k_chol_panel(int np, int k0, T* __restrict__ A, const T* __restrict__ Linv) {
    __shared__ T S[NB][NB + 1];
    __shared__ T W[NB][NB + 1];
    chol_panel_tile<T>(np, k0, k0 + NB + blockIdx.x * NB, A, Linv, S, W);
}

// Update of a set of lower 64 x 64 tiles by a block of factored columns:
//   A(bi, bj) -= sum_{c in [kc0, kc0 + kw)} L(bi, c) L(bj, c)^T
// over the trapezoid of tiles with column blocks bj in [bj0, bj0 + w) and rows
// bi in [bj, nbk).  Tiles are numbered row by row (the first w rows form a
// triangle, every later row holds w tiles) and handed out XCD-contiguously:
// workgroups are dispatched round-robin over the 8 XCDs, so consecutive tile
// numbers (same block row, same L panel rows) are given to workgroups of one
// XCD and share its L2.  The rank kw is streamed through LDS in 64-column
// chunks.  FP64 MFMA (v_mfma_f64_16x16x4f64): each of the 4 wavefronts owns a
// 32x32 quarter of the tile as 2x2 blocks of 16x16.  Operand layout per lane:
// A(i = lane%16, k = lane/16), B(k = lane/16, j = lane%16); result element v
// of a block sits at (row 4*v + lane/16, column lane%16) (measured on gfx950).
typedef double dbl4 __attribute__((ext_vector_type(4)));
typedef double dbl2 __attribute__((ext_vector_type(2)));
typedef float flt4 __attribute__((ext_vector_type(4)));

// Per-type 16x16x4 MFMA and its result layout: element v of a lane is at row
// 4*v + lane/16 (kRowFromReg) or 4*(lane/16) + v, column lane%16.
template <typename T>
struct MfmaT;
template <>
struct MfmaT<double> {
    typedef dbl4 V;
    static constexpr bool kRowFromReg = true;
    static __device__ __forceinline__ V op(double a, double b, V c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
};
template <>
struct MfmaT<float> {
    typedef flt4 V;
    static constexpr bool kRowFromReg = MFMA_F32_ROW_FROM_REG;
    static __device__ __forceinline__ V op(float a, float b, V c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
};

__device__ __forceinline__ double readlane_d(double v, int l) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), l);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// Cholesky factor and inverse factor of one 64 x 64 SPD block by a single
// wavefront, in FP64 MFMA tiles.  With U = L^T the 16 x 16 tiles of
// A = U^T U stay in the accumulator layout (lane (li, lk) holds elements
// (4 v + lk, li), v < 4), in which a tile X read as the A operand of
// v_mfma_f64_16x16x4f64 is X^T and read as the B operand is X: every product
// of the algorithm, U_ki^T U_kj, U_kk^-T A_kj, U_kj^T V_ki and W_jj^T S
// (V = L^-1, W_jj = U_jj^-1), has the form X^T Y and needs no data movement.
// Only the 16 x 16 diagonal tiles are worked on element by element: lane li
// takes column li (through LDS), pivots and rows are broadcast by readlane.
// The four-columns-a-step form (chol_diag_block, a workgroup of 256 with two
// barriers a step) was bound by that barrier chain, 27 us a block and 250 us
// for 4096 of them at three workgroups per compute unit; this one has no
// barrier, so the wavefronts of a SIMD fill each other's waits: 30 -> 16 us a
// block alone, evaluation 166 -> 157 us (122 atoms), 4096 molecules 6.49 -> 6.16
// ms mixed and 7.51 -> 7.13 ms FP64.
// A: lower triangle, row-major, leading dimension ld; L is written back when
// write_L; Linv: 64 x 64 row-major, zero above the diagonal.  buf: 16 x 17
// doubles of LDS of the wavefront.  Returns whether every pivot was positive.
__device__ __forceinline__ void xty(const dbl4& x, const dbl4& y, dbl4& c) {  // c += X^T Y
#pragma unroll
    for (int v = 0; v < 4; ++v) c = MfmaT<double>::op(x[v], y[v], c);
}
// W = U^-1 of an upper 16 x 16 factor D = U^T U: on return d holds U and w W,
// vt V = W^T, all in accumulator layout
__device__ __forceinline__ bool chol16(dbl4& d, dbl4& w, dbl4& vt, double* buf) {
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    constexpr int S = 17;
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int v = 0; v < 4; ++v) buf[(4 * v + lk) * S + li] = d[v];
    __builtin_amdgcn_wave_barrier();
    double a[16], iv = 0.0;
#pragma unroll
    for (int r = 0; r < 16; ++r) a[r] = buf[r * S + li];
    __builtin_amdgcn_wave_barrier();
    bool ok = true;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        double piv = readlane_d(a[k], k);
        if (!(piv > 0.0)) {
            ok = false;
            piv = 1.0;
        }
        const double inv = rsqrt_nr(piv);
        if (li == k) iv = inv;
        a[k] = li >= k ? a[k] * inv : 0.0;  // U(k, li)
#pragma unroll
        for (int r = k + 1; r < 16; ++r) a[r] -= readlane_d(a[k], r) * a[k];
    }
    double x[16];  // column li of W
#pragma unroll
    for (int r = 15; r >= 0; --r) {
        double s = li == r ? 1.0 : 0.0;
#pragma unroll
        for (int m = r + 1; m < 16; ++m) s -= readlane_d(a[r], m) * x[m];
        x[r] = s * readlane_d(iv, r);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        d[v] = lk == 0 ? a[4 * v] : lk == 1 ? a[4 * v + 1] : lk == 2 ? a[4 * v + 2] : a[4 * v + 3];
        w[v] = lk == 0 ? x[4 * v] : lk == 1 ? x[4 * v + 1] : lk == 2 ? x[4 * v + 2] : x[4 * v + 3];
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) buf[(4 * v + lk) * S + li] = w[v];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int v = 0; v < 4; ++v) vt[v] = buf[li * S + 4 * v + lk];
    __builtin_amdgcn_wave_barrier();
    return ok;
}
__device__ __forceinline__ bool chol64_wave(double* A, int ld, double* Linv, bool write_L, double* buf) {
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    dbl4 U[4][4], W[4], V[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = i; j < 4; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = 16 * i + 4 * v + lk, c = 16 * j + li;
                U[i][j][v] = A[(size_t)max(r, c) * ld + min(r, c)];
            }
    bool ok = true;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        dbl4 vt;
        ok = chol16(U[k][k], W[k], vt, buf) && ok;
        V[k] = vt;
#pragma unroll
        for (int j = k + 1; j < 4; ++j) {
            dbl4 t = {0.0, 0.0, 0.0, 0.0};
            xty(W[k], U[k][j], t);
            U[k][j] = t;
        }
#pragma unroll
        for (int i = k + 1; i < 4; ++i) {
            const dbl4 m = {-U[k][i][0], -U[k][i][1], -U[k][i][2], -U[k][i][3]};
#pragma unroll
            for (int j = i; j < 4; ++j) xty(m, U[k][j], U[i][j]);
        }
    }
    if (write_L) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = i; j < 4; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int r = 16 * i + 4 * v + lk, c = 16 * j + li;
                    if (r <= c) A[(size_t)c * ld + r] = U[i][j][v];
                }
    }
    // V = L^-1 by block columns: V_ji = -W_jj^T sum_k U_kj^T V_ki
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        dbl4 col[4];
        col[i] = V[i];
#pragma unroll
        for (int j = i + 1; j < 4; ++j) {
            dbl4 sum = {0.0, 0.0, 0.0, 0.0}, t = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int k = i; k < j; ++k) xty(U[k][j], col[k], sum);
            const dbl4 m = {-sum[0], -sum[1], -sum[2], -sum[3]};
            xty(W[j], m, t);
            col[j] = t;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) Linv[(16 * j + 4 * v + lk) * NB + 16 * i + li] = j < i ? 0.0 : col[j][v];
    }
    return ok;
}

__device__ inline int xcd_tile(int b, int nb) {
    const int x = b & 7, l = b >> 3, per = nb >> 3, rem = nb & 7;
    return x * per + min(x, rem) + l;
}

// A(ri.., rj..) -= sum_{c in [kc0, kc0 + kw)} L(ri.., c) L(rj.., c)^T for one
// 64 x 64 tile (lower triangle only when ri == rj), FP64/FP32 MFMA
template <typename T>
__device__ __forceinline__ void chol_update_tile(int np, int ri, int rj, int kc0, int kw, T* __restrict__ A, T (*P)[NB + 1],
                                 T (*Q)[NB + 1]) {
    using M = MfmaT<T>;
    const int bi = ri, bj = rj;  // only compared for equality (diagonal tile)
    const int tid = threadIdx.x;
    const int wave = tid / 64, lane = tid % 64;
    const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
    const int li = lane % 16, lk = lane / 16;
    typename M::V acc[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[x][y] = typename M::V{0, 0, 0, 0};
    // chunk kc of both panels: element u of this thread is row tid/64 + 4u,
    // column tid%64; the next chunk is fetched into registers while the
    // current one feeds the MFMAs
    T pr[NB * NB / 256], qr[NB * NB / 256];
    auto fetch = [&](int kc) {
#pragma unroll
        for (int u = 0; u < NB * NB / 256; ++u) {
            const int r = (tid >> 6) + 4 * u, c = tid & 63;
            pr[u] = A[(size_t)(ri + r) * np + kc + c];
            qr[u] = A[(size_t)(rj + r) * np + kc + c];
        }
    };
    fetch(kc0);
    for (int kc = kc0; kc < kc0 + kw; kc += NB) {
        __syncthreads();
#pragma unroll
        for (int u = 0; u < NB * NB / 256; ++u) {
            const int r = (tid >> 6) + 4 * u, c = tid & 63;
            P[r][c] = pr[u];
            Q[r][c] = qr[u];
        }
        __syncthreads();
        if (kc + NB < kc0 + kw) fetch(kc + NB);
#pragma unroll 4
        for (int k = 0; k < NB; k += 4) {
            const T fa0 = P[wr + li][k + lk], fa1 = P[wr + 16 + li][k + lk];
            const T fb0 = Q[wc + li][k + lk], fb1 = Q[wc + 16 + li][k + lk];
            acc[0][0] = M::op(fa0, fb0, acc[0][0]);
            acc[0][1] = M::op(fa0, fb1, acc[0][1]);
            acc[1][0] = M::op(fa1, fb0, acc[1][0]);
            acc[1][1] = M::op(fa1, fb1, acc[1][1]);
        }
    }
    // off-diagonal tiles: all 16 read-modify-writes issued unconditionally;
    // diagonal tiles keep the lower triangle only
    T old[2][2][4];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = ri + wr + 16 * x + (M::kRowFromReg ? 4 * v + lk : 4 * lk + v);
                const int c = rj + wc + 16 * y + li;
                old[x][y][v] = A[(size_t)r * np + c];
            }
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = ri + wr + 16 * x + (M::kRowFromReg ? 4 * v + lk : 4 * lk + v);
                const int c = rj + wc + 16 * y + li;
                if (bi != bj || c <= r) A[(size_t)r * np + c] = old[x][y][v] - acc[x][y][v];
            }
}

template <typename T>
__global__ __launch_bounds__(256) void k_chol_update(int np, int kc0, int kw, int bj0, int w, int nbk,
                                                     T* __restrict__ A) {
    const int t = xcd_tile(blockIdx.x, gridDim.x);
    const int head = w * (w + 1) / 2;
    int bi, bj;
    if (t < head) {
        int r = (int)((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
        while ((r + 1) * (r + 2) / 2 <= t) ++r;
        while (r * (r + 1) / 2 > t) --r;
        bi = bj0 + r;
        bj = bj0 + (t - r * (r + 1) / 2);
    } else {
        const int t2 = t - head;
        bi = bj0 + w + t2 / w;
        bj = bj0 + t2 % w;
    }
    if (bi >= nbk) return;
    __shared__ T P[NB][NB + 1];
    __shared__ T Q[NB][NB + 1];
    chol_update_tile<T>(np, bi * NB, bj * NB, kc0, kw, A, P, Q);
}

// Blocked right-looking Cholesky of the padded np x np matrix in two levels:
// column blocks of NB = 64 are factored (diag + panel) and applied at once
// only to the remaining columns of their super-panel of SP blocks; the rest of
// the matrix receives one rank-(SP NB) update per super-panel.  Every element
// of the trailing matrix is then read and written once per 256 columns
// instead of once per 64, which lifts the update above the HBM roofline.
constexpr int SP = 4;
constexpr int SYMV_SPLIT = 8;   // tile split of the refinement matvec
constexpr int REFINE_STEPS = 3; // FP32 solves per mixed-precision EEQ solve

// ---------------------------------------------------------------------------
// K4: triangular solves with the blocked factor
// ---------------------------------------------------------------------------
// Blocked substitution with the stored inverses of the diagonal blocks.
// Forward, block k: y_k = Linv_k b_k (every workgroup recomputes the 64x64
// product from LDS; workgroup 0 stores it), then rows below the block get
// b_r -= L(r, k) y_k.  Backward, block k (descending): x_k = Linv_k^T c_k,
// then c_j -= L(k, j)^T x_k for j < k0.
// Forward, block k: y_k = Linv_k b_k, then b_r -= L(r, k-block) y_k for the
// 64-row tile of this workgroup (rows r0 = k0 + NB + 64 blockIdx.x ...).  The
// tile is staged in LDS with coalesced row reads; thread (row, q) sums the
// products p = 4u + q and quad shuffles combine the four shares.  Every
// workgroup forms y_k itself (64 x 64 product from LDS); workgroup 0 stores it.
template <typename T>
__global__ __launch_bounds__(256) void k_trsv_fwd(int np, int k0, const T* __restrict__ A,
                                                  const T* __restrict__ Linv, T* __restrict__ b,
                                                  T* __restrict__ y) {
    __shared__ T W[NB][NB + 1];
    __shared__ T Tt[NB][NB + 1];
    __shared__ T bk[NB], yk[NB];
    const int tid = threadIdx.x, t = tid >> 2, q = tid & 3;
    const int r0 = k0 + NB + blockIdx.x * NB;
    const T* Li = Linv + (size_t)(k0 / NB) * NB * NB;
    _Pragma("unroll") for (int u_ = 0, e = tid; u_ < NB * NB / 256; ++u_, e += 256) {
        const int rr = e / NB, p = e % NB;
        W[rr][p] = Li[e];
        const T v = A[(size_t)min(r0 + rr, np - 1) * np + k0 + p];  // clamped: unconditional load
        Tt[rr][p] = (r0 + rr < np) ? v : T(0);
    }
    if (tid < NB) bk[tid] = b[k0 + tid];
    __syncthreads();
    T s = T(0);
#pragma unroll
    for (int u = 0; u < NB / 4; ++u) s += W[t][4 * u + q] * bk[4 * u + q];
    s += __shfl_xor(s, 1);
    s += __shfl_xor(s, 2);
    if (q == 0) {
        yk[t] = s;
        if (blockIdx.x == 0) y[k0 + t] = s;
    }
    __syncthreads();
    s = T(0);
#pragma unroll
    for (int u = 0; u < NB / 4; ++u) s += Tt[t][4 * u + q] * yk[4 * u + q];
    s += __shfl_xor(s, 1);
    s += __shfl_xor(s, 2);
    if (q == 0 && r0 + t < np) b[r0 + t] -= s;
}
// Backward, block k (descending): x_k = Linv_k^T c_k, then c_j -= L(k-block, j)^T x_k
// for the 64 columns j of this workgroup (j < k0).  Wave g sums rows p in
// [16 g, 16 g + 16) with coalesced row reads; the four partial sums are
// combined in LDS in a fixed order.
template <typename T>
__global__ __launch_bounds__(256) void k_trsv_bwd(int np, int k0, const T* __restrict__ A,
                                                  const T* __restrict__ Linv, T* __restrict__ c,
                                                  T* __restrict__ xout) {
    __shared__ T W[NB][NB + 1];
    __shared__ T ck[NB], xk[NB];
    __shared__ T part[4][NB];
    const int tid = threadIdx.x, t = tid >> 2, q = tid & 3;
    const T* Li = Linv + (size_t)(k0 / NB) * NB * NB;
    _Pragma("unroll") for (int u_ = 0, e = tid; u_ < NB * NB / 256; ++u_, e += 256) W[e / NB][e % NB] = Li[e];
    if (tid < NB) ck[tid] = c[k0 + tid];
    __syncthreads();
    T s = T(0);
#pragma unroll
    for (int u = 0; u < NB / 4; ++u) s += W[4 * u + q][t] * ck[4 * u + q];
    s += __shfl_xor(s, 1);
    s += __shfl_xor(s, 2);
    if (q == 0) {
        xk[t] = s;
        if (blockIdx.x == 0) xout[k0 + t] = s;
    }
    __syncthreads();
    const int jj = tid & 63, g = tid >> 6;
    const int col = blockIdx.x * NB + jj;
    T acc = T(0);
    if (col < k0) {
#pragma unroll
        for (int p = 16 * g; p < 16 * g + 16; ++p) acc += A[(size_t)(k0 + p) * np + col] * xk[p];
    }
    part[g][jj] = acc;
    __syncthreads();
    if (g == 0 && col < k0) c[col] -= ((part[0][jj] + part[1][jj]) + part[2][jj]) + part[3][jj];
}

// Single-launch sweeps.  One workgroup per 64-row block; block w needs the
// solution blocks k < w (forward) or k > w (backward).  Each workgroup stages
// the L tile of the next dependency in LDS before waiting for its ready flag,
// folds L(w,k) y_k into its right-hand side as soon as y_k is published, then
// applies the stored inverse of its diagonal block and publishes y_w with an
// agent-scope release.  Workgroups wait only for blocks published by
// lower-numbered workgroups (the backward sweep numbers blocks in descending
// order), so progress never depends on a workgroup that has not started.
// Every wait is bounded: after SPIN_MAX polls the workgroup sets FLAG_SOLVE
// and continues, so the launch always terminates.
constexpr int SPIN_MAX = 1 << 18;

// Waits for ready flag f; gives up at once when any workgroup has already
// flagged a failed wait, so a broken sweep ends after one bounded wait.
__device__ inline bool wait_ready(const int* f, int* flags) {
    for (int it = 0; it < SPIN_MAX; ++it) {
        if (__hip_atomic_load(f, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) != 0) return true;
        if (__hip_atomic_load(flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & FLAG_SOLVE) return false;
        __builtin_amdgcn_s_sleep(1);
    }
    atomicOr(flags, FLAG_SOLVE);
    return false;
}

template <typename T>
__global__ __launch_bounds__(256) void k_trsv_fwd_sweep(int np, const T* __restrict__ A, const T* __restrict__ Linv,
                                                        const T* __restrict__ b, T* __restrict__ y,
                                                        int* __restrict__ ready, int* __restrict__ flags) {
    __shared__ T Tt[NB][NB + 1];
    __shared__ T Wi[NB][NB + 1];  // inverse of the diagonal block, fetched first
    __shared__ T yk[NB];
    __shared__ T bw[NB];
    const int w = blockIdx.x, tid = threadIdx.x, t = tid >> 2, q = tid & 3;
    T acc = (q == 0) ? b[w * NB + t] : T(0);  // thread (t, q): share of row t
    {
        const T* Li = Linv + (size_t)w * NB * NB;
        _Pragma("unroll") for (int u_ = 0, e = tid; u_ < NB * NB / 256; ++u_, e += 256) Wi[e / NB][e % NB] = Li[e];
    }
    bool ok = true;
    for (int k = 0; k < w; ++k) {
        __syncthreads();
        _Pragma("unroll") for (int u_ = 0, e = tid; u_ < NB * NB / 256; ++u_, e += 256)
            Tt[e / NB][e % NB] = A[(size_t)(w * NB + e / NB) * np + k * NB + e % NB];
        if (tid < NB) {
            ok = wait_ready(ready + k, flags) && ok;
            yk[tid] = __hip_atomic_load(y + k * NB + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < NB / 4; ++u) acc -= Tt[t][4 * u + q] * yk[4 * u + q];
    }
    acc += __shfl_xor(acc, 1);
    acc += __shfl_xor(acc, 2);
    __syncthreads();
    if (q == 0) bw[t] = acc;
    __syncthreads();
    T s = T(0);
#pragma unroll
    for (int u = 0; u < NB / 4; ++u) s += Wi[t][4 * u + q] * bw[4 * u + q];
    s += __shfl_xor(s, 1);
    s += __shfl_xor(s, 2);
    if (q == 0) {
        __hip_atomic_store(y + w * NB + t, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __threadfence();  // the block is visible device-wide before the flag
    }
    __syncthreads();
    if (tid == 0) __hip_atomic_store(ready + w, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    if (!ok && tid < NB) atomicOr(flags, FLAG_SOLVE);
}

// Backward: x_w = Linv_w^T (c_w - sum_{k > w} L(k, w)^T x_k), workgroup g
// handles block w = nbk - 1 - g.
template <typename T>
__global__ __launch_bounds__(256) void k_trsv_bwd_sweep(int np, const T* __restrict__ A, const T* __restrict__ Linv,
                                                        const T* __restrict__ c, T* __restrict__ x,
                                                        int* __restrict__ ready, int* __restrict__ flags) {
    __shared__ T Tt[NB][NB + 1];
    __shared__ T Wi[NB][NB + 1];  // inverse of the diagonal block, fetched first
    __shared__ T xk[NB];
    __shared__ T cw[NB];
    const int nbk = np / NB;
    const int w = nbk - 1 - (int)blockIdx.x, tid = threadIdx.x, t = tid >> 2, q = tid & 3;
    T acc = (q == 0) ? c[w * NB + t] : T(0);  // thread (t, q): share of column t
    {
        const T* Li = Linv + (size_t)w * NB * NB;
        _Pragma("unroll") for (int u_ = 0, e = tid; u_ < NB * NB / 256; ++u_, e += 256) Wi[e / NB][e % NB] = Li[e];
    }
    bool ok = true;
    for (int k = nbk - 1; k > w; --k) {
        __syncthreads();
        _Pragma("unroll") for (int u_ = 0, e = tid; u_ < NB * NB / 256; ++u_, e += 256)
            Tt[e / NB][e % NB] = A[(size_t)(k * NB + e / NB) * np + w * NB + e % NB];
        if (tid < NB) {
            ok = wait_ready(ready + k, flags) && ok;
            xk[tid] = __hip_atomic_load(x + k * NB + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < NB / 4; ++u) acc -= Tt[4 * u + q][t] * xk[4 * u + q];
    }
    acc += __shfl_xor(acc, 1);
    acc += __shfl_xor(acc, 2);
    __syncthreads();
    if (q == 0) cw[t] = acc;
    __syncthreads();
    T s = T(0);
#pragma unroll
    for (int u = 0; u < NB / 4; ++u) s += Wi[4 * u + q][t] * cw[4 * u + q];
    s += __shfl_xor(s, 1);
    s += __shfl_xor(s, 2);
    if (q == 0) {
        __hip_atomic_store(x + w * NB + t, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __threadfence();  // the block is visible device-wide before the flag
    }
    __syncthreads();
    if (tid == 0) __hip_atomic_store(ready + w, 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    if (!ok && tid < NB) atomicOr(flags, FLAG_SOLVE);
}

// ---------------------------------------------------------------------------
// K4c: iterative EEQ solve.  The reduced EEQ matrices of non-bonded clusters
// are well conditioned (water clusters: kappa ~ 6), so preconditioned CG
// converges in ~15 matrix-vector products.  Each product streams the matrix
// once from HBM (row-major, both triangles stored), which replaces the
// latency-bound chain of the blocked factorisation.
// ---------------------------------------------------------------------------
constexpr int PCG_THREADS = 512;
constexpr int PCG_WAVES = PCG_THREADS / 64;
constexpr int PCGS_THREADS = 256;  // the streaming form, k_eeq_pcg
constexpr int PCGS_WAVES = PCGS_THREADS / 64;
constexpr int PCGS_PP = 8;  // from this many blocks per wavefront on, two register buffers stream in turn

// Sum over the 64 lanes of a wavefront (fixed butterfly; every lane gets it).
__device__ inline double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// Fixed-order sum over a workgroup of 256 threads: wavefront butterflies,
// then the four wavefront totals in order (every thread returns the total).
__device__ double wg_sum256(double v, double* red) {
    v = wave_sum(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
}

// Device-coherent access for data shared between the workgroups of a
// persistent kernel: relaxed agent-scope atomics, i.e. loads and stores that
// bypass the non-coherent caches (no cache write-back or invalidation, whose
// cost grows with the number of workgroups on a multi-die GPU).
__device__ inline double ld_c(const double* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ inline void st_c(double* p, double v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ inline unsigned long long ld_cu(const unsigned long long* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void st_cu(unsigned long long* p, unsigned long long v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// s_waitcnt vmcnt(0): this wave's loads and stores have completed (device-
// coherent stores are then visible to every device-coherent load).
__device__ inline void wait_vm() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// Grid-wide sum of two values per thread for a persistent kernel whose
// G <= 256 workgroups are all resident.  Mailboxes are 128-byte lines of
// 64-bit words holding MB_EMPTY (a NaN pattern no arithmetic produces) until
// written: at barrier j workgroup g writes its sums to line (g, j mod 4), and
// thread t of every workgroup polls line (t, j mod 4) and reads producer t's
// values; every workgroup then adds the G values in the same fixed order, so
// all hold identical sums.  (The words of all workgroups side by side were
// slower: one line then has many writers; H-(Gly)200-OH 660 against 637 us.)
// A writer clears its line (g, (j + 2) mod 4), last written at barrier j - 2, behind its value of barrier j: having passed
// barrier j - 1 it has seen every workgroup's barrier j - 1 value, each
// written after its writer finished reading barrier j - 2, so no reader still
// needs the cleared line; and the clear completes (the wait at the head of
// barrier j + 1) before the value of barrier j + 1 is written, which every
// reader has seen before it polls for barrier j + 2.  With three lines the
// clear has to complete before the value of its own barrier, one more trip to
// memory in each barrier.  Every wait is bounded (FLAG_SOLVE on a timeout).
// Ordering without cache maintenance: the data a workgroup shares is written
// with device-coherent stores that complete (vmcnt) before its mailbox value
// is written, and read with device-coherent loads issued after all values
// were seen, so every shared write before the barrier is visible to every
// workgroup after it.
constexpr unsigned long long MB_EMPTY = 0x7ff0deadbeef0001ull;
constexpr int MB_LINE = 16;                  // 64-bit words per 128-byte line
constexpr int MB_WORDS = 4 * 256 * MB_LINE;  // lines (g, k), k < 4, at (4 g + k) MB_LINE

// between: issued behind the publication and ahead of the polls (loads whose
// latency the barrier covers; ahead of the publication they would delay it).
// red: 4 PCGS_WAVES doubles of LDS, used in halves by the barrier's parity, so
// that a barrier writes the half that was last read before the barrier ahead
// of it.
template <class F>
__device__ __forceinline__ bool grid_allreduce2(double v0, double v1, double* sums, unsigned long long* mb, int j,
                                                int* flags, double* red, F between) {
    const int G = gridDim.x, g = blockIdx.x, tid = threadIdx.x, k = j & 3;
    double* const rd = red + (j & 1) * 2 * PCGS_WAVES;
    v0 = wave_sum(v0);
    v1 = wave_sum(v1);
    if ((tid & 63) == 0) {
        rd[tid >> 6] = v0;
        rd[PCGS_WAVES + (tid >> 6)] = v1;
    }
    wait_vm();
    __syncthreads();
    if (tid == 0) {
        unsigned long long* const own = mb + (4 * g + k) * MB_LINE;
        unsigned long long* const old = mb + (4 * g + ((k + 2) & 3)) * MB_LINE;
        double s0 = rd[0], s1 = rd[PCGS_WAVES];
#pragma unroll
        for (int w = 1; w < PCGS_WAVES; ++w) {
            s0 += rd[w];
            s1 += rd[PCGS_WAVES + w];
        }
        st_cu(own, __double_as_longlong(s0));
        st_cu(own + 1, __double_as_longlong(s1));
        st_cu(old, MB_EMPTY);
        st_cu(old + 1, MB_EMPTY);
    }
    between();
    double u0 = 0.0, u1 = 0.0;
    int bad = 0;
    if (tid < G) {
        const unsigned long long* const in = mb + (4 * tid + k) * MB_LINE;
        unsigned long long a0 = MB_EMPTY, a1 = MB_EMPTY;
        for (int it = 0;; ++it) {
            a0 = ld_cu(in);
            a1 = ld_cu(in + 1);
            if (a0 != MB_EMPTY && a1 != MB_EMPTY) break;
            if (it > SPIN_MAX ||
                ((it & 63) == 63 &&
                 (__hip_atomic_load(flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & FLAG_SOLVE))) {
                bad = 1;
                atomicOr(flags, FLAG_SOLVE);
                break;
            }
        }
        u0 = __longlong_as_double(a0);
        u1 = __longlong_as_double(a1);
    }
    __syncthreads();  // thread 0 has read this workgroup's partial sums
    if (tid < 256) {
        u0 = wave_sum(u0);
        u1 = wave_sum(u1);
        if ((tid & 63) == 0) {
            rd[tid >> 6] = u0;
            rd[PCGS_WAVES + (tid >> 6)] = u1;
        }
    }
    const bool ok = __syncthreads_or(bad) == 0;
    sums[0] = (rd[0] + rd[1]) + (rd[2] + rd[3]);
    sums[1] = (rd[PCGS_WAVES] + rd[PCGS_WAVES + 1]) + (rd[PCGS_WAVES + 2] + rd[PCGS_WAVES + 3]);
    return ok;
}

// z_b = Linv_b^T (Linv_b r_b) for the 64-block b (r_b and the result in LDS;
// threads 0..255 compute, every thread synchronises).  ld: row length of Li
// (LDC for the copy in LDS, whose rows must not start on the same bank).
constexpr int LDC = NB + 1;
__device__ void bjacobi_apply(const double* __restrict__ Li, int ld, const double* rb, double* wb, double* zb) {
    const int tid = threadIdx.x, t = (tid >> 2) & 63, q = tid & 3;
    const bool act = tid < 256;
    double s = 0.0;
    if (act) {
#pragma unroll
        for (int u = 0; u < NB / 4; ++u) s += Li[t * ld + 4 * u + q] * rb[4 * u + q];
    }
    s += __shfl_xor(s, 1);
    s += __shfl_xor(s, 2);
    __syncthreads();
    if (act && q == 0) wb[t] = s;
    __syncthreads();
    s = 0.0;
    if (act) {
#pragma unroll
        for (int u = 0; u < NB / 4; ++u) s += Li[(4 * u + q) * ld + t] * wb[4 * u + q];
    }
    s += __shfl_xor(s, 1);
    s += __shfl_xor(s, 2);
    if (act && q == 0) zb[t] = s;
    __syncthreads();
}

// Fallback solve of a reduced EEQ system that is not positive definite
// (FLAG_CHOL raised by the Cholesky of a diagonal block or of the matrix): the
// reference falls back to an LU with partial pivoting of its bordered system
// when the Cholesky of A fails (eeq_solver.cpp:2143-2165, the augmented-system
// PartialPivLU).  The reduced system R p = b is the bordered system with the
// constraints eliminated, so Gaussian elimination with partial pivoting on it
// gives the same charges.  One workgroup: behind the Cholesky solve a kernel
// that does nothing unless the flag is set and clears it when it succeeds (a
// zero pivot keeps it: singular system); in the iterative solve the first
// workgroup of k_eeq_pcg, which leaves the flag to the workgroups that have
// yet to read it and raises FLAG_LU beside it.
// R: layout 0 = packed lower 64x64 blocks (block I >= J at (I(I+1)/2 + J) 64^2,
// row-major inside), layout 1 = row-major np x np, lower triangle used.
// W: nr x (nr + 1) work (the system augmented with b).  nr <= LU_MAX.
constexpr int LU_MAX = 1024;
constexpr int LU_T = 1024;
// The update of a step with at most LU_FLAT columns left takes its elements one
// after another (two trips to memory hold a step then), with more LU_ROWS rows
// of a wavefront at a time, whose loads are in flight together.  Measured,
// evaluation of hydrogen chains in the 512 threads of the iterative solve: all
// elements one after another 70 atoms 343 us, 300 5.5 ms, 1000 230 ms; all by
// rows 380 us, 4.1 and 97 ms.
constexpr int LU_FLAT = 128;
constexpr int LU_ROWS = 8;
template <int NT>
__device__ __noinline__ bool eeq_lu(int np, int nr, int layout, const double* __restrict__ R,
                                    const double* __restrict__ b, double* __restrict__ W, double* __restrict__ x) {
    __shared__ int s_piv;
    __shared__ double s_best[NT / 64];
    __shared__ int s_idx[NT / 64];
    __shared__ double xs[LU_MAX];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int m = nr, ld = nr + 1;
    for (long e = tid; e < (long)m * m; e += NT) {
        const int i = (int)(e / m), j = (int)(e % m);
        const int r = max(i, j), c = min(i, j);
        double v;
        if (layout == 0) {
            const long I = r / NB, J = c / NB;
            v = R[(I * (I + 1) / 2 + J) * NB * NB + (r % NB) * NB + (c % NB)];
        } else {
            v = R[(long)r * np + c];
        }
        W[(long)i * ld + j] = v;
    }
    for (int i = tid; i < m; i += NT) W[(long)i * ld + m] = b[i];
    __syncthreads();
    int ok = 1;
    for (int k = 0; k < m; ++k) {
        // pivot row: largest |W(i, k)| for i >= k, the lowest index on ties
        double best = -1.0;
        int bi = m;
        for (int i = k + tid; i < m; i += NT) {
            const double a = fabs(W[(long)i * ld + k]);
            if (a > best) {
                best = a;
                bi = i;
            }
        }
        for (int o = 32; o > 0; o >>= 1) {
            const double ob = __shfl_xor(best, o);
            const int oi = __shfl_xor(bi, o);
            if (ob > best || (ob == best && oi < bi)) {
                best = ob;
                bi = oi;
            }
        }
        if (lane == 0) {
            s_best[wv] = best;
            s_idx[wv] = bi;
        }
        __syncthreads();
        if (tid == 0) {
            double bb = s_best[0];
            int ii = s_idx[0];
            for (int w = 1; w < NT / 64; ++w)
                if (s_best[w] > bb || (s_best[w] == bb && s_idx[w] < ii)) {
                    bb = s_best[w];
                    ii = s_idx[w];
                }
            s_piv = (bb > 0.0 && ii < m) ? ii : -1;
        }
        __syncthreads();
        const int p = s_piv;
        if (p < 0) {
            ok = 0;
            break;
        }
        if (p != k)
            for (int j = k + tid; j <= m; j += NT) {
                const double t = W[(long)k * ld + j];
                W[(long)k * ld + j] = W[(long)p * ld + j];
                W[(long)p * ld + j] = t;
            }
        __syncthreads();
        const double inv = 1.0 / W[(long)k * ld + k];
        // rows k + 1 .. m - 1, columns k + 1 .. m (the last is b)
        const int cols = m - k;
        if (cols <= LU_FLAT) {
            for (int e = tid; e < (cols - 1) * cols; e += NT) {
                const int i = k + 1 + e / cols, j = k + 1 + e % cols;
                W[(long)i * ld + j] -= (W[(long)i * ld + k] * inv) * W[(long)k * ld + j];
            }
        } else {
            // LU_ROWS rows of a wavefront at a time, all loaded before the first is stored
            for (int i0 = k + 1 + wv; i0 < m; i0 += LU_ROWS * (NT / 64)) {
                double f[LU_ROWS];
                double* row[LU_ROWS];
#pragma unroll
                for (int u = 0; u < LU_ROWS; ++u) {
                    const int i = i0 + u * (NT / 64);
                    row[u] = W + (long)min(i, m - 1) * ld;
                    f[u] = i < m ? row[u][k] * inv : 0.0;
                }
                for (int j = k + 1 + lane; j <= m; j += 64) {
                    const double p = W[(long)k * ld + j];
                    double v[LU_ROWS];
#pragma unroll
                    for (int u = 0; u < LU_ROWS; ++u) v[u] = row[u][j];
#pragma unroll
                    for (int u = 0; u < LU_ROWS; ++u)
                        if (i0 + u * (NT / 64) < m) row[u][j] = v[u] - f[u] * p;
                }
            }
        }
        __syncthreads();
    }
    if (!ok) return false;
    for (int i = m - 1; i >= 0; --i) {
        double sacc = 0.0;
        for (int j = i + 1 + tid; j < m; j += NT) sacc += W[(long)i * ld + j] * xs[j];
        for (int o = 32; o > 0; o >>= 1) sacc += __shfl_xor(sacc, o);
        if (lane == 0) s_best[wv] = sacc;
        __syncthreads();
        if (tid == 0) {
            double t = 0.0;
            for (int w = 0; w < NT / 64; ++w) t += s_best[w];
            xs[i] = (W[(long)i * ld + m] - t) / W[(long)i * ld + i];
        }
        __syncthreads();
    }
    for (int i = tid; i < np; i += NT) x[i] = (i < m) ? xs[i] : 0.0;
    return true;
}

__global__ __launch_bounds__(LU_T) void k_eeq_lu_fallback(int np, int nr, const double* __restrict__ R,
                                                          const double* __restrict__ b, double* __restrict__ W,
                                                          double* __restrict__ x, int* __restrict__ flags) {
    __shared__ int s_flag;
    if (threadIdx.x == 0) s_flag = __hip_atomic_load(flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (!(s_flag & FLAG_CHOL) || nr > LU_MAX) return;
    // the LU result replaces whatever the failed solve left (its bounded waits included)
    if (eeq_lu<LU_T>(np, nr, 1, R, b, W, x) && threadIdx.x == 0) atomicAnd(flags, ~(FLAG_CHOL | FLAG_SOLVE));
}

// Persistent PCG on R x = b with R in packed symmetric storage: the 64x64
// blocks (I, J), I >= J, at Rp + (I (I + 1) / 2 + J) 64^2, row-major, the
// diagonal blocks full.  Workgroup g owns the 64-row blocks g, g + G, ... (at
// most PCG_MAXB) for the vector updates.  The matrix-vector product runs over
// the stored blocks, each block read once by one wavefront (contiguous,
// balanced ranges of the packed order): lane (rg, cg) holds 8 rows x 8
// columns of the block, and the row sums R_IJ p_J and column sums
// R_IJ^T p_I come from 8-lane transpose-reduces.  Every (row block X, column block Y)
// product goes to its own partial part[X][Y][64], which the owner of X adds
// in Y order after the barrier; p.q is formed from the partials (it is
// linear in them).  Per iteration: (1) p = z + beta p_prev (formed on the fly
// by every reader; owners store their rows), block products; barrier;
// (2) alpha = rz / pq; owners: q, x += alpha p, r -= alpha q, z = M^-1 r,
// partials r.z and r.r; barrier; beta = rz_new / rz.  Stops when
// r.r <= tol2 * b.b (uniform decision from identical sums) or after maxit
// iterations (FLAG_SOLVE).  Cross-workgroup vectors (z, p, part) are written
// and read with device-coherent accesses (ld_c, st_c); an owner keeps its
// rows of x and r, and the Linv of a single owned block, in LDS for the
// whole solve and writes x at the end.
//
// Streaming (np > 4032): one wavefront per SIMD with the whole register file.
// Up to PCGS_PP blocks per wavefront its first block stays in registers for
// the whole solve (water_3000, 4.4 blocks each: a quarter of the matrix), and
// the next one is loaded behind the publication of the barrier ahead of it,
// which hides its latency; with more, two register buffers take the blocks in
// turn.  water_3000 1324 -> 1259 us against eight wavefronts with one buffer
// (mixed 1019 -> 970); in turn from two blocks on 1282 and 987.  The first form
// takes 30 us an iteration on water_3000 (113 MB of blocks through the memory,
// 120 MB read and 5 MB written with partials and vectors: 4.1 TB/s between two
// barriers); 80 chains of C80H162 run at 0.34 ms either way: 1.49 GB of blocks
// and 0.09 GB of partials at 4.6 TB/s, where a device copy moves 5.2.
//
// Preconditioner.  M = D, the diagonal blocks of R, cuts a fragment of more
// than 64 variables into pieces, and every variable of the fragment carries
// the terms of the same last atom l, R = A - u 1^T - 1 u^T + A_ll 1 1^T: the
// rank-one part couples all pieces.  Over such "split" fragments f
// (SM) M = D + sum_f A_ll(f) 1_f 1_f^T with D the diagonal blocks of A
// itself within the fragment (k_bjacobi_setup), and by Sherman-Morrison
//   z = y - sum_f sigma_f s_f w_f,  y = D^-1 r, w_f = D^-1 1_f,
//   s_f = 1_f . y,  sigma_f = 1 / (1 / A_ll(f) + 1_f . w_f),
//   r.z = r.y - sum_f sigma_f s_f^2.
// Owners publish y and their pieces' parts of s_f; after the barrier every
// workgroup forms the same sigma_f s_f, and z on the fly.  Together with the
// order of the variables along the bond graph (reduced_order): 80 chains of
// C80H162 (mixed) 467 -> 76 to 80 iterations by the geometry and 159 -> 27 ms,
// C300H602 148 -> 38, H-(Gly)200-OH 97 -> 39, C40H82 39 -> 15.
constexpr int PCG_MAXB = 8;
constexpr double PCG_TOL_FP64 = 1e-13;   // default |r| / |b| of the FP64 path
constexpr double PCG_TOL_MIXED = 1e-10;  // default of the mixed path (EEQ energy is variational in q)
constexpr int PCG_MAXIT = 1000;
constexpr int SM_MAXF = 512;        // split fragments and 64-variable blocks of the Sherman-Morrison form
constexpr int SM_MAXB = 1024;       // (beyond: plain diagonal blocks)
constexpr int SM_MAXP = SM_MAXB + SM_MAXF;  // pieces: one per block and one more per fragment boundary inside a block

struct PcgArgs {
    int np, nr, maxit;
    double* lu_w;        // work of the dense fallback (nullptr: nr > LU_MAX)
    double tol2;
    const double *Rp, *Lj, *b;
    double *x, *z, *pb, *part;
    unsigned long long* mb;  // mailboxes; with resident blocks the exchanged vectors z, sp and part lie behind them
    int nmb;                 // words to clear
    int *iters, *flags;
    // split fragments
    int nsf;
    const int* rowf;     // [np] 2 f + slot of the row's piece in its block, or -1
    const int* poff;     // [nsf + 1] pieces of a fragment in pidx
    const int* pidx;     // a piece's place 2 block + slot
    const double* w;     // [np] D^-1 1_f (k_bjacobi_setup)
    const double* w1;    // [2 nbk] 1_f . w of each piece
    const double* all;   // [nsf] A_ll of the fragment's last atom
    const int* smon;     // [nbk] 0: the block's A was not positive definite and its R was factored instead
    double* sp;          // [2 nbk] parts of s_f
};

// Sum of 8 per-lane values v[k] over the 8 lanes that differ in lane bits
// s, s + 1, s + 2 (recursive halving): lane l ends with the total of
// k(l) = 4 b(s+2) + 2 b(s+1) + b(s), b the bits of l; the eight lanes of a
// group hold the same bits.
template <int S>
__device__ inline double tr_reduce8(const double (&v)[8], int l) {
    double a4[4], a2[2];
    const bool h2 = (l >> (S + 2)) & 1, h1 = (l >> (S + 1)) & 1, h0 = (l >> S) & 1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const double keep = h2 ? v[i + 4] : v[i], send = h2 ? v[i] : v[i + 4];
        a4[i] = keep + __shfl_xor(send, 4 << S);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const double keep = h1 ? a4[i + 2] : a4[i], send = h1 ? a4[i] : a4[i + 2];
        a2[i] = keep + __shfl_xor(send, 2 << S);
    }
    return (h0 ? a2[1] : a2[0]) + __shfl_xor(h0 ? a2[0] : a2[1], 1 << S);
}

// Products of one 64 x 64 block held as rv by a wavefront (see k_eeq_pcg) with
// the p of its rows (pw[0]) and columns (pw[1]): rs = (R p_J) of row l and,
// for an off-diagonal block, cs = (R^T p_I) of column
// cend = 2 cg + (rg & 1) + 16 (rg >> 1), whose p is pjc.
__device__ __forceinline__ void block_products(const double (&rv)[8][8], const double (*pw)[NB], int l, bool cols,
                                               double& rs, double& cs, double& pjc) {
    const int rg = l >> 3, cg = l & 7;
    double v[8], o[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = pw[1][2 * cg + (k & 1) + 16 * (k >> 1)];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        double s = 0.0;
#pragma unroll
        for (int m = 0; m < 8; ++m) s += rv[k][m] * v[m];
        o[k] = s;
    }
    rs = tr_reduce8<0>(o, l);  // row 8 rg + cg = l
    __builtin_amdgcn_sched_barrier(0);  // rows before columns: both at once do not fit the registers
    cs = pjc = 0.0;
    if (!cols) return;
    pjc = pw[1][2 * cg + (rg & 1) + 16 * (rg >> 1)];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = pw[0][8 * rg + k];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        double s = 0.0;
#pragma unroll
        for (int m = 0; m < 8; ++m) s += rv[m][k] * v[m];
        o[k] = s;
    }
    cs = tr_reduce8<3>(o, l);
    __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ void load_block(double (&rv)[8][8], const double* __restrict__ R, int l) {
    const int rg = l >> 3, cg = l & 7;
    const double2* Rb = reinterpret_cast<const double2*>(R);
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const double2 v2 = Rb[((8 * rg + i) * NB + 16 * j + 2 * cg) / 2];
            rv[i][2 * j] = v2.x;
            rv[i][2 * j + 1] = v2.y;
        }
}
// block t of the packed lower order: t = I (I + 1) / 2 + J
__device__ inline void packed_block(int t, int& I, int& J) {
    I = (int)((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
    while ((long)(I + 1) * (I + 2) / 2 <= t) ++I;
    while ((long)I * (I + 1) / 2 > t) --I;
    J = t - I * (I + 1) / 2;
}

// sigma_f s_f of every split fragment into sfs, from the published parts;
// returns sum_f sigma_f s_f^2 (the same in every workgroup).  sig: sigma_f.
// pbuf: the parts, in LDS.
template <int NT>
__device__ double sm_sums(const PcgArgs& a, double* sfs, const double* sig, const double* pbuf, double* red) {
    const int tid = threadIdx.x, l8 = tid & 7;
    double e = 0.0;
    for (int f0 = 0; f0 < a.nsf; f0 += NT / 8) {
        const int f = f0 + (tid >> 3);
        double s = 0.0;
        if (f < a.nsf)
            for (int k = a.poff[f] + l8; k < a.poff[f + 1]; k += 8) s += pbuf[k];
        s += __shfl_xor(s, 1);
        s += __shfl_xor(s, 2);
        s += __shfl_xor(s, 4);
        if (f < a.nsf && l8 == 0) {
            sfs[f] = sig[f] * s;
            e += sig[f] * s * s;
        }
    }
    e = wave_sum(e);
    if ((tid & 63) == 0) red[tid >> 6] = e;
    __syncthreads();
    double t = red[0];
#pragma unroll
    for (int w = 1; w < NT / 64; ++w) t += red[w];
    return t;
}

template <int NT>
__device__ double sm_gather(const PcgArgs& a, int npc, double* sfs, const double* sig, double* pbuf, double* red) {
    for (int k = threadIdx.x; k < npc; k += NT) pbuf[k] = ld_c(a.sp + a.pidx[k]);
    __syncthreads();
    return sm_sums<NT>(a, sfs, sig, pbuf, red);
}

template <bool SM, bool PP>
__global__ __launch_bounds__(PCGS_THREADS, 1) void k_eeq_pcg(PcgArgs a) {
    __shared__ double red[4 * PCGS_WAVES], red2[2][PCGS_WAVES];
    __shared__ double pown[PCG_MAXB][NB];
    __shared__ double qs[PCGS_WAVES][NB];
    __shared__ double rb[NB], wb[NB], zb[NB];
    __shared__ double xo[PCG_MAXB][NB], ro[PCG_MAXB][NB];  // owned rows of x and r, resident for the solve
    __shared__ double Lc[NB * LDC];                         // Linv of the owned block when there is one
    __shared__ __align__(16) double pw[PCGS_WAVES][2][NB];    // per wavefront: p of the block's rows and columns
    __shared__ double sfs[SM ? SM_MAXF : 1], sig[SM ? SM_MAXF : 1], pbuf[SM ? SM_MAXP : 1];
    // a diagonal block that is not positive definite (FLAG_CHOL, set before
    // this launch and not cleared in it, so every workgroup reads the same
    // value) leaves the solve to the dense fallback
    if (__hip_atomic_load(a.flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & FLAG_CHOL) {
        if (blockIdx.x == 0 && a.lu_w && eeq_lu<PCGS_THREADS>(a.np, a.nr, 0, a.Rp, a.b, a.lu_w, a.x) && threadIdx.x == 0)
            atomicOr(a.flags, FLAG_LU);
        return;
    }
    const int np = a.np, G = gridDim.x, g = blockIdx.x, nbk = np / NB;
    const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63;
    const int nown = (nbk - g + G - 1) / G;
    // this wavefront's blocks of the packed order: [t0, t1)
    const long T = (long)nbk * (nbk + 1) / 2, W = (long)PCGS_WAVES * G, gw = (long)PCGS_WAVES * g + wv;
    const int t0 = (int)(T * gw / W), t1 = (int)(T * (gw + 1) / W);
    int I0, J0;
    packed_block(t0, I0, J0);
    // lane (rg, cg) holds rows 8 rg + i (i < 8) and columns 2 cg + (k & 1) + 16 (k >> 1) (k < 8) of a
    // block: every 16-byte load instruction reads whole 128-byte row segments
    const int rg = l >> 3, cg = l & 7;
    // PP: rv and ra take the blocks of the range in turn, the next one in
    // flight; otherwise ra keeps the first for the whole solve
    double ra[8][8], rv[8][8];
    constexpr int S0 = PP ? 0 : 1;  // first streamed block
    if (!PP && t0 < t1) load_block(ra, a.Rp + (size_t)t0 * NB * NB, l);
    auto first_stream = [&]() {
        if (t0 + S0 < t1) load_block(rv, a.Rp + (size_t)(t0 + S0) * NB * NB, l);
    };
    auto nothing = []() {};
    const bool lcache = nown == 1;
    if (lcache)
        for (int e = tid; e < NB * NB; e += PCGS_THREADS) Lc[(e >> 6) * LDC + (e & 63)] = a.Lj[(size_t)g * NB * NB + e];
    const int npc = SM ? a.poff[a.nsf] : 0;
    if (SM)
        for (int f = tid; f < a.nsf; f += PCGS_THREADS) {
            double s = 1.0 / a.all[f];
            for (int k = a.poff[f]; k < a.poff[f + 1]; ++k) s += a.w1[a.pidx[k]];
            sig[f] = 1.0 / s;
        }
    // z of a row: y, less the fragment's rank-one part
    auto zrow = [&](int row) {
        double v = ld_c(a.z + row);
        if (SM) {
            const int rf = a.rowf[row];
            if (rf >= 0) v -= sfs[rf >> 1] * a.w[row];
        }
        return v;
    };
    // owners publish y = D^-1 r of a block (rb -> z) and its pieces' parts of s_f
    auto publish = [&](int kb, double& lrz, double& lrr) {
        bjacobi_apply(lcache ? Lc : a.Lj + (size_t)kb * NB * NB, lcache ? LDC : NB, rb, wb, zb);
        if (tid < NB) {
            const double y = zb[tid], r = rb[tid];
            st_c(a.z + kb * NB + tid, y);
            lrz += r * y;
            lrr += r * r;
            if (SM) {
                const int rf = a.smon[kb] ? a.rowf[kb * NB + tid] : -1;
                const double s0 = wave_sum(rf >= 0 && !(rf & 1) ? y : 0.0), s1 = wave_sum(rf >= 0 && (rf & 1) ? y : 0.0);
                if (tid < 2) st_c(a.sp + 2 * kb + tid, tid ? s1 : s0);
            }
        }
    };
    // init: x = 0, r = b, z = M^-1 b; partials r.z and b.b
    double lrz = 0.0, lbb = 0.0;
    for (int o = 0; o < nown; ++o) {
        const int kb = g + o * G;
        if (tid < NB) {
            const double bv = a.b[kb * NB + tid];
            rb[tid] = bv;
            xo[o][tid] = 0.0;
            ro[o][tid] = bv;
        }
        __syncthreads();
        publish(kb, lrz, lbb);
    }
    int nbar = 0;  // barriers passed
    double sums[2];
    if (!grid_allreduce2(lrz, lbb, sums, a.mb, nbar++, a.flags, red, first_stream)) return;
    double rz = sums[0];
    const double bb = sums[1];
    if (SM) rz -= sm_gather<PCGS_THREADS>(a, npc, sfs, sig, pbuf, red2[0]);
    double beta = 0.0;
    int it = 0;
    bool done = !(bb > 0.0);
    for (; !done && it < a.maxit; ++it) {
        const double* pprev = a.pb + (size_t)((it + 1) & 1) * np;
        double* pcur = a.pb + (size_t)(it & 1) * np;
        // (1) owners: p rows; every wavefront: its blocks' products
        for (int o = 0; o < nown; ++o) {
            if (tid < NB) {
                const int row = (g + o * G) * NB + tid;
                const double pc = (it == 0) ? 0.0 : pown[o][tid];
                const double pv = zrow(row) + beta * pc;
                pown[o][tid] = pv;
                st_c(pcur + row, pv);
            }
        }
        double lpq = 0.0;
        int I = I0, J = J0;
        // what a block's product needs of z and p (y, p, w and fragment of its
        // columns and rows), loaded ahead of the next block's loads: loads
        // return in order
        struct Raw {
            double zj, pj, zi, pi, wj, wi;
            int fj, fi;
        };
        auto fetch = [&](int I, int J) {
            Raw r;
            const int cj = J * NB + l, ci = I * NB + l;
            r.zj = ld_c(a.z + cj);
            r.zi = ld_c(a.z + ci);
            r.pj = it == 0 ? 0.0 : ld_c(pprev + cj);
            r.pi = it == 0 ? 0.0 : ld_c(pprev + ci);
            r.fj = SM ? a.rowf[cj] : -1;
            r.fi = SM ? a.rowf[ci] : -1;
            r.wj = SM && r.fj >= 0 ? a.w[cj] : 0.0;
            r.wi = SM && r.fi >= 0 ? a.w[ci] : 0.0;
            return r;
        };
        auto next = [&](int& I, int& J) {
            if (++J > I) {
                ++I;
                J = 0;
            }
        };
        auto product = [&](const double (&blk)[8][8], const Raw& r) {
            // p of row I * 64 + l and column J * 64 + l
            double zj = r.zj, zi = r.zi;
            if (SM) {
                if (r.fj >= 0) zj -= sfs[r.fj >> 1] * r.wj;
                if (r.fi >= 0) zi -= sfs[r.fi >> 1] * r.wi;
            }
            const double pjl = zj + beta * r.pj, pil = zi + beta * r.pi;
            pw[wv][0][l] = pil;
            pw[wv][1][l] = pjl;
            __builtin_amdgcn_wave_barrier();
            double rs, cs, pjc;
            block_products(blk, pw[wv], l, I != J, rs, cs, pjc);
            st_c(a.part + ((size_t)I * nbk + J) * NB + l, rs);
            lpq += pil * rs;
            if (I != J) {
                st_c(a.part + ((size_t)J * nbk + I) * NB + 2 * cg + (rg & 1) + 16 * (rg >> 1), cs);
                lpq += pjc * cs;
            }
            next(I, J);
        };
        if (!PP) {
            if (t0 < t1) product(ra, fetch(I, J));
            for (int t = t0 + 1; t < t1; ++t) {
                if (t > t0 + 1) load_block(rv, a.Rp + (size_t)t * NB * NB, l);  // the first: behind the last barrier
                product(rv, fetch(I, J));
            }
        } else if (t0 < t1) {
            Raw r0 = fetch(I, J);
            for (int t = t0; t < t1; t += 2) {
                int I1 = I, J1 = J;
                next(I1, J1);
                Raw r1{};
                if (t + 1 < t1) {
                    r1 = fetch(I1, J1);
                    load_block(ra, a.Rp + (size_t)(t + 1) * NB * NB, l);
                }
                product(rv, r0);
                if (t + 1 >= t1) break;
                I1 = I;
                J1 = J;
                next(I1, J1);
                if (t + 2 < t1) {
                    r0 = fetch(I1, J1);
                    load_block(rv, a.Rp + (size_t)(t + 2) * NB * NB, l);
                }
                product(ra, r1);
            }
        }
        if (!grid_allreduce2(lpq, 0.0, sums, a.mb, nbar++, a.flags, red, nothing)) return;
        const double pq = sums[0];
        const double alpha = rz / pq;
        // (2) owners: q rows from the partials (Y order), x, r, z and the
        // partials r.z, r.r
        double lrz2 = 0.0, lrr = 0.0;
        for (int o = 0; o < nown; ++o) {
            const int kb = g + o * G;
            {
                // thread (row l, part wv) adds Y = wv, wv + PCGS_WAVES, ... in batches of 16 loads
                const double* pr = a.part + (size_t)kb * nbk * NB + l;
                double acc = 0.0;
                for (int y0 = wv; y0 < nbk; y0 += 16 * PCGS_WAVES) {
                    double t16[16];
#pragma unroll
                    for (int u = 0; u < 16; ++u) t16[u] = ld_c(pr + (size_t)min(y0 + PCGS_WAVES * u, nbk - 1) * NB);
#pragma unroll
                    for (int u = 0; u < 16; ++u) acc += (y0 + PCGS_WAVES * u < nbk) ? t16[u] : 0.0;
                }
                qs[wv][l] = acc;
            }
            __syncthreads();
            if (tid < NB) {
                double qv = qs[0][tid];
#pragma unroll
                for (int w = 1; w < PCGS_WAVES; ++w) qv += qs[w][tid];
                xo[o][tid] += alpha * pown[o][tid];
                const double rn = ro[o][tid] - alpha * qv;
                ro[o][tid] = rn;
                rb[tid] = rn;
            }
            __syncthreads();
            publish(kb, lrz2, lrr);
        }
        if (!grid_allreduce2(lrz2, lrr, sums, a.mb, nbar++, a.flags, red, first_stream)) return;
        const double rr = sums[1];
        double rz2 = sums[0];
        done = rr <= a.tol2 * bb;
        if (SM && !done) rz2 -= sm_gather<PCGS_THREADS>(a, npc, sfs, sig, pbuf, red2[it & 1]);
        beta = rz2 / rz;
        rz = rz2;
    }
    for (int o = 0; o < nown; ++o)
        if (tid < NB) a.x[(g + o * G) * NB + tid] = xo[o][tid];
    if (g == 0 && tid == 0) a.iters[0] = it;
    if (!done && g == 0 && tid == 0) atomicOr(a.flags, FLAG_SOLVE);
}

// The same solve with every block resident: each wavefront holds at most one
// block of R in registers (np <= 4032 with 2048 wavefronts) and its slices of
// p for the whole solve, and a workgroup owns at most one row block.  An
// iteration is then bound by the two exchanges between workgroups, each a
// trip to memory and back, so the exchanged words carry their own arrival:
// every word of y, of the partial products and of the parts of s_f holds
// MB_EMPTY until it is written, and its readers poll the words they need
// (poll_c) instead of waiting for a barrier and then reading: one trip per
// exchange instead of three (complete the stores; flag; read).  The sums of
// p.q, r.z and r.r go through the mailboxes of grid_allreduce2.
// Buffers rotate over four iterations.  A writer clears the words it wrote
// two iterations ago behind each publication: their readers have since
// published something the writer has read (an owner's y needs the partials,
// a partial needs its owners' y, p.q needs the parts of s_f).  The clear is
// complete (wait_vm) before the writer's next publication, which every reader
// reads before it polls for the one after, so no reader sees a word of four
// iterations ago.  Measured, evaluation, against blocks resident behind full
// barriers: 216 H2O 261 -> 240 us, H-(Gly)200-OH 726 -> 637, C300H602 650 ->
// 590; two exchanges of about 4 us each bound an iteration.  A block is half of
// a lane's 256 registers; 17 others are spilled without split fragments (80
// bytes of scratch per lane) and 36 with them (128 bytes).
__device__ __forceinline__ double poll_c(const double* p, int& bad, const int* flags) {
    const unsigned long long* u = reinterpret_cast<const unsigned long long*>(p);
    unsigned long long v = ld_cu(u);
    for (int it = 0; v == MB_EMPTY; ++it) {
        if (it > SPIN_MAX ||
            ((it & 63) == 63 && (__hip_atomic_load(flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & FLAG_SOLVE))) {
            bad = 1;
            return 0.0;
        }
        v = ld_cu(u);
    }
    return __longlong_as_double(v);
}
__device__ inline void clear_c(double* p) { st_cu(reinterpret_cast<unsigned long long*>(p), MB_EMPTY); }
// mailbox value of exchange j (thread 0 of the workgroup)
__device__ inline void mb_put(unsigned long long* mb, int j, double v0, double v1) {
    unsigned long long* const own = mb + (4 * blockIdx.x + (j & 3)) * MB_LINE;
    unsigned long long* const old = mb + (4 * blockIdx.x + ((j + 2) & 3)) * MB_LINE;
    wait_vm();
    st_cu(own, __double_as_longlong(v0));
    st_cu(own + 1, __double_as_longlong(v1));
    st_cu(old, MB_EMPTY);
    st_cu(old + 1, MB_EMPTY);
}
// every workgroup's values of exchange j, summed over each of the first four
// wavefronts into rd[w], rd[4 + w]
__device__ inline void mb_get(const unsigned long long* mb, int j, double* rd, int& bad, const int* flags) {
    const int tid = threadIdx.x;
    if (tid >= 256) return;
    double u0 = 0.0, u1 = 0.0;
    if (tid < (int)gridDim.x) {
        const double* in = reinterpret_cast<const double*>(mb + (4 * tid + (j & 3)) * MB_LINE);
        u0 = poll_c(in, bad, flags);
        u1 = poll_c(in + 1, bad, flags);
    }
    u0 = wave_sum(u0);
    u1 = wave_sum(u1);
    if ((tid & 63) == 0) {
        rd[tid >> 6] = u0;
        rd[4 + (tid >> 6)] = u1;
    }
}

template <bool SM>
__global__ __launch_bounds__(PCG_THREADS) void k_eeq_pcg_res(PcgArgs a) {
    __shared__ double red[2][8], redq[PCG_WAVES], red2[PCG_WAVES];
    __shared__ double qs[PCG_WAVES][NB];
    __shared__ double rb[NB], wb[NB], zb[NB];
    __shared__ double Lc[NB * LDC];
    __shared__ __align__(16) double pw[PCG_WAVES][2][NB];
    __shared__ double sfs[SM ? SM_MAXF : 1], sig[SM ? SM_MAXF : 1], pbuf[SM ? SM_MAXP : 1];
    if (__hip_atomic_load(a.flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & FLAG_CHOL) {
        if (blockIdx.x == 0 && a.lu_w && eeq_lu<PCG_THREADS>(a.np, a.nr, 0, a.Rp, a.b, a.lu_w, a.x) && threadIdx.x == 0)
            atomicOr(a.flags, FLAG_LU);
        return;
    }
    const int np = a.np, G = gridDim.x, g = blockIdx.x, nbk = np / NB;
    const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63;
    const bool owner = g < nbk;  // of row block g
    const int T = nbk * (nbk + 1) / 2;
    // block of this wavefront: workgroup g takes every G-th
    const int t = wv * G + g;
    const bool has = t < T;
    int I = 0, J = 0;
    double rv[8][8];
    if (has) {
        packed_block(t, I, J);
        load_block(rv, a.Rp + (size_t)t * NB * NB, l);
    }
    const int cend = 2 * (l & 7) + ((l >> 3) & 1) + 16 * (l >> 4);
    const size_t pstride = (size_t)nbk * np;
    const int npc = SM ? a.poff[a.nsf] : 0;
    double wI = 0.0, wJ = 0.0, wO = 0.0;  // w and fragment of this lane's rows
    int fI = -1, fJ = -1, fO = -1, s01 = 0;
    if (SM) {
        if (has) {
            fI = a.rowf[I * NB + l];
            fJ = a.rowf[J * NB + l];
            if (fI >= 0) wI = a.w[I * NB + l];
            if (fJ >= 0) wJ = a.w[J * NB + l];
        }
        if (owner) {
            fO = a.rowf[g * NB + l];
            if (fO >= 0) wO = a.w[g * NB + l];
            s01 = a.smon[g];
        }
        for (int f = tid; f < a.nsf; f += PCG_THREADS) {
            double s = 1.0 / a.all[f];
            for (int k = a.poff[f]; k < a.poff[f + 1]; ++k) s += a.w1[a.pidx[k]];
            sig[f] = 1.0 / s;
        }
    }
    if (owner)
        for (int e = tid; e < NB * NB; e += PCG_THREADS) Lc[(e >> 6) * LDC + (e & 63)] = a.Lj[(size_t)g * NB * NB + e];
    double ro = 0.0, xo = 0.0, po = 0.0;  // the owner's rows of r, x and p (wavefront 0)
    if (owner && tid < NB) {
        ro = a.b[g * NB + tid];
        rb[tid] = ro;
    }
    __syncthreads();
    int nex = 0, bad = 0;  // mailbox exchanges published
    // y of buffer k from rb, published with its parts of s_f and the sums r.y, r.r
    auto publish = [&](int k) {
        if (owner) bjacobi_apply(Lc, LDC, rb, wb, zb);
        if (tid < NB) {
            double rz = 0.0, rr = 0.0;
            if (owner) {
                const double y = zb[tid];
                wait_vm();
                st_c(a.z + (size_t)(k & 3) * np + g * NB + tid, y);
                if (SM) {
                    const int rf = s01 ? fO : -1;
                    const double s0 = wave_sum(rf >= 0 && !(rf & 1) ? y : 0.0);
                    const double s1 = wave_sum(rf >= 0 && (rf & 1) ? y : 0.0);
                    if (tid < 2) {
                        st_c(a.sp + (size_t)(k & 3) * 2 * nbk + 2 * g + tid, tid ? s1 : s0);
                        clear_c(a.sp + (size_t)((k + 2) & 3) * 2 * nbk + 2 * g + tid);
                    }
                }
                clear_c(a.z + (size_t)((k + 2) & 3) * np + g * NB + tid);
                rz = wave_sum(ro * y);
                rr = wave_sum(ro * ro);
            }
            if (tid == 0) mb_put(a.mb, nex, rz, rr);
        }
        ++nex;
    };
    publish(0);
    double rzold = 1.0, pir = 0.0, pjr = 0.0, bb = 0.0;
    int it = 0;
    bool done = false;
    for (;; ++it) {
        // y of this lane's rows and columns, the parts of s_f, the sums
        const double* yb = a.z + (size_t)(it & 3) * np;
        double yI = 0.0, yJ = 0.0;
        if (has) {
            yJ = poll_c(yb + J * NB + l, bad, a.flags);
            yI = poll_c(yb + I * NB + l, bad, a.flags);
        }
        if (SM)
            for (int k = tid; k < npc; k += PCG_THREADS)
                pbuf[k] = poll_c(a.sp + (size_t)(it & 3) * 2 * nbk + a.pidx[k], bad, a.flags);
        mb_get(a.mb, nex - 1, red[0], bad, a.flags);
        if (__syncthreads_or(bad)) break;
        double rz = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
        const double rr = (red[0][4] + red[0][5]) + (red[0][6] + red[0][7]);
        if (it == 0) {
            bb = rr;
            done = !(bb > 0.0);
        } else {
            done = rr <= a.tol2 * bb;
        }
        if (done || it >= a.maxit) break;
        if (SM) {
            rz -= sm_sums<PCG_THREADS>(a, sfs, sig, pbuf, red2);
            if (fI >= 0) yI -= sfs[fI >> 1] * wI;
            if (fJ >= 0) yJ -= sfs[fJ >> 1] * wJ;
        }
        const double beta = it == 0 ? 0.0 : rz / rzold;
        rzold = rz;
        if (owner && tid < NB) {
            double z = zb[tid];
            if (SM && fO >= 0) z -= sfs[fO >> 1] * wO;
            po = z + beta * po;
        }
        double lpq = 0.0;
        if (has) {
            pjr = yJ + beta * pjr;
            pir = yI + beta * pir;
            pw[wv][0][l] = pir;
            pw[wv][1][l] = pjr;
            __builtin_amdgcn_wave_barrier();
            double rs, cs, pjc;
            block_products(rv, pw[wv], l, I != J, rs, cs, pjc);
            double* const pb = a.part + (size_t)(it & 3) * pstride;
            double* const pc = a.part + (size_t)((it + 2) & 3) * pstride;
            wait_vm();
            st_c(pb + ((size_t)I * nbk + J) * NB + l, rs);
            lpq = pir * rs;
            if (I != J) {
                st_c(pb + ((size_t)J * nbk + I) * NB + cend, cs);
                lpq += pjc * cs;
                clear_c(pc + ((size_t)J * nbk + I) * NB + cend);
            }
            clear_c(pc + ((size_t)I * nbk + J) * NB + l);
        }
        lpq = wave_sum(lpq);
        if (l == 0) redq[wv] = lpq;
        __syncthreads();
        if (tid == 0) {
            double v = redq[0];
#pragma unroll
            for (int w = 1; w < PCG_WAVES; ++w) v += redq[w];
            mb_put(a.mb, nex, v, 0.0);
        }
        ++nex;
        // owners: the products of their rows (thread (row l, part wv): Y = wv, wv + PCG_WAVES, ..)
        if (owner) {
            const double* pr = a.part + (size_t)(it & 3) * pstride + (size_t)g * nbk * NB + l;
            double t8[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) t8[u] = ld_c(pr + (size_t)min(wv + PCG_WAVES * u, nbk - 1) * NB);
            double acc = 0.0;
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (wv + PCG_WAVES * u < nbk) {
                    if ((unsigned long long)__double_as_longlong(t8[u]) == MB_EMPTY)
                        t8[u] = poll_c(pr + (size_t)(wv + PCG_WAVES * u) * NB, bad, a.flags);
                    acc += t8[u];
                }
            qs[wv][l] = acc;
        }
        mb_get(a.mb, nex - 1, red[1], bad, a.flags);
        if (__syncthreads_or(bad)) break;
        if (owner) {
            const double alpha = rz / ((red[1][0] + red[1][1]) + (red[1][2] + red[1][3]));
            if (tid < NB) {
                double qv = qs[0][tid];
#pragma unroll
                for (int w = 1; w < PCG_WAVES; ++w) qv += qs[w][tid];
                xo += alpha * po;
                ro -= alpha * qv;
                rb[tid] = ro;
            }
            __syncthreads();
        }
        publish(it + 1);
    }
    if (owner && tid < NB) a.x[g * NB + tid] = xo;
    if (g == 0 && tid == 0) a.iters[0] = it;
    if (!done && tid == 0) atomicOr(a.flags, FLAG_SOLVE);
}

// And with everything in one workgroup (np <= 64 NBK_ONE): the blocks in the
// registers of one wavefront each, vectors and factors in LDS, a barrier of
// the workgroup where the others cross the chip.  122 atoms: evaluation 297 ->
// 169 us; an iteration takes 4.3 us there (15: 64 us) and 5.7 with three row
// blocks, which fill the registers and LDS of a compute unit.
constexpr int NBK_ONE = 3;
template <int NBK>
__global__ __launch_bounds__(PCG_THREADS) void k_eeq_pcg_one(PcgArgs a) {
    constexpr int NT = NBK * (NBK + 1) / 2, N = NBK * NB;
    __shared__ double Ls[NBK][NB * LDC];
    __shared__ double part[NBK][NBK][NB], pv[N], rvec[N], wv_[N], zv[N], redq[NT], red[2][NBK];
    __shared__ __align__(16) double pw[NT][2][NB];
    if (__hip_atomic_load(a.flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & FLAG_CHOL) {
        if (a.lu_w && eeq_lu<PCG_THREADS>(a.np, a.nr, 0, a.Rp, a.b, a.lu_w, a.x) && threadIdx.x == 0)
            atomicOr(a.flags, FLAG_LU);
        return;
    }
    const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63;
    int I = 0, J = 0;
    double rv[8][8];
    if (wv < NT) {
        packed_block(wv, I, J);
        load_block(rv, a.Rp + (size_t)wv * NB * NB, l);
    }
    for (int e = tid; e < NBK * NB * NB; e += PCG_THREADS)
        Ls[e >> 12][((e >> 6) & 63) * LDC + (e & 63)] = a.Lj[e];
    double r = 0.0, x = 0.0, p = 0.0, z = 0.0;  // row tid
    if (tid < N) {
        r = a.b[tid];
        rvec[tid] = r;
    }
    __syncthreads();
    const int half = tid >> 8, t = (tid >> 2) & 63, q = tid & 3;
    // z = M^-1 r (two blocks at a time), and the sums r.z and r.r
    auto precond = [&](double& rz, double& rr) {
#pragma unroll
        for (int pass = 0; pass < 2; ++pass) {
            const double* in = pass ? wv_ : rvec;
            double* out = pass ? zv : wv_;
#pragma unroll
            for (int b0 = 0; b0 < NBK; b0 += 2) {
                const int b = b0 + half;
                if (b < NBK) {
                    double s = 0.0;
#pragma unroll
                    for (int u = 0; u < NB / 4; ++u)
                        s += (pass ? Ls[b][(4 * u + q) * LDC + t] : Ls[b][t * LDC + 4 * u + q]) * in[b * NB + 4 * u + q];
                    s += __shfl_xor(s, 1);
                    s += __shfl_xor(s, 2);
                    if (q == 0) out[b * NB + t] = s;
                }
            }
            __syncthreads();
        }
        if (tid < N) {
            z = zv[tid];
            const double s0 = wave_sum(r * z), s1 = wave_sum(r * r);
            if (l == 0) {
                red[0][wv] = s0;
                red[1][wv] = s1;
            }
        }
        __syncthreads();
        rz = red[0][0];
        rr = red[1][0];
#pragma unroll
        for (int w = 1; w < NBK; ++w) {
            rz += red[0][w];
            rr += red[1][w];
        }
    };
    double rz, bb;
    precond(rz, bb);
    double beta = 0.0;
    int it = 0;
    bool done = !(bb > 0.0);
    for (; !done && it < a.maxit; ++it) {
        if (tid < N) {
            p = z + beta * p;
            pv[tid] = p;
        }
        __syncthreads();
        double lpq = 0.0;
        if (wv < NT) {
            const double pil = pv[I * NB + l], pjl = pv[J * NB + l];
            pw[wv][0][l] = pil;
            pw[wv][1][l] = pjl;
            __builtin_amdgcn_wave_barrier();
            double rs, cs, pjc;
            block_products(rv, pw[wv], l, I != J, rs, cs, pjc);
            part[I][J][l] = rs;
            lpq = pil * rs;
            if (I != J) {
                part[J][I][2 * (l & 7) + ((l >> 3) & 1) + 16 * (l >> 4)] = cs;
                lpq += pjc * cs;
            }
            lpq = wave_sum(lpq);
            if (l == 0) redq[wv] = lpq;
        }
        __syncthreads();
        double pq = redq[0];
#pragma unroll
        for (int w = 1; w < NT; ++w) pq += redq[w];
        const double alpha = rz / pq;
        if (tid < N) {
            double qv = part[wv][0][l];
#pragma unroll
            for (int c = 1; c < NBK; ++c) qv += part[wv][c][l];
            x += alpha * p;
            r -= alpha * qv;
            rvec[tid] = r;
        }
        __syncthreads();
        double rz2, rr;
        precond(rz2, rr);
        beta = rz2 / rz;
        rz = rz2;
        done = rr <= a.tol2 * bb;
    }
    if (tid < N) a.x[tid] = x;
    if (tid == 0) {
        a.iters[0] = it;
        if (!done) atomicOr(a.flags, FLAG_SOLVE);
    }
}

// ---------------------------------------------------------------------------
// K4b: mixed-precision EEQ.  The reduced matrix R is factored in FP32 and the
// FP64 solution is won back by iterative refinement against the FP64 R:
//   x = 0, r = b;  repeat: x += L32^-T L32^-1 r;  r = b - R x.
// ---------------------------------------------------------------------------
// FP32 copy of the lower tiles (bi >= bj) of R; tile t numbered row by row.
__global__ __launch_bounds__(256) void k_lower_to_f32(int np, const double* __restrict__ A, float* __restrict__ A32) {
    const int t = blockIdx.x;
    int bi = (int)((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
    while ((bi + 1) * (bi + 2) / 2 <= t) ++bi;
    while (bi * (bi + 1) / 2 > t) --bi;
    const int bj = t - bi * (bi + 1) / 2;
    _Pragma("unroll") for (int u_ = 0, e = (int)threadIdx.x; u_ < NB * NB / 256; ++u_, e += 256) {
        const size_t o = (size_t)(bi * NB + e / NB) * np + bj * NB + e % NB;
        A32[o] = (float)A[o];
    }
}

// Partial products of the symmetric matvec y = R x from the lower tiles of R:
// workgroup (I, sp) sums, for the 64 rows of block row I, the tiles J = sp,
// sp + nsplit, ...: (I, J) by rows when J < I, the diagonal tile completed
// symmetrically from its lower triangle, and (J, I)^T by columns when J > I.
// part[sp][row]; summed in a fixed order by k_eeq_resid.
__global__ __launch_bounds__(256) void k_symv_part(int np, int nsplit, const double* __restrict__ R,
                                                   const double* __restrict__ x, double* __restrict__ part) {
    __shared__ double Tt[NB][NB + 1];
    __shared__ double xs[NB];
    const int I = blockIdx.x, sp = blockIdx.y, nbk = np / NB;
    const int tid = threadIdx.x, t = tid >> 2, q = tid & 3;
    double acc = 0.0;
    for (int J = sp; J < nbk; J += nsplit) {
        __syncthreads();
        const bool below = J > I;
        const int r0 = below ? J * NB : I * NB, c0 = below ? I * NB : J * NB;
        _Pragma("unroll") for (int u_ = 0, e = tid; u_ < NB * NB / 256; ++u_, e += 256) {
            const int r = e / NB, c = e % NB;
            // diagonal tile: symmetric completion from its lower triangle
            Tt[r][c] = (J == I && c > r) ? R[(size_t)(r0 + c) * np + c0 + r] : R[(size_t)(r0 + r) * np + c0 + c];
        }
        if (tid < NB) xs[tid] = x[J * NB + tid];
        __syncthreads();
        if (!below) {
#pragma unroll
            for (int u = 0; u < NB / 4; ++u) acc += Tt[t][4 * u + q] * xs[4 * u + q];
        } else {
#pragma unroll
            for (int u = 0; u < NB / 4; ++u) acc += Tt[4 * u + q][t] * xs[4 * u + q];
        }
    }
    acc += __shfl_xor(acc, 1);
    acc += __shfl_xor(acc, 2);
    if (q == 0) part[(size_t)sp * np + I * NB + t] = acc;
}

// r = b - sum_sp part[sp] (fixed order); rf = (float) r for the next FP32 solve.
__global__ __launch_bounds__(256) void k_eeq_resid(int np, int nsplit, const double* __restrict__ part,
                                                   const double* __restrict__ b, double* __restrict__ r,
                                                   float* __restrict__ rf) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    double y = 0.0;
    for (int sp = 0; sp < nsplit; ++sp) y += part[(size_t)sp * np + i];
    const double v = b[i] - y;
    r[i] = v;
    rf[i] = (float)v;
}

// x (+)= d for the FP32 correction d; first == 1 starts from x = d.
__global__ __launch_bounds__(256) void k_refine_add(int np, int first, const float* __restrict__ d,
                                                    double* __restrict__ x) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= np) return;
    x[i] = first ? (double)d[i] : x[i] + (double)d[i];
}

__global__ __launch_bounds__(256) void k_to_f32(int n, const double* __restrict__ a, float* __restrict__ b) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] = (float)a[i];
}

// ---------------------------------------------------------------------------
// K5: charges, self energy (ff_workspace.cpp:426-449) and qtmp (:459-507)
// ---------------------------------------------------------------------------
// Charges from the reduced solution, one thread per atom; the last atom of a
// fragment takes qp minus the sum over the others, formed by a wavefront per
// fragment (workgroups natb ..: lanes stride the fragment's atoms, fixed
// butterfly) that also finishes that atom.
struct ChargeArgs {
    int n, nfrag, natb;
    const int *frag_off, *frag_atoms, *red_of;
    const double *qp, *p, *chi_base, *cnf, *gam, *alp, *cn;
    double *q, *e_self, *qtmp;
};
__device__ inline void charge_atom(const ChargeArgs& a, int i, double qi) {
    a.q[i] = qi;
    const double c = a.cn[i];
    const double chi = a.chi_base[i] + a.cnf[i] * sqrt(fmax(c, 0.0));
    a.e_self[i] = -qi * chi + 0.5 * qi * qi * (a.gam[i] + TSQRT2PI_SELF / sqrt(a.alp[i]));
    a.qtmp[i] = qi * a.cnf[i] / (2.0 * sqrt(fmax(c, 0.0)) + 1e-16);
}
__global__ __launch_bounds__(256) void k_charges(ChargeArgs a) {
    if ((int)blockIdx.x < a.natb) {
        const int i = blockIdx.x * 256 + threadIdx.x;
        if (i >= a.n) return;
        const int ri = a.red_of[i];
        if (ri >= 0) charge_atom(a, i, a.qp[i] + a.p[ri]);
        return;
    }
    const int f = (blockIdx.x - a.natb) * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (f >= a.nfrag) return;
    double s = 0.0;
    for (int k = a.frag_off[f] + lane; k < a.frag_off[f + 1]; k += 64) {
        const int ra = a.red_of[a.frag_atoms[k]];
        if (ra >= 0) s += a.p[ra];
    }
    s = wave_sum(s);
    if (lane == 0) {
        const int i = a.frag_atoms[a.frag_off[f + 1] - 1];
        charge_atom(a, i, a.qp[i] - s);
    }
}

// ---------------------------------------------------------------------------
// K6: pair terms.  Row atom i per thread, partners j staged in LDS tiles.
//   Coulomb  (r <= 100)  ff_workspace_gfnff.cpp:850-898
//   D4       (r <= 50)   :715-767 with C6 from the current Gaussian weights
//   repulsion (r <= 20)  :814-842 with the element-pair factor; bonded and
//                        1,3/1,4 H-H pairs are corrected by k_atom_tail
// Each pair is evaluated from both sides; a row keeps half of each pair
// energy and its own full gradient and dE/dCN, so no atomics are needed.
// ---------------------------------------------------------------------------
struct PairArgs {
    int n, nelem;
    const double* x;
    const double* q;
    const double* alp;
    const double* gw;
    const double* dgw;
    const double* zeta;
    const double* szr;
    const double* anb;
    const double* repz;
    const int* Z;
    const int* elem;
    const int* nref;
    const int* metal;
    const double* c6ref;
    const double* h;  // [n][nelem][7] D4 half contraction (k_terms)
    const double* dh;
    const int* mol_of;   // batches: molecule of each atom (nullptr: one molecule)
    const int* mol_off;  // batches: atom offsets of the molecules
    double* g;        // [3n]
    double* dEdcn;    // [n]
    double* e_coul;   // [n]
    double* e_disp;   // [n]
    double* e_rep;    // [n]
};

__device__ inline double rep_ff(int zi, int zj, int mi, int mj) {
    if (zi == 1 && zj == 1) return 0.6290;
    if ((zi == 1 && mj > 0) || (zj == 1 && mi > 0)) return 0.85;
    if ((zi == 1 && zj == 6) || (zj == 1 && zi == 6)) return 0.91;
    if ((zi == 1 && zj == 8) || (zj == 1 && zi == 8)) return 1.04;
    return 1.0;
}

// Partner range of a pair-kernel workgroup: the j chunk of a single molecule,
// or, in a batch, the union of the molecules of the workgroup's rows (each
// row then keeps only partners of its own molecule).
__device__ inline void pair_range(const PairArgs& a, int cj, int& j0, int& j1) {
    if (!a.mol_of) {
        j0 = blockIdx.y * cj;
        j1 = min(a.n, j0 + cj);
    } else {
        const int first = blockIdx.x * TILE, last = min(a.n, first + TILE) - 1;
        j0 = a.mol_off[a.mol_of[first]];
        j1 = a.mol_off[a.mol_of[last] + 1];
    }
}

// D4 half contraction per atom i and partner element e:
//   h[i][e][b]  = sum_a gw_i[a]  c6ref[ei, e, a, b]
//   dh[i][e][b] = sum_a dgw_i[a] c6ref[ei, e, a, b]
// so that C6_ij = h[i][ej] . gw_j and dC6_ij/dCN_i = dh[i][ej] . gw_j
// (the reference's half-contraction, d4param_generator.cpp:1235).
__device__ __forceinline__ void d4_half_entry(int t, int n, int ne, const int* __restrict__ elem,
                                              const int* __restrict__ nref, const double* __restrict__ c6ref,
                                              const double* __restrict__ gw, const double* __restrict__ dgw,
                                              double* __restrict__ h, double* __restrict__ dh) {
    if (t >= n * ne) return;
    int i = t / ne, e = t % ne;
    int ei = elem[i], nri = nref[ei];
    const double* c = c6ref + (size_t)(ei * ne + e) * 49;
    double hb[7] = {}, dhb[7] = {};
    for (int aa = 0; aa < nri; ++aa) {
        double g = gw[(size_t)i * 7 + aa], dg = dgw[(size_t)i * 7 + aa];
#pragma unroll
        for (int bb = 0; bb < 7; ++bb) {
            hb[bb] += g * c[aa * 7 + bb];
            dhb[bb] += dg * c[aa * 7 + bb];
        }
    }
#pragma unroll
    for (int bb = 0; bb < 7; ++bb) {
        h[(size_t)t * 7 + bb] = hb[bb];
        dh[(size_t)t * 7 + bb] = dhb[bb];
    }
}

// Pair terms over full rows, split into j chunks so that the launch fills the
// chip: block (bx, by) owns rows i in [256 bx, 256 bx + 256) and partners j in
// [by cj, by cj + cj).  Each thread accumulates its row's gradient, dE/dCN and
// three energies over the chunk and writes them to part[by][k][i]; the chunks
// are summed in a fixed order by k_pairs_reduce (no atomics, deterministic).
// NE > 0: the D4 half contraction of row i for every partner element sits in
// registers and is selected by the partner's element, which is uniform across
// the wavefront because all lanes visit the same j; NE == 0: read from memory.
constexpr int PART_K = 7;
template <int NE>
__global__ __launch_bounds__(TILE) void k_pairs_part(PairArgs a, int cj, double* __restrict__ part) {
    __shared__ double sx[TILE], sy[TILE], sz[TILE], sq[TILE], sal[TILE], szt[TILE], ssz[TILE], san[TILE],
        srz[TILE];
    __shared__ double sgw[TILE * 7];
    __shared__ int sZ[TILE], sel[TILE], smt[TILE];
    const int n = a.n, ne = a.nelem;
    const int i = blockIdx.x * TILE + threadIdx.x;
    const bool act = i < n;
    int j0, j1;
    pair_range(a, cj, j0, j1);
    const int mlo = (a.mol_of && act) ? a.mol_off[a.mol_of[i]] : 0;
    const int mhi = (a.mol_of && act) ? a.mol_off[a.mol_of[i] + 1] : n;
    double3 xi = act ? ld3(a.x, i) : make_double3(0, 0, 0);
    double qi = act ? a.q[i] : 0.0, ali = act ? a.alp[i] : 1.0, zti = act ? a.zeta[i] : 0.0;
    double szi = act ? a.szr[i] : 0.0, ani = act ? a.anb[i] : 0.0, rzi = act ? a.repz[i] : 0.0;
    int zi = act ? a.Z[i] : 0, mi = act ? a.metal[i] : 0;
    constexpr int NH = NE > 0 ? NE * 7 : 1;
    double hr[NH], dhr[NH];
    if (NE > 0) {
#pragma unroll
        for (int k = 0; k < NH; ++k) {
            hr[k] = act ? a.h[(size_t)i * NH + k] : 0.0;
            dhr[k] = act ? a.dh[(size_t)i * NH + k] : 0.0;
        }
    }
    double gx = 0, gy = 0, gz = 0, dcn = 0, ec = 0, ed = 0, er = 0;
    for (int t0 = j0; t0 < j1; t0 += TILE) {
        __syncthreads();
        int j = t0 + threadIdx.x;
        if (j < j1) {
            sx[threadIdx.x] = a.x[3 * j];
            sy[threadIdx.x] = a.x[3 * j + 1];
            sz[threadIdx.x] = a.x[3 * j + 2];
            sq[threadIdx.x] = a.q[j];
            sal[threadIdx.x] = a.alp[j];
            szt[threadIdx.x] = a.zeta[j];
            ssz[threadIdx.x] = a.szr[j];
            san[threadIdx.x] = a.anb[j];
            srz[threadIdx.x] = a.repz[j];
            sZ[threadIdx.x] = a.Z[j];
            sel[threadIdx.x] = a.elem[j];
            smt[threadIdx.x] = a.metal[j];
#pragma unroll
            for (int r = 0; r < 7; ++r) sgw[threadIdx.x * 7 + r] = a.gw[(size_t)j * 7 + r];
        }
        __syncthreads();
        if (!act) continue;
        const int m = min(TILE, j1 - t0);
        for (int jj = 0; jj < m; ++jj) {
            if (t0 + jj == i || t0 + jj < mlo || t0 + jj >= mhi) continue;
            double dx = xi.x - sx[jj], dy = xi.y - sy[jj], dz = xi.z - sz[jj];
            double r2 = dx * dx + dy * dy + dz * dz;
            if (r2 > 10000.0) continue;  // beyond every pair cut-off (Coulomb 100 Bohr)
            double r = sqrt(r2);
            double dEdr = 0.0;
            // Coulomb
            if (r <= 100.0 && r >= 1e-10) {
                double gij = 1.0 / sqrt(ali + sal[jj]);
                double gr = gij * r;
                double ef, eg;
                erf_exp(gr, ef, eg);
                double qq = qi * sq[jj];
                ec += 0.5 * qq * ef / r;
                dEdr += qq * (gij * eg * (2.0 / 1.772453850905516) / r - ef / r2);
            }
            // D4 dispersion
            if (r <= 50.0 && r >= 1e-10) {
                const int ej = sel[jj];
                double c6 = 0.0, dci = 0.0;
                if (NE > 0) {
#pragma unroll
                    for (int e = 0; e < (NE > 0 ? NE : 1); ++e)
                        if (e == ej) {
#pragma unroll
                            for (int bb = 0; bb < 7; ++bb) {
                                double gj = sgw[jj * 7 + bb];
                                c6 += hr[e * 7 + bb] * gj;
                                dci += dhr[e * 7 + bb] * gj;
                            }
                        }
                } else {
                    const double* hp = a.h + ((size_t)i * ne + ej) * 7;
                    const double* dp = a.dh + ((size_t)i * ne + ej) * 7;
#pragma unroll
                    for (int bb = 0; bb < 7; ++bb) {
                        double gj = sgw[jj * 7 + bb];
                        c6 += hp[bb] * gj;
                        dci += dp[bb] * gj;
                    }
                }
                double r4r2 = 3.0 * szi * ssz[jj];
                double r0 = 0.58 * sqrt(r4r2) + 4.80;
                double r0s = r0 * r0;
                double zc = zti * szt[jj];
                double r6 = r2 * r2 * r2, r06 = r0s * r0s * r0s;
                double t6 = 1.0 / (r6 + r06), t8 = 1.0 / (r6 * r2 + r06 * r0s);
                double sum = t6 + 2.0 * r4r2 * t8;
                ed += 0.5 * (-c6 * sum * zc);
                double d6 = -6.0 * r2 * r2 * t6 * t6, d8 = -8.0 * r2 * r2 * r2 * t8 * t8;
                dEdr += -c6 * zc * (d6 + 2.0 * r4r2 * d8) * r;
                dcn -= dci * sum * zc;
            }
            // non-bonded repulsion (generic pair factor; bonded / 1,3 / 1,4
            // corrections follow in k_atom_tail)
            if (r2 <= 400.0 && r >= 1e-8) {
                double ff = rep_ff(zi, sZ[jj], mi, smt[jj]);
                double al = sqrt(ani * san[jj]) * ff;
                double ab = rzi * srz[jj] * 0.4270;
                double e = ab * exp(-al * r * sqrt(r)) / r;
                er += 0.5 * e;
                dEdr += -e / r - 1.5 * al * sqrt(r) * e;
            }
            double s = dEdr / r;
            gx += s * dx;
            gy += s * dy;
            gz += s * dz;
        }
    }
    if (!act) return;
    double* p = part + (size_t)blockIdx.y * PART_K * n + i;
    p[0] = gx;
    p[(size_t)n] = gy;
    p[(size_t)2 * n] = gz;
    p[(size_t)3 * n] = dcn;
    p[(size_t)4 * n] = ec;
    p[(size_t)5 * n] = ed;
    p[(size_t)6 * n] = er;
}

// Mixed-precision pair terms: the same rows, chunks and partial-sum layout as
// k_pairs_part.  Coordinate differences are formed in FP64 (no loss of the
// absolute positions), every term is evaluated in FP32 (hardware rsqrt, rcp,
// exp, erf paths) and the row sums are accumulated in FP64.
template <int NE>
__global__ __launch_bounds__(TILE) void k_pairs_part32(PairArgs a, int cj, double* __restrict__ part) {
    __shared__ double sx[TILE], sy[TILE], sz[TILE];
    __shared__ float sq[TILE], sal[TILE], szt[TILE], ssz[TILE], san[TILE], srz[TILE];
    __shared__ float sgw[TILE * 7];
    __shared__ int sZ[TILE], sel[TILE], smt[TILE];
    const int n = a.n, ne = a.nelem;
    const int i = blockIdx.x * TILE + threadIdx.x;
    const bool act = i < n;
    int j0, j1;
    pair_range(a, cj, j0, j1);
    const int mlo = (a.mol_of && act) ? a.mol_off[a.mol_of[i]] : 0;
    const int mhi = (a.mol_of && act) ? a.mol_off[a.mol_of[i] + 1] : n;
    const double3 xi = act ? ld3(a.x, i) : make_double3(0, 0, 0);
    const float qi = act ? (float)a.q[i] : 0.f, ali = act ? (float)a.alp[i] : 1.f;
    const float zti = act ? (float)a.zeta[i] : 0.f, szi = act ? (float)a.szr[i] : 0.f;
    const float ani = act ? (float)a.anb[i] : 0.f, rzi = act ? (float)a.repz[i] : 0.f;
    const int zi = act ? a.Z[i] : 0, mi = act ? a.metal[i] : 0;
    constexpr int NH = NE > 0 ? NE * 7 : 1;
    float hr[NH], dhr[NH];
    if (NE > 0) {
#pragma unroll
        for (int k = 0; k < NH; ++k) {
            hr[k] = act ? (float)a.h[(size_t)i * NH + k] : 0.f;
            dhr[k] = act ? (float)a.dh[(size_t)i * NH + k] : 0.f;
        }
    }
    double gx = 0, gy = 0, gz = 0, dcn = 0, ec = 0, ed = 0, er = 0;
    for (int t0 = j0; t0 < j1; t0 += TILE) {
        __syncthreads();
        const int j = t0 + threadIdx.x;
        if (j < j1) {
            sx[threadIdx.x] = a.x[3 * j];
            sy[threadIdx.x] = a.x[3 * j + 1];
            sz[threadIdx.x] = a.x[3 * j + 2];
            sq[threadIdx.x] = (float)a.q[j];
            sal[threadIdx.x] = (float)a.alp[j];
            szt[threadIdx.x] = (float)a.zeta[j];
            ssz[threadIdx.x] = (float)a.szr[j];
            san[threadIdx.x] = (float)a.anb[j];
            srz[threadIdx.x] = (float)a.repz[j];
            sZ[threadIdx.x] = a.Z[j];
            sel[threadIdx.x] = a.elem[j];
            smt[threadIdx.x] = a.metal[j];
#pragma unroll
            for (int r = 0; r < 7; ++r) sgw[threadIdx.x * 7 + r] = (float)a.gw[(size_t)j * 7 + r];
        }
        __syncthreads();
        if (!act) continue;
        const int m = min(TILE, j1 - t0);
        for (int jj = 0; jj < m; ++jj) {
            if (t0 + jj == i || t0 + jj < mlo || t0 + jj >= mhi) continue;
            const double dxd = xi.x - sx[jj], dyd = xi.y - sy[jj], dzd = xi.z - sz[jj];
            const double r2d = dxd * dxd + dyd * dyd + dzd * dzd;
            if (r2d > 10000.0) continue;  // beyond every pair cut-off (Coulomb 100 Bohr)
            const float r2 = (float)r2d;
            const float rinv = __builtin_amdgcn_rsqf(r2);
            const float r = r2 * rinv;
            float dEdr = 0.f;
            if (r2d >= 1e-20) {
                // Coulomb (r <= 100)
                const float gij = __builtin_amdgcn_rsqf(ali + sal[jj]);
                const float gr = gij * r;
                float ef, eg;
                erf_exp(gr, ef, eg);
                const float qq = qi * sq[jj];
                ec += (double)(0.5f * qq * ef * rinv);
                dEdr += qq * (gij * eg * 1.1283791671f * rinv - ef * rinv * rinv);
            }
            if (r2d <= 2500.0 && r2d >= 1e-20) {
                // D4 dispersion (r <= 50)
                const int ej = sel[jj];
                float c6 = 0.f, dci = 0.f;
                if (NE > 0) {
#pragma unroll
                    for (int e = 0; e < (NE > 0 ? NE : 1); ++e)
                        if (e == ej) {
#pragma unroll
                            for (int bb = 0; bb < 7; ++bb) {
                                const float gj = sgw[jj * 7 + bb];
                                c6 += hr[e * 7 + bb] * gj;
                                dci += dhr[e * 7 + bb] * gj;
                            }
                        }
                } else {
                    const double* hp = a.h + ((size_t)i * ne + ej) * 7;
                    const double* dp = a.dh + ((size_t)i * ne + ej) * 7;
#pragma unroll
                    for (int bb = 0; bb < 7; ++bb) {
                        const float gj = sgw[jj * 7 + bb];
                        c6 += (float)hp[bb] * gj;
                        dci += (float)dp[bb] * gj;
                    }
                }
                const float r4r2 = 3.f * szi * ssz[jj];
                const float r0 = 0.58f * __builtin_sqrtf(r4r2) + 4.80f;
                const float r0s = r0 * r0;
                const float zc = zti * szt[jj];
                const float r6 = r2 * r2 * r2, r06 = r0s * r0s * r0s;
                const float t6 = __builtin_amdgcn_rcpf(r6 + r06), t8 = __builtin_amdgcn_rcpf(r6 * r2 + r06 * r0s);
                const float sum = t6 + 2.f * r4r2 * t8;
                ed += (double)(0.5f * (-c6 * sum * zc));
                const float d6 = -6.f * r2 * r2 * t6 * t6, d8 = -8.f * r2 * r2 * r2 * t8 * t8;
                dEdr += -c6 * zc * (d6 + 2.f * r4r2 * d8) * r;
                dcn -= (double)(dci * sum * zc);
            }
            if (r2d <= 400.0 && r2d >= 1e-16) {
                // non-bonded repulsion (r <= 20), generic pair factor
                const float ff = (float)rep_ff(zi, sZ[jj], mi, smt[jj]);
                const float al = __builtin_sqrtf(ani * san[jj]) * ff;
                const float ab = rzi * srz[jj] * 0.4270f;
                const float sr = __builtin_sqrtf(r);
                const float e = ab * __expf(-al * r * sr) * rinv;
                er += (double)(0.5f * e);
                dEdr += -e * rinv - 1.5f * al * sr * e;
            }
            const double sgrad = (double)(dEdr * rinv);
            gx += sgrad * dxd;
            gy += sgrad * dyd;
            gz += sgrad * dzd;
        }
    }
    if (!act) return;
    double* p = part + (size_t)blockIdx.y * PART_K * n + i;
    p[0] = gx;
    p[(size_t)n] = gy;
    p[(size_t)2 * n] = gz;
    p[(size_t)3 * n] = dcn;
    p[(size_t)4 * n] = ec;
    p[(size_t)5 * n] = ed;
    p[(size_t)6 * n] = er;
}

// ---------------------------------------------------------------------------
// Pair terms with each unordered pair evaluated once (single molecules).
// Tiles of 64 rows x 64 columns of the lower triangle (row block R >= column
// block C, tile t = R (R + 1) / 2 + C), one wavefront each.  The column
// atoms' data sit in LDS; at step s lane l pairs its row atom with column
// (l + s) mod 64, so every lane meets every column once and the 64 lanes of
// one step touch 64 distinct columns: the column-side sums accumulate in LDS
// without atomics, in a fixed order.  Diagonal tiles take s = 1 .. 31 and,
// for l < 32, s = 32 (each unordered pair once).  Every tile writes its
// row-side and column-side sums (PART_K quantities x 64 atoms) to partials of
// its own, which k_pairs_sym_reduce adds per atom in a fixed order.  The pair
// arithmetic is that of k_pairs_part (T = double) or k_pairs_part32
// (T = float: FP64 coordinate differences, FP32 terms, every sum in FP64,
// row side and column side); the partner's dC6/dCN
// uses sum_b h_i[e_j][b] dgw_j[b], the transposed half contraction.
// FP64: the kernel issues instructions most of its time, and divisions and
// square roots were more than half of them.  One reciprocal square root
// serves r and every division by it, both damping denominators share one
// reciprocal, and the pair's square roots of per-atom parameters are
// products of the atoms'.  9000 atoms 497 -> 360 us, 4096 molecules 1.63 ->
// 1.2 ms.
constexpr int PS_B = 64;
__device__ inline float ps_rsqrt(float v) { return __builtin_amdgcn_rsqf(v); }
__device__ inline double ps_rsqrt(double v) { return rsqrt_c(v); }
__device__ inline float ps_sqrt(float v) { return __builtin_sqrtf(v); }
__device__ inline double ps_sqrt(double v) { return v * rsqrt_c(v); }
__device__ inline float ps_rcp(float v) { return __builtin_amdgcn_rcpf(v); }
__device__ inline double ps_rcp(double v) { return rcp_c(v); }
__device__ inline float ps_exp(float v) { return __expf(v); }
__device__ inline double ps_exp(double v) { return exp(v); }

// terms: PT_COUL | PT_DISP | PT_REP select the pair terms evaluated (all three
// in one pass, or the charge-independent dispersion and repulsion before the
// EEQ solve and the Coulomb term after it, into separate partials).
//
// split: the 64 steps of a tile are dealt in equal runs to split wavefronts
// (blocks t * split .. t * split + split - 1), each with partials of its own.
// A step is a chain of reciprocal square roots, the D4 contraction of every
// element among the step's columns and, near by, erf and exp: about 1.1 us when
// one wavefront has its SIMD to itself (122 atoms, both types: 80 us of 64 steps,
// 18 of 8), so a launch of few tiles is bound by that chain and not by
// throughput (ps_split).
constexpr int PT_COUL = 1, PT_DISP = 2, PT_REP = 4, PT_ALL = 7;
template <typename T, int NE>
__global__ __launch_bounds__(PS_B) void k_pairs_sym(PairArgs a, double* __restrict__ part,
                                                    const int4* __restrict__ tiles, int terms, int split) {
    __shared__ double cx[PS_B], cy[PS_B], cz[PS_B];
    __shared__ T cq[PS_B], cal[PS_B], czt[PS_B], csz[PS_B], can[PS_B], crz[PS_B];
    __shared__ T cgw[7][PS_B], cdgw[7][PS_B];
    constexpr bool F64 = sizeof(T) == 8;
    __shared__ T crs[F64 ? PS_B : 1];
    __shared__ int czem[PS_B];        // Z | element << 8 | metal << 16
    __shared__ double acc[PART_K][PS_B];  // column-side sums of this tile, in FP64 on both paths
    const int t = blockIdx.x / split, sub = blockIdx.x % split, l = threadIdx.x;
    // the tile's molecule (atoms a0 .. a0 + n - 1) and its row and column blocks
    int a0 = 0, n = a.n, R, C;
    if (tiles) {
        const int4 tt = tiles[t];
        a0 = tt.x;
        n = tt.y;
        R = tt.z;
        C = tt.w;
    } else {
        R = (int)((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
        while ((R + 1) * (R + 2) / 2 <= t) ++R;
        while (R * (R + 1) / 2 > t) --R;
        C = t - R * (R + 1) / 2;
    }
    const int ne = a.nelem;
    const int i = a0 + R * PS_B + l, jl = a0 + C * PS_B + l;
    const bool acti = R * PS_B + l < n;
    {
        const bool actj = C * PS_B + l < n;
        const int js = actj ? jl : a0;
        cx[l] = a.x[3 * js];
        cy[l] = a.x[3 * js + 1];
        cz[l] = a.x[3 * js + 2];
        cq[l] = (T)a.q[js];
        cal[l] = (T)a.alp[js];
        czt[l] = (T)a.zeta[js];
        // FP64: the pair's square roots as products of the atoms' (rsz, ran)
        csz[l] = (T)a.szr[js];
        can[l] = F64 ? (T)sqrt(a.anb[js]) : (T)a.anb[js];
        if (F64) crs[l] = (T)sqrt(a.szr[js]);
        crz[l] = (T)a.repz[js];
        czem[l] = a.Z[js] | (a.elem[js] << 8) | (a.metal[js] << 16);
#pragma unroll
        for (int r = 0; r < 7; ++r) {
            cgw[r][l] = (T)a.gw[(size_t)js * 7 + r];
            cdgw[r][l] = (T)a.dgw[(size_t)js * 7 + r];
        }
#pragma unroll
        for (int k = 0; k < PART_K; ++k) acc[k][l] = 0.0;
    }
    __syncthreads();
    const int is = acti ? i : a0;
    const double3 xi = ld3(a.x, is);
    const T qi = (T)a.q[is], ali = (T)a.alp[is], zti = (T)a.zeta[is], szi = (T)a.szr[is];
    const T ani = F64 ? (T)sqrt(a.anb[is]) : (T)a.anb[is], rzi = (T)a.repz[is];
    const T rsi = F64 ? (T)(0.58 * 1.7320508075688772 * sqrt(a.szr[is])) : T(0);  // 0.58 sqrt(3 szr_i)
    const int zi = a.Z[is], mi = a.metal[is];
    constexpr int NH = NE > 0 ? NE * 7 : 1;
    T hr[NH], dhr[NH];
    if (NE > 0) {
#pragma unroll
        for (int k = 0; k < NH; ++k) {
            hr[k] = (T)a.h[(size_t)is * NH + k];
            dhr[k] = (T)a.dh[(size_t)is * NH + k];
        }
    }
    const int jmax = min(PS_B, n - C * PS_B);  // columns present in this tile
    const bool diag = R == C;
    // this wavefront's run of the steps 1 .. 32 (diagonal tile) or 0 .. 63
    const int run = (diag ? PS_B / 2 : PS_B) / split;
    const int s0 = (diag ? 1 : 0) + sub * run;
    const int s1 = min(s0 + run - 1, diag ? (l < 32 ? 32 : 31) : PS_B - 1);
    double gx = 0, gy = 0, gz = 0, dcn = 0, ec = 0, ed = 0, er = 0;
    for (int s = s0; s <= s1; ++s) {
        __atomic_signal_fence(__ATOMIC_SEQ_CST);  // keep the LDS updates of consecutive steps in order
        const int jj = (l + s) & (PS_B - 1);
        if (!acti || jj >= jmax) continue;
        const double dxd = xi.x - cx[jj], dyd = xi.y - cy[jj], dzd = xi.z - cz[jj];
        const double r2d = dxd * dxd + dyd * dyd + dzd * dzd;
        if (r2d > ((terms & PT_COUL) ? 10000.0 : 2500.0)) continue;  // beyond every pair cut-off (Coulomb 100 Bohr)
        T dEdr = 0, hec = 0, hed = 0, her = 0, dci = 0, dcj = 0;
        const T r2 = (T)r2d;
        const T rinv = ps_rsqrt(r2), r = r2 * rinv;
        // cut-offs on the squares: r is within rounding of the root, not the rounded root
        const bool coul = (terms & PT_COUL) && r2d >= 1e-20;
        const bool disp = (terms & PT_DISP) && r2d <= 2500.0 && r2d >= 1e-20;
        const bool rep = (terms & PT_REP) && r2d <= 400.0 && r2d >= 1e-16;
        if (coul) {
            const T gij = ps_rsqrt(ali + cal[jj]);
            const T gr = gij * r;
            T ef, eg;
            erf_exp(gr, ef, eg);
            const T qq = qi * cq[jj];
            hec = T(0.5) * qq * ef * rinv;
            dEdr += qq * (gij * eg * (F64 ? T(2.0 / 1.772453850905516) : T(1.1283791671)) * rinv - ef * rinv * rinv);
        }
        if (disp) {
            const int ej = (czem[jj] >> 8) & 0xff;
            T c6 = 0;
            if (NE > 0) {
#pragma unroll
                for (int e = 0; e < (NE > 0 ? NE : 1); ++e)
                    if (e == ej) {
#pragma unroll
                        for (int bb = 0; bb < 7; ++bb) {
                            const T gj = cgw[bb][jj], dgj = cdgw[bb][jj];
                            c6 += hr[e * 7 + bb] * gj;
                            dci += dhr[e * 7 + bb] * gj;
                            dcj += hr[e * 7 + bb] * dgj;
                        }
                    }
            } else {
                const double* hp = a.h + ((size_t)is * ne + ej) * 7;
                const double* dp = a.dh + ((size_t)is * ne + ej) * 7;
#pragma unroll
                for (int bb = 0; bb < 7; ++bb) {
                    const T gj = cgw[bb][jj], dgj = cdgw[bb][jj];
                    c6 += (T)hp[bb] * gj;
                    dci += (T)dp[bb] * gj;
                    dcj += (T)hp[bb] * dgj;
                }
            }
            const T r4r2 = T(3) * szi * csz[jj];
            const T r0 = F64 ? rsi * crs[jj] + T(4.80) : T(0.58) * ps_sqrt(r4r2) + T(4.80);
            const T r0s = r0 * r0;
            const T zc = zti * czt[jj];
            const T r6 = r2 * r2 * r2, r06 = r0s * r0s * r0s;
            T t6, t8;
            if (F64) {  // both reciprocals from one
                const T p6 = r6 + r06, p8 = r6 * r2 + r06 * r0s, pi = ps_rcp(p6 * p8);
                t6 = p8 * pi;
                t8 = p6 * pi;
            } else {
                t6 = ps_rcp(r6 + r06);
                t8 = ps_rcp(r6 * r2 + r06 * r0s);
            }
            const T sum = t6 + T(2) * r4r2 * t8;
            hed = T(0.5) * (-c6 * sum * zc);
            const T d6 = T(-6) * r2 * r2 * t6 * t6, d8 = T(-8) * r2 * r2 * r2 * t8 * t8;
            dEdr += -c6 * zc * (d6 + T(2) * r4r2 * d8) * r;
            dci = dci * sum * zc;
            dcj = dcj * sum * zc;
        }
        if (rep) {
            const T ff = (T)rep_ff(zi, czem[jj] & 0xff, mi, czem[jj] >> 16);
            const T al = (F64 ? ani * can[jj] : ps_sqrt(ani * can[jj])) * ff;
            const T ab = rzi * crz[jj] * T(0.4270);
            const T sr = ps_sqrt(r);
            const T e = ab * ps_exp(-al * r * sr) * rinv;
            dEdr += -e * rinv - T(1.5) * al * sr * e;
            her = T(0.5) * e;
        }
        const double sg = (double)(dEdr * rinv);
        const double fx = sg * dxd, fy = sg * dyd, fz = sg * dzd;
        gx += fx;
        gy += fy;
        gz += fz;
        ec += (double)hec;
        ed += (double)hed;
        er += (double)her;
        dcn -= (double)dci;
        acc[0][jj] -= fx;
        acc[1][jj] -= fy;
        acc[2][jj] -= fz;
        if (disp) acc[3][jj] -= (double)dcj;
        acc[4][jj] += (double)hec;
        if (disp) acc[5][jj] += (double)hed;
        if (rep) acc[6][jj] += (double)her;
    }
    __syncthreads();
    double* pr = part + (size_t)blockIdx.x * 2 * PART_K * PS_B;
    const double iv[PART_K] = {gx, gy, gz, dcn, ec, ed, er};
#pragma unroll
    for (int k = 0; k < PART_K; ++k) {
        pr[k * PS_B + l] = iv[k];
        pr[(PART_K + k) * PS_B + l] = acc[k][l];
    }
}

// Wavefronts per tile: doubled until the launch has 2048 of them (two per
// SIMD of the chip), at most 8.  Measured, pair kernel and evaluation: 122
// atoms (3 tiles) 96 -> 14 us and 531 -> 450 us; 216 H2O (66 tiles) 406 -> 326
// us per dynamics step, 334 us with at most 16 and 360 with 32 (the partial
// sets cost the reduction more than the shorter chain gains); 512 H2O mixed
// (300 tiles) 370 -> 331 us, 353 us with 4096 wavefronts.
static int ps_split(int ntiles) {
    int split = 1;
    while (split < 8 && ntiles * split < 2048) split *= 2;
    return split;
}

// ---------------------------------------------------------------------------
// K7: repulsion corrections over the topological neighbourhood
// (gfnff_method.cpp:9781-9872: bonded pairs excluded, H-H 1,3 / 1,4 factors)
// ---------------------------------------------------------------------------
// share w of nw of atom i's neighbours: out = gradient and energy corrections
__device__ inline void nbrep_fix_part(int i, int w, int nw, const double* __restrict__ x, const int* __restrict__ Z,
                                      const int* __restrict__ metal, const double* __restrict__ anb,
                                      const double* __restrict__ repz, const int* __restrict__ toff,
                                      const int* __restrict__ tidx, const int* __restrict__ tdist, double out[4]) {
    double3 xi = ld3(x, i);
    double gx = 0, gy = 0, gz = 0, er = 0;
    for (int k = toff[i] + w; k < toff[i + 1]; k += nw) {
        int j = tidx[k], td = tdist[k];
        int zi = Z[i], zj = Z[j];
        double fgen = rep_ff(zi, zj, metal[i], metal[j]);
        double fnew;
        if (td == 1) fnew = 0.0;
        else if (zi == 1 && zj == 1 && td == 2) fnew = 0.6290 * 1.4580;
        else if (zi == 1 && zj == 1 && td == 3) fnew = 0.6290 * 0.7080;
        else continue;
        double3 d = xi - ld3(x, j);
        double r = nrm(d);
        if (r > 20.0 || r < 1e-8) continue;
        double ab = repz[i] * repz[j] * 0.4270;
        double base = sqrt(anb[i] * anb[j]);
        double de = 0.0, dEdr = 0.0;
        {
            double al = base * fgen;
            double e = ab * exp(-al * r * sqrt(r)) / r;
            de -= e;
            dEdr -= -e / r - 1.5 * al * sqrt(r) * e;
        }
        if (fnew != 0.0) {
            double al = base * fnew;
            double e = ab * exp(-al * r * sqrt(r)) / r;
            de += e;
            dEdr += -e / r - 1.5 * al * sqrt(r) * e;
        }
        er += 0.5 * de;
        double s = dEdr / r;
        gx += s * d.x;
        gy += s * d.y;
        gz += s * d.z;
    }
    out[0] = gx;
    out[1] = gy;
    out[2] = gz;
    out[3] = er;
}
__device__ inline void nbrep_fix_atom(int i, const double* __restrict__ x, const int* __restrict__ Z,
                                      const int* __restrict__ metal, const double* __restrict__ anb,
                                      const double* __restrict__ repz, const int* __restrict__ toff,
                                      const int* __restrict__ tidx, const int* __restrict__ tdist,
                                      double* __restrict__ g, double* __restrict__ e_rep) {
    double o[4];
    nbrep_fix_part(i, 0, 1, x, Z, metal, anb, repz, toff, tidx, tdist, o);
    g[3 * i] += o[0];
    g[3 * i + 1] += o[1];
    g[3 * i + 2] += o[2];
    e_rep[i] += o[3];
}

// Tail of an atom after the pair terms: the repulsion corrections of its
// topological neighbourhood (its gradient and e_rep) and its dE/dCN total
// with the chain vector, which touch disjoint data.
struct AtomTailArgs {
    const double* x;
    const int *Z, *metal;
    const double *anb, *repz;
    const int *toff, *tidx, *tdist;
    double *g, *e_rep;
    const int *doff, *didx;
    const double* dcn_slot;
    double* dEdcn;
    const double* qtmp;
    double* v;
};
__device__ inline void dcn_total_atom(int i, double s, const AtomTailArgs& a) {
    for (int k = a.doff[i]; k < a.doff[i + 1]; ++k) s += a.dcn_slot[a.didx[k]];
    a.dEdcn[i] = s;
    a.v[i] = s - a.qtmp[i];
}
// one thread per atom (behind the row kernels of batches)
__global__ __launch_bounds__(256) void k_atom_tail(int n, AtomTailArgs a) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    nbrep_fix_atom(i, a.x, a.Z, a.metal, a.anb, a.repz, a.toff, a.tidx, a.tdist, a.g, a.e_rep);
    dcn_total_atom(i, a.dEdcn[i], a);
}

// f(0) + .. + f(W - 1) in groups of four
template <int W, class F>
__device__ __forceinline__ double ordered_sum(F f) {
    double s = 0.0;
#pragma unroll
    for (int u = 0; u < W; u += 4) s += (f(u) + f(u + 1)) + (f(u + 2) + f(u + 3));
    return s;
}

// Per atom a = A 64 + l: the row-side partials of tiles (A, C), C = 0 .. A,
// then the column-side partials of tiles (R, A), R = A .. nb - 1, in that
// order, dealt to W wavefronts whose sums are added in order: W = 16 where the
// tiles are split (few blocks, many partial sets: 512 H2O, 200 sets a block, 26
// us with four wavefronts; evaluation 256 -> 242 us), 4 otherwise.
// Batches (blocks != nullptr): one workgroup per 64-atom block {a0, n, A, base}
// of a molecule (atoms a0 .. a0 + n - 1, its tiles numbered from base).
// part2 (nullable): a second set of tile partials (the split pair terms),
// added tile by tile after the first.
// The atom's tail follows in the same launch, its neighbours dealt to the W
// wavefronts (by one thread per atom in a launch of its own it took 15 us at
// any size: a chain of square roots and exponentials per neighbour).  W = 16
// leaves a lane 128 registers, 12 of them spilled.
template <int W>
__global__ __launch_bounds__(64 * W) void k_pairs_sym_reduce(int n, int nb, const double* __restrict__ part,
                                                          const double* __restrict__ part2,
                                                          double* __restrict__ e_coul, double* __restrict__ e_disp,
                                                          const int4* __restrict__ blocks, int split, AtomTailArgs at) {
    __shared__ double qs[W][PART_K][PS_B], fs[W][4][PS_B];
    int A = blockIdx.x, a0 = 0, base = 0;
    if (blocks) {
        const int4 bb = blocks[blockIdx.x];
        a0 = bb.x;
        n = bb.y;
        A = bb.z;
        base = bb.w;
        nb = (n + PS_B - 1) / PS_B;
    }
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int nset = (nb + 1) * split;  // A + 1 row-side tiles and nb - A column-side tiles, split sets each
    double s[PART_K] = {0, 0, 0, 0, 0, 0, 0};
#pragma unroll 2
    for (int v = w; v < nset; v += W) {
        const int u = v / split, sub = v % split;
        const bool rowside = u <= A;
        const int Rr = u - 1;  // column side: tile (R, A), R = u - 1 = A .. nb - 1
        const int t = base + (rowside ? A * (A + 1) / 2 + u : Rr * (Rr + 1) / 2 + A);
        const size_t o = (((size_t)t * split + sub) * 2 + (rowside ? 0 : 1)) * PART_K * PS_B + l;
        const double* p = part + o;
#pragma unroll
        for (int k = 0; k < PART_K; ++k) s[k] += p[k * PS_B];
        if (part2) {
#pragma unroll
            for (int k = 0; k < PART_K; ++k) s[k] += part2[o + k * PS_B];
        }
    }
#pragma unroll
    for (int k = 0; k < PART_K; ++k) qs[w][k][l] = s[k];
    {
        double o[4] = {0, 0, 0, 0};
        if (A * PS_B + l < n)
            nbrep_fix_part(a0 + A * PS_B + l, w, W, at.x, at.Z, at.metal, at.anb, at.repz, at.toff, at.tidx, at.tdist, o);
#pragma unroll
        for (int k = 0; k < 4; ++k) fs[w][k][l] = o[k];
    }
    __syncthreads();
    if (threadIdx.x >= PS_B || A * PS_B + (int)threadIdx.x >= n) return;
    const int i = a0 + A * PS_B + threadIdx.x;
    double v[PART_K];
#pragma unroll
    for (int k = 0; k < PART_K; ++k) v[k] = ordered_sum<W>([&](int u) { return qs[u][k][l]; });
    double c[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) c[k] = ordered_sum<W>([&](int u) { return fs[u][k][l]; });
    at.g[3 * i] = v[0] + c[0];
    at.g[3 * i + 1] = v[1] + c[1];
    at.g[3 * i + 2] = v[2] + c[2];
    e_coul[i] = v[4];
    e_disp[i] = v[5];
    at.e_rep[i] = v[6] + c[3];
    dcn_total_atom(i, v[3], at);
}

// Sums the j-chunk partials of k_pairs_part in chunk order.
__global__ __launch_bounds__(256) void k_pairs_reduce(int n, int nchunk, const double* __restrict__ part,
                                                      double* __restrict__ g, double* __restrict__ dEdcn,
                                                      double* __restrict__ e_coul, double* __restrict__ e_disp,
                                                      double* __restrict__ e_rep) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double acc[PART_K] = {};
    for (int c = 0; c < nchunk; ++c) {
        const double* p = part + (size_t)c * PART_K * n + i;
#pragma unroll
        for (int k = 0; k < PART_K; ++k) acc[k] += p[(size_t)k * n];
    }
    g[3 * i] = acc[0];
    g[3 * i + 1] = acc[1];
    g[3 * i + 2] = acc[2];
    dEdcn[i] = acc[3];
    e_coul[i] = acc[4];
    e_disp[i] = acc[5];
    e_rep[i] = acc[6];
}

// ---------------------------------------------------------------------------
// K8: bonded term lists.  Each entry writes its atom gradients to fixed slots
// (gathered per atom in k_finish in a fixed order) and its energy to e_out.
// ---------------------------------------------------------------------------
// HB coordination of X-H hydrogens (ff_workspace_gfnff.cpp:46-97) and bonds (:104-180)
// bonds with an X-H hydrogen and a non-empty hydrogen-bond partner list
// (bsel: their indices): one wavefront per bond,
// lanes stride the bond's hydrogen-bond partner list (HB coordination and
// its gradient), fixed butterflies; lane 0 writes the bond's own slots

__device__ __forceinline__ void bond_hb_wave(int w, int nsel, const int* __restrict__ bsel,
                                             const int* __restrict__ ij, const double* __restrict__ par,
                                             const int* __restrict__ hb_off, const int* __restrict__ hb_B,
                                             const int* __restrict__ slot0, const double* __restrict__ x,
                                             const double* __restrict__ cn, const double* __restrict__ rcov_d3,
                                             const int* __restrict__ bond_H, double* __restrict__ slots,
                                             double* __restrict__ dcn_slot, double* __restrict__ e_out) {
    const int lane = threadIdx.x & 63;
    if (w >= nsel) return;
    const int b = bsel[w];
    int i = ij[2 * b], j = ij[2 * b + 1];
    const double* p = par + 8 * b;
    double3 d = ld3(x, i) - ld3(x, j);
    double r = nrm(d);
    double r0 = (p[0] + p[2] * cn[i] + p[1] + p[3] * cn[j] + p[4]) * p[5];
    double dr = r - r0;
    double a0 = p[6], al = a0;
    const int H = bond_H[b];
    const int k0 = (H >= 0) ? hb_off[b] : 0, k1 = (H >= 0) ? hb_off[b + 1] : 0;
    if (H >= 0) {
        const double3 xh = ld3(x, H);
        double hbcn = 0.0;
        for (int k = k0 + lane; k < k1; k += 64) {
            int B = hb_B[k];
            double3 v = ld3(x, B) - xh;
            double rr2 = dot(v, v);
            if (rr2 > 900.0) continue;
            double rr = sqrt(rr2);
            double rc = 1.78 * (4.0 / 3.0) * (rcov_d3[H] + rcov_d3[B]);
            hbcn += cn_count(-27.5 * (rr - rc) / rc);
        }
        hbcn = wave_sum(hbcn);
        al = (-(1.0 - 0.9) * hbcn + 1.0) * a0;
    }
    double e = p[7] * exp(-al * dr * dr);
    double dEdr = -2.0 * al * dr * e;
    int s = slot0[b];
    if (lane == 0) {
        e_out[b] = e;
        st3(slots, s, (dEdr / r) * d);
        st3(slots, s + 1, (-dEdr / r) * d);
        double yy = -dEdr;
        dcn_slot[2 * b] = yy * p[5] * p[2];
        dcn_slot[2 * b + 1] = yy * p[5] * p[3];
    }
    if (H >= 0) {
        double zz = 0.1 * a0 * dr * dr * e;
        const double3 xh = ld3(x, H);
        double3 gH = make_double3(0, 0, 0);
        for (int k = k0 + lane; k < k1; k += 64) {
            int B = hb_B[k];
            double3 v = ld3(x, B) - xh;
            double rr2 = dot(v, v);
            double3 gB = make_double3(0, 0, 0);
            if (rr2 <= 900.0) {
                double rr = sqrt(rr2);
                double rc = 1.78 * (4.0 / 3.0) * (rcov_d3[H] + rcov_d3[B]);
                double arg = -27.5 * (rr - rc) / rc;
                // exp(-arg^2) underflows to 0 for |arg| > 27.5: skipped there
                double dc = 0.0;
                if (arg > -27.5) dc = 0.5641895835477563 * (-27.5 / rc) * exp(-arg * arg) / rr;
                gH = gH + (-zz * dc) * v;
                gB = (zz * dc) * v;
            }
            st3(slots, s + 3 + (k - k0), gB);
        }
        gH.x = wave_sum(gH.x);
        gH.y = wave_sum(gH.y);
        gH.z = wave_sum(gH.z);
        if (lane == 0) st3(slots, s + 2, gH);
    }
}

// bonds without HB coordination (no X-H hydrogen, or an empty partner list,
// where hbcn = 0 leaves alpha = a0 exactly; bsel: their indices), one thread
// each: the arithmetic of bond_hb_wave's lane 0; an X-H bond's hydrogen slot gets
// its zero gradient
__device__ __forceinline__ void bond_plain(int t, int nsel, const int* __restrict__ bsel, const int* __restrict__ ij,
                                           const double* __restrict__ par, const int* __restrict__ slot0,
                                           const int* __restrict__ bond_H, const double* __restrict__ x,
                                           const double* __restrict__ cn, double* __restrict__ slots,
                                           double* __restrict__ dcn_slot, double* __restrict__ e_out) {
    if (t >= nsel) return;
    const int b = bsel[t];
    const int i = ij[2 * b], j = ij[2 * b + 1];
    const double* p = par + 8 * b;
    const double3 d = ld3(x, i) - ld3(x, j);
    const double r = nrm(d);
    const double r0 = (p[0] + p[2] * cn[i] + p[1] + p[3] * cn[j] + p[4]) * p[5];
    const double dr = r - r0;
    const double al = p[6];
    const double e = p[7] * exp(-al * dr * dr);
    const double dEdr = -2.0 * al * dr * e;
    const int s = slot0[b];
    e_out[b] = e;
    st3(slots, s, (dEdr / r) * d);
    st3(slots, s + 1, (-dEdr / r) * d);
    const double yy = -dEdr;
    dcn_slot[2 * b] = yy * p[5] * p[2];
    dcn_slot[2 * b + 1] = yy * p[5] * p[3];
    if (bond_H[b] >= 0) st3(slots, s + 2, make_double3(0, 0, 0));
}

// angles: ff_workspace_gfnff.cpp:187-275
__device__ __forceinline__ void angle_entry(int t, int na, const int* __restrict__ ijk,
                                            const double* __restrict__ par, const int* __restrict__ slot0,
                                            const double* __restrict__ x, const double* __restrict__ rcov_d3,
                                            double* __restrict__ slots, double* __restrict__ e_out) {
    if (t >= na) return;
    int i = ijk[3 * t], j = ijk[3 * t + 1], k = ijk[3 * t + 2];
    double fc = par[2 * t], th0 = par[2 * t + 1];
    double3 u = ld3(x, i) - ld3(x, j), v = ld3(x, k) - ld3(x, j);
    double ru = nrm(u), rv = nrm(v);
    double cth = (ru < 1e-10 || rv < 1e-10) ? 1.0 : dot(u, v) / (ru * rv);
    cth = fmin(1.0, fmax(-1.0, cth));
    double th = acos(cth), e, dEdcos;
    if (fabs(M_PI - th0) < 1e-6) {
        double dt = th - th0;
        e = fc * dt * dt;
        double sn = sin(th);
        dEdcos = (sn > 1e-14) ? -2.0 * fc * dt / sn : 0.0;
    } else {
        double c0 = cos(th0);
        e = fc * (cth - c0) * (cth - c0);
        dEdcos = 2.0 * fc * (cth - c0);
    }
    double rci = rcov_d3[i] * (4.0 / 3.0), rcj = rcov_d3[j] * (4.0 / 3.0), rck = rcov_d3[k] * (4.0 / 3.0);
    double rc1 = 0.595 * (rci + rcj) * (rci + rcj), rc2 = 0.595 * (rcj + rck) * (rcj + rck);
    double r12 = ru * ru, r22 = rv * rv;
    double rr1 = r12 / rc1, rr2 = r22 / rc2;
    rr1 *= rr1;
    rr2 *= rr2;
    double d1 = 1.0 / (1.0 + rr1), d2 = 1.0 / (1.0 + rr2), damp = d1 * d2;
    e_out[t] = e * damp;
    double dd1 = (r12 > 1e-8) ? -4.0 * rr1 / (r12 * (1.0 + rr1) * (1.0 + rr1)) : 0.0;
    double dd2 = (r22 > 1e-8) ? -4.0 * rr2 / (r22 * (1.0 + rr2) * (1.0 + rr2)) : 0.0;
    double sinth = sqrt(fmax(0.0, 1.0 - cth * cth));
    double pre = (sinth < 1e-14 || ru < 1e-10 || rv < 1e-10) ? 0.0 : dEdcos * damp;
    double3 gi = (pre / ru) * ((1.0 / rv) * v - (cth / ru) * u) + (e * dd1 * d2) * u;
    double3 gk = (pre / rv) * ((1.0 / ru) * u - (cth / rv) * v) + (e * dd2 * d1) * v;
    int s = slot0[t];
    st3(slots, s, gi);
    st3(slots, s + 1, (-1.0) * (gi + gk));
    st3(slots, s + 2, gk);
}

// signed dihedral and its gradient (phi as in gfnff_geometry.h:60-110)
__device__ __forceinline__ double dihed(double3 ri, double3 rj, double3 rk, double3 rl, double3 g[4], bool& ok) {
    double3 v1 = rj - ri, v2 = rk - rj, v3 = rl - rk;
    double3 n1 = cross(v1, v2), n2 = cross(v2, v3);
    double nn1 = nrm(n1), nn2 = nrm(n2), nv2 = nrm(v2);
    ok = !(nn1 < 1e-10 || nn2 < 1e-10 || nv2 < 1e-10);
    if (!ok) {
        for (int a = 0; a < 4; ++a) g[a] = make_double3(0, 0, 0);
        return 0.0;
    }
    double c = dot(n1, n2) / (nn1 * nn2);
    double s = nv2 * dot(n1, v3) / nn1 / nn2;
    s = fmin(1.0, fmax(-1.0, s));
    double phi = atan2(s, c);
    double n1s = nn1 * nn1, n2s = nn2 * nn2, b2 = nv2 * nv2;
    double3 gi = (-nv2 / n1s) * n1, gl = (nv2 / n2s) * n2;
    double aa = dot(v1, v2) / b2, bb = dot(v3, v2) / b2;
    g[0] = gi;
    g[3] = gl;
    g[1] = (-1.0 - aa) * gi + bb * gl;
    g[2] = aa * gi + (-1.0 - bb) * gl;
    return phi;
}

// torsions (primary and extra): ff_workspace_gfnff.cpp:282-482
__device__ __forceinline__ void torsion_entry(int t, int nt, const int* __restrict__ ijkl,
                                              const double* __restrict__ par, const int* __restrict__ slot0,
                                              const double* __restrict__ x, const double* __restrict__ rcov_d3,
                                              double* __restrict__ slots, double* __restrict__ e_out) {
    if (t >= nt) return;
    int id[4] = {ijkl[4 * t], ijkl[4 * t + 1], ijkl[4 * t + 2], ijkl[4 * t + 3]};
    const double* p = par + 4 * t;
    double3 r[4];
    for (int a = 0; a < 4; ++a) r[a] = ld3(x, id[a]);
    double3 gp[4];
    bool ok;
    double phi = dihed(r[0], r[1], r[2], r[3], gp, ok);
    double V = p[0], nn = p[1], phi0 = p[2], atc = p[3];
    double c1 = nn * (phi - phi0) + M_PI;
    double e = V * (1.0 + cos(c1));
    double3 v[3] = {r[0] - r[1], r[1] - r[2], r[2] - r[3]};
    double dmp[3], rr[3], r2[3];
    for (int s = 0; s < 3; ++s) {
        r2[s] = dot(v[s], v[s]);
        double rs = rcov_d3[id[s]] * (4.0 / 3.0) + rcov_d3[id[s + 1]] * (4.0 / 3.0);
        double rc = atc * rs * rs;
        rr[s] = r2[s] / rc;
        rr[s] *= rr[s];
        dmp[s] = 1.0 / (1.0 + rr[s]);
    }
    double damp = dmp[0] * dmp[1] * dmp[2];
    e_out[t] = e * damp;
    double dEdphi = ok ? -V * nn * sin(c1) * damp : 0.0;
    double dd[3];
    for (int s = 0; s < 3; ++s) dd[s] = (r2[s] > 1e-8) ? -4.0 * rr[s] / (r2[s] * (1.0 + rr[s]) * (1.0 + rr[s])) : 0.0;
    double f0 = e * dd[0] * dmp[1] * dmp[2], f1 = e * dmp[0] * dd[1] * dmp[2], f2 = e * dmp[0] * dmp[1] * dd[2];
    int s = slot0[t];
    st3(slots, s, dEdphi * gp[0] + f0 * v[0]);
    st3(slots, s + 1, dEdphi * gp[1] + (-f0) * v[0] + f1 * v[1]);
    st3(slots, s + 2, dEdphi * gp[2] + (-f1) * v[1] + f2 * v[2]);
    st3(slots, s + 3, dEdphi * gp[3] + (-f2) * v[2]);
}

// out-of-plane angle of centre ri against the plane through its first
// neighbour rj (gfnff_geometry.h:207-300): n = (ri - rj) x (rk - rj),
// v = rl - ri, omega = asin(n.v / (|n||v|)), with its gradient from
// gn = v/(|n||v|) - s n/|n|^2, gv = n/(|n||v|) - s v/|v|^2.
__device__ __forceinline__ double oop(double3 ri, double3 rj, double3 rk, double3 rl, double3 g[4]) {
    double3 re = ri - rj, rd = rk - rj, rv = rl - ri;
    double3 nn = cross(re, rd);
    double N = nrm(nn), V = nrm(rv);
    for (int a = 0; a < 4; ++a) g[a] = make_double3(0, 0, 0);
    if (N < 1e-10 || V < 1e-10) return 0.0;
    double s = fmin(1.0, fmax(-1.0, dot(nn, rv) / (N * V)));
    double om = asin(s), co = cos(om);
    if (fabs(N * V * co) < 1e-14) return om;
    double3 gn = (1.0 / (N * V)) * rv + (-s / (N * N)) * nn;
    double3 gv = (1.0 / (N * V)) * nn + (-s / (V * V)) * rv;
    double3 dre = cross(rd, gn), drd = cross(gn, re);
    double ic = 1.0 / co;
    g[0] = ic * (dre + (-1.0) * gv);
    g[1] = (-ic) * (dre + drd);
    g[2] = ic * drd;
    g[3] = ic * gv;
    return om;
}

// inversions: ff_workspace_gfnff.cpp:489-604.  par: fc, omega0, type
// (0: V (1 - cos w), -1: V (cos w - cos w0)^2); damping over the distances of
// the first neighbour j to the centre and the other two neighbours.
__device__ __forceinline__ void inversion_entry(int t, int nv, const int* __restrict__ ijkl,
                                                const double* __restrict__ par, const int* __restrict__ slot0,
                                                const double* __restrict__ x, const double* __restrict__ rcov_d3,
                                                double* __restrict__ slots, double* __restrict__ e_out) {
    if (t >= nv) return;
    int id[4] = {ijkl[4 * t], ijkl[4 * t + 1], ijkl[4 * t + 2], ijkl[4 * t + 3]};
    const double* p = par + 3 * t;
    double3 r[4];
    double rc[4];
    for (int a = 0; a < 4; ++a) {
        r[a] = ld3(x, id[a]);
        rc[a] = rcov_d3[id[a]] * (4.0 / 3.0);
    }
    double3 go[4];
    double om = oop(r[0], r[1], r[2], r[3], go);
    const int other[3] = {0, 2, 3};
    double3 dv[3];
    double r2[3], rr[3], dmp[3];
    for (int s = 0; s < 3; ++s) {
        int o = other[s];
        dv[s] = r[1] - r[o];
        r2[s] = dot(dv[s], dv[s]);
        double rcut = 0.505 * (rc[1] + rc[o]) * (rc[1] + rc[o]);
        rr[s] = (r2[s] / rcut) * (r2[s] / rcut);
        dmp[s] = 1.0 / (1.0 + rr[s]);
    }
    double damp = dmp[0] * dmp[1] * dmp[2];
    double V = p[0], et, dEdom;
    if (p[2] == 0.0) {
        et = V * (1.0 - cos(om));
        dEdom = V * sin(om) * damp;
    } else {
        double df = cos(om) - cos(p[1]);
        et = V * df * df;
        dEdom = -2.0 * V * sin(om) * df * damp;
    }
    e_out[t] = et * damp;
    double f[3];
    for (int s = 0; s < 3; ++s) {
        double dd = (r2[s] < 1e-8) ? 0.0 : -4.0 * rr[s] / (r2[s] * (1.0 + rr[s]) * (1.0 + rr[s]));
        f[s] = et * dd * dmp[(s + 1) % 3] * dmp[(s + 2) % 3];
    }
    int s = slot0[t];
    st3(slots, s, dEdom * go[0] + (-f[0]) * dv[0]);
    st3(slots, s + 1, dEdom * go[1] + f[0] * dv[0] + f[1] * dv[1] + f[2] * dv[2]);
    st3(slots, s + 2, dEdom * go[2] + (-f[1]) * dv[1]);
    st3(slots, s + 3, dEdom * go[3] + (-f[2]) * dv[2]);
}

// triple-bond torsions: ff_workspace_gfnff.cpp:611-648 (undamped),
// E = erefhalf (1 - cos 2 phi)
__device__ __forceinline__ void stors_entry(int t, int nt, const int* __restrict__ ijkl,
                                            const double* __restrict__ eh, const int* __restrict__ slot0,
                                            const double* __restrict__ x, double* __restrict__ slots,
                                            double* __restrict__ e_out) {
    if (t >= nt) return;
    double3 gp[4];
    bool ok;
    double phi = dihed(ld3(x, ijkl[4 * t]), ld3(x, ijkl[4 * t + 1]), ld3(x, ijkl[4 * t + 2]), ld3(x, ijkl[4 * t + 3]),
                       gp, ok);
    double e = eh[t];
    e_out[t] = e - e * cos(2.0 * phi);
    double d = ok ? 2.0 * e * sin(2.0 * phi) : 0.0;
    int s = slot0[t];
    for (int a = 0; a < 4; ++a) st3(slots, s + a, d * gp[a]);
}

// bonded repulsion: ff_workspace_gfnff.cpp:774-807
__device__ __forceinline__ void brep_entry(int b, int nb, const int* __restrict__ ij, const double* __restrict__ par,
                                           const int* __restrict__ slot0, const double* __restrict__ x,
                                           double* __restrict__ slots, double* __restrict__ e_out) {
    if (b >= nb) return;
    int i = ij[2 * b], j = ij[2 * b + 1];
    double3 d = ld3(x, i) - ld3(x, j);
    double r = nrm(d);
    double e = 0.0, dEdr = 0.0;
    if (!(r > 20.0 || r < 1e-8)) {
        double al = par[2 * b], ab = par[2 * b + 1];
        e = ab * exp(-al * r * sqrt(r)) / r;
        dEdr = -e / r - 1.5 * al * sqrt(r) * e;
    }
    e_out[b] = e;
    int s = slot0[b];
    st3(slots, s, (dEdr / r) * d);
    st3(slots, s + 1, (-dEdr / r) * d);
}

// hydrogen bonds, cases 1-4: ff_workspace_gfnff.cpp:938-1404
// hb_core evaluates one triplet A-H...B: returns its energy and the gradient
// on A, H and B; with XTRA it also writes the gradient of the acceptor's
// neighbours to xs[k] (k-th neighbour of B) and, for case 3, of the
// neighbours D of the carbonyl carbon other than B to xs[nnb + d].  Case 3: B
// is a carbonyl O whose only neighbour is the carbon C; case 4: sp2 N
// acceptor with a virtual lone pair opposite its neighbours.  The per-triplet
// parameters of the reference (basicity, acidity, topology charges) are
// per-atom values, and the neighbour lists depend on B only.
struct HBArgs {
    const double* cb;      // basicity per atom
    const double* ca;      // acidity per atom
    const double* Qh;      // per atom e^(15 q) / (e^(15 q) + 1), q the topology charge (role H)
    const double* Qab;     // per atom e^(-15 q) / (e^(-15 q) + 1) (roles A, B)
    const int* nb_off;     // per atom: neighbours of an acceptor of cases 2-4 (CSR)
    const int* nb_idx;
    const int* parentC;    // per atom: carbonyl carbon of a case-3 acceptor, else -1
    const int* nbc_off;    // per atom: neighbours of parentC other than the acceptor (CSR)
    const int* nbc_idx;
    const double* hb_rad;
    const double* lpd;     // per atom: case-4 lone-pair distance (element table)
    const int* Z;
    const float4* pk;      // FP32 per atom {basicity, acidity, Qab, hb_rad} (roles A, B of the FP32 cores)
    const float* qh32;     // FP32 Qh (role H of the FP32 cores)
};
__device__ inline double pow6(double t) {
    const double t2 = t * t;
    return t2 * t2 * t2;
}

template <bool XTRA>
__device__ double hb_core(int A, int H, int B, int cs, const HBArgs& a, const double* __restrict__ x,
                          double3& ga_out, double3& gh_out, double3& gb_out, double* __restrict__ xs) {
    const double basA = a.cb[A], basB = a.cb[B], aciA = a.ca[A], aciB = a.ca[B];

    double3 pA = ld3(x, A), pH = ld3(x, H), pB = ld3(x, B);
    double rAH = nrm(pH - pA), rHB = nrm(pB - pH), rAB = nrm(pB - pA);
    const int nb0 = (cs >= 2) ? a.nb_off[B] : 0, nb1 = (cs >= 2) ? a.nb_off[B + 1] : 0;
    const int C3 = (cs == 3) ? a.parentC[B] : -1;
    const int c0 = (C3 >= 0) ? a.nbc_off[B] : 0, c1 = (C3 >= 0) ? a.nbc_off[B + 1] : 0;
    const int sD = nb1 - nb0;  // first extra slot of the D atoms
    double3 z3 = make_double3(0, 0, 0);
    double3 ga = z3, gb = z3, gh = z3;
    double E = 0.0;
    bool nb_written = false;
    if (rAB <= 50.0) {
        double rAH4 = rAH * rAH * rAH * rAH, rHB4 = rHB * rHB * rHB * rHB;
        double den = 1.0 / (rAH4 + rHB4);
        const double QH = a.Qh[H], QA = a.Qab[A], QB = a.Qab[B];
        double bas = (QA * basA * rAH4 + QB * basB * rHB4) * den;
        double aci = (aciB * rAH4 + aciA * rHB4) * den;
        double radab = a.hb_rad[A] + a.hb_rad[B];
        const double ratio3 = pow6(22.0 * radab / (rAB * rAB)), ratio1 = pow6(rAB * rAB / 85.0);
        double dsh = 1.0 / (1.0 + ratio3);
        double dlg = 1.0 / (1.0 + ratio1);
        double denv = dsh * dlg;
        double expo0 = (49.0 / radab) * ((rAH + rHB) / rAB - 1.0);
        double doutl = (expo0 > 15.0) ? 0.0 : 2.0 / (1.0 + exp(expo0));
        double outl_nb = 1.0;
        double nbcut = (a.Z[B] == 7 && nb1 - nb0 == 1) ? 2.0 : 11.20;
        if (cs >= 2)
            for (int k = nb0; k < nb1; ++k) {
                double3 pn = ld3(x, a.nb_idx[k]);
                double ex = (nbcut / radab) * ((nrm(pn - pA) + nrm(pn - pB)) / rAB - 1.0);
                outl_nb *= (2.0 / (1.0 + exp(-ex)) - 1.0);
            }
        double rdamp = (cs >= 2) ? denv * (1.8 / (rHB * rHB * rHB) - 0.8 / (rAB * rAB * rAB)) : denv / (rAB * rAB * rAB);
        // case 4: virtual lone pair lp = B - lpd v/|v|, v = sum_nb (x_nb - x_B)
        double outl_lp = 1.0, lpd = 0.0, xlp = 0.0;
        double3 lpv = z3, lp = pB;
        int nlp = 0;
        if (cs == 4) {
            lpd = a.lpd[B];
            for (int k = nb0; k < nb1; ++k) lpv = lpv + (ld3(x, a.nb_idx[k]) - pB);
            double vn = nrm(lpv);
            if (vn > 1e-10 && nb1 > nb0) {
                nlp = nb1 - nb0;
                lp = pB + (-lpd / vn) * lpv;
                xlp = (56.0 / radab) * ((nrm(pA - lp) + lpd + 1e-12) / rAB - 1.0);
                outl_lp = 2.0 / (1.0 + exp(xlp));
            }
        }
        // case 3: H...O=C bend and D-C=O...H torsion factors
        double eangl = 1.0, etors = 1.0;
        double3 dB3 = z3, dC3 = z3, dH3 = z3;  // d eangl / d(B, C, H)
        const double tfc = (1.0 - 0.94) / 2.0;
        if (C3 >= 0) {
            const double cc0 = cos(120.0 * M_PI / 180.0);
            const double kb = (1.0 - 0.20) / ((1.0 - cc0) * (1.0 - cc0));
            double3 u = ld3(x, C3) - pB, w = pH - pB;
            double ru = nrm(u), rw = nrm(w);
            double ca = fmin(1.0, fmax(-1.0, dot(u, w) / (ru * rw + 1e-14)));
            eangl = 1.0 - kb * (ca - cc0) * (ca - cc0);
            double dea = 2.0 * kb * (ca - cc0);
            dC3 = (-dea / ru) * ((1.0 / rw) * w + (-ca / ru) * u);
            dH3 = (-dea / rw) * ((1.0 / ru) * u + (-ca / rw) * w);
            dB3 = (-1.0) * (dC3 + dH3);
            double3 pC = ld3(x, C3);
            for (int k = c0; k < c1; ++k) {
                double3 gp[4];
                bool ok;
                double phi = dihed(ld3(x, a.nbc_idx[k]), pB, pC, pH, gp, ok);
                etors *= (1.0 + cos(2.0 * (phi - M_PI / 2.0) + M_PI)) * tfc + 0.94;
            }
        }
        double qhoutl = QH * doutl * outl_nb * outl_lp;
        double gscale = (cs == 2 || cs == 4) ? 0.268 : (cs == 3 ? 0.350 : 1.0);
        double cval = aciA * basB * QA * QB * gscale;
        E = (cs >= 2) ? -rdamp * qhoutl * cval * eangl * etors : -bas * aci * rdamp * qhoutl;
        double3 drab = pA - pB, drah = pA - pH, drbh = pB - pH;
        double rab2 = rAB * rAB, rbh2 = rHB * rHB, rah2 = rAH * rAH;
        double rahprbh = rAH + rHB + 1e-12;
        double ddamp = (-2.0 * 6.0 * ratio1 / (1.0 + ratio1)) + (2.0 * 6.0 * ratio3 / (1.0 + ratio3));
        double expo = (49.0 / radab) * (rahprbh / rAB - 1.0);
        if (!(expo > 15.0)) {
            double ratio2 = exp(expo);
            if (cs >= 2) {
                double ct = cval * eangl * etors;
                double rbhdamp = denv * 1.8 / (rbh2 * rHB), rabdamp = denv * -0.8 / (rab2 * rAB);
                double dterm = -qhoutl * ct, aterm = -rdamp * QH * outl_nb * outl_lp * ct;
                double nbterm = -rdamp * QH * doutl * outl_lp * ct;
                double gi = ((rabdamp + rbhdamp) * ddamp - 3.0 * rabdamp) / rab2 * dterm;
                ga = gi * drab;
                gb = (-gi) * drab;
                gi = -3.0 * rbhdamp / rbh2 * dterm;
                gb = gb + gi * drbh;
                gh = (-gi) * drbh;
                double tmp1 = -2.0 * aterm * ratio2 * expo / ((1.0 + ratio2) * (1.0 + ratio2)) / (rahprbh - rAB);
                gi = -tmp1 * rahprbh / rab2;
                ga = ga + gi * drab;
                gb = gb + (-gi) * drab;
                double3 dga = (tmp1 / rAH) * drah, dgb = (tmp1 / rHB) * drbh;
                ga = ga + dga;
                gb = gb + dgb;
                gh = gh + (-1.0) * (dga + dgb);
                // case 4: d outl_lp through s = |A - lp| + lpd and rAB
                double3 pg = z3;
                if (nlp > 0) {
                    double lpterm = -rdamp * QH * doutl * outl_nb * cval;
                    double3 dal = pA - lp;
                    double ral = nrm(dal), sl = ral + lpd + 1e-12;
                    double el = exp(xlp), fe = 2.0 * lpterm * el / ((1.0 + el) * (1.0 + el)) * (56.0 / radab);
                    double dEds = -fe / rAB, dEdrab = fe * sl / rab2;
                    double3 gA = (dEds / (ral + 1e-12)) * dal;
                    ga = ga + (dEdrab / rAB) * drab + gA;
                    gb = gb + (-dEdrab / rAB) * drab;
                    double3 glp = (-1.0) * gA;
                    double vn = nrm(lpv), vg = dot(lpv, glp);
                    pg = (lpd / vn) * (glp + (-vg / (vn * vn)) * lpv);
                    gb = gb + glp + (double)nlp * pg;
                }
                // case 3: bend and torsion factors
                double3 gC = z3;
                if (C3 >= 0) {
                    double bterm = -rdamp * qhoutl * etors * cval, tterm = -rdamp * qhoutl * eangl * cval;
                    gb = gb + bterm * dB3;
                    gC = bterm * dC3;
                    gh = gh + bterm * dH3;
                    double3 pC = ld3(x, C3);
                    for (int k = c0; k < c1; ++k) {
                        double3 gp[4];
                        bool ok;
                        double phi = dihed(ld3(x, a.nbc_idx[k]), pB, pC, pH, gp, ok);
                        double cc = 2.0 * (phi - M_PI / 2.0) + M_PI;
                        double etk = (1.0 + cos(cc)) * tfc + 0.94;
                        double f = ok ? (etors / etk) * tterm * (-2.0 * sin(cc) * tfc) : 0.0;
                        if (XTRA) st3(xs, sD + (k - c0), f * gp[0]);
                        gb = gb + f * gp[1];
                        gC = gC + f * gp[2];
                        gh = gh + f * gp[3];
                    }
                }
                nb_written = true;
                int kk = 3;
                for (int k = nb0; k < nb1; ++k, ++kk) {
                    double3 pn = ld3(x, a.nb_idx[k]);
                    double3 dranb = pA - pn, drbnb = pB - pn;
                    double ranb = nrm(dranb), rbnb = nrm(drbnb), sm = ranb + rbnb + 1e-12;
                    double ex = (nbcut / radab) * (sm / rAB - 1.0);
                    double r2n = exp(-ex);
                    double oi = 2.0 / (1.0 + r2n) - 1.0;
                    double others = (fabs(oi) > 1e-12) ? outl_nb / oi : 1.0;
                    double tmp2 = 2.0 * nbterm * others * r2n * ex / ((1.0 + r2n) * (1.0 + r2n)) / (sm - rAB);
                    double gi2 = -tmp2 * sm / rab2;
                    ga = ga + gi2 * drab;
                    gb = gb + (-gi2) * drab;
                    double3 da = (tmp2 / ranb) * dranb, db = (tmp2 / rbnb) * drbnb;
                    ga = ga + da;
                    gb = gb + db;
                    double3 gn = (-1.0) * (da + db + pg);
                    if (kk == 3 && C3 >= 0) gn = gn + gC;
                    if (XTRA) st3(xs, kk - 3, gn);
                }
            } else {
                double caa = QA * basA, cbb = QB * basB;
                double rterm = -aci * rdamp * qhoutl, dterm = -aci * bas * qhoutl, sterm = -rdamp * bas * qhoutl;
                double aterm = -aci * bas * rdamp * QH;
                double tmp = den * den * 4.0;
                double dd24a = rah2 * rHB4 * tmp, dd24b = rbh2 * rAH4 * tmp;
                ga = ((caa - cbb) * dd24a * rterm) * drah;
                gb = ((cbb - caa) * dd24b * rterm) * drbh;
                gh = (-1.0) * (ga + gb);
                double3 dga = ((aciB - aciA) * dd24a * sterm) * drah, dgb = ((aciA - aciB) * dd24b * sterm) * drbh;
                ga = ga + dga;
                gb = gb + dgb;
                gh = gh + (-1.0) * (dga + dgb);
                double gi = rdamp * (ddamp - 3.0) / rab2;
                ga = ga + (gi * dterm) * drab;
                gb = gb + (-gi * dterm) * drab;
                gi = aterm * 2.0 * ratio2 * expo * rahprbh / ((1.0 + ratio2) * (1.0 + ratio2)) / (rahprbh - rAB) / rab2;
                ga = ga + gi * drab;
                gb = gb + (-gi) * drab;
                double to = -2.0 * aterm * ratio2 * expo / ((1.0 + ratio2) * (1.0 + ratio2)) / (rahprbh - rAB);
                double3 da = (to / rAH) * drah, db = (to / rHB) * drbh;
                ga = ga + da;
                gb = gb + db;
                gh = gh + (-1.0) * (da + db);
            }
        }
    }
    ga_out = ga;
    gh_out = gh;
    gb_out = gb;
    if (XTRA && !nb_written) {
        for (int kk = 0; kk < nb1 - nb0; ++kk) st3(xs, kk, z3);
        for (int k = c0; k < c1; ++k) st3(xs, sD + (k - c0), z3);
    }
    return E;
}

// halogen bonds A-X...B: ff_workspace_gfnff.cpp:1411-1519.  The gradient is
// the reference's: its short- and long-range damping derivatives
// (-12 f_s t_s / (r (1 + t_s)) and -12 r f_l t_l / (70 (1 + t_l))) are kept as
// they are, so along r_XB it is not the derivative of the energy.
__device__ __forceinline__ void xb_entry(int b, int nx, const int* __restrict__ axb, const double* __restrict__ par,
                                         const int* __restrict__ slot0, const double* __restrict__ x,
                                         const double* __restrict__ hb_rad, double* __restrict__ slots,
                                         double* __restrict__ e_out) {
    if (b >= nx) return;
    int A = axb[3 * b], X = axb[3 * b + 1], B = axb[3 * b + 2];
    const double* p = par + 3 * b;
    double3 pA = ld3(x, A), pX = ld3(x, X), pB = ld3(x, B);
    double3 vax = pX - pA, vxb = pB - pX, vab = pB - pA;
    double rax = nrm(vax), rxb = nrm(vxb), rab = nrm(vab);
    double3 z3 = make_double3(0, 0, 0), gA = z3, gX = z3, gB = z3;
    double E = 0.0;
    double radab = hb_rad[A] + hb_rad[B];
    double ex = 70.0 * ((rax + rxb) / rab - 1.0);
    if (!(rxb > 20.0) && !(ex > 15.0)) {
        double ts = pow(5.0 * radab / (rxb * rxb), 6.0), tl = pow(rxb * rxb / 70.0, 6.0);
        double fs = 1.0 / (1.0 + ts), fl = 1.0 / (1.0 + tl);
        double fo = 2.0 / (1.0 + exp(ex));
        double eX = exp(15.0 * p[1]), eB = exp(15.0 * -p[2]);
        double QX = eX / (eX + 0.03), QB = eB / (eB + 0.03);
        double r3 = rxb * rxb * rxb;
        double Rd = fs * fl * fo / r3;
        double pre = -QB * p[0] * QX;
        E = pre * Rd;
        double dfs = -2.0 * 6.0 * fs * ts / (rxb * (1.0 + ts));
        double dfl = -2.0 * 6.0 * rxb * fl * tl / (70.0 * (1.0 + tl));
        double et = exp(ex), de = (1.0 + et) * (1.0 + et);
        double dfo_ax = -2.0 * et * 70.0 / (rab * de);
        double dfo_ab = 2.0 * et * 70.0 * (rax + rxb) / (rab * rab * de);
        double dR_xb = (dfs * fl * fo + fs * dfl * fo + fs * fl * dfo_ax) / r3 - 3.0 * Rd / rxb;
        double gxb = pre * dR_xb / (rxb + 1e-14), gax = pre * (fs * fl * dfo_ax / r3) / (rax + 1e-14);
        double gab = pre * (fs * fl * dfo_ab / r3) / (rab + 1e-14);
        gA = (-gax) * vax + (-gab) * vab;
        gX = gax * vax + (-gxb) * vxb;
        gB = gxb * vxb + gab * vab;
    }
    e_out[b] = E;
    int s0 = slot0[b];
    st3(slots, s0, gA);
    st3(slots, s0 + 1, gX);
    st3(slots, s0 + 2, gB);
}

// Case-1 triplet (H bonded to neither A nor B): the cs = 1 path of hb_core
// without the neighbour, lone-pair and carbonyl factors (all 1).  T = double
// is the reference arithmetic; T = float (mixed path) forms the coordinate
// differences in FP64 and evaluates the term in FP32 with hardware rsqrt,
// rcp and exp.
// The FP64 cores are bound by instruction issue: a divide or square-root
// sequence is 14 and 20 of their FP64 instructions, the refined estimates
// (about 1 ulp) 4 for the reciprocal and 8 for the square root.
__device__ inline double hb_sqrt(double v) { return v * rsqrt_c(fmax(v, 1e-300)); }
__device__ inline float hb_sqrt(float v) { return __builtin_sqrtf(v); }
__device__ inline double hb_rcp(double v) { return rcp_c(v); }
__device__ inline float hb_rcp(float v) { return __builtin_amdgcn_rcpf(v); }
__device__ inline double hb_exp(double v) { return exp(v); }
__device__ inline float hb_exp(float v) { return __expf(v); }
// r_AB <= 50 Bohr; FP64 on the square, as r is within rounding of the root, not the rounded root
__device__ inline bool hb_near(double rab2, double) { return rab2 <= 2500.0; }
__device__ inline bool hb_near(float, float rAB) { return rAB <= 50.0f; }
template <typename T>
struct V3 {
    T x, y, z;
};
template <typename T>
__device__ inline V3<T> v3(double3 d) {
    return {(T)d.x, (T)d.y, (T)d.z};
}
template <typename T>
__device__ inline double3 d3(T s, V3<T> v) {
    return make_double3((double)(s * v.x), (double)(s * v.y), (double)(s * v.z));
}
// per-atom HB parameters of a triplet: FP64 arrays for the FP64 cores, the
// packed FP32 copies (two 16-byte loads and one 4-byte load) for T = float
template <typename T>
__device__ inline void hb_params(int A, int H, int B, const HBArgs& a, T& basA, T& basB, T& aciA, T& aciB, T& QH,
                                 T& QA, T& QB, T& radab) {
    if constexpr (sizeof(T) == sizeof(float)) {
        const float4 pa = a.pk[A], pb = a.pk[B];
        basA = pa.x;
        aciA = pa.y;
        QA = pa.z;
        basB = pb.x;
        aciB = pb.y;
        QB = pb.z;
        radab = pa.w + pb.w;
        QH = a.qh32[H];
    } else {
        basA = a.cb[A];
        basB = a.cb[B];
        aciA = a.ca[A];
        aciB = a.ca[B];
        QH = a.Qh[H];
        QA = a.Qab[A];
        QB = a.Qab[B];
        radab = a.hb_rad[A] + a.hb_rad[B];
    }
}
template <typename T>
__device__ double hb_core1(int A, int H, int B, const HBArgs& a, const double* __restrict__ x, double3& ga,
                           double3& gh, double3& gb) {
    const double3 z3 = make_double3(0, 0, 0);
    ga = z3;
    gh = z3;
    gb = z3;
    const double3 pA = ld3(x, A), pH = ld3(x, H), pB = ld3(x, B);
    // difference vectors drah = A - H, drbh = B - H, drab = A - B
    const V3<T> drah = v3<T>(pA - pH), drbh = v3<T>(pB - pH), drab = v3<T>(pA - pB);
    const T rah2 = drah.x * drah.x + drah.y * drah.y + drah.z * drah.z;
    const T rbh2 = drbh.x * drbh.x + drbh.y * drbh.y + drbh.z * drbh.z;
    const T rab2 = drab.x * drab.x + drab.y * drab.y + drab.z * drab.z;
    const T rAH = hb_sqrt(rah2), rHB = hb_sqrt(rbh2), rAB = hb_sqrt(rab2);
    if (!hb_near(rab2, rAB)) return 0.0;
    T basA, basB, aciA, aciB, QH, QA, QB, radab;
    hb_params<T>(A, H, B, a, basA, basB, aciA, aciB, QH, QA, QB, radab);
    const T rAH4 = rah2 * rah2, rHB4 = rbh2 * rbh2;
    const T den = hb_rcp(rAH4 + rHB4);
    const T bas = (QA * basA * rAH4 + QB * basB * rHB4) * den;
    const T aci = (aciB * rAH4 + aciA * rHB4) * den;
    const T irab2 = hb_rcp(rab2), irAB = hb_rcp(rAB);
    const T t3 = T(22) * radab * irab2, t1 = rab2 * T(1.0 / 85.0);
    const T ratio3 = (t3 * t3) * (t3 * t3) * (t3 * t3), ratio1 = (t1 * t1) * (t1 * t1) * (t1 * t1);
    const T denv = hb_rcp(T(1) + ratio3) * hb_rcp(T(1) + ratio1);
    const T c49 = T(49) * hb_rcp(radab);
    const T expo0 = c49 * ((rAH + rHB) * irAB - T(1));
    const T doutl = (expo0 > T(15)) ? T(0) : T(2) * hb_rcp(T(1) + hb_exp(expo0));
    const T rdamp = denv * irab2 * irAB;
    const T qhoutl = QH * doutl;
    const double E = (double)(-bas * aci * rdamp * qhoutl);
    const T rahprbh = rAH + rHB + T(1e-12);
    const T ddamp = (T(-12) * ratio1 * hb_rcp(T(1) + ratio1)) + (T(12) * ratio3 * hb_rcp(T(1) + ratio3));
    const T expo = c49 * (rahprbh * irAB - T(1));
    if (expo > T(15)) return E;
    const T ratio2 = hb_exp(expo);
    const T caa = QA * basA, cbb = QB * basB;
    const T rterm = -aci * rdamp * qhoutl, dterm = -aci * bas * qhoutl, sterm = -rdamp * bas * qhoutl;
    const T aterm = -aci * bas * rdamp * QH;
    const T tmp = den * den * T(4);
    const T dd24a = rah2 * rHB4 * tmp, dd24b = rbh2 * rAH4 * tmp;
    // coefficients of drah, drbh, drab in the gradient on A and B (H: minus the sum)
    // expo / (rAH + rHB - rAB) = 49 / (radab rAB): the reference divides the two
    // (with a 1e-12 guard); the closed form stays finite for collinear A-H-B
    const T ie2 = hb_rcp((T(1) + ratio2) * (T(1) + ratio2)), eir = c49 * irAB;
    const T gi1 = rdamp * (ddamp - T(3)) * irab2 * dterm;
    const T gi2 = aterm * T(2) * ratio2 * eir * rahprbh * ie2 * irab2;
    const T to = T(-2) * aterm * ratio2 * ie2 * eir;
    const T cah = (caa - cbb) * dd24a * rterm + (aciB - aciA) * dd24a * sterm + to * hb_rcp(rAH);
    const T cbh = (cbb - caa) * dd24b * rterm + (aciA - aciB) * dd24b * sterm + to * hb_rcp(rHB);
    const T cab = gi1 + gi2;
    ga = make_double3((double)(cah * drah.x + cab * drab.x), (double)(cah * drah.y + cab * drab.y),
                      (double)(cah * drah.z + cab * drab.z));
    gb = make_double3((double)(cbh * drbh.x - cab * drab.x), (double)(cbh * drbh.y - cab * drab.y),
                      (double)(cbh * drbh.z - cab * drab.z));
    gh = make_double3(-(double)(cah * drah.x + cbh * drbh.x), -(double)(cah * drah.y + cbh * drbh.y),
                      -(double)(cah * drah.z + cbh * drbh.z));
    return E;
}

// Case-2 triplet (acceptor B with covalent neighbours, no lone-pair or
// carbonyl factor): the cs = 2 path of hb_core in the arithmetic of
// hb_core1 (T = float on the mixed path: FP64 coordinate differences, FP32
// terms).  The quotients expo / (rAH + rHB - rAB) and ex_k / (s_k - rAB) are
// taken in closed form, 49 / (radab rAB) and cnb / rAB.  xs[k]: gradient on
// the k-th neighbour of B.
template <typename T>
__device__ double hb_core2(int A, int H, int B, const HBArgs& a, const double* __restrict__ x, double3& ga,
                           double3& gh, double3& gb, double* __restrict__ xs) {
    const double3 z3 = make_double3(0, 0, 0);
    ga = z3;
    gh = z3;
    gb = z3;
    const int nb0 = a.nb_off[B], nb1 = a.nb_off[B + 1];
    const double3 pA = ld3(x, A), pH = ld3(x, H), pB = ld3(x, B);
    const V3<T> drah = v3<T>(pA - pH), drbh = v3<T>(pB - pH), drab = v3<T>(pA - pB);
    const T rah2 = drah.x * drah.x + drah.y * drah.y + drah.z * drah.z;
    const T rbh2 = drbh.x * drbh.x + drbh.y * drbh.y + drbh.z * drbh.z;
    const T rab2 = drab.x * drab.x + drab.y * drab.y + drab.z * drab.z;
    const T rAH = hb_sqrt(rah2), rHB = hb_sqrt(rbh2), rAB = hb_sqrt(rab2);
    double E = 0.0;
    bool written = false;
    if (hb_near(rab2, rAB)) {
        T basA, basB, aciA, aciB, QH, QA, QB, radab;
        hb_params<T>(A, H, B, a, basA, basB, aciA, aciB, QH, QA, QB, radab);
        const T irab2 = hb_rcp(rab2), irAB = hb_rcp(rAB), irHB = hb_rcp(rHB), irbh2 = irHB * irHB;
        const T t3 = T(22) * radab * irab2, t1 = rab2 * T(1.0 / 85.0);
        const T ratio3 = (t3 * t3) * (t3 * t3) * (t3 * t3), ratio1 = (t1 * t1) * (t1 * t1) * (t1 * t1);
        const T denv = hb_rcp(T(1) + ratio3) * hb_rcp(T(1) + ratio1);
        const T irad = hb_rcp(radab), c49 = T(49) * irad;
        const T expo0 = c49 * ((rAH + rHB) * irAB - T(1));
        const T doutl = (expo0 > T(15)) ? T(0) : T(2) * hb_rcp(T(1) + hb_exp(expo0));
        const T cnb = ((a.Z[B] == 7 && nb1 - nb0 == 1) ? T(2.0) : T(11.20)) * irad;
        T outl_nb = T(1);
        for (int k = nb0; k < nb1; ++k) {
            const double3 pn = ld3(x, a.nb_idx[k]);
            const V3<T> dan = v3<T>(pA - pn), dbn = v3<T>(pB - pn);
            const T sm = hb_sqrt(dan.x * dan.x + dan.y * dan.y + dan.z * dan.z) +
                         hb_sqrt(dbn.x * dbn.x + dbn.y * dbn.y + dbn.z * dbn.z);
            const T ex = cnb * (sm * irAB - T(1));
            outl_nb *= T(2) * hb_rcp(T(1) + hb_exp(-ex)) - T(1);
        }
        const T rbhdamp = denv * T(1.8) * irbh2 * irHB, rabdamp = denv * T(-0.8) * irab2 * irAB;
        const T rdamp = rbhdamp + rabdamp;
        const T cval = aciA * basB * QA * QB * T(0.268);
        const T qhoutl = QH * doutl * outl_nb;
        E = (double)(-rdamp * qhoutl * cval);
        const T rahprbh = rAH + rHB + T(1e-12);
        const T ddamp = (T(-12) * ratio1 * hb_rcp(T(1) + ratio1)) + (T(12) * ratio3 * hb_rcp(T(1) + ratio3));
        const T expo = c49 * (rahprbh * irAB - T(1));
        if (!(expo > T(15))) {
            written = true;
            const T ratio2 = hb_exp(expo);
            const T dterm = -qhoutl * cval, aterm = -rdamp * QH * outl_nb * cval;
            const T nbterm = -rdamp * QH * doutl * cval;
            const T ie2 = hb_rcp((T(1) + ratio2) * (T(1) + ratio2));
            const T tmp1 = T(-2) * aterm * ratio2 * ie2 * c49 * irAB;
            // coefficients of drab (A: +, B: -), drah (A: +, H: -), drbh (B: +, H: -)
            T cab = ((rabdamp + rbhdamp) * ddamp - T(3) * rabdamp) * irab2 * dterm - tmp1 * rahprbh * irab2;
            const T cah = tmp1 * hb_rcp(rAH);
            const T cbh = T(-3) * rbhdamp * irbh2 * dterm + tmp1 * irHB;
            T gax = T(0), gay = T(0), gaz = T(0), gbx = T(0), gby = T(0), gbz = T(0);
            int kk = 0;
            for (int k = nb0; k < nb1; ++k, ++kk) {
                const double3 pn = ld3(x, a.nb_idx[k]);
                const V3<T> dan = v3<T>(pA - pn), dbn = v3<T>(pB - pn);
                const T ranb = hb_sqrt(dan.x * dan.x + dan.y * dan.y + dan.z * dan.z);
                const T rbnb = hb_sqrt(dbn.x * dbn.x + dbn.y * dbn.y + dbn.z * dbn.z);
                const T sm = ranb + rbnb + T(1e-12);
                const T ex = cnb * (sm * irAB - T(1));
                const T r2n = hb_exp(-ex), ir = hb_rcp(T(1) + r2n);
                const T oi = T(2) * ir - T(1);
                const T others = (fabs(oi) > T(1e-12)) ? outl_nb * hb_rcp(oi) : T(1);
                const T tmp2 = T(2) * nbterm * others * r2n * ir * ir * cnb * irAB;
                cab -= tmp2 * sm * irab2;
                const T fa = tmp2 * hb_rcp(ranb), fb = tmp2 * hb_rcp(rbnb);
                gax += fa * dan.x;
                gay += fa * dan.y;
                gaz += fa * dan.z;
                gbx += fb * dbn.x;
                gby += fb * dbn.y;
                gbz += fb * dbn.z;
                st3(xs, kk, make_double3(-(double)(fa * dan.x + fb * dbn.x), -(double)(fa * dan.y + fb * dbn.y),
                                         -(double)(fa * dan.z + fb * dbn.z)));
            }
            ga = make_double3((double)(cah * drah.x + cab * drab.x + gax), (double)(cah * drah.y + cab * drab.y + gay),
                              (double)(cah * drah.z + cab * drab.z + gaz));
            gb = make_double3((double)(cbh * drbh.x - cab * drab.x + gbx), (double)(cbh * drbh.y - cab * drab.y + gby),
                              (double)(cbh * drbh.z - cab * drab.z + gbz));
            gh = make_double3(-(double)(cah * drah.x + cbh * drbh.x), -(double)(cah * drah.y + cbh * drbh.y),
                              -(double)(cah * drah.z + cbh * drbh.z));
        }
    }
    if (!written)
        for (int kk = 0; kk < nb1 - nb0; ++kk) st3(xs, kk, z3);
    return E;
}

// Case-1 hydrogen bonds by role: the case-1 triplets are kept three times,
// grouped by the atom in role A, H or B (entries: the other two atoms), each
// group cut into chunks of at most HB_CHUNK triplets.  One wavefront per
// chunk evaluates every triplet of its chunk (lanes
// stride the chunk; a triplet is evaluated once per role, which costs less
// than storing and gathering per-triplet gradients), adds the gradient on its
// own atom (and, for role A, the energy) with a fixed butterfly and writes
// one result per chunk.
constexpr int HB_CHUNK = 256;
struct HBRoles {
    const int2* ent;
    const int* goff;    // [ngt + 1]
    const int* gatom;   // [ngt]
    int ng0, ng1, ngt;  // role A chunks [0, ng0), H [ng0, ng1), B [ng1, ngt)
};
template <int ROLE, typename T>
__device__ __forceinline__ void hb_role_chunk(int w, const HBRoles& r, const HBArgs& a, const double* __restrict__ x,
                                              double* __restrict__ gout, double* __restrict__ egrp) {
    const int lane = threadIdx.x & 63;
    const int g1 = (ROLE == 0) ? r.ng0 : (ROLE == 1 ? r.ng1 : r.ngt);
    if (w >= g1) return;
    const int at = r.gatom[w], e0 = r.goff[w], e1 = r.goff[w + 1];
    double3 g = make_double3(0, 0, 0);
    double E = 0.0;
    for (int e = e0 + lane; e < e1; e += 64) {
        const int2 en = r.ent[e];
        double3 ga, gh, gb;
        if (ROLE == 0) {
            E += hb_core1<T>(at, en.x, en.y, a, x, ga, gh, gb);
            g = g + ga;
        } else if (ROLE == 1) {
            hb_core1<T>(en.x, at, en.y, a, x, ga, gh, gb);
            g = g + gh;
        } else {
            hb_core1<T>(en.x, en.y, at, a, x, ga, gh, gb);
            g = g + gb;
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        g.x += __shfl_xor(g.x, o);
        g.y += __shfl_xor(g.y, o);
        g.z += __shfl_xor(g.z, o);
        if (ROLE == 0) E += __shfl_xor(E, o);
    }
    if (lane == 0) {
        st3(gout, w, g);
        if (ROLE == 0) egrp[w] = E;
    }
}

// the three roles in one launch (four chunks per workgroup, a role's last
// workgroup partly idle): the roles' tails overlap
template <typename T>
__global__ __launch_bounds__(256) void k_hb_roles(HBRoles r, HBArgs a, const double* __restrict__ x,
                                                  double* __restrict__ gout, double* __restrict__ egrp) {
    const int b0 = (r.ng0 + 3) / 4, b1 = b0 + (r.ng1 - r.ng0 + 3) / 4, wv = threadIdx.x >> 6;
    const int blk = blockIdx.x;
    if (blk < b0)
        hb_role_chunk<0, T>(blk * 4 + wv, r, a, x, gout, egrp);
    else if (blk < b1)
        hb_role_chunk<1, T>(r.ng0 + (blk - b0) * 4 + wv, r, a, x, gout, egrp);
    else
        hb_role_chunk<2, T>(r.ng1 + (blk - b1) * 4 + wv, r, a, x, gout, egrp);
}

// Hydrogen bonds of cases 2-4, one thread each: energy, and the gradient in
// the triplet's slots s0 (A), s0 + 1 (H), s0 + 2 (B), s0 + 3 + k (k-th
// neighbour of B), then the carbonyl's D atoms.  MODE 0: every entry by the
// general FP64 core; MODE 1: case-2 entries only, by hb_core2<T> (FP32 terms
// on the mixed path); MODE 2: entries of cases 3 and 4 only, FP64.  ord (MODE 1
// and 2): the entries of the mode, case 2 first, so that no lane idles on
// an entry of the other mode; nh counts the mode's entries.
// Bound by FP64 instruction issue.  The general core holds 256 VGPRs (two
// wavefronts per SIMD) and divides throughout; the lean one 152.  With it and
// the estimates of hb_rcp in the case-1 roles an FP64 evaluation of 9000
// atoms of water goes 1258 -> 1236 us, of 4096 molecules 7.14 -> 7.10 ms.
template <typename T, int MODE>
__global__ __launch_bounds__(256, 2) void k_hb_full(int nh, const int* __restrict__ ord, const int4* __restrict__ ahbc,
                                                 const int* __restrict__ slot0, HBArgs a, const double* __restrict__ x,
                                                 double* __restrict__ slots, double* __restrict__ e_out) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nh) return;
    const int h = MODE == 0 ? k : ord[k];
    const int4 t = ahbc[h];
    const int s0 = slot0[h];
    double3 ga, gh, gb;
    double* xs = slots + 3 * ((size_t)s0 + 3);
    if ((MODE == 1 && t.w != 2) || (MODE == 2 && t.w == 2)) return;
    if (MODE == 1)
        e_out[h] = hb_core2<T>(t.x, t.y, t.z, a, x, ga, gh, gb, xs);
    else
        e_out[h] = hb_core<true>(t.x, t.y, t.z, t.w, a, x, ga, gh, gb, xs);
    st3(slots, s0, ga);
    st3(slots, s0 + 1, gh);
    st3(slots, s0 + 2, gb);
}

// per-atom hydrogen-bond gradient, one wavefront per atom: the atom's
// case-1 chunk results in roles A, H, B (chunks [crange[r (n + 1) + i],
// crange[r (n + 1) + i + 1])) and its slots of cases 2-4; lanes stride the
// lists, fixed butterfly
struct HBGather {
    const int* crange;  // nullptr: no hydrogen bonds
    const double* gout;
    const int *xoff, *xidx;
    const double* xslots;
};
template <int LPA>
__device__ __forceinline__ double3 hb_gather(int i, int lane, int n, const HBGather& h) {
    double3 s = make_double3(0, 0, 0);
#pragma unroll
    for (int role = 0; role < 3; ++role) {
        const int* cr = h.crange + role * (n + 1);
        for (int k = cr[i] + lane; k < cr[i + 1]; k += LPA) s = s + ld3(h.gout, k);
    }
    for (int k = h.xoff[i] + lane; k < h.xoff[i + 1]; k += LPA) s = s + ld3(h.xslots, h.xidx[k]);
    return s;
}
template <int LPA>
__global__ __launch_bounds__(256) void k_hb_gather(int n, HBGather h, double* __restrict__ g) {
    const int lane = threadIdx.x & (LPA - 1);
    const int i = blockIdx.x * (256 / LPA) + threadIdx.x / LPA;
    if (i >= n) return;
    double3 s = hb_gather<LPA>(i, lane, n, h);
#pragma unroll
    for (int o = LPA / 2; o > 0; o >>= 1) {
        s.x += __shfl_xor(s.x, o);
        s.y += __shfl_xor(s.y, o);
        s.z += __shfl_xor(s.z, o);
    }
    if (lane == 0) st3(g, i, s);
}

// D4 ATM over bonded triplets (energy +c9, gradient -c9 as in
// ff_workspace_gfnff.cpp:1526-1658) and bonded ATM (:1665-1739)
__device__ inline double c6_pair(int i, int j, int ne, const int* elem, const int* nref, const double* c6ref,
                                 const double* gw) {
    int ei = elem[i], ej = elem[j];
    const double* c = c6ref + ((size_t)ei * ne + ej) * 49;
    double s = 0.0;
    for (int a = 0; a < nref[ei]; ++a)
        for (int b = 0; b < nref[ej]; ++b) s += gw[(size_t)i * 7 + a] * gw[(size_t)j * 7 + b] * c[a * 7 + b];
    return s;
}

__device__ __forceinline__ void atm_entry(int t, int nt, const int* __restrict__ ijk, const double* __restrict__ sc,
                                          const int* __restrict__ slot0, const double* __restrict__ x,
                                          const double* __restrict__ rcov_d3, int ne, const int* __restrict__ elem,
                                          const int* __restrict__ nref, const double* __restrict__ c6ref,
                                          const double* __restrict__ gw, double* __restrict__ slots,
                                          double* __restrict__ e_out) {
    if (t >= nt) return;
    int i = ijk[3 * t], j = ijk[3 * t + 1], k = ijk[3 * t + 2];
    double c9 = sqrt(fabs(c6_pair(i, j, ne, elem, nref, c6ref, gw) * c6_pair(i, k, ne, elem, nref, c6ref, gw) *
                          c6_pair(j, k, ne, elem, nref, c6ref, gw)));
    double3 vij = ld3(x, j) - ld3(x, i), vik = ld3(x, k) - ld3(x, i), vjk = ld3(x, k) - ld3(x, j);
    double rij = nrm(vij), rik = nrm(vik), rjk = nrm(vjk);
    double r2ij = rij * rij, r2ik = rik * rik, r2jk = rjk * rjk;
    double r0ij = 0.58 * sqrt(3.0 * rcov_d3[i] * rcov_d3[j]) + 4.80;
    double r0ik = 0.58 * sqrt(3.0 * rcov_d3[i] * rcov_d3[k]) + 4.80;
    double r0jk = 0.58 * sqrt(3.0 * rcov_d3[j] * rcov_d3[k]) + 4.80;
    double rijk = rij * rik * rjk, r2ijk = r2ij * r2ik * r2jk, r3ijk = rijk * r2ijk, r5ijk = r2ijk * r3ijk;
    double tmp = pow(r0ij * r0ik * r0jk / rijk, 14.0 / 3.0);
    double fdmp = 1.0 / (1.0 + 6.0 * tmp);
    double Aa = r2ij + r2jk - r2ik, Bb = r2ij + r2ik - r2jk, Cc = r2ik + r2jk - r2ij;
    double ang = (0.375 * Aa * Bb * Cc / r2ijk + 1.0) / r3ijk;
    double s = sc[t];
    e_out[t] = ang * fdmp * c9 / 3.0 * s;
    double dfdmp = -2.0 * 14.0 * tmp * fdmp * fdmp;
    double dij = -0.375 * (cube(r2ij) + sq(r2ij) * (r2jk + r2ik) +
                           r2ij * (3.0 * sq(r2jk) + 2.0 * r2jk * r2ik + 3.0 * sq(r2ik)) -
                           5.0 * sq(r2jk - r2ik) * (r2jk + r2ik)) / r5ijk;
    double dik = -0.375 * (cube(r2ik) + sq(r2ik) * (r2jk + r2ij) +
                           r2ik * (3.0 * sq(r2jk) + 2.0 * r2jk * r2ij + 3.0 * sq(r2ij)) -
                           5.0 * sq(r2jk - r2ij) * (r2jk + r2ij)) / r5ijk;
    double djk = -0.375 * (cube(r2jk) + sq(r2jk) * (r2ik + r2ij) +
                           r2jk * (3.0 * sq(r2ik) + 2.0 * r2ik * r2ij + 3.0 * sq(r2ij)) -
                           5.0 * sq(r2ik - r2ij) * (r2ik + r2ij)) / r5ijk;
    double pre = -c9 * s / 3.0;
    double a1 = pre * (-dij * fdmp + ang * dfdmp) / r2ij, a2 = pre * (-dik * fdmp + ang * dfdmp) / r2ik,
           a3 = pre * (-djk * fdmp + ang * dfdmp) / r2jk;
    int q = slot0[t];
    st3(slots, q, (-1.0) * (a1 * vij + a2 * vik));
    st3(slots, q + 1, a1 * vij + (-a3) * vjk);
    st3(slots, q + 2, a2 * vik + a3 * vjk);
}

__device__ __forceinline__ void batm_entry(int t, int nt, const int* __restrict__ ijk, const double* __restrict__ zb,
                                           const int* __restrict__ slot0, const double* __restrict__ x,
                                           const double* __restrict__ qa, double* __restrict__ slots,
                                           double* __restrict__ e_out) {
    if (t >= nt) return;
    int i = ijk[3 * t], j = ijk[3 * t + 1], k = ijk[3 * t + 2];
    double3 vij = ld3(x, j) - ld3(x, i), vik = ld3(x, k) - ld3(x, i), vjk = ld3(x, k) - ld3(x, j);
    double r2ij = dot(vij, vij), r2jk = dot(vjk, vjk), r2ik = dot(vik, vik);
    double rij = sqrt(r2ij), rjk = sqrt(r2jk), rik = sqrt(r2ik);
    double rijk3 = r2ij * r2jk * r2ik;
    double mijk = -r2ij + r2jk + r2ik, imjk = r2ij - r2jk + r2ik, ijmk = r2ij + r2jk - r2ik;
    double ang = 0.375 * ijmk * imjk * mijk / rijk3;
    double rav3 = rijk3 * sqrt(rijk3);
    double angr9 = (ang + 1.0) / rav3;
    double fi = fmin(fmax(1.0 - 3.0 * qa[i], -4.0), 4.0);
    double fj = fmin(fmax(1.0 - 3.0 * qa[j], -4.0), 4.0);
    double fk = fmin(fmax(1.0 - 3.0 * qa[k], -4.0), 4.0);
    double c9 = fi * fj * fk * zb[3 * t] * zb[3 * t + 1] * zb[3 * t + 2];
    e_out[t] = c9 * angr9;
    double dij = -0.375 * (cube(r2ij) + sq(r2ij) * (r2jk + r2ik) +
                           r2ij * (3.0 * sq(r2jk) + 2.0 * r2jk * r2ik + 3.0 * sq(r2ik)) -
                           5.0 * sq(r2jk - r2ik) * (r2jk + r2ik)) / (rij * rijk3 * rav3);
    double djk = -0.375 * (cube(r2jk) + sq(r2jk) * (r2ik + r2ij) +
                           r2jk * (3.0 * sq(r2ik) + 2.0 * r2ik * r2ij + 3.0 * sq(r2ij)) -
                           5.0 * sq(r2ik - r2ij) * (r2ik + r2ij)) / (rjk * rijk3 * rav3);
    double dik = -0.375 * (cube(r2ik) + sq(r2ik) * (r2jk + r2ij) +
                           r2ik * (3.0 * sq(r2jk) + 2.0 * r2jk * r2ij + 3.0 * sq(r2ij)) -
                           5.0 * sq(r2jk - r2ij) * (r2jk + r2ij)) / (rik * rijk3 * rav3);
    double3 gij = (-dij * c9 / rij) * vij, gjk = (-djk * c9 / rjk) * vjk, gik = (-dik * c9 / rik) * vik;
    int q = slot0[t];
    st3(slots, q, gij + gik);                 // i
    st3(slots, q + 1, (-1.0) * gij + gjk);    // j
    st3(slots, q + 2, (-1.0) * (gik + gjk));  // k
}

// Every list term that needs only coordinates, CN and D4 weights, the D4 half
// contraction and the reduced EEQ right-hand side in one launch: the lists are
// short next to the chip (hundreds of entries for 100 atoms, one wavefront or
// two per list and SIMD), and ten launches of 4 to 18 us in a row took 60 to
// 90 us where the longest single chain, a torsion's or an ATM triple's, takes
// about 16.  Workgroups are dealt to the lists in the order below, the
// longest chains first.  Launches of many workgroups are bound by throughput
// instead: there each list runs in a launch of its own with its own register
// count (the torsions' 114 registers hold the fused kernel at four wavefronts
// per SIMD): 4096 molecules, 52,000 workgroups, 6.51 against 6.65 ms fused;
// 122 to 1536 atoms, up to 500 workgroups, 331 -> 280 us fused on 512 H2O.
constexpr int TERMS_FUSED_MAX = 2048;
struct TermArgs {
    int end[12];  // workgroups of the sections 0 .. k
    int n, ne, nr, np;
    int nb_hb, nb_plain, nangle, ntors, ninv, nstors, nxb, nbrep, natm, nbatm;
    const double *x, *cn, *rcov_d3, *hb_rad, *gw, *dgw, *qa, *c6ref;
    const int *elem, *nref;
    const int *bsel_hb, *bsel_plain, *bond_ij, *bond_H, *bond_hboff, *bond_hbB, *bond_slot;
    const double* bond_par;
    const int *ang_ijk, *ang_slot, *tor_ijkl, *tor_slot, *inv_ijkl, *inv_slot, *st_ijkl, *st_slot, *xb_axb, *xb_slot;
    const double *ang_par, *tor_par, *inv_par, *st_par, *xb_par;
    const int *brep_ij, *brep_slot, *atm_ijk, *atm_slot, *batm_ijk, *batm_slot;
    const double *brep_par, *atm_sc, *batm_zb;
    double *slots, *dcn_slot, *e_bond, *e_ang, *e_tor, *e_inv, *e_st, *e_xb, *e_brep, *e_atm, *e_batm;
    double *h6, *dh6;
    const int *red_atom, *red_last;
    const double* rhs;
    double* b;
};
// ONE >= 0: that section alone (blockIdx.x counts its workgroups)
template <int ONE>
__global__ __launch_bounds__(256) void k_terms(TermArgs a) {
    int sec = ONE, first = 0;
    if (ONE < 0) {
        sec = 0;
#pragma unroll
        for (int k = 0; k < 11; ++k)
            if ((int)blockIdx.x >= a.end[k]) {
                sec = k + 1;
                first = a.end[k];
            }
    }
    const int blk = blockIdx.x - first, t = blk * 256 + threadIdx.x;
    switch (sec) {
        case 0:
            atm_entry(t, a.natm, a.atm_ijk, a.atm_sc, a.atm_slot, a.x, a.rcov_d3, a.ne, a.elem, a.nref, a.c6ref, a.gw,
                      a.slots, a.e_atm);
            break;
        case 1:
            torsion_entry(t, a.ntors, a.tor_ijkl, a.tor_par, a.tor_slot, a.x, a.rcov_d3, a.slots, a.e_tor);
            break;
        case 2:
            bond_hb_wave(blk * 4 + (threadIdx.x >> 6), a.nb_hb, a.bsel_hb, a.bond_ij, a.bond_par, a.bond_hboff,
                         a.bond_hbB, a.bond_slot, a.x, a.cn, a.rcov_d3, a.bond_H, a.slots, a.dcn_slot, a.e_bond);
            break;
        case 3:
            inversion_entry(t, a.ninv, a.inv_ijkl, a.inv_par, a.inv_slot, a.x, a.rcov_d3, a.slots, a.e_inv);
            break;
        case 4:
            stors_entry(t, a.nstors, a.st_ijkl, a.st_par, a.st_slot, a.x, a.slots, a.e_st);
            break;
        case 5:
            xb_entry(t, a.nxb, a.xb_axb, a.xb_par, a.xb_slot, a.x, a.hb_rad, a.slots, a.e_xb);
            break;
        case 6:
            angle_entry(t, a.nangle, a.ang_ijk, a.ang_par, a.ang_slot, a.x, a.rcov_d3, a.slots, a.e_ang);
            break;
        case 7:
            batm_entry(t, a.nbatm, a.batm_ijk, a.batm_zb, a.batm_slot, a.x, a.qa, a.slots, a.e_batm);
            break;
        case 8:
            brep_entry(t, a.nbrep, a.brep_ij, a.brep_par, a.brep_slot, a.x, a.slots, a.e_brep);
            break;
        case 9:
            bond_plain(t, a.nb_plain, a.bsel_plain, a.bond_ij, a.bond_par, a.bond_slot, a.bond_H, a.x, a.cn, a.slots,
                       a.dcn_slot, a.e_bond);
            break;
        case 10:
            d4_half_entry(t, a.n, a.ne, a.elem, a.nref, a.c6ref, a.gw, a.dgw, a.h6, a.dh6);
            break;
        default:
            rhs_reduce_entry(t, a.nr, a.np, a.red_atom, a.red_last, a.rhs, a.b);
            break;
    }
}

// ---------------------------------------------------------------------------
// K11: batches of independent molecules (one launch per kernel for the whole
// batch).  Molecule m owns atoms [mol_off[m], mol_off[m+1]); every all-pairs
// loop is restricted to the molecule, the bonded lists are concatenated.  Its
// reduced EEQ system occupies the padded block [vo_m, vo_m + np_m) of the
// concatenated reduced index space, its matrix lies at A + mo_m (np_m x np_m,
// row-major) and the inverses of its diagonal blocks at Linv + vo_m NB.
// ---------------------------------------------------------------------------
constexpr int BATCH_MAX_NP = 512;  // largest padded reduced system of a batched molecule

// One 64 x 64 lower tile (m, bi, bj) of a molecule's reduced matrix per
// workgroup.  When the tile's rows share one last atom la and its columns
// one last atom lb (always within one fragment, so for every tile of a
// one-fragment molecule), the entries A(ia, lb), A(la, ib) and A(la, lb) are
// evaluated once per row, column and tile into LDS and every element needs
// one fresh A(ia, ib); the sum keeps the order of the direct four-term form,
// so R is the same bit for bit.  Other tiles use the direct form.  A32 (the
// mixed path) receives the same entries rounded to FP32.
__global__ __launch_bounds__(256) void k_eeq_reduced_batch(const int4* __restrict__ tiles, const int* __restrict__ mnr,
                                                           const int* __restrict__ mnp,
                                                           const long long* __restrict__ mo,
                                                           const int* __restrict__ vo, const int* __restrict__ ra,
                                                           const int* __restrict__ rl, const double* __restrict__ x,
                                                           const double* __restrict__ alp,
                                                           const double* __restrict__ diag, double* __restrict__ A,
                                                           float* __restrict__ A32) {
    __shared__ double urow[NB], wcol[NB];
    __shared__ double sll;
    const int4 tt = tiles[blockIdx.x];
    const int m = tt.x, bi = tt.y, bj = tt.z;
    const int nr = mnr[m], np = mnp[m], base = vo[m];
    const int tid = threadIdx.x;
    double* Am = A + mo[m];
    // shared last atoms of the tile's valid rows and columns (-1 when none is valid)
    const int r0 = bi * NB, c0 = bj * NB;
    const int la0 = r0 < nr ? rl[base + r0] : -1, lb0 = c0 < nr ? rl[base + c0] : -1;
    bool same = true;
    if (tid < NB) same = !(r0 + tid < nr) || rl[base + r0 + tid] == la0;
    else if (tid < 2 * NB) same = !(c0 + tid - NB < nr) || rl[base + c0 + tid - NB] == lb0;
    const bool uni = __syncthreads_and(same) && la0 >= 0 && lb0 >= 0;
    if (uni) {
        if (tid < NB) {
            const int r = r0 + tid;
            urow[tid] = r < nr ? eeq_a(ra[base + r], lb0, x, alp, diag) : 0.0;
        } else if (tid < 2 * NB) {
            const int c = c0 + tid - NB;
            wcol[tid - NB] = c < nr ? eeq_a(la0, ra[base + c], x, alp, diag) : 0.0;
        } else if (tid == 2 * NB) {
            sll = eeq_a(la0, lb0, x, alp, diag);
        }
        __syncthreads();
    }
    for (int e = tid; e < NB * NB; e += blockDim.x) {
        const int r = r0 + e / NB, c = c0 + e % NB;
        if (c > r) continue;
        double v;
        if (r >= nr || c >= nr) {
            v = (r == c) ? 1.0 : 0.0;
        } else if (uni) {
            v = eeq_a(ra[base + r], ra[base + c], x, alp, diag) - urow[e / NB] - wcol[e % NB] + sll;
        } else {
            const int ia = ra[base + r], la = rl[base + r], ib = ra[base + c], lb = rl[base + c];
            v = eeq_a(ia, ib, x, alp, diag) - eeq_a(ia, lb, x, alp, diag) - eeq_a(la, ib, x, alp, diag) +
                eeq_a(la, lb, x, alp, diag);
        }
        Am[(size_t)r * np + c] = v;
        if (A32) A32[mo[m] + (size_t)r * np + c] = (float)v;  // the mixed path factors this copy
    }
}

// ---- per-molecule factorisation: tile phases shared out over wavefronts ----
// One 64 x 64 output tile per wavefront on MFMA (v_mfma_f64_16x16x4f64 or
// v_mfma_f32_16x16x4f32), in two 32-row halves, operands read from memory
// (L2).  Lane layout: A(i = lane%16, k = lane/16), B(k = lane/16,
// j = lane%16); result element v of a 16 x 16 block at row 4 v + lane/16
// (FP64) or 4 (lane/16) + v (FP32), column lane%16.  Operands are read DEPTH 4-column steps
// ahead (the L2 latency exceeds one step's eight MFMAs); DEPTH 1 keeps the
// register footprint of three workgroups per CU.
//   SUB = true : A(ri.., rj..) -= P(ri.., 0..63) Q(rj.., 0..63)^T (trailing
//                update; P = Q = the panel, leading dimension ldq = np;
//                diagonal tiles keep the lower triangle)
//   SUB = false: A(ri.., rj..)  = P(ri.., 0..63) Q(0.., 0..63)^T (panel
//                solve, Q = the inverse of the diagonal block, ldq = 64)
template <typename T, bool SUB, int DEPTH>
__device__ __forceinline__ void batch_tile_mfma(T* __restrict__ Am, int np, int ri, int rj,
                                                const T* __restrict__ P, const T* __restrict__ Q, int ldq) {
    using M = MfmaT<T>;
    using V = typename M::V;
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    const bool lower_only = SUB && ri == rj;
#pragma unroll 1
    for (int h = 0; h < 2; ++h) {
        const T* Pi = P + (size_t)(32 * h) * np;
        V acc[2][4];
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 4; ++y) acc[x][y] = V{0, 0, 0, 0};
        if constexpr (DEPTH == 1) {
            // the next step's operands are loaded before the current step's MFMAs
            T fa[2], fb[4];
#pragma unroll
            for (int x = 0; x < 2; ++x) fa[x] = Pi[(size_t)(16 * x + li) * np + lk];
#pragma unroll
            for (int y = 0; y < 4; ++y) fb[y] = Q[(size_t)(16 * y + li) * ldq + lk];
#pragma unroll 2
            for (int kk = 0; kk < NB; kk += 4) {
                T na[2], nb[4];
                if (kk + 4 < NB) {
#pragma unroll
                    for (int x = 0; x < 2; ++x) na[x] = Pi[(size_t)(16 * x + li) * np + kk + 4 + lk];
#pragma unroll
                    for (int y = 0; y < 4; ++y) nb[y] = Q[(size_t)(16 * y + li) * ldq + kk + 4 + lk];
                }
#pragma unroll
                for (int x = 0; x < 2; ++x)
#pragma unroll
                    for (int y = 0; y < 4; ++y)
                        acc[x][y] = M::op(fa[x], fb[y], acc[x][y]);
                if (kk + 4 < NB) {
#pragma unroll
                    for (int x = 0; x < 2; ++x) fa[x] = na[x];
#pragma unroll
                    for (int y = 0; y < 4; ++y) fb[y] = nb[y];
                }
            }
        } else {
            // operands of DEPTH 4-column steps in flight (ring of registers)
            T fa[DEPTH][2], fb[DEPTH][4];
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) {
#pragma unroll
                for (int x = 0; x < 2; ++x) fa[d][x] = Pi[(size_t)(16 * x + li) * np + 4 * d + lk];
#pragma unroll
                for (int y = 0; y < 4; ++y) fb[d][y] = Q[(size_t)(16 * y + li) * ldq + 4 * d + lk];
            }
#pragma unroll
            for (int st = 0; st < NB / 4; ++st) {
                const int sl = st % DEPTH;
#pragma unroll
                for (int x = 0; x < 2; ++x)
#pragma unroll
                    for (int y = 0; y < 4; ++y)
                        acc[x][y] = M::op(fa[sl][x], fb[sl][y], acc[x][y]);
                if (st + DEPTH < NB / 4) {
                    const int kk = 4 * (st + DEPTH);
#pragma unroll
                    for (int x = 0; x < 2; ++x) fa[sl][x] = Pi[(size_t)(16 * x + li) * np + kk + lk];
#pragma unroll
                    for (int y = 0; y < 4; ++y) fb[sl][y] = Q[(size_t)(16 * y + li) * ldq + kk + lk];
                }
            }
        }
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 4; ++y)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int r = 32 * h + 16 * x + (M::kRowFromReg ? 4 * v + lk : 4 * lk + v), c = 16 * y + li;
                    T* p = Am + (size_t)(ri + r) * np + rj + c;
                    if (!SUB) *p = acc[x][y][v];
                    else if (!lower_only || c <= r) *p = *p - acc[x][y][v];
                }
    }
}

// The diagonal-block routine as a call of its own, so that its register
// footprint is not added to the state of the surrounding phases.
template <typename T>
__device__ __noinline__ void batch_diag_block(int np, int k0, T* __restrict__ A, T* __restrict__ Linv,
                                              int* __restrict__ flags, T (*S0)[NB + 1], T (*col)[NB], T* rdiag) {
    chol_diag_block<T>(np, k0, A, Linv, flags, S0, col, rdiag);
}

// z = L^-T L^-1 v for one molecule (blocked substitutions with the stored
// inverses of the diagonal blocks): v in vec (LDS, type T), result in vec.
template <typename T>
__device__ __forceinline__ void batch_substitute(int np, const T* __restrict__ Am, const T* __restrict__ Lm, T* vec,
                                                 T* tmp) {
    const int tid = threadIdx.x, t = tid >> 2, q = tid & 3, nb = np / NB;
    // forward: y_kb = Linv_kb (v_kb - sum_{k < kb} L(kb, k) y_k)
    for (int kb = 0; kb < nb; ++kb) {
        T acc = (q == 0) ? vec[kb * NB + t] : T(0);
        for (int k = 0; k < kb; ++k)
#pragma unroll
            for (int u = 0; u < NB / 4; ++u)
                acc -= Am[(size_t)(kb * NB + t) * np + k * NB + 4 * u + q] * vec[k * NB + 4 * u + q];
        acc += __shfl_xor(acc, 1);
        acc += __shfl_xor(acc, 2);
        if (q == 0) tmp[t] = acc;
        __syncthreads();
        const T* Li = Lm + (size_t)kb * NB * NB;
        T s = 0;
#pragma unroll
        for (int u = 0; u < NB / 4; ++u) s += Li[t * NB + 4 * u + q] * tmp[4 * u + q];
        s += __shfl_xor(s, 1);
        s += __shfl_xor(s, 2);
        if (q == 0) vec[kb * NB + t] = s;
        __syncthreads();
    }
    // backward: x_kb = Linv_kb^T (y_kb - sum_{k > kb} L(k, kb)^T x_k)
    for (int kb = nb - 1; kb >= 0; --kb) {
        T acc = (q == 0) ? vec[kb * NB + t] : T(0);
        for (int k = nb - 1; k > kb; --k)
#pragma unroll
            for (int u = 0; u < NB / 4; ++u)
                acc -= Am[(size_t)(k * NB + 4 * u + q) * np + kb * NB + t] * vec[k * NB + 4 * u + q];
        acc += __shfl_xor(acc, 1);
        acc += __shfl_xor(acc, 2);
        if (q == 0) tmp[t] = acc;
        __syncthreads();
        const T* Li = Lm + (size_t)kb * NB * NB;
        T s = 0;
#pragma unroll
        for (int u = 0; u < NB / 4; ++u) s += Li[(4 * u + q) * NB + t] * tmp[4 * u + q];
        s += __shfl_xor(s, 1);
        s += __shfl_xor(s, 2);
        if (q == 0) vec[kb * NB + t] = s;
        __syncthreads();
    }
}

// Factorisation of one molecule's reduced system per workgroup of four
// wavefronts, right-looking by 64-column blocks.  Step k: the workgroup
// factors the diagonal block and forms its inverse (chol_diag_block, a call
// of its own so that its registers do not add to the other phases'); the
// panel tiles L(i, k) = A(i, k) L(k, k)^-T and then the trailing tiles
// A(i, j) -= L(i, k) L(j, k)^T are computed one tile per wavefront on MFMA,
// dealt round-robin, with one barrier after each phase.  T = double factors
// the FP64 matrix in place; T = float (mixed path, batch_fp32 = 1) factors
// the FP32 copy.  The factorisation needs only the matrix, so it runs on the
// side stream right after the matrix build, alongside CN and the bonded
// terms; the substitutions (k_bsolve_subst) follow once the right-hand side
// is known.  Registers and LDS let MINB workgroups share a CU, so the
// diagonal-block phases of one molecule overlap the MFMA phases of others.
constexpr int BSOLVE_T = 256;
constexpr int BSOLVE_NREF = 2;  // refinement steps of the FP32 factor
template <typename T, int MINB, int DEPTH>
__global__ __launch_bounds__(BSOLVE_T, MINB) void k_eeq_batch_factor(const int* __restrict__ order,
                                                                  const int* __restrict__ mnp,
                                                                  const long long* __restrict__ mo,
                                                                  const int* __restrict__ vo, T* __restrict__ A,
                                                                  T* __restrict__ Linv, int* __restrict__ flags) {
    __shared__ T S0[NB][NB + 1];
    __shared__ T col[2][NB];
    __shared__ T rdiag[NB];
    constexpr int NW = BSOLVE_T / 64;
    const int m = order[blockIdx.x], np = mnp[m], nb = np / NB, base = vo[m];  // largest systems first
    T* Am = A + mo[m];
    T* Lm = Linv + (size_t)base * NB;
    const int wave = threadIdx.x >> 6;
    for (int kb = 0; kb < nb; ++kb) {
        const int k0 = kb * NB;
        batch_diag_block<T>(np, k0, Am, Lm, flags, S0, col, rdiag);
        __syncthreads();
        for (int bi = kb + 1 + wave; bi < nb; bi += NW)
            batch_tile_mfma<T, false, DEPTH>(Am, np, bi * NB, k0, Am + (size_t)bi * NB * np + k0,
                                             Lm + (size_t)kb * NB * NB, NB);
        __syncthreads();
        int tile = 0;
        for (int bi = kb + 1; bi < nb; ++bi)
            for (int bj = kb + 1; bj <= bi; ++bj, ++tile)
                if (tile % NW == wave)
                    batch_tile_mfma<T, true, DEPTH>(Am, np, bi * NB, bj * NB, Am + (size_t)bi * NB * np + k0,
                                                    Am + (size_t)bj * NB * np + k0, np);
        __syncthreads();
    }
}

// Substitutions of one molecule's factored system (workgroup of BSOLVE_T
// threads): x = L^-T L^-1 b, and for T = float BSOLVE_NREF FP64 refinement
// steps against Rm (FP64, lower triangle).
template <typename T>
__device__ __forceinline__ void batch_solve_tail(int np, const T* __restrict__ Am, const T* __restrict__ Lm,
                                                 const double* __restrict__ Rm, const double* __restrict__ b,
                                                 double* __restrict__ x, T* vec, T* tmp, double* xs) {
    const int tid = threadIdx.x, t = tid >> 2, q = tid & 3;
    for (int r = tid; r < np; r += BSOLVE_T) vec[r] = (T)b[r];
    __syncthreads();
    batch_substitute<T>(np, Am, Lm, vec, tmp);
    if constexpr (sizeof(T) == 4) {
        for (int r = tid; r < np; r += BSOLVE_T) xs[r] = (double)vec[r];
        __syncthreads();
        for (int it = 0; it < BSOLVE_NREF; ++it) {
            // r_i = b_i - (sum_{j <= i} R(i, j) x_j + sum_{j > i} R(j, i) x_j), four lanes per row
            for (int i0 = 0; i0 < np; i0 += NB) {
                const int i = i0 + t;
                double acc = 0.0;
                for (int j = q; j <= i; j += 4) acc += Rm[(size_t)i * np + j] * xs[j];
                for (int j = i + 1 + q; j < np; j += 4) acc += Rm[(size_t)j * np + i] * xs[j];
                acc += __shfl_xor(acc, 1);
                acc += __shfl_xor(acc, 2);
                if (q == 0) vec[i] = (T)(b[i] - acc);
            }
            __syncthreads();
            batch_substitute<T>(np, Am, Lm, vec, tmp);
            for (int r = tid; r < np; r += BSOLVE_T) xs[r] += (double)vec[r];
            __syncthreads();
        }
        for (int r = tid; r < np; r += BSOLVE_T) x[r] = xs[r];
    } else {
        for (int r = tid; r < np; r += BSOLVE_T) x[r] = (double)vec[r];
    }
}

// ---- per-molecule factorisation by steps over the whole batch (batch_solver 3)
// Step k is three launches over every molecule with more than k column
// blocks: the diagonal blocks (one workgroup each), the panel tiles and the
// trailing tiles (one wavefront per tile, four per workgroup, any molecule).
// Every tile of a phase is independent, so a launch holds thousands of
// independent tiles and needs no barrier inside a molecule.  The
// substitutions follow in one launch (k_bsolve_subst) on the evaluation
// stream.
template <typename T>
__global__ __launch_bounds__(256, 3) void k_bstep_diag(const int* __restrict__ mols, int k, const int* __restrict__ mnp,
                                                    const long long* __restrict__ mo, const int* __restrict__ vo,
                                                    T* __restrict__ A, T* __restrict__ Linv, int* __restrict__ flags) {
    __shared__ T S0[NB][NB + 1];
    __shared__ T col[2][NB];
    __shared__ T rdiag[NB];
    const int m = mols[blockIdx.x];
    chol_diag_block<T>(mnp[m], k * NB, A + mo[m], Linv + (size_t)vo[m] * NB, flags, S0, col, rdiag);
}

// the same in FP64, one wavefront per block
__global__ __launch_bounds__(64, 2) void k_bstep_diag64(const int* __restrict__ mols, int k, const int* __restrict__ mnp,
                                                        const long long* __restrict__ mo, const int* __restrict__ vo,
                                                        double* __restrict__ A, double* __restrict__ Linv,
                                                        int* __restrict__ flags) {
    __shared__ double buf[16 * 17];
    const int m = mols[blockIdx.x], np = mnp[m], k0 = k * NB;
    const bool ok = chol64_wave(A + mo[m] + (size_t)k0 * np + k0, np, Linv + ((size_t)vo[m] + k0) * NB, true, buf);
    if (!ok && threadIdx.x == 0) atomicOr(flags, FLAG_CHOL);
}

// FP64 panel tile over the whole 64-row tile in one product (the column
// panel of the inverse read once per tile instead of once per half):
// A(ri.., rj..) = P(ri.., 0..63) Q(0..63, 0..63)^T, P the tile itself (leading
// dimension np), Q the inverse of the diagonal block (64 x 64, zero above the
// diagonal); operands eight columns at a time, the next eight in flight.
__device__ __forceinline__ void panel_tile_whole(double* __restrict__ Am, int np, int ri, int rj,
                                                 const double* __restrict__ P, const double* __restrict__ Q) {
    using M = MfmaT<double>;
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    dbl4 acc[4][4];
#pragma unroll
    for (int xx = 0; xx < 4; ++xx)
#pragma unroll
        for (int y = 0; y < 4; ++y) acc[xx][y] = dbl4{0.0, 0.0, 0.0, 0.0};
    dbl2 fa[4], fb[4];
#pragma unroll
    for (int xx = 0; xx < 4; ++xx) fa[xx] = *(const dbl2*)(P + (size_t)(16 * xx + li) * np + 2 * lk);
#pragma unroll
    for (int y = 0; y < 4; ++y) fb[y] = *(const dbl2*)(Q + (16 * y + li) * NB + 2 * lk);
#pragma unroll 1
    for (int kc = 0; kc < NB; kc += 8) {
        const bool more = kc + 8 < NB;
        dbl2 na[4], nb[4];
        if (more) {
#pragma unroll
            for (int xx = 0; xx < 4; ++xx) na[xx] = *(const dbl2*)(P + (size_t)(16 * xx + li) * np + kc + 8 + 2 * lk);
#pragma unroll
            for (int y = 0; y < 4; ++y) nb[y] = *(const dbl2*)(Q + (16 * y + li) * NB + kc + 8 + 2 * lk);
        }
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int xx = 0; xx < 4; ++xx)
#pragma unroll
                for (int y = 0; y < 4; ++y) acc[xx][y] = M::op(fa[xx][st], fb[y][st], acc[xx][y]);
        if (more) {
#pragma unroll
            for (int xx = 0; xx < 4; ++xx) fa[xx] = na[xx];
#pragma unroll
            for (int y = 0; y < 4; ++y) fb[y] = nb[y];
        }
    }
#pragma unroll
    for (int xx = 0; xx < 4; ++xx)
#pragma unroll
        for (int y = 0; y < 4; ++y)
#pragma unroll
            for (int v = 0; v < 4; ++v) Am[(size_t)(ri + 16 * xx + 4 * v + lk) * np + rj + 16 * y + li] = acc[xx][y][v];
}

// tiles {m, bi, bj}: panel tiles (SUB = false, bj unused) or trailing tiles of step k
template <typename T, bool SUB>
__global__ __launch_bounds__(256, 2) void k_bstep_tiles(const int4* __restrict__ tl, int ntl, int k,
                                                     const int* __restrict__ mnp, const long long* __restrict__ mo,
                                                     const int* __restrict__ vo, T* __restrict__ A,
                                                     const T* __restrict__ Linv) {
    const int w = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (w >= ntl) return;  // wavefront-local work: no barrier follows
    const int4 tt = tl[w];
    const int m = tt.x, bi = tt.y, bj = tt.z, np = mnp[m], k0 = k * NB;
    T* Am = A + mo[m];
    if constexpr (!SUB && sizeof(T) == 8)
        panel_tile_whole(Am, np, bi * NB, k0, Am + (size_t)bi * NB * np + k0,
                         Linv + (size_t)vo[m] * NB + (size_t)k * NB * NB);
    else if (!SUB)
        batch_tile_mfma<T, false, 4>(Am, np, bi * NB, k0, Am + (size_t)bi * NB * np + k0,
                                     Linv + (size_t)vo[m] * NB + (size_t)k * NB * NB, NB);
    else
        batch_tile_mfma<T, true, 4>(Am, np, bi * NB, bj * NB, Am + (size_t)bi * NB * np + k0,
                                    Am + (size_t)bj * NB * np + k0, np);
}

template <typename T>
__global__ __launch_bounds__(BSOLVE_T) void k_bsolve_subst(const int* __restrict__ order, const int* __restrict__ mnp,
                                                           const long long* __restrict__ mo,
                                                           const int* __restrict__ vo, const T* __restrict__ A,
                                                           const T* __restrict__ Linv,
                                                           const double* __restrict__ A64,
                                                           const double* __restrict__ b, double* __restrict__ x) {
    __shared__ T vec[BATCH_MAX_NP];
    __shared__ T tmp[NB];
    __shared__ double xs[sizeof(T) == 4 ? BATCH_MAX_NP : 1];
    const int m = order[blockIdx.x], base = vo[m];
    batch_solve_tail<T>(mnp[m], A + mo[m], Linv + (size_t)base * NB, A64 ? A64 + mo[m] : nullptr, b + base, x + base,
                        vec, tmp, xs);
}

// ---- per-molecule left-looking factorisation with the matrix formed in place (batch_solver 4)
// Tile (i, j), i >= j, of column block j on one wavefront:
//   C = R(i, j) - L(i, 0:K) L(j, 0:K)^T,  K = 64 j,
// stored at the tile, in two 32-row halves.  First the half's entries of R
// are evaluated from the coordinates with the operations of
// k_eeq_reduced_batch, lane = column, one row at a time: one-fragment
// molecules (uni) as A(ia, ib) - u_a - u_b + A(L, L) with u_r = A(ia_r, L),
// the row's data (coordinates, alpha, u) read from the lane of the half that
// loaded it (readlane, no dependent gather per row); other molecules in the
// direct four-term form; padded rows and columns as the identity.  They are
// stored at the tile (the lines stay in L2) and read back in the MFMA
// accumulator layout as -R; the product adds L(i, :) L(j, :)^T over the whole
// K on FP64 MFMA, and C = -acc is stored.  The operands are read eight
// columns at a time as 16-byte vectors (lane group g holds columns 2 g and
// 2 g + 1 of the eight, MFMA step s takes column 2 g + s: a permutation of
// the columns that both operands share), the next eight columns in flight
// while the current ones are multiplied.

// C = -(R - L(r0:r0+16XX, 0:K) L(j, 0:K)^T) over 16 XX rows from r0: element v
// of block (xx, y) at row r0 + 16 xx + 4 v + lk, column 64 j + 16 y + li, read
// in the MFMA accumulator layout after the wavefront's own entry stores;
// the operands eight columns at a time, the next eight in flight.
template <int XX>
__device__ __forceinline__ void fused_product(double* __restrict__ Am, int np, int r0, int j) {
    using M = MfmaT<double>;
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    const int K = j * NB;
    if (K == 0) return;  // column block 0: C = R, already stored by the entry pass
    const double* Qj = Am + (size_t)(j * NB) * np;
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_wave_barrier();
    double* pt = Am + (size_t)(r0 + lk) * np + j * NB + li;  // this lane's element (0, 0, 0)
    dbl4 acc[XX][4];
#pragma unroll
    for (int xx = 0; xx < XX; ++xx)
#pragma unroll
        for (int y = 0; y < 4; ++y)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[xx][y][v] = -pt[(size_t)(16 * xx + 4 * v) * np + 16 * y];
    if (K > 0) {
        const double* Pi = Am + (size_t)r0 * np;
        dbl2 fa[XX], fb[4];
#pragma unroll
        for (int xx = 0; xx < XX; ++xx) fa[xx] = *(const dbl2*)(Pi + (size_t)(16 * xx + li) * np + 2 * lk);
#pragma unroll
        for (int y = 0; y < 4; ++y) fb[y] = *(const dbl2*)(Qj + (size_t)(16 * y + li) * np + 2 * lk);
#pragma unroll 1
        for (int kc = 0; kc < K; kc += 8) {
            const bool more = kc + 8 < K;
            dbl2 na[XX], nb[4];
            if (more) {
#pragma unroll
                for (int xx = 0; xx < XX; ++xx)
                    na[xx] = *(const dbl2*)(Pi + (size_t)(16 * xx + li) * np + kc + 8 + 2 * lk);
#pragma unroll
                for (int y = 0; y < 4; ++y) nb[y] = *(const dbl2*)(Qj + (size_t)(16 * y + li) * np + kc + 8 + 2 * lk);
            }
#pragma unroll
            for (int st = 0; st < 2; ++st)
#pragma unroll
                for (int xx = 0; xx < XX; ++xx)
#pragma unroll
                    for (int y = 0; y < 4; ++y) acc[xx][y] = M::op(fa[xx][st], fb[y][st], acc[xx][y]);
            if (more) {
#pragma unroll
                for (int xx = 0; xx < XX; ++xx) fa[xx] = na[xx];
#pragma unroll
                for (int y = 0; y < 4; ++y) fb[y] = nb[y];
            }
        }
    }
    // the element addresses are formed again here rather than kept in
    // registers across the product (an empty asm makes pt opaque)
    asm volatile("" : "+v"(pt));
#pragma unroll
    for (int xx = 0; xx < XX; ++xx)
#pragma unroll
        for (int y = 0; y < 4; ++y)
#pragma unroll
            for (int v = 0; v < 4; ++v) pt[(size_t)(16 * xx + 4 * v) * np + 16 * y] = -acc[xx][y][v];
}

// MODE 2 of fused_tile: the tile is formed transposed, D = C^T (rows the
// column block's 64 rows cj, columns the tile's rows ri), so that the
// accumulator is directly the B operand of the panel product
//   L(i, j)^T = Linv(j) C^T,   i.e.  L(i, j) = C(i, j) Linv(j)^T,
// the product of the panel launch of the other column orders, without the
// round trip of C through memory.  Lj: the inverse of the diagonal block,
// 64 x 64 row-major, zero above the diagonal.
__device__ __forceinline__ void fused_product_panel(double* __restrict__ Am, int np, int r0, int j,
                                                    const double* __restrict__ Lj) {
    using M = MfmaT<double>;
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
    const int K = j * NB;
    const double* Qj = Am + (size_t)(j * NB) * np;
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_wave_barrier();
    // element v of block (yy, xx): D(16 yy + 4 v + lk, 16 xx + li) = C(r0 + 16 xx + li, 64 j + 16 yy + 4 v + lk)
    double* pr = Am + (size_t)(r0 + li) * np + j * NB + lk;
    dbl4 acc[4][4];
#pragma unroll
    for (int yy = 0; yy < 4; ++yy)
#pragma unroll
        for (int xx = 0; xx < 4; ++xx)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[yy][xx][v] = -pr[(size_t)(16 * xx) * np + 16 * yy + 4 * v];
    if (K > 0) {
        const double* Pi = Am + (size_t)r0 * np;
        dbl2 fa[4], fb[4];
#pragma unroll
        for (int xx = 0; xx < 4; ++xx) fa[xx] = *(const dbl2*)(Pi + (size_t)(16 * xx + li) * np + 2 * lk);
#pragma unroll
        for (int y = 0; y < 4; ++y) fb[y] = *(const dbl2*)(Qj + (size_t)(16 * y + li) * np + 2 * lk);
#pragma unroll 1
        for (int kc = 0; kc < K; kc += 8) {
            const bool more = kc + 8 < K;
            dbl2 na[4], nb[4];
            if (more) {
#pragma unroll
                for (int xx = 0; xx < 4; ++xx)
                    na[xx] = *(const dbl2*)(Pi + (size_t)(16 * xx + li) * np + kc + 8 + 2 * lk);
#pragma unroll
                for (int y = 0; y < 4; ++y) nb[y] = *(const dbl2*)(Qj + (size_t)(16 * y + li) * np + kc + 8 + 2 * lk);
            }
#pragma unroll
            for (int st = 0; st < 2; ++st)
#pragma unroll
                for (int yy = 0; yy < 4; ++yy)
#pragma unroll
                    for (int xx = 0; xx < 4; ++xx) acc[yy][xx] = M::op(fb[yy][st], fa[xx][st], acc[yy][xx]);
            if (more) {
#pragma unroll
                for (int xx = 0; xx < 4; ++xx) fa[xx] = na[xx];
#pragma unroll
                for (int y = 0; y < 4; ++y) fb[y] = nb[y];
            }
        }
    }
    // acc = -C^T.  Per column block xx of the tile's rows: out(mm) = sum over
    // the 16 four-row chunks (yy, v) of Linv(16 mm + li, 16 yy + 4 v + lk)
    // times chunk (yy, v) of acc, = -L(i, j)^T block (mm, xx)
    asm volatile("" : "+v"(pr));
#pragma unroll
    for (int xx = 0; xx < 4; ++xx) {
        dbl4 out[4];
#pragma unroll
        for (int mm = 0; mm < 4; ++mm) out[mm] = dbl4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int yy = 0; yy < 4; ++yy)
#pragma unroll
            for (int v = 0; v < 4; ++v)
#pragma unroll
                for (int mm = 0; mm < 4; ++mm)
                    out[mm] = M::op(Lj[(16 * mm + li) * NB + 16 * yy + 4 * v + lk], acc[yy][xx][v], out[mm]);
#pragma unroll
        for (int mm = 0; mm < 4; ++mm)
#pragma unroll
            for (int v = 0; v < 4; ++v) pr[(size_t)(16 * xx) * np + 16 * mm + 4 * v] = -out[mm][v];
    }
}

// MODE 0: product per 32-row half; 1: one product over the 64-row tile, so
// that the column's own row panel L(j, 0:K) is read once per tile (needs the
// registers of two wavefronts per SIMD); 2: as 1, transposed, followed by
// the panel product with Lj (fused_product_panel)
template <int MODE>
__device__ __forceinline__ void fused_tile(double* __restrict__ Am, int np, int nr, int i, int j,
                                           const int* __restrict__ rab, const int* __restrict__ rlb,
                                           const double* __restrict__ x, const double* __restrict__ alp,
                                           const double* __restrict__ diag, const double* su, double sll, bool uni,
                                           const double* __restrict__ Lj = nullptr) {
    const int lane = threadIdx.x & 63;
    // this lane's column of the entry pass
    const int Cc = j * NB + lane;
    const bool cin = Cc < nr;
    const int ib = cin ? rab[Cc] : 0, lb = (cin && !uni) ? rlb[Cc] : 0;
    const double3 cx = (cin && uni) ? ld3(x, ib) : make_double3(0.0, 0.0, 0.0);
    const double ca = (cin && uni) ? alp[ib] : 0.0, cu = (cin && uni) ? su[Cc] : 0.0;
    const double cdg = (cin && uni) ? diag[ib] : 0.0;
#pragma unroll 1
    for (int h = 0; h < 2; ++h) {
        const int r0 = i * NB + 32 * h;
        if (uni) {
            // row r0 + (lane & 31) loaded by this lane
            const int Rl = r0 + (lane & 31);
            const bool rinl = Rl < nr;
            const int ial = rinl ? rab[Rl] : 0;
            const double3 rxl = rinl ? ld3(x, ial) : make_double3(0.0, 0.0, 0.0);
            const double ral = rinl ? alp[ial] : 0.0, rul = rinl ? su[Rl] : 0.0;
#pragma unroll 4
            for (int rr = 0; rr < 32; ++rr) {
                const int R = r0 + rr;
                const double3 rx = make_double3(readlane_d(rxl.x, rr), readlane_d(rxl.y, rr), readlane_d(rxl.z, rr));
                const double ra = readlane_d(ral, rr), ru = readlane_d(rul, rr);
                double a;
                if (R >= nr || !cin) {
                    a = (R == Cc) ? 1.0 : 0.0;
                } else {
                    const double3 d = rx - cx;
                    const double aij = (R == Cc) ? cdg : eeq_a_r2(dot(d, d), ra, ca);
                    a = aij - ru - cu + sll;
                }
                Am[(size_t)R * np + Cc] = a;
            }
        } else {
#pragma unroll 2
            for (int rr = 0; rr < 32; ++rr) {
                const int R = r0 + rr;
                double a;
                if (R >= nr || !cin) {
                    a = (R == Cc) ? 1.0 : 0.0;
                } else {
                    const int ia = rab[R], la = rlb[R];
                    a = eeq_a(ia, ib, x, alp, diag) - eeq_a(ia, lb, x, alp, diag) - eeq_a(la, ib, x, alp, diag) +
                        eeq_a(la, lb, x, alp, diag);
                }
                Am[(size_t)R * np + Cc] = a;
            }
        }
        if (MODE == 0) fused_product<2>(Am, np, r0, j);
    }
    if (MODE == 1) fused_product<4>(Am, np, i * NB, j);
    if (MODE == 2) fused_product_panel(Am, np, i * NB, j, Lj);
}

// One workgroup of four wavefronts per molecule (largest systems first),
// left-looking by 64-column blocks.  Column block j: the tiles (i, j), i >= j,
// are formed (fused_tile, one per wavefront, dealt round-robin); the diagonal
// block is factored and inverted (chol_diag_block); the tiles below it become
// L(i, j) = C(i, j) L(j, j)^-T (MFMA, one per wavefront).  Against the
// right-looking form every tile is written once, the factored panels are read
// once per column block with the product accumulated in registers over the
// whole K, and the matrix is never built as a separate pass (no R in HBM):
// the only matrix traffic is L, so the kernel reads and writes about a third
// of the bytes.  The substitutions follow in k_bsolve_subst<double>.
template <int MINB>
__global__ __launch_bounds__(BSOLVE_T, MINB) void k_eeq_batch_fused(
    const int* __restrict__ order, const int* __restrict__ mnr, const int* __restrict__ mnp,
    const long long* __restrict__ mo, const int* __restrict__ vo, const int* __restrict__ ra,
    const int* __restrict__ rl, const double* __restrict__ x, const double* __restrict__ alp,
    const double* __restrict__ diag, double* __restrict__ A, double* __restrict__ Linv, int* __restrict__ flags) {
    __shared__ double S0[NB][NB + 1];
    __shared__ double col[2][NB];
    __shared__ double rdiag[NB];
    __shared__ double su[BATCH_MAX_NP];
    constexpr int NW = BSOLVE_T / 64;
    const int m = order[blockIdx.x], nr = mnr[m], np = mnp[m], nb = np / NB, base = vo[m];
    const int tid = threadIdx.x, wave = tid >> 6;
    double* Am = A + mo[m];
    double* Lm = Linv + (size_t)base * NB;
    const int* rab = ra + base;
    const int* rlb = rl + base;
    // one fragment: every row's last atom is row 0's
    const int L0 = nr > 0 ? rlb[0] : 0;
    bool same = true;
    for (int r = tid; r < nr; r += BSOLVE_T) same = same && rlb[r] == L0;
    const bool uni = __syncthreads_and(same) && nr > 0;
    if (uni)
        for (int r = tid; r < nr; r += BSOLVE_T) su[r] = eeq_a(rab[r], L0, x, alp, diag);
    const double sll = uni ? eeq_a(L0, L0, x, alp, diag) : 0.0;
    __syncthreads();
    for (int j = 0; j < nb; ++j) {
        for (int i = j + wave; i < nb; i += NW) fused_tile<0>(Am, np, nr, i, j, rab, rlb, x, alp, diag, su, sll, uni);
        __syncthreads();
        batch_diag_block<double>(np, j * NB, Am, Lm, flags, S0, col, rdiag);
        __syncthreads();
        for (int i = j + 1 + wave; i < nb; i += NW)
            batch_tile_mfma<double, false, 1>(Am, np, i * NB, j * NB, Am + (size_t)i * NB * np + j * NB,
                                              Lm + (size_t)j * NB * NB, NB);
        __syncthreads();
    }
}

// ---- left-looking factorisation by column blocks over the whole batch (batch_solver 5)
// Column block j is three launches over every molecule with more than j
// column blocks: the tiles (i, j), i >= j, formed by fused_tile (one
// wavefront per tile, any molecule), the diagonal blocks (k_bstep_diag64) and
// the panel tiles L(i, j) = C(i, j) L(j, j)^-T (k_bstep_tiles<double,
// false>).  The per-molecule form's parallelism (four wavefronts) becomes
// thousands of independent tiles per launch, and the entries of R are still
// evaluated once, inside the tile that needs them.
// u_v = A(ia_v, last atom of v's fragment) for every reduced row (0 on padding)
__global__ __launch_bounds__(256) void k_red_u(int nv, const int* __restrict__ ra, const int* __restrict__ rl,
                                               const double* __restrict__ x, const double* __restrict__ alp,
                                               const double* __restrict__ diag, double* __restrict__ u) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= nv) return;
    u[v] = (ra[v] >= 0) ? eeq_a(ra[v], rl[v], x, alp, diag) : 0.0;
}

// tiles {m, i, one-fragment flag, 0} of column block j
__global__ __launch_bounds__(256, 2) void k_lstep_tiles(const int4* __restrict__ tl, int ntl, int j,
                                                     const int* __restrict__ mnr, const int* __restrict__ mnp,
                                                     const long long* __restrict__ mo, const int* __restrict__ vo,
                                                     const int* __restrict__ ra, const int* __restrict__ rl,
                                                     const double* __restrict__ x, const double* __restrict__ alp,
                                                     const double* __restrict__ diag, const double* __restrict__ u,
                                                     double* __restrict__ A) {
    const int w = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (w >= ntl) return;  // wavefront-local work: no barrier follows
    const int4 tt = tl[w];
    const int m = tt.x, base = vo[m];
    const bool uni = tt.z != 0;
    const double sll = uni ? eeq_a(rl[base], rl[base], x, alp, diag) : 0.0;
    fused_tile<1>(A + mo[m], mnp[m], mnr[m], tt.y, j, ra + base, rl + base, x, alp, diag, u + base, sll, uni);
}

// batch_solver 6: the tiles below the diagonal of column block j after its
// diagonal block is factored: formed and multiplied by Linv(j) in one pass,
// L(i, j) stored directly (fused_tile MODE 2)
__global__ __launch_bounds__(256, 2) void k_lpanel_tiles(const int4* __restrict__ tl, int ntl, int j,
                                                      const int* __restrict__ mnr, const int* __restrict__ mnp,
                                                      const long long* __restrict__ mo, const int* __restrict__ vo,
                                                      const int* __restrict__ ra, const int* __restrict__ rl,
                                                      const double* __restrict__ x, const double* __restrict__ alp,
                                                      const double* __restrict__ diag, const double* __restrict__ u,
                                                      double* __restrict__ A, const double* __restrict__ Linv) {
    const int w = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (w >= ntl) return;  // wavefront-local work: no barrier follows
    const int4 tt = tl[w];
    const int m = tt.x, base = vo[m];
    const bool uni = tt.z != 0;
    const double sll = uni ? eeq_a(rl[base], rl[base], x, alp, diag) : 0.0;
    fused_tile<2>(A + mo[m], mnp[m], mnr[m], tt.y, j, ra + base, rl + base, x, alp, diag, u + base, sll, uni,
                  Linv + (size_t)base * NB + (size_t)j * NB * NB);
}

// Previous per-molecule solve (whole workgroup per tile step), kept for
// comparison: the blocked right-looking Cholesky (diag / panel / MFMA tile
// update, the routines of the single-molecule path) and both substitutions,
// all inside the workgroup.  b, x: concatenated padded vectors.
__global__ __launch_bounds__(256) void k_eeq_batch_solve_tiles(const int* __restrict__ order,
                                                         const int* __restrict__ mnp, const long long* __restrict__ mo,
                                                         const int* __restrict__ vo, double* __restrict__ A,
                                                         double* __restrict__ Linv, const double* __restrict__ b,
                                                         double* __restrict__ x, int* __restrict__ flags) {
    __shared__ double S0[NB][NB + 1];
    __shared__ double S1[NB][NB + 1];
    __shared__ double col[2][NB];
    __shared__ double rdiag[NB];
    __shared__ double vec[BATCH_MAX_NP];
    __shared__ double tmp[NB];
    const int m = order[blockIdx.x], np = mnp[m], nb = np / NB, base = vo[m];  // largest systems first
    double* Am = A + mo[m];
    double* Lm = Linv + (size_t)base * NB;
    const int tid = threadIdx.x, t = tid >> 2, q = tid & 3;
    for (int kb = 0; kb < nb; ++kb) {
        chol_diag_block<double>(np, kb * NB, Am, Lm, flags, S0, col, rdiag);
        __syncthreads();
        for (int bi = kb + 1; bi < nb; ++bi) {
            chol_panel_tile<double>(np, kb * NB, bi * NB, Am, Lm, S0, S1);
            __syncthreads();
        }
        for (int bi = kb + 1; bi < nb; ++bi)
            for (int bj = kb + 1; bj <= bi; ++bj) {
                chol_update_tile<double>(np, bi * NB, bj * NB, kb * NB, NB, Am, S0, S1);
                __syncthreads();
            }
    }
    for (int r = tid; r < np; r += 256) vec[r] = b[base + r];
    __syncthreads();
    // forward: y_kb = Linv_kb (b_kb - sum_{k < kb} L(kb, k) y_k), y kept in vec
    for (int kb = 0; kb < nb; ++kb) {
        double acc = (q == 0) ? vec[kb * NB + t] : 0.0;
        for (int k = 0; k < kb; ++k)
#pragma unroll
            for (int u = 0; u < NB / 4; ++u)
                acc -= Am[(size_t)(kb * NB + t) * np + k * NB + 4 * u + q] * vec[k * NB + 4 * u + q];
        acc += __shfl_xor(acc, 1);
        acc += __shfl_xor(acc, 2);
        if (q == 0) tmp[t] = acc;
        __syncthreads();
        const double* Li = Lm + (size_t)kb * NB * NB;
        double s = 0.0;
#pragma unroll
        for (int u = 0; u < NB / 4; ++u) s += Li[t * NB + 4 * u + q] * tmp[4 * u + q];
        s += __shfl_xor(s, 1);
        s += __shfl_xor(s, 2);
        if (q == 0) vec[kb * NB + t] = s;
        __syncthreads();
    }
    // backward: x_kb = Linv_kb^T (y_kb - sum_{k > kb} L(k, kb)^T x_k)
    for (int kb = nb - 1; kb >= 0; --kb) {
        double acc = (q == 0) ? vec[kb * NB + t] : 0.0;
        for (int k = nb - 1; k > kb; --k)
#pragma unroll
            for (int u = 0; u < NB / 4; ++u)
                acc -= Am[(size_t)(k * NB + 4 * u + q) * np + kb * NB + t] * vec[k * NB + 4 * u + q];
        acc += __shfl_xor(acc, 1);
        acc += __shfl_xor(acc, 2);
        if (q == 0) tmp[t] = acc;
        __syncthreads();
        const double* Li = Lm + (size_t)kb * NB * NB;
        double s = 0.0;
#pragma unroll
        for (int u = 0; u < NB / 4; ++u) s += Li[(4 * u + q) * NB + t] * tmp[4 * u + q];
        s += __shfl_xor(s, 1);
        s += __shfl_xor(s, 2);
        if (q == 0) vec[kb * NB + t] = s;
        __syncthreads();
    }
    for (int r = tid; r < np; r += 256) x[base + r] = vec[r];
}

// Per-molecule total energy: one wavefront per molecule sums the per-atom
// terms over its atoms and the per-entry terms over its list segments
// (seg[t * (nmol + 1) + m]) in a fixed order.
struct MolEnergyArgs {
    int nmol;
    const int* mol_off;
    const int* seg;        // [11][nmol + 1]: bond, angle, torsion, brep, hb case 1 (role-A groups), atm, batm,
                           // inversion, stors, xb, hb cases 2-4
    const double* atom_terms[4];   // coul, disp, rep, self
    const double* list_terms[11];
    double* e_mol;
};
__device__ inline void mol_energy(const MolEnergyArgs& a, int m, int lane) {
    if (m >= a.nmol) return;
    double acc = 0.0;
    for (int k = 0; k < 4; ++k)
        for (int i = a.mol_off[m] + lane; i < a.mol_off[m + 1]; i += 64) acc += a.atom_terms[k][i];
    for (int k = 0; k < 11; ++k) {
        const int* sg = a.seg + k * (a.nmol + 1);
        for (int i = sg[m] + lane; i < sg[m + 1]; i += 64) acc += a.list_terms[k][i];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
    if (lane == 0) a.e_mol[m] = acc;
}

// ---------------------------------------------------------------------------
// K10: parameter adjoint.  For per-element scale factors theta of the
// repulsion charge (repz), the repulsion exponent (rep_anb / repa) and the D4
// sqrt(Z r4r2), and a weight field w (w_i = dLoss/dg_i of a loss on the
// gradient g, e.g. 2 (g - g_ref) for force matching), the kernels accumulate
//   dLoss/dln(theta_p) = sum_i w_i . d g_i / d ln(theta_p).
// Only the D4 pair term (energy gradient and its dE/dCN chain) and the bonded
// and non-bonded repulsion depend on these parameters; ATM uses rcov_d3, the
// EEQ and CN are parameter-free here.  Output layout: [p * ne + e] with
// p = 0 repz, 1 exponent, 2 sqrt(Z r4r2).
// ---------------------------------------------------------------------------
constexpr int ADJ_P = 3;

// u_a = dlog_a sum_{b in nb(a)} dd(r_ab) (w_a - w_b) . (x_a - x_b) / r_ab:
// the contraction of w with d CN_a / dx (same arithmetic as k_finish).
__global__ __launch_bounds__(256) void k_adj_u(int n, const double* __restrict__ x, const double* __restrict__ rcov,
                                               const double* __restrict__ dlog, const int* __restrict__ nbn,
                                               const int* __restrict__ nbl, const double* __restrict__ w,
                                               double* __restrict__ u) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= n) return;
    const double3 xa = ld3(x, a), wa = ld3(w, a);
    double acc = 0.0;
    for (int k = 0; k < nbn[a]; ++k) {
        const int b = nbl[(size_t)a * MAXNB_CN + k];
        const double3 d = xa - ld3(x, b);
        const double r = nrm(d);
        const double rs = rcov[a] + rcov[b];
        const double dr = (r - rs) / rs;
        const double dd = (KN / SQRTPI_TRUNC) * exp(-KN * KN * dr * dr) / rs;
        acc += dd * dot(wa - ld3(w, b), d) / r;
    }
    u[a] = dlog[a] * acc;
}

// derivatives of the repulsion pair term e = ab exp(-al r^1.5) / r:
//   dE'/d ln ab = E',  dE'/d al = -0.5 sqrt(r) e + 1.5 al r^2 e
__device__ inline void rep_adj(double ab, double al, double r, double& dp_lnab, double& dp_al) {
    const double sr = sqrt(r), rinv = rcp_c(r);
    const double e = ab * exp(-al * r * sr) * rinv;
    dp_lnab = -e * rinv - 1.5 * al * sr * e;
    dp_al = -0.5 * sr * e + 1.5 * al * r * r * e;
}

// D4 pair, derivatives with respect to q = r4r2 of E' (=dE/dr) and of the row
// atom's dE/dCN share -dci sum zeta (ff_workspace_gfnff.cpp:715-767):
__device__ inline void d4_adj(double c6, double dci, double zc, double q, double r2, double r, double& dEp_dq,
                              double& ddcn_dq) {
    const double rq = rsqrt_c(q);
    const double r0 = 0.58 * (q * rq) + 4.80;
    const double dr0 = 0.29 * rq;
    const double r0s = r0 * r0;
    const double r6 = r2 * r2 * r2, r06 = r0s * r0s * r0s;
    const double p6 = r6 + r06, p8 = r6 * r2 + r06 * r0s, pi = rcp_c(p6 * p8);
    const double t6 = p8 * pi, t8 = p6 * pi;  // 1 / p6, 1 / p8
    const double dt6 = -t6 * t6 * 6.0 * (r0s * r0s * r0) * dr0;  // d t6 / dq
    const double dt8 = -t8 * t8 * 8.0 * r06 * r0 * dr0;        // d t8 / dq
    const double d8 = -8.0 * r2 * r2 * r2 * t8 * t8;
    const double dd6 = -6.0 * r2 * r2 * 2.0 * t6 * dt6;
    const double dd8 = -8.0 * r2 * r2 * r2 * 2.0 * t8 * dt8;
    dEp_dq = -c6 * zc * (dd6 + 2.0 * d8 + 2.0 * q * dd8) * r;
    ddcn_dq = -dci * zc * (dt6 + 2.0 * t8 + 2.0 * q * dt8);
}

// Pair adjoint over full rows, the partners (all atoms, or the molecules of
// the workgroup's rows) cut into up to 16 chunks (gridDim.y, adj_chunks), until
// the launch has 1024 workgroups: 256 conformers, 33,700 atoms, 132 row
// blocks, ran 432 us in one chunk on half of the chip's compute units; one
// fitting step with this and the reduction below 2.39 -> 1.65 ms.
// Row i collects sum_j (w_i . r_hat_ij) dE'_ij/dln(theta) + u_i d(dEdcn_i)/dln(theta)
// for its own element and the partner's; part[chunk][k * n + i], k = p * ne + e.
template <int NE>
__global__ __launch_bounds__(TILE) void k_adj_pairs(PairArgs a, const double* __restrict__ w,
                                                    const double* __restrict__ u, double* __restrict__ part) {
    __shared__ double sx[TILE], sy[TILE], sz[TILE], ssz[TILE], san[TILE], srz[TILE], szt[TILE];
    __shared__ double sgw[TILE * 7];
    __shared__ int sZ[TILE], sel[TILE], smt[TILE];
    const int n = a.n;
    const int i = blockIdx.x * TILE + threadIdx.x;
    const bool act = i < n;
    int j0, j1;
    if (a.mol_of)
        pair_range(a, a.n, j0, j1);
    else
        j0 = 0, j1 = n;
    {
        const int len = (j1 - j0 + gridDim.y - 1) / gridDim.y;
        j0 += blockIdx.y * len;
        j1 = min(j1, j0 + len);
    }
    const int mlo = (a.mol_of && act) ? a.mol_off[a.mol_of[i]] : 0;
    const int mhi = (a.mol_of && act) ? a.mol_off[a.mol_of[i] + 1] : n;
    const double3 xi = act ? ld3(a.x, i) : make_double3(0, 0, 0);
    const double3 wi = act ? ld3(w, i) : make_double3(0, 0, 0);
    const double ui = act ? u[i] : 0.0, zti = act ? a.zeta[i] : 0.0, szi = act ? a.szr[i] : 0.0;
    const double ani = act ? a.anb[i] : 0.0, rzi = act ? a.repz[i] : 0.0;
    const int zi = act ? a.Z[i] : 0, mi = act ? a.metal[i] : 0, ei = act ? a.elem[i] : 0;
    double hr[NE * 7], dhr[NE * 7];
#pragma unroll
    for (int k = 0; k < NE * 7; ++k) {
        hr[k] = act ? a.h[(size_t)i * NE * 7 + k] : 0.0;
        dhr[k] = act ? a.dh[(size_t)i * NE * 7 + k] : 0.0;
    }
    double own[ADJ_P] = {0.0, 0.0, 0.0};    // contributions through the row atom's element
    double oth[ADJ_P][NE];                  // through the partner's element
#pragma unroll
    for (int p = 0; p < ADJ_P; ++p)
#pragma unroll
        for (int e = 0; e < NE; ++e) oth[p][e] = 0.0;
    for (int t0 = j0; t0 < j1; t0 += TILE) {
        __syncthreads();
        const int j = t0 + threadIdx.x;
        if (j < j1) {
            sx[threadIdx.x] = a.x[3 * j];
            sy[threadIdx.x] = a.x[3 * j + 1];
            sz[threadIdx.x] = a.x[3 * j + 2];
            ssz[threadIdx.x] = a.szr[j];
            san[threadIdx.x] = a.anb[j];
            srz[threadIdx.x] = a.repz[j];
            szt[threadIdx.x] = a.zeta[j];
            sZ[threadIdx.x] = a.Z[j];
            sel[threadIdx.x] = a.elem[j];
            smt[threadIdx.x] = a.metal[j];
#pragma unroll
            for (int r = 0; r < 7; ++r) sgw[threadIdx.x * 7 + r] = a.gw[(size_t)j * 7 + r];
        }
        __syncthreads();
        if (!act) continue;
        const int m = min(TILE, j1 - t0);
        for (int jj = 0; jj < m; ++jj) {
            if (t0 + jj == i || t0 + jj < mlo || t0 + jj >= mhi) continue;
            const double dx = xi.x - sx[jj], dy = xi.y - sy[jj], dz = xi.z - sz[jj];
            const double r2 = dx * dx + dy * dy + dz * dz;
            if (r2 > 2500.0) continue;  // beyond the D4 and repulsion cut-offs
            const double rinv = rsqrt_c(r2), r = r2 * rinv;
            if (!(r >= 1e-10)) continue;
            const double sw = (wi.x * dx + wi.y * dy + wi.z * dz) * rinv;
            const int ej = sel[jj];
            double dd4 = 0.0, dz_ = 0.0, da_ = 0.0;
            {   // D4 (r <= 50)
                double c6 = 0.0, dci = 0.0;
#pragma unroll
                for (int e = 0; e < NE; ++e)
                    if (e == ej) {
#pragma unroll
                        for (int bb = 0; bb < 7; ++bb) {
                            const double gj = sgw[jj * 7 + bb];
                            c6 += hr[e * 7 + bb] * gj;
                            dci += dhr[e * 7 + bb] * gj;
                        }
                    }
                const double q = 3.0 * szi * ssz[jj];
                double dEp_dq, ddcn_dq;
                d4_adj(c6, dci, zti * szt[jj], q, r2, r, dEp_dq, ddcn_dq);
                dd4 = (sw * dEp_dq + ui * ddcn_dq) * q;  // d / d ln(theta) of one factor of q
            }
            if (r2 <= 400.0 && r >= 1e-8) {   // non-bonded repulsion, generic pair factor
                const double ff = rep_ff(zi, sZ[jj], mi, smt[jj]);
                const double al = sqrt(ani * san[jj]) * ff;
                const double ab = rzi * srz[jj] * 0.4270;
                double dp_lnab, dp_al;
                rep_adj(ab, al, r, dp_lnab, dp_al);
                dz_ = sw * dp_lnab;
                da_ = sw * dp_al * 0.5 * al;
            }
            own[0] += dz_;
            own[1] += da_;
            own[2] += dd4;
#pragma unroll
            for (int e = 0; e < NE; ++e)
                if (e == ej) {
                    oth[0][e] += dz_;
                    oth[1][e] += da_;
                    oth[2][e] += dd4;
                }
        }
    }
    if (!act) return;
    double* pp = part + (size_t)blockIdx.y * ADJ_P * NE * n + i;
#pragma unroll
    for (int p = 0; p < ADJ_P; ++p)
#pragma unroll
        for (int e = 0; e < NE; ++e) pp[(size_t)(p * NE + e) * n] = oth[p][e] + (e == ei ? own[p] : 0.0);
}

// Topological corrections of the non-bonded repulsion (bonded pairs removed,
// H-H 1,3 / 1,4 factors), mirroring nbrep_fix_atom; row-wise, appended as one
// more chunk of partials.
template <int NE>
__global__ __launch_bounds__(256) void k_adj_nbrep_fix(int n, const double* __restrict__ x,
                                                       const int* __restrict__ Z, const int* __restrict__ metal,
                                                       const int* __restrict__ elem, const double* __restrict__ anb,
                                                       const double* __restrict__ repz, const int* __restrict__ toff,
                                                       const int* __restrict__ tidx, const int* __restrict__ tdist,
                                                       const double* __restrict__ w, double* __restrict__ part) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double3 xi = ld3(x, i), wi = ld3(w, i);
    double acc[ADJ_P - 1][NE];
#pragma unroll
    for (int p = 0; p < ADJ_P - 1; ++p)
#pragma unroll
        for (int e = 0; e < NE; ++e) acc[p][e] = 0.0;
    const int ei = elem[i];
    for (int k = toff[i]; k < toff[i + 1]; ++k) {
        const int j = tidx[k], td = tdist[k];
        const int zi = Z[i], zj = Z[j];
        const double fgen = rep_ff(zi, zj, metal[i], metal[j]);
        double fnew;
        if (td == 1) fnew = 0.0;
        else if (zi == 1 && zj == 1 && td == 2) fnew = 0.6290 * 1.4580;
        else if (zi == 1 && zj == 1 && td == 3) fnew = 0.6290 * 0.7080;
        else continue;
        const double3 d = xi - ld3(x, j);
        const double r = nrm(d);
        if (r > 20.0 || r < 1e-8) continue;
        const double sw = dot(wi, d) / r;
        const double ab = repz[i] * repz[j] * 0.4270;
        const double base = sqrt(anb[i] * anb[j]);
        double dz_ = 0.0, da_ = 0.0, dp_lnab, dp_al;
        rep_adj(ab, base * fgen, r, dp_lnab, dp_al);
        dz_ -= sw * dp_lnab;
        da_ -= sw * dp_al * 0.5 * base * fgen;
        if (fnew != 0.0) {
            rep_adj(ab, base * fnew, r, dp_lnab, dp_al);
            dz_ += sw * dp_lnab;
            da_ += sw * dp_al * 0.5 * base * fnew;
        }
        const int ej = elem[j];
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            const double c = (e == ei ? 1.0 : 0.0) + (e == ej ? 1.0 : 0.0);
            acc[0][e] += c * dz_;
            acc[1][e] += c * da_;
        }
    }
#pragma unroll
    for (int e = 0; e < NE; ++e) {
        part[(size_t)(0 * NE + e) * n + i] = acc[0][e];
        part[(size_t)(1 * NE + e) * n + i] = acc[1][e];
        part[(size_t)(2 * NE + e) * n + i] = 0.0;
    }
}

// Bonded repulsion list: entry b couples atoms i, j with al = sqrt(repa_i repa_j),
// ab = repz_i repz_j 1.7583; its gradient contributes (w_i - w_j) . r_hat dE'/dtheta.
// One row of partials per entry: bpart[k * nb + b].
template <int NE>
__global__ __launch_bounds__(256) void k_adj_brep(int nb, const int* __restrict__ ij, const double* __restrict__ par,
                                                  const int* __restrict__ elem, const double* __restrict__ x,
                                                  const double* __restrict__ w, double* __restrict__ bpart) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nb) return;
    const int i = ij[2 * b], j = ij[2 * b + 1];
    const double3 d = ld3(x, i) - ld3(x, j);
    const double r = nrm(d);
    double dz_ = 0.0, da_ = 0.0;
    if (!(r > 20.0 || r < 1e-8)) {
        const double al = par[2 * b], ab = par[2 * b + 1];
        const double sw = dot(ld3(w, i) - ld3(w, j), d) / r;
        double dp_lnab, dp_al;
        rep_adj(ab, al, r, dp_lnab, dp_al);
        dz_ = sw * dp_lnab;
        da_ = sw * dp_al * 0.5 * al;
    }
    const int ei = elem[i], ej = elem[j];
#pragma unroll
    for (int e = 0; e < NE; ++e) {
        const double c = (e == ei ? 1.0 : 0.0) + (e == ej ? 1.0 : 0.0);
        bpart[(size_t)(0 * NE + e) * nb + b] = c * dz_;
        bpart[(size_t)(1 * NE + e) * nb + b] = c * da_;
        bpart[(size_t)(2 * NE + e) * nb + b] = 0.0;
    }
}

// Fixed-order reduction of the adjoint partials: workgroup (k, b) adds share b
// of the rows of output component k (by one wavefront per component it took
// 390 us for 33,700 atoms), then one wavefront per component adds the shares.
// Up to ADJ_ONE_MAX rows of all chunks one share is the sum, which saves the
// second launch and the idle workgroups of the first (whole call, one and 64
// shares: 6 atoms 46 and 73 us, 195 atoms 90 and 111, 900 atoms, 15,000 rows,
// 131 and 138; 1500 atoms, 26,500 rows, the same).
constexpr int ADJ_RB = 64;
constexpr int ADJ_ONE_MAX = 16384;
template <int RB>  // shares, 1 or ADJ_RB
__global__ __launch_bounds__(256) void k_adj_reduce(int n, int nchunk, const double* __restrict__ part, int nb,
                                                    const double* __restrict__ bpart, int nk,
                                                    double* __restrict__ share) {
    __shared__ double red[4];
    const int k = blockIdx.x, b = blockIdx.y, tid = threadIdx.x;
    double acc = 0.0;
    for (int c = 0; c < nchunk; ++c)
        for (int i = b * 256 + tid; i < n; i += RB * 256) acc += part[((size_t)c * nk + k) * n + i];
    for (int i = b * 256 + tid; i < nb; i += RB * 256) acc += bpart[(size_t)k * nb + i];
    acc = wg_sum256(acc, red);
    if (tid == 0) share[k * RB + b] = acc;
}
__global__ __launch_bounds__(64) void k_adj_final(const double* __restrict__ share, double* __restrict__ out) {
    const double v = wave_sum(share[blockIdx.x * ADJ_RB + threadIdx.x]);
    if (threadIdx.x == 0) out[blockIdx.x] = v;
}

// ---------------------------------------------------------------------------
// K9: gradient assembly: CN chain rule with Coulomb term 1b
// (ff_workspace.cpp:459-507), fixed order per atom, and the energies.
// ---------------------------------------------------------------------------
// LPA lanes per atom (64: one wavefront; 16 for short lists, four atoms per
// wavefront): lanes stride the atom's slot list and its CN neighbour list
// (chain rule), fixed butterfly over the atom's lanes
template <int W>
__device__ inline double group_sum(double v) {
#pragma unroll
    for (int o = W / 2; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}
// Per-atom sum of the bonded-list gradient slots (every slot writer runs
// before the EEQ solve, so this gather runs there too, off the solve's path),
// and of a single molecule's hydrogen-bond gradients (h.crange nullptr: none).
template <int LPA>
__global__ __launch_bounds__(256) void k_slot_gather(int n, const int* __restrict__ soff, const int* __restrict__ sidx,
                                                     const double* __restrict__ slots, HBGather h,
                                                     double* __restrict__ gslot) {
    const int lane = threadIdx.x & (LPA - 1);
    const int i = blockIdx.x * (256 / LPA) + threadIdx.x / LPA;
    if (i >= n) return;
    double3 g = make_double3(0, 0, 0);
    for (int k = soff[i] + lane; k < soff[i + 1]; k += LPA) g = g + ld3(slots, sidx[k]);
    if (h.crange) g = g + hb_gather<LPA>(i, lane, n, h);
    g.x = group_sum<LPA>(g.x);
    g.y = group_sum<LPA>(g.y);
    g.z = group_sum<LPA>(g.z);
    if (lane == 0) st3(gslot, i, g);
}

// Last launch of an evaluation, workgroups dealt to three jobs that do not
// depend on each other:
//  * the energies: NPARTS segments of up to RED_BLOCKS workgroups each, fixed
//    shape; the last workgroup to arrive adds the partial sums in a fixed order
//    and forms out[0] = total and out[1..15] = terms.  The partials are written
//    and read with device-coherent accesses, complete before the arrival is
//    counted, so no cache maintenance is needed;
//  * batches: the energy of every molecule, a wavefront each;
//  * the gradient: CN chain rule over an atom's neighbour list plus the
//    gathered slot, pair, hydrogen-bond and solvation gradients, LPA lanes per atom.
// Results go to the engine's buffers and to the caller's (out2, grad2).  Five
// launches of 4.5 us each before, for 122 atoms 24 us behind the pair terms.
constexpr int RED_BLOCKS = 64;
constexpr int NPARTS = 16;  // energy segments reduced per evaluation
struct FinishArgs {
    int n, nred, nmolb;  // workgroups per energy segment, and of the molecules' energies
    int first;           // workgroups ahead of this launch's (0; the energies', where their class is timed)
    const double *x, *rcov, *dlog, *v;
    const int *nbn, *nbl;
    const double *gslot, *gpair, *ghb, *gsolv;
    double *grad, *grad2;
    const double* seg[NPARTS];
    int cnt[NPARTS];
    double *part, *out, *out2;
    const int* flags;
    int *sticky, *arrived;
    MolEnergyArgs mol;
};

__device__ void reduce_segment(const FinishArgs& a, int sg, int b) {
    __shared__ double red[256];
    __shared__ int last;
    const double* p = a.seg[sg];
    const int n = a.cnt[sg], nb = a.nred, tid = threadIdx.x;
    const int chunk = (n + nb - 1) / nb;
    const int lo = b * chunk, hi = min(n, lo + chunk);
    // eight independent partial sums per thread keep eight loads in flight
    double a8[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int k = lo + tid; k < hi; k += 8 * 256) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const double v = p[min(k + u * 256, hi - 1)];  // unconditional load, masked add
            a8[u] += (k + u * 256 < hi) ? v : 0.0;
        }
    }
    red[tid] = ((a8[0] + a8[1]) + (a8[2] + a8[3])) + ((a8[4] + a8[5]) + (a8[6] + a8[7]));
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (tid < w) red[tid] += red[tid + w];
        __syncthreads();
    }
    if (tid == 0) {
        st_c(a.part + sg * RED_BLOCKS + b, red[0]);
        wait_vm();
        last = __hip_atomic_fetch_add(a.arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == NPARTS * nb - 1;
    }
    __syncthreads();
    if (!last) return;
    // 16 lanes per segment
    __shared__ double sp[NPARTS];
    {
        const int g = tid >> 4, l = tid & 15;
        double v = 0.0;
        for (int k = l; k < nb; k += 16) v += ld_c(a.part + g * RED_BLOCKS + k);
        v = group_sum<16>(v);
        if (l == 0) sp[g] = v;
    }
    __syncthreads();
    if (tid != 0) return;
    double t[GFNFF_NTERMS];
    for (int k = 0; k < GFNFF_NTERMS; ++k) t[k] = 0.0;
    // segments: 0 bond,1 angle,2 tors,3 inv,4 disp(pairs),5 brep,6 nbrep(pairs incl fix),7 coul pairs,
    // 8 self,9 hb case 1,10 atm,11 batm,12 triple-bond torsions,13 xb,14 hb cases 2-4,15 solvation
    t[GFNFF_E_BOND] = sp[0];
    t[GFNFF_E_ANGLE] = sp[1];
    t[GFNFF_E_TORSION] = sp[2];
    t[GFNFF_E_INVERSION] = sp[3];
    t[GFNFF_E_DISPERSION] = sp[4];
    t[GFNFF_E_BONDED_REP] = sp[5];
    t[GFNFF_E_NONBONDED_REP] = sp[6];
    t[GFNFF_E_COULOMB] = sp[7] + sp[8];
    t[GFNFF_E_HBOND] = sp[9] + sp[14];
    t[GFNFF_E_ATM] = sp[10];
    t[GFNFF_E_BATM] = sp[11];
    t[GFNFF_E_STORS] = sp[12];
    t[GFNFF_E_XBOND] = sp[13];
    t[GFNFF_E_SOLVATION] = sp[15];
    double tot = 0.0;
    for (int k = 0; k < GFNFF_NTERMS; ++k) tot += t[k];
    // a status flag raised in this evaluation (CN list overflow, EEQ pivot,
    // solver timeout) makes the total NaN and is kept in the sticky word
    // until the host reads and clears it
    const int f = final_flags(__hip_atomic_load(a.flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    if (f) {
        tot = __builtin_nan("");
        atomicOr(a.sticky, f);
    }
    a.out[0] = tot;
    for (int k = 0; k < GFNFF_NTERMS; ++k) a.out[1 + k] = t[k];
    if (a.out2) {
        a.out2[0] = tot;
        for (int k = 0; k < GFNFF_NTERMS; ++k) a.out2[1 + k] = t[k];
    }
}

template <int LPA>
__global__ __launch_bounds__(256) void k_finish(FinishArgs a) {
    int blk = blockIdx.x + a.first;
    if (blk < NPARTS * a.nred) {
        reduce_segment(a, blk / a.nred, blk % a.nred);
        return;
    }
    blk -= NPARTS * a.nred;
    if (blk < a.nmolb) {
        mol_energy(a.mol, blk * 4 + (threadIdx.x >> 6), threadIdx.x & 63);
        return;
    }
    blk -= a.nmolb;
    const int lane = threadIdx.x & (LPA - 1);
    const int i = blk * (256 / LPA) + threadIdx.x / LPA;
    if (i >= a.n) return;
    double3 g = make_double3(0, 0, 0);
    const double3 xi = ld3(a.x, i);
    const double ai = a.dlog[i] * a.v[i];
    const int nn = a.nbn[i];
    for (int k = lane; k < nn; k += LPA) {
        int j = a.nbl[(size_t)i * MAXNB_CN + k];
        double3 d = ld3(a.x, j) - xi;
        double r = nrm(d);
        double rs = a.rcov[i] + a.rcov[j];
        double dr = (r - rs) / rs;
        double dd = (KN / SQRTPI_TRUNC) * exp(-KN * KN * dr * dr) / rs;
        double s = dd * (ai + a.dlog[j] * a.v[j]);
        g = g + (-s / r) * d;
    }
    g.x = group_sum<LPA>(g.x);
    g.y = group_sum<LPA>(g.y);
    g.z = group_sum<LPA>(g.z);
    if (lane == 0) {
        g = g + ld3(a.gslot, i) + ld3(a.gpair, i);
        if (a.ghb) g = g + ld3(a.ghb, i);
        if (a.gsolv) g = g + ld3(a.gsolv, i);
        st3(a.grad, i, g);
        if (a.grad2) st3(a.grad2, i, g);
    }
}

__global__ void k_copy(int n, const double* __restrict__ a, double* __restrict__ b) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) b[i] = a[i];
}
__global__ void k_fill_i(int n, int* __restrict__ a, int v) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = v;
}

// ---------------------------------------------------------------------------
// K12: device-resident molecular dynamics.  Velocity Verlet as in
// SimpleMD::Verlet (simplemd.cpp:2580-2673) with the optional Berendsen bath
// of SimpleMD::Berendson (:3967-3975), in atomic units (Bohr, electron
// masses, atomic time units; gradient in Eh/Bohr).  One step:
//   k_md_drift   x += dt v - dt^2/2 g/m,  v -= dt/2 g/m   (g of the old x)
//   evaluation   g, Epot at the new x
//   k_md_kick    v -= dt/2 g/m; per-block partial sums of m v^2 and of the
//                displacement |x - x_ref|^2 since the last HB/XB detection
//   k_md_finish  Ekin, T = 2 Ekin / (kB dof), Berendsen factor, the step's
//                record (Epot, Ekin, T, Epot + Ekin), and GFNFF flag 8 when
//                sqrt(sum dx^2) / N exceeds the re-detection threshold
//                (gfnff_method.cpp:2243-2251)
//   k_md_scale   v *= lambda (bath only)
// Sums are formed in a fixed order; nothing is copied to the host.
// ---------------------------------------------------------------------------
constexpr int FLAG_HB_STALE = 8;
constexpr int MD_T = 256;

__global__ __launch_bounds__(MD_T) void k_md_drift(int n3, double dt, const double* __restrict__ im3,
                                                   const double* __restrict__ g, double* __restrict__ x,
                                                   double* __restrict__ v) {
    const int k = blockIdx.x * MD_T + threadIdx.x;
    if (k >= n3) return;
    const double a = g[k] * im3[k];
    x[k] = x[k] + dt * v[k] - 0.5 * a * dt * dt;
    v[k] = v[k] - 0.5 * dt * a;
}

__global__ __launch_bounds__(MD_T) void k_md_kick(int n3, double dt, const double* __restrict__ im3,
                                                  const double* __restrict__ m3, const double* __restrict__ g,
                                                  const double* __restrict__ x, const double* __restrict__ xref,
                                                  double* __restrict__ v, double* __restrict__ part) {
    __shared__ double sk[MD_T / 64], sd[MD_T / 64];
    const int k = blockIdx.x * MD_T + threadIdx.x;
    double ek = 0.0, dd = 0.0;
    if (k < n3) {
        const double vk = v[k] - 0.5 * dt * g[k] * im3[k];
        v[k] = vk;
        ek = m3[k] * vk * vk;
        const double dx = x[k] - xref[k];
        dd = dx * dx;
    }
    ek = wave_sum(ek);
    dd = wave_sum(dd);
    if ((threadIdx.x & 63) == 0) {
        sk[threadIdx.x >> 6] = ek;
        sd[threadIdx.x >> 6] = dd;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = (sk[0] + sk[1]) + (sk[2] + sk[3]);
        part[2 * blockIdx.x + 1] = (sd[0] + sd[1]) + (sd[2] + sd[3]);
    }
}

__global__ __launch_bounds__(64) void k_md_finish(int nb, const double* __restrict__ part,
                                                  const double* __restrict__ epot, double kb_dof, double dt, double T0,
                                                  double tau, double disp2_max, double* __restrict__ lambda,
                                                  double* __restrict__ rec, int* __restrict__ sticky) {
    const int lane = threadIdx.x;
    double ek = 0.0, dd = 0.0;
    for (int b = lane; b < nb; b += 64) {
        ek += part[2 * b];
        dd += part[2 * b + 1];
    }
    ek = 0.5 * wave_sum(ek);
    dd = wave_sum(dd);
    if (lane != 0) return;
    const double T = 2.0 * ek / kb_dof;
    double lam = 1.0;
    if (T0 > 0.0 && T > 0.0) lam = sqrt(1.0 + (dt / 2.0 * (T0 - T)) / (T * tau));
    *lambda = lam;
    rec[0] = epot[0];
    rec[1] = ek;
    rec[2] = T;
    rec[3] = epot[0] + ek;
    if (dd > disp2_max) atomicOr(sticky, FLAG_HB_STALE);
}

__global__ __launch_bounds__(MD_T) void k_md_scale(int n3, const double* __restrict__ lambda, double* __restrict__ v) {
    const int k = blockIdx.x * MD_T + threadIdx.x;
    if (k < n3) v[k] *= *lambda;
}

// ---------------------------------------------------------------------------
// K13: ALPB implicit solvation of one molecule, FP64 on both precision
// paths.  Born radii from the OBC-II transform of the pairwise descreening
// sum (alpb_solvation.cpp:502-690), surface areas on the 230-point angular
// grid with the smooth neighbour switching (:696-801), the H-bond diagonal
// (:873-881) and the shape descriptor (:908-938).  The Born matrix
// (P16 kernel, :810-867) is never stored: its entries are formed where they
// are used, added to the reduced EEQ matrix and right-hand side (the
// reference's A + B, eeq_solver.cpp:3774-3784), and contracted with the
// solved charges for the energy and the gradient at fixed charges
// (:1016-1041, :1139-1201, :1265-1300).  Every sum runs in a fixed order.
// ---------------------------------------------------------------------------
constexpr int SOLV_NB = 512;     // surface neighbours per atom (LDS list)
constexpr int SOLV_NANG = 230;   // angular grid points per atom
constexpr int FLAG_SOLV_NB = 16; // more than SOLV_NB surface neighbours
constexpr double ALPB_W = 0.3 / 0.52917726;
constexpr double ALPB_AH0 = 0.5;
constexpr double ALPB_AH1 = 3.0 / (4.0 * ALPB_W);
constexpr double ALPB_AH3 = -1.0 / (4.0 * ALPB_W * ALPB_W * ALPB_W);
constexpr double ALPB_ZETA = 1.028;
constexpr double ALPB_TOLSESP = 1.0e-6;

struct SolvArgs {
    int n;
    double keps, alpbet, c1, gshift, lr2, sr2;
    const double* x;
    const double *vdwr, *rho, *svdw, *vdwsa, *wrp, *trjlo, *trjhi, *gam, *hbmag, *grid;
    double *brad, *dbr, *sasa, *hbw;  // Born radius, d radius / d psi, surface area, H-bond diagonal
    double* sv;                       // [n][SOLV_NB][3] d sasa_i / d x_i per neighbour slot
    int *sj, *sn;                     // [n][SOLV_NB] neighbour of each slot (ascending), [n] count
    double* shape;                    // adet, totrad3, centre[3], inertia[9], gradient scale, cofactors[9]
    double *w, *c, *eat, *gs;         // radius weight, surface weight, atom energy, direct gradient [3n]
    double *e_solv, *parts;           // total, {gborn, ghb, gsasa, gshift}
    int* flags;
};

// One descreening contribution to psi of atom s from atom o at distance r
// (rho_o: descreening radius of o, rv: van der Waals radius of s), the
// non-overlapping or overlapping integral; dg = (d g / d r) / r.
__device__ inline double alpb_psi(double r, double rho_o, double rv, double& dg) {
    if (r >= rv + rho_o) {
        const double r1 = 1.0 / r, ap = r + rho_o, am = r - rho_o, ab = ap * am, rhab = rho_o / ab;
        const double lnab = 0.5 * log(am / ap) * r1;
        dg = -2.0 * rhab / ab + (rhab - lnab) * r1 * r1;
        return rhab + lnab;
    }
    if (r + rho_o <= rv) {
        dg = 0.0;
        return 0.0;
    }
    const double r1 = 1.0 / r, r12 = 0.5 * r1, r24 = r12 * r12, ap = r + rho_o, am = r - rho_o;
    const double rh1 = 1.0 / rv, rhr1 = 1.0 / ap, aprh1 = ap * rh1, lnab = log(aprh1);
    dg = (rhr1 * rhr1 * (1.0 - 0.25 * am * r1 * (1.0 + aprh1 * aprh1)) + rho_o * r24 * (rhr1 - rh1 * aprh1) +
          r12 * (r1 * lnab - rhr1)) *
         r1;
    return rh1 - rhr1 + r12 * (0.5 * am * (rhr1 - rh1 * aprh1) - lnab);
}

// P16 interaction a16 = (ab / (ab + zeta r / 16))^16; returns a1 = the base
__device__ inline double p16_pow(double ab, double r, double& a16) {
    const double a1 = ab / (ab + (ALPB_ZETA / 16.0) * r);
    double t = a1 * a1;
    t = t * t;
    t = t * t;
    a16 = t * t;
    return a1;
}

// Born matrix entry without the shape constant (which cancels in the
// reduced EEQ system: every reduced row and column sums entries with total
// weight zero)
__device__ inline double born_b(const SolvArgs& a, int i, int j) {
    if (i == j) return a.keps / a.brad[i] + 2.0 * a.hbw[i];
    const double3 d = ld3(a.x, i) - ld3(a.x, j);
    const double r = sqrt(dot(d, d)), ab = sqrt(a.brad[i] * a.brad[j]);
    double a16;
    (void)p16_pow(ab, r, a16);
    return a.keps / (r + ab * a16);
}

// Born radii: one wavefront per atom over all partners within lrcut
__device__ void solv_born(const SolvArgs& a, int blk) {
    const int i = blk * 4 + (threadIdx.x >> 6), l = threadIdx.x & 63;
    if (i >= a.n) return;  // wavefront-uniform
    const double3 xi = ld3(a.x, i);
    const double rvi = a.vdwr[i];
    double psi = 0.0;
    for (int j = l; j < a.n; j += 64) {
        if (j == i) continue;
        const double3 d = xi - ld3(a.x, j);
        const double r2 = dot(d, d);
        if (r2 >= a.lr2) continue;
        double dg;
        psi += alpb_psi(sqrt(r2), a.rho[j], rvi, dg);
    }
    psi = wave_sum(psi);
    if (l != 0) return;
    // OBC-II: R = c1 / (1/svdw - tanh(arg) / vdwr), arg a cubic in psi svdw / 2
    const double s1 = 1.0 / a.svdw[i], v1 = 1.0 / rvi, s2 = 0.5 * a.svdw[i];
    const double br = psi * s2;
    double arg2 = br * (4.85 * br - 0.8);
    const double arg = br * (1.0 + arg2);
    arg2 = 2.0 * arg2 + 1.0 + 4.85 * br * br;
    const double th = tanh(arg), ch = cosh(arg);
    a.brad[i] = a.c1 / (s1 - v1 * th);
    const double dp = ch * (s1 - v1 * th);
    a.dbr[i] = a.c1 * s2 * v1 * arg2 / (dp * dp);
}

// Surface area of atom i (one workgroup): the neighbours within srcut are
// compacted into LDS in ascending order; one thread per grid point forms
// the switched product; one thread per neighbour then sums its derivative
// over the grid points (no atomics).
__device__ void solv_shape(const SolvArgs& a);
// Geometry parts of one evaluation in one launch: the surface areas (a
// workgroup per atom), then the shape descriptor, then the Born radii.
__global__ __launch_bounds__(256) void k_solv_geom(SolvArgs a) {
    if ((int)blockIdx.x >= a.n) {
        if ((int)blockIdx.x == a.n)
            solv_shape(a);
        else
            solv_born(a, blockIdx.x - a.n - 1);
        return;
    }
    __shared__ double3 nx[SOLV_NB];
    __shared__ double nlo[SOLV_NB], nhi[SOLV_NB], nsa[SOLV_NB];
    __shared__ int nj[SOLV_NB];
    __shared__ double3 px[256];
    __shared__ double pw[256];
    __shared__ int wcnt[4];
    __shared__ double red[4];
    const int i = blockIdx.x, tid = threadIdx.x, l = tid & 63, wv = tid >> 6;
    const double3 xi = ld3(a.x, i);
    int cnt = 0;
    for (int j0 = 0; j0 < a.n; j0 += 256) {
        const int j = j0 + tid;
        bool in = false;
        if (j < a.n && j != i) {
            const double3 d = xi - ld3(a.x, j);
            const double r2 = dot(d, d);
            in = r2 < a.lr2 && r2 < a.sr2;
        }
        const unsigned long long b = __ballot(in);
        const int pre = __popcll(b & ((1ull << l) - 1ull));
        if (l == 0) wcnt[wv] = __popcll(b);
        __syncthreads();
        int off = cnt;
        for (int w = 0; w < wv; ++w) off += wcnt[w];
        const int tot = wcnt[0] + wcnt[1] + wcnt[2] + wcnt[3];
        if (in && off + pre < SOLV_NB) {
            const int s = off + pre;
            nx[s] = ld3(a.x, j);
            nlo[s] = a.trjlo[j];
            nhi[s] = a.trjhi[j];
            nsa[s] = a.vdwsa[j];
            nj[s] = j;
        }
        cnt += tot;
        __syncthreads();
    }
    if (cnt > SOLV_NB) {
        if (tid == 0) atomicOr(a.flags, FLAG_SOLV_NB);
        cnt = SOLV_NB;
    }
    const double rsa = a.vdwsa[i];
    double wsa = 0.0;
    double3 xp = xi;
    if (tid < SOLV_NANG) {
        const double* g = a.grid + 4 * tid;
        xp = make_double3(xi.x + rsa * g[0], xi.y + rsa * g[1], xi.z + rsa * g[2]);
        double sp = 1.0;
        for (int s = 0; s < cnt; ++s) {
            const double3 t = xp - nx[s];
            const double t2 = dot(t, t);
            if (t2 < nhi[s]) {
                if (t2 <= nlo[s]) {
                    sp = 0.0;
                    break;
                }
                const double u = sqrt(t2) - nsa[s], ah3u2 = ALPB_AH3 * u * u;
                sp *= ALPB_AH0 + (ALPB_AH1 + ah3u2) * u;
            }
        }
        if (sp > ALPB_TOLSESP) wsa = g[3] * a.wrp[i] * sp;
    }
    px[tid] = xp;
    pw[tid] = wsa;
    const double sasa = wg_sum256(wsa, red);  // its barriers also publish px and pw
    for (int s = tid; s < cnt; s += 256) {
        const double3 xj = nx[s];
        const double hi = nhi[s], sa = nsa[s];
        double vx = 0.0, vy = 0.0, vz = 0.0;
        for (int p = 0; p < SOLV_NANG; ++p) {
            const double w = pw[p];
            if (w == 0.0) continue;
            const double3 t = px[p] - xj;
            const double t2 = dot(t, t);
            if (t2 < hi) {
                const double sq = sqrt(t2), u = sq - sa, ah3u2 = ALPB_AH3 * u * u;
                const double f = ALPB_AH0 + (ALPB_AH1 + ah3u2) * u;
                const double df = w * (ALPB_AH1 + 3.0 * ah3u2) / (f * sq);
                vx += df * t.x;
                vy += df * t.y;
                vz += df * t.z;
            }
        }
        const size_t o = (size_t)i * SOLV_NB + s;
        a.sv[3 * o] = vx;
        a.sv[3 * o + 1] = vy;
        a.sv[3 * o + 2] = vz;
        a.sj[o] = nj[s];
    }
    if (tid == 0) {
        a.sasa[i] = sasa;
        a.hbw[i] = a.hbmag[i] * sasa / (rsa * rsa);
        a.sn[i] = cnt;
    }
}

// Shape descriptor (one workgroup): the inertia tensor of spheres with the
// van der Waals radii about their volume-weighted centre, and
// adet = sqrt(det^(1/3) / (2/5 sum r^3)).
__device__ void solv_shape(const SolvArgs& a) {
    __shared__ double red[4];
    const int tid = threadIdx.x;
    double tr = 0.0, cx = 0.0, cy = 0.0, cz = 0.0;
    for (int i = tid; i < a.n; i += 256) {
        const double r3 = a.vdwr[i] * a.vdwr[i] * a.vdwr[i];
        tr += r3;
        cx += a.x[3 * i] * r3;
        cy += a.x[3 * i + 1] * r3;
        cz += a.x[3 * i + 2] * r3;
    }
    tr = wg_sum256(tr, red);
    cx = wg_sum256(cx, red) / tr;
    cy = wg_sum256(cy, red) / tr;
    cz = wg_sum256(cz, red) / tr;
    double I[6] = {0, 0, 0, 0, 0, 0};  // xx, yy, zz, xy, xz, yz
    for (int i = tid; i < a.n; i += 256) {
        const double r2v = a.vdwr[i] * a.vdwr[i], r3 = r2v * a.vdwr[i];
        const double vx = a.x[3 * i] - cx, vy = a.x[3 * i + 1] - cy, vz = a.x[3 * i + 2] - cz;
        const double d = vx * vx + vy * vy + vz * vz + 0.4 * r2v;
        I[0] += r3 * (d - vx * vx);
        I[1] += r3 * (d - vy * vy);
        I[2] += r3 * (d - vz * vz);
        I[3] -= r3 * vx * vy;
        I[4] -= r3 * vx * vz;
        I[5] -= r3 * vy * vz;
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) I[k] = wg_sum256(I[k], red);
    if (tid != 0) return;
    const double xx = I[0], yy = I[1], zz = I[2], xy = I[3], xz = I[4], yz = I[5];
    const double det = xx * (yy * zz - yz * yz) - xy * (xy * zz - yz * xz) + xz * (xy * yz - yy * xz);
    double* s = a.shape;
    s[0] = sqrt(cbrt(det) / (0.4 * tr));
    s[1] = tr;
    s[2] = cx;
    s[3] = cy;
    s[4] = cz;
    const double full[9] = {xx, xy, xz, xy, yy, yz, xz, yz, zz};
    for (int k = 0; k < 9; ++k) s[5 + k] = full[k];
}

// Reduced Born matrix added to the reduced EEQ matrix, in the storage of
// k_eeq_reduced (full == 0: lower triangle of the row-major matrix, 1: also
// the upper triangle, 2: packed tiles with full diagonal tiles); gridDim.y
// workgroups share a tile (16 entries per thread in a row took 30 us at any
// size)
__global__ __launch_bounds__(256) void k_solv_red_add(int nr, int np, const int* __restrict__ ra,
                                                      const int* __restrict__ rl, SolvArgs a, double* __restrict__ A,
                                                      int full) {
    const int t = blockIdx.x;
    int bi = (int)((sqrt(8.0 * t + 1.0) - 1.0) * 0.5);
    while ((bi + 1) * (bi + 2) / 2 <= t) ++bi;
    while (bi * (bi + 1) / 2 > t) --bi;
    const int bj = t - bi * (bi + 1) / 2;
    for (int e = blockIdx.y * 256 + threadIdx.x; e < NB * NB; e += gridDim.y * 256) {
        const int rr = e >> 6, cc = e & 63, r = bi * NB + rr, c = bj * NB + cc;
        if (c > r || r >= nr || c >= nr) continue;
        const int ia = ra[r], la = rl[r], ib = ra[c], lb = rl[c];
        const double v = born_b(a, ia, ib) - born_b(a, ia, lb) - born_b(a, la, ib) + born_b(a, la, lb);
        if (full == 2) {
            A[(size_t)t * NB * NB + rr * NB + cc] += v;
            if (bi == bj && cc != rr) A[(size_t)t * NB * NB + cc * NB + rr] += v;
        } else {
            A[(size_t)r * np + c] += v;
            if (full == 1 && c != r) A[(size_t)c * np + r] += v;
        }
    }
}

// Preconditioner of the iterative EEQ solve: the inverse factors of the
// 64 x 64 diagonal blocks D of k_eeq_pcg (one workgroup per block; R is left
// intact).  Rows of split fragments (rowf >= 0) take A of their own fragment
// instead of R and nothing of the others; such a block also gets w = D^-1 1_f
// and 1_f . w for its pieces.  A need not be positive definite where R is: a
// block whose D fails is factored as it stands in R and takes no part in the
// rank-one terms (smon 0).
__global__ __launch_bounds__(256, 2) void k_bjacobi_setup(double* __restrict__ Rp, double* __restrict__ Lj,
                                                       int* __restrict__ flags, int nsf, PcgArgs pa,
                                                       const int* __restrict__ ra, const int* __restrict__ rl,
                                                       const double* __restrict__ x, const double* __restrict__ alp,
                                                       const double* __restrict__ diag, int solv, SolvArgs sv,
                                                       double* __restrict__ w, double* __restrict__ w1,
                                                       double* __restrict__ all, int* __restrict__ smon) {
    __shared__ double buf[16 * 17], v0[2 * NB];
    __shared__ int bad;
    const size_t I = blockIdx.x;
    double* const Rb = Rp + (I * (I + 1) / 2 + I) * NB * NB;
    double* const Li = Lj + I * NB * NB;
    const int tid = threadIdx.x;
    for (int k = (int)I * 256 + tid; k < pa.nmb; k += gridDim.x * 256) pa.mb[k] = MB_EMPTY;  // the solver's exchange buffers
    bool any = false;
    if (nsf > 0) any = __syncthreads_or(pa.rowf[I * NB + (tid & 63)] >= 0);
    if (!any) {  // uniform over the workgroup
        if (nsf > 0 && tid == 0) smon[I] = 0;
        if (tid < 64 && !chol64_wave(Rb, NB, Li, false, buf) && tid == 0) atomicOr(flags, FLAG_CHOL);
        return;
    }
    if (tid == 0) bad = 0;
    // D into Li, which chol64_wave reads before it writes the inverse there
    for (int e = tid; e < NB * NB; e += 256) {
        const int r = e >> 6, c = e & 63, fr = pa.rowf[I * NB + r], fc = pa.rowf[I * NB + c];
        double v;
        if (fr < 0 && fc < 0) {
            v = Rb[e];
        } else if (fr >= 0 && fr == fc) {
            const int ia = ra[I * NB + r], ib = ra[I * NB + c];
            v = eeq_a(ia, ib, x, alp, diag);
            if (solv) v += born_b(sv, ia, ib);
        } else {
            v = 0.0;
        }
        Li[e] = v;
        // the fragment's last atom, by its first row
        if (c == 0 && fr >= 0 && pa.pidx[pa.poff[fr >> 1]] == (int)(2 * I + (fr & 1)) &&
            (r == 0 || pa.rowf[I * NB + r - 1] != fr)) {
            const int la = rl[I * NB + r];
            const double d = diag[la] + (solv ? born_b(sv, la, la) : 0.0);
            all[fr >> 1] = d > 0.0 ? d : diag[la];
        }
    }
    __syncthreads();
    if (tid < 64 && !chol64_wave(Li, NB, Li, false, buf) && tid == 0) bad = 1;
    __syncthreads();
    const bool on = bad == 0;
    if (!on && tid < 64 && !chol64_wave(Rb, NB, Li, false, buf) && tid == 0) atomicOr(flags, FLAG_CHOL);
    __syncthreads();
    if (tid == 0) smon[I] = on;
    // w = L^-T (L^-1 1_f) per piece, the pieces of a block being disjoint: one
    // pass with both indicators, thread (t, q) a quarter of row t's products
    const int t = tid >> 2, q = tid & 3;
    double p0 = 0.0, p1 = 0.0;
    for (int u = 0; u < NB / 4; ++u) {
        const int c = 4 * u + q, fc = pa.rowf[I * NB + c];
        const double lv = Li[t * NB + c];
        if (fc >= 0) (fc & 1 ? p1 : p0) += lv;
    }
    p0 += __shfl_xor(p0, 1);
    p0 += __shfl_xor(p0, 2);
    p1 += __shfl_xor(p1, 1);
    p1 += __shfl_xor(p1, 2);
    if (q == 0) {
        v0[t] = p0;
        v0[NB + t] = p1;
    }
    __syncthreads();
    // rows of one piece couple only to their own indicator (D is block diagonal over the fragments)
    const int ft = pa.rowf[I * NB + t];
    double wt = 0.0;
    for (int u = 0; u < NB / 4; ++u) wt += Li[(4 * u + q) * NB + t] * v0[(ft & 1) * NB + 4 * u + q];
    wt += __shfl_xor(wt, 1);
    wt += __shfl_xor(wt, 2);
    if (ft < 0 || !on) wt = 0.0;
    __syncthreads();
    if (q == 0) {
        w[I * NB + t] = wt;
        v0[t] = wt;
    }
    __syncthreads();
    if (tid < NB) {
        const int f = pa.rowf[I * NB + tid];
        const double s0 = wave_sum(f >= 0 && !(f & 1) ? v0[tid] : 0.0), s1 = wave_sum(f >= 0 && (f & 1) ? v0[tid] : 0.0);
        if (tid < 2) w1[2 * I + tid] = tid ? s1 : s0;
    }
}

// Charged fragments: the Born part of A qp leaves the right-hand side
__global__ __launch_bounds__(256) void k_solv_rhs(SolvArgs a, const double* __restrict__ qp, double* __restrict__ r) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    double s = 0.0;
    for (int j = 0; j < a.n; ++j)
        if (qp[j] != 0.0) s += born_b(a, i, j) * qp[j];
    r[i] -= s;
}

// Born pair terms at the solved charges (one wavefront per atom i over all
// partners): atom energy, direct gradient, and d E / d R_i folded with
// d R_i / d psi_i; the surface weight gamma_i + d(H-bond)/d sasa_i.
__global__ __launch_bounds__(256) void k_solv_pairs(SolvArgs a, const double* __restrict__ q) {
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6), l = threadIdx.x & 63;
    if (i >= a.n) return;
    const double3 xi = ld3(a.x, i);
    const double Ri = a.brad[i], qi = q[i];
    double e = 0.0, gx = 0.0, gy = 0.0, gz = 0.0, dr = 0.0;
    for (int j = l; j < a.n; j += 64) {
        if (j == i) continue;
        const double3 d = xi - ld3(a.x, j);
        const double r = sqrt(dot(d, d)), Rj = a.brad[j], ab = sqrt(Ri * Rj), qj = q[j];
        double a16;
        const double a1 = p16_pow(ab, r, a16);
        const double df = 1.0 / (r + ab * a16), df2 = df * df;
        e += qj * df;
        const double ap = (1.0 - ALPB_ZETA * a1 * a16) * df2 * qj / r;
        gx -= ap * d.x;
        gy -= ap * d.y;
        gz -= ap * d.z;
        dr += Rj * (-0.5 * (r * ALPB_ZETA / ab * a1 + 1.0) / ab * a16 * df2) * qj;
    }
    e = wave_sum(e);
    gx = wave_sum(gx);
    gy = wave_sum(gy);
    gz = wave_sum(gz);
    dr = wave_sum(dr);
    if (l != 0) return;
    const double kq = a.keps * qi;
    a.eat[i] = 0.5 * kq * e + 0.5 * qi * qi * (a.keps / Ri + 2.0 * a.hbw[i]);
    a.gs[3 * i] = kq * gx;
    a.gs[3 * i + 1] = kq * gy;
    a.gs[3 * i + 2] = kq * gz;
    a.w[i] = (kq * dr - 0.5 * kq * qi / (Ri * Ri)) * a.dbr[i];
    a.c[i] = a.gam[i] + a.hbmag[i] / (a.vdwsa[i] * a.vdwsa[i]) * qi * qi;
}

// Solvation energy (one workgroup, fixed order) and the shape gradient's scale
__global__ __launch_bounds__(256) void k_solv_energy(SolvArgs a, const double* __restrict__ q) {
    __shared__ double red[4];
    double eb = 0.0, ehb = 0.0, es = 0.0, qt = 0.0;
    for (int i = threadIdx.x; i < a.n; i += 256) {
        eb += a.eat[i];
        ehb += a.hbw[i] * q[i] * q[i];
        es += a.gam[i] * a.sasa[i];
        qt += q[i];
    }
    eb = wg_sum256(eb, red);
    ehb = wg_sum256(ehb, red);
    es = wg_sum256(es, red);
    qt = wg_sum256(qt, red);
    if (threadIdx.x != 0) return;
    double* s = a.shape;
    const double ad = s[0], tr = s[1];
    double esh = 0.0;
    s[14] = 0.0;
    if (a.alpbet > 0.0) {
        esh = 0.5 * a.keps * a.alpbet * qt * qt / ad;
        s[14] = (250.0 / (48.0 * tr * tr * tr * pow(ad, 5.0))) * (-0.5 * a.keps * a.alpbet * qt * qt / (ad * ad));
    }
    // cofactor-type matrix of the inertia tensor (gbsa.f90:769-779)
    const double* I = s + 5;
    double* D = s + 15;
    D[0] = I[0] * (I[4] + I[8]) - I[1] * I[1] - I[2] * I[2];
    D[1] = I[1] * I[8] - I[2] * I[5];
    D[2] = I[2] * I[4] - I[1] * I[7];
    D[3] = D[1];
    D[4] = I[4] * (I[0] + I[8]) - I[1] * I[1] - I[5] * I[5];
    D[5] = I[0] * I[5] - I[1] * I[2];
    D[6] = D[2];
    D[7] = D[5];
    D[8] = I[8] * (I[0] + I[4]) - I[2] * I[2] - I[5] * I[5];
    a.parts[0] = eb - ehb + esh;
    a.parts[1] = ehb;
    a.parts[2] = es;
    a.parts[3] = a.gshift;
    a.e_solv[0] = ((eb + esh) + es) + a.gshift;
}

// Solvation gradient of atom k (one wavefront): the Born-radius chain rule
// over all partners within lrcut, the surface terms of k's own sphere and of
// every neighbour's sphere (k's slot in the neighbour's ascending list by
// bisection), the direct pair gradient and the shape term, into gs (k_finish
// adds it).
__global__ __launch_bounds__(256) void k_solv_grad(SolvArgs a) {
    const int k = blockIdx.x * 4 + (threadIdx.x >> 6), l = threadIdx.x & 63;
    if (k >= a.n) return;
    const double3 xk = ld3(a.x, k);
    const double wk = a.w[k], rvk = a.vdwr[k], rhok = a.rho[k], ck = a.c[k];
    double gx = 0.0, gy = 0.0, gz = 0.0;
    for (int j = l; j < a.n; j += 64) {
        if (j == k) continue;
        const double3 d = xk - ld3(a.x, j);
        const double r2 = dot(d, d);
        if (r2 >= a.lr2) continue;
        const double r = sqrt(r2);
        double d1, d2;
        (void)alpb_psi(r, a.rho[j], rvk, d1);
        (void)alpb_psi(r, rhok, a.vdwr[j], d2);
        const double f = wk * d1 + a.w[j] * d2;
        gx += f * d.x;
        gy += f * d.y;
        gz += f * d.z;
    }
    const int nk = a.sn[k];
    for (int s = l; s < nk; s += 64) {
        const size_t o = (size_t)k * SOLV_NB + s;
        gx += ck * a.sv[3 * o];
        gy += ck * a.sv[3 * o + 1];
        gz += ck * a.sv[3 * o + 2];
        const int j = a.sj[o];
        const int* lj = a.sj + (size_t)j * SOLV_NB;
        int lo = 0, hi = a.sn[j];
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (lj[mid] < k)
                lo = mid + 1;
            else
                hi = mid;
        }
        if (lo < a.sn[j] && lj[lo] == k) {
            const size_t oj = (size_t)j * SOLV_NB + lo;
            const double cj = a.c[j];
            gx -= cj * a.sv[3 * oj];
            gy -= cj * a.sv[3 * oj + 1];
            gz -= cj * a.sv[3 * oj + 2];
        }
    }
    gx = wave_sum(gx);
    gy = wave_sum(gy);
    gz = wave_sum(gz);
    if (l != 0) return;
    const double* s = a.shape;
    const double r3 = rvk * rvk * rvk * s[14];
    const double vx = xk.x - s[2], vy = xk.y - s[3], vz = xk.z - s[4];
    const double* D = s + 15;
    a.gs[3 * k] += gx + r3 * (D[0] * vx + D[1] * vy + D[2] * vz);
    a.gs[3 * k + 1] += gy + r3 * (D[3] * vx + D[4] * vy + D[5] * vz);
    a.gs[3 * k + 2] += gz + r3 * (D[6] * vx + D[7] * vy + D[8] * vz);
}

inline int cdiv(long a, long b) { return (int)((a + b - 1) / b); }

}  // namespace

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
// Kernel classes that can be timed with HIP events (one class at a time).
enum KernelClass {
    KC_CN, KC_EEQ_BUILD, KC_CHOL_DIAG, KC_CHOL_PANEL, KC_CHOL_UPDATE, KC_TRSV, KC_CHARGES, KC_PAIRS, KC_PAIRS_AUX,
    KC_NBREP, KC_REFINE, KC_BONDS, KC_ANGLES, KC_TORS, KC_BREP, KC_HB, KC_ATM, KC_BATM, KC_CHAIN, KC_REDUCE, KC_PCG,
    KC_BATCH_SOLVE, KC_SOLV, KC_COUNT
};
const char* const kKernelClassNames[KC_COUNT] = {
    "cn",    "eeq_build", "chol_diag", "chol_panel", "chol_update", "trsv", "charges", "pairs", "pairs_aux", "nbrep", "refine",
    "bonds", "angles",    "torsions",  "brep",       "hb",          "atm",  "batm",    "chain", "reduce", "pcg",
    "batch_solve", "solvation"};

// Start/stop event pairs around every launch of the selected class, recorded
// on the stream the kernels run on.
struct KernelTimer {
    int cls = -1;
    std::vector<hipEvent_t> ev;
    size_t used = 0;
    void mark(int c, hipStream_t s) {
        if (c != cls) return;
        if (used == ev.size()) {
            hipEvent_t e = nullptr;
            if (hipEventCreate(&e) != hipSuccess) {
                cls = -1;  // timing silently off when no event can be created; read() reports it
                return;
            }
            ev.push_back(e);
        }
        (void)hipEventRecord(ev[used++], s);
    }
    ~KernelTimer() {
        for (hipEvent_t e : ev) (void)hipEventDestroy(e);
    }
};

// Side stream and fork/join events for the factorisation lookahead.
struct Lookahead {
    hipStream_t side = nullptr;
    hipEvent_t fork = nullptr, join = nullptr;
};

#define LAUNCH(cls, kern, grid, block, stream, ...)                           \
    do {                                                                      \
        E->timer.mark(cls, stream);                                           \
        hipLaunchKernelGGL(kern, grid, block, 0, stream, __VA_ARGS__);        \
        E->timer.mark(cls, stream);                                           \
    } while (0)
#define LAUNCH_SHM(cls, kern, grid, block, shm, stream, ...)                  \
    do {                                                                      \
        E->timer.mark(cls, stream);                                           \
        hipLaunchKernelGGL(kern, grid, block, shm, stream, __VA_ARGS__);      \
        E->timer.mark(cls, stream);                                           \
    } while (0)

struct DeviceEngine {
    KernelTimer timer;
    int n = 0, nelem = 0, nfrag = 0;
    int nr = 0, np = 0;                 // reduced EEQ size, padded size
    int nbond = 0, nangle = 0, ntors = 0, nbrep = 0, nhb = 0, natm = 0, nbatm = 0, ninv = 0, nstors = 0, nxb = 0;
    int nslots = 0;
    int pair_cj = 0, pair_nchunk = 0;   // j-chunk size and count of the pair kernel
    int ps_nb = 0;                      // 64-atom blocks of the symmetric pair kernel (single molecules)
    int ps_split = 1;                   // wavefronts per tile
    int ps_ntiles = 0, ps_nblocks = 0;  // its tiles and 64-atom blocks (0 tiles: batches on the row kernel)
    const int4* ps_tiles = nullptr;     // batches: tiles {a0, n, R, C} of every molecule
    const int4* ps_blocks = nullptr;    // batches: blocks {a0, n, A, first tile of the molecule}
    double* tbox = nullptr;             // bounding boxes of the 256-atom tiles (CN partner pruning)
    hipStream_t side = nullptr;         // builds the reduced EEQ matrix alongside the evaluation stream
    hipEvent_t ev_fork = nullptr, ev_join = nullptr;
    hipEvent_t ev_fact = nullptr;       // batches: the factorisations on the side stream are done
    // batch_streams 2: the second half of the batch's factorisation on a third stream, forked from
    // and joined back to the side stream; per half h the column lists of batch_solver 5
    hipStream_t side2 = nullptr;
    hipEvent_t ev_h2f = nullptr, ev_h2j = nullptr;
    int batch_streams = 1;
    std::vector<int> h2_doff[2], h2_poff[2], h2_loff[2];
    int* h2_dmols[2] = {nullptr, nullptr};
    int4 *h2_ptiles[2] = {nullptr, nullptr}, *h2_ltiles[2] = {nullptr, nullptr};
    double* ps_part = nullptr;          // its per-tile row and column partials
    double* ps_part2 = nullptr;         // pair_split: the partials of dispersion and repulsion
    bool pair_split = false;            // dispersion and repulsion before the EEQ solve, Coulomb after
    bool mixed = false;                 // FP32 pair terms + FP32 factorisation with FP64 refinement
    Lookahead la;                       // side stream of the factorisation
    bool use_lookahead = false;
    bool use_cg = false;                // iterative EEQ solve (single molecules)
    int batch_solver = 5;               // batches: 0 / 1 variants of k_eeq_batch_factor, 2 k_eeq_batch_solve_tiles,
                                        // 3 factorisation by steps over the batch, 4 k_eeq_batch_fused,
                                        // 5 left-looking by column blocks over the batch
    bool batch_fp32 = false;            // mixed batches: FP32 factor with FP64 refinement
    bool solv = false;                  // ALPB solvation (single molecules)
    SolvArgs sa{};                      // its parameters and buffers
    int cg_groups = 0;                  // workgroups of the persistent PCG kernel
    double cg_tol2 = 0.0;               // squared relative residual at which the PCG solve stops
    double *cg_z = nullptr, *cg_p = nullptr;
    double* cg_part = nullptr;          // block-product partials [nbk][nbk][64]
    unsigned long long* cg_mb = nullptr;  // all-reduce mailboxes of the persistent PCG
    int* cg_iters = nullptr;
    PcgArgs cg{};                       // k_eeq_pcg
    bool cg_res = false, cg_one = false;  // k_eeq_pcg_res, k_eeq_pcg_one
    TermArgs terms{};                   // k_terms
    double *cg_w = nullptr, *cg_w1 = nullptr, *cg_all = nullptr;
    int* cg_smon = nullptr;
    int* ready = nullptr;               // per-block ready flags of the solve sweeps
    // batches of molecules (nmol > 1)
    int nmol = 1, nbtiles = 0;
    size_t mat_size = 0;                // doubles of the reduced EEQ matrix (or matrices)
    int *mol_of = nullptr, *mol_off = nullptr, *mol_seg = nullptr, *mnr = nullptr, *mnp = nullptr, *mvo = nullptr;
    int* morder = nullptr;  // batch: molecules by decreasing reduced size (solve launch order)
    bool cn_by_mol = false;  // batch of molecules of at most CNMOL_MAX atoms: k_cn_mol
    int cn_cap = 0;          // its LDS capacity in atoms (the largest molecule, rounded up to 64)
    long long* mmo = nullptr;
    int4* btiles = nullptr;
    // batch_solver 3: work of step k over the batch, at [off[k], off[k + 1]) of each list
    std::vector<int> bs_doff, bs_poff, bs_uoff;
    int* bs_dmols = nullptr;            // molecules with more than k column blocks
    int4* bs_ptiles = nullptr;          // panel tiles {m, bi, 0, 0}
    int4* bs_utiles = nullptr;          // trailing tiles {m, bi, bj, 0}
    // batch_solver 5: tiles {m, i, one-fragment flag, 0} of column block j at [ls_off[j], ls_off[j + 1])
    std::vector<int> ls_off;
    int4* ls_tiles = nullptr;
    // batch_solver 6: diagonal tiles and the tiles below them, per column block
    std::vector<int> l6d_off, l6o_off;
    int4 *l6d_tiles = nullptr, *l6o_tiles = nullptr;
    double* ured = nullptr;             // u of every reduced row (k_red_u)
    double* e_mol = nullptr;
    double *adj_w = nullptr, *adj_u = nullptr, *adj_part = nullptr, *adj_bpart = nullptr, *adj_share = nullptr, *adj_out = nullptr;
    float *Ared32 = nullptr, *Linv32 = nullptr, *b32 = nullptr, *y32 = nullptr, *d32 = nullptr;
    double *rvec = nullptr, *symv = nullptr;
    bool charged = false;
    hipStream_t own = nullptr;
    double* hpin = nullptr;  // pinned: coordinates and results of a host-buffer evaluation
    std::vector<void*> bufs;
    // parameters (device)
    int *Z, *elem, *nref, *metal, *toff, *tidx, *tdist;
    double *chi_base, *gam, *alp, *cnf, *rcov_cn, *rcov_d3, *hb_rad, *hb_lpd, *qa, *zeta, *szr, *anb, *repz, *refcn, *c6ref;
    int *red_atom, *red_last, *red_of, *frag_off, *frag_atoms;
    int *red_lidx, *red_ul, *red_nul;  // distinct last atoms per 64-block of reduced variables
    double* qp;
    int *bond_ij, *bond_H, *bond_hboff, *bond_hbB, *bond_slot;
    int *bsel_hb, *bsel_plain, nb_hb, nb_plain;  // bond indices with / without HB coordination
    int fin_lpa, hbg_lpa, slot_lpa;                // lanes per atom of k_finish, k_hb_gather and k_slot_gather
    double* bond_par;
    int *ang_ijk, *ang_slot;
    double* ang_par;
    int *tor_ijkl, *tor_slot;
    double* tor_par;
    int *inv_ijkl, *inv_slot, *st_ijkl, *st_slot, *xb_axb, *xb_slot;
    double *inv_par, *st_par, *xb_par;
    int *brep_ij, *brep_slot;
    double* brep_par;
    // hydrogen bonds by role (k_hb_roles): per-acceptor lists (CSR by atom),
    // role-grouped entries, group results, extra slots and the gather maps
    int *hb_nboff, *hb_nbidx, *hb_parc, *hb_nbcoff, *hb_nbcidx;
    int *hb_goff, *hb_gatom, *hb_crange, *hb_s0, *hb_xoff, *hb_xidx;
    int2* hb_ent;
    int4* hb_ahbc;
    int hb_ng0, hb_ng1, hb_ngt, nhb2, nhb2_c2;  // nhb2_c2: case-2 entries of the cases 2-4 list
    int* hb_ord = nullptr;                      // entries of the cases 2-4 list, case 2 first
    double *hb_cb, *hb_ca, *hb_Qh, *hb_Qab, *hb_gout, *hb_xslots, *e_hb2;
    float4* hb_pk;
    float* hb_qh32;
    int *atm_ijk, *atm_slot;
    double* atm_sc;
    int *batm_ijk, *batm_slot;
    double* batm_zb;
    int *slot_off, *slot_idx, *dcn_off, *dcn_idx;
    // work
    double *x, *cn, *dlog, *gw, *dgw, *rhs, *Ared, *Linv, *b, *rres, *q, *eself, *qtmp, *gpair, *dEdcn, *vchain,
        *slots, *dcn_slot, *grad, *e_coul, *e_disp, *e_rep, *e_bond, *e_ang, *e_tor, *e_brep, *e_hb, *e_atm,
        *e_batm, *e_inv, *e_st, *e_xb, *rpart, *out, *diag, *ghb, *gslot, *ybuf, *xbuf, *h6, *dh6, *ppart;
    int *nbn, *nbl, *flags;
    int* arrived = nullptr;  // workgroups of the energy reduction that have arrived (k_finish)
    int* sticky = nullptr;  // status flags of every evaluation since the last device_status read
    double *lu_w = nullptr, *lu_src = nullptr;  // LU fallback of a non-SPD reduced system (nr <= LU_MAX)

    PairArgs pair_args() const {
        PairArgs a;
        a.n = n;
        a.nelem = nelem;
        a.x = x;
        a.q = q;
        a.alp = alp;
        a.gw = gw;
        a.dgw = dgw;
        a.zeta = zeta;
        a.szr = szr;
        a.anb = anb;
        a.repz = repz;
        a.Z = Z;
        a.elem = elem;
        a.nref = nref;
        a.metal = metal;
        a.c6ref = c6ref;
        a.h = h6;
        a.dh = dh6;
        a.mol_of = mol_of;
        a.mol_off = mol_off;
        a.g = gpair;
        a.dEdcn = dEdcn;
        a.e_coul = e_coul;
        a.e_disp = e_disp;
        a.e_rep = e_rep;
        return a;
    }
    template <class T>
    T* alloc(size_t count) {
        void* p = nullptr;
        size_t bytes = std::max<size_t>(count, 1) * sizeof(T);
        if (hipMalloc(&p, bytes) != hipSuccess) throw std::bad_alloc();
        bufs.push_back(p);
        return (T*)p;
    }
    template <class T>
    T* upload(const std::vector<T>& v) {
        T* d = alloc<T>(v.size());
        if (!v.empty() && hipMemcpy(d, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice) != hipSuccess)
            throw std::runtime_error("upload failed");
        return d;
    }
    double *md_im3 = nullptr, *md_m3 = nullptr, *md_xref = nullptr, *md_part = nullptr, *md_e = nullptr,
           *md_lambda = nullptr;        // molecular dynamics state (device_md_steps)
    hipGraph_t graph = nullptr;         // captured device-resident evaluation (gfnff_graph_capture)
    hipGraphExec_t gexec = nullptr;
    void drop_graph() {
        if (gexec) (void)hipGraphExecDestroy(gexec);
        if (graph) (void)hipGraphDestroy(graph);
        gexec = nullptr;
        graph = nullptr;
    }
    ~DeviceEngine() {
        drop_graph();
        if (la.side) {
            (void)hipStreamSynchronize(la.side);
            (void)hipStreamDestroy(la.side);
        }
        if (la.fork) (void)hipEventDestroy(la.fork);
        if (la.join) (void)hipEventDestroy(la.join);
        if (side) {
            (void)hipStreamSynchronize(side);
            (void)hipStreamDestroy(side);
        }
        if (ev_fork) (void)hipEventDestroy(ev_fork);
        if (ev_join) (void)hipEventDestroy(ev_join);
        if (ev_fact) (void)hipEventDestroy(ev_fact);
        if (side2) {
            (void)hipStreamSynchronize(side2);
            (void)hipStreamDestroy(side2);
        }
        if (ev_h2f) (void)hipEventDestroy(ev_h2f);
        if (ev_h2j) (void)hipEventDestroy(ev_h2j);
        if (own) {
            (void)hipStreamSynchronize(own);
            (void)hipStreamDestroy(own);
        }
        if (hpin) (void)hipHostFree(hpin);
        for (void* p : bufs) (void)hipFree(p);
    }
};

// Order of the reduced variables of the iterative solve: the atoms of a
// fragment of more than 64 variables in breadth-first order over its bonds
// from an end of the molecule (the last atom of two searches), so that a
// 64-variable block holds neighbouring atoms; in an alkane's own order one
// block holds carbons and another their hydrogens, and the block-Jacobi
// preconditioner misses the coupling between them.  The last atom, whose
// variable is eliminated, stays the last.
static void reduced_order(const ParamSet& P, std::vector<std::vector<int>>& fa) {
    std::vector<std::vector<int>> nb;
    for (std::vector<int>& at : fa) {
        if ((int)at.size() - 1 <= NB) continue;
        if (nb.empty()) {
            nb.resize(P.n);
            for (size_t k = 0; k + 1 < P.bond_ij.size(); k += 2) {
                nb[P.bond_ij[k]].push_back(P.bond_ij[k + 1]);
                nb[P.bond_ij[k + 1]].push_back(P.bond_ij[k]);
            }
            for (auto& v : nb) std::sort(v.begin(), v.end());
        }
        const int last = at.back();
        std::vector<int> order;
        std::vector<char> seen(P.n, 0), mine(P.n, 0);
        for (int i : at) mine[i] = 1;
        int start = at[0];
        for (int pass = 0; pass < 3; ++pass) {
            order.assign(1, start);
            std::fill(seen.begin(), seen.end(), 0);
            seen[start] = 1;
            for (size_t k = 0; k < order.size(); ++k)
                for (int j : nb[order[k]])
                    if (mine[j] && !seen[j]) {
                        seen[j] = 1;
                        order.push_back(j);
                    }
            start = order.back();
        }
        for (int i : at)  // atoms that no bond of the list reaches keep their order
            if (!seen[i]) order.push_back(i);
        order.erase(std::find(order.begin(), order.end(), last));
        order.push_back(last);
        at.swap(order);
    }
}

DeviceEngine* device_create(const ParamSet& P, int precision, const Options& opt, int& status, std::string& msg) {
    const bool lookahead = opt.cholesky_lookahead;
    const int solver = opt.eeq_solver;
    const double pcg_tol = opt.pcg_tol;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) {
        status = kErrDevice;
        msg = "no HIP device available";
        return nullptr;
    }
    if (precision != 0 && precision != 1) {
        status = kErrArgs;
        msg = "unknown precision mode";
        return nullptr;
    }
    for (size_t h = 0; h < P.hb_case.size(); ++h)
        if (P.hb_case[h] == 3 && P.hb_parentC[h] >= 0 &&
            (P.hb_nbB_off[h + 1] - P.hb_nbB_off[h] != 1 || P.hb_nbB_idx[P.hb_nbB_off[h]] != P.hb_parentC[h])) {
            status = kErrArgs;
            msg = "hydrogen-bond case 3 needs the carbonyl carbon as the acceptor's only neighbour";
            return nullptr;
        }
    auto* E = new DeviceEngine();
    E->mixed = precision == 1;
    E->use_lookahead = lookahead;
    E->use_cg = solver == 0 && P.nmol == 1;
    E->batch_solver = opt.batch_solver;
    E->batch_streams = (opt.batch_streams == 2 && opt.batch_solver == 5 && P.nmol > 1) ? 2 : 1;
    E->batch_fp32 = opt.batch_fp32 != 0;
    {
        const double tol = pcg_tol > 0.0 ? pcg_tol : (E->mixed ? PCG_TOL_MIXED : PCG_TOL_FP64);
        E->cg_tol2 = tol * tol;
    }
    const bool default_tol = !(pcg_tol > 0.0);
    try {
        const int n = P.n;
        E->n = n;
        E->nelem = P.nelem;
        E->nfrag = P.nfrag;
        if (P.nelem * P.nelem * 49 > 16 * 49) {
            status = kErrUnsupported;
            msg = "more than 4 distinct elements are not supported by the pair kernel yet";
            delete E;
            return nullptr;
        }
        E->Z = E->upload(P.Z);
        E->elem = E->upload(P.elem);
        E->nref = E->upload(P.nref);
        E->metal = E->upload(P.metal);
        E->toff = E->upload(P.topo_off);
        E->tidx = E->upload(P.topo_idx);
        E->tdist = E->upload(P.topo_dist);
        E->chi_base = E->upload(P.chi_base);
        E->gam = E->upload(P.gam_eff);
        E->alp = E->upload(P.alpeeq);
        E->cnf = E->upload(P.cnf);
        E->rcov_cn = E->upload(P.rcov_cn);
        E->rcov_d3 = E->upload(P.rcov_d3);
        E->hb_rad = E->upload(P.hb_rad);
        E->hb_lpd = E->upload(P.hb_lpd);
        E->qa = E->upload(P.qa);
        E->zeta = E->upload(P.zeta);
        E->szr = E->upload(P.sqrt_zr4r2);
        E->anb = E->upload(P.rep_anb);
        E->repz = E->upload(P.repz);
        E->refcn = E->upload(P.refcn);
        E->c6ref = E->upload(P.c6ref);

        // fragment null-space reduction
        std::vector<std::vector<int>> fa(P.nfrag);
        for (int i = 0; i < n; ++i) fa[P.frag[i]].push_back(i);
        std::vector<int> red_atom, red_last, red_of(n, -1), foff(P.nfrag + 1, 0), fatoms;
        std::vector<double> qp(n, 0.0);
        // On the mixed path the pair terms take the charges rounded to FP32, so that
        // two solves that agree to the tolerance can round a charge to
        // neighbouring values; one such step moves the gradient by up to 1.6e-7 of
        // its RMS where charges reach 0.5 e (a peptide), by 4e-9 where they stay
        // below 0.1 e (hydrocarbons).  There the order and the preconditioner of
        // long fragments apply on both paths, for polar molecules on the FP64 path
        // only, whose charges converge to rounding: a long polar molecule keeps its
        // results and its iterations on the mixed path (H-(Gly)200-OH 97, FP64 39).
        double qmax = 0.0;
        for (double v : P.qa) qmax = std::max(qmax, std::fabs(v));
        const bool long_frag = E->use_cg && (!E->mixed || qmax <= 0.1);
        if (long_frag) reduced_order(P, fa);
        for (int f = 0; f < P.nfrag; ++f) {
            int m = (int)fa[f].size();
            int last = fa[f].back();
            for (int k = 0; k + 1 < m; ++k) {
                red_of[fa[f][k]] = (int)red_atom.size();
                red_atom.push_back(fa[f][k]);
                red_last.push_back(last);
            }
            for (int a : fa[f]) {
                qp[a] = P.qfrag[f] / m;
                fatoms.push_back(a);
            }
            foff[f + 1] = (int)fatoms.size();
            if (P.qfrag[f] != 0.0) E->charged = true;
        }
        E->nr = (int)red_atom.size();
        E->np = std::max(NB, cdiv(std::max(E->nr, 1), NB) * NB);
        E->mat_size = (size_t)E->np * E->np;
        if (P.nmol > 1) {
            // batch: each molecule's fragments form their own padded block
            E->nmol = P.nmol;
            std::vector<int> ra2, rl2, mnr(P.nmol), mnp(P.nmol), vo(P.nmol);
            std::vector<long long> mo(P.nmol);
            std::vector<int> fr_first(P.nmol + 1, 0);
            for (int f = 0; f < P.nfrag; ++f) fr_first[P.mol_of_atom(fa[f][0]) + 1] = f + 1;
            for (int m = 0; m < P.nmol; ++m) fr_first[m + 1] = std::max(fr_first[m + 1], fr_first[m]);
            long long off = 0;
            for (int m = 0; m < P.nmol; ++m) {
                vo[m] = (int)ra2.size();
                int loc = 0;
                for (int f = fr_first[m]; f < fr_first[m + 1]; ++f) {
                    const int cnt = (int)fa[f].size(), last = fa[f].back();
                    for (int k = 0; k + 1 < cnt; ++k) {
                        red_of[fa[f][k]] = (int)ra2.size();
                        ra2.push_back(fa[f][k]);
                        rl2.push_back(last);
                        ++loc;
                    }
                }
                mnr[m] = loc;
                mnp[m] = std::max(NB, cdiv(std::max(loc, 1), NB) * NB);
                if (mnp[m] > BATCH_MAX_NP) throw std::runtime_error("batched molecule too large");
                while ((int)ra2.size() < vo[m] + mnp[m]) {
                    ra2.push_back(-1);
                    rl2.push_back(-1);
                }
                mo[m] = off;
                off += (long long)mnp[m] * mnp[m];
            }
            red_atom.swap(ra2);
            red_last.swap(rl2);
            E->nr = (int)red_atom.size();
            E->np = E->nr;
            E->mat_size = (size_t)off;
            std::vector<int4> tiles;
            for (int m = 0; m < P.nmol; ++m)
                for (int bi = 0; bi < mnp[m] / NB; ++bi)
                    for (int bj = 0; bj <= bi; ++bj) tiles.push_back(make_int4(m, bi, bj, 0));
            E->nbtiles = (int)tiles.size();
            E->btiles = E->upload(tiles);
            {
                int maxnb = 0;
                for (int m = 0; m < P.nmol; ++m) maxnb = std::max(maxnb, mnp[m] / NB);
                std::vector<std::vector<int>> dm(maxnb);
                std::vector<std::vector<int4>> pt(maxnb), ut(maxnb);
                for (int m = 0; m < P.nmol; ++m) {
                    const int nbm = mnp[m] / NB;
                    for (int k = 0; k < nbm; ++k) {
                        dm[k].push_back(m);
                        for (int bi = k + 1; bi < nbm; ++bi) {
                            pt[k].push_back(make_int4(m, bi, 0, 0));
                            for (int bj = k + 1; bj <= bi; ++bj) ut[k].push_back(make_int4(m, bi, bj, 0));
                        }
                    }
                }
                std::vector<int> dflat;
                std::vector<int4> pflat, uflat;
                E->bs_doff.assign(1, 0);
                E->bs_poff.assign(1, 0);
                E->bs_uoff.assign(1, 0);
                for (int k = 0; k < maxnb; ++k) {
                    dflat.insert(dflat.end(), dm[k].begin(), dm[k].end());
                    pflat.insert(pflat.end(), pt[k].begin(), pt[k].end());
                    uflat.insert(uflat.end(), ut[k].begin(), ut[k].end());
                    E->bs_doff.push_back((int)dflat.size());
                    E->bs_poff.push_back((int)pflat.size());
                    E->bs_uoff.push_back((int)uflat.size());
                }
                E->bs_dmols = E->upload(dflat);
                if (!pflat.empty()) E->bs_ptiles = E->upload(pflat);
                if (!uflat.empty()) E->bs_utiles = E->upload(uflat);
                // left-looking column tiles; a molecule is one-fragment when
                // all its reduced rows share the last atom
                std::vector<int4> lflat;
                E->ls_off.assign(1, 0);
                std::vector<int> uni(P.nmol, 1);
                for (int m = 0; m < P.nmol; ++m)
                    for (int r = 1; r < mnr[m]; ++r)
                        if (red_last[vo[m] + r] != red_last[vo[m]]) uni[m] = 0;
                for (int j = 0; j < maxnb; ++j) {
                    for (int m = 0; m < P.nmol; ++m)
                        for (int i = j; i < mnp[m] / NB; ++i) lflat.push_back(make_int4(m, i, uni[m] && mnr[m] > 0, 0));
                    E->ls_off.push_back((int)lflat.size());
                }
                E->ls_tiles = E->upload(lflat);
                // batch_solver 6: per column block the diagonal tiles, then the tiles below them
                std::vector<int4> dl, ol;
                E->l6d_off.assign(1, 0);
                E->l6o_off.assign(1, 0);
                for (int j = 0; j < maxnb; ++j) {
                    for (int k = E->ls_off[j]; k < E->ls_off[j + 1]; ++k) (lflat[k].y == j ? dl : ol).push_back(lflat[k]);
                    E->l6d_off.push_back((int)dl.size());
                    E->l6o_off.push_back((int)ol.size());
                }
                E->l6d_tiles = E->upload(dl);
                if (!ol.empty()) E->l6o_tiles = E->upload(ol);
                // batch_streams 2: molecules dealt alternately, by decreasing size, to two halves
                if (E->batch_streams == 2) {
                    std::vector<int> ordm(P.nmol), half(P.nmol);
                    for (int m = 0; m < P.nmol; ++m) ordm[m] = m;
                    std::stable_sort(ordm.begin(), ordm.end(), [&](int a, int b) { return mnp[a] > mnp[b]; });
                    for (int k = 0; k < P.nmol; ++k) half[ordm[k]] = k & 1;
                    for (int h = 0; h < 2; ++h) {
                        std::vector<int> d2;
                        std::vector<int4> p2, l2;
                        E->h2_doff[h].assign(1, 0);
                        E->h2_poff[h].assign(1, 0);
                        E->h2_loff[h].assign(1, 0);
                        for (int j = 0; j < maxnb; ++j) {
                            for (int m : dm[j])
                                if (half[m] == h) d2.push_back(m);
                            for (const int4& t : pt[j])
                                if (half[t.x] == h) p2.push_back(t);
                            for (int k = E->ls_off[j]; k < E->ls_off[j + 1]; ++k)
                                if (half[lflat[k].x] == h) l2.push_back(lflat[k]);
                            E->h2_doff[h].push_back((int)d2.size());
                            E->h2_poff[h].push_back((int)p2.size());
                            E->h2_loff[h].push_back((int)l2.size());
                        }
                        if (!d2.empty()) E->h2_dmols[h] = E->upload(d2);
                        if (!p2.empty()) E->h2_ptiles[h] = E->upload(p2);
                        if (!l2.empty()) E->h2_ltiles[h] = E->upload(l2);
                    }
                }
            }
            E->mnr = E->upload(mnr);
            E->mnp = E->upload(mnp);
            {
                // workgroup order of the per-molecule solves: largest reduced
                // systems first, so the long factorizations start early
                std::vector<int> order(P.nmol);
                std::iota(order.begin(), order.end(), 0);
                std::stable_sort(order.begin(), order.end(), [&](int a2, int b2) { return mnp[a2] > mnp[b2]; });
                E->morder = E->upload(order);
            }
            int maxat = 0;
            for (int m2 = 0; m2 < P.nmol; ++m2) maxat = std::max(maxat, P.mol_off[m2 + 1] - P.mol_off[m2]);
            E->cn_by_mol = maxat <= CNMOL_MAX;
            E->cn_cap = std::max(64, (maxat + 63) / 64 * 64);
            E->mvo = E->upload(vo);
            E->mmo = E->upload(mo);
            E->mol_off = E->upload(P.mol_off);
            std::vector<int> mof(n);
            for (int m = 0; m < P.nmol; ++m)
                for (int i = P.mol_off[m]; i < P.mol_off[m + 1]; ++i) mof[i] = m;
            E->mol_of = E->upload(mof);
            E->mol_seg = E->upload(P.mol_seg);
            E->e_mol = E->alloc<double>(P.nmol);
        }
        E->red_atom = E->upload(red_atom);
        E->red_last = E->upload(red_last);
        {
            // per 64-block of reduced variables: its distinct last atoms (in
            // order of appearance) and each variable's index among them
            const int nbk0 = E->np / NB;
            std::vector<int> lidx(E->np, 0), ul((size_t)E->np, -1), nul(std::max(nbk0, 1), 0);
            for (int bk = 0; bk < nbk0; ++bk) {
                int cnt = 0;
                for (int r = bk * NB; r < std::min((bk + 1) * NB, E->nr); ++r) {
                    const int la = red_last[r];
                    int u = 0;
                    while (u < cnt && ul[(size_t)bk * NB + u] != la) ++u;
                    if (u == cnt) ul[(size_t)bk * NB + cnt++] = la;
                    lidx[r] = u;
                }
                nul[bk] = cnt;
            }
            E->red_lidx = E->upload(lidx);
            E->red_ul = E->upload(ul);
            E->red_nul = E->upload(nul);
        }
        E->red_of = E->upload(red_of);
        E->frag_off = E->upload(foff);
        E->frag_atoms = E->upload(fatoms);
        E->qp = E->upload(qp);

        // term lists and gradient slots
        int slot = 0;
        std::vector<int> slot_atom;
        auto add_slot = [&](int atom) {
            slot_atom.push_back(atom);
            return slot++;
        };
        // bonds: i, j, (H, B...) for HB-modulated bonds
        E->nbond = (int)P.bond_hbH.size();
        std::vector<int> bhoff(E->nbond + 1, 0), bhB, bslot(E->nbond);
        {
            std::vector<std::vector<int>> byH(n);
            for (size_t k = 0; k + 1 < P.hbcn_pair.size(); k += 2) byH[P.hbcn_pair[k]].push_back(P.hbcn_pair[k + 1]);
            for (int b = 0; b < E->nbond; ++b) {
                int H = P.bond_hbH[b];
                bslot[b] = add_slot(P.bond_ij[2 * b]);
                add_slot(P.bond_ij[2 * b + 1]);
                if (H >= 0) {
                    add_slot(H);
                    for (int B : byH[H]) {
                        bhB.push_back(B);
                        add_slot(B);
                    }
                }
                bhoff[b + 1] = (int)bhB.size();
            }
        }
        E->bond_ij = E->upload(P.bond_ij);
        E->bond_par = E->upload(P.bond_par);
        E->bond_H = E->upload(P.bond_hbH);
        E->bond_hboff = E->upload(bhoff);
        E->bond_hbB = E->upload(bhB);
        E->bond_slot = E->upload(bslot);
        {
            std::vector<int> bh, bp;
            for (int b = 0; b < (int)P.bond_hbH.size(); ++b)
                (P.bond_hbH[b] >= 0 && bhoff[b + 1] > bhoff[b] ? bh : bp).push_back(b);
            E->nb_hb = (int)bh.size();
            E->nb_plain = (int)bp.size();
            E->bsel_hb = E->upload(bh);
            E->bsel_plain = E->upload(bp);
        }
        E->nangle = (int)(P.angle_par.size() / 2);
        std::vector<int> aslot(E->nangle);
        for (int t = 0; t < E->nangle; ++t) {
            aslot[t] = add_slot(P.angle_ijk[3 * t]);
            add_slot(P.angle_ijk[3 * t + 1]);
            add_slot(P.angle_ijk[3 * t + 2]);
        }
        E->ang_ijk = E->upload(P.angle_ijk);
        E->ang_par = E->upload(P.angle_par);
        E->ang_slot = E->upload(aslot);
        E->ntors = (int)(P.tors_par.size() / 4);
        std::vector<int> tslot(E->ntors);
        for (int t = 0; t < E->ntors; ++t) {
            tslot[t] = add_slot(P.tors_ijkl[4 * t]);
            for (int a = 1; a < 4; ++a) add_slot(P.tors_ijkl[4 * t + a]);
        }
        E->tor_ijkl = E->upload(P.tors_ijkl);
        E->tor_par = E->upload(P.tors_par);
        E->tor_slot = E->upload(tslot);
        E->ninv = (int)(P.inv_par.size() / 3);
        std::vector<int> islot(E->ninv);
        for (int t = 0; t < E->ninv; ++t) {
            islot[t] = add_slot(P.inv_ijkl[4 * t]);
            for (int a = 1; a < 4; ++a) add_slot(P.inv_ijkl[4 * t + a]);
        }
        E->inv_ijkl = E->upload(P.inv_ijkl);
        E->inv_par = E->upload(P.inv_par);
        E->inv_slot = E->upload(islot);
        E->nstors = (int)P.stors_par.size();
        std::vector<int> sslot(E->nstors);
        for (int t = 0; t < E->nstors; ++t) {
            sslot[t] = add_slot(P.stors_ijkl[4 * t]);
            for (int a = 1; a < 4; ++a) add_slot(P.stors_ijkl[4 * t + a]);
        }
        E->st_ijkl = E->upload(P.stors_ijkl);
        E->st_par = E->upload(P.stors_par);
        E->st_slot = E->upload(sslot);
        E->nxb = (int)(P.xb_par.size() / 3);
        std::vector<int> xslot(E->nxb);
        for (int t = 0; t < E->nxb; ++t) {
            xslot[t] = add_slot(P.xb_axb[3 * t]);
            add_slot(P.xb_axb[3 * t + 1]);
            add_slot(P.xb_axb[3 * t + 2]);
        }
        E->xb_axb = E->upload(P.xb_axb);
        E->xb_par = E->upload(P.xb_par);
        E->xb_slot = E->upload(xslot);
        E->nbrep = (int)(P.brep_par.size() / 2);
        std::vector<int> rslot(E->nbrep);
        for (int b = 0; b < E->nbrep; ++b) {
            rslot[b] = add_slot(P.brep_ij[2 * b]);
            add_slot(P.brep_ij[2 * b + 1]);
        }
        E->brep_ij = E->upload(P.brep_ij);
        E->brep_par = E->upload(P.brep_par);
        E->brep_slot = E->upload(rslot);
        E->nhb = (int)P.hb_case.size();
        {
            // Hydrogen bonds.  The reference's per-triplet parameters are
            // per-atom values and its neighbour lists depend on the acceptor
            // only; both are checked while they are gathered.  Case-1 triplets
            // go to the role lists, cases 2-4 to a compact list with slots.
            const int nh = E->nhb;
            if (nh && n >= (1 << 28)) throw std::runtime_error("hydrogen-bond lists need atom indices below 2^28");
            std::vector<double> cb(n, 0.0), ca(n, 0.0), qt(n, 0.0);
            std::vector<char> s_cb(n, 0), s_ca(n, 0), s_qt(n, 0);
            auto put = [](std::vector<double>& v, std::vector<char>& set, int i, double val) {
                if (set[i] && v[i] != val) throw std::runtime_error("hydrogen-bond parameter is not a per-atom value");
                v[i] = val;
                set[i] = 1;
            };
            std::vector<std::vector<int>> bnb(n), bD(n);
            std::vector<int> bC(n, -1);
            std::vector<char> s_nb(n, 0), s_c(n, 0);
            for (int h = 0; h < nh; ++h) {
                const int A = P.hb_ahb[3 * h], H = P.hb_ahb[3 * h + 1], B = P.hb_ahb[3 * h + 2], cs = P.hb_case[h];
                const double* q = &P.hb_par[7 * (size_t)h];
                put(cb, s_cb, A, q[0]);
                put(cb, s_cb, B, q[1]);
                put(ca, s_ca, A, q[2]);
                put(ca, s_ca, B, q[3]);
                put(qt, s_qt, H, q[4]);
                put(qt, s_qt, A, q[5]);
                put(qt, s_qt, B, q[6]);
                if (cs < 1 || cs > 4) throw std::runtime_error("unknown hydrogen-bond case");
                if (cs >= 2) {
                    std::vector<int> l(P.hb_nbB_idx.begin() + P.hb_nbB_off[h], P.hb_nbB_idx.begin() + P.hb_nbB_off[h + 1]);
                    if (s_nb[B] && bnb[B] != l) throw std::runtime_error("acceptor neighbour lists differ between hydrogen bonds");
                    bnb[B] = l;
                    s_nb[B] = 1;
                }
                if (cs == 3) {
                    std::vector<int> l(P.hb_nbC_idx.begin() + P.hb_nbC_off[h], P.hb_nbC_idx.begin() + P.hb_nbC_off[h + 1]);
                    if (s_c[B] && (bC[B] != P.hb_parentC[h] || bD[B] != l))
                        throw std::runtime_error("carbonyl lists differ between hydrogen bonds");
                    bC[B] = P.hb_parentC[h];
                    bD[B] = l;
                    s_c[B] = 1;
                }
            }
            // charge switches Q(+q) for H and Q(-q) for A and B
            std::vector<double> Qh(n), Qab(n);
            for (int i = 0; i < n; ++i) {
                const double eh = std::exp(15.0 * qt[i]), em = std::exp(15.0 * -qt[i]);
                Qh[i] = eh / (eh + 1.0);
                Qab[i] = em / (em + 1.0);
            }
            auto csr = [&](const std::vector<std::vector<int>>& L, std::vector<int>& off, std::vector<int>& idx) {
                off.assign(n + 1, 0);
                for (int i = 0; i < n; ++i) off[i + 1] = off[i] + (int)L[i].size();
                idx.clear();
                for (int i = 0; i < n; ++i) idx.insert(idx.end(), L[i].begin(), L[i].end());
            };
            std::vector<int> nboff, nbidx, nbcoff, nbcidx;
            csr(bnb, nboff, nbidx);
            csr(bD, nbcoff, nbcidx);
            // case 1: role lists (counting sort by the role's atom, triplet order within a group)
            std::vector<int> c1;
            for (int h = 0; h < nh; ++h)
                if (P.hb_case[h] == 1) c1.push_back(h);
            std::vector<int2> ent((size_t)3 * c1.size());
            std::vector<int> goff(1, 0), gatom, crange((size_t)3 * (n + 1), 0);
            int ngr[3] = {0, 0, 0};
            size_t eo = 0;
            for (int role = 0; role < 3; ++role) {
                std::vector<int> cnt(n + 1, 0);
                for (int h : c1) cnt[P.hb_ahb[3 * h + role] + 1]++;
                for (int i = 0; i < n; ++i) cnt[i + 1] += cnt[i];
                std::vector<int> order(c1.size()), fill(cnt.begin(), cnt.end() - 1);
                for (int h : c1) order[fill[P.hb_ahb[3 * h + role]]++] = h;
                for (int i = 0; i < n; ++i) {
                    crange[(size_t)role * (n + 1) + i] = (int)gatom.size();
                    for (int k = cnt[i]; k < cnt[i + 1]; ++k) {
                        const int h = order[k];
                        const int A = P.hb_ahb[3 * h], H = P.hb_ahb[3 * h + 1], B = P.hb_ahb[3 * h + 2];
                        ent[eo++] = role == 0 ? make_int2(H, B) : (role == 1 ? make_int2(A, B) : make_int2(A, H));
                        if ((k - cnt[i]) % HB_CHUNK == HB_CHUNK - 1 || k + 1 == cnt[i + 1]) {
                            gatom.push_back(i);
                            goff.push_back((int)eo);
                        }
                    }
                }
                crange[(size_t)role * (n + 1) + n] = (int)gatom.size();
                ngr[role] = (int)gatom.size();
            }
            E->hb_ng0 = ngr[0];
            E->hb_ng1 = ngr[1];
            E->hb_ngt = ngr[2];
            // cases 2-4: compact list, slots triplet-major (A, H, B, neighbours
            // of B, carbonyl D atoms) and the per-atom CSR over them
            std::vector<int4> ahbc;
            std::vector<int> s0v, xatom, c2mol;
            for (int h = 0; h < nh; ++h) {
                const int cs = P.hb_case[h];
                if (cs == 1) continue;
                const int A = P.hb_ahb[3 * h], H = P.hb_ahb[3 * h + 1], B = P.hb_ahb[3 * h + 2];
                ahbc.push_back(make_int4(A, H, B, cs));
                s0v.push_back((int)xatom.size());
                xatom.push_back(A);
                xatom.push_back(H);
                xatom.push_back(B);
                for (int a2 : bnb[B]) xatom.push_back(a2);
                if (cs == 3)
                    for (int a2 : bD[B]) xatom.push_back(a2);
                c2mol.push_back(h);
                if (xatom.size() > (size_t)INT32_MAX / 4)
                    throw std::runtime_error("hydrogen-bond slot count exceeds the index range");
            }
            E->nhb2 = (int)ahbc.size();
            E->nhb2_c2 = 0;
            std::vector<int> ord;
            for (size_t h = 0; h < ahbc.size(); ++h)
                if (ahbc[h].w == 2) ord.push_back((int)h);
            E->nhb2_c2 = (int)ord.size();
            for (size_t h = 0; h < ahbc.size(); ++h)
                if (ahbc[h].w != 2) ord.push_back((int)h);
            E->hb_ord = E->upload(ord);
            std::vector<int> xoff(n + 1, 0), xidx(xatom.size());
            for (int at : xatom) xoff[at + 1]++;
            for (int i = 0; i < n; ++i) xoff[i + 1] += xoff[i];
            {
                std::vector<int> fill(xoff.begin(), xoff.end() - 1);
                for (size_t k = 0; k < xatom.size(); ++k) xidx[fill[xatom[k]]++] = (int)k;
            }
            E->hb_cb = E->upload(cb);
            E->hb_ca = E->upload(ca);
            E->hb_Qh = E->upload(Qh);
            E->hb_Qab = E->upload(Qab);
            {
                std::vector<float4> pk(n);
                std::vector<float> qh32(n);
                for (int i = 0; i < n; ++i) {
                    pk[i] = make_float4((float)cb[i], (float)ca[i], (float)Qab[i], (float)P.hb_rad[i]);
                    qh32[i] = (float)Qh[i];
                }
                E->hb_pk = E->upload(pk);
                E->hb_qh32 = E->upload(qh32);
            }
            E->hb_nboff = E->upload(nboff);
            E->hb_nbidx = E->upload(nbidx);
            E->hb_parc = E->upload(bC);
            E->hb_nbcoff = E->upload(nbcoff);
            E->hb_nbcidx = E->upload(nbcidx);
            E->hb_ent = E->upload(ent);
            E->hb_goff = E->upload(goff);
            E->hb_gatom = E->upload(gatom);
            E->hb_crange = E->upload(crange);
            E->hb_ahbc = E->upload(ahbc);
            E->hb_s0 = E->upload(s0v);
            E->hb_xoff = E->upload(xoff);
            E->hb_xidx = E->upload(xidx);
            // lanes per atom of the gather: 16 when the atoms' lists are short on average
            E->hbg_lpa = ((long long)crange[(size_t)2 * (n + 1) + n] + xoff[n] < 192LL * n) ? 16 : 64;
            if (opt.gather_lanes) E->hbg_lpa = opt.gather_lanes;
            E->hb_gout = E->alloc<double>(3 * (size_t)std::max(E->hb_ngt, 1));
            E->hb_xslots = E->alloc<double>(3 * std::max<size_t>(xatom.size(), 1));
            E->e_hb2 = E->alloc<double>(std::max(E->nhb2, 1));
            if (E->nmol > 1) {
                // per-molecule segments: row 4 the case-1 role-A chunks of the
                // molecule's atoms (chunks ascend in atom index), row 10 its
                // triplets of cases 2-4 (in triplet order, molecule-major)
                const int nm1 = E->nmol + 1;
                std::vector<int> ms(P.mol_seg.begin(), P.mol_seg.begin() + 10 * nm1);
                ms.resize(11 * nm1);
                for (int m = 0; m <= E->nmol; ++m) {
                    const int a0 = (m < E->nmol) ? P.mol_off[m] : n;
                    ms[4 * nm1 + m] = (int)(std::lower_bound(gatom.begin(), gatom.begin() + ngr[0], a0) - gatom.begin());
                    const int h0 = P.mol_seg[4 * nm1 + m];
                    ms[10 * nm1 + m] = (int)(std::lower_bound(c2mol.begin(), c2mol.end(), h0) - c2mol.begin());
                }
                E->mol_seg = E->upload(ms);
            }
        }
        E->natm = (int)P.atm_scale.size();
        std::vector<int> atslot(E->natm);
        for (int t = 0; t < E->natm; ++t) {
            atslot[t] = add_slot(P.atm_ijk[3 * t]);
            add_slot(P.atm_ijk[3 * t + 1]);
            add_slot(P.atm_ijk[3 * t + 2]);
        }
        E->atm_ijk = E->upload(P.atm_ijk);
        E->atm_sc = E->upload(P.atm_scale);
        E->atm_slot = E->upload(atslot);
        E->nbatm = (int)(P.batm_par.size() / 3);
        std::vector<int> btslot(E->nbatm);
        for (int t = 0; t < E->nbatm; ++t) {
            btslot[t] = add_slot(P.batm_ijk[3 * t]);
            add_slot(P.batm_ijk[3 * t + 1]);
            add_slot(P.batm_ijk[3 * t + 2]);
        }
        E->batm_ijk = E->upload(P.batm_ijk);
        E->batm_zb = E->upload(P.batm_par);
        E->batm_slot = E->upload(btslot);
        E->nslots = slot;
        // per-atom CSR over slots (ascending slot order)
        std::vector<int> soff(n + 1, 0), sidx(slot);
        for (int a : slot_atom) soff[a + 1]++;
        for (int i = 0; i < n; ++i) soff[i + 1] += soff[i];
        {
            std::vector<int> fill(soff.begin(), soff.end() - 1);
            for (int s = 0; s < slot; ++s) sidx[fill[slot_atom[s]]++] = s;
        }
        E->slot_off = E->upload(soff);
        E->fin_lpa = ((long long)soff[n] < 192LL * n) ? 16 : 64;  // lanes per atom of k_finish
        if (opt.gather_lanes) E->fin_lpa = opt.gather_lanes;
        // the gather of the slots (and a single molecule's hydrogen bonds): a
        // wavefront per atom also for short lists while that is at most four per
        // SIMD, where the lists' length and not their number sets the time
        // (evaluation with 16 lanes and with 64: 216 H2O 220.2 and 217.7 us, 512
        // 289.5 and 283.5; 64 and 1000 to 3000 H2O, alkanes of 122 to 1802 atoms and
        // batches of 828 to 20,777 the same within 0.4 %)
        E->slot_lpa = E->nmol == 1 && E->nhb ? std::max(E->fin_lpa, E->hbg_lpa) : E->fin_lpa;
        if (n <= 4096 && !opt.gather_lanes) E->slot_lpa = 64;
        E->slot_idx = E->upload(sidx);
        std::vector<int> doff(n + 1, 0), didx(2 * E->nbond);
        for (int b = 0; b < E->nbond; ++b) {
            doff[P.bond_ij[2 * b] + 1]++;
            doff[P.bond_ij[2 * b + 1] + 1]++;
        }
        for (int i = 0; i < n; ++i) doff[i + 1] += doff[i];
        {
            std::vector<int> fill(doff.begin(), doff.end() - 1);
            for (int b = 0; b < E->nbond; ++b) {
                didx[fill[P.bond_ij[2 * b]]++] = 2 * b;
                didx[fill[P.bond_ij[2 * b + 1]]++] = 2 * b + 1;
            }
        }
        E->dcn_off = E->upload(doff);
        E->dcn_idx = E->upload(didx);

        // work buffers
        E->x = E->alloc<double>(3 * (size_t)n);
        E->cn = E->alloc<double>(n);
        E->dlog = E->alloc<double>(n);
        E->gw = E->alloc<double>(7 * (size_t)n);
        E->dgw = E->alloc<double>(7 * (size_t)n);
        E->rhs = E->alloc<double>(n);
        E->diag = E->alloc<double>(n);
        if (E->use_cg) {
            // every workgroup of the persistent kernel must be resident at once
            const int nbk = E->np / NB;
            int dev = 0, ncu = 0, per_cu = 0;
            if (hipGetDevice(&dev) != hipSuccess ||
                hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
                hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_eeq_pcg<true, true>, PCGS_THREADS, 0) !=
                    hipSuccess) {
                status = kErrDevice;
                msg = "PCG occupancy query failed";
                delete E;
                return nullptr;
            }
            const long T = (long)nbk * (nbk + 1) / 2;
            // workgroups: enough wavefronts for one block each, so that the blocks
            // stay in registers, and two per owned 64-row block; more only add lines
            // to the all-reduce (512 H2O, 136 blocks: 16 groups 354 us per
            // evaluation, 32 312, 136 320; H-(Gly)200-OH, 253 blocks: 32 734, 64 726,
            // 253 782; 8 chains, 496 blocks: 32 1220, 64 925, 256 1045)
            E->cg_groups = (int)std::min<long>({(long)ncu * per_cu, 256L, T, std::max(2L * nbk, (T + PCG_WAVES - 1) / PCG_WAVES)});
            if (opt.pcg_groups > 0) E->cg_groups = std::min(E->cg_groups, opt.pcg_groups);
            if (E->cg_groups < 1 || cdiv(nbk, E->cg_groups) > PCG_MAXB) E->use_cg = false;
            if (E->use_cg) E->mat_size = (size_t)T * NB * NB;  // packed symmetric storage
        }
        E->Ared = E->alloc<double>(E->mat_size);
        E->Linv = E->alloc<double>((size_t)E->np * NB);
        E->b = E->alloc<double>(E->np);
        E->ybuf = E->alloc<double>(E->np);
        E->xbuf = E->alloc<double>(E->np);
        E->ready = E->alloc<int>(E->np / NB);
        if (E->nmol > 1) E->ured = E->alloc<double>(E->np);
        if (E->nmol == 1 && E->nr <= LU_MAX) {
            E->lu_w = E->alloc<double>((size_t)std::max(E->nr, 1) * (std::max(E->nr, 1) + 1));
            // the FP64 Cholesky factors R in place: keep a copy for the fallback
            if (!E->use_cg && !E->mixed) E->lu_src = E->alloc<double>(E->mat_size);
        }
        if (E->use_cg) {
            const int nbk0 = E->np / NB;
            E->cg_one = nbk0 <= NBK_ONE;
            E->cg_res = !E->cg_one && (long)nbk0 * (nbk0 + 1) / 2 <= (long)PCG_WAVES * E->cg_groups &&
                        E->cg_groups >= nbk0;
            const size_t pw = (size_t)nbk0 * E->np;
            if (E->cg_res) {
                // mailboxes and four buffers each of y, s_f parts and partials, cleared together
                const size_t words = MB_WORDS + 4 * ((size_t)E->np + 2 * nbk0 + pw);
                E->cg_mb = E->alloc<unsigned long long>(words);
                E->cg.nmb = (int)words;
                E->cg_z = (double*)(E->cg_mb + MB_WORDS);
                E->cg.sp = E->cg_z + 4 * (size_t)E->np;
                E->cg_part = E->cg.sp + 8 * (size_t)nbk0;
            } else if (!E->cg_one) {
                E->cg_z = E->alloc<double>(E->np);
                E->cg_p = E->alloc<double>(2 * (size_t)E->np);
                E->cg_part = E->alloc<double>(pw);
                E->cg_mb = E->alloc<unsigned long long>(MB_WORDS);
                E->cg.nmb = MB_WORDS;
            }
            E->cg_iters = E->alloc<int>(1);
            const int nbk = E->np / NB;
            // split fragments: more than 64 variables, so never inside one block
            std::vector<int> rowf(E->np, -1), poff(1, 0), pidx;
            int nsf = 0;
            for (int r0 = 0; r0 < E->nr;) {
                int r1 = r0 + 1;
                while (r1 < E->nr && red_last[r1] == red_last[r0]) ++r1;
                if (r1 - r0 > NB && long_frag) {
                    for (int r = r0; r < r1; ++r) {
                        const int bk = r / NB;
                        // second piece of its block when another split fragment, which then
                        // holds the block's first row, comes before it there
                        const int slot = rowf[bk * NB] >= 0 && (rowf[bk * NB] >> 1) != nsf ? 1 : 0;
                        rowf[r] = 2 * nsf + slot;
                        if (r == r0 || r % NB == 0) pidx.push_back(2 * bk + slot);
                    }
                    poff.push_back((int)pidx.size());
                    ++nsf;
                }
                r0 = r1;
            }
            PcgArgs& a = E->cg;
            a.np = E->np;
            a.nr = E->nr;
            a.lu_w = E->lu_w;
            a.maxit = PCG_MAXIT;
            a.tol2 = E->cg_tol2;
            a.Rp = E->Ared;
            a.Lj = E->Linv;
            a.b = E->b;
            a.x = E->xbuf;
            a.z = E->cg_z;
            a.pb = E->cg_p;
            a.part = E->cg_part;
            a.mb = E->cg_mb;
            a.iters = E->cg_iters;
            a.nsf = (nsf <= SM_MAXF && nbk <= SM_MAXB && !E->cg_one) ? nsf : 0;
            // long fragments converge by a factor of 4 in three or four iterations
            // and are worse conditioned: there the mixed path's default stops a
            // little later, so that its charges stay as close to the exact ones as
            // those of the plain block-Jacobi iteration (19,360 atoms: gradient off
            // by 1e-11 instead of 8e-11)
            if (a.nsf > 0 && E->mixed && default_tol) a.tol2 = E->cg_tol2 * 0.09;
            if (a.nsf > 0) {
                a.rowf = E->upload(rowf);
                a.poff = E->upload(poff);
                a.pidx = E->upload(pidx);
                a.w = E->cg_w = E->alloc<double>(E->np);
                a.w1 = E->cg_w1 = E->alloc<double>(2 * (size_t)nbk);
                a.all = E->cg_all = E->alloc<double>(nsf);
                a.smon = E->cg_smon = E->alloc<int>(nbk);
                if (!E->cg_res) a.sp = E->alloc<double>(2 * (size_t)nbk);
            }
        } else if (E->mixed && E->nmol > 1 && E->batch_fp32 && E->batch_solver != 2 && E->batch_solver < 4) {
            E->Ared32 = E->alloc<float>(E->mat_size);  // FP32 copies of the molecules' matrices and factors
            E->Linv32 = E->alloc<float>((size_t)E->np * NB);
        } else if (E->mixed && E->nmol == 1) {
            E->Ared32 = E->alloc<float>((size_t)E->np * E->np);
            E->Linv32 = E->alloc<float>((size_t)E->np * NB);
            E->b32 = E->alloc<float>(E->np);
            E->y32 = E->alloc<float>(E->np);
            E->d32 = E->alloc<float>(E->np);
            E->rvec = E->alloc<double>(E->np);
            E->symv = E->alloc<double>((size_t)SYMV_SPLIT * E->np);
        }
        E->rres = E->alloc<double>(n);
        E->q = E->alloc<double>(n);
        E->eself = E->alloc<double>(n);
        E->qtmp = E->alloc<double>(n);
        E->gpair = E->alloc<double>(3 * (size_t)n);
        E->dEdcn = E->alloc<double>(n);
        E->vchain = E->alloc<double>(n);
        E->slots = E->alloc<double>(3 * (size_t)std::max(slot, 1));
        E->dcn_slot = E->alloc<double>(2 * (size_t)std::max(E->nbond, 1));
        E->grad = E->alloc<double>(3 * (size_t)n);
        E->e_coul = E->alloc<double>(n);
        E->e_disp = E->alloc<double>(n);
        E->e_rep = E->alloc<double>(n);
        E->h6 = E->alloc<double>((size_t)n * E->nelem * 7);
        E->dh6 = E->alloc<double>((size_t)n * E->nelem * 7);
        {
            // j chunks: the grid (row blocks x chunks) should fill whole
            // rounds of the resident-workgroup capacity of the pair kernel in
            // use (at most two rounds, at least 128 partners per chunk; ties
            // to fewer chunks)
            const int rowblk = cdiv(n, TILE);
            const void* fn = nullptr;
            switch (E->mixed ? std::min(P.nelem, 5) : 10 + std::min(P.nelem, 5)) {
                case 1: fn = (const void*)k_pairs_part32<1>; break;
                case 2: fn = (const void*)k_pairs_part32<2>; break;
                case 3: fn = (const void*)k_pairs_part32<3>; break;
                case 4: fn = (const void*)k_pairs_part32<4>; break;
                case 5: fn = (const void*)k_pairs_part32<0>; break;
                case 11: fn = (const void*)k_pairs_part<1>; break;
                case 12: fn = (const void*)k_pairs_part<2>; break;
                case 13: fn = (const void*)k_pairs_part<3>; break;
                case 14: fn = (const void*)k_pairs_part<4>; break;
                default: fn = (const void*)k_pairs_part<0>; break;
            }
            int dev = 0, ncu = 0, per_cu = 0;
            if (hipGetDevice(&dev) != hipSuccess ||
                hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
                hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, TILE, 0) != hipSuccess || per_cu < 1)
                throw std::runtime_error("pair kernel occupancy query failed");
            const long cap = (long)ncu * per_cu;
            int best = 1;
            double best_eff = -1.0;
            for (int nck = 1; nck <= std::min(n, (int)(2 * cap)); ++nck) {
                const int cj = cdiv(n, nck), real = cdiv(n, cj);
                const long wg = (long)rowblk * real, rounds = (wg + cap - 1) / cap;
                if (rounds > 2 || cj < std::min(n, 128)) break;  // at least 128 partners per chunk
                const double eff = (double)wg / (double)(rounds * cap);
                if (eff > best_eff + 1e-9) {
                    best_eff = eff;
                    best = real;
                }
            }
            E->pair_cj = cdiv(n, best);
            E->pair_nchunk = cdiv(n, E->pair_cj);
            if (E->nmol > 1) {  // rows see only their molecule: one chunk
                E->pair_cj = n;
                E->pair_nchunk = 1;
            }
        }
        E->ppart = E->alloc<double>((size_t)E->pair_nchunk * PART_K * n);
        if (E->nmol == 1) {
            // each unordered pair once: 64 x 64 tiles of the lower triangle
            E->ps_nb = cdiv(n, PS_B);
            E->ps_ntiles = E->ps_nb * (E->ps_nb + 1) / 2;
            E->ps_nblocks = E->ps_nb;
            E->tbox = E->alloc<double>(6 * (size_t)cdiv(n, 256));
        } else if (opt.batch_pairs == 0) {
            // batches: the same tiles per molecule, listed {a0, n, R, C}, and the
            // molecules' 64-atom blocks {a0, n, A, first tile} for the reduction
            std::vector<int4> tl, bl;
            for (int m = 0; m < P.nmol; ++m) {
                const int a0 = P.mol_off[m], nm = P.mol_off[m + 1] - a0, nbm = cdiv(nm, PS_B);
                const int base = (int)tl.size();
                for (int R = 0; R < nbm; ++R)
                    for (int C = 0; C <= R; ++C) tl.push_back(make_int4(a0, nm, R, C));
                for (int A = 0; A < nbm; ++A) bl.push_back(make_int4(a0, nm, A, base));
            }
            E->ps_ntiles = (int)tl.size();
            E->ps_nblocks = (int)bl.size();
            E->ps_tiles = E->upload(tl);
            E->ps_blocks = E->upload(bl);
        }
        if (E->ps_ntiles > 0) {
            E->ps_split = ps_split(E->ps_ntiles);
            E->ps_part = E->alloc<double>((size_t)E->ps_ntiles * E->ps_split * 2 * PART_K * PS_B);
        }
        E->pair_split = opt.pair_split != 0 && E->ps_ntiles > 0;
        if (E->pair_split) E->ps_part2 = E->alloc<double>((size_t)E->ps_ntiles * E->ps_split * 2 * PART_K * PS_B);
        E->e_bond = E->alloc<double>(std::max(E->nbond, 1));
        E->e_ang = E->alloc<double>(std::max(E->nangle, 1));
        E->e_tor = E->alloc<double>(std::max(E->ntors, 1));
        E->e_inv = E->alloc<double>(std::max(E->ninv, 1));
        E->e_st = E->alloc<double>(std::max(E->nstors, 1));
        E->e_xb = E->alloc<double>(std::max(E->nxb, 1));
        E->e_brep = E->alloc<double>(std::max(E->nbrep, 1));
        E->e_hb = E->alloc<double>(std::max(E->hb_ng0, 1));
        E->e_atm = E->alloc<double>(std::max(E->natm, 1));
        E->e_batm = E->alloc<double>(std::max(E->nbatm, 1));
        if (P.solv.n > 0) {
            if (P.nmol != 1 || P.solv.n != n) {
                status = kErrUnsupported;
                msg = "ALPB solvation is built for single molecules";
                delete E;
                return nullptr;
            }
            const AlpbSet& A = P.solv;
            SolvArgs& a = E->sa;
            E->solv = true;
            a.n = n;
            a.keps = A.keps;
            a.alpbet = A.alpbet;
            a.c1 = A.born_scale;
            a.gshift = A.gshift;
            a.lr2 = A.lrcut * A.lrcut;
            a.sr2 = A.srcut * A.srcut;
            a.x = E->x;
            a.vdwr = E->upload(A.vdwr);
            a.rho = E->upload(A.rho);
            a.svdw = E->upload(A.svdw);
            a.vdwsa = E->upload(A.vdwsa);
            a.wrp = E->upload(A.wrp);
            a.trjlo = E->upload(A.trj_lo);
            a.trjhi = E->upload(A.trj_hi);
            a.gam = E->upload(A.gamsasa);
            a.hbmag = E->upload(A.hbmag);
            if (A.nang != SOLV_NANG) throw std::runtime_error("ALPB grid size");
            a.grid = E->upload(A.grid);
            a.brad = E->alloc<double>(n);
            a.dbr = E->alloc<double>(n);
            a.sasa = E->alloc<double>(n);
            a.hbw = E->alloc<double>(n);
            a.sv = E->alloc<double>((size_t)n * SOLV_NB * 3);
            a.sj = E->alloc<int>((size_t)n * SOLV_NB);
            a.sn = E->alloc<int>(n);
            a.shape = E->alloc<double>(32);
            a.w = E->alloc<double>(n);
            a.c = E->alloc<double>(n);
            a.eat = E->alloc<double>(n);
            a.gs = E->alloc<double>(3 * (size_t)n);
            a.e_solv = E->alloc<double>(1);
            a.parts = E->alloc<double>(4);
        }
        E->rpart = E->alloc<double>(16 * RED_BLOCKS);
        E->ghb = E->alloc<double>(3 * (size_t)n);
        E->gslot = E->alloc<double>(3 * (size_t)n);
        E->out = E->alloc<double>(GFNFF_NTERMS + 1);
        E->nbn = E->alloc<int>(n);
        E->nbl = E->alloc<int>((size_t)n * MAXNB_CN);
        E->flags = E->alloc<int>(1);
        E->sticky = E->alloc<int>(1);
        E->arrived = E->alloc<int>(1);
        E->sa.flags = E->flags;
        E->cg.flags = E->flags;
        {
            TermArgs& a = E->terms;
            const int cnt[12] = {cdiv(E->natm, 256),  cdiv(E->ntors, 256), cdiv(E->nb_hb, 4),   cdiv(E->ninv, 256),
                                 cdiv(E->nstors, 256), cdiv(E->nxb, 256),  cdiv(E->nangle, 256), cdiv(E->nbatm, 256),
                                 cdiv(E->nbrep, 256), cdiv(E->nb_plain, 256), cdiv(n * E->nelem, 256), cdiv(E->np, 256)};
            for (int k = 0, at = 0; k < 12; ++k) a.end[k] = at += cnt[k];
            a.n = n; a.ne = E->nelem; a.nr = E->nr; a.np = E->np;
            a.nb_hb = E->nb_hb; a.nb_plain = E->nb_plain; a.nangle = E->nangle; a.ntors = E->ntors;
            a.ninv = E->ninv; a.nstors = E->nstors; a.nxb = E->nxb; a.nbrep = E->nbrep; a.natm = E->natm;
            a.nbatm = E->nbatm;
            a.x = E->x; a.cn = E->cn; a.rcov_d3 = E->rcov_d3; a.hb_rad = E->hb_rad; a.gw = E->gw; a.dgw = E->dgw;
            a.qa = E->qa; a.c6ref = E->c6ref; a.elem = E->elem; a.nref = E->nref;
            a.bsel_hb = E->bsel_hb; a.bsel_plain = E->bsel_plain; a.bond_ij = E->bond_ij; a.bond_H = E->bond_H;
            a.bond_hboff = E->bond_hboff; a.bond_hbB = E->bond_hbB; a.bond_slot = E->bond_slot; a.bond_par = E->bond_par;
            a.ang_ijk = E->ang_ijk; a.ang_slot = E->ang_slot; a.ang_par = E->ang_par;
            a.tor_ijkl = E->tor_ijkl; a.tor_slot = E->tor_slot; a.tor_par = E->tor_par;
            a.inv_ijkl = E->inv_ijkl; a.inv_slot = E->inv_slot; a.inv_par = E->inv_par;
            a.st_ijkl = E->st_ijkl; a.st_slot = E->st_slot; a.st_par = E->st_par;
            a.xb_axb = E->xb_axb; a.xb_slot = E->xb_slot; a.xb_par = E->xb_par;
            a.brep_ij = E->brep_ij; a.brep_slot = E->brep_slot; a.brep_par = E->brep_par;
            a.atm_ijk = E->atm_ijk; a.atm_slot = E->atm_slot; a.atm_sc = E->atm_sc;
            a.batm_ijk = E->batm_ijk; a.batm_slot = E->batm_slot; a.batm_zb = E->batm_zb;
            a.slots = E->slots; a.dcn_slot = E->dcn_slot; a.e_bond = E->e_bond; a.e_ang = E->e_ang; a.e_tor = E->e_tor;
            a.e_inv = E->e_inv; a.e_st = E->e_st; a.e_xb = E->e_xb; a.e_brep = E->e_brep; a.e_atm = E->e_atm;
            a.e_batm = E->e_batm; a.h6 = E->h6; a.dh6 = E->dh6;
            a.red_atom = E->red_atom; a.red_last = E->red_last; a.b = E->b;
        }
        if (hipStreamCreate(&E->own) != hipSuccess || hipStreamCreate(&E->la.side) != hipSuccess ||
            hipEventCreateWithFlags(&E->la.fork, hipEventDisableTiming) != hipSuccess ||
            hipEventCreateWithFlags(&E->la.join, hipEventDisableTiming) != hipSuccess ||
            hipStreamCreateWithFlags(&E->side, hipStreamNonBlocking) != hipSuccess ||
            hipEventCreateWithFlags(&E->ev_fork, hipEventDisableTiming) != hipSuccess ||
            hipEventCreateWithFlags(&E->ev_join, hipEventDisableTiming) != hipSuccess ||
            hipEventCreateWithFlags(&E->ev_fact, hipEventDisableTiming) != hipSuccess)
            throw std::runtime_error("stream");
        if (E->batch_streams == 2 &&
            (hipStreamCreateWithFlags(&E->side2, hipStreamNonBlocking) != hipSuccess ||
             hipEventCreateWithFlags(&E->ev_h2f, hipEventDisableTiming) != hipSuccess ||
             hipEventCreateWithFlags(&E->ev_h2j, hipEventDisableTiming) != hipSuccess))
            throw std::runtime_error("stream");
        hipLaunchKernelGGL(k_fill_i, dim3(1), dim3(64), 0, E->own, 1, E->flags, 0);
        hipLaunchKernelGGL(k_fill_i, dim3(1), dim3(64), 0, E->own, 1, E->sticky, 0);
        hipLaunchKernelGGL(k_eeq_diag, dim3(cdiv(n, 256)), dim3(256), 0, E->own, n, E->gam, E->alp, E->diag);
        if (hipStreamSynchronize(E->own) != hipSuccess) throw std::runtime_error("init sync");
    } catch (const std::bad_alloc&) {
        status = kErrDevice;
        msg = "device allocation failed";
        delete E;
        return nullptr;
    } catch (const std::exception& ex) {
        status = kErrDevice;
        msg = ex.what();
        delete E;
        return nullptr;
    }
    status = kOk;
    return E;
}

void device_destroy(DeviceEngine* e) { delete e; }

// Queues the two-level blocked factorisation of the lower triangle of A
// (np x np, np a multiple of NB) on stream s; Linv receives the inverses of the
// diagonal blocks, flags FLAG_CHOL on a non-positive pivot.  tm (optional)
// times the kernel classes.
//
// Lookahead (la != nullptr): once super-panel K is factored, the columns of the
// next super-panel receive their rank-(SP NB) update first on s; the rest of
// the trailing matrix is updated on the side stream while s factors the next
// super-panel, which touches only its own columns.  The side stream is joined
// before the next trailing update and at the end.
template <typename T>
static void queue_cholesky(KernelTimer* tm, hipStream_t s, int np, T* A, T* Linv, int* flags,
                           const Lookahead* la = nullptr) {
    auto mark = [&](int c, hipStream_t st) {
        if (tm) tm->mark(c, st);
    };
    const int nbk = np / NB;
    bool pending = false;  // side-stream update not yet joined
    for (int K = 0; K < nbk; K += SP) {
        const int kend = std::min(K + SP, nbk);
        for (int k = K; k < kend; ++k) {
            const int k0 = k * NB;
            mark(KC_CHOL_DIAG, s);
            hipLaunchKernelGGL(k_chol_diag<T>, dim3(1), dim3(256), 0, s, np, k0, A, Linv, flags);
            mark(KC_CHOL_DIAG, s);
            const int rem = nbk - k - 1;
            if (rem == 0) continue;
            mark(KC_CHOL_PANEL, s);
            hipLaunchKernelGGL(k_chol_panel<T>, dim3(rem), dim3(256), 0, s, np, k0, A, Linv);
            mark(KC_CHOL_PANEL, s);
            const int w = kend - k - 1;
            if (w > 0) {
                const int ntiles = w * (w + 1) / 2 + (rem - w) * w;
                mark(KC_CHOL_UPDATE, s);
                hipLaunchKernelGGL(k_chol_update<T>, dim3(ntiles), dim3(256), 0, s, np, k0, NB, k + 1, w, nbk, A);
                mark(KC_CHOL_UPDATE, s);
            }
        }
        if (kend >= nbk) break;
        if (pending) {  // the previous side update wrote the tiles updated next
            (void)hipStreamWaitEvent(s, la->join, 0);
            pending = false;
        }
        const int M = nbk - kend;
        const int kend2 = std::min(kend + SP, nbk);
        if (!la || kend2 >= nbk) {
            mark(KC_CHOL_UPDATE, s);
            hipLaunchKernelGGL(k_chol_update<T>, dim3(M * (M + 1) / 2), dim3(256), 0, s, np, K * NB,
                               (kend - K) * NB, kend, M, nbk, A);
            mark(KC_CHOL_UPDATE, s);
            continue;
        }
        // rest of the trailing matrix (column blocks >= kend2) on the side stream
        const int M2 = nbk - kend2;
        (void)hipEventRecord(la->fork, s);
        (void)hipStreamWaitEvent(la->side, la->fork, 0);
        mark(KC_CHOL_UPDATE, la->side);
        hipLaunchKernelGGL(k_chol_update<T>, dim3(M2 * (M2 + 1) / 2), dim3(256), 0, la->side, np, K * NB,
                           (kend - K) * NB, kend2, M2, nbk, A);
        mark(KC_CHOL_UPDATE, la->side);
        (void)hipEventRecord(la->join, la->side);
        pending = true;
        // columns of the next super-panel (column blocks [kend, kend2), all rows) on s
        const int w = kend2 - kend;
        mark(KC_CHOL_UPDATE, s);
        hipLaunchKernelGGL(k_chol_update<T>, dim3(w * (w + 1) / 2 + (M - w) * w), dim3(256), 0, s, np, K * NB,
                           (kend - K) * NB, kend, w, nbk, A);
        mark(KC_CHOL_UPDATE, s);
    }
    if (pending) (void)hipStreamWaitEvent(s, la->join, 0);
}

// Forward and backward substitution with the blocked factor, one launch per
// sweep (k_trsv_*_sweep); the ready flags are cleared by a fill kernel, not a
// memset, so that the sequence can be captured in a graph.
template <typename T>
static void queue_solve(DeviceEngine* E, hipStream_t s, const T* A, const T* Linv, const T* b, T* y, T* x) {
    const int np = E->np, nbk = np / NB;
    LAUNCH(KC_TRSV, k_fill_i, dim3(cdiv(nbk, 256)), dim3(256), s, nbk, E->ready, 0);
    LAUNCH(KC_TRSV, k_trsv_fwd_sweep<T>, dim3(nbk), dim3(256), s, np, A, Linv, b, y, E->ready, E->flags);
    LAUNCH(KC_TRSV, k_fill_i, dim3(cdiv(nbk, 256)), dim3(256), s, nbk, E->ready, 0);
    LAUNCH(KC_TRSV, k_trsv_bwd_sweep<T>, dim3(nbk), dim3(256), s, np, A, Linv, y, x, E->ready, E->flags);
}

static void queue_diag(DeviceEngine* E, hipStream_t s, const int* mols, int nd, int k, double* A, double* Linv) {
    LAUNCH(KC_BATCH_SOLVE, k_bstep_diag64, dim3(nd), dim3(64), s, mols, k, E->mnp, E->mmo, E->mvo, A, Linv, E->flags);
}
static void queue_diag(DeviceEngine* E, hipStream_t s, const int* mols, int nd, int k, float* A, float* Linv) {
    LAUNCH(KC_BATCH_SOLVE, k_bstep_diag<float>, dim3(nd), dim3(256), s, mols, k, E->mnp, E->mmo, E->mvo, A, Linv,
           E->flags);
}

// batch_solver 3: the per-molecule factorisations advanced one column block at
// a time over the whole batch (three launches per step), then the
// substitutions (and, for FP32 factors, the FP64 refinement) in one launch.
template <typename T>
static void queue_batch_steps(DeviceEngine* E, hipStream_t s, T* A, T* Linv) {
    const int nsteps = (int)E->bs_doff.size() - 1;
    for (int k = 0; k < nsteps; ++k) {
        const int nd = E->bs_doff[k + 1] - E->bs_doff[k];
        const int npn = E->bs_poff[k + 1] - E->bs_poff[k];
        const int nu = E->bs_uoff[k + 1] - E->bs_uoff[k];
        queue_diag(E, s, E->bs_dmols + E->bs_doff[k], nd, k, A, Linv);
        if (npn)
            LAUNCH(KC_BATCH_SOLVE, (k_bstep_tiles<T, false>), dim3(cdiv(npn, 4)), dim3(256), s,
                   E->bs_ptiles + E->bs_poff[k], npn, k, E->mnp, E->mmo, E->mvo, A, Linv);
        if (nu)
            LAUNCH(KC_BATCH_SOLVE, (k_bstep_tiles<T, true>), dim3(cdiv(nu, 4)), dim3(256), s,
                   E->bs_utiles + E->bs_uoff[k], nu, k, E->mnp, E->mmo, E->mvo, A, Linv);
    }
}

// The batch factorisation (every variant but the whole-workgroup solve, which
// includes its substitutions) on stream s.
static void queue_batch_factor(DeviceEngine* E, hipStream_t s) {
    const dim3 g(E->nmol), b(BSOLVE_T);
    if (E->batch_solver == 4) {  // left-looking, matrix formed in place (FP64 on both paths)
        LAUNCH(KC_BATCH_SOLVE, k_eeq_batch_fused<3>, g, b, s, E->morder, E->mnr, E->mnp, E->mmo, E->mvo,
               E->red_atom, E->red_last, E->x, E->alp, E->diag, E->Ared, E->Linv, E->flags);
    } else if (E->batch_solver == 5 && E->batch_streams == 2) {  // two halves of the batch on two streams
        LAUNCH(KC_BATCH_SOLVE, k_red_u, dim3(cdiv(E->np, 256)), dim3(256), s, E->np, E->red_atom, E->red_last, E->x,
               E->alp, E->diag, E->ured);
        (void)hipEventRecord(E->ev_h2f, s);
        (void)hipStreamWaitEvent(E->side2, E->ev_h2f, 0);
        const int ncol = (int)E->h2_doff[0].size() - 1;
        for (int j = 0; j < ncol; ++j)
            for (int h = 0; h < 2; ++h) {
                hipStream_t st = h ? E->side2 : s;
                const int nt = E->h2_loff[h][j + 1] - E->h2_loff[h][j];
                const int nd = E->h2_doff[h][j + 1] - E->h2_doff[h][j];
                const int npn = E->h2_poff[h][j + 1] - E->h2_poff[h][j];
                if (nt)
                    LAUNCH(KC_BATCH_SOLVE, k_lstep_tiles, dim3(cdiv(nt, 4)), dim3(256), st,
                           E->h2_ltiles[h] + E->h2_loff[h][j], nt, j, E->mnr, E->mnp, E->mmo, E->mvo, E->red_atom,
                           E->red_last, E->x, E->alp, E->diag, E->ured, E->Ared);
                if (nd)
                    LAUNCH(KC_BATCH_SOLVE, k_bstep_diag64, dim3(nd), dim3(64), st,
                           E->h2_dmols[h] + E->h2_doff[h][j], j, E->mnp, E->mmo, E->mvo, E->Ared, E->Linv, E->flags);
                if (npn)
                    LAUNCH(KC_BATCH_SOLVE, (k_bstep_tiles<double, false>), dim3(cdiv(npn, 4)), dim3(256), st,
                           E->h2_ptiles[h] + E->h2_poff[h][j], npn, j, E->mnp, E->mmo, E->mvo, E->Ared, E->Linv);
            }
        (void)hipEventRecord(E->ev_h2j, E->side2);
        (void)hipStreamWaitEvent(s, E->ev_h2j, 0);
    } else if (E->batch_solver == 5) {  // left-looking by column blocks over the batch (FP64 on both paths)
        LAUNCH(KC_BATCH_SOLVE, k_red_u, dim3(cdiv(E->np, 256)), dim3(256), s, E->np, E->red_atom, E->red_last, E->x,
               E->alp, E->diag, E->ured);
        const int ncol = (int)E->ls_off.size() - 1;
        for (int j = 0; j < ncol; ++j) {
            const int nt = E->ls_off[j + 1] - E->ls_off[j];
            const int nd = E->bs_doff[j + 1] - E->bs_doff[j];
            const int npn = E->bs_poff[j + 1] - E->bs_poff[j];
            LAUNCH(KC_BATCH_SOLVE, k_lstep_tiles, dim3(cdiv(nt, 4)), dim3(256), s, E->ls_tiles + E->ls_off[j], nt, j,
                   E->mnr, E->mnp, E->mmo, E->mvo, E->red_atom, E->red_last, E->x, E->alp, E->diag, E->ured, E->Ared);
            LAUNCH(KC_BATCH_SOLVE, k_bstep_diag64, dim3(nd), dim3(64), s, E->bs_dmols + E->bs_doff[j], j,
                   E->mnp, E->mmo, E->mvo, E->Ared, E->Linv, E->flags);
            if (npn)
                LAUNCH(KC_BATCH_SOLVE, (k_bstep_tiles<double, false>), dim3(cdiv(npn, 4)), dim3(256), s,
                       E->bs_ptiles + E->bs_poff[j], npn, j, E->mnp, E->mmo, E->mvo, E->Ared, E->Linv);
        }
    } else if (E->batch_solver == 6) {  // as 5, the panel product inside the tiles below the diagonal
        LAUNCH(KC_BATCH_SOLVE, k_red_u, dim3(cdiv(E->np, 256)), dim3(256), s, E->np, E->red_atom, E->red_last, E->x,
               E->alp, E->diag, E->ured);
        const int ncol = (int)E->l6d_off.size() - 1;
        for (int j = 0; j < ncol; ++j) {
            const int ndt = E->l6d_off[j + 1] - E->l6d_off[j];
            const int not_ = E->l6o_off[j + 1] - E->l6o_off[j];
            const int nd = E->bs_doff[j + 1] - E->bs_doff[j];
            LAUNCH(KC_BATCH_SOLVE, k_lstep_tiles, dim3(cdiv(ndt, 4)), dim3(256), s, E->l6d_tiles + E->l6d_off[j], ndt,
                   j, E->mnr, E->mnp, E->mmo, E->mvo, E->red_atom, E->red_last, E->x, E->alp, E->diag, E->ured,
                   E->Ared);
            LAUNCH(KC_BATCH_SOLVE, k_bstep_diag64, dim3(nd), dim3(64), s, E->bs_dmols + E->bs_doff[j], j,
                   E->mnp, E->mmo, E->mvo, E->Ared, E->Linv, E->flags);
            if (not_)
                LAUNCH(KC_BATCH_SOLVE, k_lpanel_tiles, dim3(cdiv(not_, 4)), dim3(256), s,
                       E->l6o_tiles + E->l6o_off[j], not_, j, E->mnr, E->mnp, E->mmo, E->mvo, E->red_atom,
                       E->red_last, E->x, E->alp, E->diag, E->ured, E->Ared, E->Linv);
        }
    } else if (E->mixed && E->batch_fp32) {
        if (E->batch_solver == 3)
            queue_batch_steps<float>(E, s, E->Ared32, E->Linv32);
        else if (E->batch_solver == 1)  // two workgroups per CU, operands four steps ahead
            LAUNCH(KC_BATCH_SOLVE, (k_eeq_batch_factor<float, 2, 4>), g, b, s, E->morder, E->mnp, E->mmo, E->mvo,
                   E->Ared32, E->Linv32, E->flags);
        else  // three workgroups per CU, operands one step ahead
            LAUNCH(KC_BATCH_SOLVE, (k_eeq_batch_factor<float, 3, 1>), g, b, s, E->morder, E->mnp, E->mmo, E->mvo,
                   E->Ared32, E->Linv32, E->flags);
    } else {
        if (E->batch_solver == 3)
            queue_batch_steps<double>(E, s, E->Ared, E->Linv);
        else if (E->batch_solver == 1)
            LAUNCH(KC_BATCH_SOLVE, (k_eeq_batch_factor<double, 2, 4>), g, b, s, E->morder, E->mnp, E->mmo, E->mvo,
                   E->Ared, E->Linv, E->flags);
        else
            LAUNCH(KC_BATCH_SOLVE, (k_eeq_batch_factor<double, 3, 1>), g, b, s, E->morder, E->mnp, E->mmo, E->mvo,
                   E->Ared, E->Linv, E->flags);
    }
}

// k_pairs_sym over the engine's tiles for the selected pair terms
static void queue_pairs_sym(DeviceEngine* E, hipStream_t s, const PairArgs& pa, double* part, int terms) {
    const dim3 grid(E->ps_ntiles * E->ps_split);
    if (!E->mixed) {
        switch (E->nelem) {
            case 1: LAUNCH(KC_PAIRS, (k_pairs_sym<double, 1>), grid, dim3(PS_B), s, pa, part, E->ps_tiles, terms, E->ps_split); break;
            case 2: LAUNCH(KC_PAIRS, (k_pairs_sym<double, 2>), grid, dim3(PS_B), s, pa, part, E->ps_tiles, terms, E->ps_split); break;
            case 3: LAUNCH(KC_PAIRS, (k_pairs_sym<double, 3>), grid, dim3(PS_B), s, pa, part, E->ps_tiles, terms, E->ps_split); break;
            case 4: LAUNCH(KC_PAIRS, (k_pairs_sym<double, 4>), grid, dim3(PS_B), s, pa, part, E->ps_tiles, terms, E->ps_split); break;
            default: LAUNCH(KC_PAIRS, (k_pairs_sym<double, 0>), grid, dim3(PS_B), s, pa, part, E->ps_tiles, terms, E->ps_split); break;
        }
    } else {
        switch (E->nelem) {
            case 1: LAUNCH(KC_PAIRS, (k_pairs_sym<float, 1>), grid, dim3(PS_B), s, pa, part, E->ps_tiles, terms, E->ps_split); break;
            case 2: LAUNCH(KC_PAIRS, (k_pairs_sym<float, 2>), grid, dim3(PS_B), s, pa, part, E->ps_tiles, terms, E->ps_split); break;
            case 3: LAUNCH(KC_PAIRS, (k_pairs_sym<float, 3>), grid, dim3(PS_B), s, pa, part, E->ps_tiles, terms, E->ps_split); break;
            case 4: LAUNCH(KC_PAIRS, (k_pairs_sym<float, 4>), grid, dim3(PS_B), s, pa, part, E->ps_tiles, terms, E->ps_split); break;
            default: LAUNCH(KC_PAIRS, (k_pairs_sym<float, 0>), grid, dim3(PS_B), s, pa, part, E->ps_tiles, terms, E->ps_split); break;
        }
    }
}

// One evaluation of the coordinates xin (device-accessible) on stream s; the
// energy terms and the gradient also go to energy_out and grad_out (nullable).
static int launch_eval(DeviceEngine* E, const double* xin, double* energy_out, double* grad_out, hipStream_t s,
                       std::string& msg) {
    const int n = E->n;
    hipLaunchKernelGGL(k_start, dim3(cdiv(3 * n, 256)), dim3(256), 0, s, n, xin, E->x, E->flags, E->arrived,
                       E->mol_of ? (double*)nullptr : E->tbox);
    // The reduced EEQ matrix needs only the coordinates: it is built on the
    // side stream while this stream computes CN, the EEQ right-hand side and
    // every term that does not depend on the EEQ charges; the solve waits
    // for both (and runs alone, as the persistent solver requires).
    // Born radii, surface areas and shape: geometry only, and the matrix needs
    // the radii and the hydrogen-bond weights of the surfaces, so on the side
    // stream; a charged molecule's right-hand side needs the radii on this one
    if (E->solv && E->charged) LAUNCH(KC_SOLV, k_solv_geom, dim3(n + 1 + cdiv(n, 4)), dim3(256), s, E->sa);
    HIP_OK(hipEventRecord(E->ev_fork, s));
    HIP_OK(hipStreamWaitEvent(E->side, E->ev_fork, 0));
    // EEQ
    const int np = E->np, nbk = np / NB;
    if (E->nmol == 1) {
        if (E->solv && !E->charged) LAUNCH(KC_SOLV, k_solv_geom, dim3(n + 1 + cdiv(n, 4)), dim3(256), E->side, E->sa);
        LAUNCH(KC_EEQ_BUILD, k_eeq_reduced, dim3(nbk * (nbk + 1) / 2), dim3(RED_T), E->side, E->nr, np,
               E->red_atom, E->red_last, E->red_lidx, E->red_ul, E->red_nul, E->x, E->alp, E->diag, E->Ared,
               E->use_cg ? 2 : 0);
        if (E->solv)
            LAUNCH(KC_SOLV, k_solv_red_add, dim3(nbk * (nbk + 1) / 2, 8), dim3(256), E->side, E->nr, np, E->red_atom,
                   E->red_last, E->sa, E->Ared, E->use_cg ? 2 : 0);
        if (E->use_cg) {
            // block-Jacobi factors of R's diagonal blocks and the solver's
            // mailboxes, also off the evaluation stream
            LAUNCH(KC_CHOL_DIAG, k_bjacobi_setup, dim3(nbk), dim3(256), E->side, E->Ared, E->Linv, E->flags,
                   E->cg.nsf, E->cg, E->red_atom, E->red_last, E->x, E->alp, E->diag, E->solv ? 1 : 0, E->sa, E->cg_w,
                   E->cg_w1, E->cg_all, E->cg_smon);
        }
    }
    else if (E->batch_solver < 4)  // batch_solver 4 and 5 form the matrix inside their factorisations
        LAUNCH(KC_EEQ_BUILD, k_eeq_reduced_batch, dim3(E->nbtiles), dim3(256), E->side, E->btiles, E->mnr, E->mnp,
               E->mmo, E->mvo, E->red_atom, E->red_last, E->x, E->alp, E->diag, E->Ared,
               E->Ared32);  // the FP32 copy exists only when the mixed path factors in FP32
    const bool split = E->nmol > 1 && E->batch_solver != 2;
    if (split) {
        queue_batch_factor(E, E->side);
        HIP_OK(hipEventRecord(E->ev_fact, E->side));
    }
    if (E->cn_by_mol)
        LAUNCH_SHM(KC_CN, k_cn_mol, dim3(E->nmol), dim3(256), (size_t)E->cn_cap * CNMOL_LDS_BYTES, s, E->cn_cap,
                   E->mol_off, E->x, E->rcov_cn, E->elem, E->nref,
               E->refcn, E->chi_base, E->cnf, E->cn, E->dlog, E->gw, E->dgw, E->rhs, E->nbn, E->nbl, E->flags);
    else
        LAUNCH(KC_CN, k_cn, dim3(cdiv(n, 4)), dim3(256), s, n, E->x, E->rcov_cn, E->elem, E->nref, E->refcn,
               E->chi_base, E->cnf, E->cn, E->dlog, E->gw, E->dgw, E->rhs, E->nbn, E->nbl, E->flags, E->mol_of,
               E->mol_off, E->tbox);
    const double* rsrc = E->rhs;
    if (E->charged) {
        LAUNCH(KC_EEQ_BUILD, k_eeq_rhs_qp, dim3(cdiv(n, 256)), dim3(256), s, n, E->x, E->alp, E->diag, E->qp,
                           E->rhs, E->rres, E->mol_of, E->mol_off);
        if (E->solv) LAUNCH(KC_SOLV, k_solv_rhs, dim3(cdiv(n, 256)), dim3(256), s, E->sa, E->qp, E->rres);
        rsrc = E->rres;
    }
    const PairArgs pa = E->pair_args();
    {
        TermArgs ta = E->terms;
        ta.rhs = rsrc;
        // a launch per list also where one of these classes is timed
        const int tc = E->timer.cls;
        const bool timed = tc == KC_EEQ_BUILD || tc == KC_PAIRS_AUX || tc == KC_BONDS || tc == KC_ANGLES ||
                           tc == KC_TORS || tc == KC_HB || tc == KC_BREP || tc == KC_ATM || tc == KC_BATM;
        if (ta.end[11] <= TERMS_FUSED_MAX && !timed) {
            LAUNCH(KC_BONDS, k_terms<-1>, dim3(ta.end[11]), dim3(256), s, ta);
        } else {
            auto wgs = [&](int k) { return dim3(ta.end[k] - (k ? ta.end[k - 1] : 0)); };
            LAUNCH(KC_EEQ_BUILD, k_terms<11>, wgs(11), dim3(256), s, ta);
            LAUNCH(KC_PAIRS_AUX, k_terms<10>, wgs(10), dim3(256), s, ta);
            if (ta.nb_hb) LAUNCH(KC_BONDS, k_terms<2>, wgs(2), dim3(256), s, ta);
            if (ta.nb_plain) LAUNCH(KC_BONDS, k_terms<9>, wgs(9), dim3(256), s, ta);
            if (ta.nangle) LAUNCH(KC_ANGLES, k_terms<6>, wgs(6), dim3(256), s, ta);
            if (ta.ntors) LAUNCH(KC_TORS, k_terms<1>, wgs(1), dim3(256), s, ta);
            if (ta.ninv) LAUNCH(KC_TORS, k_terms<3>, wgs(3), dim3(256), s, ta);
            if (ta.nstors) LAUNCH(KC_TORS, k_terms<4>, wgs(4), dim3(256), s, ta);
            if (ta.nxb) LAUNCH(KC_HB, k_terms<5>, wgs(5), dim3(256), s, ta);
            if (ta.nbrep) LAUNCH(KC_BREP, k_terms<8>, wgs(8), dim3(256), s, ta);
            if (ta.natm) LAUNCH(KC_ATM, k_terms<0>, wgs(0), dim3(256), s, ta);
            if (ta.nbatm) LAUNCH(KC_BATM, k_terms<7>, wgs(7), dim3(256), s, ta);
        }
    }
    // a single molecule's hydrogen bonds are gathered with the slots (below)
    const HBGather hg{E->nhb ? E->hb_crange : nullptr, E->hb_gout, E->hb_xoff, E->hb_xidx, E->hb_xslots};
    auto slot_gather = [&](const HBGather& h, int lpa) {
        if (lpa == 64)
            LAUNCH(KC_CHAIN, k_slot_gather<64>, dim3(cdiv(n, 4)), dim3(256), s, n, E->slot_off, E->slot_idx, E->slots,
                   h, E->gslot);
        else
            LAUNCH(KC_CHAIN, k_slot_gather<16>, dim3(cdiv(n, 16)), dim3(256), s, n, E->slot_off, E->slot_idx, E->slots,
                   h, E->gslot);
    };
    if (E->nmol > 1) slot_gather(HBGather{}, E->slot_lpa);
    // pair_split: the charge-independent pair terms (dispersion, repulsion)
    // last before the solve, beside the factorisation's smaller column blocks
    if (E->pair_split) queue_pairs_sym(E, s, pa, E->ps_part2, PT_DISP | PT_REP);
    // Hydrogen bonds (all kernels and their gather) need only the coordinates
    // and set-up data: a single molecule evaluates them on this stream while
    // the side stream builds the EEQ matrix; a batch appends them to the side
    // stream behind its matrix build and factorisation (run beside the
    // factorisation, they slowed it, and it is the longer chain), and they
    // join this stream before k_finish.
    hipStream_t hs = (E->nmol > 1) ? E->side : s;
    if (E->nhb) {
        HBArgs ha{E->hb_cb, E->hb_ca, E->hb_Qh, E->hb_Qab, E->hb_nboff, E->hb_nbidx, E->hb_parc,
                  E->hb_nbcoff, E->hb_nbcidx, E->hb_rad, E->hb_lpd, E->Z, E->hb_pk, E->hb_qh32};
        HBRoles hr{E->hb_ent, E->hb_goff, E->hb_gatom, E->hb_ng0, E->hb_ng1, E->hb_ngt};
        // case-1 roles (FP32 terms on the mixed path, FP64 otherwise)
        const int nrole = cdiv(E->hb_ng0, 4) + cdiv(E->hb_ng1 - E->hb_ng0, 4) + cdiv(E->hb_ngt - E->hb_ng1, 4);
        if (nrole) {
            if (E->mixed)
                LAUNCH(KC_HB, k_hb_roles<float>, dim3(nrole), dim3(256), hs, hr, ha, E->x, E->hb_gout, E->e_hb);
            else
                LAUNCH(KC_HB, k_hb_roles<double>, dim3(nrole), dim3(256), hs, hr, ha, E->x, E->hb_gout, E->e_hb);
        }
        // cases 2-4: the case-2 entries by the lean core (FP32 terms on the
        // mixed path), those of cases 3 and 4 by the general FP64 one; a short
        // FP64 list that holds both by the general core in one launch, which
        // saves a launch of the chain (peptides of 38 atoms, 40 entries: 96 us
        // against 99.7 with two; 143 atoms 208.7 against 211.0; 283 to 1403 atoms
        // and batches of 56 to 57,000 entries the same within 0.3 %)
        const int n34 = E->nhb2 - E->nhb2_c2;
        constexpr int HB_ONE_MAX = 16384;
        const bool one = !E->mixed && n34 > 0 && E->nhb2 <= HB_ONE_MAX;
        if (one)
            LAUNCH(KC_HB, (k_hb_full<double, 0>), dim3(cdiv(E->nhb2, 256)), dim3(256), hs, E->nhb2, E->hb_ord,
                   E->hb_ahbc, E->hb_s0, ha, E->x, E->hb_xslots, E->e_hb2);
        if (!one && E->nhb2_c2 && !E->mixed)
            LAUNCH(KC_HB, (k_hb_full<double, 1>), dim3(cdiv(E->nhb2_c2, 256)), dim3(256), hs, E->nhb2_c2, E->hb_ord,
                   E->hb_ahbc, E->hb_s0, ha, E->x, E->hb_xslots, E->e_hb2);
        if (E->mixed && E->nhb2_c2)
            LAUNCH(KC_HB, (k_hb_full<float, 1>), dim3(cdiv(E->nhb2_c2, 256)), dim3(256), hs, E->nhb2_c2, E->hb_ord,
                   E->hb_ahbc, E->hb_s0, ha, E->x, E->hb_xslots, E->e_hb2);
        if (!one && n34 > 0)
            LAUNCH(KC_HB, (k_hb_full<double, 2>), dim3(cdiv(n34, 256)), dim3(256), hs, n34, E->hb_ord + E->nhb2_c2,
                   E->hb_ahbc, E->hb_s0, ha, E->x, E->hb_xslots, E->e_hb2);
    }
    if (E->nmol == 1)
        slot_gather(hg, E->slot_lpa);
    else if (E->nhb) {
        if (E->hbg_lpa == 64)
            LAUNCH(KC_HB, k_hb_gather<64>, dim3(cdiv(n, 4)), dim3(256), hs, n, hg, E->ghb);
        else
            LAUNCH(KC_HB, k_hb_gather<16>, dim3(cdiv(n, 16)), dim3(256), hs, n, hg, E->ghb);
    }
    const double* ghb = (E->nmol > 1 && E->nhb) ? E->ghb : nullptr;
    HIP_OK(hipEventRecord(E->ev_join, E->side));
    // batches wait here for the factorisation only; the hydrogen-bond work
    // queued behind it on the side stream joins before k_finish
    HIP_OK(hipStreamWaitEvent(s, split ? E->ev_fact : E->ev_join, 0));
    if (E->nmol > 1) {
        // batch: every molecule's system factored (side stream, above) and
        // solved by one workgroup per molecule
        if (E->batch_solver == 2)
            LAUNCH(KC_BATCH_SOLVE, k_eeq_batch_solve_tiles, dim3(E->nmol), dim3(256), s, E->morder, E->mnp, E->mmo,
                   E->mvo, E->Ared, E->Linv, E->b, E->xbuf, E->flags);
        else if (E->mixed && E->batch_fp32 && E->batch_solver < 4)
            LAUNCH(KC_BATCH_SOLVE, k_bsolve_subst<float>, dim3(E->nmol), dim3(BSOLVE_T), s, E->morder, E->mnp,
                   E->mmo, E->mvo, E->Ared32, E->Linv32, E->Ared, E->b, E->xbuf);
        else
            LAUNCH(KC_BATCH_SOLVE, k_bsolve_subst<double>, dim3(E->nmol), dim3(BSOLVE_T), s, E->morder, E->mnp,
                   E->mmo, E->mvo, E->Ared, E->Linv, (const double*)nullptr, E->b, E->xbuf);
    } else if (E->use_cg) {
        // the persistent PCG (block-Jacobi factors and mailboxes were set up on the side stream)
        const dim3 grid(E->cg_groups), block(PCG_THREADS);
        if (E->cg_one) {
            switch (nbk) {
                case 1: LAUNCH(KC_PCG, k_eeq_pcg_one<1>, dim3(1), block, s, E->cg); break;
                case 2: LAUNCH(KC_PCG, k_eeq_pcg_one<2>, dim3(1), block, s, E->cg); break;
                default: LAUNCH(KC_PCG, k_eeq_pcg_one<3>, dim3(1), block, s, E->cg); break;
            }
        } else if (E->cg_res && E->cg.nsf)
            LAUNCH(KC_PCG, k_eeq_pcg_res<true>, grid, block, s, E->cg);
        else if (E->cg_res)
            LAUNCH(KC_PCG, k_eeq_pcg_res<false>, grid, block, s, E->cg);
        else {
            const dim3 sb(PCGS_THREADS);
            const bool pp = (long)nbk * (nbk + 1) / 2 >= (long)PCGS_PP * PCGS_WAVES * E->cg_groups;
            if (E->cg.nsf && pp)
                LAUNCH(KC_PCG, (k_eeq_pcg<true, true>), grid, sb, s, E->cg);
            else if (E->cg.nsf)
                LAUNCH(KC_PCG, (k_eeq_pcg<true, false>), grid, sb, s, E->cg);
            else if (pp)
                LAUNCH(KC_PCG, (k_eeq_pcg<false, true>), grid, sb, s, E->cg);
            else
                LAUNCH(KC_PCG, (k_eeq_pcg<false, false>), grid, sb, s, E->cg);
        }
    } else if (!E->mixed) {
        if (E->lu_src)
            LAUNCH(KC_CHOL_DIAG, k_copy, dim3(cdiv((long)E->mat_size, 256)), dim3(256), s, (int)E->mat_size, E->Ared,
                   E->lu_src);
        queue_cholesky(&E->timer, s, np, E->Ared, E->Linv, E->flags, E->use_lookahead ? &E->la : nullptr);
        queue_solve<double>(E, s, E->Ared, E->Linv, E->b, E->ybuf, E->xbuf);
    } else {
        LAUNCH(KC_EEQ_BUILD, k_lower_to_f32, dim3(nbk * (nbk + 1) / 2), dim3(256), s, np, E->Ared, E->Ared32);
        queue_cholesky(&E->timer, s, np, E->Ared32, E->Linv32, E->flags, E->use_lookahead ? &E->la : nullptr);
        LAUNCH(KC_REFINE, k_to_f32, dim3(cdiv(np, 256)), dim3(256), s, np, E->b, E->b32);
        for (int it = 0; it < REFINE_STEPS; ++it) {
            queue_solve<float>(E, s, E->Ared32, E->Linv32, E->b32, E->y32, E->d32);
            LAUNCH(KC_REFINE, k_refine_add, dim3(cdiv(np, 256)), dim3(256), s, np, it == 0 ? 1 : 0, E->d32,
                   E->xbuf);
            if (it + 1 < REFINE_STEPS) {
                LAUNCH(KC_REFINE, k_symv_part, dim3(nbk, SYMV_SPLIT), dim3(256), s, np, SYMV_SPLIT, E->Ared,
                       E->xbuf, E->symv);
                LAUNCH(KC_REFINE, k_eeq_resid, dim3(cdiv(np, 256)), dim3(256), s, np, SYMV_SPLIT, E->symv, E->b,
                       E->rvec, E->b32);
            }
        }
    }
    if (E->lu_w && !E->use_cg)  // no work unless the system was found not positive definite
        LAUNCH(KC_CHARGES, k_eeq_lu_fallback, dim3(1), dim3(LU_T), s, np, E->nr,
               E->lu_src ? E->lu_src : E->Ared, E->b, E->lu_w, E->xbuf, E->flags);
    {
        const int natb = cdiv(n, 256);
        const ChargeArgs ca{n,     E->nfrag,  natb,        E->frag_off, E->frag_atoms, E->red_of, E->qp, E->xbuf,
                            E->chi_base, E->cnf, E->gam, E->alp, E->cn, E->q, E->eself, E->qtmp};
        LAUNCH(KC_CHARGES, k_charges, dim3(natb + cdiv(E->nfrag, 4)), dim3(256), s, ca);
    }
    if (E->solv) {
        // the solvation terms need the charges and what the side stream holds:
        // there, beside the pair terms, joined before k_finish
        HIP_OK(hipEventRecord(E->ev_fork, s));
        HIP_OK(hipStreamWaitEvent(E->side, E->ev_fork, 0));
        LAUNCH(KC_SOLV, k_solv_pairs, dim3(cdiv(n, 4)), dim3(256), E->side, E->sa, E->q);
        LAUNCH(KC_SOLV, k_solv_energy, dim3(1), dim3(256), E->side, E->sa, E->q);
        LAUNCH(KC_SOLV, k_solv_grad, dim3(cdiv(n, 4)), dim3(256), E->side, E->sa);
        HIP_OK(hipEventRecord(E->ev_join, E->side));
    }
    // pair terms
    const AtomTailArgs tail{E->x,    E->Z,       E->metal,   E->anb,      E->repz,  E->toff,
                            E->tidx, E->tdist,   E->gpair,   E->e_rep,    E->dcn_off, E->dcn_idx,
                            E->dcn_slot, E->dEdcn, E->qtmp, E->vchain};
    if (E->ps_ntiles > 0) {  // each unordered pair once (single molecules; batches unless batch_pairs = 1)
        queue_pairs_sym(E, s, pa, E->ps_part, E->pair_split ? PT_COUL : PT_ALL);
        const double* part2 = E->pair_split ? E->ps_part2 : nullptr;
        if (E->ps_split > 1)
            LAUNCH(KC_PAIRS_AUX, k_pairs_sym_reduce<16>, dim3(E->ps_nblocks), dim3(1024), s, n, E->ps_nb, E->ps_part,
                   part2, E->e_coul, E->e_disp, E->ps_blocks, E->ps_split, tail);
        else
            LAUNCH(KC_PAIRS_AUX, k_pairs_sym_reduce<4>, dim3(E->ps_nblocks), dim3(256), s, n, E->ps_nb, E->ps_part,
                   part2, E->e_coul, E->e_disp, E->ps_blocks, E->ps_split, tail);
    } else {
        const dim3 grid(cdiv(n, TILE), E->pair_nchunk);
        if (!E->mixed) {
            switch (E->nelem) {
                case 1: LAUNCH(KC_PAIRS, k_pairs_part<1>, grid, dim3(TILE), s, pa, E->pair_cj, E->ppart); break;
                case 2: LAUNCH(KC_PAIRS, k_pairs_part<2>, grid, dim3(TILE), s, pa, E->pair_cj, E->ppart); break;
                case 3: LAUNCH(KC_PAIRS, k_pairs_part<3>, grid, dim3(TILE), s, pa, E->pair_cj, E->ppart); break;
                case 4: LAUNCH(KC_PAIRS, k_pairs_part<4>, grid, dim3(TILE), s, pa, E->pair_cj, E->ppart); break;
                default: LAUNCH(KC_PAIRS, k_pairs_part<0>, grid, dim3(TILE), s, pa, E->pair_cj, E->ppart); break;
            }
        } else {
            switch (E->nelem) {
                case 1: LAUNCH(KC_PAIRS, k_pairs_part32<1>, grid, dim3(TILE), s, pa, E->pair_cj, E->ppart); break;
                case 2: LAUNCH(KC_PAIRS, k_pairs_part32<2>, grid, dim3(TILE), s, pa, E->pair_cj, E->ppart); break;
                case 3: LAUNCH(KC_PAIRS, k_pairs_part32<3>, grid, dim3(TILE), s, pa, E->pair_cj, E->ppart); break;
                case 4: LAUNCH(KC_PAIRS, k_pairs_part32<4>, grid, dim3(TILE), s, pa, E->pair_cj, E->ppart); break;
                default: LAUNCH(KC_PAIRS, k_pairs_part32<0>, grid, dim3(TILE), s, pa, E->pair_cj, E->ppart); break;
            }
        }
        LAUNCH(KC_PAIRS_AUX, k_pairs_reduce, dim3(cdiv(n, 256)), dim3(256), s, n, E->pair_nchunk, E->ppart, E->gpair,
               E->dEdcn, E->e_coul, E->e_disp, E->e_rep);
        LAUNCH(KC_CHAIN, k_atom_tail, dim3(cdiv(n, 256)), dim3(256), s, n, tail);
    }
    if (split || E->solv) HIP_OK(hipStreamWaitEvent(s, E->ev_join, 0));
    FinishArgs fa{};
    fa.n = n;
    fa.x = E->x;
    fa.rcov = E->rcov_cn;
    fa.dlog = E->dlog;
    fa.v = E->vchain;
    fa.nbn = E->nbn;
    fa.nbl = E->nbl;
    fa.gslot = E->gslot;
    fa.gpair = E->gpair;
    fa.ghb = ghb;
    fa.gsolv = E->solv ? E->sa.gs : nullptr;
    fa.grad = E->grad;
    fa.grad2 = grad_out;
    const double* ptrs[NPARTS] = {E->e_bond, E->e_ang,  E->e_tor, E->e_inv, E->e_disp, E->e_brep,
                                  E->e_rep,  E->e_coul, E->eself, E->e_hb,  E->e_atm,  E->e_batm,
                                  E->e_st,   E->e_xb,   E->e_hb2, E->solv ? E->sa.e_solv : E->e_bond};
    const int cnts[NPARTS] = {E->nbond, E->nangle, E->ntors, E->ninv, n, E->nbrep, n, n, n, E->hb_ng0, E->natm,
                              E->nbatm, E->nstors, E->nxb, E->nhb2, E->solv ? 1 : 0};
    int most = 0;
    for (int k = 0; k < NPARTS; ++k) {
        fa.seg[k] = ptrs[k];
        fa.cnt[k] = cnts[k];
        most = std::max(most, cnts[k]);
    }
    fa.nred = std::min(RED_BLOCKS, std::max(1, cdiv(most, 1024)));
    fa.part = E->rpart;
    fa.out = E->out;
    fa.out2 = energy_out;
    fa.flags = E->flags;
    fa.sticky = E->sticky;
    fa.arrived = E->arrived;
    if (E->nmol > 1) {
        MolEnergyArgs& ma = fa.mol;
        ma.nmol = E->nmol;
        ma.mol_off = E->mol_off;
        ma.seg = E->mol_seg;
        ma.atom_terms[0] = E->e_coul;
        ma.atom_terms[1] = E->e_disp;
        ma.atom_terms[2] = E->e_rep;
        ma.atom_terms[3] = E->eself;
        const double* lists[11] = {E->e_bond, E->e_ang,  E->e_tor, E->e_brep, E->e_hb, E->e_atm,
                                   E->e_batm, E->e_inv, E->e_st,  E->e_xb,   E->e_hb2};
        for (int k = 0; k < 11; ++k) ma.list_terms[k] = lists[k];
        ma.e_mol = E->e_mol;
        fa.nmolb = cdiv(E->nmol, 4);
    }
    const int head = NPARTS * fa.nred + fa.nmolb;
    int left = head + cdiv(n, E->fin_lpa == 64 ? 4 : 16);
    if (E->timer.cls == KC_REDUCE || E->timer.cls == KC_CHAIN) {  // the energies in a launch of their own
        LAUNCH(KC_REDUCE, k_finish<64>, dim3(head), dim3(256), s, fa);
        fa.first = head;
        left -= head;
    }
    if (E->fin_lpa == 64)
        LAUNCH(KC_CHAIN, k_finish<64>, dim3(left), dim3(256), s, fa);
    else
        LAUNCH(KC_CHAIN, k_finish<16>, dim3(left), dim3(256), s, fa);
    if (hipGetLastError() != hipSuccess) {
        msg = "kernel launch failed";
        return kErrDevice;
    }
    return kOk;
}

// Host-buffer evaluations of up to HOST_PINNED_MAX atoms go through pinned
// memory that the device reads and writes itself: the head of the evaluation
// reads the coordinates there and one launch at its end writes every result,
// side by side, so that a call is one queue of launches and one wait.  By
// pageable copies it was five transfers with a wait in the runtime each.  By
// copies and by pinned memory: 38 atoms 209 and 135 us, 648 345 and 256, 3,000
// 589 and 430, batches of 3,415 877 and 751 us, 53,797 1.44 and 1.38 ms, 124,193
// 2.22 and 2.19, 204,392 3.15 and 3.07, 409,164 5.70 and 5.73, 819,770 11.2 and
// 11.5 ms.  Larger systems keep the copies, whose bandwidth counts there and
// whose staging belongs to the runtime.
constexpr int HOST_PINNED_MAX = 131072;
// results of one evaluation: [0, 16) energies, [16] flags, then charges, CN
// and, unless grad is nullptr, the gradient
__global__ __launch_bounds__(256) void k_host_out(int n, const double* __restrict__ out, const int* __restrict__ flags,
                                                  const double* __restrict__ grad, const double* __restrict__ q,
                                                  const double* __restrict__ cn, double* __restrict__ dst) {
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e < GFNFF_NTERMS + 1) dst[e] = out[e];
    if (e == GFNFF_NTERMS + 1) dst[e] = (double)flags[0];
    double* const r = dst + GFNFF_NTERMS + 2;
    if (e < n)
        r[e] = q[e];
    else if (e < 2 * n)
        r[e] = cn[e - n];
    else if (grad && e < 5 * n)
        r[e] = grad[e - 2 * n];
}

int device_eval_host(DeviceEngine* E, const double* xyz_bohr, bool want_grad, double* e_terms, double* grad,
                     double* q, double* cn, std::string& msg) {
    const int n = E->n;
    int flags = 0;
    if (!E->hpin && n <= HOST_PINNED_MAX) {
        void* p = nullptr;
        if (hipHostMalloc(&p, sizeof(double) * (8 * (size_t)n + GFNFF_NTERMS + 2), hipHostMallocDefault) == hipSuccess)
            E->hpin = (double*)p;
        else
            (void)hipGetLastError();  // no pinned memory: by copies
    }
    if (E->hpin) {
        double* const o = E->hpin + 3 * (size_t)n;
        std::memcpy(E->hpin, xyz_bohr, sizeof(double) * 3 * n);
        const int st = launch_eval(E, E->hpin, nullptr, nullptr, E->own, msg);
        if (st) return st;
        const double* const g = want_grad && grad ? E->grad : nullptr;
        hipLaunchKernelGGL(k_host_out, dim3(cdiv(std::max((g ? 5 : 2) * n, GFNFF_NTERMS + 2), 256)), dim3(256), 0,
                           E->own, n, E->out, E->flags, g, E->q, E->cn, o);
        HIP_OK(hipGetLastError());
        HIP_OK(hipStreamSynchronize(E->own));
        const double* const r = o + GFNFF_NTERMS + 2;
        std::memcpy(e_terms, o, sizeof(double) * (GFNFF_NTERMS + 1));
        flags = (int)o[GFNFF_NTERMS + 1];
        if (q) std::memcpy(q, r, sizeof(double) * n);
        if (cn) std::memcpy(cn, r + n, sizeof(double) * n);
        if (g) std::memcpy(grad, r + 2 * (size_t)n, sizeof(double) * 3 * n);
    } else {
        HIP_OK(hipMemcpyAsync(E->gpair, xyz_bohr, 3 * sizeof(double) * n, hipMemcpyHostToDevice, E->own));
        // gpair is overwritten by the pair reduction after the head of the evaluation has consumed it
        const int st = launch_eval(E, E->gpair, nullptr, nullptr, E->own, msg);
        if (st) return st;
        HIP_OK(hipMemcpyAsync(e_terms, E->out, sizeof(double) * (GFNFF_NTERMS + 1), hipMemcpyDeviceToHost, E->own));
        HIP_OK(hipMemcpyAsync(&flags, E->flags, sizeof(int), hipMemcpyDeviceToHost, E->own));
        if (want_grad && grad)
            HIP_OK(hipMemcpyAsync(grad, E->grad, 3 * sizeof(double) * n, hipMemcpyDeviceToHost, E->own));
        if (q) HIP_OK(hipMemcpyAsync(q, E->q, sizeof(double) * n, hipMemcpyDeviceToHost, E->own));
        if (cn) HIP_OK(hipMemcpyAsync(cn, E->cn, sizeof(double) * n, hipMemcpyDeviceToHost, E->own));
        HIP_OK(hipStreamSynchronize(E->own));
    }
    flags = final_flags(flags);
    if (flags & FLAG_CHOL) {
        msg = "EEQ matrix is not positive definite on the constraint space";
        return kErrEEQ;
    }
    if (flags & FLAG_CNOVF) {
        msg = "more than 128 atoms within the 6 Bohr CN cut-off of one atom";
        return kErrGeometry;
    }
    if (flags & FLAG_SOLVE) {
        msg = "EEQ triangular solve did not complete (a block waited beyond its bound)";
        return kErrDevice;
    }
    return kOk;
}

int device_eval(DeviceEngine* E, const double* xyz_bohr_dev, double* energy_dev, double* grad_dev, void* stream,
                std::string& msg) {
    hipStream_t s = (hipStream_t)stream;
    return launch_eval(E, xyz_bohr_dev, energy_dev, grad_dev, s, msg);
}

// Records one device-resident evaluation with fixed buffers into a HIP graph
// (both streams: the fork and join events become graph dependencies) and
// instantiates it; nothing runs during the capture.  The evaluation queues
// no memset or host synchronisation, and the kernel-class timer is off
// while recording.
int device_graph_capture(DeviceEngine* E, const double* xyz_bohr_dev, double* energy_dev, double* grad_dev,
                         void* stream, std::string& msg) {
    hipStream_t s = (hipStream_t)stream;
    if (!s) {
        msg = "graph capture needs a created stream (not the default stream)";
        return kErrArgs;
    }
    if (E->batch_streams == 2) {
        // its capture ended in a crash inside the runtime whose cause is not
        // established: the two-stream factorisation runs eagerly only
        msg = "graph capture is not available with batch_streams 2";
        return kErrArgs;
    }
    E->drop_graph();
    const int cls = E->timer.cls;
    E->timer.cls = -1;
    HIP_OK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
    const int st = device_eval(E, xyz_bohr_dev, energy_dev, grad_dev, stream, msg);
    hipGraph_t g = nullptr;
    const hipError_t ce = hipStreamEndCapture(s, &g);
    E->timer.cls = cls;
    if (st != kOk || ce != hipSuccess || !g) {
        if (g) (void)hipGraphDestroy(g);
        if (st == kOk) msg = std::string("hipStreamEndCapture: ") + hipGetErrorString(ce);
        return st != kOk ? st : kErrDevice;
    }
    hipGraphExec_t ex = nullptr;
    const hipError_t ie = hipGraphInstantiate(&ex, g, nullptr, nullptr, 0);
    if (ie != hipSuccess) {
        (void)hipGraphDestroy(g);
        msg = std::string("hipGraphInstantiate: ") + hipGetErrorString(ie);
        return kErrDevice;
    }
    E->graph = g;
    E->gexec = ex;
    return kOk;
}

int device_graph_launch(DeviceEngine* E, void* stream, std::string& msg) {
    if (!E->gexec) {
        msg = "no captured evaluation (the engine was rebuilt, or gfnff_graph_capture was not called)";
        return kErrArgs;
    }
    HIP_OK(hipGraphLaunch(E->gexec, (hipStream_t)stream));
    return kOk;
}

int device_md_steps(DeviceEngine* E, double* x_dev, double* v_dev, double* grad_dev, const double* mass_amu,
                    const double* xref_bohr, double dt_fs, double T0, double tau_fs, double disp_thresh, int nsteps,
                    double* rec_dev, void* stream, std::string& msg) {
    const int n = E->n, n3 = 3 * n;
    hipStream_t s = (hipStream_t)stream;
    constexpr double kAmuToMe = 1822.8884850;    // electron masses per amu (global.h:46)
    constexpr double kFsToAu = 41.34137314;      // atomic time units per fs (global.h:50)
    constexpr double kBoltzEh = 3.166811e-6;     // Hartree per Kelvin (global.h:47)
    if (!E->md_im3) {
        try {
            E->md_im3 = E->alloc<double>(n3);
            E->md_m3 = E->alloc<double>(n3);
            E->md_xref = E->alloc<double>(n3);
            E->md_part = E->alloc<double>(2 * (size_t)cdiv(n3, MD_T));
            E->md_e = E->alloc<double>(GFNFF_NTERMS + 1);
            E->md_lambda = E->alloc<double>(1);
        } catch (const std::bad_alloc&) {
            msg = "device allocation failed";
            return kErrDevice;
        }
    }
    std::vector<double> m3(n3), im3(n3);
    for (int i = 0; i < n; ++i) {
        if (!(mass_amu[i] > 0.0)) {
            msg = "masses must be positive";
            return kErrArgs;
        }
        for (int c = 0; c < 3; ++c) {
            m3[3 * i + c] = mass_amu[i] * kAmuToMe;
            im3[3 * i + c] = 1.0 / (mass_amu[i] * kAmuToMe);
        }
    }
    // once per call (not per step): masses and the coordinates of the last HB/XB detection
    HIP_OK(hipStreamSynchronize(s));
    HIP_OK(hipMemcpy(E->md_m3, m3.data(), sizeof(double) * n3, hipMemcpyHostToDevice));
    HIP_OK(hipMemcpy(E->md_im3, im3.data(), sizeof(double) * n3, hipMemcpyHostToDevice));
    HIP_OK(hipMemcpy(E->md_xref, xref_bohr, sizeof(double) * n3, hipMemcpyHostToDevice));
    const double dt = dt_fs * kFsToAu, tau = tau_fs * kFsToAu;
    const int dof = n > 2 ? 3 * n - 6 : (n == 2 ? 1 : 3);
    const double disp2_max = (disp_thresh * n) * (disp_thresh * n);
    const int nb = cdiv(n3, MD_T);
    for (int step = 0; step < nsteps; ++step) {
        hipLaunchKernelGGL(k_md_drift, dim3(nb), dim3(MD_T), 0, s, n3, dt, E->md_im3, grad_dev, x_dev, v_dev);
        const int st = device_eval(E, x_dev, E->md_e, grad_dev, stream, msg);
        if (st) return st;
        hipLaunchKernelGGL(k_md_kick, dim3(nb), dim3(MD_T), 0, s, n3, dt, E->md_im3, E->md_m3, grad_dev, x_dev,
                           E->md_xref, v_dev, E->md_part);
        hipLaunchKernelGGL(k_md_finish, dim3(1), dim3(64), 0, s, nb, E->md_part, E->md_e, kBoltzEh * dof, dt, T0, tau,
                           disp2_max, E->md_lambda, rec_dev + 4 * (size_t)step, E->sticky);
        if (T0 > 0.0) hipLaunchKernelGGL(k_md_scale, dim3(nb), dim3(MD_T), 0, s, n3, E->md_lambda, v_dev);
    }
    HIP_OK(hipGetLastError());
    return kOk;
}

int device_status(DeviceEngine* E, int* flags, bool clear, std::string& msg) {
    HIP_OK(hipDeviceSynchronize());
    HIP_OK(hipMemcpy(flags, E->sticky, sizeof(int), hipMemcpyDeviceToHost));
    if (clear) {
        hipLaunchKernelGGL(k_fill_i, dim3(1), dim3(64), 0, E->own, 1, E->sticky, 0);
        HIP_OK(hipGetLastError());
        HIP_OK(hipStreamSynchronize(E->own));
    }
    return kOk;
}

int device_solver_iterations(DeviceEngine* E) {
    if (!E->use_cg) return 0;
    int it = -1;
    if (hipDeviceSynchronize() != hipSuccess || hipMemcpy(&it, E->cg_iters, sizeof(int), hipMemcpyDeviceToHost) != hipSuccess)
        return -1;
    return it;
}

int device_cn_neighbours(DeviceEngine* E, int* counts, int* idx, int maxnb, std::string& msg) {
    const int n = E->n;
    std::vector<int> nbl((size_t)n * MAXNB_CN);
    HIP_OK(hipDeviceSynchronize());
    HIP_OK(hipMemcpy(counts, E->nbn, sizeof(int) * n, hipMemcpyDeviceToHost));
    HIP_OK(hipMemcpy(nbl.data(), E->nbl, sizeof(int) * nbl.size(), hipMemcpyDeviceToHost));
    for (int i = 0; i < n; ++i)
        for (int k = 0; k < maxnb; ++k)
            idx[(size_t)i * maxnb + k] = (k < counts[i] && k < MAXNB_CN) ? nbl[(size_t)i * MAXNB_CN + k] : -1;
    return kOk;
}

int device_batch_energies(DeviceEngine* E, double* e_mol, bool device_dst, void* stream, std::string& msg) {
    if (E->nmol < 2) {
        msg = "not a batch";
        return kErrArgs;
    }
    if (device_dst) {
        hipLaunchKernelGGL(k_copy, dim3(cdiv(E->nmol, 256)), dim3(256), 0, (hipStream_t)stream, E->nmol, E->e_mol,
                           e_mol);
        HIP_OK(hipGetLastError());
    } else {
        HIP_OK(hipDeviceSynchronize());
        HIP_OK(hipMemcpy(e_mol, E->e_mol, sizeof(double) * E->nmol, hipMemcpyDeviceToHost));
    }
    return kOk;
}

int device_update_params(DeviceEngine* E, const ParamSet& P, std::string& msg) {
    HIP_OK(hipDeviceSynchronize());
    HIP_OK(hipMemcpy(E->szr, P.sqrt_zr4r2.data(), sizeof(double) * P.n, hipMemcpyHostToDevice));
    HIP_OK(hipMemcpy(E->anb, P.rep_anb.data(), sizeof(double) * P.n, hipMemcpyHostToDevice));
    HIP_OK(hipMemcpy(E->repz, P.repz.data(), sizeof(double) * P.n, hipMemcpyHostToDevice));
    if (!P.brep_par.empty())
        HIP_OK(hipMemcpy(E->brep_par, P.brep_par.data(), sizeof(double) * P.brep_par.size(),
                         hipMemcpyHostToDevice));
    return kOk;
}

// partner chunks of the pair adjoint: at most 16, of at least 64 partners of
// one large molecule
static int adj_chunks(int n) {
    const int rows = cdiv(n, TILE);
    return std::max(1, std::min({16, cdiv(1024, rows), cdiv(n, 64)}));
}

template <int NE>
static void queue_adjoint(DeviceEngine* E, hipStream_t s, const PairArgs& pa, double* part, double* bpart) {
    const int n = E->n;
    const int nc = adj_chunks(n);
    hipLaunchKernelGGL(k_adj_pairs<NE>, dim3(cdiv(n, TILE), nc), dim3(TILE), 0, s, pa, E->adj_w, E->adj_u, part);
    hipLaunchKernelGGL(k_adj_nbrep_fix<NE>, dim3(cdiv(n, 256)), dim3(256), 0, s, n, E->x, E->Z, E->metal, E->elem,
                       E->anb, E->repz, E->toff, E->tidx, E->tdist, E->adj_w, part + (size_t)nc * ADJ_P * NE * n);
    if (E->nbrep)
        hipLaunchKernelGGL(k_adj_brep<NE>, dim3(cdiv(E->nbrep, 256)), dim3(256), 0, s, E->nbrep, E->brep_ij,
                           E->brep_par, E->elem, E->x, E->adj_w, bpart);
    if ((long)(nc + 1) * n + E->nbrep <= ADJ_ONE_MAX) {
        hipLaunchKernelGGL(k_adj_reduce<1>, dim3(ADJ_P * NE), dim3(256), 0, s, n, nc + 1, part, E->nbrep, bpart,
                           ADJ_P * NE, E->adj_out);
        return;
    }
    hipLaunchKernelGGL(k_adj_reduce<ADJ_RB>, dim3(ADJ_P * NE, ADJ_RB), dim3(256), 0, s, n, nc + 1, part, E->nbrep,
                       bpart, ADJ_P * NE, E->adj_share);
    hipLaunchKernelGGL(k_adj_final, dim3(ADJ_P * NE), dim3(64), 0, s, E->adj_share, E->adj_out);
}

// dLoss/dln(theta) = sum_i w_i . dg_i/dln(theta) at the state of the last
// evaluation (coordinates, charges, CN and D4 weights on the device).
int device_param_adjoint(DeviceEngine* E, const double* w, double* out, std::string& msg) {
    const int n = E->n, ne = E->nelem;
    if (ne < 1 || ne > 4) {
        msg = "the parameter adjoint is built for up to 4 elements";
        return kErrUnsupported;
    }
    hipStream_t s = E->own;
    HIP_OK(hipDeviceSynchronize());
    if (!E->adj_w) {
        try {
            E->adj_w = E->alloc<double>(3 * (size_t)n);
            E->adj_u = E->alloc<double>(n);
            E->adj_part = E->alloc<double>((size_t)(adj_chunks(n) + 1) * ADJ_P * ne * n);
            E->adj_share = E->alloc<double>(ADJ_P * ne * ADJ_RB);
            E->adj_bpart = E->alloc<double>((size_t)ADJ_P * ne * std::max(E->nbrep, 1));
            E->adj_out = E->alloc<double>(ADJ_P * ne);
        } catch (const std::bad_alloc&) {
            msg = "device allocation failed";
            return kErrDevice;
        }
    }
    HIP_OK(hipMemcpyAsync(E->adj_w, w, sizeof(double) * 3 * n, hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_adj_u, dim3(cdiv(n, 256)), dim3(256), 0, s, n, E->x, E->rcov_cn, E->dlog, E->nbn, E->nbl,
                       E->adj_w, E->adj_u);
    PairArgs pa = E->pair_args();
    switch (ne) {
        case 1: queue_adjoint<1>(E, s, pa, E->adj_part, E->adj_bpart); break;
        case 2: queue_adjoint<2>(E, s, pa, E->adj_part, E->adj_bpart); break;
        case 3: queue_adjoint<3>(E, s, pa, E->adj_part, E->adj_bpart); break;
        default: queue_adjoint<4>(E, s, pa, E->adj_part, E->adj_bpart); break;
    }
    HIP_OK(hipGetLastError());
    HIP_OK(hipMemcpyAsync(out, E->adj_out, sizeof(double) * ADJ_P * ne, hipMemcpyDeviceToHost, s));
    HIP_OK(hipStreamSynchronize(s));
    return kOk;
}

int device_profile_select(DeviceEngine* E, const char* name, std::string& msg) {
    E->timer.used = 0;
    E->timer.cls = -1;
    if (!name || !*name) return kOk;
    for (int c = 0; c < KC_COUNT; ++c)
        if (std::strcmp(name, kKernelClassNames[c]) == 0) {
            E->timer.cls = c;
            return kOk;
        }
    msg = std::string("unknown kernel class: ") + name;
    return kErrArgs;
}

int device_profile_read(DeviceEngine* E, double* total_ms, int* launches, std::string& msg) {
    KernelTimer& T = E->timer;
    *total_ms = 0.0;
    *launches = 0;
    for (size_t i = 0; i + 1 < T.used; i += 2) {
        float ms = 0.0f;
        HIP_OK(hipEventSynchronize(T.ev[i + 1]));  // launches of a class may sit on different streams
        HIP_OK(hipEventElapsedTime(&ms, T.ev[i], T.ev[i + 1]));
        *total_ms += ms;
        ++*launches;
    }
    T.used = 0;
    return kOk;
}

int device_solvation_parts(DeviceEngine* E, double* parts, std::string& msg) {
    if (!E->solv) {
        msg = "no solvent";
        return kErrArgs;
    }
    if (hipMemcpy(parts, E->sa.parts, 4 * sizeof(double), hipMemcpyDeviceToHost) != hipSuccess) {
        msg = "download failed";
        return kErrDevice;
    }
    return kOk;
}

int device_count() {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

// Blocked Cholesky of a dense SPD matrix (the EEQ factorisation kernels on an
// arbitrary input).  a: n x n row-major; l_out receives the lower factor.
template <typename T>
static int dense_cholesky(int n, const T* a, T* l_out, std::string& msg) {
    if (n <= 0) {
        msg = "n must be positive";
        return kErrArgs;
    }
    const int np = cdiv(n, NB) * NB;
    std::vector<T> h((size_t)np * np, 0.0);
    for (int i = 0; i < np; ++i)
        for (int j = 0; j < np; ++j) h[(size_t)i * np + j] = (i < n && j < n) ? a[(size_t)i * n + j] : (i == j ? T(1) : T(0));
    T *dA = nullptr, *dL = nullptr;
    int* dflag = nullptr;
    hipStream_t s = nullptr;
    int st = kOk;
    auto cleanup = [&]() {
        if (s) (void)hipStreamDestroy(s);
        if (dA) (void)hipFree(dA);
        if (dL) (void)hipFree(dL);
        if (dflag) (void)hipFree(dflag);
    };
    if (hipStreamCreate(&s) != hipSuccess || hipMalloc(&dA, h.size() * sizeof(T)) != hipSuccess ||
        hipMalloc(&dL, (size_t)np * NB * sizeof(T)) != hipSuccess || hipMalloc(&dflag, sizeof(int)) != hipSuccess) {
        cleanup();
        msg = "device allocation failed";
        return kErrDevice;
    }
    int zero = 0, flag = 0;
    (void)hipMemcpyAsync(dA, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice, s);
    (void)hipMemcpyAsync(dflag, &zero, sizeof(int), hipMemcpyHostToDevice, s);
    queue_cholesky(nullptr, s, np, dA, dL, dflag);
    (void)hipMemcpyAsync(h.data(), dA, h.size() * sizeof(T), hipMemcpyDeviceToHost, s);
    (void)hipMemcpyAsync(&flag, dflag, sizeof(int), hipMemcpyDeviceToHost, s);
    if (hipStreamSynchronize(s) != hipSuccess) {
        msg = "kernel failure";
        st = kErrDevice;
    } else if (flag & FLAG_CHOL) {
        msg = "matrix is not positive definite";
        st = kErrEEQ;
    }
    for (int i = 0; i < n; ++i)
        for (int j = 0; j < n; ++j) l_out[(size_t)i * n + j] = (j <= i) ? h[(size_t)i * np + j] : T(0);
    cleanup();
    return st;
}

int device_dense_cholesky(int n, const double* a, double* l_out, std::string& msg) {
    return dense_cholesky<double>(n, a, l_out, msg);
}

int device_dense_cholesky_f32(int n, const float* a, float* l_out, std::string& msg) {
    return dense_cholesky<float>(n, a, l_out, msg);
}

// ---------------------------------------------------------------------------
// Allocation-free variant of the dense Cholesky: the padded working matrix,
// the inverses of its diagonal blocks and the status word sit in one
// file-scope device array (8.5 MB on every device the library runs on, held
// until the process ends).  Host code never uses the array's name as an
// address: the device address comes from hipGetSymbolAddress, taken once per
// device at the first call there, and the kernels receive that address.
// Calls that overlap on one device share the array and race.
// ---------------------------------------------------------------------------
constexpr int NOALLOC_MAX_N = 1024;
constexpr size_t NOALLOC_MAT = (size_t)NOALLOC_MAX_N * NOALLOC_MAX_N;  // padded np x np matrix
constexpr size_t NOALLOC_LINV = (size_t)NOALLOC_MAX_N * NB;           // np / 64 inverses of 64 x 64 blocks
constexpr size_t NOALLOC_DOUBLES = NOALLOC_MAT + NOALLOC_LINV + 32;    // + status word (256-byte line)
static __device__ __align__(256) double scratch[NOALLOC_DOUBLES];

namespace {
// A = a padded to np x np with the identity; clears the status word (a store,
// not a memset, so that the sequence can be captured in a graph).
__global__ __launch_bounds__(256) void k_noalloc_pad(int n, int np, const double* __restrict__ a,
                                                     double* __restrict__ A, int* __restrict__ flag) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e == 0) flag[0] = 0;
    if (e >= (size_t)np * np) return;
    const int i = (int)(e / np), j = (int)(e % np);
    A[e] = (i < n && j < n) ? a[(size_t)i * n + j] : (i == j ? 1.0 : 0.0);
}

// l = lower triangle of the factored A (zeros above the diagonal); status
// GFNFF_STATUS_EEQ (3) when a pivot was not positive, else 0.
__global__ __launch_bounds__(256) void k_noalloc_out(int n, int np, const double* __restrict__ A,
                                                     double* __restrict__ l, const int* __restrict__ flag,
                                                     int* __restrict__ status) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e == 0) status[0] = (flag[0] & FLAG_CHOL) ? kErrEEQ : kOk;
    if (e >= (size_t)n * n) return;
    const int i = (int)(e / n), j = (int)(e % n);
    l[e] = (j <= i) ? A[(size_t)i * np + j] : 0.0;
}

constexpr int NOALLOC_MAX_DEVICES = 64;
std::mutex g_noalloc_mu;
double* g_noalloc_base[NOALLOC_MAX_DEVICES] = {};
}  // namespace

int device_dense_cholesky_noalloc(int n, const double* a_dev, double* l_dev, int* status_dev, void* stream,
                                  std::string& msg) {
    if (n <= 0 || n > NOALLOC_MAX_N) {
        msg = "n must be in 1.." + std::to_string(NOALLOC_MAX_N);
        return kErrArgs;
    }
    int dev = 0;
    HIP_OK(hipGetDevice(&dev));
    if (dev < 0 || dev >= NOALLOC_MAX_DEVICES) {
        msg = "device index out of range";
        return kErrArgs;
    }
    double* base = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_noalloc_mu);
        if (!g_noalloc_base[dev]) {
            void* p = nullptr;
            HIP_OK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
            if (!p) {
                msg = "no device address for the scratch array";
                return kErrDevice;
            }
            g_noalloc_base[dev] = static_cast<double*>(p);
        }
        base = g_noalloc_base[dev];
    }
    const int np = cdiv(n, NB) * NB;
    double* A = base;
    double* Linv = base + NOALLOC_MAT;
    int* flag = reinterpret_cast<int*>(base + NOALLOC_MAT + NOALLOC_LINV);
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(k_noalloc_pad, dim3(cdiv((long)np * np, 256)), dim3(256), 0, s, n, np, a_dev, A, flag);
    queue_cholesky<double>(nullptr, s, np, A, Linv, flag);
    hipLaunchKernelGGL(k_noalloc_out, dim3(cdiv((long)n * n, 256)), dim3(256), 0, s, n, np, A, l_dev, flag,
                       status_dev);
    HIP_OK(hipGetLastError());
    return kOk;
}

}  // namespace gfnff
