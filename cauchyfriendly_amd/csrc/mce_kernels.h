// HIP kernels of the MCE term-propagation step (gfx950).
//
// Per scalar measurement update the host drives, in order:
//   k_tp               time propagation + Gamma coalignment, one thread per parent
//   k_btab_simple      B-tables that need no enumeration (copy / identity / empty)
//   k_btab_enum        time-propagation B-table by vertex enumeration, one block per parent
//   k_mu               measurement update, one thread per output slot (parent x child)
//   k_mom_sum          fz / mean / covariance summands and their in-order sums per
//                      reference thread (second stream, overlapped with reduction)
//   k_ftr_*            fast term reduction of all shape buckets: keys, components, groups
//   k_group_btab       B-table of each reduction group's root, one wavefront per group
//   k_group_eval       g-tables of each group: root, replacement chain, member sums
//   k_group_sort       key order for groups whose root was replaced
//   k_compact          survivors become the next step's parents
#pragma once
#include <climits>

#include <hipcub/block/block_radix_sort.hpp>

#include "mce_device.h"
#include "mce_multi.h"
#include "mce_pool.h"

namespace mce {

constexpr int kWave = 64;
// Gather key of a slot that holds no term: above every term's ((m T + tid) 2 + child), which
// stays below 336 for shapes up to 20 hyperplanes and T <= 8, so the sort needs 10 bits.
constexpr uint32_t kGatherKeyNone = 0x3ffu;
constexpr int kGatherKeyBits = 10;
// Default: groups with more members than this add them with one wavefront per member.
constexpr int kBigGroupMembers = 16;
// Slots of an engine's device counters that more than one kernel knows.
constexpr int kCtrMuErr = 17;     // measurement-update error bits
constexpr int kCtrNanP = 24;      // set when a child's p holds a NaN
constexpr int kCtrBigComp = 25;   // reduction components beyond one wavefront

enum BtabMode : uint8_t { kModeNone = 0, kModeCopy = 1, kModeIdent = 2, kModeTrivial = 3, kModeEmpty = 4, kModeEnum = 5 };

// Per-update constants (one small device buffer).
struct StepConst {
    double Phi[kMaxD * kMaxD];
    double H[kMaxD];
    double G[kMaxM * kMaxD];   // pre-coaligned Gamma rows
    double beta[kMaxM];
    double Bu[kMaxD];          // B u, computed once per update
    double root[kMaxD];
    double msmt, gamma, gscale;
    int d, ng, cmcc, with_tp, skip, first, T, threaded;
    int order[kMaxD];          // fast-term-reduction axis order
    int in_off[kMaxM + 2];     // parents' shape bucket offsets (bucket m: [in_off[m], in_off[m+1]))
    int64_t rk_base[kMaxM + 2];  // first rank-arena word of each shape bucket's rank structures
};

// ------------------------------------------------------------------ small dense linear algebra
// Column-sum one-norm, cauchy_linalg.hpp:1301-1314.
template <int D>
__device__ inline double dev_one_norm(const double* A) {
    double best = -1;
#pragma unroll
    for (int c = 0; c < D; c++) {
        double s = 0;
#pragma unroll
        for (int r = 0; r < D; r++) s += fabs(A[r * D + c]);
        if (s > best) best = s;
    }
    return best;
}

// In-place partial-pivot LU, cauchy_linalg.hpp:1180-1232.  Row exchanges are
// written as predicated swaps over compile-time indices so the matrix stays in
// registers; the arithmetic and its order are the reference's.
template <int D>
__device__ inline bool dev_lu(double* A, int* piv) {
#pragma unroll
    for (int j = 0; j < D; ++j) {
        double pv = kPluEps;
        int pi = -1;
#pragma unroll
        for (int i = j; i < D; ++i)
            if (fabs(A[i * D + j]) > fabs(pv)) {
                pv = A[i * D + j];
                pi = i;
            }
        if (pi == -1) return false;
#pragma unroll
        for (int r = j + 1; r < D; ++r) {
            const bool sw = (r == pi);
#pragma unroll
            for (int k = 0; k < D; k++) {
                const double a = A[j * D + k], b = A[r * D + k];
                A[j * D + k] = sw ? b : a;
                A[r * D + k] = sw ? a : b;
            }
        }
        piv[j] = pi;
#pragma unroll
        for (int k = j + 1; k < D; ++k) {
            A[k * D + j] /= A[j * D + j];
            const double t = A[k * D + j];
#pragma unroll
            for (int q = j + 1; q < D; q++) A[k * D + q] -= t * A[j * D + q];
        }
    }
    return true;
}

template <int D>
__device__ inline void dev_fwd(const double* LU, double* b) {
#pragma unroll
    for (int i = 0; i < D; i++) {
        double s = b[i];
#pragma unroll
        for (int j = 0; j < i; j++) s -= LU[i * D + j] * b[j];
        b[i] = s;
    }
}
template <int D>
__device__ inline void dev_bwd(const double* LU, double* b) {
#pragma unroll
    for (int i = D - 1; i >= 0; i--) {
        double s = b[i];
#pragma unroll
        for (int j = D - 1; j > i; j--) s -= LU[i * D + j] * b[j];
        b[i] = s / LU[i * D + i];
    }
}
// Inverse of the LAPACK-style pivot sequence (cauchy_linalg.hpp:1258-1277):
// pt[r] = position row r of the original matrix ends up at.
template <int D>
__device__ inline void dev_pivot_inverse(const int* piv, int* pt) {
    int preg[D];
#pragma unroll
    for (int i = 0; i < D; i++) preg[i] = i;
#pragma unroll
    for (int i = 0; i < D; i++) {
        // swap preg[i] and preg[piv[i]] (piv[i] >= i)
        const int a = preg[i];
        int b = a;
#pragma unroll
        for (int r = i; r < D; r++) b = (r == piv[i]) ? preg[r] : b;
#pragma unroll
        for (int r = i; r < D; r++) preg[r] = (r == piv[i]) ? a : preg[r];
        preg[i] = b;
    }
#pragma unroll
    for (int r = 0; r < D; r++) {
        int v = 0;
#pragma unroll
        for (int i = 0; i < D; i++) v = (preg[i] == r) ? i : v;
        pt[r] = v;
    }
}

// One-norm condition number via explicit inverse, cauchy_linalg.hpp:1337-1392.
// The callers only compare it with kCondEps.  A cheap bound decides first: every
// entry of A^-1 is a cofactor over det A, and by Hadamard's inequality a cofactor is
// at most rn^(D-1), rn the largest row 1-norm, so cond1 <= ||A||_1 * D * rn^(D-1) /
// |det A|, with |det A| the product of the LU pivots.  When that bound is below
// kCondScreen (three orders of magnitude under kCondEps, far beyond the rounding of
// the pivots) the bound is returned; otherwise the reference's value is computed.
constexpr double kCondScreen = 1e9;
template <int D>
__device__ inline double dev_cond1(double* A, int* piv) {
    const double na = dev_one_norm<D>(A);
    double rn = 0;
#pragma unroll
    for (int r = 0; r < D; r++) {
        double s = 0;
#pragma unroll
        for (int c = 0; c < D; c++) s += fabs(A[r * D + c]);
        rn = fmax(rn, s);
    }
    if (!dev_lu<D>(A, piv)) return 1.7976931348623157e308;
    {
        double det = 1.0, bnd = na * (double)D;
#pragma unroll
        for (int i = 0; i < D; i++) det *= fabs(A[i * D + i]);
#pragma unroll
        for (int i = 0; i < D - 1; i++) bnd *= rn;
        if (bnd <= kCondScreen * det) return bnd / det;
    }
    int pt[D];
    dev_pivot_inverse<D>(piv, pt);
    // one-norm of the inverse = largest absolute row sum of W, whose row i solves
    // A w = e_i (W is the transpose of the inverse before reflect_array)
    double best = -1;
#pragma unroll
    for (int i = 0; i < D; i++) {
        double w[D];
#pragma unroll
        for (int c = 0; c < D; c++) w[c] = (c == pt[i]) ? 1.0 : 0.0;
        dev_fwd<D>(A, w);
        dev_bwd<D>(A, w);
        double s = 0;
#pragma unroll
        for (int r = 0; r < D; r++) s += fabs(w[r]);
        if (s > best) best = s;
    }
    return na * best;
}

template <int D>
__device__ inline void dev_lu_solve(const double* LU, const int* piv, const double* b, double* x) {
    int pt[D];
    dev_pivot_inverse<D>(piv, pt);
#pragma unroll
    for (int c = 0; c < D; c++) {
        double v = 0.0;
#pragma unroll
        for (int i = 0; i < D; i++) v = (pt[i] == c) ? b[i] : v;
        x[c] = v;
    }
    dev_fwd<D>(LU, x);
    dev_bwd<D>(LU, x);
}

template <int D>
__device__ inline double dev_dot(const double* x, const double* y) {
    double z = 0.0;
    for (int i = 0; i < D; i++) z += x[i] * y[i];
    return z;
}

// ------------------------------------------------------------------ wave helpers
__device__ inline int wave_lane() { return threadIdx.x & (kWave - 1); }

__device__ inline int wave_excl_scan(int v, int* total) {
    const int lane = wave_lane();
    int x = v;
    for (int o = 1; o < kWave; o <<= 1) {
        int y = __shfl_up(x, o, kWave);
        if (lane >= o) x += y;
    }
    *total = __shfl(x, kWave - 1, kWave);
    return x - v;
}

// A value that every lane of the wavefront holds alike, in scalar registers.
__device__ __forceinline__ int wave_uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int64_t wave_uniform(int64_t v) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    return ((int64_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32) | lo;
}

// Orders the LDS accesses of the lanes of one wavefront (for workgroups of one wavefront):
// a wavefront's LDS operations complete in issue order, so only the compiler has to be
// held back, and the wavefront does not wait for its global loads and stores as a
// workgroup barrier makes it.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Inclusive scan of one value per lane across a wavefront (shuffles, no barrier).
template <class T>
__device__ __forceinline__ T wave_incl_scan(T x) {
    const int lane = (int)(threadIdx.x & (kWave - 1));
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const T y = __shfl_up(x, o, kWave);
        if (lane >= o) x += y;
    }
    return x;
}

// Largest input of the one-workgroup scans, and their threads.
constexpr int kSmallScan = 65536;
constexpr int kSmallScanThreads = 1024;

// Exclusive prefix of each thread's `v` over a block of kSmallScanThreads threads, and the
// block total: wavefront scans, then one wavefront scans the wavefront totals (two
// barriers).  Every thread of the block must call it.
template <class T>
__device__ __forceinline__ T block_excl_scan(T v, T* total) {
    constexpr int kWaves = kSmallScanThreads / kWave;
    __shared__ T wsum[kWaves];
    const int lane = (int)(threadIdx.x & (kWave - 1)), w = (int)(threadIdx.x / kWave);
    const T x = wave_incl_scan(v);
    if (lane == kWave - 1) wsum[w] = x;
    __syncthreads();
    if (w == 0) {
        T y = lane < kWaves ? wsum[lane] : (T)0;
        y = wave_incl_scan(y);
        if (lane < kWaves) wsum[lane] = y;
    }
    __syncthreads();
    *total = wsum[kWaves - 1];
    return (w > 0 ? wsum[w - 1] : (T)0) + x - v;
}

// Exclusive prefix of each thread's v over a block of whole wavefronts (at most 4) and the
// block total, through wsum[4] in LDS (two barriers).  Every thread of the block calls it.
__device__ __forceinline__ int block4_excl_scan(int v, int* total, int* wsum) {
    const int lane = (int)(threadIdx.x & (kWave - 1)), w = (int)(threadIdx.x / kWave);
    const int nw = (int)(blockDim.x / kWave);
    const int x = wave_incl_scan(v);
    __syncthreads();  // wsum of an earlier scan has been read
    if (lane == kWave - 1) wsum[w] = x;
    __syncthreads();
    int before = 0, tot = 0;
    for (int k = 0; k < nw; k++) {
        const int sk = wsum[k];
        before += k < w ? sk : 0;
        tot += sk;
    }
    *total = tot;
    return before + x - v;
}

// ------------------------------------------------------------------ first term
// The term a window starts from (setup_first_term, cauchy_term.hpp:772-785), by value with
// the launch: one launch and one wait per reset, where a copy per field waited seven times.
struct FirstTerm {
    double A[kMaxD * kMaxD], p[kMaxD], b[kMaxD];
};
__global__ __launch_bounds__(64) void k_first_term(TermPool P, int d, FirstTerm f) {
    const int t = threadIdx.x;
    for (int i = t; i < P.MM * d; i += 64) P.A[i] = i < d * d ? f.A[i] : 0.0;
    for (int i = t; i < P.MM; i += 64) P.p[i] = i < d ? f.p[i] : 0.0;
    if (t < d) P.b[t] = f.b[t];
    if (t == 0) {
        P.m[0] = d;
        P.gp_n[0] = 0;
        P.gp_off[0] = 0;
    }
}

// ------------------------------------------------------------------ time propagation
// cauchy_term.hpp:435-531 (time_prop, normalize_hps, tp_coalign), with the B-table
// mode decision of cauchy_estimator.hpp:678-708 (serial) / 1614-1637 (threaded).
template <int D>
__device__ __forceinline__ void k_tp(MG<1024, 1> mg, TermPool P, int n, const StepConst* __restrict__ sc, const int* __restrict__ cen_half,
                     int* __restrict__ slots, int* __restrict__ btcap, int* __restrict__ err) {
    const int i = mg.bx * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int MM = P.MM;
    int m = P.m[i];
    const int phc = m;
    P.phc[i] = phc;
    double* A = P.A + (int64_t)i * MM * D;
    double* p = P.p + (int64_t)i * MM;
    double* b = P.b + (int64_t)i * D;
    if (sc->with_tp) {
        double t[D];
        for (int r = 0; r < m; r++) {
            for (int k = 0; k < D; k++) t[k] = A[r * D + k];
            for (int j = 0; j < D; j++) {
                double s = 0.0;
                for (int k = 0; k < D; k++) s += t[k] * sc->Phi[k + j * D];
                A[r * D + j] = s;
            }
        }
        for (int k = 0; k < D; k++) t[k] = b[k];
        for (int r = 0; r < D; r++) {
            double s = 0.0;
            for (int j = 0; j < D; j++) s += sc->Phi[r * D + j] * t[j];
            b[r] = s;
        }
        if (sc->cmcc > 0)
            for (int r = 0; r < D; r++) b[r] += 1.0 * sc->Bu[r];
        for (int r = 0; r < m; r++) {
            double n1 = 0;
            for (int k = 0; k < D; k++) n1 += fabs(A[r * D + k]);
            p[r] *= n1;
            for (int k = 0; k < D; k++) A[r * D + k] /= n1;
        }
        uint32_t F = (sc->ng >= 32) ? 0xffffffffu : ((1u << sc->ng) - 1u);
        for (int j = 0; j < sc->ng; j++)
            for (int k = 0; k < m; k++) {
                if (!((F >> j) & 1u)) continue;
                bool pos, neg;
                coalign_gates(&sc->G[j * D], &A[k * D], D, pos, neg);
                if (pos || neg) {
                    F &= ~(1u << j);
                    p[k] += sc->beta[j];
                }
            }
        for (int j = 0; j < sc->ng; j++)
            if ((F >> j) & 1u) {
                if (m >= MM) {
                    atomicOr(err, 4);
                    break;
                }
                for (int k = 0; k < D; k++) A[m * D + k] = sc->G[j * D + k];
                p[m] = sc->beta[j];
                m++;
            }
        P.m[i] = m;
    }
    int tid = 0;
    if (sc->threaded) tid = (i - sc->in_off[phc]) % sc->T;
    P.tid[i] = tid;
    uint8_t mode;
    int cap;
    const int gn = P.gp_n[i];
    if (sc->skip) {
        mode = kModeNone;
        cap = 0;
    } else if (!sc->with_tp) {
        mode = kModeCopy;
        cap = gn;
    } else if (sc->threaded && m <= D) {
        mode = kModeIdent;
        cap = gn;
    } else if (m == phc) {
        mode = kModeCopy;
        cap = gn;
    } else if (m < D) {
        mode = kModeTrivial;
        cap = max(1 << (m - 1), gn);
    } else if (m == D) {
        mode = kModeEmpty;
        cap = 0;
    } else {
        mode = kModeEnum;
        cap = cen_half[m];
    }
    P.mode[i] = mode;
    btcap[i] = cap;
    slots[i] = m + 1;
}

// B-tables that need no enumeration; enumeration jobs are appended to a list.
__device__ __forceinline__ void k_btab_simple(MG<1024, 1> mg, TermPool P, int n, const int64_t* __restrict__ bt_base, const uint32_t* __restrict__ gkeys,
                              uint32_t* __restrict__ Barena, int* __restrict__ enum_list, int* __restrict__ enum_count) {
    const int i = mg.bx * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint8_t mode = P.mode[i];
    const int64_t off = bt_base[i];
    P.bt_off[i] = off;
    P.bt_sgn[i] = 0;
    const int gn = P.gp_n[i];
    uint32_t* B = Barena + off;
    switch (mode) {
        case kModeCopy: {
            const uint32_t* src = gkeys + P.gp_off[i];
            for (int k = 0; k < gn; k++) B[k] = src[k];
            P.bt_n[i] = gn;
        } break;
        case kModeIdent:
            for (int k = 0; k < gn; k++) B[k] = (uint32_t)k;
            P.bt_n[i] = gn;
            break;
        case kModeTrivial: {
            const int m = P.m[i];
            const int nn = max(1 << (m - 1), gn);
            for (int k = 0; k < nn; k++) B[k] = (uint32_t)k;
            P.bt_n[i] = gn;
        } break;
        case kModeEnum: {
            const int slot = atomicAdd(enum_count, 1);
            enum_list[slot] = i;
            // the enumerator's LDS is sized by the largest shape and parent hyperplane
            // count among the parents it visits
            atomicMax(enum_count + 4, P.m[i]);
            atomicMax(enum_count + 5, P.phc[i]);
            P.bt_n[i] = 0;
        } break;
        default:
            P.bt_n[i] = 0;
            break;
    }
}

// The sign vectors of the cells around one vertex v of the arrangement: every hyperplane
// not among the vertex's D (cmask) takes the side of v; the D of the vertex take both.
template <int D>
__device__ __forceinline__ void enum_vertex_cells(const double* __restrict__ A, const double* __restrict__ bp, int m,
                                                  const uint8_t* __restrict__ cb, const double* v, uint32_t* bits) {
    uint32_t cbit[D], cmask = 0;
#pragma unroll
    for (int k = 0; k < D; k++) {
        cbit[k] = 1u << cb[k];
        cmask |= cbit[k];
    }
    // every hyperplane's side is computed (m is uniform, so no lane waits on another);
    // those of the vertex are dropped
    uint32_t niv = 0;
    for (int ac = 0; ac < m; ac++)
        if ((dev_dot<D>(A + ac * D, v) - bp[ac]) < 0) niv |= (1u << ac);
    niv &= ~cmask;
    for (int s = 0; s < (1 << D); s++) {
        uint32_t sv = niv;
#pragma unroll
        for (int k = 0; k < D; k++)
            if ((s >> k) & 1) sv |= cbit[k];
        atomicOr(&bits[sv >> 5], 1u << (sv & 31));
    }
}

// Cells of the time-propagated arrangement by vertex enumeration,
// cell_enumeration.hpp:676-855.  One block per parent; the sign vectors seen are
// an LDS bitset of 2^m bits, so the output comes out sorted and de-duplicated.
// The parent's g-table keys are a second LDS bitset, `pofs` words after the first,
// or, when `psearch` is set (both sets would not fit in LDS: 2^20 + 2^18 bits), are
// looked up by binary search in the parent's sorted keys in global memory.
//
// A vertex is kept when the one-norm condition number of its D hyperplanes is at most
// kCondEps.  The block decides that for T = blockDim.x combinations at a time, cheapest
// test first, each test exact against the reference's value:
//   * the LU factorisation fails (a pivot under kPluEps): the reference's value is the
//     largest double, rejected;
//   * the upper bound of dev_cond1 is under kCondScreen: kept;
//   * ||A||_1 / |u_DD| > kCondEps, u_DD the last pivot: rejected.  The reference's inverse
//     has the entry fl(1 / u_DD) (the solve of the unit vector that the pivots move to the
//     last row: forward substitution leaves it a unit vector, back substitution divides
//     it by u_DD), its norm is a sum of absolute values no smaller than that entry, and
//     rounding is monotone, so the reference's product ||A||_1 ||A^-1||_1 is at least this
//     product;
//   * otherwise the reference's value is computed (dev_cond1).
// On the window workloads about 28% of the combinations fail to factor, 63% pass the
// bound, 8% are rejected by the last pivot and 2% need the full value.  The kept vertices
// (with their solution) and the undecided combinations go to two LDS queues, which are
// worked off T at a time, so that the vertex work and the full condition number run on
// full wavefronts rather than on the lanes that one combination in each wavefront keeps.
template <int D>
__device__ __forceinline__ void k_btab_enum(MG<256, 3> mg, TermPool P, const int* __restrict__ list,
                                                   const double* __restrict__ bpert, const uint8_t* __restrict__ combos,
                                                   const int64_t* __restrict__ combo_off, const int* __restrict__ combo_cnt,
                                                   const uint32_t* __restrict__ gkeys, uint32_t* __restrict__ Barena,
                                                   const int* __restrict__ btcap, int* __restrict__ err, int pofs,
                                                   int psearch) {
    extern __shared__ double enum_lds[];
    __shared__ int wsum[4];
    const int T = (int)blockDim.x, Q = 2 * T;
    // queues: kept vertices (combination, solution) and undecided combinations, 2T each
    double* qv = enum_lds;                    // [D][Q]
    int* qa = (int*)(qv + (size_t)D * Q);     // [Q]
    int* qs = qa + Q;                         // [Q]
    uint32_t* bits = (uint32_t*)(qs + Q);
    const int i = list[mg.bx];
    const int MM = P.MM;
    const int m = P.m[i];
    const int phc = P.phc[i];
    const int W = m >= 5 ? (1 << (m - 5)) : 1;
    // bitset of the parent's g-table keys (all below 2^(phc-1)), after the 2^m-bit
    // sets of candidate sign vectors of every parent of the launch
    uint32_t* pbits = bits + pofs;
    const uint32_t ptop = 1u << (phc - 1);
    const int PW = psearch ? 0 : (int)((ptop + 31u) >> 5);
    for (int w = threadIdx.x; w < W; w += blockDim.x) bits[w] = 0;
    for (int w = threadIdx.x; w < PW; w += blockDim.x) pbits[w] = 0;
    __syncthreads();
    const uint32_t* gk = gkeys + P.gp_off[i];
    const int gn = P.gp_n[i];
    // a parent key at or above 2^(phc-1) (a coaligned child's cell kept with bit phc-1
    // set) can never equal a looked-up sign vector, which is reversed below it
    if (!psearch)
        for (int q = threadIdx.x; q < gn; q += blockDim.x) {
            const uint32_t key = gk[q];
            if (key < ptop) atomicOr(&pbits[key >> 5], 1u << (key & 31));
        }
    const double* A = P.A + (int64_t)i * MM * D;
    const double* bp = bpert + (int64_t)P.tid[i] * MM;
    const uint8_t* cmb = combos + combo_off[m];
    const int nc = combo_cnt[m];
    auto load = [&](int ci, double* Ac, double* bc) {
        const uint8_t* cb = cmb + ci * D;
#pragma unroll
        for (int j = 0; j < D; j++) {
            const int r = cb[j];
#pragma unroll
            for (int k = 0; k < D; k++) Ac[j * D + k] = A[r * D + k];
            bc[j] = bp[r];
        }
    };
    // appends this thread's kept vertex and / or undecided combination (block-wide call)
    int na = 0, ns = 0;
    auto push = [&](bool keep, bool slow, int ci, const double* v) {
        int tot;
        const int pre = block4_excl_scan((keep ? 1 : 0) | (slow ? 1 << 16 : 0), &tot, wsum);
        if (keep) {
            const int q = na + (pre & 0xffff);
            qa[q] = ci;
#pragma unroll
            for (int k = 0; k < D; k++) qv[k * Q + q] = v[k];
        }
        if (slow) qs[ns + (pre >> 16)] = ci;
        na += tot & 0xffff;
        ns += tot >> 16;
        __syncthreads();
    };
    // the cells around the last `cnt` kept vertices (block-wide call)
    auto drain = [&](int cnt) {
        const int q = na - cnt + (int)threadIdx.x;
        if ((int)threadIdx.x < cnt) {
            double v[D];
#pragma unroll
            for (int k = 0; k < D; k++) v[k] = qv[k * Q + q];
            enum_vertex_cells<D>(A, bp, m, cmb + qa[q] * D, v, bits);
        }
        na -= cnt;
        __syncthreads();
    };
    // the reference's condition number of the last `cnt` undecided combinations
    auto settle = [&](int cnt) {
        const int q = ns - cnt + (int)threadIdx.x;
        bool keep = false;
        int ci = 0;
        double v[D];
        if ((int)threadIdx.x < cnt) {
            ci = qs[q];
            double Ac[D * D], bc[D];
            int piv[D];
            load(ci, Ac, bc);
            if (dev_cond1<D>(Ac, piv) <= kCondEps) {
                dev_lu_solve<D>(Ac, piv, bc, v);
                keep = true;
            }
        }
        ns -= cnt;
        push(keep, false, ci, v);
    };
    for (int base = 0; base < nc; base += T) {
        const int ci = base + (int)threadIdx.x;
        bool keep = false, slow = false;
        double v[D];
        if (ci < nc) {
            double Ac[D * D], bc[D];
            int piv[D];
            load(ci, Ac, bc);
            const double na1 = dev_one_norm<D>(Ac);
            double rn = 0;
#pragma unroll
            for (int r = 0; r < D; r++) {
                double sr = 0;
#pragma unroll
                for (int c = 0; c < D; c++) sr += fabs(Ac[r * D + c]);
                rn = fmax(rn, sr);
            }
            if (dev_lu<D>(Ac, piv)) {
                double det = 1.0, bnd = na1 * (double)D;
#pragma unroll
                for (int k = 0; k < D; k++) det *= fabs(Ac[k * D + k]);
#pragma unroll
                for (int k = 0; k < D - 1; k++) bnd *= rn;
                if (bnd <= kCondScreen * det) {
                    dev_lu_solve<D>(Ac, piv, bc, v);
                    keep = true;
                } else if (!(na1 * (1.0 / fabs(Ac[D * D - 1])) > kCondEps)) {
                    slow = true;
                }
            }
        }
        push(keep, slow, ci, v);
        if (na >= T) drain(T);
        if (ns >= T) {
            settle(T);
            if (na >= T) drain(T);
        }
    }
    if (ns > 0) settle(ns);
    while (na > 0) drain(min(na, T));
    __syncthreads();
    // keep sign vectors whose parent part is a cell of the parent arrangement
    const uint32_t top_phc = 1u << (phc - 1), rev_phc = (phc >= 32) ? 0xffffffffu : ((1u << phc) - 1u);
    const uint32_t valid_mask = (m >= 5) ? 0xffffffffu : ((1u << (1 << m)) - 1u);
    for (int w = threadIdx.x; w < W; w += blockDim.x) {
        uint32_t x = bits[w] & valid_mask, keep = 0;
        while (x) {
            const int bt = __ffs(x) - 1;
            x &= x - 1;
            uint32_t psv = ((uint32_t)(w * 32 + bt)) & rev_phc;
            if (psv & top_phc) psv ^= rev_phc;
            bool in_parent;
            if (!psearch) {
                in_parent = (pbits[psv >> 5] >> (psv & 31)) & 1u;
            } else {
                int lo = 0, hi = gn;  // first key >= psv
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (gk[mid] < psv) lo = mid + 1;
                    else hi = mid;
                }
                in_parent = lo < gn && gk[lo] == psv;
            }
            if (in_parent) keep |= (1u << bt);
        }
        bits[w] = keep;
    }
    __syncthreads();
    // antipodal pairs; the half-storage representative has bit m-1 clear
    const uint32_t rev_m = (m >= 32) ? 0xffffffffu : ((1u << m) - 1u);
    const int nlow = 1 << (m - 1);  // candidate keys [0, 2^(m-1))
    const int WL = (nlow + 31) >> 5;
    const int per = (WL + blockDim.x - 1) / blockDim.x;
    const int w0 = threadIdx.x * per, w1 = min(WL, w0 + per);
    int cnt = 0;
    for (int w = w0; w < w1; w++) {
        uint32_t x = bits[w];
        if (nlow < 32) x &= (1u << nlow) - 1u;
        while (x) {
            const int bt = __ffs(x) - 1;
            x &= x - 1;
            const uint32_t sv = (uint32_t)(w * 32 + bt);
            const uint32_t pr = sv ^ rev_m;
            if ((bits[pr >> 5] >> (pr & 31)) & 1u) cnt++;
        }
    }
    int total;
    int pos = block4_excl_scan(cnt, &total, wsum);
    uint32_t* out = Barena + P.bt_off[i];
    const int cap = btcap[i];
    for (int w = w0; w < w1; w++) {
        uint32_t x = bits[w];
        if (nlow < 32) x &= (1u << nlow) - 1u;
        while (x) {
            const int bt = __ffs(x) - 1;
            x &= x - 1;
            const uint32_t sv = (uint32_t)(w * 32 + bt);
            const uint32_t pr = sv ^ rev_m;
            if ((bits[pr >> 5] >> (pr & 31)) & 1u) {
                if (pos < cap) out[pos] = sv;
                pos++;
            }
        }
    }
    if (threadIdx.x == 0) {
        P.bt_n[i] = min(total, cap);
        if (total > cap) atomicOr(err, 8);
    }
}

// ------------------------------------------------------------------ g evaluation helpers
// g value and y_ei of one term at the estimator's root point, cauchy_term.hpp:312-401.
template <int D>
__device__ inline cplx dev_eval_g_yei(const double* A, const double* p, const double* b, double c, double dv, int m,
                                      uint32_t hf, int phc, int z, int lhp, const uint32_t* gk, const cplx* gv,
                                      int gn, const double* root, bool first, double* ty) {
    for (int k = 0; k < D; k++) ty[k] = 0.0;
    double ygi = 0.0;
    uint32_t neg = 0;
    for (int l = 0; l < m; l++) {
        const double s = dev_dot<D>(A + l * D, root) > 0 ? 1 : -1;
        if (s < 0) neg |= (1u << l);
        const double scl = p[l] * s;
        for (int k = 0; k < D; k++) ty[k] += scl * A[l * D + k];
        if (!((hf >> l) & 1u)) ygi += p[l] * s;
    }
    cplx gp, gm;
    if (first) {
        gp = cmake(1, 0);
        gm = cmake(1, 0);
    } else {
        const int top = 1 << (phc - 1), rev = (phc >= 32) ? -1 : ((1 << phc) - 1);
        int lp = 0, lmv = 0, k = 0;
        for (int l = 0; l < m; l++) {
            if (k < phc) {
                if (k == z) {
                    lmv |= (1 << k);
                    k++;
                    if (k == phc) continue;
                }
                if ((neg >> l) & 1u) {
                    lp |= (1 << k);
                    lmv |= (1 << k);
                }
                k++;
            }
        }
        gp = lookup_num(lp ^ lhp, top, rev, gk, gv, gn);
        gm = lookup_num(lmv ^ lhp, top, rev, gk, gv, gn);
    }
    cplx g = csub(cdiv(gp, cmake(ygi + dv, c)), cdiv(gm, cmake(ygi - dv, c)));
    return cscale(g, kInvTwoPi);
}

// Measurement-update coalignment in place, cauchy_term.hpp:533-745.  Returns the
// new shape; sets *cm when hyperplanes were merged (c_map kept).
template <int D>
__device__ inline int dev_mu_coalign(double* A, double* p, double* q, uint8_t* cmap, int8_t* csmap, uint32_t* hfp,
                                     int m, int* err) {
    for (int r = 0; r < m; r++) {
        q[r] = p[r];
        double n1 = 0;
        for (int k = 0; k < D; k++) n1 += fabs(A[r * D + k]);
        p[r] *= n1;
        for (int k = 0; k < D; k++) A[r * D + k] /= n1;
        cmap[r] = 255;
        csmap[r] = 1;
    }
    const uint32_t hf = *hfp;
    uint32_t hu = hf;
    uint32_t F = (m >= 32) ? 0xffffffffu : ((1u << m) - 1u);
    int u = 0;
    for (int j = 0; j < m - 1; j++) {
        if (!((F >> j) & 1u)) continue;
        cmap[j] = (uint8_t)u;
        for (int k = j + 1; k < m; k++) {
            if (!((F >> k) & 1u)) continue;
            bool pos, neg;
            coalign_gates(A + j * D, A + k * D, D, pos, neg);
            if (pos) {
                if (hf) {
                    const bool hj = (hu >> j) & 1u, hk = (hu >> k) & 1u;
                    if (!hj && !hk) q[j] += q[k];
                    else if (hj && !hk) {
                        q[j] = q[k];
                        hu &= ~(1u << j);
                    } else if (!hj && hk) {
                        hu &= ~(1u << k);
                    } else {
                        hu &= ~(1u << k);
                        q[j] += q[k];
                    }
                } else {
                    q[j] += q[k];
                }
                F &= ~(1u << k);
                p[j] += p[k];
                cmap[k] = (uint8_t)u;
                csmap[k] = 1;
            }
            if (neg) {
                if (hf) {
                    const bool hj = (hu >> j) & 1u, hk = (hu >> k) & 1u;
                    if (!hj && !hk) q[j] -= q[k];
                    else if (hj && !hk) {
                        q[j] = -q[k];
                        hu &= ~(1u << j);
                    } else if (!hj && hk) {
                        hu &= ~(1u << k);
                    } else {
                        atomicOr(err, 1);  // the reference exits here (cauchy_term.hpp:676-685)
                    }
                } else {
                    q[j] -= q[k];
                }
                F &= ~(1u << k);
                p[j] += p[k];
                cmap[k] = (uint8_t)u;
                csmap[k] = -1;
            }
        }
        u += 1;
    }
    if ((F >> (m - 1)) & 1u) cmap[m - 1] = (uint8_t)u;
    const int ns = __popc(F);
    if (ns != m) {
        int w = 1;
        for (int j = 1; j < m; j++)
            if ((F >> j) & 1u) {
                if (w < j) {
                    for (int k = 0; k < D; k++) A[w * D + k] = A[j * D + k];
                    p[w] = p[j];
                    q[w] = q[j];
                }
                w++;
            }
        if (hf) {
            uint32_t nh = 0;
            int cc = 0;
            for (int j = 0; j < m; j++)
                if ((F >> j) & 1u) nh |= (((hu >> j) & 1u) << cc++);
            *hfp = nh;
        }
    }
    return ns;
}

// ------------------------------------------------------------------ moment chains
// Moment sums run in the reference's exact order.  Reference thread t owns parents
// i = t, t+T, ... of every shape bucket (cauchy_estimator.hpp:1575-1604) and adds,
// per parent, the parent's own term before its children (cache_moments,
// cauchy_estimator.hpp:307-338 and 1436-1468): chain t is the output slots (parent first) of
// its parents in order.  The measurement update writes a slot's moment inputs at its chain's
// position, so the sums read them as they come; one chain (T == 1) is the slots themselves.
//
// rel[i]: slots of chain t before parent i's, len[t]: slots of the chain.  One workgroup per
// chain over its parents.  Sorting the slots by chain instead took three launches of a small
// update and a radix sort of every slot of a large one.
__device__ __forceinline__ void k_chain_pos(MG<1024, 1> mg, const int* __restrict__ slots,
                                            const StepConst* __restrict__ sc, int sr, int* __restrict__ rel,
                                            int* __restrict__ len) {
    __shared__ int cum[kMaxM + 2];  // parents of the chain in the buckets before each
    const int t = mg.bx, T = sc->T;
    if (threadIdx.x == 0) {
        int c = 0;
        for (int b = 0; b < sr; b++) {
            cum[b] = c;
            const int n = sc->in_off[b + 1] - sc->in_off[b];
            c += n > t ? (n - t - 1) / T + 1 : 0;
        }
        cum[sr] = c;
    }
    __syncthreads();
    const int n = cum[sr];
    int carry = 0;
    for (int q0 = 0; q0 < n; q0 += blockDim.x) {
        const int q = q0 + threadIdx.x;
        int i = -1;
        if (q < n) {
            int b = 0;
            while (cum[b + 1] <= q) b++;
            i = sc->in_off[b] + t + T * (q - cum[b]);
        }
        int total;
        const int x = block_excl_scan(i >= 0 ? slots[i] : 0, &total);
        if (i >= 0) rel[i] = carry + x;
        carry += total;
        __syncthreads();
    }
    if (threadIdx.x == 0) len[t] = carry;
}

// First position of chain t.
__device__ __forceinline__ int chain_begin(const int* __restrict__ len, int t) {
    int o = 0;
    for (int u = 0; u < t; u++) o += len[u];
    return o;
}

// Position of slot s, the ts-th of parent P of chain t.
__device__ __forceinline__ int64_t chain_pos(const StepConst* __restrict__ sc, const int* __restrict__ rel,
                                             const int* __restrict__ len, int t, int P, int s, int ts) {
    return sc->T > 1 ? chain_begin(len, t) + rel[P] + ts : s;
}

// ------------------------------------------------------------------ measurement update
// cauchy_term.hpp:84-310 (msmt_update) + cache_moments inputs + MU coalignment,
// one thread per output slot.  Slot t < m of parent P is its child t; slot m is
// the parent itself.  Writes the gather key (shape, reference thread, is_child)
// that reproduces the reference's term order (cauchy_estimator.hpp:898-937, 1683-1704).
template <int D>
__device__ __forceinline__ void k_mu(MG<1024, 1> mg, TermPool IN, int np, const int* __restrict__ slot_base, TermPool OUT, int nslots,
                     const StepConst* __restrict__ sc, const uint32_t* __restrict__ gk_prev,
                     const cplx* __restrict__ gv_prev, double* __restrict__ gy, uint32_t* __restrict__ keys_out,
                     const int* __restrict__ chain_rel, const int* __restrict__ chain_len, int* __restrict__ err) {
    const int s = mg.bx * blockDim.x + threadIdx.x;
    if (s >= nslots) return;
    int lo = 0, hi = np - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (slot_base[mid] <= s) lo = mid;
        else hi = mid - 1;
    }
    const int P = lo;
    const int MM = IN.MM;
    const int m = IN.m[P];
    // slot 0 of a parent holds the parent itself (child m), slots 1..m its children 0..m-1
    const int ts = s - slot_base[P];
    const int t = (ts == 0) ? m : ts - 1;
    const double* A = IN.A + (int64_t)P * MM * D;
    const double* p = IN.p + (int64_t)P * MM;
    const double* b = IN.b + (int64_t)P * D;
    const double* H = sc->H;
    uint32_t integ = 0, negs = 0;
    for (int l = 0; l < m; l++) {
        const double h = dev_dot<D>(H, A + l * D);
        if (!(fabs(h) < kMuEps)) {
            integ |= (1u << l);
            if (!(h > 0)) negs |= (1u << l);
        }
    }
    double* g_out = gy + chain_pos(sc, chain_rel, chain_len, IN.tid[P], P, s, ts) * (2 + 2 * D);
    if (t < m && !((integ >> t) & 1u)) {
        OUT.flags[s] = 0;
        keys_out[s] = kGatherKeyNone;
        for (int k = 0; k < 2 + 2 * D; k++) g_out[k] = 0.0;
        return;
    }
    const double zeta = sc->msmt - dev_dot<D>(H, b);
    double mut[D];
    double rho_t;
    if (t == m) {
        for (int k = 0; k < D; k++) mut[k] = 0.0;
        rho_t = sc->gamma;
    } else {
        const double h = dev_dot<D>(H, A + t * D);
        const double r = 1.0 / h;
        for (int k = 0; k < D; k++) mut[k] = A[t * D + k] * r;
        rho_t = p[t] * fabs(h);
    }
    double* oA = OUT.A + (int64_t)s * MM * D;
    double* op = OUT.p + (int64_t)s * MM;
    double* oq = OUT.q + (int64_t)s * MM;
    double* ob = OUT.b + (int64_t)s * D;
    for (int k = 0; k < D; k++) ob[k] = b[k] + zeta * mut[k];
    int lo_row = 0;
    uint32_t hf = 0;
    for (int ll = 0; ll <= m; ll++) {
        if (ll == t) continue;
        double rho;
        if (ll == m) {
            rho = sc->gamma;
            for (int k = 0; k < D; k++) oA[lo_row * D + k] = 0.0 - mut[k];
        } else {
            const double h = dev_dot<D>(H, A + ll * D);
            if (fabs(h) < kMuEps) {
                rho = p[ll];
                for (int k = 0; k < D; k++) oA[lo_row * D + k] = A[ll * D + k];
                hf |= (1u << lo_row);
            } else {
                const double r = 1.0 / h;
                rho = p[ll] * fabs(h);
                for (int k = 0; k < D; k++) oA[lo_row * D + k] = (A[ll * D + k] * r) - mut[k];
            }
        }
        op[lo_row] = rho;
        lo_row++;
    }
    const int phc = IN.phc[P];
    OUT.m[s] = m;
    OUT.c[s] = zeta;
    OUT.dv[s] = rho_t;
    OUT.phc[s] = phc;
    OUT.pbc[s] = m;
    OUT.z[s] = t;
    OUT.gp_off[s] = IN.gp_off[P];
    OUT.rk_off[s] = IN.rk_off[P];
    OUT.gp_n[s] = IN.gp_n[P];
    const uint32_t enc = negs;
    uint32_t lhp = enc;
    if (phc < m) lhp &= (1u << phc) - 1u;
    uint32_t sg = enc;
    const uint32_t rev_m = (m >= 32) ? 0xffffffffu : ((1u << m) - 1u);
    if (sg & (1u << (m - 1))) sg ^= rev_m;
    OUT.lhp[s] = (int)lhp;
    OUT.bt_off[s] = IN.bt_off[P];
    OUT.bt_n[s] = IN.bt_n[P];
    OUT.bt_sgn[s] = (int)sg;
    OUT.tid[s] = IN.tid[P];
    // moments: g and y_ei of this term (cache_moments, cauchy_estimator.hpp:307-338)
    {
        double ty[D];
        const int64_t go = IN.gp_off[P];
        const cplx g = dev_eval_g_yei<D>(oA, op, ob, zeta, rho_t, m, hf, phc, t, (int)lhp, gk_prev + go, gv_prev + go,
                                         IN.gp_n[P], sc->root, sc->first != 0, ty);
        g_out[0] = g.re;
        g_out[1] = g.im;
        for (int k = 0; k < D; k++) {
            g_out[2 + 2 * k] = -ty[k];
            g_out[3 + 2 * k] = ob[k];
        }
    }
    int mnew = m;
    uint8_t fl = kValid | ((t != m) ? kIsNew : 0);
    if (!sc->first) {
        uint8_t* cm = OUT.cmap + (int64_t)s * MM;
        int8_t* cs = OUT.csmap + (int64_t)s * MM;
        if (t == m) {
            for (int r = 0; r < m; r++) {
                oq[r] = op[r];
                double n1 = 0;
                for (int k = 0; k < D; k++) n1 += fabs(oA[r * D + k]);
                op[r] *= n1;
                for (int k = 0; k < D; k++) oA[r * D + k] /= n1;
            }
        } else {
            mnew = dev_mu_coalign<D>(oA, op, oq, cm, cs, &hf, m, err);
            if (mnew < m) fl |= kHasCmap;
        }
        bool nan_p = false;
        for (int r = 0; r < mnew; r++) nan_p |= op[r] != op[r];
        if (nan_p) atomicOr(err + (kCtrNanP - kCtrMuErr), 1);
    }
    OUT.hflag[s] = hf;
    OUT.flags[s] = fl;
    OUT.m[s] = mnew;
    keys_out[s] = (uint32_t)(((mnew * sc->T) + IN.tid[P]) * 2 + ((t != m) ? 1 : 0));
}

// Rows of the parents of one block of output slots, staged in LDS by k_mu_r and k_mu_last.
// Slot s of parent P is s - slot_base[P] in 0..m: 0 the parent itself, t + 1 its child t.
// A child's row r is parent row src (r below t, r + 1 from t on; src == m is the
// measurement-noise row) as mu_src - mu_t with mu_l = A_l / (H . A_l), so everything but a
// subtraction depends on the parent's row alone: mu_l, rho_l = p_l |H . A_l| and whether the
// row is H-orthogonal are formed once per parent and block here, where m + 1 threads each
// formed all of them (a product with H, a division and D products per row and slot) out of
// global memory.  Entry q holds row q - slot_base[P] of the parent that slot base0 + q belongs
// to (the last slot of each parent stands empty): a block's slots and the other slots of its
// first and last parent, at most 31 each.
constexpr int kMuThreads = 256;
constexpr int kMuRowCap = kMuThreads + 64;
template <int D>
struct MuRows {
    double mu[D][kMuRowCap];
    double rho[kMuRowCap];
    uint8_t cls[kMuRowCap];  // 0: H-orthogonal (mu holds A itself), 1: H . A > 0, 2: not
    int base0, last;         // first slot of the first parent, last parent
};

// Largest i in [0, n) with base[i] <= x (base ascending, base[0] <= x), by a whole wavefront:
// 64 probes a round, three rounds up to 262,144 entries, where a binary search has 18
// dependent loads.
__device__ __forceinline__ int wave_floor(const int* __restrict__ base, int n, int x) {
    const int lane = threadIdx.x & 63;
    int lo = 0, len = n;  // the answer lies in [lo, lo + len)
    while (len > 1) {
        const int step = (len + 63) >> 6;
        const int i = lane * step;
        const int cnt = __popcll(__ballot(i < len && base[lo + i] <= x));  // lane 0 always counts
        lo += (cnt - 1) * step;
        len = min(step, len - (cnt - 1) * step);
    }
    return lo;
}

// Stages the rows behind the block's slots [mg.bx * 256, + 256) and returns the parent of this
// thread's slot (of the last slot for threads past the end).  All threads of the block.
template <int D>
__device__ __forceinline__ int mu_stage(MuRows<D>& R, const TermPool& IN, int np, const int* __restrict__ slot_base,
                                        int s0, int nslots, const double* H) {
    const int tid = threadIdx.x;
    const int P0 = wave_floor(slot_base, np, s0);
    auto parent = [&](int lo, int hi, int x) {
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (slot_base[mid] <= x) lo = mid;
            else hi = mid - 1;
        }
        return lo;
    };
    const int sl = min(s0 + kMuThreads, nslots) - 1;
    const int P = parent(P0, min(np - 1, P0 + kMuThreads - 1), min(s0 + tid, sl));
    if (s0 + tid == sl) R.last = P;
    if (tid == 0) R.base0 = slot_base[P0];
    __syncthreads();
    const int base0 = R.base0, Pl = R.last;
    const int end = slot_base[Pl + 1];
    const int MM = IN.MM;
    for (int q = base0 + tid; q < end; q += kMuThreads) {
        const int Q = parent(P0, Pl, q);
        const int l = q - slot_base[Q];
        if (l >= IN.m[Q] || q - base0 >= kMuRowCap) continue;
        const double* A = IN.A + ((int64_t)Q * MM + l) * D;
        double row[D];
#pragma unroll
        for (int k = 0; k < D; k++) row[k] = A[k];
        const double pl = IN.p[(int64_t)Q * MM + l];
        const double h = dev_dot<D>(H, row);
        const int i = q - base0;
        if (fabs(h) < kMuEps) {
            R.cls[i] = 0;
            R.rho[i] = pl;
        } else {
            const double r = 1.0 / h;
            R.cls[i] = h > 0 ? 1 : 2;
            R.rho[i] = pl * fabs(h);
#pragma unroll
            for (int k = 0; k < D; k++) row[k] *= r;
        }
#pragma unroll
        for (int k = 0; k < D; k++) R.mu[k][i] = row[k];
    }
    __syncthreads();
    return P;
}

// Masks of the parent's rows: integ has the rows that are not H-orthogonal, the result those
// of them with H . A not positive.
template <int D>
__device__ __forceinline__ uint32_t mu_masks(const MuRows<D>& R, int i0, int m, uint32_t* integ) {
    uint32_t in = 0, neg = 0;
    for (int l = 0; l < m; l++) {
        const int c = R.cls[i0 + l];
        in |= (uint32_t)(c != 0) << l;
        neg |= (uint32_t)(c == 2) << l;
    }
    *integ = in;
    return neg;
}

// Row r of child t from the staged rows; returns its p.
template <int D>
__device__ __forceinline__ double mu_row(const MuRows<D>& R, int i0, const double* mut, double gamma, int m, int t,
                                         int r, double* row, bool* horth) {
    const int src = (t < m && r >= t) ? r + 1 : r;
    if (src == m) {
#pragma unroll
        for (int k = 0; k < D; k++) row[k] = 0.0 - mut[k];
        *horth = false;
        return gamma;
    }
    const int i = i0 + src;
    *horth = R.cls[i] == 0;
#pragma unroll
    for (int k = 0; k < D; k++) {
        const double v = R.mu[k][i];
        row[k] = *horth ? v : v - mut[k];
    }
    return R.rho[i];
}

// row /= n1, to the same bits: the steps a double division takes (two Newton steps on the
// estimate of 1 / n1, the product, one correction by its exact remainder; Markstein, IBM
// J. Res. Dev. 34, 1990), with the estimate's part done once for the row's D quotients.
// Outside the range where no step can overflow or lose a subnormal's bits the row is divided
// as it stands.
template <int D>
__device__ __forceinline__ void div_row(double* row, double n1) {
    bool plain = n1 > 1e-120 && n1 < 1e120;
#pragma unroll
    for (int k = 0; k < D; k++) plain &= row[k] == 0.0 || fabs(row[k]) > 1e-150;
    if (plain) {
        double y = __builtin_amdgcn_rcp(n1);
        y = __builtin_fma(__builtin_fma(-n1, y, 1.0), y, y);
        y = __builtin_fma(__builtin_fma(-n1, y, 1.0), y, y);
#pragma unroll
        for (int k = 0; k < D; k++) {
            const double q = row[k] * y;
            const double v = __builtin_fma(__builtin_fma(-n1, q, row[k]), y, q);
            row[k] = row[k] == 0.0 ? row[k] : v;
        }
    } else {
#pragma unroll
        for (int k = 0; k < D; k++) row[k] /= n1;
    }
}

// g and -Re y, Im y of one slot (eval_g_yei, cauchy_term.hpp:312-401) from its sums over the
// child rows: written where the moment sums read them.
template <int D>
__device__ __forceinline__ void mu_moment(const TermPool& IN, int P, bool first, int m, int t, uint32_t neg,
                                          uint32_t lhp, double ygi, double rho_t, double zeta, const double* ty,
                                          const double* cb, const uint32_t* __restrict__ gk_prev,
                                          const cplx* __restrict__ gv_prev, double* __restrict__ g_out) {
    cplx gpl, gmn;
    if (first) {
        gpl = cmake(1, 0);
        gmn = cmake(1, 0);
    } else {
        const int phc = IN.phc[P];
        const int top = 1 << (phc - 1), rev = (phc >= 32) ? -1 : ((1 << phc) - 1);
        int lp = 0, lmv = 0, kq = 0;
        for (int l = 0; l < m; l++) {
            if (kq < phc) {
                if (kq == t) {
                    lmv |= (1 << kq);
                    kq++;
                    if (kq == phc) continue;
                }
                if ((neg >> l) & 1u) {
                    lp |= (1 << kq);
                    lmv |= (1 << kq);
                }
                kq++;
            }
        }
        const int64_t go = IN.gp_off[P];
        gpl = lookup_num(lp ^ (int)lhp, top, rev, gk_prev + go, gv_prev + go, IN.gp_n[P]);
        gmn = lookup_num(lmv ^ (int)lhp, top, rev, gk_prev + go, gv_prev + go, IN.gp_n[P]);
    }
    const cplx g = cscale(csub(cdiv(gpl, cmake(ygi + rho_t, zeta)), cdiv(gmn, cmake(ygi - rho_t, zeta))), kInvTwoPi);
    g_out[0] = g.re;
    g_out[1] = g.im;
#pragma unroll
    for (int k = 0; k < D; k++) {
        g_out[2 + 2 * k] = -ty[k];
        g_out[3 + 2 * k] = cb[k];
    }
}

// Measurement update streamed row by row (KM >= m, compile-time bound).  The same
// operations in the same order as k_mu: each child row is built, enters the moment
// sums, is L1-normalised and written once; only the normalised first coordinates
// are kept, for the coalignment filter.  When the filter finds a possible merge (a
// rare case) the rows are rebuilt in memory and coaligned there, as k_mu does.
// Bound by its double-precision arithmetic: the row's share that does not depend on the
// child is staged (MuRows) and the normalisation's D divisions share a reciprocal.
template <int D, int KM>
__device__ __forceinline__ void k_mu_r(MG<256, 3> mg, TermPool IN, int np, const int* __restrict__ slot_base, TermPool OUT,
                                             int nslots, const StepConst* __restrict__ sc,
                                             const uint32_t* __restrict__ gk_prev, const cplx* __restrict__ gv_prev,
                                             double* __restrict__ gy, uint32_t* __restrict__ keys_out,
                                             const int* __restrict__ chain_rel, const int* __restrict__ chain_len,
                                             int* __restrict__ err) {
    __shared__ MuRows<D> R;
    const int s = mg.bx * kMuThreads + threadIdx.x;
    const int P = mu_stage<D>(R, IN, np, slot_base, mg.bx * kMuThreads, nslots, sc->H);
    if (s >= nslots) return;
    const int MM = IN.MM;
    const int m = IN.m[P];
    if (m > KM) {
        atomicOr(err, 2);
        return;
    }
    const int ts = s - slot_base[P];
    const int t = (ts == 0) ? m : ts - 1;
    const int i0 = slot_base[P] - R.base0;
    const double* b = IN.b + (int64_t)P * D;
    const double* H = sc->H;
    uint32_t integ;
    const uint32_t negs = mu_masks<D>(R, i0, m, &integ);
    double* g_out = gy + chain_pos(sc, chain_rel, chain_len, IN.tid[P], P, s, ts) * (2 + 2 * D);
    if (t < m && !((integ >> t) & 1u)) {
        OUT.flags[s] = 0;
        keys_out[s] = kGatherKeyNone;
        for (int kk = 0; kk < 2 + 2 * D; kk++) g_out[kk] = 0.0;
        return;
    }
    const double zeta = sc->msmt - dev_dot<D>(H, b);
    double mut[D];
#pragma unroll
    for (int kk = 0; kk < D; kk++) mut[kk] = t == m ? 0.0 : R.mu[kk][i0 + t];
    const double rho_t = t == m ? sc->gamma : R.rho[i0 + t];
    double cb[D];
#pragma unroll
    for (int kk = 0; kk < D; kk++) cb[kk] = b[kk] + zeta * mut[kk];
    const int phc = IN.phc[P];
    OUT.c[s] = zeta;
    OUT.dv[s] = rho_t;
    OUT.phc[s] = phc;
    OUT.pbc[s] = m;
    OUT.z[s] = t;
    OUT.gp_off[s] = IN.gp_off[P];
    OUT.rk_off[s] = IN.rk_off[P];
    OUT.gp_n[s] = IN.gp_n[P];
    const uint32_t enc = negs;
    uint32_t lhp = enc;
    if (phc < m) lhp &= (1u << phc) - 1u;
    uint32_t sg = enc;
    const uint32_t rev_m = (m >= 32) ? 0xffffffffu : ((1u << m) - 1u);
    if (sg & (1u << (m - 1))) sg ^= rev_m;
    OUT.lhp[s] = (int)lhp;
    OUT.bt_off[s] = IN.bt_off[P];
    OUT.bt_n[s] = IN.bt_n[P];
    OUT.bt_sgn[s] = (int)sg;
    OUT.tid[s] = IN.tid[P];
    double* ob = OUT.b + (int64_t)s * D;
#pragma unroll
    for (int kk = 0; kk < D; kk++) ob[kk] = cb[kk];
    double* oA = OUT.A + (int64_t)s * MM * D;
    double* op = OUT.p + (int64_t)s * MM;
    double* oq = OUT.q + (int64_t)s * MM;
    const bool normalise = !sc->first;
    // rows: moment contributions (eval_g_yei, cauchy_term.hpp:312-401), then
    // q <- p and the L1 normalisation (normalize_hps, cauchy_term.hpp:458-474)
    double ty[D];
#pragma unroll
    for (int kk = 0; kk < D; kk++) ty[kk] = 0.0;
    double ygi = 0.0;
    uint32_t neg = 0, hf = 0;
    bool nan_p = false;
    double x0[KM];
#pragma unroll
    for (int r = 0; r < KM; r++) {
        x0[r] = 0.0;
        if (r < m) {
            double row[D];
            bool ho;
            double pr = mu_row<D>(R, i0, mut, sc->gamma, m, t, r, row, &ho);
            if (ho) hf |= (1u << r);
            double dr = 0.0;
#pragma unroll
            for (int kk = 0; kk < D; kk++) dr += row[kk] * sc->root[kk];
            const double sgn = dr > 0 ? 1 : -1;
            if (sgn < 0) neg |= (1u << r);
            const double scl = pr * sgn;
#pragma unroll
            for (int kk = 0; kk < D; kk++) ty[kk] += scl * row[kk];
            if (!ho) ygi += pr * sgn;
            if (normalise) {
                double n1 = 0;
#pragma unroll
                for (int kk = 0; kk < D; kk++) n1 += fabs(row[kk]);
                oq[r] = pr;
                pr *= n1;
                nan_p |= pr != pr;
                div_row<D>(row, n1);
                x0[r] = fabs(row[0]);
            }
#pragma unroll
            for (int kk = 0; kk < D; kk++) oA[r * D + kk] = row[kk];
            op[r] = pr;
        }
    }
    mu_moment<D>(IN, P, sc->first != 0, m, t, neg, lhp, ygi, rho_t, zeta, ty, cb, gk_prev, gv_prev, g_out);
    int mnew = m;
    uint8_t fl = kValid | ((t != m) ? kIsNew : 0);
    if (normalise && t != m) {
        // Two normalised rows coalign (mu_coalign, cauchy_term.hpp:533-745) only if
        // |x_j - x_k| < eps or |x_j + x_k| < eps on every coordinate, so only if
        // ||x_j0| - |x_k0|| < eps on the first (in floating point the latter equals
        // one of the former exactly).  Without such a pair nothing merges.
        bool cand = false;
#pragma unroll
        for (int j = 0; j < KM - 1; j++)
#pragma unroll
            for (int kx = j + 1; kx < KM; kx++)
                if (kx < m && fabs(x0[j] - x0[kx]) < kCoalignEps) cand = true;
        uint8_t* cm = OUT.cmap + (int64_t)s * MM;
        int8_t* cs = OUT.csmap + (int64_t)s * MM;
        if (cand) {
            // possible merge: rebuild the rows as built before normalisation and run
            // the in-memory coalignment
            for (int r = 0; r < m; r++) {
                double row[D];
                bool ho;
                op[r] = mu_row<D>(R, i0, mut, sc->gamma, m, t, r, row, &ho);
#pragma unroll
                for (int kk = 0; kk < D; kk++) oA[r * D + kk] = row[kk];
            }
            mnew = dev_mu_coalign<D>(oA, op, oq, cm, cs, &hf, m, err);
            if (mnew < m) fl |= kHasCmap;
        } else {
            // a new child's maps are the identity
            for (int r = 0; r < m; r++) {
                cm[r] = (uint8_t)r;
                cs[r] = 1;
            }
        }
    }
    if (nan_p) atomicOr(err + (kCtrNanP - kCtrMuErr), 1);
    OUT.hflag[s] = hf;
    OUT.flags[s] = fl;
    OUT.m[s] = mnew;
    keys_out[s] = (uint32_t)(((mnew * sc->T) + IN.tid[P]) * 2 + ((t != m) ? 1 : 0));
}

// A window's last update: its terms are summed into the moments and not kept, so only the
// moment inputs and the shape of each slot are formed; the rows are never
// written, and the output pool holds nothing but flags and shapes.  The same operations in
// the same order as k_mu and k_mu_r for any shape.
template <int D>
__device__ __forceinline__ void k_mu_last(MG<256, 4> mg, TermPool IN, int np, const int* __restrict__ slot_base,
                                          uint8_t* __restrict__ flags, int* __restrict__ shape, int nslots,
                                          const StepConst* __restrict__ sc, const uint32_t* __restrict__ gk_prev,
                                          const cplx* __restrict__ gv_prev, double* __restrict__ gy,
                                          const int* __restrict__ chain_rel, const int* __restrict__ chain_len) {
    __shared__ MuRows<D> R;
    const int s = mg.bx * kMuThreads + threadIdx.x;
    const int P = mu_stage<D>(R, IN, np, slot_base, mg.bx * kMuThreads, nslots, sc->H);
    if (s >= nslots) return;
    const int m = IN.m[P];
    const int ts = s - slot_base[P];
    const int t = (ts == 0) ? m : ts - 1;
    const int i0 = slot_base[P] - R.base0;
    const double* b = IN.b + (int64_t)P * D;
    uint32_t integ;
    const uint32_t negs = mu_masks<D>(R, i0, m, &integ);
    double* g_out = gy + chain_pos(sc, chain_rel, chain_len, IN.tid[P], P, s, ts) * (2 + 2 * D);
    if (t < m && !((integ >> t) & 1u)) {
        flags[s] = 0;
        for (int k = 0; k < 2 + 2 * D; k++) g_out[k] = 0.0;
        return;
    }
    const double zeta = sc->msmt - dev_dot<D>(sc->H, b);
    double mut[D], cb[D], ty[D];
#pragma unroll
    for (int k = 0; k < D; k++) {
        mut[k] = t == m ? 0.0 : R.mu[k][i0 + t];
        cb[k] = b[k] + zeta * mut[k];
        ty[k] = 0.0;
    }
    const double rho_t = t == m ? sc->gamma : R.rho[i0 + t];
    const int phc = IN.phc[P];
    const uint32_t lhp = phc < m ? negs & ((1u << phc) - 1u) : negs;
    double ygi = 0.0;
    uint32_t neg = 0;
    for (int r = 0; r < m; r++) {
        double row[D];
        bool ho;
        const double pr = mu_row<D>(R, i0, mut, sc->gamma, m, t, r, row, &ho);
        double dr = 0.0;
#pragma unroll
        for (int k = 0; k < D; k++) dr += row[k] * sc->root[k];
        const double sgn = dr > 0 ? 1 : -1;
        if (sgn < 0) neg |= (1u << r);
        const double scl = pr * sgn;
#pragma unroll
        for (int k = 0; k < D; k++) ty[k] += scl * row[k];
        if (!ho) ygi += pr * sgn;
    }
    mu_moment<D>(IN, P, sc->first != 0, m, t, neg, lhp, ygi, rho_t, zeta, ty, cb, gk_prev, gv_prev, g_out);
    flags[s] = kValid | ((t != m) ? kIsNew : 0);
    shape[s] = m;
}

// ------------------------------------------------------------------ moments
constexpr int kSumCW = 16;    // doubles (twice the components) one workgroup sums
constexpr int kSumTP = 224;   // positions per LDS tile
constexpr int kSumWaves = 8;  // the adding wave and seven that form the summands
static_assert(kSumTP % 32 == 0, "the adding wave takes a full tile 32 positions at a time");
constexpr int kSumDepth = 3;  // tiles whose inputs are in flight in registers

template <int D>
__host__ __device__ constexpr int mom_blocks() {
    return (2 * (1 + D + D * D) + kSumCW - 1) / kSumCW;
}

// Moments after term reduction (debug mode), cauchy_term.hpp:403-433 (eval_g_yei_after_ftr)
// over every parent term: the sign vector of its hyperplanes at the root point (bit l set
// where A_l . root <= 0), y_j = -(sum_l (p_l s_l) A_lj) + i b_j, and g its own g-table's value
// at that sign vector.  Writes (g, y) per term in the layout k_mom_sum reads.
template <int D>
__device__ __forceinline__ void k_after_ftr_gy(MG<1024, 1> mg, const TermPool P, int n,
                                               const StepConst* __restrict__ sc, const uint32_t* __restrict__ gk,
                                               const cplx* __restrict__ gv, double* __restrict__ gy) {
    const int t = mg.bx * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const int m = P.m[t];
    const int MM = P.MM;
    const double* A = P.A + (int64_t)t * MM * D;
    const double* p = P.p + (int64_t)t * MM;
    const double* b = P.b + (int64_t)t * D;
    double tmp[D];
#pragma unroll
    for (int j = 0; j < D; j++) tmp[j] = 0.0;
    int enc = 0;
    for (int l = 0; l < m; l++) {
        double dp = 0.0;
#pragma unroll
        for (int k = 0; k < D; k++) dp += A[l * D + k] * sc->root[k];
        const double s = dp > 0 ? 1.0 : -1.0;
        const double w = p[l] * s;
#pragma unroll
        for (int j = 0; j < D; j++) tmp[j] += w * A[l * D + j];
        if (s < 0) enc |= 1 << l;
    }
    const int top = 1 << (m - 1);
    const int rev = (m >= 32) ? -1 : ((1 << m) - 1);
    const int64_t go = P.gp_off[t];
    const cplx g = lookup_num(enc, top, rev, gk + go, gv + go, P.gp_n[t]);
    double* rec = gy + (int64_t)t * (2 + 2 * D);
    rec[0] = g.re;
    rec[1] = g.im;
#pragma unroll
    for (int j = 0; j < D; j++) {
        rec[2 + 2 * j] = -tmp[j];
        rec[3 + 2 * j] = b[j];
    }
}

// In-order sums of g, g*y_j and the negated (g*y_j)*y_k over each chain (the reference
// subtracts the latter; a - b == a + (-b) exactly), with the reference's operations.  Grid
// (T, mom_blocks): a workgroup sums kSumCW doubles of chain blockIdx.x.  Seven waves form the
// summands of a tile of positions out of the slots' (g, y) and leave them in a two-tile LDS
// ring, with the inputs of the next kSumDepth tiles in flight; wave 0 adds, a lane per
// double, bound by the latency of dependent double-precision additions (the last
// update of a 5-state window, 1.45M slots in 8 chains of 62 doubles: 2.0 ms; 1.0 ms of summands
// written to memory and read back and 3.1 ms of sums before, whose adding wave waited for LDS
// reads under a condition).
// Slots without a term hold zeros and add +-0.0, which leaves a sum that starts at +0.0
// unchanged; padding is +0.0.  part[t][c] receives the sum of chain t, and part[T * NC2] the
// measurement update's error bits (*mu_err), so one copy brings both back.  `len` is not read
// when T == 1: the chain is all n slots.
template <int D>
__device__ __forceinline__ void k_mom_sum(MG<64 * kSumWaves, 2> mg, const double* __restrict__ gy,
                                          const int* __restrict__ len, int T, int n, double* __restrict__ part,
                                          const int* __restrict__ mu_err) {
    constexpr int NS = 2 + 2 * D;
    constexpr int NC = 1 + D + D * D;
    constexpr int CB = kSumCW / 2;                        // components of the workgroup
    constexpr int PT = 64 * (kSumWaves - 1) / CB;         // positions the producers take at once
    constexpr int PER = kSumTP / PT;                      // ... and times per tile
    static_assert(PER * PT == kSumTP, "a tile is an exact multiple of the producers");
    __shared__ __align__(16) double ring[2][kSumTP * kSumCW];
    const int t = mg.bx;
    const int yb = mg.by;
    const int tid = threadIdx.x;
    if (t == 0 && yb == 0 && tid == 0) part[(int64_t)T * 2 * NC] = (double)mu_err[0];
    const int beg = T > 1 ? chain_begin(len, t) : 0;
    const int cnt = T > 1 ? len[t] : n;
    const int ntiles = (cnt + kSumTP - 1) / kSumTP;
    const bool adder = __builtin_amdgcn_readfirstlane(tid >> 6) == 0;
    // LDS-only barrier: global loads stay in flight across it
    auto lds_barrier = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };
    // The two roles run separate loops; each performs exactly nsteps + 1 barriers.  The step
    // count is padded to a multiple of kSumDepth so that every unrolled step is unconditional
    // (the compiler then keeps the later tiles' loads in flight).
    const int nsteps = (ntiles + kSumDepth - 1) / kSumDepth * kSumDepth;
    if (!adder) {
        const int l = tid - 64;
        const int c = l % CB, p0 = l / CB;
        const int cc = yb * CB + c;
        // operands of this thread's component: g, y_j where jo, y_k where ko
        const bool live = cc < NC, jo = live && cc > 0, ko = live && cc > D;
        const int j = !jo ? 0 : ko ? (cc - 1 - D) / D : cc - 1, k = ko ? (cc - 1 - D) % D : 0;
        const double* base = gy + (int64_t)beg * NS;
        double2 rg[kSumDepth][PER], rj[kSumDepth][PER], rk[kSumDepth][PER];
        // Loads are unconditional (position clamped into the chain) so that no load is
        // skipped and the wait for the oldest tile stays exact.
        auto load = [&](int u, int tile) {
#pragma unroll
            for (int q = 0; q < PER; q++) {
                const int pos = min(tile * kSumTP + q * PT + p0, cnt - 1);
                const double* rec = base + (int64_t)pos * NS;
                rg[u][q] = *(const double2*)rec;
                rj[u][q] = *(const double2*)(rec + 2 + 2 * j);
                rk[u][q] = *(const double2*)(rec + 2 + 2 * k);
            }
        };
        auto form = [&](int u, int tile, double* dst) {
#pragma unroll
            for (int q = 0; q < PER; q++) {
                const int pos = q * PT + p0;
                cplx x = cmake(rg[u][q].x, rg[u][q].y);
                const cplx xj = cmul(x, cmake(rj[u][q].x, rj[u][q].y));
                if (jo) x = xj;
                const cplx xk = cmul(x, cmake(rk[u][q].x, rk[u][q].y));
                if (ko) x = cmake(-xk.re, -xk.im);
                if (!live || tile * kSumTP + pos >= cnt) x = cmake(0.0, 0.0);
                *(double2*)(dst + pos * kSumCW + 2 * c) = make_double2(x.re, x.im);
            }
        };
        if (nsteps > 0) {
#pragma unroll
            for (int u = 0; u < kSumDepth; u++) load(u, u);
            form(0, 0, ring[0]);
            load(0, kSumDepth);
        }
        lds_barrier();
        for (int k0 = 0; k0 < nsteps; k0 += kSumDepth) {
#pragma unroll
            for (int u = 0; u < kSumDepth; u++) {
                const int s = k0 + u;
                // u is a compile-time index once the loop is unrolled
                form((u + 1) % kSumDepth, s + 1, ring[(s + 1) & 1]);
                load((u + 1) % kSumDepth, s + 1 + kSumDepth);
                lds_barrier();
            }
        }
    } else {
        const int lane = tid;
        double acc = 0.0;
        lds_barrier();
        for (int s = 0; s < nsteps; s++) {
            if (lane < kSumCW && s < ntiles) {
                const double* src = ring[s & 1] + lane;
                const int left = cnt - s * kSumTP;
                double ev[16], od[16];
                auto take = [&](double (&v)[16], int blk) {
#pragma unroll
                    for (int q = 0; q < 16; q++) v[q] = src[(blk * 16 + q) * kSumCW];
                };
                auto add = [&](const double (&v)[16]) {
#pragma unroll
                    for (int q = 0; q < 16; q++) acc += v[q];
                };
                if (left >= kSumTP) {
                    // reads of the next 16 summands are always in flight, none of them under
                    // a condition, so the additions wait for nothing but each other
                    take(ev, 0);
                    for (int r = 0; r < kSumTP / 16; r += 2) {
                        take(od, r + 1);
                        add(ev);
                        take(ev, min(r + 2, kSumTP / 16 - 1));
                        add(od);
                    }
                } else {
                    for (int r = 0; r * 16 < left; r++) {
                        take(ev, r);
                        add(ev);
                    }
                }
            }
            lds_barrier();
        }
        const int c2 = yb * kSumCW + lane;
        if (lane < kSumCW && c2 < 2 * NC) part[(int64_t)t * 2 * NC + c2] = acc;
    }
}

// Histogram of small integer values privatised in LDS (nbins <= 64).  mode 0: valid
// slots by shape; mode 1: surviving groups by shape.
__device__ __forceinline__ void k_hist(MG<1024, 1> mg, int n, int nbins, int mode, const uint8_t* __restrict__ flags, const int* __restrict__ vals,
                       const int* __restrict__ surv, int* __restrict__ hist) {
    __shared__ int h[64];
    for (int b = threadIdx.x; b < nbins; b += blockDim.x) h[b] = 0;
    __syncthreads();
    for (int i = mg.bx * blockDim.x + threadIdx.x; i < n; i += mg.gx * blockDim.x) {
        int v = -1;
        if (mode == 0) {
            if (flags[i] & kValid) v = vals[i];
        } else if (surv[i] >= 0) {
            v = vals[i];
        }
        if (v >= 0 && v < nbins) atomicAdd(&h[v], 1);
    }
    __syncthreads();
    for (int b = threadIdx.x; b < nbins; b += blockDim.x)
        if (h[b]) atomicAdd(&hist[b], h[b]);
}

// ------------------------------------------------------------------ gather
__device__ __forceinline__ void k_iota(MG<1024, 1> mg, uint32_t* __restrict__ v, int n) {
    const int i = mg.bx * blockDim.x + threadIdx.x;
    if (i < n) v[i] = (uint32_t)i;
}

// ------------------------------------------------------------------ fills
// Up to kFillRegions byte fills in one launch: region blockIdx.y gets `bytes` copies of
// `val`, by 32-bit words where the pointer allows, then the tail bytes.
constexpr int kFillRegions = 6;
struct FillArgs {
    uint8_t* ptr[kFillRegions];
    int64_t bytes[kFillRegions];
    uint32_t val[kFillRegions];
};
__device__ __forceinline__ void k_fill_multi(MG<1024, 1> mg, FillArgs f) {
    const int k = mg.by;
    uint8_t* p = f.ptr[k];
    const int64_t nb = f.bytes[k];
    const uint32_t v = f.val[k] & 0xffu;
    const int64_t stride = (int64_t)mg.gx * blockDim.x;
    const int64_t t = (int64_t)mg.bx * blockDim.x + threadIdx.x;
    int64_t words = 0;
    if (((uintptr_t)p & 3) == 0) {
        words = nb / 4;
        uint32_t* w = (uint32_t*)p;
        const uint32_t v4 = v * 0x01010101u;
        for (int64_t i = t; i < words; i += stride) w[i] = v4;
    }
    for (int64_t i = 4 * words + t; i < nb; i += stride) p[i] = (uint8_t)v;
}

// ------------------------------------------------------------------ fast term reduction
// All shape buckets are reduced together.  Global position p in [0, N) indexes the
// gathered order (bucket m occupies [boff[m], boff[m+1]), slot perm[p]); reduction
// decisions use bucket-local indices, as the reference reduces each bucket on its own
// (fast_term_reduction_and_create_gtables, cauchy_estimator.hpp:1001-1137).
//
// The reference looks for the terms that term i claims among those near it on one axis.
// Many terms share that coordinate (children of one parent, long windows of few states), and
// the pairs of a shared coordinate grow with the square of their number.  Here the terms are
// sorted by one number that every compared quantity enters instead (k_ftr_keys): two terms
// that reduce differ by at most a known bound in it, so every reduction stays inside a run of
// sorted neighbours that are no further apart than that bound, a component.  Components are
// the reduction groups themselves unless scales come near the tolerances.  The greedy pass then
// runs inside each component, with the reference's own comparisons on the terms' values
// (ftr_edge), so what reduces with what is unchanged: the sort only decides which pairs are
// compared.
//   k_ftr_keys      sort key of each term
//   k_ftr_comp      components of up to one wavefront: greedy pass, chunk merge, member ranks
//   k_ftr_comp_big  the others, a wavefront or a workgroup each
//   k_ftr_emit      reduction groups and member lists, after a scan over the roots
// 718k terms of a 2-state, 20-hyperplane window: the pair search, its edge lists and the
// resolution rounds took 78 ms per window (3.3 ms per pair pass, 1.2 ms per edge pass).
__device__ inline int bucket_of(const int* __restrict__ boff, int nb, int p) {
    int lo = 0, hi = nb - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (boff[mid] <= p) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Chunk of local index l in a bucket of n terms: buckets above 10000 terms are reduced
// in 8 chunks of n/8 (the last takes the rest), term_reduction.hpp:651-681.
constexpr int kFtrChunkTerms = 10000;
constexpr int kFtrChunks = 8;
__device__ inline int ftr_chunk_of(int l, int n) {
    if (n <= kFtrChunkTerms) return 0;
    const int c = l / (n / kFtrChunks);
    return c > kFtrChunks - 1 ? kFtrChunks - 1 : c;
}

// Sort key: shape, then the sum over the d coordinates of b, the m scales p and the first m
// entries of A in magnitude of w_k x_k, each x_k in whole units of 2^-kFtrFracBits and each
// w_k in whole 1024ths of [1/2, 1), in units of 2^-26 on a ring of 2^kFtrValueBits.  All of it is
// integer arithmetic, so two keys are as far apart as their terms whatever the terms' magnitude:
// states in metres are told apart as well as states of order one, where a key that squashes large
// numbers together sees thousands of distinct terms as one component.  (A 2-state window of 8
// steps whose scales were all 1e5: 9296 of 13842 terms in components of up to 4102 with the
// squashed key, whose roots a workgroup takes one by one; 2373 in 3 here, as in units of one.)
// The w_k are spread over [1/2, 1) so that terms that only exchange values get different keys.
constexpr int kFtrValueBits = 34;
constexpr int kFtrKeyBits = kFtrValueBits + 5;
constexpr uint64_t kFtrValueMask = ((uint64_t)1 << kFtrValueBits) - 1;
constexpr int kFtrFracBits = 32;
constexpr int kFtrDropBits = kFtrFracBits + 10 - 26;  // from units of 2^-kFtrFracBits / 1024 to 2^-26
__host__ __device__ constexpr uint32_t ftr_weight(int k) {  // k + 1 golden ratios, the 9 bits after the point
    return 512u + (((uint32_t)(k + 1) * 0x9E3779B9u) >> 23);
}
// Compared quantities of terms that reduce differ by at most kReductionEps = 42.9 units, those
// of b by at most 2^-26 = 64 units (b + kReductionEps is rounded, which adds up to half of b's last
// place where that is below 2^-25, and nothing but b itself is inside the window of a larger b).
// From 2^28 on they only reduce if they are equal, and any function of their bits will do.
__host__ __device__ inline uint64_t ftr_units(double x) {
    if (fabs(x) < (double)(1 << 28)) return (uint64_t)(int64_t)floor(x * (double)((uint64_t)1 << kFtrFracBits));
    union {
        double d;
        uint64_t u;
    } v = {x};
    return v.u * 0x9E3779B97F4A7C15ull;
}
// A NaN in p compares as equal to anything (ftr_edge), which no key can express: when the
// measurement update saw one, p is left out of every key.
__host__ __device__ inline uint64_t ftr_key(const double* b, const double* p, const double* A, int d, int m,
                                            const int* order, bool with_p) {
    uint64_t v = 0;
    for (int a = 0; a < d; a++) v += ftr_weight(a) * ftr_units(b[order[a]]);
    for (int k = 0; k < m; k++) {
        if (with_p) v += ftr_weight(d + 2 * k) * ftr_units(p[k]);
        v += ftr_weight(d + 2 * k + 1) * ftr_units(fabs(A[k]));
    }
    return ((uint64_t)m << kFtrValueBits) | ((v >> kFtrDropBits) & kFtrValueMask);
}
// Largest distance of the keys of two terms of shape m that reduce.  n weights in a row add up to
// at most 768 n + 512.
__host__ __device__ constexpr uint64_t ftr_link(int d, int m) {
    return (((768u * d + 512u) * 64u + (768u * 2u * m + 512u) * 43u) >> kFtrDropBits) + 1u;
}
constexpr bool ftr_weights_bounded() {
    for (int i = 0; i <= kMaxD; i++) {
        uint32_t sum = 0;
        for (int n = 1; i + n <= kMaxD + 2 * kMaxM; n++) {
            sum += ftr_weight(i + n - 1);
            if (sum > 768u * n + 512u) return false;
        }
    }
    return true;
}
static_assert(ftr_weights_bounded(), "ftr_link relies on it");

template <int D>
__device__ __forceinline__ void k_ftr_keys(MG<256, 1> mg, const TermPool OUT, const uint32_t* __restrict__ perm, int n,
                                           const int* __restrict__ boff, int nb, const StepConst* __restrict__ sc,
                                           const int* __restrict__ nan_p, uint64_t* __restrict__ keys,
                                           uint32_t* __restrict__ idx) {
    const int p = mg.bx * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const int64_t s = perm[p];
    keys[p] = ftr_key(OUT.b + s * D, OUT.p + s * OUT.MM, OUT.A + s * OUT.MM * D, D, bucket_of(boff, nb, p), sc->order,
                      *nan_p == 0);
    idx[p] = (uint32_t)p;
}

__device__ __forceinline__ int ftr_shape(uint64_t key) { return (int)(key >> kFtrValueBits); }

// Whether sorted neighbours belong to one component.
template <int D>
__device__ __forceinline__ bool ftr_linked(uint64_t prev, uint64_t cur) {
    const int m = ftr_shape(cur);
    return ftr_shape(prev) == m && cur - prev <= ftr_link(D, m);
}

// Whether two keys of shape m are near enough for their terms to reduce.
template <int D>
__device__ __forceinline__ bool ftr_near(uint64_t a, uint64_t b, int m) {
    const uint64_t x = (a - b) & kFtrValueMask;
    return x <= ftr_link(D, m) || kFtrValueMask + 1 - x <= ftr_link(D, m);
}

// Whether the last and the first key of a shape are neighbours on the ring: the run at the
// bucket's end goes on at its beginning.  (They are different runs: one around the whole ring
// would need 2^kFtrValueBits / ftr_link terms of a shape, which no device holds.)
template <int D>
__device__ __forceinline__ bool ftr_joined(uint64_t first, uint64_t last) {
    return ((first - last) & kFtrValueMask) <= ftr_link(D, ftr_shape(first)) && first != last;
}

// Whether term si (earlier) claims term sj (later) of shape m, term_reduction.hpp:89-276:
// b_j inside (b_i - ep, b_i + ep] on every axis, |p_j - p_i| <= ep on the first m, and the
// element-wise check over the first m flattened entries of A.
template <int D>
__device__ inline bool ftr_edge(const TermPool& O, int64_t si, int64_t sj, int m, const StepConst* __restrict__ sc,
                                const uint32_t* __restrict__ perm, int beg, int end) {
    const double ep = kReductionEps;
    const double* bi = O.b + si * D;
    const double* bj = O.b + sj * D;
    bool ok = true;
#pragma unroll
    for (int a = 0; a < D; a++) {
        const int ax = sc->order[a];
        const double v = bi[ax], x = bj[ax];
        ok &= x > v - ep && x <= v + ep;
    }
    if (!ok) return false;
    const double* pi = O.p + si * O.MM;
    const double* pj = O.p + sj * O.MM;
    const double* Ai = O.A + si * O.MM * D;
    const double* Aj = O.A + sj * O.MM * D;
    for (int k = 0; k < m; k++) {
        const double x = Ai[k], y = Aj[k];
        ok &= !(fabs(pj[k] - pi[k]) > ep) && (fabs(x - y) < ep || fabs(x + y) < ep);
    }
    if (!ok) return false;
    // The window on the first axis must hold two points.  It holds i and j, unless b_i - ep
    // rounds to b_i (magnitudes above 2^27), where i itself is outside its window.
    const int a0 = sc->order[0];
    const double v = bi[a0], lo = v - ep, hi = v + ep;
    if (!(v > lo)) {
        int c = 0;
        for (int p = beg; p < end && c < 2; p++) {
            const double x = O.b[(int64_t)perm[p] * D + a0];
            c += x > lo && x <= hi;
        }
        return c >= 2;
    }
    return true;
}

// Components that begin in the first kCompOwn of 64 sorted positions are reduced by the
// wavefront that looks at these 64, a lane per term; the next wavefront begins kCompOwn
// positions on.  A component that does not end inside the 64, or that goes on at its bucket's
// beginning, goes to big_list (at most one of the former per wavefront, one of the latter per
// shape).  No list of all components is made or counted.
//
// Greedy pass: the least unclaimed term of a component is a root and claims every later
// unclaimed term that ftr_edge accepts.  In a bucket above kFtrChunkTerms terms each chunk c
// has its own pass (roots of chunk c claim terms of chunks >= c), and the eight results are
// merged pairwise, term_reduction.hpp:592-649: F_c[j] is the root claiming j, else j, every
// value of F_c is a fixed point of it, so a merge level is data parallel.  Roots, members and
// merges never leave a component.
constexpr int kCompOwn = 48;
// Reduces the components that begin in the first `own` of the 64 sorted positions from `base`
// (< n).  Returns the lanes at which those to be listed begin.
template <int D>
__device__ __forceinline__ uint64_t ftr_comp_wave(const TermPool& OUT, const uint32_t* __restrict__ perm, int n,
                                                  const int* __restrict__ boff, const StepConst* __restrict__ sc,
                                                  const uint64_t* __restrict__ skeys,
                                                  const uint32_t* __restrict__ sidx, int* __restrict__ rootpos,
                                                  int* __restrict__ rank, int64_t* __restrict__ gval, int base,
                                                  int own_starts) {
    const int lane = wave_lane();
    const int r = base + lane;
    const bool in = r < n;
    const uint64_t q = in ? skeys[r] : 0;
    const uint64_t before = in && r > 0 ? skeys[r - 1] : 0;
    const uint64_t beyond = base + kWave < n ? skeys[base + kWave] : 0;
    const bool start = !(in && r > 0 && ftr_linked<D>(before, q));  // past the end: a start
    const uint64_t starts = __ballot(start);
    const uint64_t upto = starts & (~0ull >> (kWave - 1 - lane));
    const int sb = upto ? kWave - 1 - __clzll((long long)upto) : -1;
    const uint64_t after = lane == kWave - 1 ? 0ull : starts >> (lane + 1);
    const int se = after ? lane + __ffsll((unsigned long long)after) : kWave;
    const int m = ftr_shape(q);
    // the first and the last term of a bucket (no shape is 0) whose ends are joined
    const uint64_t down = __shfl_down(q, 1, kWave);
    const bool head = in && ftr_shape(before) != m, tail = in && ftr_shape(lane == kWave - 1 ? beyond : down) != m;
    const bool joined = (head || tail) && ftr_joined<D>(skeys[boff[m]], skeys[boff[m + 1] - 1]);
    const uint64_t heads = __ballot(head && joined), tails = __ballot(tail && joined);
    const bool ends = base + kWave >= n || !ftr_linked<D>(__shfl(q, kWave - 1, kWave), beyond);
    const bool own = in && sb >= 0 && sb < own_starts;
    const bool closed = se < kWave || ends;
    const bool from_end = own && ((heads >> sb) & 1u), goes_on = own && ((tails >> (se - 1)) & 1u);
    // a bucket's last run takes in its first one
    const bool mine = own && closed && !from_end && !goes_on;
    const uint64_t listed = __ballot(own && lane == sb && !from_end && (!closed || goes_on));
    const int size = mine ? se - sb : 1;
    const uint64_t seg = mine ? ((se == kWave ? ~0ull : (1ull << se) - 1ull) & ~((1ull << sb) - 1ull)) : 0ull;
    const int p = mine ? (int)sidx[r] : INT_MAX;
    const int beg = mine ? boff[m] : 0, end = mine ? boff[m + 1] : 0;
    const int slot = mine ? (int)perm[p] : 0;
    const int last = mine ? se - 1 : lane;
    // one greedy pass over every component of the wavefront: `cand` may become roots, `open`
    // may be claimed; returns the lane of each lane's root (its own if unclaimed)
    auto greedy = [&](bool cand, bool open) {
        int f = lane;
        for (;;) {
            int v = cand ? p : INT_MAX;
#pragma unroll
            for (int o = 1; o < kWave; o <<= 1) {
                const int y = __shfl_up(v, o, kWave);
                if (lane - o >= sb) v = min(v, y);
            }
            const int mn = __shfl(v, last, kWave);
            const uint64_t roots = __ballot(cand && p == mn);
            if (!roots) return f;
            const uint64_t mr = roots & seg;
            const int rl = mr ? __ffsll((unsigned long long)mr) - 1 : lane;
            const int rs = __shfl(slot, rl, kWave);
            if (mr) {
                if (rl == lane) {
                    cand = open = false;
                } else if (open && p > mn && ftr_edge<D>(OUT, rs, slot, m, sc, perm, beg, end)) {
                    f = rl;
                    cand = open = false;
                }
            }
        }
    };
    const int nbk = end - beg;
    const bool multi = mine && size > 1;
    int f0;
    if (!__any(multi && nbk > kFtrChunkTerms)) {
        f0 = greedy(multi, multi);
    } else {
        const int c0 = multi ? ftr_chunk_of(p - beg, nbk) : -1;
        int F[kFtrChunks];
#pragma unroll
        for (int c = 0; c < kFtrChunks; c++) F[c] = __any(c0 == c) ? greedy(c0 == c, c0 >= c) : lane;
#pragma unroll
        for (int lvl = 0; lvl < 3; lvl++)
#pragma unroll
            for (int k = 0; k < (kFtrChunks >> (lvl + 1)); k++) {
                const int rt = k << (lvl + 1), cm = rt + (1 << lvl);
                const int f2 = F[cm];
                const int x = __shfl(F[rt], f2, kWave);
                if (nbk > kFtrChunkTerms && p - beg >= cm * (nbk / kFtrChunks) && f2 != lane && F[rt] == lane)
                    F[rt] = x == f2 ? f2 : x;
            }
        f0 = F[0];
    }
    // members of each root, and each member's rank among them
    int cnt = 0, less = 0;
    for (int k = 1; __any(k < size); k++) {
        int pl = lane + k;
        if (pl >= se) pl -= size;
        pl = k < size ? pl : lane;
        const int pf = __shfl(f0, pl, kWave), pp = __shfl(p, pl, kWave);
        if (k < size) {
            cnt += pf == lane;
            less += pf == f0 && pl != f0 && pp < p;
        }
    }
    const int rp = __shfl(p, f0, kWave);
    if (mine) {
        rootpos[p] = rp;
        rank[p] = less;
        gval[p] = ((int64_t)(f0 == lane) << 32) | (uint32_t)cnt;
    }
    return listed;
}

template <int D>
__device__ __forceinline__ void k_ftr_comp(MG<256, 1> mg, const TermPool OUT, const uint32_t* __restrict__ perm, int n,
                                           const int* __restrict__ boff, const StepConst* __restrict__ sc,
                                           const uint64_t* __restrict__ skeys, const uint32_t* __restrict__ sidx,
                                           int* __restrict__ rootpos, int* __restrict__ rank,
                                           int64_t* __restrict__ gval, int* __restrict__ big_count,
                                           int* __restrict__ big_list) {
    const int base = (mg.bx * (blockDim.x / kWave) + threadIdx.x / kWave) * kCompOwn;
    if (base >= n) return;
    const uint64_t listed =
        ftr_comp_wave<D>(OUT, perm, n, boff, sc, skeys, sidx, rootpos, rank, gval, base, kCompOwn);
    if ((listed >> wave_lane()) & 1u) big_list[atomicAdd(big_count, 1)] = base + wave_lane();
}

// LDS of one wavefront for a component of any size: up to kWave terms that may become roots
// together (key, b on the first two search axes, slot, place in term order, which of them each
// one claims; in the order of their keys, who they are and the entries with keys near theirs),
// and a sort pass's digit counts.
struct FtrLds {
    uint64_t key[kWave], row[kWave];
    double b0[kWave], b1[kWave];
    int slot[kWave], idx[kWave];
    int who[kWave], lo[kWave], hi[kWave];
    int base[kWave], cnt[kWave];
};

// The component that begins at sorted position r0 and ends before r1, of any size, by T
// threads: one wavefront, or (T > 64) a workgroup.  Positions beyond the bucket's end stand for
// those from its beginning on (a component across the ring's zero).
//
// The terms are brought into term order.  Then the first kWave unclaimed ones are taken at a
// time: which of them claims which follows from the pairs among them, and every later term looks
// at those roots among them whose keys are near its own, with most of what tells them apart in
// LDS.  The first time a single one is taken: a long window's largest components are one group.
// At last a stable sort by root leaves each group's members together and in order.  Bound by the
// latency of a pass's dependent loads and barriers, so a pass serves 64 roots.  Components whose
// terms all differ are few, but where the scales come near the tolerances, or rounding at
// large ones exceeds it, they hold thousands: with a pass and two barriers per root, and ranks by
// comparing all pairs, a 2-state window of 8 steps with scales of 1e-5 took 125 ms (10.0 ms here),
// with 1e6 66 ms (3.6 ms, most of it the key's), with 1 3.6 ms (3.6 ms).
//
// F: kFtrArrays arrays of n ints (8 where a bucket is reduced in chunks), O: kFtrOrders;
// the component has its own positions in each.
constexpr int kFtrArrays = 3;
constexpr int kFtrOrders = 3;
template <int D, int T>
__device__ __forceinline__ void ftr_comp_many(const TermPool& OUT, const uint32_t* __restrict__ perm, int n,
                                              const int* __restrict__ boff, const StepConst* __restrict__ sc,
                                              const uint64_t* __restrict__ skeys, const uint32_t* __restrict__ sidx,
                                              int* __restrict__ rootpos, int* __restrict__ rank,
                                              int64_t* __restrict__ gval, int* F, int* O, int r0, int r1, FtrLds* lds,
                                              int* wsum) {
    constexpr int kWaves = T / kWave;
    const int lane = wave_lane(), t = T == kWave ? lane : (int)threadIdx.x, w = t / kWave;
    FtrLds& L = lds[0];
    auto sync = [&]() {
        if constexpr (T == kWave) {
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
            __builtin_amdgcn_wave_barrier();
        } else {
            __syncthreads();
        }
    };
    // set flags before this thread's, and of all threads
    auto count = [&](bool flag, int* total) {
        const uint64_t b = __ballot(flag);
        int x = __popcll(b & ((1ull << lane) - 1ull)), all = __popcll(b);
        if constexpr (T > kWave) {
            __syncthreads();
            if (lane == 0) wsum[w] = all;
            __syncthreads();
            all = 0;
            for (int k = 0; k < kWaves; k++) {
                x += k < w ? wsum[k] : 0;
                all += wsum[k];
            }
        }
        *total = all;
        return x;
    };
    // the sum over all threads; what they wrote before is visible afterwards
    auto sum = [&](int v) {
        for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
        sync();
        if constexpr (T > kWave) {
            if (lane == 0) wsum[w] = v;
            __syncthreads();
            v = 0;
            for (int k = 0; k < kWaves; k++) v += wsum[k];
        }
        return v;
    };
    const uint64_t key0 = skeys[r0];
    const int m = ftr_shape(key0);
    const int beg = boff[m], end = boff[m + 1], nbk = end - beg;
    const int nc = nbk > kFtrChunkTerms ? kFtrChunks : 1, per = nbk / kFtrChunks;
    const int size = r1 - r0;
    // entry e of the component, and of its stretch of an array
    auto at = [&](int e) { return r0 + e < end ? r0 + e : r0 + e - nbk; };
    auto dist = [&](int e) { return (skeys[at(e)] - key0) & kFtrValueMask; };  // ascending
    // Stable sort of the entries of a by of(entry) < 2^bits, 6 bits a pass, through b; returns
    // the one that holds the result.
    auto sort = [&](int* a, int* b, int bits, auto of) {
        for (int shift = 0; shift < bits; shift += 6) {
            sync();
            if (t < kWave) L.base[t] = 0;
            sync();
            for (int i = t; i < size; i += T) atomicAdd(&L.base[(of(a[at(i)]) >> shift) & 63], 1);
            sync();
            if (t < kWave) {
                const int c = L.base[t];
                L.base[t] = wave_incl_scan(c) - c;
            }
            for (int i0 = 0; i0 < size; i0 += T) {
                const bool in = i0 + t < size;
                const int e = in ? a[at(i0 + t)] : 0;
                const int dg = in ? (of(e) >> shift) & 63 : 0;
                uint64_t same = __ballot(in);
                for (int k = 0; k < 6; k++) {
                    const uint64_t set = __ballot((dg >> k) & 1);
                    same &= (dg >> k) & 1 ? set : ~set;
                }
                const int before = __popcll(same & ((1ull << lane) - 1ull));
                lds[w].cnt[lane] = 0;
                sync();
                if (in && before == 0) lds[w].cnt[dg] = __popcll(same);
                sync();
                if (in) {
                    int o = L.base[dg] + before;
                    for (int k = 0; k < w; k++) o += lds[k].cnt[dg];
                    b[at(o)] = e;
                }
                sync();
                if (t < kWave)
                    for (int k = 0; k < kWaves; k++) L.base[t] += lds[k].cnt[t];
                sync();
            }
            int* const was = a;
            a = b;
            b = was;
        }
        sync();
        return a;
    };
    auto bits_of = [](int x) { return 32 - __clz(x); };

    // P: the entries in term order, place: each one's place in it.  Equal keys are in order
    // already, the sort was stable.
    int* const place = O + 2 * (int64_t)n;
    for (int e = t; e < size; e += T) O[at(e)] = e;
    const bool in_order = r1 <= end && key0 == skeys[r1 - 1];
    int* const P = in_order ? O : sort(O, O + n, bits_of(nbk - 1), [&](int e) { return (int)sidx[at(e)] - beg; });
    sync();
    for (int i = t; i < size; i += T) {
        place[at(P[at(i)])] = i;
        for (int c = 0; c < nc; c++) F[(int64_t)c * n + at(i)] = i;
    }
    auto term = [&](int i) { return (int)sidx[at(P[at(i)])]; };
    // whether a term with x0 and x1 on the first search axes may be claimed by candidate i
    const int a0 = sc->order[0], a1 = sc->order[D > 1 ? 1 : 0];
    auto window = [&](int i, double x0, double x1) {
        const double ep = kReductionEps, v0 = L.b0[i], v1 = L.b1[i];
        return x0 > v0 - ep && x0 <= v0 + ep && x1 > v1 - ep && x1 <= v1 + ep;
    };
    sync();
    if (t <= nc) {  // places of the chunks' first terms
        int lo = t == nc ? size : 0, hi = t == 0 ? 0 : size;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (term(mid) - beg < t * per) lo = mid + 1;
            else hi = mid;
        }
        L.base[t] = lo;
    }
    sync();
    int roots = 0;  // with one chunk: of the component
    for (int c = 0; c < nc; c++) {
        int* Fc = F + (int64_t)c * n;
        const int cb = L.base[c], ce = L.base[c + 1];
        int left = ce - cb;  // neither roots nor claimed
        int most = 1;
        for (int next = cb; left > 0; most = kWave) {
            // the first unclaimed terms, at most `most`
            int k = 0;
            for (; next < ce && k < most; next += T) {
                const int i = next + t;
                const bool un = i < ce && Fc[at(i)] == i;
                int found;
                const int x = k + count(un, &found);
                if (un && x < most) {
                    const int slot = (int)perm[term(i)];
                    L.idx[x] = i;
                    L.slot[x] = slot;
                    L.key[x] = skeys[at(P[at(i)])];
                    L.b0[x] = OUT.b[(int64_t)slot * D + a0];
                    L.b1[x] = OUT.b[(int64_t)slot * D + a1];
                }
                k += found;
            }
            k = min(k, most);
            sync();
            next = L.idx[k - 1] + 1;
            // the entries near each, and which of them claims which later one
            if (t < k) {
                const uint64_t d = (L.key[t] - key0) & kFtrValueMask, link = ftr_link(D, m);
                int place_of = 0;
                for (int i = 0; i < k; i++) {
                    const uint64_t di = (L.key[i] - key0) & kFtrValueMask;
                    place_of += di < d || (di == d && i < t);
                }
                int lo = 0, hi = most == 1 ? 0 : size;
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (dist(mid) + link < d) lo = mid + 1;
                    else hi = mid;
                }
                L.who[place_of] = t;
                L.lo[place_of] = lo;
                hi = size;
                while (lo < hi && most > 1) {
                    const int mid = (lo + hi) >> 1;
                    if (dist(mid) <= d + link) lo = mid + 1;
                    else hi = mid;
                }
                L.hi[place_of] = hi;
            }
            for (int i = w; i < k; i += kWaves) {
                const bool e = lane > i && lane < k && window(i, L.b0[lane], L.b1[lane]) &&
                               ftr_near<D>(L.key[i], L.key[lane], m) &&
                               ftr_edge<D>(OUT, L.slot[i], L.slot[lane], m, sc, perm, beg, end);
                const uint64_t row = __ballot(e);
                if (lane == 0) L.row[i] = row;
            }
            sync();
            uint64_t is_root = 0, claimed = 0;
            for (int i = 0; i < k; i++) {
                if ((claimed >> i) & 1u) continue;
                is_root |= 1ull << i;
                claimed |= L.row[i];
            }
            // the earliest root that has an edge to a term claims it; those near entry e are
            // the ones from the first that ends beyond it to the last that begins at or before it
            auto beyond = [&](const int* ends, int e) {
                int lo = 0, hi = k;
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (ends[mid] <= e) lo = mid + 1;
                    else hi = mid;
                }
                return lo;
            };
            int fewer = 0;
            for (int e = t; e < size; e += T) {
                const int j = place[at(e)];
                if (j <= L.idx[0] || Fc[at(j)] != j) continue;
                int s = beyond(L.hi, e);
                const int send = beyond(L.lo, e);
                if (s >= send) continue;
                const int64_t slot = perm[sidx[at(e)]];
                const double x0 = OUT.b[slot * D + a0], x1 = OUT.b[slot * D + a1];
                int f = j;
                for (; s < send; s++) {
                    const int i = L.who[s];
                    if (((is_root >> i) & 1u) && L.idx[i] < f && window(i, x0, x1) &&
                        ftr_edge<D>(OUT, L.slot[i], slot, m, sc, perm, beg, end))
                        f = L.idx[i];
                }
                if (f < j) {
                    Fc[at(j)] = f;
                    fewer += j < ce;
                }
            }
            left -= sum(fewer) + __popcll(is_root);
            roots += __popcll(is_root);
        }
    }
    for (int lvl = 0; nc > 1 && lvl < 3; lvl++) {
        sync();
        for (int k = 0; k < (kFtrChunks >> (lvl + 1)); k++) {
            const int rt = k << (lvl + 1), cm = rt + (1 << lvl);
            int* F1 = F + (int64_t)rt * n;
            const int* F2 = F + (int64_t)cm * n;
            for (int i = t; i < size; i += T) {
                if (term(i) - beg < cm * per) continue;
                const int f2 = F2[at(i)];
                if (f2 != i && F1[at(i)] == i) F1[at(i)] = F1[at(f2)] == f2 ? f2 : F1[at(f2)];
            }
        }
    }
    if (nc > 1) {
        sync();
        roots = 0;
        for (int i = t; i < size; i += T) roots += F[at(i)] == i;
        roots = sum(roots);
    }
    if (roots == 1) {
        const int pf = term(0);
        for (int i = t; i < size; i += T) {
            const int p = term(i);
            rootpos[p] = pf;
            rank[p] = max(i - 1, 0);
            gval[p] = i == 0 ? ((int64_t)1 << 32) | (uint32_t)(size - 1) : 0;
        }
        sync();
        return;
    }
    // groups: a root and its members, all later than it, in order
    int* Q = P == O ? O + n : O;
    int* const G = F + 2 * (int64_t)n;  // where each root's group begins
    for (int i = t; i < size; i += T) Q[at(i)] = i;
    Q = sort(Q, F + n, bits_of(size - 1), [&](int i) { return F[at(i)]; });
    sync();
    for (int x = t; x < size; x += T)
        if (F[at(Q[at(x)])] == Q[at(x)]) G[at(Q[at(x)])] = x;
    sync();
    for (int x = t; x < size; x += T) {
        const int i = Q[at(x)], f = F[at(i)], g = G[at(f)];
        const int p = term(i), pf = term(f);
        rootpos[p] = pf;
        rank[p] = i == f ? 0 : x - g - 1;
        if (i != f) gval[p] = 0;
        if (x + 1 == size || F[at(Q[at(x + 1)])] != f) gval[pf] = ((int64_t)1 << 32) | (uint32_t)(x - g);
    }
    sync();
}

// The listed components.  Most only straddled the end of their wavefront's positions: a
// wavefront takes each and reduces it as above from its own first position.  Up to
// kCompWave terms it goes through them 64 at a time; a workgroup takes what is larger.
// Long windows of few states have components of thousands of terms that all reduce into one
// (16269 in a 10-step window of 2 states).  The arrays F and O belong to these components alone.
constexpr int kCompWave = 1024;
constexpr int kCompThreads = 512;
template <int D>
__device__ __forceinline__ void k_ftr_comp_big(MG<kCompThreads, 1> mg, const TermPool OUT,
                                               const uint32_t* __restrict__ perm, int n, const int* __restrict__ boff,
                                               const StepConst* __restrict__ sc, const uint64_t* __restrict__ skeys,
                                               const uint32_t* __restrict__ sidx,
                                               int* __restrict__ rootpos, int* __restrict__ rank,
                                               int64_t* __restrict__ gval, const int* __restrict__ big_count,
                                               const int* __restrict__ big_list, int* F, int* O) {
    constexpr int kWaves = kCompThreads / kWave;
    __shared__ int wsum[kWaves];
    __shared__ int2 large[kWaves];
    __shared__ FtrLds lds[kWaves];
    const int lane = wave_lane(), w = threadIdx.x / kWave;
    const int count = *big_count;
    for (int e0 = mg.bx * kWaves; e0 < count; e0 += mg.gx * kWaves) {
        int r0 = -1, r1 = -1;
        if (e0 + w < count && (ftr_comp_wave<D>(OUT, perm, n, boff, sc, skeys, sidx, rootpos, rank, gval,
                                                big_list[e0 + w], 1) & 1u))
            r0 = big_list[e0 + w];
        if (r0 >= 0) {
            auto run_end = [&](int b) {  // positions past n stop it
                for (;; b += kWave) {
                    const int r = b + lane;
                    const uint64_t stop = __ballot(r >= n || !ftr_linked<D>(skeys[r - 1], skeys[r]));
                    if (stop) return min(n, b + __ffsll((unsigned long long)stop) - 1);
                }
            };
            r1 = run_end(r0 + 1);
            const int m = ftr_shape(skeys[r0]);
            const int beg = boff[m];
            if (r1 == boff[m + 1] && ftr_joined<D>(skeys[beg], skeys[r1 - 1])) r1 += run_end(beg + 1) - beg;
        }
        if (r0 >= 0) {
            if (r1 - r0 <= kCompWave) {
                ftr_comp_many<D, kWave>(OUT, perm, n, boff, sc, skeys, sidx, rootpos, rank, gval, F, O, r0, r1, lds + w,
                                        nullptr);
                r0 = -1;
            }
        }
        __syncthreads();  // the previous round's list has been read
        if (lane == 0) large[w] = make_int2(r0, r1);
        __syncthreads();
        for (int e = 0; e < kWaves; e++)
            if (large[e].x >= 0)
                ftr_comp_many<D, kCompThreads>(OUT, perm, n, boff, sc, skeys, sidx, rootpos, rank, gval, F, O,
                                               large[e].x, large[e].y, lds, wsum);
    }
}

// Reduction groups in the reference's order: buckets ascending, roots ascending, members
// ascending per root.  goff is the exclusive scan of gval: groups before position p in its
// upper half, members before it in its lower.  gbase[m]: first group of shape m; gbase[nb]:
// their number.
__device__ __forceinline__ void k_ftr_emit(MG<256, 1> mg, int n, const int* __restrict__ boff, int nb,
                                           const uint32_t* __restrict__ perm, const int64_t* __restrict__ gval,
                                           const int64_t* __restrict__ goff, const int* __restrict__ rootpos,
                                           const int* __restrict__ rank, int* __restrict__ grp_root,
                                           int* __restrict__ grp_moff, int* __restrict__ grp_mcnt,
                                           int* __restrict__ grp_m, int* __restrict__ mem_slots,
                                           int* __restrict__ gbase) {
    const int p = mg.bx * blockDim.x + threadIdx.x;
    if (p <= nb) {
        const int f = boff[p];
        gbase[p] = (int)((f < n ? goff[f] : goff[n - 1] + gval[n - 1]) >> 32);
    }
    if (p >= n) return;
    const int64_t v = gval[p];
    const int slot = (int)perm[p];
    if (v >> 32) {
        const int64_t o = goff[p];
        const int g = (int)(o >> 32);
        grp_root[g] = slot;
        grp_moff[g] = (int)(uint32_t)o;
        grp_mcnt[g] = (int)(uint32_t)v;
        grp_m[g] = bucket_of(boff, nb, p);
    } else {
        mem_slots[(int)(uint32_t)goff[rootpos[p]] + rank[p]] = slot;
    }
}

// ------------------------------------------------------------------ group B-tables
// Upper bound of each group's B-table size.
__device__ __forceinline__ void k_group_ub(MG<1024, 1> mg, const TermPool OUT, int ng, const int* __restrict__ grp_root, const int* __restrict__ grp_m,
                           int d, int* __restrict__ ub) {
    const int g = mg.bx * blockDim.x + threadIdx.x;
    if (g >= ng) return;
    const int s = grp_root[g];
    const int m = grp_m[g];
    int u = OUT.bt_n[s];
    if ((OUT.flags[s] & kIsNew) && m <= d) u = max(u, 1 << (m - 1));
    ub[g] = max(u, 1);
}

// B-table of a group root: new children pair the parent's post-update cells
// across their defining hyperplane and, when coaligned, project through c_map
// (make_new_child_btable, cell_enumeration.hpp:206-371); parents keep their own
// post-update cells.  One wavefront per group, an LDS bitset of 2^m bits per
// wavefront, sorted output.
__device__ __forceinline__ void k_group_btab(MG<1024, 1> mg, const TermPool OUT, int g0, int ngb, int m, int d, const int* __restrict__ grp_root,
                             const uint32_t* __restrict__ Barena, const int64_t* __restrict__ b2_off,
                             const int64_t* __restrict__ ub, uint32_t* __restrict__ B2, int* __restrict__ b2_n,
                             int words_per_wave, int* __restrict__ err) {
    extern __shared__ uint32_t sh[];
    const int wv = threadIdx.x / kWave;
    const int lane = wave_lane();
    const int g = g0 + mg.bx * (blockDim.x / kWave) + wv;
    if (g >= g0 + ngb) return;
    uint32_t* bits = sh + wv * words_per_wave;
    const int s = grp_root[g];
    uint32_t* out = B2 + b2_off[g];
    const bool is_new = OUT.flags[s] & kIsNew;
    if (is_new && m <= d) {
        const int nn = (int)min((int64_t)(1 << (m - 1)), ub[g]);
        for (int k = lane; k < nn; k += kWave) out[k] = (uint32_t)k;
        if (lane == 0) b2_n[g] = nn;
        return;
    }
    const int W = m >= 5 ? (1 << (m - 5)) : 1;
    for (int w = lane; w < W; w += kWave) bits[w] = 0;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    const uint32_t* Bt = Barena + OUT.bt_off[s];
    const int nb = OUT.bt_n[s];
    const uint32_t sg = (uint32_t)OUT.bt_sgn[s];
    if (is_new) {
        const int pbc = OUT.pbc[s], z = OUT.z[s];
        const bool coal = m < pbc;
        int bitpos[kMaxM];
        int ncoal = 0;
        if (coal) {
            const uint8_t* cm = OUT.cmap + (int64_t)s * OUT.MM;
            uint32_t seen = 0;
            for (int j = 0; j < pbc; j++) {
                const int ci = cm[j];
                if (!((seen >> ci) & 1u)) {
                    seen |= (1u << ci);
                    bitpos[ncoal++] = j;
                }
            }
        }
        const uint32_t mask_z = 1u << z, top = 1u << (pbc - 1);
        const uint32_t rev = (pbc >= 32) ? 0xffffffffu : ((1u << pbc) - 1u);
        const uint32_t low = mask_z - 1u;
        for (int j = lane; j < nb; j += kWave) {
            const uint32_t bb = Bt[j] ^ sg;
            uint32_t qv = bb ^ mask_z;
            if (qv & top) qv ^= rev;
            if (bsearch_u32(Bt, qv ^ sg, nb) < 0) continue;
            const uint32_t zb = (bb & mask_z) >> z;
            const uint32_t c1 = ((bb >> (z + 1)) << z) | (bb & low) | (zb << (pbc - 1));
            const uint32_t c2 = c1 ^ top;
            uint32_t cs[2] = {(c1 & top) ? (c1 ^ rev) : c1, (c2 & top) ? (c2 ^ rev) : c2};
            for (int e = 0; e < 2; e++) {
                uint32_t key = cs[e];
                if (coal) {
                    uint32_t bc = 0;
                    for (int l = 0; l < ncoal; l++)
                        if ((key >> bitpos[l]) & 1u) bc |= (1u << l);
                    key = bc;
                }
                if (key >= (1u << m)) {
                    atomicOr(err, 16);
                    continue;
                }
                atomicOr(&bits[key >> 5], 1u << (key & 31));
            }
        }
    } else {
        for (int j = lane; j < nb; j += kWave) {
            const uint32_t key = Bt[j] ^ sg;
            if (key >= (1u << m)) {
                atomicOr(err, 16);
                continue;
            }
            atomicOr(&bits[key >> 5], 1u << (key & 31));
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int per = (W + kWave - 1) / kWave;
    const int w0 = lane * per, w1 = min(W, w0 + per);
    int cnt = 0;
    for (int w = w0; w < w1; w++) cnt += __popc(bits[w]);
    int total;
    int pos = wave_excl_scan(cnt, &total);
    const int64_t cap = ub[g];
    for (int w = w0; w < w1; w++) {
        uint32_t x = bits[w];
        while (x) {
            const int bt = __ffs(x) - 1;
            x &= x - 1;
            if (pos < cap) out[pos] = (uint32_t)(w * 32 + bt);
            pos++;
        }
    }
    if (lane == 0) {
        b2_n[g] = (int)min((int64_t)total, cap);
        if (total > cap) atomicOr(err, 32);
    }
}

// ------------------------------------------------------------------ group g-tables
// Parent g-table lookup modes of the g-table kernel.
//   kLookupSearch     binary search over the parent keys in global memory
//   kLookupSearchLds  binary search over an LDS copy of the parent keys
//   kLookupRank       rank structure in LDS (bitset of the parent keys + per-word
//                     prefix counts), values read from global memory
//   kLookupRankVals   rank structure and an LDS copy of the parent values
// Every mode finds the same entry; they differ only in where the index comes from.
// Largest shape of an estimator, and the largest for which the rank structure is used.  A rank
// structure has 2^(shape-1) bits and as many prefix words / 32: beyond kRankShape 16 KiB and more
// for tables of some hundred keys, which a binary search of the staged keys finds in 5 to 9
// steps.  The limit is not a measured crossover: the instantiation for 17 and more rows faulted
// the GPU once, for a reason that was not found, and does not exist.
constexpr int kMaxShape = 20;
constexpr int kRankShape = 16;
enum LookupMode { kLookupSearch = 0, kLookupSearchLds = 1, kLookupRank = 2, kLookupRankVals = 3 };

// Per-term data of one g-table evaluation, staged once per evaluated term: its
// q, coalignment maps and its parent g-table (keys, or rank structure and values)
// live in LDS, the rest in registers.
struct EvalTerm {
    const uint32_t* pkeys;  // parent g-table keys (LDS copy or global)
    const cplx* pvals;      // parent g-table values (LDS copy or global)
    const uint32_t* rbits;  // rank structure: key bitset
    const uint32_t* rpre;   // rank structure: keys in the words before each word
    uint32_t klim;          // 2^(phc-1): every stored key is below it (half storage)
    uint32_t fm;            // rows that enter ygi: below m and not H-orthogonal
    int pn;                 // parent g-table size
    int m, phc, z, lhp;
    uint32_t hf;
    bool is_new, has_cmap;
    double c, dv, gscale;
};

// Half-storage g numerator lookup in the parent g-table, eval_gs.hpp:94-153.
template <int MODE>
__device__ inline cplx lookup_g(const EvalTerm& T, int enc, int top_bit, int rev_mask) {
    if (MODE >= kLookupRank) {
        // branchless: both LDS reads are issued together, the value read uses
        // entry 0 when the key is absent and the result is then replaced by zero
        const bool cj = (enc & top_bit) != 0;
        const uint32_t key0 = (uint32_t)(cj ? (rev_mask ^ enc) : enc);
        const bool inr = key0 < T.klim;
        const uint32_t key = inr ? key0 : 0u;
        const uint32_t wv = T.rbits[key >> 5];
        const uint32_t pre = T.rpre[key >> 5];
        const uint32_t bit = 1u << (key & 31);
        const bool found = inr && (wv & bit) != 0;
        const int idx = found ? (int)(pre + __popc(wv & (bit - 1u))) : 0;
        // the LDS value copy always holds entry 0; a global table may be empty
        const cplx v = (MODE == kLookupRankVals || found) ? T.pvals[idx] : cmake(0, 0);
        const double re = found ? v.re : 0.0;
        const double im = found ? (cj ? -v.im : v.im) : 0.0;
        return cmake(re, im);
    }
    return lookup_num(enc, top_bit, rev_mask, T.pkeys, T.pvals, T.pn);
}

// g value of one term at one cell (make_gtable loop body, flattening.hpp:129-248).
// ygi is summed in row order as in the reference.  qr holds q for the rows that
// enter the sum and -0.0 for the others (KM >= m, compile-time bound): adding
// -0.0 leaves any double unchanged, and q * (-1) is q with its sign bit flipped.
template <int MODE, int KM>
__device__ inline cplx eval_cell(const EvalTerm& T, const double (&qr)[KM], const uint8_t* cm, const int8_t* cs,
                                 uint32_t key) {
    double ygi = 0;
    const uint32_t kb = key & T.fm;
#pragma unroll
    for (int k = 0; k < KM; k++) {
        const unsigned long long sb = (unsigned long long)((kb >> k) & 1u) << 63;
        ygi += __longlong_as_double((long long)((unsigned long long)__double_as_longlong(qr[k]) ^ sb));
    }
    const int phc = T.phc;
    const int rev_phc = (phc >= 32) ? -1 : ((1 << phc) - 1);
    const int top_phc = 1 << (phc - 1);
    int lp = 0, lmv = 0;
    if (!T.is_new) {
        lp = (int)key & rev_phc;
        lmv = lp;
    } else if (!T.has_cmap) {
        // the child's key with bit z of the parent inserted: parent bit k is child
        // bit k below z and child bit k-1 above it; bit z is 0 in lp and 1 in lmv
        if (T.z < phc) {
            const uint32_t low = key & ((1u << T.z) - 1u);
            const uint32_t high = (key >> T.z) << (T.z + 1);
            lp = (int)((low | high) & (uint32_t)rev_phc);
            lmv = lp | (1 << T.z);
        } else {
            lp = (int)key & rev_phc;
            lmv = lp;
        }
    } else {
        int k = 0, l = 0;
        while (k < phc) {
            if (k == T.z) {
                lmv |= (1 << k);
                k++;
                if (k == phc) break;
            }
            const int bv = (((key >> cm[l]) & 1u) ? -1 : 1) * (int)cs[l];
            if (bv < 0) {
                lp |= (1 << k);
                lmv |= (1 << k);
            }
            k++;
            l++;
        }
    }
    const cplx a = lookup_g<MODE>(T, lp ^ T.lhp, top_phc, rev_phc);
    const cplx bm = lookup_g<MODE>(T, lmv ^ T.lhp, top_phc, rev_phc);
    const cplx v = csub(cdiv(a, cmake(ygi + T.dv, T.c)), cdiv(bm, cmake(ygi - T.dv, T.c)));
    return cscale(v, T.gscale);
}

// (sum of p over the first m rows)^2 of term s, summed in row order.  A wavefront's lanes load
// the rows at once; the sum then takes them from the lanes one by one.
__device__ __forceinline__ double wave_psum2(const TermPool& T, int64_t s, int m) {
    const int lane = wave_lane();
    const double x = lane < m ? T.p[s * T.MM + lane] : 0.0;
    const int lo = __double2loint(x), hi = __double2hiint(x);
    double ps = 0;
    for (int k = 0; k < m; k++)
        ps += __hiloint2double(__builtin_amdgcn_readlane(hi, k), __builtin_amdgcn_readlane(lo, k));
    return ps * ps;
}

// Orientation mask between two +/- equal arrangements: per row, sign of the first element
// non-negligible in both, cell_enumeration.hpp:586-599, by a whole wavefront, lane k on row k.
// `ai` holds Ai[k d] on lane k (kept by the caller for its root, which meets every member of its
// group).
__device__ __forceinline__ int wave_orientation(const double* Ai, double ai, const double* Aj, int m, int d) {
    const int k = wave_lane();
    const bool row = k < m;
    const double aj = row ? Aj[k * d] : 1.0;
    bool neg = row && ai * aj < 0;
    if (__any(row && (fabs(ai) < kReductionEps || fabs(aj) < kReductionEps))) {
        neg = false;
        if (row) {
            int e = k * d;
            while (e < m * d && ((fabs(Ai[e]) < kReductionEps) || (fabs(Aj[e]) < kReductionEps))) e++;
            neg = e < m * d && (Ai[e] * Aj[e]) < 0;
        }
    }
    return (int)__ballot(neg);
}

// Whether any lane's value v (of the lanes in `on`) is large, ps |v| > kApproxEps.  |v| is at
// least either part, so a part that is large by more than the rounding of hypot and of the
// products decides it; only if no lane's is, the reference's test is taken.
__device__ __forceinline__ bool wave_large(bool on, double ps, cplx v) {
    constexpr double lim = kApproxEps * (1.0 + 1e-10);
    const bool sure = on && v.re == v.re && v.im == v.im && (ps * fabs(v.re) > lim || ps * fabs(v.im) > lim);
    if (__any(sure)) return true;
    return __any(on && (ps * hypot(v.re, v.im)) > kApproxEps);
}

// Stages term s for evaluation (a workgroup of one wavefront, blockDim == 64).  `lds` is the
// kernel's dynamic LDS: parent keys (kLookupSearchLds), or the rank structure of
// `wmax` words of bits and `wmax` prefix counts, then the parent values.
template <int MODE, int KM>
__device__ inline EvalTerm stage_term(const TermPool& O, int64_t s, int m, const uint32_t* gk_prev,
                                      const cplx* gv_prev, const uint2* rank, double gscale, uint32_t* lds, int wmax,
                                      double (&qr)[KM], uint8_t* cm_s, int8_t* cs_s) {
    EvalTerm T;
    // every lane loads the same record; its scalars go to scalar registers
    const int64_t go = wave_uniform(O.gp_off[s]);
    T.pn = wave_uniform(O.gp_n[s]);
    T.pvals = gv_prev + go;
    T.pkeys = gk_prev + go;
    T.rbits = nullptr;
    T.rpre = nullptr;
    T.m = m;
    T.phc = wave_uniform(O.phc[s]);
    T.z = wave_uniform(O.z[s]);
    T.lhp = wave_uniform(O.lhp[s]);
    T.hf = (uint32_t)wave_uniform((int)O.hflag[s]);
    const int fl = wave_uniform((int)O.flags[s]);
    T.is_new = fl & kIsNew;
    T.has_cmap = fl & kHasCmap;
    T.c = O.c[s];
    T.dv = O.dv[s];
    T.gscale = gscale;
    T.klim = 1u << (T.phc - 1);
    wave_lds_sync();
    const int lane = threadIdx.x;
    if (MODE == kLookupSearchLds) {
        const uint32_t* src = gk_prev + go;
        for (int i = lane; i < T.pn; i += kWave) lds[i] = src[i];
        T.pkeys = lds;
    } else if (MODE >= kLookupRank) {
        // the parent's rank structure, built once per update by k_rank_build
        const int W = (int)((T.klim + 31u) >> 5);
        uint32_t* bits = lds;
        uint32_t* pre = lds + wmax;
        const uint2* R = rank + wave_uniform(O.rk_off[s]);
        for (int w = lane; w < W; w += kWave) {
            const uint2 v = R[w];
            bits[w] = v.x;
            pre[w] = v.y;
        }
        T.rbits = bits;
        T.rpre = pre;
        if (MODE == kLookupRankVals) {
            cplx* dst = reinterpret_cast<cplx*>(lds + 2 * wmax);
            const cplx* vs = gv_prev + go;
            for (int i = lane; i < T.pn; i += kWave) dst[i] = vs[i];
            if (T.pn == 0 && lane == 0) dst[0] = cmake(0, 0);
            T.pvals = dst;
        }
    }
    const int MM = O.MM;
    T.fm = (m >= 32 ? 0xffffffffu : ((1u << m) - 1u)) & ~T.hf;
#pragma unroll
    for (int kk = 0; kk < KM; kk++) qr[kk] = ((T.fm >> kk) & 1u) ? O.q[s * MM + kk] : -0.0;
    if (T.has_cmap && lane < O.pbc[s]) {
        cm_s[lane] = O.cmap[s * MM + lane];
        cs_s[lane] = O.csmap[s * MM + lane];
    }
    wave_lds_sync();
    return T;
}

// Rank structure of each parent's g-table, once per update: a bitset of its keys below
// 2^(phc-1) and, per 32-bit word, the index of its first key at or after the word's first
// key value.  Every child of the parent evaluated by the g-table kernel reads it from here
// (stage_term) instead of rebuilding it from the keys.  One wavefront per parent; the
// structure is built in LDS (wmax words of bits, then wmax of prefix counts) and written
// out as (bits, prefix) pairs at sc->rk_base[phc] + (index in its shape bucket) * W.
__device__ __forceinline__ void k_rank_build(MG<64, 1> mg, const TermPool P, int n, const StepConst* __restrict__ sc,
                                             const uint32_t* __restrict__ gkeys, uint2* __restrict__ rank, int wmax) {
    extern __shared__ __align__(16) uint32_t lds_dyn[];
    const int t = mg.bx;
    if (t >= n) return;
    const int lane = threadIdx.x;
    const int phc = P.phc[t];
    const uint32_t klim = 1u << (phc - 1);
    const int W = (int)((klim + 31u) >> 5);
    const int64_t off = sc->rk_base[phc] + (int64_t)(t - sc->in_off[phc]) * W;
    if (lane == 0) P.rk_off[t] = off;
    const int pn = P.gp_n[t];
    const uint32_t* src = gkeys + P.gp_off[t];
    // keys are sorted ascending; W words cover those below klim.  A key at or above klim (a
    // coaligned child's cell whose bit m-1 was left set, kept as a parent key) sorts after
    // every key below it and is never looked up (lookups reverse their key below klim,
    // eval_gs.hpp:116-151), so it only ends the prefix counts.
    uint32_t* bits = lds_dyn;
    uint32_t* pre = lds_dyn + wmax;
    for (int w = lane; w < W; w += kWave) bits[w] = 0;
    __syncthreads();
    // eight keys per lane per round; all loads of a round are issued before the LDS updates
    constexpr int U = 8;
    for (int i0 = 0; i0 < pn; i0 += U * kWave) {
        uint32_t kc[U], kp[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = min(i0 + lane + u * kWave, pn - 1);
            kc[u] = src[i];
            kp[u] = src[i > 0 ? i - 1 : 0];
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = i0 + lane + u * kWave;
            if (i >= pn) continue;
            const uint32_t key = kc[u];
            if (key < klim) atomicOr(&bits[key >> 5], 1u << (key & 31));
            // pre[x] = index of the first key in word >= x, filled for the words between the
            // previous key's word and this key's word
            const int w = min((int)(key >> 5), W - 1);
            const int wp = i ? min((int)(kp[u] >> 5), W - 1) : -1;
            for (int x = wp + 1; x <= w; x++) pre[x] = i;
        }
    }
    const int lastw = pn ? min((int)(src[pn - 1] >> 5), W - 1) : -1;
    for (int w = lane; w < W; w += kWave)
        if (w > lastw) pre[w] = pn;
    __syncthreads();
    for (int w = lane; w < W; w += kWave) rank[off + w] = make_uint2(bits[w], pre[w]);
}

// One member of a reduction group, added into the group's root table (add_gtables,
// flattening.hpp:259-315) in the root's orientation sig: root cell bi takes the member's value
// at bi ^ sig, reversed and conjugated when that key is in the upper half; a key outside the
// member's table adds nothing.  A negligible member (term approximation) adds nothing at all.
// add(i, v) receives the values.  The approximation test looks at the member's own cells
// B ^ own, which are the same keys wherever bi is in the lower half: the values it evaluates
// are the ones that are added.  (A coaligned child's projected cells are not re-normalised,
// cell_enumeration.hpp:206-371, so a key of B can have bit m-1 set.)  Returns whether the
// member is negligible.
template <int MODE, int KM, class Add>
__device__ __forceinline__ bool eval_member(const EvalTerm& T, const double (&qr)[KM], const uint8_t* cm_s,
                                            const int8_t* cs_s, const uint32_t* __restrict__ B, int n, int m,
                                            uint32_t X, uint32_t sig, double ps, Add add) {
    const int lane = wave_lane();
    const uint32_t top = 1u << (m - 1), rev = (m >= 32) ? 0xffffffffu : ((1u << m) - 1u);
    const uint32_t own = X ^ ((sig & top) ? (sig ^ rev) : sig);  // a cell of B is the member's key B ^ own
    // the first 64 cells with a large one among them
    int at = 0;
    uint32_t b = 0;
    cplx v = cmake(0, 0);
    for (; at < n; at += kWave) {
        const int i = at + lane;
        b = B[min(i, n - 1)];
        if (i < n) v = eval_cell<MODE, KM>(T, qr, cm_s, cs_s, b ^ own);
        if (wave_large(i < n, ps, v)) break;
    }
    if (at >= n) return true;
    for (int i0 = 0; i0 < n; i0 += kWave) {
        const int i = i0 + lane;
        const uint32_t bi = i0 == at ? b : B[min(i, n - 1)];
        uint32_t x = bi ^ X ^ sig;
        const bool cj = (x & top) != 0;
        if (cj) x ^= rev;
        bool on = i < n, known = i0 == at;
        if (x != (bi ^ own)) {
            on = on && bsearch_u32(B, x ^ own, n) >= 0;
            known = false;
        }
        cplx c = v;
        if (__any(on && !known) && on && !known) c = eval_cell<MODE, KM>(T, qr, cm_s, cs_s, x);
        if (on) add(i, cj ? cconj(c) : c);
    }
    return false;
}

// Flattening of one reduction group, make_gtables (flattening.hpp:351-564):
// the root's g-table; if the root is negligible (term approximation), the
// members in order re-orient the group B-table until one is not (root
// replacement); then every later non-negligible member's g-table is added into
// the root's in member order (add_gtables, flattening.hpp:259-315).
// One wavefront per group; lanes own cells.  What bounds it is the chain of loads that each
// evaluated term waits for (its record, then its parent's rank structure, then the parent
// values its cells look up), so a term's p, A and q are loaded by all lanes at once, and every
// cell of a member is evaluated once.
template <int MODE, int KM>
__device__ __forceinline__ void k_group_eval(MG<64, 1> mg, const TermPool OUT, int ng, int d, int wmax,
                                                  const int* __restrict__ grp_root,
                                                  const int* __restrict__ grp_moff, const int* __restrict__ grp_mcnt,
                                                  const int* __restrict__ grp_m, const int* __restrict__ mem_slots,
                                                  const uint32_t* __restrict__ B2, const int64_t* __restrict__ b2_off,
                                                  const int* __restrict__ b2_n, const int64_t* __restrict__ g_off,
                                                  const uint32_t* __restrict__ gk_prev, const cplx* __restrict__ gv_prev,
                                                  uint32_t* __restrict__ gk_out, cplx* __restrict__ gv_out,
                                                  double gscale, int* __restrict__ surv,
                                                  int* __restrict__ gxor, int* __restrict__ sort_list,
                                                  int* __restrict__ sort_count, int* __restrict__ rare,
                                                  int big_members, int* __restrict__ defer_k0,
                                                  uint8_t* __restrict__ mem_add, const uint2* __restrict__ rank) {
    extern __shared__ __align__(16) uint32_t lds_dyn[];
    double qr[KM];
    __shared__ uint8_t cm_s[kMaxM];
    __shared__ int8_t cs_s[kMaxM];
    const int g = mg.bx;
    if (g >= ng) return;
    const int lane = threadIdx.x;
    const int m = grp_m[g];
    const int MM = OUT.MM;
    const uint32_t* B = B2 + b2_off[g];
    const int n = b2_n[g];
    uint32_t* ok = gk_out + g_off[g];
    cplx* ov = gv_out + g_off[g];
    const int* mem = mem_slots + grp_moff[g];
    const int nmem = grp_mcnt[g];
    const uint32_t top = 1u << (m - 1);
    const uint32_t rev = (m >= 32) ? 0xffffffffu : ((1u << m) - 1u);
    int r = grp_root[g];
    uint32_t X = 0;
    // The root's cells are written as the group's table.  While a root is negligible (every cell
    // is small; the test stops at the first large one), the next member re-orients the group and
    // replaces it (replacement chain, flattening.hpp:412-489).
    int k = 0;
    for (;;) {
        const EvalTerm T = stage_term<MODE, KM>(OUT, r, m, gk_prev, gv_prev, rank, gscale, lds_dyn, wmax, qr, cm_s, cs_s);
        const double ps = wave_psum2(OUT, r, m);
        bool negl = true;
        uint32_t bnext = n > 0 ? B[min(lane, n - 1)] : 0u;  // cell key of the next pass, loaded a pass ahead
        for (int i0 = 0; i0 < n; i0 += kWave) {
            const int i = i0 + lane;
            const uint32_t bcur = bnext;
            bnext = B[min(i + kWave, n - 1)];
            cplx v = cmake(0, 0);
            if (i < n) {
                v = eval_cell<MODE, KM>(T, qr, cm_s, cs_s, bcur ^ X);
                ov[i] = v;
            }
            if (negl) negl = !wave_large(i < n, ps, v);
        }
        if (!negl) break;
        if (k >= nmem) {
            if (lane == 0) surv[g] = -1;
            return;
        }
        const int sk = wave_uniform(mem[k++]);
        if (!(OUT.flags[sk] & kIsNew) && lane == 0) atomicOr(rare, 1);
        const double* Al = OUT.A + (int64_t)r * MM * d;
        int sig = wave_orientation(Al, lane < m ? Al[lane * d] : 1.0, OUT.A + (int64_t)sk * MM * d, m, d);
        if ((uint32_t)sig & top) sig ^= (int)rev;
        X ^= (uint32_t)sig;
        r = sk;
    }
    // later members are added into the root's table; in a group with more than
    // big_members members that is left to k_group_members / k_group_sum
    const double* Ar = OUT.A + (int64_t)r * MM * d;
    const double ar = lane < m ? Ar[lane * d] : 1.0;
    if (nmem > big_members) {
        if (lane == 0) defer_k0[g] = k;
        k = nmem;
    }
    for (; k < nmem; k++) {
        const int sk = wave_uniform(mem[k]);
        if (!(OUT.flags[sk] & kIsNew) && lane == 0) atomicOr(rare, 2);
        const int sig = wave_orientation(Ar, ar, OUT.A + (int64_t)sk * MM * d, m, d);
        const EvalTerm T = stage_term<MODE, KM>(OUT, sk, m, gk_prev, gv_prev, rank, gscale, lds_dyn, wmax, qr, cm_s, cs_s);
        const bool negl = eval_member<MODE, KM>(T, qr, cm_s, cs_s, B, n, m, X, (uint32_t)sig, wave_psum2(OUT, sk, m),
                                                [&](int i, cplx v) { ov[i] = cadd(ov[i], v); });
        if (mem_add && lane == 0) mem_add[grp_moff[g] + k] = negl ? 0 : 1;
    }
    for (int i = lane; i < n; i += kWave) ok[i] = B[i] ^ X;
    if (lane == 0) {
        surv[g] = r;
        gxor[g] = (int)X;
        if (X != 0) {
            const int slot = atomicAdd(sort_count, 1);
            sort_list[slot] = g;
        }
    }
}

// Work lists of the groups whose members are added in parallel: per group the
// member count, the contribution entries (members x cells) and the 64-cell chunks.
__device__ __forceinline__ void k_big_prep(MG<1024, 1> mg, int ng, int big_members, const int* __restrict__ grp_mcnt, const int* __restrict__ b2_n,
                           int* __restrict__ icnt, int64_t* __restrict__ ccnt, int* __restrict__ hcnt) {
    const int g = mg.bx * blockDim.x + threadIdx.x;
    if (g >= ng) return;
    const int nm = grp_mcnt[g];
    const bool big = nm > big_members;
    icnt[g] = big ? nm : 0;
    ccnt[g] = big ? (int64_t)nm * b2_n[g] : 0;
    hcnt[g] = big ? (b2_n[g] + kWave - 1) / kWave : 0;
}

// Largest g with off[g] <= item (off ascending, off[0] == 0).
__device__ inline int owner_of(const int* __restrict__ off, int n, int item) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (off[mid] <= item) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// One wavefront per (large group, member k): the member's g-table contribution to
// every cell of the group's root, in the root's orientation (add_gtables,
// flattening.hpp:259-315), written to contrib[coff[g] + k * n + i].  A cell that receives
// nothing, and every cell of a negligible member, gets (-0.0, -0.0), which leaves any sum
// unchanged.
template <int MODE, int KM>
__device__ __forceinline__ void k_group_members(MG<64, 1> mg, const TermPool OUT, int ng, int d, int wmax,
                                                     const int* __restrict__ ioff, int nitems,
                                                     const int64_t* __restrict__ coff,
                                                     const int* __restrict__ grp_moff, const int* __restrict__ grp_mcnt,
                                                     const int* __restrict__ grp_m, const int* __restrict__ mem_slots,
                                                     const uint32_t* __restrict__ B2, const int64_t* __restrict__ b2_off,
                                                     const int* __restrict__ b2_n, const uint32_t* __restrict__ gk_prev,
                                                     const cplx* __restrict__ gv_prev, double gscale,
                                                     const int* __restrict__ surv, const int* __restrict__ gxor,
                                                     const int* __restrict__ defer_k0, cplx* __restrict__ contrib,
                                                     int* __restrict__ rare,
                                                     uint8_t* __restrict__ mem_add, const uint2* __restrict__ rank) {
    extern __shared__ __align__(16) uint32_t lds_dyn[];
    double qr[KM];
    __shared__ uint8_t cm_s[kMaxM];
    __shared__ int8_t cs_s[kMaxM];
    const int item = mg.bx;
    if (item >= nitems) return;
    const int g = owner_of(ioff, ng, item);
    const int k = item - ioff[g];
    const int r = surv[g];
    if (r < 0 || k < defer_k0[g]) return;
    const int lane = threadIdx.x;
    const int m = grp_m[g];
    const int MM = OUT.MM;
    const uint32_t* B = B2 + b2_off[g];
    const int n = b2_n[g];
    const int sk = mem_slots[grp_moff[g] + k];
    if (!(OUT.flags[sk] & kIsNew) && lane == 0) atomicOr(rare, 2);
    const double* Ar = OUT.A + (int64_t)r * MM * d;
    const int sig = wave_orientation(Ar, lane < m ? Ar[lane * d] : 1.0, OUT.A + (int64_t)sk * MM * d, m, d);
    const EvalTerm T = stage_term<MODE, KM>(OUT, sk, m, gk_prev, gv_prev, rank, gscale, lds_dyn, wmax, qr, cm_s, cs_s);
    cplx* out = contrib + coff[g] + (int64_t)k * n;
    for (int i = lane; i < n; i += kWave) out[i] = cmake(-0.0, -0.0);
    const bool negl = eval_member<MODE, KM>(T, qr, cm_s, cs_s, B, n, m, (uint32_t)gxor[g], (uint32_t)sig,
                                            wave_psum2(OUT, sk, m), [&](int i, cplx v) { out[i] = v; });
    if (mem_add && lane == 0) mem_add[grp_moff[g] + k] = negl ? 0 : 1;
}

// Adds the member contributions of each large group into its root's table, one
// lane per cell, members in order (the sum order of add_gtables): a serial chain of adds, fed
// by kSumBatch loads in flight.
__device__ __forceinline__ void k_group_sum(MG<64, 1> mg, int ng, const int* __restrict__ hoff, int nchunks,
                                                 const int64_t* __restrict__ coff,
                                                 const int* __restrict__ grp_mcnt, const int* __restrict__ b2_n,
                                                 const int64_t* __restrict__ g_off, const int* __restrict__ surv,
                                                 const int* __restrict__ defer_k0, const cplx* __restrict__ contrib,
                                                 cplx* __restrict__ gv_out) {
    const int item = mg.bx;
    if (item >= nchunks) return;
    const int g = owner_of(hoff, ng, item);
    if (surv[g] < 0) return;
    const int n = b2_n[g];
    const int i = (item - hoff[g]) * kWave + threadIdx.x;
    if (i >= n) return;
    const int nm = grp_mcnt[g];
    const cplx* cb = contrib + coff[g] + i;
    cplx acc = gv_out[g_off[g] + i];
    constexpr int kSumBatch = 16;
    int k = defer_k0[g];
    for (; k + kSumBatch <= nm; k += kSumBatch) {
        cplx c[kSumBatch];
#pragma unroll
        for (int u = 0; u < kSumBatch; u++) c[u] = cb[(int64_t)(k + u) * n];
#pragma unroll
        for (int u = 0; u < kSumBatch; u++) acc = cadd(acc, c[u]);
    }
    for (; k < nm; k++) acc = cadd(acc, cb[(int64_t)k * n]);
    gv_out[g_off[g] + i] = acc;
}

// Restores ascending key order of a group table whose keys were re-oriented by
// a root replacement.  One block per listed group; rank from an LDS bitset.
__device__ __forceinline__ void k_group_sort(MG<1024, 1> mg, int nlist, const int* __restrict__ list, const int* __restrict__ grp_m,
                             const int* __restrict__ b2_n, const int64_t* __restrict__ g_off,
                             uint32_t* __restrict__ gk, cplx* __restrict__ gv, uint32_t* __restrict__ tmpk,
                             cplx* __restrict__ tmpv) {
    extern __shared__ uint32_t bits[];
    __shared__ int wbase[1024];
    const int g = list[mg.bx];
    const int m = grp_m[g];
    const int n = b2_n[g];
    const int W = m >= 5 ? (1 << (m - 5)) : 1;
    uint32_t* k = gk + g_off[g];
    cplx* v = gv + g_off[g];
    uint32_t* tk = tmpk + g_off[g];
    cplx* tv = tmpv + g_off[g];
    for (int w = threadIdx.x; w < W; w += blockDim.x) bits[w] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        tk[i] = k[i];
        tv[i] = v[i];
        atomicOr(&bits[k[i] >> 5], 1u << (k[i] & 31));
    }
    __syncthreads();
    // prefix popcounts over words, in chunks of blockDim
    const int per = (W + blockDim.x - 1) / blockDim.x;
    const int w0 = threadIdx.x * per, w1 = min(W, w0 + per);
    int c = 0;
    for (int w = w0; w < w1; w++) c += __popc(bits[w]);
    wbase[threadIdx.x] = c;
    __syncthreads();
    for (int o = 1; o < (int)blockDim.x; o <<= 1) {
        int t = (threadIdx.x >= (unsigned)o) ? wbase[threadIdx.x - o] : 0;
        __syncthreads();
        wbase[threadIdx.x] += t;
        __syncthreads();
    }
    const int tb = wbase[threadIdx.x] - c;
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const uint32_t key = tk[i];
        const int w = key >> 5;
        const int owner = w / per;
        int pos = (owner > 0 ? wbase[owner - 1] : 0);
        for (int ww = owner * per; ww < w; ww++) pos += __popc(bits[ww]);
        pos += __popc(bits[w] & ((1u << (key & 31)) - 1u));
        k[pos] = key;
        v[pos] = tv[i];
    }
    (void)tb;
}

// ------------------------------------------------------------------ compaction
template <int D>
__device__ __forceinline__ void k_compact(MG<1024, 1> mg, const TermPool OUT, int ng, const int* __restrict__ surv, const int* __restrict__ pos,
                          const int* __restrict__ grp_m, const int64_t* __restrict__ g_off,
                          const int* __restrict__ b2_n, TermPool NEXT) {
    const int g = mg.bx * blockDim.x + threadIdx.x;
    if (g >= ng) return;
    const int r = surv[g];
    if (r < 0) return;
    const int o = pos[g];
    const int m = grp_m[g];
    const int MM = OUT.MM;
    const double* A = OUT.A + (int64_t)r * MM * D;
    const double* p = OUT.p + (int64_t)r * MM;
    const double* b = OUT.b + (int64_t)r * D;
    double* nA = NEXT.A + (int64_t)o * MM * D;
    double* np_ = NEXT.p + (int64_t)o * MM;
    double* nb = NEXT.b + (int64_t)o * D;
    for (int k = 0; k < m * D; k++) nA[k] = A[k];
    for (int k = 0; k < m; k++) np_[k] = p[k];
    for (int k = 0; k < D; k++) nb[k] = b[k];
    NEXT.m[o] = m;
    NEXT.gp_off[o] = g_off[g];
    NEXT.gp_n[o] = b2_n[g];
}

// g-tables of the first update's terms (make_gtable_first, flattening.hpp:14-67).
template <int D>
__device__ __forceinline__ void k_gtable_first(MG<1024, 1> mg, const TermPool OUT, int n, const uint32_t* __restrict__ perm, double gscale,
                               uint32_t* __restrict__ gk, cplx* __restrict__ gv, TermPool NEXT) {
    const int r = mg.bx * blockDim.x + threadIdx.x;
    if (r >= n) return;
    const int64_t s = perm[r];
    const int cells = 1 << (D - 1);
    const int MM = OUT.MM;
    const double* p = OUT.p + s * MM;
    const uint32_t hf = OUT.hflag[s];
    const double c = OUT.c[s], dv = OUT.dv[s];
    const int64_t off = (int64_t)r * cells;
    for (int j = 0; j < cells; j++) {
        double ygi = 0;
        for (int k = 0; k < D; k++)
            if (!((hf >> k) & 1u)) {
                const double sb = ((j >> k) & 1) == 0 ? 1 : -1;
                ygi += p[k] * sb;
            }
        cplx v = csub(cdiv(cmake(1.0, 0.0), cmake(ygi + dv, c)), cdiv(cmake(1.0, 0.0), cmake(ygi - dv, c)));
        gk[off + j] = (uint32_t)j;
        gv[off + j] = cscale(v, gscale);
    }
    const double* A = OUT.A + s * MM * D;
    const double* b = OUT.b + s * D;
    for (int k = 0; k < D * D; k++) NEXT.A[(int64_t)r * MM * D + k] = A[k];
    for (int k = 0; k < D; k++) NEXT.p[(int64_t)r * MM + k] = p[k];
    for (int k = 0; k < D; k++) NEXT.b[(int64_t)r * D + k] = b[k];
    NEXT.m[r] = D;
    NEXT.gp_off[r] = off;
    NEXT.gp_n[r] = cells;
}

// Algorithmic bytes of k_group_eval: per group, the B-table keys (4 B/cell) and the
// output table (key + complex value, 20 B/cell); per evaluated term (root and every
// member), its record (q, p, A rows, scalars, coalignment maps) and, per cell, the two
// parent g-table entries its numerators need (2 x 20 B).
__device__ __forceinline__ void k_geval_bytes(MG<1024, 1> mg, int ng, int d, const int* __restrict__ grp_m, const int* __restrict__ grp_mcnt,
                              const int* __restrict__ b2_n, const int* __restrict__ surv,
                              const int* __restrict__ defer_k0, int big_members, unsigned long long* __restrict__ acc) {
    const int g = mg.bx * blockDim.x + threadIdx.x;
    unsigned long long v = 0;
    if (g < ng) {
        const unsigned long long n = (unsigned long long)b2_n[g];
        const unsigned long long m = (unsigned long long)grp_m[g];
        const unsigned long long rec = m * (16ull + 8ull * d) + 2ull * m + 52ull;
        // terms evaluated by k_group_eval: the root and the members it adds itself (a
        // large group's later members are evaluated by k_group_members)
        const int nm = grp_mcnt[g];
        const int own = (nm > big_members && surv[g] >= 0) ? defer_k0[g] : nm;
        const unsigned long long evals = 1ull + (unsigned long long)own;
        v = 24ull * n + evals * (40ull * n + rec);
    }
    // one atomic per wavefront: the counter is shared by every group of the launch
    for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_down(v, o, kWave);
    if ((threadIdx.x & (kWave - 1)) == 0 && v) atomicAdd(acc, v);
}

// acc += sum over i < n of a[i] * (b ? b[i] : 1), over the i with keep[i] >= 0 when keep is
// given: the cell counts of the update's byte accounting (profiling only).
__device__ __forceinline__ void k_prof_sum(MG<1024, 1> mg, int n, const int* __restrict__ a, const int* __restrict__ b,
                                           const int* __restrict__ keep, unsigned long long* __restrict__ acc) {
    const int i = mg.bx * blockDim.x + threadIdx.x;
    unsigned long long v = 0;
    if (i < n && (!keep || keep[i] >= 0))
        v = (unsigned long long)max(a[i], 0) * (unsigned long long)(b ? max(b[i], 0) : 1);
    for (int o = kWave / 2; o > 0; o >>= 1) v += __shfl_down(v, o, kWave);
    if ((threadIdx.x & (kWave - 1)) == 0 && v) atomicAdd(acc, v);
}

// ------------------------------------------------------------------ small helpers
// Total of an exclusive scan: off[n-1] + cnt[n-1].
template <class A, class B>
__device__ __forceinline__ void k_scan_total(MG<1024, 1> mg, const A* __restrict__ off, const B* __restrict__ cnt, int n, int64_t* __restrict__ out) {
    out[0] = n > 0 ? (int64_t)off[n - 1] + (int64_t)cnt[n - 1] : 0;
}

// The same total, also stored into a device-mapped host slot when one is given.
template <class A, class B>
__device__ __forceinline__ void k_scan_total_mapped(MG<1024, 1> mg, const A* __restrict__ off,
                                                    const B* __restrict__ cnt, int n, int64_t* __restrict__ out,
                                                    int64_t* host_out) {
    const int64_t v = n > 0 ? (int64_t)off[n - 1] + (int64_t)cnt[n - 1] : 0;
    out[0] = v;
    if (host_out) *(volatile int64_t*)host_out = v;
}

// Items per thread of one tile of the small scan.  Above one tile, tiles of
// kSmallScanThreads x kScanItems items are loaded coalesced (consecutive threads,
// consecutive items) into LDS, each thread scans its kScanItems consecutive items there,
// and the results go back out coalesced.
constexpr int kScanItems = 4;

// Scan of up to kSmallScan items by one workgroup: the small arrays of small estimators,
// where a library scan costs more launches than work.  Each thread sums a contiguous run, a
// block scan of the run sums gives each run's offset, and the run is written out.  With
// `wide`, the input is also stored widened; with `out_total` / `host_total`, the sum of all
// items goes to a device scalar and a device-mapped host slot.  Integer sums, so the result
// is the same as any other summation order's.
template <class In, class Out, bool Inclusive>
__device__ __forceinline__ void k_small_scan(MG<kSmallScanThreads, 1> mg, const In* __restrict__ in,
                                             Out* __restrict__ out, int n, Out* __restrict__ wide,
                                             int64_t* __restrict__ out_total, int64_t* host_total) {
    (void)mg;
    constexpr int kTile = kSmallScanThreads * kScanItems;
    __shared__ Out tile[kTile];
    const int t = threadIdx.x;
    if (n <= kTile) {
        // one tile or less: each thread scans at most kScanItems consecutive items in place,
        // which costs fewer barriers than staging them.  The items are loaded once, all
        // loads issued before the first is used.
        const int per = (n + kSmallScanThreads - 1) / kSmallScanThreads;
        const int b = min(n, t * per), e = min(n, b + per);
        Out x[kScanItems];
#pragma unroll
        for (int j = 0; j < kScanItems; j++) x[j] = b + j < e ? (Out)in[b + j] : (Out)0;
        Out sum = 0;
#pragma unroll
        for (int j = 0; j < kScanItems; j++) sum += x[j];
        Out tot;
        Out run = block_excl_scan(sum, &tot);
#pragma unroll
        for (int j = 0; j < kScanItems; j++) {
            const int i = b + j;
            if (i < e) {
                if (wide) wide[i] = x[j];
                if (Inclusive) {
                    run += x[j];
                    out[i] = run;
                } else {
                    out[i] = run;
                    run += x[j];
                }
            }
        }
        if (t == kSmallScanThreads - 1) {
            if (out_total) out_total[0] = (int64_t)tot;
            if (host_total) *(volatile int64_t*)host_total = (int64_t)tot;
        }
        return;
    }
    // Tiles: the next tile's loads are issued before the current tile is scanned, so their
    // latency overlaps the scan's barriers and stores.
    Out nx[kScanItems];
#pragma unroll
    for (int j = 0; j < kScanItems; j++) {
        const int i = j * kSmallScanThreads + t;
        nx[j] = i < n ? (Out)in[i] : (Out)0;
    }
    Out carry = 0;
    for (int base = 0; base < n; base += kTile) {
#pragma unroll
        for (int j = 0; j < kScanItems; j++) {
            const int i = base + j * kSmallScanThreads + t;
            if (wide && i < n) wide[i] = nx[j];
            tile[j * kSmallScanThreads + t] = nx[j];
        }
        if (base + kTile < n) {
#pragma unroll
            for (int j = 0; j < kScanItems; j++) {
                const int i = base + kTile + j * kSmallScanThreads + t;
                nx[j] = i < n ? (Out)in[i] : (Out)0;
            }
        }
        __syncthreads();
        Out v[kScanItems], sum = 0;
#pragma unroll
        for (int j = 0; j < kScanItems; j++) {
            v[j] = tile[t * kScanItems + j];
            sum += v[j];
        }
        Out tot;
        Out run = block_excl_scan(sum, &tot) + carry;
#pragma unroll
        for (int j = 0; j < kScanItems; j++) {
            if (Inclusive) {
                run += v[j];
                tile[t * kScanItems + j] = run;
            } else {
                tile[t * kScanItems + j] = run;
                run += v[j];
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kScanItems; j++) {
            const int i = base + j * kSmallScanThreads + t;
            if (i < n) out[i] = tile[j * kSmallScanThreads + t];
        }
        carry += tot;
        __syncthreads();  // the tile is rewritten
    }
    if (t == kSmallScanThreads - 1) {
        if (out_total) out_total[0] = (int64_t)carry;
        if (host_total) *(volatile int64_t*)host_total = (int64_t)carry;
    }
}

__device__ __forceinline__ void k_widen(MG<1024, 1> mg, const int* __restrict__ src, int64_t* __restrict__ dst, int n) {
    const int i = mg.bx * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = (int64_t)src[i];
}
__device__ __forceinline__ void k_surv_flags(MG<1024, 1> mg, int n, const int* __restrict__ surv, int* __restrict__ f) {
    const int i = mg.bx * blockDim.x + threadIdx.x;
    if (i < n) f[i] = surv[i] >= 0 ? 1 : 0;
}
template <int D>
__global__ void k_det_tp(TermPool P, int n, const double* __restrict__ Tr, const double* __restrict__ bias) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int m = P.m[i];
    double* A = P.A + (int64_t)i * P.MM * D;
    double* b = P.b + (int64_t)i * D;
    double t[D];
    for (int r = 0; r < m; r++) {
        for (int k = 0; k < D; k++) t[k] = A[r * D + k];
        for (int j = 0; j < D; j++) {
            double s = 0.0;
            for (int k = 0; k < D; k++) s += t[k] * Tr[k + j * D];
            A[r * D + j] = s;
        }
    }
    for (int k = 0; k < D; k++) t[k] = b[k];
    for (int r = 0; r < D; r++) {
        double s = 0.0;
        for (int j = 0; j < D; j++) s += Tr[r * D + j] * t[j];
        b[r] = s;
    }
    if (bias)
        for (int r = 0; r < D; r++) b[r] += bias[r];
}

// A d-vector passed by value as a kernel argument.
struct VecArg {
    double v[kMaxD];
};

// ------------------------------------------------------------ 1D marginal CPDF
// Per-term closed form of the 1D marginal density (cpdf_ndim.hpp:1233-1368): the
// arrangement is cut along state `marg`; w = sum_j p_j |A_j,marg|, the sign vectors of
// the two half-lines select the numerators, and the term contributes
// Re(g_lhs / (w + i(b_marg - x)) - g_rhs / (-w + i(b_marg - x))) at x.  The second form,
// (a x + bb) / (w^2 + (x - s)^2) with s = b_marg, a = Im(g_rhs) / pi and
// bb = (Re(g_rhs) w - Im(g_rhs) s) / pi, is the one every later grid point uses.
struct CpdfTerm1D {
    double a, bb, w2, s;
};

template <int D>
__global__ void k_cpdf1d_terms(TermPool P, int n, int marg, VecArg bar_nu, const uint32_t* __restrict__ gkeys,
                               const cplx* __restrict__ gvals, double x0, double* __restrict__ direct,
                               CpdfTerm1D* __restrict__ cached) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int m = P.m[i];
    const double* A = P.A + (int64_t)i * P.MM * D;
    const double* p = P.p + (int64_t)i * P.MM;
    const double bm = P.b[(int64_t)i * D + marg];
    double w = 0.0;
    int lhs = 0, rhs = 0;
    for (int j = 0; j < m; j++) {
        const double acj = A[j * D + marg];
        const double fa = fabs(acj);
        w += p[j] * fa;
        bool pos;
        if (fa > 1e-15) {
            pos = acj > 0;
        } else {
            // a row orthogonal to the state: its side is taken from the drawn direction
            double ip = 0.0;
            for (int k = 0; k < D; k++) ip += A[j * D + k] * bar_nu.v[k];
            pos = ip > 0;
        }
        if (pos) lhs |= 1 << j;
        else rhs |= 1 << j;
    }
    const int top = 1 << (m - 1), rev = (1 << m) - 1;
    const int64_t go = P.gp_off[i];
    const int gn = P.gp_n[i];
    const cplx gl = lookup_num(lhs, top, rev, gkeys + go, gvals + go, gn);
    const cplx gr = lookup_num(rhs, top, rev, gkeys + go, gvals + go, gn);
    const double bc = bm - x0;
    const cplx v = csub(cdiv(gl, cmake(w, bc)), cdiv(gr, cmake(-w, bc)));
    direct[i] = v.re;
    CpdfTerm1D c;
    c.s = bm;
    c.a = gr.im / kPi;
    c.bb = (gr.re * w - gr.im * bm) / kPi;
    c.w2 = w * w;
    cached[i] = c;
}

// Deterministic sum of n values by one block (fixed strided partials, then a fixed tree).
__global__ void k_sum_fixed(const double* __restrict__ v, int n, double* __restrict__ out) {
    __shared__ double sh[1024];
    const int t = threadIdx.x;
    double s = 0.0;
    int i = t;
    for (; i + 15 * (int)blockDim.x < n; i += 16 * blockDim.x) {  // sixteen loads in flight
        double x[16];
#pragma unroll
        for (int u = 0; u < 16; u++) x[u] = v[i + u * blockDim.x];
#pragma unroll
        for (int u = 0; u < 16; u++) s += x[u];
    }
    for (; i < n; i += blockDim.x) s += v[i];
    sh[t] = s;
    __syncthreads();
    for (int h = blockDim.x / 2; h > 0; h >>= 1) {
        if (t < h) sh[t] += sh[t + h];
        __syncthreads();
    }
    if (t == 0) out[0] = sh[0];
}

// 1 / d to the last bit or two: the hardware's 2^-24 estimate x with error e = 1 - d x, then
// x (1 + e + e^2), three fused operations where a division takes about ten.  Not finite where
// d is zero, infinite or not a number, or 1 / d beyond the largest double; the callers look for
// that in their sums.  Above 2^1022 1 / d is subnormal, and correct to its fewer bits at most: a
// sum of such terms stays finite and is not formed again by divisions.
__device__ __forceinline__ double fast_rcp(double d) {
    const double x = __builtin_amdgcn_rcp(d);
    const double e = __builtin_fma(-d, x, 1.0);
    return __builtin_fma(x, __builtin_fma(e, e, e), x);
}
__device__ __forceinline__ bool is_finite(double x) { return fabs(x) < __builtin_inf(); }

constexpr int kCpdfChunk = 1024;   // terms staged in LDS per block
constexpr int kCpdfPoints = 256;   // grid points per block (one per thread)

// Partial sums over one chunk of terms for a block of grid points:
// part[chunk * npts + k] = sum over the chunk of (a x_k + bb) / (w2 + (x_k - s)^2).
__global__ void __launch_bounds__(kCpdfPoints) k_cpdf1d_grid(const CpdfTerm1D* __restrict__ cached, int n,
                                                             const double* __restrict__ xs, int npts,
                                                             double* __restrict__ part) {
    __shared__ CpdfTerm1D sh[kCpdfChunk];
    const int chunk = blockIdx.y;
    const int t0 = chunk * kCpdfChunk;
    const int nt = min(kCpdfChunk, n - t0);
    for (int j = threadIdx.x; j < nt; j += blockDim.x) sh[j] = cached[t0 + j];
    __syncthreads();
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= npts) return;
    const double x = xs[k];
    double acc = 0.0;
    // Terms in pairs, n0 / d0 + n1 / d1 = (n0 d1 + n1 d0) / (d0 d1), each d = w^2 + (x - s)^2: one
    // reciprocal per two terms.  Where d0 d1 leaves the range of a double the reciprocal is not
    // a number, and the run of pairs is added again by divisions.
    constexpr int kRun = 32;
    for (int j0 = 0; j0 < nt; j0 += kRun) {
        const int j1 = min(nt, j0 + kRun);
        double run = 0.0;
        int j = j0;
        for (; j + 1 < j1; j += 2) {
            const CpdfTerm1D c0 = sh[j], c1 = sh[j + 1];
            const double x0 = x - c0.s, x1 = x - c1.s;
            const double d0 = __builtin_fma(x0, x0, c0.w2), d1 = __builtin_fma(x1, x1, c1.w2);
            const double n0 = __builtin_fma(c0.a, x, c0.bb), n1 = __builtin_fma(c1.a, x, c1.bb);
            run = __builtin_fma(__builtin_fma(n0, d1, n1 * d0), fast_rcp(d0 * d1), run);
        }
        if (j < j1) {
            const CpdfTerm1D c = sh[j];
            const double xm = x - c.s;
            run += (c.a * x + c.bb) / (c.w2 + xm * xm);
        }
        if (!is_finite(run)) {
            run = 0.0;
            for (j = j0; j < j1; j++) {
                const CpdfTerm1D c = sh[j];
                const double xm = x - c.s;
                run += (c.a * x + c.bb) / (c.w2 + xm * xm);
            }
        }
        acc += run;
    }
    part[(int64_t)chunk * npts + k] = acc;
}

// y_k = (sum over chunks of part) / norm.  Workgroup of kFinishPoints points x kFinishSlices
// wavefronts; slice w adds chunks w, w + kFinishSlices, ... in order, then the slices are added
// in order.  (One thread per point left a 21 x 21 grid's 441 points to two workgroups, which
// took 606 us over 1600 chunks.)
constexpr int kFinishPoints = 64;
constexpr int kFinishSlices = 16;
__global__ void __launch_bounds__(kFinishPoints* kFinishSlices) k_cpdf1d_finish(const double* __restrict__ part,
                                                                                int nchunks, int npts, double norm,
                                                                                double* __restrict__ y) {
    __shared__ double sh[kFinishSlices][kFinishPoints];
    const int lane = threadIdx.x % kFinishPoints, w = threadIdx.x / kFinishPoints;
    const int k = blockIdx.x * kFinishPoints + lane;
    double s = 0.0;
    if (k < npts) {
        int c = w;
        for (; c + 7 * kFinishSlices < nchunks; c += 8 * kFinishSlices) {
            double x[8];
#pragma unroll
            for (int u = 0; u < 8; u++) x[u] = part[(int64_t)(c + u * kFinishSlices) * npts + k];
#pragma unroll
            for (int u = 0; u < 8; u++) s += x[u];
        }
        for (; c < nchunks; c += kFinishSlices) s += part[(int64_t)c * npts + k];
    }
    sh[w][lane] = s;
    __syncthreads();
    if (w == 0 && k < npts) {
        for (int u = 1; u < kFinishSlices; u++) s += sh[u][lane];
        y[k] = s / norm;
    }
}


// Grid abscissae of the 1D density, x_k = min(low + k res, high), as the host forms them
// (no multiply-add is fused), for callers that keep the grid in device memory.
__global__ void k_cpdf1d_xs(double* __restrict__ xs, int npts, double lo, double res, double hi) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= npts) return;
    const double v = lo + (double)k * res;
    xs[k] = hi < v ? hi : v;
}

// The density at the first grid point from the direct sum, (sum / 2 pi) / norm, or
// zero everywhere when the estimator holds no terms.
__global__ void k_cpdf1d_first(const double* __restrict__ direct_sum, double norm, double* __restrict__ y,
                               int zero_n) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (zero_n > 0) {
        if (k < zero_n) y[k] = 0.0;
        return;
    }
    if (k == 0) y[0] = direct_sum[0] * kInvTwoPi / norm;
}

// b <- b - dx for every term (cauchy_estimator.hpp:1371-1380, sub_vecs).
template <int D>
__device__ __forceinline__ void k_sub_b(MG<1024, 1> mg, TermPool P, int n, VecArg dx) {
    const int i = mg.bx * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double* b = P.b + (int64_t)i * D;
#pragma unroll
    for (int r = 0; r < D; r++) b[r] -= dx.v[r];
}

// ------------------------------------------------------------ 2D marginal CPDF
// Per-term cell data of the 2D marginal density (cpdf_ndim.hpp:1400-1700): the
// arrangement cut to states (i1, i2), zero rows removed and +/- equal rows merged
// (marg2d_remove_zeros_and_coalign), the cell walls' angles sorted over a full turn,
// and for each of the m' cells of a half turn its g numerator and the real parts of
// gamma1, gamma2.  Arrays have a stride of MM cells per term (MM + 1 angles).
// A cell's integral is sin(t2 - t1) g / (D1 D2), Dk = gamma1 cos tk + gamma2 sin tk at its two
// walls.  Re gamma changes from cell to cell by the rows whose sides change there, and those
// vanish at the wall between: the two cells of a wall have the same D there.  So a wall holds
// its direction and Re D, and with the cell after it the numerator; a grid point adds Im D =
// (b1 - x) cos t + (b2 - y) sin t.
struct Wall2D {
    double c, s;      // cos, sin of the wall's angle
    double r, r2;     // Re D and its square
    double nre, nim;  // g sin(t2 - t1) of the cell that begins here
};
// What the reference's other form of the integral needs (gamma1 near zero), per cell.
struct Cell2D {
    double g1r, g2r;  // Re gamma
    cplx g;           // g numerator
};

struct Cpdf2D {
    int MM;
    int* mc;       // cells per term
    double* b2;    // b of the two states
    Wall2D* wall;  // MM + 1 walls per term
    Cell2D* cell;  // MM cells per term
};

__device__ inline Wall2D wall2d(double s1, double c1, double s2, double c2, double g1re, double g2re, cplx g) {
    const double sd = s2 * c1 - s1 * c2, r = g1re * c1 + g2re * s1;
    return Wall2D{c1, s1, r, r * r, g.re * sd, g.im * sd};
}

constexpr double kIntegralGammaEps = 1e-8;  // INTEGRAL_GAMMA_EPS, cauchy_constants.hpp:76
constexpr int kZeroHpMarker = 32;           // ZERO_HP_MARKER_VALUE, cpdf_ndim.hpp:371

// Integral of one cell at (x1, x2) (marg2d_eval_term_for_cpdf, cpdf_ndim.hpp:1603-1636);
// `singular` is set where the reference stops with a singularity error.
__device__ inline double cpdf2d_cell(double s1, double c1, double s2, double c2, double g1re, double g2re,
                                     double g1im, double g2im, cplx g, bool check_g1, bool& singular) {
    cplx ga1 = cmake(g1re, g1im), ga2 = cmake(g2re, g2im);
    if (check_g1 && fabs(g1re) < kIntegralGammaEps) {
        if (fabs(g2re) < kIntegralGammaEps && fabs(g2im) < kIntegralGammaEps) {
            singular = true;
            return 0.0;
        }
        const cplx lo = cdiv(csub(cscale(ga1, s1), cscale(ga2, c1)), cadd(cscale(ga1, c1), cscale(ga2, s1)));
        const cplx hi = cdiv(csub(cscale(ga1, s2), cscale(ga2, c2)), cadd(cscale(ga1, c2), cscale(ga2, s2)));
        const cplx sq = cadd(cmul(ga1, ga1), cmul(ga2, ga2));
        return cmul(csub(hi, lo), cdiv(g, sq)).re;
    }
    // The reference's form, sin t2 / (g1 (g1 cos t2 + g2 sin t2)) - (the same at t1), equals
    // sin(t2 - t1) / (D1 D2) with Dk = g1 cos tk + g2 sin tk exactly: one complex quotient
    // instead of two, and no cancellation between the two limits.
    const cplx d1 = cadd(cscale(ga1, c1), cscale(ga2, s1));
    const cplx d2 = cadd(cscale(ga1, c2), cscale(ga2, s2));
    const double sd = s2 * c1 - s1 * c2;
    return cdiv(cscale(g, sd), cmul(d1, d2)).re;
}

template <int D>
__global__ void k_cpdf2d_terms(TermPool P, int n, int i1, int i2, VecArg bar_nu, const uint32_t* __restrict__ gkeys,
                               const cplx* __restrict__ gvals, double x0, double y0, Cpdf2D C,
                               double* __restrict__ direct, int* __restrict__ err) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int m = P.m[i];
    const int MM = C.MM;
    const double* A = P.A + (int64_t)i * P.MM * D;
    const double* p = P.p + (int64_t)i * P.MM;
    double wa[2 * kMaxM], wp[kMaxM], wa2[2 * kMaxM], wp2[kMaxM], th[2 * kMaxM];
    int cmap[kMaxM], csm[kMaxM], fidx[kMaxM];
    bool F[kMaxM];
    // columns of the two states; zero rows marked, the others L1-normalised
    for (int r = 0; r < m; r++) {
        double a0 = A[r * D + i1], a1 = A[r * D + i2];
        const double f0 = fabs(a0), f1 = fabs(a1);
        wp[r] = p[r];
        if (f0 < kMuEps && f1 < kMuEps) {
            cmap[r] = csm[r] = fidx[r] = kZeroHpMarker;
            F[r] = false;
        } else {
            const double sa = f0 + f1;
            wa[2 * r] = a0 / sa;
            wa[2 * r + 1] = a1 / sa;
            wp[r] *= sa;
            F[r] = true;
        }
    }
    // +/- equal rows merged into the first of them
    int u = 0;
    for (int r = 0; r < m; r++) {
        if (!F[r]) continue;
        cmap[r] = u;
        csm[r] = 1;
        fidx[r] = r;
        wp2[u] = wp[r];
        for (int j = r + 1; j < m; j++) {
            if (!F[j]) continue;
            const bool pos = (fabs(wa[2 * r] - wa[2 * j]) < kCoalignEps) && (fabs(wa[2 * r + 1] - wa[2 * j + 1]) < kCoalignEps);
            if (pos) {
                cmap[j] = u;
                csm[j] = 1;
                F[j] = false;
                fidx[j] = r;
                wp2[u] += wp[j];
                continue;
            }
            const bool neg = (fabs(wa[2 * r] + wa[2 * j]) < kCoalignEps) && (fabs(wa[2 * r + 1] + wa[2 * j + 1]) < kCoalignEps);
            if (neg) {
                cmap[j] = u;
                csm[j] = -1;
                F[j] = false;
                fidx[j] = r;
                wp2[u] += wp[j];
            }
        }
        u++;
    }
    {
        int k = 0;
        for (int r = 0; r < m; r++)
            if (fidx[r] == r) {
                wa2[2 * k] = wa[2 * r];
                wa2[2 * k + 1] = wa[2 * r + 1];
                k++;
            }
    }
    // cell wall angles over a full turn, ascending (marg2d_get_cell_wall_angles)
    for (int r = 0; r < u; r++) {
        const double a0 = wa2[2 * r], a1 = wa2[2 * r + 1];
        double px, py;
        if (fabs(a0) < fabs(a1)) {
            px = 1.0;
            py = -a0 / a1;
        } else {
            px = -a1 / a0;
            py = 1.0;
        }
        double t1 = atan2(py, px);
        if (t1 < 0) t1 += kPi;
        th[2 * r] = t1;
        th[2 * r + 1] = t1 + kPi;
    }
    for (int a = 1; a < 2 * u; a++) {
        const double v = th[a];
        int b = a - 1;
        while (b >= 0 && th[b] > v) {
            th[b + 1] = th[b];
            b--;
        }
        th[b + 1] = v;
    }
    const double bx = P.b[(int64_t)i * D + i1], by = P.b[(int64_t)i * D + i2];
    const double g1im = bx - x0, g2im = by - y0;
    const bool check_g1 = fabs(g1im) < kIntegralGammaEps;
    const int top = 1 << (m - 1), rev = (1 << m) - 1;
    const int64_t go = P.gp_off[i];
    const int gn = P.gp_n[i];
    const int64_t co = (int64_t)i * MM;
    double total = 0.0;
    bool singular = false;
    double s1 = 0.0, c1 = 0.0;
    if (u > 0) {
        s1 = sin(th[0]);
        c1 = cos(th[0]);
    }
    for (int c = 0; c < u; c++) {
        // sign vector of the cell from its middle direction (marg2d_get_SVs)
        const double t = (th[c + 1] + th[c]) / 2.0;
        const double ptx = cos(t), pty = sin(t);
        uint32_t neg = 0;  // bit j: row j of the cut arrangement is negative in this cell
        for (int j = 0; j < u; j++)
            if (!(wa2[2 * j] * ptx + wa2[2 * j + 1] * pty > 0)) neg |= 1u << j;
        int enc = 0;
        for (int j = 0; j < m; j++) {
            if (cmap[j] == kZeroHpMarker) {
                double ip = 0.0;
                for (int k = 0; k < D; k++) ip += A[j * D + k] * bar_nu.v[k];
                if (ip < 0) enc |= 1 << j;
            } else {
                const int sv = ((neg >> cmap[j]) & 1u) ? -1 : 1;
                if (sv * csm[j] < 0) enc |= 1 << j;
            }
        }
        const cplx g = lookup_num(enc, top, rev, gkeys + go, gvals + go, gn);
        double g1re = 0.0, g2re = 0.0;
        for (int j = 0; j < u; j++) {
            const double sv = ((neg >> j) & 1u) ? -1.0 : 1.0;
            g1re -= (wa2[2 * j] * wp2[j]) * sv;
            g2re -= (wa2[2 * j + 1] * wp2[j]) * sv;
        }
        const double s2 = sin(th[c + 1]), c2 = cos(th[c + 1]);
        total += cpdf2d_cell(s1, c1, s2, c2, g1re, g2re, g1im, g2im, g, check_g1, singular);
        C.wall[co + i + c] = wall2d(s1, c1, s2, c2, g1re, g2re, g);
        C.cell[co + c] = Cell2D{g1re, g2re, g};
        s1 = s2;
        c1 = c2;
        if (c == u - 1) {
            const double r = g1re * c2 + g2re * s2;
            C.wall[co + i + u] = Wall2D{c2, s2, r, r * r, 0.0, 0.0};
        }
    }
    C.mc[i] = u;
    C.b2[2 * i] = bx;
    C.b2[2 * i + 1] = by;
    direct[i] = total;
    if (singular) atomicOr(err, 1);
}

// Partial sums over one chunk of terms for kGridLanes * P grid points (the cached cell
// integrals, marg2d_cached_eval_term_for_cpdf, cpdf_ndim.hpp:1654-1735).
//
// FP64 VALU bound.  A wavefront holds P points per lane and goes through a quarter of the
// chunk's terms, whose walls it reads as scalars (every lane is at the same term).  The sum over a
// term's cells is sum_c Re(n_c q_c q_c+1) with q = 1 / D, one q per wall instead of one quotient
// per cell, and two walls share a reciprocal: about 16 operations a wall and point, where the
// quotient per cell took about 35.  A sum that is not finite (some |D|^2 left the range of a
// double) and a term with |b1 - x| < kIntegralGammaEps (the reference's other form) are
// evaluated cell by cell.  101 x 101 points, 579k terms of 13 cells: 110.5 ms before.
constexpr int kGridLanes = 64;
constexpr int kGridWaves = 4;
template <int P>
__global__ void __launch_bounds__(kGridLanes* kGridWaves) k_cpdf2d_grid(Cpdf2D C, int n, int chunk_terms,
                                                                        const double* __restrict__ px,
                                                                        const double* __restrict__ py, int npts,
                                                                        double* __restrict__ part,
                                                                        int* __restrict__ err) {
    __shared__ double sh[kGridWaves][P][kGridLanes];
    const int lane = threadIdx.x % kGridLanes;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kGridLanes));
    const int chunk = blockIdx.y;
    const int per = (chunk_terms + kGridWaves - 1) / kGridWaves;
    const int t0 = min(n, chunk * chunk_terms + w * per);
    const int t1 = min(min(n, (chunk + 1) * chunk_terms), t0 + per);
    const int k0 = blockIdx.x * kGridLanes * P + lane;
    const int MM = C.MM;
    double x[P], y[P], acc[P];
#pragma unroll
    for (int j = 0; j < P; j++) {
        const int k = min(k0 + j * kGridLanes, npts - 1);
        x[j] = px[k];
        y[j] = py[k];
        acc[j] = 0.0;
    }
    bool singular = false;
    for (int64_t t = t0; t < t1; t++) {
        const int u = C.mc[t];
        if (u <= 0) continue;
        const Wall2D* __restrict__ W = C.wall + t * (MM + 1);
        const double bx = C.b2[2 * t], by = C.b2[2 * t + 1];
        double gx[P], gy[P], sum[P], qr[P], qi[P];
        bool plain = true;
#pragma unroll
        for (int j = 0; j < P; j++) {
            gx[j] = bx - x[j];
            gy[j] = by - y[j];
            plain &= !(fabs(gx[j]) < kIntegralGammaEps);
            sum[j] = 0.0;
            const double i0 = __builtin_fma(gx[j], W[0].c, gy[j] * W[0].s);
            const double v = fast_rcp(__builtin_fma(i0, i0, W[0].r2));
            qr[j] = W[0].r * v;
            qi[j] = -(i0 * v);
        }
        if (__all(plain)) {
            int c = 0;
            for (; c + 1 < u; c += 2) {
                const Wall2D wa = W[c + 1], wb = W[c + 2];
                const double n0r = W[c].nre, n0i = W[c].nim;
#pragma unroll
                for (int j = 0; j < P; j++) {
                    const double ia = __builtin_fma(gx[j], wa.c, gy[j] * wa.s);
                    const double ib = __builtin_fma(gx[j], wb.c, gy[j] * wb.s);
                    const double da = __builtin_fma(ia, ia, wa.r2), db = __builtin_fma(ib, ib, wb.r2);
                    const double v = fast_rcp(da * db);
                    const double va = v * db, vb = v * da;
                    const double ar = wa.r * va, ai = -(ia * va), br = wb.r * vb, bi = -(ib * vb);
                    const double ur = __builtin_fma(n0r, qr[j], -(n0i * qi[j]));
                    const double ui = __builtin_fma(n0r, qi[j], n0i * qr[j]);
                    const double vr = __builtin_fma(wa.nre, br, -(wa.nim * bi));
                    const double vi = __builtin_fma(wa.nre, bi, wa.nim * br);
                    // Re((n0 q + na qb) qa): both cells share the wall between them
                    const double er = ur + vr, ei = ui + vi;
                    sum[j] = __builtin_fma(er, ar, __builtin_fma(-ei, ai, sum[j]));
                    qr[j] = br;
                    qi[j] = bi;
                }
            }
            if (c < u) {
                const Wall2D wa = W[c + 1];
                const double n0r = W[c].nre, n0i = W[c].nim;
#pragma unroll
                for (int j = 0; j < P; j++) {
                    const double ia = __builtin_fma(gx[j], wa.c, gy[j] * wa.s);
                    const double v = fast_rcp(__builtin_fma(ia, ia, wa.r2));
                    const double ar = wa.r * v, ai = -(ia * v);
                    const double ur = __builtin_fma(n0r, qr[j], -(n0i * qi[j]));
                    const double ui = __builtin_fma(n0r, qi[j], n0i * qr[j]);
                    sum[j] = __builtin_fma(ur, ar, __builtin_fma(-ui, ai, sum[j]));
                }
            }
#pragma unroll
            for (int j = 0; j < P; j++) plain &= is_finite(sum[j]);
        }
        if (!__all(plain)) {
            const Cell2D* __restrict__ L = C.cell + t * MM;
#pragma unroll 1
            for (int j = 0; j < P; j++) {
                double z = 0.0;
                const bool check_g1 = fabs(gx[j]) < kIntegralGammaEps;
                for (int c = 0; c < u; c++)
                    z += cpdf2d_cell(W[c].s, W[c].c, W[c + 1].s, W[c + 1].c, L[c].g1r, L[c].g2r, gx[j], gy[j], L[c].g,
                                     check_g1, singular);
                sum[j] = z;
            }
        }
#pragma unroll
        for (int j = 0; j < P; j++) acc[j] += sum[j];
    }
#pragma unroll
    for (int j = 0; j < P; j++) sh[w][j][lane] = acc[j];
    __syncthreads();
    if (w == 0)
#pragma unroll
        for (int j = 0; j < P; j++) {
            const int k = k0 + j * kGridLanes;
            double z = sh[0][j][lane];
            for (int v = 1; v < kGridWaves; v++) z += sh[v][j][lane];
            if (k < npts) part[(int64_t)chunk * npts + k] = z;
        }
    if (singular) atomicOr(err, 1);
}


// ------------------------------------------------------------ relative system (two estimators)
// The relative system rel = secondary - primary, transformed to 2D by Trel (2 x d),
// as get_marg2d_relative_and_transformed_cpdf builds it (cauchy_prediction.hpp:497-650):
// one relative term per (primary term, secondary term) pair, A = [-A_p; A_s] Trel^T,
// p = [p_p; p_s], b = Trel (b_s - b_p).  Per pair: its moment contribution
// (eval_rel_sys_moments_for_term, 207-286), its cell data for the density
// (cache_rel_marg2d_term_for_cpdf, 306-443) and whether the term is approximated out
// (approx_out_rel_marg2d_term_for_cpdf, 445-471).
struct RsysArgs {
    double T[2 * kMaxD];   // Trel, row-major 2 x d
    double nu2[2];         // Trel bar_nu
    double nu[kMaxD];      // bar_nu (full state)
    double norm_fact;      // (1 / 2pi)^2 / (Re fz_p Re fz_s)
    double eps;            // term approximation threshold
};

__device__ inline double sgn_d(double x) { return (double)((x > 0) - (x < 0)); }

// A pair's rows are its two terms' rows, so everything about a row is formed once per term
// (k_rsys_terms), where one thread per pair formed all of it in private memory: u angles, 2 u
// sines and cosines, a sort and u^2 sums and merge tests (u rows): 119 ms for two 5-state
// estimators of three steps, 4.6 ms in the two passes below.  A row vanishes on a line through the origin, at angle th in [0, pi]; going
// round, its side flips there and nowhere else within half a turn.  So a term's lines in order,
// with its Re gamma sums and g value before each, are all that the cells of a pair need: the
// cells lie between the merged lines of both terms, sums add and g values multiply.
struct RsysStep {
    double th, s, c;    // the line's angle (infinity after the last line), sin, cos
    double a0, a1;      // its row, L1-normalised
    double g1, g2;      // Re gamma of the term's rows before the line
    double gre, gim, gabs;  // the term's g value before the line, and its modulus
};
struct RsysTerm {
    double ty0, ty1;  // the rows' shares of Re y at bar_nu, summed
    cplx g;           // the term's g value there
};

// One wavefront per term; sg: -1 for the primary's rows, +1 for the secondary's.
// steps: [term][MM + 1]; shares ([term][MM], may be null): every row's share of Re y.
__global__ __launch_bounds__(64) void k_rsys_terms(TermPool P, int n, int d, double sg,
                                                   const uint32_t* __restrict__ keys, const cplx* __restrict__ vals,
                                                   RsysArgs R, RsysStep* __restrict__ steps,
                                                   RsysTerm* __restrict__ terms, double2* __restrict__ shares) {
    __shared__ double ty[2][kMaxM];
    __shared__ double th[kMaxM], sn[kMaxM], cs[kMaxM], a0s[kMaxM], a1s[kMaxM], bp[kMaxM];
    __shared__ int row[kMaxM];
    const int t = blockIdx.x;
    if (t >= n) return;
    const int r = threadIdx.x;
    const int MM = P.MM;
    const int m = P.m[t];
    const int mask = (1 << m) - 1, top = 1 << (m - 1);
    double a0 = 0, a1 = 0, p = 0, ang = 0, c = 1, s = 0, beta = 0;
    bool zero = true, neg_nu = false, neg = false;
    if (r < m) {
        const double* A = P.A + ((int64_t)t * MM + r) * d;
        for (int j = 0; j < d; j++) a0 += (A[j] * sg) * R.T[j];
        for (int j = 0; j < d; j++) a1 += (A[j] * sg) * R.T[d + j];
        p = P.p[(int64_t)t * MM + r];
        // rows that vanish under Trel keep the side of bar_nu, the others are L1-normalised
        const double f0 = fabs(a0), f1 = fabs(a1);
        zero = f0 < kMuEps && f1 < kMuEps;
        double ds = 0.0;
        if (zero) {
            for (int j = 0; j < d; j++) ds += (A[j] * sg) * R.nu[j];
        } else {
            const double sa = f0 + f1;
            a0 /= sa;
            a1 /= sa;
            p *= sa;
            ds = a0 * R.nu2[0] + a1 * R.nu2[1];
            const bool flat = fabs(a0) < fabs(a1);
            ang = flat ? atan2(-a0 / a1, 1.0) : atan2(1.0, -a1 / a0);
            if (ang < 0) ang += kPi;
            sincos(ang, &s, &c);
            beta = a0 * s - a1 * c > 0 ? 1.0 : -1.0;  // the row's side before its line
        }
        const double sgi = sgn_d(ds);
        neg_nu = sgi < 0;
        neg = zero ? ds < 0 : beta < 0;
        ty[0][r] = a0 * (p * sgi);
        ty[1][r] = a1 * (p * sgi);
        if (shares) shares[(int64_t)t * MM + r] = make_double2(ty[0][r], ty[1][r]);
    }
    const int enc_nu = (int)__ballot(neg_nu), enc0 = (int)__ballot(neg);
    const bool line = r < m && !zero;
    const int u = __popcll(__ballot(line));
    // the lines in order of their angles (of the rows, where equal)
    int rank = 0;
    for (int q = 0; q < m; q++) {
        const double o = __shfl(ang, q, kWave);
        const bool lq = __shfl((int)line, q, kWave) != 0;
        rank += lq && (o < ang || (o == ang && q < r));
    }
    if (line) {
        th[rank] = ang;
        sn[rank] = s;
        cs[rank] = c;
        a0s[rank] = a0;
        a1s[rank] = a1;
        bp[rank] = beta * p;
        row[rank] = r;
    }
    __syncthreads();
    const uint32_t* pk = keys + P.gp_off[t];
    const cplx* pv = vals + P.gp_off[t];
    const int pn = P.gp_n[t];
    if (r <= u) {
        // before line r: lines 0 .. r-1 crossed
        int enc = enc0;
        double g1 = 0.0, g2 = 0.0;
        for (int j = 0; j < u; j++) {
            const double w = j < r ? bp[j] : -bp[j];
            g1 += a0s[j] * w;
            g2 += a1s[j] * w;
            if (j < r) enc ^= 1 << row[j];
        }
        const cplx g = lookup_num(enc, top, mask, pk, pv, pn);
        RsysStep o;
        const bool end = r == u;
        o.th = end ? __builtin_inf() : th[r];
        o.s = end ? 0.0 : sn[r];
        o.c = end ? 1.0 : cs[r];
        o.a0 = end ? 0.0 : a0s[r];
        o.a1 = end ? 0.0 : a1s[r];
        o.g1 = g1;
        o.g2 = g2;
        o.gre = g.re;
        o.gim = g.im;
        o.gabs = hypot(g.re, g.im);
        steps[(int64_t)t * (MM + 1) + r] = o;
    }
    if (r == 0) {
        RsysTerm o;
        o.ty0 = o.ty1 = 0.0;
        for (int j = 0; j < m; j++) {
            o.ty0 += ty[0][j];
            o.ty1 += ty[1][j];
        }
        o.g = lookup_num(enc_nu, top, mask, pk, pv, pn);
        terms[t] = o;
    }
}

// One thread per pair walks the lines of both terms in order: per line one 80-byte step of
// either term, two sums, a product and the cell it closes, in registers.  Lines that are the
// same, the last and the first included, bound no cell between them.  Rows that agree within
// kCoalignEps up to sign count as one, the first of them in row order; where neighbouring lines
// agree so far but differ by more than kSameLine, the pair is left to k_rsys_near (keep 2, or -1
// cells).  First (CELLS false) every pair's moments and whether the approximation keeps
// it; then (CELLS true) the cells of the n kept pairs idx[0 .. n), which the grid reads.  The
// cells are 80 bytes each in separate stretches per lane, and writing them bounds the second
// pass, so pairs that are dropped write none: 2.6 + 1.9 ms, where one pass that wrote every
// pair's took 19.8 ms.  The first is bound by the latency of the steps' loads.
constexpr double kSameLine = 1e-12;
constexpr uint8_t kKeepNear = 2;
__device__ inline bool same_line(double x0, double x1, double y0, double y1, double eps) {
    return (fabs(x0 - y0) < eps && fabs(x1 - y1) < eps) || (fabs(x0 + y0) < eps && fabs(x1 + y1) < eps);
}

template <bool CELLS>
__global__ __launch_bounds__(256) void k_rsys_pairs(TermPool P, TermPool S, int ns, int64_t n, int d,
                                                    const int* __restrict__ idx,
                                                    const RsysStep* __restrict__ psteps,
                                                    const RsysTerm* __restrict__ pterms,
                                                    const RsysStep* __restrict__ ssteps,
                                                    const RsysTerm* __restrict__ sterms,
                                                    const double2* __restrict__ sshares, RsysArgs R, Cpdf2D C,
                                                    double* __restrict__ mom, uint8_t* __restrict__ keep) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int64_t q = CELLS ? idx[k] : k;
    const int tp = (int)(q / ns), ts = (int)(q % ns);
    double b2[2] = {0.0, 0.0};
    for (int j = 0; j < d; j++) {
        const double br = S.b[(int64_t)ts * d + j] - P.b[(int64_t)tp * d + j];
        b2[0] += R.T[j] * br;
        b2[1] += R.T[d + j] * br;
    }
    if constexpr (!CELLS) {
        const RsysTerm a = pterms[tp], b = sterms[ts];
        const cplx g = cmul(a.g, b.g);
        // one sum over the primary's rows, then the secondary's: the covariance, a difference
        // of far larger numbers, shows its rounding
        double ty0 = a.ty0, ty1 = a.ty1;
        const int ms = S.m[ts];
        for (int j = 0; j < ms; j++) {
            const double2 v = sshares[(int64_t)ts * S.MM + j];
            ty0 += v.x;
            ty1 += v.y;
        }
        const cplx y0 = cmake(-ty0, b2[0]), y1 = cmake(-ty1, b2[1]);
        // component c of pair q at mom[c * npairs + q] (column-major: contiguous column sums)
        const cplx gy0 = cmul(g, y0), gy1 = cmul(g, y1);
        const cplx c00 = cmul(gy0, y0), c01 = cmul(gy0, y1), c10 = cmul(gy1, y0), c11 = cmul(gy1, y1);
        const double v[14] = {g.re,   g.im,   gy0.re, gy0.im, gy1.re, gy1.im, c00.re,
                              c00.im, c01.re, c01.im, c10.re, c10.im, c11.re, c11.im};
#pragma unroll
        for (int c = 0; c < 14; c++) mom[c * n + q] = v[c];
    }
    const RsysStep* pp = psteps + (int64_t)tp * (P.MM + 1);
    const RsysStep* ps = ssteps + (int64_t)ts * (S.MM + 1);
    RsysStep A = *pp, B = *ps;
    const int64_t w0 = k * (C.MM + 1), c0 = k * C.MM;
    double total = 0.0, g1 = 0.0, g2 = 0.0;
    bool keep_term = false;
    int u = 0;
    // takes cell u between the lower and the upper line, both terms' states being those in it
    auto cell = [&](double s1, double c1, double s2, double c2) {
        g1 = A.g1 + B.g1;
        g2 = A.g2 + B.g2;
        if constexpr (CELLS) {
            const cplx g = cmul(cmake(A.gre, A.gim), cmake(B.gre, B.gim));
            C.wall[w0 + u] = wall2d(s1, c1, s2, c2, g1, g2, g);
            C.cell[c0 + u] = Cell2D{g1, g2, g};
        } else {
            // the approximation's bound on the cell's contribution
            const double den1 = g1 * (g1 * c1 + g2 * s1);
            const double den2 = g1 * (g1 * c2 + g2 * s2);
            if (fabs(den1) < 1e-14 || fabs(den2) < 1e-14) keep_term = true;
            const double gr = A.gabs * B.gabs;
            total += fabs((gr * s2) / den2) + fabs((gr * s1) / den1);
        }
        u++;
    };
    bool near = false;
    // whether the row x, neighbour of y, has the same line
    auto coaligned = [&](double x0, double x1, double y0, double y1) {
        if (!same_line(x0, x1, y0, y1, kCoalignEps)) return false;
        near |= !same_line(x0, x1, y0, y1, kSameLine);
        return true;
    };
    double fs = 0, fc = 1, fa0 = 0, fa1 = 0;  // the first line
    double ls = 0, lc = 1, la0 = 0, la1 = 0;  // the line the open cell begins at
    bool open = false;
    bool fromA = A.th <= B.th;
    while (fmin(A.th, B.th) < __builtin_inf()) {
        const double s = fromA ? A.s : B.s, c = fromA ? A.c : B.c;
        const double a0 = fromA ? A.a0 : B.a0, a1 = fromA ? A.a1 : B.a1;
        if (open) {
            cell(ls, lc, s, c);
        } else {
            fs = s;
            fc = c;
            fa0 = a0;
            fa1 = a1;
        }
        open = true;
        ls = s;
        lc = c;
        la0 = a0;
        la1 = a1;
        // cross the line and those coaligned with it
        double n0, n1, nt;
        do {
            const RsysStep N = *(fromA ? ++pp : ++ps);
            if (fromA) A = N;
            else B = N;
            fromA = A.th <= B.th;
            n0 = fromA ? A.a0 : B.a0;
            n1 = fromA ? A.a1 : B.a1;
            nt = fromA ? A.th : B.th;
        } while (nt < __builtin_inf() && coaligned(n0, n1, la0, la1));
        if (near) break;
    }
    if (open) coaligned(la0, la1, fa0, fa1);
    if (near) {
        if constexpr (CELLS) C.mc[k] = -1;
        else keep[k] = kKeepNear;
        return;
    }
    if (open) {
        // the last cell ends at the first line's other half, or, where that is coaligned with
        // the last line, has ended there
        const bool ended = u > 0 && same_line(la0, la1, fa0, fa1, kCoalignEps);
        const double es = ended ? ls : -fs, ec = ended ? lc : -fc;
        if (!ended) cell(ls, lc, es, ec);
        if constexpr (CELLS) {
            const double r = g1 * ec + g2 * es;
            C.wall[w0 + u] = Wall2D{ec, es, r, r * r, 0.0, 0.0};
        }
    }
    if constexpr (CELLS) {
        C.mc[k] = u;
        C.b2[2 * k] = b2[0];
        C.b2[2 * k + 1] = b2[1];
    } else {
        total *= (2 * R.norm_fact);
        keep[k] = (keep_term || !(fabs(total) < R.eps)) ? 1 : 0;
    }
}

// The pairs that k_rsys_pairs left: rows that agree within kCoalignEps up to sign, but not to
// rounding, are merged as the reference merges them (marg2d_remove_zeros_and_coalign,
// cpdf_ndim.hpp:405-517): in row order, the primary's rows first, each row that is left takes
// in every later one that agrees with it, and the cells are those of the rows that are left.  A
// wavefront per pair, a lane per row and then per cell; two estimators of nearly equal systems
// have such pairs, others hardly any, and then a wavefront only reads 64 pairs' flags at a time.
// (Private arrays with computed indices, a thread per pair, are not an option: this compiler
// keeps them in registers and gave wrong densities.)
template <bool CELLS>
__global__ __launch_bounds__(256) void k_rsys_near(TermPool P, TermPool S, int ns, int64_t n, int d,
                                                   const int* __restrict__ idx, const uint32_t* __restrict__ pkeys,
                                                   const cplx* __restrict__ pvals, const uint32_t* __restrict__ skeys,
                                                   const cplx* __restrict__ svals, RsysArgs R, Cpdf2D C,
                                                   uint8_t* __restrict__ keep) {
    const int lane = wave_lane();
    const int64_t waves = (int64_t)gridDim.x * (blockDim.x / kWave);
    int64_t k0 = ((int64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave) * kWave;
    for (; k0 < n; k0 += waves * kWave) {
        const bool mine = k0 + lane < n && (CELLS ? C.mc[k0 + lane] < 0 : keep[k0 + lane] == kKeepNear);
        for (uint64_t todo = __ballot(mine); todo; todo &= todo - 1) {
            const int64_t k = k0 + __ffsll((unsigned long long)todo) - 1;
            const int64_t q = CELLS ? idx[k] : k;
            const int tp = (int)(q / ns), ts = (int)(q % ns);
            const int mp = P.m[tp], ms = S.m[ts], m = mp + ms;
            // this lane's row, normalised; those that vanish keep the side of nu
            const bool pr = lane < mp, row = lane < m;
            double x0 = 0.0, x1 = 0.0, w = 0.0, ip = 0.0;
            if (row) {
                const double* A = pr ? P.A + ((int64_t)tp * P.MM + lane) * d : S.A + ((int64_t)ts * S.MM + lane - mp) * d;
                const double sg = pr ? -1.0 : 1.0;
                for (int j = 0; j < d; j++) {
                    x0 += (A[j] * sg) * R.T[j];
                    x1 += (A[j] * sg) * R.T[d + j];
                    ip += (A[j] * sg) * R.nu[j];
                }
                w = pr ? P.p[(int64_t)tp * P.MM + lane] : S.p[(int64_t)ts * S.MM + lane - mp];
            }
            const bool line = row && !(fabs(x0) < kMuEps && fabs(x1) < kMuEps);
            if (line) {
                const double sa = fabs(x0) + fabs(x1);
                x0 /= sa;
                x1 /= sa;
                w *= sa;
            }
            // the row that takes this one in, and whether they point opposite ways
            int into = lane;
            bool opposite = false;
            for (int r = 0; r < m; r++) {
                const double y0 = __shfl(x0, r, kWave), y1 = __shfl(x1, r, kWave);
                const bool free_row = line && into == lane;
                const uint64_t free_rows = __ballot(free_row);
                if (!((free_rows >> r) & 1u) || !free_row || lane <= r) continue;
                const bool pos = fabs(y0 - x0) < kCoalignEps && fabs(y1 - x1) < kCoalignEps;
                if (pos || (fabs(y0 + x0) < kCoalignEps && fabs(y1 + x1) < kCoalignEps)) {
                    into = r;
                    opposite = !pos;
                }
            }
            const bool left = line && into == lane;
            const uint64_t lefts = __ballot(left);
            const int u = __popcll(lefts);
            for (int j = 0; j < m; j++) {  // the weights of what it took in, in row order
                const double wj = __shfl(w, j, kWave);
                const int rj = __shfl(into, j, kWave);
                const bool lj = __shfl((int)line, j, kWave) != 0;
                if (left && lj && rj == lane && j > lane) w += wj;
            }
            double t = 0.0, sn = 0.0, cs = 1.0;
            if (left) {
                const bool flat = fabs(x0) < fabs(x1);
                t = flat ? atan2(-x0 / x1, 1.0) : atan2(1.0, -x1 / x0);
                if (t < 0) t += kPi;
                sn = sin(t);
                cs = cos(t);
            }
            // place of its line going round; side of the row before the line
            int place = 0;
            for (int j = 0; j < m; j++) {
                const double tj = __shfl(t, j, kWave);
                place += ((lefts >> j) & 1u) && (tj < t || (tj == t && j < lane));
            }
            const bool neg = left && !(x0 * sn - x1 * cs > 0);
            const bool neg_into = __shfl((int)neg, into, kWave) != 0;
            const bool before = line ? neg_into != opposite : row && ip < 0;
            const int at = __shfl(place, into, kWave);  // of the line it changes sides at
            const double signedw = neg ? -w : w;
            // lane c takes the cell between line c and the next, the last one half a turn on
            double s1 = 0.0, c1 = 1.0, s2 = 0.0, c2 = 1.0, g1 = 0.0, g2 = 0.0;
            uint32_t enc = 0;
            for (int j = 0; j < m; j++) {
                const bool lj = __shfl((int)line, j, kWave) != 0;
                const bool crossed = __shfl(at, j, kWave) <= lane;
                const bool bj = __shfl((int)before, j, kWave) != 0;
                const double y0 = __shfl(x0, j, kWave), y1 = __shfl(x1, j, kWave), wj = __shfl(signedw, j, kWave);
                const double tj = __shfl(t, j, kWave), sj = __shfl(sn, j, kWave), cj = __shfl(cs, j, kWave);
                const int pj = __shfl(place, j, kWave);
                enc |= (uint32_t)(bj != (lj && crossed)) << j;
                if ((lefts >> j) & 1u) {
                    const double v = crossed ? -wj : wj;
                    g1 -= y0 * v;
                    g2 -= y1 * v;
                    if (pj == lane) {
                        s1 = sj;
                        c1 = cj;
                    }
                    if (pj == lane + 1) {
                        s2 = sj;
                        c2 = cj;
                    }
                    if (pj == 0 && lane == u - 1) {
                        s2 = sin(tj + kPi);
                        c2 = cos(tj + kPi);
                    }
                }
            }
            cplx g = cmake(0.0, 0.0);
            if (lane < u) {
                const int pmask = (1 << mp) - 1, smask = (1 << ms) - 1;
                const int64_t po = P.gp_off[tp], so = S.gp_off[ts];
                g = cmul(lookup_num((int)enc & pmask, 1 << (mp - 1), pmask, pkeys + po, pvals + po, P.gp_n[tp]),
                         lookup_num((int)(enc >> mp), 1 << (ms - 1), smask, skeys + so, svals + so, S.gp_n[ts]));
            }
            if constexpr (CELLS) {
                if (lane < u) {
                    C.wall[k * (C.MM + 1) + lane] = wall2d(s1, c1, s2, c2, g1, g2, g);
                    C.cell[k * C.MM + lane] = Cell2D{g1, g2, g};
                }
                if (lane == u - 1) {
                    const double r = g1 * c2 + g2 * s2;
                    C.wall[k * (C.MM + 1) + u] = Wall2D{c2, s2, r, r * r, 0.0, 0.0};
                }
                if (lane == 0) {
                    double b0 = 0.0, b1 = 0.0;
                    for (int j = 0; j < d; j++) {
                        const double br = S.b[(int64_t)ts * d + j] - P.b[(int64_t)tp * d + j];
                        b0 += R.T[j] * br;
                        b1 += R.T[d + j] * br;
                    }
                    C.mc[k] = u;
                    C.b2[2 * k] = b0;
                    C.b2[2 * k + 1] = b1;
                }
            } else {
                // the approximation's bound on the pair's contribution, as in k_rsys_pairs
                const double den1 = g1 * (g1 * c1 + g2 * s1), den2 = g1 * (g1 * c2 + g2 * s2);
                const bool stays = __any(lane < u && (fabs(den1) < 1e-14 || fabs(den2) < 1e-14));
                const double gr = hypot(g.re, g.im);
                const double bound = fabs((gr * s2) / den2) + fabs((gr * s1) / den1);
                double total = 0.0;
                for (int c = 0; c < u; c++) total += __shfl(bound, c, kWave);
                total *= (2 * R.norm_fact);
                if (lane == 0) keep[k] = (stays || !(fabs(total) < R.eps)) ? 1 : 0;
            }
        }
    }
}

// Partial sums of the columns of a column-major n x cols array: block (b, c) adds the
// fixed slice b of column c; k_colsum_finish adds the slices in order.
constexpr int kColSlices = 256;
__global__ void k_colsum_part(const double* __restrict__ v, int64_t n, double* __restrict__ part) {
    __shared__ double sh[256];
    const int b = blockIdx.x, c = blockIdx.y, t = threadIdx.x;
    const int64_t per = (n + kColSlices - 1) / kColSlices;
    const int64_t lo = b * per, hi = min(n, lo + per);
    const double* col = v + c * n;
    double s = 0.0;
    for (int64_t i = lo + t; i < hi; i += blockDim.x) s += col[i];
    sh[t] = s;
    __syncthreads();
    for (int h = blockDim.x / 2; h > 0; h >>= 1) {
        if (t < h) sh[t] += sh[t + h];
        __syncthreads();
    }
    if (t == 0) part[c * kColSlices + b] = sh[0];
}

__global__ void k_colsum_finish(const double* __restrict__ part, int cols, double* __restrict__ out) {
    const int c = threadIdx.x;
    if (c >= cols) return;
    double s = 0.0;
    for (int b = 0; b < kColSlices; b++) s += part[c * kColSlices + b];
    out[c] = s;
}

// ------------------------------------------------------------------ merged-launch plumbing
// Byte copy of one staged payload or readback (8-byte words when both ends and the length
// allow).
__device__ __forceinline__ void k_copy_bytes(MG<256, 1> mg, const uint8_t* __restrict__ src, uint8_t* __restrict__ dst,
                                             int64_t bytes) {
    const int64_t t = (int64_t)mg.bx * blockDim.x + threadIdx.x;
    const int64_t stride = (int64_t)mg.gx * blockDim.x;
    if ((((uintptr_t)src | (uintptr_t)dst | (uintptr_t)bytes) & 7) == 0) {
        const uint64_t* s = (const uint64_t*)src;
        uint64_t* d = (uint64_t*)dst;
        for (int64_t i = t; i < bytes / 8; i += stride) d[i] = s[i];
    } else {
        for (int64_t i = t; i < bytes; i += stride) dst[i] = src[i];
    }
}

// Stable sort of up to kSmallSort (key, value) pairs by key bits [begin_bit, end_bit) in one
// workgroup: the order a stable device radix sort over the same bits gives.  Slots past n
// hold all-ones keys, which sort after every real key of the same digits (stability keeps
// the real ones first), and are not written back.
constexpr int kSmallSortThreads = 256;
constexpr int kSmallSortItems = 16;
constexpr int kSmallSort = kSmallSortThreads * kSmallSortItems;
template <class K, class V>
__device__ __forceinline__ void k_small_sort(MG<kSmallSortThreads, 1> mg, const K* __restrict__ kin,
                                             K* __restrict__ kout, const V* __restrict__ vin, V* __restrict__ vout,
                                             int n, int begin_bit, int end_bit) {
    (void)mg;
    using Sort = hipcub::BlockRadixSort<K, kSmallSortThreads, kSmallSortItems, V>;
    __shared__ typename Sort::TempStorage tmp;
    K k[kSmallSortItems];
    V v[kSmallSortItems];
    const int base = threadIdx.x * kSmallSortItems;
#pragma unroll
    for (int j = 0; j < kSmallSortItems; j++) {
        const int i = base + j;
        k[j] = i < n ? kin[i] : (K)~(K)0;
        v[j] = i < n ? vin[i] : (V)0;
    }
    Sort(tmp).Sort(k, v, begin_bit, end_bit);
#pragma unroll
    for (int j = 0; j < kSmallSortItems; j++) {
        const int i = base + j;
        if (i < n) {
            kout[i] = k[j];
            vout[i] = v[j];
        }
    }
}

// Largest of n ints in one workgroup (INT_MIN when n = 0, as a device max
// reduction gives).
__device__ __forceinline__ void k_small_max(MG<1024, 1> mg, const int* __restrict__ in, int* __restrict__ out,
                                            int n) {
    (void)mg;
    __shared__ int part[1024];
    int m = INT_MIN;
    for (int i = threadIdx.x; i < n; i += blockDim.x) m = max(m, in[i]);
    part[threadIdx.x] = m;
    __syncthreads();
    for (int o = blockDim.x / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) part[threadIdx.x] = max(part[threadIdx.x], part[threadIdx.x + o]);
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = part[0];
}

// Stable LSD radix sort of (key, value) pairs for inputs of kSmallSort .. kRadixMax items,
// one digit of up to 8 bits per pass, in chunks of kRadixChunk items per block, for many
// estimators at once: (1) each chunk's digit histogram, stored digit-major; (2) an exclusive
// scan over it (k_small_scan) gives every (digit, chunk) its first output slot; (3) each
// chunk sorts itself stably by the digit and writes every item to its digit's slot plus its
// rank among the chunk's items of that digit.  Equal digits keep chunk order and in-chunk
// order, so each pass is stable and the passes over bits [0, end) give the order of a stable
// sort over those bits.
constexpr int kRadixThreads = 256;
constexpr int kRadixItems = 16;
constexpr int kRadixChunk = kRadixThreads * kRadixItems;
constexpr int kRadixBins = 256;
constexpr int kRadixMax = kSmallScan / kRadixBins * kRadixChunk;  // the digit-major scan fits k_small_scan
template <class K>
__device__ __forceinline__ void k_radix_hist(MG<kRadixThreads, 1> mg, const K* __restrict__ keys, int n, int shift,
                                             int bits, int* __restrict__ hist, int nchunks) {
    __shared__ int h[kRadixBins];
    h[threadIdx.x] = 0;
    __syncthreads();
    const int base = mg.bx * kRadixChunk;
    const K mask = (K)((1u << bits) - 1u);
    for (int j = threadIdx.x; j < kRadixChunk; j += kRadixThreads) {
        const int i = base + j;
        if (i < n) atomicAdd(&h[(int)((keys[i] >> shift) & mask)], 1);
    }
    __syncthreads();
    hist[threadIdx.x * nchunks + mg.bx] = h[threadIdx.x];
}
template <class K>
__device__ __forceinline__ void k_radix_scatter(MG<kRadixThreads, 1> mg, const K* __restrict__ kin,
                                                const uint32_t* __restrict__ vin, K* __restrict__ kout,
                                                uint32_t* __restrict__ vout, int n, int shift, int bits,
                                                const int* __restrict__ offs, int nchunks) {
    using Sort = hipcub::BlockRadixSort<K, kRadixThreads, kRadixItems, uint32_t>;
    __shared__ typename Sort::TempStorage tmp;
    __shared__ int first[kRadixBins];
    const int base = mg.bx * kRadixChunk;
    const int nreal = min(n - base, kRadixChunk);
    const K mask = (K)((1u << bits) - 1u);
    K k[kRadixItems];
    uint32_t v[kRadixItems];
    first[threadIdx.x] = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kRadixItems; j++) {
        const int p = threadIdx.x * kRadixItems + j;
        const bool real = p < nreal;
        k[j] = real ? kin[base + p] : (K)~(K)0;
        v[j] = real ? vin[base + p] : 0u;
        if (real) atomicAdd(&first[(int)((k[j] >> shift) & mask)], 1);
    }
    __syncthreads();
    // exclusive scan of the chunk's digit counts: first[d] = items of smaller digits
    const int c = first[threadIdx.x];
    for (int o = 1; o < kRadixBins; o <<= 1) {
        const int add = (int)threadIdx.x >= o ? first[threadIdx.x - o] : 0;
        __syncthreads();
        first[threadIdx.x] += add;
        __syncthreads();
    }
    first[threadIdx.x] -= c;
    // padding keys are all ones: they sort after every real item of the last digit
    Sort(tmp).Sort(k, v, shift, shift + bits);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kRadixItems; j++) {
        const int p = threadIdx.x * kRadixItems + j;
        if (p < nreal) {
            const int dg = (int)((k[j] >> shift) & mask);
            const int dst = offs[dg * nchunks + mg.bx] + (p - first[dg]);
            kout[dst] = k[j];
            vout[dst] = v[j];
        }
    }
}

}  // namespace mce
