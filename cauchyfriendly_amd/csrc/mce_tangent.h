// Forward-mode (tangent-linear) derivatives of the measurement update.
//
// For P directions at once, every term carries the derivatives of its continuous fields
// (A, p, q, b, c, d) and every g-table cell the derivative of its value, with respect to
// the parameters the caller seeds per update (Phi, H, the process scales beta and the
// measurement scale gamma).  Every discrete decision (signs, coalignment, cells, term
// reduction, negligibility, root replacement) is the nominal forward's, taken from the
// same kernels or recomputed with the same arithmetic, so the derivative is that of the
// estimator with its term structure held fixed.  The derivative of a step's measurement
// likelihood fz comes out of the moment sum; nothing is stored between steps except the
// current terms' tangents (the forward is recomputed, step by step, with its tangents).
//
// Forward being differentiated: time_prop / normalize_hps / tp_coalign
// (cauchy_term.hpp:435-531), msmt_update and eval_g_yei (cauchy_term.hpp:84-401),
// mu_coalign (cauchy_term.hpp:533-745), make_gtable_first / make_gtable / add_gtables /
// make_gtables (flattening.hpp:14-568), cache_moments (cauchy_estimator.hpp:307-338).
#pragma once
#include "mce_kernels.h"

namespace mce {

constexpr int kMaxTan = 16;  // directions per estimator

// Per-update seeds: direction k moves Phi by Phi[k], the measurement row by H[k], the
// pre-coaligned process scales by beta[k] and the measurement scale by gamma[k].
struct StepTan {
    double Phi[kMaxTan][kMaxD * kMaxD];
    double H[kMaxTan][kMaxD];
    double beta[kMaxTan][kMaxM];
    double gamma[kMaxTan];
};

// Tangents of a term pool, [term][direction][field].
struct TanPool {
    double *A, *p, *q, *b, *c, *dv;
    int P, MM, d;
    __device__ __host__ double* tA(int64_t i, int k) const { return A + ((i * P + k) * MM) * d; }
    __device__ __host__ double* tp(int64_t i, int k) const { return p + (i * P + k) * MM; }
    __device__ __host__ double* tq(int64_t i, int k) const { return q + (i * P + k) * MM; }
    __device__ __host__ double* tb(int64_t i, int k) const { return b + (i * P + k) * d; }
    __device__ __host__ double* tc(int64_t i, int k) const { return c + i * P + k; }
    __device__ __host__ double* tdv(int64_t i, int k) const { return dv + i * P + k; }
};

__device__ inline double sgn0(double x) { return x > 0 ? 1.0 : (x < 0 ? -1.0 : 0.0); }

// d(a / D) = (da - (a / D) dD) / D for complex a, D.
__device__ inline cplx dquot(cplx a, cplx da, cplx D, cplx dD) {
    const cplx w = cdiv(a, D);
    return cdiv(csub(da, cmul(w, dD)), D);
}

// Index of the parent g-table entry of a half-storage key (eval_gs.hpp:94-153): -1 when
// absent; *cj when the key was reversed (the value enters conjugated).
__device__ inline int lookup_idx(int enc, int top_bit, int rev_mask, const uint32_t* keys, int size, bool* cj) {
    *cj = (enc & top_bit) != 0;
    return bsearch_u32(keys, (uint32_t)(*cj ? (rev_mask ^ enc) : enc), size);
}

// ------------------------------------------------------------------ time propagation
// Tangents through time_prop / normalize_hps / tp_coalign, launched before k_tp on the
// same parents: the nominal rows are formed with k_tp's arithmetic, so the coalignment
// decisions are k_tp's.  Row r: u = A_r Phi^T, n1 = |u|_1, A'_r = u / n1, p'_r = p_r n1,
// then p'_k += beta_j for a coaligned Gamma row j, else the row (Gamma_j, beta_j) is
// appended; b' = Phi b (+ B u, which carries no tangent).
// One wavefront per parent: lanes form the nominal rows, then take a (row, direction) each.
// One thread per parent walked all of them (3-state windows with 14 directions: 79 -> 5 us per
// launch).
template <int D>
__global__ __launch_bounds__(64) void k_tp_tan(TermPool P, TanPool T, int n, const StepConst* __restrict__ sc,
                                               const StepTan* __restrict__ st) {
    __shared__ double An[kMaxShape * D], Ao[kMaxShape * D], n1s[kMaxShape], po[kMaxShape];
    const int i = blockIdx.x;
    if (i >= n || !sc->with_tp) return;
    const int lane = threadIdx.x;
    const int MM = P.MM, NP = T.P;
    const int m = P.m[i];
    const double* b = P.b + (int64_t)i * D;
    if (lane < m) {
        const double* A = P.A + ((int64_t)i * MM + lane) * D;
        double t[D], u[D];
        double n1 = 0;
        for (int k = 0; k < D; k++) t[k] = A[k];
        for (int j = 0; j < D; j++) {
            double s = 0.0;
            for (int k = 0; k < D; k++) s += t[k] * sc->Phi[k + j * D];
            u[j] = s;
        }
        for (int k = 0; k < D; k++) n1 += fabs(u[k]);
        n1s[lane] = n1;
        po[lane] = P.p[(int64_t)i * MM + lane];
        for (int k = 0; k < D; k++) {
            Ao[lane * D + k] = t[k];
            An[lane * D + k] = u[k] / n1;
        }
    }
    __syncthreads();
    // the row that Gamma row j coaligns with (the first), or where it is appended; -1: nowhere
    int crow = -1;  // lane j holds row j's
    int mm = m;
    for (int j = 0; j < sc->ng; j++) {
        bool pos = false, neg = false;
        if (lane < m) coalign_gates(&sc->G[j * D], &An[lane * D], D, pos, neg);
        const unsigned long long hit = __ballot(pos || neg);
        const int r = hit ? __ffsll((long long)hit) - 1 : mm < MM ? mm++ : -1;
        if (lane == j) crow = r;
    }
    for (int it = lane; it < m * NP; it += 64) {
        const int r = it % m, kk = it / m;
        const double* dPhi = st->Phi[kk];
        double* dA = T.tA(i, kk) + r * D;
        double* dp = T.tp(i, kk) + r;
        double t[D], du[D];
        for (int k = 0; k < D; k++) t[k] = dA[k];
        double dn1 = 0;
        for (int j = 0; j < D; j++) {
            double s = 0.0;
            for (int k = 0; k < D; k++) s += t[k] * sc->Phi[k + j * D] + Ao[r * D + k] * dPhi[k + j * D];
            du[j] = s;
            dn1 += sgn0(An[r * D + j]) * s;
        }
        for (int j = 0; j < D; j++) dA[j] = (du[j] - An[r * D + j] * dn1) / n1s[r];
        dp[0] = dp[0] * n1s[r] + po[r] * dn1;
    }
    for (int kk = lane; kk < NP; kk += 64) {
        const double* dPhi = st->Phi[kk];
        double* db = T.tb(i, kk);
        double t[D];
        for (int k = 0; k < D; k++) t[k] = db[k];
        for (int r = 0; r < D; r++) {
            double s = 0.0;
            for (int j = 0; j < D; j++) s += dPhi[r * D + j] * b[j] + sc->Phi[r * D + j] * t[j];
            db[r] = s;
        }
    }
    __syncthreads();
    for (int j = 0; j < sc->ng; j++) {
        const int r = __builtin_amdgcn_readlane(crow, j);
        if (r < 0) continue;
        for (int kk = lane; kk < NP; kk += 64) {
            double* dp = T.tp(i, kk) + r;
            if (r < m) {
                dp[0] += st->beta[kk][j];
            } else {
                for (int k = 0; k < D; k++) T.tA(i, kk)[r * D + k] = 0.0;
                dp[0] = st->beta[kk][j];
            }
        }
    }
}

// ------------------------------------------------------------------ measurement update
// mu_coalign's merges (cauchy_term.hpp:533-745) applied to one direction's tangents of
// the L1-normalised rows: the decisions come from the nominal normalised rows An and
// the H-orthogonality mask, exactly as dev_mu_coalign takes them.
template <int D>
__device__ inline void mu_coalign_tan(const double* An, uint32_t hf, int m, double* dA, double* dp, double* dq) {
    uint32_t hu = hf;
    uint32_t F = (m >= 32) ? 0xffffffffu : ((1u << m) - 1u);
    for (int j = 0; j < m - 1; j++) {
        if (!((F >> j) & 1u)) continue;
        for (int k = j + 1; k < m; k++) {
            if (!((F >> k) & 1u)) continue;
            bool pos, neg;
            coalign_gates(An + j * D, An + k * D, D, pos, neg);
            if (pos) {
                if (hf) {
                    const bool hj = (hu >> j) & 1u, hk = (hu >> k) & 1u;
                    if (!hj && !hk) dq[j] += dq[k];
                    else if (hj && !hk) {
                        dq[j] = dq[k];
                        hu &= ~(1u << j);
                    } else if (!hj && hk) {
                        hu &= ~(1u << k);
                    } else {
                        hu &= ~(1u << k);
                        dq[j] += dq[k];
                    }
                } else {
                    dq[j] += dq[k];
                }
                F &= ~(1u << k);
                dp[j] += dp[k];
            }
            if (neg) {
                if (hf) {
                    const bool hj = (hu >> j) & 1u, hk = (hu >> k) & 1u;
                    if (!hj && !hk) dq[j] -= dq[k];
                    else if (hj && !hk) {
                        dq[j] = -dq[k];
                        hu &= ~(1u << j);
                    } else if (!hj && hk) {
                        hu &= ~(1u << k);
                    }
                } else {
                    dq[j] -= dq[k];
                }
                F &= ~(1u << k);
                dp[j] += dp[k];
            }
        }
    }
    if (__popc(F) != m) {
        int w = 1;
        for (int j = 1; j < m; j++)
            if ((F >> j) & 1u) {
                if (w < j) {
                    for (int k = 0; k < D; k++) dA[w * D + k] = dA[j * D + k];
                    dp[w] = dp[j];
                    dq[w] = dq[j];
                }
                w++;
            }
    }
}

// A double divisor with the estimate of its reciprocal kept: quot(x) is x / d to the same
// bits (see div_row), the estimate's part done once for the several quotients by d.
struct Divisor {
    double d, y;
    bool plain;
    __device__ explicit Divisor(double v) : d(v) {
        plain = fabs(v) > 1e-120 && fabs(v) < 1e120;
        double t = __builtin_amdgcn_rcp(v);
        t = __builtin_fma(__builtin_fma(-v, t, 1.0), t, t);
        y = __builtin_fma(__builtin_fma(-v, t, 1.0), t, t);
    }
    Divisor() = default;
    __device__ double quot(double x) const {
        const double ax = fabs(x);
        const double q = x * y;
        if (plain && x == 0.0) return q;
        if (plain && ax > 1e-150 && ax < 1e150) return __builtin_fma(__builtin_fma(-d, q, x), y, q);
        return x / d;
    }
};

// A complex divisor of several quotients: cdiv's steps, those of the divisor alone once.
struct CDivisor {
    double r;
    Divisor den;
    bool small_c;
    __device__ explicit CDivisor(cplx b) {
        const double c = b.re, d = b.im;
        small_c = fabs(c) < fabs(d);
        const double p = small_c ? c : d, q = small_c ? d : c;
        r = p / q;
        den = Divisor((p * r) + q);
    }
    CDivisor() = default;
    __device__ cplx quot(cplx a) const {
        const double pr = a.re * r, pi = a.im * r;
        const double xn = small_c ? (pr + a.im) : (pi + a.re);
        const double yn = small_c ? (pi - a.re) : (a.im - pr);
        return cmake(den.quot(xn), den.quot(yn));
    }
};

// Tangents of every measurement-update output slot (after k_mu, which wrote the nominal
// outputs; the parents are read post propagation), and of each slot's g value at the
// root point, whose sum is the tangent of fz (eval_g_yei, cauchy_term.hpp:312-401).
// dg: [slot][direction] complex.
//
// One workgroup per parent.  Row r of child t is mu_src - mu_t (parent row r below t, r + 1
// from t on, parent row m standing for the measurement-noise row), so mu_l, rho_l and their
// tangents in every direction are formed once per parent in LDS; each thread then takes a
// (slot, direction) and streams the rows, where one thread per slot walked all directions
// with the rows in scratch memory (3-state windows with 14 directions: 289 -> 24 us per launch,
// orbit windows: 715 -> 133 us).
template <int D>
__global__ __launch_bounds__(128) void k_mu_tan(TermPool IN, TanPool TI, int np, const int* __restrict__ slot_base,
                                                TermPool OUT, TanPool TO, const StepConst* __restrict__ sc,
                                                const StepTan* __restrict__ st, const uint32_t* __restrict__ gk_prev,
                                                const cplx* __restrict__ gv_prev, const cplx* __restrict__ dgv_prev,
                                                cplx* __restrict__ dg) {
    extern __shared__ double tan_lds[];
    const int Pp = blockIdx.x;
    if (Pp >= np) return;
    const int tid = threadIdx.x;
    const int NP = TO.P, MM = IN.MM;
    const int m = IN.m[Pp];
    // [m][D] mu, [m] rho, [m] H . A (0 where H-orthogonal), then per direction [m][D], [m]
    double* mu = tan_lds;
    double* rho = mu + MM * D;
    double* hh = rho + MM;
    double* dmu = hh + MM;
    double* drho = dmu + (size_t)NP * MM * D;
    const double* A = IN.A + (int64_t)Pp * MM * D;
    const double* p = IN.p + (int64_t)Pp * MM;
    const double* b = IN.b + (int64_t)Pp * D;
    const double* H = sc->H;
    for (int l = tid; l < m; l += 128) {
        const double h = dev_dot<D>(H, A + l * D);
        const bool orth = fabs(h) < kMuEps;
        const double rr = 1.0 / h;
        for (int k = 0; k < D; k++) mu[l * D + k] = orth ? A[l * D + k] : A[l * D + k] * rr;
        rho[l] = orth ? p[l] : p[l] * fabs(h);
        hh[l] = orth ? 0.0 : h;
    }
    for (int it = tid; it < m * NP; it += 128) {
        const int l = it % m, kk = it / m;
        const double* dH = st->H[kk];
        const double* Al = A + l * D;
        const double* dA = TI.tA(Pp, kk) + l * D;
        const double dpl = TI.tp(Pp, kk)[l];
        double* dm = dmu + ((size_t)kk * MM + l) * D;
        const double h = dev_dot<D>(H, Al);
        if (fabs(h) < kMuEps) {
            for (int k = 0; k < D; k++) dm[k] = dA[k];
            drho[kk * MM + l] = dpl;
        } else {
            double dh = 0;
            for (int k = 0; k < D; k++) dh += dH[k] * Al[k] + H[k] * dA[k];
            const double rr = 1.0 / h;
            for (int k = 0; k < D; k++) {
                const double v = Al[k] * rr;
                dm[k] = (dA[k] - v * dh) * rr;
            }
            drho[kk * MM + l] = dpl * fabs(h) + p[l] * sgn0(h) * dh;
        }
    }
    __syncthreads();
    const int s0 = slot_base[Pp];
    const double zeta = sc->msmt - dev_dot<D>(H, b);
    const bool first = sc->first != 0;
    const int phc = IN.phc[Pp];
    int lhp = 0;
    for (int l = 0; l < m && l < phc; l++) lhp |= (hh[l] != 0.0 && !(hh[l] > 0)) ? 1 << l : 0;
    const int64_t go = IN.gp_off[Pp];
    const int gn = IN.gp_n[Pp];
    for (int it = tid; it < (m + 1) * NP; it += 128) {
        const int ts = it / NP, kk = it - ts * NP;
        const int64_t s = s0 + ts;
        const int fl = OUT.flags[s];
        if (fl == 0) {  // a child of an H-orthogonal row: no term
            dg[s * NP + kk] = cmake(0, 0);
            continue;
        }
        const int t = ts == 0 ? m : ts - 1;
        const double* dmk = dmu + (size_t)kk * MM * D;
        const double* drk = drho + kk * MM;
        const double* db = TI.tb(Pp, kk);
        const double dgamma = st->gamma[kk];
        double dzeta = 0;
        for (int k = 0; k < D; k++) dzeta -= st->H[kk][k] * b[k] + H[k] * db[k];
        double mut[D], dmut[D];
        for (int k = 0; k < D; k++) {
            mut[k] = t == m ? 0.0 : mu[t * D + k];
            dmut[k] = t == m ? 0.0 : dmk[t * D + k];
        }
        const double rho_t = t == m ? sc->gamma : rho[t], drho_t = t == m ? dgamma : drk[t];
        auto child_row = [&](int r, double* row, double* drow, double& rh, double& drh) {
            const int src = (t < m && r >= t) ? r + 1 : r;
            if (src == m) {
                for (int k = 0; k < D; k++) {
                    row[k] = 0.0 - mut[k];
                    drow[k] = -dmut[k];
                }
                rh = sc->gamma;
                drh = dgamma;
                return false;
            }
            const bool orth = hh[src] == 0.0;
            for (int k = 0; k < D; k++) {
                row[k] = orth ? mu[src * D + k] : mu[src * D + k] - mut[k];
                drow[k] = orth ? dmk[src * D + k] : dmk[src * D + k] - dmut[k];
            }
            rh = rho[src];
            drh = drk[src];
            return orth;
        };
        // g at the root point: signs of the child rows, ygi over the rows that are not
        // H-orthogonal, the two parent-table numerators
        double row[D], drow[D], rh, drh;
        double ygi = 0, dygi = 0;
        uint32_t neg = 0, hf = 0;
        for (int l = 0; l < m; l++) {
            const bool orth = child_row(l, row, drow, rh, drh);
            const double sl = dev_dot<D>(row, sc->root) > 0 ? 1 : -1;
            if (sl < 0) neg |= (1u << l);
            if (orth) {
                hf |= 1u << l;
            } else {
                ygi += rh * sl;
                dygi += drh * sl;
            }
        }
        cplx gp = cmake(1, 0), gm = cmake(1, 0), dgp = cmake(0, 0), dgm = cmake(0, 0);
        if (!first) {
            const int top = 1 << (phc - 1), rev = (phc >= 32) ? -1 : ((1 << phc) - 1);
            int lp = 0, lmv = 0, k = 0;
            for (int l = 0; l < m; l++) {
                if (k < phc) {
                    if (k == t) {
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
            bool cj;
            int ix = lookup_idx(lp ^ lhp, top, rev, gk_prev + go, gn, &cj);
            gp = ix < 0 ? cmake(0, 0) : (cj ? cconj(gv_prev[go + ix]) : gv_prev[go + ix]);
            dgp = ix < 0 ? cmake(0, 0) : (cj ? cconj(dgv_prev[(go + ix) * NP + kk]) : dgv_prev[(go + ix) * NP + kk]);
            ix = lookup_idx(lmv ^ lhp, top, rev, gk_prev + go, gn, &cj);
            gm = ix < 0 ? cmake(0, 0) : (cj ? cconj(gv_prev[go + ix]) : gv_prev[go + ix]);
            dgm = ix < 0 ? cmake(0, 0) : (cj ? cconj(dgv_prev[(go + ix) * NP + kk]) : dgv_prev[(go + ix) * NP + kk]);
        }
        const cplx D1 = cmake(ygi + rho_t, zeta), D2 = cmake(ygi - rho_t, zeta);
        const cplx dD1 = cmake(dygi + drho_t, dzeta), dD2 = cmake(dygi - drho_t, dzeta);
        const cplx v = csub(dquot(gp, dgp, D1, dD1), dquot(gm, dgm, D2, dD2));
        dg[s * NP + kk] = cscale(v, kInvTwoPi);
        if (sc->skip) continue;  // a window's last update keeps no terms: TO may be empty
        double* tb_ = TO.tb(s, kk);
        for (int k = 0; k < D; k++) tb_[k] = db[k] + dzeta * mut[k] + zeta * dmut[k];
        *TO.tc(s, kk) = dzeta;
        *TO.tdv(s, kk) = drho_t;
        double* oA = TO.tA(s, kk);
        double* op = TO.tp(s, kk);
        double* oq = TO.tq(s, kk);
        for (int r = 0; r < m; r++) {
            child_row(r, row, drow, rh, drh);
            if (!first) {
                // normalize_hps(true): q = p, p *= |row|_1, row /= |row|_1
                double n1 = 0, dn1 = 0;
                for (int k = 0; k < D; k++) {
                    n1 += fabs(row[k]);
                    dn1 += sgn0(row[k]) * drow[k];
                }
                const Divisor N(n1);
                for (int k = 0; k < D; k++) drow[k] = N.quot(drow[k] - N.quot(row[k]) * dn1);
                oq[r] = drh;
                drh = drh * n1 + rh * dn1;
            }
            for (int k = 0; k < D; k++) oA[r * D + k] = drow[k];
            op[r] = drh;
        }
        if (!first && (fl & kHasCmap)) {
            // hyperplanes merged (k_mu's decisions, from the normalised rows)
            double An[kMaxShape * D];
            for (int r = 0; r < m; r++) {
                child_row(r, row, drow, rh, drh);
                double n1 = 0;
                for (int k = 0; k < D; k++) n1 += fabs(row[k]);
                for (int k = 0; k < D; k++) An[r * D + k] = row[k] / n1;
            }
            mu_coalign_tan<D>(An, hf, m, oA, op, oq);
        }
    }
}

// LDS bytes of k_mu_tan.
inline size_t mu_tan_lds(int MM, int D, int NP) { return sizeof(double) * (size_t)MM * ((D + 2) + (size_t)NP * (D + 1)); }

// Column sums of the [slot][direction] tangents: out[k] = sum over slots of dg[s][k], in a
// fixed order.  Blocks read whole stretches of slots (one block per direction read every
// NP-th entry of the array: 188 us per launch on orbit windows, 19 us with both kernels), then one wavefront adds
// their partial sums.
constexpr int kTanSumBlocks = 128;
__global__ __launch_bounds__(256) void k_tan_colsum(const cplx* __restrict__ dg, int n, int NP,
                                                    cplx* __restrict__ part) {
    __shared__ double sr[256], si[256];
    const int t = threadIdx.x;
    const int lanes = 256 / NP;  // slots side by side
    const int k = t % NP, j = t / NP;
    const int per = (n + gridDim.x - 1) / gridDim.x;
    const int s0 = blockIdx.x * per, s1 = min(n, s0 + per);
    double a = 0, c = 0;
    if (j < lanes)
        for (int s = s0 + j; s < s1; s += lanes) {
            const cplx v = dg[(int64_t)s * NP + k];
            a += v.re;
            c += v.im;
        }
    sr[t] = a;
    si[t] = c;
    __syncthreads();
    if (t < NP) {
        for (int i = 1; i < lanes; i++) {
            a += sr[i * NP + t];
            c += si[i * NP + t];
        }
        part[blockIdx.x * NP + t] = cmake(a, c);
    }
}
__global__ __launch_bounds__(64) void k_tan_colsum_finish(const cplx* __restrict__ part, int nb, int NP,
                                                          cplx* __restrict__ out) {
    const int k = threadIdx.x;
    if (k >= NP) return;
    cplx a = part[k];
    for (int b = 1; b < nb; b++) a = cadd(a, part[b * NP + k]);
    out[k] = a;
}

// ------------------------------------------------------------------ g-tables
// Tangents of the first update's g-tables and of the next parents (make_gtable_first,
// flattening.hpp:14-67): g_j = (1 / (ygi + d + i c) - 1 / (ygi - d + i c)) * gscale.
// One workgroup per slot, a thread per (cell, direction).
template <int D>
__global__ __launch_bounds__(256) void k_gtable_first_tan(const TermPool OUT, TanPool TO, int n,
                                                          const uint32_t* __restrict__ perm, double gscale,
                                                          const double* __restrict__ dgscale, cplx* __restrict__ dgv,
                                                          TanPool TN) {
    const int r = blockIdx.x;
    if (r >= n) return;
    const int64_t s = perm[r];
    const int NP = TO.P;
    const int cells = 1 << (D - 1);
    const int MM = OUT.MM;
    const double* p = OUT.p + s * MM;
    const uint32_t hf = OUT.hflag[s];
    const double c = OUT.c[s], dv = OUT.dv[s];
    for (int it = threadIdx.x; it < cells * NP; it += 256) {
        const int j = it / NP, kk = it - j * NP;
        const double* dp = TO.tp(s, kk);
        const double dc = *TO.tc(s, kk), ddv = *TO.tdv(s, kk);
        double ygi = 0, dygi = 0;
        for (int k = 0; k < D; k++)
            if (!((hf >> k) & 1u)) {
                const double sb = ((j >> k) & 1) == 0 ? 1 : -1;
                ygi += p[k] * sb;
                dygi += dp[k] * sb;
            }
        const cplx one = cmake(1.0, 0.0), zero = cmake(0, 0);
        const cplx D1 = cmake(ygi + dv, c), D2 = cmake(ygi - dv, c);
        const cplx v = csub(cdiv(one, D1), cdiv(one, D2));
        const cplx dvv = csub(dquot(one, zero, D1, cmake(dygi + ddv, dc)), dquot(one, zero, D2, cmake(dygi - ddv, dc)));
        dgv[((int64_t)r * cells + j) * NP + kk] = cadd(cscale(dvv, gscale), cscale(v, dgscale[kk]));
    }
    for (int it = threadIdx.x; it < NP * D * D; it += 256) {
        const int kk = it / (D * D), k = it - kk * D * D;
        TN.tA(r, kk)[k] = TO.tA(s, kk)[k];
    }
    for (int it = threadIdx.x; it < NP * D; it += 256) {
        const int kk = it / D, k = it - kk * D;
        TN.tp(r, kk)[k] = TO.tp(s, kk)[k];
        TN.tb(r, kk)[k] = TO.tb(s, kk)[k];
    }
}

// Parent-side key pair of a child cell (make_gtable's lambda_p / lambda_m,
// flattening.hpp:155-216): an old term keeps its key below phc; a new child gets
// parent bit z inserted (0 in lp, 1 in lm), through its coalignment maps if merged.
__device__ inline void parent_keys(uint32_t key, bool is_new, bool has_cmap, int z, int phc, const uint8_t* cm,
                                   const int8_t* cs, int* lp_, int* lm_) {
    const int rev_phc = (phc >= 32) ? -1 : ((1 << phc) - 1);
    int lp = 0, lmv = 0;
    if (!is_new) {
        lp = (int)key & rev_phc;
        lmv = lp;
    } else if (!has_cmap) {
        int k = 0, l = 0;
        while (k < phc) {
            if (k == z) {
                lmv |= (1 << k);
                k++;
                if (k == phc) break;
            }
            if ((key >> l) & 1u) {
                lp |= (1 << k);
                lmv |= (1 << k);
            }
            k++;
            l++;
        }
    } else {
        int k = 0, l = 0;
        while (k < phc) {
            if (k == z) {
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
    *lp_ = lp;
    *lm_ = lmv;
}

// Tangents of each reduction group's g-table (make_gtables, flattening.hpp:318-568), one
// workgroup per group, after k_group_eval (and k_group_sort) settled it: the surviving
// root's values at B ^ X (X: the replacement chain's orientation), plus, in member order,
// every member k_group_eval / k_group_members added (mem_add), at bi ^ sigma reversed and
// conjugated when in the lower half, where the member's table holds that key
// (add_gtables, flattening.hpp:259-315).  Written at the cell's position in the final
// (key-sorted) table; dgv: [cell][direction].
//
// A term's value at a cell is g = (a / (ygi + d + i c) - b / (ygi - d + i c)) * gscale
// (make_gtable's loop body, flattening.hpp:129-248), with ygi = sum of q_k s_k over the rows
// that are not H-orthogonal and a, b looked up in its parent's table.  All of it but the
// tangents themselves is common to the directions: for W terms (the root, then the added
// members) at a time, each of the W wavefronts leaves one term's cells in LDS, 64 at once,
// with the divisors ready for further quotients; then the threads take a (cell, direction)
// each and add the W in order.  Bound by the latency of the searches and of the terms'
// fields.  One wavefront per group that walked directions, members and cells in turn, both
// searches and six complex divisions each, took 739 us per launch on 3-state windows with 14
// directions (35 us now) and 1231 us on orbit windows (889 us).  Four wavefronts share a group
// (and its members) while there are fewer than kTanOneWave groups; beyond, one per group fills
// the chip, and four only wait for each other (orbit windows: 1770 us with four throughout).
struct TanCell {
    CDivisor D1, D2;
    cplx w1, w2;       // a / D1, b / D2
    uint32_t key;
    int ix1, ix2;      // entries of a and b in the parent's table, -1: absent
    uint8_t on, cj, cj1, cj2;
    double pad;        // a stride of 34 words: 64 lanes leave their cells without meeting in one bank
};
constexpr int kTanOneWave = 4096;
template <int W>
__global__ __launch_bounds__(64 * W, 4) void k_group_tan(
    const TermPool OUT, TanPool TO, int ng, int d, const int* __restrict__ grp_moff, const int* __restrict__ grp_mcnt,
    const int* __restrict__ grp_m, const int* __restrict__ mem_slots, const uint8_t* __restrict__ mem_add,
    const int* __restrict__ surv, const int* __restrict__ gxor, const uint32_t* __restrict__ B2,
    const int64_t* __restrict__ b2_off, const int* __restrict__ b2_n, const int64_t* __restrict__ g_off,
    const uint32_t* __restrict__ gk_prev, const cplx* __restrict__ gv_prev, const cplx* __restrict__ dgv_prev,
    const uint32_t* __restrict__ gk_out, double gscale, const double* __restrict__ dgscale,
    cplx* __restrict__ dgv_out) {
    __shared__ TanCell cells[W][64];
    __shared__ double dqs[W][kMaxTan][kMaxShape];
    __shared__ double dcs[W][kMaxTan], ddvs[W][kMaxTan];
    __shared__ int64_t gos[W];
    __shared__ uint32_t hfs[W];
    __shared__ int poss[64];
    const int g = blockIdx.x;
    if (g >= ng) return;
    const int r = surv[g];
    if (r < 0) return;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int NP = TO.P;
    const int m = grp_m[g];
    const int MM = OUT.MM;
    const uint32_t* B = B2 + b2_off[g];
    const int n = b2_n[g];
    const uint32_t X = (uint32_t)gxor[g];
    const uint32_t top = 1u << (m - 1);
    const uint32_t rev = (m >= 32) ? 0xffffffffu : ((1u << m) - 1u);
    const uint32_t* ok = gk_out + g_off[g];
    const int* mem = mem_slots + grp_moff[g];
    const uint8_t* add = mem_add + grp_moff[g];
    const int nmem = grp_mcnt[g];
    const double* Ar = OUT.A + (int64_t)r * MM * d;
    const double ar = lane < m ? Ar[lane * d] : 1.0;
    cplx* out = dgv_out + g_off[g] * NP;
    for (int c0 = 0; c0 < n; c0 += 64) {
        const int nc = min(64, n - c0);
        // the terms in order: the root (-1), then the added members, found 64 flags at a time
        // by every wavefront alike
        int base = 0;
        unsigned long long left = __ballot(lane < nmem && add[lane]);
        for (bool first = true, more = true; more; first = false) {
            int e = -2, ne = 0;  // this wavefront's term, terms of this pass
            for (; ne < W; ne++) {
                int next = -1;
                if (!first || ne > 0) {
                    while (!left && base + 64 < nmem) {
                        base += 64;
                        left = __ballot(base + lane < nmem && add[base + lane]);
                    }
                    if (!left) break;
                    next = base + __ffsll((long long)left) - 1;
                    left &= left - 1;
                }
                if (ne == w) e = next;
            }
            more = ne == W;
            if (ne == 0) break;
            TanCell C;
            C.on = 0;
            if (e >= -1) {
                const int s = wave_uniform(e < 0 ? r : mem[e]);
                const int phc = OUT.phc[s];
                const uint32_t hf = OUT.hflag[s];
                const int64_t go = OUT.gp_off[s];
                const int gn = OUT.gp_n[s];
                for (int it = lane; it < NP * m; it += 64) {
                    const int kk = it / m, k = it - kk * m;
                    dqs[w][kk][k] = TO.tq(s, kk)[k];
                }
                if (lane < NP) {
                    dcs[w][lane] = *TO.tc(s, lane);
                    ddvs[w][lane] = *TO.tdv(s, lane);
                }
                if (lane == 0) {
                    gos[w] = go;
                    hfs[w] = hf;
                }
                const uint32_t sig =
                    e < 0 ? 0u : (uint32_t)wave_orientation(Ar, ar, OUT.A + (int64_t)s * MM * d, m, d);
                const uint32_t sh = (sig & top) ? (sig ^ rev) : sig;
                if (lane < nc) {
                    const uint32_t bi = B[c0 + lane] ^ X;
                    const int pos = X == 0 ? c0 + lane : bsearch_u32(ok, bi, n);
                    if (e < 0) poss[lane] = pos;
                    uint32_t x = bi ^ sig;
                    C.cj = e >= 0 && (x & top);
                    if (C.cj) x ^= rev;
                    C.on = pos >= 0 && (e < 0 || bsearch_u32(B, x ^ sh ^ X, n) >= 0);
                    if (C.on) {
                        const double* q = OUT.q + (int64_t)s * MM;
                        double ygi = 0;
                        for (int k = 0; k < m; k++)
                            if (!((hf >> k) & 1u)) ygi += q[k] * (((x >> k) & 1u) ? -1.0 : 1.0);
                        const int fl = OUT.flags[s];
                        int lp, lmv;
                        parent_keys(x, fl & kIsNew, fl & kHasCmap, OUT.z[s], phc, OUT.cmap + (int64_t)s * MM,
                                    OUT.csmap + (int64_t)s * MM, &lp, &lmv);
                        const int lhp = OUT.lhp[s];
                        const int ptop = 1 << (phc - 1), prev = (phc >= 32) ? -1 : ((1 << phc) - 1);
                        bool c1, c2;
                        C.key = x;
                        C.ix1 = lookup_idx(lp ^ lhp, ptop, prev, gk_prev + go, gn, &c1);
                        C.ix2 = lookup_idx(lmv ^ lhp, ptop, prev, gk_prev + go, gn, &c2);
                        C.cj1 = c1;
                        C.cj2 = c2;
                        cplx a = cmake(0, 0), b = cmake(0, 0);
                        if (C.ix1 >= 0) a = c1 ? cconj(gv_prev[go + C.ix1]) : gv_prev[go + C.ix1];
                        if (C.ix2 >= 0) b = c2 ? cconj(gv_prev[go + C.ix2]) : gv_prev[go + C.ix2];
                        const double c = OUT.c[s], dv = OUT.dv[s];
                        C.D1 = CDivisor(cmake(ygi + dv, c));
                        C.D2 = CDivisor(cmake(ygi - dv, c));
                        C.w1 = C.D1.quot(a);
                        C.w2 = C.D2.quot(b);
                    }
                }
            }
            cells[w][lane] = C;
            __syncthreads();
            for (int it = tid; it < nc * NP; it += 64 * W) {
                const int cl = it / NP, kk = it - cl * NP;
                const int pos = poss[cl];
                if (pos < 0) continue;
                cplx sum = first ? cmake(0, 0) : out[(int64_t)pos * NP + kk];
                for (int u = 0; u < ne; u++) {
                    const TanCell& T = cells[u][cl];
                    if (!T.on) continue;
                    const uint32_t key = T.key, hf = hfs[u];
                    double dygi = 0;
                    for (int k = 0; k < m; k++)
                        if (!((hf >> k) & 1u)) dygi += dqs[u][kk][k] * (((key >> k) & 1u) ? -1.0 : 1.0);
                    const int64_t go = gos[u];
                    cplx da = cmake(0, 0), db = cmake(0, 0);
                    if (T.ix1 >= 0) {
                        da = dgv_prev[(go + T.ix1) * NP + kk];
                        if (T.cj1) da = cconj(da);
                    }
                    if (T.ix2 >= 0) {
                        db = dgv_prev[(go + T.ix2) * NP + kk];
                        if (T.cj2) db = cconj(db);
                    }
                    const double dc = dcs[u][kk], ddv = ddvs[u][kk];
                    const cplx t1 = T.D1.quot(csub(da, cmul(T.w1, cmake(dygi + ddv, dc))));
                    const cplx t2 = T.D2.quot(csub(db, cmul(T.w2, cmake(dygi - ddv, dc))));
                    cplx v = cadd(cscale(csub(t1, t2), gscale), cscale(csub(T.w1, T.w2), dgscale[kk]));
                    if (T.cj) v = cconj(v);
                    sum = first && u == 0 ? v : cadd(sum, v);
                }
                out[(int64_t)pos * NP + kk] = sum;
            }
            __syncthreads();
        }
    }
}

// Survivors' tangents follow k_compact into the next parents' slots, one wavefront per group
// (each direction's rows are one stretch of memory).
template <int D>
__global__ __launch_bounds__(256) void k_compact_tan(TanPool TO, int ng, const int* __restrict__ surv,
                                                     const int* __restrict__ pos, const int* __restrict__ grp_m,
                                                     TanPool TN) {
    const int g = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (g >= ng) return;
    const int r = surv[g];
    if (r < 0) return;
    const int o = pos[g];
    const int m = grp_m[g];
    for (int kk = 0; kk < TO.P; kk++) {
        for (int k = lane; k < m * D; k += 64) TN.tA(o, kk)[k] = TO.tA(r, kk)[k];
        if (lane < m) TN.tp(o, kk)[lane] = TO.tp(r, kk)[lane];
        if (lane < D) TN.tb(o, kk)[lane] = TO.tb(r, kk)[lane];
    }
}

}  // namespace mce
