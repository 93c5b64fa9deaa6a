// Direct eigensolver of the Gram method (gfx950).
//
// The Gram method needs the unitary Y whose rows are the (conjugated)
// eigenvectors of H = X X^H (n x n Hermitian, FP64), after which X <- Y X has
// orthogonal rows. Instead of rotating H sweep by sweep, problems of up to
// EIG_MAX_N rows take the classical direct route, all in FP64:
//
//   tridiagonal  H = Q T Q^H by n - 1 Householder reflectors, T real
//                symmetric tridiagonal (Golub & Van Loan, 4th ed., 8.3.1,
//                in the one-pass form: the rank-2 update of step j and the
//                product A v of step j + 1 share one pass over A);
//   T = S L S^T  divide and conquer (Cuppen 1981) with the deflation of
//                Dongarra & Sorensen (1987), the secular roots by rational
//                interpolation at the two neighbouring poles (Bunch, Nielsen
//                & Sorensen 1978) inside a bracket, and the eigenvectors of
//                every rank-one update from the weights recomputed from the
//                roots (Gu & Eisenstat 1994), which keeps S orthogonal to
//                FP64 rounding without extended precision;
//   Y = (Q S)^H  the reflectors applied in blocks of 16 (compact WY), on the
//                FP64 matrix cores.
//
// Both halves are backward stable: Y is unitary to FP64 rounding and the
// eigenvalues carry an absolute error of a few eps ||H||. The flops are
// about 16/3 n^3 + 8 n^3 complex-real mixed per problem, against 8-10 sweeps of
// 12 n^3 for the two-sided Jacobi iteration, and the launches do not depend
// on the data, so nothing is polled.
//
// Storage, all inside the problem's region: H region: H (both triangles),
// then the reflectors V as n/16 panels [Cp][16]; the Y part of Z: while
// tridiagonalising the exchange slots (below), then S^T (row i = eigenvector
// i, real) in two buffers, doubles [0, Cp) and [Cp, 2 Cp) of each Y row, and
// at the end Y; the rotation region: the small vectors (EigVec).
#include <hip/hip_runtime.h>

#include <cstddef>

#include "common.h"
#include "launch.h"

namespace {

constexpr double kEps = 2.220446049250313e-16;
// Deflation threshold for T scaled to unit norm.
constexpr double kDeflate = 8.0 * kEps;

// Small vectors of a problem in its rotation region.
struct EigVec {
    double *d, *e, *es;  // diagonal (then eigenvalues), off-diagonal, scaled off-diagonal
    double2 *tau;        // reflector scalars
    double *dl, *zl;     // per merge: poles and weights of the secular equation
    double *zh, *rt;     // recomputed weights; roots as offsets from a pole
    int *src, *base;     // row of S^T each new row comes from; pole a root is offset from
    int *kn;             // per merge (at index lo): non-deflated count
    double *rho;         // per merge (at index lo)
    int *nref;           // reflectors made
    double2 *t;          // T factors of the panels, 16 x 16 each
};
MPSX_DEV EigVec eig_vec(char *ws, const mpsx_plan &p) {
    EigVec v;
    const int Cp = p.Cp;
    // (a tall problem of method 3 has a smaller rotation region: its V ring)
    double *b = reinterpret_cast<double *>(ws + (p.method == 3 ? qv_off(p) : qmat_off(p)));
    v.t = reinterpret_cast<double2 *>(b);
    b += 2 * 16 * Cp;  // Cp / 16 panels of 256
    v.tau = reinterpret_cast<double2 *>(b);
    b += 2 * Cp;
    v.d = b;
    v.e = b + Cp;
    v.es = b + 2 * Cp;
    v.dl = b + 3 * Cp;
    v.zl = b + 4 * Cp;
    v.zh = b + 5 * Cp;
    v.rt = b + 6 * Cp;
    v.rho = b + 7 * Cp;
    int *i = reinterpret_cast<int *>(b + 8 * Cp);
    v.src = i;
    v.base = i + Cp;
    v.kn = i + 2 * Cp;
    v.nref = i + 3 * Cp;
    return v;
}
// 256 + 16 + 64 + 12 bytes per padded row and a counter, in a rotation region
// of 1024 bytes per padded row or a V ring of 2048.
static_assert(256 + 16 + 64 + 16 <= 1024 && 1024 <= QR_RING * 16 * 16, "the small vectors fit the rotation region");

MPSX_DEV double2 *eig_h(char *ws, const mpsx_plan &p) {
    return reinterpret_cast<double2 *>(ws + h_off(p));
}
// First double of Y (rows 2 LD doubles apart).
MPSX_DEV double *eig_y(char *ws, const mpsx_plan &p) {
    return reinterpret_cast<double *>(reinterpret_cast<double2 *>(ws + z_off(p)) + p.R);
}
// Merge levels above the 64-row leaves, so also the buffer S^T ends in.
MPSX_DEV int eig_levels(int n) {
    int l = 0;
    while ((64 << l) < n) ++l;
    return l;
}

template <int CTRL>
MPSX_DEV double dpp_f64(double x) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}
// Sum over groups of L consecutive lanes, the same in every lane of the
// group (quad permutes, then the half-row and row mirrors).
template <int L>
MPSX_DEV double group_sum(double x) {
    if (L >= 2) x += dpp_f64<0xB1>(x);
    if (L >= 4) x += dpp_f64<0x4E>(x);
    if (L >= 8) x += dpp_f64<0x141>(x);
    if (L >= 16) x += dpp_f64<0x140>(x);
    return x;
}
template <int L>
MPSX_DEV double group_prod(double x) {
    if (L >= 2) x *= dpp_f64<0xB1>(x);
    if (L >= 4) x *= dpp_f64<0x4E>(x);
    if (L >= 8) x *= dpp_f64<0x141>(x);
    if (L >= 16) x *= dpp_f64<0x140>(x);
    return x;
}
MPSX_DEV double wave_sum64(double x) {
    x = group_sum<16>(x);
    x += __shfl_xor(x, 16, 64);
    x += __shfl_xor(x, 32, 64);
    return x;
}
// a' = [a.lower, b.lower], b' = [a.upper, b.upper] halves of the wave, added:
// the lower half then holds a's pairwise sums, the upper half b's.
MPSX_DEV double fold32(double a, double b) {
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b), false, false);
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
// The same on rows of 16 lanes: even rows hold a's sums, odd rows b's.
MPSX_DEV double fold16(double a, double b) {
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b), false, false);
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
// Wave sums of four complex values at once: lanes 16 q .. 16 q + 15 receive
// the sum of x[q]. Folding two values into one register halves the work of
// every level (12 exchanges of 64-bit values instead of 48).
MPSX_DEV double2 wave_sum4(const double2 (&x)[4]) {
    const double re = fold16(fold32(x[0].x, x[2].x), fold32(x[1].x, x[3].x));
    const double im = fold16(fold32(x[0].y, x[2].y), fold32(x[1].y, x[3].y));
    return make_double2(group_sum<16>(re), group_sum<16>(im));
}
MPSX_DEV double uniform_f64(double x) {
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(x)),
                            __builtin_amdgcn_readfirstlane(__double2loint(x)));
}
MPSX_DEV double2 uniform_z(double2 v) { return make_double2(uniform_f64(v.x), uniform_f64(v.y)); }

// ------------------------------------------------------- tridiagonal form
// A group of G workgroups (eig_group: 128, 64, 32 or 16 rows each) holds one
// problem's whole trailing matrix in registers: wave g of the group's 8 G owns
// the rows g, g + 8 G, ..., lane l the columns l, l + 64, .... Step j
//   1. takes p = A v (of the previous reflector v) and column j of A, both
//      as they were before the pending rank-2 update;
//   2. w = tau p - (tau/2)(tau p)^H v) v; column j brought up to date; its
//      reflector (tau', v');
//   3. one pass over the registers: A -= v w^H + w v^H, p' = A v'.
// Step 2 is repeated by every workgroup of the group (n-vectors only), so
// the only exchange between workgroups is p' and column j + 1: 2 (n - j)
// complex values a step, published by the owner of each row and awaited by
// all.
//
// The exchange carries no flags: every slot is used once, starts as a NaN
// of one fixed bit pattern (EIG_EMPTY, written by k_init_rows) and is written
// by one 64-bit store at device scope; a reader polls until the pattern is
// gone (a published NaN is given other bits). Slots of step J: p_i and c_i
// for i = J .. n-1. Steps J and n - J share two Y rows of Cp complex values.
//
// Workgroups take their place by a ticket in the order they start, so a
// workgroup waits only for others that have the tickets next to its own:
// all groups but the last started one are whole and run to their end
// whatever else holds the GPU, and four launches at once leave fewer than
// 4 (64 - 1) workgroups waiting on the 256 compute units. A wait that is not
// served within kSpin polls (seconds) gives up for good and the problem's
// results become NaN.
//
// The iteration stops where the trailing matrix is zero to working precision
// (its trace, what the diagonal has left of tr H, is at most 64 eps tr H; H is
// positive semidefinite, so its entries are no larger): on an H of rank r that
// is after about r steps, whatever n. Tall theta and the zero singular
// values that gates of low Schmidt rank leave make such H.
//
// Bound: the step's latency, an exchange (about 2 us) and four barriers;
// the arithmetic of step 3 is under a microsecond.
constexpr int kSpin = 1 << 21;

MPSX_DEV void publish(double *at, double v) {
    unsigned long long b = (unsigned long long)__double_as_longlong(v);
    if (v != v) b = 0x7ff8000000000000ULL;
    __hip_atomic_store(reinterpret_cast<unsigned long long *>(at), b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
MPSX_DEV unsigned long long peek(const double *at) {
    return __hip_atomic_load(reinterpret_cast<const unsigned long long *>(at), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
}

struct TriShared {
    double2 v[2][EIG_MAX_N];  // reflectors of the previous and this step
    double2 w[EIG_MAX_N];
    double2 p[128], c[128];   // the exchange of a one-workgroup group
    double2 red1[8];
    double red2[8];
    double2 xj, al;
    double dj;
    int fail;
    int slot;
};

// Slot of (step J, row i): four doubles (p re, p im, c re, c im).
MPSX_DEV double *xslot(double *y, int64_t ld2, int Cp, int n, int J, int i) {
    const bool late = J > n - J;
    const int q = late ? n - J : J;
    int pos = 2 * (i - J) + (late ? 2 * (n - q) : 0);
    int row = 2 * q - 2;
    if (pos >= Cp) {
        pos -= Cp;
        ++row;
    }
    return y + row * ld2 + 2 * pos;
}

// Step 3 on NL live rows (the last of the four rows at r0): update, product
// and the publication of column J.
template <int CH, int RW, int NL, int NG>
MPSX_DEV void tri_rows(double2 (&a)[RW][CH], int r0, const double2 *v, const double2 *w, const double2 *vn,
                       int lane, const int (&row)[4], double2 (&acc)[4], int t0, int J, int n, bool alone,
                       TriShared &sm, double *y, int64_t ld2, int Cp) {
    double2 vi[4], wi[4];
#pragma unroll
    for (int q = NG - NL; q < NG; ++q) {
        const int r = row[q] < n ? row[q] : n;  // entry n and above are zero
        vi[q] = uniform_z(v[r < EIG_MAX_N ? r : 0]);
        wi[q] = uniform_z(w[r < EIG_MAX_N ? r : 0]);
    }
    const int tc = J >> 6, lc = J & 63;
#pragma unroll
    for (int t = 0; t < CH; ++t) {
        if (t < t0) continue;
        const int k = lane + 64 * t;
        const double2 vk = v[k], wk = w[k], nk = vn[k];
#pragma unroll
        for (int q = NG - NL; q < NG; ++q) {
            double2 x = a[r0 + q][t];
            x.x = fma(-vi[q].x, wk.x, fma(-vi[q].y, wk.y, fma(-wi[q].x, vk.x, fma(-wi[q].y, vk.y, x.x))));
            x.y = fma(-vi[q].y, wk.x, fma(vi[q].x, wk.y, fma(-wi[q].y, vk.x, fma(wi[q].x, vk.y, x.y))));
            acc[q].x = fma(x.x, nk.x, fma(-x.y, nk.y, acc[q].x));
            acc[q].y = fma(x.x, nk.y, fma(x.y, nk.x, acc[q].y));
            a[r0 + q][t] = x;
        }
        if (t == tc && lane == lc) {
#pragma unroll
            for (int q = NG - NL; q < NG; ++q) {
                if (row[q] >= n) continue;
                const double2 x = a[r0 + q][t];
                if (alone) {
                    sm.c[row[q]] = x;
                } else {
                    double *s = xslot(y, ld2, Cp, n, J, row[q]);
                    publish(s + 2, x.x);
                    publish(s + 3, x.y);
                }
            }
        }
    }
}

template <int CH, int RW>
MPSX_DEV void tridiag(const mpsx_plan &p, char *ws, int member, int G, TriShared &sm) {
    constexpr int EPT = CH > 8 ? 2 : 1;  // vector elements per thread
    constexpr int NG = RW < 4 ? RW : 4;  // rows per reduction
    const int n = p.C, Cp = p.Cp;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int gw = member * 8 + wave, NW = 8 * G;
    const bool alone = G == 1;
    double2 *H = eig_h(ws, p);
    double *y = eig_y(ws, p);
    const int64_t ld2 = 2 * (int64_t)p.LD;
    const EigVec ev = eig_vec(ws, p);

    double2 a[RW][CH];
#pragma unroll
    for (int r = 0; r < RW; ++r)
#pragma unroll
        for (int t = 0; t < CH; ++t) {
            const int row = gw + NW * r, k = lane + 64 * t;
            a[r][t] = (row < n && k < n) ? H[(int64_t)row * Cp + k] : make_double2(0.0, 0.0);
        }
    double2 c0[EPT], vown[EPT];
#pragma unroll
    for (int s = 0; s < EPT; ++s) {
        const int i = tid + 512 * s;
        c0[s] = i < n ? H[(int64_t)i * Cp] : make_double2(0.0, 0.0);
        vown[s] = make_double2(0.0, 0.0);
    }
    for (int i = tid; i < EIG_MAX_N; i += 512) {
        sm.v[0][i] = make_double2(0.0, 0.0);
        sm.v[1][i] = make_double2(0.0, 0.0);
        sm.w[i] = make_double2(0.0, 0.0);
    }
    double trace = 0.0;
    for (int i = lane; i < n; i += 64) trace += H[(int64_t)i * Cp + i].x;
    double rem = wave_sum64(trace);  // trace of the trailing matrix; the same in every wave
    const double floor_tr = 64.0 * kEps * rem;
    int nref = n - 1;
    if (tid == 0) {
        sm.fail = 0;
        sm.xj = make_double2(0.0, 0.0);
        sm.al = make_double2(0.0, 0.0);
    }
    __syncthreads();
    double2 tau = make_double2(0.0, 0.0);
    int cur = 0;
    for (int j = 0; j < n; ++j) {
        // ---- 1. p and column j
        double2 x[EPT], c[EPT], dot = make_double2(0.0, 0.0);
        const bool failed = sm.fail != 0;
#pragma unroll
        for (int s = 0; s < EPT; ++s) {
            const int i = tid + 512 * s;
            double2 pv = make_double2(0.0, 0.0);
            c[s] = make_double2(0.0, 0.0);
            if (i >= j && i < n) {
                if (j == 0) {
                    c[s] = c0[s];
                } else if (alone) {
                    pv = sm.p[i];
                    c[s] = sm.c[i];
                } else {
                    const double *at = xslot(y, ld2, Cp, n, j, i);
                    unsigned long long b0, b1, b2, b3;
                    int spin = failed ? kSpin : 0;
                    while (true) {
                        b0 = peek(at);
                        b1 = peek(at + 1);
                        b2 = peek(at + 2);
                        b3 = peek(at + 3);
                        if (b0 != EIG_EMPTY && b1 != EIG_EMPTY && b2 != EIG_EMPTY && b3 != EIG_EMPTY) break;
                        if (++spin > kSpin) {
                            sm.fail = 1;
                            break;
                        }
                    }
                    pv = make_double2(__longlong_as_double((long long)b0), __longlong_as_double((long long)b1));
                    c[s] = make_double2(__longlong_as_double((long long)b2), __longlong_as_double((long long)b3));
                }
            }
            x[s] = zmul(tau, pv);
            // conj(x) v
            dot.x = fma(x[s].x, vown[s].x, fma(x[s].y, vown[s].y, dot.x));
            dot.y = fma(x[s].x, vown[s].y, fma(-x[s].y, vown[s].x, dot.y));
            if (i == j) sm.xj = x[s];
        }
        dot = make_double2(wave_sum64(dot.x), wave_sum64(dot.y));
        if (lane == 0) sm.red1[wave] = dot;
        __syncthreads();
        // ---- 2. w, column j, its reflector
        dot = make_double2(0.0, 0.0);
#pragma unroll
        for (int u = 0; u < 8; ++u) dot = zadd(dot, sm.red1[u]);
        const double2 alpha = zscale(zmul(tau, dot), -0.5);
        const double2 wj = zadd(sm.xj, alpha);  // v_j = 1 for j > 0; zero otherwise
        double2 col[EPT];
        double nrm = 0.0;
        const bool writer = j > 0 && member == j % G;
        const bool stop = rem <= floor_tr;
#pragma unroll
        for (int s = 0; s < EPT; ++s) {
            const int i = tid + 512 * s;
            const double2 v = vown[s];
            const double2 w = zadd(x[s], zmul(alpha, v));
            // c - v conj(w_j) - w conj(v_j), v_j = 1
            col[s].x = c[s].x - (v.x * wj.x + v.y * wj.y) - (j > 0 ? w.x : 0.0);
            col[s].y = c[s].y - (v.y * wj.x - v.x * wj.y) - (j > 0 ? w.y : 0.0);
            if (i < EIG_MAX_N) sm.w[i] = (i > j && i < n) ? w : make_double2(0.0, 0.0);
            if (i > j + 1 && i < n) nrm = fma(col[s].x, col[s].x, fma(col[s].y, col[s].y, nrm));
            if (i == j + 1) sm.al = col[s];
            if (i == j) sm.dj = col[s].x;
            if (member == 0 && i == j && !stop) ev.d[j] = col[s].x;
            // reflector j - 1 to its panel (every workgroup has read H by now)
            if (writer && i < n && i >= ((j - 1) & ~15))
                H[(int64_t)((j - 1) >> 4) * 16 * Cp + (int64_t)i * 16 + ((j - 1) & 15)] = v;
        }
        if (stop) {
            nref = j;
            if (member == 0)
                for (int i = j + tid; i < n; i += 512) {
                    ev.d[i] = 0.0;
                    ev.e[i] = 0.0;
                }
            break;
        }
        nrm = wave_sum64(nrm);
        if (lane == 0) sm.red2[wave] = nrm;
        __syncthreads();
        if (j == n - 1) break;
        rem -= sm.dj;
        nrm = ((sm.red2[0] + sm.red2[1]) + (sm.red2[2] + sm.red2[3])) +
              ((sm.red2[4] + sm.red2[5]) + (sm.red2[6] + sm.red2[7]));
        const double2 al = sm.al;
        double beta = al.x;
        double2 sc = make_double2(0.0, 0.0);
        tau = make_double2(0.0, 0.0);
        if (!(nrm == 0.0 && al.y == 0.0)) {
            beta = -copysign(sqrt(fma(al.x, al.x, fma(al.y, al.y, nrm))), al.x);
            const double ib = 1.0 / beta;
            tau = make_double2((beta - al.x) * ib, -al.y * ib);
            const double2 df = make_double2(al.x - beta, al.y);
            const double id = 1.0 / fma(df.x, df.x, df.y * df.y);
            sc = make_double2(df.x * id, -df.y * id);
        }
        if (member == 0 && tid == 0) {
            ev.e[j] = beta;
            ev.tau[j] = tau;
        }
        double2 *vn = sm.v[cur ^ 1];
#pragma unroll
        for (int s = 0; s < EPT; ++s) {
            const int i = tid + 512 * s;
            vown[s] = i == j + 1 ? make_double2(1.0, 0.0)
                                 : ((i > j + 1 && i < n) ? zmul(col[s], sc) : make_double2(0.0, 0.0));
            if (i < EIG_MAX_N) vn[i] = vown[s];
        }
        __syncthreads();
        // ---- 3. A -= v w^H + w v^H, p' = A v'; publish p' and column j + 1
        const double2 *v = sm.v[cur];
        const int J = j + 1, t0 = J >> 6;
#pragma unroll
        for (int g = 0; g < RW / NG; ++g) {
            int row[4] = {n, n, n, n};
#pragma unroll
            for (int q = 0; q < NG; ++q) row[q] = gw + NW * (g * NG + q);
            double2 acc[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) acc[q] = make_double2(0.0, 0.0);
            int live = 0;  // rows of index >= J: the last ones
#pragma unroll
            for (int q = 0; q < NG; ++q) live += row[q] >= J;
            if (live == 0) continue;
            if (live == 1)
                tri_rows<CH, RW, 1, NG>(a, g * NG, v, sm.w, vn, lane, row, acc, t0, J, n, alone, sm, y, ld2, Cp);
            else if (live == 2)
                tri_rows<CH, RW, 2, NG>(a, g * NG, v, sm.w, vn, lane, row, acc, t0, J, n, alone, sm, y, ld2, Cp);
            else if (live == 3)
                tri_rows<CH, RW, (NG < 3 ? NG : 3), NG>(a, g * NG, v, sm.w, vn, lane, row, acc, t0, J, n, alone, sm,
                                                        y, ld2, Cp);
            else
                tri_rows<CH, RW, NG, NG>(a, g * NG, v, sm.w, vn, lane, row, acc, t0, J, n, alone, sm, y, ld2, Cp);
            const double2 s = wave_sum4(acc);
            const int q = lane >> 4;
            int rq = row[0];
            if (q == 1) rq = row[1];
            if (q == 2) rq = row[2];
            if (q == 3) rq = row[3];
            if ((lane & 15) == 0 && q < NG && rq >= J && rq < n) {
                if (alone) {
                    sm.p[rq] = s;
                } else {
                    double *at = xslot(y, ld2, Cp, n, J, rq);
                    publish(at, s.x);
                    publish(at + 1, s.y);
                }
            }
        }
        cur ^= 1;
        if (alone) __syncthreads();
    }
    if (member == 0 && tid == 0) *ev.nref = nref;
}

}  // namespace

// Table of the workgroups of k_tridiag: entry s = (problem, member << 8 |
// group size), the problems with the largest groups first. One workgroup.
__global__ void __launch_bounds__(256)
k_eig_map(const mpsx_two_site_op *ops, int count, int2 *map, int max_n) {
    __shared__ int wsum[4];
    __shared__ int total;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (tid == 0) total = 0;
    __syncthreads();
    for (int cls = 3; cls >= 0; --cls)
        for (int b = 0; b < count; b += 256) {
            const int pi = b + tid;
            int g = 0;
            if (pi < count) {
                const mpsx_plan p = ops[pi].plan;
                if (eig_direct(p, max_n) && eig_class(p.C) == cls) g = eig_group(p.C);
            }
            int inc = g;
            for (int o = 1; o < 64; o <<= 1) {
                const int up = __shfl_up(inc, o, 64);
                if (lane >= o) inc += up;
            }
            if (lane == 63) wsum[wave] = inc;
            __syncthreads();
            int at = total + inc - g;
            for (int u = 0; u < wave; ++u) at += wsum[u];
            for (int m = 0; m < g; ++m) map[at + m] = make_int2(pi, (m << 8) | g);
            __syncthreads();
            if (tid == 0) total += wsum[0] + wsum[1] + wsum[2] + wsum[3];
            __syncthreads();
        }
}

__global__ void __launch_bounds__(512, 2)
k_tridiag(const mpsx_two_site_op *ops, const int2 *map, char *ws, int slots) {
    __shared__ TriShared sm;
    if (threadIdx.x == 0) sm.slot = atomicAdd(&reinterpret_cast<TwoSiteHeader *>(ws)->ticket, 1);
    __syncthreads();
    const int slot = sm.slot;
    if (slot >= slots) return;
    const int2 m = map[slot];
    const mpsx_plan p = ops[m.x].plan;
    const int member = m.y >> 8, G = m.y & 255;
    switch (eig_class(p.C)) {
        case 0: tridiag<2, 16>(p, ws, member, G, sm); break;
        case 1: tridiag<4, 8>(p, ws, member, G, sm); break;
        case 2: tridiag<8, 4>(p, ws, member, G, sm); break;
        default: tridiag<16, 2>(p, ws, member, G, sm); break;
    }
}

// T factors of the reflector panels (H_0 ... H_15 = I - V T V^H, T upper
// triangular): V^H V on the matrix cores, four waves over the rows, then T by
// columns, T[0:j, j] = -tau_j T[0:j, 0:j] (V^H v_j). x: panel, y: problem.
__global__ void __launch_bounds__(256)
k_eig_t(const mpsx_two_site_op *ops, char *ws, int max_n) {
    __shared__ double2 part[4][16][17];
    __shared__ double2 g[16][17];
    const mpsx_plan p = ops[blockIdx.y].plan;
    if (!eig_direct(p, max_n)) return;
    const int n = p.C, Cp = p.Cp, q = (int)blockIdx.x;
    const EigVec ev = eig_vec(ws, p);
    const int nref = *ev.nref;
    if (16 * q >= nref) return;
    const int ncols = min(16, nref - 16 * q);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, lq = lane >> 4;
    const double2 *V = eig_h(ws, p) + (int64_t)q * 16 * Cp;
    mfma_d4 m1 = {0.0, 0.0, 0.0, 0.0}, m2 = m1, m3 = m1, m4 = m1;
    for (int r0 = 16 * q + 4 * wave; r0 < n; r0 += 16) {
        const int row = r0 + lq;
        const double2 v = (row < n && l16 < ncols) ? V[(int64_t)row * 16 + l16] : make_double2(0.0, 0.0);
        m1 = mfma16d(v.x, v.x, m1);
        m2 = mfma16d(v.y, v.y, m2);
        m3 = mfma16d(v.x, v.y, m3);
        m4 = mfma16d(v.y, v.x, m4);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) part[wave][4 * r + lq][l16] = make_double2(m1[r] + m2[r], m3[r] - m4[r]);
    __syncthreads();
    {
        const int i = tid >> 4, j = tid & 15;
        g[i][j] = zadd(zadd(part[0][i][j], part[1][i][j]), zadd(part[2][i][j], part[3][i][j]));  // v_i^H v_j
    }
    __syncthreads();
    if (tid >= 16) return;
    // row tid of T
    double2 tr[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        double2 sum = make_double2(0.0, 0.0);
#pragma unroll
        for (int m = 0; m < j; ++m) sum = zadd(sum, zmul(tr[m], g[m][j]));
        const double2 tj = j < ncols ? ev.tau[16 * q + j] : make_double2(0.0, 0.0);
        const double2 off = zmul(sum, make_double2(-tj.x, -tj.y));
        const bool on = j < ncols && j >= tid;
        tr[j] = make_double2(!on ? 0.0 : (j == tid ? tj.x : off.x), !on ? 0.0 : (j == tid ? tj.y : off.y));
    }
    double2 *T = ev.t + (int64_t)q * 256 + tid * 16;
#pragma unroll
    for (int j = 0; j < 16; ++j) T[j] = tr[j];
}

// ---------------------------------------------------- divide and conquer
namespace {

// Rank-one update diag(d) + rho z z^T of a merge, poles in ascending order
// (ds, zs, id): deflates the entries with negligible weight and, of poles
// closer than the weights resolve, one of each pair after a rotation. K
// poles stay (dl, zl, src[0 .. K-1]); the deflated ones fill dd and src from
// the end. rot_i, rot_c: the rotations (row a, row b, c, s) in order. Serial.
MPSX_DEV int deflate(int m, double rho, const double *ds, const double *zs, const int *id, double *dl,
                     double *zl, int *src, double *dd, int2 *rot_i, double2 *rot_c, int *nrot) {
    int K = 0, e = m, nr = 0, pj = -1;
    double pd = 0.0, pz = 0.0;
    int in = id[0];
    double dn = ds[0], zn = zs[0];
    for (int r = 0; r < m; ++r) {
        const int i = in;
        const double dr = dn, zr = zn;
        if (r + 1 < m) {
            in = id[r + 1];
            dn = ds[r + 1];
            zn = zs[r + 1];
        }
        if (rho * fabs(zr) <= kDeflate) {
            --e;
            src[e] = i;
            dd[e] = dr;
            continue;
        }
        if (pj >= 0) {
            const double n2 = fma(pz, pz, zr * zr);
            if (fabs((dr - pd) * pz * zr) <= kDeflate * n2) {
                const double t = sqrt(n2), c = zr / t, s = -pz / t;
                rot_i[nr] = make_int2(pj, i);
                rot_c[nr] = make_double2(c, s);
                ++nr;
                --e;
                src[e] = pj;
                dd[e] = pd * c * c + dr * s * s;
                pd = pd * s * s + dr * c * c;
                pz = t;
                pj = i;
                continue;
            }
            dl[K] = pd;
            zl[K] = pz;
            src[K] = pj;
            ++K;
        }
        pj = i;
        pd = dr;
        pz = zr;
    }
    if (pj >= 0) {
        dl[K] = pd;
        zl[K] = pz;
        src[K] = pj;
        ++K;
    }
    *nrot = nr;
    return K;
}

MPSX_DEV double recip(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(r, fma(-x, r, 1.0), r);
    return fma(r, fma(-x, r, 1.0), r);
}

// Root j of 1 + rho sum_i z_i^2 / (d_i - lambda), 0 <= j < K, by L lanes (sub
// = lane in the group): lambda = dl[base] + tau with base the nearer of the
// two poles around it, so that every difference d_i - lambda is accurate.
template <int L>
MPSX_DEV void secular_root(int K, const double *dl, const double *zl, double rho, int j, int sub, int *base,
                           double *root) {
    const bool last = j == K - 1;
    const double dj = dl[j];
    int org = j;
    double lo, hi, t;
    if (last) {
        double s = 0.0;
        for (int i = sub; i < K; i += L) s = fma(zl[i], zl[i], s);
        s = group_sum<L>(s);
        lo = 0.0;
        hi = rho * s * (1.0 + 4.0 * kEps);
        t = K == 1 ? rho * s : 0.5 * hi;
    } else {
        const double gap = dl[j + 1] - dj, mid = 0.5 * gap;
        double c0 = 0.0;
        for (int i = sub; i < K; i += L) {
            if (i == j || i == j + 1) continue;
            c0 = fma(zl[i] * zl[i], recip((dl[i] - dj) - mid), c0);
        }
        c0 = group_sum<L>(c0);
        const double s = rho * zl[j] * zl[j], v = rho * zl[j + 1] * zl[j + 1], c = fma(rho, c0, 1.0);
        const bool left = c + (v - s) / mid >= 0.0;
        org = left ? j : j + 1;
        lo = left ? 0.0 : -mid;
        hi = left ? mid : 0.0;
        // c + s / (p1 - t) + v / (p2 - t) = 0 with the poles at 0 and +-gap
        const double A = left ? fma(c, gap, s + v) : fma(-c, gap, s + v);
        const double B = left ? s * gap : -v * gap;
        const double sq = sqrt(fmax(fma(A, A, -4.0 * c * B), 0.0));
        t = A > 0.0 ? 2.0 * B / (A + sq) : (A - sq) / (2.0 * c);
    }
    if (K > 1) {
        if (!(t > lo && t < hi)) t = 0.5 * (lo + hi);
        const double dorg = dl[org], p1 = dj - dorg, p2 = last ? 0.0 : dl[j + 1] - dorg;
        for (int it = 0; it < 64; ++it) {
            double psi = 0.0, dpsi = 0.0, phi = 0.0, dphi = 0.0;
            for (int i = sub; i < K; i += L) {
                const double r = recip((dl[i] - dorg) - t), q = zl[i] * zl[i] * r, dq = q * r;
                if (i <= j) {
                    psi += q;
                    dpsi += dq;
                } else {
                    phi += q;
                    dphi += dq;
                }
            }
            psi = rho * group_sum<L>(psi);
            phi = rho * group_sum<L>(phi);
            dpsi = rho * group_sum<L>(dpsi);
            dphi = rho * group_sum<L>(dphi);
            const double g = 1.0 + psi + phi;
            if (fabs(g) <= kEps * (8.0 * (1.0 + fabs(psi) + fabs(phi)) + fabs(t) * (dpsi + dphi))) break;
            if (g < 0.0)
                lo = t;
            else
                hi = t;
            double tn;
            if (last) {
                // c - s / t = 0 through the pole at the origin
                tn = dpsi * t * t / fma(dpsi, t, g);
            } else {
                const double D1 = p1 - t, D2 = p2 - t;
                const double s = dpsi * D1 * D1, v = dphi * D2 * D2, c = g - dpsi * D1 - dphi * D2;
                const double A = fma(c, D1 + D2, s + v), B = D1 * D2 * g;
                const double sq = sqrt(fmax(fma(A, A, -4.0 * c * B), 0.0));
                const double q = 0.5 * (A + copysign(sq, A));
                double eta = B / q;  // of the two roots, the one between the poles
                if (!(eta > D1 && eta < D2)) eta = q / c;
                tn = t + eta;
            }
            if (!(tn > lo && tn < hi)) tn = 0.5 * (lo + hi);
            if (tn == t || hi - lo <= 2.0 * kEps * fmax(fabs(lo), fabs(hi))) break;
            t = tn;
        }
    }
    *base = org;
    *root = t;
}

// |z_i| for which the computed roots are the exact ones (Gu & Eisenstat), by
// L lanes.
template <int L>
MPSX_DEV double zhat(int K, const double *dl, const int *base, const double *rt, int i, int sub) {
    const double di = dl[i];
    double pr = 1.0;
    for (int j = sub; j < K; j += L) {
        const double num = (dl[base[j]] - di) + rt[j];
        const double den = j < i ? dl[j] - di : (j < K - 1 ? dl[j + 1] - di : 1.0);
        pr *= num / den;
    }
    return sqrt(fmax(group_prod<L>(pr), 0.0));
}

// Sort key: NaN below everything, so that ranks are a permutation.
MPSX_DEV double sort_key(double x) { return x == x ? x : -__builtin_huge_val(); }

}  // namespace

// Leaves: the eigensystem of every 64 x 64 diagonal block of T, torn at each
// entry, by six levels of merges in LDS. x: block, y: problem. Also scales T to
// unit norm (es, d) for the merges above.
__global__ void __launch_bounds__(256)
k_eig_leaf(const mpsx_two_site_op *ops, char *ws, int max_n) {
    constexpr int M = 64;
    __shared__ double S[2][M][M + 1];
    __shared__ double U[M][M + 1];
    __shared__ double d[M], z[M], ds[M], zs[M], dl[M], zl[M], dd[M], zh[M], rt[M];
    __shared__ int id[M], src[M], base[M], kn[M], nrot[M];
    __shared__ int2 rot_i[M];
    __shared__ double2 rot_c[M];
    __shared__ double red[4];
    const mpsx_plan p = ops[blockIdx.y].plan;
    if (!eig_direct(p, max_n)) return;
    const int n = p.C, b0 = (int)blockIdx.x * M;
    if (b0 >= n) return;
    const int m = min(M, n - b0), tid = threadIdx.x;
    const EigVec ev = eig_vec(ws, p);
    double mx = 0.0;
    for (int i = tid; i < n; i += 256) {
        mx = fmax(mx, fabs(ev.d[i]));
        if (i + 1 < n) mx = fmax(mx, fabs(ev.e[i]));
    }
    for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o, 64));
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
    mx = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
    const double scale = mx > 0.0 ? 1.0 / mx : 1.0;
    auto off = [&](int i) { return (i >= 0 && i + 1 < n) ? ev.e[i] * scale : 0.0; };
    if (tid < M) {
        const int i = b0 + tid;
        // d stays unscaled in memory (other leaves read it): this leaf's
        // eigenvalues go to rt, where the first merge takes them
        d[tid] = i < n ? ev.d[i] * scale - fabs(off(i - 1)) - fabs(off(i)) : 0.0;
        if (i < n) ev.es[i] = off(i);
    }
    for (int e = tid; e < M * M; e += 256) {
        S[0][e >> 6][e & 63] = (e >> 6) == (e & 63) ? 1.0 : 0.0;
    }
    __syncthreads();
    int cur = 0;
    for (int s = 1; s < m; s <<= 1) {
        const int h = 2 * s;
        const int ni = tid < M ? tid : (tid >> 2);  // index this thread serves in the 1-per-index steps
        const int lo = ni & ~(h - 1), mid = lo + s, hi = min(lo + h, m), sz = hi - lo;
        const bool merge = mid < hi;
        const double ee = (lo < m && merge) ? off(b0 + mid - 1) : 0.0;
        if (tid < m) {
            z[tid] = merge ? S[cur][tid][tid < mid ? mid - 1 : mid] *
                                 (tid >= mid && ee < 0.0 ? -0.7071067811865476 : 0.7071067811865476)
                           : 0.0;
        }
        __syncthreads();
        if (tid < m) {
            const double key = sort_key(d[tid]);
            int rank = 0;
            for (int o = lo; o < hi; ++o) {
                const double ko = sort_key(d[o]);
                rank += (ko < key) || (ko == key && o < tid);
            }
            ds[lo + rank] = d[tid];
            zs[lo + rank] = z[tid];
            id[lo + rank] = tid;
        }
        __syncthreads();
        if (tid < m && tid == lo) {
            kn[lo] = deflate(sz, merge ? 2.0 * fabs(ee) : 0.0, ds + lo, zs + lo, id + lo, dl + lo, zl + lo, src + lo,
                             dd + lo, rot_i + lo, rot_c + lo, &nrot[lo]);
        }
        __syncthreads();
        if (tid < m) {  // component tid of the node's rows
            for (int r = 0; r < nrot[lo]; ++r) {
                const int2 ab = rot_i[lo + r];
                const double2 cs = rot_c[lo + r];
                const double xa = S[cur][ab.x][tid], xb = S[cur][ab.y][tid];
                S[cur][ab.x][tid] = cs.x * xa + cs.y * xb;
                S[cur][ab.y][tid] = cs.x * xb - cs.y * xa;
            }
        }
        __syncthreads();
        // four lanes per root from here on
        const int g = tid >> 2, sub = tid & 3;
        const int glo = g & ~(h - 1), gmid = glo + s;
        const int K = g < m ? kn[glo] : 0, gj = g - glo;
        const double grho = (g < m && gmid < min(glo + h, m)) ? 2.0 * fabs(off(b0 + gmid - 1)) : 0.0;
        if (gj < K) {
            int bs;
            double root;
            secular_root<4>(K, dl + glo, zl + glo, grho, gj, sub, &bs, &root);
            if (sub == 0) {
                base[g] = bs;
                rt[g] = root;
            }
        }
        __syncthreads();
        if (gj < K) {
            const double v = zhat<4>(K, dl + glo, base + glo, rt + glo, gj, sub);
            if (sub == 0) zh[g] = copysign(v, zl[g]);
        }
        __syncthreads();
        if (gj < K) {
            const double db = dl[glo + base[g]], tj = rt[g];
            double nn = 0.0;
            for (int i = sub; i < K; i += 4) {
                const double u = zh[glo + i] / ((dl[glo + i] - db) - tj);
                U[g][i] = u;
                nn = fma(u, u, nn);
            }
            nn = group_sum<4>(nn);
            const double f = 1.0 / sqrt(nn);
            for (int i = sub; i < K; i += 4) U[g][i] *= f;
        }
        __syncthreads();
        for (int e = tid; e < M * M; e += 256) {
            const int j = e >> 6, r = e & 63;
            const int jlo = j & ~(h - 1);
            double v = 0.0;
            if (j < m && r >= jlo && r < min(jlo + h, m)) {
                const int Kj = kn[jlo];
                if (j - jlo < Kj) {
                    for (int i = 0; i < Kj; ++i) v = fma(U[j][i], S[cur][src[jlo + i]][r], v);
                } else {
                    v = S[cur][src[j]][r];
                }
            }
            S[cur ^ 1][j][r] = v;
        }
        if (tid < m) d[tid] = (tid - lo) < kn[lo] ? dl[lo + base[tid]] + rt[tid] : dd[tid];
        __syncthreads();
        cur ^= 1;
    }
    double *y = eig_y(ws, p);
    const int64_t ld2 = 2 * (int64_t)p.LD;
    // both buffers of S^T: zero outside the block (the merges write their
    // own blocks only)
    for (int j = tid >> 6; j < m; j += 4)
        for (int r = tid & 63; r < 2 * p.Cp; r += 64) {
            const int rr = r - b0;
            y[(int64_t)(b0 + j) * ld2 + r] = (rr >= 0 && rr < m) ? S[cur][j][rr] : 0.0;
        }
    if (tid < m) ev.rt[b0 + tid] = d[tid];
}

// Merge of the blocks [lo, lo + s) and [lo + s, lo + 2 s): z, sorting,
// deflation and its rotations. One workgroup per merge (x) and problem (y).
// `first`: the eigenvalues come from the leaves (rt). Buffer `buf` of S^T is
// read; deflated rows and eigenvalues go to the end of the block.
__global__ void __launch_bounds__(512)
k_eig_merge(const mpsx_two_site_op *ops, char *ws, int max_n, int s, int buf, int first) {
    __shared__ double d0[EIG_MAX_N], ds[EIG_MAX_N], zs[EIG_MAX_N], dl[EIG_MAX_N], zl[EIG_MAX_N], dd[EIG_MAX_N];
    __shared__ int id[EIG_MAX_N], src[EIG_MAX_N];
    __shared__ int2 rot_i[EIG_MAX_N];
    __shared__ double2 rot_c[EIG_MAX_N];
    __shared__ int sK, sR;
    const mpsx_plan p = ops[blockIdx.y].plan;
    if (!eig_direct(p, max_n)) return;
    const int n = p.C, lo = (int)blockIdx.x * 2 * s;
    if (s >= n || lo >= n) return;
    const int mid = lo + s, hi = min(lo + 2 * s, n), m = hi - lo, tid = threadIdx.x;
    const bool merge = mid < hi;
    const EigVec ev = eig_vec(ws, p);
    double *y = eig_y(ws, p) + (int64_t)buf * p.Cp;
    const int64_t ld2 = 2 * (int64_t)p.LD;
    const double ee = merge ? ev.es[mid - 1] : 0.0;
    for (int i = tid; i < m; i += 512) d0[i] = first ? ev.rt[lo + i] : ev.d[lo + i];
    __syncthreads();
    if (tid == 0) {
        sK = 0;
        sR = 0;
    }
    if (!merge) {  // no right half: the block passes on as it is
        for (int i = tid; i < m; i += 512) {
            ev.d[lo + i] = d0[i];
            ev.src[lo + i] = lo + i;
        }
        if (tid == 0) {
            ev.kn[lo] = 0;
            ev.rho[lo] = 0.0;
        }
        return;
    }
    for (int i = tid; i < m; i += 512) {
        const double x = d0[i], key = sort_key(x);
        double zv = y[(int64_t)(lo + i) * ld2 + (lo + i < mid ? mid - 1 : mid)];
        zv *= (lo + i >= mid && ee < 0.0) ? -0.7071067811865476 : 0.7071067811865476;
        int rank = 0;
#pragma unroll 16
        for (int o = 0; o < m; ++o) {
            const double ko = sort_key(d0[o]);
            rank += (ko < key) || (ko == key && o < i);
        }
        ds[rank] = x;
        zs[rank] = zv;
        id[rank] = lo + i;
    }
    __syncthreads();
    const double rho = 2.0 * fabs(ee);
    if (tid == 0) sK = deflate(m, rho, ds, zs, id, dl, zl, src, dd, rot_i, rot_c, &sR);
    __syncthreads();
    const int K = sK, nr = sR;
    for (int r = tid; r < m; r += 512)
        for (int q = 0; q < nr; ++q) {
            const int2 ab = rot_i[q];
            const double2 cs = rot_c[q];
            double *pa = y + (int64_t)ab.x * ld2 + lo + r, *pb = y + (int64_t)ab.y * ld2 + lo + r;
            const double xa = *pa, xb = *pb;
            *pa = cs.x * xa + cs.y * xb;
            *pb = cs.x * xb - cs.y * xa;
        }
    for (int i = tid; i < m; i += 512) {
        ev.src[lo + i] = src[i];
        if (i < K) {
            ev.dl[lo + i] = dl[i];
            ev.zl[lo + i] = zl[i];
        } else {
            ev.d[lo + i] = dd[i];
        }
    }
    if (tid == 0) {
        ev.kn[lo] = K;
        ev.rho[lo] = rho;
    }
}

// The secular roots of a level's merges, 16 lanes per root: 16 roots per
// workgroup (x; a merge's 2 s >= 128 rows are whole workgroups), y: problem.
__global__ void __launch_bounds__(256)
k_eig_roots(const mpsx_two_site_op *ops, char *ws, int max_n, int s) {
    __shared__ double dl[EIG_MAX_N], zl[EIG_MAX_N];
    const mpsx_plan p = ops[blockIdx.y].plan;
    if (!eig_direct(p, max_n)) return;
    const int n = p.C, r0 = (int)blockIdx.x * 16;
    if (s >= n || r0 >= n) return;
    const int lo = r0 & ~(2 * s - 1);
    const EigVec ev = eig_vec(ws, p);
    const int K = ev.kn[lo];
    if (r0 - lo >= K) return;
    for (int i = threadIdx.x; i < K; i += 256) {
        dl[i] = ev.dl[lo + i];
        zl[i] = ev.zl[lo + i];
    }
    __syncthreads();
    const int j = r0 - lo + ((int)threadIdx.x >> 4), sub = threadIdx.x & 15;
    if (j >= K) return;
    int bs;
    double root;
    secular_root<16>(K, dl, zl, ev.rho[lo], j, sub, &bs, &root);
    if (sub == 0) {
        ev.base[lo + j] = bs;
        ev.rt[lo + j] = root;
        ev.d[lo + j] = dl[bs] + root;
    }
}

// The recomputed weights, 16 lanes per pole, split as k_eig_roots.
__global__ void __launch_bounds__(256)
k_eig_weights(const mpsx_two_site_op *ops, char *ws, int max_n, int s) {
    __shared__ double dl[EIG_MAX_N], rt[EIG_MAX_N];
    __shared__ int base[EIG_MAX_N];
    const mpsx_plan p = ops[blockIdx.y].plan;
    if (!eig_direct(p, max_n)) return;
    const int n = p.C, r0 = (int)blockIdx.x * 16;
    if (s >= n || r0 >= n) return;
    const int lo = r0 & ~(2 * s - 1);
    const EigVec ev = eig_vec(ws, p);
    const int K = ev.kn[lo];
    if (r0 - lo >= K) return;
    for (int i = threadIdx.x; i < K; i += 256) {
        dl[i] = ev.dl[lo + i];
        rt[i] = ev.rt[lo + i];
        base[i] = ev.base[lo + i];
    }
    __syncthreads();
    const int i = r0 - lo + ((int)threadIdx.x >> 4), sub = threadIdx.x & 15;
    if (i >= K) return;
    const double v = zhat<16>(K, dl, base, rt, i, sub);
    if (sub == 0) ev.zh[lo + i] = copysign(v, ev.zl[lo + i]);
}

// Rows of the merged S^T (buffer buf ^ 1): row j < K is sum_i u_ij S^T[src_i],
// u_ij = zh_i / (d_i - lambda_j), normalised; the deflated rows are copied. A
// 64 x 64 tile per workgroup on the FP64 matrix cores, the entries of u formed
// while they are staged (one division each, repeated by the tile's few
// column neighbours, instead of a pass over memory). x: row tile * column
// tiles + column tile of a merge, z: merge, y: problem.
__global__ void __launch_bounds__(256)
k_eig_vectors(const mpsx_two_site_op *ops, char *ws, int max_n, int s, int buf) {
    constexpr int TK = 16;
    __shared__ double As[64][TK + 1];
    __shared__ double Bs[TK][64 + 1];
    __shared__ double nrm[64];
    const mpsx_plan p = ops[blockIdx.y].plan;
    if (!eig_direct(p, max_n)) return;
    const int n = p.C, lo = (int)blockIdx.z * 2 * s;
    if (s >= n || lo >= n) return;
    const int hi = min(lo + 2 * s, n), m = hi - lo;
    const int ct = (2 * s) / 64, j0 = ((int)blockIdx.x / ct) * 64, c0 = ((int)blockIdx.x % ct) * 64;
    if (j0 >= m || c0 >= m) return;
    const EigVec ev = eig_vec(ws, p);
    const int64_t ld2 = 2 * (int64_t)p.LD;
    const double *in = eig_y(ws, p) + (int64_t)buf * p.Cp + lo;
    double *out = eig_y(ws, p) + (int64_t)(buf ^ 1) * p.Cp + lo;
    const int K = ev.kn[lo];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, lq = lane >> 4;
    const int wm = wave >> 1, wn = wave & 1;
    if (j0 < K) {
        // thread: row j of the tile, 4 of the 16 poles of a stage
        const int aj = tid >> 2, ai = (tid & 3) * 4;
        const bool jok = j0 + aj < K;
        double db = 0.0, tj = 0.0, nn = 0.0;
        if (jok) {
            db = ev.dl[lo + ev.base[lo + j0 + aj]];
            tj = ev.rt[lo + j0 + aj];
        }
        mfma_d4 acc[2][2];
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b) acc[a][b] = mfma_d4{0.0, 0.0, 0.0, 0.0};
        for (int k0 = 0; k0 < K; k0 += TK) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int i = k0 + ai + t;
                double u = 0.0;
                if (jok && i < K) u = ev.zh[lo + i] * recip((ev.dl[lo + i] - db) - tj);
                nn = fma(u, u, nn);
                As[aj][ai + t] = u;
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int bk = (tid >> 6) + 4 * t, bc = tid & 63;
                const int i = k0 + bk;
                Bs[bk][bc] = (i < K && c0 + bc < m) ? in[(int64_t)ev.src[lo + i] * ld2 + c0 + bc] : 0.0;
            }
            __syncthreads();
#pragma unroll
            for (int q = 0; q < TK / 4; ++q) {
                const int kk = 4 * q + lq;
                double av[2], bv[2];
#pragma unroll
                for (int a = 0; a < 2; ++a) av[a] = As[32 * wm + 16 * a + l16][kk];
#pragma unroll
                for (int b = 0; b < 2; ++b) bv[b] = Bs[kk][32 * wn + 16 * b + l16];
#pragma unroll
                for (int a = 0; a < 2; ++a)
#pragma unroll
                    for (int b = 0; b < 2; ++b) acc[a][b] = mfma16d(av[a], bv[b], acc[a][b]);
            }
            __syncthreads();
        }
        nn = group_sum<4>(nn);
        if ((tid & 3) == 0) nrm[aj] = jok ? 1.0 / sqrt(nn) : 0.0;
        __syncthreads();
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int jj = 32 * wm + 16 * a + 4 * r + lq, cc = c0 + 32 * wn + 16 * b + l16;
                    if (j0 + jj < K && cc < m) out[(int64_t)(lo + j0 + jj) * ld2 + cc] = acc[a][b][r] * nrm[jj];
                }
    }
    if (j0 + 64 > K)  // deflated rows
        for (int e = tid; e < 64 * 64; e += 256) {
            const int j = j0 + (e >> 6), cc = c0 + (e & 63);
            if (j >= K && j < m && cc < m) out[(int64_t)(lo + j) * ld2 + cc] = in[(int64_t)ev.src[lo + j] * ld2 + cc];
        }
}

// ---------------------------------------------------- back transformation
// Y rows i0 .. i0 + 15 = (Q s_i)^H: the strip [s_i0 .. s_i0+15] (n x 16, one
// eigenvector a column) in the matrix-core output layout in registers (eight
// waves; wave w the 16-row chunks w, w + 8, ...), the panels' block
// reflectors I - V T V^H from the last to the first. x: strip, y: problem.
// CH chunks a wave: 4 up to 512 rows, 8 up to 1024. Bound: the three
// barriers a panel at two workgroups per CU (CH = 4) and the FP64 matrix
// cores; V is read once per strip, from the L2.
template <int CH>
__global__ void __launch_bounds__(512, CH == 4 ? 4 : 2)
k_eig_back(const mpsx_two_site_op *ops, char *ws, int max_n) {
    __shared__ double2 Wp[8][16][17];
    __shared__ double2 Wt[16][17], Ws[16][17], Ts[16][17];
    const mpsx_plan p = ops[blockIdx.y].plan;
    if (!eig_direct(p, max_n) || (CH == 4) != (p.C <= 512)) return;
    const int n = p.C, Cp = p.Cp, i0 = 16 * (int)blockIdx.x;
    if (i0 >= n) return;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, l16 = lane & 15, lq = lane >> 4;
    const EigVec ev = eig_vec(ws, p);
    double *y = eig_y(ws, p);
    const int64_t ld2 = 2 * (int64_t)p.LD;
    const bool vec_ok = i0 + l16 < n;
    const double *sv = y + (int64_t)(i0 + l16) * ld2 + (int64_t)(eig_levels(n) & 1) * Cp;
    double2 a[CH][4];
#pragma unroll
    for (int i = 0; i < CH; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * (w + 8 * i) + 4 * r + lq;
            a[i][r] = make_double2((row < n && vec_ok) ? sv[row] : 0.0, 0.0);
        }
    __syncthreads();  // the rows are read before any of them is written
    const int nref = *ev.nref;
    for (int q = (nref + 15) / 16 - 1; q >= 0; --q) {
        const double2 *V = eig_h(ws, p) + (int64_t)q * 16 * Cp;
        const double2 *T = ev.t + (int64_t)q * 256;
        const int vr0 = 16 * q, ncols = min(16, nref - vr0);
        mfma_d4 m1 = {0.0, 0.0, 0.0, 0.0}, m2 = m1, m3 = m1;
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const int b = 16 * (w + 8 * i);
            if (b < vr0 || b >= n) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = b + 4 * r + lq;
                const double2 v = (row < n && l16 < ncols) ? V[(int64_t)row * 16 + l16] : make_double2(0.0, 0.0);
                m1 = mfma16d(v.x, a[i][r].x, m1);
                m2 = mfma16d(v.y, a[i][r].y, m2);
                m3 = mfma16d(v.x - v.y, a[i][r].x + a[i][r].y, m3);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
            Wp[w][4 * r + lq][l16] = make_double2(m1[r] + m2[r], m3[r] - m1[r] + m2[r]);
        if (tid < 256) Ts[tid >> 4][tid & 15] = T[tid];
        __syncthreads();
        if (tid < 256) {
            const int i = tid >> 4, c = tid & 15;
            double2 s = make_double2(0.0, 0.0);
#pragma unroll
            for (int u = 0; u < 8; ++u) s = zadd(s, Wp[u][i][c]);
            Wt[i][c] = s;
        }
        __syncthreads();
        if (tid < 256) {  // Ws = T Wt
            const int i = tid >> 4, c = tid & 15;
            double2 s = make_double2(0.0, 0.0);
#pragma unroll
            for (int k = 0; k < 16; ++k) s = zadd(s, zmul(Ts[i][k], Wt[k][c]));
            Ws[i][c] = s;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const int b = 16 * (w + 8 * i);
            if (b < vr0 || b >= n) continue;
            mfma_d4 n1 = {0.0, 0.0, 0.0, 0.0}, n2 = n1, n3 = n1;
            const int vrow = b + l16;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const double2 v = (vrow < n && 4 * t + lq < ncols) ? V[(int64_t)vrow * 16 + 4 * t + lq]
                                                                   : make_double2(0.0, 0.0);
                const double2 x = Ws[4 * t + lq][l16];
                n1 = mfma16d(v.x, x.x, n1);
                n2 = mfma16d(v.y, x.y, n2);
                n3 = mfma16d(v.x + v.y, x.x + x.y, n3);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                a[i][r].x -= n1[r] - n2[r];
                a[i][r].y -= n3[r] - n1[r] - n2[r];
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (!vec_ok) return;
    double2 *yr = reinterpret_cast<double2 *>(y + (int64_t)(i0 + l16) * ld2);
#pragma unroll
    for (int i = 0; i < CH; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = 16 * (w + 8 * i) + 4 * r + lq;  // zero beyond n
            if (row < Cp) yr[row] = make_double2(a[i][r].x, -a[i][r].y);
        }
}

// ---------------------------------------------------------------- launchers
hipError_t launch_eig_tridiag(hipStream_t s, const mpsx_two_site_op *d, int count, char *ws, void *map, int max_n,
                              int slots) {
    hipLaunchKernelGGL(k_eig_map, dim3(1), dim3(256), 0, s, d, count, static_cast<int2 *>(map), max_n);
    hipLaunchKernelGGL(k_tridiag, dim3((unsigned)slots), dim3(512), 0, s, d, static_cast<const int2 *>(map), ws,
                       slots);
    return hipGetLastError();
}

hipError_t launch_eig_conquer(hipStream_t s, const mpsx_two_site_op *d, int count, char *ws, int max_n, int n) {
    const unsigned y = (unsigned)count;
    hipLaunchKernelGGL(k_eig_leaf, dim3((unsigned)((n + 63) / 64), y), dim3(256), 0, s, d, ws, max_n);
    int buf = 0;
    for (int h = 64; h < n; h *= 2, buf ^= 1) {
        const unsigned nodes = (unsigned)((n + 2 * h - 1) / (2 * h)), tiles = (unsigned)(2 * h / 64);
        const unsigned roots = (unsigned)((n + 15) / 16);
        hipLaunchKernelGGL(k_eig_merge, dim3(nodes, y), dim3(512), 0, s, d, ws, max_n, h, buf, h == 64 ? 1 : 0);
        hipLaunchKernelGGL(k_eig_roots, dim3(roots, y), dim3(256), 0, s, d, ws, max_n, h);
        hipLaunchKernelGGL(k_eig_weights, dim3(roots, y), dim3(256), 0, s, d, ws, max_n, h);
        hipLaunchKernelGGL(k_eig_vectors, dim3(tiles * tiles, y, nodes), dim3(256), 0, s, d, ws, max_n, h, buf);
    }
    return hipGetLastError();
}

hipError_t launch_eig_back(hipStream_t s, const mpsx_two_site_op *d, int count, char *ws, int max_n, int n,
                           bool small, bool large) {
    hipLaunchKernelGGL(k_eig_t, dim3((unsigned)((n + 14) / 16), (unsigned)count), dim3(256), 0, s, d, ws, max_n);
    if (small)
        hipLaunchKernelGGL(k_eig_back<4>, dim3((unsigned)((min(n, 512) + 15) / 16), (unsigned)count), dim3(512), 0, s,
                           d, ws, max_n);
    if (large)
        hipLaunchKernelGGL(k_eig_back<8>, dim3((unsigned)((n + 15) / 16), (unsigned)count), dim3(512), 0, s, d, ws,
                           max_n);
    return hipGetLastError();
}
