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
//   T = S L S^T  divide and conquer (eig_dc.h), merges above 64 rows spread
//                over the GPU;
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

#include <atomic>
#include <cstddef>

#include "common.h"
#include "eig_dc.h"
#include "launch.h"

namespace {

// Small vectors of a problem in its rotation region.
struct EigVec {
    double *d, *e, *es;  // diagonal (then eigenvalues), off-diagonal, scaled off-diagonal
    double2 *tau;        // reflector scalars
    double *dl, *zl;     // per merge: poles and weights of the secular equation
    double *zh, *rt;     // recomputed weights; roots as offsets from a pole
    double *pb;          // pole a root is offset from
    int *src;            // row of S^T each new row comes from
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
    v.pb = b + 8 * Cp;
    int *i = reinterpret_cast<int *>(b + 9 * Cp);
    v.src = i;
    v.kn = i + Cp;
    v.nref = i + 2 * Cp;
    return v;
}
// 256 + 16 + 72 + 8 bytes per padded row and a counter, in a rotation region
// of 1024 bytes per padded row or a V ring of 2048.
static_assert(256 + 16 + 72 + 16 <= 1024 && 1024 <= QR_RING * 16 * 16, "the small vectors fit the rotation region");

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

// ------------------------------------------------------- tridiagonal form
// A group of G workgroups (eig_group: 128, 64, 32 or 16 rows each) holds one
// problem's whole trailing matrix in registers: the rows in blocks of eight,
// dealt out to the workgroups in turn, a row of a block a wave; lane l the
// columns l, l + 64, .... Step j
//   1. takes p = A v (of the previous reflector v) and column j of A, both
//      as they were before the pending rank-2 update;
//   2. w = tau p - (tau/2)(tau p)^H v) v; column j brought up to date; its
//      reflector (tau', v');
//   3. one pass over the registers: A -= v w^H + w v^H, p' = A v'.
// Step 2 is repeated by every workgroup of the group (n-vectors only), so
// the only exchange between workgroups is p' and column j + 1: 2 (n - j)
// complex values a step, published by the owner of each row and awaited by
// all. In a workgroup the vectors of up to 256 elements are the work of its
// first four waves: a SIMD issues for one of them as fast as for two.
//
// The exchange carries no flags: every slot is used once, starts as a NaN
// of one fixed bit pattern (EIG_EMPTY, written by k_init_rows) and is written
// by one 64-bit store at device scope; a reader polls until the pattern is
// gone (a published NaN is given other bits). Slots of step J: four arrays of n
// - J doubles (p re, p im, c re, c im). Steps J and n - J share two Y rows.
//
// A group starts its work only when all its workgroups have started: from then on it
// holds its compute units and waits for nothing but itself. Before that a
// workgroup may hold a compute unit that a missing member needs. In a launch
// whose largest problem has more than 256 rows the groups are stretches of the
// workgroups as they are numbered: each XCD is dealt every eighth and starts its share in
// order, so the first group that is not done is whole before later ones hold
// anything it needs. (By order of start, the last groups could be left with more
// workgroups on one XCD than that has compute units: one launch of 11 problems of 900
// rows took 28 ms and now and then 316; now 21.4.) Members are numbered XCD by XCD, so that
// the owners of neighbouring rows share an L2 (1024 rows: 7.7 -> 7.4 ms). Groups of
// up to four are formed by tickets in the order of start instead, which leaves fewer
// compute units waiting where launches of several streams mix (four streams of 100 problems
// of 150 rows: 3.9 ms a call, 4.9 by number).
// Several launches can still block each other, each with an incomplete group (the
// host holds back those of large groups, launch_big_groups), so the wait has an end: after
// kFormTicks, once to four times by the launch's turn so that launches under way
// together do not all give up at once, the group is given up for good, its workgroups leave, and
// k_tridiag_one does the problem. The flag and the count are one word (ctl->group), so a
// group is either whole or given up for all its members.
//
// The iteration stops where the trailing matrix is zero to working precision
// (its trace, what the diagonal has left of tr H, is at most 64 eps tr H; H is
// positive semidefinite, so its entries are no larger): on an H of rank r that
// is after about r steps, whatever n. Tall theta and the zero singular
// values that gates of low Schmidt rank leave make such H.
//
// Bound: the step's latency: an exchange (about 2 us), three barriers, and
// instruction issue; 4.5 us a step at n = 512, 3.1 at 128. The whole update
// of 512 x 512 takes 3.0 ms, with the Jacobi rounds (300 launches of 37 us,
// behind a QR of 1.6 ms) it took 13.2. k_tridiag_one: 28 ms at 512, 0.3 s at
// 1024.
constexpr int kSpin = 1 << 21;  // polls of a slot of a whole group (seconds): never reached
constexpr long long kFormTicks = 4000000;  // 40 ms at 100 MHz

// Whether the group is whole; one thread of each of its workgroups asks.
MPSX_DEV bool form_group(int *state, int G, int spread) {
    if (G == 1) return true;
    int s = __hip_atomic_fetch_add(state, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
    const long long start = wall_clock64(), limit = kFormTicks * (1 + spread);
    while (true) {
        if (s & EIG_GROUP_LOST) return false;
        if (s >= G) return true;
        if (wall_clock64() - start > limit) {
            if (__hip_atomic_compare_exchange_strong(state, &s, s | EIG_GROUP_LOST, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                     __HIP_MEMORY_SCOPE_AGENT))
                return false;
            continue;  // s is the newer value
        }
        __builtin_amdgcn_s_sleep(4);
        s = __hip_atomic_load(state, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

MPSX_DEV void publish(double *at, double v) {
    unsigned long long b = (unsigned long long)__double_as_longlong(v);
    if (v != v) b = 0x7ff8000000000000ULL;
    __hip_atomic_store(reinterpret_cast<unsigned long long *>(at), b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
MPSX_DEV unsigned long long peek(const double *at) {
    return __hip_atomic_load(reinterpret_cast<const unsigned long long *>(at), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
}

// NX: rows a one-workgroup group may have; PW: parts their product with v is
// summed from.
template <int NX, int PW>
struct TriShared {
    double2 v[2][EIG_MAX_N];  // reflectors of the previous and this step
    double2 w[EIG_MAX_N];
    double2 p[PW][NX], c[NX];  // the exchange of a one-workgroup group
    double2 red1[8];
    double red2[8];
    double2 xj, al;
    double dj;
    int fail, stop, whole;
    int slot;
};

// The slots of step J in the Y rows: doubles first .. of a stretch that starts in
// row `row` and goes on in the next at Cp complex values.
struct Slots {
    double *y;
    int64_t ld2;
    int first, split, m;
};
MPSX_DEV Slots slots_of(double *y, int64_t ld2, int Cp, int n, int J) {
    const bool late = J > n - J;
    const int q = late ? n - J : J;
    Slots s;
    s.y = y + (int64_t)(2 * q - 2) * ld2;
    s.ld2 = ld2;
    s.first = late ? 4 * (n - q) : 0;
    s.split = 2 * Cp;
    s.m = n - J;
    return s;
}
MPSX_DEV double *slot_at(const Slots &s, int array, int i) {
    const int pos = s.first + array * s.m + i;
    return s.y + (pos >= s.split ? s.ld2 + (pos - s.split) : (int64_t)pos);
}

// Step 3 on NL live rows (the last of the NG at r0), and the publication of
// column J. MEM: the rows are in memory (A, row stride lda)
// instead of registers.
template <int CH, int RW, int NL, int NG, bool MEM, class SM>
MPSX_DEV void tri_rows(double2 (&a)[RW][CH], double2 *A, int64_t lda, int r0, const double2 *v, const double2 *w, const double2 *vn,
                       int lane, const int (&row)[4], double2 (&acc)[4], int t0, int J, int n, SM &sm,
                       const Slots &sl) {
    double2 vi[4], wi[4];
#pragma unroll
    for (int q = NG - NL; q < NG; ++q) {
        const int r = row[q] < n ? row[q] : 0;  // entry 0 is zero from the second step on, a row beyond n always
        vi[q] = uniform_z(v[r]);
        wi[q] = uniform_z(w[r]);
    }
    // Column J: up to 256 rows the wave that holds row J writes that,
    // conjugated, chunk by chunk (the others save the instructions: 10.8
    // instead of 12.7 thousand cycles a step at n = 256); above, where the row is long
    // (1.1 us at n = 1024), every row its entry.
    constexpr bool ROW = CH <= 4;
    constexpr int qj = NG - NL;  // the only row here that can be row J
    const bool has_j = ROW && row[qj] == J;
    const int tc = J >> 6, lc = J & 63;
#pragma unroll
    for (int t = 0; t < CH; ++t) {
        if (t < t0) continue;
        const int k = lane + 64 * t;
        const double2 vk = v[k], wk = w[k], nk = vn[k];
#pragma unroll
        for (int q = NG - NL; q < NG; ++q) {
            double2 x;
            if constexpr (MEM)
                x = (row[q] < n && k < n) ? A[row[q] * lda + k] : make_double2(0.0, 0.0);
            else
                x = a[r0 + q][t];
            x.x = fma(-vi[q].x, wk.x, fma(-vi[q].y, wk.y, fma(-wi[q].x, vk.x, fma(-wi[q].y, vk.y, x.x))));
            x.y = fma(-vi[q].y, wk.x, fma(vi[q].x, wk.y, fma(-wi[q].y, vk.x, fma(wi[q].x, vk.y, x.y))));
            acc[q].x = fma(x.x, nk.x, fma(-x.y, nk.y, acc[q].x));
            acc[q].y = fma(x.x, nk.y, fma(x.y, nk.x, acc[q].y));
            if constexpr (MEM) {
                if (row[q] < n && k < n) A[row[q] * lda + k] = x;
            } else {
                a[r0 + q][t] = x;
            }
            if (ROW && q == qj && has_j && k >= J && k < n) {
                if (MEM) {
                    sm.c[k] = zconj(x);
                } else {
                    publish(slot_at(sl, 2, k - J), x.x);
                    publish(slot_at(sl, 3, k - J), -x.y);
                }
            }
        }
        if (!ROW && t == tc && lane == lc) {
#pragma unroll
            for (int q = NG - NL; q < NG; ++q) {
                if (row[q] >= n) continue;
                double2 x;
                if constexpr (MEM)
                    x = A[row[q] * lda + k];
                else
                    x = a[r0 + q][t];
                if (MEM) {
                    sm.c[row[q]] = x;
                } else {
                    publish(slot_at(sl, 2, row[q] - J), x.x);
                    publish(slot_at(sl, 3, row[q] - J), x.y);
                }
            }
        }
    }
}

// Step 3 of a one-workgroup group: A is Hermitian, so p' = A v' is summed down the
// columns, in the lanes, without a reduction across them; the eight waves' parts
// meet in LDS. Row J, conjugated, is column J.
template <int RW, int T0, class SM>
MPSX_DEV void tri_rows_alone(double2 (&a)[RW][2], const double2 *v, const double2 *w, const double2 *vn, int lane,
                             int wave, int J, int n, SM &sm) {
    double2 acc[2], vk[2], wk[2];
#pragma unroll
    for (int t = T0; t < 2; ++t) {
        acc[t] = make_double2(0.0, 0.0);
        vk[t] = v[lane + 64 * t];
        wk[t] = w[lane + 64 * t];
    }
#pragma unroll
    for (int r = 0; r < RW; ++r) {
        const int row = 8 * r + wave;
        if (row < J || row >= n) continue;
        const double2 vi = v[row], wi = w[row], ni = vn[row];
#pragma unroll
        for (int t = T0; t < 2; ++t) {
            double2 x = a[r][t];
            x.x = fma(-vi.x, wk[t].x, fma(-vi.y, wk[t].y, fma(-wi.x, vk[t].x, fma(-wi.y, vk[t].y, x.x))));
            x.y = fma(-vi.y, wk[t].x, fma(vi.x, wk[t].y, fma(-wi.y, vk[t].x, fma(wi.x, vk[t].y, x.y))));
            acc[t].x = fma(x.x, ni.x, fma(x.y, ni.y, acc[t].x));
            acc[t].y = fma(x.x, ni.y, fma(-x.y, ni.x, acc[t].y));
            a[r][t] = x;
            if (row == J) sm.c[lane + 64 * t] = zconj(x);
        }
    }
#pragma unroll
    for (int t = T0; t < 2; ++t) sm.p[wave][lane + 64 * t] = acc[t];
}

// MEM: one workgroup, the matrix copied to the Y rows (which hold no slots
// then); every sum is formed in the same order as by a group. spin_limit: looks at a
// slot after which the group is reported as not converged.
template <int CH, int RW, bool MEM, class SM>
MPSX_DEV void tridiag(const mpsx_plan &p, char *ws, int member, int G, int spin_limit, SM &sm) {
    constexpr int VW = CH > 4 ? 8 : 4;        // waves that hold the vectors
    constexpr int EPT = CH > VW ? CH / VW : 1;  // vector elements per thread of theirs
    constexpr int NG = RW < 4 ? RW : 4;       // rows per reduction
    const int n = p.C, Cp = p.Cp;
    const int tid = threadIdx.x;
    int wave = tid >> 6;
    constexpr bool LANES = CH == 2 && !MEM;   // a group of one (up to 128 rows)
    constexpr bool alone = CH == 2 || MEM;
    const bool vec = VW == 8 || wave < VW;
    double2 *H = eig_h(ws, p);
    double *y = eig_y(ws, p);
    const int64_t ld2 = 2 * (int64_t)p.LD;
    const EigVec ev = eig_vec(ws, p);

    double2 a[RW][CH], vown[EPT];
    double2 *A = reinterpret_cast<double2 *>(y);
    double rem;  // trace of the trailing matrix
    {
        const int lane = tid & 63;
        if constexpr (MEM) {
            for (int row = wave; row < n; row += 8)
                for (int k = lane; k < n; k += 64) A[(int64_t)row * p.LD + k] = H[(int64_t)row * Cp + k];
        } else {
#pragma unroll
            for (int r = 0; r < RW; ++r)
#pragma unroll
                for (int t = 0; t < CH; ++t) {
                    const int row = 8 * (member + G * r) + wave, k = lane + 64 * t;
                    a[r][t] = (row < n && k < n) ? H[(int64_t)row * Cp + k] : make_double2(0.0, 0.0);
                }
        }
#pragma unroll
        for (int s = 0; s < EPT; ++s) vown[s] = make_double2(0.0, 0.0);
        for (int i = tid; i < EIG_MAX_N; i += 512) {
            sm.v[0][i] = make_double2(0.0, 0.0);
            sm.v[1][i] = make_double2(0.0, 0.0);
            sm.w[i] = make_double2(0.0, 0.0);
        }
        rem = 0.0;
        if (vec)
            for (int i = lane; i < n; i += 64) rem += H[(int64_t)i * Cp + i].x;
        rem = wave_sum64(rem);  // the same in each of these waves
    }
    const double floor_tr = 64.0 * kEps * rem;
    if (tid == 0) {
        sm.fail = 0;
        sm.xj = make_double2(0.0, 0.0);
        sm.al = make_double2(0.0, 0.0);
        sm.dj = 0.0;
    }
    __syncthreads();
    double2 tau = make_double2(0.0, 0.0);
    // This workgroup's rows of reflector q to its panel: 256 bytes apart, so
    // that they are shared out and come after what others wait for (one member in turn writing
    // all of them before its pass cost 0.4 us a step at n = 512). Every
    // workgroup has read H once the slots of step 1 are full.
    auto panel = [&](int q, const double2 *v) {
        for (int i = tid; i < n; i += 512)
            if (i >= (q & ~15) && (alone || (i >> 3) % G == member))
                H[(int64_t)(q >> 4) * 16 * Cp + (int64_t)i * 16 + (q & 15)] = v[i];
    };
    int cur = 0, nref = n - 1;
    for (int j = 0; j < n; ++j) {
        // the lane and the wave through an empty asm statement: addresses are
        // formed in the step rather than held (and spilled) across it
        int lane = tid & 63;
        asm volatile("" : "+v"(lane), "+v"(wave));
        const int ti = 64 * wave + lane;  // this thread's first vector element
        double2 x[EPT], c[EPT];
        if (vec) {
            // ---- 1. p and column j
            double2 dot = make_double2(0.0, 0.0);
            const bool failed = sm.fail != 0;
            const Slots sl = slots_of(y, ld2, Cp, n, j);
            double2 pv[EPT];
            if (j == 0 || alone) {
#pragma unroll
                for (int s = 0; s < EPT; ++s) {
                    const int i = ti + 64 * VW * s;
                    pv[s] = make_double2(0.0, 0.0);
                    c[s] = make_double2(0.0, 0.0);
                    if (i < j || i >= n) continue;
                    if (j == 0) {
                        c[s] = H[(int64_t)i * Cp];
                    } else {
                        pv[s] = sm.p[0][i];
                        if constexpr (LANES) {
#pragma unroll
                            for (int u = 1; u < 8; ++u) pv[s] = zadd(pv[s], sm.p[u][i]);
                        }
                        c[s] = sm.c[i];
                    }
                }
            } else {
                // all of this thread's slots in each look
                unsigned long long b[EPT][4];
                bool here[EPT];
#pragma unroll
                for (int s = 0; s < EPT; ++s) {
                    const int i = ti + 64 * VW * s;
                    here[s] = i < j || i >= n;
                    b[s][0] = b[s][1] = b[s][2] = b[s][3] = 0;
                }
                int spin = failed ? spin_limit : 0;
                while (true) {
#pragma unroll
                    for (int s = 0; s < EPT; ++s)
                        if (!here[s])
#pragma unroll
                            for (int u = 0; u < 4; ++u) b[s][u] = peek(slot_at(sl, u, ti + 64 * VW * s - j));
                    bool all = true;
#pragma unroll
                    for (int s = 0; s < EPT; ++s) {
                        here[s] = b[s][0] != EIG_EMPTY && b[s][1] != EIG_EMPTY && b[s][2] != EIG_EMPTY &&
                                  b[s][3] != EIG_EMPTY;
                        all = all && here[s];
                    }
                    if (all) break;
                    if (++spin > spin_limit) {
                        sm.fail = 1;
                        break;
                    }
                }
#pragma unroll
                for (int s = 0; s < EPT; ++s) {
                    pv[s] = make_double2(__longlong_as_double((long long)b[s][0]), __longlong_as_double((long long)b[s][1]));
                    c[s] = make_double2(__longlong_as_double((long long)b[s][2]), __longlong_as_double((long long)b[s][3]));
                }
            }
#pragma unroll
            for (int s = 0; s < EPT; ++s) {
                x[s] = zmul(tau, pv[s]);
                // conj(x) v
                dot.x = fma(x[s].x, vown[s].x, fma(x[s].y, vown[s].y, dot.x));
                dot.y = fma(x[s].x, vown[s].y, fma(-x[s].y, vown[s].x, dot.y));
                if (ti + 64 * VW * s == j) sm.xj = x[s];
            }
            double f = fold32(dot.x, dot.y);  // the two halves of the wave
            f = group_sum<16>(fold16(f, f));
            if (lane == 0) sm.red1[wave].x = f;
            if (lane == 32) sm.red1[wave].y = f;
            if (ti == 0) sm.stop = rem <= floor_tr;
        }
        __syncthreads();
        const bool stop = sm.stop != 0;
        double2 col[EPT];
        if (vec) {
            // ---- 2. w, column j, its reflector
            double2 dot = zadd(zadd(sm.red1[0], sm.red1[1]), zadd(sm.red1[2], sm.red1[3]));
            if (VW == 8)
                dot = zadd(dot, zadd(zadd(sm.red1[4], sm.red1[5]), zadd(sm.red1[6], sm.red1[7])));
            const double2 alpha = zscale(zmul(tau, dot), -0.5);
            const double2 wj = zadd(sm.xj, alpha);  // v_j = 1 for j > 0; zero otherwise
            double nrm = 0.0;
#pragma unroll
            for (int s = 0; s < EPT; ++s) {
                const int i = ti + 64 * VW * s;
                const double2 v = vown[s];
                const double2 w = zadd(x[s], zmul(alpha, v));
                // c - v conj(w_j) - w conj(v_j), v_j = 1
                col[s].x = c[s].x - (v.x * wj.x + v.y * wj.y) - (j > 0 ? w.x : 0.0);
                col[s].y = c[s].y - (v.y * wj.x - v.x * wj.y) - (j > 0 ? w.y : 0.0);
                sm.w[i] = (i > j && i < n) ? w : make_double2(0.0, 0.0);
                if (i > j + 1 && i < n) nrm = fma(col[s].x, col[s].x, fma(col[s].y, col[s].y, nrm));
                if (i == j + 1) sm.al = col[s];
                // (one workgroup: reflector j - 1 to its panel from the register)
                if (LANES && j > 0 && i < n && i >= ((j - 1) & ~15))
                    H[(int64_t)((j - 1) >> 4) * 16 * Cp + (int64_t)i * 16 + ((j - 1) & 15)] = v;
                if (i == j) sm.dj = col[s].x;
                if (member == 0 && i == j && !stop) ev.d[j] = col[s].x;
            }
            nrm = wave_sum64(nrm);
            if (lane == 0) sm.red2[wave] = nrm;
        }
        __syncthreads();
        // one exit only: with two, the registers' array is kept twice
        nref = stop ? j : n - 1;
        if (stop || j == n - 1) break;
        double2 *vn = sm.v[cur ^ 1];
        if (vec) {
            rem -= sm.dj;
            double nrm = (sm.red2[0] + sm.red2[1]) + (sm.red2[2] + sm.red2[3]);
            if (VW == 8) nrm += (sm.red2[4] + sm.red2[5]) + (sm.red2[6] + sm.red2[7]);
            const double2 al = sm.al;
            double beta = al.x;
            double2 sc = make_double2(0.0, 0.0);
            tau = make_double2(0.0, 0.0);
            if (!(fma(al.y, al.y, nrm) <= kTiny)) {
                beta = -copysign(sqrt(fma(al.x, al.x, fma(al.y, al.y, nrm))), al.x);
                const double ib = recip(beta);
                tau = make_double2((beta - al.x) * ib, -al.y * ib);
                const double2 df = make_double2(al.x - beta, al.y);
                const double id = recip(fma(df.x, df.x, df.y * df.y));
                sc = make_double2(df.x * id, -df.y * id);
            }
            if (member == 0 && ti == 0) {
                ev.e[j] = beta;
                ev.tau[j] = tau;
            }
#pragma unroll
            for (int s = 0; s < EPT; ++s) {
                const int i = ti + 64 * VW * s;
                vown[s] = i == j + 1 ? make_double2(1.0, 0.0)
                                     : ((i > j + 1 && i < n) ? zmul(col[s], sc) : make_double2(0.0, 0.0));
                vn[i] = vown[s];
            }
        }
        __syncthreads();
        // ---- 3. A -= v w^H + w v^H, p' = A v'; publish p' and column j + 1
        const double2 *v = sm.v[cur];
        const int J = j + 1, t0 = J >> 6;
        const Slots sl = slots_of(y, ld2, Cp, n, J);
        auto rows = [&](int g) {
            int row[4] = {n, n, n, n};
#pragma unroll
            for (int q = 0; q < NG; ++q) row[q] = 8 * (member + G * (g * NG + q)) + wave;
            double2 acc[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) acc[q] = make_double2(0.0, 0.0);
            int live = 0;  // rows of index >= J: the last ones
#pragma unroll
            for (int q = 0; q < NG; ++q) live += row[q] >= J;
            if (live == 0) return;
            if (live == 1)
                tri_rows<CH, RW, 1, NG, MEM>(a, A, p.LD, g * NG, v, sm.w, vn, lane, row, acc, t0, J, n, sm, sl);
            else if (live == 2)
                tri_rows<CH, RW, 2, NG, MEM>(a, A, p.LD, g * NG, v, sm.w, vn, lane, row, acc, t0, J, n, sm, sl);
            else if (live == 3)
                tri_rows<CH, RW, (NG < 3 ? NG : 3), NG, MEM>(a, A, p.LD, g * NG, v, sm.w, vn, lane, row, acc, t0, J, n, sm, sl);
            else
                tri_rows<CH, RW, NG, NG, MEM>(a, A, p.LD, g * NG, v, sm.w, vn, lane, row, acc, t0, J, n, sm, sl);
            const double s = wave_sum4(acc);
            const int q = lane >> 4, im = (lane >> 3) & 1;
            const int rq = 8 * (member + G * (g * NG + q)) + wave;
            if ((lane & 7) == 0 && q < NG && rq >= J && rq < n) {
                if (alone)
                    (im ? sm.p[0][rq].y : sm.p[0][rq].x) = s;
                else
                    publish(slot_at(sl, im, rq - J), s);
            }
        };
        if constexpr (LANES) {
            if (J < 64)
                tri_rows_alone<RW, 0>(a, v, sm.w, vn, lane, wave, J, n, sm);
            else
                tri_rows_alone<RW, 1>(a, v, sm.w, vn, lane, wave, J, n, sm);
        } else if constexpr (MEM) {
            for (int g = 0; g < (n + 8 * NG - 1) / (8 * NG); ++g) rows(g);
        } else {
#pragma unroll
            for (int g = 0; g < RW / NG; ++g) rows(g);
        }
        if (!LANES && j > 0) panel(j - 1, v);
        cur ^= 1;
        if (alone) __syncthreads();
    }
    if (!LANES && nref > 0) panel(nref - 1, sm.v[cur]);
    if (!alone && tid == 0 && sm.fail) reinterpret_cast<ProblemCtl *>(ws + p.ws_off)->conv = 0;
    if (member != 0) return;
    if (tid == 0) *ev.nref = nref;
    if (nref < n - 1 || sm.stop)
        for (int i = nref + tid; i < n; i += 512) {
            ev.d[i] = 0.0;
            ev.e[i] = 0.0;
        }
}

}  // namespace

// ---------------------------------------------- H = X X^H and X <- Y X
// A 32 x 32 tile of the result a workgroup, its four waves 16 of every 64 k:
// fragments straight from memory (lane l k = 4 (l / 16) .. + 3 of a wave's
// block in its four matrix instructions), three real products a complex one,
// the waves' sums meeting in LDS in a fixed order.
//   GRAM:  H (both triangles, from the tiles ti <= tj), A = B^H = X
//   else:  X = Y Xc, Xc the copy of X in the H region (row stride R)
// x: tile, y: problem. (A problem's tiles on one XCD, for its L2, gained nothing at 28
// problems of 512 rows and left XCDs idle beside fewer or uneven ones.)
// Bound: the FP64 matrix cores. Against 16 x 16 tiles of H and 32 x 32 or
// LDS-staged ones of X (us): 28 of 512 x 512: H 629 -> 266, X 631 -> 387; one: 30 -> 25
// and 31 -> 24; a layer with four of 1024 x 1024: 754 -> 250 and 1193 -> 358.
template <bool GRAM>
__global__ void __launch_bounds__(256, 2)
k_eig_gemm(const mpsx_two_site_op *ops, char *ws, int max_n) {
    __shared__ double2 part[4][32][33];
    const mpsx_plan p = ops[blockIdx.y].plan;
    int t = (int)blockIdx.x;
    if (!eig_direct(p, max_n)) return;
    const int n = p.C, Cp = p.Cp, R = p.R, nt = (n + 31) / 32;
    int ti, tj;
    if (GRAM) {
        ti = 0;
        while (ti < nt && t >= nt - ti) t -= nt - ti++;
        if (ti >= nt) return;
        tj = ti + t;
    } else {
        const int nc = (R + 31) / 32;
        ti = t / nc;
        tj = t % nc;
        if (ti >= nt) return;
    }
    double2 *Z = reinterpret_cast<double2 *>(ws + z_off(p));
    double2 *H = eig_h(ws, p);
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_id(), l16 = lane & 15, q = lane >> 4;
    const int64_t LD = p.LD;
    const int K = GRAM ? R : n;
    // rows and columns beyond the matrix repeat its last one (never stored)
    const double2 *A[2], *B[2];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        const int i = min(32 * ti + 16 * a + l16, n - 1), j = 32 * tj + 16 * a + l16;
        A[a] = Z + (GRAM ? 0 : R) + i * LD;
        B[a] = GRAM ? Z + min(j, n - 1) * LD : H + min(j, R - 1);
    }
    mfma_d4 acc[2][2][3];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int u = 0; u < 3; ++u) acc[a][b][u] = mfma_d4{0.0, 0.0, 0.0, 0.0};
    auto multiply = [&](const double2 (&x)[2][4], const double2 (&y)[2][4]) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            double xs[2], ys[2];
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                xs[a] = x[a][u].x + x[a][u].y;
                ys[a] = GRAM ? y[a][u].x - y[a][u].y : y[a][u].x + y[a][u].y;
            }
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    acc[a][b][0] = mfma16d(x[a][u].x, y[b][u].x, acc[a][b][0]);
                    acc[a][b][1] = mfma16d(x[a][u].y, y[b][u].y, acc[a][b][1]);
                    acc[a][b][2] = mfma16d(xs[a], ys[b], acc[a][b][2]);
                }
        }
    };
    double2 x[2][4], y[2][4];
    int k0 = 16 * wave;
    for (; k0 + 16 <= K; k0 += 64) {
        const int k = k0 + 4 * q;
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                x[a][u] = A[a][k + u];
                y[a][u] = GRAM ? B[a][k + u] : B[a][(int64_t)(k + u) * R];
            }
        multiply(x, y);
    }
    if (k0 < K) {
        const int k = k0 + 4 * q;
        const double2 zero = make_double2(0.0, 0.0);
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                x[a][u] = k + u < K ? A[a][k + u] : zero;
                y[a][u] = k + u < K ? (GRAM ? B[a][k + u] : B[a][(int64_t)(k + u) * R]) : zero;
            }
        multiply(x, y);
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const double p1 = acc[a][b][0][r], p2 = acc[a][b][1][r], p3 = acc[a][b][2][r];
                part[wave][16 * a + 4 * r + q][16 * b + l16] =
                    GRAM ? make_double2(p1 + p2, p3 - p1 + p2) : make_double2(p1 - p2, p3 - p1 - p2);
            }
    __syncthreads();
    auto entry = [&](int i, int j) {
        return zadd(zadd(part[0][i][j], part[2][i][j]), zadd(part[1][i][j], part[3][i][j]));
    };
    for (int e = tid; e < 32 * 32; e += 256) {
        const int i = e >> 5, j = e & 31, gi = 32 * ti + i, gj = 32 * tj + j;
        if (GRAM) {
            if (gi < n && gj < n) {
                double2 v = entry(i, j);
                if (gi == gj) v.y = 0.0;
                H[(int64_t)gi * Cp + gj] = v;
            }
            // the mirrored tile, by rows of its own
            if (ti != tj && 32 * tj + i < n && 32 * ti + j < n)
                H[(int64_t)(32 * tj + i) * Cp + 32 * ti + j] = zconj(entry(j, i));
        } else if (gi < n && gj < R) {
            Z[gi * LD + gj] = entry(i, j);
        }
    }
}

// Table of the workgroups of k_tridiag: entry s = (problem, member << 8 |
// group size), the problems with the largest groups first. One workgroup.
__global__ void __launch_bounds__(256)
k_eig_map(const mpsx_two_site_op *ops, int count, char *ws, int2 *map, int max_n, int spread) {
    __shared__ int wsum[4];
    __shared__ int total;
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
    if (tid == 0) {
        total = 0;
        reinterpret_cast<TwoSiteHeader *>(ws)->spread = spread;
    }
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
k_tridiag(const mpsx_two_site_op *ops, const int2 *map, char *ws, int slots, int ticket, int spread,
          int spin_limit) {
    __shared__ TriShared<128, 8> sm;
    int slot = (int)blockIdx.x;
    if (ticket) {  // by order of start
        if (threadIdx.x == 0) sm.slot = atomicAdd(&reinterpret_cast<TwoSiteHeader *>(ws)->ticket, 1);
        __syncthreads();
        slot = sm.slot;
    }
    if (slot >= slots) return;
    const int2 m = map[slot];
    const mpsx_plan p = ops[m.x].plan;
    const int G = m.y & 255;
    int member = m.y >> 8;
    if (!ticket) member = (member & 7) * (G >> 3) + min(member & 7, G & 7) + (member >> 3);  // XCD by XCD
    if (threadIdx.x == 0)
        sm.whole = form_group(&reinterpret_cast<ProblemCtl *>(ws + p.ws_off)->group, G, spread);
    __syncthreads();
    if (!sm.whole) return;
    switch (eig_class(p.C)) {
        case 0: tridiag<2, 16, false>(p, ws, member, G, spin_limit, sm); break;
        case 1: tridiag<4, 8, false>(p, ws, member, G, spin_limit, sm); break;
        case 2: tridiag<8, 4, false>(p, ws, member, G, spin_limit, sm); break;
        default: tridiag<16, 2, false>(p, ws, member, G, spin_limit, sm); break;
    }
}

// The problems whose group was given up, one workgroup each, the matrix in
// memory: it waits for no other workgroup. The results have the same bits.
__global__ void __launch_bounds__(512, 2)
k_tridiag_one(const mpsx_two_site_op *ops, char *ws, int max_n) {
    __shared__ TriShared<EIG_MAX_N, 1> sm;
    const mpsx_plan p = ops[blockIdx.x].plan;
    if (!eig_direct(p, max_n)) return;
    if (!(reinterpret_cast<const ProblemCtl *>(ws + p.ws_off)->group & EIG_GROUP_LOST)) return;
    switch (eig_class(p.C)) {
        case 0: break;  // a group of one
        case 1: tridiag<4, 8, true>(p, ws, 0, 1, 0, sm); break;
        case 2: tridiag<8, 4, true>(p, ws, 0, 1, 0, sm); break;
        default: tridiag<16, 2, true>(p, ws, 0, 1, 0, sm); break;
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
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_id(), l16 = lane & 15, lq = lane >> 4;
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
// Leaves: the eigensystem of every 64 x 64 diagonal block of T, torn at each
// entry, by six levels of merges in LDS. x: block, y: problem. Also scales T to
// unit norm (es, d) for the merges above.
__global__ void __launch_bounds__(LEAF_THREADS)
k_eig_leaf(const mpsx_two_site_op *ops, char *ws, int max_n, int leaves) {
    constexpr int M = LEAF;
    __shared__ double S[M][M + 1], U[M][M + 1];
    __shared__ LeafShared L;
    __shared__ double red[8];
    const mpsx_plan p = ops[blockIdx.y].plan;
    if (!eig_direct(p, max_n)) return;
    const int n = p.C;
    if ((int)blockIdx.x >= leaves) {
        // both buffers of S^T are zero outside the leaves' blocks (the merges
        // write their own blocks only): eight rows a workgroup
        const int row = 8 * ((int)blockIdx.x - leaves) + (threadIdx.x >> 6);
        if (row >= n) return;
        double *yr = eig_y(ws, p) + (int64_t)row * 2 * p.LD;
        const int l0 = row & ~(M - 1);
        for (int r = threadIdx.x & 63; r < 2 * p.Cp; r += 64)
            if (r < l0 || r >= min(l0 + M, n)) yr[r] = 0.0;
        return;
    }
    const int b0 = (int)blockIdx.x * M;
    if (b0 >= n) return;
    const int m = min(M, n - b0), tid = threadIdx.x;
    const EigVec ev = eig_vec(ws, p);
    double mx = 0.0;
    for (int i = tid; i < n; i += LEAF_THREADS) {
        mx = fmax(mx, fabs(ev.d[i]));
        if (i + 1 < n) mx = fmax(mx, fabs(ev.e[i]));
    }
    for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o, 64));
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
    mx = fmax(fmax(fmax(red[0], red[1]), fmax(red[2], red[3])), fmax(fmax(red[4], red[5]), fmax(red[6], red[7])));
    const double scale = mx > 0.0 ? 1.0 / mx : 1.0;
    auto off = [&](int i) { return (i >= 0 && i + 1 < n) ? ev.e[i] * scale : 0.0; };
    if (tid < M) {
        const int i = b0 + tid;
        // d stays unscaled in memory (other leaves read it): this leaf's
        // eigenvalues go to rt, where the first merge takes them
        L.d[tid] = i < n ? ev.d[i] * scale - fabs(off(i - 1)) - fabs(off(i)) : 0.0;
        L.e[tid] = off(i);
        if (i < n) ev.es[i] = off(i);
    }
    leaf_conquer(m, S, U, L);
    double *y = eig_y(ws, p);
    const int64_t ld2 = 2 * (int64_t)p.LD;
    for (int j = tid >> 6; j < m; j += 8) {
        const int rr = tid & 63;
        if (rr < m) y[(int64_t)(b0 + j) * ld2 + b0 + rr] = S[j][rr];
    }
    if (tid < m) ev.rt[b0 + tid] = L.d[tid];
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
    __shared__ int sK, sR, kept[8];
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
    // The entries of negligible weight go to the end (from it here, in order when
    // they are written out); only if two of the others then have to be rotated
    // together is the serial pass made (0.2 us an entry).
    int before = 0;
    for (int b = 0; b < m; b += 512) {
        const int i = b + tid;
        const bool keep = i < m && rho * fabs(zs[i]) > kDeflate;
        const unsigned long long mask = __ballot(keep);
        if ((tid & 63) == 0) kept[tid >> 6] = __popcll(mask);
        __syncthreads();
        int at = before + __popcll(mask & ((1ULL << (tid & 63)) - 1)), all = 0;
        for (int u = 0; u < 8; ++u) {
            if (u < (tid >> 6)) at += kept[u];
            all += kept[u];
        }
        if (keep) {
            dl[at] = ds[i];
            zl[at] = zs[i];
            src[at] = id[i];
        } else if (i < m) {
            const int e = m - 1 - (i - at);
            dd[e] = ds[i];
            src[e] = id[i];
        }
        before += all;
        __syncthreads();
    }
    bool some = false;
    for (int i = tid; i + 1 < before; i += 512) some = some || may_deflate(before, i, rho, dl, zl);
    if (tid == 0) sK = before;
    const bool serial = __syncthreads_or(some);
    if (serial) {
        if (tid == 0) sK = deflate(m, m - before, rho, ds, zs, id, dl, zl, src, dd, rot_i, rot_c, &sR);
        __syncthreads();
    }
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
        const int o = i < K || serial ? i : m - 1 - (i - K);
        ev.src[lo + i] = src[o];
        if (i < K) {
            ev.dl[lo + i] = dl[i];
            ev.zl[lo + i] = zl[i];
        } else {
            ev.d[lo + i] = dd[o];
        }
    }
    if (tid == 0) {
        ev.kn[lo] = K;
        ev.rho[lo] = rho;
    }
}

// (The four kernels of a level at 512 rows, us, with the poles one by one, staged
// rows and a serial deflation -> now: merge 101 -> 26, roots 41 -> 10, weights 18 -> 5,
// vectors 66 -> 21.)
//
// The secular roots of a level's merges, a wave per root: 4 roots per workgroup
// (x; all of one merge, whose first row is a multiple of 128), y: problem.
__global__ void __launch_bounds__(256)
k_eig_roots(const mpsx_two_site_op *ops, char *ws, int max_n, int s) {
    const mpsx_plan p = ops[blockIdx.y].plan;
    if (!eig_direct(p, max_n)) return;
    const int n = p.C, row = (int)blockIdx.x * 4 + wave_id(), sub = threadIdx.x & 63;
    if (s >= n || row >= n) return;
    const int lo = row & ~(2 * s - 1), j = row - lo;
    const EigVec ev = eig_vec(ws, p);
    const int K = ev.kn[lo];
    if (j >= K) return;
    const double *dl = ev.dl + lo, *zl = ev.zl + lo;
    double d[EIG_MAX_N / 64], z2[EIG_MAX_N / 64];
#pragma unroll
    for (int u = 0; u < EIG_MAX_N / 64; ++u) {
        const int i = sub + 64 * u;
        d[u] = 1e200;
        z2[u] = 0.0;
        if (64 * u >= K) continue;
        if (i < K) {
            const double z = zl[i];
            d[u] = dl[i];
            z2[u] = z * z;
        }
    }
    const int nx = min(j + 1, K - 1);
    const double dj = dl[j], dn = dl[nx];
    double root;
    const double pole = secular_root<64, EIG_MAX_N / 64>(K, d, z2, dj, dn, zl[j], zl[nx], ev.rho[lo], j, sub, &root) ? dn : dj;
    if (sub == 0) {
        ev.pb[row] = pole;
        ev.rt[row] = root;
        ev.d[row] = pole + root;
    }
}

// The recomputed weights, a wave per pole, split as k_eig_roots.
__global__ void __launch_bounds__(256)
k_eig_weights(const mpsx_two_site_op *ops, char *ws, int max_n, int s) {
    const mpsx_plan p = ops[blockIdx.y].plan;
    if (!eig_direct(p, max_n)) return;
    const int n = p.C, row = (int)blockIdx.x * 4 + wave_id(), sub = threadIdx.x & 63;
    if (s >= n || row >= n) return;
    const int lo = row & ~(2 * s - 1), i = row - lo;
    const EigVec ev = eig_vec(ws, p);
    const int K = ev.kn[lo];
    if (i >= K) return;
    double v = group_prod<16>(zhat_factors<64>(K, ev.dl + lo, ev.pb + lo, ev.rt + lo, i, sub));
    v *= __shfl_xor(v, 16, 64);
    v *= __shfl_xor(v, 32, 64);
    if (sub == 0) ev.zh[row] = copysign(sqrt(fmax(v, 0.0)), ev.zl[row]);
}

// Rows of the merged S^T (buffer buf ^ 1): row j < K is sum_i u_ij S^T[src_i],
// u_ij = zh_i / (d_i - lambda_j), normalised; the deflated rows are copied. A
// wave has 16 rows and 32 columns on the FP64 matrix cores and the entries of u
// formed in its lanes (lane l poles 4 (l / 16) .. + 3 of a block of 16); the
// rows of S^T are on their way a block ahead, their indices two. Staged through
// LDS in 64 x 64 tiles a block of 16 poles took 2 us. x: 64-row tile * column
// tiles + 32-column tile of a merge, z: merge, y: problem.
__global__ void __launch_bounds__(256)
k_eig_vectors(const mpsx_two_site_op *ops, char *ws, int max_n, int s, int buf) {
    const mpsx_plan p = ops[blockIdx.y].plan;
    if (!eig_direct(p, max_n)) return;
    const int n = p.C, lo = (int)blockIdx.z * 2 * s;
    if (s >= n || lo >= n) return;
    const int hi = min(lo + 2 * s, n), m = hi - lo;
    const int ct = (2 * s) / 32, j0 = ((int)blockIdx.x / ct) * 64, c0 = ((int)blockIdx.x % ct) * 32;
    if (j0 >= m || c0 >= m) return;
    const EigVec ev = eig_vec(ws, p);
    const int64_t ld2 = 2 * (int64_t)p.LD;
    const double *in = eig_y(ws, p) + (int64_t)buf * p.Cp + lo;
    double *out = eig_y(ws, p) + (int64_t)(buf ^ 1) * p.Cp + lo;
    const int K = ev.kn[lo];
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, q = lane >> 4;
    const int j1 = j0 + 16 * wave_id();  // this wave's rows
    if (j1 < K) {
        const int j = min(j1 + l16, K - 1);
        const double db = ev.pb[lo + j], tj = ev.rt[lo + j];
        // columns beyond the merge repeat its last (never stored)
        const double *col[2] = {in + min(c0 + l16, m - 1), in + min(c0 + 16 + l16, m - 1)};
        const int blocks = (K + 15) / 16;
        struct Poles {
            double zh[4], dl[4];
            int src[4];
        };
        auto poles = [&](int b, Poles &x) {  // of block b, or of the last again
            const int i0 = lo + 16 * min(b, blocks - 1) + 4 * q;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const bool on = i0 + t < lo + K;
                x.zh[t] = on ? ev.zh[i0 + t] : 0.0;
                x.dl[t] = on ? ev.dl[i0 + t] : 1e200;
                x.src[t] = on ? ev.src[i0 + t] : lo;
            }
        };
        auto rows = [&](const Poles &x, double (&v)[2][4]) {
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int c = 0; c < 2; ++c) v[c][t] = col[c][x.src[t] * ld2];
        };
        mfma_d4 acc[2] = {{0.0, 0.0, 0.0, 0.0}, {0.0, 0.0, 0.0, 0.0}};
        double nn = 0.0;
        auto multiply = [&](const Poles &x, const double (&v)[2][4]) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const double u = x.zh[t] * recip((x.dl[t] - db) - tj);
                nn = fma(u, u, nn);
#pragma unroll
                for (int c = 0; c < 2; ++c) acc[c] = mfma16d(u, v[c][t], acc[c]);
            }
        };
        Poles x0, x1, x2;
        double v0[2][4], v1[2][4];
        poles(0, x0);
        poles(1, x1);
        rows(x0, v0);
        for (int b = 0; b < blocks; b += 2) {
            rows(x1, v1);
            poles(b + 2, x2);
            multiply(x0, v0);
            if (b + 1 >= blocks) break;
            rows(x2, v0);
            x0 = x2;
            poles(b + 3, x2);
            multiply(x1, v1);
            x1 = x2;
        }
        nn += __shfl_xor(nn, 16, 64);
        nn += __shfl_xor(nn, 32, 64);
        const double f = 1.0 / sqrt(nn);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int jj = 4 * r + q;
            const double fj = __shfl(f, jj, 64);
#pragma unroll
            for (int c = 0; c < 2; ++c)
                if (j1 + jj < K && c0 + 16 * c + l16 < m)
                    out[(int64_t)(lo + j1 + jj) * ld2 + c0 + 16 * c + l16] = acc[c][r] * fj;
        }
    }
    if (j0 + 64 > K)  // deflated rows
        for (int e = tid; e < 64 * 32; e += 256) {
            const int j = j0 + (e >> 5), cc = c0 + (e & 31);
            if (j >= K && j < m && cc < m) out[(int64_t)(lo + j) * ld2 + cc] = in[(int64_t)ev.src[lo + j] * ld2 + cc];
        }
}

// ---------------------------------------------------- back transformation
// Y rows i0 .. i0 + 15 = (Q s_i)^H: the strip [s_i0 .. s_i0+15] (n x 16, one
// eigenvector a column) in the matrix-core output layout in registers (eight
// waves; wave w the 16-row chunks w, w + 8, ...), the panels' block
// reflectors I - V T V^H from the last to the first. x: strip, y: problem.
// CH chunks a wave: 4 up to 512 rows, 8 up to 1024. Registers for two waves a
// SIMD: for four, CH = 4 spilled (one strip set of 512 rows 333 us, now 274;
// 28 of them 944, now 990). Bound: the FP64 matrix cores of a strip's one
// compute unit and the three barriers a panel; V is read once per strip, from
// the L2.
template <int CH>
__global__ void __launch_bounds__(512, 2)
k_eig_back(const mpsx_two_site_op *ops, char *ws, int max_n) {
    __shared__ double2 Wp[8][16][17];
    __shared__ double2 Wt[16][17], Ws[16][17], Ts[16][17];
    const mpsx_plan p = ops[blockIdx.y].plan;
    if (!eig_direct(p, max_n) || (CH == 4) != (p.C <= 512)) return;
    const int n = p.C, Cp = p.Cp, i0 = 16 * (int)blockIdx.x;
    if (i0 >= n) return;
    const int tid = threadIdx.x, lane = tid & 63, w = wave_id(), l16 = lane & 15, lq = lane >> 4;
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
                              int slots, bool grouped, bool ticket, bool no_wait) {
    static std::atomic<unsigned> launches{0};
    const int spread = (int)(launches.fetch_add(1, std::memory_order_relaxed) & 3);
    hipLaunchKernelGGL(k_eig_map, dim3(1), dim3(256), 0, s, d, count, ws, static_cast<int2 *>(map), max_n, spread);
    hipLaunchKernelGGL(k_tridiag, dim3((unsigned)slots), dim3(512), 0, s, d, static_cast<const int2 *>(map), ws,
                       slots, ticket ? 1 : 0, spread, no_wait ? 0 : kSpin);
    if (grouped)
        hipLaunchKernelGGL(k_tridiag_one, dim3((unsigned)count), dim3(512), 0, s, d, ws, max_n);
    return hipGetLastError();
}

hipError_t launch_eig_conquer(hipStream_t s, const mpsx_two_site_op *d, int count, char *ws, int max_n, int n) {
    const unsigned y = (unsigned)count;
    const int leaves = (n + 63) / 64;
    hipLaunchKernelGGL(k_eig_leaf, dim3((unsigned)(leaves + (n + 7) / 8), y), dim3(LEAF_THREADS), 0, s, d, ws, max_n,
                       leaves);
    int buf = 0;
    for (int h = 64; h < n; h *= 2, buf ^= 1) {
        const unsigned nodes = (unsigned)((n + 2 * h - 1) / (2 * h)), tiles = (unsigned)(2 * h / 64);
        const unsigned roots = (unsigned)((n + 3) / 4);
        hipLaunchKernelGGL(k_eig_merge, dim3(nodes, y), dim3(512), 0, s, d, ws, max_n, h, buf, h == 64 ? 1 : 0);
        hipLaunchKernelGGL(k_eig_roots, dim3(roots, y), dim3(256), 0, s, d, ws, max_n, h);
        hipLaunchKernelGGL(k_eig_weights, dim3(roots, y), dim3(256), 0, s, d, ws, max_n, h);
        hipLaunchKernelGGL(k_eig_vectors, dim3(2 * tiles * tiles, y, nodes), dim3(256), 0, s, d, ws, max_n, h, buf);
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

hipError_t launch_eig_gram(hipStream_t s, const mpsx_two_site_op *d, int count, char *ws, int max_n, int n) {
    const unsigned nt = (unsigned)((n + 31) / 32), tiles = nt * (nt + 1) / 2;
    hipLaunchKernelGGL(k_eig_gemm<true>, dim3(tiles, (unsigned)count), dim3(256), 0, s, d, ws, max_n);
    return hipGetLastError();
}

hipError_t launch_eig_apply(hipStream_t s, const mpsx_two_site_op *d, int count, char *ws, int max_n, int64_t tiles) {
    hipLaunchKernelGGL(k_eig_gemm<false>, dim3((unsigned)tiles, (unsigned)count), dim3(256), 0, s, d, ws, max_n);
    return hipGetLastError();
}
