// Two-site updates of at most 64 rows (gfx950): everything after theta in one
// workgroup and one launch.
//
// Z = [X | Y] stays in the problem's workspace rows (L2), Y starting as the
// identity; the 64 x 64 working matrices are in LDS. Repeated until the rows
// of X are orthogonal (the test of the Jacobi rounds: every pair within tol of
// the norms' product, rows below null2 aside):
//   H = X X^H (FP64 matrix cores);
//   the m rows of some pair that fails the test; W, the eigenvectors of their
//   block of H, by the direct route of eig.hip (tridiagonal form, divide and
//   conquer), up to m = 8 by Jacobi sweeps until nothing rotates;
//   those rows of Z <- W (those rows of Z).
// The direct route leaves rows orthogonal to FP64 rounding of the largest of
// them. The rows below that (a graded spectrum, the rounding noise of a
// rank-deficient theta) still fail and are the next pass's block, which
// resolves them on their own scale: a pass covers about seven decades. Every
// fourth pass is a Jacobi sweep over the block, whose convergence needs no such
// argument.
// Then the norms, the order, the truncation and the two factors. The rows are
// formed again from Z before every test, so nothing is lost to H's rounding.
//
// Bound: latency. A column of the tridiagonal form is about 2 us (instruction
// issue and a barrier), the leaf's six levels 60 us; the kernel takes 280 us
// at 64 x 64, 75 at 16, 20 at 4. The launch sequence of the same steps
// (16 launches of 5 us and more, a poll per sweep) took 1100 us at 64 x 64 and
// 170 at 4 x 4.
#include <hip/hip_runtime.h>

#include <cstddef>

#include "common.h"
#include "eig_dc.h"
#include "launch.h"

namespace {

constexpr int SN = 64;    // rows
constexpr int kPasses = 30;  // then the problem is reported as not converged
constexpr int ST = LEAF_THREADS;  // 512
constexpr int SW = ST / 64;

struct SmallShared {
    double2 A[SN][SN + 1];  // H; then the reflectors, column j = reflector j
    union {
        double2 Q[SN][SN + 1];  // W
        struct {
            double S[SN][SN + 1], U[SN][SN + 1];
        };
    };
    LeafShared L;
    double2 p[2][SN], c[2][SN];  // A v and the next column, two steps
    double d[SN], e[SN];
    double2 tau[SN];
    double sig[SN];
    int perm[SN];
    int row8[7][4];           // the index pairs of a sweep over at most 8 rows
    int row[SN], pos[SN];  // the block's rows; the place of a row in it, or -1
    int fail[SN];
    double prm_c[SN / 2];
    double2 prm_s[SN / 2];
    int any, nref;
};

MPSX_DEV double2 lane_z(double2 v, int lane) { return make_double2(lane_f64(v.x, lane), lane_f64(v.y, lane)); }

// H = X X^H from the rows of Z, both triangles. Wave w forms the 16 x 16 tiles
// w, w + 8, ... of the upper block triangle.
MPSX_DEV void small_gram(const double2 *Z, int64_t LD, int n, int R, SmallShared &sm) {
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_id(), l16 = lane & 15, lq = lane >> 4;
    const int nt = (n + 15) / 16, tiles = nt * (nt + 1) / 2;
    for (int t = wave; t < tiles; t += SW) {
        int rem = t, ti = 0;
        while (rem >= nt - ti) {
            rem -= nt - ti;
            ++ti;
        }
        const int tj = ti + rem;
        const int ra = 16 * ti + l16, rb = 16 * tj + l16;
        const double2 *za = Z + (int64_t)ra * LD, *zb = Z + (int64_t)rb * LD;
        mfma_d4 p1 = {0.0, 0.0, 0.0, 0.0}, p2 = p1, p3 = p1;
        auto load = [&](int c0, double2 (&va)[4], double2 (&vb)[4]) {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int c = c0 + 4 * lq + k;
                va[k] = (ra < n && c < R) ? za[c] : make_double2(0.0, 0.0);
                vb[k] = (rb < n && c < R) ? zb[c] : make_double2(0.0, 0.0);
            }
        };
        double2 va[4], vb[4], na[4], nb[4];
        load(0, va, vb);
        for (int c0 = 0; c0 < R; c0 += 16) {
            load(c0 + 16, na, nb);  // the next columns are in flight during these products
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                p1 = mfma16d(va[k].x, vb[k].x, p1);
                p2 = mfma16d(va[k].y, vb[k].y, p2);
                p3 = mfma16d(va[k].x + va[k].y, vb[k].x - vb[k].y, p3);
                va[k] = na[k];
                vb[k] = nb[k];
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = 16 * ti + 4 * r + lq, j = 16 * tj + l16;
            double2 v = make_double2(p1[r] + p2[r], p3[r] - p1[r] + p2[r]);
            if (ti == tj) {  // the diagonal tile from its upper triangle
                if (i > j) continue;
                if (i == j) v.y = 0.0;
            }
            sm.A[i][j] = v;
            sm.A[j][i] = zconj(v);
        }
    }
    __syncthreads();
}

// Tridiagonal form of H (n <= 64) and its reflectors in A: the steps of
// tridiag() in eig.hip with the matrix in one workgroup's registers (wave w the
// rows w, w + 8, ..., a column a lane) and the vectors repeated by every wave,
// an element a lane, so that a step has one barrier.
MPSX_DEV void small_tridiag(int n, SmallShared &sm) {
    const int tid = threadIdx.x, lane0 = tid & 63, wave = wave_id();
    constexpr int RW = SN / SW;  // rows a wave
    double2 a[RW];
#pragma unroll
    for (int q = 0; q < RW; ++q) {
        const int row = wave + SW * q;
        a[q] = (row < n && lane0 < n) ? sm.A[row][lane0] : make_double2(0.0, 0.0);
    }
    double2 c0 = lane0 < n ? sm.A[lane0][0] : make_double2(0.0, 0.0);
    double rem = wave_sum64(lane0 < n ? sm.A[lane0][lane0].x : 0.0);
    const double floor_tr = 64.0 * kEps * rem;
    __syncthreads();  // A is free for the reflectors
    double2 tau = make_double2(0.0, 0.0), v = tau;
    int nref = n - 1;
    for (int j = 0; j < n; ++j) {
        // the lane through an empty asm statement: addresses are formed in the
        // step rather than held (and spilled) across it
        int lane = tid & 63;
        asm volatile("" : "+v"(lane));
        const bool on = lane >= j && lane < n;
        double2 pv = make_double2(0.0, 0.0), c = c0;
        if (j > 0) {
            c = make_double2(0.0, 0.0);
            if (on) {
                pv = sm.p[j & 1][lane];
                c = sm.c[j & 1][lane];
            }
        }
        const double2 x = zmul(tau, pv);
        // x^H v, real and imaginary part in the two halves of the wave
        const double dre = fma(x.x, v.x, x.y * v.y), dim = fma(x.x, v.y, -x.y * v.x);
        double f = fold32(dre, dim);
        f = group_sum<16>(fold16(f, f));
        const double2 dot = make_double2(lane_f64(f, 0), lane_f64(f, 32));
        const double2 alpha = zscale(zmul(tau, dot), -0.5);
        const double2 w = zadd(x, zmul(alpha, v));
        const double2 wj = lane_z(w, j);
        double2 col = c;
        if (j > 0) {
            col.x = c.x - (v.x * wj.x + v.y * wj.y) - w.x;
            col.y = c.y - (v.y * wj.x - v.x * wj.y) - w.y;
        }
        const double dj = lane_f64(col.x, j);
        if (rem <= floor_tr) {
            nref = j;
            if (wave == 0 && on) {
                sm.d[lane] = 0.0;
                sm.e[lane] = 0.0;
            }
            break;
        }
        if (tid == 0) sm.d[j] = dj;
        if (j == n - 1) {
            if (tid == 0) sm.e[j] = 0.0;
            break;
        }
        rem -= dj;
        const double nrm = wave_sum64((lane > j + 1 && lane < n) ? fma(col.x, col.x, col.y * col.y) : 0.0);
        const double2 al = lane_z(col, j + 1);
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
        const double2 vo = v;
        v = lane == j + 1 ? make_double2(1.0, 0.0)
                          : ((lane > j + 1 && lane < n) ? zmul(col, sc) : make_double2(0.0, 0.0));
        if (tid == 0) {
            sm.e[j] = beta;
            sm.tau[j] = tau;
        }
        if (wave == (j & (SW - 1))) sm.A[lane][j] = v;
        // A -= v w^H + w v^H, p = A v', column j + 1
        const int nx = (j + 1) & 1;
        double2 acc[RW];
#pragma unroll
        for (int q = 0; q < RW; ++q) {
            const int row = wave + SW * q;
            acc[q] = make_double2(0.0, 0.0);
            if (row <= j || row >= n) continue;
            const double2 vi = lane_z(vo, row), wi = lane_z(w, row);
            double2 y = a[q];
            y.x = fma(-vi.x, w.x, fma(-vi.y, w.y, fma(-wi.x, vo.x, fma(-wi.y, vo.y, y.x))));
            y.y = fma(-vi.y, w.x, fma(vi.x, w.y, fma(-wi.y, vo.x, fma(wi.x, vo.y, y.y))));
            a[q] = y;
            acc[q].x = fma(y.x, v.x, -y.y * v.y);
            acc[q].y = fma(y.x, v.y, y.y * v.x);
            if (row == j + 1) sm.c[nx][lane] = zconj(y);  // column j + 1 is this row, conjugated
        }
        const double s = wave_sum8(acc);
        const int q = (lane >> 4) + 4 * ((lane >> 3) & 1), row = wave + SW * q;
        if ((lane & 3) == 0 && row > j && row < n) (lane & 4 ? sm.p[nx][row].y : sm.p[nx][row].x) = s;
        __syncthreads();
    }
    if (tid == 0) sm.nref = nref;
    __syncthreads();
}

// W = (Q S)^H from the eigenvectors S of T and the reflectors in A: eight lanes
// an eigenvector, the reflectors from the last to the first.
MPSX_DEV void small_back(int n, SmallShared &sm) {
    constexpr int LV = ST / SN, XR = SN / LV;  // lanes an eigenvector, rows a lane
    const int tid = threadIdx.x, j = tid / LV, sub = tid % LV;
    double2 x[XR];
#pragma unroll
    for (int t = 0; t < XR; ++t) {
        const int r = sub + LV * t;
        x[t] = make_double2((j < n && r < n) ? sm.S[j][r] : 0.0, 0.0);
    }
    __syncthreads();  // S shares its memory with Q
    for (int q = sm.nref - 1; q >= 0; --q) {
        double2 dot = make_double2(0.0, 0.0);
        double2 vr[XR];
        const int t0 = (q + 1) / LV;
#pragma unroll
        for (int t = 0; t < XR; ++t) {
            if (t < t0) continue;
            vr[t] = sm.A[sub + LV * t][q];
            dot.x = fma(vr[t].x, x[t].x, fma(vr[t].y, x[t].y, dot.x));
            dot.y = fma(vr[t].x, x[t].y, fma(-vr[t].y, x[t].x, dot.y));
        }
        dot = make_double2(group_sum<LV>(dot.x), group_sum<LV>(dot.y));
        const double2 f = zmul(sm.tau[q], dot);
#pragma unroll
        for (int t = 0; t < XR; ++t) {
            if (t < t0) continue;
            x[t].x = fma(-vr[t].x, f.x, fma(vr[t].y, f.y, x[t].x));
            x[t].y = fma(-vr[t].x, f.y, fma(-vr[t].y, f.x, x[t].y));
        }
    }
    if (j < n)
#pragma unroll
        for (int t = 0; t < XR; ++t) {
            const int r = sub + LV * t;
            if (r < n) sm.Q[j][r] = zconj(x[t]);
        }
    __syncthreads();
}

// Rotation [[c, s], [-conj(s), c]] that diagonalises [[a, h], [conj(h), b]], T = (b
// - a) / 2, g2 = |h|^2 > 0: tan of its angle t = w |h| with w = sign(T) / (|T| +
// sqrt(T^2 + |h|^2)), s = w c h.
MPSX_DEV void jacobi_angle(double T, double g2, double2 h, double *c, double2 *s) {
    const double w = copysign(1.0 / (fabs(T) + sqrt(fma(T, T, g2))), T);
    *c = 1.0 / sqrt(fma(w * w, g2, 1.0));
    *s = make_double2(w * *c * h.x, w * *c * h.y);
}
// H <- J1^H H J2 on the block of the index pairs (p1, q1), (p2, q2); index n (the
// idle partner of an odd n) has an identity rotation.
MPSX_DEV void jacobi_block(int n, SmallShared &sm, int p1, int q1, int p2, int q2, double c1, double2 s1, double c2,
                           double2 s2) {
    if (s1.x == 0.0 && s1.y == 0.0 && s2.x == 0.0 && s2.y == 0.0) return;
    const bool i1 = q1 < n, i2 = q2 < n;
    const double2 z = make_double2(0.0, 0.0);
    const double2 h00 = sm.A[p1][p2], h01 = i2 ? sm.A[p1][q2] : z, h10 = i1 ? sm.A[q1][p2] : z,
                  h11 = i1 && i2 ? sm.A[q1][q2] : z;
    const double2 ms2 = make_double2(-s2.x, s2.y);
    const double2 m00 = zadd(zscale(h00, c2), zmul(h01, ms2)), m01 = zadd(zmul(h00, s2), zscale(h01, c2));
    const double2 m10 = zadd(zscale(h10, c2), zmul(h11, ms2)), m11 = zadd(zmul(h10, s2), zscale(h11, c2));
    const double2 ns1 = make_double2(-s1.x, -s1.y), cs1 = zconj(s1);
    sm.A[p1][p2] = zadd(zscale(m00, c1), zmul(ns1, m10));
    if (i2) sm.A[p1][q2] = zadd(zscale(m01, c1), zmul(ns1, m11));
    if (i1) sm.A[q1][p2] = zadd(zmul(cs1, m00), zscale(m10, c1));
    if (i1 && i2) sm.A[q1][q2] = zadd(zmul(cs1, m01), zscale(m11, c1));
}
// Rows p, q of W <- J^H (rows p, q), column c.
MPSX_DEV void jacobi_rows(SmallShared &sm, int p, int q, int c, double cs, double2 s) {
    if (s.x == 0.0 && s.y == 0.0) return;
    const double2 xp = sm.Q[p][c], xq = sm.Q[q][c];
    sm.Q[p][c] = zadd(zscale(xp, cs), zmul(make_double2(-s.x, -s.y), xq));
    sm.Q[q][c] = zadd(zmul(zconj(s), xp), zscale(xq, cs));
}

// Two-sided Jacobi on H in A until nothing rotates, W accumulated in Q, for n <=
// 8 rows: one wave, no barriers (a wave's LDS accesses stay in order); lanes 0 .. 3 the rotations of a step, then one 2 x 2 block of
// H or one column of a pair of W's rows a lane.
MPSX_DEV void small_jacobi8(int n, SmallShared &sm, double null2, double tol) {
    const int tid = threadIdx.x, m = n + (n & 1), np = m / 2;
    if (tid < 64) {
        if (tid < n * n) sm.Q[tid / n][tid % n] = make_double2(tid / n == tid % n ? 1.0 : 0.0, 0.0);
        for (int e = tid; e < (m - 1) * np; e += 64) {
            int p, q;
            rr_pair(e % np, e / np, m, &p, &q);
            sm.row8[e / np][e % np] = p | (q << 8);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        // this lane's item: block (k1, k2) of H, or column c of pair k1 of W
        const bool blk = tid < np * np, qit = tid >= 16 && tid < 16 + np * n;
        const int k1 = blk ? tid / np : (qit ? (tid - 16) / n : 0), k2 = blk ? tid % np : 0;
        const int c = qit ? (tid - 16) % n : 0;
        for (int sw = 0; sw < 12; ++sw) {
            bool rotated = false;
            for (int step = 0; step < m - 1; ++step) {
                bool on = false;
                if (tid < np) {
                    const int pq = sm.row8[step][tid], p = pq & 255, q = pq >> 8;
                    double cs = 1.0;
                    double2 s = make_double2(0.0, 0.0);
                    if (q < n) {
                        const double a = sm.A[p][p].x, b = sm.A[q][q].x;
                        const double2 h = sm.A[p][q];
                        const double g2 = fma(h.x, h.x, h.y * h.y);
                        on = a > null2 && b > null2 && g2 > tol * tol * a * b && g2 > 0.0;
                        if (on) jacobi_angle(0.5 * (b - a), g2, h, &cs, &s);
                    }
                    sm.prm_c[tid] = cs;
                    sm.prm_s[tid] = s;
                }
                if (!__any(on)) continue;
                rotated = true;
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
                const int pq1 = sm.row8[step][k1], p1 = pq1 & 255, q1 = pq1 >> 8;
                const double c1 = sm.prm_c[k1];
                const double2 s1 = sm.prm_s[k1];
                if (blk)
                    jacobi_block(n, sm, p1, q1, sm.row8[step][k2] & 255, sm.row8[step][k2] >> 8, c1, s1, sm.prm_c[k2],
                                 sm.prm_s[k2]);
                else if (qit && q1 < n)
                    jacobi_rows(sm, p1, q1, c, c1, s1);
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
            if (!rotated) break;
        }
    }
    __syncthreads();
}

// Cyclic two-sided Jacobi on H in A, W accumulated in Q (identity at first):
// `sweeps` sweeps at most, ended by one that rotates nothing.
MPSX_DEV void small_jacobi(int n, SmallShared &sm, double null2, double tol, int sweeps) {
    const int tid = threadIdx.x, m = n + (n & 1), np = m / 2;
    for (int e = tid; e < n * n; e += ST) sm.Q[e / n][e % n] = make_double2(e / n == e % n ? 1.0 : 0.0, 0.0);
    __syncthreads();
    for (int sw = 0; sw < sweeps; ++sw) {
        int rotated = 0;
        for (int step = 0; step < m - 1; ++step) {
            int on = 0;
            if (tid < np) {
                int p, q;
                rr_pair(tid, step, m, &p, &q);
                double cs = 1.0;
                double2 s = make_double2(0.0, 0.0);
                if (q < n) {
                    const double a = sm.A[p][p].x, c = sm.A[q][q].x;
                    const double2 h = sm.A[p][q];
                    const double g2 = fma(h.x, h.x, h.y * h.y);
                    if (a > null2 && c > null2 && g2 > tol * tol * a * c && g2 > 0.0) {
                        jacobi_angle(0.5 * (c - a), g2, h, &cs, &s);
                        on = 1;
                    }
                }
                sm.prm_c[tid] = cs;
                sm.prm_s[tid] = s;
            }
            if (!__syncthreads_or(on)) continue;
            rotated = 1;
            // H <- J^H H J on the 2 x 2 blocks (k1, k2), W <- J^H W, with J =
            // [[c, s], [-conj(s), c]] for each pair
            for (int e = tid; e < np * np; e += ST) {
                const int k1 = e / np, k2 = e % np;
                int p1, q1, p2, q2;
                rr_pair(k1, step, m, &p1, &q1);
                rr_pair(k2, step, m, &p2, &q2);
                jacobi_block(n, sm, p1, q1, p2, q2, sm.prm_c[k1], sm.prm_s[k1], sm.prm_c[k2], sm.prm_s[k2]);
            }
            for (int e = tid; e < np * n; e += ST) {
                const int k = e / n, c = e % n;
                int p, q;
                rr_pair(k, step, m, &p, &q);
                if (q < n) jacobi_rows(sm, p, q, c, sm.prm_c[k], sm.prm_s[k]);
            }
            __syncthreads();
        }
        if (!rotated) break;
    }
}

// The block's m rows of Z <- W (those rows), 16 columns a wave; with `first`, Y
// is still the identity.
MPSX_DEV void small_apply(double2 *Z, int64_t LD, int rows, int n, int R, bool first, SmallShared &sm) {
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_id(), l16 = lane & 15, lq = lane >> 4;
    const int nt = (n + 15) / 16, to = first ? R : R + rows;
    for (int c0 = 16 * wave; c0 < to; c0 += 16 * SW) {
        const int c = c0 + l16;
        double2 x[SN / 4];
#pragma unroll
        for (int s = 0; s < SN / 4; ++s) {
            const int row = 4 * s + lq;
            x[s] = (row < n && c < to) ? Z[(int64_t)sm.row[row] * LD + c] : make_double2(0.0, 0.0);
        }
        for (int tm = 0; tm < nt; ++tm) {
            mfma_d4 a1 = {0.0, 0.0, 0.0, 0.0}, a2 = a1, a3 = a1;
            const int ar = 16 * tm + l16;
#pragma unroll
            for (int s = 0; s < SN / 4; ++s) {
                if (4 * s >= n) break;
                const double2 q = (ar < n && 4 * s + lq < n) ? sm.Q[ar][4 * s + lq] : make_double2(0.0, 0.0);
                a1 = mfma16d(q.x, x[s].x, a1);
                a2 = mfma16d(q.y, x[s].y, a2);
                a3 = mfma16d(q.x + q.y, x[s].x + x[s].y, a3);
            }
            if (c < to)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = 16 * tm + 4 * r + lq;
                    if (row < n) Z[(int64_t)sm.row[row] * LD + c] = make_double2(a1[r] - a2[r], a3[r] - a1[r] - a2[r]);
                }
        }
    }
    if (first)
        for (int e = tid; e < rows * rows; e += ST) {
            const int i = e / rows, c = e % rows, pi = sm.pos[i], pc = sm.pos[c];
            Z[(int64_t)i * LD + R + c] = pi >= 0 && pc >= 0 ? sm.Q[pi][pc] : make_double2(i == c ? 1.0 : 0.0, 0.0);
        }
    __syncthreads();
}

}  // namespace

// One workgroup per problem; theta (X) is in the workspace.
__global__ void __launch_bounds__(ST, 2)
k_small(const mpsx_two_site_op *ops, char *ws, double tol, double null_rel, int *unconverged, int *late) {
    __shared__ SmallShared sm;
    const mpsx_two_site_op &op = ops[blockIdx.x];
    const mpsx_plan p = op.plan;
    if (!small_route(p, 1)) return;
    const int n = p.C, R = p.R, tid = threadIdx.x, lane = tid & 63, wave = wave_id();
    const int64_t LD = p.LD;
    double2 *Z = reinterpret_cast<double2 *>(ws + z_off(p));
    double null2 = 0.0;
    bool first = true, done = false;
    for (int it = 0; it < kPasses && !done; ++it) {
        small_gram(Z, LD, n, R, sm);
        if (it == 0) {
            const double fro2 = wave_sum64(lane < n ? sm.A[lane][lane].x : 0.0);
            null2 = null_rel * null_rel * fro2;
        }
        if (tid < SN) sm.fail[tid] = 0;
        __syncthreads();
        int rot = 0;
        for (int e = tid; e < n * n; e += ST) {
            const int i = e / n, j = e % n;
            if (i >= j) continue;
            const double hi = sm.A[i][i].x, hj = sm.A[j][j].x;
            const double2 h = sm.A[i][j];
            const double g2 = fma(h.x, h.x, h.y * h.y);
            if (hi > null2 && hj > null2 && g2 > tol * tol * hi * hj) {
                rot = 1;
                sm.fail[i] = 1;
                sm.fail[j] = 1;
            }
        }
        if (!__syncthreads_or(rot)) {
            done = true;
            break;
        }
        const unsigned long long in = __ballot(sm.fail[lane] != 0);
        const int m = __popcll(in);
        if (tid < SN) {
            const int at = __popcll(in & ((1ULL << tid) - 1));
            const bool on = (in >> tid) & 1;
            sm.pos[tid] = on ? at : -1;
            if (on) sm.row[at] = tid;
        }
        __syncthreads();
        if (m < n) {  // the block of H to the front
            double2 b[SN * SN / ST];
#pragma unroll
            for (int t = 0; t < SN * SN / ST; ++t) {
                const int e = tid + ST * t;
                b[t] = e < m * m ? sm.A[sm.row[e / m]][sm.row[e % m]] : make_double2(0.0, 0.0);
            }
            __syncthreads();
#pragma unroll
            for (int t = 0; t < SN * SN / ST; ++t) {
                const int e = tid + ST * t;
                if (e < m * m) sm.A[e / m][e % m] = b[t];
            }
            __syncthreads();
        }
        if (m > 8 && it % 4 != 3) {
            small_tridiag(m, sm);
            if (tid < LEAF) {
                // T scaled to unit norm and torn
                const double dv = tid < m ? sm.d[tid] : 0.0, ev = tid + 1 < m ? sm.e[tid] : 0.0;
                double mx = fmax(fabs(dv), fabs(ev));
                for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o, 64));
                const double f = mx > 0.0 ? 1.0 / mx : 1.0;
                const double below = __shfl_up(ev, 1, 64);
                sm.L.e[tid] = ev * f;
                sm.L.d[tid] = dv * f - fabs(ev * f) - (tid > 0 ? fabs(below * f) : 0.0);
            }
            leaf_conquer(m, sm.S, sm.U, sm.L);
            small_back(m, sm);
        } else if (m <= 8) {
            small_jacobi8(m, sm, null2, 0.01 * tol);
        } else {
            small_jacobi(m, sm, null2, 0.01 * tol, 1);
        }
        small_apply(Z, LD, n, m, R, first, sm);
        first = false;
    }
    if (!done && tid == 0) {
        if (unconverged) atomicAdd(unconverged, 1);
        tell_host(late);
    }

    // norms, order, factors
    for (int row = wave; row < n; row += SW) {
        double s = 0.0;
#pragma unroll 4
        for (int c = lane; c < R; c += 64) {
            const double2 v = Z[(int64_t)row * LD + c];
            s = fma(v.x, v.x, fma(v.y, v.y, s));
        }
        s = wave_sum64(s);
        if (lane == 0) sm.sig[row] = s;
    }
    __syncthreads();
    const int k = op.k;
    if (wave == 0) {
        const double s = lane < n ? sm.sig[lane] : 0.0, key = sort_key(s);
        int rank = 0;
        for (int o = 0; o < n; ++o) {
            const double ko = sort_key(sm.sig[o]);
            rank += (ko > key) || (ko == key && o < lane);
        }
        if (lane < n) sm.perm[rank] = lane;
        const double disc = wave_sum64((lane < n && rank >= k) ? s : 0.0);
        if (lane == 0 && op.discarded) *op.discarded = disc;
        if (lane < n && rank < k && op.s_out) op.s_out[rank] = (float)sqrt(s);
    }
    __syncthreads();
    const bool left = (op.flags & 1) != 0;
    const int M = op.d * op.chi_l, N = op.d * op.chi_r;
    // absorb right: a_out[m][j] = conj(Y[perm j][m]), b_out[j][c] = X[perm j][c];
    // absorb left: a_out[m][j] = X[perm j][m], b_out[j][c] = conj(Y[perm j][c]).
    // The unscaled factor of a problem that never rotated is the identity's rows.
    auto y_at = [&](int row, int c) {
        return first ? make_double2(row == c ? 1.0 : 0.0, 0.0) : Z[(int64_t)row * LD + R + c];
    };
    float2 *a_out = reinterpret_cast<float2 *>(op.a_out), *b_out = reinterpret_cast<float2 *>(op.b_out);
#pragma unroll 4
    for (int e = tid; e < M * k; e += ST) {
        const int m = e / k, row = sm.perm[e % k];
        const double2 v = left ? Z[(int64_t)row * LD + m] : zconj(y_at(row, m));
        a_out[e] = make_float2((float)v.x, (float)v.y);
    }
#pragma unroll 4
    for (int e = tid; e < k * N; e += ST) {
        const int c = e % N, row = sm.perm[e / N];
        const double2 v = left ? zconj(y_at(row, c)) : Z[(int64_t)row * LD + c];
        b_out[e] = make_float2((float)v.x, (float)v.y);
    }
}

hipError_t launch_small(hipStream_t s, const mpsx_two_site_op *d, int count, char *ws, double tol, double null_rel,
                        int *unconverged, int *late) {
    hipLaunchKernelGGL(k_small, dim3((unsigned)count), dim3(ST), 0, s, d, ws, tol, null_rel, unconverged, late);
    return hipGetLastError();
}
