// Device pieces of the real symmetric tridiagonal eigensolver, shared by the
// direct solver of the Gram method (eig.hip) and the one-workgroup kernel of
// small problems (small.hip).
//
// Divide and conquer (Cuppen 1981): T is torn at an entry e into two halves and
// a rank-one update |e| u u^T; the halves' eigensystems turn it into diag(d) +
// rho z z^T. Deflation of Dongarra & Sorensen (1987); the secular roots by
// rational interpolation at the two neighbouring poles (Bunch, Nielsen &
// Sorensen 1978) inside a bracket; the eigenvectors of the update from the
// weights recomputed from the roots (Gu & Eisenstat 1994), which keeps S
// orthogonal to FP64 rounding without extended precision.
#pragma once

#include "common.h"

namespace {

constexpr double kEps = 2.220446049250313e-16;
// Deflation threshold for T scaled to unit norm.
constexpr double kDeflate = 8.0 * kEps;
// Squares below this are not worth a reflector: H is made of FP32 data, so its
// trace is zero or above 1e-90, and sqrt(kTiny) is zero beside that. (An
// underflow to zero would be divided by.)
constexpr double kTiny = 1e-290;

// Wave of the workgroup, as a scalar: what depends on it alone (rows, branches,
// addresses) then stays out of the vector registers.
MPSX_DEV int wave_id() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }
template <int CTRL>
MPSX_DEV double dpp_f64(double x) {
    // permutes within a row of 16: every lane has a source, nothing to keep
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(x), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(x), CTRL, 0xf, 0xf, true);
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
// The same inside rows of 16 (lanes 0-7 a, 8-15 b) and of 8 (lanes 0-3 a, 4-7 b).
MPSX_DEV double fold8(double a, double b) {
    const bool hi = (threadIdx.x & 8) != 0;
    return (hi ? b : a) + dpp_f64<0x128>(hi ? a : b);  // row_ror 8
}
MPSX_DEV double fold4(double a, double b) {
    const bool hi = (threadIdx.x & 4) != 0;
    return (hi ? b : a) + dpp_f64<0x141>(hi ? a : b);  // half-row mirror
}
// Wave sums of several complex values at once. Folding two values into one
// register halves the work of every level that follows, so that eight sums
// take about as many instructions as two would one by one.
//   wave_sum4: lane 16 q + 8 h (and the seven after it) holds the sum of x[q],
//   real (h = 0) or imaginary (h = 1) part;
//   wave_sum8: lane 16 q + 8 u + 4 h (and the three after it) that of x[q + 4 u].
MPSX_DEV double wave_sum4(const double2 (&x)[4]) {
    const double re = fold16(fold32(x[0].x, x[2].x), fold32(x[1].x, x[3].x));
    const double im = fold16(fold32(x[0].y, x[2].y), fold32(x[1].y, x[3].y));
    return group_sum<8>(fold8(re, im));
}
MPSX_DEV double wave_sum8(const double2 (&x)[8]) {
    double re[2], im[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const double2 *y = x + 4 * u;
        re[u] = fold16(fold32(y[0].x, y[2].x), fold32(y[1].x, y[3].x));
        im[u] = fold16(fold32(y[0].y, y[2].y), fold32(y[1].y, y[3].y));
    }
    return group_sum<4>(fold4(fold8(re[0], re[1]), fold8(im[0], im[1])));
}
MPSX_DEV double wave_sum64(double x) {
    x = fold32(x, x);
    return group_sum<16>(fold16(x, x));
}
MPSX_DEV double uniform_f64(double x) {
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(x)),
                            __builtin_amdgcn_readfirstlane(__double2loint(x)));
}
MPSX_DEV double2 uniform_z(double2 v) { return make_double2(uniform_f64(v.x), uniform_f64(v.y)); }


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

// Whether deflate() would drop entry r of the m sorted ones, or merge it with
// the next: if none, the update has all m poles as they stand.
MPSX_DEV bool may_deflate(int m, int r, double rho, const double *ds, const double *zs) {
    const double z = zs[r];
    if (rho * fabs(z) <= kDeflate) return true;
    if (r + 1 >= m) return false;
    const double zn = zs[r + 1];
    return fabs((ds[r + 1] - ds[r]) * z * zn) <= kDeflate * fma(z, z, zn * zn);
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

// The eigensystem of a tridiagonal block of m <= 64 rows, torn at every entry.
constexpr int LEAF = 64;
struct LeafShared {
    double d[LEAF], e[LEAF];  // in: the torn diagonal and the off-diagonal, scaled; out: the eigenvalues in d
    double z[LEAF], ds[LEAF], zs[LEAF], dl[LEAF], zl[LEAF], dd[LEAF], zh[LEAF], rt[LEAF];
    int id[LEAF], src[LEAF], base[LEAF], kn[LEAF], nrot[LEAF];
    int2 rot_i[LEAF];
    double2 rot_c[LEAF];
};
// Merges of 1, 2, 4, ... rows in LDS by a workgroup of NT threads (a multiple
// of 256); on return row j of S is eigenvector j. L.d and L.e are written by
// the first LEAF threads before the call.
template <int NT>
MPSX_DEV void leaf_conquer(int m, double (*S)[LEAF + 1], double (*U)[LEAF + 1], LeafShared &L) {
    constexpr int M = LEAF;
    const int tid = threadIdx.x;
    for (int e = tid; e < M * M; e += NT) S[e >> 6][e & 63] = (e >> 6) == (e & 63) ? 1.0 : 0.0;
    __syncthreads();
    for (int s = 1; s < m; s <<= 1) {
        const int h = 2 * s;
        // the first threads serve one index each: index tid, its merge [lo, hi)
        const int lo = tid & ~(h - 1), mid = lo + s, hi = min(lo + h, m);
        const bool merge = tid < m && mid < hi;
        const double ee = merge ? L.e[mid - 1] : 0.0;
        if (tid < m)
            L.z[tid] = merge ? S[tid][tid < mid ? mid - 1 : mid] *
                                   (tid >= mid && ee < 0.0 ? -0.7071067811865476 : 0.7071067811865476)
                             : 0.0;
        __syncthreads();
        if (tid < m) {
            const double key = sort_key(L.d[tid]);
            int rank = 0;
            for (int o = lo; o < hi; ++o) {
                const double ko = sort_key(L.d[o]);
                rank += (ko < key) || (ko == key && o < tid);
            }
            L.ds[lo + rank] = L.d[tid];
            L.zs[lo + rank] = L.z[tid];
            L.id[lo + rank] = tid;
        }
        if (tid < m && tid == lo) L.kn[lo] = hi - lo;  // until something deflates
        __syncthreads();
        if (tid < m) {
            if (may_deflate(hi - lo, tid - lo, 2.0 * fabs(ee), L.ds + lo, L.zs + lo)) L.kn[lo] = -1;
            L.dl[tid] = L.ds[tid];
            L.zl[tid] = L.zs[tid];
            L.src[tid] = L.id[tid];
            if (tid == lo) L.nrot[lo] = 0;
        }
        __syncthreads();
        if (tid < m && tid == lo && L.kn[lo] < 0)
            L.kn[lo] = deflate(hi - lo, 2.0 * fabs(ee), L.ds + lo, L.zs + lo, L.id + lo, L.dl + lo, L.zl + lo,
                               L.src + lo, L.dd + lo, L.rot_i + lo, L.rot_c + lo, &L.nrot[lo]);
        __syncthreads();
        if (tid < m) {  // component tid of the merge's rows
            for (int r = 0; r < L.nrot[lo]; ++r) {
                const int2 ab = L.rot_i[lo + r];
                const double2 cs = L.rot_c[lo + r];
                const double xa = S[ab.x][tid], xb = S[ab.y][tid];
                S[ab.x][tid] = cs.x * xa + cs.y * xb;
                S[ab.y][tid] = cs.x * xb - cs.y * xa;
            }
        }
        // four lanes per root
        const int g = tid >> 2, sub = tid & 3;
        const int glo = g & ~(h - 1), gmid = glo + s, gj = g - glo;
        const int K = g < m ? L.kn[glo] : 0;
        if (gj < K) {
            int bs;
            double root;
            secular_root<4>(K, L.dl + glo, L.zl + glo, 2.0 * fabs(L.e[gmid - 1]), gj, sub, &bs, &root);
            if (sub == 0) {
                L.base[g] = bs;
                L.rt[g] = root;
            }
        }
        __syncthreads();
        if (gj < K) {
            const double v = zhat<4>(K, L.dl + glo, L.base + glo, L.rt + glo, gj, sub);
            if (sub == 0) L.zh[g] = copysign(v, L.zl[g]);
        }
        __syncthreads();
        if (gj < K) {
            const double db = L.dl[glo + L.base[g]], tj = L.rt[g];
            double nn = 0.0;
            for (int i = sub; i < K; i += 4) {
                const double u = L.zh[glo + i] * recip((L.dl[glo + i] - db) - tj);
                U[g][i] = u;
                nn = fma(u, u, nn);
            }
            nn = group_sum<4>(nn);
            const double f = 1.0 / sqrt(nn);
            for (int i = sub; i < K; i += 4) U[g][i] *= f;
        }
        __syncthreads();
        // The new rows, held in registers until every old row has been read:
        // thread (wave, lane r) the rows wave, wave + NT / 64, ... of column
        // r's merge (the columns outside a merge stay zero), so that a pole
        // costs one read of S and a broadcast of u for each row.
        constexpr int W = NT / 64;
        const int r = tid & 63, wv = wave_id(), rlo = r & ~(h - 1);
        const int Kr = r < m ? L.kn[rlo] : 0, nr = r < m ? min(h, m - rlo) : 0;
        double v[M / W];
#pragma unroll
        for (int t = 0; t < M / W; ++t) v[t] = 0.0;
#pragma unroll 4
        for (int i = 0; i < Kr; ++i) {
            const double x = S[L.src[rlo + i]][r];
#pragma unroll
            for (int t = 0; t < M / W; ++t) {
                if (W * t >= h) break;
                v[t] = fma(U[(rlo + wv + W * t) & (M - 1)][i], x, v[t]);
            }
        }
#pragma unroll
        for (int t = 0; t < M / W; ++t) {
            const int jj = wv + W * t;
            if (jj >= Kr && jj < nr) v[t] = S[L.src[rlo + jj]][r];  // deflated: copied
        }
        const double dn = tid < m ? ((tid - lo) < L.kn[lo] ? L.dl[lo + L.base[tid]] + L.rt[tid] : L.dd[tid]) : 0.0;
        __syncthreads();
#pragma unroll
        for (int t = 0; t < M / W; ++t) {
            const int jj = wv + W * t;
            if (jj < nr) S[rlo + jj][r] = v[t];
        }
        if (tid < m) L.d[tid] = dn;
        __syncthreads();
    }
}

}  // namespace
