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
// poles stay (dl, zl, src[0 .. K-1]); of dd and src the `none` entries of
// negligible weight (as many as the same test counts) fill the end, in order, so
// that rows which nothing couples keep theirs, and the rotated ones the places before
// them. rot_i, rot_c: the rotations (row a, row b, c, s) in order. Serial.
MPSX_DEV int deflate(int m, int none, double rho, const double *ds, const double *zs, const int *id, double *dl,
                     double *zl, int *src, double *dd, int2 *rot_i, double2 *rot_c, int *nrot) {
    int K = 0, f = m - none, e = f, nr = 0, pj = -1;
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
        if (!(rho * fabs(zr) > kDeflate)) {
            src[f] = i;
            dd[f] = dr;
            ++f;
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

// A lane's value as a wave-uniform one.
MPSX_DEV double lane_f64(double x, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), lane),
                            __builtin_amdgcn_readlane(__double2loint(x), lane));
}

// Root j of 1 + rho sum_i z_i^2 / (d_i - lambda), 0 <= j < K, by L lanes (sub
// = lane in the group): lambda = d_org + root with org the nearer of the two
// poles around it, so that every difference d_i - lambda is accurate. A lane
// has the poles sub, sub + L, ... and their squared weights in registers (far
// away and zero beyond K) and works on four at a time: one by one from LDS, the
// chain of a reciprocal took 440 cycles a pole. d is shifted by the origin.
// dj, dn, zj, zn: pole j and j + 1 and their weights. Returns org - j.
template <int L, int U>
MPSX_DEV int secular_root(int K, double (&d)[U], const double (&z2)[U], double dj, double dn, double zj, double zn,
                          double rho, int j, int sub, double *root) {
    static_assert(U % 4 == 0 && (L == 8 || L == 64), "poles a lane");
    const bool last = j == K - 1;
    int org = 0;
    double lo, hi, t;
    auto sum = [](double x) { return L == 64 ? wave_sum64(x) : group_sum<8>(x); };
    if (last) {
        double s = 0.0;
#pragma unroll
        for (int u = 0; u < U; ++u) s += z2[u];
        s = sum(s);
        lo = 0.0;
        hi = rho * s * (1.0 + 4.0 * kEps);
        t = K == 1 ? rho * s : 0.5 * hi;
    } else {
        const double gap = dn - dj, mid = 0.5 * gap;
        double c0 = 0.0;
#pragma unroll
        for (int u0 = 0; u0 < U; u0 += 4) {
            if (L * u0 >= K) break;
#pragma unroll
            for (int u = u0; u < u0 + 4; ++u) {
                const int i = sub + L * u;
                const double q = z2[u] * recip((d[u] - dj) - mid);
                c0 += (i == j || i == j + 1) ? 0.0 : q;
            }
        }
        c0 = sum(c0);
        const double s = rho * zj * zj, v = rho * zn * zn, c = fma(rho, c0, 1.0);
        const bool left = c + (v - s) / mid >= 0.0;
        org = left ? 0 : 1;
        lo = left ? 0.0 : -mid;
        hi = left ? mid : 0.0;
        // c + s / (p1 - t) + v / (p2 - t) = 0 with the poles at 0 and +-gap
        const double A = left ? fma(c, gap, s + v) : fma(-c, gap, s + v);
        const double B = left ? s * gap : -v * gap;
        const double sq = sqrt(fmax(fma(A, A, -4.0 * c * B), 0.0));
        t = A > 0.0 ? 2.0 * B * recip(A + sq) : (A - sq) * recip(2.0 * c);
    }
    if (K > 1) {
        if (!(t > lo && t < hi)) t = 0.5 * (lo + hi);
        const double dorg = org ? dn : dj, p1 = dj - dorg, p2 = last ? 0.0 : dn - dorg;
#pragma unroll
        for (int u = 0; u < U; ++u) d[u] -= dorg;
        for (int it = 0; it < 64; ++it) {
            double psi = 0.0, dpsi = 0.0, phi = 0.0, dphi = 0.0;
#pragma unroll
            for (int u0 = 0; u0 < U; u0 += 4) {
                if (L * u0 >= K) break;
#pragma unroll
                for (int u = u0; u < u0 + 4; ++u) {
                    const double zl = sub + L * u <= j ? z2[u] : 0.0, zr = z2[u] - zl;
                    const double r = recip(d[u] - t), ql = zl * r, qr = zr * r;
                    psi += ql;
                    phi += qr;
                    dpsi = fma(ql, r, dpsi);
                    dphi = fma(qr, r, dphi);
                }
            }
            if (L == 64) {
                const double f = group_sum<16>(fold16(fold32(psi, phi), fold32(dpsi, dphi)));
                psi = rho * lane_f64(f, 0);
                dpsi = rho * lane_f64(f, 16);
                phi = rho * lane_f64(f, 32);
                dphi = rho * lane_f64(f, 48);
            } else {
                psi = rho * group_sum<8>(psi);
                phi = rho * group_sum<8>(phi);
                dpsi = rho * group_sum<8>(dpsi);
                dphi = rho * group_sum<8>(dphi);
            }
            const double g = 1.0 + psi + phi;
            if (fabs(g) <= kEps * (8.0 * (1.0 + fabs(psi) + fabs(phi)) + fabs(t) * (dpsi + dphi))) break;
            if (g < 0.0)
                lo = t;
            else
                hi = t;
            double tn;
            if (last) {
                // c - s / t = 0 through the pole at the origin
                tn = dpsi * t * t * recip(fma(dpsi, t, g));
            } else {
                const double D1 = p1 - t, D2 = p2 - t;
                const double s = dpsi * D1 * D1, v = dphi * D2 * D2, c = g - dpsi * D1 - dphi * D2;
                const double A = fma(c, D1 + D2, s + v), B = D1 * D2 * g;
                const double sq = sqrt(fmax(fma(A, A, -4.0 * c * B), 0.0));
                const double q = 0.5 * (A + copysign(sq, A));
                double eta = B * recip(q);  // of the two roots, the one between the poles
                if (!(eta > D1 && eta < D2)) eta = q * recip(c);
                tn = t + eta;
            }
            if (!(tn > lo && tn < hi)) tn = 0.5 * (lo + hi);
            if (tn == t || hi - lo <= 2.0 * kEps * fmax(fabs(lo), fabs(hi))) break;
            t = tn;
        }
    }
    *root = t;
    return org;
}

// |z_i| for which the computed roots are the exact ones (Gu & Eisenstat): the
// factors sub, sub + L, ... of its square. pb, rt: pole and offset of a root.
template <int L>
MPSX_DEV double zhat_factors(int K, const double *dl, const double *pb, const double *rt, int i, int sub) {
    const double di = dl[i];
    double pr = 1.0;
#pragma unroll 4
    for (int j = sub; j < K; j += L) {
        const double num = (pb[j] - di) + rt[j];
        const double den = j < i ? dl[j] - di : (j < K - 1 ? dl[j + 1] - di : 1.0);
        pr *= num * recip(den);
    }
    return pr;
}

// The eigensystem of a tridiagonal block of m <= 64 rows, torn at every entry.
constexpr int LEAF = 64, LEAF_THREADS = 512;
struct LeafShared {
    double d[LEAF], e[LEAF];  // in: the torn diagonal and the off-diagonal, scaled; out: the eigenvalues in d
    double ds[LEAF], zs[LEAF], dl[LEAF], zl[LEAF], dd[LEAF], zh[LEAF], rt[LEAF], pb[LEAF];
    int id[LEAF], src[LEAF], kn[LEAF], nrot[LEAF];
    int2 rot_i[LEAF];
    double2 rot_c[LEAF];
};
// Merges of 1, 2, 4, ... rows in LDS by a workgroup of LEAF_THREADS, eight
// lanes a row; on return row j of S is eigenvector j. L.d and L.e are written by
// the first LEAF threads before the call.
// Bound: latency, about 8 us a level (18 with the poles one by one and the
// rows on the vector units); the deflation in one wave rather than one lane takes 30 us
// off a block with negligible weights.
MPSX_DEV void leaf_conquer(int m, double (*S)[LEAF + 1], double (*U)[LEAF + 1], LeafShared &L) {
    constexpr int M = LEAF;
    const int tid = threadIdx.x, g = tid >> 3, sub = tid & 7;
    for (int e = tid; e < M * M; e += LEAF_THREADS) S[e >> 6][e & 63] = (e >> 6) == (e & 63) ? 1.0 : 0.0;
    __syncthreads();
    for (int s = 1; s < m; s <<= 1) {
        const int h = 2 * s;
        // index g, its merge [lo, hi)
        const int lo = g & ~(h - 1), mid = lo + s, hi = min(lo + h, m), gj = g - lo;
        const double ee = mid < hi ? L.e[mid - 1] : 0.0, rho = 2.0 * fabs(ee);
        if (g < m) {
            const double dg = L.d[g], key = sort_key(dg);
            int rank = 0;
            for (int o = lo + sub; o < hi; o += 8) {
                const double ko = sort_key(L.d[o]);
                rank += (ko < key) || (ko == key && o < g);
            }
            rank += __builtin_amdgcn_mov_dpp(rank, 0xB1, 0xf, 0xf, true);
            rank += __builtin_amdgcn_mov_dpp(rank, 0x4E, 0xf, 0xf, true);
            rank += __builtin_amdgcn_mov_dpp(rank, 0x141, 0xf, 0xf, true);
            if (sub == 0) {
                L.ds[lo + rank] = dg;
                L.zs[lo + rank] = mid < hi ? S[g][g < mid ? mid - 1 : mid] *
                                                 (g >= mid && ee < 0.0 ? -0.7071067811865476 : 0.7071067811865476)
                                           : 0.0;
                L.id[lo + rank] = g;
            }
        }
        __syncthreads();
        // The first wave, a lane a sorted entry: those of negligible weight go to the end
        // of their merge, in order; if two of the others have to be rotated together
        // (kn < 0: -1 - the number of others), deflate() starts over.
        if (tid < M) {
            const int r = tid, rl = r & ~(h - 1), rm = rl + s, rh = min(rl + h, m);
            const bool on = r < m;
            const double rr = rm < rh ? 2.0 * fabs(L.e[rm - 1]) : 0.0;
            const double z = on ? L.zs[r] : 0.0, d = on ? L.ds[r] : 0.0;
            const bool keep = on && rr * fabs(z) > kDeflate;
            const unsigned long long mine = __ballot(keep) & ((h == 64 ? ~0ULL : (1ULL << h) - 1) << rl);
            const int before = __popcll(mine & ((1ULL << r) - 1));
            const unsigned long long after = r < 63 ? mine >> (r + 1) : 0ULL;
            const int nx = after ? r + __ffsll((long long)after) : r;
            const double zn = __shfl(z, nx, 64), dn = __shfl(d, nx, 64);
            const bool pair = keep && after && fabs((dn - d) * z * zn) <= kDeflate * fma(z, z, zn * zn);
            const unsigned long long pairs = __ballot(pair) & ((h == 64 ? ~0ULL : (1ULL << h) - 1) << rl);
            if (keep) {
                L.dl[rl + before] = d;
                L.zl[rl + before] = z;
                L.src[rl + before] = L.id[r];
            } else if (on) {
                const int e = rl + __popcll(mine) + (r - rl - before);
                L.dd[e] = d;
                L.src[e] = L.id[r];
            } else {
                L.src[r] = r;
            }
            if (on && r == rl) {
                L.kn[r] = pairs ? -1 - __popcll(mine) : __popcll(mine);
                L.nrot[r] = 0;
            }
        }
        __syncthreads();
        if (sub == 0 && g < m && gj == 0 && L.kn[lo] < 0)
            L.kn[lo] = deflate(hi - lo, hi - lo + L.kn[lo] + 1, rho, L.ds + lo, L.zs + lo, L.id + lo, L.dl + lo,
                               L.zl + lo, L.src + lo, L.dd + lo, L.rot_i + lo, L.rot_c + lo, &L.nrot[lo]);
        __syncthreads();
        if (tid < m) {  // component tid of its merge's rows
            const int tlo = tid & ~(h - 1);
            for (int r = 0; r < L.nrot[tlo]; ++r) {
                const int2 ab = L.rot_i[tlo + r];
                const double2 cs = L.rot_c[tlo + r];
                const double xa = S[ab.x][tid], xb = S[ab.y][tid];
                S[ab.x][tid] = cs.x * xa + cs.y * xb;
                S[ab.y][tid] = cs.x * xb - cs.y * xa;
            }
        }
        const int K = g < m ? L.kn[lo] : 0;
        double db = 0.0, tj = 0.0;
        if (gj < K) {
            double d[8], z2[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int i = sub + 8 * u;
                d[u] = i < K ? L.dl[lo + i] : 1e200;
                const double z = i < K ? L.zl[lo + i] : 0.0;
                z2[u] = z * z;
            }
            const int nx = min(gj + 1, K - 1);
            const double dj = L.dl[g], dn = L.dl[lo + nx];
            db = secular_root<8, 8>(K, d, z2, dj, dn, L.zl[g], L.zl[lo + nx], rho, gj, sub, &tj) ? dn : dj;
            if (sub == 0) {
                L.pb[g] = db;
                L.rt[g] = tj;
            }
        }
        __syncthreads();
        if (gj < K) {
            const double v = group_prod<8>(zhat_factors<8>(K, L.dl + lo, L.pb + lo, L.rt + lo, gj, sub));
            if (sub == 0) L.zh[g] = copysign(sqrt(fmax(v, 0.0)), L.zl[g]);
        }
        __syncthreads();
        // Row g of the blocks of max(h, 16) columns that multiply the old rows:
        // u over the merge's poles, a unit vector for a deflated row, zero elsewhere.
        const int hb = max(h, 16), off = lo & (hb - 1);
        {
            double u[8], nn = 0.0;
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const int i = sub + 8 * t - off;
                u[t] = 0.0;
                if (8 * t < hb && gj < K) {
                    if (i >= 0 && i < K) u[t] = L.zh[lo + i] * recip((L.dl[lo + i] - db) - tj);
                    nn = fma(u[t], u[t], nn);
                }
            }
            nn = group_sum<8>(nn);
            const double f = gj < K ? 1.0 / sqrt(nn) : 0.0;
#pragma unroll
            for (int t = 0; t < 8; ++t)
                if (8 * t < hb) U[g][sub + 8 * t] = gj < K ? u[t] * f : (sub + 8 * t - off == gj ? 1.0 : 0.0);
        }
        const double dn = g < m ? (gj < K ? db + tj : L.dd[g]) : 0.0;
        __syncthreads();
        // New rows = U (old rows in the order of src) on the matrix cores, block by
        // block: hb / 16 squared tiles a block, hb / 4 in all, two at most a wave.
        const int lane = tid & 63, wave = wave_id(), l16 = lane & 15, q = lane >> 4;
        const int tb = hb / 16, per = tb * tb;
        mfma_d4 acc[2];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const int t = wave + 8 * w;
            acc[w] = mfma_d4{0.0, 0.0, 0.0, 0.0};
            if (t >= hb / 4) continue;
            const int b0 = (t / per) * hb, ti = (t % per) / tb, tj2 = (t % per) % tb;
            for (int k = 0; k < hb; k += 16)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    acc[w] = mfma16d(U[b0 + 16 * ti + l16][k + 4 * v + q],
                                     S[L.src[b0 + k + 4 * v + q]][b0 + 16 * tj2 + l16], acc[w]);
        }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const int t = wave + 8 * w;
            if (t >= hb / 4) continue;
            const int b0 = (t / per) * hb, ti = (t % per) / tb, tj2 = (t % per) % tb;
#pragma unroll
            for (int r = 0; r < 4; ++r) S[b0 + 16 * ti + 4 * r + q][b0 + 16 * tj2 + l16] = acc[w][r];
        }
        if (sub == 0 && g < m) L.d[g] = dn;
        __syncthreads();
    }
}

}  // namespace
