// Grouped complex64 GEMM for the read-out contractions.
//
// C = alpha * op(A) op(B) (+ C), op = identity or conjugate-transpose.
// Used for the left-to-right chain of MPS.wavefunction (core.py:483-500) and
// the two contractions per site of the transfer sweep in
// MPS.inner_product (core.py:553-559).
#include <hip/hip_runtime.h>

#include "common.h"
#include "launch.h"

// FP32 matrix cores (FP32 products and sums), four real products a complex
// one. No LDS staging: a wave loads its fragments from global memory (L1 and
// L2 hold what its neighbours share) GemmShape::PD blocks of 16 k ahead, and waits
// for no other wave. The order of k within a product is free, so lane l of a
// 16 x 16 tile takes k = 4 (l / 16) .. + 3 of a block in its four matrix
// instructions: where k is the contiguous index a lane reads 32 bytes and a
// row's four lanes one 128-byte line; where it is not, 16 lanes read one.
//   T    16 x 16 tiles a wave holds along each side
//   W    waves along each side of the workgroup's tile
//   KS   waves that share a tile's k, blocks dealt out in turn; their sums
//        meet in LDS
//   PD   blocks loaded ahead
//   OCC  waves a SIMD the registers are for
// Bound: small products by the latency of one pass over k, large ones by the
// matrix cores (157 TFLOP/s) and L1. Staged through LDS in 32 x 32 tiles on
// the vector units it was (us, before -> now): 256 x 512 x 256 30.7 -> 6.8,
// 256 x 256 x 256 31.2 -> 4.5, 4096 x 512 x 256 98 -> 50, 12 of
// 1024 x 1024 x 512 900 -> 480 (107 TFLOP/s), 1 x 1 x 65536 8000 -> 370; the error
// against FP64 fell by a third (the real products are summed apart).
template <int T_, int W_, int KS_, int PD_, int OCC_>
struct GemmShape {
    static constexpr int T = T_, W = W_, KS = KS_, PD = PD_, OCC = OCC_;
    static constexpr int TILE = 16 * T_ * W_, THREADS = 64 * W_ * W_ * KS_;
};

// Four k of one row (or column) of an operand: contiguous and 16-byte aligned
// (VEC), or anywhere (ks: stride of k).
template <bool VEC>
MPSX_DEV void gemm_load(const float2 *p, int64_t ks, float2 (&out)[4]) {
    if constexpr (VEC) {
        const float4 u = gload4(p), v = gload4(p + 2);
        out[0] = make_float2(u.x, u.y);
        out[1] = make_float2(u.z, u.w);
        out[2] = make_float2(v.x, v.y);
        out[3] = make_float2(v.z, v.w);
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) out[j] = gload2(p + j * ks);
    }
}

template <class S, bool VA, bool VB>
MPSX_DEV void gemm_tile(const mpsx_gemm_op &op, int64_t m0, int64_t n0, float2 (*red)[16][17]) {
    constexpr int T = S::T, W = S::W, KS = S::KS, PD = S::PD;
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int share = wave % KS, wm = wave / KS / W, wn = wave / KS % W;
    const bool ta = (op.flags & 1) != 0, tb = (op.flags & 2) != 0, accum = (op.flags & 4) != 0;
    const int64_t K = op.k, aks = ta ? op.lda : 1, bks = tb ? 1 : op.ldb;
    m0 += 16 * T * wm;
    n0 += 16 * T * wn;
    // rows and columns beyond the matrix repeat its last one (never stored)
    const float2 *pa[T], *pb[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const int64_t i = min(m0 + 16 * t + l16, op.m - 1), j = min(n0 + 16 * t + l16, op.n - 1);
        pa[t] = reinterpret_cast<const float2 *>(op.A) + (ta ? i : i * op.lda);
        pb[t] = reinterpret_cast<const float2 *>(op.B) + (tb ? j * op.ldb : j);
    }
    // the four real products apart: shorter sums, and conjugation is a sign at the end
    mfma_f4 rr[T][T], ii[T][T], ri[T][T], ir[T][T];
#pragma unroll
    for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j) rr[i][j] = ii[i][j] = ri[i][j] = ir[i][j] = mfma_f4{0.f, 0.f, 0.f, 0.f};
    float2 a[PD][T][4], b[PD][T][4];
    auto load = [&](int64_t blk, float2 (&x)[T][4], float2 (&y)[T][4]) {
        const int64_t k0 = 16 * blk + 4 * q;
#pragma unroll
        for (int t = 0; t < T; ++t) {
            gemm_load<VA>(pa[t] + k0 * aks, aks, x[t]);
            gemm_load<VB>(pb[t] + k0 * bks, bks, y[t]);
        }
    };
    auto multiply = [&](const float2 (&a)[T][4], const float2 (&b)[T][4]) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int x = 0; x < T; ++x)
#pragma unroll
                for (int y = 0; y < T; ++y) {
                    rr[x][y] = mfma16(a[x][j].x, b[y][j].x, rr[x][y]);
                    ii[x][y] = mfma16(a[x][j].y, b[y][j].y, ii[x][y]);
                    ri[x][y] = mfma16(a[x][j].x, b[y][j].y, ri[x][y]);
                    ir[x][y] = mfma16(a[x][j].y, b[y][j].x, ir[x][y]);
                }
    };
    // whole blocks; a load past this wave's last one repeats that
    const int64_t blocks = K / 16;
    const int64_t mine = blocks > share ? (blocks - share + KS - 1) / KS : 0;
    if (mine > 0) {
#pragma unroll
        for (int u = 0; u < PD; ++u) load(share + min((int64_t)u, mine - 1) * KS, a[u], b[u]);
        int64_t s = 0;
        for (; s + PD <= mine; s += PD) {
#pragma unroll
            for (int u = 0; u < PD; ++u) {
                multiply(a[u], b[u]);
                load(share + min(s + u + PD, mine - 1) * KS, a[u], b[u]);
            }
        }
#pragma unroll
        for (int u = 0; u < PD - 1; ++u)
            if (s + u < mine) multiply(a[u], b[u]);
    }
    // the rest of k, by the wave whose turn it is
    if (K % 16 != 0 && share == blocks % KS) {
        const int64_t k0 = 16 * blocks + 4 * q;
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool in = k0 + j < K;
                a[0][t][j] = in ? gload2(pa[t] + (k0 + j) * aks) : make_float2(0.f, 0.f);
                b[0][t][j] = in ? gload2(pb[t] + (k0 + j) * bks) : make_float2(0.f, 0.f);
            }
        multiply(a[0], b[0]);
    }
    const float si = ta == tb ? -1.f : 1.f, sri = tb ? -1.f : 1.f, sir = ta ? -1.f : 1.f;
    auto entry = [&](int x, int y, int r) {
        return make_float2(fmaf(si, ii[x][y][r], rr[x][y][r]), fmaf(sri, ri[x][y][r], sir * ir[x][y][r]));
    };
    const float2 alpha = make_float2(op.alpha_re, op.alpha_im);
    float2 *C = reinterpret_cast<float2 *>(op.C);
    auto store = [&](int64_t i, int64_t j, float2 v) {
        if (i >= op.m || j >= op.n) return;
        v = cmul(alpha, v);
        float2 *dst = C + i * op.ldc + j;
        if (accum) {
            const float2 old = gload2(dst);
            v.x += old.x;
            v.y += old.y;
        }
        gstore2(dst, v);
    };
    if constexpr (KS == 1) {
#pragma unroll
        for (int x = 0; x < T; ++x)
#pragma unroll
            for (int y = 0; y < T; ++y)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    store(m0 + 16 * x + 4 * q + r, n0 + 16 * y + l16, entry(x, y, r));
    } else {
        static_assert(T == 1 && W == 1, "waves share the k of one tile");
#pragma unroll
        for (int r = 0; r < 4; ++r) red[share][4 * q + r][l16] = entry(0, 0, r);
        __syncthreads();
        if (tid < 256) {
            float2 v = red[0][tid >> 4][tid & 15];
#pragma unroll
            for (int u = 1; u < KS; ++u) {
                v.x += red[u][tid >> 4][tid & 15].x;
                v.y += red[u][tid >> 4][tid & 15].y;
            }
            store(m0 + (tid >> 4), n0 + (tid & 15), v);
        }
    }
}

// Grid: x = (m tile, n tile) folded as m_tile * gn + n_tile (so m may need
// more than 65535 tiles, as the last steps of a wavefunction do), y = op.
template <class S>
__global__ void __launch_bounds__(S::THREADS, S::OCC) k_gemm(const mpsx_gemm_op *ops, int64_t gn) {
    __shared__ float2 red[S::KS > 1 ? S::KS : 1][16][17];
    const mpsx_gemm_op op = ops[blockIdx.y];
    const int64_t tile = blockIdx.x;
    const int64_t m0 = (tile / gn) * S::TILE, n0 = (tile % gn) * S::TILE;
    if (m0 >= op.m || n0 >= op.n) return;
    const bool va = !(op.flags & 1) && reinterpret_cast<uintptr_t>(op.A) % 16 == 0 && op.lda % 2 == 0;
    const bool vb = (op.flags & 2) && reinterpret_cast<uintptr_t>(op.B) % 16 == 0 && op.ldb % 2 == 0;
    if (va && vb)
        gemm_tile<S, true, true>(op, m0, n0, red);
    else if (va)
        gemm_tile<S, true, false>(op, m0, n0, red);
    else if (vb)
        gemm_tile<S, false, true>(op, m0, n0, red);
    else
        gemm_tile<S, false, false>(op, m0, n0, red);
}

// Tall, narrow products (no conjugation, k <= ROWS_KMAX, n <= 256): the
// late steps of the wavefunction chain, m up to d^(n-1) rows with k and n of
// a few. A workgroup takes a block of rows_per_block(k, n) consecutive rows:
// it copies their k entries of A into LDS with 16-byte loads (one
// contiguous, coalesced block when the rows are packed, lda = k), then
// thread t computes column j = t % n of rows t / n, t / n + 256 / n, ...
// from LDS (row-mates read the same entries, a broadcast) with column j of
// B in registers; a wave's stores cover consecutive outputs. Bound by HBM
// for small k and n.
constexpr int ROWS_KMAX = 32;
constexpr int ROWS_LDS_ELEMS = 8192;  // complex entries of A staged per workgroup (64 KiB)

MPSX_HD int rows_per_block(int km, int n) {
    const int per = 256 / n;
    int passes = ROWS_LDS_ELEMS / (km * per);
    passes = passes < 1 ? 1 : (passes > 8 ? 8 : passes);
    return per * passes;
}

// KM: the op's k rounded up to a power of two (the unrolled length).
template <int KM>
__global__ void __launch_bounds__(256) k_gemm_rows(const mpsx_gemm_op *ops) {
    extern __shared__ float2 As[];  // [rows of the block][KM]
    const mpsx_gemm_op op = ops[blockIdx.y];
    if (op.m <= 0 || op.n <= 0) return;
    const int n = (int)op.n, k = (int)op.k, per = 256 / n;
    const int rb = rows_per_block(KM, n);
    const int64_t rbase = (int64_t)blockIdx.x * rb;
    if (rbase >= op.m) return;
    const int nrows = (int)((op.m - rbase) < rb ? (op.m - rbase) : rb);
    const float2 *A = reinterpret_cast<const float2 *>(op.A);
    const float2 *B = reinterpret_cast<const float2 *>(op.B);
    float2 *C = reinterpret_cast<float2 *>(op.C);
    const int t = threadIdx.x;
    // stage A rows [rbase, rbase + nrows) as As[row][kk], kk < KM (zero-padded)
    if (op.lda == k && (k & 1) == 0) {
        const float4 *src = reinterpret_cast<const float4 *>(A + rbase * k);
        const int pairs = nrows * k / 2;
        for (int e = t; e < pairs; e += 256) {
            const float4 v = src[e];
            const int c = 2 * e, row = c / k, kk = c % k;
            As[row * KM + kk] = make_float2(v.x, v.y);
            As[row * KM + kk + 1] = make_float2(v.z, v.w);
        }
        if (k < KM)
            for (int e = t; e < nrows * (KM - k); e += 256)
                As[(e / (KM - k)) * KM + k + e % (KM - k)] = make_float2(0.f, 0.f);
    } else {
        for (int e = t; e < nrows * KM; e += 256) {
            const int row = e / KM, kk = e % KM;
            As[e] = kk < k ? A[(rbase + row) * op.lda + kk] : make_float2(0.f, 0.f);
        }
    }
    __syncthreads();
    if (t >= per * n) return;
    const int j = t % n;
    float2 bcol[KM];
#pragma unroll
    for (int kk = 0; kk < KM; ++kk)
        bcol[kk] = kk < k ? B[(int64_t)kk * op.ldb + j] : make_float2(0.f, 0.f);
    const float2 alpha = make_float2(op.alpha_re, op.alpha_im);
    const bool accum = (op.flags & 4) != 0;
    for (int row = t / n; row < nrows; row += per) {
        float2 acc = make_float2(0.f, 0.f);
#pragma unroll
        for (int kk = 0; kk < KM; ++kk) acc = cfma(As[row * KM + kk], bcol[kk], acc);
        float2 v = cmul(alpha, acc);
        float2 *dst = C + (rbase + row) * op.ldc + j;
        if (accum) {
            const float2 old = *dst;
            v.x += old.x;
            v.y += old.y;
        }
        *dst = v;
    }
}

bool gemm_rows_fit(const mpsx_gemm_op &o) {
    return (o.flags & 3) == 0 && o.k <= ROWS_KMAX && o.n >= 1 && o.n <= 256;
}

hipError_t launch_gemm_rows(hipStream_t s, const mpsx_gemm_op *h, const mpsx_gemm_op *d,
                            int count) {
    int64_t kmax = 1;
    for (int i = 0; i < count; ++i) kmax = kmax > h[i].k ? kmax : h[i].k;
    const int km = kmax <= 2 ? 2 : kmax <= 4 ? 4 : kmax <= 8 ? 8 : kmax <= 16 ? 16 : 32;
    int64_t blocks = 1;
    int rb_max = 1;
    for (int i = 0; i < count; ++i) {
        if (h[i].m <= 0 || h[i].n <= 0) continue;
        const int rb = rows_per_block(km, (int)h[i].n);
        rb_max = rb_max > rb ? rb_max : rb;
        blocks = blocks > (h[i].m + rb - 1) / rb ? blocks : (h[i].m + rb - 1) / rb;
    }
    if (blocks > 2147483647LL || count > 65535) return hipErrorInvalidValue;
    const dim3 g((unsigned)blocks, (unsigned)count), blk(256);
    const size_t lds = sizeof(float2) * (size_t)rb_max * km;
    if (km == 2)
        hipLaunchKernelGGL(k_gemm_rows<2>, g, blk, lds, s, d);
    else if (km == 4)
        hipLaunchKernelGGL(k_gemm_rows<4>, g, blk, lds, s, d);
    else if (km == 8)
        hipLaunchKernelGGL(k_gemm_rows<8>, g, blk, lds, s, d);
    else if (km == 16)
        hipLaunchKernelGGL(k_gemm_rows<16>, g, blk, lds, s, d);
    else
        hipLaunchKernelGGL(k_gemm_rows<32>, g, blk, lds, s, d);
    return hipGetLastError();
}

using GemmWide = GemmShape<2, 2, 1, 2, 2>;  // 64 x 64
using GemmMid = GemmShape<1, 2, 1, 2, 5>;   // 32 x 32
using GemmThin = GemmShape<1, 1, 4, 2, 5>;  // 16 x 16, four waves along k

template <class S>
static hipError_t gemm_run(hipStream_t s, const mpsx_gemm_op *d, int count, int64_t max_m, int64_t max_n) {
    const int64_t gm = (max_m + S::TILE - 1) / S::TILE, gn = (max_n + S::TILE - 1) / S::TILE;
    if (gm * gn > 2147483647LL || count > 65535) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_gemm<S>, dim3((unsigned)(gm * gn), (unsigned)count), dim3(S::THREADS), 0, s, d, gn);
    return hipGetLastError();
}

// The tile of a call. First the largest that still makes about a workgroup a
// compute unit: above that the wider tile reads less (4096 x 512 x 256: 50 us wide, 60
// mid; 16 of 256 x 256 x 256: 26 and 32), below it the narrower one has the waves
// (1024 x 512 x 256, 128 wide tiles: 17 us mid, 23 wide; 256 x 512 x 256, 128
// mid ones: 6.8 thin, 9.1 mid). Then a smaller one where the matrices leave much of that
// tile empty: an element of a full tile takes about 1 : 1.25 : 1.5 wide : mid : thin (64
// columns, k = 256: 135, 160 and 199 us of 100000 rows), and so do the elements of padding.
// In us, wide tiles -> this choice: 2^20 x 3 x 33 361 -> 135, 100000 x 24 x 64 52 -> 37,
// 100000 x 80 x 40 77 -> 70, 2000 of 8 x 8 x 40 52 -> 13, of 65 x 65 x 40 205 -> 108.
// Not where the launch, sized for the largest m and the largest n, would be mostly
// workgroups without a tile.
constexpr int64_t GEMM_FILL = 192;

hipError_t launch_gemm(hipStream_t s, const mpsx_gemm_op *h, const mpsx_gemm_op *d, int count, int64_t max_m,
                       int64_t max_n) {
    if (max_m < 1 || max_n < 1) return hipSuccess;
    constexpr int64_t edge[3] = {GemmWide::TILE, GemmMid::TILE, GemmThin::TILE};
    constexpr double cost[3] = {1.0, 1.25, 1.5};  // of an element
    int64_t tiles[3] = {0, 0, 0};
    for (int i = 0; i < count; ++i)
        for (int t = 0; t < 3; ++t) tiles[t] += ((h[i].m + edge[t] - 1) / edge[t]) * ((h[i].n + edge[t] - 1) / edge[t]);
    const int fill = tiles[0] >= GEMM_FILL ? 0 : tiles[1] >= GEMM_FILL ? 1 : 2;
    int pick = fill;
    for (int t = fill + 1; t < 3; ++t) {
        const int64_t grid = ((max_m + edge[t] - 1) / edge[t]) * ((max_n + edge[t] - 1) / edge[t]);
        if (grid > 2147483647LL || (double)grid * count > 2.0 * (double)tiles[t]) continue;
        if (cost[t] * (double)(tiles[t] * edge[t] * edge[t]) < cost[pick] * (double)(tiles[pick] * edge[pick] * edge[pick]))
            pick = t;
    }
    if (pick == 0) return gemm_run<GemmWide>(s, d, count, max_m, max_n);
    if (pick == 1) return gemm_run<GemmMid>(s, d, count, max_m, max_n);
    return gemm_run<GemmThin>(s, d, count, max_m, max_n);
}
