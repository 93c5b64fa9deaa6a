// One-site gate and elementwise scale kernels (HBM-bound).
//
//   one-site   out[l, o, r] = sum_p G[o, p] a[l, p, r]
//              (mpsim/core.py:753-826, the tensordot of core.py:825)
//   scale      x <- f * x or f * conj(x)
//              (MPS.renormalize core.py:591-594, MPS.dagger core.py:502-505)
#include <hip/hip_runtime.h>

#include <cstring>

#include "common.h"
#include "launch.h"

constexpr int SITE_MAXD = 16;

// Each thread owns one (l, r) column of a site tensor and reads its d
// physical entries (stride chi_r: consecutive threads take consecutive r,
// so every load and store instruction is coalesced).
template <int D>
MPSX_DEV void one_site_body(const mpsx_site_op &op, const float2 *g, int64_t e) {
    const int64_t chi_r = op.chi_r;
    const int64_t l = e / chi_r, r = e - l * chi_r;
    const float2 *src = reinterpret_cast<const float2 *>(op.a) + l * D * chi_r + r;
    float2 *dst = reinterpret_cast<float2 *>(op.out) + l * D * chi_r + r;
    float2 v[D];
#pragma unroll
    for (int p = 0; p < D; ++p) v[p] = src[p * chi_r];
#pragma unroll
    for (int o = 0; o < D; ++o) {
        float2 acc = make_float2(0.f, 0.f);
#pragma unroll
        for (int p = 0; p < D; ++p) acc = cfma(g[o * D + p], v[p], acc);
        dst[o * chi_r] = acc;
    }
}

MPSX_DEV void one_site_generic(const mpsx_site_op &op, const float2 *g, int64_t e) {
    const int d = op.d;
    const int64_t chi_r = op.chi_r;
    const int64_t l = e / chi_r, r = e - l * chi_r;
    const float2 *src = reinterpret_cast<const float2 *>(op.a) + l * d * chi_r + r;
    float2 *dst = reinterpret_cast<float2 *>(op.out) + l * d * chi_r + r;
    float2 v[SITE_MAXD];
    for (int p = 0; p < d; ++p) v[p] = src[p * chi_r];
    for (int o = 0; o < d; ++o) {
        float2 acc = make_float2(0.f, 0.f);
        for (int p = 0; p < d; ++p) acc = cfma(g[o * d + p], v[p], acc);
        dst[o * chi_r] = acc;
    }
}

// One kernel per qudit dimension 2..4 (ops of other dimensions return at
// once), launched for the dimensions a call has.
// Ops: the descriptors in device memory, or in the launch's arguments
// (SiteArgs: for one gate at a time, which a launch of k_put before it, 5 us,
// would double).
struct SiteArgs {
    mpsx_site_op op[MPSX_SITE_NOW];
    MPSX_DEV const mpsx_site_op &operator[](unsigned i) const { return op[i]; }
};
template <int D, class Ops>
__global__ void __launch_bounds__(256) k_one_site(Ops ops) {
    __shared__ float2 g[D * D];
    const mpsx_site_op op = ops[blockIdx.y];
    if (op.d != D) return;
    const float2 *G = reinterpret_cast<const float2 *>(op.gate);
    for (int i = threadIdx.x; i < D * D; i += blockDim.x) g[i] = G[i];
    __syncthreads();
    const int64_t pairs = op.chi_l * op.chi_r;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < pairs;
         e += (int64_t)gridDim.x * blockDim.x)
        one_site_body<D>(op, g, e);
}

// Every other dimension (1, and 5..16). Kept apart from the unrolled kernels
// because its runtime-indexed input array lives in scratch memory, which
// every launch of a kernel that has it must reserve.
template <class Ops>
__global__ void __launch_bounds__(256) k_one_site_gen(Ops ops) {
    __shared__ float2 g[SITE_MAXD * SITE_MAXD];
    const mpsx_site_op op = ops[blockIdx.y];
    const int d = op.d;
    if (d >= 2 && d <= 4) return;
    const float2 *G = reinterpret_cast<const float2 *>(op.gate);
    for (int i = threadIdx.x; i < d * d; i += blockDim.x) g[i] = G[i];
    __syncthreads();
    const int64_t pairs = op.chi_l * op.chi_r;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < pairs;
         e += (int64_t)gridDim.x * blockDim.x)
        one_site_generic(op, g, e);
}

__global__ void __launch_bounds__(256) k_scale(const mpsx_scale_op *ops) {
    const mpsx_scale_op op = ops[blockIdx.y];
    float2 *x = reinterpret_cast<float2 *>(op.x);
    const float2 f = make_float2(op.re, op.im);
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < op.n;
         e += (int64_t)gridDim.x * blockDim.x) {
        float2 v = x[e];
        if (op.conj) v.y = -v.y;
        x[e] = cmul(f, v);
    }
}

// A small table from the host in the launch's own arguments: no staging
// buffer, no copy engine and no wait on either side. Latency only: a call
// preceded by a blocking copy of its table cost 40-50 us of host time and left the
// GPU idle between calls; 24 state vectors of 8-12 qubits (217 such calls and a graph
// replay) take 5.0 ms instead of 9.4, a 16-qubit circuit gate by gate 11.9 instead of 15.8.
struct PutChunk {
    uint32_t w[PUT_CHUNK / 4];
};
__global__ void __launch_bounds__(256) k_put(uint32_t *dst, int words, PutChunk c) {
    for (int i = threadIdx.x; i < words; i += 256) dst[i] = c.w[i];
}

hipError_t launch_put(hipStream_t s, void *dst, const void *src, size_t bytes) {
    for (size_t at = 0; at < bytes; at += PUT_CHUNK) {
        const size_t n = bytes - at < (size_t)PUT_CHUNK ? bytes - at : (size_t)PUT_CHUNK;
        PutChunk c;
        memcpy(c.w, static_cast<const char *>(src) + at, n);
        hipLaunchKernelGGL(k_put, dim3(1), dim3(256), 0, s,
                           reinterpret_cast<uint32_t *>(static_cast<char *>(dst) + at), (int)(n / 4), c);
    }
    return hipGetLastError();
}

static unsigned blocks_for(int64_t n, int64_t per_block, unsigned cap) {
    int64_t b = (n + per_block - 1) / per_block;
    if (b < 1) b = 1;
    if (b > cap) b = cap;
    return (unsigned)b;
}

template <class Ops>
static hipError_t launch_one_site_t(hipStream_t s, Ops ops, int count, int64_t max_pairs, uint32_t dmask) {
    dim3 grid(blocks_for(max_pairs, 256, 8192), (unsigned)count);
    if (dmask & (1u << 2)) hipLaunchKernelGGL((k_one_site<2, Ops>), grid, dim3(256), 0, s, ops);
    if (dmask & (1u << 3)) hipLaunchKernelGGL((k_one_site<3, Ops>), grid, dim3(256), 0, s, ops);
    if (dmask & (1u << 4)) hipLaunchKernelGGL((k_one_site<4, Ops>), grid, dim3(256), 0, s, ops);
    if (dmask & ~((1u << 2) | (1u << 3) | (1u << 4)))
        hipLaunchKernelGGL(k_one_site_gen<Ops>, grid, dim3(256), 0, s, ops);
    return hipGetLastError();
}

hipError_t launch_one_site(hipStream_t s, const mpsx_site_op *h, const mpsx_site_op *d, int count,
                           int64_t max_pairs, uint32_t dmask) {
    if (d) return launch_one_site_t(s, d, count, max_pairs, dmask);
    SiteArgs args = {};
    memcpy(args.op, h, sizeof(mpsx_site_op) * (size_t)count);
    return launch_one_site_t(s, args, count, max_pairs, dmask);
}

hipError_t launch_scale(hipStream_t s, const mpsx_scale_op *d, int count, int64_t max_n) {
    dim3 grid(blocks_for(max_n, 256 * 4, 8192), (unsigned)count);
    hipLaunchKernelGGL(k_scale, grid, dim3(256), 0, s, d);
    return hipGetLastError();
}
