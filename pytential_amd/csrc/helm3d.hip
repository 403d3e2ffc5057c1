// 3D Helmholtz point sums for smooth (far) targets and their adjoints: the
// forward and backward kernels of the differentiable single-layer evaluation
// at targets that need no QBX (pytential evaluates such targets through the
// plain FMM part of the QBX-FMM, qbx/fmm.py:216-225, P2P/M2P/L2P with
// HelmholtzKernel(3) = e^{ikr} / (4 pi r)).
//
//   pot[t]    = sum_s G_k(t, s) q_s,          G_k = e^{ik|t-s|} / (4 pi |t-s|)
//   dpot_dk[t] = sum_s dG_k/dk q_s = sum_s i e^{ik|t-s|} / (4 pi) q_s
//   v[s]      = sum_t conj(G_k(t, s)) u_t     (the adjoint, G^H u)
//
// Both directions are a point per thread against the other set, staged
// through LDS in tiles.  Forward: few targets (thousands) against many
// sources, so the sources are split into chunks across blocks until they
// fill the chip: block (tile of 256 targets, chunk) sums its chunk and writes
// a partial, and a second kernel adds the partials of each target in chunk
// order.  Adjoint: a source takes 1, 4 or 16 threads of a block, whichever
// first gives blocks to fill the chip, added in LDS in order (no scratch
// memory: calls on several streams share nothing).  Deterministic, no
// atomics.  Coincident points contribute zero.
//
// FP64 VALU bound: a pair is 59 (forward with the k-derivative) or 57
// instructions.  4096 targets and 737280 sources, 3.0e9 pairs: forward
// 8.1 -> 5.4 ms, adjoint 8.0 -> 5.2 ms against two Newton steps, nine-term
// Taylor series and a branch per pair for coincidence and for the range of
// the sine.
#include "qbx_internal.h"
#include "qbx_math.h"

#include <algorithm>

namespace qbx {

constexpr int H3_THREADS = 256;   // targets (forward) / sources (adjoint) per block
constexpr int H3_TILE = 256;      // staged points per LDS tile
constexpr double INV4PI = 0.07957747154594766788;

struct H3Sums {
    double pr = 0, pi = 0, dr = 0, di = 0;
};

// e^{+-ikr} q / r (and i e^{ikr} q) of one pair, added.  FAST leaves out the
// test for coincident points and large k r and reports either (a coincident
// pair's k r is a NaN) for the tile to be summed again without FAST.
template <bool FAST, bool ADJ>
__device__ __forceinline__ bool h3_pair(double dx, double dy, double dz, double k, double qr,
                                        double qi, H3Sums &a)
{
    const double r2 = dx * dx + dy * dy + dz * dz;
    if (!FAST && r2 == 0.0) return false;
    const double ir = qbx_rsqrt(r2);
    const double x = k * (r2 * ir);
    double sn, cs;
    if (FAST)
        qbx_sincos_core(x, &sn, &cs);
    else
        qbx_sincos(x, &sn, &cs);
    const double si = ADJ ? -sn : sn;
    const double er = cs * qr - si * qi;
    const double ei = cs * qi + si * qr;
    a.pr += er * ir;
    a.pi += ei * ir;
    if (!ADJ) {
        a.dr -= ei;
        a.di += er;
    }
    return FAST && !(__builtin_fabs(x) <= QBX_SINCOS_MAX);
}

// part[chunk][point] = the sum over the chunk's points b (values q) at point
// a of set A, SPL threads to a point; ADJ false: part_dk likewise
template <bool ADJ, int SPL>
__global__ void __launch_bounds__(H3_THREADS)
k_h3_p2p(int nb, const double *ptb, const double *q, int na, const double *pta, double k,
         int chunk, double scale, double *part, double *part_dk)
{
    __shared__ double2 bxy[H3_TILE], bq[H3_TILE];
    __shared__ double bz[H3_TILE];
    constexpr int PP = H3_THREADS / SPL;
    const int sub = threadIdx.x / PP;
    const int t = blockIdx.x * PP + threadIdx.x % PP;
    const int c = blockIdx.y;
    const int b0 = c * chunk, b1 = min(nb, b0 + chunk);
    const bool act = t < na;
    const double ax = act ? pta[t] : 0.0, ay = act ? pta[(size_t)na + t] : 0.0,
                 az = act ? pta[2 * (size_t)na + t] : 0.0;
    H3Sums tot;
    for (int b = b0; b < b1; b += H3_TILE) {
        const int n = min(H3_TILE, b1 - b);
        __syncthreads();
        for (int j = threadIdx.x; j < n; j += H3_THREADS) {
            const size_t s = b + j;
            bxy[j] = {ptb[s], ptb[(size_t)nb + s]};
            bz[j] = ptb[2 * (size_t)nb + s];
            bq[j] = {q[2 * s], q[2 * s + 1]};
        }
        __syncthreads();
        H3Sums a;
        bool again = false;
#pragma unroll 2
        for (int j = sub; j < n; j += SPL)
            again |= h3_pair<true, ADJ>(ax - bxy[j].x, ay - bxy[j].y, az - bz[j], k, bq[j].x,
                                        bq[j].y, a);
        if (again && act) {
            a = H3Sums();
            for (int j = sub; j < n; j += SPL)
                h3_pair<false, ADJ>(ax - bxy[j].x, ay - bxy[j].y, az - bz[j], k, bq[j].x,
                                    bq[j].y, a);
        }
        tot.pr += a.pr;
        tot.pi += a.pi;
        tot.dr += a.dr;
        tot.di += a.di;
    }
    if (SPL > 1) {
        __syncthreads();
        bq[threadIdx.x] = {tot.pr, tot.pi};
        __syncthreads();
        if (sub > 0) return;
        for (int w = 1; w < SPL; ++w) {
            tot.pr += bq[w * PP + t % PP].x;
            tot.pi += bq[w * PP + t % PP].y;
        }
    }
    if (act) {
        const size_t o = (size_t)c * na + t;
        part[2 * o] = tot.pr * scale;
        part[2 * o + 1] = tot.pi * scale;
        if (!ADJ && part_dk) {
            part_dk[2 * o] = tot.dr * scale;
            part_dk[2 * o + 1] = tot.di * scale;
        }
    }
}

__global__ void k_h3_reduce(int nchunks, int nt, const double *part, double *out)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nt) return;
    double re = 0, im = 0;
    for (int c = 0; c < nchunks; ++c) {
        re += part[2 * ((size_t)c * nt + t)];
        im += part[2 * ((size_t)c * nt + t) + 1];
    }
    out[2 * (size_t)t] = re * INV4PI;
    out[2 * (size_t)t + 1] = im * INV4PI;
}

// out[e, j, r] = sum_i mat[i, j] in[e, i, r]  (the transpose of qbx_upsample)
__global__ void k_upsample_adjoint(int nel, int n1, int nf, int nr, const double *mat,
                                   const double *in, double *out)
{
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)nel * n1 * nr) return;
    const long ej = idx / nr;
    const int r = (int)(idx % nr);
    const int e = (int)(ej / n1), j = (int)(ej % n1);
    double re = 0, im = 0;
    for (int i = 0; i < nf; ++i) {
        const double m = mat[i * n1 + j];
        const size_t kk = ((size_t)e * nf + i) * nr + r;
        re += m * in[2 * kk];
        im += m * in[2 * kk + 1];
    }
    out[2 * idx] = re;
    out[2 * idx + 1] = im;
}

}  // namespace qbx

using namespace qbx;

extern "C" {

int qbx_helmholtz3d_p2p(qbx_ctx *ctx, void *stream, int nsources, const double *sources,
                        const double *strengths, int ntargets, const double *targets, double k,
                        double *pot, double *dpot_dk)
{
    QBX_CHECK(ctx && pot, "qbx_helmholtz3d_p2p: null argument");
    QBX_CHECK(nsources >= 0 && ntargets >= 0, "qbx_helmholtz3d_p2p: negative size");
    QBX_CHECK(nsources == 0 || (sources && strengths), "qbx_helmholtz3d_p2p: null sources");
    QBX_CHECK(ntargets == 0 || targets, "qbx_helmholtz3d_p2p: null targets");
    hipStream_t st = S(stream);
    if (ntargets == 0) return QBX_OK;
    if (nsources == 0) {
        QBX_TRY(zero_fill(pot, 2L * ntargets, st));
        if (dpot_dk) QBX_TRY(zero_fill(dpot_dk, 2L * ntargets, st));
        return QBX_OK;
    }
    const int tiles = cdiv(ntargets, H3_THREADS);
    // enough blocks to fill the chip (8 per CU on 256 CUs), chunks of at
    // least one LDS tile
    int nchunks = std::max(1, 2048 / tiles);
    nchunks = std::min(nchunks, cdiv(nsources, H3_TILE));
    const int chunk = cdiv(nsources, nchunks);
    nchunks = cdiv(nsources, chunk);
    const size_t pb = sizeof(double) * 2 * (size_t)nchunks * ntargets;
    void *scr;
    QBX_TRY(scratch_reserve(ctx, st, dpot_dk ? 2 * pb : pb, &scr));
    double *ppot = (double *)scr;
    double *pdk = dpot_dk ? ppot + 2 * (size_t)nchunks * ntargets : nullptr;
    hipLaunchKernelGGL((k_h3_p2p<false, 1>), dim3(tiles, nchunks), dim3(H3_THREADS), 0, st,
                       nsources, sources, strengths, ntargets, targets, k, chunk, 1.0, ppot, pdk);
    hipLaunchKernelGGL(k_h3_reduce, dim3(cdiv(ntargets, 256)), dim3(256), 0, st, nchunks,
                       ntargets, ppot, pot);
    if (dpot_dk)
        hipLaunchKernelGGL(k_h3_reduce, dim3(cdiv(ntargets, 256)), dim3(256), 0, st, nchunks,
                           ntargets, pdk, dpot_dk);
    QBX_HIP(hipGetLastError());
    return QBX_OK;
}

int qbx_helmholtz3d_p2p_adjoint(qbx_ctx *ctx, void *stream, int nsources, const double *sources,
                                int ntargets, const double *targets, double k, const double *u,
                                double *v)
{
    QBX_CHECK(ctx && v, "qbx_helmholtz3d_p2p_adjoint: null argument");
    QBX_CHECK(nsources >= 0 && ntargets >= 0, "qbx_helmholtz3d_p2p_adjoint: negative size");
    QBX_CHECK(nsources == 0 || sources, "qbx_helmholtz3d_p2p_adjoint: null sources");
    QBX_CHECK(ntargets == 0 || (targets && u), "qbx_helmholtz3d_p2p_adjoint: null targets");
    if (nsources == 0) return QBX_OK;
    hipStream_t st = S(stream);
#define H3_ADJ(SPL)                                                                       \
    hipLaunchKernelGGL((k_h3_p2p<true, SPL>), dim3(cdiv(nsources, H3_THREADS / (SPL))),    \
                       dim3(H3_THREADS), 0, st, ntargets, targets, u, nsources, sources, k, \
                       ntargets, INV4PI, v, nullptr)
    // 1024 blocks (four per CU) at 1 and 4 threads a source, else 16
    if (nsources >= 1024 * H3_THREADS)
        H3_ADJ(1);
    else if (nsources >= 256 * H3_THREADS)
        H3_ADJ(4);
    else
        H3_ADJ(16);
#undef H3_ADJ
    QBX_HIP(hipGetLastError());
    return QBX_OK;
}

int qbx_upsample_adjoint(qbx_ctx *ctx, void *stream, int nelements, int n1, int nf, int nrhs,
                         const double *mat, const double *in, double *out)
{
    QBX_CHECK(ctx && mat && in && out, "qbx_upsample_adjoint: null argument");
    QBX_CHECK(nelements >= 0 && n1 > 0 && nf > 0 && nrhs >= 1, "qbx_upsample_adjoint: bad size");
    const long n = (long)nelements * n1 * nrhs;
    if (n == 0) return QBX_OK;
    hipLaunchKernelGGL(k_upsample_adjoint, dim3(cdiv(n, 256)), dim3(256), 0, S(stream),
                       nelements, n1, nf, nrhs, mat, in, out);
    QBX_HIP(hipGetLastError());
    return QBX_OK;
}

}  // extern "C"
