// QBX-FMM wrangler stages for 3D Laplace (pytential/qbx/fmm.py drive_fmm and
// pytential/qbx/interactions.py), FP64 / complex128.
//
// Expansions in solid harmonics (coefficient (n, m) at n*n + n + m):
//   Y_n^m(x) = r^n P_n^m(cos th) e^{i m phi} / (n+m)!        regular
//   T_n^m(x) = (n-m)! P_n^m(cos th) e^{i m phi} / r^{n+1}    irregular
//   Y_n^{-m} = (-1)^m conj(Y_n^m), T_n^{-m} = (-1)^m conj(T_n^m)
//   1/|x-y| = sum conj(Y_n^m(y)) T_n^m(x) for |y| < |x|
//   multipole  M_n^m = sum q conj(Y_n^m(s-c)),  phi(x) = sum M T(x-c)
//   local      L_n^m = sum q T_n^m(s-c),        phi(x) = sum L conj(Y(x-c))
//   M2M  M'_n^m = sum_{k,l} conj(Y_k^l(c-c')) M_{n-k}^{m-l}
//   M2L  L_k^l  = (-1)^k sum_{n,m} M_n^m T_{n+k}^{m+l}(c'-c)
//   L2L  L'_a^b = sum_{j,i} L_{a+j}^{b+i} conj(Y_j^i(c'-c))
// Double layer: q nu . grad_s through
//   d_z Y_n^m = Y_{n-1}^m, (d_x +- i d_y) Y_n^m = +-Y_{n-1}^{m+-1},
//   d_z T_n^m = -T_{n+1}^m, (d_x +- i d_y) T_n^m = +-T_{n+1}^{m+-1}.
// Potentials carry G = 1/(4 pi r).
//
// Recurrences (no trigonometry, w = x + i y, r^2 = |x|^2):
//   Y_m^m = -(w/2m) Y_{m-1}^{m-1}, (n-m)(n+m) Y_n^m = (2n-1) z Y_{n-1}^m - r^2 Y_{n-2}^m
//   T_m^m = -(2m-1)(w/r^2) T_{m-1}^{m-1},
//   T_n^m = ((2n-1) z T_{n-1}^m - (n+m-1)(n-m-1) T_{n-2}^m) / r^2
//
// Right-hand sides: as in the 2D stages, nr densities share one evaluation,
// arrays carry them innermost, and each kernel applies an interaction's
// geometry (harmonics, translation weights) to a chunk of right-hand sides
// held in registers; the host launches one chunk [r0, r0 + rc) at a time.
//
// Storage (HBM): box expansions level-compact, (p_l+1)^2 complex per box of
// level l (times nr); QBX expansions [ncenters][(p_q+1)^2][nr].
//
// Thread mappings:
//  P2M, P2L        one thread per (box, coefficient)
//  M2M, L2L        one thread per (box, coefficient), child offsets from a
//                  table of Y at the 8 unit child offsets
//  M2L             one 64-lane block per target box; each list-2 multipole is
//                  staged (rescaled by h^-n) in LDS and contracted against
//                  the irregular harmonics of its integer offset class, read
//                  from a table T(delta), |delta_i| <= 2 nsep + 1
//  P2P, M2P, L2P   one block per target box, lane groups per target
//  P2QBXL          16 lanes per QBX center over its list-1 sources, the
//                  order-p_q expansion in registers, shuffle reduction
//  M2QBXL          16 lanes per QBX center: per list-3 box the irregular
//                  harmonics of the offset are built in LDS, then each lane
//                  contracts its output coefficients
//  L2QBXL          one thread per QBX center, expansion in registers
//  QBXL2P          one thread per (center, target) pair
#include "qbx_internal.h"
#include "qbx_math.h"

#include <complex>
#include <cstring>
#include <vector>

namespace qbx {
namespace f3 {

constexpr int MAXP = 20;       // box expansion orders
constexpr int MAXPQ = 8;       // QBX expansion orders (templated)
constexpr int FML = 21;        // levels of a 3D tree (19-bit coordinates)
constexpr int NRC_S = 8;       // RHS chunk of the scalar-accumulator kernels
constexpr int NRC_Q = 2;       // RHS chunk of the QBX-expansion kernels
constexpr double INV4PI = 0.079577471545947667884;

__host__ __device__ constexpr int IDX(int n, int m) { return n * n + n + m; }

// accumulator of v_mfma_f64_16x16x4f64 (4 doubles per lane)
typedef double f3_d4 __attribute__((ext_vector_type(4)));

struct KD {
    int dip, pq, nlevels, ncq, nsep, W, pmax, tabn;   // tabn = 2 pmax + 1
    int nr, r0, rc;            // right-hand sides; the chunk of this launch
    int order[FML];
    int ncl[FML];
    int lbox[FML + 1];
    long lcoef[FML + 1];
    double h[FML];
    const double *tab_m2l;   // [(2W+1)^3][tabn^2] complex: T(delta), unit box size
    const double *tab_ch;    // [8][(pmax+1)^2] complex: Y(bit - 1/2), unit child size
};

struct TD {
    int nboxes;
    const int *level, *parent, *child, *coords;
    const double *centers;  // [3][nboxes]
    const int *sstart, *scount, *scumul;
};

struct v3 {
    double x, y, z;
};
__device__ __forceinline__ v3 ld3(const double *p, long n, long i)
{
    return {p[i], p[n + i], p[2 * n + i]};
}
__device__ __forceinline__ v3 sub(v3 a, v3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ v3 boxc(const TD &t, int b) { return ld3(t.centers, t.nboxes, b); }

// coefficient 0, right-hand side 0 of box b; coefficient i, right-hand side
// r at [2 (i nr + r)]
__device__ __forceinline__ long ecoef_off(const KD &kd, int b, int lv)
{
    return 2 * (kd.lcoef[lv] + (long)(b - kd.lbox[lv]) * kd.ncl[lv]) * kd.nr;
}

__device__ __forceinline__ cplx ldq(const KD &kd, const double *str, int s, int r)
{
    return ldc(str + 2 * ((size_t)s * kd.nr + r));
}

__device__ __forceinline__ cplx ldcn(const KD &kd, const double *a, int i, int r)
{
    return ldc(a + 2 * ((long)i * kd.nr + r));
}

__device__ __forceinline__ void nm_of(int i, int &n, int &m)
{
    n = (int)sqrt((double)i);
    while (n * n > i) --n;
    while ((n + 1) * (n + 1) <= i) ++n;
    m = i - n * n - n;
}

__device__ __forceinline__ cplx neg_m(cplx v, int am)  // (-1)^m conj(v)
{
    return (am & 1) ? cplx{-v.x, v.y} : cplx{v.x, -v.y};
}

// full table T_n^m(d), n <= P, in registers
template <int P>
__device__ __forceinline__ void the_table(v3 d, cplx *T)
{
    const double r2 = d.x * d.x + d.y * d.y + d.z * d.z;
    const double ir2 = 1.0 / r2;
    const cplx w = {d.x * ir2, d.y * ir2};
    cplx tmm = {sqrt(ir2), 0};
#pragma unroll
    for (int m = 0; m <= P; ++m) {
        if (m > 0) tmm = (-(2.0 * m - 1.0)) * (tmm * w);
        T[IDX(m, m)] = tmm;
        cplx a = {0, 0}, b = tmm;
#pragma unroll
        for (int n = m + 1; n <= P; ++n) {
            const cplx c = ir2 * (((2.0 * n - 1.0) * d.z) * b -
                                  ((double)(n + m - 1) * (n - m - 1)) * a);
            T[IDX(n, m)] = c;
            a = b;
            b = c;
        }
    }
#pragma unroll
    for (int n = 1; n <= P; ++n)
#pragma unroll
        for (int m = 1; m <= n; ++m) T[IDX(n, -m)] = neg_m(T[IDX(n, m)], m);
}

// out[q] += sum_{n<=p,m} coef[n,m][r0+q] T_n^m(d); coef strided by nr,
// streamed column by column with O(1) harmonic state
template <int NRC>
__device__ void sum_irregular_n(const KD &kd, const double *coef, int p, v3 d, cplx *out)
{
    const double r2 = d.x * d.x + d.y * d.y + d.z * d.z;
    const double ir2 = 1.0 / r2;
    const cplx w = {d.x * ir2, d.y * ir2};
    cplx tmm = {sqrt(ir2), 0};
    for (int m = 0; m <= p; ++m) {
        if (m > 0) tmm = (-(2.0 * m - 1.0)) * (tmm * w);
        cplx a = {0, 0}, b = tmm;
        for (int n = m; n <= p; ++n) {
            if (n > m) {
                const cplx c = ir2 * (((2.0 * n - 1.0) * d.z) * b -
                                      ((double)(n + m - 1) * (n - m - 1)) * a);
                a = b;
                b = c;
            }
            const cplx bn = neg_m(b, m);
#pragma unroll
            for (int q = 0; q < NRC; ++q)
                if (q < kd.rc) {
                    out[q] += ldcn(kd, coef, IDX(n, m), kd.r0 + q) * b;
                    if (m > 0) out[q] += ldcn(kd, coef, IDX(n, -m), kd.r0 + q) * bn;
                }
        }
    }
}

// out[q] += sum_{n<=p,m} coef[n,m][r0+q] conj(Y_n^m(d)); conj(Y_n^{-m}) = (-1)^m Y_n^m
template <int NRC>
__device__ void sum_regular_conj_n(const KD &kd, const double *coef, int p, v3 d, cplx *out)
{
    const double r2 = d.x * d.x + d.y * d.y + d.z * d.z;
    const cplx hw = {-0.5 * d.x, -0.5 * d.y};
    cplx ymm = {1, 0};
    for (int m = 0; m <= p; ++m) {
        if (m > 0) ymm = (1.0 / m) * (ymm * hw);
        cplx a = {0, 0}, b = ymm;
        for (int n = m; n <= p; ++n) {
            if (n > m) {
                const cplx c = (1.0 / ((double)(n - m) * (n + m))) *
                               (((2.0 * n - 1.0) * d.z) * b - r2 * a);
                a = b;
                b = c;
            }
            const cplx bc = conj(b);
            const cplx bs = (m & 1) ? -b : b;
#pragma unroll
            for (int q = 0; q < NRC; ++q)
                if (q < kd.rc) {
                    out[q] += ldcn(kd, coef, IDX(n, m), kd.r0 + q) * bc;
                    if (m > 0) out[q] += ldcn(kd, coef, IDX(n, -m), kd.r0 + q) * bs;
                }
        }
    }
}

__device__ __forceinline__ double p2p_value(const KD &kd, v3 s, v3 nu, v3 t)
{
    const v3 d = sub(t, s);
    const double r2 = d.x * d.x + d.y * d.y + d.z * d.z;
    if (r2 == 0.0) return 0.0;
    const double ir = qbx_rsqrt(r2);
    if (!kd.dip) return INV4PI * ir;
    return INV4PI * ir * ir * ir * (nu.x * d.x + nu.y * d.y + nu.z * d.z);
}

template <int NRC>
__device__ __forceinline__ void store_add(const KD &kd, double *o, const cplx *acc)
{
#pragma unroll
    for (int q = 0; q < NRC; ++q)
        if (q < kd.rc) {
            double *p = o + 2 * (kd.r0 + q);
            stc(p, ldc(p) + acc[q]);
        }
}

// P2M and P2L, a block per box, on the FP64 matrix cores for any number of
// densities.  S sources at a time (the box's own, or those of its list-4
// boxes, dealt without regard to box borders) the block forms the harmonics
// of source - center once, real rows H[n^2 + 2m - 1 or + 2m][source] (Re, Im
// of Y_n^m or T_n^m, m >= 0, n <= pt), and stages real weights: each
// density's strength (S), or the strength times each component of the source
// normal (D), real parts in one tile of 16 columns and imaginary parts in
// another that is skipped while they are all zero (up to 8 weights: both in
// one tile).  U = H weights, then the coefficients: the negative orders from
// (-1)^m conj, and for D
//   P2L: -U_z(n+1,m) + ((U_x - i U_y)(n+1,m+1) - (U_x + i U_y)(n+1,m-1)) / 2
//   P2M: conj of U_z(n-1,m) + ((U_x - i U_y)(n-1,m+1) - (U_x + i U_y)(n-1,m-1)) / 2.
// The waves split the row tiles RG ways and the sources 4 / RG ways; their
// sums meet in LDS.  Bound by the tables' recurrences and the latency of a
// step's loads at two blocks a CU (216 registers), not by the matrix cores.
//
// Row stride S + 2 doubles (even, and odd multiples of 2 mod 32 banks): the
// harmonics are written along the sources and read down the rows without
// bank conflicts.
//
// The one-lane-per-source tables and the gathered operands of the kernels
// before kept most lanes waiting: 14.8e6 (box, source) pairs at order 8 with
// 32 real densities (91 GFLOP here) took 13.9 ms, now 5.0; 1.06e6 pairs,
// one dipole density at order 10, 4.3 ms, now 0.88.
struct P2EShape {
    int S, SS, rows, RT, RG, RTW, NB, pt;
    size_t bytes;
};

template <bool LOCAL, bool DIP, int NB, int RTW>
__global__ void __launch_bounds__(256)
k3_p2e(KD kd, TD t, int i0, P2EShape sh, const int *boxes, const int *starts,
       const int *lists, const double *src, int ns, const double *str, const double *nrm,
       double *expn)
{
    extern __shared__ double lds[];
    __shared__ int pre[257], first[256], wsum[4], idx[2][32];
    const int i = i0 + blockIdx.x;
    const int Bx = boxes[i];
    int e0 = 0, e1 = 1;
    if (LOCAL) {
        e0 = starts[i];
        e1 = starts[i + 1];
        if (e0 == e1) return;
    }
    const int lv = t.level[Bx], p = kd.order[lv], pt = sh.pt;
    const int S = sh.S, SS = sh.SS, RT = sh.RT, RG = sh.RG, KG = 4 / RG;
    double *H = lds, *W = H + RT * 16 * SS;          // W[S][2 NB 16]
    constexpr int WC = 2 * NB * 16, ND = DIP ? 3 : 1;
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
    const int col = lane & 15, kr = lane >> 4;
    const int rg = wv / KG, kg = wv % KG;
    const int nr = kd.nr, rc = kd.rc, r0 = kd.r0;
    const bool pack = NB == 1 && ND * rc <= 8;
    const v3 c = boxc(t, Bx);
    f3_d4 acc[RTW][2 * NB];
#pragma unroll
    for (int a = 0; a < RTW; ++a)
#pragma unroll
        for (int b = 0; b < 2 * NB; ++b) acc[a][b] = f3_d4{0, 0, 0, 0};
    // rows beyond the table stay zero
    for (int e = sh.rows * SS + tid; e < RT * 16 * SS; e += 256) H[e] = 0.0;

    for (int eb = e0; eb < e1; eb += 256) {
        const int e = eb + tid;
        int cnt = 0;
        if (e < e1) {
            const int Sb = LOCAL ? lists[e] : Bx;
            cnt = t.scount[Sb];
            first[tid] = t.sstart[Sb];
        }
        int run = cnt;
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(run, o);
            if (lane >= o) run += y;
        }
        if (lane == 63) wsum[wv] = run;
        __syncthreads();
        for (int w = 0; w < wv; ++w) run += wsum[w];
        pre[tid + 1] = run;
        if (tid == 0) pre[0] = 0;
        __syncthreads();
        const int total = pre[256];
        // the source of the chunk's place v (the last one again beyond the end)
        auto source = [&](int v) {
            v = min(v, total - 1);
            int lo = 0, hi = 256;
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (pre[mid] <= v) lo = mid; else hi = mid;
            }
            return first[lo] + v - pre[lo];
        };
        if (total == 0) continue;
        // a chunk's points and weights pass through registers: the next
        // chunk's are loaded while this one's are multiplied
        constexpr int NW = NB * 2;               // weights of a thread (S <= 32)
        const int s = tid & (S - 1), g = tid / S, ng = 256 / S;
        v3 x;
        double wr[NW], wi[NW];
        auto fetch = [&](int v0, const int *ix) {
            x = ld3(src, ns, ix[s]);
            const int n_ = min(S, total - v0);
#pragma unroll
            for (int u = 0; u < NW; ++u) {
                const int e2 = tid + 256 * u, k = e2 / (NB * 16), cc = e2 % (NB * 16);
                // 16 / ND densities to a tile of 16 columns
                const int in = pack ? cc & 7 : cc & 15, dir = in % ND;
                const int r = (cc >> 4) * (16 / ND) + in / ND;
                wr[u] = wi[u] = 0.0;
                if (k < n_ && r < rc && in / ND < 16 / ND) {
                    const int si = ix[k];
                    const double *q = str + 2 * ((size_t)si * nr + r0 + r);
                    const double f = DIP ? nrm[(size_t)dir * ns + si] : 1.0;
                    wr[u] = f * q[0];
                    wi[u] = f * q[1];
                }
            }
        };
        if (tid < S) {
            idx[0][tid] = source(tid);
            idx[1][tid] = source(S + tid);
        }
        __syncthreads();
        fetch(0, idx[0]);
        for (int v0 = 0, buf = 1; v0 < total; v0 += S, buf ^= 1) {
            // harmonics: thread (source s, orders m = g, g + 256 / S, ...)
            {
                const v3 d = sub(x, c);
                const double r2 = d.x * d.x + d.y * d.y + d.z * d.z;
                double ir2 = 0.0;
                cplx w, mm = {1.0, 0.0};
                if (LOCAL) {
                    const double ir = qbx_rsqrt(r2);
                    ir2 = ir * ir;
                    w = {d.x * ir2, d.y * ir2};
                    mm = {ir, 0.0};
                } else {
                    w = {-0.5 * d.x, -0.5 * d.y};
                }
                const double z2 = 2.0 * d.z;
                int m = 0;
                for (int mt = g; mt <= pt; mt += ng) {
                    while (m < mt) {
                        ++m;
                        mm = LOCAL ? (-(2.0 * m - 1.0)) * (mm * w) : qbx_rcp(m) * (mm * w);
                    }
                    const double m2 = (double)(m * m);
                    cplx a = {0, 0}, b = mm;
                    double z = (2.0 * m - 1.0) * d.z, k1 = m;   // (2n-1) d.z, n
                    double *h = H + (m * m + (m > 0 ? 2 * m - 1 : 0)) * SS + s;
                    for (int n = m;;) {
                        h[0] = b.x;
                        if (m > 0) h[SS] = b.y;
                        if (++n > pt) break;
                        z += z2;
                        cplx v;
                        if (LOCAL) {
                            // (n + m - 1) (n - m - 1) = (n - 1)^2 - m^2
                            v = ir2 * (z * b - (k1 * k1 - m2) * a);
                            k1 += 1.0;
                        } else {
                            k1 += 1.0;
                            v = qbx_rcp(k1 * k1 - m2) * (z * b - r2 * a);
                        }
                        a = b;
                        b = v;
                        h += (2 * n - 1) * SS;
                    }
                }
            }
            int imag = 0;
#pragma unroll
            for (int u = 0; u < NW; ++u) {
                const int e2 = tid + 256 * u, k = e2 / (NB * 16), cc = e2 % (NB * 16);
                if (k >= S) continue;
                if (pack) {
                    W[k * WC + cc] = cc < 8 ? wr[u] : wi[u];
                } else {
                    imag |= wi[u] != 0.0;
                    W[k * WC + cc] = wr[u];
                    W[k * WC + NB * 16 + cc] = wi[u];
                }
            }
            imag = __syncthreads_or(imag);
            if (v0 + S < total) fetch(v0 + S, idx[buf]);
            for (int ks = kg; ks < S / 4; ks += KG) {
                const int k = ks * 4 + kr;
                double b[2 * NB];
#pragma unroll
                for (int j = 0; j < 2 * NB; ++j) b[j] = W[k * WC + j * 16 + col];
#pragma unroll
                for (int a = 0; a < RTW; ++a) {
                    const int rt = rg * RTW + a;
                    if (rt < RT) {
                        const double h = H[(rt * 16 + col) * SS + k];
#pragma unroll
                        for (int j = 0; j < NB; ++j) {
                            acc[a][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(h, b[j], acc[a][j],
                                                                             0, 0, 0);
                            if (imag)
                                acc[a][NB + j] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                                    h, b[NB + j], acc[a][NB + j], 0, 0, 0);
                        }
                    }
                }
            }
            if (tid < S) idx[buf ^ 1][tid] = source(v0 + 2 * S + tid);
            __syncthreads();
        }
    }
    __syncthreads();

    // the waves' sums of one column tile at a time (over H), then the
    // coefficients (n, +-m) of its densities
    double(*red)[17] = reinterpret_cast<double(*)[17]>(lds);
    double *o = expn + ecoef_off(kd, Bx, lv);
    const int nh = (p + 1) * (p + 2) / 2;
#pragma unroll
    for (int j = 0; j < 2 * NB; ++j) {
        if (pack && j == 1) break;
        const bool im = j >= NB;
        for (int w = 0; w < KG; ++w) {
            __syncthreads();
            if (kg == w) {
#pragma unroll
                for (int a = 0; a < RTW; ++a) {
                    const int rt = rg * RTW + a;
                    if (rt < RT) {
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            double &x = red[rt * 16 + 4 * q + kr][col];
                            x = (w == 0 ? 0.0 : x) + acc[a][j][q];
                        }
                    }
                }
            }
        }
        __syncthreads();
        // U(n, m) of column cc, any m, zero outside the table
        auto U = [&](int n, int m, int cc) -> cplx {
            const int am = m < 0 ? -m : m;
            if (n < 0 || am > n) return {0, 0};
            const int row = n * n + (am > 0 ? 2 * am - 1 : 0);
            const cplx v = {red[row][cc], am > 0 ? red[row + 1][cc] : 0.0};
            return m < 0 ? neg_m(v, am) : v;
        };
        auto coef = [&](int n, int m, int cc) -> cplx {
            if (!DIP) return LOCAL ? U(n, m, cc) : conj(U(n, m, cc));
            const int n1 = LOCAL ? n + 1 : n - 1;
            const cplx I = {0, 1};
            const cplx up = U(n1, m + 1, cc) - I * U(n1, m + 1, cc + 1);
            const cplx dn = U(n1, m - 1, cc) + I * U(n1, m - 1, cc + 1);
            const cplx uz = U(n1, m, cc + 2);
            if (LOCAL) return 0.5 * (up - dn) - uz;
            return conj(uz + 0.5 * (up - dn));
        };
        const int perd = pack ? rc : 16 / ND;   // densities of a tile
        const int d0 = (im ? j - NB : j) * perd;
        for (int q = tid; q < nh * 16; q += 256) {
            const int ii = q >> 4, r = q & 15;
            if (r >= perd || d0 + r >= rc) continue;
            int n = (int)sqrt(2.0 * ii);
            while (n * (n + 1) / 2 > ii) --n;
            while ((n + 1) * (n + 2) / 2 <= ii) ++n;
            const int m = ii - n * (n + 1) / 2;
            cplx x = coef(n, m, r * ND), y = {0, 0};
            if (pack) {
                y = coef(n, m, 8 + r * ND);
            } else if (im) {
                y = x;
                x = {0, 0};
            }
            const cplx vp = {x.x - y.y, x.y + y.x};
            const double sg = (m & 1) ? -1.0 : 1.0;
            const cplx vm = {sg * (x.x + y.y), sg * (y.x - x.y)};
            double *dp = o + 2 * ((long)IDX(n, m) * nr + r0 + d0 + r);
            double *dm = o + 2 * ((long)IDX(n, -m) * nr + r0 + d0 + r);
            const bool add = LOCAL || im;
            stc(dp, add ? ldc(dp) + vp : vp);
            if (m > 0) stc(dm, add ? ldc(dm) + vm : vm);
        }
        __syncthreads();
    }
}

// child offset index bits: bit d set = upper half in dimension d
__device__ __forceinline__ const double *child_tab(const KD &kd, int ci)
{
    return kd.tab_ch + 2L * ci * (kd.pmax + 1) * (kd.pmax + 1);
}

// M2M into parents of level lvp: thread per (parent, coefficient)
template <int NRC>
__global__ void k3_m2m(KD kd, TD t, int lvp, int i0, int i1, const int *spb, double *mpole,
                       const int *allreal)
{
    if (allreal && *allreal) return;  // k3_trans_real's case
    const long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int ncp = kd.ncl[lvp];
    const long nthr = (long)(i1 - i0) * ncp;
    if (gid >= nthr) return;
    const int P = spb[i0 + (int)(gid / ncp)];
    const int j = (int)(gid % ncp);
    int n, m;
    nm_of(j, n, m);
    const int lvc = lvp + 1;
    const int pc = kd.order[lvc];
    const double hc = kd.h[lvc];
    cplx acc[NRC];
#pragma unroll
    for (int q = 0; q < NRC; ++q) acc[q] = {0, 0};
    for (int ci = 0; ci < 8; ++ci) {
        const int C = t.child[(size_t)ci * t.nboxes + P];
        if (C < 0 || t.scumul[C] == 0) continue;
        const double *a = mpole + ecoef_off(kd, C, lvc);
        const double *U = child_tab(kd, ci);
        // conj(Y_k^l(c_child - c_parent)) = conj(U_k^l) hc^k
        double hk = 1.0;
        for (int k = 0; k <= n; ++k) {
            const int nn = n - k;
            if (nn <= pc) {
                for (int l = -k; l <= k; ++l) {
                    const int mm = m - l;
                    if (mm < -nn || mm > nn) continue;
                    const cplx wgt = hk * conj(ldc(U + 2 * IDX(k, l)));
#pragma unroll
                    for (int q = 0; q < NRC; ++q)
                        if (q < kd.rc) acc[q] += wgt * ldcn(kd, a, IDX(nn, mm), kd.r0 + q);
                }
            }
            hk *= hc;
        }
    }
    double *o = mpole + ecoef_off(kd, P, lvp) + 2L * j * kd.nr;
#pragma unroll
    for (int q = 0; q < NRC; ++q)
        if (q < kd.rc) stc(o + 2 * (kd.r0 + q), acc[q]);
}

// L2L into ttp boxes of level lv: thread per (box, coefficient), accumulating
template <int NRC>
__global__ void k3_l2l(KD kd, TD t, int lv, int i0, int i1, const int *ttp, double *local,
                       const int *allreal)
{
    if (allreal && *allreal) return;  // k3_trans_real's case
    const long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int nc = kd.ncl[lv];
    const long nthr = (long)(i1 - i0) * nc;
    if (gid >= nthr) return;
    const int Bx = ttp[i0 + (int)(gid / nc)];
    const int j = (int)(gid % nc);
    int a, b;
    nm_of(j, a, b);
    const int Pp = t.parent[Bx];
    const int lvp = lv - 1;
    const int pp = kd.order[lvp];
    const double hc = kd.h[lv];
    // child index of Bx within its parent from coordinates
    int ci = 0;
    ci |= (t.coords[Bx] & 1);
    ci |= (t.coords[(size_t)t.nboxes + Bx] & 1) << 1;
    ci |= (t.coords[2 * (size_t)t.nboxes + Bx] & 1) << 2;
    const double *U = child_tab(kd, ci);
    const double *L = local + ecoef_off(kd, Pp, lvp);
    cplx acc[NRC];
#pragma unroll
    for (int q = 0; q < NRC; ++q) acc[q] = {0, 0};
    double hj = 1.0;
    for (int jj = 0; a + jj <= pp; ++jj) {
        for (int i = -jj; i <= jj; ++i) {
            const int mm = b + i;
            if (mm < -(a + jj) || mm > a + jj) continue;
            const cplx wgt = hj * conj(ldc(U + 2 * IDX(jj, i)));
#pragma unroll
            for (int q = 0; q < NRC; ++q)
                if (q < kd.rc) acc[q] += wgt * ldcn(kd, L, IDX(a + jj, mm), kd.r0 + q);
        }
        hj *= hc;
    }
    store_add<NRC>(kd, local + ecoef_off(kd, Bx, lv) + 2L * j * kd.nr, acc);
}

constexpr int M2L_THREADS = 64;

// M2L: one 64-lane block per ttp box with list-2 entries; NO output
// coefficients per lane, NRC right-hand sides; LDS holds the rescaled source
// multipole [ncl][NRC]
template <int NO, int NRC>
__global__ void __launch_bounds__(M2L_THREADS) k3_m2l(KD kd, TD t, const int *ttp,
                                                      const int *starts, const int *lists,
                                                      const double *mpole, double *local)
{
    extern __shared__ double Ms[];
    const int i = blockIdx.x;
    const int e0 = starts[i], e1 = starts[i + 1];
    if (e0 == e1) return;
    const int Bx = ttp[i];
    const int lv = t.level[Bx];
    const int p = kd.order[lv];
    const int nc = kd.ncl[lv];
    const double h = kd.h[lv];
    const double ih = 1.0 / h;
    const int W = kd.W, S1 = 2 * W + 1;
    const int tn = kd.tabn;
    const int bx = t.coords[Bx], by = t.coords[(size_t)t.nboxes + Bx],
              bz = t.coords[2 * (size_t)t.nboxes + Bx];
    cplx acc[NO][NRC];
#pragma unroll
    for (int r = 0; r < NO; ++r)
#pragma unroll
        for (int q = 0; q < NRC; ++q) acc[r][q] = {0, 0};
    for (int e = e0; e < e1; ++e) {
        const int A = lists[e];
        const int dx = bx - t.coords[A] + W;
        const int dy = by - t.coords[(size_t)t.nboxes + A] + W;
        const int dz = bz - t.coords[2 * (size_t)t.nboxes + A] + W;
        // list 2 offsets satisfy |delta_i| <= 2 nsep + 1 by construction
        if ((unsigned)dx >= (unsigned)S1 || (unsigned)dy >= (unsigned)S1 ||
            (unsigned)dz >= (unsigned)S1)
            continue;
        const double *a = mpole + ecoef_off(kd, A, lv);
        __syncthreads();
        for (int qq = threadIdx.x; qq < nc; qq += M2L_THREADS) {
            int n, m;
            nm_of(qq, n, m);
            double s = 1.0;
            for (int k = 0; k < n; ++k) s *= ih;
#pragma unroll
            for (int q = 0; q < NRC; ++q)
                stc(Ms + 2 * (qq * NRC + q),
                    q < kd.rc ? s * ldcn(kd, a, qq, kd.r0 + q) : cplx{0, 0});
        }
        __syncthreads();
        const double *T = kd.tab_m2l + 2L * ((dx * S1 + dy) * S1 + dz) * tn * tn;
#pragma unroll
        for (int r = 0; r < NO; ++r) {
            const int qo = threadIdx.x + r * M2L_THREADS;
            if (qo < nc) {
                int k, l;
                nm_of(qo, k, l);
                for (int n = 0; n <= p; ++n) {
                    const int N = n + k;
                    for (int m = -n; m <= n; ++m) {
                        const int M = m + l;
                        if (M < -N || M > N) continue;
                        const cplx tv = ldc(T + 2 * IDX(N, M));
#pragma unroll
                        for (int q = 0; q < NRC; ++q)
                            acc[r][q] += ldc(Ms + 2 * (IDX(n, m) * NRC + q)) * tv;
                    }
                }
            }
        }
    }
#pragma unroll
    for (int r = 0; r < NO; ++r) {
        const int qo = threadIdx.x + r * M2L_THREADS;
        if (qo < nc) {
            int k, l;
            nm_of(qo, k, l);
            double s = (k & 1) ? -ih : ih;  // (-1)^k h^{-k-1}
            for (int kk = 0; kk < k; ++kk) s *= ih;
            cplx v[NRC];
#pragma unroll
            for (int q = 0; q < NRC; ++q) v[q] = s * acc[r][q];
            store_add<NRC>(kd, local + ecoef_off(kd, Bx, lv) + 2L * qo * kd.nr, v);
        }
    }
}

// Box translations on the FP64 matrix cores.  Real strengths give M_n^{-m} = (-1)^m conj(M_n^m) and L_n^{-m} = (-1)^m
// conj(L_n^m) for every multipole and local, so a translation out = A in
// forms only the output rows i = (k, l), l >= 0, from the input columns
// j = (n, m), m >= 0: out_i = sum_j A1 a_j + A2 conj(a_j) with A1 = A(i, j)
// and A2 = (-1)^m A(i, (n, -m)) (0 for m = 0), a real-linear map
//   [Re out]   [A1r + A2r   A2i - A1i] [Re a]
//   [Im out] = [A1i + A2i   A1r - A2r] [Im a]
// of (P+1)(P+2) rows and columns -- about a third of the real products of
// the complex (P+1)^2 square.  The operator of one entry, read from a table
// staged in LDS:
//   M2L (OPK 0)  A = T_{n+k}^{m+l}(delta), the unit-offset irregular
//                harmonics of the list-2 offset; B scaled h^-n, output
//                (-1)^k h^-(k+1); entries: the list-2 boxes
//   M2M (OPK 1)  A = conj(Y_{k-n}^{l-m}(child offset)) for n <= k (unit
//                child size); B scaled hc^-n, output hc^k; entries: the
//                children, output the parent (stored)
//   L2L (OPK 2)  A = conj(Y_{n-k}^{m-l}(child offset)) for n >= k; B (the
//                parent's locals) scaled hc^n, output hc^-k; entry: the
//                parent, output the box (added)
// (row i = (k, l), column j = (n, m); for M2M and L2L the tiles on the zero
// side of n = k are skipped).  Rows and columns interleave (re, im) of each
// coefficient (row 2i + pr, column 2j + pk).  A block per output box of one
// level and 16 NCT right-hand sides.  Per entry the table and the input
// box's m >= 0 coefficients (scaled, split into re / im rows) are staged in
// LDS; the next entry's are loaded into registers while the current one is
// contracted.  The K-steps of each entry are dealt round-robin to the four
// waves, each wave holding every row tile; the waves' sums are added in LDS
// at the end and the epilogue writes row (k, l) and its mirror (k, -l).
//
// SPLIT (M2L): strengths of any kind, two columns to a density.  Every expansion is
// M = Mr + i Mi with both parts conjugate-symmetric, Mr = (M + J M)/2, Mi =
// (M - J M)/(2i), (J M)_n^m = (-1)^m conj(M_n^{-m}); the columns of Mr and Mi
// are translated as real densities and the epilogue adds Lr + i Li.  One to
// three densities take this route too: 2 of 16 columns filled, yet a third of
// the serial vector kernel's time (M2M and L2L of few densities stay on it:
// few boxes a level, and there the vector kernels are twice as fast): 38170
// list-2 pairs at order 10, one density, 5.3 -> 1.7 ms.
//
// With allreal given the kernel runs only when *allreal is set, SPLIT only
// when it is not; without, the caller has stated which.
//
// M2L's operand gather: T_{n+k}^{m+l} lies at n^2 + n + m + (k^2 + k + l) +
// 2nk, so that a row tile costs three integer operations a K-step instead of
// twenty (the masks of the general form are not needed: rows and columns
// beyond the last meet zeros of B or are not stored).  32 real densities at
// order 8, 875275 pairs (495 GFLOP executed): 17.6 -> 12.9 ms, 38 TFLOP/s.
constexpr int TR3_ECH = 256;  // entries whose offsets are staged at once

__host__ __device__ constexpr int tri_n(int j)  // n of triangular index j
{
    int n = 0;
    while ((n + 1) * (n + 2) / 2 <= j) ++n;
    return n;
}

template <int OPK, int P, int NCT, bool SPLIT>
__global__ void __launch_bounds__(256)
k3_trans_real(KD kd, TD t, int i0, const int *boxes, const int *starts,
              const int *lists, const double *in, double *out, const int *allreal)
{
    constexpr int R = (P + 1) * (P + 2) / 2;      // coefficients with m >= 0
    constexpr int R2 = 2 * R;                     // real rows / columns
    constexpr int RT = (R2 + 15) / 16;            // row tiles
    constexpr int KS = (R2 + 3) / 4;              // K-steps
    // high orders split the row tiles over RG groups of waves (fewer
    // accumulators per wave) and the K-steps over the KG waves of a group
    constexpr int RG = (OPK == 0 && P >= 10) ? 2 : 1, KG = 4 / RG;
    constexpr int RTW = (RT + RG - 1) / RG;       // row tiles per wave
    constexpr int RC = 16 * NCT;                  // right-hand sides per block
    constexpr int TNL = OPK == 0 ? (2 * P + 1) * (2 * P + 1) : (P + 1) * (P + 1);
    constexpr int NT = (2 * TNL + 255) / 256;       // table doubles per thread
    constexpr int NB = (R * RC + 255) / 256;        // (coefficient, rhs) pairs per thread
    // staging area, reused for the reduction at the end
    constexpr int LDSN = (2 * TNL + R2 * RC) > RT * 16 * 17 ? (2 * TNL + R2 * RC)
                                                            : RT * 16 * 17;
    __shared__ double lds[LDSN];
    __shared__ double bsc[P + 1], osc[P + 1];
    __shared__ short jn[R];
    __shared__ int etab[TR3_ECH];
    __shared__ long eoff[TR3_ECH];
    __shared__ int nent;
    double *Ts = lds, *Bs = lds + 2 * TNL;
    if (allreal && (*allreal != 0) == SPLIT) return;
    const int i = i0 + blockIdx.x;
    const int Bx = boxes[i];
    const int lv = t.level[Bx];
    // the entry range: list 2, the children, or the parent
    int e0 = 0, e1 = 0;
    if (OPK == 0) {
        e0 = starts[i];
        e1 = starts[i + 1];
        if (e0 == e1) return;
    } else if (OPK == 1) {
        e1 = 8;
    } else {
        e1 = 1;
    }
    const int W = kd.W, S1 = 2 * W + 1, tn = kd.tabn;
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
    const int col = lane & 15, kr = lane >> 4;
    const int rg = wv / KG, kg = wv % KG;
    const int rc = kd.rc, r0 = kd.r0, nr = kd.nr;
    // the level of the input boxes and the scalings
    const int lin = OPK == 0 ? lv : (OPK == 1 ? lv + 1 : lv - 1);
    if (tid <= P) {
        const double h = OPK == 0 ? kd.h[lv] : (OPK == 1 ? kd.h[lv + 1] : kd.h[lv]);
        const double ih = 1.0 / h;
        double pw = 1.0, ipw = 1.0;
        for (int k = 0; k < tid; ++k) {
            pw *= h;
            ipw *= ih;
        }
        if (OPK == 0) {
            bsc[tid] = ipw;
            osc[tid] = ((tid & 1) ? -ipw : ipw) * ih;
        } else if (OPK == 1) {
            bsc[tid] = ipw;
            osc[tid] = pw;
        } else {
            bsc[tid] = pw;
            osc[tid] = ipw;
        }
    }
    for (int j = tid; j < R; j += 256) jn[j] = (short)tri_n(j);
    // this lane's A rows: (k, l, pr) of row (rg RTW + rt) 16 + col
    int rowk[RTW], rowl[RTW], rowpr[RTW];
#pragma unroll
    for (int rt = 0; rt < RTW; ++rt) {
        const int rho = (rg * RTW + rt) * 16 + col;
        const int ii = rho >> 1;
        const int k = tri_n(ii);
        rowk[rt] = rho < R2 ? k : -1;
        rowl[rt] = ii - k * (k + 1) / 2;
        rowpr[rt] = rho & 1;
        if (OPK == 0) {
            // the row's share of the table offset, and 2k, in bytes
            const int kk = rho < R2 ? k : 0, ll = rho < R2 ? rowl[rt] : 0;
            rowk[rt] = 16 * (kk * kk + kk + ll) + ((col ^ kr) & 1 ? 8 : 0);
            rowl[rt] = 32 * kk;
        }
    }
    // M2L: the sign of column part kr % 2 (re, im) in row part col % 2
    const double sneg = (col & 1) == 0 && (kr & 1) ? -1.0 : 1.0;
    const int bx = t.coords[Bx], by = t.coords[(size_t)t.nboxes + Bx],
              bz = t.coords[2 * (size_t)t.nboxes + Bx];
    // the staged data of an entry: table doubles and (re, im) of the B pairs;
    // the entries' table and coefficient offsets come from LDS (filled per
    // chunk of TR3_ECH entries), so the loads of the next entry depend on no
    // global read and overlap the current entry's products
    double tr[NT], br[NB][2];
    auto fetch = [&](int ee) -> bool {
        const int tix = etab[ee];
        if (tix < 0) return false;  // uniform over the block
        const double *T = OPK == 0 ? kd.tab_m2l + 2L * tix * tn * tn
                                   : kd.tab_ch + 2L * tix * (kd.pmax + 1) * (kd.pmax + 1);
#pragma unroll
        for (int u = 0; u < NT; ++u) {
            const int q = tid + 256 * u;
            // the child table holds Y: stage conj(Y) (flip the imaginary parts)
            tr[u] = q < 2 * TNL ? ((OPK != 0 && (q & 1)) ? -T[q] : T[q]) : 0.0;
        }
        const double *a = in + eoff[ee];
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            const int f = tid + 256 * u;
            const int j = f / RC, r = f % RC;
            br[u][0] = br[u][1] = 0.0;
            if (f < R * RC && (SPLIT ? r >> 1 : r) < rc) {
                const int n = jn[j];
                const int m = j - n * (n + 1) / 2;
                const long i1 = (long)(n * n + n + m) * nr + r0;
                if (SPLIT) {
                    const double *z = a + 2 * (i1 + (r >> 1)), *y = z - 4L * m * nr;
                    const double sg = (m & 1) ? -1.0 : 1.0;
                    if (r & 1) {
                        br[u][0] = 0.5 * (z[1] + sg * y[1]);
                        br[u][1] = -0.5 * (z[0] - sg * y[0]);
                    } else {
                        br[u][0] = 0.5 * (z[0] + sg * y[0]);
                        br[u][1] = 0.5 * (z[1] - sg * y[1]);
                    }
                } else {
                    br[u][0] = a[2 * (i1 + r)];
                    br[u][1] = a[2 * (i1 + r) + 1];
                }
            }
        }
        return true;
    };
    f3_d4 acc[RTW][NCT];
#pragma unroll
    for (int rt = 0; rt < RTW; ++rt)
#pragma unroll
        for (int c = 0; c < NCT; ++c) acc[rt][c] = f3_d4{0, 0, 0, 0};
    int step = 0;  // K-steps dealt so far (rotates the round-robin start)
    for (int cb = e0; cb < e1; cb += TR3_ECH) {
        __syncthreads();  // the previous chunk's entries consumed (bsc, jn written)
        if (OPK == 0) {
            const int cn = min(TR3_ECH, e1 - cb);
            for (int q = tid; q < cn; q += 256) {
                const int A = lists[cb + q];
                const int dx = bx - t.coords[A] + W;
                const int dy = by - t.coords[(size_t)t.nboxes + A] + W;
                const int dz = bz - t.coords[2 * (size_t)t.nboxes + A] + W;
                const bool ok = (unsigned)dx < (unsigned)S1 && (unsigned)dy < (unsigned)S1 &&
                                (unsigned)dz < (unsigned)S1;
                etab[q] = ok ? (dx * S1 + dy) * S1 + dz : -1;
                eoff[q] = ecoef_off(kd, A, lin);
            }
            if (tid == 0) nent = cn;
        } else if (OPK == 1) {
            // the nonempty children, octant ci = child slot ci
            if (tid == 0) {
                int c = 0;
                for (int ci = 0; ci < 8; ++ci) {
                    const int C = t.child[(size_t)ci * t.nboxes + Bx];
                    if (C < 0 || t.scumul[C] == 0) continue;
                    etab[c] = ci;
                    eoff[c] = ecoef_off(kd, C, lin);
                    ++c;
                }
                nent = c;
            }
        } else {
            if (tid == 0) {
                etab[0] = (bx & 1) | ((by & 1) << 1) | ((bz & 1) << 2);
                eoff[0] = ecoef_off(kd, t.parent[Bx], lin);
                nent = 1;
            }
        }
        __syncthreads();
        const int cn = nent;
        bool have = cn > 0 ? fetch(0) : false;
        for (int ee = 0; ee < cn; ++ee) {
            __syncthreads();  // the previous entry's staging consumed
            if (have) {
#pragma unroll
                for (int u = 0; u < NT; ++u) {
                    const int q = tid + 256 * u;
                    if (q < 2 * TNL) Ts[q] = tr[u];
                }
#pragma unroll
                for (int u = 0; u < NB; ++u) {
                    const int f = tid + 256 * u;
                    if (f < R * RC) {
                        const int j = f / RC, r = f % RC;
                        const double sc = bsc[jn[j]];
                        Bs[(2 * j) * RC + r] = sc * br[u][0];
                        Bs[(2 * j + 1) * RC + r] = sc * br[u][1];
                    }
                }
            }
            const bool cur = have;
            __syncthreads();
            have = ee + 1 < cn ? fetch(ee + 1) : false;
            if (!cur) continue;
            if (OPK == 0) {
                for (int ks = kg; ks < KS; ks += KG) {
                    const int kap = ks * 4 + kr;  // B row / A column
                    const bool kin = kap < R2;
                    const int j = kin ? kap >> 1 : 0;
                    double b[NCT];
#pragma unroll
                    for (int c = 0; c < NCT; ++c)
                        b[c] = kin ? Bs[kap * RC + c * 16 + col] : 0.0;
                    const int n = jn[j], m = j - n * (n + 1) / 2;
                    const int cb = 16 * (n * n + n + m);   // bytes
                    const double s2 = m == 0 ? 0.0 : ((m + kr) & 1) ? -sneg : sneg;
                    const char *tb = reinterpret_cast<const char *>(Ts);
                    double c1[RTW], c2[RTW];
#pragma unroll
                    for (int rt = 0; rt < RTW; ++rt) {
                        const int o1 = rowk[rt] + cb + n * rowl[rt];
                        c1[rt] = *reinterpret_cast<const double *>(tb + o1);
                        c2[rt] = *reinterpret_cast<const double *>(tb + o1 - 32 * m);
                    }
#pragma unroll
                    for (int rt = 0; rt < RTW; ++rt) {
                        const double v = s2 * c2[rt] + sneg * c1[rt];
                        if (rg * RTW + rt < RT) {
#pragma unroll
                            for (int c = 0; c < NCT; ++c)
                                acc[rt][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                                    v, b[c], acc[rt][c], 0, 0, 0);
                        }
                    }
                }
                continue;
            }
            for (int ks = (kg - step + KG * 4) % KG; ks < KS; ks += KG) {
                const int kap = ks * 4 + kr;  // B row / A column
                const int j = kap >> 1, pk = kap & 1;
                const bool kin = kap < R2;
                int n = 0, m = 0;
                double b[NCT];
#pragma unroll
                for (int c = 0; c < NCT; ++c) b[c] = 0.0;
                if (kin) {
                    n = jn[j];
                    m = j - n * (n + 1) / 2;
#pragma unroll
                    for (int c = 0; c < NCT; ++c) b[c] = Bs[kap * RC + c * 16 + col];
                }
                const double sm = (m == 0) ? 0.0 : ((m & 1) ? -1.0 : 1.0);
                // the K-step's column orders (uniform): M2M and L2L skip the
                // row tiles on the zero side of n = k
                const int nlo = tri_n(min(2 * ks, R - 1)), nhi = tri_n(min(2 * ks + 1, R - 1));
                // branch-free gather: every row tile's two table reads are
                // issued together (invalid entries read 0 and are masked),
                // then the matrix products follow
                double c1[RTW], c2[RTW];
                bool v1[RTW], v2[RTW];
#pragma unroll
                for (int rt = 0; rt < RTW; ++rt) {
                    const int k = rowk[rt], l = rowl[rt];
                    const int off = rowpr[rt] == pk ? 0 : 1;
                    int i1, i2;
                    bool ok1, ok2;
                    if (OPK == 1) {
                        const int K = k - n, base = K * K + K;
                        i1 = base + l - m;
                        i2 = base + l + m;
                        ok1 = kin && k >= 0 && K >= 0 && l - m <= K && m - l <= K;
                        ok2 = kin && k >= 0 && K >= 0 && l + m <= K;
                    } else {
                        const int K = n - k, base = K * K + K;
                        i1 = base + m - l;
                        i2 = base - m - l;
                        ok1 = kin && k >= 0 && K >= 0 && m - l <= K && l - m <= K;
                        ok2 = kin && k >= 0 && K >= 0 && m + l <= K;
                    }
                    v1[rt] = ok1;
                    v2[rt] = ok2;
                    c1[rt] = Ts[ok1 ? 2 * i1 + off : 0];
                    c2[rt] = Ts[ok2 ? 2 * i2 + off : 0];
                }
                const double s2 = pk ? -sm : sm;
#pragma unroll
                for (int rt = 0; rt < RTW; ++rt) {
                    // row orders of the tile
                    const int rtg = rg * RTW + rt;
                    const int rklo = tri_n(min(8 * rtg, R - 1)),
                              rkhi = tri_n(min(8 * rtg + 7, R - 1));
                    const bool live =
                        rtg < RT && (OPK == 1 ? nlo <= rkhi : nhi >= rklo);
                    double v = (v1[rt] ? c1[rt] : 0.0) + s2 * (v2[rt] ? c2[rt] : 0.0);
                    v = (rowpr[rt] == 0 && pk == 1) ? -v : v;
                    if (live) {
#pragma unroll
                        for (int c = 0; c < NCT; ++c)
                            acc[rt][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(v, b[c], acc[rt][c],
                                                                               0, 0, 0);
                    }
                }
            }
            step = (step + KS) % KG;
        }
    }
    // the sums of a row group's waves, one 16-column tile at a time (in the
    // staging area): D register j of lane i is row 4 j + i / 16, column
    // i % 16 of its tile
    double(*red)[17] = reinterpret_cast<double(*)[17]>(lds);
    double *o = out + ecoef_off(kd, Bx, lv);
#pragma unroll
    for (int c = 0; c < NCT; ++c) {
        for (int w = 0; w < KG; ++w) {
            __syncthreads();
            if (kg == w) {
#pragma unroll
                for (int rt = 0; rt < RTW; ++rt) {
                    const int rtg = rg * RTW + rt;
                    if (rtg < RT) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            double &d = red[rtg * 16 + 4 * j + kr][col];
                            d = (w == 0 ? 0.0 : d) + acc[rt][c][j];
                        }
                    }
                }
            }
        }
        __syncthreads();
        constexpr int DC = SPLIT ? 8 : 16;   // densities of a tile
        for (int q = tid; q < R * DC; q += 256) {
            const int ii = q / DC, cc = q % DC;
            const int r = c * DC + cc;
            if (r >= rc) continue;
            const int k = jn[ii];
            const int l = ii - k * (k + 1) / 2;
            const double sc = osc[k], sl = (l & 1) ? -sc : sc;
            const int cx = SPLIT ? 2 * cc : cc;
            cplx v = {red[2 * ii][cx], red[2 * ii + 1][cx]};
            cplx u = conj(v);                   // (k, -l): (-1)^l of it
            if (SPLIT) {
                const cplx y = {red[2 * ii][cx + 1], red[2 * ii + 1][cx + 1]};
                v += cplx{-y.y, y.x};
                u += cplx{y.y, y.x};
            }
            double *dst = o + 2 * ((long)(k * k + k + l) * nr + r0 + r);
            double *dm = o + 2 * ((long)(k * k + k - l) * nr + r0 + r);
            stc(dst, OPK == 1 ? sc * v : ldc(dst) + sc * v);
            if (l > 0) stc(dm, OPK == 1 ? sl * u : ldc(dm) + sl * u);
        }
    }
}

// P2P (MODE 0, list 1), M2P (1, list 3), L2P (2) for non-QBX targets, a
// wavefront per target box: L2P, and the others where the geometry's work
// units are those of another traversal
template <int MODE, int NRC>
__global__ void __launch_bounds__(64) k3_eval_targets(KD kd, TD t, int ntb, const int *tboxes,
                                                      const int *starts, const int *lists,
                                                      const int *fstart, const int *fcount,
                                                      const int *unfilt, const double *tgt,
                                                      int nt, const double *src, int ns,
                                                      const double *str, const double *nrm,
                                                      const double *expn, double *pot)
{
    const int it = blockIdx.x;
    if (it >= ntb) return;
    const int B = tboxes[it];
    const int f0 = fstart[B], nf = fcount[B];
    if (nf == 0) return;
    const int lane = threadIdx.x;
    if (MODE == 2) {
        const int lv = t.level[B];
        const v3 c = boxc(t, B);
        for (int f = f0 + lane; f < f0 + nf; f += 64) {
            const int ti = unfilt[f];
            cplx v[NRC];
#pragma unroll
            for (int q = 0; q < NRC; ++q) v[q] = {0, 0};
            sum_regular_conj_n<NRC>(kd, expn + ecoef_off(kd, B, lv), kd.order[lv],
                                    sub(ld3(tgt, nt, ti), c), v);
#pragma unroll
            for (int q = 0; q < NRC; ++q) v[q] = INV4PI * v[q];
            store_add<NRC>(kd, pot + 2 * (size_t)ti * kd.nr, v);
        }
        return;
    }
    int G = 64;
    while (G > 1 && G * nf > 64) G >>= 1;
    const int tpr = 64 / G;
    const int tsub = lane / G, sub_ = lane % G;
    const int e0 = starts[it], e1 = starts[it + 1];
    for (int base = 0; base < nf; base += tpr) {
        const bool active = base + tsub < nf;
        int ti = 0;
        cplx acc[NRC];
#pragma unroll
        for (int q = 0; q < NRC; ++q) acc[q] = {0, 0};
        if (active) {
            ti = unfilt[f0 + base + tsub];
            const v3 tp = ld3(tgt, nt, ti);
            if (MODE == 0) {
                for (int e = e0; e < e1; ++e) {
                    const int Sb = lists[e];
                    const int s0 = t.sstart[Sb], s1 = s0 + t.scount[Sb];
                    for (int s = s0 + sub_; s < s1; s += G) {
                        const v3 nu = kd.dip ? ld3(nrm, ns, s) : v3{0, 0, 0};
                        const double g = p2p_value(kd, ld3(src, ns, s), nu, tp);
#pragma unroll
                        for (int q = 0; q < NRC; ++q)
                            if (q < kd.rc) acc[q] += g * ldq(kd, str, s, kd.r0 + q);
                    }
                }
            } else {
                for (int e = e0 + sub_; e < e1; e += G) {
                    const int D = lists[e];
                    const int lv = t.level[D];
                    sum_irregular_n<NRC>(kd, expn + ecoef_off(kd, D, lv), kd.order[lv],
                                         sub(tp, boxc(t, D)), acc);
                }
#pragma unroll
                for (int q = 0; q < NRC; ++q) acc[q] = INV4PI * acc[q];
            }
        }
#pragma unroll
        for (int q = 0; q < NRC; ++q)
            for (int m = G / 2; m >= 1; m >>= 1) {
                acc[q].x += __shfl_xor(acc[q].x, m);
                acc[q].y += __shfl_xor(acc[q].y, m);
            }
        if (active && sub_ == 0) store_add<NRC>(kd, pot + 2 * (size_t)ti * kd.nr, acc);
    }
}

// P2P (MODE 0, list 1) and M2P (1, list 3) over the geometry's work units
// (unit_plan): G lanes per target, each walking every G-th source of a list-1
// box or every G-th list-3 box, reduced by shuffles.  A target in a coarse
// box against all of a surface's sources is a long walk: with a wavefront per
// target box the 3001 loose points around 46080 sources kept a few
// wavefronts busy for 32 ms (P2P) and 2.1 ms (M2P); over units 0.61 and
// 0.18 ms, one target's walk on 64 lanes.
template <int MODE, int NRC>
__global__ void __launch_bounds__(64) k3_eval_units(KD kd, TD t, const int *ubox, const int *ut0,
                                                    const int *box_g, const int *tboxes,
                                                    const int *starts, const int *lists,
                                                    const int *fstart, const int *fcount,
                                                    const int *unfilt, const double *tgt, int nt,
                                                    const double *src, int ns,
                                                    const double *str, const double *nrm,
                                                    const double *expn, double *pot)
{
    const int u = blockIdx.x;
    const int it = ubox[u];
    const int B = tboxes[it];
    const int G = box_g[it];
    const int lane = threadIdx.x;
    const int tsub = lane / G, sub_ = lane & (G - 1);
    const int tl = ut0[u] + tsub;
    const bool active = tl < fcount[B];
    const int ti = active ? unfilt[fstart[B] + tl] : 0;
    const v3 tp = active ? ld3(tgt, nt, ti) : v3{0, 0, 0};
    cplx acc[NRC];
#pragma unroll
    for (int q = 0; q < NRC; ++q) acc[q] = {0, 0};
    const int e0 = starts[it], e1 = starts[it + 1];
    if (active && MODE == 0) {
        for (int e = e0; e < e1; ++e) {
            const int Sb = lists[e];
            const int s0 = t.sstart[Sb], s1 = s0 + t.scount[Sb];
            for (int s = s0 + sub_; s < s1; s += G) {
                const v3 nu = kd.dip ? ld3(nrm, ns, s) : v3{0, 0, 0};
                const double g = p2p_value(kd, ld3(src, ns, s), nu, tp);
#pragma unroll
                for (int q = 0; q < NRC; ++q)
                    if (q < kd.rc) acc[q] += g * ldq(kd, str, s, kd.r0 + q);
            }
        }
    } else if (active) {
        for (int e = e0 + sub_; e < e1; e += G) {
            const int D = lists[e];
            const int lv = t.level[D];
            sum_irregular_n<NRC>(kd, expn + ecoef_off(kd, D, lv), kd.order[lv],
                                 sub(tp, boxc(t, D)), acc);
        }
#pragma unroll
        for (int q = 0; q < NRC; ++q) acc[q] = INV4PI * acc[q];
    }
#pragma unroll
    for (int q = 0; q < NRC; ++q)
        for (int m = G >> 1; m >= 1; m >>= 1) {
            acc[q].x += __shfl_xor(acc[q].x, m);
            acc[q].y += __shfl_xor(acc[q].y, m);
        }
    if (active && sub_ == 0) store_add<NRC>(kd, pot + 2 * (size_t)ti * kd.nr, acc);
}

// ---- QBX stages
template <int PQ, int NRC>
struct QAcc {
    cplx v[NRC][(PQ + 1) * (PQ + 1)];
};

template <int PQ, int NRC>
__device__ void qbx_store(const KD &kd, double *qexp, int c, const QAcc<PQ, NRC> &A,
                          int accumulate)
{
    constexpr int NQ = (PQ + 1) * (PQ + 1);
    double *o = qexp + 2 * (size_t)c * NQ * kd.nr;
#pragma unroll
    for (int i = 0; i < NQ; ++i)
#pragma unroll
        for (int q = 0; q < NRC; ++q)
            if (q < kd.rc) {
                double *p = o + 2 * ((long)i * kd.nr + kd.r0 + q);
                cplx v = A.v[q][i];
                if (accumulate) v += ldc(p);
                stc(p, v);
            }
}

// P2QBXL over balanced work units (unit_plan over the global QBX centers of
// each target box): the unit's TG centers take G lanes apiece; the box's
// list-1 sources are staged through LDS in chunks (positions, normals,
// strengths, coalesced) and each center's lanes split a chunk; the expansions
// are reduced by shuffles within the G-lane groups.
template <int NRC>
struct P2QTile3 {
    static constexpr int CH = NRC == 1 ? 256 : 64;
};

template <int PQ, int NRC>
__global__ void __launch_bounds__(64) k3_p2qbxl(KD kd, TD t, const int *ubox, const int *ut0,
                                                const int *box_g, const int *gcs,
                                                const int *gcl, const double *ctr, int nc,
                                                const int *l1s, const int *l1l,
                                                const double *src, int ns, const double *str,
                                                const double *nrm, double *qexp, int accumulate)
{
    constexpr int NQ = (PQ + 1) * (PQ + 1);
    constexpr int CH = P2QTile3<NRC>::CH;
    __shared__ double sx[CH], sy[CH], sz[CH], snx[CH], sny[CH], snz[CH];
    __shared__ double sq[CH * 2 * NRC];
    const int u = blockIdx.x;
    const int it = ubox[u];
    const int G = box_g[it];
    const int lane = threadIdx.x;
    const int tsub = lane / G, sub = lane & (G - 1);
    const int cl = ut0[u] + tsub;
    const bool active = cl < gcs[it + 1] - gcs[it];
    const bool dip = kd.dip;
    const int rc = kd.rc, r0 = kd.r0, nr = kd.nr;
    int c = 0;
    v3 cc = {0, 0, 0};
    if (active) {
        c = gcl[gcs[it] + cl];
        cc = ld3(ctr, nc, c);
    }
    QAcc<PQ, NRC> A;
#pragma unroll
    for (int q = 0; q < NRC; ++q)
#pragma unroll
        for (int i = 0; i < NQ; ++i) A.v[q][i] = {0, 0};

    auto flush = [&](int n) {
        __syncthreads();
        if (active) {
            for (int j = sub; j < n; j += G) {
                const v3 d = {sx[j] - cc.x, sy[j] - cc.y, sz[j] - cc.z};
                cplx qs[NRC];
#pragma unroll
                for (int q = 0; q < NRC; ++q)
                    qs[q] = q < rc ? cplx{sq[2 * (j * NRC + q)], sq[2 * (j * NRC + q) + 1]}
                                   : cplx{0, 0};
                if (!dip) {
                    cplx T[NQ];
                    the_table<PQ>(d, T);
#pragma unroll
                    for (int i = 0; i < NQ; ++i)
#pragma unroll
                        for (int q = 0; q < NRC; ++q) A.v[q][i] += qs[q] * T[i];
                } else {
                    constexpr int P1 = PQ + 1;
                    cplx T[(P1 + 1) * (P1 + 1)];
                    the_table<P1>(d, T);
                    const cplx nmn = {snx[j], -sny[j]}, npl = {snx[j], sny[j]};
                    const double nz = snz[j];
#pragma unroll
                    for (int n = 0; n <= PQ; ++n)
#pragma unroll
                        for (int m = -n; m <= n; ++m) {
                            const cplx g2 = (-nz) * T[IDX(n + 1, m)] +
                                            0.5 * (nmn * T[IDX(n + 1, m + 1)] -
                                                   npl * T[IDX(n + 1, m - 1)]);
#pragma unroll
                            for (int q = 0; q < NRC; ++q) A.v[q][IDX(n, m)] += qs[q] * g2;
                        }
                }
            }
        }
        __syncthreads();
    };

    int fill = 0;
    const int e1 = l1s[it + 1];
    for (int e = l1s[it]; e < e1; ++e) {
        const int Sb = l1l[e];
        int s = t.sstart[Sb];
        const int s1 = s + t.scount[Sb];
        while (s < s1) {
            const int take = min(s1 - s, CH - fill);
            for (int j = lane; j < take; j += 64) {
                const int si = s + j, dd = fill + j;
                sx[dd] = src[si];
                sy[dd] = src[(size_t)ns + si];
                sz[dd] = src[2 * (size_t)ns + si];
                if (dip) {
                    snx[dd] = nrm[si];
                    sny[dd] = nrm[(size_t)ns + si];
                    snz[dd] = nrm[2 * (size_t)ns + si];
                }
#pragma unroll
                for (int q = 0; q < NRC; ++q)
                    if (q < rc) {
                        const double *pq = str + 2 * ((size_t)si * nr + r0 + q);
                        sq[2 * (dd * NRC + q)] = pq[0];
                        sq[2 * (dd * NRC + q) + 1] = pq[1];
                    }
            }
            fill += take;
            s += take;
            if (fill == CH) {
                flush(CH);
                fill = 0;
            }
        }
    }
    if (fill > 0) flush(fill);
#pragma unroll
    for (int q = 0; q < NRC; ++q)
#pragma unroll
        for (int i = 0; i < NQ; ++i)
            for (int m = G / 2; m >= 1; m >>= 1) {
                A.v[q][i].x += __shfl_xor(A.v[q][i].x, m);
                A.v[q][i].y += __shfl_xor(A.v[q][i].y, m);
            }
    if (active && sub == 0) qbx_store<PQ, NRC>(kd, qexp, c, A, accumulate);
}

// Batched P2QBXL (many right-hand sides), a complex contraction per target
// box: for one group of up to GC_GROUP global centers of a box and MR_RB
// right-hand sides, the box's list-1 sources are taken SC at a time; phase A
// builds the basis of every (center, source) pair once into LDS,
// A[k][row] with row = (center, coefficient), and stages the chunk's
// strengths B[k][rhs]; phase B accumulates C[row][rhs] += sum_k A[k][row]
// B[k][rhs] on the FP64 matrix cores (v_mfma_f64_16x16x4f64, 16 x 16 output
// tiles, the complex product as four real ones).  The basis is computed once
// for all right-hand sides instead of once per register chunk of them.
constexpr int MR_RB = 32;

template <int PQ>
struct MRShape {
    static constexpr int NQ = (PQ + 1) * (PQ + 1);
    static constexpr int R = GC_GROUP * NQ;
    static constexpr int SC = PQ <= 3 ? 32 : 16;
};

template <int PQ>
__global__ void __launch_bounds__(256) k3_p2qbxl_mr(KD kd, TD t, const int *ubox,
                                                    const int *uc0, const int *gcs,
                                                    const int *gcl, const double *ctr, int nc,
                                                    const int *l1s, const int *l1l,
                                                    const double *src, int ns, const double *str,
                                                    const double *nrm, double *qexp,
                                                    int accumulate)
{
    using SH = MRShape<PQ>;
    constexpr int NQ = SH::NQ, R = SH::R, SC = SH::SC;
    __shared__ double As[SC * R * 2];
    __shared__ double Bs[SC * MR_RB * 2];
    __shared__ int sidx[SC];
    const int u = blockIdx.x;
    const int it = ubox[u];
    const int c0 = uc0[u];
    const int ncen = min(GC_GROUP, gcs[it + 1] - gcs[it] - c0);
    const int nr = kd.nr;
    const int rb0 = blockIdx.y * MR_RB;
    const int nrb = min(MR_RB, nr - rb0);
    const int tid = threadIdx.x;
    const int wv = tid >> 6, lane = tid & 63;
    const int col = lane & 15, kr = lane >> 4;
    const bool dip = kd.dip;
    // phase B on the matrix cores: output tiles (16 rows x 16 right-hand
    // sides); wave w takes the row tiles w, w + 4, ... for both column tiles
    constexpr int RT = (R + 15) / 16, RTW = (RT + 3) / 4;
    f3_d4 cre[RTW][2], cim[RTW][2];
#pragma unroll
    for (int j = 0; j < RTW; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h) cre[j][h] = cim[j][h] = f3_d4{0, 0, 0, 0};

    auto flush = [&](int n) {
        __syncthreads();
        for (int pr = tid; pr < GC_GROUP * n; pr += 256) {
            const int ci = pr / n, k = pr - ci * n;
            if (ci >= ncen) continue;
            const int si = sidx[k];
            const v3 cc = ld3(ctr, nc, gcl[gcs[it] + c0 + ci]);
            const v3 d = sub(ld3(src, ns, si), cc);
            double *a = As + 2 * ((size_t)k * R + ci * NQ);
            if (!dip) {
                cplx T[NQ];
                the_table<PQ>(d, T);
#pragma unroll
                for (int i = 0; i < NQ; ++i) stc(a + 2 * i, T[i]);
            } else {
                constexpr int P1 = PQ + 1;
                cplx T[(P1 + 1) * (P1 + 1)];
                the_table<P1>(d, T);
                const v3 nu = ld3(nrm, ns, si);
                const cplx nmn = {nu.x, -nu.y}, npl = {nu.x, nu.y};
#pragma unroll
                for (int nn = 0; nn <= PQ; ++nn)
#pragma unroll
                    for (int m = -nn; m <= nn; ++m)
                        stc(a + 2 * IDX(nn, m),
                            (-nu.z) * T[IDX(nn + 1, m)] +
                                0.5 * (nmn * T[IDX(nn + 1, m + 1)] - npl * T[IDX(nn + 1, m - 1)]));
            }
        }
        int imag = 0;
        for (int e = tid; e < n * nrb; e += 256) {
            const int k = e / nrb, r = e - k * nrb;
            const double *pq = str + 2 * ((size_t)sidx[k] * nr + rb0 + r);
            Bs[2 * (k * MR_RB + r)] = pq[0];
            Bs[2 * (k * MR_RB + r) + 1] = pq[1];
            imag |= pq[1] != 0.0;
        }
        // real strengths (a real density): the products with the zero
        // imaginary parts are skipped (block-uniform)
        imag = __syncthreads_or(imag);
        // C[row][rhs] += sum_k A[k][row] B[k][rhs]: lane holds A[row0 + col][k]
        // and B[k][16 h + col], k = 4 ks + kr; slots k >= n hold stale data
        // and are masked (rows and columns past the valid ones only reach
        // outputs that are not stored)
        for (int ks = 0; ks < (SC + 3) / 4; ++ks) {
            const int k = ks * 4 + kr;
            const bool kin = k < n;
            double bre[2], bim[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                bre[h] = kin ? Bs[2 * (k * MR_RB + 16 * h + col)] : 0.0;
                bim[h] = kin ? Bs[2 * (k * MR_RB + 16 * h + col) + 1] : 0.0;
            }
#pragma unroll
            for (int j = 0; j < RTW; ++j) {
                const int rtile = wv + 4 * j;
                if (rtile < RT) {
                    const int row = rtile * 16 + col;
                    double are = 0.0, aim = 0.0;
                    if (kin && row < R) {
                        are = As[2 * (k * R + row)];
                        aim = As[2 * (k * R + row) + 1];
                    }
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        cre[j][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(are, bre[h], cre[j][h], 0, 0, 0);
                        if (imag) {
                            cre[j][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(-aim, bim[h], cre[j][h], 0, 0, 0);
                            cim[j][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(are, bim[h], cim[j][h], 0, 0, 0);
                        }
                        cim[j][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(aim, bre[h], cim[j][h], 0, 0, 0);
                    }
                }
            }
        }
    };

    int fill = 0;
    const int e1 = l1s[it + 1];
    for (int e = l1s[it]; e < e1; ++e) {
        const int Sb = l1l[e];
        int s = t.sstart[Sb];
        const int s1 = s + t.scount[Sb];
        while (s < s1) {
            const int take = min(s1 - s, SC - fill);
            for (int j = tid; j < take; j += 256) sidx[fill + j] = s + j;
            fill += take;
            s += take;
            if (fill == SC) {
                flush(SC);
                fill = 0;
            }
        }
    }
    if (fill > 0) flush(fill);
#pragma unroll
    for (int j = 0; j < RTW; ++j) {
        const int rtile = wv + 4 * j;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int row = rtile * 16 + 4 * g + kr;  // D row of register g
                const int r = 16 * h + col;
                if (rtile >= RT || row >= R || r >= nrb) continue;
                const int ci = row / NQ, i = row - ci * NQ;
                if (ci >= ncen) continue;
                const int c = gcl[gcs[it] + c0 + ci];
                const cplx v = {cre[j][h][g], cim[j][h][g]};
                double *pq = qexp + 2 * (((size_t)c * NQ + i) * nr + rb0 + r);
                stc(pq, accumulate ? ldc(pq) + v : v);
            }
    }
}

constexpr int M2Q_LANES = 16;

// A lane group lives inside one wavefront: order its LDS writes before the
// group's reads (and reads before the next overwrite) without a block barrier,
// which the groups' different trip counts would make unsafe.
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// M2QBXL: 16 lanes per global center; per list-3 box the irregular harmonics
// T_N^M(c - b), N <= p_b + PQ, are built in LDS (one column m >= 0 per lane),
// then lane j contracts output coefficients j, j + 16, ...
template <int PQ, int NRC>
__global__ void __launch_bounds__(256) k3_m2qbxl(KD kd, TD t, int ng, const int *gcent,
                                                 const int *c2tb, const double *ctr, int nc,
                                                 const int *l3s, const int *l3l,
                                                 const double *mpole, double *qexp)
{
    constexpr int NQ = (PQ + 1) * (PQ + 1);
    constexpr int NO = (NQ + M2Q_LANES - 1) / M2Q_LANES;
    extern __shared__ double lds[];
    const int gid = blockIdx.x * blockDim.x + threadIdx.x;
    const int g = gid / M2Q_LANES, lane = gid % M2Q_LANES;
    const int slot = threadIdx.x / M2Q_LANES;
    const int pn = kd.pmax + PQ;
    const int ntab = (pn + 1) * (pn + 1);
    double *T = lds + 2L * slot * ntab;
    const bool active = g < ng;
    const int c = active ? gcent[g] : 0;
    const int it = active ? c2tb[c] : 0;
    const v3 cc = active ? ld3(ctr, nc, c) : v3{0, 0, 0};
    cplx acc[NO][NRC];
#pragma unroll
    for (int r = 0; r < NO; ++r)
#pragma unroll
        for (int q = 0; q < NRC; ++q) acc[r][q] = {0, 0};
    const int e0 = active ? l3s[it] : 0, e1 = active ? l3s[it + 1] : 0;
    for (int e = e0; e < e1; ++e) {
        const int D = l3l[e];
        const int lv = t.level[D];
        const int p1 = kd.order[lv];
        const int N1 = p1 + PQ;
        const v3 d = sub(cc, boxc(t, D));
        const double r2 = d.x * d.x + d.y * d.y + d.z * d.z;
        const double ir2 = 1.0 / r2;
        const cplx w = {d.x * ir2, d.y * ir2};
        // column m = lane, lane + 16, ...: T_m^m by its product formula, then up in n
        for (int m = lane; m <= N1; m += M2Q_LANES) {
            cplx tmm = {sqrt(ir2), 0};
            for (int i = 1; i <= m; ++i) tmm = (-(2.0 * i - 1.0)) * (tmm * w);
            cplx a = {0, 0}, b = tmm;
            for (int n = m; n <= N1; ++n) {
                if (n > m) {
                    const cplx cn = ir2 * (((2.0 * n - 1.0) * d.z) * b -
                                           ((double)(n + m - 1) * (n - m - 1)) * a);
                    a = b;
                    b = cn;
                }
                stc(T + 2 * IDX(n, m), b);
                if (m > 0) stc(T + 2 * IDX(n, -m), neg_m(b, m));
            }
        }
        wave_sync();
        const double *a = mpole + ecoef_off(kd, D, lv);
#pragma unroll
        for (int r = 0; r < NO; ++r) {
            const int qo = lane + r * M2Q_LANES;
            if (qo < NQ) {
                int k, l;
                nm_of(qo, k, l);
                cplx s[NRC];
#pragma unroll
                for (int q = 0; q < NRC; ++q) s[q] = {0, 0};
                for (int n = 0; n <= p1; ++n) {
                    const int N = n + k;
                    for (int m = -n; m <= n; ++m) {
                        const int M = m + l;
                        if (M < -N || M > N) continue;
                        const cplx tv = ldc(T + 2 * IDX(N, M));
#pragma unroll
                        for (int q = 0; q < NRC; ++q)
                            if (q < kd.rc) s[q] += ldcn(kd, a, IDX(n, m), kd.r0 + q) * tv;
                    }
                }
#pragma unroll
                for (int q = 0; q < NRC; ++q) acc[r][q] += (k & 1) ? -s[q] : s[q];
            }
        }
        wave_sync();
    }
    if (active) {
#pragma unroll
        for (int r = 0; r < NO; ++r) {
            const int qo = lane + r * M2Q_LANES;
            if (qo < NQ) store_add<NRC>(kd, qexp + 2 * ((size_t)c * NQ + qo) * kd.nr, acc[r]);
        }
    }
}

// M2QBXL for many right-hand sides on the FP64 matrix cores: a block per
// group of GC_GROUP global centers of one target box (gc_group_plan), wave w
// takes center w of the group and the 32 right-hand sides of blockIdx.y.
// Per list-3 box D of the target box the wave builds T_N^M(c - b_D),
// N <= p_D + PQ, in its own LDS slice (as k3_m2qbxl, one column m per lane),
// then the complex product out[(k,l)][r] += sum_(n,m) T(n+k, m+l)
// a_D[(n,m)][r] runs as four real v_mfma_f64_16x16x4f64 per K-step of four
// (n,m) (lane i holds A[i%16][k0 + i/16] and B[k0 + i/16][i%16]; D register
// j of lane i is D[4j + i/16][i%16]): rows (k,l) in 16-row tiles, columns
// two tiles of 16 right-hand sides, multipoles read straight from HBM (the
// group's waves read the same box).  The epilogue applies (-1)^k and adds
// into qexp.  Waves only touch their own LDS slice: no block barrier.
constexpr int M2QM_RB = 32;  // right-hand sides per block (blockIdx.y)

template <int PQ>
__global__ void __launch_bounds__(256) k3_m2qbxl_mfma(KD kd, TD t, const int *ubox,
                                                      const int *uc0, const int *gcs,
                                                      const int *gcl, const double *ctr, int nc,
                                                      const int *l3s, const int *l3l,
                                                      const double *mpole, double *qexp)
{
    constexpr int NQ = (PQ + 1) * (PQ + 1);
    constexpr int RT = (NQ + 15) / 16;
    extern __shared__ double lds[];
    const int u = blockIdx.x;
    const int it = ubox[u];
    const int c0 = uc0[u];
    const int ncen = min(GC_GROUP, gcs[it + 1] - gcs[it] - c0);
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
    if (wv >= ncen) return;  // no barriers below: idle waves leave at once
    const int col = lane & 15, kr = lane >> 4;
    const int nr = kd.nr;
    const int rb0 = blockIdx.y * M2QM_RB;
    const int nrb = min(M2QM_RB, nr - rb0);
    const int c = gcl[gcs[it] + c0 + wv];
    const v3 cc = ld3(ctr, nc, c);
    const int pn = kd.pmax + PQ;
    double *T = lds + 2L * wv * (pn + 1) * (pn + 1);
    // the (k, l) of this lane's A rows, tile by tile
    int rk[RT], rl[RT];
#pragma unroll
    for (int q = 0; q < RT; ++q) {
        const int row = q * 16 + col;
        if (row < NQ)
            nm_of(row, rk[q], rl[q]);
        else
            rk[q] = rl[q] = 0;
    }
    f3_d4 cre[RT][2], cim[RT][2];
#pragma unroll
    for (int q = 0; q < RT; ++q)
#pragma unroll
        for (int h = 0; h < 2; ++h) cre[q][h] = cim[q][h] = f3_d4{0, 0, 0, 0};
    const int e0 = l3s[it], e1 = l3s[it + 1];
    for (int e = e0; e < e1; ++e) {
        const int D = l3l[e];
        const int lv = t.level[D];
        const int p1 = kd.order[lv];
        const int N1 = p1 + PQ;
        const int ncf = (p1 + 1) * (p1 + 1);
        const v3 d = sub(cc, boxc(t, D));
        const double r2 = d.x * d.x + d.y * d.y + d.z * d.z;
        const double ir2 = 1.0 / r2;
        const cplx w = {d.x * ir2, d.y * ir2};
        for (int m = lane; m <= N1; m += 64) {
            cplx tmm = {sqrt(ir2), 0};
            for (int i = 1; i <= m; ++i) tmm = (-(2.0 * i - 1.0)) * (tmm * w);
            cplx a = {0, 0}, b = tmm;
            for (int n = m; n <= N1; ++n) {
                if (n > m) {
                    const cplx cn = ir2 * (((2.0 * n - 1.0) * d.z) * b -
                                           ((double)(n + m - 1) * (n - m - 1)) * a);
                    a = b;
                    b = cn;
                }
                stc(T + 2 * IDX(n, m), b);
                if (m > 0) stc(T + 2 * IDX(n, -m), neg_m(b, m));
            }
        }
        wave_sync();
        const double *am = mpole + ecoef_off(kd, D, lv);
        const int KS = (ncf + 3) / 4;
        for (int ks = 0; ks < KS; ++ks) {
            const int kq = ks * 4 + kr;  // (n, m) of the A column and B row
            int n = 0, m = 0;
            const bool kin = kq < ncf;
            if (kin) nm_of(kq, n, m);
            double bre[2], bim[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int rr = h * 16 + col;
                bre[h] = bim[h] = 0.0;
                if (kin && rr < nrb) {
                    const cplx bv = ldcn(kd, am, kq, rb0 + rr);
                    bre[h] = bv.x;
                    bim[h] = bv.y;
                }
            }
#pragma unroll
            for (int q = 0; q < RT; ++q) {
                const int row = q * 16 + col;
                double are = 0.0, aim = 0.0;
                if (kin && row < NQ) {
                    const int N = n + rk[q], M = m + rl[q];
                    if (M >= -N && M <= N) {
                        are = T[2 * IDX(N, M)];
                        aim = T[2 * IDX(N, M) + 1];
                    }
                }
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    cre[q][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(are, bre[h], cre[q][h], 0, 0, 0);
                    cre[q][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(-aim, bim[h], cre[q][h], 0, 0, 0);
                    cim[q][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(are, bim[h], cim[q][h], 0, 0, 0);
                    cim[q][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(aim, bre[h], cim[q][h], 0, 0, 0);
                }
            }
        }
        wave_sync();  // T read before the next box overwrites it
    }
    double *o = qexp + 2 * (size_t)c * NQ * nr;
#pragma unroll
    for (int q = 0; q < RT; ++q)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int row = q * 16 + 4 * j + kr;
            if (row < NQ) {
                int k, l;
                nm_of(row, k, l);
                const double sg = (k & 1) ? -1.0 : 1.0;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int rr = h * 16 + col;
                    if (rr < nrb) {
                        double *dst = o + 2 * ((long)row * nr + rb0 + rr);
                        dst[0] += sg * cre[q][h][j];
                        dst[1] += sg * cim[q][h][j];
                    }
                }
            }
        }
}

// L2QBXL for many right-hand sides on the FP64 matrix cores: a block per
// group of GC_GROUP global centers of one target box (they share the box's
// local expansion L), wave w takes center w and the 32 right-hand sides of
// blockIdx.y.  The wave builds Y_j^i(c - b), j <= p (the recurrences of
// k3_l2qbxl, one column i per lane, Y_j^-i = (-1)^i conj(Y_j^i)) in its LDS
// slice; then out[(a,b)][r] += sum_(n,m) conj(Y_(n-a)^(m-b)) L[(n,m)][r]
// (zero unless n >= a and |m - b| <= n - a) as four real
// v_mfma_f64_16x16x4f64 per K-step (lane layout as k3_m2qbxl_mfma).
template <int PQ>
__global__ void __launch_bounds__(256) k3_l2qbxl_mfma(KD kd, TD t, const int *ubox,
                                                      const int *uc0, const int *gcs,
                                                      const int *gcl, const int *tboxes,
                                                      const double *ctr, int nc,
                                                      const double *local, double *qexp)
{
    constexpr int NQ = (PQ + 1) * (PQ + 1);
    constexpr int RT = (NQ + 15) / 16;
    extern __shared__ double lds[];
    const int u = blockIdx.x;
    const int it = ubox[u];
    const int c0 = uc0[u];
    const int ncen = min(GC_GROUP, gcs[it + 1] - gcs[it] - c0);
    const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
    if (wv >= ncen) return;  // no barriers below: idle waves leave at once
    const int col = lane & 15, kr = lane >> 4;
    const int nr = kd.nr;
    const int rb0 = blockIdx.y * M2QM_RB;
    const int nrb = min(M2QM_RB, nr - rb0);
    const int c = gcl[gcs[it] + c0 + wv];
    const int Bx = tboxes[it];
    const int lv = t.level[Bx];
    const int p1 = kd.order[lv];
    const int ncf = (p1 + 1) * (p1 + 1);
    double *Y = lds + 2L * wv * (kd.pmax + 1) * (kd.pmax + 1);
    const v3 d = sub(ld3(ctr, nc, c), boxc(t, Bx));
    const double r2 = d.x * d.x + d.y * d.y + d.z * d.z;
    const cplx hw = {-0.5 * d.x, -0.5 * d.y};
    for (int i = lane; i <= p1; i += 64) {
        cplx ymm = {1, 0};
        for (int q = 1; q <= i; ++q) ymm = (1.0 / q) * (ymm * hw);
        cplx ya = {0, 0}, yb = ymm;
        for (int j = i; j <= p1; ++j) {
            if (j > i) {
                const cplx cn = (1.0 / ((double)(j - i) * (j + i))) *
                                (((2.0 * j - 1.0) * d.z) * yb - r2 * ya);
                ya = yb;
                yb = cn;
            }
            stc(Y + 2 * IDX(j, i), yb);
            if (i > 0) stc(Y + 2 * IDX(j, -i), (i & 1) ? -conj(yb) : conj(yb));
        }
    }
    wave_sync();
    int ra[RT], rb[RT];
#pragma unroll
    for (int q = 0; q < RT; ++q) {
        const int row = q * 16 + col;
        if (row < NQ)
            nm_of(row, ra[q], rb[q]);
        else
            ra[q] = rb[q] = 0;
    }
    f3_d4 cre[RT][2], cim[RT][2];
#pragma unroll
    for (int q = 0; q < RT; ++q)
#pragma unroll
        for (int h = 0; h < 2; ++h) cre[q][h] = cim[q][h] = f3_d4{0, 0, 0, 0};
    const double *L = local + ecoef_off(kd, Bx, lv);
    const int KS = (ncf + 3) / 4;
    for (int ks = 0; ks < KS; ++ks) {
        const int kq = ks * 4 + kr;
        int n = 0, m = 0;
        const bool kin = kq < ncf;
        if (kin) nm_of(kq, n, m);
        double bre[2], bim[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int rr = h * 16 + col;
            bre[h] = bim[h] = 0.0;
            if (kin && rr < nrb) {
                const cplx bv = ldcn(kd, L, kq, rb0 + rr);
                bre[h] = bv.x;
                bim[h] = bv.y;
            }
        }
#pragma unroll
        for (int q = 0; q < RT; ++q) {
            const int row = q * 16 + col;
            double are = 0.0, aim = 0.0;
            const int j = n - ra[q], i = m - rb[q];
            if (kin && row < NQ && j >= 0 && i >= -j && i <= j) {
                are = Y[2 * IDX(j, i)];
                aim = -Y[2 * IDX(j, i) + 1];  // conj
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                cre[q][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(are, bre[h], cre[q][h], 0, 0, 0);
                cre[q][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(-aim, bim[h], cre[q][h], 0, 0, 0);
                cim[q][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(are, bim[h], cim[q][h], 0, 0, 0);
                cim[q][h] = __builtin_amdgcn_mfma_f64_16x16x4f64(aim, bre[h], cim[q][h], 0, 0, 0);
            }
        }
    }
    double *o = qexp + 2 * (size_t)c * NQ * nr;
#pragma unroll
    for (int q = 0; q < RT; ++q)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int row = q * 16 + 4 * j + kr;
            if (row < NQ) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int rr = h * 16 + col;
                    if (rr < nrb) {
                        double *dst = o + 2 * ((long)row * nr + rb0 + rr);
                        dst[0] += cre[q][h][j];
                        dst[1] += cim[q][h][j];
                    }
                }
            }
        }
}

// L2QBXL: one thread per global center
template <int PQ, int NRC>
__global__ void k3_l2qbxl(KD kd, TD t, int ng, const int *gcent, const int *c2tb,
                          const int *tboxes, const double *ctr, int nc, const double *local,
                          double *qexp)
{
    constexpr int NQ = (PQ + 1) * (PQ + 1);
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= ng) return;
    const int c = gcent[g];
    const int Bx = tboxes[c2tb[c]];
    const int lv = t.level[Bx];
    const int p1 = kd.order[lv];
    const v3 d = sub(ld3(ctr, nc, c), boxc(t, Bx));
    const double *L = local + ecoef_off(kd, Bx, lv);
    QAcc<PQ, NRC> A;
#pragma unroll
    for (int q = 0; q < NRC; ++q)
#pragma unroll
        for (int i = 0; i < NQ; ++i) A.v[q][i] = {0, 0};
    const double r2 = d.x * d.x + d.y * d.y + d.z * d.z;
    const cplx hw = {-0.5 * d.x, -0.5 * d.y};
    cplx ymm = {1, 0};
    for (int i = 0; i <= p1; ++i) {        // column i >= 0 of Y_j^i, j = i..p1
        if (i > 0) ymm = (1.0 / i) * (ymm * hw);
        cplx ya = {0, 0}, yb = ymm;
        for (int j = i; j <= p1; ++j) {
            if (j > i) {
                const cplx cn = (1.0 / ((double)(j - i) * (j + i))) *
                                (((2.0 * j - 1.0) * d.z) * yb - r2 * ya);
                ya = yb;
                yb = cn;
            }
            const cplx yc = conj(yb);                  // conj(Y_j^i)
            const cplx yn = (i & 1) ? -yb : yb;        // conj(Y_j^{-i}) = (-1)^i Y_j^i
#pragma unroll
            for (int a = 0; a <= PQ; ++a) {
                if (a + j > p1) continue;
#pragma unroll
                for (int b = -a; b <= a; ++b) {
                    const int n = a + j;
                    const int m1 = b + i;
                    const int m2 = b - i;
#pragma unroll
                    for (int q = 0; q < NRC; ++q) {
                        if (q >= kd.rc) continue;
                        if (m1 >= -n && m1 <= n)
                            A.v[q][IDX(a, b)] += ldcn(kd, L, IDX(n, m1), kd.r0 + q) * yc;
                        if (i > 0 && m2 >= -n && m2 <= n)
                            A.v[q][IDX(a, b)] += ldcn(kd, L, IDX(n, m2), kd.r0 + q) * yn;
                    }
                }
            }
        }
    }
    qbx_store<PQ, NRC>(kd, qexp, c, A, 1);
}

// QBXL2P: one thread per (center, target) entry
template <int NRC>
__global__ void k3_qbxl2p(KD kd, int nctt, const int *ctt_lists, const int *tree_ttc,
                          const double *tgt, int nt, const double *ctr, int nc,
                          const double *qexp, double *pot)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nctt) return;
    const int ti = ctt_lists[j];
    const int c = tree_ttc[ti];
    const v3 d = sub(ld3(tgt, nt, ti), ld3(ctr, nc, c));
    cplx v[NRC];
#pragma unroll
    for (int q = 0; q < NRC; ++q) v[q] = {0, 0};
    sum_regular_conj_n<NRC>(kd, qexp + 2 * (size_t)c * kd.ncq * kd.nr, kd.pq, d, v);
#pragma unroll
    for (int q = 0; q < NRC; ++q)
        if (q < kd.rc) stc(pot + 2 * ((size_t)ti * kd.nr + kd.r0 + q), INV4PI * v[q]);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
using zc = std::complex<double>;

static void host_irregular(int p, const double *x, zc *T)
{
    const double r2 = x[0] * x[0] + x[1] * x[1] + x[2] * x[2];
    const double ir2 = 1.0 / r2;
    const zc w(x[0] * ir2, x[1] * ir2);
    zc tmm(std::sqrt(ir2), 0.0);
    for (int m = 0; m <= p; ++m) {
        if (m > 0) tmm = -(2.0 * m - 1.0) * w * tmm;
        zc a = 0.0, b = tmm;
        T[IDX(m, m)] = tmm;
        for (int n = m + 1; n <= p; ++n) {
            zc c = ir2 * ((2.0 * n - 1.0) * x[2] * b - (double)(n + m - 1) * (n - m - 1) * a);
            T[IDX(n, m)] = c;
            a = b;
            b = c;
        }
    }
    for (int n = 1; n <= p; ++n)
        for (int m = 1; m <= n; ++m) T[IDX(n, -m)] = ((m & 1) ? -1.0 : 1.0) * std::conj(T[IDX(n, m)]);
}

static void host_regular(int p, const double *x, zc *Y)
{
    const double r2 = x[0] * x[0] + x[1] * x[1] + x[2] * x[2];
    const zc hw(-0.5 * x[0], -0.5 * x[1]);
    zc ymm = 1.0;
    for (int m = 0; m <= p; ++m) {
        if (m > 0) ymm = (1.0 / m) * hw * ymm;
        zc a = 0.0, b = ymm;
        Y[IDX(m, m)] = ymm;
        for (int n = m + 1; n <= p; ++n) {
            zc c = ((2.0 * n - 1.0) * x[2] * b - r2 * a) / ((double)(n - m) * (n + m));
            Y[IDX(n, m)] = c;
            a = b;
            b = c;
        }
    }
    for (int n = 1; n <= p; ++n)
        for (int m = 1; m <= n; ++m) Y[IDX(n, -m)] = ((m & 1) ? -1.0 : 1.0) * std::conj(Y[IDX(n, m)]);
}

static int make_kd(const qbx_kernel_desc *d, const qbx_tree *T, KD *kd, int nsep = 2)
{
    QBX_CHECK(d, "null kernel description");
    QBX_CHECK(!d->target_deriv, "3D stages: target derivatives are not supported (the "
                                "target-specific stage gives 3D gradients)");
    QBX_CHECK(d->kernel == QBX_LAPLACE3D, "3D stages support QBX_LAPLACE3D only (got %d)",
              d->kernel);
    QBX_CHECK(d->source_kind == QBX_SOURCE_S || d->source_kind == QBX_SOURCE_D,
              "unsupported source kind %d", d->source_kind);
    QBX_CHECK(d->qbx_order >= 0 && d->qbx_order <= MAXPQ, "3D qbx_order must be in [0, %d]",
              MAXPQ);
    QBX_CHECK(d->level_orders && d->nlevels >= 1, "level_orders missing");
    QBX_CHECK(d->nrhs >= 0, "nrhs must be >= 0 (0 means 1)");
    if (T) {
        QBX_CHECK(T->dim == 3, "3D kernels need a 3D tree");
        QBX_CHECK(T->nlevels <= FML, "tree has too many levels (%d)", T->nlevels);
        QBX_CHECK(d->nlevels >= T->nlevels, "level_orders has %d entries, tree has %d levels",
                  d->nlevels, T->nlevels);
    }
    memset(kd, 0, sizeof(*kd));
    kd->dip = d->source_kind == QBX_SOURCE_D;
    kd->pq = d->qbx_order;
    kd->nsep = nsep;
    kd->W = 2 * nsep + 1;
    kd->nr = d->nrhs > 0 ? d->nrhs : 1;
    kd->r0 = 0;
    kd->rc = 1;
    const int nl = T ? T->nlevels : std::min(d->nlevels, FML);
    kd->nlevels = nl;
    long coef = 0;
    int pmax = 0;
    for (int l = 0; l < nl; ++l) {
        const int p = d->level_orders[l];
        QBX_CHECK(p >= 1 && p <= MAXP, "3D fmm order %d at level %d outside [1, %d]", p, l, MAXP);
        kd->order[l] = p;
        pmax = std::max(pmax, p);
        kd->ncl[l] = (p + 1) * (p + 1);
        kd->h[l] = T ? ldexp(T->root_extent, -l) : 1.0;
        kd->lbox[l] = T ? T->level_start_box_nrs[l] : 0;
        kd->lcoef[l] = coef;
        if (T)
            coef += (long)(T->level_start_box_nrs[l + 1] - T->level_start_box_nrs[l]) * kd->ncl[l];
    }
    kd->lbox[nl] = T ? T->nboxes : 0;
    kd->lcoef[nl] = coef;
    kd->pmax = pmax;
    kd->tabn = 2 * pmax + 1;
    kd->ncq = (kd->pq + 1) * (kd->pq + 1);
    return QBX_OK;
}

// unit-offset tables, cached in the context per (nsep, pmax)
static int ensure_tables(qbx_ctx *ctx, hipStream_t st, KD *kd)
{
    std::vector<double> key = {3.0, (double)kd->nsep, (double)kd->pmax};
    QBX_TRY(note_capture(ctx, st));
    if (key != ctx->tab3_key) {
        // a graph replays the tables it captured: never rebuild under one
        QBX_TRY(may_replace(ctx, st, "3D translation tables"));
        const int W = kd->W, S1 = 2 * W + 1, tn = kd->tabn;
        const long ncls = (long)S1 * S1 * S1;
        std::vector<zc> tab((size_t)ncls * tn * tn, zc(0.0, 0.0));
        for (int ix = -W; ix <= W; ++ix)
            for (int iy = -W; iy <= W; ++iy)
                for (int iz = -W; iz <= W; ++iz) {
                    if (!ix && !iy && !iz) continue;
                    const double x[3] = {(double)ix, (double)iy, (double)iz};
                    const long cl = ((long)(ix + W) * S1 + (iy + W)) * S1 + (iz + W);
                    host_irregular(2 * kd->pmax, x, tab.data() + cl * tn * tn);
                }
        const int nc1 = (kd->pmax + 1) * (kd->pmax + 1);
        std::vector<zc> ch((size_t)8 * nc1);
        for (int ci = 0; ci < 8; ++ci) {
            const double x[3] = {(ci & 1) ? 0.5 : -0.5, (ci & 2) ? 0.5 : -0.5,
                                 (ci & 4) ? 0.5 : -0.5};
            host_regular(kd->pmax, x, ch.data() + (size_t)ci * nc1);
        }
        QBX_TRY(ctx->ws_tab3_m2l.alloc(2L * (long)tab.size()));
        QBX_TRY(ctx->ws_tab3_ch.alloc(2L * (long)ch.size()));
        QBX_HIP(hipMemcpy(ctx->ws_tab3_m2l.p, tab.data(), sizeof(zc) * tab.size(),
                          hipMemcpyHostToDevice));
        QBX_HIP(hipMemcpy(ctx->ws_tab3_ch.p, ch.data(), sizeof(zc) * ch.size(),
                          hipMemcpyHostToDevice));
        ctx->tab3_key = key;
    }
    kd->tab_m2l = ctx->ws_tab3_m2l.p;
    kd->tab_ch = ctx->ws_tab3_ch.p;
    return QBX_OK;
}

static TD make_td(const qbx_tree *T)
{
    TD t;
    t.nboxes = T->nboxes;
    t.level = T->box_levels.p;
    t.parent = T->box_parent_ids.p;
    t.child = T->box_child_ids.p;
    t.coords = T->box_coords.p;
    t.centers = T->box_centers.p;
    t.sstart = T->box_source_starts.p;
    t.scount = T->box_source_counts_nonchild.p;
    t.scumul = T->box_source_counts_cumul.p;
    return t;
}

// Run LAUNCH(N) over the right-hand-side chunks: N = 1 for a single
// right-hand side, CH otherwise; kd.r0 / kd.rc are set per chunk.
#define FOR_RHS_CHUNKS3(kd, CH, LAUNCH)                                                 \
    do {                                                                                 \
        if ((kd).nr == 1) {                                                              \
            (kd).r0 = 0;                                                                 \
            (kd).rc = 1;                                                                 \
            LAUNCH(1);                                                                   \
        } else {                                                                         \
            for (int r0_ = 0; r0_ < (kd).nr; r0_ += (CH)) {                             \
                (kd).r0 = r0_;                                                           \
                (kd).rc = std::min((CH), (kd).nr - r0_);                                 \
                LAUNCH(CH);                                                              \
            }                                                                            \
        }                                                                                \
    } while (0)

#define DISPATCH3_PQ_NR(pq, NR, KERNEL, ...)                                            \
    switch (pq) {                                                                        \
    case 0: hipLaunchKernelGGL((KERNEL<0, NR>), __VA_ARGS__); break;                     \
    case 1: hipLaunchKernelGGL((KERNEL<1, NR>), __VA_ARGS__); break;                     \
    case 2: hipLaunchKernelGGL((KERNEL<2, NR>), __VA_ARGS__); break;                     \
    case 3: hipLaunchKernelGGL((KERNEL<3, NR>), __VA_ARGS__); break;                     \
    case 4: hipLaunchKernelGGL((KERNEL<4, NR>), __VA_ARGS__); break;                     \
    case 5: hipLaunchKernelGGL((KERNEL<5, NR>), __VA_ARGS__); break;                     \
    case 6: hipLaunchKernelGGL((KERNEL<6, NR>), __VA_ARGS__); break;                     \
    case 7: hipLaunchKernelGGL((KERNEL<7, NR>), __VA_ARGS__); break;                     \
    case 8: hipLaunchKernelGGL((KERNEL<8, NR>), __VA_ARGS__); break;                     \
    default: set_error("qbx_order out of range"); return QBX_ERR_INVALID;               \
    }

#define DISPATCH3_NO_NR(no, NR, KERNEL, ...)                                            \
    switch (no) {                                                                        \
    case 1: hipLaunchKernelGGL((KERNEL<1, NR>), __VA_ARGS__); break;                     \
    case 2: hipLaunchKernelGGL((KERNEL<2, NR>), __VA_ARGS__); break;                     \
    case 3: hipLaunchKernelGGL((KERNEL<3, NR>), __VA_ARGS__); break;                     \
    case 4: hipLaunchKernelGGL((KERNEL<4, NR>), __VA_ARGS__); break;                     \
    case 5: hipLaunchKernelGGL((KERNEL<5, NR>), __VA_ARGS__); break;                     \
    case 6: hipLaunchKernelGGL((KERNEL<6, NR>), __VA_ARGS__); break;                     \
    case 7: hipLaunchKernelGGL((KERNEL<7, NR>), __VA_ARGS__); break;                     \
    default: set_error("M2L: order out of range"); return QBX_ERR_INVALID;              \
    }

static inline long exp_bytes(const KD &kd) { return 16L * kd.lcoef[kd.nlevels] * kd.nr; }

}  // namespace f3

using namespace f3;

long f3_expansion_size(const qbx_kernel_desc *d, const qbx_tree *T)
{
    KD kd;
    if (!T || make_kd(d, T, &kd) != QBX_OK) return -1;
    return kd.lcoef[kd.nlevels] * kd.nr;
}

int f3_expansion_level_offsets(const qbx_kernel_desc *d, const qbx_tree *T, long *offsets)
{
    KD kd;
    QBX_TRY(make_kd(d, T, &kd));
    for (int l = 0; l <= kd.nlevels; ++l) offsets[l] = kd.lcoef[l] * kd.nr;
    return QBX_OK;
}

int f3_ncoeff_qbx(const qbx_kernel_desc *d)
{
    KD kd;
    if (make_kd(d, nullptr, &kd) != QBX_OK) return -1;
    return kd.ncq;
}

// k3_p2e over the boxes of every level: its shape at each level's order and
// the densities' chunks.  32 sources at a time while their table fits 40 KiB of
// LDS (16 above order 11, 8 above 16).  Two column tiles (32 weights) where
// they are filled and three row tiles a wave suffice.
template <bool LOCAL>
static int launch_p2e(hipStream_t st, KD kd, const TD &td, const std::vector<int> &lstart,
                      const int *boxes, const int *starts, const int *lists, const double *src,
                      int ns, const double *str, const double *nrm, double *expn)
{
    const int nd = kd.dip ? 3 : 1;
    for (int l = 0, l1; l < kd.nlevels; l = l1) {
        // the boxes of consecutive levels of one order in one launch
        for (l1 = l + 1; l1 < kd.nlevels && kd.order[l1] == kd.order[l];) ++l1;
        const int i0 = lstart[l], nb = lstart[l1] - i0;
        if (nb == 0) continue;
        P2EShape h;
        h.pt = LOCAL ? kd.order[l] + (kd.dip ? 1 : 0) : kd.order[l];
        h.rows = (h.pt + 1) * (h.pt + 1);
        h.RT = (h.rows + 15) / 16;
        h.S = 32;
        while (h.S > 8 && h.RT * 16 * (h.S + 2) * 8 > 40960) h.S /= 2;
        h.SS = h.S + 2;
        for (int r0 = 0; r0 < kd.nr;) {
            const bool two = (kd.nr - r0) * nd > 16 && h.RT <= 12;
            h.NB = two ? 2 : 1;
            h.RTW = two ? 3 : h.RT <= 24 ? 6 : 8;
            h.RG = h.RT <= h.RTW ? 1 : h.RT <= 2 * h.RTW ? 2 : 4;
            const int per = h.NB * (16 / nd);
            kd.r0 = r0;
            kd.rc = std::min(per, kd.nr - r0);
            h.bytes = 8UL * std::max(h.RT * 16 * h.SS + h.S * 32 * h.NB, h.RT * 16 * 17);
#define P2E3_GO(D, N, T)                                                                   \
    hipLaunchKernelGGL((k3_p2e<LOCAL, D, N, T>), dim3(nb), dim3(256), h.bytes, st, kd, td, i0, \
                       h, boxes, starts, lists, src, ns, str, nrm, expn)
            if (kd.dip) {
                if (two) P2E3_GO(true, 2, 3);
                else if (h.RTW == 6) P2E3_GO(true, 1, 6);
                else P2E3_GO(true, 1, 8);
            } else {
                if (two) P2E3_GO(false, 2, 3);
                else if (h.RTW == 6) P2E3_GO(false, 1, 6);
                else P2E3_GO(false, 1, 8);
            }
#undef P2E3_GO
            r0 += kd.rc;
        }
    }
    QBX_HIP(hipGetLastError());
    return QBX_OK;
}

int f3_form_multipoles(qbx_ctx *ctx, void *stream, const qbx_tree *T, const qbx_trav *R,
                       const qbx_kernel_desc *d, const double *str, const double *nrm,
                       double *mpole)
{
    KD kd;
    QBX_TRY(make_kd(d, T, &kd));
    QBX_CHECK(!kd.dip || nrm, "double layer needs normals");
    hipStream_t st = S(stream);
    QBX_TRY(zero_fill(mpole, (exp_bytes(kd)) / 8, st));
    return launch_p2e<false>(st, kd, make_td(T), R->h_level_start_source_box_nrs,
                             R->source_boxes.p, nullptr, nullptr, T->sources.p, T->nsources, str,
                             nrm, mpole);
}

// Launch k3_trans_real<OPK, p> over nb output boxes of level l (orders p <= 15;
// 32 right-hand sides per block, 16 for M2M and L2L above order 9).
template <int OPK, bool SPLIT>
static int launch_trans_real(hipStream_t st, KD kd, const TD &td, int p, int i0, int nb,
                             const int *boxes, const int *starts, const int *lists,
                             const double *in, double *out, const int *allreal)
{
    const int rcb = SPLIT ? 8 : (OPK != 0 && p >= 10) ? 16 : 32;
    for (int r0 = 0; r0 < kd.nr; r0 += rcb) {
        kd.r0 = r0;
        kd.rc = std::min(rcb, kd.nr - r0);
#define TR_CASE(PP)                                                                        \
    case PP:                                                                               \
        hipLaunchKernelGGL(                                                                \
            (k3_trans_real<OPK, PP, (SPLIT || (OPK != 0 && PP >= 10)) ? 1 : 2, SPLIT>),    \
            dim3(nb), dim3(256), 0, st, kd, td, i0, boxes, starts, lists, in, out, allreal); \
        break;
        switch (p) {
            TR_CASE(1) TR_CASE(2) TR_CASE(3) TR_CASE(4) TR_CASE(5) TR_CASE(6) TR_CASE(7)
            TR_CASE(8) TR_CASE(9) TR_CASE(10) TR_CASE(11) TR_CASE(12) TR_CASE(13)
            TR_CASE(14) TR_CASE(15)
        default: set_error("matrix-core translation: order %d out of range", p);
            return QBX_ERR_INVALID;
        }
#undef TR_CASE
    }
    QBX_HIP(hipGetLastError());
    return QBX_OK;
}

// Which kernels run a box translation: the real-strength matrix-core kernel
// (stated by the caller, or decided on the device by *flag), the one for any
// strengths, or both, each returning at once in the other's case.
struct RealSel {
    bool real, other;
    const int *flag;  // passed to both kernels (null: no device decision)
};

static RealSel real_sel(const qbx_kernel_desc *d, const KD &kd, const int *flag, bool fits)
{
    const bool ok = fits && kd.nr >= 4;
    if (ok && d->real_strengths) return {true, false, nullptr};
    if (ok && flag) return {true, true, flag};
    return {false, true, nullptr};
}

int f3_coarsen_multipoles(qbx_ctx *ctx, void *stream, const qbx_tree *T, const qbx_trav *R,
                          const qbx_kernel_desc *d, double *mpole, int lmin, const int *allreal)
{
    KD kd;
    QBX_TRY(make_kd(d, T, &kd, R->nsep));
    QBX_TRY(ensure_tables(ctx, S(stream), &kd));
    hipStream_t st = S(stream);
    const TD td = make_td(T);
    for (int l = T->nlevels - 2; l >= std::max(lmin, 0); --l) {
        const int i0 = R->h_level_start_source_parent_box_nrs[l];
        const int i1 = R->h_level_start_source_parent_box_nrs[l + 1];
        const long nthr = (long)(i1 - i0) * kd.ncl[l];
        if (nthr > 0) {
            // the real-strength kernel where parent and child orders agree
            const int p = kd.order[l];
            const RealSel rs = real_sel(d, kd, allreal, p <= 15 && kd.order[l + 1] == p);
            if (rs.real)
                QBX_TRY((launch_trans_real<1, false>(st, kd, td, p, i0, i1 - i0,
                                                     R->source_parent_boxes.p, nullptr, nullptr,
                                                     mpole, mpole, rs.flag)));
            if (rs.other) {
#define L3_M2M(N)                                                                          \
    hipLaunchKernelGGL(k3_m2m<N>, dim3(cdiv(nthr, 128)), dim3(128), 0, st, kd, td, l, i0,  \
                       i1, R->source_parent_boxes.p, mpole, rs.flag)
                FOR_RHS_CHUNKS3(kd, NRC_S, L3_M2M);
#undef L3_M2M
            }
        }
    }
    QBX_HIP(hipGetLastError());
    return QBX_OK;
}

int f3_eval_targets(qbx_ctx *ctx, void *stream, const qbx_tree *T, const qbx_trav *R,
                    const qbx_geo *G, const qbx_kernel_desc *d, int mode, const double *str,
                    const double *nrm, const double *expn, double *pot, int accumulate)
{
    KD kd;
    QBX_TRY(make_kd(d, T, &kd));
    hipStream_t st = S(stream);
    if (!accumulate)
        QBX_TRY(zero_fill(pot, (sizeof(double) * 2 * (size_t)T->ntargets * kd.nr) / 8, st));
    const int ntb = R->ntarget_boxes;
    if (ntb == 0 || G->nfiltered == 0) return QBX_OK;
    const TD td = make_td(T);
    const int *starts = mode == 1 ? R->l3_starts.p : R->l1_starts.p;
    const int *lists = mode == 1 ? R->l3_lists.p : R->l1_lists.p;
    if (mode != 2 && G->trav == R) {
        const unit_plan &U = mode == 0 ? G->p2p_plan : G->m2p_plan;
        if (U.nunits == 0) return QBX_OK;
#define EVAL3_UNITS(M, N)                                                                  \
    hipLaunchKernelGGL((k3_eval_units<M, N>), dim3(U.nunits), dim3(64), 0, st, kd, td,     \
                       U.unit_box.p, U.unit_t0.p, U.box_g.p, R->target_boxes.p, starts,   \
                       lists, G->nqbtl_box_target_starts.p,                               \
                       G->nqbtl_box_target_counts_nonchild.p, G->nqbtl_unfiltered.p,      \
                       T->targets.p, T->ntargets, T->sources.p, T->nsources, str, nrm, expn, \
                       pot)
#define EV3U0(N) EVAL3_UNITS(0, N)
#define EV3U1(N) EVAL3_UNITS(1, N)
        if (mode == 0) FOR_RHS_CHUNKS3(kd, NRC_S, EV3U0);
        else FOR_RHS_CHUNKS3(kd, NRC_S, EV3U1);
#undef EV3U0
#undef EV3U1
#undef EVAL3_UNITS
        QBX_HIP(hipGetLastError());
        return QBX_OK;
    }
#define EVAL3_LAUNCH(M, N)                                                                 \
    hipLaunchKernelGGL((k3_eval_targets<M, N>), dim3(ntb), dim3(64), 0, st, kd, td, ntb,   \
                       R->target_boxes.p, starts, lists, G->nqbtl_box_target_starts.p,    \
                       G->nqbtl_box_target_counts_nonchild.p, G->nqbtl_unfiltered.p,      \
                       T->targets.p, T->ntargets, T->sources.p, T->nsources, str, nrm,    \
                       expn, pot)
#define EV30(N) EVAL3_LAUNCH(0, N)
#define EV31(N) EVAL3_LAUNCH(1, N)
#define EV32(N) EVAL3_LAUNCH(2, N)
    if (mode == 0) FOR_RHS_CHUNKS3(kd, NRC_S, EV30);
    else if (mode == 1) FOR_RHS_CHUNKS3(kd, NRC_S, EV31);
    else FOR_RHS_CHUNKS3(kd, NRC_S, EV32);
#undef EV30
#undef EV31
#undef EV32
#undef EVAL3_LAUNCH
    QBX_HIP(hipGetLastError());
    return QBX_OK;
}

int f3_multipole_to_local(qbx_ctx *ctx, void *stream, const qbx_tree *T, const qbx_trav *R,
                          const qbx_kernel_desc *d, const double *mpole, double *local,
                          const int *allreal)
{
    KD kd;
    QBX_TRY(make_kd(d, T, &kd, R->nsep));
    QBX_TRY(ensure_tables(ctx, S(stream), &kd));
    hipStream_t st = S(stream);
    QBX_TRY(zero_fill(local, (exp_bytes(kd)) / 8, st));
    const RealSel rs = real_sel(d, kd, allreal, kd.pmax <= 15);
    if (R->nttp_boxes > 0 && R->n2 > 0 && kd.pmax <= 15) {
        // the boxes of consecutive levels of one order in one launch (a
        // kernel's tile counts are fixed by its order)
        const TD td = make_td(T);
        const std::vector<int> &ls = R->h_level_start_ttp_box_nrs;
        for (int l = 0, l1; l < kd.nlevels; l = l1) {
            for (l1 = l + 1; l1 < kd.nlevels && kd.order[l1] == kd.order[l];) ++l1;
            const int i0 = ls[l], nb = ls[l1] - i0, p = kd.order[l];
            if (nb == 0) continue;
            if (rs.real)
                QBX_TRY((launch_trans_real<0, false>(st, kd, td, p, i0, nb, R->ttp_boxes.p,
                                                     R->l2_starts.p, R->l2_lists.p, mpole, local,
                                                     rs.flag)));
            if (rs.other)
                QBX_TRY((launch_trans_real<0, true>(st, kd, td, p, i0, nb, R->ttp_boxes.p,
                                                    R->l2_starts.p, R->l2_lists.p, mpole, local,
                                                    rs.flag)));
        }
    } else if (R->nttp_boxes > 0 && R->n2 > 0) {
        const TD td = make_td(T);
        const int no = ((kd.pmax + 1) * (kd.pmax + 1) + M2L_THREADS - 1) / M2L_THREADS;
#define L3_M2L(N)                                                                          \
    DISPATCH3_NO_NR(no, N, k3_m2l, dim3(R->nttp_boxes), dim3(M2L_THREADS),                 \
                    sizeof(double) * 2 * (size_t)(kd.pmax + 1) * (kd.pmax + 1) * (N), st,  \
                    kd, td, R->ttp_boxes.p, R->l2_starts.p, R->l2_lists.p, mpole, local)
        FOR_RHS_CHUNKS3(kd, NRC_S, L3_M2L);
#undef L3_M2L
    }
    QBX_HIP(hipGetLastError());
    return QBX_OK;
}

int f3_form_locals(qbx_ctx *ctx, void *stream, const qbx_tree *T, const qbx_trav *R,
                   const qbx_kernel_desc *d, const double *str, const double *nrm, double *local,
                   int accumulate)
{
    KD kd;
    QBX_TRY(make_kd(d, T, &kd));
    QBX_CHECK(!kd.dip || nrm, "double layer needs normals");
    hipStream_t st = S(stream);
    if (!accumulate) QBX_TRY(zero_fill(local, (exp_bytes(kd)) / 8, st));
    if (R->n4 == 0) return QBX_OK;
    return launch_p2e<true>(st, kd, make_td(T), R->h_level_start_ttp_box_nrs, R->ttp_boxes.p,
                            R->l4_starts.p, R->l4_lists.p, T->sources.p, T->nsources, str, nrm,
                            local);
}

int f3_refine_locals(qbx_ctx *ctx, void *stream, const qbx_tree *T, const qbx_trav *R,
                     const qbx_kernel_desc *d, double *local, int lmin, const int *allreal)
{
    KD kd;
    QBX_TRY(make_kd(d, T, &kd, R->nsep));
    QBX_TRY(ensure_tables(ctx, S(stream), &kd));
    hipStream_t st = S(stream);
    const TD td = make_td(T);
    for (int l = std::max(lmin, 0) + 1; l < T->nlevels; ++l) {
        const int i0 = R->h_level_start_ttp_box_nrs[l], i1 = R->h_level_start_ttp_box_nrs[l + 1];
        const long nthr = (long)(i1 - i0) * kd.ncl[l];
        if (nthr > 0) {
            const int p = kd.order[l];
            const RealSel rs = real_sel(d, kd, allreal, p <= 15 && kd.order[l - 1] == p);
            if (rs.real)
                QBX_TRY((launch_trans_real<2, false>(st, kd, td, p, i0, i1 - i0, R->ttp_boxes.p,
                                                     nullptr, nullptr, local, local, rs.flag)));
            if (rs.other) {
#define L3_L2L(N)                                                                          \
    hipLaunchKernelGGL(k3_l2l<N>, dim3(cdiv(nthr, 128)), dim3(128), 0, st, kd, td, l, i0,  \
                       i1, R->ttp_boxes.p, local, rs.flag)
                FOR_RHS_CHUNKS3(kd, NRC_S, L3_L2L);
#undef L3_L2L
            }
        }
    }
    QBX_HIP(hipGetLastError());
    return QBX_OK;
}

int f3_form_global_qbx_locals(qbx_ctx *ctx, void *stream, const qbx_tree *T,
                              const qbx_trav *R, const qbx_geo *G, const qbx_kernel_desc *d,
                              const double *str, const double *nrm, double *qexp, int accumulate)
{
    KD kd;
    QBX_TRY(make_kd(d, T, &kd));
    QBX_CHECK(!kd.dip || nrm, "double layer needs normals");
    hipStream_t st = S(stream);
    if (!accumulate)
        QBX_TRY(zero_fill(qexp, (sizeof(double) * 2 * (size_t)G->ncenters * kd.ncq * kd.nr) / 8, st));
    const unit_plan &U = G->p2q_plan;
    QBX_CHECK(G->trav == R, "P2QBXL: geometry was built for another traversal");
    if (G->nglobal == 0 || U.nunits == 0) return QBX_OK;
    const TD td = make_td(T);
    if (kd.nr >= 8 && kd.pq <= 5 && G->gc_group_plan.nunits > 0) {
        const unit_plan &V = G->gc_group_plan;
        const dim3 grid(V.nunits, cdiv(kd.nr, MR_RB));
#define L3_MR(PQV)                                                                         \
    hipLaunchKernelGGL(k3_p2qbxl_mr<PQV>, grid, dim3(256), 0, st, kd, td, V.unit_box.p,    \
                       V.unit_t0.p, G->gc_by_tbox_starts.p, G->gc_by_tbox.p, G->centers.p, \
                       G->ncenters, R->l1_starts.p, R->l1_lists.p, T->sources.p,            \
                       T->nsources, str, nrm, qexp, accumulate)
        switch (kd.pq) {
        case 0: L3_MR(0); break;
        case 1: L3_MR(1); break;
        case 2: L3_MR(2); break;
        case 3: L3_MR(3); break;
        case 4: L3_MR(4); break;
        default: L3_MR(5); break;
        }
#undef L3_MR
        QBX_HIP(hipGetLastError());
        return QBX_OK;
    }
#define L3_P2Q(N)                                                                          \
    DISPATCH3_PQ_NR(kd.pq, N, k3_p2qbxl, dim3(U.nunits), dim3(64), 0, st, kd, td,          \
                    U.unit_box.p, U.unit_t0.p, U.box_g.p, G->gc_by_tbox_starts.p,           \
                    G->gc_by_tbox.p, G->centers.p, G->ncenters, R->l1_starts.p,             \
                    R->l1_lists.p, T->sources.p, T->nsources, str, nrm, qexp, accumulate)
    FOR_RHS_CHUNKS3(kd, NRC_Q, L3_P2Q);
#undef L3_P2Q
    QBX_HIP(hipGetLastError());
    return QBX_OK;
}

int f3_translate_box_multipoles_to_qbx_local(qbx_ctx *ctx, void *stream, const qbx_tree *T,
                                             const qbx_trav *R, const qbx_geo *G,
                                             const qbx_kernel_desc *d, const double *mpole,
                                             double *qexp, int accumulate)
{
    KD kd;
    QBX_TRY(make_kd(d, T, &kd));
    hipStream_t st = S(stream);
    if (!accumulate)
        QBX_TRY(zero_fill(qexp, (sizeof(double) * 2 * (size_t)G->ncenters * kd.ncq * kd.nr) / 8, st));
    const int ng = G->nglobal;
    if (ng == 0 || R->n3 == 0) return QBX_OK;
    const int pn = kd.pmax + kd.pq;
    if (kd.nr >= 4 && kd.pq <= 5 && G->gc_group_plan.nunits > 0) {
        // many right-hand sides: the matrix-core kernel, one harmonic table
        // per wave (center)
        QBX_CHECK(G->trav == R, "M2QBXL: geometry was built for another traversal");
        const unit_plan &V = G->gc_group_plan;
        const size_t lds4 = sizeof(double) * 2 * (size_t)GC_GROUP * (pn + 1) * (pn + 1);
        QBX_CHECK(lds4 <= 64 * 1024, "M2QBXL: orders too high for LDS staging (%d + %d)",
                  kd.pmax, kd.pq);
        const TD td4 = make_td(T);
        const dim3 grid(V.nunits, cdiv(kd.nr, M2QM_RB));
#define L3_M2QM(PQV)                                                                       \
    hipLaunchKernelGGL(k3_m2qbxl_mfma<PQV>, grid, dim3(256), lds4, st, kd, td4, V.unit_box.p, \
                       V.unit_t0.p, G->gc_by_tbox_starts.p, G->gc_by_tbox.p, G->centers.p, \
                       G->ncenters, R->l3_starts.p, R->l3_lists.p, mpole, qexp)
        switch (kd.pq) {
        case 0: L3_M2QM(0); break;
        case 1: L3_M2QM(1); break;
        case 2: L3_M2QM(2); break;
        case 3: L3_M2QM(3); break;
        case 4: L3_M2QM(4); break;
        default: L3_M2QM(5); break;
        }
#undef L3_M2QM
        QBX_HIP(hipGetLastError());
        return QBX_OK;
    }
    // one harmonic table per 16-lane center group: 16 groups per block, or
    // 8 / 4 for the orders whose tables would not fit 64 KiB of LDS
    int block = 256;
    size_t lds = sizeof(double) * 2 * (size_t)(block / M2Q_LANES) * (pn + 1) * (pn + 1);
    while (lds > 64 * 1024 && block > 64) {
        block /= 2;
        lds /= 2;
    }
    QBX_CHECK(lds <= 64 * 1024, "M2QBXL: orders too high for LDS staging (%d + %d)", kd.pmax,
              kd.pq);
    const TD td = make_td(T);
#define L3_M2Q(N)                                                                          \
    DISPATCH3_PQ_NR(kd.pq, N, k3_m2qbxl, dim3(cdiv((long)ng * M2Q_LANES, block)), dim3(block), \
                    lds, st, kd, td, ng, G->global_qbx_centers.p, G->center_to_target_box.p, \
                    G->centers.p, G->ncenters, R->l3_starts.p, R->l3_lists.p, mpole, qexp)
    FOR_RHS_CHUNKS3(kd, NRC_Q, L3_M2Q);
#undef L3_M2Q
    QBX_HIP(hipGetLastError());
    return QBX_OK;
}

int f3_translate_box_local_to_qbx_local(qbx_ctx *ctx, void *stream, const qbx_tree *T,
                                        const qbx_trav *R, const qbx_geo *G,
                                        const qbx_kernel_desc *d, const double *local,
                                        double *qexp, int accumulate)
{
    KD kd;
    QBX_TRY(make_kd(d, T, &kd));
    hipStream_t st = S(stream);
    if (!accumulate)
        QBX_TRY(zero_fill(qexp, (sizeof(double) * 2 * (size_t)G->ncenters * kd.ncq * kd.nr) / 8, st));
    const int ng = G->nglobal;
    if (ng == 0) return QBX_OK;
    const TD td = make_td(T);
    if (kd.nr >= 4 && kd.pq <= 5 && G->gc_group_plan.nunits > 0) {
        // many right-hand sides: the matrix-core kernel (a Y table per wave)
        QBX_CHECK(G->trav == R, "L2QBXL: geometry was built for another traversal");
        const unit_plan &V = G->gc_group_plan;
        const size_t lds4 = sizeof(double) * 2 * (size_t)GC_GROUP * (kd.pmax + 1) * (kd.pmax + 1);
        QBX_CHECK(lds4 <= 64 * 1024, "L2QBXL: order too high for LDS staging (%d)", kd.pmax);
        const dim3 grid(V.nunits, cdiv(kd.nr, M2QM_RB));
#define L3_L2QM(PQV)                                                                       \
    hipLaunchKernelGGL(k3_l2qbxl_mfma<PQV>, grid, dim3(256), lds4, st, kd, td, V.unit_box.p, \
                       V.unit_t0.p, G->gc_by_tbox_starts.p, G->gc_by_tbox.p,               \
                       R->target_boxes.p, G->centers.p, G->ncenters, local, qexp)
        switch (kd.pq) {
        case 0: L3_L2QM(0); break;
        case 1: L3_L2QM(1); break;
        case 2: L3_L2QM(2); break;
        case 3: L3_L2QM(3); break;
        case 4: L3_L2QM(4); break;
        default: L3_L2QM(5); break;
        }
#undef L3_L2QM
        QBX_HIP(hipGetLastError());
        return QBX_OK;
    }
#define L3_L2Q(N)                                                                          \
    DISPATCH3_PQ_NR(kd.pq, N, k3_l2qbxl, dim3(cdiv(ng, 64)), dim3(64), 0, st, kd, td, ng,  \
                    G->global_qbx_centers.p, G->center_to_target_box.p, R->target_boxes.p, \
                    G->centers.p, G->ncenters, local, qexp)
    FOR_RHS_CHUNKS3(kd, NRC_Q, L3_L2Q);
#undef L3_L2Q
    QBX_HIP(hipGetLastError());
    return QBX_OK;
}

int f3_eval_qbx_expansions(qbx_ctx *ctx, void *stream, const qbx_tree *T, const qbx_geo *G,
                           const qbx_kernel_desc *d, const double *qexp, double *pot)
{
    KD kd;
    QBX_TRY(make_kd(d, T, &kd));
    hipStream_t st = S(stream);
    if (G->nctt > 0) {
#define L3_Q2P(N)                                                                          \
    hipLaunchKernelGGL(k3_qbxl2p<N>, dim3(cdiv(G->nctt, 64)), dim3(64), 0, st, kd,         \
                       G->nctt, G->ctt_lists.p, G->tree_ttc.p, T->targets.p, T->ntargets,  \
                       G->centers.p, G->ncenters, qexp, pot)
        FOR_RHS_CHUNKS3(kd, NRC_S, L3_Q2P);
#undef L3_Q2P
    }
    QBX_HIP(hipGetLastError());
    return QBX_OK;
}

}  // namespace qbx
