// FMM interaction lists on the GPU (boxtree FMMTraversalBuilder +
// merge_close_lists semantics as used by pytential/qbx/geometry.py:622-641).
//
// Integer spec on box index coordinates (n = well_sep_is_n_away, e = 1 when
// targets carry extent):
//   gap(A,B)   l-inf gap between boxes, in units of the smaller box
//   sep(S,X)   S not smaller than X: gap(S,X) >= n
//   sep3(D,B)  D smaller than B: gap(D, B grown by e of its own boxes) >= n
//   list1(B)   source leaves (a) not smaller than B with !sep, (b) below a
//              same-level colleague of B and under no sep3 box, (c) leaves of
//              sep3 boxes holding fewer than min_nsources_cumul sources
//   list2(P)   children of colleagues of parent(P) that are not colleagues of P
//   list3(B)   first sep3 boxes below colleagues of B
//   list4(P)   source leaves S bigger than P: sep(S,P) and !sep(S,parent(P))
// Lists are sorted by box number.  Each box's lists are built by one
// wavefront: a count pass, an exclusive scan, a fill pass, and a sort by a
// block per list.
#include "qbx_internal.h"

#include <algorithm>
#include <climits>

namespace qbx {

struct TV {
    int dim, nboxes, nlevels;
    const int *level, *parent, *child, *coords, *lstart;
    const unsigned long long *morton;
    const int *src_nonchild, *src_cumul;
};

__device__ unsigned long long tv_morton(int dim, const int *I, int level)
{
    unsigned long long k = 0;
    for (int i = 0; i < level; ++i)
        for (int d = 0; d < dim; ++d)
            k |= (unsigned long long)((I[d] >> i) & 1) << (i * dim + d);
    return k;
}

__device__ int tv_find(const TV &t, int level, const int *I)
{
    if (level >= t.nlevels) return -1;
    for (int d = 0; d < t.dim; ++d)
        if (I[d] < 0 || I[d] >= (1 << level)) return -1;
    unsigned long long key = tv_morton(t.dim, I, level);
    int lo = t.lstart[level], hi = t.lstart[level + 1], end = hi;
    while (lo < hi) {
        int mid = (lo + hi) >> 1;
        if (t.morton[mid] < key) lo = mid + 1; else hi = mid;
    }
    return (lo < end && t.morton[lo] == key) ? lo : -1;
}

__device__ bool tv_leaf(const TV &t, int b)
{
    for (int c = 0; c < (1 << t.dim); ++c)
        if (t.child[(size_t)c * t.nboxes + b] >= 0) return false;
    return true;
}

__device__ long long tv_gap(const TV &t, int a, int b, int grow)
{
    int la = t.level[a], lb = t.level[b];
    int m = la > lb ? la : lb;
    long long g = 0;
    for (int d = 0; d < t.dim; ++d) {
        long long sa = 1LL << (m - la), sb = 1LL << (m - lb);
        long long ca = t.coords[(size_t)d * t.nboxes + a], cb = t.coords[(size_t)d * t.nboxes + b];
        long long alo = ca * sa, ahi = (ca + 1) * sa;
        long long blo = (cb - grow) * sb, bhi = (cb + 1 + grow) * sb;
        long long gd = 0;
        if (alo - bhi > gd) gd = alo - bhi;
        if (blo - ahi > gd) gd = blo - ahi;
        if (gd > g) g = gd;
    }
    return g;
}

// colleague k (k in [0, (2n+1)^dim)) of box b, or -1
__device__ int tv_colleague(const TV &t, int b, int n, int k)
{
    int w = 2 * n + 1, I[3];
    for (int d = 0; d < t.dim; ++d) {
        I[d] = t.coords[(size_t)d * t.nboxes + b] + (k % w) - n;
        k /= w;
    }
    return tv_find(t, t.level[b], I);
}

struct ListOut {
    int *cnt;          // count mode: per-item count
    const int *starts; // fill mode
    int *lists;
    int fill;          // 0 count, 1 fill
};

// appends v of the lanes with `want` to the item's list (k: the entries so
// far, the same in every lane)
__device__ inline void emit(const ListOut &o, int item, int &k, bool want, int v)
{
    const unsigned long long m = __ballot(want);
    if (want && o.fill)
        o.lists[o.starts[item] + k + __popcll(m & ((1ULL << (threadIdx.x & 63)) - 1))] = v;
    k += __popcll(m);
}

// ancestors of b, b first; every lane returns their number
__device__ inline int tv_ancestors(const TV &t, int b, int *anc)
{
    int na = 0;
    for (int a = b; a >= 0 && na < MAX_LEVELS; a = t.parent[a]) {
        if (threadIdx.x == 0) anc[na] = a;
        ++na;
    }
    __syncthreads();
    return na;
}

// Lists 1 and 3, one wavefront per target box.  The searches under the box's
// colleagues run over a stack in LDS, 64 boxes a round: a coarse target box
// (centers with extent stop there) walks most of the tree, which as one
// thread per box took 40 ms a launch of serial steps on a surface of 737280
// sources (now 0.31 ms, every box's walk spread over 64 lanes).  Bit 31 of a
// stack entry marks the boxes below a sep3 box of too few sources, whose
// leaves all go to list 1.
//
// The stack holds nlevels * 64 * 2^dim entries: a round pops the top 64 and
// pushes the children of the top one last, so depths never fall towards the
// top, and boxes of a depth are pushed only when no box of that depth is left.
__global__ void __launch_bounds__(64) k_list13(TV t, int n, int e, int minsrc, int ntb,
                                               const int *target_boxes, ListOut o1, ListOut o3)
{
    extern __shared__ int stack[];
    __shared__ int anc[MAX_LEVELS];
    constexpr unsigned SUB = 0x80000000u;
    const int lane = threadIdx.x, nchild = 1 << t.dim;
    const int it = blockIdx.x;
    const int B = target_boxes[it];
    int k1 = 0, k3 = 0;
    int ncol = 1;
    for (int d = 0; d < t.dim; ++d) ncol *= (2 * n + 1);
    // (a) leaves not smaller than B: colleagues of each ancestor-or-self
    const int na = tv_ancestors(t, B, anc);
    for (int i0 = 0; i0 < na * ncol; i0 += 64) {
        const int i = i0 + lane;
        int C = -1;
        if (i < na * ncol) {
            C = tv_colleague(t, anc[i / ncol], n, i % ncol);
            if (C >= 0 && !(t.src_nonchild[C] > 0 && tv_leaf(t, C) && tv_gap(t, C, B, 0) < n))
                C = -1;
        }
        emit(o1, it, k1, C >= 0, C);
    }
    // (b) below same-level colleagues
    for (int kc = 0; kc < ncol; kc += 64) {
        int sp = 0;
        int D = kc + lane < ncol ? tv_colleague(t, B, n, kc + lane) : -1;
        bool sub = false, expand = D >= 0;
        for (;;) {
            // push the children of the lanes' boxes, lane 0's on top
            int cnt = 0;
            if (expand)
                for (int ch = 0; ch < nchild; ++ch)
                    cnt += t.child[(size_t)ch * t.nboxes + D] >= 0;
            int after = cnt;   // this lane's and the higher lanes' children
            for (int o = 1; o < 64; o <<= 1) {
                const int x = __shfl_down(after, o);
                if (lane + o < 64) after += x;
            }
            const int total = __shfl(after, 0);
            if (cnt > 0) {
                int at = sp + after - cnt;
                for (int ch = 0; ch < nchild; ++ch) {
                    const int x = t.child[(size_t)ch * t.nboxes + D];
                    if (x >= 0) stack[at++] = (int)((unsigned)x | (sub ? SUB : 0u));
                }
            }
            __syncthreads();
            sp += total;
            if (sp == 0) break;
            const int m = sp < 64 ? sp : 64;
            const unsigned v = lane < m ? (unsigned)stack[sp - 1 - lane] : 0u;
            __syncthreads();
            sp -= m;
            D = (int)(v & ~SUB);
            sub = (v & SUB) != 0;
            bool one = false, three = false;
            expand = false;
            if (lane < m && t.src_cumul[D] > 0) {
                const bool leaf = tv_leaf(t, D);
                const bool sep = !sub && tv_gap(t, D, B, e) >= n;
                three = sep && t.src_cumul[D] >= minsrc;
                sub = sub || sep;
                one = !three && leaf && t.src_nonchild[D] > 0;
                expand = !three && !leaf;
            }
            emit(o1, it, k1, one, D);
            emit(o3, it, k3, three, D);
        }
    }
    if (lane == 0 && !o1.fill) o1.cnt[it] = k1;
    if (lane == 0 && !o3.fill) o3.cnt[it] = k3;
}

// Lists 2 and 4, one wavefront per box, the candidates dealt to the lanes
__global__ void __launch_bounds__(64) k_list24(TV t, int n, int nttp, const int *ttp_boxes,
                                               ListOut o2, ListOut o4)
{
    __shared__ int anc[MAX_LEVELS];
    const int lane = threadIdx.x, nchild = 1 << t.dim;
    const int it = blockIdx.x;
    const int P = ttp_boxes[it];
    int k2 = 0, k4 = 0;
    int lp = t.level[P];
    if (lp > 0) {
        int ncol = 1;
        for (int d = 0; d < t.dim; ++d) ncol *= (2 * n + 1);
        int Q = t.parent[P];
        for (int i0 = 0; i0 < ncol; i0 += 64) {
            const int C = i0 + lane < ncol ? tv_colleague(t, Q, n, i0 + lane) : -1;
            for (int ch = 0; ch < nchild; ++ch) {
                const int A = C >= 0 ? t.child[(size_t)ch * t.nboxes + C] : -1;
                long long g = 0;
                if (A >= 0 && t.src_cumul[A] > 0)
                    for (int d = 0; d < t.dim; ++d) {
                        long long dd = (long long)t.coords[(size_t)d * t.nboxes + A] -
                                       t.coords[(size_t)d * t.nboxes + P];
                        if (dd < 0) dd = -dd;
                        if (dd > g) g = dd;
                    }
                emit(o2, it, k2, g > n, A);
            }
        }
        const int na = tv_ancestors(t, Q, anc);
        for (int i0 = 0; i0 < na * ncol; i0 += 64) {
            const int i = i0 + lane;
            bool four = false;
            int Sb = -1;
            if (i < na * ncol) {
                Sb = tv_colleague(t, anc[i / ncol], n, i % ncol);
                four = Sb >= 0 && t.src_nonchild[Sb] > 0 && tv_leaf(t, Sb) &&
                       tv_gap(t, Sb, P, 0) >= n && tv_gap(t, Sb, Q, 0) < n;
            }
            emit(o4, it, k4, four, Sb);
        }
    }
    if (lane == 0 && !o2.fill) o2.cnt[it] = k2;
    if (lane == 0 && !o4.fill) o4.cnt[it] = k4;
}

// Sorts each list (distinct box numbers) from `in` to `out`, a block per
// list.  Up to SORT_RANK entries: every entry's rank by comparison with the
// others in LDS.  More: a bitmap of the box numbers in LDS, `words` of it at
// a time, read back in order (one thread's insertion sort of the longest
// list, 12 thousand boxes, took 240 ms; a launch now takes under 45 us).
constexpr int SORT_RANK = 256, SORT_WORDS = 8192;

__global__ void __launch_bounds__(256) k_sort_lists(const int *starts, const int *in, int *out,
                                                    int nboxes, int words)
{
    extern __shared__ unsigned bits[];
    __shared__ int wsum[4];
    const int tid = threadIdx.x;
    const int a = starts[blockIdx.x], n = starts[blockIdx.x + 1] - a;
    if (n <= SORT_RANK) {
        int v = 0;
        if (tid < n) {
            v = in[a + tid];
            bits[tid] = (unsigned)v;
        }
        __syncthreads();
        if (tid < n) {
            int r = 0;
            for (int j = 0; j < n; ++j) r += (int)bits[j] < v;
            out[a + r] = v;
        }
        return;
    }
    int base = a;
    for (long lo = 0; lo < nboxes; lo += 32L * words) {
        for (int w = tid; w < words; w += 256) bits[w] = 0;
        __syncthreads();
        for (int i = tid; i < n; i += 256) {
            const long b = in[a + i] - lo;
            if (b >= 0 && b < 32L * words) atomicOr(&bits[b >> 5], 1u << (b & 31));
        }
        __syncthreads();
        for (int w0 = 0; w0 < words; w0 += 256) {
            const int w = w0 + tid;
            unsigned x = w < words ? bits[w] : 0u;
            const int c = __popc(x);
            int s = c;
            for (int o = 1; o < 64; o <<= 1) {
                const int y = __shfl_up(s, o);
                if ((tid & 63) >= o) s += y;
            }
            if ((tid & 63) == 63) wsum[tid >> 6] = s;
            __syncthreads();
            int at = base + s - c, all = 0;
            for (int k = 0; k < 4; ++k) {
                if (k < (tid >> 6)) at += wsum[k];
                all += wsum[k];
            }
            while (x) {
                out[at++] = (int)(lo + 32L * w + __ffs(x) - 1);
                x &= x - 1;
            }
            base += all;
            __syncthreads();
        }
    }
}

static void sort_lists(hipStream_t st, int nitems, int nboxes, const dbuf<int> &starts,
                       const dbuf<int> &in, dbuf<int> &out)
{
    const int words = std::max(SORT_RANK, std::min(cdiv(nboxes, 32), SORT_WORDS));
    hipLaunchKernelGGL(k_sort_lists, dim3(nitems), dim3(256), words * sizeof(unsigned), st,
                       starts.p, in.p, out.p, nboxes, words);
}

__global__ void k_box_flags(TV t, const int *tgt_nonchild, int *f_src, int *f_srcpar,
                            int *f_tgt, int *f_ttp)
{
    int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= t.nboxes) return;
    bool leaf = tv_leaf(t, b);
    f_src[b] = (leaf && t.src_nonchild[b] > 0) ? 1 : 0;
    f_srcpar[b] = (!leaf && t.src_cumul[b] > 0) ? 1 : 0;
    int tg = tgt_nonchild[b] > 0 ? 1 : 0;
    f_tgt[b] = tg;
    if (tg)
        for (int a = b; a >= 0; a = t.parent[a]) f_ttp[a] = 1;  // idempotent stores
}

__global__ void k_level_starts(int nlevels, const int *boxes, int n, const int *box_level,
                               int *out)
{
    int l = blockIdx.x * blockDim.x + threadIdx.x;
    if (l > nlevels) return;
    if (l == nlevels) { out[l] = n; return; }
    int lo = 0, hi = n;
    while (lo < hi) {
        int mid = (lo + hi) >> 1;
        if (box_level[boxes[mid]] < l) lo = mid + 1; else hi = mid;
    }
    out[l] = lo;
}

__global__ void k_inverse_map(int n, const int *boxes, int *map)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) map[boxes[i]] = i;
}

// Coarsest box level, into *out: with starts == nullptr over the n list
// entries (boxes named by entries[i]), otherwise over the boxes[i] whose list
// starts[i] .. starts[i + 1] is nonempty.  Minimum per wavefront, then one
// atomic per wavefront.
__global__ void __launch_bounds__(256) k_min_level(int n, const int *entries, const int *starts,
                                                   const int *boxes, const int *level, int *out)
{
    int m = INT_MAX;
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n;
         i += (long)gridDim.x * blockDim.x) {
        if (!starts)
            m = min(m, level[entries[i]]);
        else if (starts[i + 1] > starts[i])
            m = min(m, level[boxes[i]]);
    }
    for (int o = 32; o > 0; o >>= 1) m = min(m, __shfl_xor(m, o));
    if ((threadIdx.x & 63) == 0 && m != INT_MAX) atomicMin(out, m);
}

static void min_level(hipStream_t st, int n, const int *entries, const int *starts,
                      const int *boxes, const int *level, int *out)
{
    if (n <= 0) return;
    const int nb = (int)std::min<long>(cdiv(n, 256), 512);
    hipLaunchKernelGGL(k_min_level, dim3(nb), dim3(256), 0, st, n, entries, starts, boxes, level,
                       out);
}

static int level_starts(hipStream_t st, const qbx_tree *T, const dbuf<int> &boxes, int n,
                        dbuf<int> &d_out, std::vector<int> &h_out)
{
    QBX_TRY(d_out.alloc(T->nlevels + 1));
    hipLaunchKernelGGL(k_level_starts, dim3(1), dim3(MAX_LEVELS + 1), 0, st, T->nlevels,
                       boxes.p, n, T->box_levels.p, d_out.p);
    QBX_HIP(hipGetLastError());
    h_out.resize(T->nlevels + 1);
    QBX_HIP(hipMemcpyAsync(h_out.data(), d_out.p, sizeof(int) * (T->nlevels + 1),
                           hipMemcpyDeviceToHost, st));
    QBX_HIP(hipStreamSynchronize(st));
    return QBX_OK;
}

// starts, and room for the lists as they are found (raw) and sorted
static int build_lists(qbx_ctx *ctx, hipStream_t st, int nitems, dbuf<int> &starts,
                       dbuf<int> &raw, dbuf<int> &lists, int *total, dbuf<int> &cnt)
{
    QBX_TRY(starts.alloc(nitems + 1));
    QBX_TRY(exclusive_scan(ctx, st, cnt.p, starts.p, nitems, total));
    QBX_TRY(raw.alloc(std::max(*total, 1)));
    QBX_TRY(lists.alloc(std::max(*total, 1)));
    lists.n = *total;
    return QBX_OK;
}

static int traverse(qbx_ctx *ctx, hipStream_t st, const qbx_tree *T, int n, int ext,
                    int minsrc, qbx_trav *R)
{
    TV t;
    t.dim = T->dim;
    t.nboxes = T->nboxes;
    t.nlevels = T->nlevels;
    t.level = T->box_levels.p;
    t.parent = T->box_parent_ids.p;
    t.child = T->box_child_ids.p;
    t.coords = T->box_coords.p;
    t.lstart = T->d_level_start_box_nrs.p;
    t.morton = T->box_morton.p;
    t.src_nonchild = T->box_source_counts_nonchild.p;
    t.src_cumul = T->box_source_counts_cumul.p;
    int nb = T->nboxes;
    R->nlevels = T->nlevels;
    R->nsep = n;

    dbuf<int> f_src, f_srcpar, f_tgt, f_ttp;
    QBX_TRY(f_src.alloc(nb));
    QBX_TRY(f_srcpar.alloc(nb));
    QBX_TRY(f_tgt.alloc(nb));
    QBX_TRY(f_ttp.alloc(nb));
    QBX_HIP(hipMemsetAsync(f_ttp.p, 0, sizeof(int) * nb, st));
    hipLaunchKernelGGL(k_box_flags, dim3(cdiv(nb, 256)), dim3(256), 0, st, t,
                       T->box_target_counts_nonchild.p, f_src.p, f_srcpar.p, f_tgt.p, f_ttp.p);
    QBX_HIP(hipGetLastError());
    QBX_TRY(compact_indices(ctx, st, f_src.p, nb, R->source_boxes, &R->nsource_boxes));
    QBX_TRY(compact_indices(ctx, st, f_srcpar.p, nb, R->source_parent_boxes,
                            &R->nsource_parent_boxes));
    QBX_TRY(compact_indices(ctx, st, f_tgt.p, nb, R->target_boxes, &R->ntarget_boxes));
    QBX_TRY(compact_indices(ctx, st, f_ttp.p, nb, R->ttp_boxes, &R->nttp_boxes));
    QBX_TRY(level_starts(st, T, R->source_boxes, R->nsource_boxes, R->level_start_source_box_nrs,
                         R->h_level_start_source_box_nrs));
    QBX_TRY(level_starts(st, T, R->source_parent_boxes, R->nsource_parent_boxes,
                         R->level_start_source_parent_box_nrs,
                         R->h_level_start_source_parent_box_nrs));
    QBX_TRY(level_starts(st, T, R->target_boxes, R->ntarget_boxes, R->level_start_target_box_nrs,
                         R->h_level_start_target_box_nrs));
    QBX_TRY(level_starts(st, T, R->ttp_boxes, R->nttp_boxes, R->level_start_ttp_box_nrs,
                         R->h_level_start_ttp_box_nrs));
    QBX_TRY(R->box_to_ttp.alloc(nb));
    QBX_TRY(R->box_to_target_box.alloc(nb));
    QBX_HIP(hipMemsetAsync(R->box_to_ttp.p, 0xff, sizeof(int) * nb, st));
    QBX_HIP(hipMemsetAsync(R->box_to_target_box.p, 0xff, sizeof(int) * nb, st));
    if (R->nttp_boxes)
        hipLaunchKernelGGL(k_inverse_map, dim3(cdiv(R->nttp_boxes, 256)), dim3(256), 0, st,
                           R->nttp_boxes, R->ttp_boxes.p, R->box_to_ttp.p);
    if (R->ntarget_boxes)
        hipLaunchKernelGGL(k_inverse_map, dim3(cdiv(R->ntarget_boxes, 256)), dim3(256), 0, st,
                           R->ntarget_boxes, R->target_boxes.p, R->box_to_target_box.p);
    QBX_HIP(hipGetLastError());

    // lists 1 and 3
    {
        int ntb = R->ntarget_boxes;
        const size_t stack = sizeof(int) * 64 * (size_t)T->nlevels << T->dim;
        dbuf<int> c1, c3, r1, r3;
        QBX_TRY(c1.alloc(std::max(ntb, 1)));
        QBX_TRY(c3.alloc(std::max(ntb, 1)));
        ListOut o1{c1.p, nullptr, nullptr, 0}, o3{c3.p, nullptr, nullptr, 0};
        if (ntb)
            hipLaunchKernelGGL(k_list13, dim3(ntb), dim3(64), stack, st, t, n, ext, minsrc, ntb,
                               R->target_boxes.p, o1, o3);
        QBX_HIP(hipGetLastError());
        QBX_TRY(build_lists(ctx, st, ntb, R->l1_starts, r1, R->l1_lists, &R->n1, c1));
        QBX_TRY(build_lists(ctx, st, ntb, R->l3_starts, r3, R->l3_lists, &R->n3, c3));
        o1 = ListOut{nullptr, R->l1_starts.p, r1.p, 1};
        o3 = ListOut{nullptr, R->l3_starts.p, r3.p, 1};
        if (ntb) {
            hipLaunchKernelGGL(k_list13, dim3(ntb), dim3(64), stack, st, t, n, ext, minsrc, ntb,
                               R->target_boxes.p, o1, o3);
            sort_lists(st, ntb, nb, R->l1_starts, r1, R->l1_lists);
            sort_lists(st, ntb, nb, R->l3_starts, r3, R->l3_lists);
        }
        QBX_HIP(hipGetLastError());
    }
    // lists 2 and 4
    {
        int nt = R->nttp_boxes;
        dbuf<int> c2, c4, r2, r4;
        QBX_TRY(c2.alloc(std::max(nt, 1)));
        QBX_TRY(c4.alloc(std::max(nt, 1)));
        ListOut o2{c2.p, nullptr, nullptr, 0}, o4{c4.p, nullptr, nullptr, 0};
        if (nt)
            hipLaunchKernelGGL(k_list24, dim3(nt), dim3(64), 0, st, t, n, nt, R->ttp_boxes.p, o2,
                               o4);
        QBX_HIP(hipGetLastError());
        QBX_TRY(build_lists(ctx, st, nt, R->l2_starts, r2, R->l2_lists, &R->n2, c2));
        QBX_TRY(build_lists(ctx, st, nt, R->l4_starts, r4, R->l4_lists, &R->n4, c4));
        o2 = ListOut{nullptr, R->l2_starts.p, r2.p, 1};
        o4 = ListOut{nullptr, R->l4_starts.p, r4.p, 1};
        if (nt) {
            hipLaunchKernelGGL(k_list24, dim3(nt), dim3(64), 0, st, t, n, nt, R->ttp_boxes.p, o2,
                               o4);
            sort_lists(st, nt, nb, R->l2_starts, r2, R->l2_lists);
            sort_lists(st, nt, nb, R->l4_starts, r4, R->l4_lists);
        }
        QBX_HIP(hipGetLastError());
    }
    // the coarsest levels: qbx_trav::mpole_min_level and local_min_level
    dbuf<int> coarsest;
    QBX_TRY(coarsest.alloc(2));
    const int none[2] = {T->nlevels, T->nlevels};
    QBX_HIP(hipMemcpyAsync(coarsest.p, none, sizeof(none), hipMemcpyHostToDevice, st));
    min_level(st, R->n2, R->l2_lists.p, nullptr, nullptr, T->box_levels.p, coarsest.p);
    min_level(st, R->n3, R->l3_lists.p, nullptr, nullptr, T->box_levels.p, coarsest.p);
    min_level(st, R->nttp_boxes, nullptr, R->l2_starts.p, R->ttp_boxes.p, T->box_levels.p,
              coarsest.p + 1);
    min_level(st, R->nttp_boxes, nullptr, R->l4_starts.p, R->ttp_boxes.p, T->box_levels.p,
              coarsest.p + 1);
    QBX_HIP(hipGetLastError());
    int hc[2] = {0, 0};
    QBX_HIP(hipMemcpyAsync(hc, coarsest.p, sizeof(hc), hipMemcpyDeviceToHost, st));
    QBX_HIP(hipStreamSynchronize(st));
    R->mpole_min_level = hc[0];
    R->local_min_level = hc[1];
    return QBX_OK;
}

struct TFieldRef {
    const void *p;
    long bytes;
};

static TFieldRef trav_field(const qbx_trav *r, const char *f)
{
    std::string s(f);
    auto I = [&](const dbuf<int> &b, long n) { return TFieldRef{b.p, (long)sizeof(int) * n}; };
    int L1 = r->nlevels + 1;
    if (s == "source_boxes") return I(r->source_boxes, r->nsource_boxes);
    if (s == "source_parent_boxes") return I(r->source_parent_boxes, r->nsource_parent_boxes);
    if (s == "target_boxes") return I(r->target_boxes, r->ntarget_boxes);
    if (s == "target_or_target_parent_boxes") return I(r->ttp_boxes, r->nttp_boxes);
    if (s == "level_start_source_box_nrs") return I(r->level_start_source_box_nrs, L1);
    if (s == "level_start_source_parent_box_nrs") return I(r->level_start_source_parent_box_nrs, L1);
    if (s == "level_start_target_box_nrs") return I(r->level_start_target_box_nrs, L1);
    if (s == "level_start_target_or_target_parent_box_nrs") return I(r->level_start_ttp_box_nrs, L1);
    if (s == "neighbor_source_boxes_starts") return I(r->l1_starts, r->ntarget_boxes + 1);
    if (s == "neighbor_source_boxes_lists") return I(r->l1_lists, r->n1);
    if (s == "from_sep_siblings_starts") return I(r->l2_starts, r->nttp_boxes + 1);
    if (s == "from_sep_siblings_lists") return I(r->l2_lists, r->n2);
    if (s == "from_sep_smaller_starts") return I(r->l3_starts, r->ntarget_boxes + 1);
    if (s == "from_sep_smaller_lists") return I(r->l3_lists, r->n3);
    if (s == "from_sep_bigger_starts") return I(r->l4_starts, r->nttp_boxes + 1);
    if (s == "from_sep_bigger_lists") return I(r->l4_lists, r->n4);
    return TFieldRef{nullptr, -1};
}

}  // namespace qbx

using namespace qbx;

extern "C" {

int qbx_traverse(qbx_ctx *ctx, void *stream, const qbx_tree *tree, int well_sep_is_n_away,
                 int targets_have_extent, int from_sep_smaller_min_nsources_cumul,
                 qbx_trav **out)
{
    QBX_CHECK(ctx && tree && out, "qbx_traverse: null argument");
    QBX_CHECK(well_sep_is_n_away >= 1 && well_sep_is_n_away <= 3,
              "qbx_traverse: well_sep_is_n_away must be in [1, 3]");
    qbx_trav *R = new qbx_trav();
    int rc = traverse(ctx, S(stream), tree, well_sep_is_n_away, targets_have_extent ? 1 : 0,
                      from_sep_smaller_min_nsources_cumul, R);
    if (rc != QBX_OK) {
        delete R;
        return rc;
    }
    *out = R;
    return QBX_OK;
}

int qbx_trav_destroy(qbx_trav *t)
{
    delete t;
    return QBX_OK;
}

int qbx_trav_sizes(const qbx_trav *r, int *c)
{
    QBX_CHECK(r && c, "qbx_trav_sizes: null argument");
    c[0] = r->nsource_boxes;
    c[1] = r->nsource_parent_boxes;
    c[2] = r->ntarget_boxes;
    c[3] = r->nttp_boxes;
    c[4] = r->n1;
    c[5] = r->n2;
    c[6] = r->n3;
    c[7] = r->n4;
    return QBX_OK;
}

long qbx_trav_field_bytes(const qbx_trav *r, const char *field)
{
    if (!r || !field) return -1;
    return trav_field(r, field).bytes;
}

int qbx_trav_export(const qbx_trav *r, const char *field, void *dst, long nbytes, void *stream)
{
    QBX_CHECK(r && field, "qbx_trav_export: null argument");
    TFieldRef f = trav_field(r, field);
    QBX_CHECK(f.bytes >= 0, "qbx_trav_export: unknown field '%s'", field);
    QBX_CHECK(nbytes >= f.bytes, "qbx_trav_export: '%s' needs %ld bytes", field, f.bytes);
    if (f.bytes > 0)
        QBX_HIP(hipMemcpyAsync(dst, f.p, f.bytes, hipMemcpyDeviceToDevice, S(stream)));
    return QBX_OK;
}

}  // extern "C"
