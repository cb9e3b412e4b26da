// Device side of mesh creation: the sliced and blocked layouts that the
// kernels read are filled on the GPU from the caller's lists, which cross to
// the device once and as they are.  The host keeps what is sequential (orders,
// row offsets, colours, levels).
//
// Every kernel here moves each entry once and is bound by memory.  What they
// replace was bound by the host: for 16 cases of 48k nodes (763k nodes, 5.1M
// edges) cfd_mesh_create took 192 ms, with host passes over fresh pages and
// 0.75 GB of uploads, and takes 80 ms, with 0.30 GB of uploads and 2 ms in
// the kernels of this file.
#include "cfd_internal.h"

namespace {

constexpr int kBlock = 256;

// An incidence while its node's list is put in order: twice the index of the
// edge (E + b for boundary edge b), plus one at the R end of an interior edge.
__device__ __forceinline__ uint32_t inc_key(int e, int side) { return 2 * (uint32_t)e + (uint32_t)side; }

struct IncArgs {
    int N, E, B;
    const int *edge, *bedge;       // caller's numbering
    const double *earea, *barea;
    const int *iperm, *ip, *sptr;
    int *fill;                     // [N] incidences found (starts at zero)
    uint32_t *key;                 // SELL, becomes the edge indices
    int *nbr;
    double *sx, *sy, *sz;
    unsigned long long *bad;       // smallest internal node whose list does not fit its edges (starts at ~0)
};

// Each edge enters itself in the lists of its nodes, in any order.
__global__ __launch_bounds__(kBlock) void k_inc_edges(IncArgs a) {
    const int t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= a.E + a.B) return;
    const bool inner = t < a.E;
    for (int side = 0; side < (inner ? 2 : 1); side++) {
        const int i = a.iperm[inner ? a.edge[2 * (size_t)t + side] : a.bedge[2 * (size_t)(t - a.E)]];
        const int k = atomicAdd(&a.fill[i], 1);
        if (k < a.ip[i + 1] - a.ip[i])
            a.key[(size_t)a.sptr[i / kSlice] + (size_t)kSlice * k + i % kSlice] = inc_key(t, side);
    }
}

// Lists up to this length are sorted in LDS (one column a lane: tetrahedral
// meshes have 14 neighbours a node), longer ones by the whole wavefront where
// they are.
constexpr int kSortLds = 32;

// Ascending sort of n items by a workgroup of one wavefront: order(lo, hi) puts
// items lo < hi in order.  Bitonic merges whose comparators all put the larger
// item behind, so items past n (larger than any) stay where they are and need
// not exist.
template <class F>
__device__ void wave_sort(uint32_t n, F order) {
    auto order2 = [&](uint32_t lo, uint32_t hi) {
        if (hi < n) order(lo, hi);
    };
    uint32_t n2 = 1;
    while (n2 < n) n2 *= 2;
    for (uint32_t size = 2; size <= n2; size *= 2) {
        const uint32_t half = size / 2;
        for (uint32_t p = threadIdx.x; p < n2 / 2; p += kSlice) {
            const uint32_t g = p / half * size, j = p % half;
            order2(g + j, g + size - 1 - j);
        }
        __syncthreads();
        for (uint32_t stride = half / 2; stride; stride /= 2) {
            for (uint32_t p = threadIdx.x; p < n2 / 2; p += kSlice) {
                const uint32_t lo = p / stride * 2 * stride + p % stride;
                order2(lo, lo + stride);
            }
            __syncthreads();
        }
    }
}

// One wavefront a slice, one lane a node, so the layout is written in full
// lines: the node's list in edge order with neighbour and area vector.
__global__ __launch_bounds__(kSlice) void k_inc_lists(IncArgs a) {
    __shared__ uint32_t col[kSortLds][kSlice];
    const int sl = blockIdx.x, i = sl * kSlice + threadIdx.x;
    const size_t base = (size_t)a.sptr[sl] + threadIdx.x;
    const int w = (a.sptr[sl + 1] - a.sptr[sl]) / kSlice;
    int cnt = i < a.N ? a.ip[i + 1] - a.ip[i] : 0;
    if (i < a.N && a.fill[i] != cnt) {
        atomicMin(a.bad, (unsigned long long)i);
        cnt = 0;
    }
    const bool lds = cnt <= kSortLds;
    if (lds) {
        for (int k = 0; k < cnt; k++) {
            const uint32_t x = a.key[base + (size_t)kSlice * k];
            int q = k;
            for (; q > 0 && col[q - 1][threadIdx.x] > x; q--) col[q][threadIdx.x] = col[q - 1][threadIdx.x];
            col[q][threadIdx.x] = x;
        }
    }
    for (uint64_t hubs = __ballot(!lds); hubs; hubs &= hubs - 1) {
        const int l = __ffsll((unsigned long long)hubs) - 1;
        uint32_t *const v = a.key + a.sptr[sl] + l;
        wave_sort((uint32_t)__shfl(cnt, l), [&](uint32_t lo, uint32_t hi) {
            uint32_t &p = v[(size_t)kSlice * lo], &q = v[(size_t)kSlice * hi];
            const uint32_t x = p, y = q;
            if (y < x) {
                p = y;
                q = x;
            }
        });
    }
    for (int k = 0; k < w; k++) {
        const size_t x = base + (size_t)kSlice * k;
        int nb = 0, e = -1;  // padding, never read
        double s0 = 0.0, s1 = 0.0, s2 = 0.0;
        if (k < cnt) {
            const uint32_t key = lds ? col[k][threadIdx.x] : a.key[x];
            e = (int)(key >> 1);
            const double *S;
            if (e >= a.E) {
                nb = a.N + (e - a.E);
                S = a.barea + 3 * (size_t)(e - a.E);
            } else {
                const int side = key & 1, j = a.iperm[a.edge[2 * (size_t)e + 1 - side]];
                nb = side ? ~j : j;
                S = a.earea + 3 * (size_t)e;
            }
            s0 = S[0];
            s1 = S[1];
            s2 = S[2];
        }
        a.key[x] = (uint32_t)e;
        a.nbr[x] = nb;
        a.sx[x] = s0;
        a.sy[x] = s1;
        a.sz[x] = s2;
    }
}

// BSR block (row of the node, column of the neighbour) of each incidence.
// miss: (node << 32 | neighbour) of the first node, and of its first
// neighbour, without one (starts at ~0).
__global__ __launch_bounds__(kBlock) void k_off_slots(int N, const int *__restrict__ ip, const int *__restrict__ sptr,
                                                      const int *__restrict__ nbr, const int *__restrict__ order,
                                                      const int *__restrict__ ia, const int *__restrict__ ja,
                                                      int *__restrict__ soff, unsigned long long *miss) {
    const int ii = blockIdx.x * kBlock + threadIdx.x, sl = ii / kSlice;
    if (sl >= (N + kSlice - 1) / kSlice) return;
    const size_t base = (size_t)sptr[sl] + ii % kSlice;
    const int w = (sptr[sl + 1] - sptr[sl]) / kSlice;
    const int cnt = ii < N ? ip[ii + 1] - ip[ii] : 0;
    const int i = ii < N ? order[ii] : 0;
    const int b0 = ia[i], b1 = ia[i + 1];
    bool whole = true;
    for (int k = 0; k < w; k++) {
        const size_t x = base + (size_t)kSlice * k;
        int slot = -1;
        if (k < cnt && nbr[x] < N) {
            const int j = order[nbr[x] < 0 ? ~nbr[x] : nbr[x]];
            int lo = b0, hi = b1;
            while (lo < hi) {
                const int mid = lo + (hi - lo) / 2;
                if (ja[mid] < j) lo = mid + 1;
                else hi = mid;
            }
            if (lo < b1 && ja[lo] == j) {
                slot = lo;
            } else if (whole) {
                atomicMin(miss, (unsigned long long)ii << 32 | (unsigned)j);
                whole = false;
            }
        }
        soff[x] = slot;
    }
}

// Block-SELL pattern of the slots first(i) .. last(i)-1 of each row: column 0
// and source -1 in padding.
__global__ __launch_bounds__(kBlock) void k_block_sell(int n, BsrPart part, const int *__restrict__ ia,
                                                       const int *__restrict__ iau, const int *__restrict__ ja,
                                                       const int *__restrict__ off, int *__restrict__ col,
                                                       int *__restrict__ src) {
    const int i = blockIdx.x * kBlock + threadIdx.x, sl = i / 64;
    if (sl >= (n + 63) / 64) return;
    const int w = (off[sl + 1] - off[sl]) / 64;
    int b = 0, e = 0;
    if (i < n) {
        b = part == BsrPart::kUpper ? iau[i] + 1 : ia[i];
        e = part == BsrPart::kLower ? iau[i] : ia[i + 1];
    }
    for (int k = 0; k < w; k++) {
        const size_t q = (size_t)off[sl] + 64 * (size_t)k + i % 64;
        const bool in = k < e - b;
        col[q] = in ? ja[b + k] : 0;
        src[q] = in ? b + k : -1;
    }
}

// Multicolour pattern: row t is row perm[t] with its blocks in ascending new
// column (src: the slot a block comes from; equal columns keep their order).
// A block's place is the number of blocks before it, counted in LDS by the
// row's lane; rows that do not fit are sorted where they are by the whole
// wavefront (counting took 0.5 s for a row of 15,000 blocks).
__global__ __launch_bounds__(kSlice) void k_mc_pattern(int N, const int *__restrict__ perm,
                                                       const int *__restrict__ iperm, const int *__restrict__ ia,
                                                       const int *__restrict__ ja, const int *__restrict__ mia,
                                                       int *mja, int *__restrict__ miau, int *src) {
    __shared__ int col[kSortLds][kSlice];
    const int lane = threadIdx.x, t = blockIdx.x * kSlice + lane;
    int from = 0, to = 0, n = 0;
    if (t < N) {
        from = ia[perm[t]];
        n = ia[perm[t] + 1] - from;
        to = mia[t];
    }
    const bool lds = n <= kSortLds;
    if (lds) {
        for (int k = 0; k < n; k++) col[k][lane] = iperm[ja[from + k]];
        for (int k = 0; k < n; k++) {
            const int c = col[k][lane];
            int q = to;
            for (int u = 0; u < n; u++) q += col[u][lane] < c || (col[u][lane] == c && u < k);
            mja[q] = c;
            src[q] = from + k;
            if (c == t) miau[t] = q;
        }
    }
    for (uint64_t big = __ballot(!lds); big; big &= big - 1) {
        const int l = __ffsll((unsigned long long)big) - 1;
        const int f = __shfl(from, l), m = __shfl(n, l), o = __shfl(to, l), row = blockIdx.x * kSlice + l;
        int *const c = mja + o, *const b = src + o;
        for (int k = lane; k < m; k += kSlice) {
            c[k] = iperm[ja[f + k]];
            b[k] = f + k;
        }
        __syncthreads();
        wave_sort((uint32_t)m, [&](uint32_t lo, uint32_t hi) {
            const int x = c[lo], y = c[hi], p = b[lo], q = b[hi];
            if (y < x || (y == x && q < p)) {
                c[lo] = y;
                c[hi] = x;
                b[lo] = q;
                b[hi] = p;
            }
        });
        for (int k = lane; k < m; k += kSlice)
            if (c[k] == row) miau[row] = o + k;
    }
}

// Levels of the upper sweep of the rows [r0, r1) of one colour, the later
// colours' being there: one more than the largest of the rows it needs.
__global__ __launch_bounds__(kBlock) void k_mc_levels(int r0, int r1, const int *__restrict__ mia,
                                                      const int *__restrict__ miau, const int *__restrict__ mja,
                                                      int *lev) {
    const int t = r0 + blockIdx.x * kBlock + threadIdx.x;
    if (t >= r1) return;
    int l = 0;
    for (int k = miau[t] + 1; k < mia[t + 1]; k++) l = max(l, lev[mja[k]] + 1);
    lev[t] = l;
}

// Neighbour lists in internal numbering, the order within a list unchanged.
__global__ __launch_bounds__(kBlock) void k_neighbours(int N, const int *__restrict__ order,
                                                       const int *__restrict__ iperm, const int *__restrict__ ria,
                                                       const int *__restrict__ rja, const int *__restrict__ nia,
                                                       int *__restrict__ nja) {
    const int ii = blockIdx.x * kBlock + threadIdx.x;
    if (ii >= N) return;
    const int r = ria[order[ii]], b = nia[ii], n = nia[ii + 1] - b;
    for (int k = 0; k < n; k++) nja[b + k] = iperm[rja[r + k]];
}

struct Five {
    double v[5];
};

// Node records: freestream state, coordinates (none in ghosts), and volumes.
__global__ __launch_bounds__(kBlock) void k_node_records(int N, int NT, const int *__restrict__ order,
                                                         const double *__restrict__ xyz,
                                                         const double *__restrict__ vref, Five q,
                                                         double *__restrict__ qa, double *__restrict__ vol) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= NT) return;
    const int r = i < N ? order[i] : 0;
    for (int k = 0; k < 5; k++) qa[(size_t)kQA * i + k] = q.v[k];
    for (int k = 0; k < 3; k++) qa[(size_t)kQA * i + 5 + k] = i < N ? xyz[3 * (size_t)r + k] : 0.0;
    if (i < N) vol[i] = vref[r];
}

// ---------------------------------------------------------------------------
// Work-edge patches in node order (PatchSet).  A work edge belongs to its
// first end in the patch, so it is in that node's own incidence list and its
// place among the node's work edges is a count over that list: by (L, R), and
// among equal pairs by place in the list.  Both ends of an edge count the same
// place, so no lane waits for another and nothing is sorted but a node's slots.
// The lists are short and their neighbours' are near (Morton order): the counts
// are reads of cached lines.  4.17M nodes (41M work edges): 3.7 ms and 0.1 ms
// in the kernels, 6 ms in all; the host's build, with the lists fetched from
// the device and the arrays sent back, took 800 ms.
// ---------------------------------------------------------------------------
struct WorkEdge {
    uint64_t lr;  // L << 32 | R
    int owner;
};

// Incidence nb of node i, in the patch of nodes [n0, n1).
__device__ __forceinline__ WorkEdge work_edge(int i, int nb, int N, int n0, int n1) {
    const bool left = nb >= 0;
    const int j = left ? nb : ~nb;
    const bool inside = j < N && j >= n0 && j < n1;
    const uint32_t l = left ? i : j, r = left ? j : i;
    return {(uint64_t)l << 32 | r, inside && j < i ? j : i};
}

// own[i]: work edges of the patch that belong to nodes before i; cnt[p]: of patch p.
__global__ __launch_bounds__(kPatch) void k_patch_own(PatchBuild a) {
    __shared__ int part[kPatch];
    const int p = blockIdx.x, t = threadIdx.x, n0 = a.pstart[p], n1 = a.pstart[p + 1], i = n0 + t;
    int c = 0;
    if (i < n1) {
        const int *const nb = a.nbr + a.sptr[i / kSlice] + i % kSlice;
        for (int k = a.ip[i + 1] - a.ip[i] - 1; k >= 0; k--)
            c += work_edge(i, nb[(size_t)kSlice * k], a.N, n0, n1).owner == i;
    }
    part[t] = c;
    for (int d = 1; d < kPatch; d *= 2) {
        __syncthreads();
        const int before = t >= d ? part[t - d] : 0;
        __syncthreads();
        part[t] += before;
    }
    if (i < n1) a.own[i] = part[t] - c;
    if (t == kPatch - 1) a.cnt[p] = part[t];
}

// One wavefront a slice, one lane a node: the node's work edges, and its slots
// in ascending order (dynamic LDS: one column a lane, as long as the slice is wide).
__global__ __launch_bounds__(kSlice) void k_patch_edges(PatchBuild a) {
    extern __shared__ uint32_t slots[];
    const int sl = blockIdx.x, lane = threadIdx.x, i = sl * kSlice + lane;
    const size_t base = (size_t)a.sptr[sl] + lane;
    const int w = (a.sptr[sl + 1] - a.sptr[sl]) / kSlice;
    int cnt = 0;
    if (i < a.N) {
        cnt = a.ip[i + 1] - a.ip[i];
        int p = 0;  // the patch: pstart[p] <= i < pstart[p + 1]
        for (int hi = a.P; hi - p > 1;) {
            const int mid = p + (hi - p) / 2;
            if (a.pstart[mid] <= i) p = mid;
            else hi = mid;
        }
        const int n0 = a.pstart[p], n1 = a.pstart[p + 1];
        for (int k = 0; k < cnt; k++) {
            const size_t x = base + (size_t)kSlice * k;
            const WorkEdge e = work_edge(i, a.nbr[x], a.N, n0, n1);
            int q = a.own[e.owner];
            for (int u = 0; u < k; u++) q += work_edge(i, a.nbr[base + (size_t)kSlice * u], a.N, n0, n1).lr == e.lr;
            const int *const nb = a.nbr + a.sptr[e.owner / kSlice] + e.owner % kSlice;
            for (int u = a.ip[e.owner + 1] - a.ip[e.owner] - 1; u >= 0; u--) {
                const WorkEdge o = work_edge(e.owner, nb[(size_t)kSlice * u], a.N, n0, n1);
                q += o.owner == e.owner && o.lr < e.lr;
            }
            const int r = (int)(uint32_t)e.lr;
            if (e.owner == i) {
                const size_t o = (size_t)a.wptr[p] + q;
                a.wl[o] = (int)(e.lr >> 32);
                a.wr[o] = r;
                a.ws[3 * o] = a.sx[x];
                a.ws[3 * o + 1] = a.sy[x];
                a.ws[3 * o + 2] = a.sz[x];
            }
            const uint32_t v = 2 * (uint32_t)q + (r == i);
            int b = k;
            for (; b > 0 && slots[(b - 1) * kSlice + lane] > v; b--)
                slots[b * kSlice + lane] = slots[(b - 1) * kSlice + lane];
            slots[b * kSlice + lane] = v;
        }
    }
    for (int k = 0; k < w; k++) {
        const uint32_t v = k < cnt ? slots[k * kSlice + lane] : 0;
        a.slot[base + (size_t)kSlice * k] = (int)(v >> 1 | v << 31);  // sign bit: the node is R
    }
}

__global__ __launch_bounds__(kBlock) void k_to_float(size_t n, const double *__restrict__ in, float *__restrict__ out) {
    const size_t i = blockIdx.x * (size_t)kBlock + threadIdx.x;
    if (i < n) out[i] = (float)in[i];
}

inline dim3 blocks(int64_t n) { return dim3((unsigned)((n + kBlock - 1) / kBlock)); }

}  // namespace

int launch_incidences(cfd_mesh *m, const IncidenceInput &in) {
    IncArgs a{m->N, m->E, m->B, in.edge, in.bedge, in.earea, in.barea, m->iperm, m->inc_ptr, m->sptr, in.fill,
              (uint32_t *)m->sell_edge, m->nbr, m->d.isx, m->d.isy, m->d.isz, in.bad};
    if (m->E + m->B) hipLaunchKernelGGL(k_inc_edges, blocks((int64_t)m->E + m->B), dim3(kBlock), 0, m->stream, a);
    hipLaunchKernelGGL(k_inc_lists, dim3((m->N + kSlice - 1) / kSlice), dim3(kSlice), 0, m->stream, a);
    CFD_HIP(m, hipGetLastError());
    return CFD_OK;
}

int launch_off_slots(cfd_mesh *m, unsigned long long *miss) {
    hipLaunchKernelGGL(k_off_slots, blocks(m->N), dim3(kBlock), 0, m->stream, m->N, m->inc_ptr, m->sptr, m->nbr,
                       m->order, m->ia, m->ja, m->soff, miss);
    CFD_HIP(m, hipGetLastError());
    return CFD_OK;
}

int launch_block_sell(cfd_mesh *m, BsrPart part, const int *ia, const int *iau, const int *ja, const BlockSell &bs) {
    hipLaunchKernelGGL(k_block_sell, blocks(m->N), dim3(kBlock), 0, m->stream, m->N, part, ia, iau, ja, bs.off, bs.col,
                       bs.src);
    CFD_HIP(m, hipGetLastError());
    return CFD_OK;
}

int launch_mc_pattern(cfd_mesh *m, const int *iperm, int *lev) {
    hipLaunchKernelGGL(k_mc_pattern, dim3((m->N + kSlice - 1) / kSlice), dim3(kSlice), 0, m->stream, m->N, m->mc_perm,
                       iperm, m->ia, m->ja, m->mc_ia, m->mc_ja, m->mc_iau, m->mc_src);
    for (int c = m->ncolor - 1; c >= 0; c--) {
        const int r0 = m->mc_cstart[c], r1 = m->mc_cstart[c + 1];
        if (r1 > r0)
            hipLaunchKernelGGL(k_mc_levels, blocks(r1 - r0), dim3(kBlock), 0, m->stream, r0, r1, m->mc_ia, m->mc_iau,
                               m->mc_ja, lev);
    }
    CFD_HIP(m, hipGetLastError());
    return CFD_OK;
}

int launch_neighbours(cfd_mesh *m, const int *ref_ia, const int *ref_ja) {
    hipLaunchKernelGGL(k_neighbours, blocks(m->N), dim3(kBlock), 0, m->stream, m->N, m->order, m->iperm, ref_ia, ref_ja,
                       m->n2n_ia, m->n2n_ja);
    CFD_HIP(m, hipGetLastError());
    return CFD_OK;
}

int launch_node_records(cfd_mesh *m, const double *xyz, const double *vol, const double *q5) {
    Five q;
    for (int k = 0; k < 5; k++) q.v[k] = q5[k];
    hipLaunchKernelGGL(k_node_records, blocks(m->NT), dim3(kBlock), 0, m->stream, m->N, m->NT, m->order, xyz, vol, q,
                       m->d.qa, m->d.vol);
    CFD_HIP(m, hipGetLastError());
    return CFD_OK;
}

int launch_patch_own(cfd_mesh *m, const PatchBuild &a) {
    hipLaunchKernelGGL(k_patch_own, dim3(a.P), dim3(kPatch), 0, m->stream, a);
    CFD_HIP(m, hipGetLastError());
    return CFD_OK;
}

int launch_patch_edges(cfd_mesh *m, const PatchBuild &a) {
    hipLaunchKernelGGL(k_patch_edges, dim3((m->N + kSlice - 1) / kSlice), dim3(kSlice),
                       sizeof(uint32_t) * kSlice * (size_t)m->widest, m->stream, a);
    CFD_HIP(m, hipGetLastError());
    return CFD_OK;
}

int launch_to_float(cfd_mesh *m, size_t n, const double *in, float *out) {
    if (n) hipLaunchKernelGGL(k_to_float, blocks((int64_t)n), dim3(kBlock), 0, m->stream, n, in, out);
    CFD_HIP(m, hipGetLastError());
    return CFD_OK;
}
