// dhip_batch.hpp -- many independent P1 trace-FEM problems assembled and solved together.
//
// Each problem has its own Kuhn brick, level set and sizes.  The assembly runs step by step over all
// problems at once with the single-problem path's per-item code (cell_cut_mask, local_p1_one, qualify_one,
// first_one, row_wave), so every assembled array equals what the single-problem entry points produce.
// Then one workgroup owns one problem at a time and runs a Jacobi PCG with FP32 inner iterations and FP64
// refinement, with workgroup barriers only; workgroups take problems from a queue ordered largest first
// (longest-processing-time order), so uneven sizes balance over the grid.
//
//   k_batch_cells / k_batch_verts   planning: cut tets and cut-tet vertices per problem (sizes of
//                                   the per-problem scratch; the rows of a problem are at most its
//                                   cut-tet vertices, each row has at most 15 entries)
//   k_batch_cut_count .. k_batch_rows   assembly, every step over all problems
//   k_batch_solve                   the PCGs, one problem per CU at a time, largest first
#pragma once

#include "dhip_assembly.hpp"
#include "dhip_krylov.hpp"

namespace dhip {

struct BatchProb {
    MeshP m;
    int64_t phi_off;    // first level-set value of the problem
    int64_t cell_off;   // first cell word
    int64_t cut_off;    // first cut-tet slot (capacity ncut_cap)
    int64_t ncut_cap;
    int64_t row_off;    // first row slot (capacity row_cap; row pointers at row_off + problem index)
    int64_t row_cap;
    int64_t nz_off;     // first entry slot (capacity nz_cap)
    int64_t nz_cap;
    double lc[3];       // the solved operator combination
    int64_t sell_off;   // first SELL-64 slot (capacity 16 * 64 * ceil(row_cap / 64) + 16 * BPT)
    int64_t slice_off;  // first slice offset (capacity ceil(row_cap / 64) + 1)
};

struct BatchStat {
    int32_t status;     // DHIP_OK, DHIP_E_NOT_CONVERGED, DHIP_E_ZERO_NODE, DHIP_E_ZERO_PATTERN, DHIP_E_CAPACITY
    int32_t ncut, ndof, nnz;
    int32_t iters, outer;
    double resid;
    uint64_t t0, t1;    // wall clock (100 MHz) at the start and end of the problem
    uint64_t t_asm;     // wall clock when its CSR system was complete
};

// ---------------------------------------------------------------------------
// planning
// ---------------------------------------------------------------------------
constexpr int BPLAN = 256;

__global__ void __launch_bounds__(BPLAN) k_batch_cells(const BatchProb *prob, const double *phi, uint8_t *mask,
                                                       int32_t *ncut, int32_t *zero) {
    const BatchProb &P = prob[blockIdx.y];
    const int64_t cell = (int64_t)blockIdx.x * BPLAN + threadIdx.x;
    int mk = 0;
    bool z = false;
    if (cell < P.m.ncell) {
        mk = cell_cut_mask(P.m, phi + P.phi_off, cell, z);
        mask[P.cell_off + cell] = (uint8_t)mk;
    }
    const double cnt = block_sum<BPLAN>((double)__popc(mk));
    const double zs = block_sum<BPLAN>(z ? 1.0 : 0.0);
    if (threadIdx.x == 0) {
        if (cnt > 0.0) atomicAdd(&ncut[blockIdx.y], (int32_t)cnt);
        if (zs > 0.0) atomicOr(&zero[blockIdx.y], 1);
    }
}

__global__ void __launch_bounds__(BPLAN) k_batch_verts(const BatchProb *prob, const uint8_t *mask, int32_t *nvert) {
    const BatchProb &P = prob[blockIdx.y];
    const MeshP &m = P.m;
    const int64_t nv = (int64_t)(m.n[0] + 1) * (m.n[1] + 1) * (m.n[2] + 1);
    const int64_t v = (int64_t)blockIdx.x * BPLAN + threadIdx.x;
    bool in = false;
    if (v < nv) {
        const int64_t x1 = v % (m.n[0] + 1), x2 = (v / (m.n[0] + 1)) % (m.n[1] + 1),
                      x3 = v / ((int64_t)(m.n[0] + 1) * (m.n[1] + 1));
        for (int d = 0; d < 8 && !in; ++d) {
            const int64_t c1 = x1 - (d & 1), c2 = x2 - ((d >> 1) & 1), c3 = x3 - ((d >> 2) & 1);
            if (c1 < 0 || c2 < 0 || c3 < 0 || c1 >= m.n[0] || c2 >= m.n[1] || c3 >= m.n[2]) continue;
            const int mk = mask[P.cell_off + (c3 * m.n[1] + c2) * m.n[0] + c1];
            for (int k = 0; k < 6; ++k)
                if (((mk >> k) & 1) && c_tab.inc[d][k] >= 0) in = true;
        }
    }
    const double cnt = block_sum<BPLAN>(in ? 1.0 : 0.0);
    if (threadIdx.x == 0 && cnt > 0.0) atomicAdd(&nvert[blockIdx.y], (int32_t)cnt);
}

// ---------------------------------------------------------------------------
// assembly over the whole grid
//
// Every step of the single-problem assembly as one launch over all problems: a problem's workgroup had
// to walk its own steps one after the other, the largest one for 8 ms while the others had long ended, and
// kept the local matrices' and the rows' registers in one kernel (1,272 bytes of scratch a lane).  The same
// per-item functions produce the same arrays as the single-problem entry points.
//   k_batch_cut_count   per (problem, block of cells): cell masks, the block's cut-tet count,
//                       the problem's exact-zero flag
//   k_batch_cut_scan    per problem: exclusive scan of its block counts; opens its stat entry
//   k_batch_cut_fill    per (problem, block of cells): cut list in cell order and cell words
//   k_batch_local       one thread per cut tet of any problem: local matrices and qualification
//   k_batch_first       one thread per (cut tet, vertex): first-encounter owner
//   k_batch_rank        per problem: owner ranks, DOF count
//   k_batch_dofs        one thread per (cut tet, vertex)
//   k_batch_rows<>      one wave per row: count, then (k_batch_rowptr per problem) fill
// Threads find their problem from the offsets' table; a problem that failed a step (exact zero, capacity)
// is skipped from there on.  512 problems of 16^3 to 64^3 cells (5.1 M cut
// tets, 1.8 M rows): 27.0 -> 8.0 ms, local matrices 2.9 (5.1 before they list their facets), rows 1.1 + 2.1, cells
// 0.83 + 0.25, owners 0.55, the rest 0.3.
// ---------------------------------------------------------------------------
struct BatchArgs {
    const BatchProb *prob;
    const int32_t *order;       // problem ids, largest first
    int32_t nprob;
    int32_t *queue;             // next position in `order` (zeroed before the launch)
    const double *phi;
    uint8_t *cellmask;          // per problem cell (cell_off layout)
    int32_t *blkcnt;            // [nprob][max_blocks]
    int32_t max_blocks;
    int32_t *zero, *perr;       // per problem: exact-zero node in a cut tet; local error bits (2: all-zero sub-tet)
    int64_t cut_total, row_total;
    uint32_t *cellinfo;
    int64_t *cut;
    uint8_t *flags;
    double *loc;                // SoA [LOC_N][ncut_cap] per problem
    int32_t *first, *slot, *dofs;
    int32_t *rowowner, *rowlen, *rowptr;
    int32_t *col;
    double *vm, *vl, *vs, *vc;
    double *rhs, *diag, *x, *r64;
    float *d32, *r32, *z32, *p32, *q32;
    int32_t *scol, *soff;       // FP32 inner matrix in memory: streamed rows, or a SELL-64 copy of the whole
    float *sval;
    BatchStat *stat;
    double coef0, coef1, coef2;
    int rhs_kind;
    double rhs_p0;
    double omit_bound;
    int zero_throw;
    double tol;
    int max_iter;
    int rel;
    double inner_tol;
    int inner_max;
};

__global__ void __launch_bounds__(BPLAN) k_batch_cut_count(BatchArgs a) {
    const int p = blockIdx.y;
    const BatchProb &P = a.prob[p];
    const int64_t cell = (int64_t)blockIdx.x * BPLAN + threadIdx.x;
    if (blockIdx.x == 0 && threadIdx.x == 0) a.stat[p].t0 = wall_clock64();
    if ((int64_t)blockIdx.x * BPLAN >= P.m.ncell) return;
    int mk = 0;
    bool z = false;
    if (cell < P.m.ncell) {
        mk = cell_cut_mask(P.m, a.phi + P.phi_off, cell, z);
        a.cellmask[P.cell_off + cell] = (uint8_t)mk;
    }
    int tot;
    block_excl_scan<BPLAN>(__popc(mk), &tot);
    if (threadIdx.x == 0) a.blkcnt[(int64_t)p * a.max_blocks + blockIdx.x] = tot;
    if (z) atomicOr(&a.zero[p], 1);
}

// exclusive scan of in[0..n) into out (may alias) by a workgroup of 1024, four items a thread at a time;
// returns the total
constexpr int BSCAN = 1024;
__device__ inline int64_t wg_scan4(const int32_t *in, int32_t *out, int64_t n) {
    int64_t carry = 0;
    for (int64_t i0 = 0; i0 < n; i0 += 4 * BSCAN) {
        const int64_t i = i0 + 4 * threadIdx.x;
        int v[4], s = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            v[k] = i + k < n ? in[i + k] : 0;
            s += v[k];
        }
        int tot;
        int off = (int)carry + block_excl_scan<BSCAN>(s, &tot);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (i + k < n) out[i + k] = off;
            off += v[k];
        }
        carry += tot;
    }
    return carry;
}

__global__ void __launch_bounds__(BSCAN) k_batch_cut_scan(BatchArgs a) {
    const int p = blockIdx.x;
    const BatchProb &P = a.prob[p];
    int32_t *cnt = a.blkcnt + (int64_t)p * a.max_blocks;
    const int64_t ncut = wg_scan4(cnt, cnt, (P.m.ncell + BPLAN - 1) / BPLAN);
    if (threadIdx.x != 0) return;
    BatchStat &st = a.stat[p];
    st.ncut = (int32_t)ncut;
    st.ndof = st.nnz = st.iters = st.outer = 0;
    st.resid = 0.0;
    st.status = ncut > P.ncut_cap ? DHIP_E_CAPACITY : a.zero_throw && a.zero[p] ? DHIP_E_ZERO_NODE : DHIP_OK;
    st.t1 = st.t_asm = wall_clock64();
}

__global__ void __launch_bounds__(BPLAN) k_batch_cut_fill(BatchArgs a) {
    const int p = blockIdx.y;
    const BatchProb &P = a.prob[p];
    if ((int64_t)blockIdx.x * BPLAN >= P.m.ncell || a.stat[p].status != DHIP_OK) return;
    const int64_t cell = (int64_t)blockIdx.x * BPLAN + threadIdx.x;
    const int mask = cell < P.m.ncell ? a.cellmask[P.cell_off + cell] : 0;
    const int off = block_excl_scan<BPLAN>(__popc(mask), nullptr);
    if (cell >= P.m.ncell) return;
    int64_t b = (int64_t)a.blkcnt[(int64_t)p * a.max_blocks + blockIdx.x] + off;
    a.cellinfo[P.cell_off + cell] = ((uint32_t)b << 6) | (uint32_t)mask;
    for (int k = 0; k < 6; ++k)
        if (mask & (1 << k)) a.cut[P.cut_off + b++] = cell * 6 + k;   // (the counts are within the capacity)
}

// The problem whose range of a flat index holds g, ranges starting at off(problem): the last one that starts at
// or before g.  The wave's first index is searched for all lanes together.
template <class F>
__device__ __forceinline__ int batch_find(int nprob, int64_t g, F &&off) {
    const uint32_t lo32 = __builtin_amdgcn_readfirstlane((int)(uint32_t)g);
    const int64_t g0 = (int64_t)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(g >> 32)) << 32 | lo32);
    int lo = 0, hi = nprob - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (off(mid) <= g0) lo = mid;
        else hi = mid - 1;
    }
    while (lo + 1 < nprob && off(lo + 1) <= g) ++lo;
    return lo;
}

// problem and cut tet of flat cut slot g; false for the unused capacity and failed problems
__device__ __forceinline__ bool batch_tet(const BatchArgs &a, int64_t g, int &p, int64_t &c) {
    p = batch_find(a.nprob, g, [&](int k) { return a.prob[k].cut_off; });
    c = g - a.prob[p].cut_off;
    return a.stat[p].status == DHIP_OK && c < a.stat[p].ncut;
}

__global__ void __launch_bounds__(LOCAL_BLOCK) k_batch_local(BatchArgs a) {
    __shared__ LocalP1Shared sh;
    local_p1_tables(sh);
    const int64_t g = (int64_t)blockIdx.x * LOCAL_BLOCK + threadIdx.x;
    if (g >= a.cut_total) return;
    int p;
    int64_t c;
    if (!batch_tet(a, g, p, c)) return;
    const BatchProb &P = a.prob[p];
    double *loc = a.loc + (int64_t)LOC_N * P.cut_off;
    LocalArgs la{P.m, a.phi + P.phi_off, a.cut + P.cut_off, P.ncut_cap, a.coef0, a.coef1, a.coef2, a.rhs_kind,
                 a.rhs_p0, loc, a.flags + P.cut_off, &a.perr[p]};
    local_p1_one(la, c, sh);
    QualArgs qa{P.m, a.cut + P.cut_off, P.ncut_cap, loc, a.flags + P.cut_off, a.omit_bound};
    qualify_one(qa, c);
}

constexpr int BFLAT = 256;

__global__ void __launch_bounds__(BFLAT) k_batch_first(BatchArgs a) {
    const int64_t g = (int64_t)blockIdx.x * BFLAT + threadIdx.x;
    if (g >= 4 * a.cut_total) return;
    int p;
    int64_t c;
    if (!batch_tet(a, g >> 2, p, c)) return;
    const BatchProb &P = a.prob[p];
    FirstArgs fa{P.m, a.cut + P.cut_off, a.stat[p].ncut, a.cellinfo + P.cell_off, a.flags + P.cut_off,
                 a.first + 4 * P.cut_off, a.slot + 4 * P.cut_off};
    first_one(fa, 4 * c + (g & 3));
}

__global__ void __launch_bounds__(BSCAN) k_batch_rank(BatchArgs a) {
    const int p = blockIdx.x;
    const BatchProb &P = a.prob[p];
    BatchStat &st = a.stat[p];
    if (st.status != DHIP_OK) return;
    if (a.perr[p] & 2) {
        if (threadIdx.x == 0) st.status = DHIP_E_ZERO_PATTERN;
        return;
    }
    int32_t *slot = a.slot + 4 * P.cut_off;   // owner flag -> owner rank
    const int64_t nd = wg_scan4(slot, slot, 4 * (int64_t)st.ncut);
    if (threadIdx.x == 0) {
        st.ndof = (int32_t)nd;
        if (nd > P.row_cap) st.status = DHIP_E_CAPACITY;
    }
}

__global__ void __launch_bounds__(BFLAT) k_batch_dofs(BatchArgs a) {
    const int64_t g = (int64_t)blockIdx.x * BFLAT + threadIdx.x;
    if (g >= 4 * a.cut_total) return;
    int p;
    int64_t c;
    if (!batch_tet(a, g >> 2, p, c)) return;
    const BatchProb &P = a.prob[p];
    const int64_t s = 4 * c + (g & 3), o = 4 * P.cut_off;
    const int32_t f = a.first[o + s];
    a.dofs[o + s] = f >= 0 ? a.slot[o + f] : -1;
    if (f == s) a.rowowner[P.row_off + a.slot[o + s]] = (int32_t)s;
}

template <bool FILL>
__global__ void __launch_bounds__(64 * ROWW_WAVES) k_batch_rows(BatchArgs a) {
    __shared__ RowWShared shm[ROWW_WAVES];
    const int w = threadIdx.x >> 6;
    const int64_t g = (int64_t)xcd_position(blockIdx.x, gridDim.x) * ROWW_WAVES + w;
    if (g >= a.row_total) return;
    const int p = __builtin_amdgcn_readfirstlane(
        batch_find(a.nprob, g, [&](int k) { return a.prob[k].row_off; }));
    const BatchProb &P = a.prob[p];
    const BatchStat &st = a.stat[p];
    const int64_t r = g - P.row_off;
    if (st.status != DHIP_OK || r >= st.ndof) return;
    RowArgs ra{P.m, a.cut + P.cut_off, P.ncut_cap, a.cellinfo + P.cell_off, a.flags + P.cut_off,
               a.dofs + 4 * P.cut_off, a.rowowner + P.row_off, st.ndof, a.loc + (int64_t)LOC_N * P.cut_off,
               a.rowlen + P.row_off, a.rowptr + P.row_off + p, a.col + P.nz_off, a.vm + P.nz_off, a.vl + P.nz_off,
               a.vs + P.nz_off, a.vc + P.nz_off, a.rhs + P.row_off, a.diag + P.row_off, P.lc[0], P.lc[1], P.lc[2]};
    row_wave<FILL>(ra, r, shm[w]);
}

__global__ void __launch_bounds__(BSCAN) k_batch_rowptr(BatchArgs a) {
    const int p = blockIdx.x;
    const BatchProb &P = a.prob[p];
    BatchStat &st = a.stat[p];
    if (st.status != DHIP_OK) return;
    int32_t *rowptr = a.rowptr + P.row_off + p;
    const int64_t nnz = wg_scan4(a.rowlen + P.row_off, rowptr, st.ndof);
    if (threadIdx.x == 0) {
        rowptr[st.ndof] = (int32_t)nnz;
        st.nnz = (int32_t)nnz;
        if (nnz > P.nz_cap) st.status = DHIP_E_CAPACITY;
    }
}

// exclusive scan of a[0..n) in place by the whole workgroup; returns the total
template <int BB>
__device__ inline int64_t wg_scan_inplace(int32_t *a, int64_t n) {
    int64_t carry = 0;
    for (int64_t i0 = 0; i0 < n; i0 += BB) {
        const int64_t i = i0 + threadIdx.x;
        const int v = i < n ? a[i] : 0;
        int tot;
        const int off = block_excl_scan<BB>(v, &tot);
        if (i < n) a[i] = (int32_t)(carry + off);
        carry += tot;
    }
    __syncthreads();
    return carry;
}

// Relative residual at which an FP32 inner solve of the batch stops, from the FP64 relative residual `resid` it starts
// at: half of what is left to `tol` where FP32 reaches that, else `base`.  With `base` alone most problems end their
// second solve just below 1e-8 and some take a third of 1e-4 for a factor of little over one: 512 problems 34.4 ms
// instead of 28.6, and the batch's solutions are further from the exact ones, in all (listed 3.1e-9 against 2.4e-9;
// nine sets of 5 to 85 problems 1.6e-9 to 6.4e-9 against 1.2e-9 to 3.1e-9), in the median and in the worst
// problem (1.9e-8 against 1e-8).  The single solver keeps `base`: a solve that a third pass had
// taken to 4e-13 ended at 6.6e-10 with this rule.
__device__ __forceinline__ double inner_tolerance(double tol, double resid, double base) {
    const double left = tol / resid;
    return left >= 0.1 * base ? 0.5 * left : base;
}

// two workgroup sums with one LDS round
template <int BB>
__device__ inline void block_sum2(double &u, double &v) {
    __shared__ double ws[2][BB / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    u = wave_sum(u);
    v = wave_sum(v);
    if (lane == 0) {
        ws[0][w] = u;
        ws[1][w] = v;
    }
    __syncthreads();
    double su = 0.0, sv = 0.0;
#pragma unroll
    for (int i = 0; i < BB / 64; ++i) {
        su += ws[0][i];
        sv += ws[1][i];
    }
    __syncthreads();
    u = su;
    v = sv;
}

// Row loops of the inner iteration in groups: a thread's rows r = tid + (g + u BB) are handled G at a
// time with every load of the group issued before the first use, so a group costs one memory round
// trip instead of one per row (the loops are latency-bound: a few dozen rows per thread).
constexpr int SELL_MAXW = 15;   // entries per row of a P1 interface matrix on a Kuhn mesh

template <int BB, int G>
__device__ __forceinline__ double sell_spmv_group(const int32_t *soff, const int32_t *scol, const float *sval,
                                                  const int32_t *rowptr, const float *pv, float *q32, int64_t nd) {
    double p_lam = 0.0;
    for (int64_t r0 = threadIdx.x; r0 < nd; r0 += (int64_t)G * BB) {
        int64_t base[G];
        int32_t len[G];
#pragma unroll
        for (int u = 0; u < G; ++u) {
            const int64_t r = r0 + (int64_t)u * BB;
            len[u] = 0;
            base[u] = 0;
            if (r < nd) {
                base[u] = (int64_t)soff[r >> 6] + (r & 63);
                len[u] = rowptr[r + 1] - rowptr[r];
            }
        }
        int32_t cc[G][SELL_MAXW];
        float vv[G][SELL_MAXW];
#pragma unroll
        for (int u = 0; u < G; ++u)
#pragma unroll
            for (int k = 0; k < SELL_MAXW; ++k)
                if (k < len[u]) {
                    cc[u][k] = scol[base[u] + 64 * k];
                    vv[u][k] = sval[base[u] + 64 * k];
                }
#pragma unroll
        for (int u = 0; u < G; ++u) {
            const int64_t r = r0 + (int64_t)u * BB;
            float s = 0.0f;
#pragma unroll
            for (int k = 0; k < SELL_MAXW; ++k)
                if (k < len[u]) s += vv[u][k] * pv[cc[u][k]];
            if (r < nd) {
                q32[r] = s;
                p_lam += (double)s * (double)pv[r];
            }
        }
    }
    return p_lam;
}

// The same PCG for a problem whose search direction does not fit the workgroup's LDS: every vector in
// memory, the inner matrix as a SELL-64 copy.
template <int BB>
__device__ __noinline__ void batch_pcg_memory(const BatchArgs &a, int p, BatchStat &st) {
    const BatchProb P = a.prob[p];
    const int tid = threadIdx.x;
    const int64_t nd = st.ndof;
    const int32_t *rowptr = a.rowptr + P.row_off + p;
    const int32_t *col = a.col + P.nz_off;
    const double *vc = a.vc + P.nz_off;
    const double *rhs = a.rhs + P.row_off, *diag = a.diag + P.row_off;
    double *x = a.x + P.row_off, *r64 = a.r64 + P.row_off;
    float *d32 = a.d32 + P.row_off, *r32 = a.r32 + P.row_off, *z32 = a.z32 + P.row_off;
    float *p32 = a.p32 + P.row_off, *q32 = a.q32 + P.row_off;
    // SELL-64 copy of the FP32 matrix: entry k of row r at soff[r / 64] + 64 k + r % 64, so the
    // thread-per-row loads of a wave (64 consecutive rows) coalesce
    int32_t *scol = a.scol + P.sell_off, *soff = a.soff + P.slice_off;
    float *sval = a.sval + P.sell_off;
    const int64_t nsl = (nd + 63) / 64;
    for (int64_t sl = tid; sl < nsl; sl += BB) {
        int32_t w = 0;
        for (int64_t r = 64 * sl; r < 64 * sl + 64 && r < nd; ++r) {
            const int32_t len = rowptr[r + 1] - rowptr[r];
            w = len > w ? len : w;
        }
        soff[sl] = 64 * w;
    }
    __syncthreads();
    wg_scan_inplace<BB>(soff, nsl);
    for (int64_t r = tid; r < nd; r += BB) {
        const int64_t base = (int64_t)soff[r >> 6] + (r & 63);
        for (int32_t e = rowptr[r], k = 0; e < rowptr[r + 1]; ++e, ++k) {
            scol[base + 64 * (int64_t)k] = col[e];
            sval[base + 64 * (int64_t)k] = (float)vc[e];
        }
    }
    __syncthreads();
    for (int64_t r = tid; r < nd; r += BB) x[r] = 0.0;
    __syncthreads();
    {
        int total_it = 0, outer = 0, status = 1;
        double normb = 1.0, resid = 0.0;
        bool firstpass = true;
        for (;;) {
            double p_rr = 0.0, p_bb = 0.0;
            for (int64_t r = tid; r < nd; r += BB) {
                const double s =
                    row_product<double, 8>(rowptr, col, vc, 0, r, [&](int32_t c) { return x[c]; });
                const double bv = rhs[r];
                const double rv = bv - s;
                r64[r] = rv;
                p_rr += rv * rv;
                p_bb += bv * bv;
            }
            p_rr = block_sum<BB>(p_rr);
            if (firstpass) {
                p_bb = block_sum<BB>(p_bb);
                normb = sqrt(p_bb);
                if (normb == 0.0 || !a.rel) normb = 1.0;
                firstpass = false;
            }
            const double rnorm = sqrt(p_rr);
            resid = rnorm / normb;
            if (resid <= a.tol) { status = 0; break; }
            if (total_it >= a.max_iter) { status = 1; break; }
            ++outer;
            const double scale = 1.0 / rnorm;
            float *pv = p32;
            double p_zr = 0.0;
            for (int64_t r = tid; r < nd; r += BB) {
                const float rin = (float)(r64[r] * scale);
                const float zv = rin / (float)diag[r];
                r32[r] = rin;
                z32[r] = zv;
                d32[r] = 0.0f;
                pv[r] = 0.0f;
                p_zr += (double)zv * (double)rin;
            }
            double rho = block_sum<BB>(p_zr);
            float beta = 0.0f;
            for (int it = 1; it <= a.inner_max && total_it < a.max_iter; ++it) {
                ++total_it;
                constexpr int GU = 4;   // rows per group of the vector loops
                for (int64_t r0 = tid; r0 < nd; r0 += (int64_t)GU * BB) {
                    float zl[GU], pl[GU];
#pragma unroll
                    for (int u = 0; u < GU; ++u) {
                        const int64_t r = r0 + (int64_t)u * BB;
                        if (r < nd) {
                            zl[u] = z32[r];
                            pl[u] = pv[r];
                        }
                    }
#pragma unroll
                    for (int u = 0; u < GU; ++u) {
                        const int64_t r = r0 + (int64_t)u * BB;
                        if (r < nd) pv[r] = zl[u] + beta * pl[u];
                    }
                }
                __syncthreads();
                const double lam =
                    block_sum<BB>(sell_spmv_group<BB, 2>(soff, scol, sval, rowptr, pv, q32, nd));
                const float alpha = (float)(rho / lam);
                double p_rr2 = 0.0, p_zr2 = 0.0;
                for (int64_t r0 = tid; r0 < nd; r0 += (int64_t)GU * BB) {
                    float dl[GU], rl[GU], ql[GU], pl[GU];
                    double gl[GU];
#pragma unroll
                    for (int u = 0; u < GU; ++u) {
                        const int64_t r = r0 + (int64_t)u * BB;
                        if (r < nd) {
                            dl[u] = d32[r];
                            rl[u] = r32[r];
                            ql[u] = q32[r];
                            gl[u] = diag[r];
                            pl[u] = pv[r];
                        }
                    }
#pragma unroll
                    for (int u = 0; u < GU; ++u) {
                        const int64_t r = r0 + (int64_t)u * BB;
                        if (r < nd) {
                            d32[r] = dl[u] + alpha * pl[u];
                            const float rin = rl[u] - alpha * ql[u];
                            r32[r] = rin;
                            const float zv = rin / (float)gl[u];
                            z32[r] = zv;
                            p_rr2 += (double)rin * (double)rin;
                            p_zr2 += (double)zv * (double)rin;
                        }
                    }
                }
                block_sum2<BB>(p_rr2, p_zr2);
                if (sqrt(p_rr2) <= inner_tolerance(a.tol, resid, a.inner_tol)) break;
                const double rho1 = rho;
                rho = p_zr2;
                beta = (float)(rho / rho1);
            }
            for (int64_t r = tid; r < nd; r += BB) x[r] += rnorm * (double)d32[r];
            __syncthreads();
        }
        st.iters = total_it;
        st.outer = outer;
        st.resid = resid;
        st.status = status == 0 ? DHIP_OK : DHIP_E_NOT_CONVERGED;
    }
}

// ---------------------------------------------------------------------------
// the PCG of a problem inside one CU
//
// One workgroup of BPT threads runs a problem's Jacobi PCG with FP32 inner iterations and FP64
// refinement (residuals, dot products and the solution in FP64).  What an inner iteration touches stays
// on the CU: the search direction in LDS, and of thread t's rows t, t + BPT, ... the first R with their
// matrix entries (16 values, 16 column indices of 16 bits) and their vectors in registers, the next L with
// their entries in LDS.  The rows of larger problems beyond these are streamed each iteration from a copy laid
// out for their own thread (four values and four columns a load, 96 B a row); S rows a thread of those keep
// their vectors in registers, and past 19 rows a thread (MEM) the vectors are streamed too.  The classes are
// what 256 registers hold without spilling.
// An iteration is three barriers, two workgroup sums and the LDS gathers of the search direction (about 7
// cycles a wave's 64 against 2 without bank conflicts).  Measured a row count's iteration with 200 problems at
// once: 765 rows 1.9 us, 1,543 2.5, 2,471 3.4, 3,555 4.7, 4,682 9.7, 7,604 13.7, 9,372 20, 12,936 30; with
// every vector and the matrix in memory 15 to 60 us.  512 problems of 16^3 to 64^3 cells: all PCGs 70 -> 18.5 ms,
// 13.4 with inner_tolerance.
// ---------------------------------------------------------------------------
constexpr int BPT = 512;
constexpr int BPW = BPT / 64;
constexpr int BP_W = 16, BP_Q = BP_W / 4;   // entries per row (a P1 interface row has at most 15), in quads
constexpr int BP_G = 4;               // streamed rows whose vector loads are issued together
constexpr int BP_MAX_SLOTS = 76;      // rows per thread: 76 * 512 floats of search direction fit the LDS
struct BpShared {
    double red[2][BPW][2];
    uint8_t quads[BP_MAX_SLOTS * BPW];
    __align__(16) unsigned char end[16];
};

// bytes of LDS: the search direction of `slots` rows a thread, and l rows' entries
constexpr int64_t bp_lds(int64_t slots, int l) {
    return (int64_t)sizeof(BpShared) + slots * BPT * 4 + (int64_t)l * BP_Q * BPT * 24;
}

// dynamic LDS of k_batch_solve: its largest class, on a CU of 160 KiB
constexpr int64_t BP_LDS = bp_lds(BP_MAX_SLOTS, 0) > bp_lds(28, 2) ? bp_lds(BP_MAX_SLOTS, 0) : bp_lds(28, 2);
static_assert(BP_LDS + 2048 <= 160 * 1024, "k_batch_solve's LDS");

// sum over the wave in lane 63 (row shifts, then the row broadcasts)
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, ROWS, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, ROWS, 0xf, true);
    return v + __builtin_bit_cast(double, ((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
}
__device__ __forceinline__ double wave_sum_last(double v) {
    v = dpp_add<0x111, 0xf>(v);
    v = dpp_add<0x112, 0xf>(v);
    v = dpp_add<0x114, 0xf>(v);
    v = dpp_add<0x118, 0xf>(v);
    v = dpp_add<0x142, 0xa>(v);
    return dpp_add<0x143, 0xc>(v);
}

// Workgroup sums of u and v in every thread: the eight waves' sums go through LDS once, every lane takes one
// of them and the lanes add up in a fixed pattern.  One barrier: successive calls use the two halves of `red`
// in turn, and a half is written again only after the other half's barrier.
__device__ __forceinline__ void bp_sum2(double (*red)[2], double &u, double &v) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    u = wave_sum_last(u);
    v = wave_sum_last(v);
    if (lane == 63) {
        red[w][0] = u;
        red[w][1] = v;
    }
    __syncthreads();
    u = red[lane & 7][0];
    v = red[lane & 7][1];
    u = dpp_add<0xB1, 0xf>(u);    // lane ^ 1
    v = dpp_add<0xB1, 0xf>(v);
    u = dpp_add<0x4E, 0xf>(u);    // lane ^ 2
    v = dpp_add<0x4E, 0xf>(v);
    u = dpp_add<0x141, 0xf>(u);   // the other half of the eight
    v = dpp_add<0x141, 0xf>(v);
}
static_assert(BPW == 8, "bp_sum2 adds eight waves");

// u / v for positive normal v, to a rounding of FP64 (the quotient is used as FP32)
__device__ __forceinline__ double bp_quot(double u, double v) {
    double r = __builtin_amdgcn_rcp(v);
    r = __builtin_fma(__builtin_fma(-v, r, 1.0), r, r);
    r = __builtin_fma(__builtin_fma(-v, r, 1.0), r, r);
    return u * r;
}

// Global pointers of a called function: without the address space the loads would be flat ones, which wait
// for every load in flight.
template <class T>
using GlobalPtr = __attribute__((address_space(1))) T *;
typedef float BpF4 __attribute__((ext_vector_type(4)));
typedef uint32_t BpU2 __attribute__((ext_vector_type(2)));

// A row's FP32 entries and columns, four at a time; entries past the row's end are (0, column 0).  Every load
// is issued (an index past the row's end is clamped to it), so that a row's loads overlap.
struct BpQuad {
    BpF4 v;
    BpU2 c;
};
__device__ __forceinline__ BpQuad bp_load_quad(GlobalPtr<const int32_t> col, GlobalPtr<const double> vc, int32_t e,
                                               int32_t end) {
    double v[4];
    uint32_t cc[4];
    const int32_t last = end > 0 ? end - 1 : 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int32_t i = e + k < last ? e + k : last;
        v[k] = vc[i];
        cc[k] = (uint32_t)col[i];
    }
    BpQuad q;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const bool in = e + k < end;
        q.v[k] = in ? (float)v[k] : 0.0f;
        cc[k] = in ? cc[k] : 0u;
    }
    q.c[0] = cc[0] | cc[1] << 16;
    q.c[1] = cc[2] | cc[3] << 16;
    return q;
}
__device__ __forceinline__ float bp_quad_dot(float s, const BpF4 &v, const BpU2 &c, const float *pv) {
    s = __builtin_fmaf(v[0], pv[c[0] & 0xffffu], s);
    s = __builtin_fmaf(v[1], pv[c[0] >> 16], s);
    s = __builtin_fmaf(v[2], pv[c[1] & 0xffffu], s);
    return __builtin_fmaf(v[3], pv[c[1] >> 16], s);
}
// (A x)_r in FP64, in column order
__device__ __forceinline__ double bp_row64(GlobalPtr<const int32_t> col, GlobalPtr<const double> vc, int32_t e,
                                           int32_t end, GlobalPtr<const double> x) {
    constexpr int B = 8;
    double s = 0.0;
    for (; e < end; e += B) {
        double v[B], xx[B];
        int32_t cc[B];
#pragma unroll
        for (int k = 0; k < B; ++k) {
            const int32_t i = e + k < end ? e + k : end - 1;
            cc[k] = col[i];
            v[k] = vc[i];
        }
#pragma unroll
        for (int k = 0; k < B; ++k) xx[k] = x[cc[k]];
#pragma unroll
        for (int k = 0; k < B; ++k)
            if (e + k < end) s += v[k] * xx[k];
    }
    return s;
}

// the widest row of the wave's 64, in quads (uniform)
__device__ __forceinline__ int bp_wave_quads(int len) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const int t = __shfl_xor(len, o, 64);
        len = t > len ? t : len;
    }
    return __builtin_amdgcn_readfirstlane((len + 3) >> 2);
}

template <int R, int L, int S, bool MEM>
__device__ __noinline__ void batch_pcg_chip(const BatchArgs &a, int p, BatchStat &st) {
    extern __shared__ __align__(16) unsigned char lds[];
    BpShared &sh = *reinterpret_cast<BpShared *>(lds);
    float *pv = reinterpret_cast<float *>(lds + sizeof(BpShared));
    double (*red)[BPW][2] = sh.red;
    uint8_t *quads = sh.quads;
    constexpr int V0 = R + L;   // rows per thread whose entries are on the CU
    constexpr int V = V0 + S;   // rows per thread whose vectors are in registers
    const BatchProb &P = a.prob[p];
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));   // nothing of one size's code is formed ahead of the queue loop
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int nd = st.ndof;
    const int slots = MEM ? (nd + BPT - 1) / BPT : V;
    const auto rowptr = (GlobalPtr<const int32_t>)(a.rowptr + P.row_off + p);
    const auto col = (GlobalPtr<const int32_t>)(a.col + P.nz_off);
    const auto vc = (GlobalPtr<const double>)(a.vc + P.nz_off);
    const auto rhs = (GlobalPtr<const double>)(a.rhs + P.row_off);
    const auto diag = (GlobalPtr<const double>)(a.diag + P.row_off);
    const auto x = (GlobalPtr<double>)(a.x + P.row_off);
    const auto r64 = (GlobalPtr<double>)(a.r64 + P.row_off);
    // streamed rows: entries as four floats / four uint16 per (slice, quad, lane); MEM: the vectors too (z32
    // holds the inverse diagonal)
    const auto d32 = (GlobalPtr<float>)(a.d32 + P.row_off), r32 = (GlobalPtr<float>)(a.r32 + P.row_off);
    const auto z32 = (GlobalPtr<float>)(a.z32 + P.row_off), q32 = (GlobalPtr<float>)(a.q32 + P.row_off);
    const auto sv = (GlobalPtr<BpF4>)(a.sval + P.sell_off);
    const auto sc = (GlobalPtr<BpU2>)(a.scol + P.sell_off);
    // LDS rows: the same quads behind the search direction
    BpF4 *lv = reinterpret_cast<BpF4 *>(pv + slots * BPT);
    BpU2 *lc = reinterpret_cast<BpU2 *>(lv + L * BP_Q * BPT);

    // entries of the LDS and streamed rows, once per problem
    for (int u = R; u < slots; ++u) {
        const int r = tid + u * BPT;
        int32_t e = 0, end = 0;
        if (r < nd) {
            e = rowptr[r];
            end = rowptr[r + 1];
            if (MEM && u >= V) z32[r] = 1.0f / (float)diag[r];
        }
        const int w = bp_wave_quads(end - e);
        if (lane == 0) quads[u * BPW + wv] = (uint8_t)w;
        for (int q = 0; q < (S > 0 || MEM ? BP_Q : w); ++q) {   // (streamed rows are loaded whole, padding included)
            const BpQuad b = bp_load_quad(col, vc, e + 4 * q, end);
            const BpF4 bv = b.v;
            const BpU2 bc = b.c;
            if (u < V0) {
                lv[((u - R) * BP_Q + q) * BPT + tid] = bv;
                lc[((u - R) * BP_Q + q) * BPT + tid] = bc;
            } else {
                const int64_t at = (int64_t)(((u - V0) * BPW + wv) * BP_Q + q) * 64 + lane;
                sv[at] = bv;
                sc[at] = bc;
            }
        }
    }
    int total_it = 0, outer = 0, status = 1;
    double normb = 1.0, resid = 0.0;
    bool firstpass = true;
    for (;;) {
        // ---- FP64 residual (the start is x = 0: b itself) ----
        double p_rr = 0.0, p_bb = 0.0;
        for (int r = tid; r < nd; r += BPT) {
            const double bv = rhs[r];
            double rv = bv;
            if (firstpass) {
                x[r] = 0.0;
                p_bb += bv * bv;
            } else {
                rv = bv - bp_row64(col, vc, rowptr[r], rowptr[r + 1], x);
            }
            r64[r] = rv;
            p_rr += rv * rv;
        }
        bp_sum2(red[0], p_rr, p_bb);
        if (firstpass) {
            normb = sqrt(p_bb);
            if (normb == 0.0 || !a.rel) normb = 1.0;
            firstpass = false;
        }
        const double rnorm = sqrt(p_rr);
        resid = rnorm / normb;
        if (resid <= a.tol) { status = 0; break; }
        if (total_it >= a.max_iter) { status = 1; break; }
        ++outer;
        const double scale = 1.0 / rnorm;
        const double inner_tol = inner_tolerance(a.tol, resid, a.inner_tol), inner_tol2 = inner_tol * inner_tol;
        // ---- the register rows' entries and vectors ----
        BpF4 val[R][BP_Q];
        BpU2 cc[R][BP_Q];
        float rv[V], dv[V], di[V], qv[V];
        int wq[V];
        double p_zr = 0.0, unused = 0.0;
        int t0 = tid;
        asm volatile("" : "+v"(t0));   // (row addresses are formed here, not kept over the iterations)
#pragma unroll
        for (int u = 0; u < V; ++u) {
            const int r = t0 + u * BPT;
            int32_t e = 0, end = 0;
            rv[u] = dv[u] = di[u] = 0.0f;
            if (r < nd) {
                e = rowptr[r];
                end = rowptr[r + 1];
                rv[u] = (float)(r64[r] * scale);
                di[u] = 1.0f / (float)diag[r];
            }
            wq[u] = bp_wave_quads(end - e);
            if (u < R) {
#pragma unroll
                for (int q = 0; q < BP_Q; ++q) {
                    const BpQuad b = bp_load_quad(col, vc, e + 4 * q, end);
                    val[u < R ? u : 0][q] = b.v;
                    cc[u < R ? u : 0][q] = b.c;
                    if (R >= 4 && (q & 1)) __builtin_amdgcn_sched_barrier(0);   // (two quads' FP64 loads in flight)
                }
            }
            pv[r] = 0.0f;
            p_zr += (double)(rv[u] * di[u]) * (double)rv[u];
        }
        for (int u = V; MEM && u < slots; ++u) {
            const int r = tid + u * BPT;
            pv[r] = 0.0f;
            if (r < nd) {
                const float rin = (float)(r64[r] * scale);
                r32[r] = rin;
                d32[r] = 0.0f;
                p_zr += (double)(rin * z32[r]) * (double)rin;
            }
        }
        bp_sum2(red[1], p_zr, unused);
        double rho = p_zr;
        float beta = 0.0f;
        for (int it = 1; it <= a.inner_max && total_it < a.max_iter; ++it) {
            ++total_it;
            // p = z + beta p
#pragma unroll
            for (int u = 0; u < V; ++u) {
                const int r = tid + u * BPT;
                pv[r] = __builtin_fmaf(beta, pv[r], rv[u] * di[u]);
                if (V > 8 && u % 8 == 7) __builtin_amdgcn_sched_barrier(0);
            }
            for (int u0 = V; MEM && u0 < slots; u0 += BP_G) {
                float rl[BP_G], zl[BP_G];
#pragma unroll
                for (int k = 0; k < BP_G; ++k) {
                    const int r = tid + (u0 + k) * BPT;
                    rl[k] = zl[k] = 0.0f;
                    if (r < nd) {
                        rl[k] = r32[r];
                        zl[k] = z32[r];
                    }
                }
#pragma unroll
                for (int k = 0; k < BP_G; ++k) {
                    const int r = tid + (u0 + k) * BPT;
                    if (r < nd) pv[r] = __builtin_fmaf(beta, pv[r], rl[k] * zl[k]);
                }
            }
            __syncthreads();
            // q = A p, (p, q)
            double lam = 0.0, none = 0.0;
            // The streamed rows' entries are PF rows ahead of the sums.  Their loads stand under no condition:
            // across a branch the compiler could only wait for all loads in flight.
            constexpr int PF = S >= 16 ? 1 : 2;
            BpF4 nv[PF][BP_Q];
            BpU2 nc[PF][BP_Q];
            auto fetch = [&](int u, BpF4 (&v)[BP_Q], BpU2 (&c)[BP_Q]) {
                const int64_t at = (int64_t)((u - V0) * BPW + wv) * BP_Q * 64 + lane;
#pragma unroll
                for (int q = 0; q < BP_Q; ++q) {
                    v[q] = sv[at + q * 64];
                    c[q] = sc[at + q * 64];
                }
            };
#pragma unroll
            for (int k = 0; k < PF; ++k)
                if (k < S || (MEM && k == 0)) fetch(V0 + k, nv[k], nc[k]);
#pragma unroll
            for (int u = 0; u < R; ++u) {
                // the columns stay packed: unpacked out of the loop they would take 8 more registers a row
#pragma unroll
                for (int q = 0; q < BP_Q; ++q) asm volatile("" : "+v"(cc[u][q]));
                float s = 0.0f;
#pragma unroll
                for (int q = 0; q < BP_Q; ++q)
                    if (q < wq[u]) s = bp_quad_dot(s, val[u][q], cc[u][q], pv);
                qv[u] = s;
                lam += (double)s * (double)pv[tid + u * BPT];
            }
#pragma unroll
            for (int l = 0; l < L; ++l) {
                float s = 0.0f;
#pragma unroll
                for (int q = 0; q < BP_Q; ++q)
                    if (q < wq[R + l]) s = bp_quad_dot(s, lv[(l * BP_Q + q) * BPT + tid], lc[(l * BP_Q + q) * BPT + tid], pv);
                qv[R + l] = s;
                lam += (double)s * (double)pv[tid + (R + l) * BPT];
            }
#pragma unroll
            for (int k = 0; k < S; ++k) {
                const int u = V0 + k;
                float s = 0.0f;
#pragma unroll
                for (int q = 0; q < BP_Q; ++q)
                    if (q < wq[u]) s = bp_quad_dot(s, nv[k % PF][q], nc[k % PF][q], pv);
                if (k + PF < S) fetch(u + PF, nv[k % PF], nc[k % PF]);
                qv[u] = s;
                lam += (double)s * (double)pv[tid + u * BPT];
                __builtin_amdgcn_sched_barrier(0);   // PF rows in registers, no more
            }
            for (int u = V; MEM && u < slots; ++u) {
                const int r = tid + u * BPT;
                const int w = __builtin_amdgcn_readfirstlane((int)quads[u * BPW + wv]);
                BpF4 v[BP_Q];
                BpU2 c[BP_Q];
#pragma unroll
                for (int q = 0; q < BP_Q; ++q) {
                    v[q] = nv[0][q];
                    c[q] = nc[0][q];
                }
                fetch(u + 1 < slots ? u + 1 : u, nv[0], nc[0]);
                float s = 0.0f;
#pragma unroll
                for (int q = 0; q < BP_Q; ++q)
                    if (q < w) s = bp_quad_dot(s, v[q], c[q], pv);
                if (r < nd) q32[r] = s;
                lam += (double)s * (double)pv[r];
            }
            bp_sum2(red[0], lam, none);
            const float alpha = (float)bp_quot(rho, lam);
            double p_rr2 = 0.0, p_zr2 = 0.0;
#pragma unroll
            for (int u = 0; u < V; ++u) {
                dv[u] = __builtin_fmaf(alpha, pv[tid + u * BPT], dv[u]);
                const float rin = __builtin_fmaf(-alpha, qv[u], rv[u]);
                rv[u] = rin;
                p_rr2 += (double)rin * (double)rin;
                p_zr2 += (double)(rin * di[u]) * (double)rin;
            }
            for (int u0 = V; MEM && u0 < slots; u0 += BP_G) {
                float dl[BP_G], rl[BP_G], ql[BP_G], zl[BP_G];
#pragma unroll
                for (int k = 0; k < BP_G; ++k) {
                    const int r = tid + (u0 + k) * BPT;
                    dl[k] = rl[k] = ql[k] = zl[k] = 0.0f;
                    if (r < nd) {
                        dl[k] = d32[r];
                        rl[k] = r32[r];
                        ql[k] = q32[r];
                        zl[k] = z32[r];
                    }
                }
#pragma unroll
                for (int k = 0; k < BP_G; ++k) {
                    const int r = tid + (u0 + k) * BPT;
                    if (r < nd) {
                        d32[r] = __builtin_fmaf(alpha, pv[r], dl[k]);
                        const float rin = __builtin_fmaf(-alpha, ql[k], rl[k]);
                        r32[r] = rin;
                        p_rr2 += (double)rin * (double)rin;
                        p_zr2 += (double)(rin * zl[k]) * (double)rin;
                    }
                }
            }
            bp_sum2(red[1], p_rr2, p_zr2);
            if (p_rr2 <= inner_tol2) break;
            const double rho1 = rho;
            rho = p_zr2;
            beta = (float)bp_quot(rho, rho1);
        }
        int t1 = tid;
        asm volatile("" : "+v"(t1));
#pragma unroll
        for (int u = 0; u < V; ++u) {
            const int r = t1 + u * BPT;
            if (r < nd) x[r] += rnorm * (double)dv[u];
            if (V > 8 && u % 4 == 3) __builtin_amdgcn_sched_barrier(0);
        }
        for (int u = V; MEM && u < slots; ++u) {
            const int r = tid + u * BPT;
            if (r < nd) x[r] += rnorm * (double)d32[r];
        }
        __syncthreads();
    }
    st.iters = total_it;
    st.outer = outer;
    st.resid = resid;
    st.status = status == 0 ? DHIP_OK : DHIP_E_NOT_CONVERGED;
}

// The PCG of every assembled problem: problems from the queue, largest first.
__global__ void __launch_bounds__(BPT) k_batch_solve(BatchArgs a) {
    __shared__ int sh_p;
    for (;;) {
        if (threadIdx.x == 0) {
            const int q = atomicAdd(a.queue, 1);
            sh_p = q < a.nprob ? a.order[q] : -1;
        }
        __syncthreads();
        const int p = sh_p;
        __syncthreads();
        if (p < 0) break;
        BatchStat st = a.stat[p];
        if (st.status == DHIP_OK) {
            st.t_asm = wall_clock64();
            const int slots = (st.ndof + BPT - 1) / BPT;
            // the smallest size class that holds the problem; the LDS of every class fits (asserted)
            switch (slots) {
                case 0: case 1: batch_pcg_chip<1, 0, 0, false>(a, p, st); break;
                case 2: batch_pcg_chip<2, 0, 0, false>(a, p, st); break;
                case 3: batch_pcg_chip<3, 0, 0, false>(a, p, st); break;
                case 4: batch_pcg_chip<4, 0, 0, false>(a, p, st); break;
                case 5: batch_pcg_chip<5, 0, 0, false>(a, p, st); break;
                case 6: batch_pcg_chip<6, 0, 0, false>(a, p, st); break;
                case 7: batch_pcg_chip<5, 2, 0, false>(a, p, st); break;
                case 8: batch_pcg_chip<6, 2, 0, false>(a, p, st); break;
                case 9: batch_pcg_chip<3, 2, 4, false>(a, p, st); break;
                case 10: case 11: batch_pcg_chip<2, 2, 7, false>(a, p, st); break;
                case 12: case 13: batch_pcg_chip<2, 2, 9, false>(a, p, st); break;
                case 14: case 15: batch_pcg_chip<1, 2, 12, false>(a, p, st); break;
                case 16: case 17: batch_pcg_chip<1, 2, 14, false>(a, p, st); break;
                case 18: case 19: batch_pcg_chip<1, 2, 16, false>(a, p, st); break;
                default:
                    if (slots <= 28) batch_pcg_chip<4, 2, 0, true>(a, p, st);
                    else if (slots <= BP_MAX_SLOTS) batch_pcg_chip<4, 0, 0, true>(a, p, st);
                    else batch_pcg_memory<BPT>(a, p, st);
            }
            st.t1 = wall_clock64();
            if (threadIdx.x == 0) a.stat[p] = st;
        }
        __syncthreads();
    }
}

}  // namespace dhip
