// Cell binning, deterministic cell-order sort and full neighbor-list build.
//
// Replaces GridGPU::periodicBoundaryConditions (src/GridGPU.cu:824-1103) and
// its kernels setBuildFlag (755-774), periodicWrap (138-161),
// countNumInGridCells (190-203), sortPerAtomArrays (253-322),
// countNumNeighbors / assignNeighbors (326-734).
//
// Design (gfx950):
//   * cells have edge >= r_list / reach (reach = 2), so a (2*reach+1)^3 stencil
//     holds every neighbor; columns of cells are ranked along a 2-D Morton
//     curve and z runs contiguously inside a column, so each stencil column is
//     one or two contiguous ranges of the sorted arrays (coalesced loads);
//   * the sort is a counting sort whose slots inside a cell are re-ordered by
//     atom id, so the layout depends only on positions, never on atomics order;
//   * the list is built in one pass: a team of T lanes per atom tests T
//     candidates per step with the canonical FP64 distance (no FMA contraction:
//     this file is compiled with -ffp-contract=off) and compacts hits with a
//     wave64 ballot; rows have a fixed capacity and the true count is kept so
//     overflow is detected and the host grows the rows and rebuilds;
//   * entries are index | tag << 30 with the 1-2/1-3/1-4 tag of the atom pair
//     (GridGPU.cu:471-520, globalDefs.h:40).
#include <algorithm>
#include <cstring>

#include "mdx_internal.h"

#pragma clang fp contract(off)

namespace mdx {

namespace {


__device__ __forceinline__ double mi_d(double d, double L, double invL, int periodic) {
    if (periodic) {
        double img = rint(d * invL);
        d = d - img * L;
    }
    return d;
}

// canonical squared distance, evaluated exactly as orc_dist2 in the oracle
__device__ __forceinline__ double dist2(const double4 &a, const double4 &b, const Geometry &g) {
    double dx = mi_d(b.x - a.x, g.L[0], g.invL[0], g.periodic[0]);
    double dy = mi_d(b.y - a.y, g.L[1], g.invL[1], g.periodic[1]);
    double dz = mi_d(b.z - a.z, g.L[2], g.invL[2], g.periodic[2]);
    return dx * dx + dy * dy + dz * dz;
}

__device__ __forceinline__ int cell_coord(double x, double lo, double cellInv, int nc) {
    int c = (int)floor((x - lo) * cellInv);
    return c < 0 ? 0 : (c >= nc ? nc - 1 : c);
}

// Max displacement since the last build (setBuildFlag, GridGPU.cu:755-774):
// flag when any |minImage(x - x_last)|^2 > (skin/2)^2.
__device__ __forceinline__ void check_body(int blk, int nblk, int n, const double4 *__restrict__ pos, const double4 *__restrict__ last,
                        const BoxDev *__restrict__ bx, double thr2, int *__restrict__ flags) {
    const Geometry g = bx->geo;
    int i = blk * blockDim.x + threadIdx.x;
    bool move = false;
    if (i < n) move = dist2(pos[i], last[i], g) > thr2;
    if (__any(move) && (threadIdx.x & 63) == 0) flags[0] = 1;
}

// Wrap into the box (periodicWrap) and bin into cells (countNumInGridCells),
// the first of the two launches of a re-sort.  Charged and charge-free atoms
// go to two copies of the grid (slots [0, ncell) and [ncell, 2 ncell)), so
// that after the permutation the charged atoms come first, each class sorted
// by cell: a neighbor row then lists its charged partners first, and the
// charge spread and gather see only charged atoms.
//
// Each atom is pushed onto its cell's list (head, next) and its records are
// copied to the scratch arrays pos1 ... id1, from which the second launch
// gathers them back in the new order: the sorted records end where they were,
// as the fixed buffers of captured steps need, without a copy-back pass.  The
// second launch works on chunks of 2^csh cell slots; the atoms of each chunk
// are counted here, one atomic per chunk and wave (the atoms still lie in the
// order of the previous build, so a wave meets one or two chunks).
__device__ __forceinline__ void bin_body(int blk, int nblk, const int *__restrict__ gate, int n,
                                         const double4 *__restrict__ pos, const double4 *__restrict__ vel,
                                         const float *__restrict__ q, const int *__restrict__ type,
                                         const int *__restrict__ id, double4 *__restrict__ pos1,
                                         double4 *__restrict__ vel1, float *__restrict__ q1, int *__restrict__ type1,
                                         int *__restrict__ id1, const BoxDev *__restrict__ bx, int ncell,
                                         const int *__restrict__ colRank, int *__restrict__ head,
                                         int *__restrict__ next, int *__restrict__ chunkSum, int csh,
                                         const double4 *__restrict__ cen, DecideArgs da) {
    if (da.slots) {  // the step's decisions, by every workgroup for itself
        const bool build = disp_max(da.slots) > da.half2;
        if (blk == 0 && threadIdx.x == 0) decide_write(da, build);
        if (!build) return;
    } else if (gate && *gate == 0) {
        return;
    }
    const int i = blk * blockDim.x + threadIdx.x;
    int chunk = -1;
    if (i < n) {
        const Geometry g = bx->geo;
        const CellGrid cg = bx->cg;
        double4 p = pos[i];
        const double4 v = vel[i];
        const float qi = q[i];
        const int ti = type[i], myid = id[i];
        double *pc = &p.x;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            if (g.periodic[a]) {
                double img = floor((pc[a] - g.lo[a]) * g.invL[a]);
                pc[a] = pc[a] - img * g.L[a];
            }
        }
        pos1[i] = p;
        vel1[i] = v;
        q1[i] = qi;
        type1[i] = ti;
        id1[i] = myid;
        // ring centroid lists: the atom goes to the cell of its ring's centroid
        // (already in the box)
        if (cen) p = cen[myid];
        const int cx = cell_coord(p.x, g.lo[0], cg.cellInv[0], cg.nc[0]);
        const int cy = cell_coord(p.y, g.lo[1], cg.cellInv[1], cg.nc[1]);
        const int cz = cell_coord(p.z, g.lo[2], cg.cellInv[2], cg.nc[2]);
        const int cell = colRank[cx * cg.nc[1] + cy] * cg.nc[2] + cz + (qi == 0.0f ? ncell : 0);
        next[i] = atomicExch(&head[cell], i);
        chunk = cell >> csh;
    }
    unsigned long long todo = __ballot(chunk >= 0);
    while (todo) {
        const int leader = __ffsll(todo) - 1;
        const int k = __shfl(chunk, leader, 64);
        const unsigned long long same = __ballot(chunk == k);
        if ((int)(threadIdx.x & 63) == leader) atomicAdd(&chunkSum[k], __popcll(same));
        todo &= ~same;
    }
}

// What the second launch of a re-sort reads and writes.
struct SortArgs {
    int n, nslot;        // atoms; cell slots (2 ncell)
    int cpw, csh;        // cells a workgroup takes at a time (<= 256), log2 of a chunk's cells
    int *head;           // per cell: its list of atoms (left empty for the next binning)
    const int *next;
    const int *chunkSum; // atoms per chunk
    int *start;          // nslot + 1
    const double4 *pos0, *vel0;
    const float *q0;
    const int *type0, *id0;
    double4 *pos1, *vel1;
    float *q1;
    int *type1, *id1;
    int *idToIdx;
    double4 *last;       // positions of this build (wrapped)
    float4 *xq;
    float4 *rec;         // P3M mesh records, or nullptr
    const double4 *cen;  // ring centroids by id, and the build positions made of them
    double4 *bpos;
    int *atomMolO;       // cleared for the molecule map of the build
    int *member;
    int maxExcl;         // exclusion rows by id (id | tag << 30, ~0u past the end)
    const int *exclOff;
    const uint32_t *exclIds;
    uint32_t *exclRow;
    unsigned *slots;     // the displacement maxima the binning decided from, cleared here
    const BoxDev *bx;
    BoxDev *boxLast;     // the box this build uses, kept for rebuilding the same list later
};

// Gather the record of atom o into place k (sortPerAtomArrays,
// GridGPU.cu:253-293) and refresh idToIdx, the last-build positions and xq.
__device__ __forceinline__ void place_atom(const SortArgs &a, int o, int k, int myid, const Geometry &g) {
    double4 p = a.pos0[o];
    const double4 v = a.vel0[o];
    const float qq = a.q0[o];
    const int tt = a.type0[o];
    a.pos1[k] = p;
    a.vel1[k] = v;
    a.q1[k] = qq;
    a.type1[k] = tt;
    a.id1[k] = myid;
    a.idToIdx[myid] = k;
    a.last[k] = p;
    if (a.atomMolO) a.atomMolO[k] = -1;
    if (a.member) a.member[k] = 0;
    if (a.maxExcl > 0) {
        const int o0 = a.exclOff[myid], ne = a.exclOff[myid + 1] - o0;
        for (int s = 0; s < a.maxExcl; ++s) a.exclRow[(size_t)k * a.maxExcl + s] = s < ne ? a.exclIds[o0 + s] : ~0u;
    }
    // the P3M mesh records in the new order (captured steps whose first half
    // kick refreshed them before the rebuild)
    if (a.rec && qq != 0.0f) a.rec[k] = mesh_record(p, a.bx->mesh);
    // ring centroid lists: the build works on the centroids (xq is written
    // again from the positions before the forces)
    if (a.cen) {
        p = a.cen[myid];
        a.bpos[k] = p;
    }
    a.xq[k] = make_float4((float)(p.x - g.lo[0]), (float)(p.y - g.lo[1]), (float)(p.z - g.lo[2]), qq);
}

// Scan, in-cell order and permutation of one chunk of cells per workgroup.
// The workgroup's first place is the sum of the chunk counts before its own;
// within it, one thread per cell walks the cell's list, a prefix sum over the
// cells gives the cell starts, and one thread per atom ranks the atom by id
// among its cell's (ids are unique, so the layout depends only on positions,
// never on the order of the pushes) and moves its records.
//
// This replaces a scan of all cell counts by one workgroup (15 us at 7,200
// cell slots, 126 us at 49,726, 2.8 ms at 828,478), a placing pass, a sort with
// one workgroup per slot, the permutation and a copy-back: with the binning,
// six launches of 40 us for 32,768 water sites and 3.1 ms for 500,000 LJ atoms
// became two of 18.5 us and 70 us.
// A cell slot holds about 0.6 (LJ) to 7 (water) atoms, so the walk is short; a
// round whose atoms exceed the LDS buffer (crowded cells) ranks them through
// the lists instead.
constexpr int kSortThreads = 256;
constexpr int kSortCap = 2048;  // atoms a round ranks in LDS
__device__ __forceinline__ void sort_body(int blk, int nblk, const int *__restrict__ gate, SortArgs a) {
    if (a.slots && blk == 0 && threadIdx.x < kDispSlots) {
        a.slots[threadIdx.x * kDispStride] = 0u;
        a.slots[threadIdx.x * kDispStride + 1] = 0u;
    }
    if (gate && *gate == 0) return;
    __shared__ int sIdx[kSortCap], sKey[kSortCap];
    __shared__ unsigned char sCell[kSortCap];
    __shared__ int sStart[kSortThreads + 1], wsum[kSortThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    if (blk == 0) {
        constexpr int kBoxWords = (int)(sizeof(BoxDev) / sizeof(int));
        static_assert(sizeof(BoxDev) % sizeof(int) == 0, "BoxDev copied as words");
        for (int k = tid; k < kBoxWords; k += kSortThreads)
            reinterpret_cast<int *>(a.boxLast)[k] = reinterpret_cast<const int *>(a.bx)[k];
    }
    const Geometry g = a.bx->geo;
    // atoms of the chunks before this one
    int before = 0;
    constexpr int U = 8;
    for (int k0 = tid; k0 < blk; k0 += U * kSortThreads) {
        int v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = k0 + u * kSortThreads < blk ? a.chunkSum[k0 + u * kSortThreads] : 0;
#pragma unroll
        for (int u = 0; u < U; ++u) before += v[u];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o, 64);
    if (lane == 0) wsum[w] = before;
    __syncthreads();
    int base = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    const int c0 = blk << a.csh, c1 = min(c0 + (1 << a.csh), a.nslot);
    for (int cb = c0; cb < c1; cb += a.cpw) {
        const int c = cb + tid;
        const bool live = tid < a.cpw && c < c1;
        // the first entries of the cell's list stay in registers
        constexpr int R = 8;
        int e[R], m = 0, h = live ? a.head[c] : -1;
        if (live) a.head[c] = -1;
        const int first = h;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            e[r] = h;
            if (h >= 0) {
                h = a.next[h];
                ++m;
            }
        }
        while (h >= 0) {
            h = a.next[h];
            ++m;
        }
        int x = m;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(x, o, 64);
            if (lane >= o) x += y;
        }
        __syncthreads();  // wsum and the lists' buffers of the round before are free
        if (lane == 63) wsum[w] = x;
        __syncthreads();
        int pre = x - m;
        for (int k = 0; k < w; ++k) pre += wsum[k];
        const int total = wsum[0] + wsum[1] + wsum[2] + wsum[3];
        if (live) a.start[c] = base + pre;
        sStart[tid] = pre;
        if (tid == 0) sStart[kSortThreads] = total;
        if (total <= kSortCap) {  // uniform
            int k = pre;
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (r < m) {
                    sIdx[k] = e[r];
                    sCell[k++] = (unsigned char)tid;
                }
            if (m > R)
                for (h = a.next[e[R - 1]]; h >= 0; h = a.next[h]) {
                    sIdx[k] = h;
                    sCell[k++] = (unsigned char)tid;
                }
            __syncthreads();
            for (int t = tid; t < total; t += kSortThreads) sKey[t] = a.id0[sIdx[t]];
            __syncthreads();
            for (int t = tid; t < total; t += kSortThreads) {
                const int cl = sCell[t], s0 = sStart[cl], s1 = sStart[cl + 1], key = sKey[t];
                int r = s0;
                for (int j = s0; j < s1; ++j) r += sKey[j] < key;
                place_atom(a, sIdx[t], base + r, key, g);
            }
        } else {
            for (int o = first; o >= 0; o = a.next[o]) {
                const int key = a.id0[o];
                int r = pre;
                for (int j = first; j >= 0; j = a.next[j]) r += a.id0[j] < key;
                place_atom(a, o, base + r, key, g);
            }
        }
        base += total;
    }
    if (blk == nblk - 1 && tid == 0) a.start[a.nslot] = a.n;
}

__device__ __forceinline__ void xq_body(int blk, int nblk, int n, const double4 *__restrict__ pos, const float *__restrict__ q,
                     float4 *__restrict__ xq, const BoxDev *__restrict__ bx) {
    const Geometry g = bx->geo;
    int k = blk * blockDim.x + threadIdx.x;
    if (k >= n) return;
    double4 p = pos[k];
    xq[k] = make_float4((float)(p.x - g.lo[0]), (float)(p.y - g.lo[1]), (float)(p.z - g.lo[2]), q[k]);
}

// k_xq fused with the clearing of the fixed-point force rows and of the
// energy / virial accumulators that the force kernels add into; with P3M on
// (rec set) also each charged site's mesh point and offsets for the spread
// and the gather of the same force evaluation.
__device__ __forceinline__ void xq_zero_body(int blk, int nblk, int n, const double4 *__restrict__ pos, const float *__restrict__ q,
                          float4 *__restrict__ xq, const BoxDev *__restrict__ bx,
                          unsigned long long *__restrict__ force, int nacc, unsigned long long *__restrict__ acc,
                          float4 *__restrict__ rec, RowMaxArgs rm) {
    if (rm.on && blk == nblk - 1) {  // uniform over the workgroup
        if (!rm.gate || *rm.gate != 0) row_max_wg(rm.na, rm.a, rm.nb, rm.b, rm.flags);
        return;
    }
    const Geometry g = bx->geo;
    int k = blk * blockDim.x + threadIdx.x;
    if (k < nacc) acc[k] = 0ull;
    if (k >= n) return;
    double4 p = pos[k];
    const float qk = q[k];
    xq[k] = make_float4((float)(p.x - g.lo[0]), (float)(p.y - g.lo[1]), (float)(p.z - g.lo[2]), qk);
    force[3 * (size_t)k + 0] = 0ull;
    force[3 * (size_t)k + 1] = 0ull;
    force[3 * (size_t)k + 2] = 0ull;
    if (rec && qk != 0.0f) rec[k] = mesh_record(p, bx->mesh);
}

// The step decisions as a launch of their own (one wave), from the nb
// per-workgroup maxima of the displacement check.
__device__ __forceinline__ void decide_body(int blk, int nblk, int nb, DecideArgs d) {
    float d2, p2;
    part_max(nb, d.part, d2, p2);
    if (threadIdx.x == 0) decide_write(d, d2 > d.half2);
}

// Stencil walk without local arrays (a dynamically indexed local array would
// live in scratch memory): along x and y, slot s of axis_slots() is either
// one of the (2 reach + 1) cells around c with periodic wrap, or every cell
// once when the axis has fewer cells; -1 marks a slot outside a non-periodic
// box.  Along z the candidates of a column are one or two contiguous runs.
__device__ __forceinline__ int axis_slots(int nc, int reach) { return nc < 2 * reach + 1 ? nc : 2 * reach + 1; }

__device__ __forceinline__ int axis_cell(int s, int c, int nc, int reach, int periodic) {
    if (nc < 2 * reach + 1) return s;
    int cc = c - reach + s;
    if (cc < 0 || cc >= nc) {
        if (!periodic) return -1;
        cc = cc < 0 ? cc + nc : cc - nc;
    }
    return cc;
}

// One or two contiguous runs of z-cells of a column; k0 / k1 is the image
// (-1, 0, +1 box lengths) in which a run's cells sit in the unwrapped stencil.
struct ZRuns {
    int n, lo0, hi0, lo1, hi1, k0, k1;
};

__device__ __forceinline__ ZRuns z_runs(int cz, int ncz, int reach, int periodic) {
    ZRuns z;
    z.k0 = z.k1 = 0;
    if (ncz < 2 * reach + 1) {
        z.n = 1;
        z.lo0 = 0;
        z.hi0 = ncz - 1;
        z.lo1 = z.hi1 = 0;
        return z;
    }
    int lo = cz - reach, hi = cz + reach;
    z.n = 1;
    z.lo1 = z.hi1 = 0;
    if (lo < 0) {
        if (periodic) {
            z.lo1 = lo + ncz;
            z.hi1 = ncz - 1;
            z.k1 = -1;
            z.n = 2;
        }
        lo = 0;
    } else if (hi >= ncz) {
        if (periodic) {
            z.lo1 = 0;
            z.hi1 = hi - ncz;
            z.k1 = 1;
            z.n = 2;
        }
        hi = ncz - 1;
    }
    z.lo0 = lo;
    z.hi0 = hi;
    return z;
}

__device__ __forceinline__ float dist2f(const float4 &a, const float4 &b, const Prefilter &p) {
    float dx = b.x - a.x, dy = b.y - a.y, dz = b.z - a.z;
    dx -= p.L[0] * rintf(dx * p.invL[0]);
    dy -= p.L[1] * rintf(dy * p.invL[1]);
    dz -= p.L[2] * rintf(dz * p.invL[2]);
    return dx * dx + dy * dy + dz * dz;
}

// z-cells [ulo, uhi] (unwrapped, within one period of [0, nc)) as one or two
// contiguous runs of a periodic column
__device__ __forceinline__ ZRuns z_runs_cut(int ulo, int uhi, int ncz) {
    ZRuns z;
    z.n = 1;
    z.lo1 = z.hi1 = 0;
    z.k0 = z.k1 = 0;
    if (ulo > uhi) {
        z.n = 0;
        z.lo0 = z.hi0 = 0;
        return z;
    }
    if (ulo < 0) {
        if (uhi < 0) {
            z.lo0 = ulo + ncz;
            z.hi0 = uhi + ncz;
            z.k0 = -1;
        } else {
            z.lo0 = 0;
            z.hi0 = uhi;
            z.lo1 = ulo + ncz;
            z.hi1 = ncz - 1;
            z.k1 = -1;
            z.n = 2;
        }
    } else if (uhi >= ncz) {
        if (ulo >= ncz) {
            z.lo0 = ulo - ncz;
            z.hi0 = uhi - ncz;
            z.k0 = 1;
        } else {
            z.lo0 = ulo;
            z.hi0 = ncz - 1;
            z.lo1 = 0;
            z.hi1 = uhi - ncz;
            z.k1 = 1;
            z.n = 2;
        }
    } else {
        z.lo0 = ulo;
        z.hi0 = uhi;
    }
    return z;
}

__device__ __forceinline__ float axis_gap(int u, float w, float x) {
    const float a = (float)u * w;
    return fmaxf(0.0f, fmaxf(a - x, x - (a + w)));
}

// One team of T lanes per atom walks the culled stencil.  The team first
// lays out its table of candidate runs in LDS, one stencil column per lane
// (column bases and cell starts are then fetched in parallel, not as a chain
// of dependent loads per column): the runs of the charged atoms' grid, then
// those of the charge-free atoms' grid, each run padded to whole chunks of T
// so that one stream of chunks covers them all and a chunk never straddles two
// runs (the run of a chunk is uniform over the team; padding lanes test
// nothing).  The team then walks the stream U chunks at a time with all U
// loads in flight.  Hits are compacted with a ballot restricted to the team,
// so row order is (charge class, stencil column, z-run, index) -
// deterministic - and the row splits at nlCountA into charged and charge-free
// partners.
//
// SHIFT: every axis is open or holds >= 2 reach + 1 cells, so each candidate
// of a run sits in one known image of the unwrapped stencil (the run's image
// offsets are stored with it) and the FP32 pre-test is a plain difference
// against the shifted atom; otherwise it takes the minimum image by rint.
//
// Exclusion partners arrive as current indices (idx | tag << 30, rows of
// maxExcl padded with ~0u); the first four sit in registers and are compared
// only within runs flagged as holding one of them or the atom itself, further
// ones are read for hit lanes only.
constexpr int kMaxCols = 25;  // (2 reach + 1)^2 columns for an xy reach of up to 2
constexpr int kEndBits = 20;  // run ends in a team's candidate stream
constexpr uint32_t kEndMask = (1u << kEndBits) - 1u;

__device__ __forceinline__ bool in_run(uint32_t ex, int s0, int s1) {
    const int j = (int)(ex & 0x3FFFFFFFu);
    return ex != ~0u && j >= s0 && j < s1;
}

// Which parts of its row an atom needs (bit 0 charged partners, bit 1
// charge-free ones), from list_need's mask: four bits a type, the low two for
// charged atoms of the type, the high two for charge-free ones.  The pair and
// E3B kernels read only these parts (in TIP4P water a charged site reads its
// charged partners and an oxygen its charge-free ones: 0.6 of the entries), so
// a step's build leaves the rest out; nlist_complete adds it when the whole
// list is asked for.
__device__ __forceinline__ unsigned row_parts(unsigned long long need, int type, float q) {
    return (unsigned)(need >> (4 * type + (q != 0.0f ? 0 : 2))) & 3u;
}

template <int T, bool SHIFT>
__device__ __forceinline__ void build_body(int blk, int nblk, const int *__restrict__ gate, 
    int n, const double4 *__restrict__ pos, const float4 *__restrict__ xq, const BoxDev *__restrict__ bx,
    const int *__restrict__ colRank, const int *__restrict__ cellStart, int ncell,
    double rlist2, const uint32_t *__restrict__ exclIdx, int maxExcl, const int *__restrict__ type,
    unsigned long long need, int cap,
    uint32_t *__restrict__ nl, int *__restrict__ nlCount, int *__restrict__ nlCountA, int *__restrict__ flags,
    int *__restrict__ waveMax) {
    if (gate && *gate == 0) return;
    const Geometry g = bx->geo;
    const CellGrid cg = bx->cg;
    const Prefilter pf = bx->pf;
    const Cull cu = bx->cu;
    constexpr int U = T >= 32 ? 1 : 32 / T;  // chunks of T candidates per load block
    constexpr int R = 4 * kMaxCols;           // runs per table: 2 classes x 2 z-runs per column
    __shared__ int sOff[256 / T][R];          // atom index = stream position + sOff
    __shared__ uint32_t sEnd[256 / T][R];     // end of the run's candidates | code << kEndBits
    const int gtid = blk * blockDim.x + threadIdx.x;
    const int i = gtid / T;
    const int team = threadIdx.x / T;
    const int tl = threadIdx.x & (T - 1);
    const int lane = threadIdx.x & 63;
    const bool live = i < n;
    const int rx = cg.reach[0], ry = cg.reach[1], rz = cg.reach[2];
    const int sx = axis_slots(cg.nc[0], rx), sy = axis_slots(cg.nc[1], ry);
    const int ncol = sx * sy;
    const int ncz = cg.nc[2];
    // team-uniform stream lengths: runs are padded to whole chunks of T, so a
    // chunk never straddles two runs; [0, totalA) walks the charged atoms
    int total = 0, totalA = 0;
    if (live) {
        const double4 pi = pos[i];
        const float4 xi = xq[i];
        const int cx = cell_coord(pi.x, g.lo[0], cg.cellInv[0], cg.nc[0]);
        const int cy = cell_coord(pi.y, g.lo[1], cg.cellInv[1], cg.nc[1]);
        const int cz = cell_coord(pi.z, g.lo[2], cg.cellInv[2], cg.nc[2]);
        const uint32_t *exRow = exclIdx + (size_t)i * maxExcl;
        const uint32_t ex0 = maxExcl > 0 ? exRow[0] : ~0u, ex1 = maxExcl > 1 ? exRow[1] : ~0u;
        const uint32_t ex2 = maxExcl > 2 ? exRow[2] : ~0u, ex3 = maxExcl > 3 ? exRow[3] : ~0u;
        int nrun = 0;
        const unsigned parts = row_parts(need, type[i], xi.w);
#pragma unroll 1
        for (int cls = 0; cls < 2; ++cls) {
            const int *cs = cellStart + cls * ncell;
            for (int c0 = 0; (parts >> cls & 1u) && c0 < ncol; c0 += T) {
                const int col = c0 + tl;
                int st0 = 0, len0 = 0, st1 = 0, len1 = 0;
                uint32_t code0 = 0, code1 = 0;
                if (col < ncol) {
                    const int a = col / sy, b = col - a * sy;
                    const int xx = axis_cell(a, cx, cg.nc[0], rx, g.periodic[0]);
                    const int yy = axis_cell(b, cy, cg.nc[1], ry, g.periodic[1]);
                    const float gx = cu.on[0] ? axis_gap(cx - rx + a, cu.w[0], xi.x) : 0.0f;
                    const float gy = cu.on[1] ? axis_gap(cy - ry + b, cu.w[1], xi.y) : 0.0f;
                    const float gxy2 = gx * gx + gy * gy;
                    if (xx >= 0 && yy >= 0 && gxy2 <= cu.r2) {
                        ZRuns zr;
                        if (cu.on[2]) {
                            const float h = sqrtf(cu.r2 - gxy2);
                            const int ulo = max((int)floorf((xi.z - h) / cu.w[2]), cz - rz);
                            const int uhi = min((int)floorf((xi.z + h) / cu.w[2]), cz + rz);
                            zr = z_runs_cut(ulo, uhi, ncz);
                        } else {
                            zr = z_runs(cz, ncz, rz, g.periodic[2]);
                        }
                        const int colBase = colRank[xx * cg.nc[1] + yy] * ncz;
                        if (zr.n > 0) {
                            st0 = cs[colBase + zr.lo0];
                            len0 = cs[colBase + zr.hi0 + 1] - st0;
                        }
                        if (zr.n > 1) {
                            st1 = cs[colBase + zr.lo1];
                            len1 = cs[colBase + zr.hi1 + 1] - st1;
                        }
                        const int ux = cx - rx + a, uy = cy - ry + b;
                        const uint32_t kx = ux < 0 ? 0u : (ux >= cg.nc[0] ? 2u : 1u);
                        const uint32_t ky = uy < 0 ? 0u : (uy >= cg.nc[1] ? 2u : 1u);
                        // flag: the run holds the atom itself or an exclusion partner
                        const uint32_t f0 =
                            (maxExcl > 4 || (i >= st0 && i < st0 + len0) || in_run(ex0, st0, st0 + len0) ||
                             in_run(ex1, st0, st0 + len0) || in_run(ex2, st0, st0 + len0) ||
                             in_run(ex3, st0, st0 + len0)) ? 1u : 0u;
                        const uint32_t f1 =
                            (maxExcl > 4 || (i >= st1 && i < st1 + len1) || in_run(ex0, st1, st1 + len1) ||
                             in_run(ex1, st1, st1 + len1) || in_run(ex2, st1, st1 + len1) ||
                             in_run(ex3, st1, st1 + len1)) ? 1u : 0u;
                        code0 = kx | (ky << 2) | ((uint32_t)(zr.k0 + 1) << 4) | (f0 << 6);
                        code1 = kx | (ky << 2) | ((uint32_t)(zr.k1 + 1) << 4) | (f1 << 6);
                    }
                }
                // team prefix sums place the non-empty runs in column order
                const int nr = (len0 > 0 ? 1 : 0) + (len1 > 0 ? 1 : 0);
                const int pl0 = (len0 + T - 1) & ~(T - 1), pl1 = (len1 + T - 1) & ~(T - 1);
                const int ln = pl0 + pl1;
                int snr = nr, sln = ln;
#pragma unroll
                for (int o = 1; o < T; o <<= 1) {
                    const int y0 = __shfl_up(snr, o, T), y1 = __shfl_up(sln, o, T);
                    if (tl >= o) {
                        snr += y0;
                        sln += y1;
                    }
                }
                int e = nrun + snr - nr, v = total + sln - ln;
                if (len0 > 0) {
                    sOff[team][e] = st0 - v;
                    sEnd[team][e] = (uint32_t)(v + len0) | (code0 << kEndBits);
                    v += pl0;
                    ++e;
                }
                if (len1 > 0) {
                    sOff[team][e] = st1 - v;
                    sEnd[team][e] = (uint32_t)(v + len1) | (code1 << kEndBits);
                }
                nrun += __shfl(snr, T - 1, T);
                total += __shfl(sln, T - 1, T);
            }
            if (cls == 0) totalA = total;
        }
        // stream positions are kEndBits wide
        if (tl == 0 && total >= (1 << kEndBits)) atomicOr(&flags[7], 1);
    }
    // a team lies inside one wave and reads only its own table
    wave_sync();
    int cnt = 0;
    if (live && total < (1 << kEndBits)) {
        const unsigned long long teamMask =
            (T == 64) ? ~0ull : (((1ull << T) - 1ull) << (lane & ~(T - 1)));
        const uint32_t tmLo = (uint32_t)teamMask, tmHi = (uint32_t)(teamMask >> 32);
        const double4 pi = pos[i];
        const float4 xi = xq[i];
        const uint32_t *exRow = exclIdx + (size_t)i * maxExcl;
        const uint32_t ex0 = maxExcl > 0 ? exRow[0] : ~0u, ex1 = maxExcl > 1 ? exRow[1] : ~0u;
        const uint32_t ex2 = maxExcl > 2 ? exRow[2] : ~0u, ex3 = maxExcl > 3 ? exRow[3] : ~0u;
        const uint32_t e0 = ex0 & 0x3FFFFFFFu, e1 = ex1 & 0x3FFFFFFFu, e2 = ex2 & 0x3FFFFFFFu, e3 = ex3 & 0x3FFFFFFFu;
        uint32_t *row = nl + (size_t)i * cap;
        int cntA = 0;
        // the team's current run (team-uniform): offset, end of its real
        // candidates, flag bit, and the atom moved into the run's image frame;
        // the next entry is read ahead
        int r = -1, off = 0, vend = 0;
        uint32_t fl = 0, img = 0x15u;  // image code of the interior, (0, 0, 0) + 1 per axis
        float xsx = xi.x, xsy = xi.y, xsz = xi.z;
        int nOff = sOff[team][0];
        uint32_t nEnd = sEnd[team][0];
        for (int v0 = 0; v0 < total; v0 += U * T) {
            uint32_t jv[U];  // atom index, bit 31: flagged run
            float px[U], py[U], pz[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int p = v0 + u * T;
                if (p < total && p >= vend) {
                    ++r;
                    off = nOff;
                    vend = (int)(nEnd & kEndMask);
                    const uint32_t code = nEnd >> kEndBits;
                    fl = (code >> 6) << 31;
                    // most runs share the image of the previous one
                    if (SHIFT && (code & 0x3Fu) != img) {
                        img = code & 0x3Fu;
                        xsx = xi.x - (float)((int)(code & 3u) - 1) * pf.L[0];
                        xsy = xi.y - (float)((int)((code >> 2) & 3u) - 1) * pf.L[1];
                        xsz = xi.z - (float)((int)((code >> 4) & 3u) - 1) * pf.L[2];
                    }
                    const int rn = min(r + 1, R - 1);
                    nOff = sOff[team][rn];
                    nEnd = sEnd[team][rn];
                }
                const int v = p + tl;
                // padding and positions past the stream: the atom itself in a
                // flagged slot (never a hit)
                jv[u] = (p < total && v < vend) ? ((uint32_t)(v + off) | fl) : ((uint32_t)i | 0x80000000u);
                px[u] = xsx;
                py[u] = xsy;
                pz[u] = xsz;
            }
            float4 blk[U];
#pragma unroll
            for (int u = 0; u < U; ++u) blk[u] = xq[jv[u] & 0x7FFFFFFFu];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (v0 + u * T == totalA) cntA = cnt;  // first charge-free chunk
                const int j = (int)(jv[u] & 0x7FFFFFFFu);
                const float4 cur = blk[u];
                float r2f;
                if (SHIFT) {
                    const float dx = cur.x - px[u], dy = cur.y - py[u], dz = cur.z - pz[u];
                    r2f = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
                } else {
                    r2f = dist2f(xi, cur, pf);
                }
                bool hit = r2f < pf.lo2;
                if (!hit && r2f <= pf.hi2) hit = dist2(pi, pos[j], g) < rlist2;
                uint32_t tag = 0;
                if ((int)jv[u] < 0) {
                    hit = hit && j != i;
                    const uint32_t uj = (uint32_t)j;
                    tag = e0 == uj ? ex0 >> 30 : tag;
                    tag = e1 == uj ? ex1 >> 30 : tag;
                    tag = e2 == uj ? ex2 >> 30 : tag;
                    tag = e3 == uj ? ex3 >> 30 : tag;
                    if (maxExcl > 4 && hit)
                        for (int q = 4; q < maxExcl; ++q) {
                            const uint32_t e = exRow[q];
                            if ((e & 0x3FFFFFFFu) == uj) tag = e >> 30;
                        }
                }
                const unsigned long long m = __ballot(hit);
                const uint32_t mLo = (uint32_t)m & tmLo, mHi = (uint32_t)(m >> 32) & tmHi;
                if (hit) {
                    // team hits in lower lanes, counted by mbcnt on the masked ballot
                    const int k = (int)__builtin_amdgcn_mbcnt_hi(mHi, __builtin_amdgcn_mbcnt_lo(mLo, (uint32_t)cnt));
                    if (k < cap) row[k] = (uint32_t)j | (tag << 30);
                }
                cnt += __popc(mLo) + __popc(mHi);
            }
        }
        if (totalA >= total) cntA = cnt;  // no charge-free candidates
        if (tl == 0) {
            nlCount[i] = cnt;
            nlCountA[i] = cntA;
        }
    }
    // the longest row of the wave goes to the wave's own slot (k_row_max
    // reduces them): same-address device atomics serialise across the XCDs
    const int wmax = wave_max(cnt);
    if (lane == 0) waveMax[gtid >> 6] = wmax;
}

// One wave per atom (the team width 64 of the tuner).  The 64 lanes lay out
// the table in one step: lanes 0..31 take the columns of the charged atoms'
// grid, lanes 32..63 those of the charge-free atoms' grid, and a wave-wide
// prefix sum places the runs, unpadded, in one stream (class, column, z-run
// order).  Each table entry carries the run's end in the stream, the offset
// from stream position to atom index, its flag and the atom moved into the
// run's image frame (uniform over the wave, so computed once per run).  The
// wave then walks the stream 64 candidates per chunk and U chunks per block:
// a lane finds its run from the run of the chunk start (runs are rarely
// shorter than the few lanes they straddle), so the bookkeeping is a couple
// of LDS reads per lane and the compaction is one mbcnt on the wave ballot.
// the exclusion rows of the sort, translated to current indices as they are
// read (the sort has just renumbered the atoms)
struct ExclArgs {
    int maxExcl;
    const uint32_t *row;
    const int *idToIdx;
};
__device__ __forceinline__ uint32_t excl_entry(const ExclArgs &x, int i, int q) {
    const uint32_t e = x.row[(size_t)i * x.maxExcl + q];
    return e == ~0u ? e : (uint32_t)x.idToIdx[e & 0x3FFFFFFFu] | (e & 0xC0000000u);
}

// The E3B molecule list made by the wave build: for an oxygen of E3B water, the
// molecules of the oxygens among its row's hits within (r2b + skin), in row
// order (what e3b_list_body makes of a finished row).  As a launch of its own,
// reading the rows back, it took 14.2 us a rebuild for 8,192 molecules and
// 25.5 us for 32,768; here it is a second ballot in a quarter of the waves.
struct OxListArgs {
    const int *mol;  // by atom id: molecule index of an oxygen, else -1 (nullptr: no E3B)
    const int *id;
    double r2;
    float r2f;       // r2 with the pre-test's margin
    int cap;
    int *nl, *count, *wmax;
};

struct RunEntry {
    int vend;      // end of the run in the stream
    int off;       // atom index = stream position + off
    uint32_t fl;   // bit 31: the run holds the atom itself or an exclusion partner
    float xs[3];   // the atom in the run's image frame
};

// The canonical distance of the few candidates near a cutoff: the box and the
// atom are read again here (the barrier keeps the loads from moving out of the
// branch) instead of living in scalar registers through the walk, whose
// number decides how many waves a SIMD holds: 500,000 LJ atoms 651 -> 525 us.
// The builds that also make the E3B list need more vector registers and lose
// a wave to the extra addresses (313 -> 330 us at 131,072 sites), so they keep
// the values.
__device__ __forceinline__ double dist2_at(const double4 *__restrict__ pos, int i, int j, const BoxDev *bx) {
    asm volatile("" : "+s"(bx), "+s"(i));
    return dist2(pos[i], pos[j], bx->geo);
}

// OX: the set-up has E3B water (the list code costs registers).
template <bool SHIFT, bool OX>
__device__ __forceinline__ void build_wave_body(int blk, int nblk, const int *__restrict__ gate,
    int n, const double4 *__restrict__ pos, const float4 *__restrict__ xq, const BoxDev *__restrict__ bx,
    const int *__restrict__ colRank, const int *__restrict__ cellStart, int ncell,
    double rlist2, ExclArgs ex, const int *__restrict__ type, unsigned long long need, OxListArgs ox, int cap,
    uint32_t *__restrict__ nl, int *__restrict__ nlCount, int *__restrict__ nlCountA, int *__restrict__ flags,
    int *__restrict__ waveMax) {
    if (gate && *gate == 0) return;
    const Geometry g = bx->geo;
    const CellGrid cg = bx->cg;
    const Prefilter pf = bx->pf;
    const Cull cu = bx->cu;
    constexpr int U = 4;             // chunks of 64 candidates per load block
    constexpr int R = 4 * kMaxCols;  // 2 classes x 2 z-runs per column
    __shared__ RunEntry sRun[4][R + 1];
    __shared__ uint32_t sEx[4][64];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int i = __builtin_amdgcn_readfirstlane(blk * 4 + (int)(threadIdx.x >> 6));
    if (i >= n) {
        if (lane == 0) waveMax[i] = 0;
        return;
    }
    const int rx = cg.reach[0], ry = cg.reach[1], rz = cg.reach[2];
    const int sx = axis_slots(cg.nc[0], rx), sy = axis_slots(cg.nc[1], ry);
    const int ncol = sx * sy;
    const int ncz = cg.nc[2];
    const double4 pi = pos[i];
    const float4 xi = xq[i];
    const int cx = cell_coord(pi.x, g.lo[0], cg.cellInv[0], cg.nc[0]);
    const int cy = cell_coord(pi.y, g.lo[1], cg.cellInv[1], cg.nc[1]);
    const int cz = cell_coord(pi.z, g.lo[2], cg.cellInv[2], cg.nc[2]);
    // exclusion partners in current indices, one per lane: the first four are
    // uniform, further ones go to LDS
    uint32_t exv = ~0u;
    if (ex.maxExcl > 0) {
        if (lane < ex.maxExcl) exv = excl_entry(ex, i, lane);
        if (ex.maxExcl > 4) sEx[w][lane] = exv;
    }
    const int maxExcl = ex.maxExcl;
    const uint32_t ex0 = (uint32_t)__builtin_amdgcn_readlane((int)exv, 0), ex1 = (uint32_t)__builtin_amdgcn_readlane((int)exv, 1);
    const uint32_t ex2 = (uint32_t)__builtin_amdgcn_readlane((int)exv, 2), ex3 = (uint32_t)__builtin_amdgcn_readlane((int)exv, 3);
    const unsigned parts = row_parts(need, type[i], xi.w);
    const int mol = OX ? ox.mol[ox.id[i]] : -1;  // an E3B oxygen's molecule: its list is made here too
    // ---- table: one (class, column) per lane
    const int cls = lane >> 5, col = lane & 31;
    const int *cs = cellStart + cls * ncell;
    int st0 = 0, len0 = 0, st1 = 0, len1 = 0;
    uint32_t f0 = 0, f1 = 0;
    float s0x = xi.x, s0y = xi.y, s0z = xi.z, s1x = xi.x, s1y = xi.y, s1z = xi.z;
    if (col < ncol && (parts >> cls & 1u)) {
        const int a = col / sy, b = col - a * sy;
        const int xx = axis_cell(a, cx, cg.nc[0], rx, g.periodic[0]);
        const int yy = axis_cell(b, cy, cg.nc[1], ry, g.periodic[1]);
        const float gx = cu.on[0] ? axis_gap(cx - rx + a, cu.w[0], xi.x) : 0.0f;
        const float gy = cu.on[1] ? axis_gap(cy - ry + b, cu.w[1], xi.y) : 0.0f;
        const float gxy2 = gx * gx + gy * gy;
        if (xx >= 0 && yy >= 0 && gxy2 <= cu.r2) {
            ZRuns zr;
            if (cu.on[2]) {
                const float h = sqrtf(cu.r2 - gxy2);
                const int ulo = max((int)floorf((xi.z - h) / cu.w[2]), cz - rz);
                const int uhi = min((int)floorf((xi.z + h) / cu.w[2]), cz + rz);
                zr = z_runs_cut(ulo, uhi, ncz);
            } else {
                zr = z_runs(cz, ncz, rz, g.periodic[2]);
            }
            const int colBase = colRank[xx * cg.nc[1] + yy] * ncz;
            if (zr.n > 0) {
                st0 = cs[colBase + zr.lo0];
                len0 = cs[colBase + zr.hi0 + 1] - st0;
            }
            if (zr.n > 1) {
                st1 = cs[colBase + zr.lo1];
                len1 = cs[colBase + zr.hi1 + 1] - st1;
            }
            f0 = (maxExcl > 4 || (i >= st0 && i < st0 + len0) || in_run(ex0, st0, st0 + len0) ||
                  in_run(ex1, st0, st0 + len0) || in_run(ex2, st0, st0 + len0) || in_run(ex3, st0, st0 + len0))
                     ? 0x80000000u : 0u;
            f1 = (maxExcl > 4 || (i >= st1 && i < st1 + len1) || in_run(ex0, st1, st1 + len1) ||
                  in_run(ex1, st1, st1 + len1) || in_run(ex2, st1, st1 + len1) || in_run(ex3, st1, st1 + len1))
                     ? 0x80000000u : 0u;
            if (SHIFT) {
                const int ux = cx - rx + a, uy = cy - ry + b;
                const float kx = ux < 0 ? -1.0f : (ux >= cg.nc[0] ? 1.0f : 0.0f);
                const float ky = uy < 0 ? -1.0f : (uy >= cg.nc[1] ? 1.0f : 0.0f);
                s0x = s1x = xi.x - kx * pf.L[0];
                s0y = s1y = xi.y - ky * pf.L[1];
                s0z = xi.z - (float)zr.k0 * pf.L[2];
                s1z = xi.z - (float)zr.k1 * pf.L[2];
            }
        }
    }
    const int nr = (len0 > 0 ? 1 : 0) + (len1 > 0 ? 1 : 0);
    const int ln = len0 + len1;
    int snr = nr, sln = ln;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y0 = __shfl_up(snr, o, 64), y1 = __shfl_up(sln, o, 64);
        if (lane >= o) {
            snr += y0;
            sln += y1;
        }
    }
    {
        int e = snr - nr, v = sln - ln;
        if (len0 > 0) {
            RunEntry &q = sRun[w][e];
            q.vend = v + len0;
            q.off = st0 - v;
            q.fl = f0;
            q.xs[0] = s0x;
            q.xs[1] = s0y;
            q.xs[2] = s0z;
            v += len0;
            ++e;
        }
        if (len1 > 0) {
            RunEntry &q = sRun[w][e];
            q.vend = v + len1;
            q.off = st1 - v;
            q.fl = f1;
            q.xs[0] = s1x;
            q.xs[1] = s1y;
            q.xs[2] = s1z;
        }
    }
    const int nrun = __shfl(snr, 63, 64);
    const int total = __shfl(sln, 63, 64);
    const int totalA = __shfl(sln, 31, 64);
    // a sentinel past the last run stops every search
    if (lane == 0) {
        RunEntry &q = sRun[w][nrun];
        q.vend = 0x7FFFFFFF;
        q.off = 0;
        q.fl = 0x80000000u;
        q.xs[0] = xi.x;
        q.xs[1] = xi.y;
        q.xs[2] = xi.z;
    }
    wave_sync();
    // ---- walk
    const uint32_t e0 = ex0 & 0x3FFFFFFFu, e1 = ex1 & 0x3FFFFFFFu, e2 = ex2 & 0x3FFFFFFFu, e3 = ex3 & 0x3FFFFFFFu;
    uint32_t *row = nl + (size_t)i * cap;
    int cnt = 0, cntA = 0, cntO = 0;
    int ra = 0;  // run of the current chunk start (uniform)
    for (int p0 = 0; p0 < total; p0 += 64 * U) {
        uint32_t jv[U];
        float px[U], py[U], pz[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int p = p0 + 64 * u;
            // chunk start's run (uniform search)
            while (__builtin_amdgcn_readfirstlane(sRun[w][ra].vend) <= p) ++ra;
            const int v = p + lane;
            int r = ra;
            while (v >= sRun[w][r].vend) ++r;
            const RunEntry q = sRun[w][r];
            // past the stream: the atom itself in a flagged slot (never a hit)
            jv[u] = v < total ? ((uint32_t)(v + q.off) | q.fl) : ((uint32_t)i | 0x80000000u);
            px[u] = q.xs[0];
            py[u] = q.xs[1];
            pz[u] = q.xs[2];
        }
        float4 blk[U];
#pragma unroll
        for (int u = 0; u < U; ++u) blk[u] = xq[jv[u] & 0x7FFFFFFFu];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int p = p0 + 64 * u;
            const int j = (int)(jv[u] & 0x7FFFFFFFu);
            const float4 cur = blk[u];
            float r2f;
            if (SHIFT) {
                const float dx = cur.x - px[u], dy = cur.y - py[u], dz = cur.z - pz[u];
                r2f = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
            } else {
                r2f = dist2f(xi, cur, pf);
            }
            bool hit = r2f < pf.lo2;
            if (!hit && r2f <= pf.hi2) hit = (OX ? dist2(pi, pos[j], g) : dist2_at(pos, i, j, bx)) < rlist2;
            uint32_t tag = 0;
            if ((int)jv[u] < 0) {
                hit = hit && j != i;
                const uint32_t uj = (uint32_t)j;
                tag = e0 == uj ? ex0 >> 30 : tag;
                tag = e1 == uj ? ex1 >> 30 : tag;
                tag = e2 == uj ? ex2 >> 30 : tag;
                tag = e3 == uj ? ex3 >> 30 : tag;
                if (maxExcl > 4 && hit) {
                    for (int qq = 4; qq < maxExcl; ++qq) {
                        const uint32_t e = qq < 64 ? sEx[w][qq] : excl_entry(ex, i, qq);
                        if ((e & 0x3FFFFFFFu) == uj) tag = e >> 30;
                    }
                }
            }
            const unsigned long long m = __ballot(hit);
            if (hit) {
                const int k = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                             __builtin_amdgcn_mbcnt_lo((uint32_t)m, (uint32_t)cnt));
                if (k < cap) row[k] = (uint32_t)j | (tag << 30);
            }
            if (OX && mol >= 0) {  // uniform: the oxygens among the hits within the molecule list's radius
                int mj = -1;
                if (hit && r2f <= ox.r2f) {
                    mj = ox.mol[ox.id[j]];
                    if (mj >= 0 && !(dist2(pi, pos[j], g) < ox.r2)) mj = -1;
                }
                const unsigned long long mo = __ballot(mj >= 0);
                if (mj >= 0) {
                    const int k = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mo >> 32),
                                                                 __builtin_amdgcn_mbcnt_lo((uint32_t)mo, (uint32_t)cntO));
                    if (k < ox.cap) ox.nl[(size_t)mol * ox.cap + k] = mj;
                }
                cntO += __popcll(mo);
            }
            // the charged/charge-free split falls inside this chunk
            if (p <= totalA && totalA < p + 64) {
                const int below = totalA - p;
                const unsigned long long lo = below >= 64 ? ~0ull : ((1ull << below) - 1ull);
                cntA = cnt + __popcll(m & lo);
            }
            cnt += __popcll(m);
        }
    }
    if (totalA >= total) cntA = cnt;
    if (lane == 0) {
        nlCount[i] = cnt;
        nlCountA[i] = cntA;
        waveMax[i] = cnt;
        if (OX && mol >= 0) {
            ox.count[mol] = cntO;
            ox.wmax[mol] = cntO;
        }
    }
}

// Exclusion rows from ids to current indices (idx | tag << 30), in place,
// for the team builds, which read them lane by lane.
__device__ __forceinline__ void excl_idx_body(int blk, int nblk, const int *__restrict__ gate, long long n,
                                              const int *__restrict__ idToIdx, uint32_t *__restrict__ row) {
    if (gate && *gate == 0) return;
    const long long k = (long long)blk * blockDim.x + threadIdx.x;
    if (k < n && row[k] != ~0u) row[k] = (uint32_t)idToIdx[row[k] & 0x3FFFFFFFu] | (row[k] & 0xC0000000u);
}

// E3B molecule list from the atom list: for each water, the oxygens among its
// oxygen's neighbors within (r2b + skin) at build time.  Replaces the private
// molecule GridGPU of FixE3B (FixE3B.cu:656-684) that the reference rebuilds
// every step; with the skin criterion the per-step r2b set is a subset.
template <int T>
__device__ __forceinline__ void e3b_list_body(int blk, int nblk, 
    const int *__restrict__ gate, int nmol, const int4 *__restrict__ molAtoms, const int *__restrict__ atomMolO,
    const double4 *__restrict__ pos, const BoxDev *__restrict__ bx, double rcut2, int cap,
    const uint32_t *__restrict__ nl,
    const int *__restrict__ nlCount, const int *__restrict__ nlCountA, int unchargedOnly, int mcap,
    int *__restrict__ mnl, int *__restrict__ mcount, int *__restrict__ waveMax) {
    if (gate && *gate == 0) return;
    const Geometry g = bx->geo;
    const int gtid = blk * blockDim.x + threadIdx.x;
    const int m = gtid / T;
    const int tl = threadIdx.x & (T - 1);
    const int lane = threadIdx.x & 63;
    int cnt = 0;
    if (m < nmol) {
        const unsigned long long teamMask =
            (T == 64) ? ~0ull : (((1ull << T) - 1ull) << (lane & ~(T - 1)));
        const unsigned long long below = (1ull << lane) - 1ull;
        const int oi = molAtoms[m].x;
        const double4 pi = pos[oi];
        const int total = min(nlCount[oi], cap);
        const int nA = min(nlCountA[oi], total);
        const uint32_t *row = nl + (size_t)oi * cap;
        // row = [charged partners | charge-free partners]; E3B oxygens of a
        // charge-free O site need only the second part
        const int first = unchargedOnly ? nA : 0;
        for (int base = first; base < total; base += T) {
            const int v = base + tl;
            bool hit = false;
            int mj = -1;
            if (v < total) {
                const int j = (int)(row[v] & 0x3FFFFFFFu);
                mj = atomMolO[j];
                if (mj >= 0 && mj != m) hit = dist2(pi, pos[j], g) < rcut2;
            }
            const unsigned long long msk = __ballot(hit) & teamMask;
            if (hit) {
                const int s = cnt + __popcll(msk & below);
                if (s < mcap) mnl[(size_t)m * mcap + s] = mj;
            }
            cnt += __popcll(msk);
        }
        if (tl == 0) mcount[m] = cnt;
    }
    const int wmax = wave_max(cnt);
    if (lane == 0) waveMax[gtid >> 6] = wmax;
}

// Molecule to current site indices after a re-sort (E3B, rigid and flexible
// molecules), with the oxygen map and the membership flags that the re-sort
// cleared, and the chunk counts of the binning cleared for the next one.
// Extra workgroups of the list build: the maps only need the new indices, and
// what reads them comes after (one launch fewer per step).
struct MolMapArgs {
    int blocks;
    int nmol;
    const int4 *molIds;
    const int *idToIdx;
    int4 *molAtoms;
    int *atomMolO;
    int nmolR;
    const int4 *rigidIds;
    int4 *rigidAtoms;
    int *member;
    int nmolF;
    const int4 *flexIds;
    int4 *flexAtoms;
    int nchunk;
    int *chunkSum;
};

__device__ __forceinline__ int4 mol_indices(const int4 &i, const int *__restrict__ idToIdx) {
    return make_int4(idToIdx[i.x], idToIdx[i.y], idToIdx[i.z], i.w >= 0 ? idToIdx[i.w] : -1);
}

__device__ __forceinline__ void mol_map_body(int blk, int nblk, const int *__restrict__ gate, MolMapArgs mm) {
    if (gate && *gate == 0) return;
    const int m = blk * blockDim.x + threadIdx.x;
    if (m < mm.nchunk) mm.chunkSum[m] = 0;
    if (m < mm.nmolR) {
        const int4 a = mol_indices(mm.rigidIds[m], mm.idToIdx);
        mm.rigidAtoms[m] = a;
        mm.member[a.x] = 1;
        mm.member[a.y] = 1;
        mm.member[a.z] = 1;
        if (a.w >= 0) mm.member[a.w] = 1;
    }
    if (m < mm.nmolF) mm.flexAtoms[m] = mol_indices(mm.flexIds[m], mm.idToIdx);
    if (m < mm.nmol) {
        const int4 a = mol_indices(mm.molIds[m], mm.idToIdx);
        mm.molAtoms[m] = a;
        mm.atomMolO[a.x] = m;
    }
}

template <bool SHIFT, bool OX>
__device__ __forceinline__ void build_map_body(int blk, int nblk, const int *__restrict__ gate,
    int n, const double4 *__restrict__ pos, const float4 *__restrict__ xq, const BoxDev *__restrict__ bx,
    const int *__restrict__ colRank, const int *__restrict__ cellStart, int ncell,
    double rlist2, ExclArgs ex, const int *__restrict__ type, unsigned long long need, OxListArgs ox, int cap,
    uint32_t *__restrict__ nl, int *__restrict__ nlCount, int *__restrict__ nlCountA, int *__restrict__ flags,
    int *__restrict__ waveMax, MolMapArgs mm) {
    const int nb = nblk - mm.blocks;
    if (blk >= nb) {  // uniform over the workgroup
        mol_map_body(blk - nb, mm.blocks, gate, mm);
        return;
    }
    build_wave_body<SHIFT, OX>(blk, nb, gate, n, pos, xq, bx, colRank, cellStart, ncell, rlist2, ex, type, need, ox, cap, nl,
                           nlCount, nlCountA, flags, waveMax);
}

__device__ __forceinline__ void fill_int_body(int blk, int nblk, const int *__restrict__ gate, int n, int *__restrict__ p, int v) {
    if (gate && *gate == 0) return;
    int i = blk * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Longest pair row and molecule row of the build from the per-wave slots,
// folded into the running maxima flags[1], flags[2] (one workgroup), and, for
// an eager build, with the stream overflow bits into the host's pinned words.
__device__ __forceinline__ void row_max_body(int blk, int nblk, const int *__restrict__ gate, int na, const int *__restrict__ a,
                                                  int nb, const int *__restrict__ b, int *__restrict__ flags,
                                                  int *__restrict__ host) {
    if (gate && *gate == 0) return;
    row_max_wg(na, a, nb, b, flags);
    if (host && threadIdx.x == 0) {
        host_store(host, flags[1]);
        host_store(host + 1, flags[2]);
        host_store(host + 6, flags[7]);
    }
}

uint32_t morton2(uint32_t x, uint32_t y) {
    uint64_t r = 0;
    for (int b = 0; b < 16; ++b) {
        r |= (uint64_t)((x >> b) & 1u) << (2 * b);
        r |= (uint64_t)((y >> b) & 1u) << (2 * b + 1);
    }
    return (uint32_t)r;
}

// The FP32 pre-test band (box_derive) covers the FP32 error of r^2 for
// wrapped positions (x - lo in [0, L]) and r <= r_list.  Per component the
// FP32 difference is off by at most ~5 L 2^-24 (two rounded inputs, the
// subtraction, the rounded L and the image shift); r^2 is then off by at most
// 2 sqrt(3) r_list of that plus a few ulp of r^2 for the squares and the sum.
// The band takes 16 L 2^-24 and 32 r^2 2^-24, about three times both.  The
// culling margin 1e-5 (L + r_list) is far above the FP32 rounding of
// coordinates and cell bounds (~L 2^-24) and far below a cell.

// slots of the pair-list waves in c.waveMax; the molecule-list slots follow
size_t wave_slots_a(const Ctx &c) { return (size_t)c.n + 4; }

// whether every candidate of a run sits in one known image of the stencil
bool build_shifts(const Ctx &c) {
    for (int a = 0; a < 3; ++a)
        if (c.geo.periodic[a] && c.nc[a] < 2 * c.reach[a] + 1) return false;
    return true;
}

// with the molecule maps of the rebuild in the same launch, and the E3B list
void launch_build_wave(Ctx &c, const double4 *bpos, const BoxDev *box, const MolMapArgs &mm, unsigned long long need) {
    const ExclArgs ex{c.exclOff ? c.maxExcl : 0, c.exclIdx, c.idToIdx};
    OxListArgs ox{};
    if (c.e3b.on) {
        const double rc = (double)c.e3b.r2b + c.skin, lmax = std::max({c.geo.L[0], c.geo.L[1], c.geo.L[2]});
        ox.mol = c.e3b.molIdsOfO;
        ox.id = c.id[c.cur];
        ox.r2 = rc * rc;
        ox.r2f = (float)(rc * rc * (1.0 + 1e-5) + 1e-5 * rc * lmax);  // far above the FP32 rounding of r^2
        ox.cap = c.e3b.cap;
        ox.nl = c.e3b.nl;
        ox.count = c.e3b.nlCount;
        ox.wmax = c.waveMax + wave_slots_a(c);
        c.waveMaxB = c.e3b.nmol;
    }
    const int blocks = cdiv(c.n, 4);
#define MDX_BUILD(S, O) launch<build_map_body<S, O>, 256>(c, blocks + mm.blocks, 0, rebuild_gate(c), c.n, bpos, c.xq, box, c.colRank, c.cellStart, c.ncell, c.rlist * c.rlist, ex, c.type[c.cur], need, ox, c.cap, c.nl, c.nlCount, c.nlCountA, c.dFlags, c.waveMax, mm)
    const bool shift = build_shifts(c);
    if (ox.mol) {
        if (shift) MDX_BUILD(true, true); else MDX_BUILD(false, true);
    } else {
        if (shift) MDX_BUILD(true, false); else MDX_BUILD(false, false);
    }
#undef MDX_BUILD
    c.waveMaxA = blocks * 4;
}

template <int T>
void launch_build(Ctx &c, const double4 *bpos, const BoxDev *box, unsigned long long need) {
    const int threads = 256;
    const int blocks = cdiv((long long)c.n * T, threads);
    if (build_shifts(c))
        launch<build_body<T, true>, 256>(c, blocks, 0, rebuild_gate(c), c.n, bpos, c.xq, box, c.colRank, c.cellStart, c.ncell, c.rlist * c.rlist, c.exclIdx, c.exclOff ? c.maxExcl : 0, c.type[c.cur], need, c.cap, c.nl, c.nlCount, c.nlCountA, c.dFlags, c.waveMax);
    else
        launch<build_body<T, false>, 256>(c, blocks, 0, rebuild_gate(c), c.n, bpos, c.xq, box, c.colRank, c.cellStart, c.ncell, c.rlist * c.rlist, c.exclIdx, c.exclOff ? c.maxExcl : 0, c.type[c.cur], need, c.cap, c.nl, c.nlCount, c.nlCountA, c.dFlags, c.waveMax);
    c.waveMaxA = blocks * (threads / 64);
}

template <int T>
void launch_e3b_list(Ctx &c, const double4 *bpos, const BoxDev *box) {
    int threads = 256;
    int blocks = cdiv((long long)c.e3b.nmol * T, threads);
    double rc = (double)c.e3b.r2b + c.skin;
    launch<e3b_list_body<T>, 256>(c, blocks, 0, rebuild_gate(c), c.e3b.nmol, c.e3b.molAtoms, c.e3b.atomMolO, bpos, box, rc * rc, c.cap, c.nl, c.nlCount, c.nlCountA, c.e3b.oxUncharged ? 1 : 0, c.e3b.cap, c.e3b.nl, c.e3b.nlCount, c.waveMax + wave_slots_a(c));
    c.waveMaxB = blocks * (threads / 64);
}

}  // namespace

void nlist_setup(Ctx &c, const int *cells) {
    MDX_REQUIRE(c.n > 0, 3, "system not set");
    MDX_REQUIRE(c.rlist > 0, 1, "neighbor list cutoff must be positive");
    for (int a = 0; a < 3; ++a) {
        if (c.geo.periodic[a])
            MDX_REQUIRE(c.rlist < 0.5 * c.geo.L[a], 1,
                        "neighbor cutoff (rCut + padding) must be below half the box length");
        double edge = c.rlist / c.reach[a] * (1.0 + 1e-9);
        int nca = (int)std::floor(c.geo.L[a] * grid_headroom(c) / edge);
        c.nc[a] = cells ? cells[a] : std::max(1, nca);
    }
    const int ncol = c.nc[0] * c.nc[1], ncell = ncol * c.nc[2];
    if (ncell != c.ncell || ncol != c.ncol) {  // a box turned on its side keeps its cells, not its columns
        MDX_REQUIRE(!c.capture, 3, "the cell grid cannot change while a step is captured");
        if (c.ncell) {
            dfree(c, c.colXY);
            dfree(c, c.colRank);
            dfree(c, c.cellHead);
            dfree(c, c.cellStart);
        }
        c.ncell = ncell;
        c.ncol = ncol;
        c.colRank = dalloc<int>(c, ncol);
        c.colXY = dalloc<int2>(c, ncol);
        // two copies of the grid: charged atoms, then charge-free ones
        c.cellHead = dalloc<int>(c, 2 * (size_t)ncell);
        // the sort leaves the lists empty for the next binning
        MDX_HIP(hipMemsetAsync(c.cellHead, 0xFF, sizeof(int) * 2 * (size_t)ncell, c.stream));
        c.cellStart = dalloc<int>(c, 2 * (size_t)ncell + 1);
    }
    // chunks of cells for the sort: at least 512 workgroups while a workgroup
    // still has 32 cells (an 8,192-molecule box has 7,200 slots: 225 workgroups
    // of 32), then up to 256 cells at a time, then several rounds of 256
    // (about 2,048 workgroups: each sums the chunk counts before its own)
    const int nslot = 2 * ncell;
    c.sortCpw = 32;
    while (c.sortCpw < kSortThreads && cdiv(nslot, c.sortCpw) > 512) c.sortCpw *= 2;
    int chunk = c.sortCpw;
    while (cdiv(nslot, chunk) > 2048) chunk *= 2;
    c.sortCsh = 0;
    while ((1 << c.sortCsh) < chunk) ++c.sortCsh;
    c.nChunk = cdiv(nslot, chunk);
    // column ranks along a 2-D Morton curve
    std::vector<std::pair<uint32_t, int>> keys;
    for (int x = 0; x < c.nc[0]; ++x)
        for (int y = 0; y < c.nc[1]; ++y) keys.push_back({morton2(x, y), x * c.nc[1] + y});
    std::sort(keys.begin(), keys.end());
    std::vector<int> rank(keys.size());
    std::vector<int2> xy(keys.size());
    for (size_t r = 0; r < keys.size(); ++r) {
        rank[keys[r].second] = (int)r;
        xy[r] = make_int2(keys[r].second / c.nc[1], keys[r].second % c.nc[1]);
    }
    MDX_HIP(hipMemcpyAsync(c.colRank, rank.data(), sizeof(int) * rank.size(), hipMemcpyHostToDevice,
                           c.stream));
    MDX_HIP(hipMemcpyAsync(c.colXY, xy.data(), sizeof(int2) * xy.size(), hipMemcpyHostToDevice,
                           c.stream));
    MDX_HIP(hipStreamSynchronize(c.stream));
    if (!c.cellNext) {
        c.cellNext = dalloc<int>(c, c.n);
        c.chunkSum = dalloc<int>(c, 2048);
        MDX_HIP(hipMemsetAsync(c.chunkSum, 0, sizeof(int) * 2048, c.stream));
    }
    // one wave per atom (build_wave_body) measured fastest for dense water and
    // LJ alike; mdx_tune revisits the width
    if (!c.buildTeamUser) c.buildTeam = 64;
    const double dens = c.n / (c.geo.L[0] * c.geo.L[1] * c.geo.L[2]);
    if (c.cap == 0) {
        double expect = dens * 4.18879020479 * c.rlist * c.rlist * c.rlist;
        c.cap = ((int)(expect * 1.3) + 32 + 15) & ~15;
        c.nl = dalloc<uint32_t>(c, (size_t)c.n * c.cap);
        c.nlCount = dalloc<int>(c, c.n);
        c.nlCountA = dalloc<int>(c, c.n);
    }
    c.nlistConfigured = true;
    c.listValid = false;  // the cells of a list built on another grid are gone
    ++c.layoutEpoch;  // cell counts and tables are kernel arguments of captured steps
    box_upload(c);  // cell counts changed
}

void refresh_xq(Ctx &c) {
    int threads = 256;
    launch<xq_body, 256>(c, cdiv(c.n, threads), 0, c.n, c.pos[c.cur], c.q[c.cur], c.xq, c.box);
}

// the pending row maxima of a captured build for the launch that takes them
RowMaxArgs row_max_args(Ctx &c) {
    RowMaxArgs rm{};
    if (c.rowMaxPending) {
        rm.on = 1;
        rm.gate = rebuild_gate(c);
        rm.na = c.waveMaxA;
        rm.a = c.waveMax;
        rm.nb = c.waveMaxB;
        rm.b = c.waveMax + wave_slots_a(c);
        rm.flags = c.dFlags;
        c.rowMaxPending = false;
    }
    return rm;
}

void row_max_flush(Ctx &c) {
    const RowMaxArgs rm = row_max_args(c);
    if (rm.on) launch<row_max_body, 1024>(c, 1, 0, rm.gate, rm.na, rm.a, rm.nb, rm.b, rm.flags, nullptr);
}

void prepare_forces(Ctx &c) {
    const int threads = 256;
    const RowMaxArgs rm = row_max_args(c);
    launch<xq_zero_body, 256>(c, cdiv(std::max(c.n, kAccTotal), threads) + rm.on, 0, c.n, c.pos[c.cur], c.q[c.cur], c.xq, c.box, c.force, kAccTotal, c.acc,
                              c.pppm.on && c.hasCharges ? c.meshRec : nullptr, rm);
}

void nlist_check(Ctx &c) {
    int threads = 256;
    double thr = 0.5 * c.skin;
    launch<check_body, 256>(c, cdiv(c.n, threads), 0, c.n, c.pos[c.cur], c.posLast, c.box, thr * thr, c.dFlags);
}

// The rows from the sorted atoms at bpos (FP32 copies in xq), and the E3B
// list; grows them and builds again where they overflowed (sync), else leaves
// the check to the next synchronisation point.
static void build_rows(Ctx &c, const double4 *bpos, const BoxDev *box, const MolMapArgs &mm, bool sync, bool wave,
                       unsigned long long need) {
    for (;;) {
        // the builds of a run keep the running maximum of the chunk in dFlags[1..2]
        if (!c.capture && sync) fill_int(c, c.dFlags + 1, 2, 0);
        c.waveMaxB = 0;
        {
            ProfScope ps(c, PK_BUILD);
            if (wave) launch_build_wave(c, bpos, box, mm, need);
            else if (c.buildTeam == 8) launch_build<8>(c, bpos, box, need);
            else if (c.buildTeam == 32) launch_build<32>(c, bpos, box, need);
            else launch_build<16>(c, bpos, box, need);
        }
        if (c.e3b.on && !wave) {  // the wave build makes this list itself
            switch (c.e3b.listTeam) {
                case 8: launch_e3b_list<8>(c, bpos, box); break;
                case 16: launch_e3b_list<16>(c, bpos, box); break;
                default: launch_e3b_list<32>(c, bpos, box); break;
            }
        }
        if (c.capture && c.fuseStep) {
            // the row maxima ride on the position refresh that follows; the
            // host checks the rows after the chunk
            c.rowMaxPending = true;
            return;
        }
        // largest row counts -> pinned host memory; checked now (sync) or at
        // the next synchronisation point (capacity_ok)
        launch<row_max_body, 1024>(c, 1, 0, rebuild_gate(c), c.waveMaxA, c.waveMax, c.waveMaxB, c.waveMax + wave_slots_a(c), c.dFlags, c.capture ? nullptr : c.pinned);
        if (c.capture) return;  // rows checked by the host after the chunk
        if (!sync) {
            MDX_HIP(hipEventRecord(c.capEvent, c.stream));
            c.capPending = true;
            return;
        }
        MDX_HIP(hipStreamSynchronize(c.stream));
        if (!grow_if_needed(c)) return;
    }
}

// The parts of the rows that the set-up's kernels read, as row_parts' mask;
// all of them for a ring's centroid lists, whose build positions do not
// outlive the ring call, and once a program has read the list back (it may do
// so after every step, and each time pay for a completing build).
unsigned long long list_need(Ctx &c) {
    if (c.cenById || c.wholeList) return ~0ull;
    if (c.needDirty) {
        const std::vector<int> fl = pair_type_flag_table(c);
        const bool coul = c.ewaldReal && c.hasCharges;
        unsigned long long need = 0;
        for (int t = 0; t < kMaxTypes; ++t) {
            const unsigned long long lj = (unsigned long long)(c.ljOn ? fl[t] & 3 : 0);
            need |= (lj | (coul ? 1ull : 0ull)) << (4 * t) | lj << (4 * t + 2);
        }
        // the E3B list reads an oxygen's whole row, or the charge-free part of
        // charge-free oxygens
        if (c.e3b.on)
            for (int o : c.e3b.oxIds)
                need |= (c.e3b.oxUncharged ? 2ull : 3ull) << (4 * c.typeHost[o] + (c.qHost[o] != 0.0f ? 0 : 2));
        c.needMask = need;
        c.needDirty = false;
    }
    return c.needMask;
}

// The whole rows of the current list: built again from the positions and the
// box of its build, in the order that build left.
void nlist_complete(Ctx &c) {
    if (!c.listValid || c.listNeed == ~0ull) return;
    MDX_REQUIRE(!c.capture, 3, "the list cannot be completed while a step is captured");
    capacity_ok(c);
    launch<xq_body, 256>(c, cdiv(c.n, 256), 0, c.n, c.posLast, c.q[c.cur], c.xq, c.boxLast);
    c.listNeed = ~0ull;
    // the exclusion rows are as that build's kernel reads them
    build_rows(c, c.posLast, c.boxLast, MolMapArgs{}, true, !c.exclByIdx, ~0ull);
    refresh_xq(c);
}

void list_setup_changed(Ctx &c) {
    c.needDirty = true;
    if (c.listValid && !c.centroidList && (list_need(c) & ~c.listNeed)) nlist_complete(c);
}

static bool wave_build(const Ctx &c) { return c.buildTeam != 8 && c.buildTeam != 16 && c.buildTeam != 32; }

// What a build of the current set-up leaves.  A captured build leaves it only
// when it runs (run_captured asks the device after the chunk).
void list_built(Ctx &c) {
    c.listNeed = list_need(c);
    c.exclByIdx = !wave_build(c);
    c.centroidList = c.cenById != nullptr;
}

static void run_build(Ctx &c, bool sync) {
    // per-wave row maxima: n + 4 slots cover the build at up to 64 lanes per
    // atom (workgroups of 4 waves), the rest the molecule list likewise
    const size_t needSlots = wave_slots_a(c) + (size_t)(c.e3b.on ? c.e3b.nmol : 0) + 4;
    if ((size_t)c.waveMaxN < needSlots) {
        MDX_REQUIRE(!c.capture, 3, "row-maximum slots must exist before a step is captured");
        if (c.waveMax) dfree(c, c.waveMax);
        c.waveMax = dalloc<int>(c, needSlots);
        c.waveMaxN = (int)needSlots;
    }
    if (c.e3b.on && !c.e3b.nl) {
        // molecule rows for the mean density with the pair rows' margin: water
        // has 52 entries in 7.2 A, and rows of 64 overflowed now and then in
        // boxes of a few hundred molecules (each overflow replays a chunk)
        MDX_REQUIRE(!c.capture, 3, "molecule rows must exist before a step is captured");
        const double r = (double)c.e3b.r2b + c.skin;
        const double expect = c.e3b.nmol / (c.geo.L[0] * c.geo.L[1] * c.geo.L[2]) * 4.18879020479 * r * r * r;
        c.e3b.cap = ((int)(expect * 1.3) + 32 + 15) & ~15;
        c.e3b.nl = dalloc<int>(c, (size_t)c.e3b.nmol * c.e3b.cap);
    }
    const int threads = 256;
    const int cur = c.cur, scr = 1 - c.cur;  // the records are sorted in place; scr: scratch copies
    const int nslot = 2 * c.ncell;
    const double4 *cen = c.cenById;
    MDX_REQUIRE(!cen || (c.buildPos && !c.e3b.on), 3,
                "a centroid list needs its build positions and takes no E3B molecule list");
    MDX_REQUIRE(!c.e3b.on || c.rlist >= (double)c.e3b.r2b + c.skin - 1e-9, 1,
                "E3B needs rCut + padding >= 6.2 A + padding (the molecule list is taken from the "
                "pair list)");
    MDX_REQUIRE(std::min(c.nc[0], 2 * c.reach[0] + 1) * std::min(c.nc[1], 2 * c.reach[1] + 1) <= kMaxCols, 1,
                "stencil wider than the build kernel's column table");
    const bool waveBuild = wave_build(c);
    const bool excl = c.exclOff && c.maxExcl > 0;
    if (excl) {
        MDX_REQUIRE(!c.capture || c.exclIdxN == (size_t)c.n * c.maxExcl, 3,
                    "exclusion index rows must exist before a step is captured");
        if (c.exclIdxN != (size_t)c.n * c.maxExcl) {
            if (c.exclIdx) dfree(c, c.exclIdx);
            c.exclIdxN = (size_t)c.n * c.maxExcl;
            c.exclIdx = dalloc<uint32_t>(c, c.exclIdxN);
        }
    }
    const unsigned long long need = list_need(c);
    // The map workgroups of a build clear the chunk counts for the next
    // binning, so every refusal stands above it: counts left over would send
    // the next sort out of range.
    DecideArgs da{};
    if (c.capture && c.fuseCheck) {
        da = decide_args(c);
        da.slots = c.dispSlots;
    }
    launch<bin_body, 256>(c, cdiv(c.n, threads), 0, rebuild_gate(c), c.n, c.pos[cur], c.vel[cur], c.q[cur], c.type[cur], c.id[cur], c.pos[scr], c.vel[scr], c.q[scr], c.type[scr], c.id[scr], c.box, c.ncell, c.colRank, c.cellHead, c.cellNext, c.chunkSum, c.sortCsh, cen, da);
    SortArgs sa{};
    sa.n = c.n;
    sa.nslot = nslot;
    sa.cpw = c.sortCpw;
    sa.csh = c.sortCsh;
    sa.head = c.cellHead;
    sa.next = c.cellNext;
    sa.chunkSum = c.chunkSum;
    sa.start = c.cellStart;
    sa.pos0 = c.pos[scr];
    sa.vel0 = c.vel[scr];
    sa.q0 = c.q[scr];
    sa.type0 = c.type[scr];
    sa.id0 = c.id[scr];
    sa.pos1 = c.pos[cur];
    sa.vel1 = c.vel[cur];
    sa.q1 = c.q[cur];
    sa.type1 = c.type[cur];
    sa.id1 = c.id[cur];
    sa.idToIdx = c.idToIdx;
    sa.last = c.posLast;
    sa.xq = c.xq;
    sa.rec = c.refreshed && c.pppm.on && c.hasCharges ? c.meshRec : nullptr;
    sa.cen = cen;
    sa.bpos = c.buildPos;
    sa.atomMolO = c.e3b.on ? c.e3b.atomMolO : nullptr;
    sa.member = c.rigid.on ? c.rigid.member : nullptr;
    sa.maxExcl = excl ? c.maxExcl : 0;
    sa.exclOff = c.exclOff;
    sa.exclIds = c.exclIds;
    sa.exclRow = c.exclIdx;
    sa.slots = da.slots;
    sa.bx = c.box;
    sa.boxLast = c.boxLast;
    launch<sort_body, kSortThreads>(c, c.nChunk, 0, rebuild_gate(c), sa);
    // The P3M chain needs the sorted sites, their mesh records (written by the
    // sort, the first half kick having refreshed them) and the cells, not the
    // list: its stream forks here, so the list build below runs beside it.
    if (c.capture && c.refreshed && c.side && c.meshStream && !c.rec && c.pppm.on) {
        MDX_HIP(hipEventRecord(c.evFork, c.stream));
        c.forked = true;
    }
    if (excl && !waveBuild)
        launch<excl_idx_body, 256>(c, cdiv((long long)c.n * c.maxExcl, threads), 0, rebuild_gate(c), (long long)c.n * c.maxExcl, c.idToIdx, c.exclIdx);
    MolMapArgs mm{};
    mm.idToIdx = c.idToIdx;
    if (c.e3b.on) {
        mm.nmol = c.e3b.nmol;
        mm.molIds = c.e3b.molIds;
        mm.molAtoms = c.e3b.molAtoms;
        mm.atomMolO = c.e3b.atomMolO;
    }
    if (c.rigid.on) {
        mm.nmolR = c.rigid.nmol;
        mm.rigidIds = c.rigid.ids;
        mm.rigidAtoms = c.rigid.atoms;
        mm.member = c.rigid.member;
    }
    if (c.flex.on) {
        mm.nmolF = c.flex.nmol;
        mm.flexIds = c.flex.ids;
        mm.flexAtoms = c.flex.atoms;
    }
    mm.nchunk = c.nChunk;
    mm.chunkSum = c.chunkSum;
    mm.blocks = cdiv(std::max({mm.nmol, mm.nmolR, mm.nmolF, mm.nchunk}), threads);
    // the wave build takes the maps as extra workgroups; the team builds launch them first
    if (!waveBuild) launch<mol_map_body, 256>(c, mm.blocks, 0, rebuild_gate(c), mm);
    build_rows(c, cen ? c.buildPos : c.pos[cur], c.box, mm, sync, waveBuild, need);
    if (c.capture) return;
    list_built(c);
    c.nRebuilds++;
    c.listValid = true;
}

void flag7_check(int v) {
    MDX_REQUIRE(!(v & 1), 1, "an atom's stencil holds over 2^20 candidates: lower the list cutoff or the cell reach");
    MDX_REQUIRE(!(v & 2), 4,
                "a charged site's P3M stencil left the cells next to its own (a site moved beyond skin/2 "
                "between list builds)");
}

// Grows the pair / molecule rows after an overflow seen in pinned[0..1];
// returns true when something grew (the caller rebuilds).  The reference
// reallocates its list at 1.5x (GridGPU.cu:1026-1030).
bool grow_if_needed(Ctx &c) {
    flag7_check(c.pinned[6]);
    bool grew = false;
    if (c.pinned[0] > c.cap) {
        dfree(c, c.nl);
        c.cap = ((int)(c.pinned[0] * 1.25) + 15) & ~15;
        c.nl = dalloc<uint32_t>(c, (size_t)c.n * c.cap);
        grew = true;
    }
    if (c.e3b.on && c.pinned[1] > c.e3b.cap) {
        dfree(c, c.e3b.nl);
        c.e3b.cap = ((int)(c.pinned[1] * 1.25) + 15) & ~15;
        c.e3b.nl = dalloc<int>(c, (size_t)c.e3b.nmol * c.e3b.cap);
        grew = true;
    }
    return grew;
}

// True when every build since the last call fitted its rows.  Waits for the
// last asynchronous build only.
bool capacity_ok(Ctx &c) {
    if (!c.capPending) return true;
    MDX_HIP(hipEventSynchronize(c.capEvent));
    c.capPending = false;
    return !grow_if_needed(c);
}

void nlist_rebuild(Ctx &c, bool forced) {
    if (!c.nlistConfigured) nlist_setup(c);
    if (!forced) {
        int flag = 0;
        MDX_HIP(hipMemcpyAsync(&flag, c.dFlags, sizeof(int), hipMemcpyDeviceToHost, c.stream));
        MDX_HIP(hipStreamSynchronize(c.stream));
        if (!flag && c.listValid) return;
    }
    run_build(c, true);
    fill_int(c, c.dFlags, 1, 0);
}

void nlist_rebuild_async(Ctx &c) {
    if (!c.nlistConfigured) nlist_setup(c);
    run_build(c, !c.listValid);
}

void fill_int(Ctx &c, int *p, int count, int v, const int *gate) {
    launch<fill_int_body, 256>(c, cdiv(count, 256), 0, gate, count, p, v);
}

namespace {
// Lag-1 rebuild decision for the step loop: per site d = |x - x_last| and the
// prediction p = d + 2 dt |v| (an M site, moved by its molecule, never moves
// further than its fastest heavy site); max d^2 and max p^2 over all sites go
// to one of two pinned host slots.  The host reads the slot one step later.
// Grid-stride over the sites with a workgroup reduction: one atomic pair per
// workgroup (same-address atomics serialise in L2).
// Per-workgroup maxima into part[2 b], part[2 b + 1] (float bits); a
// one-wave kernel reduces them (no same-address atomics).
__device__ __forceinline__ void check_part_body(int blk, int nblk, int n, const double4 *__restrict__ pos,
                                                    const double4 *__restrict__ last,
                                                    const double4 *__restrict__ vel, const BoxDev *__restrict__ bx,
                                                    double dt2, float *__restrict__ part) {
    const Geometry g = bx->geo;
    __shared__ float red[2][4];
    const int t0 = blk * blockDim.x + threadIdx.x;
    float d2 = 0.f, p2 = 0.f;
    for (int i = t0; i < n; i += nblk * blockDim.x) {
        const double dd = dist2(pos[i], last[i], g);
        const double4 v = vel[i];
        const double p = sqrt(dd) + dt2 * sqrt(v.x * v.x + v.y * v.y + v.z * v.z);
        d2 = fmaxf(d2, (float)dd);
        p2 = fmaxf(p2, (float)(p * p));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        d2 = fmaxf(d2, __shfl_xor(d2, o, 64));
        p2 = fmaxf(p2, __shfl_xor(p2, o, 64));
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        red[0][w] = d2;
        red[1][w] = p2;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < (int)(blockDim.x >> 6); ++k) {
            d2 = fmaxf(d2, red[0][k]);
            p2 = fmaxf(p2, red[1][k]);
        }
        part[2 * blk] = d2;
        part[2 * blk + 1] = p2;
    }
}

// One wave: a check's maxima straight into the host's pinned words (a store
// of the kernel; a device-to-host copy is a launch of its own and left 5 us
// between this and the next kernel), from the per-workgroup maxima or from the
// words of a fused first half, which it clears.
__device__ __forceinline__ void check_reduce_body(int blk, int nblk, int nb, const float *__restrict__ part,
                                                  unsigned *__restrict__ slots, int *__restrict__ host) {
    float d2, p2;
    if (slots) {
        d2 = disp_max(slots, 0);
        p2 = disp_max(slots, 1);
        if (threadIdx.x < kDispSlots) {
            slots[threadIdx.x * kDispStride] = 0u;
            slots[threadIdx.x * kDispStride + 1] = 0u;
        }
    } else {
        part_max(nb, part, d2, p2);
    }
    if (threadIdx.x == 0) {
        host_store(host, __float_as_int(d2));
        host_store(host + 1, __float_as_int(p2));
    }
}
}  // namespace

static int check_blocks(const Ctx &c) { return std::max(1, std::min(cdiv(c.n, 256), kCheckBlocks)); }

static void check_part(Ctx &c) {
    launch<check_part_body, 256>(c, check_blocks(c), 0, c.n, c.pos[c.cur], c.posLast, c.vel[c.cur], c.box, 2.0 * c.dt, c.checkPart);
}

DecideArgs decide_args(const Ctx &c) {
    DecideArgs d{};
    d.part = c.checkPart;
    d.flags = c.dFlags;
    const float half = (float)(0.5 * c.skin);
    d.half2 = half * half;
    d.every = c.thermoOn ? c.thermoEvery : 0;
    d.baroEvery = c.baro.on ? c.baro.every : 0;
    d.thermo = c.fuseThermo ? c.thermo : nullptr;
    return d;
}

void skin_check(Ctx &c) { check_part(c); }

void skin_decide(Ctx &c) {
    DecideArgs d = decide_args(c);
    if (c.ringPart) d.part = c.ringPart;
    launch<decide_body, 64>(c, 1, 0, c.ringPart ? c.ringPartNb : check_blocks(c), d);
}

void decide_step(Ctx &c) {
    if (c.fuseCheck) return;  // the binning decides from the first half's maxima
    check_part(c);
    skin_decide(c);
}

void check_max(Ctx &c, int parity) {
    check_part(c);
    launch<check_reduce_body, 64>(c, 1, 0, check_blocks(c), c.checkPart, nullptr, c.pinned + 2 + 2 * parity);
}

void check_out(Ctx &c, int parity) {
    launch<check_reduce_body, 64>(c, 1, 0, 0, nullptr, c.dispSlots, c.pinned + 2 + 2 * parity);
}

}  // namespace mdx
