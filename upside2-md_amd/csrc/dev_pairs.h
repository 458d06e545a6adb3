// Pair graphs on the device: Verlet cache from LDS-tiled scans, exact edge
// refine, per-edge spline energies and the fixed-order sensitivity gather.
//
// Reference: PairlistComputation / InteractionGraph (src/interaction_graph.h).
// The edge set of a graph is {(i1,i2) acceptable : dist2 < cutoff^2} where
// dist2 is computed from the current packed coordinates exactly as the
// reference build evaluates it, fma(x,x, fma(z,z, y*y)) (the Float4 sum of
// src/interaction_graph.h:239 contracted by the compiler).  The cache (radius
// cutoff + buffer, rebuilt when any element drifts more than buffer/2,
// src/interaction_graph.h:51-169) only bounds which pairs are examined, so the
// edge set does not depend on how the cache was built.
//
// Rebuild: the other side is put into a hashed cell grid in LDS (or streamed
// in tiles when it does not fit) and every row scans it once, keeping the
// partners in a slab; after a team scan of the counts they are copied to their
// slots (a row that outgrew its slab is scanned again).  Row order is canonical
// (fixed cell-visit order, index order inside a cell).  Transposed rows (the
// forward slots of each side-2 element) are placed by their arrival in the
// column and then ordered by slot, so every order is independent of scheduling.
#pragma once
#include "dev_common.h"

namespace upside {

__device__ __forceinline__ float refine_dist2(float dx, float dy, float dz) {
    return __fmaf_rn(dx, dx, __fmaf_rn(dz, dz, __fmul_rn(dy, dy)));
}

__device__ __forceinline__ bool pg_accept(GraphC& G, int a, int b) {
    if (G.excl < 0) return (a >> 4) != (b >> 4);
    int d = a - b;
    return d > G.excl || -d > G.excl;
}

__device__ __forceinline__ ap<const float> pg_side2(const Ctx& c, GraphC& G) {
    return c.A + G.pos_pack + (G.sym ? 0 : G.n1 * 3);
}

// Copy the current coordinates of both sides into pos_pack and report whether
// the cache must be rebuilt (first use, or drift beyond half the buffer).
__device__ __forceinline__ bool pg_pack_and_check(Ctx& c, GraphC& G) {
    gp<const int> loc1 = c.CI + G.loc1;
    gp<const int> loc2 = c.CI + G.loc2;
    ap<const float> P1 = c.A + G.out1;
    ap<const float> P2 = c.A + G.out2;
    ap<float> pack = c.A + G.pos_pack;
    ap<const float> cache = c.A + G.cache_pos;
    int n = G.sym ? G.n1 : G.n1 + G.n2;
    int valid = c.I[G.state];
    int moved = 0;
    for (int i = c.gtid; i < n; i += c.gsize) {
        ap<const float> src = (i < G.n1) ? P1 + loc1[i] * G.w1 : P2 + loc2[i - G.n1] * G.w2;
        float x = src[0], y = src[1], z = src[2], old[3];
        (cache + i * 3).get<3>(old);
        pack[i * 3 + 0] = x; pack[i * 3 + 1] = y; pack[i * 3 + 2] = z;
        float dx = x - old[0], dy = y - old[1], dz = z - old[2];
        if (!(dx * dx + dy * dy + dz * dz <= G.drift2)) moved = 1;  // NaN also forces a rebuild
    }
    int any = team_or(c, moved | (valid ? 0 : 1));
    return any != 0;
}

template <class P>
__device__ __forceinline__ int lower_bound_i(P a, int n, int v) {
    int lo = 0, hi = n;
    while (lo < hi) {
        int m = (lo + hi) >> 1;
        if (a[m] < v) lo = m + 1; else hi = m;
    }
    return lo;
}

// ---- cache rebuild -------------------------------------------------------------
// Rows are scanned by groups of SG lanes: the lanes of a group stride one
// query's candidates together and emit the hits in candidate order through a
// ballot, so a row costs ceil(candidates / SG) dependent steps instead of one
// step per candidate.
constexpr int SG = 8;

struct GroupLanes {
    int gl;                    // lane within the group
    unsigned long long gmask;  // the group's lanes in the wave
    unsigned long long below;  // wave lanes below this one
};
__device__ __forceinline__ GroupLanes group_lanes(const Ctx& c) {
    GroupLanes L;
    int lane = c.tid & 63;
    L.gl = lane & (SG - 1);
    L.gmask = ((1ull << SG) - 1ull) << (lane & ~(SG - 1));
    L.below = (1ull << lane) - 1ull;
    return L;
}

// Where a scan puts the hits of a row, in candidate order.  The count scan
// keeps the first `room` partners of row q in its slab, slab[q * room ...], so
// that the fill copies them (pg_fill) instead of scanning again.
struct SlabOut {
    ap<int> slab;
    int room;
    __device__ __forceinline__ void operator()(int q, int k, int j) const {
        if (k < room) slab[q * room + k] = j;
    }
};
// A forward row's slot: partner, row, and the slot's arrival number in its
// column (any order: the columns are sorted by slot afterwards).
struct SlotOut {
    ap<int> nbr, row, toff, arrival;
    int first;
    __device__ __forceinline__ void operator()(int q, int k, int j) const {
        const int p = first + k;
        const int r = atomicAdd((int*)(toff + j).ptr(), 1);
        nbr[p] = j;
        row[p] = q;
        arrival[p] = r;
    }
};

// One SG-wide step of a row: returns the group's hits; out receives each hit
// as number cur + (hits of the lower lanes) of row q, so hits keep candidate
// order.  Every lane of the group calls it.
template <class O>
__device__ __forceinline__ int group_emit(const GroupLanes& L, bool hit, int cur, int q, int j, const O& out) {
    unsigned long long m = __ballot(hit) & L.gmask;
    if (hit) out(q, cur + __popcll(m & L.below), j);
    return __popcll(m);
}

// Fallback scan for sides too large for the LDS grid: the other side streamed
// through LDS in tiles of TILE elements, partners in increasing index.
constexpr int TILE = LDS_FLOATS / 4;

// Elements staged in LDS are 4 floats: position and an integer tag stored as
// float bits (the four stores/loads combine into 16-byte LDS accesses).
__device__ __forceinline__ void el_put(lp<float> el, int k, float x, float y, float z, int tag) {
    el[4 * k] = x; el[4 * k + 1] = y; el[4 * k + 2] = z; el[4 * k + 3] = __int_as_float(tag);
}

// Stage elements [t0, t0+n) of side pts (ids in id) as (x, y, z, id).
__device__ __forceinline__ void stage_tile(Ctx& c, ap<const float> pts, gp<const int> id, int t0, int n) {
    lp<float> tile = c.lds;
    for (int k = c.tid; k < n; k += NT) {  // every workgroup stages its own copy
        int j = t0 + k;
        el_put(tile, k, pts[j * 3], pts[j * 3 + 1], pts[j * 3 + 2], id[j]);
    }
    __syncthreads();
}

// Elements of the other side: staged in LDS, or (tiles that are gone) in memory.
struct TileEl {
    lp<const float> el;
    __device__ __forceinline__ void get(int k, float* x, int& id) const {
        x[0] = el[4 * k]; x[1] = el[4 * k + 1]; x[2] = el[4 * k + 2];
        id = __float_as_int(el[4 * k + 3]);
    }
};
struct MemEl {
    ap<const float> pts;
    gp<const int> ids;
    __device__ __forceinline__ void get(int k, float* x, int& id) const {
        (pts + k * 3).template get<3>(x);
        id = ids[k];
    }
};

// Row q (position x, id a) against elements [0, n) of el, whose first is
// element t0: a pair (q, j) is a hit when within the cache radius and
// acceptable (SYM: also j > q).  cnt: the row's hits so far; returns it advanced.
template <bool SYM, class EL, class O>
__device__ __forceinline__ int list_row(GraphC& G, const GroupLanes& L, int q, const float* x, int a, const EL& el,
                                        int t0, int n, int cnt, const O& out) {
    const float cc2 = G.cache_cut2;
    for (int k0 = 0; k0 < n; k0 += SG) {
        const int k = k0 + L.gl, j = t0 + k;
        bool hit = false;
        if (k < n) {
            float e[3];
            int id;
            el.get(k, e, id);
            const float d2 = refine_dist2(x[0] - e[0], x[1] - e[1], x[2] - e[2]);
            hit = d2 < cc2 && (!SYM || j > q) && pg_accept(G, a, id);
        }
        cnt += group_emit(L, hit, cnt, q, j, out);
    }
    return cnt;
}

// Count scan of rows q in [0, nq) (positions qp, ids qid) against the elements
// ep[0..ne) (ids eid): off[q] = hits of row q.  One tile stays in LDS for the fill.
template <bool SYM>
__device__ __forceinline__ void tile_rows(Ctx& c, GraphC& G, ap<const float> qp, gp<const int> qid, int nq,
                          ap<const float> ep, gp<const int> eid, int ne, ap<int> off, const SlabOut& out) {
    const GroupLanes L = group_lanes(c);
    const int grp = c.gtid / SG, ngrp = c.gsize / SG;
    for (int t0 = 0; t0 < ne; t0 += TILE) {
        int tn = min(TILE, ne - t0);
        if (t0) __syncthreads();  // the tile is restaged; counts visible to the group
        stage_tile(c, ep, eid, t0, tn);
        for (int q = grp; q < nq; q += ngrp) {
            float x[3];
            (qp + q * 3).get<3>(x);
            int cnt = t0 ? (int)off[q] : 0;
            cnt = list_row<SYM>(G, L, q, x, qid[q], TileEl{(lp<const float>)c.lds}, t0, tn, cnt, out);
            if (L.gl == 0) off[q] = cnt;
        }
    }
    team_sync(c);
}

// ---- cache rebuild: cell grid in LDS ----------------------------------------
// The other side is counting-sorted into hashed cells of edge >= the cache
// radius, kept in LDS as (bucket offsets, elements (x, y, z, index),
// element ids), each bucket sorted by element index.  A row visits its 27
// neighbouring cells in a fixed order, so rows come out in a canonical order.
struct LGrid {
    float ox, oy, oz, inv;
    int mask;
    lp<int> ofs;      // [mask+2]
    lp<float> el;     // [4m] (x, y, z, element index)
    lp<int> eid;      // [m]  element ids, same order (no global loads in the scan)
};

__device__ __forceinline__ int cell_coord(float x, float o, float inv) {
    // clamp keeps far outliers (and NaN) inside int range; they only cost scan time
    float t = fminf(fmaxf((x - o) * inv, -1.0e6f), 1.0e6f);
    return (int)floorf(t);
}
__device__ __forceinline__ int cell_bucket(int mask, int cx, int cy, int cz) {
    uint32_t h = ((uint32_t)cx * 73856093u) ^ ((uint32_t)cy * 19349663u) ^ ((uint32_t)cz * 83492791u);
    return (int)(h & (uint32_t)mask);
}

// Points that a grid holds: with 4096 buckets up to 7167, with 2048 the rest
// (the rows are the same).
constexpr int GRID_POINTS = 7320;
static_assert((2048 + 4) * 4 + GRID_POINTS * 20 <= LDS_FLOATS * 4, "a grid in LDS");
__device__ __forceinline__ int lgrid_buckets(int m) {
    int nb = 64;
    while (nb < m && nb < 4096) nb *= 2;
    return (nb + 4) * 4 + m * 20 <= LDS_FLOATS * 4 ? nb : nb / 2;
}
__device__ __forceinline__ bool lgrid_fits(int m) { return m <= GRID_POINTS; }

// Build the grid of the m points pts (stride 3) in this workgroup's LDS
// (every workgroup of a team builds its own copy).  All threads of the workgroup.
// Every thread keeps its points, read once, in registers.  A bucket is put in
// order by counting, for each of its elements, those with a smaller index: a
// cell holds some 25 beads, and one thread sorting it by insertion was most of
// the build.
constexpr int GRID_U = (GRID_POINTS + NT - 1) / NT;
__device__ __forceinline__ LGrid lgrid_build(Ctx& c, GraphC& G, ap<const float> pts, gp<const int> ids, int m) {
    float x[GRID_U][3];
    int id[GRID_U], at[GRID_U];
    float mn0 = 3.0e38f, mn1 = 3.0e38f, mn2 = 3.0e38f;
#pragma unroll
    for (int u = 0; u < GRID_U; ++u) {
        const int i = u * NT + c.tid;
        if (i < m) {
            (pts + i * 3).get<3>(x[u]);
            id[u] = ids[i];
        }
    }
#pragma unroll
    for (int u = 0; u < GRID_U; ++u)
        if (u * NT + c.tid < m) {
            mn0 = fminf(mn0, x[u][0]);
            mn1 = fminf(mn1, x[u][1]);
            mn2 = fminf(mn2, x[u][2]);
        }
    LGrid g;
    g.ox = -block_max(c, -mn0);
    g.oy = -block_max(c, -mn1);
    g.oz = -block_max(c, -mn2);
    // cells slightly larger than the cache radius: rounding can never put two
    // points closer than the radius more than one cell apart
    g.inv = 1.f / (G.cache_cut * 1.0001f);
    int nb = lgrid_buckets(m);
    g.mask = nb - 1;
    lp<float> L = c.lds;
    g.ofs = (lp<int>)L;
    g.el = L + ((nb + 4) & ~3);
    g.eid = (lp<int>)(g.el + 4 * m);
    for (int b = c.tid; b <= nb; b += NT) g.ofs[b] = 0;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < GRID_U; ++u)
        if (u * NT + c.tid < m) {
            at[u] = cell_bucket(g.mask, cell_coord(x[u][0], g.ox, g.inv), cell_coord(x[u][1], g.oy, g.inv),
                                cell_coord(x[u][2], g.oz, g.inv));
            atomicAdd((int*)(g.ofs + at[u] + 1), 1);
        }
    __syncthreads();
    block_exscan(c, g.ofs + 1, nb);  // ofs[b+1] = start of bucket b
#pragma unroll
    for (int u = 0; u < GRID_U; ++u)
        if (u * NT + c.tid < m)  // ofs[b+1] ends at the start of bucket b+1
            g.eid[atomicAdd((int*)(g.ofs + at[u] + 1), 1)] = u * NT + c.tid;
    __syncthreads();
    // canonical order inside every bucket: by element index
#pragma unroll
    for (int u = 0; u < GRID_U; ++u) {
        const int i = u * NT + c.tid;
        if (i < m) {
            const int lo = g.ofs[at[u]], hi = g.ofs[at[u] + 1];
            int r = lo;
            for (int k = lo; k < hi; ++k) r += g.eid[k] < i;
            at[u] = r;
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < GRID_U; ++u) {
        const int i = u * NT + c.tid;
        if (i < m) {
            el_put(g.el, at[u], x[u][0], x[u][1], x[u][2], i);
            g.eid[at[u]] = id[u];
        }
    }
    __syncthreads();
    return g;
}

// Row q against the grid; same hit rule as list_row.  Returns its hits.
constexpr int GRID_STEP = 2;  // SG elements each, loaded together
template <bool SYM, class O>
__device__ __forceinline__ int grid_row(GraphC& G, const GroupLanes& L, const LGrid& g, int q, const float* x, int a,
                                        const O& out) {
    const float cc2 = G.cache_cut2;
    int cnt = 0;
    const int cx = cell_coord(x[0], g.ox, g.inv), cy = cell_coord(x[1], g.oy, g.inv), cz = cell_coord(x[2], g.oz, g.inv);
    int ax = cx - 1, ay = cy - 1, az = cz - 1;
    int b = cell_bucket(g.mask, ax, ay, az);
    int t = g.ofs[b], t1 = g.ofs[b + 1];
    for (int cell = 0; cell < 27; ++cell) {
        // the next cell's elements are known before this cell's are tested
        int nx = ax + 1, ny = ay, nz = az;
        if (nx > cx + 1) {
            nx = cx - 1;
            if (++ny > cy + 1) { ny = cy - 1; ++nz; }
        }
        b = cell_bucket(g.mask, nx, ny, nz);
        const int s0 = g.ofs[b], s1 = g.ofs[b + 1];
        for (; t < t1; t += GRID_STEP * SG) {
            float e[GRID_STEP][4];
            int id[GRID_STEP];
#pragma unroll
            for (int h = 0; h < GRID_STEP; ++h) {
                const int k = min(t + h * SG + L.gl, t1 - 1);
#pragma unroll
                for (int d = 0; d < 4; ++d) e[h][d] = g.el[4 * k + d];
                id[h] = g.eid[k];
            }
#pragma unroll
            for (int h = 0; h < GRID_STEP; ++h) {
                const int j = __float_as_int(e[h][3]);
                const float d2 = refine_dist2(x[0] - e[h][0], x[1] - e[h][1], x[2] - e[h][2]);
                // the cell test drops elements of other cells sharing the bucket
                const bool hit = t + h * SG + L.gl < t1 && d2 < cc2 && (!SYM || j > q) &&
                                 cell_coord(e[h][0], g.ox, g.inv) == ax && cell_coord(e[h][1], g.oy, g.inv) == ay &&
                                 cell_coord(e[h][2], g.oz, g.inv) == az && pg_accept(G, a, id[h]);
                cnt += group_emit(L, hit, cnt, q, j, out);
            }
        }
        ax = nx; ay = ny; az = nz;
        t = s0; t1 = s1;
    }
    return cnt;
}

// Count scan against the grid: off[q] = hits of row q.
template <bool SYM>
__device__ __forceinline__ void grid_rows(Ctx& c, GraphC& G, const LGrid& g, ap<const float> qp, gp<const int> qid, int nq,
                          ap<int> off, const SlabOut& out) {
    const GroupLanes L = group_lanes(c);
    const int grp = c.gtid / SG, ngrp = c.gsize / SG;
    for (int q = grp; q < nq; q += ngrp) {
        float x[3];
        (qp + q * 3).get<3>(x);
        const int cnt = grid_row<SYM>(G, L, g, q, x, qid[q], out);
        if (L.gl == 0) off[q] = cnt;
    }
    team_sync(c);
}

// Fill the rows at off from their slabs, and count their columns in toff.
// Rows longer than their slab are scanned again: against the grid (use_grid),
// the tile that is still in LDS, or, where the other side takes several tiles,
// the elements in memory.
template <bool SYM>
__device__ __forceinline__ void pg_fill(Ctx& c, GraphC& G, const LGrid& g, bool use_grid, ap<const float> qp,
                          gp<const int> qid, int nq, ap<const float> ep, gp<const int> eid, int ne, ap<const int> off,
                          const SlabOut& slab, SlotOut out) {
    const GroupLanes L = group_lanes(c);
    const int grp = c.gtid / SG, ngrp = c.gsize / SG;
    constexpr int U = 4;
    for (int q = grp; q < nq; q += ngrp) {
        const int b = off[q], n = off[q + 1] - b;
        out.first = b;
        if (n <= slab.room) {
            for (int k0 = L.gl; k0 < n; k0 += U * SG) {
                int j[U], r[U];
#pragma unroll
                for (int u = 0; u < U; ++u) j[u] = k0 + u * SG < n ? (int)slab.slab[q * slab.room + k0 + u * SG] : 0;
#pragma unroll
                for (int u = 0; u < U; ++u)
                    r[u] = k0 + u * SG < n ? atomicAdd((int*)(out.toff + j[u]).ptr(), 1) : 0;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int p = b + k0 + u * SG;
                    if (k0 + u * SG < n) {
                        out.nbr[p] = j[u];
                        out.row[p] = q;
                        out.arrival[p] = r[u];
                    }
                }
            }
        } else {
            float x[3];
            (qp + q * 3).get<3>(x);
            const int a = qid[q];
            if (use_grid) grid_row<SYM>(G, L, g, q, x, a, out);
            else if (ne <= TILE) list_row<SYM>(G, L, q, x, a, TileEl{(lp<const float>)c.lds}, 0, ne, 0, out);
            else list_row<SYM>(G, L, q, x, a, MemEl{ep, eid}, 0, ne, 0, out);
        }
    }
    team_sync(c);
}

// Order every transposed row by forward slot: entry tmp[t] of column j (the
// slots whose partner is j, in arrival order) goes to tslot[toff[j] + r],
// r = number of entries of the column with a smaller slot.  Columns are split
// among the team's workgroups; each workgroup stages runs of whole columns in
// LDS.  All threads of the team.
__device__ __forceinline__ void pg_order_columns(Ctx& c, GraphC& G, int n2) {
    ap<const int> toff = c.I + G.toff;
    ap<const int> tmp = c.I + G.tmp;
    ap<const int> nbr = c.I + G.nbr;
    ap<int> tslot = c.I + G.tslot;
    lp<int> sl = (lp<int>)c.lds;
    const int CAP = LDS_FLOATS;
    int per = (n2 + c.G - 1) / c.G;
    int jb = min(c.rank * per, n2);
    const int jend = min(jb + per, n2);
    while (jb < jend) {
        const int base = uni(toff[jb]);
        // the longest run of whole columns [jb, je) that fits: largest je in
        // [jb+1, jend] with toff[je] - base <= CAP (je = jb+1 if none)
        int lo = jb + 1, hi = jend;
        while (lo < hi) {
            int mid = (lo + hi + 1) >> 1;
            if (uni(toff[mid]) - base <= CAP) lo = mid; else hi = mid - 1;
        }
        const int je = lo;
        const int n = uni(toff[je]) - base;
        if (n <= CAP) {
            for (int k = c.tid; k < n; k += NT) sl[k] = tmp[base + k];
            __syncthreads();
            constexpr int U = 4;  // loads of four entries in flight
            for (int k0 = c.tid; k0 < n; k0 += U * NT) {
                int slot[U], u0[U], u1[U];
#pragma unroll
                for (int h = 0; h < U; ++h) {
                    slot[h] = sl[min(k0 + h * NT, n - 1)];
                    const int j = nbr[slot[h]];
                    u0[h] = toff[j] - base;
                    u1[h] = toff[j + 1] - base;
                }
#pragma unroll
                for (int h = 0; h < U; ++h) {
                    if (k0 + h * NT >= n) continue;
                    int r = 0;
                    for (int u = u0[h]; u < u1[h]; ++u) r += sl[u] < slot[h];
                    tslot[base + u0[h] + r] = slot[h];
                }
            }
            __syncthreads();
        } else {  // one column longer than the LDS area: rank from memory
            for (int k = c.tid; k < n; k += NT) {
                int s = tmp[base + k];
                int r = 0;
                for (int u = 0; u < n; ++u) r += tmp[base + u] < s;
                tslot[base + r] = s;
            }
        }
        jb = je;
    }
    list_sync(c);
}

// Latency bound: a chain of short phases (scan, sums of offsets, fill, columns)
// of a few dependent loads each, so the rows are scanned once (their hits wait
// in slabs for the offsets), columns are counted while rows are filled, and
// loops over slots keep four slots' loads in flight.  Per rebuild of the
// rotamer graph of 1000 residues on 32 workgroups 200 -> 143 us, of 67 residues
// on 16 8.9 -> 7.2; sums over the other eight graphs of 1000 residues: LDS grids
// 115 -> 22, scans 205 -> 101, columns 123 -> 91.
// Rebuild rows and transposed rows from pos_pack.  False, with state[1] set,
// on overflow (the host grows the capacity and repeats the run).
//   forward rows:    side-1 element i, partners j (symmetric: j > i) in the
//                    canonical scan order;
//   transposed rows: side-2 element j, the forward slots with partner j in
//                    increasing slot order.
__device__ __forceinline__ bool pg_rebuild(Ctx& c, GraphC& G) {
    gp<const int> id1 = c.CI + G.id1;
    const bool sym = G.sym != 0;
    gp<const int> id2 = sym ? id1 : c.CI + G.id2;
    ap<const float> pack = c.A + G.pos_pack;
    ap<float> cache = c.A + G.cache_pos;
    ap<const float> p1 = pack;
    ap<const float> p2 = pg_side2(c, G);
    const int n1 = G.n1, n2 = sym ? G.n1 : G.n2;
    ap<int> off = c.I + G.off;
    ap<int> nbr = c.I + G.nbr;
    ap<int> row = c.I + G.row;
    ap<int> toff = c.I + G.toff;
    ap<int> tmp = c.I + G.tmp;
    ap<int> arrival = c.I + G.tslot;  // until the columns are ordered
    const SlabOut slab{tmp, G.ecap / max(n1, 1)};
    int npack = sym ? n1 : n1 + n2;
    for (int i = c.gtid; i < npack * 3; i += c.gsize) cache[i] = pack[i];
    for (int j = c.gtid; j <= n2; j += c.gsize) toff[j] = 0;
    if (c.gtid == 0) off[n1] = 0;
    unsigned long long t0 = ptick(c);
    // Small graphs scan every row against the whole other side staged in LDS
    // (n1 * n2 distance tests spread over the team cost less than the grid
    // build's serial phases; measured: 4-5 % of a step at 150-500 residues);
    // larger ones use the cell grid.  Either stays in LDS from the count scan
    // to the fill.  The choice depends on the sizes only, so every team size
    // builds the same rows.
    const bool use_grid = lgrid_fits(n2) && (long long)n1 * n2 > (1ll << 21);
    LGrid g{};
    if (use_grid) {
        g = lgrid_build(c, G, p2, id2, n2);
        pacc(c, PROF_RB_GRID, t0);
    }
    unsigned long long t1 = ptick(c);
    if (use_grid) {
        if (sym) grid_rows<true>(c, G, g, p1, id1, n1, off, slab);
        else grid_rows<false>(c, G, g, p1, id1, n1, off, slab);
    } else {
        if (sym) tile_rows<true>(c, G, p1, id1, n1, p2, id2, n2, off, slab);
        else tile_rows<false>(c, G, p1, id1, n1, p2, id2, n2, off, slab);
    }
    pacc(c, PROF_RB_SCAN, t1);
    const int E = team_exscan(c, off, n1 + 1);
    if (E > G.ecap) {
        if (c.gtid == 0) { c.I[G.state + 1] = 1; c.I[G.state + 0] = 0; }
        team_sync(c);
        return false;
    }
    pacc(c, PROF_RB_COUNT, t0);
    t0 = ptick(c);
    const SlotOut out{nbr, row, toff, arrival, 0};
    if (sym) pg_fill<true>(c, G, g, use_grid, p1, id1, n1, p2, id2, n2, off, slab, out);
    else pg_fill<false>(c, G, g, use_grid, p1, id1, n1, p2, id2, n2, off, slab, out);
    pacc(c, PROF_RB_FILL, t0);
    t0 = ptick(c);
    // transposed rows: column starts, arrival-order placement, slot order
    team_exscan(c, toff, n2 + 1);
    constexpr int U = 4;  // loads of four slots in flight
    for (int s0 = c.gtid; s0 < E; s0 += U * c.gsize) {
        int at[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int s = min(s0 + u * c.gsize, E - 1);
            at[u] = toff[nbr[s]] + arrival[s];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (s0 + u * c.gsize < E) tmp[at[u]] = s0 + u * c.gsize;
    }
    if (c.gtid == 0) {
        c.I[G.state + 0] = 1;
        c.I[G.state + 2] += 1;
        c.I[G.state + 3] = E;
    }
    list_sync(c);
    pg_order_columns(c, G, n2);
    pacc(c, PROF_RB_MAP, t0);
    return true;
}

// ---- edge functions -----------------------------------------------------
// quadspline (src/bead_interaction.h:31-85): radial clamped splines times
// angular splines of the two bead directions.
template <int NKA, int NK, class P, class X>
__device__ __forceinline__ float quadspline(P p, X x1, X x2, float inv_dtheta, float inv_dx, float* d1, float* d2) {
    float dx = x2[0] - x1[0], dy = x2[1] - x1[1], dz = x2[2] - x1[2];
    float r1x = x1[3], r1y = x1[4], r1z = x1[5];
    float r2x = x2[3], r2y = x2[4], r2z = x2[5];
    float dist2 = __fmaf_rn(dz, dz, __fmaf_rn(dy, dy, dx * dx));
    float inv = rsqrtf(dist2);
    float dist_coord = dist2 * (inv * inv_dx);
    float ux = inv * dx, uy = inv * dy, uz = inv * dz;
    float c1 = r1x * ux + r1y * uy + r1z * uz;
    float c2 = -(r2x * ux + r2y * uy + r2z * uz);
    // the window p[xb-1..xb+2] must stay inside the parameter row (NaN -> 1)
    float xa1 = fminf(fmaxf((c1 + 1.f) * inv_dtheta + 1.f, 1.f), (float)(NKA - 2));
    float xa2 = fminf(fmaxf((c2 + 1.f) * inv_dtheta + 1.f, 1.f), (float)(NKA - 2));
    float a1, da1, a2, da2, w, dw, nn, dn;
    deboor(p, xa1, a1, da1);
    deboor(p + NKA, xa2, a2, da2);
    clamped_deboor(p + 2 * NKA, dist_coord, NK, w, dw);
    clamped_deboor(p + 2 * NKA + NK, dist_coord, NK, nn, dn);
    float aw = a1 * a2;
    float rad = inv_dx * (dw + aw * dn);
    float ad1 = inv_dtheta * da1 * a2 * nn;
    float ad2 = inv_dtheta * a1 * da2 * nn;
    float rx = ad1 * r1x - ad2 * r2x, ry = ad1 * r1y - ad2 * r2y, rz = ad1 * r1z - ad2 * r2z;
    float ur = ux * rx + uy * ry + uz * rz;
    float ddx = rad * ux + inv * (rx - ur * ux);
    float ddy = rad * uy + inv * (ry - ur * uy);
    float ddz = rad * uz + inv * (rz - ur * uz);
    d1[0] = -ddx; d1[1] = -ddy; d1[2] = -ddz;
    d1[3] = ad1 * ux; d1[4] = ad1 * uy; d1[5] = ad1 * uz;
    d2[0] = ddx; d2[1] = ddy; d2[2] = ddz;
    d2[3] = -ad2 * ux; d2[4] = -ad2 * uy; d2[5] = -ad2 * uz;
    return w + aw * nn;
}

// ProteinHBondInteraction (src/hbond.cpp:158-246).
template <class P, class X>
__device__ __forceinline__ float protein_hbond_edge(P p, X x1, X x2, float* d1, float* d2) {
    float HOx = x1[0] - x2[0], HOy = x1[1] - x2[1], HOz = x1[2] - x2[2];
    float m2 = __fmaf_rn(HOz, HOz, __fmaf_rn(HOy, HOy, HOx * HOx)) + 1e-6f;
    float inv = rsqrtf(m2);
    float mag = m2 * inv;
    float rx = HOx * inv, ry = HOy * inv, rz = HOz * inv;
    float dHOC = rx * x2[3] + ry * x2[4] + rz * x2[5];
    float dOHN = -(rx * x1[3] + ry * x1[4] + rz * x1[5]);
    float hb = 0.f, dH[3] = {0, 0, 0}, drHN[3] = {0, 0, 0}, drOC[3] = {0, 0, 0};
    if (dHOC > 0.f && dOHN > 0.f) {
        float os, osd, is, isd, a1, da1, a2, da2;
        sigmoid((p[2] - mag) * p[3], os, osd);
        sigmoid((mag - p[0]) * p[1], is, isd);
        float rv = os * is;
        float rd = -p[3] * osd * is + p[1] * isd * os;
        sigmoid((dHOC - p[4]) * p[5], a1, da1); da1 *= p[5];
        sigmoid((dOHN - p[4]) * p[5], a2, da2); da2 *= p[5];
        hb = rv * a1 * a2;
        float c0 = rd * a1 * a2, c1 = rv * da1 * a2, c2 = -rv * a1 * da2;
        float r[3] = {rx, ry, rz};
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            drOC[k] = c1 * r[k];
            drHN[k] = c2 * r[k];
            dH[k] = c0 * r[k] + (c1 * inv) * (x2[3 + k] - dHOC * r[k]) + (c2 * inv) * (x1[3 + k] + dOHN * r[k]);
        }
    }
    float hb_log = (1.f <= hb) ? 100.f : -logf(1.f - hb);
    float pref = fminf(1.f / (1.f - hb), 1e5f);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        d1[k] = dH[k] * pref; d1[3 + k] = drHN[k] * pref;
        d2[k] = -dH[k] * pref; d2[3 + k] = drOC[k] * pref;
    }
    return hb_log;
}

// Environment coverage (src/environment.cpp:114-228); weighted: second element
// carries a probability in component 3.
template <bool WEIGHTED, class P, class X>
__device__ __forceinline__ float env_edge(P p, X x1, X x2, float* d1, float* d2) {
    float dx = x2[0] - x1[0], dy = x2[1] - x1[1], dz = x2[2] - x1[2];
    float dist2 = __fmaf_rn(dz, dz, __fmaf_rn(dy, dy, dx * dx));
    float inv = rsqrtf(dist2);
    float dist = dist2 * inv;
    float ux = inv * dx, uy = inv * dy, uz = inv * dz;
    float dp = ux * x1[3] + uy * x1[4] + uz * x1[5];
    float rs, drs, as, das;
    compact_sigmoid(dist - p[0], p[1], rs, drs);
    compact_sigmoid(p[2] - dp, p[3], as, das);
    float prob = WEIGHTED ? x2[3] : 1.f;
    float u[3] = {ux, uy, uz};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        float ddk = prob * (drs * as * u[k] - rs * das * inv * (x1[3 + k] - dp * u[k]));
        d1[k] = -ddk;
        d1[3 + k] = -prob * rs * das * u[k];
        d2[k] = ddk;
    }
    float score = rs * as;
    if (WEIGHTED) {
        d2[3] = score;
        return prob * score;
    }
    d2[3] = d2[4] = d2[5] = 0.f;
    return score;
}

// a x b with the second product of each component rounded first.
__device__ __forceinline__ void cross3_rn(const float* a, const float* b, float* o) {
    o[0] = __fmaf_rn(a[1], b[2], -__fmul_rn(a[2], b[1]));
    o[1] = __fmaf_rn(a[2], b[0], -__fmul_rn(a[0], b[2]));
    o[2] = __fmaf_rn(a[0], b[1], -__fmul_rn(a[1], b[0]));
}

// BackbonePairs residue pair (src/backbone_steric.cpp:94-140): compact-sigmoid
// repulsion between the placed backbone atoms (at most 4) of two residues;
// derivatives are (force, torque) on each residue frame.
__device__ __forceinline__ float backbone_edge(const Ctx& c, OpC& op, int r1, int r2, float* d1, float* d2) {
    ap<const float> aff = c.A + op.in_out[0];
    int w = op.in_w[0];
    gp<const float> ref = c.CF + op.ia[1];
    gp<const int> nat = c.CI + op.ia[2];
    gp<const int> res = c.CI + op.ia[0];
    int R1 = res[r1], R2 = res[r2];
    float a1[7], a2[7];
#pragma unroll
    for (int k = 0; k < 7; ++k) { a1[k] = aff[R1 * w + k]; a2[k] = aff[R2 * w + k]; }
    float U1[9], U2[9];
    quat_to_rot(a1 + 3, U1);
    quat_to_rot(a2 + 3, U2);
    float X1[4][3], X2[4][3];
    int n1 = nat[r1], n2 = nat[r2];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        gp<const float> q = ref + (r1 * 4 + a) * 3;
        gp<const float> s = ref + (r2 * 4 + a) * 3;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            X1[a][k] = U1[3 * k] * q[0] + U1[3 * k + 1] * q[1] + U1[3 * k + 2] * q[2] + a1[k];
            X2[a][k] = U2[3 * k] * s[0] + U2[3 * k + 1] * s[1] + U2[3 * k + 2] * s[2] + a2[k];
        }
    }
    const float cut2 = 3.f * 3.f + 0.1f * 3.f;
    const float sharp = 1.f / (3.0f * 0.10f);
    float pot = 0.f;
#pragma unroll
    for (int k = 0; k < 6; ++k) { d1[k] = 0.f; d2[k] = 0.f; }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (i >= n1 || j >= n2) continue;
            float rx = X1[i][0] - X2[j][0], ry = X1[i][1] - X2[j][1], rz = X1[i][2] - X2[j][2];
            float rm2 = rx * rx + ry * ry + rz * rz;
            if (rm2 > cut2) continue;
            float v, dv;
            compact_sigmoid(rm2 - 9.f, sharp, v, dv);
            pot += 4.f * v;
            float g = 2.f * 4.f * dv;
            // the roundings are fixed here: left to the compiler, which product
            // of a torque rounds first depends on the code around it, and a
            // trajectory amplifies that
            const float gv[3] = {g * rx, g * ry, g * rz};
            const float p1[3] = {X1[i][0] - a1[0], X1[i][1] - a1[1], X1[i][2] - a1[2]};
            const float p2[3] = {X2[j][0] - a2[0], X2[j][1] - a2[1], X2[j][2] - a2[2]};
            float t1[3], t2[3];
            cross3_rn(p1, gv, t1);
            const bool flip = i == 0 && j < 2;  // the first pairs add g x p2, the others subtract p2 x g
            if (flip) cross3_rn(gv, p2, t2);
            else cross3_rn(p2, gv, t2);
            const float r[3] = {rx, ry, rz};
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                d1[k] = __fmaf_rn(r[k], g, d1[k]);
                d2[k] = __fmaf_rn(-r[k], g, d2[k]);
                d1[3 + k] += t1[k];
                d2[3 + k] += flip ? t2[k] : -t2[k];
            }
        }
    }
    return pot;
}

// Refine every cached slot against the cutoff and evaluate the active edges;
// param is the coefficient table (LDS or memory).
template <int KIND, int DD1, int DD2, class P>
__device__ __forceinline__ void pg_edges_impl(Ctx& c, GraphC& G, OpC& op, P param) {
    ap<const int> nbr = c.I + G.nbr;
    ap<const int> row = c.I + G.row;
    ap<int> act = c.I + G.act;
    ap<float> val = c.A + G.val;
    ap<float> D1 = c.A + G.d1;
    ap<float> D2 = c.A + G.d2;
    ap<const float> pack = c.A + G.pos_pack;
    ap<const float> pk2 = pg_side2(c, G);
    gp<const int> loc1 = c.CI + G.loc1;
    gp<const int> loc2 = c.CI + G.loc2;
    gp<const int> t1 = c.CI + G.type1;
    gp<const int> t2 = c.CI + G.type2;
    ap<const float> P1 = c.A + G.out1;
    ap<const float> P2 = c.A + G.out2;
    const int E = uni(c.I[G.state + 3]);
    const int cap = G.ecap;
    for (int s = c.gtid; s < E; s += c.gsize) {
        int i1 = row[s], j = nbr[s];
        ap<const float> xp = pack + i1 * 3;
        ap<const float> yp = pk2 + j * 3;
        float d2 = refine_dist2(xp[0] - yp[0], xp[1] - yp[1], xp[2] - yp[2]);
        int a = d2 < G.cutoff2;
        act[s] = a;
        if (!a) { val[s] = 0.f; continue; }
        ap<const float> x1 = P1 + loc1[i1] * G.w1;
        ap<const float> x2 = P2 + loc2[j] * G.w2;
        P p = param + (t1[i1] * G.n_type2 + t2[j]) * G.n_param;
        float e1[7], e2[7];
        float v = 0.f;
        if (KIND == EDGE_ROTAMER) {
            v = quadspline<15, 12>(p, x1, x2, 6.f, 1.f / 0.7f, e1, e2);
        } else if (KIND == EDGE_HBOND_COVERAGE) {
            float cov = quadspline<15, 10>(p, x1, x2, 6.f, 1.f / 0.625f, e1, e2);
            float om = 1.f - x1[6];
            float pref = om * om;
#pragma unroll
            for (int q = 0; q < 6; ++q) { e1[q] *= pref; e2[q] *= pref; }
            e1[6] = -cov * om * 2.f;
            v = pref * cov;
        } else if (KIND == EDGE_PROTEIN_HBOND) {
            v = protein_hbond_edge(p, x1, x2, e1, e2);
        } else if (KIND == EDGE_ENV_WEIGHTED) {
            v = env_edge<true>(p, x1, x2, e1, e2);
        } else if (KIND == EDGE_ENV_HBOND) {
            v = env_edge<false>(p, x1, x2, e1, e2);
        } else {
            v = backbone_edge(c, op, i1, j, e1, e2);
        }
        val[s] = v;
#pragma unroll
        for (int q = 0; q < DD1; ++q) D1[q * cap + s] = e1[q];
#pragma unroll
        for (int q = 0; q < DD2; ++q) D2[s * DD2 + q] = e2[q];
    }
    team_sync(c);
}

// Stage the graph's coefficient table in this workgroup's LDS when it has one
// that fits, then evaluate.
template <int KIND, int DD1, int DD2>
__device__ __forceinline__ void pg_edges_t(Ctx& c, GraphC& G, OpC& op) {
    gp<const float> src = c.CF + G.param;
    if (G.param_len > 0) {
        lp<float> L = c.lds;
        for (int k = c.tid; k < G.param_len; k += NT) L[k] = src[k];
        __syncthreads();
        pg_edges_impl<KIND, DD1, DD2>(c, G, op, (lp<const float>)L);
    } else {
        pg_edges_impl<KIND, DD1, DD2>(c, G, op, src);
    }
}

__device__ __forceinline__ void pg_edges(Ctx& c, GraphC& G, OpC& op) {
    switch (G.kind) {
    case EDGE_ROTAMER: pg_edges_t<EDGE_ROTAMER, 6, 6>(c, G, op); break;
    case EDGE_HBOND_COVERAGE: pg_edges_t<EDGE_HBOND_COVERAGE, 7, 6>(c, G, op); break;
    case EDGE_PROTEIN_HBOND: pg_edges_t<EDGE_PROTEIN_HBOND, 6, 6>(c, G, op); break;
    case EDGE_ENV_WEIGHTED: pg_edges_t<EDGE_ENV_WEIGHTED, 6, 4>(c, G, op); break;
    case EDGE_ENV_HBOND: pg_edges_t<EDGE_ENV_HBOND, 6, 6>(c, G, op); break;
    default: pg_edges_t<EDGE_BACKBONE, 6, 6>(c, G, op); break;
    }
}

// Gather esens*deriv into the producers in a fixed order: groups of 16 lanes
// per element, each lane striding the element's slots, then a fixed-order
// group reduction.
constexpr int GW = 16;
static_assert(GW <= 32 && (GW & (GW - 1)) == 0, "a lane group is a power of two within half a wave");

template <int D1N, int D2N>
__device__ __forceinline__ void pg_gather_t(Ctx& c, GraphC& G) {
    ap<const int> off = c.I + G.off;
    ap<const int> toff = c.I + G.toff;
    ap<const int> tslot = c.I + G.tslot;
    ap<const int> act = c.I + G.act;
    ap<const float> es = c.A + G.esens;
    ap<const float> D1 = c.A + G.d1;
    ap<const float> D2 = c.A + G.d2;
    gp<const int> loc1 = c.CI + G.loc1;
    gp<const int> loc2 = c.CI + G.loc2;
    ap<float> S1 = c.A + G.sens1;
    ap<float> S2 = c.A + G.sens2;
    const int cap = G.ecap;
    int grp = c.gtid / GW, gl = c.gtid % GW;
    const int NG = c.gsize / GW;
    // uniform trip counts: every lane runs every group reduction
    for (int base = 0; base < G.n1; base += NG) {
        int i = base + grp;
        bool ok = i < G.n1;
        float acc[D1N];
#pragma unroll
        for (int q = 0; q < D1N; ++q) acc[q] = 0.f;
        int b = ok ? off[i] : 0, e = ok ? off[i + 1] : 0;
        // branch-free: every load of an iteration is issued at once
#pragma unroll 2
        for (int s = b + gl; s < e; s += GW) {
            bool a = act[s] != 0;
            float w = es[s];
#pragma unroll
            for (int q = 0; q < D1N; ++q) {
                float d = D1[q * cap + s];
                acc[q] += a ? w * d : 0.f;
            }
        }
        if (G.sym && ok) {
            int tb = toff[i], te = toff[i + 1];
#pragma unroll 2
            for (int t = tb + gl; t < te; t += GW) {
                int s = tslot[t];
                bool a = act[s] != 0;
                float w = es[s], d[D1N];
                (D2 + s * D1N).template get<D1N>(d);
#pragma unroll
                for (int q = 0; q < D1N; ++q) acc[q] += a ? w * d[q] : 0.f;
            }
        }
#pragma unroll
        for (int q = 0; q < D1N; ++q) acc[q] = group_sum<GW>(acc[q]);
        if (ok && gl == 0) {
            ap<float> dst = S1 + loc1[i] * G.w1;
            dst.template add<D1N>(acc);
        }
    }
    // both sides in one phase unless they accumulate into shared producer rows
    if (G.sym || G.gather_split) team_sync(c);
    if (G.sym) return;
    for (int base = 0; base < G.n2; base += NG) {
        int j = base + grp;
        bool ok = j < G.n2;
        float acc[D2N];
#pragma unroll
        for (int q = 0; q < D2N; ++q) acc[q] = 0.f;
        int tb = ok ? toff[j] : 0, te = ok ? toff[j + 1] : 0;
#pragma unroll 2
        for (int t = tb + gl; t < te; t += GW) {
            int s = tslot[t];
            bool a = act[s] != 0;
            float w = es[s], d[D2N];
            (D2 + s * D2N).template get<D2N>(d);
#pragma unroll
            for (int q = 0; q < D2N; ++q) acc[q] += a ? w * d[q] : 0.f;
        }
#pragma unroll
        for (int q = 0; q < D2N; ++q) acc[q] = group_sum<GW>(acc[q]);
        if (ok && gl == 0) {
            ap<float> dst = S2 + loc2[j] * G.w2;
            dst.template add<D2N>(acc);
        }
    }
    team_sync(c);
}

__device__ __forceinline__ void pg_gather(Ctx& c, GraphC& G) {
    unsigned long long t0 = ptick(c);
    switch (G.kind) {
    case EDGE_HBOND_COVERAGE: pg_gather_t<7, 6>(c, G); break;
    case EDGE_ENV_WEIGHTED: pg_gather_t<6, 4>(c, G); break;
    default: pg_gather_t<6, 6>(c, G); break;  // symmetric graphs: both sides 6 wide
    }
    pacc(c, PROF_PG_GATHER, t0);
}

// Sum of the active edge values of each row (side 1) or transposed row
// (side 2), in slot order: out[k*stride] = sum.  Groups of 16 lanes.
template <class O>
__device__ __forceinline__ void pg_row_sums(Ctx& c, GraphC& G, bool side2, O out, int stride) {
    ap<const int> off = c.I + (side2 ? G.toff : G.off);
    ap<const int> tslot = c.I + G.tslot;
    ap<const float> val = c.A + G.val;
    int n = side2 ? G.n2 : G.n1;
    int grp = c.gtid / GW, gl = c.gtid % GW;
    for (int base = 0; base < n; base += c.gsize / GW) {
        int r = base + grp;
        bool ok = r < n;
        float acc = 0.f;
        int k0 = ok ? off[r] : 0, k1 = ok ? off[r + 1] : 0;
        for (int k = k0 + gl; k < k1; k += GW) {
            int s = side2 ? tslot[k] : k;
            float v = val[s];  // zero on inactive slots
            acc += v;
        }
        acc = group_sum<GW>(acc);
        if (ok && gl == 0) out[r * stride] = acc;
    }
}

}  // namespace upside
