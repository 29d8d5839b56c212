// Edge and face ids in the reference's first-occurrence order, and the
// relations derived from them (include/cuda_extraction.h relation set).
//
// Edges (src/cpu_extraction.cpp:28-92): the edge {lo, hi} gets the rank of
// its first position 6c + k (cells ascending, pair k over (0,1) (0,2) (0,3)
// (1,2) (1,3) (2,3)) among all edges' first positions.  One lane per vertex
// v walks v's tets in ascending order and records, for every upper
// neighbour u > v (an entry of the ascending VV row), the first position it
// meets; first positions are flagged in a byte array, packed to bits with
// scanned counts, and an edge's id is the rank of its first position.  No atomics.
//
// Faces (src/cpu_extraction.cpp:122-222): slot s of cell c is the positional
// triple (cv[lo], cv[mid], cv[hi]) with (lo, mid, hi) = (0,1,2) (0,1,3)
// (0,2,3) (1,2,3), position 4c + s; the key is not sorted.  The cells holding
// all three vertices are ET(lo,mid) n ET(lo,hi); the first occurrence of a
// key is the smallest position among those cells' slots with the same
// positional triple, and face ids are ranks of first occurrences.
//
// The other relations with rows count, scan and write in one launch each (a
// chained scan over tiles; rows of many cells or edges in launches beside it): ET(e) = VT(lo) n VT(hi), TT and EE as joins, VE
// and VF from a vertex's VV row and cells, EF and FF from TE and TF; FT comes
// from the face matches.
#include <algorithm>

#include "ids.h"
#include "networks.h"
#include "tetra_c.h"

namespace {

constexpr int INF = INT32_MAX;

// pair index of corner positions i < j: (0,1)0 (0,2)1 (0,3)2 (1,2)3 (1,3)4 (2,3)5
__device__ __forceinline__ int pair_index(int i, int j) {
    return i == 0 ? j - 1 : (i == 1 ? j + 1 : 5);
}

__device__ __forceinline__ int32_t corner(const int4 &q, int j) {
    return j == 0 ? q.x : j == 1 ? q.y : j == 2 ? q.z : q.w;
}

// positions (lo, mid, hi) of face slot s
__device__ __forceinline__ void face_pos(int s, int &lo, int &mid, int &hi) {
    lo = s == 3 ? 1 : 0;
    mid = s <= 1 ? 1 : 2;
    hi = s == 0 ? 2 : 3;
}

// index of x in the ascending array a[0..n), or -1.  Rows shorter than 128
// take seven fixed steps (no data-dependent loop), so several searches of
// one thread overlap their loads; longer rows bisect.
__device__ __forceinline__ int32_t bsearch_i32(const int32_t *a, int32_t n, int32_t x) {
    int32_t lo = 0;
    if (n < 128) {
#pragma unroll
        for (int step = 64; step >= 1; step >>= 1) {
            const int32_t probe = lo + step - 1;
            if (probe < n && a[probe] < x) lo += step;
        }
    } else {
        int32_t hi = n;
        while (lo < hi) {
            const int32_t mid = (lo + hi) >> 1;
            if (a[mid] < x) lo = mid + 1;
            else hi = mid;
        }
    }
    return (lo < n && a[lo] == x) ? lo : -1;
}

// Unaligned 16- and 8-byte loads: dword alignment is enough for
// global_load_dwordx4/x2 on gfx950.
typedef int32_t i32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef int32_t i32x2u __attribute__((ext_vector_type(2), aligned(4)));

// A thread's row of n words in its LDS column (consecutive threads in
// consecutive banks), by independent 16-byte loads, so that it costs one memory
// latency instead of one per element.  Whole quads are read, up to three words
// past the row (the source array carries that slack).
template <int W>
__device__ __forceinline__ void stage_quads(int32_t (*buf)[W], const int32_t *__restrict__ src,
                                            int32_t n) {
#pragma unroll 4
    for (int32_t k = 0; k < n; k += 4) {
        const i32x4u v = *reinterpret_cast<const i32x4u *>(src + k);
        buf[k][threadIdx.x] = v.x;
        buf[k + 1][threadIdx.x] = v.y;
        buf[k + 2][threadIdx.x] = v.z;
        buf[k + 3][threadIdx.x] = v.w;
    }
}

// A thread's output row at its exact position: words gather in a register
// quad, full quads leave in unaligned 16-byte stores, the last one to three
// words one by one (the words after the row belong to the next row).  One
// store per four words instead of one per word: scattered per-thread rows cost
// the vector memory path per store instruction.
struct QuadOutExact {
    int32_t *row;
    int64_t n = 0;
    int4 q = make_int4(0, 0, 0, 0);
    __device__ __forceinline__ void put(int32_t v) {
        const int k = (int)(n & 3);
        q.x = k == 0 ? v : q.x;
        q.y = k == 1 ? v : q.y;
        q.z = k == 2 ? v : q.z;
        q.w = k == 3 ? v : q.w;
        if (k == 3) *reinterpret_cast<i32x4u *>(row + n - 3) = i32x4u{q.x, q.y, q.z, q.w};
        n++;
    }
    __device__ __forceinline__ void flush() {
        const int k = (int)(n & 3);
        int32_t *tail = row + (n & ~(int64_t)3);
        if (k > 0) tail[0] = q.x;
        if (k > 1) tail[1] = q.y;
        if (k > 2) tail[2] = q.z;
    }
};

// ---- edges --------------------------------------------------------------------
// Lane per vertex v: first position of every edge (v, u) of its row; upper
// ones (u > v) are flagged.
// Every pair of v's cells whose low vertex is v also records its edge's first
// position in te (replaced by the edge id, its rank, once ranks exist): the
// row search is done here, on v's own row, instead of once per cell on random
// rows, and the ranks (16 bytes per 96 positions) are a fraction of the
// VV-aligned ids that te could index instead.
// Rows up to EDGE_CAP entries are staged in LDS (one column per thread: the
// VV row and the first positions), and the vertex's cells are fetched eight
// at a time with independent loads.  A longer row is the whole wave's: its
// first positions fill the LDS, the lanes go over the vertex's cells.  (TE, EV
// and VE of 4000 cells around one vertex 0.5 ms, by one lane in global memory
// 16 with the highest id and 19 with the lowest; of a 470 k-cell Delaunay
// mesh 0.23 ms, 0.51.)
constexpr int EDGE_THREADS = 64, EDGE_CAP = 32;  // 16 KB a wave: ten waves per CU

__global__ __launch_bounds__(EDGE_THREADS) void k_edge_first(
    const int4 *__restrict__ tv4, const int32_t *__restrict__ vt_off,
    const int32_t *__restrict__ vtc, const int32_t *__restrict__ vv_off,
    const int32_t *__restrict__ vv, int64_t V, int32_t *__restrict__ efirst,
    uint8_t *__restrict__ flags, int32_t *__restrict__ te_first) {
    static_assert(EDGE_CAP % 4 == 0, "rows are staged by whole quads");
    static_assert(2 * EDGE_CAP * EDGE_THREADS >= tg::HEAVY_CAP, "one row's first positions");
    __shared__ int32_t lds[2 * EDGE_CAP * EDGE_THREADS];
    int32_t(*srow)[EDGE_THREADS] = reinterpret_cast<int32_t(*)[EDGE_THREADS]>(lds);
    int32_t(*sef)[EDGE_THREADS] = srow + EDGE_CAP;
    const int tid = threadIdx.x;
    for (int64_t v0 = (int64_t)blockIdx.x * EDGE_THREADS; v0 < V; v0 += (int64_t)gridDim.x * EDGE_THREADS) {
        const int64_t v = v0 + tid;
        const bool act = v < V;
        const int32_t rb = act ? vv_off[v] : 0, rn = act ? vv_off[v + 1] - rb : 0;
        const int32_t kb = act ? vt_off[v] : 0, ke = act ? vt_off[v + 1] : 0;
        if (act && rn <= EDGE_CAP) {
            stage_quads(srow, vv + rb, rn);
            for (int32_t i = 0; i < rn; i++) sef[i][tid] = INF;
            for (int32_t k0 = kb; k0 < ke; k0 += 8) {
                int32_t pc[8];
                int4 q[8];
#pragma unroll
                for (int c = 0; c < 8; c++) pc[c] = k0 + c < ke ? vtc[k0 + c] : -1;
#pragma unroll
                for (int c = 0; c < 8; c++) q[c] = pc[c] >= 0 ? tv4[pc[c] >> 2] : make_int4(0, 0, 0, 0);
#pragma unroll
                for (int c = 0; c < 8; c++) {
                    if (pc[c] < 0) continue;
                    const int32_t t = pc[c] >> 2, jv = pc[c] & 3;
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        if (j == jv) continue;
                        const int32_t u = corner(q[c], j);
                        int32_t lo = 0;  // place of u in the staged row (rn <= 32)
#pragma unroll
                        for (int step = 16; step >= 1; step >>= 1)
                            if (lo + step - 1 < rn && srow[lo + step - 1][tid] < u) lo += step;
                        const int32_t idx = lo < rn && srow[lo][tid] == u ? lo : -1;
                        const int32_t pos = 6 * t + pair_index(min(j, (int)jv), max(j, (int)jv));
                        int32_t p1 = INF;  // first position of the edge
                        if (idx >= 0) {
                            p1 = min(sef[idx][tid], pos);  // cells ascend
                            sef[idx][tid] = p1;
                        }
                        if (u > v) te_first[pos] = p1;
                    }
                }
            }
            QuadOutExact o;
            o.row = efirst + rb;
            for (int32_t i = 0; i < rn; i++) {
                const int32_t e = sef[i][tid];
                o.put(e);
                if (srow[i][tid] > v && e != INF) flags[e] = 1;
            }
            o.flush();
        }
        for (uint64_t b = __ballot(rn > EDGE_CAP); b; b &= b - 1) {
            const int l = __ffsll((unsigned long long)b) - 1;
            const int32_t w = (int32_t)v0 + l, wrb = tgd::lane_value(rb, l), wrn = tgd::lane_value(rn, l);
            const int32_t wkb = tgd::lane_value(kb, l), wke = tgd::lane_value(ke, l);
            const int32_t *row = vv + wrb;
            tgd::wave_sync();  // what was in the LDS has been read
            for (int32_t i = tid; i < wrn; i += EDGE_THREADS) lds[i] = INF;
            tgd::wave_sync();
            // f(position, u) for the lane's share of the vertex's cells' edges
            auto each = [&](auto f) {
                for (int32_t k = wkb + tid; k < wke; k += EDGE_THREADS) {
                    const int32_t p = vtc[k], t = p >> 2, jv = p & 3;
                    const int4 q = tv4[t];
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        if (j != jv) f(6 * t + pair_index(min(j, (int)jv), max(j, (int)jv)), corner(q, j));
                }
            };
            each([&](int32_t pos, int32_t u) {
                const int32_t idx = bsearch_i32(row, wrn, u);
                if (idx >= 0) atomicMin(&lds[idx], pos);
                if (u > w) te_first[pos] = idx;
            });
            tgd::wave_sync();
            each([&](int32_t pos, int32_t u) {
                if (u <= w) return;
                const int32_t idx = te_first[pos];
                te_first[pos] = idx >= 0 ? lds[idx] : INF;
            });
            for (int32_t i = tid; i < wrn; i += EDGE_THREADS) {
                const int32_t e = lds[i];
                efirst[wrb + i] = e;
                if (row[i] > w && e != INF) flags[e] = 1;
            }
        }
        tgd::wave_sync();
    }
}

// Rank units: 96 flags and the number of flags set before them in 16 bytes, so
// a random lookup touches one line, and 5 bytes of table hold 30 flags, where
// a count per 32-bit word takes 7.5 and keeps less of the table in each L2
// (VE of 5 M cells 274 -> 202 us, EE's rows 233 -> 132, TE 152 -> 141).
// 96 holds whole cells' flags, for edges (6) and for faces (4).
constexpr int UNIT = 96;

// bytes (0 or 1) -> a unit's flag words (y, z, w) and their number.  16-byte
// loads; the multiplication gathers the low bits of four bytes (bit 8 i moves
// to bit 28 + i; no other product bit reaches 28).
__global__ void k_pack_flags(const uint8_t *__restrict__ flags, int64_t n,
                             uint4 *__restrict__ rank, int32_t *__restrict__ pop) {
    const int64_t nu = (n + UNIT - 1) / UNIT;
    for (int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; u < nu;
         u += (int64_t)gridDim.x * blockDim.x) {
        uint32_t m[3] = {0, 0, 0};
        const int64_t b = UNIT * u;
        if (b + UNIT <= n) {
            const uint4 *p = reinterpret_cast<const uint4 *>(flags + b);
#pragma unroll
            for (int w = 0; w < 3; w++) {
                const uint4 q0 = p[2 * w], q1 = p[2 * w + 1];
                const uint32_t x[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
#pragma unroll
                for (int i = 0; i < 8; i++) m[w] |= ((x[i] * 0x10204080u) >> 28) << (4 * i);
            }
        } else {
#pragma unroll
            for (int w = 0; w < 3; w++)
                for (int i = 0; i < 32 && b + 32 * w + i < n; i++)
                    m[w] |= (uint32_t)(flags[b + 32 * w + i] != 0) << i;
        }
        rank[u] = make_uint4(0u, m[0], m[1], m[2]);
        pop[u] = __popc(m[0]) + __popc(m[1]) + __popc(m[2]);
    }
}

__global__ void k_rank_counts(const int32_t *__restrict__ before, int64_t nu,
                              uint4 *__restrict__ rank) {
    for (int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; u < nu;
         u += (int64_t)gridDim.x * blockDim.x)
        rank[u].x = (uint32_t)before[u];
}

// flags set before place i (0 .. 95) of a unit
__device__ __forceinline__ int32_t rank_in(uint4 q, uint32_t i) {
    const uint32_t a = q.y, b = q.z, c = q.w;
    const uint32_t w = i < 32 ? a : i < 64 ? b : c;
    return (int32_t)q.x + __popc(w & ((1u << (i & 31)) - 1u)) + (i >= 32 ? __popc(a) : 0) +
           (i >= 64 ? __popc(b) : 0);
}

__device__ __forceinline__ int32_t rank_of(const uint4 *__restrict__ rank, int32_t p) {
    const uint32_t u = (uint32_t)p / UNIT;
    return rank_in(rank[u], (uint32_t)p - UNIT * u);
}

// an edge's id; -1 for an entry that no cell gave a position
__device__ __forceinline__ int32_t rank_at(const uint4 *__restrict__ rank, int32_t p) {
    return p != INF ? rank_of(rank, p) : -1;
}

// TE: the first positions that k_edge_first recorded become edge ids.  A
// position per lane, read and written in whole lines: 141 us at 5 M cells (a
// cell per lane, its six lookups in flight and EV in the same launch, took 212
// against 141 + 41).
__global__ void k_te(int32_t *__restrict__ te, int64_t n, const uint4 *__restrict__ rank) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        te[i] = rank_at(rank, te[i]);
}

// EV in id order: a set flag's rank is its edge's id, and its place names the
// cell and the pair, so EV is written in sequence (from the vertices' side it
// is a line per id).  5 M cells: 41 us.
__global__ void k_ev(const int4 *__restrict__ tv4, int64_t T, const uint4 *__restrict__ rank,
                     int2 *__restrict__ ev) {
    for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < T;
         t += (int64_t)gridDim.x * blockDim.x) {
        const uint4 w = rank[t / (UNIT / 6)];
        const uint32_t i = 6 * (uint32_t)(t % (UNIT / 6));  // a cell's flags are in one unit
        const uint32_t lo = i < 32 ? w.y : i < 64 ? w.z : w.w;
        const uint32_t hi = i < 32 ? w.z : i < 64 ? w.w : 0u;
        const uint32_t f = (uint32_t)((((uint64_t)hi << 32) | lo) >> (i & 31)) & 63u;
        const int4 q = tv4[t];
        const int32_t id = rank_in(w, i);
#pragma unroll
        for (int k = 0; k < 6; k++) {
            if (!((f >> k) & 1u)) continue;
            const int pi[6] = {0, 0, 0, 1, 1, 2}, pj[6] = {1, 2, 3, 2, 3, 3};
            const int32_t x = corner(q, pi[k]), y = corner(q, pj[k]);
            ev[id + __popc(f & ((1u << k) - 1u))] = make_int2(min(x, y), max(x, y));
        }
    }
}

// Long rows of keys, all different, in order.  Up to WAVE_ROW keys by one wave:
// every lane's key is compared with every key of the row, 64 a load; more, up
// to as many as a VV row holds, by the block's bitonic sort in LDS.  EE after
// TE on the 100 k-cell fan mesh (rows of up to 313): 0.32 ms, with one lane's
// insertion in memory 7.3, with its heapsort 0.92; on 4000 cells around one
// vertex 0.16 ms, 4.1 if one wave compares there too.
constexpr int WAVE_ROW = 128;

// f(place, key) for each key of a row, place being the number of smaller ones.
template <typename F>
__device__ __forceinline__ void rank_by_wave(const int32_t *__restrict__ key, int32_t n, F f) {
    const int lane = __lane_id();
    for (int32_t i0 = 0; i0 < n; i0 += 64) {
        const int32_t x = key[min(i0 + lane, n - 1)];
        int32_t place = 0;
        for (int32_t j0 = 0; j0 < n; j0 += 64) {
            const int32_t y = j0 + lane < n ? key[j0 + lane] : INF;
#pragma unroll 16
            for (int j = 0; j < 64; j++) place += tgd::lane_value(y, j) < x;
        }
        if (i0 + lane < n) f(place, x);
    }
}

// size keys in LDS, a power of two, ascending; by a whole block, which has
// written them before a barrier.  Ends with one.
template <int THREADS>
__device__ __forceinline__ void sort_by_block(int32_t *key, int32_t size) {
    for (int32_t k = 2; k <= size; k *= 2)
        for (int32_t j = k / 2; j > 0; j /= 2) {
            for (int32_t i = threadIdx.x; i < size / 2; i += THREADS) {
                const int32_t lo = 2 * i - (i & (j - 1)), hi = lo + j;
                const int32_t x = key[lo], y = key[hi];
                if ((x > y) == ((lo & k) == 0)) {
                    key[lo] = y;
                    key[hi] = x;
                }
            }
            __syncthreads();
        }
}

template <int THREADS>
struct LongRow {
    int32_t key[tg::HEAVY_CAP];
    int32_t row[THREADS], n;
};

// The row of n keys at key + at of each lane that has more than 32:
// f(to, place, key) for all of its keys.  Every thread of the block calls it.
template <int THREADS, typename F>
__device__ __forceinline__ void order_long_rows(LongRow<THREADS> &st, const int32_t *__restrict__ key,
                                                int32_t at, int32_t n, int32_t to, F f) {
    const int tid = threadIdx.x;
    for (uint64_t b = __ballot(n > 32 && n <= WAVE_ROW); b; b &= b - 1) {
        const int l = __ffsll((unsigned long long)b) - 1;
        const int32_t lto = tgd::lane_value(to, l);
        rank_by_wave(key + tgd::lane_value(at, l), tgd::lane_value(n, l),
                     [&](int32_t place, int32_t x) { f(lto, place, x); });
    }
    if (__syncthreads_and(n <= WAVE_ROW)) return;
    if (tid == 0) st.n = 0;
    __syncthreads();
    if (n > WAVE_ROW) st.row[atomicAdd(&st.n, 1)] = tid;
    __syncthreads();
    for (int r = 0; r < st.n; r++) {
        if (tid == st.row[r]) {  // handed over by way of the staging
            st.key[0] = at;
            st.key[1] = n;
            st.key[2] = to;
        }
        __syncthreads();
        const int32_t rat = st.key[0], rn = min(st.key[1], (int32_t)tg::HEAVY_CAP), rto = st.key[2];
        __syncthreads();
        int32_t size = 2 * WAVE_ROW;
        while (size < rn) size *= 2;
        for (int32_t i = tid; i < size; i += THREADS) st.key[i] = i < rn ? key[rat + i] : INF;
        __syncthreads();
        sort_by_block<THREADS>(st.key, size);
        for (int32_t i = tid; i < rn; i += THREADS) f(rto, i, st.key[i]);
        __syncthreads();
    }
}

// Each vertex's edge ids, ascending (for EE): the upper entries' ids are VE's,
// a lower entry's is the rank of its first position, which k_edge_first noted
// for both ends of an edge.  (Searching v in each lower neighbour's row took
// 0.63 ms at 5.3 M cells, and sorting the rows in memory 0.28; VE's
// ids from a copy along VV and a count per 32-bit word 0.23; this pass 0.13.)
// Rows of up to 32 entries are sorted in registers.  In longer ones the first
// positions are ordered, as which the ids ascend, and each is looked up once.
constexpr int VX_THREADS = 256;
__global__ __launch_bounds__(VX_THREADS) void k_vertex_edges(const int32_t *__restrict__ vv_off,
                                                             int64_t V,
                                                             const int32_t *__restrict__ efirst,
                                                             const uint4 *__restrict__ rank,
                                                             const int32_t *__restrict__ ve_off,
                                                             const int2 *__restrict__ ve,
                                                             int32_t *__restrict__ out) {
    __shared__ LongRow<VX_THREADS> lng;
    const int64_t v = (int64_t)blockIdx.x * VX_THREADS + threadIdx.x;
    const int32_t rb = v < V ? vv_off[v] : 0, rn = v < V ? vv_off[v + 1] - rb : 0;
    if (rn <= 32) {
        const int32_t vb = v < V ? ve_off[v] : 0, lower = v < V ? rn - (ve_off[v + 1] - vb) : 0;
        int32_t k[32];
#pragma unroll
        for (int i = 0; i < 32; i++) {
            k[i] = INF;
            if (i < rn) k[i] = i < lower ? rank_at(rank, efirst[rb + i]) : ve[vb + (i - lower)].y;
        }
        tgn::sort_keys(k);
#pragma unroll
        for (int i = 0; i < 32; i++)
            if (i < rn) out[rb + i] = k[i];
    }
    order_long_rows(lng, efirst, rb, rn, rb, [&](int32_t to, int32_t place, int32_t p) {
        out[to + place] = rank_at(rank, p);
    });
}

// ---- faces ----------------------------------------------------------------------
// tets holding face slot s of tet t (ascending) via ET(lo,mid) n ET(lo,hi);
// returns the first matching position (smallest 4t'+s' with the same
// positional triple) and counts all matching tets.
// Ids read from TE and ET are checked against E and T: an inconsistent
// relation yields INF (reported by the callers) instead of a stray access.
constexpr int FF_ROW = 8;  // ET rows up to this length take the register path

__device__ __forceinline__ int32_t face_first(const int4 *tv4, int64_t T, const int32_t *te,
                                              int64_t E, const int64_t *et_off,
                                              const int32_t *et, int32_t t, int s,
                                              int32_t &nmatch, int32_t *tets2) {
    const int4 q = tv4[t];
    int lo, mid, hi;
    face_pos(s, lo, mid, hi);
    const int32_t a = corner(q, lo), b = corner(q, mid), c = corner(q, hi);
    const int32_t e1 = te[6 * (int64_t)t + pair_index(lo, mid)];
    const int32_t e2 = te[6 * (int64_t)t + pair_index(lo, hi)];
    int32_t best = INF;
    nmatch = 0;
    if (e1 < 0 || e1 >= E || e2 < 0 || e2 >= E) return best;
    int64_t i = et_off[e1], ie = et_off[e1 + 1], j = et_off[e2], je = et_off[e2 + 1];
    if (ie - i <= FF_ROW && je - j <= FF_ROW) {
        // short rows: both are loaded at once and intersected in registers,
        // and the cells they share are gathered together, so the slot costs
        // two dependent loads instead of one per row element
        const int na = (int)(ie - i), nb = (int)(je - j);
        int32_t ra[FF_ROW], rb[FF_ROW];
#pragma unroll
        for (int k = 0; k < FF_ROW; k++) {
            ra[k] = k < na ? et[i + k] : 0;
            rb[k] = k < nb ? et[j + k] : 0;
        }
        bool hit[FF_ROW];
        int4 r[FF_ROW];
#pragma unroll
        for (int k = 0; k < FF_ROW; k++) {
            bool h = false;
#pragma unroll
            for (int l = 0; l < FF_ROW; l++) h = h || (l < nb && rb[l] == ra[k]);
            hit[k] = k < na && h;
            if (hit[k] && (ra[k] < 0 || ra[k] >= T)) return INF;
        }
#pragma unroll
        for (int k = 0; k < FF_ROW; k++) r[k] = hit[k] ? tv4[ra[k]] : make_int4(-1, -1, -1, -1);
#pragma unroll
        for (int k = 0; k < FF_ROW; k++) {
            if (!hit[k]) continue;
            for (int s2 = 0; s2 < 4; s2++) {
                int l2, m2, h2;
                face_pos(s2, l2, m2, h2);
                if (corner(r[k], l2) == a && corner(r[k], m2) == b && corner(r[k], h2) == c) {
                    if (tets2 && nmatch == 0) tets2[0] = ra[k];
                    if (tets2 && nmatch == 1) tets2[1] = ra[k];
                    nmatch++;
                    best = min(best, 4 * ra[k] + s2);
                    break;
                }
            }
        }
        return best;
    }
    while (i < ie && j < je) {
        const int32_t x = et[i], y = et[j];
        if (x < y) i++;
        else if (y < x) j++;
        else if (x < 0 || x >= T) return INF;
        else {
            const int4 r = tv4[x];
            for (int s2 = 0; s2 < 4; s2++) {
                int l2, m2, h2;
                face_pos(s2, l2, m2, h2);
                if (corner(r, l2) == a && corner(r, m2) == b && corner(r, h2) == c) {
                    if (nmatch < 2 && tets2) tets2[nmatch] = x;
                    nmatch++;
                    best = min(best, 4 * x + s2);
                    break;
                }
            }
            i++;
            j++;
        }
    }
    return best;
}

// Per slot position p = 4t + s: the first position of its face, and the
// other cell holding it (-1 if none), so FT needs no second match.  A face
// held by more than two cells sets fterr.
__global__ void k_face_first(const int4 *__restrict__ tv4, int64_t T, const int32_t *__restrict__ te,
                             int64_t E, const int64_t *__restrict__ et_off, const int32_t *__restrict__ et,
                             int32_t *__restrict__ ffirst, uint8_t *__restrict__ flags,
                             int32_t *__restrict__ other, int32_t *__restrict__ err,
                             int32_t *__restrict__ fterr) {
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < 4 * T;
         p += (int64_t)gridDim.x * blockDim.x) {
        int32_t nm, two[2] = {-1, -1};
        const int32_t t = (int32_t)(p >> 2);
        const int32_t f = face_first(tv4, T, te, E, et_off, et, t, (int)(p & 3), nm, two);
        // the cell itself always matches; no match means ET and TE disagree
        const bool bad = f > (int32_t)p;
        if (bad) *err = 1;
        if (nm > 2) *fterr = 1;  // every writer stores the same value
        ffirst[p] = bad ? (int32_t)p : f;
        flags[p] = bad || f == (int32_t)p;
        other[p] = nm >= 2 ? (two[0] == t ? two[1] : two[0]) : -1;
    }
}

// TF; FV as (mid, hi, lo) -- the fields (middleVert, highVert, low vertex);
// FT (<= 2 tets, ascending, -1 pad)
__global__ void k_face_ids(const int4 *__restrict__ tv4, int64_t T,
                           const int32_t *__restrict__ ffirst, const int32_t *__restrict__ other,
                           const uint4 *__restrict__ rank, int32_t *__restrict__ tf,
                           int32_t *__restrict__ fv, int32_t *__restrict__ ft) {
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < 4 * T;
         p += (int64_t)gridDim.x * blockDim.x) {
        const int32_t f = ffirst[p];
        const int32_t id = rank_of(rank, f);
        tf[p] = id;
        if (f != (int32_t)p) continue;
        const int32_t t = (int32_t)(p >> 2);
        const int s = (int)(p & 3);
        const int4 q = tv4[t];
        int lo, mid, hi;
        face_pos(s, lo, mid, hi);
        fv[3 * (int64_t)id] = corner(q, mid);
        fv[3 * (int64_t)id + 1] = corner(q, hi);
        fv[3 * (int64_t)id + 2] = corner(q, lo);
        // the first position's cell is the smallest holding the face
        ft[2 * (int64_t)id] = t;
        ft[2 * (int64_t)id + 1] = other[p];
    }
}

// FE[f] = {max vertex, edge id} for the edges (lo,mid), (lo,hi), (mid,hi),
// read from TE of the face's first cell (FT[f][0]) at the slot whose
// positional triple is the face's.
__global__ void k_fe(const int4 *__restrict__ tv4, const int32_t *__restrict__ fv, int64_t F,
                     const int32_t *__restrict__ ft, const int32_t *__restrict__ te,
                     int32_t *__restrict__ fe) {
    for (int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; f < F;
         f += (int64_t)gridDim.x * blockDim.x) {
        const int32_t mid = fv[3 * f], hi = fv[3 * f + 1], lo = fv[3 * f + 2];
        const int32_t t = ft[2 * f];
        if (t < 0) {  // not reached for a built FT: every face has a first cell
            for (int k = 0; k < 6; k++) fe[6 * f + k] = -1;
            continue;
        }
        const int4 q = tv4[t];
        int s = 0;
        for (int k = 0; k < 4; k++) {
            int l, m, h;
            face_pos(k, l, m, h);
            if (corner(q, l) == lo && corner(q, m) == mid && corner(q, h) == hi) {
                s = k;
                break;
            }
        }
        int pl, pm, ph;
        face_pos(s, pl, pm, ph);
        const int32_t *tr = te + 6 * (int64_t)t;
        fe[6 * f] = max(lo, mid);
        fe[6 * f + 1] = tr[pair_index(pl, pm)];
        fe[6 * f + 2] = max(lo, hi);
        fe[6 * f + 3] = tr[pair_index(pl, ph)];
        fe[6 * f + 4] = max(mid, hi);
        fe[6 * f + 5] = tr[pair_index(pm, ph)];
    }
}

// insert x into the ascending row[0..m) unless present
__device__ __forceinline__ void insert_sorted(int32_t *row, int64_t &m, int32_t x) {
    int64_t i = m;
    while (i > 0 && row[i - 1] > x) i--;
    if (i > 0 && row[i - 1] == x) return;
    for (int64_t k = m; k > i; k--) row[k] = row[k - 1];
    row[i] = x;
    m++;
}

// ---- joins of a few short sorted rows: TT, ET and EE -------------------------------
// TT(t): union of the VT rows of t's corners, minus t.  ET(e): intersection of
// the VT rows of e's ends.  EE(e): union of its ends' edge-id rows, minus e.
// One lane per output row, one kernel: the lane's rows are loaded whole
// (16-byte quads, independent) into registers, merged by a compile-time
// bitonic network, and what the join keeps is counted; the block's total joins
// a chained scan over tiles of rows, which gives every row its exact place;
// then the rows go through an LDS window per wave to contiguous 16-byte stores.
// A wave takes the smallest network that holds its rows; what has a row beyond
// the largest one is left to LongRows' ways.
//
// What bounds it: the gathers of NR x 64 different rows per wave (TT: 4 rows of
// 96 bytes a cell, 2.0 M cells in random order 0.65 ms) and VALU issue of the
// network (560 compare-exchanges for four rows of 24).  It replaced a merge of
// LDS columns by one lane each (26-32 KB a wave, waiting on dependent LDS
// reads; longer rows from global memory), which wrote padded rows, scanned
// their lengths and packed them (TT 2.71 ms).
constexpr int JOIN_ROW = 48;  // longest row of the largest network
enum Join { UNION_LESS_SELF, INTERSECT };
// Outputs with a source row beyond JOIN_ROW: there are none, or a wave each
// joins them in launches of their own, before the main one (their lengths) and
// after it (their values; it leaves them out).
enum LongRows { NO_LONG, LISTED };

// Tiles' totals as they become known: bits 62-63 hold 0 (nothing yet), 1 (the
// tile's own sum) or 2 (the sum of all tiles up to it).
constexpr uint64_t TILE_SUM = 1ull << 62, TILE_PREFIX = 2ull << 62, TILE_VALUE = TILE_SUM - 1;

// Sum of the tiles before `tile`, by one whole wave.  Every tile with a lower
// number was started earlier (numbers are handed out by a counter) and
// publishes its sum without waiting for anything, so the wait ends.
__device__ __forceinline__ int64_t tiles_before(const uint64_t *state, int32_t tile) {
    const int lane = __lane_id();
    int64_t sum = 0;
    for (int32_t top = tile - 1;;) {
        const int32_t i = top - lane;
        const uint64_t s = i >= 0 ? tgd::load_agent(state + i) : TILE_PREFIX;
        const uint64_t full = __ballot((s >> 62) == 2), none = __ballot((s >> 62) == 0);
        const int stop = full ? __ffsll((unsigned long long)full) - 1 : 63;
        if (none & ((2ull << stop) - 1ull)) {
            tgd::pause();
            continue;
        }
        sum += tgd::wave_sum(lane <= stop ? (int64_t)(s & TILE_VALUE) : (int64_t)0);
        if (full) return sum;
        top -= 64;
    }
}

// Row of n <= R words, shifted right by SH, INF after them; DOWN: in reverse.
// Whole quads are read, up to three words past the row (the source arrays
// carry them).
template <int B, int R, bool DOWN, int SH, int N>
__device__ __forceinline__ void load_row(int32_t (&k)[N], const int32_t *__restrict__ src, int n) {
#pragma unroll
    for (int i = 0; i < R; i += 4) {
        i32x4u q = {0, 0, 0, 0};
        if (i < n) q = *reinterpret_cast<const i32x4u *>(src + i);
#pragma unroll
        for (int j = 0; j < 4; j++)
            k[B + (DOWN ? R - 1 - i - j : i + j)] = i + j < n ? q[j] >> SH : INF;
    }
}

template <int NR>
struct Rows {  // the lane's rows
    int32_t p[NR], n[NR];
    __device__ __forceinline__ int longest() const {
        int m = 0;
#pragma unroll
        for (int c = 0; c < NR; c++) m = max(m, n[c]);
        return m;
    }
};

// Block of one kernel: its threads and the words of a wave's output window.
template <int THREADS, int WIN>
struct JoinBlock {
    int32_t win[THREADS / 64][WIN];
    int32_t wtot[THREADS / 64];
    int64_t base;
    int32_t tile;
};

// One wave's share of a tile with a network for rows of up to R entries.
// Contains two workgroup barriers; every wave of the block makes one call
// (of some R), so all waves meet at both.  (The waves may be at calls in
// different branches: gfx950's barrier counts arrivals, whatever instruction
// they come from.)
template <int NR, Join J, int SH, LongRows L, int R, int THREADS, int WIN>
__device__ __forceinline__ void join_wave(JoinBlock<THREADS, WIN> &blk,
                                          const int32_t *__restrict__ src, const Rows<NR> &r,
                                          int64_t rows, int32_t mlong, uint64_t *state,
                                          int64_t *__restrict__ off, int32_t *__restrict__ out) {
    static_assert(NR == 2 || NR == 4, "merge tree");
    constexpr int N = NR * R;
    const int lane = __lane_id(), wid = threadIdx.x / 64;
    // uniform values are made scalars: the keys take nearly all vector registers
    const int32_t tile = tgd::lane_value(blk.tile, 0);
    const int64_t row = (int64_t)tile * THREADS + threadIdx.x;
    const int32_t self = (int32_t)row;
    int32_t *win = blk.win[wid];
    // outputs with a row beyond the largest network: mlong values each, left
    // out of the window
    const bool is_long = L != NO_LONG && r.longest() > JOIN_ROW;
    const uint64_t longs = L != NO_LONG ? __ballot(is_long) : 0;
    int32_t k[N], n[NR];
    int nv = 0;
#pragma unroll
    for (int c = 0; c < NR; c++) {
        n[c] = is_long ? 0 : r.n[c];
        nv += n[c];
    }
    if constexpr (NR == 4) {
        load_row<0, R, false, SH>(k, src + r.p[0], n[0]);
        load_row<R, R, true, SH>(k, src + r.p[1], n[1]);
        load_row<2 * R, R, true, SH>(k, src + r.p[2], n[2]);
        load_row<3 * R, R, false, SH>(k, src + r.p[3], n[3]);
        tgn::bitonic_merge<0, 2 * R, false>(k);
        tgn::bitonic_merge<2 * R, 2 * R, true>(k);
    } else {
        load_row<0, R, true, SH>(k, src + r.p[0], n[0]);
        load_row<R, R, false, SH>(k, src + r.p[1], n[1]);
    }
    tgn::bitonic_merge<0, N, true>(k);
    int32_t m = 0;  // distinct values, less the lane's own and the padding; or equal pairs
#pragma unroll
    for (int j = 1; j < N; j++) m += J == INTERSECT ? k[j] == k[j - 1] : k[j] != k[j - 1];
    m -= J == INTERSECT ? max(N - nv - 1, 0) : (int)(nv < N);
    if (row >= rows || is_long) m = 0;
    // places of the lane's values in the wave's window and in the wave's output
    if (!is_long) mlong = 0;
    const int32_t winc = tgd::wave_inclusive_sum(m);
    const int32_t inc = longs ? tgd::wave_inclusive_sum(m + mlong) : winc;
    if (lane == 63) blk.wtot[wid] = inc;
    __syncthreads();
    int32_t before = 0, total = 0;
#pragma unroll
    for (int i = 0; i < THREADS / 64; i++) {
        if (i < wid) before += blk.wtot[i];
        total += blk.wtot[i];
    }
    before = tgd::lane_value(before, 0);
    total = tgd::lane_value(total, 0);
    if (threadIdx.x == 0) tgd::store_agent(state + tile, TILE_SUM | (uint64_t)total);
    const int32_t first = inc - m - mlong, wfirst = winc - m;
    const int32_t wn = tgd::lane_value(winc, 63);
    // the wave's rows, one window after the other; the first one is filled
    // while the tile's place is being found
    for (int32_t w0 = 0;; w0 += WIN) {
        int32_t pos = wfirst - w0 - 1;
        // compared afresh in every window: masks kept from the count
        // above, one per key, would not fit the scalar registers
        const int32_t mv = tgd::opaque(nv);
        int32_t prev = -1;
#pragma unroll
        for (int j = 0; j < N; j++) {
            k[j] = tgd::opaque(k[j]);
            const bool keep = (J == INTERSECT ? k[j] == prev : k[j] != prev && k[j] != self) && j < mv;
            prev = k[j];
            pos += keep;
            if (keep && (uint32_t)pos < (uint32_t)WIN) win[pos] = k[j];
        }
        if (w0 == 0) {
            if (wid == 0) {
                const int64_t b = tiles_before(state, tile);
                if (lane == 0) {
                    tgd::store_agent(state + tile, TILE_PREFIX | (uint64_t)(b + total));
                    blk.base = b;
                }
            }
            __syncthreads();
            if (row < rows) off[row] = blk.base + before + first;
            if (row == rows - 1) off[rows] = blk.base + total;
        }
        tgd::wave_sync();  // the window is whole
        // words [from, to) of the windows' sequence, of which the output has
        // `shift` more before them
        auto copy = [&](int32_t from, int32_t to, int32_t shift) {
            const int32_t a = max(from - w0, 0), b = min(to - w0, WIN);
            int32_t *dst = out + (blk.base + before + w0 + shift);
            for (int32_t i = a + 4 * lane; i + 3 < b; i += 256)
                *reinterpret_cast<i32x4u *>(dst + i) = *reinterpret_cast<const i32x4u *>(win + i);
            const int32_t tail = a + ((b - a) & ~3);
            if (a < b && tail + lane < b) dst[tail + lane] = win[tail + lane];
        };
        int32_t from = 0, shift = 0;
        for (uint64_t b = longs; b; b &= b - 1) {  // the rows between the long ones
            const int l = __ffsll((unsigned long long)b) - 1;
            const int32_t to = tgd::lane_value(wfirst, l);
            copy(from, to, tgd::lane_value(first, l) - to);
            from = to;
            shift = tgd::lane_value(inc, l) - to;
        }
        copy(from, wn, shift);
        if (w0 + WIN >= wn) break;
        tgd::wave_sync();  // and has been read
    }
}

// This block's tile number, handed out in the order blocks start.
__device__ __forceinline__ int32_t take_tile(int32_t *ticket, int32_t &shared) {
    if (threadIdx.x == 0) shared = atomicAdd(ticket, 1);
    __syncthreads();
    return shared;
}

// The rows that an output joins.  TT: the VT rows of a cell's corners.
struct CellRows {
    const int4 *__restrict__ tv4;
    const int32_t *__restrict__ vt_off;
    __device__ __forceinline__ Rows<4> operator()(int64_t t, bool act) const {
        Rows<4> r;
        const int4 q = act ? tv4[t] : make_int4(0, 0, 0, 0);
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const i32x2u o = *reinterpret_cast<const i32x2u *>(vt_off + corner(q, c));
            r.p[c] = o.x;
            r.n[c] = act ? o.y - o.x : 0;
        }
        return r;
    }
};
// ET and EE: the rows of an edge's ends (corner codes by vt_off, or edge ids
// by vv_off).
struct EdgeRows {
    const int32_t *__restrict__ ev;
    int64_t V;
    const int32_t *__restrict__ row_off;
    __device__ __forceinline__ Rows<2> operator()(int64_t e, bool act) const {
        Rows<2> r;
        const int2 ends = act ? reinterpret_cast<const int2 *>(ev)[e] : make_int2(0, 0);
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int32_t v = c ? ends.y : ends.x;
            const bool ok = v >= 0 && v < V;  // always, for a built EV
            const i32x2u o = *reinterpret_cast<const i32x2u *>(row_off + (ok ? v : 0));
            r.p[c] = o.x;
            r.n[c] = act && ok ? o.y - o.x : 0;
        }
        return r;
    }
};

// Window: what two blocks per CU (as many as the registers allow) leave of
// the LDS; one window for 64 x 69 words (two windows of 2240: 0.76 ms at 2.0 M
// split cells, one 0.65).
constexpr int TT_THREADS = 256, TT_WIN = 5088;
template <LongRows L>
__global__ __launch_bounds__(TT_THREADS, 2) void k_tt(const CellRows rows_of, int64_t T,
                                                      const int32_t *__restrict__ vtc,
                                                      const int32_t *__restrict__ long_len,
                                                      int32_t *ticket, uint64_t *state,
                                                      int64_t *__restrict__ off,
                                                      int32_t *__restrict__ out) {
    __shared__ __align__(16) JoinBlock<TT_THREADS, TT_WIN> blk;
    const int64_t t = (int64_t)take_tile(ticket, blk.tile) * TT_THREADS + threadIdx.x;
    const bool act = t < T;
    const Rows<4> r = rows_of(t, act);
    const bool is_long = L != NO_LONG && r.longest() > JOIN_ROW;
    const int32_t mlong = is_long ? long_len[t] : 0;
    const int need = is_long ? 0 : r.longest();
#define TG_JOIN(R)                                                                              \
    join_wave<4, UNION_LESS_SELF, 2, L, R>(blk, vtc, r, T, mlong, state, off, out)
    if (__any(need > 40)) TG_JOIN(JOIN_ROW);
    else if (__any(need > 32)) TG_JOIN(40);
    else if (__any(need > 24)) TG_JOIN(32);
    else TG_JOIN(24);
#undef TG_JOIN
}

// 512 edges a tile: tile numbers cost 10 ns each.  Windows: one for ET (64 x 5
// words), one for EE (64 x 26).
constexpr int EJ_THREADS = 512;
template <Join J, int SH, LongRows L, int WIN>
__global__ __launch_bounds__(EJ_THREADS, 4) void k_edge_join(const EdgeRows rows_of, int64_t E,
                                                             const int32_t *__restrict__ src,
                                                             const int32_t *__restrict__ long_len,
                                                             int32_t *ticket, uint64_t *state,
                                                             int64_t *__restrict__ off,
                                                             int32_t *__restrict__ out) {
    __shared__ __align__(16) JoinBlock<EJ_THREADS, WIN> blk;
    const int64_t e = (int64_t)take_tile(ticket, blk.tile) * EJ_THREADS + threadIdx.x;
    const bool act = e < E;
    const Rows<2> r = rows_of(e, act);
    const bool is_long = L != NO_LONG && r.longest() > JOIN_ROW;
    // EE: the ends' rows share only the edge itself
    const int32_t mlong = !is_long ? 0 : J == INTERSECT ? long_len[e] : r.n[0] + r.n[1] - 2;
    const int need = is_long ? 0 : r.longest();
#define TG_JOIN(R) join_wave<2, J, SH, L, R>(blk, src, r, E, mlong, state, off, out)
    if (__any(need > 32)) TG_JOIN(JOIN_ROW);
    else if (__any(need > 24)) TG_JOIN(32);
    else if (__any(need > 16)) TG_JOIN(24);
    else TG_JOIN(16);
#undef TG_JOIN
}
constexpr int ET_WIN = 448, EE_WIN = 1728;

// Outputs with a row beyond JOIN_ROW, in any order; n has to start at 0.
constexpr int LIST_THREADS = 256;
template <typename RO>
__global__ __launch_bounds__(LIST_THREADS) void k_list_long(const RO rows_of, int64_t count,
                                                            int32_t *__restrict__ list,
                                                            int32_t *__restrict__ n) {
    const int lane = __lane_id();
    const int64_t step = (int64_t)gridDim.x * LIST_THREADS;
    for (int64_t b = (int64_t)blockIdx.x * LIST_THREADS; b < count; b += step) {
        const int64_t i = b + threadIdx.x;
        const bool is_long = rows_of(i, i < count).longest() > JOIN_ROW;
        const uint64_t m = __ballot(is_long);
        if (!m) continue;
        int32_t at = 0;
        if (lane == 0) at = atomicAdd(n, (int32_t)__popcll(m));
        at = tgd::lane_value(at, 0) + (int32_t)__popcll(m & ((1ull << lane) - 1ull));
        if (is_long) list[at] = (int32_t)i;
    }
}

// Union of the rows at at[c] .. end[c], less `self`, which every row holds, by
// one wave: returns the number of values and, with WRITE, leaves them at out,
// ascending.  A step takes 64 / NR entries of each row; those up to the
// smallest of the rows' last ones taken are sorted across the wave and
// consumed, so equal entries meet in one step.  Where one row alone has entries
// before the others' next ones, the stretch is found by a 64-way search and
// copied whole.
template <int NR, int SH, bool WRITE>
__device__ __forceinline__ int32_t union_by_wave(const int32_t *__restrict__ src, int32_t (&at)[NR],
                                                 const int32_t (&end)[NR], int32_t self,
                                                 int32_t *__restrict__ out) {
    static_assert(NR == 2 || NR == 4, "merge of halves");
    constexpr int W = 64 / NR;
    const int lane = __lane_id(), row = lane / W, j = lane % W;
    int32_t m = 0;
    while (true) {
        int32_t i = at[0], e = end[0];
#pragma unroll
        for (int c = 1; c < NR; c++) {
            i = row == c ? at[c] : i;
            e = row == c ? end[c] : e;
        }
        int32_t x = j < e - i ? src[i + j] >> SH : INF;
        int32_t head[NR], last[NR], limit = INF;
        int a = 0;  // the row with the smallest entry
#pragma unroll
        for (int c = 0; c < NR; c++) {
            head[c] = tgd::lane_value(x, W * c);
            last[c] = tgd::lane_value(x, W * c + W - 1);
            limit = min(limit, last[c]);
            if (c > 0 && head[c] < head[0]) head[0] = head[c], a = c;
        }
        if (head[0] == INF) return m;
        int32_t lo = 0, hi = 0, la = 0, others = INF;
#pragma unroll
        for (int c = 0; c < NR; c++) {
            if (c == a) lo = at[c], hi = end[c], la = last[c];
            else others = min(others, tgd::lane_value(x, W * c));
        }
        if (la < others) {  // a stretch of row a alone: [from, lo) when found
            const int32_t from = lo;
            lo += W;
            if (others == INF) lo = hi;
            while (lo < hi) {
                const int32_t step = (hi - lo + 63) / 64, p = lo + lane * step;
                const int32_t below = (int32_t)__popcll(__ballot(p < hi && src[p] >> SH < others));
                if (below == 0) break;
                hi = min(hi, lo + below * step);
                lo += (below - 1) * step + 1;
            }
            if (WRITE) {
                constexpr int U = 4;
                const int32_t n = lo - from;
                for (int32_t k = lane; k < n; k += 64 * U) {
                    int32_t y[U];
#pragma unroll
                    for (int u = 0; u < U; u++)
                        y[u] = k + 64 * u < n ? src[from + k + 64 * u] >> SH : 0;
#pragma unroll
                    for (int u = 0; u < U; u++)
                        if (k + 64 * u < n) out[m + k + 64 * u] = y[u];
                }
            }
            m += lo - from;
#pragma unroll
            for (int c = 0; c < NR; c++)
                if (c == a) at[c] = lo;
            continue;
        }
        const uint64_t taken = __ballot(x <= limit && x != INF);
        if (x > limit) x = INF;
#pragma unroll
        for (int w = 2 * W; w <= 64; w *= 2) {  // merge sorted halves of w lanes
#pragma unroll
            for (int d = w - 1; d >= 1; d = d == w - 1 ? w / 4 : d / 2) {
                const int32_t y = __shfl_xor(x, d, 64);
                // d = w - 1: partners are mirrored, the upper half keeps the larger
                const bool upper = lane & (d == w - 1 ? w / 2 : d);
                x = upper ? max(x, y) : min(x, y);
            }
        }
        const int32_t y = __shfl_up(x, 1, 64);
        const bool keep = x != INF && x != self && (lane == 0 || x != y);
        const uint64_t kept = __ballot(keep);
        if (WRITE && keep) out[m + (int32_t)__popcll(kept & ((1ull << lane) - 1ull))] = x;
        m += (int32_t)__popcll(kept);
#pragma unroll
        for (int c = 0; c < NR; c++)
            at[c] += (int32_t)__popcll(taken & ((W == 32 ? 0xFFFFFFFFull : 0xFFFFull) << (W * c)));
    }
}

// Intersection of two rows by one wave, as union_by_wave: the lanes search the
// longer row for the shorter one's entries.
template <int SH, bool WRITE>
__device__ __forceinline__ int32_t intersect_by_wave(const int32_t *__restrict__ src,
                                                     const int32_t (&at)[2], const int32_t (&end)[2],
                                                     int32_t *__restrict__ out) {
    const int lane = __lane_id();
    const int32_t n0 = end[0] - at[0], n1 = end[1] - at[1];
    const int32_t *a = src + (n0 <= n1 ? at[0] : at[1]), *b = src + (n0 <= n1 ? at[1] : at[0]);
    const int32_t na = min(n0, n1), nb = max(n0, n1);
    int32_t m = 0;
    for (int32_t i0 = 0; i0 < na; i0 += 64) {
        const int32_t x = i0 + lane < na ? a[i0 + lane] >> SH : INF;
        int32_t lo = 0, hi = nb;
        while (lo < hi) {
            const int32_t mid = (lo + hi) >> 1;
            if (b[mid] >> SH < x) lo = mid + 1;
            else hi = mid;
        }
        const bool keep = lo < nb && b[lo] >> SH == x;
        const uint64_t kept = __ballot(keep);
        if (WRITE && keep) out[m + (int32_t)__popcll(kept & ((1ull << lane) - 1ull))] = x;
        m += (int32_t)__popcll(kept);
    }
    return m;
}

// The listed outputs, a wave each: their lengths, or (WRITE) their values at
// the places that the main launch gave them.  Bound by chains of dependent
// loads, some ten a row, of which 8192 waves keep as many in flight; a lane each
// in the main launch walked a chain of a row's length once more for every window
// of its wave's output.  TT of 100 k cells, 12 % with a row beyond 48: 2620 ->
// 165 us (one lane's single merge, the rows packed afterwards: 660); of 4000
// cells around one vertex 53 -> 0.09 ms (2.3).  ET of 293 k cells around 32
// vertices of up to 2000: 2.96 -> 0.19 ms (1.26).  The list and the lengths are
// an extra pass over the outputs, so meshes without long rows leave them out.
constexpr int LONG_THREADS = 256, LONG_BLOCKS = 2048;
template <int NR, Join J, int SH, bool WRITE, typename RO>
__global__ __launch_bounds__(LONG_THREADS) void k_join_long(const RO rows_of,
                                                            const int32_t *__restrict__ src,
                                                            const int32_t *__restrict__ list,
                                                            const int32_t *__restrict__ n,
                                                            int32_t *__restrict__ len,
                                                            const int64_t *__restrict__ off,
                                                            int32_t *__restrict__ out) {
    const int32_t count = *n, waves = (int32_t)gridDim.x * (LONG_THREADS / 64);
    const int lane = __lane_id();
    for (int32_t i = (int32_t)blockIdx.x * (LONG_THREADS / 64) + threadIdx.x / 64; i < count; i += waves) {
        const int32_t id = tgd::lane_value(list[i], 0);
        const Rows<NR> r = rows_of(id, true);
        int32_t at[NR], end[NR];
#pragma unroll
        for (int c = 0; c < NR; c++) {
            at[c] = tgd::lane_value(r.p[c], 0);
            end[c] = at[c] + tgd::lane_value(r.n[c], 0);
        }
        int32_t *to = WRITE ? out + off[id] : nullptr;
        int32_t m;
        if constexpr (J == INTERSECT) m = intersect_by_wave<SH, WRITE>(src, at, end, to);
        else m = union_by_wave<NR, SH, WRITE>(src, at, end, id, to);
        if (!WRITE && lane == 0) len[id] = m;
    }
}

// EF(e): faces holding e, from the two faces of e in each cell of ET(e).  One
// lane per edge builds its sorted, duplicate-free row in an LDS column (in a
// padded slot of 2|ET(e)| words of tmp where the column is too short: by the
// wave up to 64 cells, then by the block), the block's total joins the chained scan, and the row goes to its place.  Bound
// by the lines that the gathers of ET's cells move: one a cell, from rows that
// hold its corners and faces together (TE and TF, a line each: 468 us at 2.2 M
// cells, this 303 and 25 to lay the rows out).
constexpr int EF_THREADS = 256, EF_CAP = 32;  // 32 KB a block

// Each cell's corners and faces in 32 bytes, for k_ef's gathers.
__global__ void k_cell_faces(const int4 *__restrict__ tv4, const int4 *__restrict__ tf4, int64_t T,
                             int4 *__restrict__ rows) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < 2 * T;
         i += (int64_t)gridDim.x * blockDim.x)
        rows[i] = i & 1 ? tf4[i >> 1] : tv4[i >> 1];
}

__global__ __launch_bounds__(EF_THREADS) void k_ef(const int64_t *__restrict__ et_off,
                                                   int64_t E, const int32_t *__restrict__ et,
                                                   const int2 *__restrict__ ev,
                                                   const int4 *__restrict__ rows,
                                                   int32_t *ticket, uint64_t *state,
                                                   int64_t *__restrict__ off,
                                                   int32_t *__restrict__ out,
                                                   int32_t *__restrict__ tmp) {
    __shared__ int32_t col[EF_CAP][EF_THREADS];
    __shared__ int32_t wtot[EF_THREADS / 64];
    __shared__ int32_t shared_tile, nlong, lng[EF_THREADS];
    __shared__ int64_t base;
    __shared__ struct { int64_t first; int32_t n, lo, hi; } one;
    const int tid = threadIdx.x, lane = __lane_id(), wid = tid / 64;
    const int32_t tile = take_tile(ticket, shared_tile);
    const int64_t e = (int64_t)tile * EF_THREADS + tid;
    const bool act = e < E;
    const int64_t b0 = act ? et_off[e] : 0, b1 = act ? et_off[e + 1] : 0;
    const bool lds = 2 * (b1 - b0) <= EF_CAP, by_wave = !lds && b1 - b0 <= 64;
    int32_t *grow = tmp + 2 * b0;
    int64_t m = 0;
    const int2 lh = act ? ev[e] : make_int2(-1, -1);
    // the two faces of a cell that hold the edge (lo, hi), from its row; false:
    // ET disagrees, no face of this cell
    auto faces = [](const int4 q, const int4 fr, int32_t lo, int32_t hi, int32_t (&x)[2]) {
        uint32_t apart = 0;  // corners that the edge does not have
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int32_t u = corner(q, j);
            apart |= (uint32_t)(u != lo && u != hi) << j;
        }
        if (__popc(apart) != 2) return false;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            // face slot 3 - j leaves out corner j
            const int s = 3 - (h ? 31 - __clz(apart) : __ffs(apart) - 1);
            x[h] = s == 0 ? fr.x : s == 1 ? fr.y : s == 2 ? fr.z : fr.w;
        }
        return true;
    };
    // the longest rows: sorted by the block in the columns' LDS
    const bool by_block = b1 - b0 > 64 && 2 * (b1 - b0) <= EF_CAP * EF_THREADS;
    if (!__syncthreads_and(!by_block)) {
        if (tid == 0) nlong = 0;
        __syncthreads();
        if (by_block) lng[atomicAdd(&nlong, 1)] = tid;
        __syncthreads();
        int32_t *key = &col[0][0];
        for (int r = 0; r < nlong; r++) {
            if (tid == lng[r]) {
                one.first = b0;
                one.n = (int32_t)(b1 - b0);
                one.lo = lh.x;
                one.hi = lh.y;
            }
            __syncthreads();
            int32_t size = 256;
            while (size < 2 * one.n) size *= 2;
            for (int32_t i = tid; i < size / 2; i += EF_THREADS) {
                int32_t x[2] = {INF, INF};
                if (i < one.n) {
                    const int64_t t = et[one.first + i];
                    if (!faces(rows[2 * t], rows[2 * t + 1], one.lo, one.hi, x)) x[0] = x[1] = INF;
                }
                key[2 * i] = x[0];
                key[2 * i + 1] = x[1];
            }
            __syncthreads();
            sort_by_block<EF_THREADS>(key, size);
            int32_t kept = 0;  // each face once
            for (int32_t i0 = 0; i0 < size; i0 += EF_THREADS) {
                const int32_t i = i0 + tid, x = key[i];
                const bool keep = x != INF && (i == 0 || key[i - 1] != x);
                const uint64_t mask = __ballot(keep);
                if (lane == 0) wtot[wid] = (int32_t)__popcll(mask);
                __syncthreads();
                int32_t place = kept + (int32_t)__popcll(mask & ((1ull << lane) - 1ull));
#pragma unroll
                for (int w = 0; w < EF_THREADS / 64; w++) {
                    if (w < wid) place += wtot[w];
                    kept += wtot[w];
                }
                if (keep) tmp[2 * one.first + place] = x;
                __syncthreads();
            }
            if (tid == lng[r]) m = kept;
        }
    }
    // four cells at a time, their rows loaded together (unconditional loads
    // from a clamped cell index)
    for (int64_t i0 = b0; i0 < (by_wave || by_block ? b0 : b1); i0 += 4) {
        int32_t tc[4];
        int4 q[4], fr[4];
#pragma unroll
        for (int c = 0; c < 4; c++) tc[c] = et[min(i0 + c, b1 - 1)];
#pragma unroll
        for (int c = 0; c < 4; c++) {
            q[c] = rows[2 * (int64_t)tc[c]];
            fr[c] = rows[2 * (int64_t)tc[c] + 1];
        }
#pragma unroll
        for (int c = 0; c < 4; c++) {
            if (i0 + c >= b1) break;
            int32_t two[2];
            if (!faces(q[c], fr[c], lh.x, lh.y, two)) continue;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int32_t x = two[h];
                if (lds) {  // insert into the ascending column unless present
                    int p = (int)m;
                    while (p > 0 && col[p - 1][tid] > x) p--;
                    if (p > 0 && col[p - 1][tid] == x) continue;
                    for (int q = (int)m; q > p; q--) col[q][tid] = col[q - 1][tid];
                    col[p][tid] = x;
                    m++;
                } else {
                    insert_sorted(grow, m, x);
                }
            }
        }
    }
    // rows beyond the column, of up to 64 cells: a lane per cell, the faces
    // without the repeated ones placed by comparing all pairs
    for (uint64_t b = __ballot(by_wave); b; b &= b - 1) {
        const int l = __ffsll((unsigned long long)b) - 1;
        const int64_t first = __shfl(b0, l, 64);
        const int32_t n = tgd::lane_value((int32_t)(b1 - b0), l);
        const int32_t lo = tgd::lane_value(lh.x, l), hi = tgd::lane_value(lh.y, l);
        int32_t x[2] = {INF, INF};
        if (lane < n) {
            const int64_t t = et[first + lane];
            if (!faces(rows[2 * t], rows[2 * t + 1], lo, hi, x)) x[0] = x[1] = INF;
        }
        bool again[2] = {false, false};  // an earlier cell has the face
        for (int j = 0; j < n; j++) {
            const int32_t y0 = tgd::lane_value(x[0], j), y1 = tgd::lane_value(x[1], j);
#pragma unroll
            for (int h = 0; h < 2; h++) again[h] |= j < lane && (x[h] == y0 || x[h] == y1);
        }
#pragma unroll
        for (int h = 0; h < 2; h++)
            if (again[h]) x[h] = INF;
        int32_t place[2] = {0, 0};
        for (int j = 0; j < n; j++) {
            const int32_t y0 = tgd::lane_value(x[0], j), y1 = tgd::lane_value(x[1], j);
#pragma unroll
            for (int h = 0; h < 2; h++) place[h] += (y0 < x[h]) + (y1 < x[h]);
        }
        int32_t kept = 0;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if (x[h] != INF) tmp[2 * first + place[h]] = x[h];
            kept += (int32_t)__popcll(__ballot(x[h] != INF));
        }
        if (lane == l) m = kept;
    }
    const int32_t inc = tgd::wave_inclusive_sum((int32_t)m);
    if (lane == 63) wtot[wid] = inc;
    __syncthreads();
    int32_t before = 0, total = 0;
#pragma unroll
    for (int i = 0; i < EF_THREADS / 64; i++) {
        if (i < wid) before += wtot[i];
        total += wtot[i];
    }
    if (wid == 0) {
        if (lane == 0) tgd::store_agent(state + tile, TILE_SUM | (uint64_t)total);
        const int64_t b = tiles_before(state, tile);
        if (lane == 0) {
            tgd::store_agent(state + tile, TILE_PREFIX | (uint64_t)(b + total));
            base = b;
        }
    }
    __syncthreads();
    if (!act) return;
    QuadOutExact o;
    const int64_t at = base + before + inc - m;
    o.row = out + at;
    for (int64_t q = 0; q < m; q++) o.put(lds ? col[q][tid] : grow[q]);
    o.flush();
    off[e] = at;
    if (e == E - 1) off[E] = base + total;
}

// VE rows {hi, id}: the upper entries (u > v) of v's VV row, ordered by edge
// id.  An edge's id ranks its first position, and the reference mints the
// ids of v's row in the order v's cells first meet its upper neighbours, so
// ordering by id is the reference's row order.  Lane per vertex: the upper
// entries are counted for the chained scan, their ids looked up and sorted in
// registers, longer rows of them ordered as k_vertex_edges orders its own.
// Bound by the rank lookups: their words are lines of a table that one XCD's
// L2 does not hold.  2.2 M cells: 81 us, 5 M: 202; a count, a scan, the
// ids with EV and a fill by an LDS sort in launches of their own: 142 (with EV's
// 16) and 340 (41).
constexpr int VE_THREADS = 256;

template <int N>
__device__ __forceinline__ void ve_row(const int32_t *__restrict__ vv,
                                       const int32_t *__restrict__ efirst,
                                       const uint4 *__restrict__ rank, int32_t n,
                                       int2 *__restrict__ row) {
    uint64_t k[N];  // (id << 32) | hi
#pragma unroll
    for (int i = 0; i < N; i++) {
        k[i] = ~0ull;
        if (i < n) {
            const int32_t id = rank_at(rank, efirst[i]);
            k[i] = ((uint64_t)(uint32_t)id << 32) | (uint32_t)vv[i];
        }
    }
    tgn::sort_keys(k);
#pragma unroll
    for (int i = 0; i < N; i++)
        if (i < n) row[i] = make_int2((int32_t)(uint32_t)k[i], (int32_t)(k[i] >> 32));
}

__global__ __launch_bounds__(VE_THREADS) void k_ve(const int4 *__restrict__ tv4,
                                                   const int32_t *__restrict__ vv_off,
                                                   const int32_t *__restrict__ vv, int64_t V,
                                                   const int32_t *__restrict__ efirst,
                                                   const uint4 *__restrict__ rank,
                                                   int32_t *ticket, uint64_t *state,
                                                   int32_t *__restrict__ off,
                                                   int2 *__restrict__ out) {
    __shared__ LongRow<VE_THREADS> lng;
    __shared__ int32_t wtot[VE_THREADS / 64];
    __shared__ int32_t shared_tile;
    __shared__ int64_t base;
    const int lane = __lane_id(), wid = threadIdx.x / 64;
    const int32_t tile = take_tile(ticket, shared_tile);
    const int64_t v = (int64_t)tile * VE_THREADS + threadIdx.x;
    const bool act = v < V;
    const int32_t rb = act ? vv_off[v] : 0, re = act ? vv_off[v + 1] : 0;
    int32_t n = 0;  // entries > v: the row is ascending and never holds v
    for (int32_t i0 = rb; i0 < re; i0 += 8) {
        int32_t u[8];
#pragma unroll
        for (int c = 0; c < 8; c++) u[c] = vv[min(i0 + c, re - 1)];
#pragma unroll
        for (int c = 0; c < 8; c++) n += i0 + c < re && u[c] > (int32_t)v;
    }
    const int32_t inc = tgd::wave_inclusive_sum(n);
    if (lane == 63) wtot[wid] = inc;
    __syncthreads();
    int32_t before = 0, total = 0;
#pragma unroll
    for (int i = 0; i < VE_THREADS / 64; i++) {
        if (i < wid) before += wtot[i];
        total += wtot[i];
    }
    if (wid == 0) {
        if (lane == 0) tgd::store_agent(state + tile, TILE_SUM | (uint64_t)total);
        const int64_t b = tiles_before(state, tile);
        if (lane == 0) {
            tgd::store_agent(state + tile, TILE_PREFIX | (uint64_t)(b + total));
            base = b;
        }
    }
    __syncthreads();
    const int32_t at = (int32_t)base + before + inc - n, ub = re - n;  // first upper entry
    if (act) off[v] = at;
    if (v == V - 1) off[V] = (int32_t)base + total;
    int2 *row = out + at;
    const int32_t ns = n <= 32 ? n : 0;
    if (__any(ns > 16)) ve_row<32>(vv + ub, efirst + ub, rank, ns, row);
    else ve_row<16>(vv + ub, efirst + ub, rank, ns, row);
    // longer rows: ids ascend as first positions do; a position names its edge
    order_long_rows(lng, efirst, ub, n, at, [&](int32_t to, int32_t place, int32_t p) {
        const int4 q = tv4[p / 6];
        const int k = p % 6, i = k < 3 ? 0 : k < 5 ? 1 : 2, j = k < 3 ? k + 1 : k < 5 ? k - 1 : 3;
        out[to + place] = make_int2(max(corner(q, i), corner(q, j)), rank_at(rank, p));
    });
}

// VF rows {mid, hi, id}: the row of a holds the faces whose positional low
// vertex is a.  Lane per vertex walks its tets ascending and takes the slots
// where a sits at the low position (corner 0: slots 0-2, corner 1: slot 3) and
// which are their face's first occurrence; positions ascend, so ids ascend.
// Which slots are first occurrences, and their ids, come from the rank units
// (16 bytes for 24 cells, where the first positions and TF are a line per
// cell).  The first walk counts and keeps three bits for each of the first 32
// cells; after the chained scan the second one visits only cells that give a
// face.  2.2 M cells: 0.23 ms; first positions and TF read instead, in this
// kernel or in two with a scan between them, 0.38.  The cells of a vertex with
// more than VF_ROW are the wave's, a lane each (4000 cells around the vertex of
// the lowest id: TF, FV and VF after ET 2.3 -> 0.16 ms).
constexpr int VF_THREADS = 256, VF_ROW = 96;
__global__ __launch_bounds__(VF_THREADS) void k_vf(const int4 *__restrict__ tv4,
                                                   const int32_t *__restrict__ vt_off,
                                                   const int32_t *__restrict__ vtc, int64_t V,
                                                   const uint4 *__restrict__ rank,
                                                   int32_t *ticket,
                                                   uint64_t *state, int32_t *__restrict__ off,
                                                   int32_t *__restrict__ out) {
    __shared__ int32_t wtot[VF_THREADS / 64];
    __shared__ int32_t shared_tile;
    __shared__ int64_t base;
    const int lane = __lane_id(), wid = threadIdx.x / 64;
    const int32_t tile = take_tile(ticket, shared_tile);
    const int64_t a = (int64_t)tile * VF_THREADS + threadIdx.x;
    const bool act = a < V;
    const int32_t kb = act ? vt_off[a] : 0, ke = act ? vt_off[a + 1] : 0;
    // slots of cell code p that are first occurrences with a low: bits 0-2, out
    // of the flags of the cell's rank unit
    constexpr uint32_t CELLS = UNIT / 4;
    auto word = [&](int32_t p) {  // the cell's flags are in one word
        const uint32_t t = (uint32_t)p >> 2, u = t / CELLS;
        return (const uint32_t *)(rank + u) + 1 + (t - CELLS * u) / 8;
    };
    auto firsts = [&](int32_t p, uint32_t bits) -> uint32_t {
        const uint32_t t = (uint32_t)p >> 2, f = bits >> (4 * (t % CELLS % 8));
        return (p & 3) == 0 ? f & 7u : (p & 3) == 1 ? (f >> 3) & 1u : 0u;
    };
    uint32_t m0 = 0, m1 = 0, m2 = 0;  // bit k: the cell's 1st, 2nd, 3rd slot, for the first 32 cells
    int32_t n = 0;
    const bool by_wave = ke - kb > VF_ROW;
    const int32_t le = by_wave ? kb : ke;  // end of the cells that the lane takes
    for (int32_t k0 = kb; k0 < le; k0 += 8) {
        int32_t p[8];
        uint32_t ff[8];
#pragma unroll
        for (int c = 0; c < 8; c++) p[c] = k0 + c < le ? vtc[k0 + c] : 2;
#pragma unroll
        for (int c = 0; c < 8; c++)
            ff[c] = (p[c] & 3) <= 1 ? *word(p[c]) : 0u;
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const uint32_t f = firsts(p[c], ff[c]);
            n += __popc(f);
            if (k0 + c - kb < 32) {
                m0 |= (f & 1u) << ((k0 + c - kb) & 31);
                m1 |= ((f >> 1) & 1u) << ((k0 + c - kb) & 31);
                m2 |= (f >> 2) << ((k0 + c - kb) & 31);
            }
        }
    }
    for (uint64_t b = __ballot(by_wave); b; b &= b - 1) {
        const int l = __ffsll((unsigned long long)b) - 1;
        const int32_t end = tgd::lane_value(ke, l);
        int32_t c = 0;
        for (int32_t k = tgd::lane_value(kb, l) + lane; k < end; k += 64) {
            const int32_t p = vtc[k];
            if ((p & 3) <= 1) c += __popc(firsts(p, *word(p)));
        }
        c = tgd::wave_sum(c);
        if (lane == l) n = c;
    }
    const int32_t inc = tgd::wave_inclusive_sum(n);
    if (lane == 63) wtot[wid] = inc;
    __syncthreads();
    int32_t before = 0, total = 0;
#pragma unroll
    for (int i = 0; i < VF_THREADS / 64; i++) {
        if (i < wid) before += wtot[i];
        total += wtot[i];
    }
    if (wid == 0) {
        if (lane == 0) tgd::store_agent(state + tile, TILE_SUM | (uint64_t)total);
        const int64_t b = tiles_before(state, tile);
        if (lane == 0) {
            tgd::store_agent(state + tile, TILE_PREFIX | (uint64_t)(b + total));
            base = b;
        }
    }
    __syncthreads();
    const int32_t at = (int32_t)base + before + inc - n;
    if (act) off[a] = at;
    if (a == V - 1) off[V] = (int32_t)base + total;
    auto write = [&](int32_t *&row, int32_t p, uint32_t f, const int4 q, const uint4 w) {
#pragma unroll
        for (int m = 0; m < 3; m++) {
            if (!((f >> m) & 1u)) continue;
            const int sl = (p & 3) == 0 ? m : 3;
            int lo, mid, hi;
            face_pos(sl, lo, mid, hi);
            // one 12-byte store per entry
            const int32_t id = rank_in(w, 4 * (((uint32_t)p >> 2) % CELLS) + sl);
            const int32_t ent[3] = {corner(q, mid), corner(q, hi), id};
            __builtin_memcpy(row, ent, sizeof ent);
            row += 3;
        }
    };
    int32_t *row = out + 3 * (int64_t)at;
    uint32_t any = m0 | m1 | m2;
    while (any) {  // eight cells at a time
        int32_t p[8];
        uint32_t f[8];
        int4 q[8];
        uint4 w[8];
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const int k = any ? __ffs(any) - 1 : 0;
            f[c] = any ? ((m0 >> k) & 1u) | ((m1 >> k) & 1u) << 1 | ((m2 >> k) & 1u) << 2 : 0u;
            any &= any - 1u;
            p[c] = vtc[kb + k];
        }
#pragma unroll
        for (int c = 0; c < 8; c++) {
            q[c] = tv4[p[c] >> 2];
            w[c] = rank[((uint32_t)p[c] >> 2) / CELLS];
        }
#pragma unroll
        for (int c = 0; c < 8; c++) write(row, p[c], f[c], q[c], w[c]);
    }
    for (int32_t k = kb + 32; k < le; k++) {
        const int32_t p = vtc[k];
        if ((p & 3) > 1) continue;
        const uint32_t f = firsts(p, *word(p));
        if (f) write(row, p, f, tv4[p >> 2], rank[((uint32_t)p >> 2) / CELLS]);
    }
    for (uint64_t b = __ballot(by_wave); b; b &= b - 1) {
        const int l = __ffsll((unsigned long long)b) - 1;
        const int32_t end = tgd::lane_value(ke, l);
        int32_t done = tgd::lane_value(at, l);
        for (int32_t k0 = tgd::lane_value(kb, l); k0 < end; k0 += 64) {
            const int32_t p = k0 + lane < end ? vtc[k0 + lane] : 2;
            const uint32_t f = (p & 3) <= 1 ? firsts(p, *word(p)) : 0u;
            const int32_t c = tgd::wave_inclusive_sum((int32_t)__popc(f));
            int32_t *to = out + 3 * (int64_t)(done + c - (int32_t)__popc(f));
            if (f) write(to, p, f, tv4[p >> 2], rank[((uint32_t)p >> 2) / CELLS]);
            done += tgd::lane_value(c, 63);
        }
    }
}

// Sum of squared row lengths (VT: the lengths of all cells' four rows
// together) and the longest row; one atomic of each per block of few.
constexpr int SQ_THREADS = 1024, SQ_BLOCKS = 64;
__global__ __launch_bounds__(SQ_THREADS) void k_row_squares(const int32_t *__restrict__ row_off,
                                                            int64_t rows,
                                                            unsigned long long *__restrict__ sum,
                                                            int32_t *__restrict__ longest) {
    __shared__ int64_t ws[SQ_THREADS / 64];
    __shared__ int32_t wm[SQ_THREADS / 64];
    int64_t s = 0;
    int32_t m = 0;
    for (int64_t v = (int64_t)blockIdx.x * SQ_THREADS + threadIdx.x; v < rows;
         v += (int64_t)gridDim.x * SQ_THREADS) {
        const int64_t n = row_off[v + 1] - row_off[v];
        s += n * n;
        m = max(m, (int32_t)n);
    }
    s = tgd::wave_sum(s);
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) m = max(m, __shfl_xor(m, d, 64));
    if (__lane_id() == 0) {
        ws[threadIdx.x / 64] = s;
        wm[threadIdx.x / 64] = m;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < SQ_THREADS / 64; w++) {
            s += ws[w];
            m = max(m, wm[w]);
        }
        if (s) atomicAdd(sum, (unsigned long long)s);
        if (m) atomicMax(longest, m);
    }
}

// FF(f): faces of the (at most two) cells holding f, minus f.  One lane per
// face: both TF rows are loaded at once, the six candidates sorted by a
// network and the distinct ones written at the place that the chained scan
// gives.
constexpr int FF_THREADS = 512;
__global__ __launch_bounds__(FF_THREADS) void k_ff(const int32_t *__restrict__ ft, int64_t F,
                                                   const int32_t *__restrict__ tf,
                                                   int32_t *ticket, uint64_t *state,
                                                   int64_t *__restrict__ off,
                                                   int32_t *__restrict__ out) {
    __shared__ int32_t rows[FF_THREADS * 6];
    __shared__ int32_t wtot[FF_THREADS / 64];
    __shared__ int32_t shared_tile;
    __shared__ int64_t base;
    const int tid = threadIdx.x, lane = __lane_id(), wid = tid / 64;
    const int32_t tile = take_tile(ticket, shared_tile);
    const int64_t f = (int64_t)tile * FF_THREADS + tid;
    const bool act = f < F;
    const int2 cells = act ? reinterpret_cast<const int2 *>(ft)[f] : make_int2(-1, -1);
    const int4 r0 = reinterpret_cast<const int4 *>(tf)[cells.x >= 0 ? cells.x : 0];
    const int4 r1 = reinterpret_cast<const int4 *>(tf)[cells.y >= 0 ? cells.y : 0];
    int32_t c[8] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w};
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const bool on = i < 4 ? cells.x >= 0 : cells.y >= 0;
        if (!on || c[i] == (int32_t)f) c[i] = INF;
    }
    tgn::sort_keys(c);
    int m = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) m += c[i] != INF && (i == 0 || c[i] != c[i > 0 ? i - 1 : 0]);
    const int32_t inc = tgd::wave_inclusive_sum(m);
    if (lane == 63) wtot[wid] = inc;
    __syncthreads();
    int32_t before = 0, total = 0;
#pragma unroll
    for (int i = 0; i < FF_THREADS / 64; i++) {
        if (i < wid) before += wtot[i];
        total += wtot[i];
    }
    if (tid == 0) tgd::store_agent(state + tile, TILE_SUM | (uint64_t)total);
    int p = before + inc - m;
#pragma unroll
    for (int i = 0; i < 8; i++)
        if (c[i] != INF && (i == 0 || c[i] != c[i > 0 ? i - 1 : 0])) rows[p++] = c[i];
    if (wid == 0) {
        const int64_t b = tiles_before(state, tile);
        if (lane == 0) {
            tgd::store_agent(state + tile, TILE_PREFIX | (uint64_t)(b + total));
            base = b;
        }
    }
    __syncthreads();
    if (act) off[f] = base + before + inc - m;
    if (f == F - 1) off[F] = base + total;
    for (int32_t i = tid; i < total; i += FF_THREADS) out[base + i] = rows[i];
}

unsigned grid(int64_t n, int block = 256) {
    return std::min<unsigned>(tg::grid_for(n, block), 65536u);
}

int fail(int code, const char *msg) {
    tg::set_error(msg);
    return code;
}

// rank structure over n flags (0 or 1): rank_of(rank, p) is the number of
// flags set before position p.  total, when asked for, is read back, with two
// further words in the same wait.
int build_ranks(tg_mesh &m, const uint8_t *flags, int64_t n, tg::DevArr &rank,
                int64_t *total = nullptr, const int32_t *two = nullptr,
                int32_t *two_out = nullptr) {
    const int64_t nu = (n + UNIT - 1) / UNIT;
    int rc;
    if ((rc = m.rank_tmp.ensure(sizeof(int32_t) * (size_t)(nu + 1))) ||
        (rc = rank.ensure(sizeof(uint4) * (size_t)std::max<int64_t>(nu, 1))) ||
        (rc = m.scan_tmp.ensure(tg::scan_tmp_bytes(nu))))
        return rc;
    int32_t *before = m.rank_tmp.as<int32_t>();
    if (nu > 0) {
        hipLaunchKernelGGL(k_pack_flags, dim3(grid(nu)), dim3(256), 0, m.stream, flags, n,
                           rank.as<uint4>(), before);
        TG_LAUNCH_CHECK("k_pack_flags");
    }
    if ((rc = tg::scan_exclusive_i32(before, before, nu, m.scan_tmp.p, m.stream))) return rc;
    if (nu > 0) {
        hipLaunchKernelGGL(k_rank_counts, dim3(grid(nu)), dim3(256), 0, m.stream, before, nu,
                           rank.as<uint4>());
        TG_LAUNCH_CHECK("k_rank_counts");
    }
    if (!total) return tg::OK;
    int32_t *h = (int32_t *)m.h_pinned;
    TG_HIP(hipMemcpyAsync(h, before + nu, sizeof(int32_t), hipMemcpyDeviceToHost, m.stream));
    if (two)
        TG_HIP(hipMemcpyAsync(h + 2, two, 2 * sizeof(int32_t), hipMemcpyDeviceToHost, m.stream));
    TG_HIP(hipStreamSynchronize(m.stream));
    *total = h[0];
    if (two) {
        two_out[0] = h[2];
        two_out[1] = h[3];
    }
    return tg::OK;
}

// Zeroed state of a chained scan over `tiles` tiles, in tmp_b: a sum, the
// longest row, the number of listed outputs, the tile counter, the tiles' sums.
struct Chain {
    int64_t *sum;
    int32_t *longest, *listed, *ticket;
    uint64_t *state;
};
int chain_state(tg_mesh &m, int64_t tiles, Chain &c) {
    int rc = m.tmp_b.ensure(sizeof(int64_t) * (size_t)(tiles + 3));
    if (rc) return rc;
    c.sum = m.tmp_b.as<int64_t>();
    c.longest = reinterpret_cast<int32_t *>(c.sum + 1);
    c.listed = c.longest + 1;
    c.ticket = reinterpret_cast<int32_t *>(c.sum + 2);
    c.state = reinterpret_cast<uint64_t *>(c.sum + 3);
    return tg::fill_i32((int32_t *)c.sum, 0, 2 * (tiles + 3), m.stream);
}

// Sum of squared row lengths and the longest row, read back (synchronises).
int row_squares(tg_mesh &m, const int32_t *row_off, int64_t rows, const Chain &c, int64_t &sum,
                int32_t &longest) {
    hipLaunchKernelGGL(k_row_squares, dim3(std::min(grid(rows, SQ_THREADS), (unsigned)SQ_BLOCKS)),
                       dim3(SQ_THREADS), 0, m.stream, row_off, rows, (unsigned long long *)c.sum,
                       c.longest);
    TG_LAUNCH_CHECK("k_row_squares");
    int64_t *h = (int64_t *)m.h_pinned;
    TG_HIP(hipMemcpyAsync(h, c.sum, 2 * sizeof(int64_t), hipMemcpyDeviceToHost, m.stream));
    TG_HIP(hipStreamSynchronize(m.stream));
    sum = h[0];
    longest = *(const int32_t *)(h + 1);
    return tg::OK;
}

// The outputs with a row beyond JOIN_ROW into list (room for `count`).
template <typename RO>
int list_long(tg_mesh &m, const RO &rows_of, int64_t count, const Chain &c, int32_t *list) {
    hipLaunchKernelGGL((k_list_long<RO>), dim3(std::min(grid(count, LIST_THREADS), 8192u)),
                       dim3(LIST_THREADS), 0, m.stream, rows_of, count, list, c.listed);
    TG_LAUNCH_CHECK("k_list_long");
    return tg::OK;
}

}  // namespace

namespace tg {

int ensure_edges(tg_mesh &m) {
    if (m.edges_built) return OK;
    int rc;
    const int64_t V = m.n_points, T = m.n_cells;
    int64_t nnz = 0;
    if ((rc = ensure_vv(m)) || (rc = ensure_vt_sorted(m)) ||
        (rc = sync_check_read(m, m.vv_off.as<int32_t>() + V, nnz)))
        return rc;
    // an edge is counted from both its ends' rows: with one missing, what
    // follows would be sized for fewer edges than the kernels write
    if (m.vv_short) return capacity_error();
    const size_t I = sizeof(int32_t);
    if ((rc = m.edge_first.ensure(I * (size_t)std::max<int64_t>(nnz, 1))) ||
        (rc = m.te.ensure(I * 6 * (size_t)std::max<int64_t>(T, 1))) ||
        (rc = m.tmp_a.ensure(std::max<size_t>(6 * (size_t)T, 1))) ||  // flags
        (rc = m.ve_off.ensure(I * (size_t)(V + 1))))
        return rc;
    uint8_t *flags = m.tmp_a.as<uint8_t>();
    if ((rc = fill_u8(flags, 0, 6 * T, m.stream))) return rc;
    if (V > 0) {
        hipLaunchKernelGGL(k_edge_first, dim3(grid(V, EDGE_THREADS)), dim3(EDGE_THREADS), 0, m.stream,
                           m.tv.as<const int4>(), m.vt_off.as<int32_t>(), m.vtc.as<int32_t>(),
                           m.vv_off.as<int32_t>(), m.vv_cols.as<int32_t>(), V,
                           m.edge_first.as<int32_t>(), flags, m.te.as<int32_t>());
        TG_LAUNCH_CHECK("k_edge_first");
    }
    const int64_t E = nnz / 2;  // every edge is in both its ends' rows
    if ((rc = build_ranks(m, flags, 6 * T, m.edge_rank))) return rc;
    m.n_edges = E;
    const int64_t tiles = (V + VE_THREADS - 1) / VE_THREADS;
    Chain c;
    if ((rc = m.ev.ensure(I * 2 * (size_t)std::max<int64_t>(E, 1))) ||
        (rc = m.ve_vals.ensure(I * 2 * (size_t)std::max<int64_t>(E, 1))) ||
        (rc = chain_state(m, tiles, c)))
        return rc;
    int32_t *voff = m.ve_off.as<int32_t>();
    if (V > 0) {
        hipLaunchKernelGGL(k_ve, dim3((unsigned)tiles), dim3(VE_THREADS), 0, m.stream,
                           m.tv.as<const int4>(), m.vv_off.as<int32_t>(), m.vv_cols.as<int32_t>(), V,
                           m.edge_first.as<int32_t>(), m.edge_rank.as<uint4>(), c.ticket, c.state,
                           voff, m.ve_vals.as<int2>());
        TG_LAUNCH_CHECK("k_ve");
    } else if ((rc = fill_i32(voff, 0, 1, m.stream))) {
        return rc;
    }
    if (T > 0) {
        hipLaunchKernelGGL(k_te, dim3(grid(6 * T)), dim3(256), 0, m.stream, m.te.as<int32_t>(),
                           6 * T, m.edge_rank.as<uint4>());
        TG_LAUNCH_CHECK("k_te");
        hipLaunchKernelGGL(k_ev, dim3(grid(T)), dim3(256), 0, m.stream, m.tv.as<const int4>(), T,
                           m.edge_rank.as<uint4>(), m.ev.as<int2>());
        TG_LAUNCH_CHECK("k_ev");
    }
    m.edges_built = true;
    return OK;
}

int ensure_et(tg_mesh &m) {
    if (m.et_built) return OK;
    int rc;
    // the vertex-lane VV form rewrites the corner lists unsorted: sort again
    if ((rc = ensure_edges(m)) || (rc = ensure_vt_sorted(m))) return rc;
    const int64_t E = m.n_edges;
    const int64_t nnz = 6 * m.n_cells;  // each cell holds six edges
    const int64_t tiles = (E + EJ_THREADS - 1) / EJ_THREADS;
    Chain c;
    if ((rc = m.et_off.ensure(sizeof(int64_t) * (size_t)(E + 1))) ||
        (rc = m.et_vals.ensure(sizeof(int32_t) * (size_t)std::max<int64_t>(nnz, 1))) ||
        (rc = chain_state(m, tiles, c)))
        return rc;
    int64_t *off = m.et_off.as<int64_t>();
    static_assert(JOIN_ROW >= LANE_CELLS, "few_cells: no row beyond the networks");
    bool listed = !m.few_cells;  // tmp_a: the edges with long rows, and their lengths by edge
    if (listed && !m.heavy_counted && E > 0) {  // VV came from a form that does not tell
        int64_t squares;
        int32_t longest;
        if ((rc = row_squares(m, m.vt_off.as<int32_t>(), m.n_points, c, squares, longest))) return rc;
        listed = longest > JOIN_ROW;
    }
    if (listed && (rc = m.tmp_a.ensure(sizeof(int32_t) * 2 * (size_t)std::max<int64_t>(E, 1)))) return rc;
    const EdgeRows rows_of{m.ev.as<int32_t>(), m.n_points, m.vt_off.as<int32_t>()};
    const int32_t *vtc = m.vtc.as<int32_t>();
    int32_t *list = m.tmp_a.as<int32_t>(), *len = list + E, *out = m.et_vals.as<int32_t>();
    if (E == 0) {
        if ((rc = fill_i32((int32_t *)off, 0, 2, m.stream))) return rc;
    } else if (!listed) {
        hipLaunchKernelGGL((k_edge_join<INTERSECT, 2, NO_LONG, ET_WIN>), dim3((unsigned)tiles),
                           dim3(EJ_THREADS), 0, m.stream, rows_of, E, vtc, nullptr, c.ticket, c.state,
                           off, out);
        TG_LAUNCH_CHECK("k_edge_join<ET>");
    } else {
        if ((rc = list_long(m, rows_of, E, c, list))) return rc;
        hipLaunchKernelGGL((k_join_long<2, INTERSECT, 2, false, EdgeRows>), dim3(LONG_BLOCKS),
                           dim3(LONG_THREADS), 0, m.stream, rows_of, vtc, list, c.listed, len, nullptr,
                           nullptr);
        TG_LAUNCH_CHECK("k_join_long<ET>");
        hipLaunchKernelGGL((k_edge_join<INTERSECT, 2, LISTED, ET_WIN>), dim3((unsigned)tiles),
                           dim3(EJ_THREADS), 0, m.stream, rows_of, E, vtc, len, c.ticket, c.state, off,
                           out);
        TG_LAUNCH_CHECK("k_edge_join<ET>");
        hipLaunchKernelGGL((k_join_long<2, INTERSECT, 2, true, EdgeRows>), dim3(LONG_BLOCKS),
                           dim3(LONG_THREADS), 0, m.stream, rows_of, vtc, list, c.listed, nullptr, off,
                           out);
        TG_LAUNCH_CHECK("k_join_long<ET>");
    }
    m.et_built = true;
    return OK;
}

int ensure_faces(tg_mesh &m) {
    if (m.faces_built) return OK;
    int rc;
    if ((rc = ensure_et(m)) || (rc = ensure_vt_sorted(m))) return rc;
    const int64_t V = m.n_points, T = m.n_cells;
    const size_t I = sizeof(int32_t);
    if ((rc = m.tmp_b.ensure(I * std::max<size_t>(4 * (size_t)T, 1))) ||  // ffirst
        (rc = m.tmp_a.ensure(std::max<size_t>(4 * (size_t)T, 1))) ||      // flags
        (rc = m.tf.ensure(I * std::max<size_t>(4 * (size_t)T, 1))))
        return rc;
    int32_t *ffirst = m.tmp_b.as<int32_t>();
    uint8_t *flags = m.tmp_a.as<uint8_t>();
    int32_t *err = m.counters.as<int32_t>() + C_FTERR;
    int32_t *iderr = m.counters.as<int32_t>() + C_IDERR;
    if ((rc = fill_i32(err, 0, 2, m.stream))) return rc;
    if ((rc = m.tmp_c.ensure(I * std::max<size_t>(4 * (size_t)T, 1)))) return rc;  // other cell
    int32_t *other = m.tmp_c.as<int32_t>();
    if (T > 0) {
        hipLaunchKernelGGL(k_face_first, dim3(grid(4 * T)), dim3(256), 0, m.stream,
                           m.tv.as<const int4>(), T, m.te.as<int32_t>(), m.n_edges,
                           m.et_off.as<int64_t>(), m.et_vals.as<int32_t>(), ffirst, flags, other,
                           iderr, err);
        TG_LAUNCH_CHECK("k_face_first");
    }
    int64_t F = 0;
    int32_t errs[2] = {0, 0};  // C_FTERR, C_IDERR
    static_assert(C_IDERR == C_FTERR + 1, "read together");
    if ((rc = build_ranks(m, flags, 4 * T, m.face_rank, &F, err, errs))) return rc;
    if (errs[1]) return fail(ERR_STATE, "face ids: TE and ET disagree (a cell is missing from ET)");
    m.ft_ok = errs[0] == 0;
    m.n_faces = F;
    if ((rc = m.fv.ensure(I * 3 * (size_t)std::max<int64_t>(F, 1))) ||
        (rc = m.ft.ensure(I * 2 * (size_t)std::max<int64_t>(F, 1))) ||
        (rc = m.face_off.ensure(I * (size_t)(V + 1))))
        return rc;
    if (T > 0) {
        hipLaunchKernelGGL(k_face_ids, dim3(grid(4 * T)), dim3(256), 0, m.stream,
                           m.tv.as<const int4>(), T, ffirst, other, m.face_rank.as<uint4>(),
                           m.tf.as<int32_t>(), m.fv.as<int32_t>(), m.ft.as<int32_t>());
        TG_LAUNCH_CHECK("k_face_ids");
    }
    int32_t *voff = m.face_off.as<int32_t>();
    if ((rc = m.vf_vals.ensure(I * 3 * (size_t)std::max<int64_t>(F, 1)))) return rc;
    if (V > 0) {
        const int64_t tiles = (V + VF_THREADS - 1) / VF_THREADS;
        Chain c;
        if ((rc = chain_state(m, tiles, c))) return rc;
        hipLaunchKernelGGL(k_vf, dim3((unsigned)tiles), dim3(VF_THREADS), 0, m.stream,
                           m.tv.as<const int4>(), m.vt_off.as<int32_t>(), m.vtc.as<int32_t>(), V,
                           m.face_rank.as<uint4>(), c.ticket, c.state, voff,
                           m.vf_vals.as<int32_t>());
        TG_LAUNCH_CHECK("k_vf");
    } else if ((rc = fill_i32(voff, 0, 1, m.stream))) {
        return rc;
    }
    m.face_rank.release();
    m.faces_built = true;
    return OK;
}

int ensure_fe(tg_mesh &m) {
    if (m.fe_built) return OK;
    int rc;
    if ((rc = ensure_edges(m)) || (rc = ensure_faces(m))) return rc;
    const int64_t F = m.n_faces;
    if ((rc = m.fe.ensure(sizeof(int32_t) * 6 * (size_t)std::max<int64_t>(F, 1)))) return rc;
    if (F > 0) {
        hipLaunchKernelGGL(k_fe, dim3(grid(F)), dim3(256), 0, m.stream, m.tv.as<const int4>(),
                           m.fv.as<int32_t>(), F, m.ft.as<int32_t>(), m.te.as<int32_t>(),
                           m.fe.as<int32_t>());
        TG_LAUNCH_CHECK("k_fe");
    }
    m.fe_built = true;
    return OK;
}

int ensure_ft(tg_mesh &m) {
    int rc = ensure_faces(m);
    if (rc) return rc;
    if (!m.ft_ok) return fail(ERR_MESH, "a face is held by more than two cells; FT needs <= 2");
    return OK;
}

int ensure_ef(tg_mesh &m) {
    if (m.ef_built) return OK;
    int rc;
    if ((rc = ensure_et(m)) || (rc = ensure_faces(m))) return rc;
    const int64_t E = m.n_edges;
    const int64_t tiles = (E + EF_THREADS - 1) / EF_THREADS;
    const int64_t et_nnz = 6 * m.n_cells, nnz = 3 * m.n_faces;  // a face holds three edges
    Chain c;
    // tmp_c: rows too long for LDS; tmp_a: the cells' corners and faces
    if ((rc = m.ef_off.ensure(sizeof(int64_t) * (size_t)(E + 1))) ||
        (rc = m.ef_vals.ensure(sizeof(int32_t) * (size_t)std::max<int64_t>(nnz, 1))) ||
        (rc = m.tmp_c.ensure(sizeof(int32_t) * 2 * (size_t)std::max<int64_t>(et_nnz, 1))) ||
        (rc = m.tmp_a.ensure(sizeof(int4) * 2 * (size_t)std::max<int64_t>(m.n_cells, 1))) ||
        (rc = chain_state(m, tiles, c)))
        return rc;
    int64_t *off = m.ef_off.as<int64_t>();
    if (E > 0) {
        hipLaunchKernelGGL(k_cell_faces, dim3(grid(2 * m.n_cells)), dim3(256), 0, m.stream,
                           m.tv.as<const int4>(), m.tf.as<const int4>(), m.n_cells,
                           m.tmp_a.as<int4>());
        TG_LAUNCH_CHECK("k_cell_faces");
        hipLaunchKernelGGL(k_ef, dim3((unsigned)tiles), dim3(EF_THREADS), 0, m.stream,
                           m.et_off.as<int64_t>(), E, m.et_vals.as<int32_t>(),
                           m.ev.as<const int2>(), m.tmp_a.as<const int4>(), c.ticket, c.state, off,
                           m.ef_vals.as<int32_t>(), m.tmp_c.as<int32_t>());
        TG_LAUNCH_CHECK("k_ef");
        m.tmp_a.release();  // 32 bytes a cell, which nothing else needs
    } else if ((rc = fill_i32((int32_t *)off, 0, 2, m.stream))) {
        return rc;
    }
    m.ef_nnz = nnz;
    m.ef_built = true;
    return OK;
}

int ensure_tt(tg_mesh &m) {
    if (m.tt_built) return OK;
    int rc;
    if ((rc = ensure_vt_sorted(m))) return rc;
    const int64_t T = m.n_cells, V = m.n_points;
    const int64_t tiles = (T + TT_THREADS - 1) / TT_THREADS;
    Chain c;
    if ((rc = m.tt_off.ensure(sizeof(int64_t) * (size_t)(T + 1))) || (rc = chain_state(m, tiles, c)))
        return rc;
    int64_t *off = m.tt_off.as<int64_t>();
    int64_t rows = 0;
    int32_t longest = 0;
    // the cells' rows together: every vertex's row once per entry
    if (T > 0 && (rc = row_squares(m, m.vt_off.as<int32_t>(), V, c, rows, longest))) return rc;
    const bool listed = longest > JOIN_ROW;
    // a cell's four rows hold the cell itself four times; tmp_a: the cells
    // with long rows, and their lengths by cell
    if ((rc = m.tt_vals.ensure(sizeof(int32_t) * (size_t)std::max<int64_t>(rows - 4 * T, 1))) ||
        (listed && (rc = m.tmp_a.ensure(sizeof(int32_t) * 2 * (size_t)T))))
        return rc;
    const CellRows rows_of{m.tv.as<const int4>(), m.vt_off.as<int32_t>()};
    const int32_t *vtc = m.vtc.as<int32_t>();
    int32_t *list = m.tmp_a.as<int32_t>(), *len = list + T, *out = m.tt_vals.as<int32_t>();
    if (T == 0) {
        if ((rc = fill_i32((int32_t *)off, 0, 2, m.stream))) return rc;
    } else if (!listed) {
        hipLaunchKernelGGL((k_tt<NO_LONG>), dim3((unsigned)tiles), dim3(TT_THREADS), 0, m.stream,
                           rows_of, T, vtc, nullptr, c.ticket, c.state, off, out);
        TG_LAUNCH_CHECK("k_tt");
    } else {
        if ((rc = list_long(m, rows_of, T, c, list))) return rc;
        hipLaunchKernelGGL((k_join_long<4, UNION_LESS_SELF, 2, false, CellRows>), dim3(LONG_BLOCKS),
                           dim3(LONG_THREADS), 0, m.stream, rows_of, vtc, list, c.listed, len, nullptr,
                           nullptr);
        TG_LAUNCH_CHECK("k_join_long<TT>");
        hipLaunchKernelGGL((k_tt<LISTED>), dim3((unsigned)tiles), dim3(TT_THREADS), 0, m.stream,
                           rows_of, T, vtc, len, c.ticket, c.state, off, out);
        TG_LAUNCH_CHECK("k_tt");
        hipLaunchKernelGGL((k_join_long<4, UNION_LESS_SELF, 2, true, CellRows>), dim3(LONG_BLOCKS),
                           dim3(LONG_THREADS), 0, m.stream, rows_of, vtc, list, c.listed, nullptr, off,
                           out);
        TG_LAUNCH_CHECK("k_join_long<TT>");
    }
    m.tt_nnz = T > 0 ? -1 : 0;
    m.tt_built = true;
    return OK;
}

int ensure_ff(tg_mesh &m) {
    if (m.ff_built) return OK;
    int rc;
    if ((rc = ensure_ft(m))) return rc;
    const int64_t F = m.n_faces;
    const int64_t tiles = (F + FF_THREADS - 1) / FF_THREADS;
    Chain c;
    // a cell gives each of its four faces at most the three others
    if ((rc = m.ff_off.ensure(sizeof(int64_t) * (size_t)(F + 1))) ||
        (rc = m.ff_vals.ensure(sizeof(int32_t) * (size_t)std::max<int64_t>(12 * m.n_cells, 1))) ||
        (rc = chain_state(m, tiles, c)))
        return rc;
    int64_t *off = m.ff_off.as<int64_t>();
    if (F > 0) {
        hipLaunchKernelGGL(k_ff, dim3((unsigned)tiles), dim3(FF_THREADS), 0, m.stream,
                           m.ft.as<int32_t>(), F, m.tf.as<int32_t>(), c.ticket, c.state, off,
                           m.ff_vals.as<int32_t>());
        TG_LAUNCH_CHECK("k_ff");
    } else if ((rc = fill_i32((int32_t *)off, 0, 2, m.stream))) {
        return rc;
    }
    m.ff_nnz = F > 0 ? -1 : 0;
    m.ff_built = true;
    return OK;
}

int ensure_ee(tg_mesh &m) {
    if (m.ee_built) return OK;
    int rc;
    if ((rc = ensure_edges(m))) return rc;
    const int64_t E = m.n_edges, V = m.n_points;
    const int64_t tiles = (E + EJ_THREADS - 1) / EJ_THREADS, n2 = 2 * E;
    Chain c;
    // tmp_c: each vertex's edge ids, and four words of slack (rows are loaded
    // by whole quads)
    if ((rc = m.ee_off.ensure(sizeof(int64_t) * (size_t)(E + 1))) ||
        (rc = m.tmp_c.ensure(sizeof(int32_t) * (size_t)(n2 + 4))) || (rc = chain_state(m, tiles, c)))
        return rc;
    int64_t *off = m.ee_off.as<int64_t>();
    int64_t nnz = 0;
    int32_t longest = 0;
    if (E > 0) {
        hipLaunchKernelGGL(k_vertex_edges, dim3((unsigned)((V + VX_THREADS - 1) / VX_THREADS)),
                           dim3(VX_THREADS), 0, m.stream,
                           m.vv_off.as<int32_t>(), V, m.edge_first.as<int32_t>(),
                           m.edge_rank.as<uint4>(), m.ve_off.as<int32_t>(), m.ve_vals.as<int2>(),
                           m.tmp_c.as<int32_t>());
        TG_LAUNCH_CHECK("k_vertex_edges");
        // an edge's row: its ends' edges, which share only itself
        if ((rc = row_squares(m, m.vv_off.as<int32_t>(), V, c, nnz, longest))) return rc;
        nnz -= n2;
    }
    const bool listed = longest > JOIN_ROW;  // tmp_a: the edges with long rows
    if ((rc = m.ee_vals.ensure(sizeof(int32_t) * (size_t)std::max<int64_t>(nnz, 1))) ||
        (listed && (rc = m.tmp_a.ensure(sizeof(int32_t) * (size_t)E))))
        return rc;
    const EdgeRows rows_of{m.ev.as<int32_t>(), V, m.vv_off.as<int32_t>()};
    const int32_t *ids = m.tmp_c.as<int32_t>();
    int32_t *list = m.tmp_a.as<int32_t>(), *out = m.ee_vals.as<int32_t>();
    if (E == 0) {
        if ((rc = fill_i32((int32_t *)off, 0, 2, m.stream))) return rc;
    } else if (!listed) {
        hipLaunchKernelGGL((k_edge_join<UNION_LESS_SELF, 0, NO_LONG, EE_WIN>), dim3((unsigned)tiles),
                           dim3(EJ_THREADS), 0, m.stream, rows_of, E, ids, nullptr, c.ticket, c.state,
                           off, out);
        TG_LAUNCH_CHECK("k_edge_join<EE>");
    } else {
        hipLaunchKernelGGL((k_edge_join<UNION_LESS_SELF, 0, LISTED, EE_WIN>), dim3((unsigned)tiles),
                           dim3(EJ_THREADS), 0, m.stream, rows_of, E, ids, nullptr, c.ticket, c.state,
                           off, out);
        TG_LAUNCH_CHECK("k_edge_join<EE>");
        if ((rc = list_long(m, rows_of, E, c, list))) return rc;
        hipLaunchKernelGGL((k_join_long<2, UNION_LESS_SELF, 0, true, EdgeRows>), dim3(LONG_BLOCKS), dim3(LONG_THREADS),
                           0, m.stream, rows_of, ids, list, c.listed, nullptr, off, out);
        TG_LAUNCH_CHECK("k_join_long<EE>");
    }
    m.ee_nnz = nnz;
    m.ee_built = true;
    return OK;
}

int id_relation_view(tg_mesh &m, int32_t rel, RelView &r) {
    const int64_t V = m.n_points, T = m.n_cells, E = m.n_edges, F = m.n_faces;
    auto need = [&](bool ok, const char *what) { return ok ? OK : fail(ERR_STATE, what); };
    int rc;
    switch (rel) {
    case TG_REL_TE:
        if ((rc = need(m.edges_built, "TE not built"))) return rc;
        r = {T, T, 6, nullptr, 0, m.te.as<int32_t>()};
        return OK;
    case TG_REL_EV:
        if ((rc = need(m.edges_built, "EV not built"))) return rc;
        r = {E, E, 2, nullptr, 0, m.ev.as<int32_t>()};
        return OK;
    case TG_REL_VE:
        if ((rc = need(m.edges_built, "VE not built"))) return rc;
        r = {V, E, 2, m.ve_off.p, 4, m.ve_vals.as<int32_t>()};
        return OK;
    case TG_REL_ET:
        if ((rc = need(m.et_built, "ET not built"))) return rc;
        r = {E, 6 * T, 1, m.et_off.p, 8, m.et_vals.as<int32_t>()};
        return OK;
    case TG_REL_TF:
        if ((rc = need(m.faces_built, "TF not built"))) return rc;
        r = {T, T, 4, nullptr, 0, m.tf.as<int32_t>()};
        return OK;
    case TG_REL_FV:
        if ((rc = need(m.faces_built, "FV not built"))) return rc;
        r = {F, F, 3, nullptr, 0, m.fv.as<int32_t>()};
        return OK;
    case TG_REL_VF:
        if ((rc = need(m.faces_built, "VF not built"))) return rc;
        r = {V, F, 3, m.face_off.p, 4, m.vf_vals.as<int32_t>()};
        return OK;
    case TG_REL_FE:
        if ((rc = need(m.fe_built, "FE not built"))) return rc;
        r = {F, F, 6, nullptr, 0, m.fe.as<int32_t>()};
        return OK;
    case TG_REL_FT:
        if ((rc = need(m.faces_built, "FT not built"))) return rc;
        if (!m.ft_ok) return fail(ERR_MESH, "a face is held by more than two cells");
        r = {F, F, 2, nullptr, 0, m.ft.as<int32_t>()};
        return OK;
    case TG_REL_EF:
        if ((rc = need(m.ef_built, "EF not built"))) return rc;
        r = {E, m.ef_nnz, 1, m.ef_off.p, 8, m.ef_vals.as<int32_t>()};
        return OK;
    case TG_REL_TT:
        if ((rc = need(m.tt_built, "TT not built"))) return rc;
        r = {T, m.tt_nnz, 1, m.tt_off.p, 8, m.tt_vals.as<int32_t>()};
        return OK;
    case TG_REL_FF:
        if ((rc = need(m.ff_built, "FF not built"))) return rc;
        r = {F, m.ff_nnz, 1, m.ff_off.p, 8, m.ff_vals.as<int32_t>()};
        return OK;
    case TG_REL_EE:
        if ((rc = need(m.ee_built, "EE not built"))) return rc;
        r = {E, m.ee_nnz, 1, m.ee_off.p, 8, m.ee_vals.as<int32_t>()};
        return OK;
    default:
        return fail(ERR_ARG, "unknown relation id");
    }
}

}  // namespace tg
