// pf2_kernels.hpp — device kernels of the particle stage (FP64 path).
//
// Data layout in HBM (one simulation):
//   mesh     X[n_vertices*DIM] (row-major), cell_vertices / cell_dofs [n_cells*NV],
//            vertex star CSR (ascending cells) + normalised centre directions,
//            DoF -> (cell, local vertex) CSR in ascending cell order.
//   fields   V, Vold [n_dofs*DIM] node-major (one DoF's components adjacent).
//   particles structure of arrays, component-major (x[d*cap + i]), sorted by
//            cell, ascending id inside a cell; cell_off[n_cells+1] is the CSR.
// Per time step (pf2_step):
//   k_move         one thread per particle: correction, then substeps of
//                  advection in registers until done or the first failed
//                  own-cell test; such particles are parked in a queue.
//   k_search_resume  over the queue: vertex-star search in full wavefronts,
//                  then the remaining substeps.
//                  A particle that ends in another cell takes a slot in that
//                  cell's arrival row (add_arrival).
//   k_cell_count   one 16-lane group per cell: part counts over stayers +
//                  arrivals, survivors (MAX smallest ids per part), empty
//                  parts to reseed, final count (k_cell_big: larger cells).
//   k_cell_write   survivors and new particles into the other buffer at
//                  their final positions, and the cells' projection sums in
//                  ascending id order (k_cell_partials: the sums alone, one
//                  group per cell, for a projection without a move).
//   k_node         one thread per DoF: sum of the cell partials in ascending
//                  cell order, then division by the weight.
// No floating-point atomics anywhere.  Integer atomics only build lists whose
// order is erased again by the id ordering; counters that many wavefronts
// update are sharded over separate cache lines.
//
// Times in these sources are kernel times of one MI355X per step or launch on
// the timed workloads (perf/cases.py: 101,785 quads with 2.4M particles,
// 407,140 with 11M on a moving mesh, 202,240 hexahedra, 68,992 of degree 2),
// unless they say otherwise.
#pragma once

#include "pf2_geom.hpp"
#include <stdint.h>

namespace pf2 {

constexpr int WAVE = 64;

// sum over the wavefront (all lanes must call)
__device__ __forceinline__ int wave_sum(int v) {
#pragma unroll
    for (int off = WAVE / 2; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// Counters that many wavefronts update are spread over STAT_SHARDS cache
// lines: atomics on one address serialise in the memory system (about 11 ns
// each on MI355X), so a single counter updated once per wavefront would
// cost hundreds of microseconds per launch.
constexpr int STAT_SHARDS = 256;
constexpr int NSTAT = 8;   // u64 per shard row (64 bytes)

__device__ __forceinline__ int wave_shard() {
    return (int)((blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE) & (STAT_SHARDS - 1));
}

__device__ __forceinline__ void stat_add(unsigned long long* stats, int k, unsigned long long v) {
    atomicAdd(&stats[wave_shard() * NSTAT + k], v);
}

// flush per-lane statistics with one sharded atomic per wavefront (all lanes must call)
__device__ __forceinline__ void wave_stat(unsigned long long* stats, int k, int v) {
    const int t = wave_sum(v);
    if ((threadIdx.x & (WAVE - 1)) == 0 && t) stat_add(stats, k, (unsigned long long)t);
}

// Arrivals (particles that changed cell) of the lanes with pred set: particle
// i takes a slot of cell c's row, so the census finds a cell's arrivals with
// no grouping pass; arrivals past the row go to the cell's overflow list (the
// census then handles the cell in k_cell_big).  Lanes with the same cell
// share one atomic, and the atomics of all cells of the wavefront are issued
// together, so the wavefront waits for one returning atomic.  All lanes of
// the wavefront call.
template <class W>
__device__ __forceinline__ void add_arrival(const W& w, bool pred, int c, int i) {
    const int lane = threadIdx.x & (WAVE - 1);
    unsigned long long todo = __ballot(pred);
    if (todo == 0) return;
    int leader = lane, off = 0, cnt = 0;
    while (todo) {
        const int l = __ffsll((long long)todo) - 1;
        const int key = __shfl(c, l);
        const unsigned long long same = __ballot(pred && c == key) & todo;
        if ((same >> lane) & 1) {
            leader = l;
            off = __popcll(same & ((1ull << lane) - 1));
        }
        if (lane == l) cnt = __popcll(same);
        todo &= ~same;
    }
    int base = 0;
    if (cnt) base = atomicAdd(&w.arr_cnt[c], cnt);
    base = __shfl(base, leader);
    if (!pred) return;
    const int slot = base + off;
    if (slot < w.aslots) {
        w.arr_slot[(size_t)c * w.aslots + slot] = i;
        return;
    }
    const int e = atomicAdd(&w.counters[4], 1);
    const int next = atomicExch(&w.ovf_head[c], e);
    w.ovf[e] = make_int2(i, next);
}

template <int DIM>
struct DevMesh {
    int n_cells, n_vertices, n_dofs;
    int nd;                // velocity DoFs per cell: 2^DIM (Q1) or 3^DIM (Q2)
    const double* X;
    const int* cv;
    const int* cd;         // per cell: its ND velocity DoFs (ND = QF<DIM, DEG>::ND)
    const int* star_off;
    const int* star_cell;
    const double* star_dir;
    const int* dof_off;
    const int* dof_cell;   // packed: cell * ND + local DoF
    const double* ftol;    // per cell: 2-D the tolerance of the clearly-outside test (-1: none), 3-D the
                           // HEX_N values of HexCell
    const double* cellX;   // per cell: its vertex coordinates packed [NV][DIM] (copies of X)
    const int2* cell_star; // per cell and local vertex: [begin, end) of that vertex's star
    const int4* cell_nbr;  // per cell, the neighbours across faces 0..2*DIM-1 (-1 on the boundary or past
                           // the faces): one int4 in 2-D, two in 3-D
    const double* cellV;   // per cell: V at its DoFs [ND][DIM] (refreshed when V changes); null for
                           // FP32-mixed handles, whose particle kernels read FP32 copies
    const double* cellDV;  // per cell: V - V_old at its DoFs [ND][DIM] (FP64 handles)
    const double* Vn;      // V, node-major [n_dofs][DIM]
    const unsigned char* cmoved;   // per cell: 1 if the last geometry update changed a vertex of it
};

struct DevParticles {
    int* cell;
    uint32_t* id;
    double* x;
    double* xi;
    double* v;
    double* vext;   // may be null
    long long cap;
};

struct DevParams {
    double h;           // dt / substeps
    int substeps;
    int max_per_part;
    int q[3];
    double hq[3];       // 1.0 / q[d] (the part width, correctly rounded)
    int nparts_in;      // q0*q1[*q2]
    int keep_vext;
};

// Offsets from the census's per-cell counts (fs_cnt: particles << 32 | new
// ones, whose total stays below 2^32, so the low halves never carry): an
// exclusive scan, two launches, or on meshes of up to SUMS_CELLS cells sums over
// groups of cells, from which a write workgroup reads its own offset: the tiles
// before its own and the cells before it in that, a few loads a lane at once.
//   fine     per wavefront of k_cell_count (4 cells): the cells it counted
//   tile     per TILE cells: k_cell_big adds the fine sums and the cells it
//            counts itself (which fine leaves out).  Two sets: a census adds to
//            one and the write after it clears the other for the next
//            (counters[8] says which).
// Two launches less are 3% of a step on 2,000 cells.  Whole steps of a fixed
// cylinder mesh with sums and with the scan, FP64 and FP32-mixed: 182 and 185,
// 176 and 179 us on 25,446 cells; 236 and 240, 203 and 208 on 40,000; 318 and
// 322, 238 and 242 on 60,000; 409 and 413, 287 and 289 on 80,000; the same on
// 101,785; 918 and 908, 599 and 593 on 200,000.  So they cross near 100,000
// cells, past which a workgroup's loads of the tiles before its own cost more
// than the launches (on 407,140 the census takes 14 us more and the write 17).
// The line lies below that, where a wavefront reads all tiles with two loads a
// lane; it gives away 1-2% of a step from there to 80,000 cells.
// Tiles added by the census itself, an atomic per wavefront, cost it 40 us on
// 101,785 cells: atomics on neighbouring sums serialise.
constexpr int TILE = 256;
constexpr int SUMS_CELLS = 128 * TILE;   // (two tiles a lane)
struct CellSums {
    unsigned long long* fine;   // null: scanned offsets
    unsigned long long* tile;   // 2 sets of ntile
    int nfine, ntile;
    __device__ __forceinline__ unsigned long long* tiles(int set) const { return tile + (size_t)(set & 1) * ntile; }
};
inline int fine_sums(int n_cells) { return (n_cells + 15) / 16 * 4; }
inline int tile_sums(int n_cells) { return (n_cells + TILE - 1) / TILE; }

struct DevWork {
    int* dest;          // per particle: new cell or -1
    int* pkey;          // per particle: part key of the final position
    int* spos;          // per particle: position among the cell's survivors, -1 = dropped
    int* arr_cnt;       // per cell: arrivals
    int* arr_slot;      // per cell: aslots arrival slots (particle indices)
    int aslots;
    int2* ovf;          // arrivals past a cell's slots: (particle, next entry) lists
    int* ovf_head;      // per cell: first overflow entry or -1
    unsigned long long* fs_cnt;    // per cell: final count << 32 | spawns
    unsigned long long* fs_off;    // its exclusive scan (n_cells + 1) where sums.fine is null
    CellSums sums;      // else the counts' sums over groups of cells
    int* new_off;       // n_cells + 1: particle offsets, written by the cell writes
    unsigned long long* hitmask;   // per cell: in-range parts that hold a particle
    int* nsurv;         // per cell: survivors
    double* partial;    // projection sums, DIM + 1 per cell and DoF of it (partial_at)
    int* counters;      // [0] n_particles, [1] arrivals of the last regroup, [2] overflow flags,
                        // [3] count before the last regroup, [4] overflow entries in use,
                        // [5] id counter at the last advection (ids up to it hold an inverse-mapped xi),
                        // [6] slots of a pending layout (0: none; see k_cell_pend), [7] its segment end,
                        // [8] the set of CellSums of the current census
    int* big;           // [0] number of cells listed for k_cell_big, then the cells
    int pend_mark;      // census of a pending regroup: survivors' destinations get DEST_KEPT
    uint32_t* particle_counter;
    unsigned long long* stats;   // STAT_SHARDS rows: lost, deleted, spawned, searches, zero-weight
};

// counters[2] bits 0 and 1 (particle capacity exceeded, a cell past the
// census limit) are sticky: the regroup that set them left the particle
// buffers incomplete and the new offsets beyond the capacity.  Every later
// kernel that reads particles or offsets then returns at once, so steps
// already queued (graph replays, chunks issued ahead) touch no memory out of
// bounds; the host reports PF2_E_CAPACITY at its next synchronisation.
constexpr int DEAD_FLAGS = 3;
__device__ __forceinline__ bool state_dead(const int* counters) { return (counters[2] & DEAD_FLAGS) != 0; }

// The same for the workgroups of a kernel that raises a flag itself and shares
// LDS between wavefronts: one thread reads it for all (all threads call), so
// that no wavefront leaves the others to LDS that it was to fill.
__device__ __forceinline__ bool workgroup_dead(const int* counters) {
    __shared__ int s_dead;
    if (threadIdx.x == 0) s_dead = state_dead(counters);
    __syncthreads();
    return s_dead != 0;
}

// vertex coordinates and nodal velocities of cell c, from the packed per-cell
// copies, or (GATHER: FP32-mixed handles, which keep no FP64 velocity copy)
// with the velocities gathered from V through the cell's DoF map (the same
// values).  The choice is a template argument so that the kernels of FP64
// handles carry no second path.
template <int DIM, bool GATHER = false, int DEG = 1>
__device__ __forceinline__ void load_cell(const DevMesh<DIM>& m, int c, double (*P)[DIM], double (*Fc)[DIM]) {
    constexpr int NV = Q1<DIM>::NV;
    constexpr int ND = QF<DIM, DEG>::ND;
    const double* cx = m.cellX + (size_t)c * NV * DIM;
#pragma unroll
    for (int k = 0; k < NV; ++k)
#pragma unroll
        for (int d = 0; d < DIM; ++d) P[k][d] = cx[k * DIM + d];
    if constexpr (GATHER) {
#pragma unroll
        for (int k = 0; k < ND; ++k) {
            const double* vf = m.Vn + (size_t)m.cd[(size_t)c * ND + k] * DIM;
#pragma unroll
            for (int d = 0; d < DIM; ++d) Fc[k][d] = vf[d];
        }
    } else {
        const double* cf = m.cellV + (size_t)c * ND * DIM;
#pragma unroll
        for (int k = 0; k < ND; ++k)
#pragma unroll
            for (int d = 0; d < DIM; ++d) Fc[k][d] = cf[k * DIM + d];
    }
}

// the same, choosing by whether the handle keeps the FP64 copy (seeding)
template <int DIM, int DEG = 1>
__device__ __forceinline__ void load_cell_any(const DevMesh<DIM>& m, int c, double (*P)[DIM], double (*Fc)[DIM]) {
    if (m.cellV) load_cell<DIM, false, DEG>(m, c, P, Fc);
    else load_cell<DIM, true, DEG>(m, c, P, Fc);
}

// vertex coordinates of cell c (packed per-cell copy: one dependent load level)
template <int DIM>
__device__ __forceinline__ void load_vertices(const DevMesh<DIM>& m, int c, double (*P)[DIM]) {
    constexpr int NV = Q1<DIM>::NV;
    const double* cx = m.cellX + (size_t)c * NV * DIM;
#pragma unroll
    for (int k = 0; k < NV; ++k)
#pragma unroll
        for (int d = 0; d < DIM; ++d) P[k][d] = cx[k * DIM + d];
}

// vertex coordinates gathered from X through the cell's vertex indices
template <int DIM>
__device__ __forceinline__ void gather_vertices(const DevMesh<DIM>& m, int c, double (*P)[DIM]) {
    constexpr int NV = Q1<DIM>::NV;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int gv = m.cv[(size_t)c * NV + k];
#pragma unroll
        for (int d = 0; d < DIM; ++d) P[k][d] = m.X[(size_t)gv * DIM + d];
    }
}

// sum over the wavefront (all lanes must call)
__device__ __forceinline__ unsigned long long wave_sum64(unsigned long long v) {
#pragma unroll
    for (int off = WAVE / 2; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// this lane's share of a[lo] + ... + a[hi - 1]
__device__ __forceinline__ unsigned long long lane_share(const unsigned long long* __restrict__ a, int lo, int hi,
                                                         int lane, int lanes) {
    unsigned long long v = 0;
    for (int i = lo + lane; i < hi; i += 4 * lanes) {
        unsigned long long q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] = i + u * lanes < hi ? a[i + u * lanes] : 0ull;
        v += (q[0] + q[1]) + (q[2] + q[3]);
    }
    return v;
}

// a count of cell c (one lane) added to its tile
__device__ __forceinline__ void add_cell_sum(const DevWork& w, int set, int c, unsigned long long v) {
    if (w.sums.fine && v) atomicAdd(&w.sums.tiles(set)[c / TILE], v);
}

// the fine sums into the tiles, a wavefront per tile (workgroups of 256)
__device__ __forceinline__ void add_fine_sums(const DevWork& w, int set, int bid, int nblk) {
    static_assert(TILE == 4 * WAVE, "a tile's fine sums: one per lane");
    if (!w.sums.fine) return;
    const int lane = threadIdx.x & (WAVE - 1), wv = threadIdx.x / WAVE;
    for (int t = bid * 4 + wv; t < w.sums.ntile; t += nblk * 4) {
        const int f = t * WAVE + lane;
        const unsigned long long v = wave_sum64(f < w.sums.nfine ? w.sums.fine[f] : 0ull);
        if (lane == 0 && v) atomicAdd(&w.sums.tiles(set)[t], v);
    }
}

// exclusive prefix of fs_cnt at cell c0 (a whole wavefront calls)
__device__ __forceinline__ unsigned long long cell_offset(const DevWork& w, int set, int c0) {
    if (!w.sums.fine) return w.fs_off[c0];
    const int lane = threadIdx.x & (WAVE - 1), t = c0 / TILE;
    return wave_sum64(lane_share(w.sums.tiles(set), 0, t, lane, WAVE) + lane_share(w.fs_cnt, t * TILE, c0, lane, WAVE));
}

// sum of all cells (a whole wavefront calls)
__device__ __forceinline__ unsigned long long cell_total(const DevWork& w, int set, int n_cells) {
    if (!w.sums.fine) return w.fs_off[n_cells];
    return wave_sum64(lane_share(w.sums.tiles(set), 0, w.sums.ntile, threadIdx.x & (WAVE - 1), WAVE));
}

// the first cell of a tile clears it in the set that the next census adds to
__device__ __forceinline__ void clear_next_sums(const DevWork& w, int set, int c) {
    if (w.sums.fine && c % TILE == 0) w.sums.tiles(set + 1)[c / TILE] = 0;
}

// u = sum_k N_k * F_k accumulated from zero over the cell's DoFs in order
// (velocity at a reference point)
template <int DIM, int DEG = 1>
__device__ __forceinline__ void interp(const double (*Fc)[DIM], const double* xi, double* u) {
    constexpr int ND = QF<DIM, DEG>::ND;
    double N[ND];
    shape_q<DIM, DEG>(xi, N);
#pragma unroll
    for (int d = 0; d < DIM; ++d) u[d] = 0.0;
#pragma unroll
    for (int k = 0; k < ND; ++k)
#pragma unroll
        for (int d = 0; d < DIM; ++d) u[d] += N[k] * Fc[k][d];
}

// the same with one node at a time (at(k): the velocity of node k), for a rare
// point: the nodes of a degree-2 cell held at once take the registers of a
// whole kernel (k_cell_write on degree-2 hexahedra: 408 -> 248)
template <int DIM, int DEG, class F>
__device__ __forceinline__ void interp_each(const double* xi, double* u, F at) {
#pragma unroll
    for (int d = 0; d < DIM; ++d) u[d] = 0.0;
#pragma unroll 1
    for (int k = 0; k < QF<DIM, DEG>::ND; ++k) {
        ShapeOne<DIM, DEG> N;
        N.init(k);
        const double nk = N(xi);
        const auto* f = at(k);
#pragma unroll
        for (int d = 0; d < DIM; ++d) u[d] += nk * (double)f[d];
    }
}

// Position of sum a (DoF a / (DIM + 1), component a % (DIM + 1)) of cell c
// among the cells' projection sums.  Degree-1 hexahedra: DoF by DoF, then cell
// by cell, so that k_node's neighbouring nodes, which read the same DoF of
// neighbouring cells, share 128-byte lines; with a cell's sums together each line
// was fetched by several XCDs for a quarter of it (202,240 hexahedra: k_node
// 32 -> 16 us and the write 79 either way in FP32-mixed, 35 -> 18 and 143 -> 146
// in FP64).  Elsewhere a cell's sums lie together: the
// scattered stores cost the write more than k_node gains (68,992 degree-2
// hexahedra: 97 -> 129 and 36 -> 23 us; 407,140 quads: 507 -> 520 and 25 -> 20).
template <int DIM, int DEG>
__device__ __forceinline__ size_t partial_at(int n_cells, int c, int a) {
    if constexpr (DIM == 3 && DEG == 1) {
        const int k = a / (DIM + 1);
        return ((size_t)k * n_cells + c) * (DIM + 1) + (a - k * (DIM + 1));
    }
    return (size_t)c * (QF<DIM, DEG>::ND * (DIM + 1)) + a;
}

template <int DIM>
__device__ __forceinline__ int part_key(const DevParams& pp, const double* xi) {
    // bits 0-15: part index with the phantom value q_d (the grouping key);
    // bits 16-23: 1 + ordinal of an in-range part, 0 for a phantom part
    int key = 0, stride = 1, ord = 0;
    bool in = true;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        // xi_d / h truncated: h is 1/q (middle exponents), and a xi_d below
        // them truncates to 0 either way
        const double h = pp.hq[d];
        const unsigned num = (unsigned)div_refined(xi[d], h, rcp_refined(h));
        key += (int)num * stride;
        stride *= pp.q[d] + 1;
        in = in && (int)num < pp.q[d];
        ord = ord * pp.q[d] + (int)num;
    }
    return key | ((in ? ord + 1 : 0) << 16);
}

// in-range part ordinal of a packed part key, -1 for a phantom part
__device__ __forceinline__ int part_ordinal(int pkey) { return (pkey >> 16) - 1; }

template <int DIM>
__device__ __forceinline__ void lattice_point(const DevParams& pp, int ordinal, double* xi) {
    int num[3];
    int o = ordinal;
#pragma unroll
    for (int d = DIM - 1; d >= 0; --d) {
        num[d] = o % pp.q[d];
        o /= pp.q[d];
    }
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        const double h = pp.hq[d];
        xi[d] = (num[d] + 1.0 / 2) * h;
    }
}

// Face through which the step from xold to x most likely left the cell: the
// linearised reference displacement J(xi_old)^-1 (x - xold) added to xi_old,
// the component furthest outside [0, 1] (face 2a + s is xi_a = s), -1 if
// none.  Only a guess, which the caller verifies: it rounds as it likes
// (fused multiply-adds) and scales by det J instead of dividing (a cell with
// det <= 0 gets an arbitrary face).
template <int DIM>
__device__ __forceinline__ int exit_face(const double (*P)[DIM], const double* xi_old, const double* xold,
                                         const double* x) {
    double J[DIM][DIM], Ji[DIM][DIM], dx[DIM];   // J[i][j] = d x_i / d xi_j
#pragma unroll
    for (int i = 0; i < DIM; ++i) {
        if constexpr (DIM == 2) {
            const double e0 = P[1][i] - P[0][i], e1 = P[2][i] - P[0][i], w = (P[3][i] - P[2][i]) - e0;
            J[i][0] = fma(w, xi_old[1], e0);
            J[i][1] = fma(w, xi_old[0], e1);
        } else {
            const double a = xi_old[0], b = xi_old[1], c = xi_old[2];
            // edge differences interpolated over the opposite directions
            auto lin = [&](double t, double lo, double hi) { return fma(t, hi - lo, lo); };
            J[i][0] = lin(c, lin(b, P[1][i] - P[0][i], P[3][i] - P[2][i]), lin(b, P[5][i] - P[4][i], P[7][i] - P[6][i]));
            J[i][1] = lin(c, lin(a, P[2][i] - P[0][i], P[3][i] - P[1][i]), lin(a, P[6][i] - P[4][i], P[7][i] - P[5][i]));
            J[i][2] = lin(b, lin(a, P[4][i] - P[0][i], P[5][i] - P[1][i]), lin(a, P[6][i] - P[2][i], P[7][i] - P[3][i]));
        }
    }
    auto cof = [](double a, double b, double c, double d) { return fma(a, d, -(b * c)); };
    if constexpr (DIM == 2) {
        Ji[0][0] = J[1][1];
        Ji[0][1] = -J[0][1];
        Ji[1][0] = -J[1][0];
        Ji[1][1] = J[0][0];
    } else {
        Ji[0][0] = cof(J[1][1], J[1][2], J[2][1], J[2][2]);
        Ji[0][1] = cof(J[0][2], J[0][1], J[2][2], J[2][1]);
        Ji[0][2] = cof(J[0][1], J[0][2], J[1][1], J[1][2]);
        Ji[1][0] = cof(J[1][2], J[1][0], J[2][2], J[2][0]);
        Ji[1][1] = cof(J[0][0], J[0][2], J[2][0], J[2][2]);
        Ji[1][2] = cof(J[0][2], J[0][0], J[1][2], J[1][0]);
        Ji[2][0] = cof(J[1][0], J[1][1], J[2][0], J[2][1]);
        Ji[2][1] = cof(J[0][1], J[0][0], J[2][1], J[2][0]);
        Ji[2][2] = cof(J[0][0], J[0][1], J[1][0], J[1][1]);
    }
    double det = J[0][0] * Ji[0][0];
#pragma unroll
    for (int j = 1; j < DIM; ++j) det = fma(J[0][j], Ji[j][0], det);
#pragma unroll
    for (int d = 0; d < DIM; ++d) dx[d] = x[d] - xold[d];
    int f = -1;
    double worst = 0.0;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        double e = xi_old[d] * det;   // det * (reference coordinate after the move)
#pragma unroll
        for (int j = 0; j < DIM; ++j) e = fma(Ji[d][j], dx[j], e);
        const double o = e < 0.0 ? -e : e - det;
        if (o > worst) {
            worst = o;
            f = 2 * d + (e < 0.0 ? 0 : 1);
        }
    }
    return f;
}

// The vertex of cell c that the velocity points at most from xold: the
// largest product of the normalised velocity and the normalised direction to
// the vertex, the first on ties (cylinder2D/pfem2particle.cpp:283-300).  Only
// the choice matters, so it is made with v_rsq_f64 estimates (relative error
// below 2^-20) of |velocity| times the products wherever the largest leads
// the next by more than 2^-14 |velocity| and the squares are in the middle of
// the exponent range; the definition's square roots and divisions decide the
// rest (about one in ten thousand).  9 instead of ~45 instructions a vertex.
template <int DIM>
__device__ __forceinline__ int star_vertex(const DevMesh<DIM>& m, int c, const double (*P)[DIM], const double* xold,
                                           const double* vext) {
    constexpr int NV = Q1<DIM>::NV;
    double best = -1e300, next = -1e300, lo = 1e300, sum = 0.0;
    int cvk = 0;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        double t = P[k][0] - xold[0];
        double s2 = t * t, dot = vext[0] * t;
#pragma unroll
        for (int d = 1; d < DIM; ++d) {
            t = P[k][d] - xold[d];
            s2 = fma(t, t, s2);
            dot = fma(vext[d], t, dot);
        }
        const double a = dot * __builtin_amdgcn_rsq(s2);
        const bool g = a > best;
        next = g ? best : (a > next ? a : next);
        best = g ? a : best;
        cvk = g ? k : cvk;
        lo = s2 < lo ? s2 : lo;
        sum += s2;
    }
    double v2 = vext[0] * vext[0];
#pragma unroll
    for (int d = 1; d < DIM; ++d) v2 = fma(vext[d], vext[d], v2);
    const double lead = best - next;
    if ((lead > 0.0) & (lead * lead > 0x1p-28 * v2) & (v2 > 0x1p-900) & (v2 < 0x1p900) & (lo > 0x1p-900) &
        (sum < 0x1p900))
        return cvk;
    double vn[DIM], a0 = 0.0;
    const double rv = 1.0 / vnorm<DIM>(vext);
#pragma unroll
    for (int d = 0; d < DIM; ++d) vn[d] = vext[d] * rv;
    cvk = 0;
#pragma unroll 1
    for (int k = 0; k < NV; ++k) {
        const double* p = m.cellX + ((size_t)c * NV + k) * DIM;
        double t[DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d) t[d] = p[d] - xold[d];
        const double rn = 1.0 / vnorm<DIM>(t);
#pragma unroll
        for (int d = 0; d < DIM; ++d) t[d] *= rn;
        const double a = vdot<DIM>(vn, t);
        if (k == 0 || a > a0) {
            cvk = k;
            a0 = a;
        }
    }
    return cvk;
}

// margin in reference coordinates beyond which a point inside one cell is
// inside no other cell under the containment test (the Newton acceptance
// radius is 1e-10 of a cell diameter)
constexpr double NBR_MARGIN = 1e-6;

template <int DIM>
__device__ __forceinline__ bool inside_margin(const double* r) {
    bool in = true;
#pragma unroll
    for (int d = 0; d < DIM; ++d) in = in & (r[d] >= NBR_MARGIN) & (r[d] <= 1.0 - NBR_MARGIN);
    return in;
}

// inverse_map and the unit-cell test of a candidate cell
template <int DIM>
__device__ __forceinline__ bool contains(const DevMesh<DIM>& m, int c, const double (*Q)[DIM], const double* x,
                                         double* r) {
    if constexpr (DIM == 3) {
        HexCell H;
        H.load(m.ftol + (size_t)c * HEX_N);
        return hex_map(Q, H, x, r) && inside_unit<DIM>(r);
    } else {
        return inverse_map<DIM>(Q, x, r, m.ftol[c], true) && inside_unit<DIM>(r);
    }
}

// Relocation of a particle whose position left cell c
// (pfem2ParticleHandler::sort_particles_into_subdomains_and_cells, the part
// after the own-cell test, cylinder2D/pfem2particle.cpp:278-386).  The
// reference sorts the star of the selected vertex by decreasing alignment
// (stable for equal keys) and takes the first cell that contains the point;
// that is the containing cell with the largest key, earliest star position on
// ties, which is what the loop below selects.  Returns -1 if no star cell
// contains the point.
//
// `Q` returns the vertices of the cell found.  (A caller's other data of the
// cell, loaded with each candidate's vertices to overlap the two loads, cost
// more in registers than it saved: without it the searches took 8-12% less.)
//
// OWN and own (2-D): the own-cell test's clearly-outside test said no and the
// rest of it is pending; only that test runs: c is returned if it places x in
// cell c, else RELOC_AGAIN, and the caller comes back for the search.
//
// The own cell and the star cells go through one inlined inverse map: the
// code of its Newton iteration is large, and with four copies of it the
// search kernels missed the instruction cache.
constexpr int RELOC_AGAIN = -2;

template <int DIM, bool SHORTCUT, bool OWN>
__device__ __forceinline__ int relocate(const DevMesh<DIM>& m, int c, const double (*P)[DIM], const double* xi_old,
                                        const double* vext, const double* x, double* xi_out, double (*Q)[DIM],
                                        int& searches, bool own) {
    constexpr int NV = Q1<DIM>::NV;
    constexpr int CH = 4;   // star entries read together
    int s0 = 0, n = 0, last = -1;
    double dir[DIM], lastkey = 0.0;
    // the selected vertex and its star; the face-neighbour shortcut (its cell, or -1)
    auto select = [&]() -> int {
        ++searches;
        int nb[2 * DIM];
        if constexpr (SHORTCUT) {
#pragma unroll
            for (int h = 0; h < DIM - 1; ++h) {
                const int4 q = m.cell_nbr[(size_t)c * (DIM - 1) + h];
                nb[4 * h] = q.x;
                nb[4 * h + 1] = q.y;
                if (4 * h + 2 < 2 * DIM) nb[4 * h + 2] = q.z;
                if (4 * h + 3 < 2 * DIM) nb[4 * h + 3] = q.w;
            }
        }
        double xold[DIM];
        forward<DIM>(P, xi_old, xold);
        const int cvk = star_vertex<DIM>(m, c, P, xold, vext);
        if constexpr (SHORTCUT) {
            // Face-neighbour shortcut.  The neighbour g across the exit face
            // is in the selected vertex's star when that vertex lies on the
            // face; if g contains x at least NBR_MARGIN inside, no other cell
            // contains x, so g is the first containing cell of the star in
            // any order: the star loop's result, with the same inverse map
            // (2-D: its closed form, which alone places a point there but
            // for a few that the star loop then finds).
            const int f = exit_face<DIM>(P, xi_old, xold, x);
            int g = -1;
#pragma unroll
            for (int q = 0; q < 2 * DIM; ++q)
                if (f == q && ((cvk >> (q >> 1)) & 1) == (q & 1)) g = nb[q];
            if (g >= 0) {
                load_vertices<DIM>(m, g, Q);
                double r[DIM];
                bool in;
                if constexpr (DIM == 2) {
                    QuadCell qc;
                    qc.init(Q);
                    in = closed_form(Q, qc, x, r) == 0;
                } else {
                    HexCell H;
                    H.load(m.ftol + (size_t)g * HEX_N);
                    in = hex_map(Q, H, x, r);
                }
                if (in && inside_margin<DIM>(r)) {
#pragma unroll
                    for (int d = 0; d < DIM; ++d) xi_out[d] = r[d];
                    return g;
                }
            }
        }
        const int2 se = m.cell_star[(size_t)c * NV + cvk];
        s0 = se.x;
        n = se.y - se.x;
#pragma unroll
        for (int d = 0; d < DIM; ++d) dir[d] = x[d] - m.cellX[((size_t)c * NV + cvk) * DIM + d];
        const double rn = 1.0 / vnorm<DIM>(dir);
#pragma unroll
        for (int d = 0; d < DIM; ++d) dir[d] *= rn;
        return -1;
    };
    const bool one = OWN && own;
    if (!one) {
        const int g = select();
        if (g >= 0) return g;
    }
    for (int it = 0;; ++it) {
        int cc = c;
        if (one) {
            if (it > 0) return RELOC_AGAIN;
        } else {
            // star candidates in decreasing key order (ties: star order),
            // first containing cell wins -- the reference's sorted loop,
            // stopping early.  Each pass re-reads the star (cache hits, CH
            // entries at a time) for the first entry after the last one
            // tried.  (x on the selected vertex: keys are NaN, star order.)
            if (it >= n) return -1;
            int be = -1;
            double bk = 0.0;
            for (int e0 = 0; e0 < n; e0 += CH) {
                double key[CH];
                int cell[CH];
#pragma unroll
                for (int u = 0; u < CH; ++u) {
                    const int e = e0 + u < n ? e0 + u : n - 1;
                    double sd[DIM];
#pragma unroll
                    for (int d = 0; d < DIM; ++d) sd[d] = m.star_dir[(size_t)(s0 + e) * DIM + d];
                    key[u] = vdot<DIM>(sd, dir);
                    if (!(key[u] == key[u])) key[u] = 0.0;
                    cell[u] = m.star_cell[s0 + e];
                }
#pragma unroll
                for (int u = 0; u < CH; ++u) {
                    const int e = e0 + u;
                    const bool left = it == 0 || key[u] < lastkey || (key[u] == lastkey && e > last);
                    if (e < n && left && (be < 0 || key[u] > bk)) {
                        be = e;
                        bk = key[u];
                        cc = cell[u];
                    }
                }
            }
            last = be;
            lastkey = bk;
        }
        double r[DIM];
        load_vertices<DIM>(m, cc, Q);
        if (contains<DIM>(m, cc, Q, x, r)) {
#pragma unroll
            for (int d = 0; d < DIM; ++d) xi_out[d] = r[d];
            return cc;
        }
    }
}

// ---------------------------------------------------------------------------
// Advection substeps (move_particles, TurekBenchmark/pfem2particle.cpp:813-856).
// Particles are independent within move_particles, so the substeps of one
// particle run back to back in registers: u = sum N_k V_k at the current
// reference point, velocity_ext = u, x += (dt/S) u, then the own-cell test
// (pfem2ParticleHandler::sort_particles_into_subdomains_and_cells,
// TurekBenchmark/pfem2particle.cpp:286-302).  A particle whose own-cell test
// fails is parked (position advanced, old reference point, velocity_ext and
// substep index stored) and queued; the vertex-star searches of all queued
// particles then run the vertex-star search in full wavefronts, which
// continue the remaining substeps.
//   One search round (k_search_resume, k_search_resume32), whose lanes follow
//   their particle through every further crossing and refill from the queue
//   when it is done (search_body).
// the queue segments of the refilling search (one cursor each, on its own
// cache line: a single cursor for the whole grid serialises the wavefronts'
// atomics) and the idle lanes a wavefront gathers before it refills
constexpr int RSEGS = 256;
constexpr int REFILL_MIN = 16;
// the counters of the move's queue are round 0's; the next round's hold the
// cursors (cleared with the queue counters after each regroup)
constexpr int CURSOR_ROUND = 1;
// the queue of the re-sort's relocations after a mesh move (both paths)
constexpr int RESORT_QUEUE = 2;
// rounds of the counters: the move's queue, the cursors, the re-sort
constexpr int NQROUNDS = 3;

// Queues of parked particles, the move's and the re-sort's (never filled at
// the same time) in one buffer.  A queue is QSHARDS shards of shard_cap entries plus an overflow
// region of cap entries; each shard's counter sits on its own 128-byte line
// and a wavefront appends to shard (wavefront id mod QSHARDS) with one atomic.
constexpr int QSHARDS = 256;
constexpr int QSTRIDE = 32;   // ints between shard counters

struct DevQueues {
    int2* data;           // (particle, cell): QSHARDS * shard_cap + overflow
    int* count;           // NQROUNDS rounds x (QSHARDS + 1) counters, QSTRIDE apart
    int* prefix;          // per round: QSHARDS + 2 ints (exclusive prefix, overflow start, total); round 1:
                          // QSHARDS partial counts of particles searched for again (FP32-mixed)
    int shard_cap;
    double* park_vext;    // DIM x cap: velocity_ext of a parked particle
    int* park_s;          // substep index of a parked particle
};

// Loops of wavefronts over n items (particles or queue entries): the
// wavefront handles items base + lane for base = begin, begin + step, ...
// below end, and appends to queue shard `shard`.  Shards follow the item
// order, so a queue keeps the order of the particles (stored by cell) up to
// the order within a shard, and the searches of one wavefront touch nearby
// cells.
struct WaveLoop {
    int begin, end, step, shard;
};

// The workgroups a kernel body loops over: the hardware grid, or, in a
// batched launch that steps several simulations at once, the simulation's
// own range of the launch's workgroups (index within it and its size).
struct Grid {
    unsigned bid, nblk;
};
__device__ __forceinline__ Grid hw_grid() { return Grid{blockIdx.x, gridDim.x}; }

// Both loops work in 32-bit unsigned arithmetic on wavefront-uniform values
// (grids of at most 2^16 workgroups, n < 2^31), which the compiler keeps in
// scalar registers: a 64-bit division per wavefront costs more vector
// instructions than a substep.

// grid-stride: wavefront k takes chunks k, k + W, ... of WAVE items
__device__ __forceinline__ WaveLoop stride_loop(int n, Grid G = hw_grid()) {
    const unsigned wpb = blockDim.x / WAVE, nw = G.nblk * wpb;
    const unsigned k = G.bid * wpb + (unsigned)__builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    WaveLoop L;
    L.begin = (int)(k * WAVE);
    L.end = n;
    L.step = (int)(nw * WAVE);
    L.shard = (int)(k * QSHARDS / nw);
    return L;
}

// one contiguous range of whole workgroup-sized chunks per workgroup, the
// wavefronts of a workgroup interleaved within it
__device__ __forceinline__ WaveLoop range_loop(int n, Grid G = hw_grid()) {
    const unsigned g = G.nblk, b = G.bid, un = (unsigned)n;
    const unsigned per = ((un + g - 1) / g + blockDim.x - 1) / blockDim.x * blockDim.x;
    const unsigned long long b0l = (unsigned long long)b * per;
    const unsigned b0 = b0l < un ? (unsigned)b0l : un;
    const unsigned wpb = blockDim.x / WAVE, wv = (unsigned)__builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    WaveLoop L;
    L.begin = (int)(b0 + wv * WAVE);
    L.end = (int)(un - b0 > per ? b0 + per : un);
    L.step = blockDim.x;
    L.shard = (int)((b * wpb + wv) * QSHARDS / (g * wpb));
    return L;
}

__device__ __forceinline__ int* queue_count(const DevQueues& qu, int round, int shard) {
    return qu.count + ((size_t)round * (QSHARDS + 1) + shard) * QSTRIDE;
}

// append `value` to shard `sh` for the lanes with pred set (all lanes of the
// wavefront call)
__device__ __forceinline__ void queue_push(const DevQueues& qu, int round, bool pred, int2 value, int sh) {
    const unsigned long long mask = __ballot(pred);
    if (mask == 0) return;
    const int lane = threadIdx.x & (WAVE - 1);
    const int leader = __ffsll((long long)mask) - 1;
    int base = 0;
    if (lane == leader) base = atomicAdd(queue_count(qu, round, sh), __popcll(mask));
    base = __shfl(base, leader);
    const int slot = base + __popcll(mask & ((1ull << lane) - 1));
    const bool spill = pred && slot >= qu.shard_cap;
    int2* data = qu.data;
    if (pred && !spill) data[(size_t)sh * qu.shard_cap + slot] = value;
    const unsigned long long smask = __ballot(spill);
    if (smask == 0) return;
    const int l2 = __ffsll((long long)smask) - 1;
    int ob = 0;
    if (lane == l2) ob = atomicAdd(queue_count(qu, round, QSHARDS), __popcll(smask));
    ob = __shfl(ob, l2);
    if (spill) data[(size_t)QSHARDS * qu.shard_cap + ob + __popcll(smask & ((1ull << lane) - 1))] = value;
}

// Exclusive prefix of the valid entries per shard, then the overflow start
// and the total, computed by each workgroup of the search kernel from the
// shard counters (blockDim.x == QSHARDS: one thread per shard; the counters
// are a few cache lines, so the redundant work costs less than a launch).
// Workgroup 0 also stores it for diagnostics.
__device__ __forceinline__ int queue_prefix(const DevQueues& qu, int round, int* s_pref, Grid G = hw_grid()) {
    __shared__ int s_wave[QSHARDS / WAVE];
    const int t = threadIdx.x;
    const int lane = t & (WAVE - 1), wv = t / WAVE;
    int v = *queue_count(qu, round, t);
    v = v < qu.shard_cap ? v : qu.shard_cap;
    int incl = v;
#pragma unroll
    for (int off = 1; off < WAVE; off <<= 1) {
        const int o = __shfl_up(incl, off);
        if (lane >= off) incl += o;
    }
    if (lane == WAVE - 1) s_wave[wv] = incl;
    __syncthreads();
    int wbase = 0;
    for (int q = 0; q < wv; ++q) wbase += s_wave[q];
    s_pref[t] = wbase + incl - v;
    if (t == QSHARDS - 1) {
        const int tot = wbase + incl;
        s_pref[QSHARDS] = tot;
        s_pref[QSHARDS + 1] = tot + *queue_count(qu, round, QSHARDS);
    }
    __syncthreads();
    if (G.bid == 0) {
        int* pref = qu.prefix + (size_t)round * (QSHARDS + 2);
        pref[t] = s_pref[t];
        if (t < 2) pref[QSHARDS + t] = s_pref[QSHARDS + t];
    }
    return s_pref[QSHARDS + 1];
}

// particle index of queue entry j
__device__ __forceinline__ int2 queue_get(const DevQueues& qu, const int* s_pref, int j) {
    const int2* data = qu.data;
    if (j >= s_pref[QSHARDS]) return data[(size_t)QSHARDS * qu.shard_cap + (j - s_pref[QSHARDS])];
    int lo = 0, hi = QSHARDS - 1;   // last shard with s_pref <= j
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (s_pref[mid] <= j) lo = mid;
        else hi = mid - 1;
    }
    return data[(size_t)lo * qu.shard_cap + (j - s_pref[lo])];
}

// A parked particle whose own-cell test k_move left to the search kernel
// (flag in its parked substep index)
constexpr int PARK_NEWTON = 1 << 30;
// destination mark of a particle that a pending census kept (k_cell_pend):
// destination = cell | DEST_KEPT (cell indices stay below 2^25 there)
constexpr int DEST_KEPT = 1 << 30;

// Runs substeps until done (returns 0) or the own-cell test fails (returns
// 1; s is the substep whose test failed).
// 2-D: the own-cell test takes only inverse_map's closed form and returns 2
// where inverse_map would go on to its clearly-outside test and
// Newton iteration (the point is outside the closed form's unit square, or
// closed_form leaves it undecided); the search finishes that test
// (relocate's `own`).  This keeps the Newton code, and its registers, out of
// k_move: 94 instead of 167 registers, 5 instead of 3 wavefronts per SIMD.
//
// 3-D, degree 2: the 81 nodal velocities of a cell are read in every substep
// (the lanes of a wavefront share a few cells, so the reads hit L1) instead of
// held in 162 registers, which spilled.
template <int DIM, int DEG = 1>
__device__ __forceinline__ int advance64(const DevMesh<DIM>& m, const DevParams& pp, const DevParticles& A, int i, int c,
                                         double* x, double* xi, double* vext, int& s, const double (*P)[DIM]) {
    constexpr int ND = QF<DIM, DEG>::ND;
    constexpr bool REREAD = DIM == 3 && DEG == 2;
    const double* cf = m.cellV + (size_t)c * ND * DIM;
    double Vc[REREAD ? 1 : ND][DIM];
    if constexpr (!REREAD)
#pragma unroll
        for (int k = 0; k < ND; ++k)
#pragma unroll
            for (int d = 0; d < DIM; ++d) Vc[k][d] = cf[k * DIM + d];
    QuadCell qc;
    HexCell H;
    if constexpr (DIM == 2) qc.init(P);
    else H.load(m.ftol + (size_t)c * HEX_N);
    for (; s < pp.substeps; ++s) {
        double u[DIM];
        if constexpr (REREAD) {
            // (an address the compiler cannot carry from one substep to the
            // next, or it loads the values once and spills them)
            const double* f = cf;
            asm volatile("" : "+v"(f));
            double N[ND];
            shape_q<DIM, DEG>(xi, N);
#pragma unroll
            for (int d = 0; d < DIM; ++d) u[d] = 0.0;
#pragma unroll
            for (int k = 0; k < ND; ++k)
#pragma unroll
                for (int d = 0; d < DIM; ++d) u[d] += N[k] * f[k * DIM + d];
        } else {
            interp<DIM, DEG>(Vc, xi, u);
        }
#pragma unroll
        for (int d = 0; d < DIM; ++d) vext[d] = u[d];
#pragma unroll
        for (int d = 0; d < DIM; ++d) u[d] *= pp.h;
#pragma unroll
        for (int d = 0; d < DIM; ++d) x[d] = x[d] + u[d];
        if (pp.keep_vext && s == pp.substeps - 1)
#pragma unroll
            for (int d = 0; d < DIM; ++d) A.vext[(size_t)d * A.cap + i] = vext[d];
        double r[DIM];
        int st;
        if constexpr (DIM == 2) st = closed_form(P, qc, x, r);
        else st = hex_map(P, H, x, r) && inside_unit<DIM>(r) ? 0 : 1;
        if (st) return st;
#pragma unroll
        for (int d = 0; d < DIM; ++d) xi[d] = r[d];
    }
    return 0;
}

// final bookkeeping of a particle whose substeps are complete (all lanes call)
// (seg_end: particles from it on, new particles of a pending layout, are in
// no cell's segment, so they arrive in their cell)
template <int DIM>
__device__ __forceinline__ void finish_particle(const DevParams& pp, const DevParticles& A, const DevWork& w,
                                                bool valid, int i, int c, const double* x, const double* xi,
                                                bool write_state, int seg_end = 0x7fffffff) {
    add_arrival(w, valid && c >= 0 && (c != A.cell[valid ? i : 0] || i >= seg_end), c, i);
    if (!valid) return;
    if (write_state) {
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            A.x[(size_t)d * A.cap + i] = x[d];
            A.xi[(size_t)d * A.cap + i] = xi[d];
        }
    }
    w.dest[i] = c;
    if (c >= 0) w.pkey[i] = part_key<DIM>(pp, xi);
}

// park a particle for the search of the next round (all lanes call)
template <int DIM>
__device__ __forceinline__ void park_particle(const DevParticles& A, const DevWork& w, const DevQueues& qu,
                                              int round_out, int shard, bool park, int i, int c,
                                              const double* x, const double* xi, const double* vext, int s) {
    queue_push(qu, round_out, park, make_int2(i, c), shard);
    if (!park) return;
    qu.park_s[i] = s;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        A.x[(size_t)d * A.cap + i] = x[d];
        A.xi[(size_t)d * A.cap + i] = xi[d];
        qu.park_vext[(size_t)d * A.cap + i] = vext[d];
    }
}

// k_move: [correction] + substeps until done or the first failed own-cell test.
//   correct_particles_velocities  TurekBenchmark/pfem2particle.cpp:792-811
template <int DIM, int DEG = 1>
__device__ __forceinline__ void move_body(const Grid& G, const DevMesh<DIM>& m, const DevParticles& A,
                                          const DevParams& pp, const DevWork& w, const DevQueues& qu, int do_correct, int do_move) {
    constexpr int NV = Q1<DIM>::NV;
    constexpr int ND = QF<DIM, DEG>::ND;
    // a pending layout (k_cell_pend): its slots, the current cell of a kept
    // particle in dest (with DEST_KEPT), new particles from the segment end on
    const int pn = w.counters[6];
    const int n = state_dead(w.counters) ? 0 : (pn > 0 ? pn : w.counters[0]);
    const int seg_end = pn > 0 ? w.counters[7] : 0x7fffffff;
    const int lane = threadIdx.x & (WAVE - 1);
    // every particle that exists now ends this advection with xi from an
    // inverse map (the re-sort after a mesh move relies on it)
    if (do_move && G.bid == 0 && threadIdx.x == 0) w.counters[5] = (int)*w.particle_counter;
    const WaveLoop L = stride_loop(n, G);
    for (int base = L.begin; base < L.end; base += L.step) {
        const int i = base + lane;
        bool valid = i < L.end;
        int c = 0;
        if (valid && pn > 0) {
            const int dk = w.dest[i];
            c = dk & ~DEST_KEPT;
            if (dk < 0 || !(dk & DEST_KEPT)) {
                // not kept by the pending census: gone (no cell, no arrival)
                w.dest[i] = -1;
                valid = false;
            }
        } else if (valid) {
            c = A.cell[i];
        }
        double x[DIM], xi[DIM], vext[DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d) xi[d] = valid ? A.xi[(size_t)d * A.cap + i] : 0.5;
        if (do_correct && valid) {
            double v[DIM], N[ND];
#pragma unroll
            for (int d = 0; d < DIM; ++d) v[d] = A.v[(size_t)d * A.cap + i];
            shape_q<DIM, DEG>(xi, N);
            const double* dv = m.cellDV + (size_t)c * ND * DIM;
#pragma unroll
            for (int k = 0; k < ND; ++k)
#pragma unroll
                for (int d = 0; d < DIM; ++d) v[d] = v[d] + N[k] * dv[k * DIM + d];
#pragma unroll
            for (int d = 0; d < DIM; ++d) A.v[(size_t)d * A.cap + i] = v[d];
        }
        if (!do_move) continue;
        int st = 0, s = 0;
        if (valid) {
#pragma unroll
            for (int d = 0; d < DIM; ++d) x[d] = A.x[(size_t)d * A.cap + i];
            double P[NV][DIM];
            load_vertices<DIM>(m, c, P);
            st = advance64<DIM, DEG>(m, pp, A, i, c, x, xi, vext, s, P);
        }
        park_particle<DIM>(A, w, qu, 0, L.shard, valid && st != 0, i, c, x, xi, vext, st == 2 ? s | PARK_NEWTON : s);
        finish_particle<DIM>(pp, A, w, valid && st == 0, i, c, x, xi, true, seg_end);
    }
}

template <int DIM, int DEG = 1>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(DIM == 2 ? (DEG == 1 ? 5 : 3) : 2))) k_move(DevMesh<DIM> m, DevParticles A, DevParams pp,
                                              DevWork w, DevQueues qu, int do_correct, int do_move) {
    move_body<DIM, DEG>(hw_grid(), m, A, pp, w, qu, do_correct, do_move);
}

// Queue entries for the lanes of a search wavefront that hold no particle.
// The queue is dealt in chunks of WAVE entries to segments (as many as the
// grid has wavefronts, up to RSEGS, so every segment has a wavefront), chunk k
// to segment k mod nseg: the particles with long crossing chains lie together
// (around the obstacle), and with one contiguous range a segment its few
// wavefronts were still searching when the others had left (101,785 quads: FP64
// search 208 -> 163 us, FP32-mixed 215 -> 153; 202,240 hexahedra, FP32-mixed
// 145 -> 140).  Where the long chains are few it costs the neighbourhood that
// consecutive chunks share: 407,140 quads 479 -> 490 in FP64 (FP32-mixed the
// same), 68,992 degree-2 hexahedra 198 -> 207.  The segment's cursor advances
// by one returning atomic once REFILL_MIN lanes are idle or all are (8 or 32: the
// same).
struct Refill {
    int* cursor;
    int n, seg, nseg;
    bool more;   // wavefront-uniform: the segment may hold further entries
    __device__ __forceinline__ Refill(const DevQueues& qu, int n_, const Grid& G) : n(n_), more(true) {
        const unsigned wpb = blockDim.x / WAVE, nwv = G.nblk * wpb;
        const unsigned gw = G.bid * wpb + (unsigned)__builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
        nseg = (int)(nwv < (unsigned)RSEGS ? nwv : (unsigned)RSEGS);
        seg = (int)(gw % (unsigned)nseg);
        cursor = queue_count(qu, CURSOR_ROUND, seg);
    }
    // queue entry of position p in the segment
    __device__ __forceinline__ long long entry(int p) const {
        return ((long long)(p / WAVE) * nseg + seg) * WAVE + p % WAVE;
    }
    // the queue entry for this lane or -1 (all lanes call; have: it holds a particle)
    __device__ __forceinline__ int next(bool have, int lane) {
        if (!more) return -1;
        const unsigned long long need = __ballot(!have);
        const int k = __popcll(need);
        if (need == 0 || (k < REFILL_MIN && need != ~0ull)) return -1;
        const int leader = __ffsll((long long)need) - 1;
        int base = 0;
        if (lane == leader) base = atomicAdd(cursor, k);
        base = __builtin_amdgcn_readlane(base, leader);
        more = entry(base + k) < n;
        const long long j = entry(base + __popcll(need & ((1ull << lane) - 1)));
        return !have && j < n ? (int)j : -1;
    }
};

// k_search_resume: the vertex-star search of the parked particles, then
// their remaining substeps, in one round.  A lane follows its particle
// through every further crossing and, when the particle is done, refills
// from the queue: the wavefront's segment of the queue has a cursor (one
// returning atomic per wavefront and refill, taken once REFILL_MIN lanes are
// idle or all are), so a wavefront does not wait for its longest crossing
// chain before it takes new particles, and no particle is parked twice.
// Every iteration settles a pending own-cell test or makes one search, then the
// substeps up to the next exit; a test that says no comes back as a search, and
// every other iteration consumes a substep, so each lane ends, and a wavefront leaves when its
// segment is drained and none of its lanes holds a particle.
template <int DIM, int DEG = 1, bool RESORT = false>
__device__ __forceinline__ void search_body(const Grid& G, const DevMesh<DIM>& m, const DevParticles& A,
                                            const DevParams& pp, const DevWork& w, const DevQueues& qu,
                                            int round) {
    constexpr int NV = Q1<DIM>::NV;
    __shared__ int s_pref[QSHARDS + 2];
    const int n = queue_prefix(qu, round, s_pref, G);
    // new particles of a pending layout (from its segment end on) arrive in their cell
    const int seg_end = !RESORT && w.counters[6] > 0 ? w.counters[7] : 0x7fffffff;
    const int lane = threadIdx.x & (WAVE - 1);
    Refill F(qu, n, G);
    int lost = 0, searches = 0;
    bool have = false, newton = false;
    int i = 0, c = 0, s = 0;
    double x[DIM], xi[DIM], vext[DIM], P[NV][DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) x[d] = xi[d] = vext[d] = 0.0;
    for (;;) {
        const int j = F.next(have, lane);
        if (j >= 0) {
            const int2 e = queue_get(qu, s_pref, j);
            i = e.x;
            c = e.y;
            const int ps = qu.park_s[i];
            s = ps & ~PARK_NEWTON;
            newton = (ps & PARK_NEWTON) != 0;
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                x[d] = A.x[(size_t)d * A.cap + i];
                xi[d] = A.xi[(size_t)d * A.cap + i];
                vext[d] = qu.park_vext[(size_t)d * A.cap + i];
            }
            load_vertices<DIM>(m, c, P);
            have = true;
        }
        if (__ballot(have) == 0) break;
        bool done = false;
        if (have) {
            // a particle whose own-cell test is pending (2-D): clearly
            // outside, it goes to the search; otherwise relocate runs the rest
            // of the test first
            const bool own = DIM == 2 && newton && !clearly_outside<DIM>(P, x, m.ftol[c]);
            newton = false;
            // (3-D moves go without the face-neighbour shortcut: it made this
            // kernel spill heavily before the cells' tables (HexCell).  With
            // them the two are close: 207 us without, 200 with on 68,992
            // degree-2 hexahedra, 242 and 238 on 202,240 of degree 1.)
            double Q[NV][DIM], r[DIM];
            const int cn =
                relocate<DIM, DIM == 2 || RESORT, DIM == 2>(m, c, P, xi, vext, x, r, Q, searches, own);
            done = cn == -1;
            if (cn >= 0) {
#pragma unroll
                for (int d = 0; d < DIM; ++d) xi[d] = r[d];
                if constexpr (RESORT) {
                    done = true;   // re-sort after a mesh move: no advection
                } else {
                    ++s;
#pragma unroll
                    for (int k = 0; k < NV; ++k)
#pragma unroll
                        for (int d = 0; d < DIM; ++d) P[k][d] = Q[k][d];
                    // (2-D: a test the closed form does not decide comes back
                    // as pending, as from k_move)
                    const int st = advance64<DIM, DEG>(m, pp, A, i, cn, x, xi, vext, s, P);
                    done = st == 0;
                    newton = st == 2;
                }
            }
            if (cn != RELOC_AGAIN) c = cn;
            if (cn == -1) ++lost;
        }
        finish_particle<DIM>(pp, A, w, done, i, c, x, xi, true, seg_end);
        if (done) have = false;
    }
    wave_stat(w.stats, 0, lost);
    wave_stat(w.stats, 3, searches);
}

template <int DIM, int DEG = 1>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(DIM == 2 ? 3 : 2))) k_search_resume(DevMesh<DIM> m, DevParticles A, DevParams pp, DevWork w, DevQueues qu,
                                                       int round) {
    search_body<DIM, DEG>(hw_grid(), m, A, pp, w, qu, round);
}

// the relocations of the re-sort after a mesh move (queue RESORT_QUEUE)
template <int DIM>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(DIM == 2 ? 3 : 2))) k_resort_search(DevMesh<DIM> m, DevParticles A, DevParams pp, DevWork w, DevQueues qu) {
    search_body<DIM, 1, true>(hw_grid(), m, A, pp, w, qu, RESORT_QUEUE);
}

// candidate j of cell c: stayers of the old segment first, then the
// arrivals in the cell's slots (j < n_st + min(arrivals, aslots))
__device__ __forceinline__ int candidate(const DevWork& w, const int* old_off, int c, int n_st, int j) {
    return j < n_st ? old_off[c] + j : w.arr_slot[(size_t)c * w.aslots + (j - n_st)];
}

// candidates beyond the slots: the cell's overflow list, entry t handled by
// lane t % stride
template <class F>
__device__ __forceinline__ void for_overflow(const DevWork& w, int c, int lane, int stride, F f) {
    int t = 0;
    for (int e = w.ovf_head[c]; e >= 0; ++t) {
        const int2 v = w.ovf[e];
        if (t % stride == lane) f(t, v.x);
        e = v.y;
    }
}


// ---------------------------------------------------------------------------
// Cell kernels.  A cell is handled by a group of GS = 16 lanes, so a
// wavefront works on four cells at once (the per-cell work is a short chain
// of dependent loads; several cells per wavefront hide that latency).
constexpr int GS = 16;
constexpr int GROUPS = 256 / GS;     // groups per 256-thread block
constexpr int GCAP = 64;             // candidates staged in LDS per group (small lattices, census_small_row)
constexpr int GCAP_L = 128;          // the same for larger lattices
// the census row of a lattice: GCAP for up to 16 parts, or when the
// survivors of a full cell (MAX per part) leave 8 of GCAP's entries for
// arrivals; else GCAP_L.  A cell whose candidates do not fit goes to
// k_cell_big either way; on the 5x5 lattice with MAX 2 of 407,140 quads the
// smaller rows (LDS for 7 workgroups per CU instead of 4, parts as bit masks)
// take 145 instead of 279 us a census, and their listed cells 15 instead of 5.
constexpr int SMALL_ROW_SURVIVORS = GCAP - 8;
__host__ __device__ inline bool census_small_row(int nparts, int max_per_part) {
    return nparts <= 16 || (long long)max_per_part * nparts <= SMALL_ROW_SURVIVORS;
}
constexpr int NKMAX = 272;           // part keys counted per group in the census (prod(q_d + 1))

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// sum / OR over a 16-lane group, all of whose lanes are active: a row of the
// data-parallel primitives, rotated by 8, 4, 2, 1 (no LDS permutes)
template <int N>
__device__ __forceinline__ int row_ror(int v) {
    return __builtin_amdgcn_update_dpp(0, v, 0x120 + N, 0xf, 0xf, true);
}

__device__ __forceinline__ int group_sum(int v) {
    static_assert(GS == 16, "a group is a row of 16 lanes");
    v += row_ror<8>(v);
    v += row_ror<4>(v);
    v += row_ror<2>(v);
    return v + row_ror<1>(v);
}

__device__ __forceinline__ int group_or32(int v) {
    v |= row_ror<8>(v);
    v |= row_ror<4>(v);
    v |= row_ror<2>(v);
    return v | row_ror<1>(v);
}

__device__ __forceinline__ unsigned long long group_or(unsigned long long v) {
    const unsigned lo = (unsigned)group_or32((int)(unsigned)v), hi = (unsigned)group_or32((int)(unsigned)(v >> 32));
    return ((unsigned long long)hi << 32) | lo;
}

// Staged rows of the census in LDS, compacted to the cell's valid candidates
// (stayers whose destination is c, then the arrivals): candidate index; part
// key << 32 | id; id of a survivor, all ones otherwise.  Rows are padded to a
// multiple of 4 entries with fill values (key all ones, id all ones), so the
// scans read 16 bytes at a time, and their strides put the four groups of a
// wavefront on different LDS banks.
template <int CAP>
struct CountRows {
    // particles per part key counted in rows of more than 32, one byte each
    // (four to a word, counted with word atomics; counts stay below CAP <= 128)
    // (rows of GCAP count up to 64 keys: 2-D lattices up to 7 x 7, 3-D up to
    // 3 x 3 x 3)
    static constexpr int NKC = CAP == GCAP ? 64 : NKMAX;
    // rows of GCAP on lattices of up to NKM keys: the row's entries of each
    // part key as a bit mask
    static constexpr int NKM = CAP == GCAP ? 36 : 0;
    __attribute__((aligned(16))) unsigned long long kid[GROUPS][CAP + 2];
    __attribute__((aligned(16))) uint32_t sid[GROUPS][CAP + 4];
    int idx[GROUPS][CAP + 4];
    unsigned int cnt[GROUPS][NKC / 4];
    unsigned long long mask[NKM ? GROUPS : 1][NKM + 1];
};

// k_cell_count: per-cell part census (check_cell_for_empty_parts,
// cylinder2D/pfem2particle.cpp:510-561).  Part index per direction is
// (unsigned)(xi_d / (1/q_d)) without clamping (xi = 1 gives the extra index
// q_d).  In every part the MAX particles with the smallest ids survive;
// every in-range part that holds no particle is reseeded.  With reseed = 0
// (relocation only) every particle that found a cell survives.
// A cell's candidates (stayers of its old segment, then arrivals) are staged
// in LDS when there are at most CAP of them (GCAP or GCAP_L), else listed
// for k_cell_big.
template <int DIM, int CAP, bool LIST = false>
__device__ __forceinline__ void cell_count_body(CountRows<CAP>& rows, const Grid& G, int n_cells, const int* __restrict__ old_off, const uint32_t* __restrict__ pid, const DevParams& pp, const DevWork& w, int reseed) {
    constexpr int NKC = CountRows<CAP>::NKC, NKM = CountRows<CAP>::NKM;
    auto &s_idx = rows.idx;
    auto &s_kid = rows.kid;
    auto &s_sid = rows.sid;
    auto &s_cnt = rows.cnt;
    auto &s_mask = rows.mask;
    // (LIST: cell_big_body has decided for the workgroup)
    if (!LIST && state_dead(w.counters)) return;
    const int g = threadIdx.x / GS, gl = threadIdx.x % GS;
    const unsigned long long all = pp.nparts_in >= 64 ? ~0ull : ((1ull << pp.nparts_in) - 1);
    int nk = 1;
#pragma unroll
    for (int d = 0; d < DIM; ++d) nk *= pp.q[d] + 1;
    const bool by_mask = nk <= NKM && reseed;
    const bool by_count = nk <= NKC && !by_mask;
    if constexpr (NKM > 0)
        for (int t = gl; t < NKM; t += GS) s_mask[g][t] = 0;
    for (int t = gl; t < NKC / 4; t += GS) s_cnt[g][t] = 0;
    int deleted = 0, arrivals = 0;
    const int set = w.counters[8];
    // LIST: the cells that the first pass listed (w.big), in rows of CAP
    // (those that do not fit either are left to cell_big_body)
    const int ncl = LIST ? w.big[0] : n_cells;
    for (int cb = G.bid * GROUPS; cb < ncl; cb += G.nblk * GROUPS) {
        const bool cv = cb + g < ncl;
        const int c = LIST ? (cv ? w.big[1 + cb + g] : 0) : cb + g;
        const int n_st = cv ? old_off[c + 1] - old_off[c] : 0;
        const int na = cv ? w.arr_cnt[c] : 0;
        const int k = n_st + na;
        const bool small = k <= CAP && na <= w.aslots;
        if (!LIST && cv && gl == 0) arrivals += na;
        unsigned long long hit = 0;
        // nv: valid candidates, nst of them stayers (the first nst staged
        // entries, in ascending id order like the cell's segment); the same
        // in all lanes of the group
        int nv = 0, nst = 0, nsurv = 0;
        // the group's lanes in its wavefront's ballot start at bit sh
        const int sh = (threadIdx.x & (WAVE - 1)) & ~(GS - 1);
        if (small) {
            // all loads of the row first (up to CAP / GS candidates per lane),
            // then the compaction: the candidates' dependent loads overlap
            constexpr int SU = CAP / GS;
            int idxs[SU];
            unsigned long long kids[SU];
#pragma unroll
            for (int u = 0; u < SU; ++u) {
                const int j = u * GS + gl;
                idxs[u] = -1;
                kids[u] = ~0ull;
                if (j < k) {
                    const int cidx = candidate(w, old_off, c, n_st, j);
                    const int dc = j < n_st ? w.dest[cidx] : c;
                    const unsigned long long kid = ((unsigned long long)(uint32_t)w.pkey[cidx] << 32) | pid[cidx];
                    // arrivals are listed for c because their destination is c
                    if (dc == c) {
                        idxs[u] = cidx;
                        kids[u] = kid;
                    }
                }
            }
#pragma unroll
            for (int u = 0; u < SU; ++u) {
                if (u * GS >= k) break;
                const int j = u * GS + gl;
                const int idx = idxs[u];
                const unsigned long long kid = kids[u];
                const unsigned mask = (unsigned)(__ballot(idx >= 0) >> sh) & 0xffffu;
                const unsigned smask = (unsigned)(__ballot(idx >= 0 && j < n_st) >> sh) & 0xffffu;
                if (idx >= 0) {
                    const int at = nv + __popc(mask & ((1u << gl) - 1u));
                    s_idx[g][at] = idx;
                    s_kid[g][at] = kid;
                    s_sid[g][at] = ~0u;
                }
                nv += __popc(mask);
                nst += __popc(smask);
            }
            if (gl < ((nv + 3) & ~3) - nv) {
                s_kid[g][nv + gl] = ~0ull;
                s_sid[g][nv + gl] = ~0u;
            }
        }
        const int nvr = (nv + 3) & ~3;
        wave_sync();
        // rank = particles of the same part with a smaller id, needed only
        // in a part that holds more than MAX particles: in rows of more than
        // 32 candidates the parts' counts first, then a scan of the row for
        // the particles of such parts (in shorter rows a scan for every
        // candidate costs less than the counting)
        if constexpr (NKM > 0)
            if (by_mask) {
                if (small)
                    for (int j = gl; j < nv; j += GS)
                        atomicOr(&s_mask[g][(uint32_t)(s_kid[g][j] >> 32) & 0xffffu], 1ull << j);
                wave_sync();
            }
        const bool counted = small && reseed && by_count && nv > 32;
        if (counted) {
            for (int j = gl; j < nv; j += GS) {
                const uint32_t key = (uint32_t)(s_kid[g][j] >> 32) & 0xffffu;
                atomicAdd(&s_cnt[g][key >> 2], 1u << (8 * (key & 3)));
            }
            wave_sync();
        }
        if (small)
            for (int j = gl; j < nv; j += GS) {
                const unsigned long long me = s_kid[g][j];
                const uint32_t mk = (uint32_t)(me >> 32), mi = (uint32_t)me;
                const int o = part_ordinal((int)mk);
                if (o >= 0) hit |= 1ull << o;
                // rank (fill entries carry no valid key)
                int rank = 0;
                const uint32_t key = mk & 0xffffu;
                const unsigned cnt = counted ? (s_cnt[g][key >> 2] >> (8 * (key & 3))) & 0xffu : 0xffu;
                if (by_mask) {
                    if constexpr (NKM > 0) {
                        unsigned long long mm = s_mask[g][key];
                        if (__popcll(mm) > pp.max_per_part)
                            for (; mm; mm &= mm - 1) rank += (uint32_t)s_kid[g][__ffsll((long long)mm) - 1] < mi ? 1 : 0;
                    }
                } else if (reseed && cnt > (unsigned)pp.max_per_part) {
                    for (int t = 0; t < nvr; t += 2) {
                        const ulonglong2 v = *reinterpret_cast<const ulonglong2*>(&s_kid[g][t]);
                        rank += ((uint32_t)(v.x >> 32) == mk && (uint32_t)v.x < mi) ? 1 : 0;
                        rank += ((uint32_t)(v.y >> 32) == mk && (uint32_t)v.y < mi) ? 1 : 0;
                    }
                }
                const bool surv = rank < pp.max_per_part || !reseed;
                nsurv += surv ? 1 : 0;
                if (surv) s_sid[g][j] = mi;
            }
        else if (!LIST && cv && gl == 0) {
            // more than CAP candidates: census by k_cell_big
            const int slot = atomicAdd(&w.big[0], 1);
            w.big[1 + slot] = c;
        }
        wave_sync();
        if constexpr (NKM > 0)
            if (by_mask && small)   // back to zero for the next cell
                for (int j = gl; j < nv; j += GS) s_mask[g][(uint32_t)(s_kid[g][j] >> 32) & 0xffffu] = 0;
        if (counted)   // back to zero for the next cell (the words hold only this cell's parts)
            for (int j = gl; j < nv; j += GS) s_cnt[g][((uint32_t)(s_kid[g][j] >> 32) & 0xffffu) >> 2] = 0u;
        nsurv = group_sum(nsurv);
        // positions of the survivors in ascending id order (ids are below
        // 2^32 - 1, the fill value): the survivors in that order replace the
        // cell's arrival slots (already staged) when they fit, else each
        // candidate gets its position (-1: dropped)
        const bool listed = nsurv <= w.aslots;
        // positions: with few arrivals, a stayer's is the surviving stayers
        // before it plus the surviving arrivals with a smaller id; otherwise
        // (and for the arrivals) a scan of all entries.  A pending layout
        // needs no positions, only its survivors marked.
        const bool pos_needed = small && !w.pend_mark;
        if (small && w.pend_mark)
            for (int j = gl; j < nv; j += GS)
                if (s_sid[g][j] != ~0u) w.dest[s_idx[g][j]] = c | DEST_KEPT;
        const int jp = pos_needed && nv - nst <= 4 ? nst : 0;
        if (pos_needed && jp > 0) {
            int sbase = 0;
            for (int j0 = 0; j0 < jp; j0 += GS) {
                const int j = j0 + gl;
                const bool act = j < jp;
                const uint32_t id = act ? s_sid[g][j] : ~0u;
                const bool sv = act && id != ~0u;
                const unsigned mask = (unsigned)(__ballot(sv) >> sh) & 0xffffu;
                if (sv) {
                    int pos = sbase + __popc(mask & ((1u << gl) - 1u));
                    for (int t = nst; t < nv; ++t) pos += s_sid[g][t] < id ? 1 : 0;
                    const int idx = s_idx[g][j];
                    if (listed) w.arr_slot[(size_t)c * w.aslots + pos] = idx;
                    else w.spos[idx] = pos;
                } else if (act && !listed) {
                    w.spos[s_idx[g][j]] = -1;
                }
                sbase += __popc(mask);
            }
        }
        if (pos_needed)
            for (int j = jp + gl; j < nv; j += GS) {
                const int idx = s_idx[g][j];
                const uint32_t id = s_sid[g][j];
                if (id == ~0u) {
                    if (!listed) w.spos[idx] = -1;
                    continue;
                }
                int pos = 0;
                for (int t = 0; t < nvr; t += 4) {
                    const uint4 v = *reinterpret_cast<const uint4*>(&s_sid[g][t]);
                    pos += (v.x < id ? 1 : 0) + (v.y < id ? 1 : 0) + (v.z < id ? 1 : 0) + (v.w < id ? 1 : 0);
                }
                if (listed) w.arr_slot[(size_t)c * w.aslots + pos] = idx;
                else w.spos[idx] = pos;
            }
        wave_sync();
        hit = group_or(hit);
        unsigned long long fs = 0;
        if (cv && small && gl == 0) {
            const int spawns = reseed ? __popcll(all & ~hit) : 0;
            fs = ((unsigned long long)(nsurv + spawns) << 32) | (unsigned)spawns;
            w.hitmask[c] = reseed ? hit : all;
            w.nsurv[c] = nsurv;
            w.fs_cnt[c] = fs;
            deleted += nv - nsurv;
            if (LIST) add_cell_sum(w, set, c, fs);
        }
        if (!LIST && w.sums.fine) {   // the wavefront's 4 cells
            fs += __shfl_xor(fs, GS);
            fs += __shfl_xor(fs, 2 * GS);
            if ((threadIdx.x & (WAVE - 1)) == 0) w.sums.fine[c / 4] = fs;
        }
    }
    deleted = wave_sum(deleted);
    if ((threadIdx.x & (WAVE - 1)) == 0 && deleted) stat_add(w.stats, 1, (unsigned long long)deleted);
    if (!LIST) wave_stat(w.stats, 5, arrivals);
}

template <int DIM, int CAP>
__global__ void __launch_bounds__(256) k_cell_count(int n_cells, const int* __restrict__ old_off,
                                                    const uint32_t* __restrict__ pid, DevParams pp, DevWork w,
                                                    int reseed) {
    __shared__ CountRows<CAP> rows;
    cell_count_body<DIM, CAP>(rows, hw_grid(), n_cells, old_off, pid, pp, w, reseed);
}

// k_cell_big: the census of k_cell_count for the cells it listed, candidates
// staged in LDS: a 256-thread block for each while there are blocks enough,
// and for more cells a 16-lane group for each of those with up to GCAP_L
// candidates first.  Bound by the latency of a cell's chain of dependent reads
// and barriers, so what counts is how many cells run at once: the few thousand
// listed of 101,785 cells with a 4x4 lattice took 32 us with a block each and
// take 21 with groups, the few hundred of 25,446 cells 12 with blocks and 17 with
// groups.  One launch for both: the group pass of its own on lattices of more
// than 16 parts cost 4 us.
// A cell with more than BIGCAP candidates sets overflow flag 2 and keeps no
// particle.
constexpr int BIGCAP = 2048;

template <int DIM>
__device__ __forceinline__ void cell_big_body(const Grid& G, const int* __restrict__ old_off, const uint32_t* __restrict__ pid, const DevParams& pp, const DevWork& w, int reseed) {
    struct BigRow {
        __attribute__((aligned(16))) unsigned long long kid[BIGCAP];
        __attribute__((aligned(16))) uint32_t sid[BIGCAP];
        int idx[BIGCAP];
    };
    // (one after the other: 38 KB, four workgroups a CU)
    __shared__ union {
        CountRows<GCAP_L> rows;
        BigRow row;
    } lds;
    auto &s_idx = lds.row.idx;
    auto &s_kid = lds.row.kid;
    auto &s_sid = lds.row.sid;
    __shared__ unsigned long long s_hit;
    __shared__ int s_nvalid, s_nsurv;
    const int nbig = w.big[0], set = w.counters[8];   // (read along with the flag)
    if (workgroup_dead(w.counters)) return;           // (raised below by other workgroups)
    const int tid = threadIdx.x;
    const unsigned long long all = pp.nparts_in >= 64 ? ~0ull : ((1ull << pp.nparts_in) - 1);
    add_fine_sums(w, set, (int)G.bid, (int)G.nblk);
    if (nbig == 0) return;
    const bool by_group = nbig > (int)G.nblk;
    if (by_group) {
        cell_count_body<DIM, GCAP_L, true>(lds.rows, G, 0, old_off, pid, pp, w, reseed);
        __syncthreads();
    }
    int deleted = 0;
    for (int b = G.bid; b < nbig; b += G.nblk) {
        const int c = w.big[1 + b];
        const int n_st = old_off[c + 1] - old_off[c];
        const int na = w.arr_cnt[c];
        const int k = n_st + na;
        if (by_group && k <= GCAP_L && na <= w.aslots) continue;   // done
        const int kin = n_st + (na < w.aslots ? na : w.aslots);   // candidates in the old segment and slots
        if (k > BIGCAP) {
            for (int j = tid; j < kin; j += blockDim.x) w.spos[candidate(w, old_off, c, n_st, j)] = -1;
            for_overflow(w, c, tid, blockDim.x, [&](int, int idx) { w.spos[idx] = -1; });
            if (tid == 0) {
                atomicOr(&w.counters[2], 2);
                w.hitmask[c] = all;
                w.nsurv[c] = 0;
                w.fs_cnt[c] = 0;
            }
            continue;
        }
        const int kr = (k + 3) & ~3;
        if (tid == 0) {
            s_hit = 0;
            s_nvalid = 0;
            s_nsurv = 0;
        }
        for (int j = tid; j < kr; j += blockDim.x) {
            if (j >= kin && j < k) continue;   // overflow entries, staged below
            int idx = -1;
            unsigned long long kid = ~0ull;
            if (j < k) {
                const int cidx = candidate(w, old_off, c, n_st, j);
                if (j >= n_st || w.dest[cidx] == c) {
                    idx = cidx;
                    kid = ((unsigned long long)(uint32_t)w.pkey[cidx] << 32) | pid[cidx];
                }
            }
            s_idx[j] = idx;
            s_kid[j] = kid;
            s_sid[j] = ~0u;
        }
        for_overflow(w, c, tid, blockDim.x, [&](int t, int cidx) {
            s_idx[kin + t] = cidx;
            s_kid[kin + t] = ((unsigned long long)(uint32_t)w.pkey[cidx] << 32) | pid[cidx];
            s_sid[kin + t] = ~0u;
        });
        __syncthreads();
        unsigned long long hit = 0;
        int nvalid = 0, nsurv = 0;
        for (int j = tid; j < k; j += blockDim.x) {
            if (s_idx[j] < 0) continue;
            ++nvalid;
            const unsigned long long me = s_kid[j];
            const int o = part_ordinal((int)(me >> 32));
            if (o >= 0) hit |= 1ull << o;
            int rank = 0;
            if (reseed) {
                const unsigned long long lo = me & 0xffffffff00000000ull;
                for (int t = 0; t < kr; t += 2) {
                    const ulonglong2 v = *reinterpret_cast<const ulonglong2*>(&s_kid[t]);
                    rank += (v.x >= lo && v.x < me) ? 1 : 0;
                    rank += (v.y >= lo && v.y < me) ? 1 : 0;
                }
            }
            const bool surv = rank < pp.max_per_part || !reseed;
            nsurv += surv ? 1 : 0;
            if (surv) s_sid[j] = (uint32_t)me;
        }
        if (hit) atomicOr(&s_hit, hit);
        if (nvalid) atomicAdd(&s_nvalid, nvalid);
        if (nsurv) atomicAdd(&s_nsurv, nsurv);
        __syncthreads();
        // survivors listed in the cell's (staged) arrival slots when they fit
        // (a pending layout: only marked)
        const bool listed = s_nsurv <= w.aslots;
        for (int j = tid; j < k; j += blockDim.x) {
            const int idx = s_idx[j];
            if (idx < 0) continue;
            const uint32_t id = s_sid[j];
            if (w.pend_mark) {
                if (id != ~0u) w.dest[idx] = c | DEST_KEPT;
                continue;
            }
            if (id == ~0u) {
                if (!listed) w.spos[idx] = -1;
                continue;
            }
            int pos = 0;
            for (int t = 0; t < kr; t += 4) {
                const uint4 v = *reinterpret_cast<const uint4*>(&s_sid[t]);
                pos += (v.x < id ? 1 : 0) + (v.y < id ? 1 : 0) + (v.z < id ? 1 : 0) + (v.w < id ? 1 : 0);
            }
            if (listed) w.arr_slot[(size_t)c * w.aslots + pos] = idx;
            else w.spos[idx] = pos;
        }
        if (tid == 0) {
            const unsigned long long hm = s_hit;
            const int spawns = reseed ? __popcll(all & ~hm) : 0;
            w.hitmask[c] = reseed ? hm : all;
            w.nsurv[c] = s_nsurv;
            const unsigned long long fs = ((unsigned long long)(s_nsurv + spawns) << 32) | (unsigned)spawns;
            w.fs_cnt[c] = fs;
            add_cell_sum(w, set, c, fs);
            deleted += s_nvalid - s_nsurv;
        }
        __syncthreads();
    }
    if (tid == 0 && deleted) stat_add(w.stats, 1, (unsigned long long)deleted);
}

template <int DIM>
__global__ void __launch_bounds__(256) k_cell_big(const int* __restrict__ old_off, const uint32_t* __restrict__ pid,
                                                  DevParams pp, DevWork w, int reseed) {
    cell_big_body<DIM>(hw_grid(), old_off, pid, pp, w, reseed);
}

// ---------------------------------------------------------------------------
// k_cell_write: the regroup write, survivors and reseeded particles into
// buffer B at their final positions, with the projection sums of the cells
// when SUMS is set (pf2_step).
//
// A cell's output segment starts at an arbitrary position, so stores per cell
// (a few lanes, 8 bytes each) do not cover whole cache lines and L2 fills
// every line it writes from memory first.  A workgroup therefore takes
// RegroupShape::CB consecutive cells, whose segments are one contiguous range,
// and walks that range in order: each position finds its cell by bisection of
// the offsets in LDS and its source in the cell's slot row (the census's
// survivors in id order), or creates the new particle.  The records pass
// through LDS on the way, where LPC lanes per cell add the projection sums in
// ascending id order (accumulators in registers across the passes, so any
// number of particles per cell), and no other pass reads them again.
// Bound by HBM: it moves bytes at a large copy's rate.  A 2-D FP64 particle is
// 64 bytes in and out (80 with velocity_ext); the counters show about half as
// much again read, for lines of scattered arrivals and slot rows that are used
// in part.  It takes the place of a map of the positions, a gather by it, a
// pass of sums and its own bookkeeping launch: 125 -> 92 us (FP64) and 83 -> 50
// (FP32-mixed) on 101,785 quads, 625 -> 521 and 396 -> 307 on 407,140.  One
// position per thread and pass: two or four, for more loads in flight, cost
// registers (14-44% slower).
//
// New particles: reference point at the part centre, location mapped,
// velocity interpolated from V (cylinder2D/pfem2particle.cpp:533-549), ids
// continuing the counter in ascending cell, then part, order.
template <int DIM, int DEG>
struct RegroupShape {
    static constexpr int NACC = QF<DIM, DEG>::ND * (DIM + 1);   // sums per cell
    // cells per workgroup: 16 (8 and 32 were 5-10% slower in 2-D), 32 of the
    // few particles of a hexahedron (16: 87 instead of 79 us in FP32-mixed, 161
    // instead of 146 in FP64 on 202,240)
    static constexpr int CB = DIM == 3 && DEG == 1 ? 32 : 16;
    static constexpr int LPC = 256 / CB;                        // lanes per cell in the sums
    static constexpr int NA = (NACC + LPC - 1) / LPC;           // sums per lane
};

// a workgroup's cells in LDS
template <int CB>
struct RegroupCells {
    long long base;                  // first output position
    int off[CB + 1];                 // each cell's first position after it, then the end
    int nsurv[CB];
    unsigned long long empty[CB];    // parts to reseed
    uint32_t spawn0[CB];             // new particles of earlier cells
    int dead;                        // the state was dead: nothing to write
};

// Fills s for the cells cb, cb + 1, ... (all threads call; barriers inside,
// none after the resets at the end): offsets, overflow flag, and for cells
// whose survivors outnumber the slot row (rare) their sources in omap.
// False: the state is dead.  Other workgroups of the same launch raise that
// flag, so the first wavefront reads it once and decides for the workgroup:
// were each wavefront to read it, the first could leave while the others,
// their barrier no longer waiting for it, took the cells from LDS that it
// never wrote.  (The cells' counts are read either way: they are in range in
// a dead state too.)
template <int CB>
__device__ __forceinline__ bool regroup_cells(RegroupCells<CB>& s, int cb, int nc, const int* __restrict__ old_off,
                                              long long cap, const DevParams& pp, const DevWork& w,
                                              int* __restrict__ omap) {
    constexpr int LPC = 256 / CB;
    static_assert(CB <= WAVE && (CB & (CB - 1)) == 0, "one wavefront loads the cells, bisection over them");
    const int t = threadIdx.x;
    const int last = nc - cb < CB ? nc - cb : CB;
    bool past = false;
    if (t < WAVE) {
        const int flags = w.counters[2], set = w.counters[8];
        const int c = cb + (t < last ? t : last - 1);
        const unsigned long long n = w.fs_cnt[c], v = t < last ? n : 0ull;
        const int nsurv = w.nsurv[c];
        const unsigned long long hit = w.hitmask[c];
        const unsigned long long base = cell_offset(w, set, cb);
        unsigned long long incl = v;   // particles and new ones up to cell t of the workgroup
        if (w.sums.fine) {
#pragma unroll
            for (int h = 1; h < CB; h <<= 1) {
                const unsigned long long o = __shfl_up(incl, h);
                if (t >= h) incl += o;
            }
        } else {
            incl = w.fs_off[c] - base + n;
        }
        const unsigned long long all = pp.nparts_in >= 64 ? ~0ull : ((1ull << pp.nparts_in) - 1);
        const bool dead = (__builtin_amdgcn_readfirstlane(flags) & DEAD_FLAGS) != 0;
        if (t == 0) {
            s.base = (long long)(base >> 32);
            s.dead = dead;
        }
        if (t < CB) {
            s.off[t] = (int)((incl - v) >> 32);
            if (t == CB - 1) s.off[CB] = (int)(incl >> 32);
            s.nsurv[t] = nsurv;
            s.empty[t] = all & ~hit;
            s.spawn0[t] = (uint32_t)(base + incl - v);
        }
        if (t < last && !dead) {
            const long long out0 = (long long)((base + incl - v) >> 32);
            w.new_off[c] = (int)out0;
            past = nsurv > w.aslots;
            if (out0 + (long long)(v >> 32) > cap) atomicOr(&w.counters[2], 1);
            clear_next_sums(w, set, c);
        }
    }
    const bool any_past = __syncthreads_or(past);
    if (s.dead) return false;
    if (any_past) {
        const int g = t / LPC, gl = t % LPC, c = cb + g;
        if (g < last && s.nsurv[g] > w.aslots) {
            const int n_st = old_off[c + 1] - old_off[c], na = w.arr_cnt[c];
            const long long out0 = s.base + s.off[g];
            auto put = [&](int idx) {
                const int pos = w.spos[idx];
                if (pos >= 0 && out0 + pos < cap) omap[out0 + pos] = idx;
            };
            const int kin = n_st + (na < w.aslots ? na : w.aslots);
            for (int j = gl; j < kin; j += LPC) {
                const int idx = candidate(w, old_off, c, n_st, j);
                // arrivals are in this cell's slots because their destination is c
                if (j >= n_st || w.dest[idx] == c) put(idx);
            }
            for_overflow(w, c, gl, LPC, [&](int, int idx) { put(idx); });
        }
        __syncthreads();
    }
    // (the arrival lists of the cells have been read)
    if (t < last) {
        w.arr_cnt[cb + t] = 0;
        w.ovf_head[cb + t] = -1;
    }
    return true;
}

// source of the output position p after s.base: a particle, or for a new one
// -1 - its lattice ordinal; k is its cell within the workgroup's
template <int CB>
__device__ __forceinline__ int regroup_source(const RegroupCells<CB>& s, int cb, int p, const DevWork& w,
                                              const int* __restrict__ omap, int& k) {
    k = 0;
#pragma unroll
    for (int h = CB / 2; h > 0; h >>= 1)
        if (s.off[k + h] <= p) k += h;
    const int t = p - s.off[k], ns = s.nsurv[k];
    if (t < ns) return ns <= w.aslots ? w.arr_slot[(size_t)(cb + k) * w.aslots + t] : omap[s.base + p];
    unsigned long long e = s.empty[k];
    for (int r = t - ns; r > 0; --r) e &= e - 1;
    return -__ffsll((long long)e);
}

// GATHER: velocities of new particles through the DoF map (FP32-mixed handles,
// or stale per-cell copies)
template <int DIM, bool GATHER, bool SUMS, int DEG>
__device__ __forceinline__ void cell_write_body(const Grid& G, const DevMesh<DIM>& m, const int* __restrict__ old_off,
                                                const DevParticles& A, const DevParticles& B, const DevParams& pp,
                                                const DevWork& w, int* __restrict__ omap,
                                                double* __restrict__ partial) {
    using S = RegroupShape<DIM, DEG>;
    constexpr int NV = Q1<DIM>::NV;
    constexpr int ND = QF<DIM, DEG>::ND;
    constexpr int CH = 256;   // positions per pass
    __shared__ RegroupCells<S::CB> s;
    // degree-2 hexahedra: each particle's 1-D factors in LDS, from which a lane
    // multiplies its 7 nodes' shape values; the nodes' coefficients instead took
    // 168 registers a lane, 2 wavefronts per SIMD (with interp_each 151 -> 104 us
    // on 68,992)
    constexpr bool TAB = SUMS && DIM == 3 && DEG == 2;
    static_assert(!TAB || S::LPC % (DIM + 1) == 0, "a lane's sums are of one component");
    __shared__ double s_xi[SUMS && !TAB ? DIM : 1][SUMS && !TAB ? CH : 1];
    __shared__ double s_l[TAB ? CH : 1][3 * DIM];
    __shared__ double s_v[SUMS ? DIM : 1][SUMS ? CH : 1];
    const int tid = threadIdx.x, g = tid / S::LPC, gl = tid % S::LPC;
    // the lane's sums: vertex a / (DIM + 1), component a % (DIM + 1) (the last
    // one the weight) for a = gl, gl + LPC, ...
    ShapeOne<DIM, DEG> sh[TAB ? 1 : S::NA];
    int comp[S::NA], fac[TAB ? S::NA : 1][DIM];
    if constexpr (TAB)
#pragma unroll
        for (int u = 0; u < S::NA; ++u) {
            const int a = gl + u * S::LPC;
#pragma unroll
            for (int d = 0; d < DIM; ++d) fac[u][d] = 3 * d + q2_axis(DIM, (a < S::NACC ? a : 0) / (DIM + 1), d);
        }
    else if constexpr (SUMS)
#pragma unroll
        for (int u = 0; u < S::NA; ++u) {
            const int a = gl + u * S::LPC;
            const int kk = (a < S::NACC ? a : 0) / (DIM + 1);
            comp[u] = a - kk * (DIM + 1);
            sh[u].init(kk);
        }
    for (int cb = G.bid * S::CB; cb < m.n_cells; cb += G.nblk * S::CB) {
        if (!regroup_cells<S::CB>(s, cb, m.n_cells, old_off, A.cap, pp, w, omap)) return;
        const long long base = s.base;
        const int total = base + s.off[S::CB] <= B.cap ? s.off[S::CB] : (int)(B.cap > base ? B.cap - base : 0);
        double acc[S::NA];
#pragma unroll
        for (int u = 0; u < S::NA; ++u) acc[u] = 0.0;
        for (int p0 = 0; p0 < total; p0 += CH) {
            const int p = p0 + tid;
            if (p < total) {
                int k;
                const int src = regroup_source<S::CB>(s, cb, p, w, omap, k);
                const int c = cb + k;
                uint32_t id = 0;
                double x[DIM], xi[DIM], v[DIM], e[DIM];
                if (src >= 0) {
                    id = A.id[src];
#pragma unroll
                    for (int d = 0; d < DIM; ++d) {
                        x[d] = A.x[(size_t)d * A.cap + src];
                        xi[d] = A.xi[(size_t)d * A.cap + src];
                        v[d] = A.v[(size_t)d * A.cap + src];
                        e[d] = pp.keep_vext ? A.vext[(size_t)d * A.cap + src] : 0.0;
                    }
                }
                // a new particle: most wavefronts hold one or two, so its
                // loads go out behind the records' and before any wait
                if (src < 0) {
                    double P[NV][DIM];
                    id = *w.particle_counter + s.spawn0[k] + (uint32_t)(p - s.off[k] - s.nsurv[k]) + 1u;
                    lattice_point<DIM>(pp, -1 - src, xi);
                    if constexpr (DEG == 1) {
                        double Vc[ND][DIM];
                        load_cell<DIM, GATHER, DEG>(m, c, P, Vc);
                        forward<DIM>(P, xi, x);
                        interp<DIM, DEG>(Vc, xi, v);
                    } else {
                        load_vertices<DIM>(m, c, P);
                        forward<DIM>(P, xi, x);
                        interp_each<DIM, DEG>(xi, v, [&](int n) {
                            return GATHER ? m.Vn + (size_t)m.cd[(size_t)c * ND + n] * DIM
                                          : m.cellV + ((size_t)c * ND + n) * DIM;
                        });
                    }
#pragma unroll
                    for (int d = 0; d < DIM; ++d) e[d] = 0.0;
                }
                const long long o = base + p;
                B.cell[o] = c;
                B.id[o] = id;
#pragma unroll
                for (int d = 0; d < DIM; ++d) {
                    B.x[(size_t)d * B.cap + o] = x[d];
                    B.xi[(size_t)d * B.cap + o] = xi[d];
                    B.v[(size_t)d * B.cap + o] = v[d];
                    if (pp.keep_vext) B.vext[(size_t)d * B.cap + o] = e[d];
                    if constexpr (TAB)
#pragma unroll
                        for (int q = 0; q < 3; ++q) s_l[tid][3 * d + q] = lag2(q, xi[d]);
                    else if constexpr (SUMS) s_xi[d][tid] = xi[d];
                    if constexpr (SUMS) s_v[d][tid] = v[d];
                }
            }
            if constexpr (SUMS) {
                __syncthreads();
                const int q0 = s.off[g] > p0 ? s.off[g] - p0 : 0;
                const int e = s.off[g + 1] < total ? s.off[g + 1] : total;
                const int q1 = e - p0 < CH ? e - p0 : CH;
                if constexpr (TAB) {
                    const int cp = gl % (DIM + 1);
                    for (int q = q0; q < q1; ++q) {
                        const double vc = cp < DIM ? s_v[cp < DIM ? cp : 0][q] : 1.0;
#pragma unroll
                        for (int u = 0; u < S::NA; ++u)
                            acc[u] += s_l[q][fac[u][0]] * s_l[q][fac[u][1]] * s_l[q][fac[u][2]] * vc;
                    }
                } else
                for (int q = q0; q < q1; ++q) {
                    double xi[DIM], v[DIM];
#pragma unroll
                    for (int d = 0; d < DIM; ++d) {
                        xi[d] = s_xi[d][q];
                        v[d] = s_v[d][q];
                    }
#pragma unroll
                    for (int u = 0; u < S::NA; ++u) {
                        double vc = 1.0;   // the weight term is N_k itself
#pragma unroll
                        for (int d = 0; d < DIM; ++d)
                            if (d == comp[u]) vc = v[d];
                        acc[u] += sh[u](xi) * vc;
                    }
                }
                __syncthreads();
            }
        }
        if constexpr (SUMS)
            if (cb + g < m.n_cells)
#pragma unroll
                for (int u = 0; u < S::NA; ++u)
                    if (gl + u * S::LPC < S::NACC) partial[partial_at<DIM, DEG>(m.n_cells, cb + g, gl + u * S::LPC)] = acc[u];
        __syncthreads();   // s is refilled
    }
}

template <int DIM, bool GATHER, bool SUMS, int DEG>
__global__ void __launch_bounds__(256) k_cell_write(DevMesh<DIM> m, const int* __restrict__ old_off, DevParticles A,
                                                    DevParticles B, DevParams pp, DevWork w, int* __restrict__ omap,
                                                    double* __restrict__ partial) {
    cell_write_body<DIM, GATHER, SUMS, DEG>(hw_grid(), m, old_off, A, B, pp, w, omap, partial);
}

// totals after the census: particle count, id counter, statistics; resets the
// queue counters for the next step (one workgroup of QSHARDS threads: k_finalize,
// or the last workgroup of k_node in a fused step)
__device__ __forceinline__ void finalize_block(int n_cells, const DevWork& w, int* queue_count,
                                               bool keep_pending = false) {
    static_assert(QSHARDS == STAT_SHARDS, "one thread per stat row");
    __shared__ int s_arr;
    const int t = threadIdx.x;
    for (int r = 0; r < NQROUNDS; ++r) {
        queue_count[((size_t)r * (QSHARDS + 1) + t) * QSTRIDE] = 0;
        if (t == 0) queue_count[((size_t)r * (QSHARDS + 1) + QSHARDS) * QSTRIDE] = 0;
    }
    // arrivals of this regroup (diagnostics): the stat rows' slot 5, cleared
    if (t == 0) s_arr = 0;
    __syncthreads();
    const int a = (int)w.stats[(size_t)t * NSTAT + 5];
    w.stats[(size_t)t * NSTAT + 5] = 0;
    if (a) atomicAdd(&s_arr, a);
    const int set = w.counters[8];
    const unsigned long long fo = cell_total(w, set, n_cells);
    __syncthreads();
    if (t != 0) return;
    w.counters[1] = s_arr;
    w.counters[8] = (set & 1) ^ 1;
    // a dead state publishes no particles (its total may exceed the capacity)
    const bool dead = state_dead(w.counters);
    const int total = dead ? 0 : (int)(fo >> 32);
    const int spawned = dead ? 0 : (int)(uint32_t)fo;
    w.new_off[n_cells] = total;
    w.stats[2] += (unsigned long long)spawned;
    *w.particle_counter += (uint32_t)spawned;
    w.counters[3] = w.counters[0];   // count before the step (diagnostics)
    w.counters[0] = total;
    w.counters[4] = 0;
    // a regroup consumes a pending layout; k_cell_pend has just set one up
    if (!keep_pending) w.counters[6] = 0;
    w.big[0] = 0;
}

__global__ void __launch_bounds__(QSHARDS) k_finalize(int n_cells, DevWork w, int* queue_count, int keep_pending) {
    finalize_block(n_cells, w, queue_count, keep_pending != 0);
}

// ---------------------------------------------------------------------------
// Pending layout.  After the census of a re-sort (relocation + reseed), the
// particles are not moved into a new buffer: the census's survivors are
// marked in place (destination = cell | DEST_KEPT), its
// new particles are created after the current segments (position seg_end +
// the cell's spawn offset + rank, ids and values as k_cell_write creates
// them), and counters[6], [7] record the slots and seg_end.  The next move
// takes a particle's cell from dest, skips the unmarked ones and makes the
// new ones arrive in their cell, so its census regroups the pending layout
// and the re-sort's regroup write is never done.  Any other use of the
// particles first settles the layout (k_settle + a regroup without reseed).
// (The census marks the survivors when DevWork::pend_mark is set.)

// slots and segment end of a pending layout (the first wavefront of the grid)
__device__ __forceinline__ void pend_slots(const DevWork& w, int nc, int seg_end, long long cap) {
    if (blockIdx.x != 0 || threadIdx.x >= WAVE) return;
    const unsigned long long tot = cell_total(w, w.counters[8], nc);
    if (threadIdx.x != 0) return;
    const long long slots = (long long)seg_end + (uint32_t)tot;
    if (slots > cap) atomicOr(&w.counters[2], 1);
    w.counters[6] = slots > cap ? 0 : (int)slots;
    w.counters[7] = seg_end;
}

// offsets (particles << 32 | new particles) of the cell c0 + threadIdx.x of a
// workgroup of 256 threads (all call; c0 a multiple of 256); clears its next sums
__device__ __forceinline__ unsigned long long pend_offset(const DevWork& w, int c0, int nc) {
    __shared__ unsigned long long s_base, s_w[256 / WAVE];
    const int t = threadIdx.x, lane = t & (WAVE - 1), wv = t / WAVE, c = c0 + t;
    if (!w.sums.fine) return c < nc ? w.fs_off[c] : 0ull;
    const int set = w.counters[8];
    const unsigned long long v = c < nc ? w.fs_cnt[c] : 0ull;
    if (c < nc) clear_next_sums(w, set, c);
    if (wv == 0) {
        const unsigned long long b = cell_offset(w, set, c0);
        if (lane == 0) s_base = b;
    }
    unsigned long long incl = v;
#pragma unroll
    for (int h = 1; h < WAVE; h <<= 1) {
        const unsigned long long o = __shfl_up(incl, h);
        if (lane >= h) incl += o;
    }
    if (lane == WAVE - 1) s_w[wv] = incl;
    __syncthreads();
    unsigned long long fo = s_base + incl - v;
    for (int q = 0; q < wv; ++q) fo += s_w[q];
    __syncthreads();
    return fo;
}

template <int DIM, bool GATHER, int DEG = 1>
__global__ void __launch_bounds__(256) k_cell_pend(DevMesh<DIM> m, const int* __restrict__ old_off, DevParticles A,
                                                   DevParams pp, DevWork w) {
    constexpr int NV = Q1<DIM>::NV;
    constexpr int ND = QF<DIM, DEG>::ND;
    const int nc = m.n_cells;
    const int seg_end = old_off[nc];
    if (workgroup_dead(w.counters)) return;   // (pend_slots raises the flag)
    pend_slots(w, nc, seg_end, A.cap);
    // one cell per thread: new particles are few, and most cells only get
    // their resets
    for (int c0 = blockIdx.x * 256; c0 < nc; c0 += gridDim.x * 256) {
        const int c = c0 + threadIdx.x;
        const unsigned long long fo = pend_offset(w, c0, nc);
        if (c >= nc) continue;
        if ((uint32_t)w.fs_cnt[c] != 0u) {   // spawns, in lattice order
            const unsigned long long all = pp.nparts_in >= 64 ? ~0ull : ((1ull << pp.nparts_in) - 1);
            const unsigned long long empty = all & ~w.hitmask[c];
            double P[NV][DIM], Vc[ND][DIM];
            load_cell<DIM, GATHER, DEG>(m, c, P, Vc);
            int r = 0;
            for (unsigned long long e = empty; e; e &= e - 1, ++r) {
                const int o = __ffsll((long long)e) - 1;
                const long long q = (long long)seg_end + (uint32_t)fo + r;
                if (q >= A.cap) continue;   // (flagged above)
                double xi[DIM], x[DIM], v[DIM];
                lattice_point<DIM>(pp, o, xi);
                forward<DIM>(P, xi, x);
                interp<DIM, DEG>(Vc, xi, v);
                A.cell[q] = c;
                A.id[q] = *w.particle_counter + (uint32_t)fo + (uint32_t)r + 1u;
                w.dest[q] = c | DEST_KEPT;
#pragma unroll
                for (int d = 0; d < DIM; ++d) {
                    A.x[(size_t)d * A.cap + q] = x[d];
                    A.xi[(size_t)d * A.cap + q] = xi[d];
                    A.v[(size_t)d * A.cap + q] = v[d];
                    if (pp.keep_vext) A.vext[(size_t)d * A.cap + q] = 0.0;
                }
            }
        }
        w.arr_cnt[c] = 0;
        w.ovf_head[c] = -1;
    }
}

// settles a pending layout for a regroup without reseed: every kept or new
// particle keeps its cell (destination) and gets its part key back, and the
// ones outside their cell's segment arrive there; the others are gone
template <int DIM>
__global__ void k_settle(DevParticles A, DevParams pp, DevWork w) {
    const int pn = w.counters[6];
    const int seg_end = w.counters[7];
    const int lane = threadIdx.x & (WAVE - 1);
    for (int base = blockIdx.x * blockDim.x + (threadIdx.x - lane); base < pn; base += gridDim.x * blockDim.x) {
        const int i = base + lane;
        const bool valid = i < pn;
        int c = -1;
        if (valid) {
            const int dk = w.dest[i];
            c = dk >= 0 && (dk & DEST_KEPT) ? dk & ~DEST_KEPT : -1;
            w.dest[i] = c;
            if (c >= 0) {
                double xi[DIM];
#pragma unroll
                for (int d = 0; d < DIM; ++d) xi[d] = A.xi[(size_t)d * A.cap + i];
                w.pkey[i] = part_key<DIM>(pp, xi);
            }
        }
        add_arrival(w, valid && c >= 0 && (c != A.cell[valid ? i : 0] || i >= seg_end), c, i);
    }
}

// ---------------------------------------------------------------------------
// k_cell_partials: per-cell local sums of the projection
// (TurekBenchmark/pfem2particle.cpp:880-893): for each cell vertex k,
// sum_p N_k(xi_p) v_p and sum_p N_k(xi_p), particles in ascending id order.
// A group of PGS lanes per cell stages PGS particles at a time in LDS; lane
// a = k*(DIM+1) + comp of the group then adds its terms in order.
// Q1: one lane per accumulator (12 or 32 lanes per cell); Q2: 27 (2-D, one
// lane each) or 108 accumulators (3-D: a group of 64 lanes, two each)
template <int DIM, int DEG = 1>
struct PartialsShape {
    static constexpr int NACC = QF<DIM, DEG>::ND * (DIM + 1);
    static constexpr int PGS = NACC <= 16 ? 16 : (NACC <= 32 ? 32 : 64);
    static constexpr int NA = (NACC + PGS - 1) / PGS;   // accumulators per lane
    static constexpr int NG = 256 / PGS;
};

template <int DIM, int DEG = 1>
__device__ __forceinline__ void partials_body(const Grid& G, int n_cells, const int* __restrict__ off, const DevParticles& A, double* __restrict__ partial, const int* __restrict__ counters) {
    if (state_dead(counters)) return;
    constexpr int NACC = PartialsShape<DIM, DEG>::NACC;
    constexpr int PGS = PartialsShape<DIM, DEG>::PGS;
    constexpr int NG = PartialsShape<DIM, DEG>::NG;
    constexpr int NA = PartialsShape<DIM, DEG>::NA;
    __shared__ double s_xi[NG][PGS][DIM];
    __shared__ double s_v[NG][PGS][DIM];
    const int g = threadIdx.x / PGS, gl = threadIdx.x % PGS;
    // lane gl holds accumulators gl, gl + PGS, ... (a = k * (DIM + 1) + comp)
    ShapeOne<DIM, DEG> sh[NA];
    int comp[NA];
#pragma unroll
    for (int u = 0; u < NA; ++u) {
        const int a = gl + u * PGS;
        const int kk = (a < NACC ? a : 0) / (DIM + 1);
        comp[u] = a - kk * (DIM + 1);
        sh[u].init(kk);
    }
    for (int cb = G.bid * NG; cb < n_cells; cb += G.nblk * NG) {
        const int c = cb + g;
        const bool cv = c < n_cells;
        const int b = cv ? off[c] : 0, e = cv ? off[c + 1] : 0;
        int trips = (e - b + PGS - 1) / PGS;
#pragma unroll
        for (int o = 1; o < WAVE; o <<= 1) trips = max(trips, __shfl_xor(trips, o));
        double acc[NA];
#pragma unroll
        for (int u = 0; u < NA; ++u) acc[u] = 0.0;
        for (int t = 0; t < trips; ++t) {
            const int j0 = b + t * PGS;
            const int j = j0 + gl;
            if (j < e) {
#pragma unroll
                for (int d = 0; d < DIM; ++d) {
                    s_xi[g][gl][d] = A.xi[(size_t)d * A.cap + j];
                    s_v[g][gl][d] = A.v[(size_t)d * A.cap + j];
                }
            }
            wave_sync();
            const int cnt = (e - j0) < PGS ? (e - j0) : PGS;
            if (gl < NACC)
                for (int q = 0; q < cnt; ++q) {
                    // N_k of this lane's node alone: per direction the
                    // factor of the node's axis, multiplied in shape_q's
                    // order, so the value is shape_q's N[k] (up to the sign
                    // of a zero factor, which no sum here sees: acc starts
                    // at +0)
                    double xi[DIM];
#pragma unroll
                    for (int d = 0; d < DIM; ++d) xi[d] = s_xi[g][q][d];
#pragma unroll
                    for (int u = 0; u < NA; ++u) {
                        const double nk = sh[u](xi);
                        if (comp[u] < DIM) {
                            double vc = s_v[g][q][0];
#pragma unroll
                            for (int d = 1; d < DIM; ++d)
                                if (d == comp[u]) vc = s_v[g][q][d];
                            acc[u] += nk * vc;
                        } else {
                            acc[u] += nk;
                        }
                    }
                }
            wave_sync();
        }
        if (cv)
#pragma unroll
            for (int u = 0; u < NA; ++u)
                if (gl + u * PGS < NACC) partial[partial_at<DIM, DEG>(n_cells, c, gl + u * PGS)] = acc[u];
    }
}

template <int DIM, int DEG = 1>
__global__ void __launch_bounds__(256) k_cell_partials(int n_cells, const int* __restrict__ off, DevParticles A,
                                                       double* __restrict__ partial, const int* __restrict__ counters) {
    partials_body<DIM, DEG>(hw_grid(), n_cells, off, A, partial, counters);
}

// k_node: node sums over the cells that contain the DoF (ascending cell
// order, TurekBenchmark/pfem2particle.cpp:895-909) divided by the weight.
// Writes V and V_old (both hold the projected field afterwards).
template <int DIM, bool FIN, int DEG = 1>
__device__ __forceinline__ void node_body(const Grid& G, const DevMesh<DIM>& m, const double* __restrict__ partial, double* __restrict__ V, double* __restrict__ Vold, unsigned long long* stats, const DevWork& w, int* queue_count) {
    constexpr int NV = Q1<DIM>::NV;   // cells per chunk
    constexpr int ND = QF<DIM, DEG>::ND;
    // FIN (a step whose regroup left its bookkeeping for later): the last
    // workgroup runs it; it depends on the cell write only, as the node sums do
    if (FIN && G.bid == G.nblk - 1) {
        finalize_block(m.n_cells, w, queue_count);
        return;
    }
    if (state_dead(w.counters)) return;
    const int nb = G.nblk - (FIN ? 1 : 0);
    for (int i = G.bid * blockDim.x + threadIdx.x; i < m.n_dofs; i += nb * blockDim.x) {
        double acc[DIM], wsum = 0.0;
#pragma unroll
        for (int d = 0; d < DIM; ++d) acc[d] = 0.0;
        // the node's cells in chunks of NV: the chunk's cell indices, then
        // its partials, are loaded together (two dependent levels per chunk
        // instead of two per cell); the sums keep the cell order
        const int e0 = m.dof_off[i], e1 = m.dof_off[i + 1];
        for (int e = e0; e < e1; e += NV) {
            int ck[NV];
#pragma unroll
            for (int q = 0; q < NV; ++q) ck[q] = e + q < e1 ? m.dof_cell[e + q] : -1;
            double pv[NV][DIM + 1];
#pragma unroll
            for (int q = 0; q < NV; ++q) {
                const int c = ck[q] >= 0 ? ck[q] / ND : 0, k = ck[q] >= 0 ? ck[q] - c * ND : 0;
                const double* p = partial + partial_at<DIM, DEG>(m.n_cells, c, k * (DIM + 1));
#pragma unroll
                for (int d = 0; d <= DIM; ++d) pv[q][d] = ck[q] >= 0 ? p[d] : 0.0;
            }
#pragma unroll
            for (int q = 0; q < NV; ++q)
                if (ck[q] >= 0) {
#pragma unroll
                    for (int d = 0; d < DIM; ++d) acc[d] += pv[q][d];
                    wsum += pv[q][DIM];
                }
        }
        if (wsum == 0.0) stat_add(stats, 4, 1ull);
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            const double val = acc[d] / wsum;
            V[(size_t)i * DIM + d] = val;
            Vold[(size_t)i * DIM + d] = val;
        }
    }
}

template <int DIM, bool FIN, int DEG = 1>
__global__ void __launch_bounds__(256) k_node(DevMesh<DIM> m, const double* __restrict__ partial,
                                              double* __restrict__ V, double* __restrict__ Vold,
                                              unsigned long long* stats, DevWork w, int* queue_count) {
    node_body<DIM, FIN, DEG>(hw_grid(), m, partial, V, Vold, stats, w, queue_count);
}

// ---------------------------------------------------------------------------
// wall fix-up (cylinderDyM/pfem2particle.cpp:960-992)
struct DevWalls {
    int n;
    const int* dof;         // per wall node
    const double* bc;       // n * 3
    const int* mask;        // per wall node
    int* fix;               // per wall node: deviation above 1e-5 in an enforced component
    double* val;            // n * 3 projected values before the fix
    const int* vwall;       // per vertex: wall index or -1
    int n_cells;            // cells adjacent to a wall node
    const int* cells;
    const int* counters;    // the handle's counters (dead-state flags)
};

template <int DIM>
__global__ void k_wall_flags(DevWalls wl, const double* __restrict__ V) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < wl.n; i += gridDim.x * blockDim.x) {
        const int dof = wl.dof[i];
        int fix = 0;
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            const double val = V[(size_t)dof * DIM + d];
            wl.val[i * 3 + d] = val;
            if (((wl.mask[i] >> d) & 1) && fabs(val - wl.bc[i * 3 + d]) > 1e-5) fix = 1;
        }
        wl.fix[i] = fix;
    }
}

// one wavefront per wall-adjacent cell; per particle the corrections of the
// cell's wall vertices are applied in ascending vertex order, as the
// reference loops over wall nodes in ascending order
template <int DIM>
__global__ void k_wall_particles(DevMesh<DIM> m, DevWalls wl, const int* __restrict__ off, DevParticles A) {
    constexpr int NV = Q1<DIM>::NV;
    const int lane = threadIdx.x & (WAVE - 1);
    const int t = blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
    if (t >= wl.n_cells || state_dead(wl.counters)) return;
    const int c = wl.cells[t];
    int order[NV], widx[NV], nw = 0;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const int gv = m.cv[(size_t)c * NV + k];
        const int wi = wl.vwall[gv];
        if (wi >= 0 && wl.fix[wi]) {
            // insertion by ascending global vertex index
            int p = nw;
            while (p > 0 && m.cv[(size_t)c * NV + order[p - 1]] > gv) {
                order[p] = order[p - 1];
                widx[p] = widx[p - 1];
                --p;
            }
            order[p] = k;
            widx[p] = wi;
            ++nw;
        }
    }
    if (nw == 0) return;
    for (int j = off[c] + lane; j < off[c + 1]; j += WAVE) {
        double xi[DIM], v[DIM], N[NV];
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            xi[d] = A.xi[(size_t)d * A.cap + j];
            v[d] = A.v[(size_t)d * A.cap + j];
        }
        shape<DIM>(xi, N);
        for (int q = 0; q < nw; ++q) {
            const int wi = widx[q];
            double nk = N[0];
#pragma unroll
            for (int r = 1; r < NV; ++r)
                if (r == order[q]) nk = N[r];
#pragma unroll
            for (int d = 0; d < DIM; ++d)
                if ((wl.mask[wi] >> d) & 1) v[d] = v[d] + nk * (wl.bc[wi * 3 + d] - wl.val[wi * 3 + d]);
        }
#pragma unroll
        for (int d = 0; d < DIM; ++d) A.v[(size_t)d * A.cap + j] = v[d];
    }
}

template <int DIM>
__global__ void k_wall_set(DevWalls wl, double* __restrict__ V, double* __restrict__ Vold) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < wl.n; i += gridDim.x * blockDim.x) {
        const int dof = wl.dof[i];
#pragma unroll
        for (int d = 0; d < DIM; ++d)
            if ((wl.mask[i] >> d) & 1) {
                V[(size_t)dof * DIM + d] = wl.bc[i * 3 + d];
                Vold[(size_t)dof * DIM + d] = wl.bc[i * 3 + d];
            }
    }
}

// ---------------------------------------------------------------------------
// seeding: q0*q1[*q2] particles per cell in lattice order, ids in cell order
// (cylinder2D/pfem2particle.cpp:487-508, 563-580)
template <int DIM, int DEG = 1>
__global__ void k_seed(DevMesh<DIM> m, const double* __restrict__ V, DevParticles A, DevParams pp,
                       uint32_t id_base, int* off) {
    constexpr int NV = Q1<DIM>::NV;
    constexpr int ND = QF<DIM, DEG>::ND;
    const long long total = (long long)m.n_cells * pp.nparts_in;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < total;
         i += (long long)gridDim.x * blockDim.x) {
        const int c = (int)(i / pp.nparts_in);
        const int o = (int)(i - (long long)c * pp.nparts_in);
        double xi[DIM], P[NV][DIM], Vc[ND][DIM], x[DIM], v[DIM];
        lattice_point<DIM>(pp, o, xi);
        load_cell_any<DIM, DEG>(m, c, P, Vc);
        forward<DIM>(P, xi, x);
        interp<DIM, DEG>(Vc, xi, v);
        A.cell[i] = c;
        A.id[i] = id_base + (uint32_t)i + 1u;
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            A.x[(size_t)d * A.cap + i] = x[d];
            A.xi[(size_t)d * A.cap + i] = xi[d];
            A.v[(size_t)d * A.cap + i] = v[d];
            if (pp.keep_vext) A.vext[(size_t)d * A.cap + i] = 0.0;
        }
        if (o == 0) off[c] = (int)i;
        if (i == total - 1) off[m.n_cells] = (int)total;
    }
}

// location from (cell, reference point) and, optionally, velocity from V, for
// particles placed by pf2_insert_particles
template <int DIM, int DEG = 1>
__global__ void k_init_particles(DevMesh<DIM> m, const double* __restrict__ V, DevParticles A,
                                 const unsigned char* __restrict__ need_v, long long n, int keep_vext) {
    constexpr int NV = Q1<DIM>::NV;
    constexpr int ND = QF<DIM, DEG>::ND;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        const int c = A.cell[i];
        double xi[DIM], P[NV][DIM], Vc[ND][DIM], x[DIM], v[DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d) xi[d] = A.xi[(size_t)d * A.cap + i];
        load_cell_any<DIM, DEG>(m, c, P, Vc);
        forward<DIM>(P, xi, x);
#pragma unroll
        for (int d = 0; d < DIM; ++d) A.x[(size_t)d * A.cap + i] = x[d];
        if (need_v[i]) {
            interp<DIM, DEG>(Vc, xi, v);
#pragma unroll
            for (int d = 0; d < DIM; ++d) A.v[(size_t)d * A.cap + i] = v[d];
        }
        if (keep_vext)
#pragma unroll
            for (int d = 0; d < DIM; ++d) A.vext[(size_t)d * A.cap + i] = 0.0;
    }
}

// re-sort after a mesh move: own-cell test with the stored last advection
// velocity, no advection; a particle that fails it (or, in 2-D, whose test
// needs inverse_map's clearly-outside test and Newton iteration) is parked
// with no substeps left for k_resort_search, which relocates it in full
// wavefronts.  skip_static: the geometry changed once since the last
// re-sort, so a particle whose cell kept its vertices and whose xi came from
// an inverse map in that cell (ids up to the counter of the last advection)
// keeps its xi and cell: the inverse map would return the same bits
template <int DIM>
__global__ void __launch_bounds__(256) k_resort(DevMesh<DIM> m, DevParticles A, DevParams pp, DevWork w,
                                                DevQueues qu, int skip_static) {
    constexpr int NV = Q1<DIM>::NV;
    const int n = state_dead(w.counters) ? 0 : w.counters[0];
    const int lane = threadIdx.x & (WAVE - 1);
    const uint32_t id_exact = (uint32_t)w.counters[5];
    const WaveLoop L = stride_loop(n);
    for (int base = L.begin; base < L.end; base += L.step) {
        const int i = base + lane;
        const bool valid = i < L.end;
        const int c = valid ? A.cell[i] : -1;
        double x[DIM], xi[DIM], vext[DIM], r[DIM];
        int st = 0;   // 0 stays, 1 relocate, 2 own-cell test pending
        if (valid) {
#pragma unroll
            for (int d = 0; d < DIM; ++d) xi[d] = A.xi[(size_t)d * A.cap + i];
            if (!(skip_static && !m.cmoved[c] && A.id[i] <= id_exact)) {
                double P[NV][DIM];
#pragma unroll
                for (int d = 0; d < DIM; ++d) x[d] = A.x[(size_t)d * A.cap + i];
                load_vertices<DIM>(m, c, P);
                if constexpr (DIM == 2) {
                    QuadCell qc;
                    qc.init(P);
                    st = closed_form(P, qc, x, r);
                } else {
                    st = contains<DIM>(m, c, P, x, r) ? 0 : 1;
                }
                if (st == 0) {
#pragma unroll
                    for (int d = 0; d < DIM; ++d) {
                        xi[d] = r[d];
                        A.xi[(size_t)d * A.cap + i] = r[d];
                    }
                } else {
#pragma unroll
                    for (int d = 0; d < DIM; ++d) vext[d] = A.vext ? A.vext[(size_t)d * A.cap + i] : 0.0;
                }
            }
            if (st == 0) {
                w.dest[i] = c;
                w.pkey[i] = part_key<DIM>(pp, xi);
            }
        }
        const int sp = pp.substeps - 1;
        park_particle<DIM>(A, w, qu, RESORT_QUEUE, L.shard, valid && st != 0, i, c, x, xi, vext,
                           st == 2 ? sp | PARK_NEWTON : sp);
    }
}

// dest / key of every particle for a reseed pass without movement
template <int DIM>
__global__ void k_keys(DevParticles A, DevParams pp, DevWork w) {
    const int n = state_dead(w.counters) ? 0 : w.counters[0];
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        double xi[DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d) xi[d] = A.xi[(size_t)d * A.cap + i];
        w.dest[i] = A.cell[i];
        w.pkey[i] = part_key<DIM>(pp, xi);
    }
}

// prescribed mesh motion: X = X0 + a W
__global__ void k_displace(const double* __restrict__ X0, const double* __restrict__ W, double a,
                           double* __restrict__ X, long long n) {
    for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < n; t += (long long)gridDim.x * blockDim.x)
        X[t] = X0[t] + a * W[t];
}

// V refreshed from a component-major device field: the node-major copy and
// the per-cell copies of V and V - V_old (FP32 copies when V32 is given; the
// FP64 V - V_old, read only by the FP64 correction, when cellDV is given)
template <int DIM>
__device__ __forceinline__ void refresh_body(const Grid& G, const DevMesh<DIM>& m, const double* __restrict__ Vcm, double* __restrict__ V, const double* __restrict__ Vold, double* __restrict__ cellV, double* __restrict__ cellDV, float* __restrict__ V32, float* __restrict__ DV32) {
    // A workgroup takes 256 (cell, DoF) pairs at a time and gives a lane one
    // component of one pair, so that the stores are contiguous and the DIM
    // lanes of a pair read V_old in one line: bound by the lines its gathers
    // and stores touch (one pair a lane: 74 us on 68,992 degree-2 hexahedra, now
    // 48; 2-D and degree 1 about the same).
    const long long nck = (long long)m.n_cells * m.nd, nd = m.n_dofs;
    const long long n = nck > nd ? nck : nd;
    for (long long t0 = G.bid * 256ll; t0 < n; t0 += G.nblk * 256ll) {
#pragma unroll
        for (int u = 0; u < DIM; ++u) {
            const unsigned j = u * 256u + threadIdx.x, q = j / DIM, d = j - q * DIM;
            const long long t = t0 + q, o = t0 * DIM + j;
            if (t < nd) V[o] = Vcm[(size_t)d * nd + t];
            if (t < nck) {
                const int dof = m.cd[t];
                const double a = Vcm[(size_t)d * nd + dof], b = Vold[(size_t)dof * DIM + d];
                if (cellV) cellV[o] = a;
                if (cellDV) cellDV[o] = a - b;
                if (V32) {
                    V32[o] = (float)a;
                    DV32[o] = (float)(a - b);
                }
            }
        }
    }
}

template <int DIM>
__global__ void k_refresh(DevMesh<DIM> m, const double* __restrict__ Vcm, double* __restrict__ V,
                          const double* __restrict__ Vold, double* __restrict__ cellV, double* __restrict__ cellDV,
                          float* __restrict__ V32, float* __restrict__ DV32) {
    refresh_body<DIM>(hw_grid(), m, Vcm, V, Vold, cellV, cellDV, V32, DV32);
}

// per-cell copies of V and V - V_old at the cell's DoFs (one load level in
// the particle kernels); V - V_old is the same per-node difference the
// correction forms (TurekBenchmark/pfem2particle.cpp:806-807)
template <int DIM>
__global__ void k_pack_fields(DevMesh<DIM> m, const double* __restrict__ V, const double* __restrict__ Vold,
                              double* __restrict__ cellV, double* __restrict__ cellDV) {
    const long long n = (long long)m.n_cells * m.nd;
    for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < n; t += (long long)gridDim.x * blockDim.x) {
        const int dof = m.cd[t];
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            const double a = V[(size_t)dof * DIM + d], b = Vold[(size_t)dof * DIM + d];
            if (cellV) cellV[(size_t)t * DIM + d] = a;
            if (cellDV) cellDV[(size_t)t * DIM + d] = a - b;
        }
    }
}

// nodal field layout conversion: component-major <-> node-major
template <int DIM>
__global__ void k_to_node_major(const double* __restrict__ src, double* __restrict__ dst, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
#pragma unroll
        for (int d = 0; d < DIM; ++d) dst[(size_t)i * DIM + d] = src[(size_t)d * n + i];
}

// particle vectors of a download: src (component-major, components `cap`
// apart) to rows dst[n][DIM] for up to three arrays (blockIdx.y)
struct RowCopies {
    const double* src[3];
    double* dst[3];
};
template <int DIM>
__global__ void k_particle_rows(RowCopies r, long long n, long long cap) {
    const double* __restrict__ s = r.src[blockIdx.y];
    double* __restrict__ o = r.dst[blockIdx.y];
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
#pragma unroll
        for (int d = 0; d < DIM; ++d) o[i * DIM + d] = s[(size_t)d * cap + i];
}

// the field and the overflow flags to host memory
template <int DIM>
__global__ void k_field_out(const double* __restrict__ src, double* __restrict__ dst, int n,
                            const int* __restrict__ counters, int* __restrict__ flags) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *flags = counters[2];
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
#pragma unroll
        for (int d = 0; d < DIM; ++d) dst[(size_t)d * n + i] = src[(size_t)i * DIM + d];
}

template <int DIM>
__global__ void k_to_comp_major(const double* __restrict__ src, double* __restrict__ dst, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
#pragma unroll
        for (int d = 0; d < DIM; ++d) dst[(size_t)d * n + i] = src[(size_t)i * DIM + d];
}

}  // namespace pf2
