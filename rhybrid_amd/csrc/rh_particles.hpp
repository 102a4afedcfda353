// rh_particles.hpp -- device kernels of the particle half of the step:
// Boris-Buneman push with the cell migration as a deterministic counting sort
// by subcell inside each tile, the cloud-in-cell deposit with fixed-order reductions, the FP64
// cross-tile ghost fold, particle boundary conditions and FP64 diagnostics.
//
// Storage (per species, structure of arrays, Real = float or double):
//   x,y,z    cell-local position in units of dx, in [0,1); x = -1 marks a
//            particle removed by the boundary conditions, or a place of a
//            segment that holds none
//   vx,vy,vz velocity in m/s
//   lc       the particle's cell inside its tile (implied by the sort order,
//            kept so that kernels need not search the slots' ranges)
// in one segment per tile, sorted inside it by slot; TileTables says where
// each slot's particles are.
#pragma once

#include <hip/hip_runtime.h>

#include "rh_geom.hpp"

namespace rh {

template <typename Real>
struct alignas(4 * sizeof(Real)) Real4 { Real v[4]; };
template <typename Real>
struct alignas(2 * sizeof(Real)) Real2 { Real v[2]; };

template <typename Real>
struct PArrays {
    Real *x, *y, *z, *vx, *vy, *vz;
    uint8_t* lc;  // the particle's cell inside its tile (local index, < 64)
};

template <typename Real>
struct PushFields {
    const Real *fbx, *fby, *fbz;   // faceB components
    const Real *uex, *uey, *uez;   // cellUe
    const Real *epx, *epy, *epz;   // cellEp
};

struct PushParams {
    double dt, dt_dx;
    double qmdt2;        // 0.5 q dt / m
    double max_vi2;
    double GMdt;
    int accelerate, use_e_pressure, use_gravity, initial_flow_through;
    int still;           // sort only: no acceleration, no move
};

enum DevCounter { C_MAX_VI = 0, C_MIN_CELL_RHO, C_MAX_CELL_UE, C_MIN_NODE_RHO, C_MAX_NODE_UE,
                  C_MAX_E, C_MAX_VW, C_DROPPED, C_DN_FALLBACK, C_RANK_OVERFLOW, C_N };

// Counters are spread over COUNTER_SLOTS copies (summed when read) so that
// waves of different blocks do not all hit one address.
constexpr int COUNTER_SLOTS = 64;

__device__ __forceinline__ void count_event(unsigned long long* counters, int id, bool pred) {
    // one atomic per wave: integer, so the total does not depend on order
    const unsigned long long b = __ballot(pred);
    const unsigned lane = (threadIdx.x + blockDim.x * threadIdx.y) & 63;
    if (b && lane == (unsigned)__builtin_ctzll(b)) {
        const unsigned slot = (blockIdx.x + 7u * blockIdx.y + 13u * blockIdx.z) & (COUNTER_SLOTS - 1);
        atomicAdd(counters + slot * C_N + id, (unsigned long long)__popcll(b));
    }
}

// The same for per-lane event counts, once per wave (every lane of the wave
// calls it)
__device__ __forceinline__ void count_events(unsigned long long* counters, int id, uint32_t n) {
    if (!__ballot(n != 0u)) return;
    for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off, 64);
    if (((threadIdx.x + blockDim.x * threadIdx.y) & 63) == 0) {
        const unsigned slot = (blockIdx.x + 7u * blockIdx.y + 13u * blockIdx.z) & (COUNTER_SLOTS - 1);
        atomicAdd(counters + slot * C_N + id, (unsigned long long)n);
    }
}

// 2 / (1 + t^2) of the Boris rotation: the hardware reciprocal (1 ulp) in
// FP32, the correctly rounded quotient in FP64
__device__ __forceinline__ float boris_s_factor(float t2) { return 2.0f * __builtin_amdgcn_rcpf(1.0f + t2); }
__device__ __forceinline__ double boris_s_factor(double t2) { return 2.0 / (1.0 + t2); }

template <typename Real> __device__ __forceinline__ Real below_one();
template <> __device__ __forceinline__ float below_one<float>() { return 0x1.fffffep-1f; }
template <> __device__ __forceinline__ double below_one<double>() { return 0x1.fffffffffffffp-1; }

// The push and the cell migration, one workgroup per tile and one pass over
// the particles (BorisBuneman::propagate, src/particle_propagator_boris_
// buneman.h:64-194, fields by face2r/cell2r, src/hybrid_propagator.cpp:
// 1740-1891, the move in FP64).  A tile owns one contiguous segment of the
// store, as long as the particles it held before the push, and writes the
// pushed particles into that segment of the other store in slot order: first
// those that stay, by subcell, then those that leave, by the halo cell they
// leave to.  A tile's particles are thus its own staying ones and, in up to
// 26 neighbours' segments, the ones that left towards it; the next push, the
// deposit and the boundary conditions read them there.  No tile needs
// another's counts before it writes, so the particles are read once and
// written once per step (a counting sort over the whole store needs a first
// pass that only counts, and writes into its neighbours' cache lines).
RH_HD size_t pm_align16(size_t b) { return (b + 15) & ~size_t(15); }

// A tile's push fields as one contiguous block (32-bit words): faceB of the
// (t+1)^3 cells -1..t-1 (halo on the low side), cellUe and cellEp of the
// tile's cells, and the cells' neighbourhood masks.  Written once per field
// update by k_push_fields and copied to LDS by k_push_sort.
template <typename Real>
RH_HD size_t push_field_words(const Geom& g) {
    const size_t nh = (size_t)(g.tx + 1) * (g.ty + 1) * (g.tz + 1);
    const size_t words = (sizeof(Real) * (3 * nh + 6 * (size_t)g.tc) + 4 * (size_t)g.tc) / 4;
    return (words + 3) & ~size_t(3);  // 16-byte blocks keep every tile's block aligned
}

// Neighbourhood mask of a cell: bit (a+1) + 3(b+1) + 9(c+1) is set when the
// neighbour at offset (a,b,c) exists; bit 27 when all 26 exist
// (pargrid::ALL_NEIGHBOURS_EXIST).
constexpr int NMASK_ALL = 27;
RH_HD uint32_t neighbour_mask(const Geom& g, int i, int j, int k) {
    // existence is separable: offset (a,b,c) exists iff each axis offset does
    uint32_t ax[3] = {0, 0, 0};
    const int idx[3] = {i, j, k}, n[3] = {g.nx, g.ny, g.nz};
    for (int d = 0; d < 3; ++d)
        for (int a = -1; a <= 1; ++a)
            if (g.per[d] || (idx[d] + a >= 0 && idx[d] + a < n[d])) ax[d] |= 1u << (a + 1);
    uint32_t m = 0;
    for (int c = 0; c < 3; ++c)
        for (int b = 0; b < 3; ++b)
            for (int a = 0; a < 3; ++a)
                if ((ax[0] >> a) & (ax[1] >> b) & (ax[2] >> c) & 1u) m |= 1u << (a + 3 * b + 9 * c);
    if (ax[0] == 7u && ax[1] == 7u && ax[2] == 7u) m |= 1u << NMASK_ALL;
    return m;
}

// Fields of the push in LDS order (see push_field_words).  One thread per
// grid cell (coalesced reads of the nine arrays): the cell writes its faceB,
// cellUe, cellEp and neighbourhood mask into its own tile's block, and its
// faceB into the low-side halo of the tiles above it when it lies on its
// tile's upper faces (up to seven, periodic wrap included).  Halo entries of
// cells that do not exist are never written and keep the zero of the
// allocation.
template <typename Real>
__device__ __forceinline__ void push_fields_store(const Geom& g, int i, int j, int k, Real bx, Real by, Real bz,
                                                  Real uex, Real uey, Real uez, Real epx, Real epy, Real epz,
                                                  int use_e_pressure, uint32_t* __restrict__ out,
                                                  bool write_mask = true, bool nowrap = false) {
    const int hx = g.tx + 1, hy = g.ty + 1, nh = (g.tx + 1) * (g.ty + 1) * (g.tz + 1);
    const size_t nw = push_field_words<Real>(g);
    const int li = i & (g.tx - 1), lj = j & (g.ty - 1), lk = k & (g.tz - 1);
    const int lc = li + (lj << g.ltx) + (lk << (g.ltx + g.lty));
    {
        Real* blk = reinterpret_cast<Real*>(out + (size_t)tile_of(g, i, j, k) * nw);
        const int h = (li + 1) + hx * ((lj + 1) + hy * (lk + 1));
        blk[h] = bx; blk[nh + h] = by; blk[2 * nh + h] = bz;
        Real* sue = blk + 3 * nh;
        Real* sep = sue + 3 * g.tc;
        sue[lc] = uex; sue[g.tc + lc] = uey; sue[2 * g.tc + lc] = uez;
        if (use_e_pressure) { sep[lc] = epx; sep[g.tc + lc] = epy; sep[2 * g.tc + lc] = epz; }
        else { sep[lc] = sep[g.tc + lc] = sep[2 * g.tc + lc] = Real(0); }
        // (the mask depends on the grid only: a caller that rewrites the
        // fields of blocks written once in full may leave it)
        if (write_mask) reinterpret_cast<uint32_t*>(sep + 3 * g.tc)[lc] = neighbour_mask(g, i, j, k);
    }
    // halo copies: the cell is local coordinate -1 of the tile above along
    // each axis where it is the tile's last cell (nowrap: the caller knows
    // that those tiles lie inside the grid without a wrap)
    // (the grid's last cell ends its tile even where the tile is partial)
    const int ux = li == g.tx - 1 || i == g.nx - 1, uy = lj == g.ty - 1 || j == g.ny - 1,
              uz = lk == g.tz - 1 || k == g.nz - 1;
    for (int c = 0; c <= uz; ++c)
        for (int b = 0; b <= uy; ++b)
            for (int a = 0; a <= ux; ++a) {
                if (a + b + c == 0) continue;
                int ti = i + a, tj = j + b, tk = k + c;
                if (!nowrap) {
                    ti = wrap_axis(ti, g.nx, g.per[0]); tj = wrap_axis(tj, g.ny, g.per[1]); tk = wrap_axis(tk, g.nz, g.per[2]);
                    if (ti < 0 || tj < 0 || tk < 0) continue;
                }
                Real* blk = reinterpret_cast<Real*>(out + (size_t)tile_of(g, ti, tj, tk) * nw);
                const int h = (a ? 0 : li + 1) + hx * ((b ? 0 : lj + 1) + hy * (c ? 0 : lk + 1));
                blk[h] = bx; blk[nh + h] = by; blk[2 * nh + h] = bz;
            }
}

template <typename Real>
__device__ __forceinline__ void push_fields_at(const Geom& g, int i, int j, int k, int n, const PushFields<Real>& f,
                                               int use_e_pressure, uint32_t* __restrict__ out) {
    push_fields_store(g, i, j, k, f.fbx[n], f.fby[n], f.fbz[n], f.uex[n], f.uey[n], f.uez[n],
                      use_e_pressure ? f.epx[n] : Real(0), use_e_pressure ? f.epy[n] : Real(0),
                      use_e_pressure ? f.epz[n] : Real(0), use_e_pressure, out);
}

template <typename Real>
__global__ __launch_bounds__(256) void k_push_fields(Geom g, PushFields<Real> f, int use_e_pressure,
                                                     uint32_t* __restrict__ out) {
    const int i = blockIdx.x * 32 + threadIdx.x, j = blockIdx.y * 8 + threadIdx.y, k = blockIdx.z;
    if (i >= g.nx || j >= g.ny) return;
    push_fields_at(g, i, j, k, cell_index(g, i, j, k), f, use_e_pressure, out);
}

// Injected particles waiting for their first push: per tile, the range of
// listed injection cells (cbeg, ntiles + 1 entries, null when none wait) and
// per listed cell the offset of its particles in the appendix, which has
// `places` places from store index `cap`, or lies at the store's end for the
// uniform fill (at_end).  slots > 0: fixed places per listed cell, whose
// offsets need no table.
struct InjAppendix {
    const uint32_t* cbeg;
    const uint32_t* off;
    uint32_t places;
    uint32_t slots;
    int at_end;
};

__device__ __forceinline__ uint32_t appendix_offset(const InjAppendix& app, uint32_t cell) {
    return app.slots ? cell * app.slots : app.off[cell];
}

// A species' scalars on the device.
enum DevScalar {
    SC_NP = 0,   // particles in the segments (removed ones included until the next push)
    SC_END,      // store indices in use by the segments
    SC_TICKET,   // blocks of k_tile_lists that are done
    SC_N
};

// Per tile DIR_WORDS store indices: where its halo slots of direction d begin
// (entry d; entry 27: where they end), and where its own particles begin and
// end.  Written by the push for every tile, also an empty one.
constexpr int DIR_WORDS = 32, DIR_OWN = 28;
// Per tile LIST_WORDS: where its particles are, as one sequence.  Its
// arrivals from offset j (j%3-1, (j/3)%3-1, j/9-1) are arrivals LIST_PREF + j
// to LIST_PREF + j + 1 of the sequence, arrival v at store index
// (LIST_START + j) + v; LIST_OWN: its own particles' first index and count.
constexpr int LIST_WORDS = 64, LIST_START = 0, LIST_PREF = 27, LIST_OWN = 55;

// Where a tile's particles are (written by the push, read by everything
// after it): per tile g.kt store indices, tab[T*kt + s] .. tab[T*kt + s + 1]
// the range of slot s.  Slots 0 .. 8*tc-1 are the tile's subcells; then come
// the halo cells of the tile's extended region, grouped by the direction
// (a+1) + 3(b+1) + 9(c+1) they lie in; dir[d] is the first slot of direction
// d, dir[27] the end.  slot[e] is the slot of extended cell e outside the
// tile.  The tables of a tile that held nothing (live 0) are not written.
// lists: particles may wait in halo slots (not after an upload or a merge).
struct TileTables {
    const uint32_t* tab;
    const uint8_t* live;
    const uint16_t* dir;
    const uint16_t* slot;
    int lists;
};

// Slots of a tile shape: dir (28 entries) and slot (g.next entries).
inline void tile_slots(const Geom& g, uint16_t* dir, uint16_t* slot) {
    int s = 8 * g.tc;
    for (int d = 0; d < 27; ++d) {
        dir[d] = (uint16_t)s;
        if (d == 13) continue;
        const int a[3] = {d % 3 - 1, (d / 3) % 3 - 1, d / 9 - 1}, t[3] = {g.tx, g.ty, g.tz};
        int lo[3], hi[3];
        for (int q = 0; q < 3; ++q) {
            lo[q] = a[q] < 0 ? 0 : (a[q] > 0 ? t[q] + 1 : 1);
            hi[q] = a[q] == 0 ? t[q] : lo[q];
        }
        for (int z = lo[2]; z <= hi[2]; ++z)
            for (int y = lo[1]; y <= hi[1]; ++y)
                for (int x = lo[0]; x <= hi[0]; ++x) slot[x + g.ex * (y + g.ey * z)] = (uint16_t)s++;
    }
    dir[27] = (uint16_t)s;
    for (int e = 0; e < g.next; ++e) {
        const int x = e % g.ex, y = (e / g.ex) % g.ey, z = e / (g.ex * g.ey);
        if (x >= 1 && x <= g.tx && y >= 1 && y <= g.ty && z >= 1 && z <= g.tz) slot[e] = 0;  // the tile's own
    }
}

// The source tile of the arrivals of tile (bx,by,bz) from offset (a,b,c);
// -1 where there is none.
__device__ __forceinline__ int neighbour_tile(const Geom& g, int bx, int by, int bz, int a, int b, int c) {
    int x = bx + a, y = by + b, z = bz + c;
    if (x < 0 || x >= g.ntx) { if (!g.per[0]) return -1; x += x < 0 ? g.ntx : -g.ntx; }
    if (y < 0 || y >= g.nty) { if (!g.per[1]) return -1; y += y < 0 ? g.nty : -g.nty; }
    if (z < 0 || z >= g.ntz) { if (!g.per[2]) return -1; z += z < 0 ? g.ntz : -g.ntz; }
    return x + g.ntx * (y + g.nty * z);
}

// Store index of a tile's arrival v: in the last list that starts at or before v.
__device__ __forceinline__ uint32_t arrival_index(const uint32_t* lists, uint32_t v) {
    int j = 0;
#pragma unroll
    for (int s = 16; s > 0; s >>= 1)
        if (j + s <= 26 && lists[LIST_PREF + j + s] <= v) j += s;
    return lists[LIST_START + j] + v;
}

// f(first, end) for every store range that holds particles of cell (i,j,k):
// its own subcells', then the halo cells of neighbouring tiles that it is.
template <typename F>
__device__ __forceinline__ void cell_ranges(const Geom& g, const TileTables& t, int i, int j, int k, F&& f) {
    const int c[3] = {i, j, k}, n[3] = {g.nx, g.ny, g.nz}, lt[3] = {g.ltx, g.lty, g.ltz}, nt[3] = {g.ntx, g.nty, g.ntz};
    int b[3], l[3], lo[3], hi[3];  // tile, local coordinate, whether a lower / upper neighbour's halo holds the cell
    for (int d = 0; d < 3; ++d) {
        b[d] = c[d] >> lt[d];
        l[d] = c[d] - (b[d] << lt[d]);
        lo[d] = l[d] == 0 && (b[d] > 0 || g.per[d]);
        hi[d] = l[d] == tile_width(n[d], lt[d], b[d]) - 1 && (b[d] < nt[d] - 1 || g.per[d]);
    }
    const int T = b[0] + g.ntx * (b[1] + g.nty * b[2]);
    if (t.live[T]) {
        const uint32_t* tab = t.tab + (size_t)T * g.kt + 8 * (l[0] + (l[1] << g.ltx) + (l[2] << (g.ltx + g.lty)));
        f(tab[0], tab[8]);
    }
    if (!t.lists) return;
    for (int z = -lo[2]; z <= hi[2]; ++z)
        for (int y = -lo[1]; y <= hi[1]; ++y)
            for (int x = -lo[0]; x <= hi[0]; ++x) {
                if (!x && !y && !z) continue;
                const int S = neighbour_tile(g, b[0], b[1], b[2], x, y, z);
                if (S < 0 || !t.live[S]) continue;
                const int ex = x < 0 ? g.tx + 1 : (x > 0 ? 0 : l[0] + 1), ey = y < 0 ? g.ty + 1 : (y > 0 ? 0 : l[1] + 1),
                          ez = z < 0 ? g.tz + 1 : (z > 0 ? 0 : l[2] + 1);
                const uint32_t* tab = t.tab + (size_t)S * g.kt + t.slot[ex + g.ex * (ey + g.ey * ez)];
                f(tab[0], tab[1]);
            }
}

// inclusive sum over the lanes of a wave: DPP row shifts, then row broadcasts
__device__ __forceinline__ uint32_t wave_inclusive(uint32_t v) {
    int x = (int)v;
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false);  // row_shr 1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false);  // row_shr 2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false);  // row_shr 4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false);  // row_shr 8
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false);  // lane 15 of each row to the next one
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false);  // lane 31 to the upper half
    return (uint32_t)x;
}

// a value that is the same in every lane, in a scalar register
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }

// exclusive prefix of v over the block (at most 16 waves; wsum: 16 words);
// total in every thread
template <int NT>
__device__ __forceinline__ uint32_t block_prefix(uint32_t v, uint32_t* wsum, uint32_t& total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t inc = wave_inclusive(v);
    if (lane == 63) wsum[w] = inc;
    __syncthreads();
    const uint32_t sums = wave_inclusive(lane < NT / 64 ? wsum[lane] : 0u);
    total = (uint32_t)__builtin_amdgcn_readlane((int)sums, NT / 64 - 1);
    const int wu = __builtin_amdgcn_readfirstlane(w);
    const uint32_t base = wu ? (uint32_t)__builtin_amdgcn_readlane((int)sums, wu - 1) : 0u;
    return base + inc - v;
}

// After a push: every tile's lists (half a wave per tile, one lane per
// neighbour), and its segment in the store the next push writes, as many
// places as it has particles: loc[T] + blk[T / TILES_PER_LIST_BLOCK], plus the
// injected particles of the tiles before it.  The last block to finish scans
// the block sums, so one launch does both (18,432 tiles of the 128x96x96 box
// are 576 sums; a second launch would cost more than the scan).
constexpr int LIST_THREADS = 1024;
constexpr int TILES_PER_LIST_BLOCK = LIST_THREADS / 32;

__global__ __launch_bounds__(LIST_THREADS) void k_tile_lists(Geom g, const uint32_t* __restrict__ dtab,
                                                             uint32_t* __restrict__ lists, uint32_t* __restrict__ loc,
                                                             uint32_t* __restrict__ blk, uint32_t* __restrict__ scal) {
    __shared__ uint32_t wsum[LIST_THREADS / 64], cnt[TILES_PER_LIST_BLOCK];
    __shared__ uint32_t last;
    const int tid = threadIdx.x, lane = tid & 31;
    const int T = blockIdx.x * TILES_PER_LIST_BLOCK + (tid >> 5);
    uint32_t s0 = 0, n = 0;
    if (T < g.ntiles && lane < 27) {
        int bx, by, bz;
        tile_coords(g, T, bx, by, bz);
        const int S = neighbour_tile(g, bx, by, bz, lane % 3 - 1, (lane / 3) % 3 - 1, lane / 9 - 1);
        if (S >= 0) {
            // the direction from the neighbour to the tile; the tile itself: its own particles
            const uint32_t* d = dtab + (size_t)S * DIR_WORDS + (lane == 13 ? DIR_OWN : 26 - lane);
            s0 = d[0];
            n = d[1] - s0;
        }
    }
    const uint32_t n0 = __shfl(n, 13, 32), p0 = __shfl(s0, 13, 32);
    if (lane == 13) n = 0;
    uint32_t inc = n;
#pragma unroll
    for (int off = 1; off < 32; off <<= 1) {
        const uint32_t o = __shfl_up(inc, off, 32);
        if (lane >= off) inc += o;
    }
    if (T < g.ntiles) {
        uint32_t* L = lists + (size_t)T * LIST_WORDS;
        if (lane < 27) {
            L[LIST_START + lane] = s0 - (inc - n);
            L[LIST_PREF + 1 + lane] = inc;
        } else if (lane == 27) {
            L[LIST_PREF] = 0;
        } else if (lane == 28) {
            L[LIST_OWN] = p0;
            L[LIST_OWN + 1] = n0;
        }
    }
    if (lane == 31) cnt[tid >> 5] = T < g.ntiles ? n0 + inc : 0u;
    __syncthreads();
    uint32_t total;
    const uint32_t pre = block_prefix<LIST_THREADS>(tid < TILES_PER_LIST_BLOCK ? cnt[tid] : 0u, wsum, total);
    const int Ts = blockIdx.x * TILES_PER_LIST_BLOCK + tid;
    if (tid < TILES_PER_LIST_BLOCK && Ts < g.ntiles) loc[Ts] = pre;
    if (tid == 0) {
        // (the sums go around the caches, so the ticket need not write back
        // and invalidate an L2 per block; only its order after the store
        // matters: 27 -> 15 us per launch)
        __hip_atomic_store(blk + blockIdx.x, total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        last = __hip_atomic_fetch_add(scal + SC_TICKET, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
    }
    __syncthreads();
    if (!last) return;
    uint32_t run = 0;
    for (uint32_t b0 = 0; b0 < gridDim.x; b0 += LIST_THREADS) {
        const uint32_t b = b0 + tid;
        const uint32_t v = b < gridDim.x ? __hip_atomic_load(blk + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0u;
        uint32_t tot;
        __syncthreads();  // the previous round's sums are read
        const uint32_t p = block_prefix<LIST_THREADS>(v, wsum, tot);
        if (b < gridDim.x) blk[b] = run + p;
        run += tot;
    }
    if (tid == 0) {
        scal[SC_NP] = run;  // all that the tiles hold
        scal[SC_TICKET] = 0;
    }
}

// How full the tiles are, for the choice of the push's workgroups: of about
// FILL_SAMPLE tiles spread over the grid the number that hold
// 64c-63 .. 64c particles, per class c (the last class also fuller ones;
// empty tiles are class 0), and the most that one holds.  One block, every few
// pushes; it writes to pinned memory of the host (words LOOK_*), which waits
// for an event after it: no copy that the next kernels would queue behind.
constexpr int FILL_CLASSES = 128, FILL_SAMPLE = 4096, FILL_THREADS = 1024;
enum LookWord { LOOK_NP = 0, LOOK_MOST, LOOK_CLASS, LOOK_WORDS = LOOK_CLASS + FILL_CLASSES };
RH_HD int fill_class(uint32_t n) { return n >= 64u * (FILL_CLASSES - 1) ? FILL_CLASSES - 1 : (int)((n + 63u) / 64u); }

__global__ __launch_bounds__(FILL_THREADS) void k_tile_fill(Geom g, const uint32_t* __restrict__ lists,
                                                            const uint32_t* __restrict__ scal, uint32_t* __restrict__ look) {
    __shared__ uint32_t h[FILL_CLASSES], most;
    const int tid = threadIdx.x, stride = (g.ntiles + FILL_SAMPLE - 1) / FILL_SAMPLE;
    if (tid < FILL_CLASSES) h[tid] = 0;
    if (tid == 0) most = 0;
    __syncthreads();
    for (int T = tid * stride; T < g.ntiles; T += FILL_THREADS * stride) {
        const uint32_t* L = lists + (size_t)T * LIST_WORDS;
        const uint32_t n = L[LIST_PREF + 27] + L[LIST_OWN + 1];
        atomicAdd(&h[fill_class(n)], 1u);
        if (n >= 64u * (FILL_CLASSES - 1)) atomicMax(&most, n);
    }
    __syncthreads();
    if (tid < FILL_CLASSES) look[LOOK_CLASS + tid] = h[tid];
    if (tid == 0) {
        look[LOOK_NP] = scal[SC_NP];
        look[LOOK_MOST] = most;
    }
}

// A Geom whose tile shape is known to the compiler: sides 2^LX, 2^LY, 2^LZ
// (LX < 0: as g says).
template <int LX, int LY, int LZ>
__device__ __forceinline__ Geom with_shape(const Geom& g) {
    Geom h = g;
    if constexpr (LX >= 0) {
        h.ltx = LX; h.lty = LY; h.ltz = LZ;
        h.tx = 1 << LX; h.ty = 1 << LY; h.tz = 1 << LZ;
        h.tc = h.tx * h.ty * h.tz;
        h.ex = h.tx + 2; h.ey = h.ty + 2; h.ez = h.tz + 2;
        h.next = h.ex * h.ey * h.ez;
        h.extk = 8 * h.next;
        set_slots(h);
    }
    return h;
}

// LDS of k_push_sort: one round's pushed particles (24 B in FP32) and their
// codes, its list of particles by slot (each slot's part padded to an even
// count), the slots' counts, list parts and places, the extended cells'
// codes, the tile's field block.
template <typename Real>
struct PushLds {
    size_t s2, code, list, cnt, loff, goff, codes, field, bytes;
};
template <typename Real>
RH_HD PushLds<Real> push_lds(const Geom& g, int round, int lq) {
    const size_t kq = (size_t)g.kt << lq;
    PushLds<Real> o;
    o.s2 = 4 * sizeof(Real) * (size_t)round;
    o.code = o.s2 + 2 * sizeof(Real) * (size_t)round;
    o.list = o.code + 4 * (size_t)round;
    o.cnt = o.list + pm_align16(2 * ((size_t)round + kq));
    o.loff = o.cnt + pm_align16(4 * kq);
    o.goff = o.loff + pm_align16(2 * kq);
    o.codes = o.goff + pm_align16(4 * (size_t)g.kt);
    o.field = o.codes + pm_align16(4 * ((size_t)g.next + 1));
    o.bytes = o.field + 4 * push_field_words<Real>(g);
    return o;
}

// A particle's code in the push: its slot (g.nslot: removed), in CODE_OCT the
// octant bits that the slot still lacks (7 for a cell of the tile), then its
// rank in the round and the destination's local cell.
constexpr uint32_t SLOT_BITS = 10, SLOT_MASK = (1u << SLOT_BITS) - 1u;
constexpr uint32_t CODE_OCT_SHIFT = SLOT_BITS;
constexpr uint32_t RANK_SHIFT = SLOT_BITS, RANK_ROUND_BITS = 13, RANK_MASK_ROUND = (1u << RANK_ROUND_BITS) - 1u;
constexpr uint32_t CELL_SHIFT = RANK_SHIFT + RANK_ROUND_BITS;

// Host: the codes of the extended cells of a tile with full neighbours on
// all sides, and per extended cell in which directions it leaves the tile
// (bit 0 -x, 1 +x, 2 -y, 3 +y, 4 -z, 5 +z).
inline void tile_codes(const Geom& g, const uint16_t* slots, uint32_t* code, uint32_t* side) {
    for (int e = 0; e < g.next; ++e) {
        const int t[3] = {g.tx, g.ty, g.tz};
        int l[3] = {e % g.ex - 1, (e / g.ex) % g.ey - 1, e / (g.ex * g.ey) - 1};
        side[e] = 0;
        for (int d = 0; d < 3; ++d) {
            if (l[d] < 0) { side[e] |= 1u << (2 * d); l[d] = t[d] - 1; }
            else if (l[d] >= t[d]) { side[e] |= 2u << (2 * d); l[d] = 0; }
        }
        const uint32_t nlc = (uint32_t)(l[0] + (l[1] << g.ltx) + (l[2] << (g.ltx + g.lty)));
        code[e] = side[e] ? (uint32_t)slots[e] | nlc << CELL_SHIFT : 8u * nlc | 7u << CODE_OCT_SHIFT | nlc << CELL_SHIFT;
    }
}

// The code of extended cell e of tile (bx,by,bz): a cell of the tile, of a
// neighbouring tile (with that tile's local cell), or none (outside a
// non-periodic grid, or beyond the halo of a partial tile).
__device__ __forceinline__ uint32_t cell_code(const Geom& g, int bx, int by, int bz, int e, const uint16_t* slots) {
    const int b[3] = {bx, by, bz}, n[3] = {g.nx, g.ny, g.nz}, lt[3] = {g.ltx, g.lty, g.ltz}, nt[3] = {g.ntx, g.nty, g.ntz},
              t[3] = {g.tx, g.ty, g.tz};
    const int l[3] = {e % g.ex - 1, (e / g.ex) % g.ey - 1, e / (g.ex * g.ey) - 1};
    bool own = true, exists = true;
    int c[3], x[3];  // destination's local coordinate; extended coordinate in a full tile
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const int w = tile_width(n[d], lt[d], b[d]);
        c[d] = l[d];
        x[d] = l[d] + 1;
        if (l[d] < 0) {
            own = false;
            exists = exists && (b[d] > 0 || g.per[d]);
            c[d] = tile_width(n[d], lt[d], b[d] > 0 ? b[d] - 1 : nt[d] - 1) - 1;
        } else if (l[d] >= w) {
            own = false;
            exists = exists && l[d] == w && (b[d] < nt[d] - 1 || g.per[d]);
            c[d] = 0;
            x[d] = t[d] + 1;
        }
    }
    const uint32_t nlc = (uint32_t)(c[0] + (c[1] << g.ltx) + (c[2] << (g.ltx + g.lty)));
    if (own) return 8u * nlc | 7u << CODE_OCT_SHIFT | nlc << CELL_SHIFT;
    if (!exists) return (uint32_t)g.nslot;
    return (uint32_t)slots[x[0] + g.ex * (x[1] + g.ey * x[2])] | nlc << CELL_SHIFT;
}

template <typename Real>
struct Particle {
    Real X, Y, Z, vx, vy, vz;
};

// The particle's code from its extended cell (g.next: removed) and place in it.
template <typename Real>
__device__ __forceinline__ uint32_t particle_code(const uint32_t* codes, int e, const Particle<Real>& q) {
    const uint32_t code = codes[e];
    const uint32_t o = (q.X >= Real(0.5)) + 2 * (q.Y >= Real(0.5)) + 4 * (q.Z >= Real(0.5));
    return (code & ~(7u << CODE_OCT_SHIFT)) + (o & (code >> CODE_OCT_SHIFT & 7u));
}

// One particle: push, move, code.  fl is the tile's field block, codes its
// extended cells' codes, e the extended cell it ends in; edge: the tile holds cells without all neighbours.
// PLAIN: accelerated, without gravity, and moved (the parameters of most
// runs; the others are tested for).  Without branches except for the speed
// limit, so that several particles' LDS reads are in flight.
template <typename Real, bool PLAIN>
__device__ __forceinline__ uint32_t push_particle(const Geom& g, const PushParams& pp, const int (&org)[3], bool edge,
                                                  const Real* fl, const uint32_t* codes, Particle<Real>& q, int lc,
                                                  int& e, uint32_t& n_clamped, uint32_t& n_dropped) {
    const bool act = q.X >= Real(0);
    const int hx = g.tx + 1, hy = g.ty + 1, nh = (g.tx + 1) * (g.ty + 1) * (g.tz + 1);
    const Real* sbx = fl;  // faceB of local cells -1..t-1 (halo on the low side)
    const Real* sby = fl + nh;
    const Real* sbz = fl + 2 * nh;
    const Real* sue = fl + 3 * nh;  // cellUe, cellEp of the tile's cells
    const Real* sep = sue + 3 * g.tc;
    Real X = q.X, Y = q.Y, Z = q.Z, vx = q.vx, vy = q.vy, vz = q.vz;
    int li, lj, lk;
    local_ijk(g, lc, li, lj, lk);
    bool accel = PLAIN || (pp.accelerate && !pp.initial_flow_through);
    // (the neighbourhood mask of the cell)
    if (edge) accel = accel && ((reinterpret_cast<const uint32_t*>(sep + 3 * g.tc)[lc] >> NMASK_ALL) & 1u);
    if (PLAIN || (pp.accelerate && !pp.initial_flow_through)) {
        const int h = (li + 1) + hx * ((lj + 1) + hy * (lk + 1));
        // face2r: each component linear along its own axis only
        const Real Bx = X * sbx[h] + (Real(1) - X) * sbx[h - 1];
        const Real By = Y * sby[h] + (Real(1) - Y) * sby[h - hx];
        const Real Bz = Z * sbz[h] + (Real(1) - Z) * sbz[h - hx * hy];
        // cell2r: nearest grid point; E = B x Ue (= -Ue x B) (+ Ep)
        const Real Ux = sue[lc], Uy = sue[g.tc + lc], Uz = sue[2 * g.tc + lc];
        Real Ex = By * Uz - Bz * Uy;
        Real Ey = Bz * Ux - Bx * Uz;
        Real Ez = Bx * Uy - By * Ux;
        Ex += sep[lc]; Ey += sep[g.tc + lc]; Ez += sep[2 * g.tc + lc];
        const Real qm = (Real)pp.qmdt2;
        const Real dvx = qm * Ex, dvy = qm * Ey, dvz = qm * Ez;
        const Real tx = qm * Bx, ty = qm * By, tz = qm * Bz;
        const Real t2 = tx * tx + ty * ty + tz * tz;
        const Real b2 = boris_s_factor(t2);
        const Real sx = b2 * tx, sy = b2 * ty, sz = b2 * tz;
        const Real vmx = vx + dvx, vmy = vy + dvy, vmz = vz + dvz;
        const Real v0x = vmx + vmy * tz - vmz * ty;
        const Real v0y = vmy + vmz * tx - vmx * tz;
        const Real v0z = vmz + vmx * ty - vmy * tx;
        vx = vmx + v0y * sz - v0z * sy + dvx;
        vy = vmy + v0z * sx - v0x * sz + dvy;
        vz = vmz + v0x * sy - v0y * sx + dvz;
        if (!PLAIN && pp.use_gravity) {
            const double rx = g.x0 + (org[0] + li + (double)X) * g.dx;
            const double ry = g.y0 + (org[1] + lj + (double)Y) * g.dx;
            const double rz = g.z0 + (org[2] + lk + (double)Z) * g.dx;
            const double r = sqrt(rx * rx + ry * ry + rz * rz);
            const double r3 = r * r * r;
            if (r3 > 0) {
                const double s = -pp.GMdt / r3;
                vx += (Real)(s * rx); vy += (Real)(s * ry); vz += (Real)(s * rz);
            }
        }
        const Real v2 = vx * vx + vy * vy + vz * vz;
        if (act && accel && v2 > (Real)pp.max_vi2) {
            const Real norm = sqrt((Real)pp.max_vi2 / v2);
            vx *= norm; vy *= norm; vz *= norm;
            ++n_clamped;
        }
        if (edge) {  // particles of cells without all neighbours keep their velocity
            vx = accel ? vx : q.vx; vy = accel ? vy : q.vy; vz = accel ? vz : q.vz;
        }
    }
    // move in FP64; the integer part is the cell crossing (a still pass keeps
    // every particle where it is)
    int sx = 0, sy = 0, sz = 0;
    if (PLAIN || !pp.still) {
        const double Xd = (double)X + (double)vx * pp.dt_dx;
        const double Yd = (double)Y + (double)vy * pp.dt_dx;
        const double Zd = (double)Z + (double)vz * pp.dt_dx;
        sx = (int)floor(Xd); sy = (int)floor(Yd); sz = (int)floor(Zd);
        // (a tiny negative Xd has the fraction next below one, as the
        // difference from its floor, which rounds to one, has after the limit)
        X = (Real)__builtin_amdgcn_fract(Xd); Y = (Real)__builtin_amdgcn_fract(Yd); Z = (Real)__builtin_amdgcn_fract(Zd);
    }
    // at most one cell along each axis, and nothing that is not a number (a
    // still pass keeps that too)
    const bool ok = (unsigned)(sx + 1) <= 2u && (unsigned)(sy + 1) <= 2u && (unsigned)(sz + 1) <= 2u &&
                    (X + Y + Z >= Real(0) || (!PLAIN && pp.still));
    if (PLAIN || !pp.still) {
        X = X < Real(1) ? X : below_one<Real>();
        Y = Y < Real(1) ? Y : below_one<Real>();
        Z = Z < Real(1) ? Z : below_one<Real>();
    }
    e = act && ok ? (li + sx + 1) + g.ex * ((lj + sy + 1) + g.ey * (lk + sz + 1)) : g.next;
    q.X = X; q.Y = Y; q.Z = Z; q.vx = vx; q.vy = vy; q.vz = vz;
    const uint32_t code = particle_code(codes, e, q);
    n_dropped += act && (code & SLOT_MASK) == (uint32_t)g.nslot;
    return code;
}

// How many of the slot's list entries (from `part`, c of them, padded with
// 0xFFFF to an even count) are below `me`: two to a word, two words at a time.
__device__ __forceinline__ uint32_t list_rank(const uint16_t* part, uint32_t c, uint32_t me) {
    const uint32_t m = me | me << 16, words = (c + 1) / 2;
    const uint32_t* w = reinterpret_cast<const uint32_t*>(part);
    auto below = [&](uint32_t two) {  // (me - entry, limited to 0 and 1, in each half)
        uint32_t a;
        asm("v_pk_sub_u16 %0, %1, %2 clamp" : "=v"(a) : "v"(m), "v"(two));
        asm("v_pk_min_u16 %0, %1, 1 op_sel_hi:[1,0]" : "=v"(a) : "v"(a));
        return a;
    };
    uint32_t r = 0, e = 0;
#pragma clang loop unroll(disable)
    for (; e + 2 <= words; e += 2) r += below(w[e]) + below(w[e + 1]);
    if (e < words) r += below(w[e]);
    return (r & 0xFFFFu) + (r >> 16);
}

// A tile whose particles fit one round (`round` of them, as the LDS was sized
// for) is read once: each pushed particle waits in LDS while the slots are
// counted (integer LDS atomics) and scanned, and is then written to its
// place, a wave writing 64 places in a row (written by the particles' own
// order instead, a wave's places lie in up to twice as many cache lines and
// the address units bound the kernel).  A fuller tile is pushed
// once too, for the counts, but waits in place of its input, and is then
// ranked and written round by round (pushed again in every round, for the code
// and to be written, the photoions of 160x128x128, up to 12,000 in a tile, take
// 429 us instead of 333).  A particle's
// rank in its slot is the number of the round's particles of that slot that
// come before it: the atomics hand out places of a list by slot in any order,
// and each particle then counts the smaller entries of its slot's few, so the
// sort is stable: the written order is that of the particles alone.
// Where slots hold many, neighbouring particles, which are of one slot, count
// in 2^lq parts of it in turn (fewer LDS atomics to one address); a slot's
// parts lie side by side in the list and are ranked as one, so the order does
// not depend on lq (64x32x32 with 256 per cell, ten steps: 11.65 ms, 11.88
// without parts, 11.33 ranked part by part, which is not stable; 11.47 with
// the list read two words at a time).
template <typename Real, int NT, int LX, int LY, int LZ, bool PLAIN>
__global__ __launch_bounds__(NT, sizeof(Real) == 8 ? 4 : 6) void k_push_sort(
    Geom g_, PushParams pp, const uint32_t* __restrict__ pfb, PArrays<Real> A, PArrays<Real> D,
    const uint16_t* __restrict__ dirs,
    const uint16_t* __restrict__ slots, const uint32_t* __restrict__ full_codes, uint32_t* __restrict__ tab_out,
    uint32_t* __restrict__ dtab_out, uint8_t* __restrict__ live_out, const uint32_t* __restrict__ lists,
    const uint32_t* __restrict__ seg_loc, const uint32_t* __restrict__ seg_blk, InjAppendix app,
    uint32_t* __restrict__ scal, unsigned long long* __restrict__ counters, uint32_t cap, int round, int lq) {
    const Geom g = with_shape<LX, LY, LZ>(g_);
    extern __shared__ __align__(16) unsigned char pm_smem[];
    __shared__ uint32_t wsum[16], L[LIST_WORDS];
    const int NS = 8 * g.tc, K = g.nslot;
    const int KQ = K << lq, KT = g.kt << lq, pm = (1 << lq) - 1;  // the parts of the slots
    const PushLds<Real> o = push_lds<Real>(g, round, lq);
    Real4<Real>* S4 = reinterpret_cast<Real4<Real>*>(pm_smem);         // x, y, z, vx
    Real2<Real>* S2 = reinterpret_cast<Real2<Real>*>(pm_smem + o.s2);  // vy, vz
    uint32_t* scode = reinterpret_cast<uint32_t*>(pm_smem + o.code);
    uint16_t* list = reinterpret_cast<uint16_t*>(pm_smem + o.list);
    uint32_t* cnt = reinterpret_cast<uint32_t*>(pm_smem + o.cnt);    // this round's particles per slot (entry K: the removed)
    uint16_t* loff = reinterpret_cast<uint16_t*>(pm_smem + o.loff);  // where the slot's part of the list starts
    uint32_t* goff = reinterpret_cast<uint32_t*>(pm_smem + o.goff);  // the slot's next place in the slot order
    uint32_t* codes = reinterpret_cast<uint32_t*>(pm_smem + o.codes);
    Real* fl = reinterpret_cast<Real*>(pm_smem + o.field);
    const int T = xcd_tile(g, (int)blockIdx.x);
    if (T >= g.ntiles) return;
    const int tid = threadIdx.x, lane = tid & 63;
    // the tile's lists, one word per lane, and everything else that does not
    // depend on them: one round of latency, then the particles' own
    const uint32_t lw = lists[(size_t)T * LIST_WORDS + lane];
    const uint32_t np = scal[SC_NP], sloc = seg_loc[T], sblk = seg_blk[T / TILES_PER_LIST_BLOCK];
    const int mydir = tid < 28 ? (int)dirs[tid] : 0;
    uint32_t c0 = 0, c1 = 0;
    if (app.cbeg) { c0 = app.cbeg[T]; c1 = app.cbeg[T + 1]; }
    int bx, by, bz;
    tile_coords(g, T, bx, by, bz);
    const int org[3] = {bx << g.ltx, by << g.lty, bz << g.ltz};
    const bool edge = (!g.per[0] && (org[0] < 1 || org[0] + g.tx > g.nx - 1)) ||
                      (!g.per[1] && (org[1] < 1 || org[1] + g.ty > g.ny - 1)) ||
                      (!g.per[2] && (org[2] < 1 || org[2] + g.tz > g.nz - 1));
    const uint32_t p0 = (uint32_t)__builtin_amdgcn_readlane((int)lw, LIST_OWN),
                   n0 = (uint32_t)__builtin_amdgcn_readlane((int)lw, LIST_OWN + 1),
                   na = (uint32_t)__builtin_amdgcn_readlane((int)lw, LIST_PREF + 27);
    // (uniform base pointers and 32-bit offsets for the tile's own places)
    auto own = [&](uint32_t u, Particle<Real>& q, int& lc) {
        q.X = (A.x + p0)[u]; q.Y = (A.y + p0)[u]; q.Z = (A.z + p0)[u];
        q.vx = (A.vx + p0)[u]; q.vy = (A.vy + p0)[u]; q.vz = (A.vz + p0)[u];
        lc = (A.lc + p0)[u];
    };
    Particle<Real> nq{Real(-1), Real(0), Real(0), Real(0), Real(0), Real(0)};  // the thread's next particle
    int nlc = 0;
    if ((uint32_t)tid < n0) own((uint32_t)tid, nq, nlc);
    const uint32_t room = min(cap > np ? cap - np : 0u, app.places);
    uint32_t a0 = 0, a1 = 0, before = 0;  // injected particles: the tile's, those of the tiles before it
    if (app.cbeg) {
        before = min(appendix_offset(app, c0), room);
        a0 = before;
        a1 = min(appendix_offset(app, c1), room);
    }
    const uint32_t n1 = n0 + na, N = uniform(n1 + (a1 - a0));
    a0 += app.at_end ? np : cap;
    // the segment: the places of the tiles before it
    const uint32_t seg = uniform(sloc + sblk + before);
    if (tid == 0) {
        live_out[T] = N > 0;
        if (T == 0) scal[SC_END] = np + (app.cbeg ? min(appendix_offset(app, app.cbeg[g.ntiles]), room) : 0u);
    }
    if (N == 0) {  // the slot tables of an empty tile are not read
        if (tid < DIR_WORDS) dtab_out[(size_t)T * DIR_WORDS + tid] = seg;
        return;
    }
    if (tid < LIST_WORDS) L[tid] = lw;
    // the others: arrivals, then injected particles
    auto other_place = [&](uint32_t v) { return v < na ? arrival_index(L, v) : a0 + (v - na); };
    auto place = [&](uint32_t u) { return u < n0 ? p0 + u : other_place(u - n0); };
    auto other = [&](uint32_t v, Particle<Real>& q, int& lc) {
        const uint32_t p = other_place(v);
        q.X = A.x[p]; q.Y = A.y[p]; q.Z = A.z[p];
        q.vx = A.vx[p]; q.vy = A.vy[p]; q.vz = A.vz[p];
        lc = A.lc[p];
    };
    const uint32_t places = cap > seg ? cap - seg : 0u;
    const bool one = N <= (uint32_t)round;
    for (int e = tid; e < KT; e += NT) cnt[e] = 0u;
    for (int e = tid; e < (round + KT) / 2; e += NT) reinterpret_cast<uint32_t*>(list)[e] = ~0u;
    {
        const int nw4 = (int)push_field_words<Real>(g) / 4;
        const uint4* src = reinterpret_cast<const uint4*>(pfb) + (size_t)T * nw4;
        uint4* dst = reinterpret_cast<uint4*>(fl);
        for (int e = tid; e < nw4; e += NT) dst[e] = src[e];
        // the extended cells' codes: those of a tile amid full ones, less the
        // cells that do not exist; beside a partial tile (also across a wrap)
        // they differ
        const int b[3] = {bx, by, bz}, n[3] = {g.nx, g.ny, g.nz}, lt[3] = {g.ltx, g.lty, g.ltz}, nt[3] = {g.ntx, g.nty, g.ntz};
        uint32_t missing = 0;
        bool full = true;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            if (!g.per[d] && b[d] == 0) missing |= 1u << (2 * d);
            if (!g.per[d] && b[d] == nt[d] - 1) missing |= 2u << (2 * d);
            const bool whole = (n[d] & ((1 << lt[d]) - 1)) == 0;
            full = full && (whole || (b[d] < nt[d] - 1 && !(g.per[d] && b[d] == 0)));
        }
        for (int e = tid; e <= g.next; e += NT) {
            uint32_t c = (uint32_t)K;
            if (e < g.next) {
                if (!full) c = cell_code(g, bx, by, bz, e, slots);
                else if (!(full_codes[g.next + e] & missing)) c = full_codes[e];
            }
            codes[e] = c;
        }
    }
    __syncthreads();
    uint32_t n_clamped = 0, n_dropped = 0;
    // the code with the slot's part of the round's particle i
    auto part_code = [&](uint32_t c, int i) {
        const uint32_t s = c & SLOT_MASK;
        return c + (s << lq) - s + ((uint32_t)i & (uint32_t)pm);
    };
    // the round's particle i, in part s, among all of its slot: its place in
    // the slot order
    auto rank = [&](uint32_t s, int i) {
        const uint32_t s0 = s & ~(uint32_t)pm, s1 = s | (uint32_t)pm, at = loff[s0];
        return goff[s >> lq] + list_rank(list + at, pm ? loff[s1] - at + cnt[s1] : cnt[s1], (uint32_t)i);
    };
    // The slots' places in the slot order (goff) and parts of the list (loff,
    // even) from the counts; the sum in every thread.
    auto scan_slots = [&](bool whole) {
        const int E = (KQ + NT - 1) / NT, e0 = tid * E;
        uint32_t s = 0, sp = 0;
        for (int e = e0; e < e0 + E; ++e)
            if (e < KQ) { s += cnt[e]; sp += (cnt[e] + 1u) & ~1u; }
        // (both sums in one scan, 16 bits each, unless the counts are the
        // whole tile's, whose list parts are not used)
        uint32_t total;
        uint32_t run = block_prefix<NT>(whole ? s : s | sp << 16, wsum, total);
        for (int e = e0; e < e0 + E; ++e)
            if (e < KQ) {
                const uint32_t c = cnt[e];
                const bool first = (e & pm) == 0;  // of its slot's parts
                if (whole) {
                    if (first) goff[e >> lq] = run;
                    run += c;
                } else {
                    if (one && first) goff[e >> lq] = run & 0xFFFFu;
                    loff[e] = (uint16_t)(run >> 16);
                    run += c | ((c + 1u) & ~1u) << 16;
                }
            }
        total = whole ? total : total & 0xFFFFu;
        if ((whole || one) && tid == 0) goff[K] = total;
        return total;
    };
    // the tile's tables, from the slots' places
    auto write_tables = [&](uint32_t total) {
        __syncthreads();  // goff is written
        for (int e = tid; e < K; e += NT) {
            const uint32_t f = goff[e];
            tab_out[(size_t)T * g.kt + e] = seg + f;
            if (e < NS && goff[e + 1] - f > 0xFFFFu) atomicAdd(counters + C_RANK_OVERFLOW, 1ull);  // slot 0
        }
        if (tid < 28) {
            dtab_out[(size_t)T * DIR_WORDS + tid] = seg + goff[mydir];
        } else if (tid < 30) {
            dtab_out[(size_t)T * DIR_WORDS + tid] = seg + (tid == DIR_OWN ? 0u : goff[NS]);
        } else if (tid == 30) {
            tab_out[(size_t)T * g.kt + K] = seg + total;
        }
        // places of the segment whose particles are removed
        for (uint32_t u = total + tid; u < N; u += NT)
            if (u < places) (D.x + seg)[u] = Real(-1);
    };
    if (one) {
        for (int i = tid; i < (int)N; i += NT) {
            if (i >= (int)n0) other((uint32_t)i - n0, nq, nlc);
            Particle<Real> q = nq;
            const int lc = nlc;
            const uint32_t u = (uint32_t)(i + NT);
            if (u < n0) own(u, nq, nlc);  // the next own one is loaded ahead
            int e;
            uint32_t c = push_particle<Real, PLAIN>(g, pp, org, edge, fl, codes, q, lc, e, n_clamped, n_dropped);
            S4[i] = Real4<Real>{{q.X, q.Y, q.Z, q.vx}};
            S2[i] = Real2<Real>{{q.vy, q.vz}};
            c = part_code(c, i);
            c |= atomicAdd(&cnt[c & SLOT_MASK], 1u) << RANK_SHIFT;
            scode[i] = c;
        }
        __syncthreads();
        const uint32_t total = scan_slots(false);
        write_tables(total);
        for (int i = tid; i < (int)N; i += NT) {
            const uint32_t c = scode[i], s = c & SLOT_MASK;
            if (s < (uint32_t)KQ) list[loff[s] + (c >> RANK_SHIFT & RANK_MASK_ROUND)] = (uint16_t)i;
        }
        __syncthreads();
        for (int i = tid; i < (int)N; i += NT) {
            const uint32_t c = scode[i], s = c & SLOT_MASK;
            uint32_t dst = 0xFFFFu;
            if (s < (uint32_t)KQ) dst = rank(s, i);
            scode[i] = dst | c >> CELL_SHIFT << 16;
        }
        __syncthreads();
        for (int i = tid; i < (int)N; i += NT) {
            const uint32_t dst = scode[i] & 0xFFFFu;
            if (dst != 0xFFFFu) list[dst] = (uint16_t)i;
        }
        __syncthreads();
        for (uint32_t d = tid; d < total; d += NT) {
            const uint32_t i = list[d];
            const Real4<Real> a = S4[i];
            const Real2<Real> b = S2[i];
            const uint32_t cell = scode[i] >> 16;
            if (d < places) {
                (D.x + seg)[d] = a.v[0]; (D.y + seg)[d] = a.v[1]; (D.z + seg)[d] = a.v[2];
                (D.vx + seg)[d] = a.v[3]; (D.vy + seg)[d] = b.v[0]; (D.vz + seg)[d] = b.v[1];
                (D.lc + seg)[d] = (uint8_t)cell;
            } else {
                atomicAdd(counters + C_RANK_OVERFLOW, 1ull);  // slot 0
            }
        }
    } else {
        // Pushed for the counts, and written back where it came from (no other
        // tile reads those places) with its extended cell; a removed one is
        // only marked, whatever its state was.
        for (uint32_t u = tid; u < N; u += NT) {
            if (u >= n0) other(u - n0, nq, nlc);
            Particle<Real> q = nq;
            const int lc = nlc;
            if (u + NT < n0) own(u + NT, nq, nlc);  // the next own one is loaded ahead
            int e;
            const uint32_t c = push_particle<Real, PLAIN>(g, pp, org, edge, fl, codes, q, lc, e, n_clamped, n_dropped);
            atomicAdd(&cnt[part_code(c, (int)u) & SLOT_MASK], 1u);
            const uint32_t p = place(u);
            if ((c & SLOT_MASK) == (uint32_t)K) {
                A.x[p] = Real(-1);
                continue;
            }
            A.lc[p] = put_ext_cell(e, q.X);
            A.x[p] = q.X; A.y[p] = q.Y; A.z[p] = q.Z;
            A.vx[p] = q.vx; A.vy[p] = q.vy; A.vz[p] = q.vz;
        }
        __syncthreads();
        const uint32_t total = scan_slots(true);
        write_tables(total);
        __syncthreads();
        for (int e = tid; e < KT; e += NT) cnt[e] = 0u;
        __syncthreads();
        // each round's particles then wait in LDS for their ranks
        for (uint32_t ub = 0; ub < N; ub += round) {
            const int n = (int)min((uint32_t)round, N - ub);
            for (int i = tid; i < n; i += NT) {
                const uint32_t p = place(ub + i);
                Particle<Real> q;
                q.X = A.x[p]; q.Y = A.y[p]; q.Z = A.z[p];
                q.vx = A.vx[p]; q.vy = A.vy[p]; q.vz = A.vz[p];
                const int e = take_ext_cell(A.lc[p], q.X);
                uint32_t c = part_code(q.X >= Real(0) ? particle_code(codes, e, q) : (uint32_t)K, i);
                c |= atomicAdd(&cnt[c & SLOT_MASK], 1u) << RANK_SHIFT;
                S4[i] = Real4<Real>{{q.X, q.Y, q.Z, q.vx}};
                S2[i] = Real2<Real>{{q.vy, q.vz}};
                scode[i] = c;
            }
            __syncthreads();
            scan_slots(false);
            __syncthreads();
            for (int i = tid; i < n; i += NT) {
                const uint32_t c = scode[i], s = c & SLOT_MASK;
                if (s < (uint32_t)KQ) list[loff[s] + (c >> RANK_SHIFT & RANK_MASK_ROUND)] = (uint16_t)i;
            }
            __syncthreads();
            for (int i = tid; i < n; i += NT) {
                const uint32_t c = scode[i], s = c & SLOT_MASK;
                if (s >= (uint32_t)KQ) continue;
                const uint32_t dst = rank(s, i);
                if (dst < places) {
                    const Real4<Real> a = S4[i];
                    const Real2<Real> b = S2[i];
                    (D.x + seg)[dst] = a.v[0]; (D.y + seg)[dst] = a.v[1]; (D.z + seg)[dst] = a.v[2];
                    (D.vx + seg)[dst] = a.v[3]; (D.vy + seg)[dst] = b.v[0]; (D.vz + seg)[dst] = b.v[1];
                    (D.lc + seg)[dst] = (uint8_t)(c >> CELL_SHIFT);
                } else {
                    atomicAdd(counters + C_RANK_OVERFLOW, 1ull);  // slot 0
                }
            }
            __syncthreads();
            for (int s = tid; s < g.kt; s += NT) {
                uint32_t c = 0;
                for (int e = s << lq; e <= (s << lq | pm); ++e) {
                    c += cnt[e];
                    cnt[e] = 0u;
                }
                if (s < K) goff[s] += c;
            }
            for (int e = tid; e < (round + KT) / 2; e += NT) reinterpret_cast<uint32_t*>(list)[e] = ~0u;
            __syncthreads();
        }
    }
    count_events(counters, C_MAX_VI, n_clamped);
    count_events(counters, C_DROPPED, n_dropped);
}

// axis_candidates for an axis with at least three tiles or without wrap: the
// previous tile (cell on the tile's low face), the own tile, the next tile
// (cell on the high face), in that order.
__device__ __forceinline__ int axis_candidates_fast(int i, int n, int lt, int nt, int per, int* tl, int* el) {
    const int t0 = i >> lt, l = i - (t0 << lt);
    int m = 0;
    if (l == 0 && (t0 > 0 || per)) { tl[m] = t0 > 0 ? t0 - 1 : nt - 1; el[m] = tile_width(n, lt, tl[m]) + 1; ++m; }
    tl[m] = t0; el[m++] = l + 1;
    if (l == tile_width(n, lt, t0) - 1 && (t0 < nt - 1 || per)) { tl[m] = t0 < nt - 1 ? t0 + 1 : 0; el[m++] = 0; }
    return m;
}

// Exclusive scan of uint32 counts (three passes: block sums, scan of the block
// sums, block scan plus offset).  SCAN_ITEMS elements per thread.
constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS = 16;
constexpr int SCAN_TILE = SCAN_THREADS * SCAN_ITEMS;

__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* smem, uint32_t& total) {
    const int t = threadIdx.x;
    smem[t] = v;
    __syncthreads();
    for (int off = 1; off < SCAN_THREADS; off <<= 1) {
        const uint32_t a = (t >= off) ? smem[t - off] : 0u;
        __syncthreads();
        smem[t] += a;
        __syncthreads();
    }
    total = smem[SCAN_THREADS - 1];
    const uint32_t incl = smem[t];
    __syncthreads();
    return incl - v;
}

__global__ __launch_bounds__(SCAN_THREADS) void k_scan_reduce(const uint32_t* __restrict__ in, uint32_t n,
                                                             uint32_t* __restrict__ bsum) {
    __shared__ uint32_t smem[SCAN_THREADS];
    const size_t base = (size_t)blockIdx.x * SCAN_TILE;
    uint32_t s = 0;
    for (int q = 0; q < SCAN_ITEMS; ++q) {  // coalesced: item q of thread t at base + q*threads + t
        const size_t i = base + (size_t)q * SCAN_THREADS + threadIdx.x;
        if (i < n) s += in[i];
    }
    uint32_t tot;
    block_exclusive_scan(s, smem, tot);
    if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

// In-place safe: a block reads its whole tile into LDS (coalesced) before any
// write.  LDS element j sits at j + j/SCAN_ITEMS, so that the per-thread runs
// of SCAN_ITEMS consecutive elements do not share banks.
__device__ __forceinline__ int scan_pad(int j) { return j + j / SCAN_ITEMS; }

__global__ __launch_bounds__(SCAN_THREADS) void k_scan_apply(const uint32_t* __restrict__ in, uint32_t n,
                                                            const uint32_t* __restrict__ boff,
                                                            uint32_t* __restrict__ out) {
    __shared__ uint32_t smem[SCAN_THREADS];
    __shared__ uint32_t tile[SCAN_TILE + SCAN_THREADS];
    const size_t base = (size_t)blockIdx.x * SCAN_TILE;
    for (int q = 0; q < SCAN_ITEMS; ++q) {
        const size_t i = base + (size_t)q * SCAN_THREADS + threadIdx.x;
        tile[scan_pad(q * SCAN_THREADS + threadIdx.x)] = i < n ? in[i] : 0u;
    }
    __syncthreads();
    const int t0 = threadIdx.x * (SCAN_ITEMS + 1);
    uint32_t v[SCAN_ITEMS];
    uint32_t s = 0;
    for (int q = 0; q < SCAN_ITEMS; ++q) {
        v[q] = tile[t0 + q];
        s += v[q];
    }
    uint32_t tot;
    uint32_t run = block_exclusive_scan(s, smem, tot) + boff[blockIdx.x];
    for (int q = 0; q < SCAN_ITEMS; ++q) {
        tile[t0 + q] = run;
        run += v[q];
    }
    __syncthreads();
    for (int q = 0; q < SCAN_ITEMS; ++q) {
        const size_t i = base + (size_t)q * SCAN_THREADS + threadIdx.x;
        if (i < n) out[i] = tile[scan_pad(q * SCAN_THREADS + threadIdx.x)];
    }
    // the grand total goes one past the end
    if (base + SCAN_TILE >= n && threadIdx.x == SCAN_THREADS - 1) out[n] = boff[blockIdx.x] + tot;
}

// Cloud-in-cell deposit (Accumulator::accumulateCell,
// src/particle_accumulator.cpp:43-156).  One workgroup per tile, one thread
// per subcell: a subcell's particles share one 2x2x2 footprint, so the thread
// sums, in particle order, the 8 corner weights times (1, vx, vy, vz).  The
// eight octant threads of a cell then combine their corner sums into the
// cell's 27 targets by lane exchanges, the targets are staged in LDS, and
// every cell of the tile's extended region adds the (up to 27) cell terms
// that reach it in a fixed order (crowded tiles: eight threads per subcell
// and the (up to 64) subcell terms, two quantities at a time).  The result
// is the tile's ghost partial of this species (unscaled); k_fold sums
// partials over tiles and species in FP64.  No atomics, so every run gives
// the same bits.
template <typename Real>
__device__ __forceinline__ void cic_accumulate(Real (&acc)[4][8], bool hx, bool hy, bool hz, Real X, Real Y, Real Z,
                                               Real vx, Real vy, Real vz) {
    // weights of the lower / upper target along each axis
    const Real wx1 = hx ? X - Real(0.5) : X + Real(0.5);
    const Real wy1 = hy ? Y - Real(0.5) : Y + Real(0.5);
    const Real wz1 = hz ? Z - Real(0.5) : Z + Real(0.5);
    const Real live = X >= Real(0) ? Real(1) : Real(0);  // removed particles add nothing
    const Real wx[2] = {live - live * wx1, live * wx1}, wy[2] = {Real(1) - wy1, wy1}, wz[2] = {Real(1) - wz1, wz1};
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const Real w = wx[c & 1] * wy[(c >> 1) & 1] * wz[c >> 2];
        acc[0][c] += w;
        acc[1][c] += w * vx;
        acc[2][c] += w * vy;
        acc[3][c] += w * vz;
    }
}

// Octant block of the deposit's LDS staging: the tile's cells padded by 8
// words, so that the 8 octants x 8 cells a wave writes fall in distinct banks
// (octant stride = 8 banks).
RH_HD int deposit_octant_block(const Geom& g) { return g.tc + 8; }

// Two of the four quantities (the charge and vx, or vy and vz): a and b
// are the particle's factors for them (1 and vx, or vy and vz).
template <typename Real>
__device__ __forceinline__ void cic_accumulate2(Real (&acc)[2][8], bool hx, bool hy, bool hz, Real X, Real Y,
                                                Real Z, Real a, Real b) {
    const Real wx1 = hx ? X - Real(0.5) : X + Real(0.5);
    const Real wy1 = hy ? Y - Real(0.5) : Y + Real(0.5);
    const Real wz1 = hz ? Z - Real(0.5) : Z + Real(0.5);
    const Real live = X >= Real(0) ? Real(1) : Real(0);
    const Real wx[2] = {live - live * wx1, live * wx1}, wy[2] = {Real(1) - wy1, wy1}, wz[2] = {Real(1) - wz1, wz1};
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const Real w = wx[c & 1] * wy[(c >> 1) & 1] * wz[c >> 2];
        acc[0][c] += w * a;
        acc[1][c] += w * b;
    }
}

// LDS of the deposit: half of the subcell sums (2 quantities x 8 corners) as
// [quantity*8+corner][octant][cell] (octant blocks of deposit_octant_block
// words); per extended cell four sums, the arrivals' and, on the crowded
// path, the first half's results.
template <typename Real>
RH_HD size_t deposit_lds_bytes(const Geom& g) {
    return sizeof(Real) * (16 * 8 * (size_t)deposit_octant_block(g) + 4 * (size_t)g.next);
}

// For every cell of the extended region, the LDS offsets (corner plane,
// octant block, cell) of the subcell sums that reach it: cell + half - 1 +
// corner = target along each axis.  The same for every tile of a shape;
// built once on the host, at most 64 entries per cell.
inline int deposit_gather_lists(const Geom& g, uint16_t* list, uint8_t* count) {
    const int OB = deposit_octant_block(g), QS = 8 * OB;
    for (int e = 0; e < g.next; ++e) {
        const int lx = e % g.ex - 1, ly = (e / g.ex) % g.ey - 1, lz = e / (g.ex * g.ey) - 1;
        int m = 0;
        for (int hz = 0; hz < 2; ++hz)
            for (int kz = 0; kz < 2; ++kz) {
                const int cz = lz + 1 - hz - kz;
                if (cz < 0 || cz >= g.tz) continue;
                for (int hy = 0; hy < 2; ++hy)
                    for (int ky = 0; ky < 2; ++ky) {
                        const int cy = ly + 1 - hy - ky;
                        if (cy < 0 || cy >= g.ty) continue;
                        for (int hx = 0; hx < 2; ++hx)
                            for (int kx = 0; kx < 2; ++kx) {
                                const int cx = lx + 1 - hx - kx;
                                if (cx < 0 || cx >= g.tx) continue;
                                const int cell = cx + g.tx * (cy + g.ty * cz);
                                const int corner = kx + 2 * ky + 4 * kz, oct = hx + 2 * hy + 4 * hz;
                                list[e * 64 + m++] = (uint16_t)(corner * QS + oct * OB + cell);
                            }
                    }
            }
        // ascending offsets: a fixed order that also walks LDS forward
        for (int a = 1; a < m; ++a)
            for (int b = a; b > 0 && list[e * 64 + b - 1] > list[e * 64 + b]; --b) {
                const uint16_t t = list[e * 64 + b];
                list[e * 64 + b] = list[e * 64 + b - 1];
                list[e * 64 + b - 1] = t;
            }
        count[e] = (uint8_t)m;
        // padded to a multiple of 8 entries with a word the deposit keeps at
        // zero (corner 0, octant 0, the cell past the tile's: cell padding)
        for (int t = m; t < ((m + 7) & ~7); ++t) list[e * 64 + t] = (uint16_t)g.tc;
    }
    return 0;
}

// The one-lane-per-subcell path first combines, in registers, the corner
// sums of a cell's eight octant lanes into the cell's 27 targets (cell + d,
// d in {-1, 0, 1}^3), then gathers for every cell of the extended region the
// (up to 27) cell terms that reach it.  LDS: [quantity][target][cell], cell
// blocks of deposit_octant_block words.  The lists hold, for every cell of
// the extended region, the offsets (target, cell) of its terms in ascending
// order, at most 27 per cell (stride 32), padded to a multiple of 8 entries
// with the offset of a word the deposit keeps at zero (target 0, the cell
// past the tile's: inside the padding of the cell blocks); built once on the
// host.
inline int deposit_target_lists(const Geom& g, uint16_t* list, uint8_t* count) {
    const int CB = deposit_octant_block(g);
    for (int e = 0; e < g.next; ++e) {
        const int lx = e % g.ex - 1, ly = (e / g.ex) % g.ey - 1, lz = e / (g.ex * g.ey) - 1;
        int m = 0;
        for (int dz = -1; dz <= 1; ++dz) {
            const int cz = lz - dz;
            if (cz < 0 || cz >= g.tz) continue;
            for (int dy = -1; dy <= 1; ++dy) {
                const int cy = ly - dy;
                if (cy < 0 || cy >= g.ty) continue;
                for (int dx = -1; dx <= 1; ++dx) {
                    const int cx = lx - dx;
                    if (cx < 0 || cx >= g.tx) continue;
                    const int t27 = (dx + 1) + 3 * (dy + 1) + 9 * (dz + 1);
                    list[e * 32 + m++] = (uint16_t)(t27 * CB + cx + g.tx * (cy + g.ty * cz));
                }
            }
        }
        for (int a = 1; a < m; ++a)
            for (int b = a; b > 0 && list[e * 32 + b - 1] > list[e * 32 + b]; --b) {
                const uint16_t t = list[e * 32 + b];
                list[e * 32 + b] = list[e * 32 + b - 1];
                list[e * 32 + b - 1] = t;
            }
        count[e] = (uint8_t)m;
        for (int t = m; t < ((m + 7) & ~7); ++t) list[e * 32 + t] = (uint16_t)g.tc;
    }
    return 0;
}

// The value of lane ^ M (M = 1, 2, 4: inside the 8 lanes of one cell's
// octants): DPP quad permutations for 1 and 2, a swizzle in xor mode for 4.
template <int M>
__device__ __forceinline__ int octant_xor_bits(int v) {
    if constexpr (M == 1) return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, false);  // quad_perm [1,0,3,2]
    else if constexpr (M == 2) return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, false);  // quad_perm [2,3,0,1]
    else return __builtin_amdgcn_ds_swizzle(v, (M << 10) | 0x1F);  // and 31, or 0, xor M
}
template <int M>
__device__ __forceinline__ float octant_xor(float v) { return __int_as_float(octant_xor_bits<M>(__float_as_int(v))); }
template <int M>
__device__ __forceinline__ double octant_xor(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = octant_xor_bits<M>((int)(b & 0xFFFFFFFFll)), hi = octant_xor_bits<M>((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// One exchange stage along an axis with octant bit `bit` (lane mask M):
// pairs (c0, c1) of corner 0 and 1 along the axis.  The lane with bit 0 keeps
// target -1 (its corner 0) in c0 and target 0 (its corner 1 plus the
// partner's corner 0) in c1; the lane with bit 1 keeps target +1 (its corner
// 1) in c0.  A fixed order: the same bits in every run.
template <int M, typename Real>
__device__ __forceinline__ void octant_stage(Real& c0, Real& c1, bool bit) {
    const Real p = octant_xor<M>(c0);
    const Real a0 = c0, a1 = c1;
    c0 = bit ? a1 : a0;
    c1 = bit ? Real(0) : a1 + p;
}

// Particles per chunk when the one-lane-per-subcell path stages the tile's
// particles (6 arrays) through LDS: as many as fit in the subcell-sum
// staging, which the chunks alias (it is written only after the last one).
template <typename Real>
RH_HD int deposit_chunk(const Geom& g) {
    return ((16 * 8 * deposit_octant_block(g)) / 6) & ~63;
}

// The deposit of a crowded tile (k_deposit sends tiles with at least
// dense_min particles here, whether its own or arrivals; tab null: none of
// its own): eight lanes share a subcell and read eight
// consecutive particles per array (one cache line per group instead of one
// per lane), then add their sums in a fixed butterfly order; blockDim/8
// subcells per round.  Within the same LDS as the sparse path, the two
// halves (charge and vx, then vy and vz) each read the particles once.
template <typename Real>
__device__ void deposit_dense_tile(const Geom& g, const PArrays<Real>& A, const uint32_t* __restrict__ tab,
                                   const uint16_t* __restrict__ glist, const uint8_t* __restrict__ gcount,
                                   Real* __restrict__ partial, int T, Real* S, Real4<Real>* R) {
    const int NS = g.tc * 8;
    const int OB = deposit_octant_block(g);
    const int QS = 8 * OB;
    const int tid = threadIdx.x, grp = tid >> 3, gl = tid & 7, ngrp = (int)blockDim.x >> 3;
    Real4<Real>* out = reinterpret_cast<Real4<Real>*>(partial) + (size_t)T * g.next;
    for (int half = 0; half < 2; ++half) {
        if (half) __syncthreads();  // the first half's reads are done
        for (int base = 0; base < NS; base += ngrp) {
            const int ls = base + grp;
            const bool valid = ls < NS, some = valid && tab;
            const uint32_t p0 = some ? tab[ls] : 0u, p1 = some ? tab[ls + 1] : 0u;
            const int o = ls & 7, cell = ls >> 3;
            const bool hx = o & 1, hy = (o >> 1) & 1, hz = (o >> 2) & 1;
            Real acc[2][8];
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int c = 0; c < 8; ++c) acc[q][c] = Real(0);
            for (uint32_t p = p0 + gl; p < p1; p += 8) {
                const Real a = half ? A.vy[p] : Real(1), b = half ? A.vz[p] : A.vx[p];
                cic_accumulate2(acc, hx, hy, hz, A.x[p], A.y[p], A.z[p], a, b);
            }
#pragma unroll
            for (int off = 1; off < 8; off <<= 1)
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int c = 0; c < 8; ++c) acc[q][c] += __shfl_xor(acc[q][c], off);
            if (valid && gl == 0)
#pragma unroll
                for (int q = 0; q < 2; ++q)
#pragma unroll
                    for (int c = 0; c < 8; ++c) S[(q * 8 + c) * QS + o * OB + cell] = acc[q][c];
        }
        if (tid < 2) S[tid * 8 * QS + g.tc] = Real(0);  // the lists' padding entries read these words
        __syncthreads();
        for (int e = tid; e < g.next; e += blockDim.x) {
            // eight entries at a time (the padding adds zeros after the terms)
            const int ng = (gcount[e] + 7) >> 3;
            const uint4* lst = reinterpret_cast<const uint4*>(glist + (size_t)e * 64);
            Real res[2] = {Real(0), Real(0)};
            for (int gi = 0; gi < ng; ++gi) {
                const uint4 l8 = lst[gi];
                const uint32_t w[4] = {l8.x, l8.y, l8.z, l8.w};
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    const int off = (int)((w[t >> 1] >> (16 * (t & 1))) & 0xFFFFu);
                    res[0] += S[off];
                    res[1] += S[8 * QS + off];
                }
            }
            R[e].v[2 * half] += res[0];
            R[e].v[2 * half + 1] += res[1];
            if (half) out[e] = R[e];
        }
    }
}

// The arrivals of a crowded tile, which wait in its neighbours' segments: every wave
// takes a contiguous part of the sequence and adds each particle's weights
// times (1, vx, vy, vz) to sums of its own over the extended region (in LDS,
// where the particle staging comes later): lane = corner + 8 * quantity, so
// the 32 targets of one particle are distinct words and need no atomics.  The
// waves' sums are then added in order into R.
template <typename Real>
__device__ void deposit_arrivals(const Geom& g, const PArrays<Real>& A, const uint32_t* lists,
                                 Real* S, Real4<Real>* R) {
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const uint32_t na = lists[LIST_PREF + 27];
    const int nwaves = ((int)blockDim.x + 63) >> 6;
    const int room = 16 * 8 * deposit_octant_block(g) / (4 * g.next);  // copies of the region that fit
    const int nw = nwaves < room ? nwaves : room;
    for (int e = tid; e < nw * 4 * g.next; e += blockDim.x) S[e] = Real(0);
    __syncthreads();
    const int nl = blockDim.x < 64 ? (int)blockDim.x : 64;  // lanes of this wave (8 to 64)
    if (w < nw) {
        Real* mine = S + (size_t)w * 4 * g.next;
        const uint32_t v0 = (uint32_t)((uint64_t)na * w / nw), v1 = (uint32_t)((uint64_t)na * (w + 1) / nw);
        for (uint32_t vb = v0; vb < v1; vb += nl) {
            Real X = Real(-1), Y = Real(0), Z = Real(0), vx = Real(0), vy = Real(0), vz = Real(0);
            int lc = 0;
            if (vb + lane < v1) {
                const uint32_t p = arrival_index(lists, vb + lane);
                X = A.x[p]; Y = A.y[p]; Z = A.z[p];
                vx = A.vx[p]; vy = A.vy[p]; vz = A.vz[p];
                lc = A.lc[p];
            }
            const int n = (int)min((uint32_t)nl, v1 - vb);
            for (int i = 0; i < n; ++i) {
                const Real x = __shfl(X, i), y = __shfl(Y, i), z = __shfl(Z, i);
                const Real f[4] = {Real(1), __shfl(vx, i), __shfl(vy, i), __shfl(vz, i)};
                const int l = __shfl(lc, i);
                if (x < Real(0)) continue;  // removed (the same for the whole wave)
                int li, lj, lk;
                local_ijk(g, l, li, lj, lk);
                const int hx = x >= Real(0.5), hy = y >= Real(0.5), hz = z >= Real(0.5);
                const Real wx1 = hx ? x - Real(0.5) : x + Real(0.5);
                const Real wy1 = hy ? y - Real(0.5) : y + Real(0.5);
                const Real wz1 = hz ? z - Real(0.5) : z + Real(0.5);
                for (int t = lane; t < 32; t += nl) {
                    const int kx = t & 1, ky = (t >> 1) & 1, kz = (t >> 2) & 1, qt = t >> 3;
                    const Real wt = (kx ? wx1 : Real(1) - wx1) * (ky ? wy1 : Real(1) - wy1) * (kz ? wz1 : Real(1) - wz1);
                    const int e = (li + kx + hx) + g.ex * ((lj + ky + hy) + g.ey * (lk + kz + hz));
                    mine[4 * e + qt] += wt * (qt == 0 ? f[0] : (qt == 1 ? f[1] : (qt == 2 ? f[2] : f[3])));
                }
            }
        }
    }
    __syncthreads();
    Real* Rw = reinterpret_cast<Real*>(R);
    for (int e = tid; e < 4 * g.next; e += blockDim.x) {
        Real s = Real(0);
        for (int q = 0; q < nw; ++q) s += S[(size_t)q * 4 * g.next + e];
        Rw[e] = s;
    }
    __syncthreads();
}

template <typename Real>
__global__ __launch_bounds__(512, sizeof(Real) == 8 ? 4 : 8) void k_deposit(Geom g, PArrays<Real> A, const uint32_t* __restrict__ tabs,
                                                 const uint32_t* __restrict__ lists,
                                                 const uint16_t* __restrict__ glist,
                                                 const uint8_t* __restrict__ gcount,
                                                 const uint16_t* __restrict__ tlist,
                                                 const uint8_t* __restrict__ tcount, Real* __restrict__ partial,
                                                 uint32_t dense_min) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ uint32_t L[LIST_WORDS];
    const int NS = g.tc * 8;
    const int OB = deposit_octant_block(g);  // octant block (padded)
    const int QS = 8 * OB;            // one (quantity, corner) plane
    Real* S = reinterpret_cast<Real*>(smem_raw);
    // per extended cell four words: the crowded path's arrivals' sums, or
    // this path's arrivals by subcell (below)
    Real4<Real>* R = reinterpret_cast<Real4<Real>*>(S + 16 * QS);
    const int T = xcd_tile(g, (int)blockIdx.x);
    if (T >= g.ntiles) return;
    const uint32_t* tab = tabs + (size_t)T * g.kt;
    const int ls = threadIdx.x;
    const uint32_t t0 = lists[(size_t)T * LIST_WORDS + LIST_OWN], n0 = lists[(size_t)T * LIST_WORDS + LIST_OWN + 1];
    const uint32_t na = lists[(size_t)T * LIST_WORDS + LIST_PREF + 27], t1 = t0 + n0;
    if (n0 == 0 && na == 0) {
        // an empty tile: zero ghost partials (the fold reads every tile's;
        // a per-tile flag that let the fold skip them cost it more, 35 -> 45
        // us on the dense box, than the zero stores cost here)
        Real4<Real>* out = reinterpret_cast<Real4<Real>*>(partial) + (size_t)T * g.next;
        Real4<Real> z;
        z.v[0] = z.v[1] = z.v[2] = z.v[3] = Real(0);
        for (int e = threadIdx.x; e < g.next; e += blockDim.x) out[e] = z;
        return;
    }
    uint32_t p0 = 0, p1 = 0;
    if (n0) { p0 = tab[ls]; p1 = tab[ls + 1]; }
    for (int e = ls; e < LIST_WORDS; e += blockDim.x) L[e] = lists[(size_t)T * LIST_WORDS + e];
    if (n0 + na >= dense_min) {
        if (na) {
            __syncthreads();
            deposit_arrivals(g, A, L, S, R);
        } else {
            Real* Rw = reinterpret_cast<Real*>(R);
            for (int e = ls; e < 4 * g.next; e += blockDim.x) Rw[e] = Real(0);
        }
        deposit_dense_tile(g, A, n0 ? tab : nullptr, glist, gcount, partial, T, S, R);
        return;
    }
    const int o = ls & 7, cell = ls >> 3;
    const bool hx = o & 1, hy = (o >> 1) & 1, hz = (o >> 2) & 1;
    Real acc[4][8];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int c = 0; c < 8; ++c) acc[q][c] = Real(0);
    // The tile's particles, its own and then its arrivals, go through LDS in
    // chunks (its own read with coalesced loads); each thread then takes its
    // subcell's particles of the chunk, in particle order.  A particle is
    // staged as (x, y, z, vx) and (vy, vz): two LDS reads instead of six.
    // The arrivals, about 3 % of the particles, are linked by subcell as they
    // are staged, in any order; then each walks its subcell's list once for
    // the one that follows it, and a thread takes those of its list in
    // ascending order after its own (a thread that walks its list again for
    // every four it takes needs 21 ms for 2,000 arrivals of one subcell instead
    // of 0.48, and 313 us on the box below).  The loops over the tile's own
    // particles hold nothing of the arrivals in registers (64 of them let four
    // workgroups share a CU): 128x96x96 with 35.5 M particles takes 309 us a
    // launch (2.9 TB/s; 280 where every particle lies in its own tile's
    // segment), and took 370 with both kinds in one loop, 332 with the list
    // read before the own ones, 392 with three own particles' loads in flight.
    const int CH = deposit_chunk<Real>(g);
    Real4<Real>* L4 = reinterpret_cast<Real4<Real>*>(S);          // x, y, z, vx
    Real2<Real>* L2 = reinterpret_cast<Real2<Real>*>(S + 4 * CH);  // vy, vz
    constexpr uint32_t NONE = 0xFFFFu;
    // per subcell its list's first entry as linked, and above it in order
    uint32_t* head = reinterpret_cast<uint32_t*>(R);
    uint16_t* lowest = reinterpret_cast<uint16_t*>(R) + 1;
    uint16_t* next = reinterpret_cast<uint16_t*>(head + NS);  // per arrival of the chunk the next one as linked
    // arrivals of one chunk: one a thread at most
    const uint32_t AR = min((uint32_t)((4 * sizeof(Real) * g.next - 4 * (size_t)NS) / 4), (uint32_t)NS);
    uint16_t* follow = next + AR;                             // and the next one in order
    constexpr uint32_t EMPTY = NONE | NONE << 16;
    head[ls] = EMPTY;
    uint32_t n = 0;
    for (uint32_t cs = 0; cs < n0 + na; cs += n) {
        const uint32_t qa = n0 > cs ? n0 - cs : 0u;  // the chunk's first arrival
        n = min(min((uint32_t)CH, n0 + na - cs), qa + AR);
        __syncthreads();  // the previous chunk is consumed
        const uint32_t no = min(n, qa);              // the chunk's own particles
        for (uint32_t q = ls; q < no; q += blockDim.x) {
            const uint32_t p = t0 + cs + q;
            Real4<Real> r;
            r.v[0] = A.x[p]; r.v[1] = A.y[p]; r.v[2] = A.z[p]; r.v[3] = A.vx[p];
            Real2<Real> t;
            t.v[0] = A.vy[p]; t.v[1] = A.vz[p];
            L4[q] = r;
            L2[q] = t;
        }
        const uint32_t mine = no + ls;               // the thread's arrival
        uint32_t to = 0, old = NONE;                 // its subcell, and what it was linked before
        if (mine < n) {
            const uint32_t p = arrival_index(L, cs + mine - n0);
            Real4<Real> r;
            r.v[0] = A.x[p]; r.v[1] = A.y[p]; r.v[2] = A.z[p]; r.v[3] = A.vx[p];
            Real2<Real> t;
            t.v[0] = A.vy[p]; t.v[1] = A.vz[p];
            L4[mine] = r;
            L2[mine] = t;
            const int oct = (r.v[0] >= Real(0.5)) + 2 * (r.v[1] >= Real(0.5)) + 4 * (r.v[2] >= Real(0.5));
            to = A.lc[p] * 8u + (uint32_t)oct;
            old = atomicExch(&head[to], mine | NONE << 16) & 0xFFFFu;
            next[mine - qa] = (uint16_t)old;
        }
        __syncthreads();
        if (n > no) {
            if (mine < n) {
                uint32_t above = NONE;
                bool first = true;
                for (uint32_t h = head[to] & 0xFFFFu; h != NONE; h = h == mine ? old : next[h - qa]) {
                    if (h > mine) above = min(above, h);
                    first = first && h >= mine;
                }
                follow[mine - qa] = (uint16_t)above;
                if (first) lowest[2 * to] = (uint16_t)mine;
            }
            __syncthreads();
        }
        const uint32_t a = max(p0, t0 + cs) - t0 - cs, b = min(p1, t0 + cs + n) - t0 - cs;
        const int own = p1 > t0 + cs && p0 < t0 + cs + n && p1 > p0 ? (int)(b - a) : 0;
        for (int it = 0; it < own; ++it) {
            const Real4<Real> r = L4[a + it];
            const Real2<Real> t = L2[a + it];
            cic_accumulate(acc, hx, hy, hz, r.v[0], r.v[1], r.v[2], r.v[3], t.v[0], t.v[1]);
        }
        if (n == no) continue;
        for (uint32_t h = head[ls] >> 16; h != NONE; h = follow[h - qa]) {
            const Real4<Real> r = L4[h];
            const Real2<Real> t = L2[h];
            cic_accumulate(acc, hx, hy, hz, r.v[0], r.v[1], r.v[2], r.v[3], t.v[0], t.v[1]);
        }
        head[ls] = EMPTY;
    }
    // the eight octant lanes of each cell: 64 corner sums -> 27 targets
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (int r = 0; r < 4; ++r) octant_stage<1>(acc[q][2 * r], acc[q][2 * r + 1], hx);
#pragma unroll
        for (int r = 0; r < 4; ++r) octant_stage<2>(acc[q][(r & 1) + 4 * (r >> 1)], acc[q][(r & 1) + 4 * (r >> 1) + 2], hy);
#pragma unroll
        for (int r = 0; r < 4; ++r) octant_stage<4>(acc[q][r], acc[q][r + 4], hz);
    }
    __syncthreads();  // the staging is read; the target planes may be written
    const int CB = OB, QP = 27 * CB;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const int sx = c & 1, sy = (c >> 1) & 1, sz = c >> 2;
        if ((hx && sx) || (hy && sy) || (hz && sz)) continue;  // slot unused by this octant
        const int dx = hx ? 1 : sx - 1, dy = hy ? 1 : sy - 1, dz = hz ? 1 : sz - 1;
        const int t27 = (dx + 1) + 3 * (dy + 1) + 9 * (dz + 1);
#pragma unroll
        for (int q = 0; q < 4; ++q) S[q * QP + t27 * CB + cell] = acc[q][c];
    }
    if (ls < 4) S[ls * QP + g.tc] = Real(0);  // the lists' padding entries read this word
    __syncthreads();
    Real4<Real>* out = reinterpret_cast<Real4<Real>*>(partial) + (size_t)T * g.next;
    for (int e = ls; e < g.next; e += blockDim.x) {
        // the cell terms reaching this cell: a list shared by all tiles, read
        // eight entries at a time (the padding adds zeros after the terms)
        const int ng = (tcount[e] + 7) >> 3;
        const uint4* lst = reinterpret_cast<const uint4*>(tlist + (size_t)e * 32);
        Real4<Real> r;
        r.v[0] = r.v[1] = r.v[2] = r.v[3] = Real(0);
        for (int gi = 0; gi < ng; ++gi) {
            const uint4 l8 = lst[gi];
            const uint32_t w[4] = {l8.x, l8.y, l8.z, l8.w};
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const int off = (int)((w[t >> 1] >> (16 * (t & 1))) & 0xFFFFu);
                r.v[0] += S[off];
                r.v[1] += S[QP + off];
                r.v[2] += S[2 * QP + off];
                r.v[3] += S[3 * QP + off];
            }
        }
        out[e] = r;
    }
}

// Accumulator::addRemoteUpdates (src/particle_accumulator.cpp:260-335): each
// cell sums in FP64, species by species and in a fixed tile order, the ghost
// partials of every tile whose extended region holds it, times the species'
// w*q; then rho/=dV with the rho floor, J/=dV.
constexpr int MAX_FOLD_SPECIES = 8;
template <typename Real>
struct FoldSources {
    const Real* partial[MAX_FOLD_SPECIES];
    double wq[MAX_FOLD_SPECIES];
    int n;
};

// TWO: no cell has more than two candidate tiles along an axis.
template <typename Real, bool TWO>
__global__ __launch_bounds__(256) void k_fold(Geom g, FoldSources<Real> src, double inv_dV, double min_rho,
                                             Real* __restrict__ rho, Real* __restrict__ jx, Real* __restrict__ jy,
                                             Real* __restrict__ jz, unsigned long long* __restrict__ counters) {
    const int i = blockIdx.x * 32 + threadIdx.x, j = blockIdx.y * 8 + threadIdx.y, k = blockIdx.z;
    bool floored = false;
    if (i < g.nx && j < g.ny) {
        const int n = cell_index(g, i, j, k);
        int tx[6], ex[6], ty[6], ey[6], tz[6], ez[6];
        double s0 = 0, s1 = 0, s2 = 0, s3 = 0;
        if constexpr (TWO) {
            // at most two candidate tiles per axis: all eight loads of a
            // species issued before its sum (the same order as below)
            const int mx = axis_candidates_fast(i, g.nx, g.ltx, g.ntx, g.per[0], tx, ex);
            const int my = axis_candidates_fast(j, g.ny, g.lty, g.nty, g.per[1], ty, ey);
            const int mz = axis_candidates_fast(k, g.nz, g.ltz, g.ntz, g.per[2], tz, ez);
            for (int s = 0; s < src.n; ++s) {
                const Real4<Real>* part = reinterpret_cast<const Real4<Real>*>(src.partial[s]);
                Real4<Real> v[8];
#pragma unroll
                for (int c = 0; c < 2; ++c)
#pragma unroll
                    for (int b = 0; b < 2; ++b)
#pragma unroll
                        for (int a = 0; a < 2; ++a) {
                            const int q = a + 2 * b + 4 * c;
                            if (a < mx && b < my && c < mz) {
                                const int TT = tx[a] + g.ntx * (ty[b] + g.nty * tz[c]);
                                const int e = ex[a] + g.ex * (ey[b] + g.ey * ez[c]);
                                v[q] = part[(size_t)TT * g.next + e];
                            }
                        }
                double t0 = 0, t1 = 0, t2 = 0, t3 = 0;
#pragma unroll
                for (int c = 0; c < 2; ++c)
#pragma unroll
                    for (int b = 0; b < 2; ++b)
#pragma unroll
                        for (int a = 0; a < 2; ++a) {
                            const int q = a + 2 * b + 4 * c;
                            if (!(a < mx && b < my && c < mz)) continue;
                            t0 += (double)v[q].v[0]; t1 += (double)v[q].v[1];
                            t2 += (double)v[q].v[2]; t3 += (double)v[q].v[3];
                        }
                s0 += src.wq[s] * t0; s1 += src.wq[s] * t1; s2 += src.wq[s] * t2; s3 += src.wq[s] * t3;
            }
        } else {
            const int mx = axis_candidates(i, g.nx, g.ltx, g.ntx, g.per[0], tx, ex);
            const int my = axis_candidates(j, g.ny, g.lty, g.nty, g.per[1], ty, ey);
            const int mz = axis_candidates(k, g.nz, g.ltz, g.ntz, g.per[2], tz, ez);
            for (int s = 0; s < src.n; ++s) {
                double t0 = 0, t1 = 0, t2 = 0, t3 = 0;
                for (int c = 0; c < mz; ++c)
                    for (int b = 0; b < my; ++b)
                        for (int a = 0; a < mx; ++a) {
                            const int TT = tx[a] + g.ntx * (ty[b] + g.nty * tz[c]);
                            const int e = ex[a] + g.ex * (ey[b] + g.ey * ez[c]);
                            const Real4<Real> v = reinterpret_cast<const Real4<Real>*>(src.partial[s])[(size_t)TT * g.next + e];
                            t0 += (double)v.v[0]; t1 += (double)v.v[1]; t2 += (double)v.v[2]; t3 += (double)v.v[3];
                        }
                s0 += src.wq[s] * t0; s1 += src.wq[s] * t1; s2 += src.wq[s] * t2; s3 += src.wq[s] * t3;
            }
        }
        double r = s0 * inv_dV;
        if (r < min_rho) { r = min_rho; floored = true; }
        rho[n] = (Real)r;
        jx[n] = (Real)(s1 * inv_dV);
        jy[n] = (Real)(s2 * inv_dV);
        jz[n] = (Real)(s3 * inv_dV);
    }
    count_event(counters, C_MIN_CELL_RHO, floored);
}

// WRITE_GRID_TEMPORAL_AVERAGES of the accumulator (src/particle_accumulator.
// cpp:148-151, 287-300): one species' charge and current sums of this step
// (its tile partials folded in k_fold's fixed order, times w q, before /dV
// and the floor) added to its running FP64 sums nave[n], vave[l*nc + n].
template <typename Real>
__global__ __launch_bounds__(256) void k_average_moments(Geom g, const Real* __restrict__ partial, double wq,
                                                        double* __restrict__ nave, double* __restrict__ vave) {
    const int i = blockIdx.x * 32 + threadIdx.x, j = blockIdx.y * 8 + threadIdx.y, k = blockIdx.z;
    if (i >= g.nx || j >= g.ny) return;
    const int n = cell_index(g, i, j, k);
    int tx[6], ex[6], ty[6], ey[6], tz[6], ez[6];
    const int mx = axis_candidates(i, g.nx, g.ltx, g.ntx, g.per[0], tx, ex);
    const int my = axis_candidates(j, g.ny, g.lty, g.nty, g.per[1], ty, ey);
    const int mz = axis_candidates(k, g.nz, g.ltz, g.ntz, g.per[2], tz, ez);
    double t0 = 0, t1 = 0, t2 = 0, t3 = 0;
    for (int c = 0; c < mz; ++c)
        for (int b = 0; b < my; ++b)
            for (int a = 0; a < mx; ++a) {
                const int TT = tx[a] + g.ntx * (ty[b] + g.nty * tz[c]);
                const int e = ex[a] + g.ex * (ey[b] + g.ey * ez[c]);
                const Real4<Real> v = reinterpret_cast<const Real4<Real>*>(partial)[(size_t)TT * g.next + e];
                t0 += (double)v.v[0]; t1 += (double)v.v[1]; t2 += (double)v.v[2]; t3 += (double)v.v[3];
            }
    nave[n] += wq * t0;
    vave[n] += wq * t1;
    vave[(size_t)g.nc + n] += wq * t2;
    vave[2 * (size_t)g.nc + n] += wq * t3;
}

// cellAverageB += cellB (src/hybrid_propagator.cpp:157-167), FP64 sums
template <typename Real>
__global__ __launch_bounds__(256) void k_average_cellB(int nc, const Real* __restrict__ b, double* __restrict__ ave) {
    const size_t q = blockIdx.x * (size_t)256 + threadIdx.x;
    if (q < 3 * (size_t)nc) ave[q] += (double)b[q];
}

// ParticleBoundaryCondHybrid::apply (src/particle_boundary_cond_hybrid.h:
// 112-185): empty exterior cells, remove particles inside the obstacle in
// innerFlagParticle cells.  Removed particles get x = -1; the next sort drops
// them.  16 lanes per listed cell (four cells a wave), striding through the
// cell's particles.
constexpr int BC_LANES = 16;
constexpr int BC_CELLS_PER_BLOCK = 256 / BC_LANES;
// The removed particles are counted for the logs (logCounterParticleEscape
// / Impact and their kinetic energies, :121-122,153-154): per listed cell,
// acc[4q..4q+3] += (escapes, sum v^2 of escapes, impacts, sum v^2 of
// impacts), summed over the cell's lanes in a fixed butterfly.
// rng[beg[q] .. beg[q+1]-1]: where the cell's particles may be, its own
// subcells' range first, then the halo slots of neighbouring tiles that it
// is: the tile and the table entry, which are the same in every step.
struct CellRange {
    int tile;
    uint32_t entry;
};
template <typename Real>
__global__ __launch_bounds__(256) void k_boundary(Geom g, const int* __restrict__ cells, int ncells,
                                                 const int* __restrict__ beg, const CellRange* __restrict__ rng,
                                                 TileTables tt, PArrays<Real> A,
                                                 double R2, double* __restrict__ acc) {
    const int q = blockIdx.x * BC_CELLS_PER_BLOCK + (int)(threadIdx.x / BC_LANES);
    const int lane = threadIdx.x & (BC_LANES - 1);
    const bool valid = q < ncells;
    double c[4] = {0, 0, 0, 0};
    if (valid) {
        const int b0 = beg[q], nr = tt.lists ? beg[q + 1] - b0 : 1;
        // up to 16 ranges at a time, one lane each
        uint32_t r0 = 0, r1 = 0;
        if (lane < nr) {
            const CellRange cr = rng[b0 + lane];
            if (tt.live[cr.tile]) { r0 = tt.tab[cr.entry]; r1 = tt.tab[cr.entry + (lane == 0 ? 8 : 1)]; }
        }
        const int n = cells[q];
        int i, j, k;
        cell_ijk(g, n, i, j, k);
        const bool exterior = !all_nbrs(g, i, j, k);
        const double xb = g.x0 + i * g.dx, yb = g.y0 + j * g.dx, zb = g.z0 + k * g.dx;
        for (int t = 0; t < nr; ++t) {
            if (t > 0 && (t & (BC_LANES - 1)) == 0) {  // (only cells of tiles one cell wide have more)
                r0 = r1 = 0;
                if (t + lane < nr) {
                    const CellRange cr = rng[b0 + t + lane];
                    if (tt.live[cr.tile]) { r0 = tt.tab[cr.entry]; r1 = tt.tab[cr.entry + 1]; }
                }
            }
            const uint32_t p0 = __shfl(r0, t & (BC_LANES - 1), BC_LANES), p1 = __shfl(r1, t & (BC_LANES - 1), BC_LANES);
            for (uint32_t p = p0 + lane; p < p1; p += BC_LANES) {
                if (A.x[p] < Real(0)) continue;
                const double vx = A.vx[p], vy = A.vy[p], vz = A.vz[p];
                const double v2 = vx * vx + vy * vy + vz * vz;
                if (exterior) {
                    A.x[p] = Real(-1);
                    c[0] += 1.0; c[1] += v2;
                    continue;
                }
                const double x = xb + (double)A.x[p] * g.dx, y = yb + (double)A.y[p] * g.dx, z = zb + (double)A.z[p] * g.dx;
                if (x * x + y * y + z * z < R2) {
                    A.x[p] = Real(-1);
                    c[2] += 1.0; c[3] += v2;
                }
            }
        }
    }
    // most listed cells remove nothing in a step: then the wave is done
    if (!__ballot(c[0] != 0.0 || c[2] != 0.0)) return;
    for (int t = 0; t < 4; ++t)
        for (int off = BC_LANES / 2; off > 0; off >>= 1) c[t] += __shfl_xor(c[t], off, 64);
    if (valid && lane == 0)
        for (int t = 0; t < 4; ++t) acc[(size_t)q * 4 + t] += c[t];
}

// FP64 particle sums (logCalcParticle, src/diagnostics.h:209-228), one
// partial per block, summed on the host in block order: count, sum vx, vy,
// vz, sum |v|, sum v^2 (unweighted; one weight per species) and max |v|.
constexpr int DIAG_BLOCKS = 1024;
constexpr int DIAG_Q = 7;
// Every place of the segments (*end of them; those without a particle are
// marked), and the injected particles waiting in the appendix (*extra of
// them, extra may be null, up to the store's capacity) from store index
// `base`, or from the store's end.
template <typename Real>
__global__ __launch_bounds__(256) void k_diag(PArrays<Real> A, const uint32_t* __restrict__ scal,
                                             const uint32_t* __restrict__ extra, uint32_t places, int at_end,
                                             uint32_t cap, double* __restrict__ partial) {
    __shared__ double red[DIAG_Q][256];
    const uint32_t np = scal[SC_NP], end = scal[SC_END], room = min(cap > np ? cap - np : 0u, places);
    const uint32_t nx = extra ? min(*extra, room) : 0u, base = at_end ? np : cap;
    double s[DIAG_Q] = {0, 0, 0, 0, 0, 0, 0};
    for (uint32_t u = blockIdx.x * 256u + threadIdx.x; u < end + nx; u += 256u * gridDim.x) {
        const uint32_t p = u < end ? u : base + (u - end);
        if (A.x[p] < Real(0)) continue;
        const double vx = A.vx[p], vy = A.vy[p], vz = A.vz[p];
        const double v2 = vx * vx + vy * vy + vz * vz, v = sqrt(v2);
        s[0] += 1.0; s[1] += vx; s[2] += vy; s[3] += vz; s[4] += v; s[5] += v2;
        s[6] = fmax(s[6], v);
    }
    for (int q = 0; q < DIAG_Q; ++q) red[q][threadIdx.x] = s[q];
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) {
            for (int q = 0; q < DIAG_Q - 1; ++q) red[q][threadIdx.x] += red[q][threadIdx.x + off];
            red[DIAG_Q - 1][threadIdx.x] = fmax(red[DIAG_Q - 1][threadIdx.x], red[DIAG_Q - 1][threadIdx.x + off]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int q = 0; q < DIAG_Q; ++q) partial[blockIdx.x * DIAG_Q + q] = red[q][0];
}

template <typename T>
__global__ void k_fill(T* __restrict__ p, T v, size_t n) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)blockDim.x * gridDim.x) p[i] = v;
}

}  // namespace rh
