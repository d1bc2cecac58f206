// kernels.hip -- gfx950 kernels of one DEM time step.
//
// Two ways through a step, with the same device functions and the same bits:
// k_chain (below), a chain of like launches of which a step takes as many as
// it has work for, is what steps run unless the caller chose their kernels or
// timing found the other way to be faster, which runs one kernel per stage,
// recorded as a HIP graph:
//   head       the previous step's inverse permutation and per-wall tree sums
//              of the per-particle wall forces in the reference's block order
//              (src/integration.cuh:191-221); per-cell totals.  (The previous
//              step's force kernel computed the cell ids and updated the
//              per-cell counts, src/sorting.cuh:7-43.)
//   scan       exclusive scan of the per-cell counts -> cell offsets
//   scatter    counting-sort placement of the particles
//   order      one thread per cell: order each cell's members by original
//              index, which makes the counting sort the stable sort of
//              src/device.cu:763-765; then the sorted ids, keys and FP32
//              positions (src/sorting.cuh:49-121 gathers x, vel, angvel)
//   bonds      one thread per bond: parallel-bond force, torque, breakage
//              (src/cohesion.cuh:8-233); forces go to per-bond records, no
//              scatter
//   search     27-cell search and slot update (src/contactsearch.cuh:181-355),
//              beside it the previous step's wall leapfrog
//              (src/integration.cuh:224-295)
//   force      one thread per sorted particle: contact and wall forces
//              (src/contactsearch.cuh:369-689, src/contactmodels.cuh:10-109,
//              283-493), bond forces gathered in ascending bond index,
//              leapfrog (src/integration.cuh:9-187), next cell ids
// After the last step of a call: tail (what head does for the others) and
// walls.  Steps in which no sphere changed its cell keep the previous sort:
// head, scan, scatter and order return at once.  A launch costs about 4 us of
// a step here whatever its size, and a fork to a second stream and back about
// 9: with twelve launches and that fork a step of 1,000 to 4,000 spheres took
// 80 us, with seven in a row and the skipped sort 47, as a chain 12 to 20; of
// the 1,048,576-sphere crystal 545, 475 and 428.
//
// Arithmetic keeps the reference's expression order and is built with
// -ffp-contract=off, so the FP64 path reproduces the CPU oracle bit for bit.
// Vector lengths use IEEE double sqrt (the reference narrows to float).

#include <hip/hip_runtime.h>

#include <algorithm>

#include "dem_internal.h"
#include "quad.h"
#include "vec3.h"

namespace sph {

namespace {

constexpr double PI_REF = 3.14159265358979;   // src/constants.h:14
constexpr double PI_WALL = 3.141596654;       // src/integration.cuh:258


// Workgroups are dispatched round-robin over the 8 XCDs; remap so each XCD
// walks one contiguous range of sorted particles and its L2 holds that
// range's neighbourhood.
__device__ __forceinline__ uint32_t xcd_block(uint32_t nb) {  // the first nb workgroups
    const uint32_t b = blockIdx.x;
    const uint32_t q = nb >> 3, r = nb & 7u, xcd = b & 7u, k = b >> 3;
    return xcd * q + (xcd < r ? xcd : r) + k;
}
__device__ __forceinline__ uint32_t xcd_block() { return xcd_block(gridDim.x); }
// Item of this thread among the n that a chain's launch, whose grid serves
// every phase, shares out; n or more: none.
__device__ __forceinline__ uint32_t xcd_item(uint32_t n) {
    const uint32_t nb = (n + BLOCK - 1) / BLOCK;
    return blockIdx.x < nb ? xcd_block(nb) * BLOCK + threadIdx.x : n;
}

// The system of index / sorted position i: the handle's only one, or its
// entry of the ensemble table.
template <bool B>
__device__ __forceinline__ const Sys& sys_at(const DemDev& d, uint32_t i) {
    if constexpr (B) return d.systems[d.sys_of[i]];
    else return d.sys;
}

// ------------------------------------------------------------ cell hashing
// Periodic wrap with the rule of src/integration.cuh:80-95.
__device__ __forceinline__ bool wrap_xy(const Sys& S, double& x, double& y) {
    bool changed = false;
    if (S.periodic == 1 || S.periodic == 2) {
        if (x < S.origo[0]) { x += S.L[0]; changed = true; }
        if (x > S.L[0]) { x -= S.L[0]; changed = true; }
    }
    if (S.periodic == 1) {
        if (y < S.origo[1]) { y += S.L[1]; changed = true; }
        if (y > S.L[1]) { y -= S.L[1]; changed = true; }
    }
    return changed;
}

// Start-of-step position of sorted particle q: its stored record at the
// previous position perm[q], wrapped as the step's integrate wraps it.
__device__ __forceinline__ double4 spos(const DemDev& d, const Sys& S, uint32_t q) {
    double4 x = d.ro.x[d.perm[q]];
    (void)wrap_xy(S, x.x, x.y);
    return x;
}

// The same for non-inlined helpers, which take this small view by value
// instead of the DemDev.
struct PosView {
    const double4* x;
    const uint32_t* perm;  // nullptr: the storage order is the sorted order
    double ox, oy, Lx, Ly;
    int periodic;
};

__device__ __forceinline__ PosView pos_view(const DemDev& d, const Sys& S, bool sorted) {
    PosView v;
    v.x = d.ro.x; v.perm = sorted ? d.perm : nullptr;
    v.ox = S.origo[0]; v.oy = S.origo[1]; v.Lx = S.L[0]; v.Ly = S.L[1];
    v.periodic = S.periodic;
    return v;
}

__device__ __forceinline__ double4 pv_pos(const PosView& v, uint32_t q) {
    double4 x = v.x[v.perm ? v.perm[q] : q];
    if (v.periodic == 1 || v.periodic == 2) {
        if (x.x < v.ox) x.x += v.Lx;
        if (x.x > v.Lx) x.x -= v.Lx;
    }
    if (v.periodic == 1) {
        if (x.y < v.oy) x.y += v.Ly;
        if (x.y > v.Ly) x.y -= v.Ly;
    }
    return x;
}

// floor((v - origo)/(L/num)) (src/sorting.cuh:12-14), clamped to the grid.
__device__ __forceinline__ int cell_coord(double v, double origo, double cell_len, uint32_t num, uint32_t& err) {
    const double f = floor((v - origo) / cell_len);
    if (f != f) { err |= FLAG_NAN; return 0; }
    if (f < -1.0 || f > (double)num) err |= FLAG_OUT_OF_GRID;
    if (f < 0.0) return 0;
    if (f > (double)(num - 1)) return (int)(num - 1);
    return (int)f;
}
__device__ __forceinline__ int cell_coord(const Sys& S, double v, int a, uint32_t& err) {
    return cell_coord(v, S.origo[a], S.cell_len[a], S.num[a], err);
}

__global__ __launch_bounds__(BLOCK) void k_fill_u32(uint32_t* p, uint64_t n, uint32_t v) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Cell id of a position at the start of a step: the periodic wrap the step's
// integrate applies to it (src/integration.cuh:80-95) on a copy, then
// src/sorting.cuh:7-19.  The position itself is wrapped when it is gathered
// into the sorted order.
__device__ __forceinline__ uint32_t cell_key(const Sys& S, double x, double y, double z, uint32_t& err) {
    (void)wrap_xy(S, x, y);
    const int ix = cell_coord(S, x, 0, err);
    const int iy = cell_coord(S, y, 1, err);
    const int iz = cell_coord(S, z, 2, err);
    return S.cbase + (((uint32_t)iz * S.num[1]) * S.num[0] + (uint32_t)iy * S.num[0] + (uint32_t)ix);
}

// Runs of equal keys among a wavefront's lanes (the storage order is last
// step's sorted order, so keys come in runs): one atomic per run.  The lane
// gets counter[key]'s value before the run plus its place in the run.  Every
// lane of the wavefront below the grid's end calls it (the active lanes are a
// prefix).
__device__ __forceinline__ uint32_t run_add(uint32_t* counter, uint32_t key) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t prev = __shfl_up(key, 1, 64);
    const bool head = lane == 0u || prev != key;
    const uint64_t heads = __ballot(head);
    const uint64_t acts = __ballot(true);
    const uint64_t upto = (2ull << lane) - 1ull;  // lanes 0..lane (all 64 for lane 63)
    const uint32_t start = 63u - (uint32_t)__clzll((long long)(heads & upto));
    uint32_t base = 0;
    if (head) {
        const uint64_t above = heads & ~upto;
        const uint32_t end = above ? (uint32_t)__ffsll((long long)above) - 1u : 64u - (uint32_t)__clzll((long long)acts);
        base = atomicAdd(&counter[key], end - lane);
    }
    base = __shfl(base, (int)start, 64);
    return base + (lane - start);
}

// Raises bits of a step word where any of the calling lanes' conditions holds:
// one atomic per wavefront, and none once a read shows the bits.
__device__ __forceinline__ void raise(bool cond, uint32_t* word, uint32_t bits) {
    const uint64_t any = __ballot(cond);
    if (any == 0u || (threadIdx.x & 63u) != (uint32_t)__ffsll((unsigned long long)any) - 1u) return;
    if ((__hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & bits) != bits) atomicOr(word, bits);
}

// A step sorts only when a sphere changed its cell in the last one (or the
// state was set): otherwise the storage order is the sorted order and the
// previous step's cell offsets, sorted ids and keys stand.
__device__ __forceinline__ bool sorts(const DemDev& d) { return (d.fr[FW_SORT] & SORT_CELLS) != 0u; }
// The step's words as its kernels pass them on.
struct Words {
    bool sorted, rebuild, wrap;
    bool aligned = false;  // (quads) list indices are sorted positions
};
__device__ __forceinline__ Words words_of(const DemDev& d) {
    return {sorts(d), d.fr[FW_REBUILD] != 0u, d.fr[FW_WRAP] != 0u};
}
__device__ __forceinline__ const float4* xf_sorted(const DemDev& d, Words wd) { return wd.sorted ? d.xf : d.xfs; }

// Cell ids, counts and FP32 copies of the stored positions, for a state that
// did not come out of a step (after open or a position update); steps leave
// them to the next one in the force kernel.
template <bool B>
__global__ __launch_bounds__(BLOCK) void k_cellid(DemDev d) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= d.np) return;
    const Sys& S = sys_at<B>(d, i);
    double4 x = d.ro.x[i];
    uint32_t err = 0;
    const uint32_t key = cell_key(S, x.x, x.y, x.z, err);
    d.key[i] = key;
    if (err) atomicOr(&d.fr[FW_ERR], err);
    (void)run_add(d.count, key);
    (void)wrap_xy(S, x.x, x.y);
    const_cast<float4*>(d.xfs)[i] = make_float4((float)x.x, (float)x.y, (float)x.z, (float)x.w);
}

// -------------------------------------------------------------------- scan
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* lds, uint32_t& total) {
    // wave-level inclusive scan with shuffles, then across the 4 waves
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t inc = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t t = __shfl_up(inc, o, 64);
        if (lane >= o) inc += t;
    }
    if (lane == 63) lds[wave] = inc;
    __syncthreads();
    uint32_t woff = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < BLOCK / 64; ++w) {
        const uint32_t ws = lds[w];
        if (w < wave) woff += ws;
        tot += ws;
    }
    __syncthreads();
    total = tot;
    return woff + inc - v;
}

// pos_of of the particles whose sorted position changed in the step whose
// words are `words` (most keep theirs, which spares the scattered write), by
// block b.  Until then pos_of holds the storage positions -- the previous
// step's sorted positions, where the input set's records are -- which is what
// that step's force kernel gathered partner records through.
__device__ __forceinline__ void update_pos(const DemDev& d, uint32_t b) {
    const uint32_t q = b * BLOCK + threadIdx.x;
    if (q < d.np && d.perm[q] != q) d.pos_of[d.sid[q]] = q;
}
__device__ __forceinline__ void update_pos_of(const DemDev& d, const uint32_t* words, uint32_t b) {
    if (words[FW_SORT] & SORT_CELLS) update_pos(d, b);
}

// src/integration.cuh:191-221: blocks of 256 original indices, tree halving,
// for the walls that move; one wavefront per block b of indices, each lane
// with four of them, so the halvings take no barrier and most no LDS.  (Adding
// the loaded value to 0 first, as the reference does, turns a -0 into +0.)  A
// block without a force on the wall, as most are, sums to 0.  In an ensemble
// each system's blocks start at its first index, so every system is summed
// exactly as on its own.
__device__ __forceinline__ void load_wall_block(const DemDev& d, const Sys& S, uint32_t w, uint32_t b, double* v) {
    const uint32_t i0 = S.pbase + (b - S.bbase) * BLOCK + (threadIdx.x & 63u), end = S.pbase + S.np;
    const double* pp = d.wall_pp + (size_t)w * d.np;
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = i0 + 64 * k < end ? pp[i0 + 64 * k] : 0.0;
}
__device__ __forceinline__ double wall_block_sum(const double* v) {
    double sum = 0.0;
    if (__ballot(v[0] != 0.0 || v[1] != 0.0 || v[2] != 0.0 || v[3] != 0.0)) {
        // halvings by 128 and by 64, of values added to 0
        sum = ((0.0 + v[0]) + (0.0 + v[2])) + ((0.0 + v[1]) + (0.0 + v[3]));
#pragma unroll
        for (int o = 32; o != 0; o >>= 1) sum += __shfl_down(sum, o, 64);
    }
    return sum;
}
template <bool B>
__device__ __forceinline__ void wall_partials(const DemDev& d, uint32_t b) {
    if (b >= d.nwall_blocks) return;
    const Sys& S = B ? d.systems[d.sys_of_block[b]] : d.sys;
    for (uint32_t w = 0; w < S.nw; ++w) {
        if (!((S.wmoving >> w) & 1u)) continue;
        double v[4];
        load_wall_block(d, S, w, b, v);
        const double sum = wall_block_sum(v);
        if ((threadIdx.x & 63u) == 0u) d.wall_partial[(size_t)w * d.nwall_blocks + b] = sum;
    }
}

// src/integration.cuh:224-295, one wavefront per wall; then time.current +=
// dt.  The wall force is the serial sum of the block partials in block order:
// 64 of them sit in the wavefront's lanes, and the non-zero ones are added in
// lane order (adding a zero of either sign to the sum, which is never -0,
// leaves it as it is).
__device__ __forceinline__ double serial_sum(double part, double sum) {
    for (uint64_t m = __ballot(part != 0.0); m; m &= m - 1) {
        const int l = __ffsll((unsigned long long)m) - 1;
        const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)__double2loint(part), l);
        const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)__double2hiint(part), l);
        sum += __hiloint2double((int)hi, (int)lo);
    }
    return sum;
}

// One wall's record, as its leapfrog takes and leaves it.
struct Wall {
    double4 nx, mvfd;
    double vel0;
    int mode;
};
__device__ __forceinline__ Wall load_wall(const DemDev& d, uint32_t w) { return {d.wnx[w], d.wmvfd[w], d.wvel0[w], d.wmode[w]}; }
__device__ __forceinline__ void step_wall(const DemDev& d, const Sys& S, uint32_t w, Wall wl, double fz, double t_current) {
    wl.mvfd.z = fz;
    const double dt = S.dt;
    // (without a deviatoric amplitude the product is a zero, whose sign
    // does not reach acc: fz is never -0)
    const double arg = 2.0 * PI_WALL * S.devs_f * t_current;
    const double sigma_0 = wl.mvfd.w + (S.devs_A == 0.0 && isfinite(arg) ? 0.0 : S.devs_A * sin(arg));
    const double N = -sigma_0 * S.L[0] * S.L[1];
    double acc = (wl.mvfd.z + N) / wl.mvfd.x;
    if (wl.mode == 2) acc = 0.0;
    wl.vel0 += acc * dt;
    wl.nx.w += wl.vel0 * dt;
    wl.mvfd.y = wl.vel0 + 0.5 * acc * dt;
    d.wnx[w] = wl.nx;
    d.wmvfd[w] = wl.mvfd;
    d.wvel0[w] = wl.vel0;
}

template <bool B>
__device__ __forceinline__ void walls_update(const DemDev& d, uint32_t k) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    const Sys& S = B ? d.systems[k] : d.sys;
    const double t_current = d.t_cur[k];
    __syncthreads();
    for (uint32_t w = wave; w < S.nw; w += waves) {
        if (!((S.wmoving >> w) & 1u)) continue;
        const double* src = d.wall_partial + (size_t)w * d.nwall_blocks + S.bbase;
        double fz = 0.0;
        double next = lane < S.nblocks ? src[lane] : 0.0;
        for (uint32_t c0 = 0; c0 < S.nblocks; c0 += 64) {
            const double part = next;
            next = c0 + 64 + lane < S.nblocks ? src[c0 + 64 + lane] : 0.0;
            fz = serial_sum(part, fz);
        }
        if (lane == 0) step_wall(d, S, S.wbase + w, load_wall(d, S.wbase + w), fz, t_current);
    }
    if (threadIdx.x == 0) d.t_cur[k] = t_current + S.dt;
}

// Wall sums and wall update of system `sys`, of at most WALL_BLOCKS wall-sum
// blocks, by one workgroup, the partials in LDS (part, WALL_BLOCKS of them).
template <bool B>
__device__ __forceinline__ void walls_sum_update(const DemDev& d, uint32_t sys, double* part) {
    const Sys& S = B ? d.systems[sys] : d.sys;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const double t_current = d.t_cur[sys];
    for (uint32_t w = 0; w < S.nw; ++w) {
        if (!((S.wmoving >> w) & 1u)) continue;
        const Wall wl = load_wall(d, S.wbase + w);
        __syncthreads();
        // eight blocks a wavefront at a time, their loads in flight together
        constexpr uint32_t E = 8, W = BLOCK / 64;
        for (uint32_t b0 = wave; b0 < S.nblocks; b0 += E * W) {
            double v[E][4];
#pragma unroll
            for (uint32_t k = 0; k < E; ++k) load_wall_block(d, S, w, S.bbase + b0 + k * W, v[k]);
#pragma unroll
            for (uint32_t k = 0; k < E; ++k) {
                const double sum = wall_block_sum(v[k]);
                if (lane == 0 && b0 + k * W < S.nblocks) part[b0 + k * W] = sum;
            }
        }
        __syncthreads();
        if (wave == 0) {
            double fz = 0.0;
            for (uint32_t c0 = 0; c0 < S.nblocks; c0 += 64)
                fz = serial_sum(c0 + lane < S.nblocks ? part[c0 + lane] : 0.0, fz);
            if (lane == 0) step_wall(d, S, S.wbase + w, wl, fz, t_current);
        }
    }
    if (threadIdx.x == 0) d.t_cur[sys] = t_current + S.dt;
}

__device__ __forceinline__ void scan_reduce(const DemDev& d, uint32_t b, uint32_t* lds) {
    const uint32_t base = b * SCAN_TILE + threadIdx.x * SCAN_PER_THREAD;
    uint32_t sum = 0;
#pragma unroll
    for (int j = 0; j < SCAN_PER_THREAD; ++j)
        if (base + j < d.K) sum += d.count[base + j];
    uint32_t total;
    (void)block_exclusive_scan(sum, lds, total);
    if (threadIdx.x == 0) d.scan_bsum[b] = total;
}

// The previous step's inverse permutation and wall-force partials (LEAD) and
// this step's per-cell totals, in one launch: none needs another's result.
template <bool B, bool LEAD>
__global__ __launch_bounds__(BLOCK) void k_head(DemDev d) {
    __shared__ uint32_t lds[BLOCK / 64];
    const uint32_t b = blockIdx.x;
    if (b == 0 && threadIdx.x == 0) {
        // the errors of the last step's new positions belong to this step
        const uint32_t f = d.fr[FW_ERR];
        if (f) atomicOr(d.flags, f);
        if (d.search_mode == 5 && d.fr[FW_REBUILD]) d.nstate[NSTATE_BUILDS] += 1u;
        if (sorts(d)) d.nstate[NSTATE_ALIGNED] = 0u;
    }
    if constexpr (LEAD) {
        update_pos_of(d, d.fw, b);
        wall_partials<B>(d, b * (BLOCK / 64) + (threadIdx.x >> 6));
    }
    if (b < d.scan_blocks && sorts(d)) scan_reduce(d, b, lds);
}

// The end of a call's last step: what k_head<B, true> does for the others.
template <bool B>
__global__ __launch_bounds__(BLOCK) void k_tail(DemDev d) {
    update_pos_of(d, d.fr, blockIdx.x);
    wall_partials<B>(d, blockIdx.x * (BLOCK / 64) + (threadIdx.x >> 6));
}

template <bool B>
__global__ __launch_bounds__(BLOCK) void k_walls(DemDev d) { walls_update<B>(d, blockIdx.x); }

// off[c] = first sorted position of cell c, off[K] = np.  Each block adds
// the totals of the blocks before it (integer sums: any order).
__device__ __forceinline__ void scan_down(const DemDev& d, uint32_t block, uint32_t* lds) {
    uint32_t before = 0;
    for (uint32_t b = threadIdx.x; b < block; b += BLOCK) before += d.scan_bsum[b];
    uint32_t prefix;
    (void)block_exclusive_scan(before, lds, prefix);
    const uint32_t base = block * SCAN_TILE + threadIdx.x * SCAN_PER_THREAD;
    uint32_t c[SCAN_PER_THREAD];
    uint32_t sum = 0;
#pragma unroll
    for (int j = 0; j < SCAN_PER_THREAD; ++j) {
        c[j] = base + j < d.K ? d.count[base + j] : 0u;
        sum += c[j];
    }
    uint32_t total;
    uint32_t off = block_exclusive_scan(sum, lds, total) + prefix;
#pragma unroll
    for (int j = 0; j < SCAN_PER_THREAD; ++j) {
        if (base + j < d.K) {
            d.off[base + j] = off;
            d.cursor[base + j] = off;
        }
        off += c[j];
        if (base + j + 1 == d.K) d.off[d.K] = off;
    }
}

__global__ __launch_bounds__(BLOCK) void k_scan_down(DemDev d) {
    __shared__ uint32_t lds[BLOCK / 64];
    if (blockIdx.x == 0 && threadIdx.x < FW_WORDS) d.fw[threadIdx.x] = 0u;
    if (sorts(d)) scan_down(d, blockIdx.x, lds);
}

__device__ __forceinline__ void place(const DemDev& d, uint32_t i) {
    const uint32_t q = run_add(d.cursor, d.key[i]);
    if (q < d.np) d.perm[q] = i;  // (counts and keys agree by construction; never write past perm)
}

// Places the particles of each cell, in any order (k_order sorts them).
__global__ __launch_bounds__(BLOCK) void k_scatter(DemDev d) {
    if (!sorts(d)) return;
    const uint32_t i = xcd_block() * blockDim.x + threadIdx.x;
    if (i < d.np) place(d, i);
}

// Order one cell's members by original index: odd-even transposition network
// on (id, position) pairs in registers for up to W members, insertion sort in
// memory beyond that.
template <int W>
__device__ __forceinline__ void sort_small(const DemDev& d, uint32_t* p, uint32_t n) {
    uint64_t v[W];
#pragma unroll
    for (int j = 0; j < W; ++j)
        v[j] = (uint32_t)j < n ? ((uint64_t)d.ro.id[p[j]] << 32) | p[j] : ~0ull;
#pragma unroll
    for (int r = 0; r < W; ++r) {
#pragma unroll
        for (int j = (r & 1); j + 1 < W; j += 2) {
            const uint64_t a = v[j], b = v[j + 1];
            v[j] = a < b ? a : b;
            v[j + 1] = a < b ? b : a;
        }
    }
#pragma unroll
    for (int j = 0; j < W; ++j)
        if ((uint32_t)j < n) p[j] = (uint32_t)v[j];
}

__device__ __forceinline__ void sort_cell(const DemDev& d, uint32_t c) {
    const uint32_t st = d.off[c];
    const uint32_t n = d.off[c + 1] - st;
    uint32_t* p = d.perm + st;
    if (n < 2) return;
    if (n <= 4) sort_small<4>(d, p, n);
    else if (n <= 8) sort_small<8>(d, p, n);
    else if (n <= 16) sort_small<16>(d, p, n);
    else {
        for (uint32_t i = 1; i < n; ++i) {
            const uint32_t v = p[i];
            const uint32_t key = d.ro.id[v];
            uint32_t j = i;
            while (j > 0 && d.ro.id[p[j - 1]] > key) { p[j] = p[j - 1]; --j; }
            p[j] = v;
        }
    }
}

__device__ __forceinline__ void gather_sorted(const DemDev& d, uint32_t q) {
    const uint32_t p = d.perm[q];
    d.xf[q] = d.xfs[p];
    d.sid[q] = d.ro.id[p];
    d.skey[q] = d.key[p];
    if (d.search_mode == 5) {
        const uint32_t li = d.ro.lidx[p];
        d.linv[li] = q;
        d.slidx[q] = li;
    }
}

__device__ __forceinline__ void order_cells(const DemDev& d, uint32_t b) {
    const uint32_t c0 = b * BLOCK, c = c0 + threadIdx.x;
    if (c0 >= d.K) return;
    const uint32_t q0 = d.off[c0], q1 = d.off[c0 + BLOCK < d.K ? c0 + BLOCK : d.K];
    if (c < d.K) sort_cell(d, c);
    __syncthreads();
    for (uint32_t q = q0 + threadIdx.x; q < q1; q += BLOCK) gather_sorted(d, q);
}

// The members of BLOCK cells, one thread per cell, into original-index order
// (with the counting sort's placement the stable sort of src/device.cu:
// 763-765); then the block's run of sorted positions, one thread each: ids,
// keys and FP32 positions (src/sorting.cuh:49-121 gathers x, vel, angvel) and,
// in search mode 5, the list index.  On a step that does not sort nothing is
// left to do but to reset a permutation that an earlier step left.
__global__ __launch_bounds__(BLOCK) void k_order(DemDev d) {
    const uint32_t word = d.fr[FW_SORT];
    if (word == 0u) return;
    const uint32_t b = xcd_block();
    if (word & SORT_CELLS) {
        order_cells(d, b);
        return;
    }
    const uint32_t c0 = b * BLOCK;
    const uint32_t q0 = d.off[c0], q1 = d.off[c0 + BLOCK < d.K ? c0 + BLOCK : d.K];
    for (uint32_t q = q0 + threadIdx.x; q < q1; q += BLOCK) d.perm[q] = q;
}

// ------------------------------------------------------------------- bonds
// src/cohesion.cuh:8-233.  The force and torque of an intact bond go to
// bond_f/bond_t; the contact kernel adds them per particle in ascending bond
// index (the reference adds them with racing += at :220-226).
__device__ __forceinline__ void bond_force(const DemDev& d, uint32_t k) {
    const Sys& S = d.sys;
    const uint2 bond = d.bonds[k];
    if (!(bond.x < d.np)) return;
    const double dt = S.dt;
    const double4 d0 = d.bdelta[k], o0 = d.bomega[k];
    V3<double> delta0_t = mk(d0.x, d0.y, d0.z);
    const double delta0_n = d0.w;
    V3<double> omega0_t = mk(o0.x, o0.y, o0.z);
    const double omega0_n = o0.w;
    const uint32_t pi = d.pos_of[bond.x], pj = d.pos_of[bond.y];
    const double4 x_i = d.ro.x[pi], x_j = d.ro.x[pj];
    const double4 vel_i = d.ro.vel[pi], vel_j = d.ro.vel[pj];
    const V3<double> angvel_i = xyz(d.ro.angvel[pi]), angvel_j = xyz(d.ro.angvel[pj]);
    const double R_bar = d.lambda_bar * fmin(x_i.w, x_j.w);
    const double A = PI_REF * R_bar * R_bar;
    const double I = 0.25 * PI_REF * R_bar * R_bar * R_bar * R_bar;
    const double J = I * 2.0;
    const V3<double> x = mk(x_i.x - x_j.x, x_i.y - x_j.y, x_i.z - x_j.z);
    const double x_length = vlen(x);
    const double overlap = fmin(0.0, x_length - (x_i.w + x_j.w));
    const V3<double> n = x / x_length;
    delta0_t = delta0_t - (n * dot(n, delta0_t));
    const V3<double> ddelta = (mk(vel_i.x - vel_j.x, vel_i.y - vel_j.y, vel_i.z - vel_j.z)
                               + (x_i.w + overlap / 2.0) * cross(n, angvel_i)
                               + (x_j.w + overlap / 2.0) * cross(n, angvel_j)) * dt;
    const double ddelta_n = -dot(ddelta, n);
    const double delta_n = delta0_n + ddelta_n;
    const V3<double> ddelta_t = ddelta - n * dot(n, ddelta);
    const V3<double> delta_t = delta0_t + ddelta_t;
    const V3<double> f_n = (S.k_n * A * delta_n + S.gamma_n * ddelta_n / dt) * n;
    const V3<double> f_t = -S.k_t * A * delta_t - S.gamma_t * ddelta_t / dt;
    const V3<double> f = f_n + f_t;
    const V3<double> mn = -n;
    omega0_t = omega0_t - mn * dot(omega0_t, mn);
    const V3<double> domega = mk(angvel_j.x - angvel_i.x, angvel_j.y - angvel_i.y, angvel_j.z - angvel_i.z) * dt;
    const double domega_n = dot(domega, mn);
    const double omega_n = omega0_n + domega_n;
    const V3<double> domega_t = domega - domega_n * mn;
    const V3<double> omega_t = omega0_t + domega_t;
    const V3<double> t_n = -S.k_t * J * omega_n * mn;
    const V3<double> t_t = -S.k_n * I * omega_t;
    const V3<double> t_j = t_n + t_t;
    const double sigma_max = vlen(f_n) / A + vlen(t_t) * R_bar / I;
    const double tau_max = vlen(f_t) / A + vlen(t_n) * R_bar / J;
    if (sigma_max >= d.sigma_b || tau_max >= d.tau_b) {
        d.bonds[k].x = d.bond_broken;
        return;
    }
    d.bdelta[k] = make_double4(delta_t.x, delta_t.y, delta_t.z, delta_n);
    d.bomega[k] = make_double4(omega_t.x, omega_t.y, omega_t.z, omega_n);
    d.bond_f[k] = make_double4(f.x, f.y, f.z, 0.0);
    d.bond_t[k] = make_double4(t_j.x, t_j.y, t_j.z, 0.0);
}

__global__ __launch_bounds__(BLOCK) void k_bonds(DemDev d) {
    const uint32_t k = xcd_block() * blockDim.x + threadIdx.x;
    if (k < d.nb0) bond_force(d, k);
}

// --------------------------------------------------------- contact models
struct Acc {
    V3<double> F, T;
    double es_dot, ev_dot, p;
};

// src/contactmodels.cuh:283-493 in arithmetic T (double: the reference's
// FP64 path; float: the mixed mode's pair force).  Sums go to FP64.  What
// cannot change a bit of the result is left out: a length is compared with 0
// by its square; without cohesion the capillary term is a zero of some sign,
// which neither a length nor a sum that started at +0 sees (so the normal
// force's own length is the friction limit's); and the pressure is summed only
// if the step keeps it.  That is three square roots and three divisions a
// sticking contact instead of seven and four: the pair force was half of the
// FP64 instructions' issue time of a twelve-contact crystal's force kernel
// (1,048,576 spheres: 396 -> 388 us, which the gathers bound now; in FP32,
// 500,000 spheres: 152 -> 149).
template <class T>
__device__ __forceinline__ void contact_linear(const Sys& S, Acc& acc, V3<T> vel_a, V3<T> angvel_a,
                                               V3<T> vel_b, V3<T> angvel_b, T radius_a, T radius_b,
                                               V3<T> x, T x_length, T delta, V3<T>& delta_t_io, bool keep_p) {
    const T k_n = (T)S.k_n, k_t = (T)S.k_t, gamma_n = (T)S.gamma_n, gamma_t = (T)S.gamma_t;
    const T mu_s = (T)S.mu_s, mu_d = (T)S.mu_d, kappa = (T)S.kappa, dt = (T)S.dt;
    const V3<T> delta_t0_uncor = delta_t_io;
    const V3<T> n = x / x_length;
    const V3<T> vel_linear = vel_a - vel_b;
    const V3<T> vel = vel_linear + (radius_a + delta / (T)2.0) * cross(n, angvel_a)
                      + (radius_b + delta / (T)2.0) * cross(n, angvel_b);
    const T vel_n = -dot(vel_linear, n);
    const V3<T> vel_t = vel - n * dot(n, vel);
    const V3<T> delta_t0 = delta_t0_uncor - (n * dot(n, delta_t0_uncor));
    V3<T> delta_t = delta_t0;
    V3<T> f_n = (-k_n * delta - gamma_n * vel_n) * n;
    acc.ev_dot += (double)(gamma_n * vel_n * vel_n);
    if (dot(f_n, n) < (T)0.0) f_n = mk<T>(0, 0, 0);
    const T f_n_length = vlen(f_n);
    T hold = f_n_length;  // |f_n - f_c|
    V3<T> f_c = mk<T>(0, 0, 0);
    if (kappa != (T)0.0) {
        f_c = (-kappa * (T)sqrt(radius_a * radius_b)) * n;
        hold = vlen(f_n - f_c);
    }
    V3<T> f_t = mk<T>(0, 0, 0);
    if (dot(delta_t0, delta_t0) > (T)0.0 || dot(vel_t, vel_t) > (T)0.0) {
        delta_t = delta_t0 + vel_t * dt;
        const V3<T> f_t_elast = -k_t * delta_t;
        const V3<T> f_t_visc = -gamma_t * vel_t;
        f_t = f_t_elast + f_t_visc;
        const T f_t_length = vlen(f_t);
        const T f_t_limit = mu_s * hold;
        delta_t = delta_t0 + vel_t * dt;
        if (f_t_length > f_t_limit) {
            const V3<T> t = f_t / f_t_length;
            f_t = f_t_limit * t;
            delta_t = (T)-1.0 / k_t * (mu_d * hold * t + gamma_t * vel_t);
            acc.es_dot += (double)(vlen(vlen(f_t) * vel_t * dt) / dt);
        }
    }
    V3<T> fsum = f_n + f_t;
    if (kappa != (T)0.0) fsum = fsum + f_c;
    acc.F = acc.F + mk<double>(fsum.x, fsum.y, fsum.z);
    const V3<T> tq = cross(-(radius_a + delta * (T)0.5) * n, f_t);
    acc.T = acc.T + mk<double>(tq.x, tq.y, tq.z);
    if (keep_p) acc.p += (double)(f_n_length / ((T)4.0 * (T)PI_REF * radius_a * radius_a));
    delta_t_io = delta_t;
}

// src/contactmodels.cuh:499-666 contactHertz (contact model 3), FP64, for a
// positive overlap xi = -delta.  The reference raises the negative overlap
// itself to the powers 3/2, 1/4 and 1/2 (powf of a negative number: NaN
// forces); each power is taken here of xi, with the sign the linear law's
// terms carry (elastic normal term k_n xi^(3/2) repulsive, positive viscous
// and tangential coefficients), as xi sqrt(xi), sqrt(sqrt(xi)), sqrt(xi).
// The rolling resistance (:642-653) opposes the relative spin with the
// smaller of gamma_r r_a |w_ab| and mu_r r_a |f_n|.
__device__ __forceinline__ void contact_hertz(const Sys& S, Acc& acc, V3<double> vel_a, V3<double> angvel_a,
                                              V3<double> vel_b, V3<double> angvel_b, double radius_a,
                                              double radius_b, V3<double> x, double x_length, double delta,
                                              V3<double>& delta_t_io) {
    const double xi = -delta;
    const double sq = sqrt(xi);
    const double xi32 = xi * sq, xi14 = sqrt(sq), xi12 = sq;
    const V3<double> delta_t0_uncor = delta_t_io;
    const V3<double> n = x / x_length;
    const V3<double> vel_linear = vel_a - vel_b;
    const V3<double> vel = vel_linear + (radius_a + delta / 2.0) * cross(n, angvel_a)
                           + (radius_b + delta / 2.0) * cross(n, angvel_b);
    const V3<double> angvel_ab = angvel_a - angvel_b;
    const double angvel_ab_length = vlen(angvel_ab);
    const double vel_n = dot(vel_linear, n);
    const V3<double> vel_t = vel - n * dot(vel, n);
    const double vel_t_length = vlen(vel_t);
    const V3<double> delta_t0 = delta_t0_uncor - n * dot(delta_t0_uncor, n);
    const double delta_t0_length = vlen(delta_t0);
    V3<double> delta_t = delta_t0;
    V3<double> f_n = (S.k_n * xi32 - S.gamma_n * xi14 * vel_n) * n;
    acc.ev_dot += S.gamma_n * vel_n * vel_n;
    if (dot(f_n, n) < 0.0) f_n = mk(0.0, 0.0, 0.0);
    const double f_n_length = vlen(f_n);
    const V3<double> f_c = (-S.kappa * sqrt(radius_a * radius_b)) * n;
    V3<double> f_t = mk(0.0, 0.0, 0.0), t_res = mk(0.0, 0.0, 0.0);
    if (delta_t0_length > 0.0 || vel_t_length > 0.0) {
        const V3<double> f_t_elast = (-S.k_t * xi12) * delta_t0;
        const V3<double> f_t_visc = (-S.gamma_t * xi14) * vel_t;
        const double f_t_limit = vel_t_length > (double)0.001f ? S.mu_d * vlen(f_n - f_c) : S.mu_s * vlen(f_n - f_c);
        f_t = f_t_elast + f_t_visc;
        const double f_t_length = vlen(f_t);
        if (f_t_length > f_t_limit) {
            f_t = f_t * (f_t_limit / f_t_length);
            delta_t = (f_t + (S.gamma_t * xi14) * vel_t) / (-S.k_t * xi12);
            acc.es_dot += vlen(delta_t0 - delta_t) * S.k_t / S.dt;
        } else {
            delta_t = delta_t0 + vel_t * S.dt;
        }
    }
    if (angvel_ab_length > 0.0)
        t_res = ((-1.0 * fmin(S.gamma_r * radius_a * angvel_ab_length, S.mu_r * radius_a * f_n_length)) * angvel_ab) /
                angvel_ab_length;
    acc.F = acc.F + ((f_n + f_t) + f_c);
    acc.T = acc.T + ((-(radius_a + delta / 2.0)) * cross(n, f_t) + t_res);
    acc.p += f_n_length / (4.0 * PI_REF * radius_a * radius_a);
    delta_t_io = delta_t;
}

// src/contactmodels.cuh:10-109 contactLinear_wall (FP64 in both modes).
__device__ __forceinline__ double contact_wall(const Sys& S, Acc& acc, V3<double> linvel, V3<double> angvel,
                                               double radius_a, V3<double> n, double delta, double wvel) {
    const V3<double> v0 = linvel + radius_a * cross(n, angvel);
    // operator+(Float3, Float) adds the scalar wall velocity to every component
    const V3<double> vel = mk(v0.x + wvel, v0.y + wvel, v0.z + wvel);
    const double vel_n = dot(vel, n);
    const V3<double> vel_t = vel - n * dot(vel, n);
    const double vel_t_length = vlen(vel_t);
    V3<double> f_n = (-S.k_n * delta - S.gamma_wn * vel_n) * n;
    if (dot(f_n, n) < 0.0) f_n = mk(0.0, 0.0, 0.0);
    const double f_n_length = vlen(f_n);
    V3<double> f_t = mk(0.0, 0.0, 0.0);
    if (vel_t_length > 0.0) {
        const double f_t_visc = S.gamma_wt * vel_t_length;
        const double f_t_limit = vel_t_length > (double)0.001f ? S.mu_wd * f_n_length : S.mu_ws * f_n_length;
        if (f_t_visc < f_t_limit) f_t = (-1.0 * f_t_visc) * vel_t / vel_t_length;
        else f_t = (-1.0 * f_t_limit) * vel_t / vel_t_length;
    }
    acc.F = acc.F + (f_n + f_t);
    const V3<double> tq = (-radius_a) * cross(n, f_t);
    acc.T = acc.T + mk(tq.x + 0.0, tq.y + 0.0, tq.z + 0.0);
    acc.p += f_n_length / (4.0 * PI_REF * radius_a * radius_a);
    return dot(f_n, n);
}

// The exponential of the capillary bond (the reference calls expf on a
// double): fixed steps, the same as the oracle's -- Cody-Waite reduction
// x = k ln2 + r with |r| <= ln2/2, the Taylor series of e^r to degree 13 by
// Horner's rule, scaling by 2^k -- so both sides get the same bits.
__device__ __forceinline__ double det_exp(double x) {
    const double inv_ln2 = 1.4426950408889634074;
    const double ln2_hi = 6.93147180369123816490e-01, ln2_lo = 1.90821492927058770002e-10;
    const double k = rint(x * inv_ln2);
    const double r = (x - k * ln2_hi) - k * ln2_lo;
    double q = 1.0 / 6227020800.0;  // 1/13!
    q = q * r + 1.0 / 479001600.0;
    q = q * r + 1.0 / 39916800.0;
    q = q * r + 1.0 / 3628800.0;
    q = q * r + 1.0 / 362880.0;
    q = q * r + 1.0 / 40320.0;
    q = q * r + 1.0 / 5040.0;
    q = q * r + 1.0 / 720.0;
    q = q * r + 1.0 / 120.0;
    q = q * r + 1.0 / 24.0;
    q = q * r + 1.0 / 6.0;
    q = q * r + 0.5;
    q = q * r + 1.0;
    q = q * r + 1.0;
    return ldexp(q, (int)k);
}

// src/contactmodels.cuh:114-253 contactLinearViscous (contact model 1, FP64
// in both precision modes): no spring history, no torque (commented out in
// the reference), viscous tangential force capped by Coulomb friction.
__device__ __forceinline__ void contact_viscous(const Sys& S, Acc& acc, V3<double> vel_a, V3<double> angvel_a,
                                                V3<double> vel_b, V3<double> angvel_b, double radius_a,
                                                double radius_b, V3<double> x, double x_length, double delta) {
    const V3<double> n = x / x_length;
    const V3<double> vel_linear = vel_a - vel_b;
    const V3<double> vel = vel_linear + (radius_a + delta / 2.0) * cross(n, angvel_a)
                           + (radius_b + delta / 2.0) * cross(n, angvel_b);
    const double vel_n = dot(vel_linear, n);
    const V3<double> vel_t = vel - n * dot(vel, n);
    const double vel_t_length = vlen(vel_t);
    V3<double> f_n = (-S.k_n * delta - S.gamma_n * vel_n) * n;
    if (dot(f_n, n) < 0.0) f_n = mk(0.0, 0.0, 0.0);
    const double f_n_length = vlen(f_n);
    const V3<double> f_c = (-S.kappa * sqrt(radius_a * radius_b)) * n;
    V3<double> f_t = mk(0.0, 0.0, 0.0);
    if (vel_t_length > 0.0) {
        const double f_t_visc = S.gamma_t * vel_t_length;
        const double f_t_limit = vel_t_length > (double)0.001f ? S.mu_d * vlen(f_n - f_c) : S.mu_s * vlen(f_n - f_c);
        if (f_t_visc < f_t_limit) f_t = ((-f_t_visc) * vel_t) / vel_t_length;
        else f_t = ((-f_t_limit) * vel_t) / vel_t_length;
    }
    acc.F = acc.F + (f_n + f_t + f_c);
    acc.p += f_n_length / (4.0 * PI_REF * radius_a * radius_a);
}

// src/cohesion.cuh:314-350 capillaryCohesion_exp, as written (the decay
// length has h = -sqrt(r) < 0).
__device__ __forceinline__ void capillary(const Sys& S, Acc& acc, double radius_a, double radius_b, double delta,
                                          V3<double> x, double x_length) {
    const V3<double> n = x / x_length;
    const double r = (radius_a / radius_b) > (radius_b / radius_a) ? radius_a / radius_b : radius_b / radius_a;
    const double h = -sqrt(r);
    const double R_har = (2.0 * radius_a * radius_b) / (radius_a + radius_b);
    const double R_geo = sqrt(radius_a * radius_b);
    const double lambda = (double)0.9f * h * sqrt(S.V_b / R_har);
    acc.F = acc.F + (-S.kappa * R_geo * det_exp(-delta / lambda)) * n;
}

__device__ __forceinline__ void decode_image(const Sys& S, uint32_t code, double& dx, double& dy) {
    const uint32_t cx = code & 3u, cy = (code >> 2) & 3u;
    dx = cx == 1u ? S.L[0] : (cx == 2u ? -S.L[0] : 0.0);
    dy = cy == 1u ? S.L[1] : (cy == 2u ? -S.L[1] : 0.0);
}

// A partner's velocity records as the pair force of arithmetic T reads
// them: the FP64 records, or (mixed mode) their FP32 copies, which the
// previous step's force kernel wrote next to them -- the same values the
// pair force would round them to, in half the bytes.
template <class T> struct PartnerVel;
template <> struct PartnerVel<double> {
    using type = double4;
    static __device__ __forceinline__ double4 vel(const DemDev& d, uint32_t p) { return d.ro.vel[p]; }
    static __device__ __forceinline__ double4 angvel(const DemDev& d, uint32_t p) { return d.ro.angvel[p]; }
    static __device__ __forceinline__ double4 zero() { return make_double4(0.0, 0.0, 0.0, 0.0); }
    static __device__ __forceinline__ V3<double> v3(double4 a) { return xyz(a); }
};
template <> struct PartnerVel<float> {
    using type = float4;
    static __device__ __forceinline__ float4 vel(const DemDev& d, uint32_t p) { return d.ro.vf[p]; }
    static __device__ __forceinline__ float4 angvel(const DemDev& d, uint32_t p) { return d.ro.wf[p]; }
    static __device__ __forceinline__ float4 zero() { return make_float4(0.f, 0.f, 0.f, 0.f); }
    static __device__ __forceinline__ V3<float> v3(float4 a) { return mk<float>(a.x, a.y, a.z); }
};

// Stores of what only the next step's own thread reads: springs and private
// records.  In a system whose steps' state no longer fits the 256 MB of the
// memory-side cache they would only push out of the caches what the step still
// reads (its neighbours' records, the lists); below, the next step finds them
// there.  us a step without and with: crystal of 171,500 spheres 59 and 73, of
// 256,000 110 and 107, of 364,500 150 and 141, of 500,000 201 and 191, of
// 1,048,576 398 and 382 (mixed precision 47 and 54, 68 and 83, 110 and 104, 150
// and 146, 296 and 291); bonded 256,000 382 and 374; lattice of 262,144 51 and
// 58, of 512,000 105 and 99, of 1,000,000 210 and 205; loose packing of 131,071
// 36 and 38, of 300,000 61 and 73; ensemble of 328,596 66 and 75.  The line is
// that of packings with few contacts, which lose most on the wrong side of it;
// crystals pass it at about 240,000 spheres in FP64 and 330,000 in mixed
// precision and lose up to 6 % below it.  (Streaming their loads as well made
// the crystal slower: 473 against 450 a step, as stages.)
constexpr uint32_t STREAM_NP = 400000;
using nt4 = double __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void put(const DemDev& d, double4* p, double4 v) {
    if (d.np >= STREAM_NP) {
        const nt4 w = {v.x, v.y, v.z, v.w};
        __builtin_nontemporal_store(w, reinterpret_cast<nt4*>(p));
    } else {
        *p = v;
    }
}
template <class T> __device__ __forceinline__ void put3(const DemDev& d, T* p, V3<T> v) {
    if (d.np >= STREAM_NP) {
        __builtin_nontemporal_store(v.x, p);
        __builtin_nontemporal_store(v.y, p + 1);
        __builtin_nontemporal_store(v.z, p + 2);
    } else {
        p[0] = v.x; p[1] = v.y; p[2] = v.z;
    }
}

// The spring of contact slot k: read at the particle's storage position in
// the step's input set, written at its sorted position in the output set.
template <class T> struct SlotStore;
template <> struct SlotStore<double> {
    static __device__ __forceinline__ V3<double> load(const DemDev& d, int k, uint32_t q) {
        const double* p = d.ro.cdt + 3 * ((size_t)k * d.np + q);
        return mk(p[0], p[1], p[2]);
    }
    static __device__ __forceinline__ void store(const DemDev& d, int k, uint32_t q, V3<double> v) {
        put3(d, d.wo.cdt + 3 * ((size_t)k * d.np + q), v);
    }
};
template <> struct SlotStore<float> {
    static __device__ __forceinline__ V3<float> load(const DemDev& d, int k, uint32_t q) {
        const float* p = d.ro.cdt32 + 3 * ((size_t)k * d.np + q);
        return mk(p[0], p[1], p[2]);
    }
    static __device__ __forceinline__ void store(const DemDev& d, int k, uint32_t q, V3<float> v) {
        put3(d, d.wo.cdt32 + 3 * ((size_t)k * d.np + q), v);
    }
};

// The search kernels that run once per step carry the previous step's wall
// update, which only the force kernel after them reads: the first lead_blocks
// blocks (one per system) make it, beside the others' search.
template <bool B>
__device__ __forceinline__ bool lead_walls(const DemDev& d) {
    if (blockIdx.x >= d.lead_blocks) return false;
    walls_update<B>(d, blockIdx.x);
    return true;
}
// xcd_block of the blocks after those.
__device__ __forceinline__ uint32_t work_block(const DemDev& d) {
    const uint32_t nb = gridDim.x - d.lead_blocks, b = blockIdx.x - d.lead_blocks;
    const uint32_t q = nb >> 3, r = nb & 7u, xcd = b & 7u, k = b >> 3;
    return xcd * q + (xcd < r ? xcd : r) + k;
}

// ----------------------------------------------------------- contact search
// One block per tile of tile_x x tile_y cells in one z plane.  The positions
// of every particle in the 3 x (tile_y+2) x (tile_x+2) cells around the tile
// are staged once into LDS (each staged cell is a contiguous run of the
// sorted arrays); each thread then walks its particle's 27 cells from LDS in
// the reference's z, y, x order and, within a cell, in sorted order
// (src/contactsearch.cuh:181-355).  A tile whose neighbourhood exceeds the
// LDS capacity reads the same candidates from HBM instead.
struct TopoShared {
    double4 pos[TOPO_CAP];
    uint32_t cstart[TOPO_MAX_CELLS + 1];  // LDS offset of each staged cell
    uint32_t cglob[TOPO_MAX_CELLS];       // first sorted index of each staged cell
    uint8_t ccode[TOPO_MAX_CELLS];        // periodic image code of each staged cell
    uint32_t scan[BLOCK / 64];
};

// The slot words of one particle in the step's input set: word k of the
// particle stored at q is cslot[k * np + q] (slot-major, like the springs).
// A search updates the row in place (each particle's row is its own); the
// force kernel carries the words of the contacts that last into the output
// set at the particle's sorted position.
struct SlotRow {
    uint32_t* p;
    size_t ld;
    __device__ __forceinline__ uint32_t& operator[](int k) const { return p[(size_t)k * ld]; }
};
__device__ __forceinline__ SlotRow slot_row(const DemDev& d, uint32_t s) { return {d.ro.cslot + d.perm[s], d.np}; }

// Slot bookkeeping of one confirmed overlap (src/contactsearch.cuh:252-284):
// the slot already holding b (lowest), else the highest empty slot.
struct SlotState {
    uint32_t mask, fresh, nc, err;
    bool stop;
};

__device__ __noinline__ void slot_insert(SlotRow slot, SlotState& st, uint32_t bo, uint32_t code) {
    int cpos = -1;
    for (uint32_t m = st.mask; m; m &= m - 1) {
        const int i = __ffs(m) - 1;
        if ((slot[i] & SLOT_IDX_MASK) == bo) { cpos = i; break; }
    }
    if (cpos < 0) {
        const uint32_t empty = ~st.mask;
        if (empty == 0u) { st.err |= FLAG_CONTACT_OVERFLOW; st.stop = true; return; }
        cpos = 31 - __clz(empty);
        st.fresh |= 1u << cpos;
    }
    slot[cpos] = bo | (code << 28);
    st.mask |= 1u << cpos;
    if (++st.nc > (uint32_t)NC) { st.err |= FLAG_CONTACT_OVERFLOW; st.stop = true; }
}

template <bool FROM_LDS>
__device__ __forceinline__ double4 staged_pos(const DemDev& d, const TopoShared& sh, uint32_t lb, uint32_t sb) {
    if constexpr (FROM_LDS) return sh.pos[lb];
    else return spos(d, d.sys, sb);
}

// Walks the 27 cells of every home particle of the tile: 9 rows (z, y order),
// each row the contiguous run of cells x-1, x, x+1, within a cell in sorted
// order -- the candidate order of src/contactsearch.cuh:340-353.  Candidates
// come from LDS (FROM_LDS) or from HBM.  The hot loop only rejects pairs whose
// squared distance exceeds (ra+rb)^2 by more than rounding; the exact test
// sqrt(d2) - (ra+rb) < 0 runs on the few that remain.
template <bool FROM_LDS>
__device__ __forceinline__ void topo_search(const DemDev& d, const TopoShared& sh, int W, int H, int nxh,
                                            int nyh) {
    uint32_t home_total = 0;
    for (int hr = 0; hr < nyh; ++hr) {
        const int e0 = (1 * H + hr + 1) * W + 1;
        home_total += sh.cstart[e0 + nxh] - sh.cstart[e0];
    }
    for (uint32_t h = threadIdx.x; h < home_total; h += BLOCK) {
        int hr = 0, e0 = 0;
        uint32_t li = 0, rem = h;
        for (; hr < nyh; ++hr) {
            e0 = (1 * H + hr + 1) * W + 1;
            const uint32_t n_row = sh.cstart[e0 + nxh] - sh.cstart[e0];
            if (rem < n_row) { li = sh.cstart[e0] + rem; break; }
            rem -= n_row;
        }
        int eh = e0;
        while (sh.cstart[eh + 1] <= li) ++eh;
        const int colh = eh - (1 * H + hr + 1) * W;  // 1..nxh
        const uint32_t s = sh.cglob[eh] + (li - sh.cstart[eh]);
        const double4 xa = staged_pos<FROM_LDS>(d, sh, li, s);
        const double ra = xa.w;
        const SlotRow slot = slot_row(d, s);
        SlotState st;
        st.mask = d.ro.cmask[d.perm[s]];
        st.fresh = 0; st.nc = 0; st.err = 0; st.stop = false;
        for (int lay = 0; lay < 3 && !st.stop; ++lay) {
            for (int dy = 0; dy < 3 && !st.stop; ++dy) {
                const int e = (lay * H + hr + dy) * W + colh - 1;
                const uint32_t b0 = sh.cstart[e], b3 = sh.cstart[e + 3];
                if (b0 == b3) continue;
                const uint32_t codes = (uint32_t)sh.ccode[e] | ((uint32_t)sh.ccode[e + 1] << 8) |
                                       ((uint32_t)sh.ccode[e + 2] << 16);
                for (int c = 0; c < 3 && !st.stop; ++c) {
                    const uint32_t lo = c == 0 ? b0 : sh.cstart[e + c];
                    const uint32_t hi = c == 2 ? b3 : sh.cstart[e + c + 1];
                    if (lo == hi) continue;
                    const uint32_t code = (codes >> (8 * c)) & 0xffu;
                    double dmx, dmy;
                    decode_image(d.sys, code, dmx, dmy);
                    const uint32_t gb = sh.cglob[e + c] - lo;
                    for (uint32_t lb = lo; lb < hi; ++lb) {
                        const double4 xb = staged_pos<FROM_LDS>(d, sh, lb, gb + lb);
                        const double ex = (xa.x - xb.x) + dmx;
                        const double ey = (xa.y - xb.y) + dmy;
                        const double ez = xa.z - xb.z;
                        // (ez + 0.0)^2 == ez^2, so d2 equals dot(xab, xab) of the exact test
                        const double d2 = ex * ex + ey * ey + ez * ez;
                        const double rsum = ra + xb.w;
                        if (__builtin_expect(d2 <= rsum * rsum * 1.0000001, 0) && lb != li) {
                            // exact test of src/contactsearch.cuh:242-248 (double sqrt)
                            if (sqrt(d2) - rsum < 0.0) {
                                slot_insert(slot, st, d.sid[gb + lb], code);
                                if (st.stop) break;
                            }
                        }
                    }
                }
            }
        }
        d.tmask[s] = st.mask;
        d.tfresh[s] = st.fresh;
        if (st.err) atomicOr(d.flags, st.err);
    }
}

__global__ __launch_bounds__(BLOCK) void k_topo(DemDev d) {
    __shared__ TopoShared sh;
    const Sys& S = d.sys;
    const uint32_t bt = xcd_block();
    const uint32_t txi = bt % d.tiles_x, rest = bt / d.tiles_x;
    const uint32_t tyi = rest % d.tiles_y, tz = rest / d.tiles_y;
    const int nx = (int)S.num[0], ny = (int)S.num[1], nz = (int)S.num[2];
    const int x0 = (int)(txi * d.tile_x), y0 = (int)(tyi * d.tile_y);
    const int nxh = min((int)d.tile_x, nx - x0), nyh = min((int)d.tile_y, ny - y0);
    const int W = nxh + 2, H = nyh + 2;
    const int ncell = 3 * H * W;  // <= TOPO_MAX_CELLS (host-checked)

    // 1. staged cells: global run, image code, count -> LDS offsets
    uint32_t cnt2[2] = {0u, 0u};
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const int e = 2 * (int)threadIdx.x + k;
        if (e >= ncell) continue;
        const int col = e % W, rr = e / W, row = rr % H, lay = rr / H;
        int cx = x0 - 1 + col, cy = y0 - 1 + row;
        const int cz = (int)tz - 1 + lay;
        uint32_t code = 0, g0 = 0, cnt = 0;
        bool ok = cz >= 0 && cz < nz;
        if (ok && (cy < 0 || cy >= ny)) {
            if (S.periodic == 1) { code |= (cy < 0 ? 1u : 2u) << 2; cy = cy < 0 ? ny - 1 : 0; }
            else ok = false;
        }
        if (ok && (cx < 0 || cx >= nx)) {
            if (S.periodic != 0) { code |= cx < 0 ? 1u : 2u; cx = cx < 0 ? nx - 1 : 0; }
            else ok = false;
        }
        if (ok) {
            const uint32_t cid = (uint32_t)cx + (uint32_t)cy * S.num[0] + (S.num[0] * S.num[1]) * (uint32_t)cz;
            g0 = d.off[cid];
            cnt = d.off[cid + 1] - g0;
        }
        sh.cglob[e] = g0;
        sh.ccode[e] = (uint8_t)code;
        cnt2[k] = cnt;
    }
    uint32_t total;
    const uint32_t ex = block_exclusive_scan(cnt2[0] + cnt2[1], sh.scan, total);
    if (2 * (int)threadIdx.x < ncell) sh.cstart[2 * threadIdx.x] = ex;
    if (2 * (int)threadIdx.x + 1 < ncell) sh.cstart[2 * threadIdx.x + 1] = ex + cnt2[0];
    if (threadIdx.x == 0) sh.cstart[ncell] = total;
    __syncthreads();
    const bool use_lds = total <= (uint32_t)TOPO_CAP;

    // 2. stage positions
    if (use_lds) {
        for (uint32_t i = threadIdx.x; i < total; i += BLOCK) {
            int lo = 0, hi = ncell - 1;  // last cell with cstart <= i
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (sh.cstart[mid] <= i) lo = mid; else hi = mid - 1;
            }
            sh.pos[i] = spos(d, S, sh.cglob[lo] + (i - sh.cstart[lo]));
        }
    }
    __syncthreads();

    // 3. home particles: cells (lay 1, rows 1..nyh, cols 1..nxh), row by row
    if (use_lds) topo_search<true>(d, sh, W, H, nxh, nyh);
    else topo_search<false>(d, sh, W, H, nxh, nyh);
}

// One thread per sorted particle; the 27 cells are walked as 9 runs of the
// sorted arrays (cells x-1, x, x+1 of a row have consecutive ids), the same
// candidate order as k_topo, candidates read through L1/L2.  The hot loop
// reads the FP32 copy of the positions and keeps only pairs within
// (r_a + r_b + search_eps), a margin larger than the FP32 rounding of the
// distance, so it never drops an overlap; the reference's exact test
// sqrt(d2) - (r_a + r_b) < 0 then runs in FP64 on the few that remain
// (rows_try).  The particle's slot words are cached in LDS from its first
// overlap on and written back once.
struct RowSlots {
    uint32_t mask, fresh, nc, err, dirty;
    bool stop, loaded;
    uint32_t ld;  // stride of the LDS slot column (threads per block)
};

// (Inlined: as a call it had the caller's registers saved to memory around
// it, and the batch below lived there when a variable indexed it: a rebuild of
// the 1,048,576-sphere crystal wrote 3.1 GB and took 1,540 us more than a list
// step, without the batch's part 930, without either 530.)
__device__ __forceinline__ void rows_try(PosView pv, const uint32_t* __restrict__ sid, uint32_t* sw,
                                      SlotRow gslot, RowSlots& st, double4 xa, uint32_t sb, uint32_t code) {
    const double4 xb = pv_pos(pv, sb);
    const uint32_t cx = code & 3u, cy = (code >> 2) & 3u;
    const double dmx = cx == 1u ? pv.Lx : (cx == 2u ? -pv.Lx : 0.0);
    const double dmy = cy == 1u ? pv.Ly : (cy == 2u ? -pv.Ly : 0.0);
    const double ex = (xa.x - xb.x) + dmx, ey = (xa.y - xb.y) + dmy, ez = xa.z - xb.z;
    // ((e + 0.0)^2 == e^2: d2 equals dot(xab, xab) of src/contactsearch.cuh:242-248)
    const double d2 = ex * ex + ey * ey + ez * ez;
    if (!(sqrt(d2) - (xa.w + xb.w) < 0.0)) return;
    if (!st.loaded) {
        for (uint32_t m = st.mask; m; m &= m - 1) {
            const int i = __ffs(m) - 1;
            sw[i * st.ld] = gslot[i];
        }
        st.loaded = true;
    }
    // slot rule of src/contactsearch.cuh:252-271
    const uint32_t bo = sid[sb];
    int cpos = -1;
    for (uint32_t m = st.mask; m; m &= m - 1) {
        const int i = __ffs(m) - 1;
        if ((sw[i * st.ld] & SLOT_IDX_MASK) == bo) { cpos = i; break; }
    }
    if (cpos < 0) {
        const uint32_t empty = ~st.mask;
        if (empty == 0u) { st.err |= FLAG_CONTACT_OVERFLOW; st.stop = true; return; }
        cpos = 31 - __clz(empty);
        st.fresh |= 1u << cpos;
    }
    const uint32_t w = bo | (code << 28);
    if (sw[cpos * st.ld] != w || !((st.mask >> cpos) & 1u)) {  // unchanged kept slots are not written back
        sw[cpos * st.ld] = w;
        st.dirty |= 1u << cpos;
    }
    st.mask |= 1u << cpos;
    if (++st.nc > (uint32_t)NC) { st.err |= FLAG_CONTACT_OVERFLOW; st.stop = true; }
}

// Candidates [lo, hi) of one run with periodic image (dmx, dmy), in batches
// of ROW_BATCH independent loads; overlaps go to rows_try in candidate order.
constexpr int ROW_BATCH = 8;

// With BUILD, the pass also records every candidate within the list reach
// (r_a + r_b + skin, same prefilter margin) in the particle's neighbour list.
template <bool BUILD>
__device__ __forceinline__ void rows_run(const DemDev& d, Words wd, const float4* __restrict__ xf, const Sys& S, uint32_t lo, uint32_t hi, float dmx, float dmy,
                                         uint32_t code, uint32_t s, float4 xaf, float ra_eps, float ra_skin,
                                         double4 xa, uint32_t* sw, SlotRow gslot, RowSlots& st,
                                         uint32_t* list, uint32_t& lcnt) {
    for (uint32_t sb0 = lo; sb0 < hi; sb0 += ROW_BATCH) {
        float4 c[ROW_BATCH];
#pragma unroll
        for (int k = 0; k < ROW_BATCH; ++k)
            c[k] = sb0 + k < hi ? xf[sb0 + k] : make_float4(1e30f, 1e30f, 1e30f, 0.0f);
        uint32_t hits = 0, near = 0;
#pragma unroll
        for (int k = 0; k < ROW_BATCH; ++k) {
            const float ex = (xaf.x - c[k].x) + dmx, ey = (xaf.y - c[k].y) + dmy, ez = xaf.z - c[k].z;
            const float d2 = ex * ex + ey * ey + ez * ez;
            const float rs = ra_eps + c[k].w;
            hits |= d2 <= rs * rs ? 1u << k : 0u;
            if constexpr (BUILD) {
                const float rl = ra_skin + c[k].w;
                near |= d2 <= rl * rl ? 1u << k : 0u;
            }
        }
        if constexpr (BUILD) {
#pragma unroll
            for (int k = 0; k < ROW_BATCH; ++k) {  // (unrolled: see rows_try)
                const uint32_t sb = sb0 + (uint32_t)k;
                if (!((near >> k) & 1u) || sb == s) continue;
                if (lcnt < (uint32_t)NLIST) {
                    list[(size_t)lcnt * d.np] = sb;  // the partner's list index
                    d.nhint[(size_t)lcnt * d.np + s] = 0xffu;  // no slot known yet
                    const float ex = (xaf.x - c[k].x) + dmx, ey = (xaf.y - c[k].y) + dmy, ez = xaf.z - c[k].z;
                    d.nlistg[(size_t)lcnt * d.np + s] = sqrtf(ex * ex + ey * ey + ez * ez) - (xaf.w + c[k].w);
                }
                ++lcnt;
            }
        }
        if (__builtin_expect(hits != 0u, 0)) {
            for (; hits; hits &= hits - 1) {
                const uint32_t sb = sb0 + (uint32_t)(__ffs(hits) - 1);
                if (sb == s) continue;
                rows_try(pos_view(d, S, wd.sorted), d.sid, sw, gslot, st, xa, sb, code);
                if (st.stop) return;
            }
        }
    }
}

// Distance along one axis from the coordinate v to the box of cell t (of n)
// seen through the periodic shift dm (the image of a sphere at c is c - dm),
// widened by mg.  Spheres of the edge cells may lie beyond the grid (cell
// ids clamp), so those cells are open on their outer side.
__device__ __forceinline__ float cell_gap(float v, int t, int n, float o, float cl, float dm, float mg) {
    const float lo = t == 0 ? -INFINITY : o + (float)t * cl - dm - mg;
    const float hi = t == n - 1 ? INFINITY : o + (float)(t + 1) * cl - dm + mg;
    return fmaxf(0.0f, fmaxf(lo - v, v - hi));
}

// Second pass of a list build: the spheres two cells away (the outer shell of
// the 5 x 5 x 5 cells around the particle's cell) within the list reach.  A
// pair two cells apart is more than a cell apart; when a cell is narrower
// than the largest pair plus 0.9 skin such a pair can meet before the next
// rebuild, so the host asks for this pass (list_shell) instead of shrinking
// the rebuild distance to fit the 27 cells.  It does so only when every
// periodic axis has at least 5 cells: no cell is then reached twice.
// Cells whose widened box lies farther than the list reach with the largest
// partner (reach2 = (r_a + eps + skin + r_max)^2, rounded up) hold no list
// entry and are skipped.
struct CellBox {
    float o[3], cl[3], mg, reach2;
};

__device__ __noinline__ void list_shell(const uint32_t* __restrict__ off, const float4* __restrict__ xf,
                                        uint8_t* hint,
                                        uint32_t* list, float* gap, uint32_t np, uint32_t& lcnt, int gx, int gy, int gz, int nx,
                                        int ny, int nz, int periodic, float Lx, float Ly, uint32_t cbase,
                                        float4 xaf, float ra_skin, CellBox cb3) {
    for (int dz = -2; dz <= 2; ++dz) {
        const int tz = gz + dz;
        if (tz < 0 || tz >= nz) continue;
        const float gzz = cell_gap(xaf.z, tz, nz, cb3.o[2], cb3.cl[2], 0.0f, cb3.mg);
        for (int dy = -2; dy <= 2; ++dy) {
            int ty = gy + dy;
            float dmy = 0.0f;
            if (ty < 0 || ty >= ny) {
                if (periodic != 1) continue;
                dmy = ty < 0 ? Ly : -Ly;
                ty = ty < 0 ? ty + ny : ty - ny;
            }
            const float gyy = cell_gap(xaf.y, ty, ny, cb3.o[1], cb3.cl[1], dmy, cb3.mg);
            if (gyy * gyy + gzz * gzz > cb3.reach2) continue;
            for (int dx = -2; dx <= 2; ++dx) {
                if (dx > -2 && dx < 2 && dy > -2 && dy < 2 && dz > -2 && dz < 2) continue;  // the 27 cells
                int tx = gx + dx;
                float dmx = 0.0f;
                if (tx < 0 || tx >= nx) {
                    if (periodic == 0) continue;
                    dmx = tx < 0 ? Lx : -Lx;
                    tx = tx < 0 ? tx + nx : tx - nx;
                }
                const float gxx = cell_gap(xaf.x, tx, nx, cb3.o[0], cb3.cl[0], dmx, cb3.mg);
                if (gxx * gxx + gyy * gyy + gzz * gzz > cb3.reach2) continue;
                const uint32_t c = cbase + (uint32_t)tx + (uint32_t)ty * (uint32_t)nx + (uint32_t)tz * (uint32_t)(nx * ny);
                const uint32_t hi = off[c + 1];
                for (uint32_t sb = off[c]; sb < hi; ++sb) {
                    const float4 cb = xf[sb];
                    const float ex = (xaf.x - cb.x) + dmx, ey = (xaf.y - cb.y) + dmy, ez = xaf.z - cb.z;
                    const float rl = ra_skin + cb.w;
                    const float d2 = ex * ex + ey * ey + ez * ez;
                    if (d2 <= rl * rl) {
                        if (lcnt < (uint32_t)NLIST) {
                            list[(size_t)lcnt * np] = sb;
                            hint[(size_t)lcnt * np] = 0xffu;
                            gap[(size_t)lcnt * np] = sqrtf(d2) - (xaf.w + cb.w);
                        }
                        ++lcnt;
                    }
                }
            }
        }
    }
}

// The search of sorted particle s, its slot words in the LDS column sw of
// stride ld.  BUILD: it also rebuilds the particle's neighbour list.
template <bool BUILD, bool B>
__device__ __forceinline__ void rows_search(const DemDev& d, Words wd, uint32_t s, uint32_t* sw, uint32_t ld) {
    const Sys& S = sys_at<B>(d, s);
    const float4* xfp = xf_sorted(d, wd);
    const int nx = (int)S.num[0], ny = (int)S.num[1], nz = (int)S.num[2];
    const uint32_t key = d.skey[s] - S.cbase;
    const int gx = (int)(key % S.num[0]), gy = (int)((key / S.num[0]) % S.num[1]), gz = (int)(key / (S.num[0] * S.num[1]));
    const uint32_t p = wd.sorted ? d.perm[s] : s;
    double4 xa = d.ro.x[p];
    (void)wrap_xy(S, xa.x, xa.y);
    const float4 xaf = xfp[s];
    const float ra_eps = xaf.w + d.search_eps;
    const float ra_skin = ra_eps + d.list_skin;
    const SlotRow gslot{d.ro.cslot + p, d.np};
    uint32_t* list = BUILD ? d.nlist + s : nullptr;  // entry k at list[k * np]
    uint32_t lcnt = 0;
    // rows of cells farther than any hit (or list entry) can reach are skipped
    CellBox cb3;
    for (int a = 0; a < 3; ++a) {
        cb3.o[a] = (float)S.origo[a];
        cb3.cl[a] = (float)S.cell_len[a];
    }
    cb3.mg = d.cell_margin;
    {
        const float reach = (BUILD ? ra_skin : ra_eps) + d.rmax_f;
        cb3.reach2 = reach * reach * 1.001f;
    }
    RowSlots st;
    st.mask = d.ro.cmask[p];
    st.fresh = 0; st.nc = 0; st.err = 0; st.dirty = 0; st.stop = false; st.loaded = false;
    st.ld = ld;
    for (int dz = -1; dz <= 1 && !st.stop; ++dz) {
        const int tz = gz + dz;
        if (tz < 0 || tz == nz) continue;
        for (int dy = -1; dy <= 1 && !st.stop; ++dy) {
            int ty = gy + dy;
            uint32_t cy = 0;
            if (ty < 0 || ty == ny) {
                if (S.periodic != 1) continue;
                cy = ty < 0 ? 1u : 2u;
                ty = ty < 0 ? ny - 1 : 0;
            }
            {
                const float dmy = cy == 1u ? S.Lf[1] : (cy == 2u ? -S.Lf[1] : 0.0f);
                const float gyy = cell_gap(xaf.y, ty, ny, cb3.o[1], cb3.cl[1], dmy, cb3.mg);
                const float gzz = cell_gap(xaf.z, tz, nz, cb3.o[2], cb3.cl[2], 0.0f, cb3.mg);
                if (gyy * gyy + gzz * gzz > cb3.reach2) continue;
            }
            const uint32_t row = S.cbase + (uint32_t)ty * S.num[0] + (S.num[0] * S.num[1]) * (uint32_t)tz;
            if (gx >= 1 && gx + 1 < nx && cy == 0) {
                // no periodic image anywhere in the run: one contiguous range
                rows_run<BUILD>(d, wd, xfp, S, d.off[row + gx - 1], d.off[row + gx + 2], 0.0f, 0.0f, 0u, s, xaf, ra_eps,
                                ra_skin, xa, sw, gslot, st, list, lcnt);
                continue;
            }
            for (int dx = -1; dx <= 1 && !st.stop; ++dx) {
                int tx = gx + dx;
                uint32_t cx = 0;
                if (tx < 0 || tx == nx) {
                    if (S.periodic == 0) continue;
                    cx = tx < 0 ? 1u : 2u;
                    tx = tx < 0 ? nx - 1 : 0;
                }
                const float dmx = cx == 1u ? S.Lf[0] : (cx == 2u ? -S.Lf[0] : 0.0f);
                const float dmy = cy == 1u ? S.Lf[1] : (cy == 2u ? -S.Lf[1] : 0.0f);
                rows_run<BUILD>(d, wd, xfp, S, d.off[row + tx], d.off[row + tx + 1], dmx, dmy, cx | (cy << 2), s, xaf,
                                ra_eps, ra_skin, xa, sw, gslot, st, list, lcnt);
            }
        }
    }
    for (uint32_t m = st.dirty; m; m &= m - 1) {
        const int i = __ffs(m) - 1;
        gslot[i] = sw[i * st.ld];
    }
    d.tmask[s] = st.mask;
    d.tfresh[s] = st.fresh;
    if (st.err) atomicOr(d.flags, st.err);
    if constexpr (BUILD) {  // list index = this sorted position
        if (d.list_shell && !st.stop)
            list_shell(d.off, xfp, d.nhint + s, list, d.nlistg + s, d.np, lcnt, gx, gy, gz, nx, ny, nz, S.periodic, S.Lf[0],
                       S.Lf[1], S.cbase, xaf, ra_skin, cb3);
        d.ncnt[s] = lcnt < (uint32_t)NLIST ? lcnt : (uint32_t)NLIST;
        d.nfree[s] = 0.0f;
        d.xref[s] = make_float4(xaf.x, xaf.y, xaf.z, 0.0f);
        d.slidx[s] = s;
        d.linv[s] = s;
        if (lcnt > (uint32_t)NLIST || st.stop) atomicOr(&d.fw[FW_REBUILD], 1u);  // list unusable: rebuild next step
    }
}

// BUILD (search mode 5): runs only on steps whose neighbour lists must be
// rebuilt.
template <bool BUILD, bool B>
__global__ __launch_bounds__(BLOCK) void k_topo_rows(DemDev d) {
    extern __shared__ uint32_t sw_all[];  // NC x blockDim: slot i of thread t at [i * blockDim + t]
    const Words wd = words_of(d);
    if constexpr (BUILD) {
        if (!wd.rebuild) return;
    } else if (lead_walls<B>(d)) return;
    if (BUILD && blockIdx.x == 0u && threadIdx.x == 0u) d.nstate[NSTATE_ALIGNED] = 1u;
    const uint32_t s = work_block(d) * blockDim.x + threadIdx.x;
    if (s < d.np) rows_search<BUILD, B>(d, wd, s, sw_all + threadIdx.x, blockDim.x);
}

// ---------------------------------------------------- half-shell search
// Every unordered pair is tested once, by its lower sorted position, with the
// same FP32 prefilter and FP64 exact test as k_topo_rows (the exact test is
// symmetric: swapping a and b negates every component of the distance
// exactly).  An overlap is recorded in both particles' hit lists under its
// key in each one's reference visiting order -- cell offset index
// (dz+1)*9 + (dy+1)*3 + (dx+1), then sorted position (src/contactsearch.cuh:
// 340-353) -- and k_topo_apply replays each list in key order through the
// slot rule.
constexpr uint32_t NO_SPLIT = 0xffffffffu;

__device__ __noinline__ uint32_t half_hit(PosView pv, uint32_t* hcnt, uint64_t* hits, double4 xa, uint32_t s,
                                          uint32_t sb, uint32_t vi, uint32_t code) {
    const double4 xb = pv_pos(pv, sb);
    const uint32_t cx = code & 3u, cy = (code >> 2) & 3u;
    const double dmx = cx == 1u ? pv.Lx : (cx == 2u ? -pv.Lx : 0.0);
    const double dmy = cy == 1u ? pv.Ly : (cy == 2u ? -pv.Ly : 0.0);
    const double ex = (xa.x - xb.x) + dmx, ey = (xa.y - xb.y) + dmy, ez = xa.z - xb.z;
    const double d2 = ex * ex + ey * ey + ez * ez;
    if (!(sqrt(d2) - (xa.w + xb.w) < 0.0)) return 0u;
    const uint32_t rx = cx == 1u ? 2u : (cx == 2u ? 1u : 0u), ry = cy == 1u ? 2u : (cy == 2u ? 1u : 0u);
    const uint32_t rcode = rx | (ry << 2);
    uint32_t err = 0;
    const uint32_t k = atomicAdd(&hcnt[s], 1u);
    if (k < (uint32_t)NC) hits[(size_t)s * NC + k] = ((uint64_t)vi << 40) | ((uint64_t)code << 32) | sb;
    else err |= FLAG_CONTACT_OVERFLOW;
    const uint32_t k2 = atomicAdd(&hcnt[sb], 1u);
    if (k2 < (uint32_t)NC) hits[(size_t)sb * NC + k2] = ((uint64_t)(26u - vi) << 40) | ((uint64_t)rcode << 32) | s;
    else err |= FLAG_CONTACT_OVERFLOW;
    return err;
}

// Candidates (s, hi) of one run; the run's cells start their offset index at
// vi0 and advance at sorted positions m1 and m2.
__device__ __forceinline__ uint32_t half_run(const DemDev& d, const float4* __restrict__ xf, const Sys& S, uint32_t lo, uint32_t hi, uint32_t m1, uint32_t m2,
                                             uint32_t vi0, float dmx, float dmy, uint32_t code, uint32_t s,
                                             float4 xaf, float ra_eps, double4 xa) {
    uint32_t err = 0;
    if (lo <= s) lo = s + 1;
    for (uint32_t sb0 = lo; sb0 < hi; sb0 += ROW_BATCH) {
        float4 c[ROW_BATCH];
#pragma unroll
        for (int k = 0; k < ROW_BATCH; ++k)
            c[k] = sb0 + k < hi ? xf[sb0 + k] : make_float4(1e30f, 1e30f, 1e30f, 0.0f);
        uint32_t hits = 0;
#pragma unroll
        for (int k = 0; k < ROW_BATCH; ++k) {
            const float ex = (xaf.x - c[k].x) + dmx, ey = (xaf.y - c[k].y) + dmy, ez = xaf.z - c[k].z;
            const float d2 = ex * ex + ey * ey + ez * ez;
            const float rs = ra_eps + c[k].w;
            hits |= d2 <= rs * rs ? 1u << k : 0u;
        }
        if (__builtin_expect(hits != 0u, 0)) {
            for (; hits; hits &= hits - 1) {
                const uint32_t sb = sb0 + (uint32_t)(__ffs(hits) - 1);
                const uint32_t vi = vi0 + (sb >= m1 ? 1u : 0u) + (sb >= m2 ? 1u : 0u);
                err |= half_hit(pos_view(d, S, true), d.hcnt, d.hits, xa, s, sb, vi, code);
            }
        }
    }
    return err;
}

template <bool B>
__global__ __launch_bounds__(BLOCK) void k_topo_half(DemDev d) {
    const uint32_t s = xcd_block() * blockDim.x + threadIdx.x;
    if (s >= d.np) return;
    const Sys& S = sys_at<B>(d, s);
    const int nx = (int)S.num[0], ny = (int)S.num[1], nz = (int)S.num[2];
    const uint32_t key = d.skey[s] - S.cbase;
    const int gx = (int)(key % S.num[0]), gy = (int)((key / S.num[0]) % S.num[1]), gz = (int)(key / (S.num[0] * S.num[1]));
    const double4 xa = spos(d, S, s);
    const float4* xfp = xf_sorted(d, words_of(d));
    const float4 xaf = xfp[s];
    const float ra_eps = xaf.w + d.search_eps;
    uint32_t err = 0;
    for (int dz = -1; dz <= 1; ++dz) {
        const int tz = gz + dz;
        if (tz < 0 || tz == nz) continue;
        for (int dy = -1; dy <= 1; ++dy) {
            int ty = gy + dy;
            uint32_t cy = 0;
            if (ty < 0 || ty == ny) {
                if (S.periodic != 1) continue;
                cy = ty < 0 ? 1u : 2u;
                ty = ty < 0 ? ny - 1 : 0;
            }
            const uint32_t row = S.cbase + (uint32_t)ty * S.num[0] + (S.num[0] * S.num[1]) * (uint32_t)tz;
            const uint32_t vrow = (uint32_t)((dz + 1) * 9 + (dy + 1) * 3);
            if (gx >= 1 && gx + 1 < nx && cy == 0) {
                const uint32_t hi = d.off[row + gx + 2];
                if (hi <= s + 1) continue;  // the whole run lies at or below s
                err |= half_run(d, xfp, S, d.off[row + gx - 1], hi, d.off[row + gx], d.off[row + gx + 1], vrow, 0.0f, 0.0f,
                                0u, s, xaf, ra_eps, xa);
                continue;
            }
            for (int dx = -1; dx <= 1; ++dx) {
                int tx = gx + dx;
                uint32_t cx = 0;
                if (tx < 0 || tx == nx) {
                    if (S.periodic == 0) continue;
                    cx = tx < 0 ? 1u : 2u;
                    tx = tx < 0 ? nx - 1 : 0;
                }
                const float dmx = cx == 1u ? S.Lf[0] : (cx == 2u ? -S.Lf[0] : 0.0f);
                const float dmy = cy == 1u ? S.Lf[1] : (cy == 2u ? -S.Lf[1] : 0.0f);
                err |= half_run(d, xfp, S, d.off[row + tx], d.off[row + tx + 1], NO_SPLIT, NO_SPLIT, vrow + (uint32_t)(dx + 1),
                                dmx, dmy, cx | (cy << 2), s, xaf, ra_eps, xa);
            }
        }
    }
    if (err) atomicOr(d.flags, err);
}

// Replays each particle's hits in visiting-key order through the slot rule
// (src/contactsearch.cuh:252-271); the keys (at most NC) are insertion-sorted
// in place, the slot words cached in LDS.
constexpr int APPLY_BLOCK = 128;

// Copies the occupied slot words of a row into the particle's LDS column
// (stride LD), eight independent loads at a time.
template <int LD>
__device__ __forceinline__ void stage_slots(SlotRow gslot, uint32_t mask, uint32_t* sw) {
    constexpr int G = 8;
    for (uint32_t m = mask; m;) {
        int si[G];
        uint32_t w[G];
        int cnt = 0;
#pragma unroll
        for (int k = 0; k < G; ++k) {
            si[k] = m ? __ffs(m) - 1 : 0;
            if (m) { m &= m - 1; ++cnt; }
        }
#pragma unroll
        for (int k = 0; k < G; ++k) w[k] = k < cnt ? gslot[si[k]] : 0u;
#pragma unroll
        for (int k = 0; k < G; ++k)
            if (k < cnt) sw[si[k] * LD] = w[k];
    }
}

// Applies the n (<= NC) hit keys k of sorted particle s through the slot
// rule as if in key order.  A partner occurs at most once among the hits, so
// a hit whose partner already holds a slot lands in that slot whatever the
// order; only the new contacts take empty slots in key order, and only they
// are sorted.  sw is the particle's LDS column of slot words (stride
// APPLY_BLOCK).
__device__ __forceinline__ void apply_hits(const DemDev& d, uint32_t s, uint64_t* k, uint32_t n, uint32_t mask0,
                                           uint32_t* sw, uint32_t err) {
    const SlotRow gslot = slot_row(d, s);
    stage_slots<APPLY_BLOCK>(gslot, mask0, sw);
    uint32_t mask = mask0, fresh = 0, dirty = 0, nnew = 0;
    for (uint32_t h = 0; h < n; ++h) {
        const uint64_t v = k[h];
        const uint32_t sb = (uint32_t)(v & 0xffffffffu), code = (uint32_t)(v >> 32) & 15u;
        const uint32_t bo = d.sid[sb];
        int cpos = -1;
        for (uint32_t m = mask0; m; m &= m - 1) {
            const int i = __ffs(m) - 1;
            if ((sw[i * APPLY_BLOCK] & SLOT_IDX_MASK) == bo) { cpos = i; break; }
        }
        if (cpos >= 0) {  // kept; written back only if its image changed
            const uint32_t w = bo | (code << 28);
            if (sw[cpos * APPLY_BLOCK] != w) {
                sw[cpos * APPLY_BLOCK] = w;
                dirty |= 1u << cpos;
            }
        } else {
            k[nnew++] = v;  // compacted in place (nnew <= h)
        }
    }
    for (uint32_t i = 1; i < nnew; ++i) {
        const uint64_t v = k[i];
        uint32_t j = i;
        while (j > 0 && k[j - 1] > v) { k[j] = k[j - 1]; --j; }
        k[j] = v;
    }
    for (uint32_t h = 0; h < nnew; ++h) {
        const uint64_t v = k[h];
        const uint32_t sb = (uint32_t)(v & 0xffffffffu), code = (uint32_t)(v >> 32) & 15u;
        const uint32_t empty = ~mask;
        if (empty == 0u) { err |= FLAG_CONTACT_OVERFLOW; break; }
        const int cpos = 31 - __clz(empty);
        fresh |= 1u << cpos;
        sw[cpos * APPLY_BLOCK] = d.sid[sb] | (code << 28);
        dirty |= 1u << cpos;
        mask |= 1u << cpos;
    }
    for (uint32_t m = dirty; m; m &= m - 1) {
        const int i = __ffs(m) - 1;
        gslot[i] = sw[i * APPLY_BLOCK];
    }
    d.tmask[s] = mask;
    d.tfresh[s] = fresh;
    if (err) atomicOr(d.flags, err);
}

template <bool B>
__global__ __launch_bounds__(APPLY_BLOCK) void k_topo_apply(DemDev d) {
    __shared__ uint32_t sw_all[NC * APPLY_BLOCK];
    if (lead_walls<B>(d)) return;
    const uint32_t s = work_block(d) * APPLY_BLOCK + threadIdx.x;
    if (s >= d.np) return;
    const uint32_t cnt = d.hcnt[s];
    const uint32_t mask0 = d.ro.cmask[d.perm[s]];
    if (cnt != 0u) d.hcnt[s] = 0u;  // zero for the next search
    if (cnt == 0u) {
        d.tmask[s] = mask0;
        d.tfresh[s] = 0u;
        return;
    }
    const uint32_t n = cnt < (uint32_t)NC ? cnt : (uint32_t)NC;
    apply_hits(d, s, d.hits + (size_t)s * NC, n, mask0, sw_all + threadIdx.x, 0u);
}

// ------------------------------------------------- neighbour-list search
// Search mode 5.  k_topo_rows<true> rebuilds, per particle, the list of every
// sphere within r_a + r_b + skin (original indices) and keeps the position of
// the build; the force kernel requests a rebuild once any sphere has moved
// more than list_lim since.  list_lim is at most 0.45 skin, so no pair
// outside the reach can overlap before the rebuild (both spheres would have
// had to close a gap of more than skin).  A pair more than a cell apart at the
// build cannot overlap either: the build also scans the cells two away
// (list_shell) when a cell leaves less room than 0.9 skin beyond the largest
// pair, and where it cannot (a periodic axis of fewer than 5 cells) list_lim
// is at most half that room.  Testing the list pairs then finds exactly the
// overlaps the full search finds.
// The overlaps are keyed by the reference's visiting order -- the offset of
// the partner's cell (periodic wrap included, as findDistMod resolves it,
// src/contactsearch.cuh:12-74) and its sorted position -- and replayed
// through the slot rule in that order.
__device__ __forceinline__ bool cell_offset(int g, int b, int n, bool wrap, int& dxo, uint32_t& code) {
    const int raw = b - g;
    code = 0u;
    if (raw >= -1 && raw <= 1) { dxo = raw; return true; }
    if (wrap && g == 0 && b == n - 1) { dxo = -1; code = 1u; return true; }   // x - 1 wraps to n - 1: +L
    if (wrap && g == n - 1 && b == 0) { dxo = 1; code = 2u; return true; }    // x + 1 wraps to 0: -L
    return false;
}

constexpr int LIST_BATCH = 4;


// Cell coordinates of a system-local cell id (x fastest, then y, then z).
__device__ __forceinline__ void cell_xyz(const Sys& S, uint32_t key, int& gx, int& gy, int& gz) {
    const uint32_t z = fdiv(key, S.div_xy), r = key - z * S.div_xy.d, y = fdiv(r, S.div_x);
    gx = (int)(r - y * S.div_x.d);
    gy = (int)y;
    gz = (int)z;
}

// Full FP64 treatment of one list partner that passed the prefilter: its cell
// offset and image as the reference's search would reach it and the exact
// overlap test; returns the hit key, or 0 for no overlap (a real key is
// never 0: its sorted position differs from the particle's own).
__device__ __forceinline__ uint64_t list_pair(const Sys& S, uint32_t sb, uint32_t kb, double4 x, double4 xa,
                                              int gx, int gy, int gz) {
    int bx, by, bz, dx, dy, dz;
    uint32_t cx, cy, cz;
    cell_xyz(S, kb, bx, by, bz);
    if (!cell_offset(gz, bz, (int)S.num[2], false, dz, cz)) return 0ull;
    if (!cell_offset(gy, by, (int)S.num[1], S.periodic == 1, dy, cy)) return 0ull;
    if (!cell_offset(gx, bx, (int)S.num[0], S.periodic != 0, dx, cx)) return 0ull;
    const uint32_t code = cx | (cy << 2);
    (void)wrap_xy(S, x.x, x.y);
    const double dmx = cx == 1u ? S.L[0] : (cx == 2u ? -S.L[0] : 0.0);
    const double dmy = cy == 1u ? S.L[1] : (cy == 2u ? -S.L[1] : 0.0);
    const double ex = (xa.x - x.x) + dmx, ey = (xa.y - x.y) + dmy, ez = xa.z - x.z;
    const double d2 = ex * ex + ey * ey + ez * ez;
    if (!(sqrt(d2) - (xa.w + x.w) < 0.0)) return 0ull;  // exact test of src/contactsearch.cuh:242-248
    const uint32_t vi = (uint32_t)((dz + 1) * 9 + (dy + 1) * 3 + (dx + 1));
    return ((uint64_t)vi << 40) | ((uint64_t)code << 32) | sb;
}

// An overlap whose partner already holds a slot is applied on the spot (its
// slot does not depend on the order, a partner occurs once); the others are
// collected and given empty slots in key order at the end.  Each list entry
// keeps the slot its partner was last found in, with the partner's original
// index (both written when the search finds the partner in a slot; a build
// marks them unknown): one slot-word compare confirms the slot, and only a
// stale or unknown hint scans the occupied slots.
// Held contacts are skipped outright where the search could only rewrite
// their slot word unchanged.  That is so when no sphere crossed a periodic
// face in the last step: the image through which two overlapping spheres
// meet changes only when one of them wraps, and the word was written (or
// confirmed) by the last step's search, while the pair overlapped.  It is
// also so, in any step, when the word carries no periodic image and the
// particle's cell is off the periodic faces: any overlap the search finds
// with that partner has no image either (and one it does not find leaves
// the word as it is).  Skipped entries are not counted; a contact overflow is
// still caught when a new contact finds no empty slot.
// FREE (one lane a sphere): the whole list of a particle with contacts is
// passed over where its entries cannot matter: a search leaves in nfree the
// smallest gap of the entries whose partner holds no slot (negative if one of
// the slots carries a periodic image; 0 if some gap could close before the
// lists are built again).  Until a contact of the particle ends, which the
// force phase notes there, those gaps stay the only way to a new contact.  (Kept
// by chains of one lane a sphere alone: stages may give a slot an image without
// a word of it here, so the first chain after them starts from 0s, and quads
// neither read nor write it -- a handle's spheres, and with them its lanes a
// sphere, are the same from open to close.)  A
// dense packing at rest then reads 4 bytes of search a sphere instead of 13 a
// list entry and its slot words: crystal of 1,048,576 spheres 424 -> 394 us a
// step, mixed precision 332 -> 293.  A particle without contacts has a short
// list, and four lanes a sphere are bound by the launch: both lost 2 to 4 % by
// the extra load and test.
__device__ __forceinline__ bool list_free(float nfree, float dfar, bool wraps, bool skip_held) {
    return (wraps ? nfree : fabsf(nfree)) > dfar && (!wraps || skip_held);
}
struct Slots {
    uint32_t mask, fresh;  // occupied, and taken from empty by this step's search
};
template <bool B, int LD, bool FREE>
__device__ __forceinline__ Slots list_search(const DemDev& d, Words wd, uint32_t s, uint32_t* sw) {
    const Sys& S = sys_at<B>(d, s);
    const float4* xf = xf_sorted(d, wd);
    const uint32_t p = wd.sorted ? d.perm[s] : s;
    const float4 xaf = xf[s];
    const float ra_eps = xaf.w + d.search_eps;
    const uint32_t li = d.slidx[s];
    const uint32_t* list = d.nlist + li;  // entry k at list[k * np]
    uint8_t* hint = d.nhint + li;
    uint32_t* lorig = d.nlo + li;
    const uint32_t nl = d.ncnt[li];
    const uint32_t mask0 = d.ro.cmask[p];
    const bool px = S.periodic != 0, py = S.periodic == 1;
    uint64_t* hk = d.hits + (size_t)s * NC;
    uint32_t n = 0, nnew = 0, err = 0, dirty = 0;
    bool have_a = false;
    double4 xa = make_double4(0.0, 0.0, 0.0, 0.0);
    int gx = 0, gy = 0, gz = 0;
    bool have_cell = false;
    bool skip_held = false;
    const bool no_wraps = !wd.wrap;
    const uint32_t held_bits = no_wraps ? SLOT_IDX_MASK : 0xffffffffu;  // with wraps: the word must carry no image
    const SlotRow gslot{d.ro.cslot + p, d.np};
    if (mask0) {
        skip_held = no_wraps;
        if (!no_wraps) {
            cell_xyz(S, d.skey[s] - S.cbase, gx, gy, gz);
            have_cell = true;
            skip_held = (!px || (gx > 0 && gx < (int)S.num[0] - 1)) && (!py || (gy > 0 && gy < (int)S.num[1] - 1));
        }
    }
    // A pair whose gap at the build exceeds the two spheres' displacements
    // since then cannot overlap now: skip it without touching the partner's
    // record (margins of three FP32 prefilter widths for the rounding of the
    // gap and of the displacements)
    const float da = d.ldisp[li] + 3.0f * d.search_eps;
    // No sphere has moved more than list_lim since the build (a step after
    // one that did rebuilds the lists instead): a gap beyond this cannot
    // close, whatever the partner's displacement, which is then not read.
    const float dfar = da + d.list_lim + 3.0f * d.search_eps;
    const float was_free = FREE && mask0 ? d.nfree[li] : 0.0f;
    if (FREE && list_free(was_free, dfar, !no_wraps, skip_held)) return {mask0, 0u};
    if (mask0) stage_slots<LD>(gslot, mask0, sw);
    float gfree = 1e30f;
    bool moved_in = false;  // a partner without the held test was found in a slot
    const float* gap = d.nlistg + li;
    // the next batch's entries are loaded while the current one is processed
    uint32_t qlb[LIST_BATCH], qhb[LIST_BATCH], qlw[LIST_BATCH];
    float qg[LIST_BATCH];
    auto fetch = [&](uint32_t i0) {
#pragma unroll
        for (int k = 0; k < LIST_BATCH; ++k) {
            const bool in = i0 + k < nl;
            qlb[k] = in ? list[(size_t)(i0 + k) * d.np] : li;
            qg[k] = in ? gap[(size_t)(i0 + k) * d.np] : 1e30f;
            qhb[k] = in && mask0 ? hint[(size_t)(i0 + k) * d.np] : 0xffu;
            qlw[k] = in && mask0 && skip_held ? lorig[(size_t)(i0 + k) * d.np] : 0xffffffffu;
        }
    };
    fetch(0);
    for (uint32_t i0 = 0; i0 < nl; i0 += LIST_BATCH) {
        uint32_t lb[LIST_BATCH], sb[LIST_BATCH], hb[LIST_BATCH], lw[LIST_BATCH];
        float g[LIST_BATCH];
        float4 c[LIST_BATCH];
#pragma unroll
        for (int k = 0; k < LIST_BATCH; ++k) {
            lb[k] = qlb[k];
            g[k] = qg[k];
            hb[k] = qhb[k];
            lw[k] = qlw[k];
        }
        if (i0 + LIST_BATCH < nl) fetch(i0 + LIST_BATCH);
        uint32_t held = 0, near = 0;
        if (mask0) {
#pragma unroll
            for (int k = 0; k < LIST_BATCH; ++k)
                held |= hb[k] < 32u && ((mask0 >> hb[k]) & 1u) && (sw[(hb[k] & 31u) * LD] & held_bits) == lw[k]
                            ? 1u << k : 0u;
        }
#pragma unroll
        for (int k = 0; k < LIST_BATCH && FREE; ++k) gfree = (held >> k) & 1u ? gfree : fminf(gfree, g[k]);
#pragma unroll
        for (int k = 0; k < LIST_BATCH; ++k)
            near |= !((held >> k) & 1u) && g[k] <= dfar && g[k] <= da + d.ldisp[lb[k]] ? 1u << k : 0u;
        if (near == 0u) continue;
#pragma unroll
        for (int k = 0; k < LIST_BATCH; ++k) sb[k] = (near >> k) & 1u ? d.linv[lb[k]] : s;
#pragma unroll
        for (int k = 0; k < LIST_BATCH; ++k) c[k] = xf[sb[k]];
        // FP32 prefilter at the minimum image (an overlap is always closer
        // than half a period), the same margin as the cell search
        uint32_t pass = 0;
#pragma unroll
        for (int k = 0; k < LIST_BATCH; ++k) {
            float ex = xaf.x - c[k].x, ey = xaf.y - c[k].y;
            const float ez = xaf.z - c[k].z;
            if (px) ex -= S.Lf[0] * rintf(ex / S.Lf[0]);
            if (py) ey -= S.Lf[1] * rintf(ey / S.Lf[1]);
            const float d2 = ex * ex + ey * ey + ez * ez;
            const float rs = ra_eps + c[k].w;
            pass |= ((near >> k) & 1u) && d2 <= rs * rs ? 1u << k : 0u;
        }
        if (pass == 0u) continue;
        if (!have_a) {
            xa = d.ro.x[p];
            (void)wrap_xy(S, xa.x, xa.y);
            if (!have_cell) cell_xyz(S, d.skey[s] - S.cbase, gx, gy, gz);
            have_a = true;
        }
        // the batch's keys, FP64 positions and original indices, independent loads
        uint32_t kb[LIST_BATCH], bo[LIST_BATCH];
        double4 xb[LIST_BATCH];
#pragma unroll
        for (int k = 0; k < LIST_BATCH; ++k) {
            kb[k] = d.skey[sb[k]];
            xb[k] = d.ro.x[wd.sorted ? d.perm[sb[k]] : sb[k]];
            bo[k] = d.sid[sb[k]];
        }
#pragma unroll
        for (int k = 0; k < LIST_BATCH; ++k) {
            if (!((pass >> k) & 1u)) continue;
            const uint64_t v = list_pair(S, sb[k], kb[k] - S.cbase, xb[k], xa, gx, gy, gz);
            if (v == 0ull) continue;
            ++n;
            int cpos = -1;
            if (hb[k] < 32u && ((mask0 >> hb[k]) & 1u) && (sw[(hb[k] & 31u) * LD] & SLOT_IDX_MASK) == bo[k]) {
                cpos = (int)hb[k];
            } else {
                for (uint32_t m = mask0; m; m &= m - 1) {
                    const int i = __ffs(m) - 1;
                    if ((sw[i * LD] & SLOT_IDX_MASK) == bo[k]) { cpos = i; break; }
                }
                if (cpos >= 0) {  // the entry's hint and partner, written together
                    hint[(size_t)(i0 + k) * d.np] = (uint8_t)cpos;
                    lorig[(size_t)(i0 + k) * d.np] = bo[k];
                }
            }
            if (cpos >= 0) {  // kept; written back only if its image changed
                moved_in = true;
                const uint32_t w = bo[k] | ((uint32_t)(v >> 32) & 15u) << 28;
                if (sw[cpos * LD] != w) {
                    sw[cpos * LD] = w;
                    dirty |= 1u << cpos;
                }
            } else if (nnew < (uint32_t)NC) {
                hk[nnew++] = v;
            }
        }
    }
    if (n > (uint32_t)NC) err |= FLAG_CONTACT_OVERFLOW;
    auto leave = [&](uint32_t mask) {
        if (!FREE || mask0 == 0u) return;
        uint32_t images = 0u;
        const bool free = gfree > dfar && !moved_in;
        if (free)
            for (uint32_t m = mask; m; m &= m - 1) images |= sw[(__ffs(m) - 1) * LD] & ~SLOT_IDX_MASK;
        const float now = !free ? 0.0f : images ? -gfree : gfree;
        if (now != was_free) d.nfree[li] = now;
    };
    if (!have_a) {
        leave(mask0);
        return {mask0, 0u};
    }
    // new contacts: empty slots in key order
    for (uint32_t i = 1; i < nnew; ++i) {
        const uint64_t v = hk[i];
        uint32_t j = i;
        while (j > 0 && hk[j - 1] > v) { hk[j] = hk[j - 1]; --j; }
        hk[j] = v;
    }
    uint32_t mask = mask0, fresh = 0;
    for (uint32_t h = 0; h < nnew; ++h) {
        const uint64_t v = hk[h];
        const uint32_t empty = ~mask;
        if (empty == 0u) { err |= FLAG_CONTACT_OVERFLOW; break; }
        const int cpos = 31 - __clz(empty);
        fresh |= 1u << cpos;
        sw[cpos * LD] = d.sid[(uint32_t)(v & 0xffffffffu)] | ((uint32_t)(v >> 32) & 15u) << 28;
        dirty |= 1u << cpos;
        mask |= 1u << cpos;
    }
    for (uint32_t m = dirty; m; m &= m - 1) {
        const int i = __ffs(m) - 1;
        gslot[i] = sw[i * LD];
    }
    leave(mask);
    if (err) atomicOr(d.flags, err);
    return {mask, fresh};
}

template <bool B>
__global__ __launch_bounds__(APPLY_BLOCK, 4) void k_list_search(DemDev d) {  // four waves per SIMD: <= 128 VGPRs
    __shared__ uint32_t sw_all[NC * APPLY_BLOCK];
    if (lead_walls<B>(d)) return;
    const Words wd = words_of(d);
    if (wd.rebuild) return;  // k_topo_rows<true> rebuilds the lists this step
    const uint32_t s = work_block(d) * APPLY_BLOCK + threadIdx.x;
    if (s < d.np) {
        const Slots r = list_search<B, APPLY_BLOCK, false>(d, wd, s, sw_all + threadIdx.x);
        d.tmask[s] = r.mask;
        d.tfresh[s] = r.fresh;
    }
}

// One wavefront per cell.  The candidates of the cell's 27-cell neighbourhood,
// in the reference's visiting order (z, y, x cells, sorted order within a
// cell; src/contactsearch.cuh:340-353), are up to 27 runs of the sorted
// arrays; candidate t of the concatenation sits in lane t % 64 of chunk
// t / 64, in registers for the first SEARCH_REG_CHUNKS chunks.  Each member of
// the cell tests all candidates at once, one lane per candidate, and applies
// the overlaps (a ballot) in lane order, i.e. in the serial loop's order.
// While a member is processed its 32 slot words sit in lanes 0..31, so the
// slot rule (src/contactsearch.cuh:252-271) is one ballot per overlap.
constexpr int SEARCH_REG_CHUNKS = 2;

struct Cand {
    double x, y, z, r, dmx, dmy;
    uint32_t sb, bid, code;
    bool ok;
};

// Candidate t of the run list held in lanes 0..26 (start, exclusive prefix,
// length, image code); `runs` has a bit per non-empty run.
__device__ __forceinline__ Cand load_cand(const DemDev& d, uint32_t t, uint32_t T, uint64_t runs, uint32_t r_lo,
                                          uint32_t r_pre, uint32_t r_len, uint32_t r_code) {
    Cand c;
    uint32_t sb = 0, code = 0;
    for (uint64_t m = runs; m; m &= m - 1) {
        const int j = __ffsll((unsigned long long)m) - 1;
        const uint32_t pre = __builtin_amdgcn_readlane(r_pre, j);
        const uint32_t len = __builtin_amdgcn_readlane(r_len, j);
        if (t - pre < len) {
            sb = __builtin_amdgcn_readlane(r_lo, j) + (t - pre);
            code = __builtin_amdgcn_readlane(r_code, j);
        }
    }
    c.ok = t < T;
    c.sb = sb;
    c.code = code;
    if (c.ok) {
        const double4 xb = spos(d, d.sys, sb);
        c.x = xb.x; c.y = xb.y; c.z = xb.z; c.r = xb.w;
        c.bid = d.sid[sb];
    } else {
        c.x = c.y = c.z = c.r = 0.0;
        c.bid = 0;
    }
    decode_image(d.sys, code, c.dmx, c.dmy);
    return c;
}

struct MemberState {
    uint32_t mask, fresh, nc, err;
    bool stop, loaded;
};

// Overlaps of the member at sorted position m with one chunk of candidates.
__device__ __forceinline__ void member_chunk(const Cand& cb, uint32_t lane, uint32_t m, double4 xa,
                                             SlotRow slot, uint32_t& w, bool& dirty, MemberState& st) {
    const double ex = (xa.x - cb.x) + cb.dmx, ey = (xa.y - cb.y) + cb.dmy, ez = xa.z - cb.z;
    const double d2 = ex * ex + ey * ey + ez * ez;
    const double rsum = xa.w + cb.r;
    bool hit = false;
    if (__builtin_expect(cb.ok && d2 <= rsum * rsum * 1.0000001 && cb.sb != m, 0))
        hit = sqrt(d2) - rsum < 0.0;  // exact test of src/contactsearch.cuh:242-248 (double sqrt)
    uint64_t hits = __ballot(hit);
    while (hits) {
        const int l = __ffsll((unsigned long long)hits) - 1;
        hits &= hits - 1;
        const uint32_t bo = __builtin_amdgcn_readlane(cb.bid, l);
        const uint32_t code = __builtin_amdgcn_readlane(cb.code, l);
        if (!st.loaded) {
            w = lane < (uint32_t)NC ? slot[(int)lane] : 0u;
            st.loaded = true;
        }
        const uint64_t match = __ballot(lane < (uint32_t)NC && ((st.mask >> lane) & 1u) && (w & SLOT_IDX_MASK) == bo);
        int cpos;
        if (match) {
            cpos = __ffsll((unsigned long long)match) - 1;
        } else {
            const uint32_t empty = ~st.mask;
            if (empty == 0u) { st.err |= FLAG_CONTACT_OVERFLOW; st.stop = true; return; }
            cpos = 31 - __clz(empty);
            st.fresh |= 1u << cpos;
        }
        if (lane == (uint32_t)cpos) { w = bo | (code << 28); dirty = true; }
        st.mask |= 1u << cpos;
        if (++st.nc > (uint32_t)NC) { st.err |= FLAG_CONTACT_OVERFLOW; st.stop = true; return; }
    }
}

__global__ __launch_bounds__(BLOCK) void k_topo_wave(DemDev d) {
    const Sys& S = d.sys;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t c = xcd_block() * (BLOCK / 64) + (threadIdx.x >> 6);
    if (c >= d.K) return;
    const uint32_t m0 = d.off[c], m1 = d.off[c + 1];
    if (m0 == m1) return;
    const int nx = (int)S.num[0], ny = (int)S.num[1], nz = (int)S.num[2];
    const int gx = (int)(c % S.num[0]), gy = (int)((c / S.num[0]) % S.num[1]), gz = (int)(c / (S.num[0] * S.num[1]));

    // run j = lane (0..26): cell (gx + j%3 - 1, gy + (j/3)%3 - 1, gz + j/9 - 1);
    // a row without periodic image is one run, held by its dx = -1 lane
    uint32_t r_lo = 0, r_len = 0, r_code = 0;
    if (lane < 27u) {
        const int dz = (int)(lane / 9u) - 1, dy = (int)((lane / 3u) % 3u) - 1, dx = (int)(lane % 3u) - 1;
        const int tz = gz + dz;
        int ty = gy + dy, tx = gx + dx;
        bool ok = tz >= 0 && tz < nz;
        uint32_t cy = 0, cx = 0;
        if (ok && (ty < 0 || ty == ny)) {
            if (S.periodic == 1) { cy = ty < 0 ? 1u : 2u; ty = ty < 0 ? ny - 1 : 0; }
            else ok = false;
        }
        if (ok) {
            const uint32_t row = S.cbase + (uint32_t)ty * S.num[0] + (S.num[0] * S.num[1]) * (uint32_t)tz;
            if (gx >= 1 && gx + 1 < nx && cy == 0) {
                if (dx == -1) { r_lo = d.off[row + gx - 1]; r_len = d.off[row + gx + 2] - r_lo; }
            } else {
                if (tx < 0 || tx == nx) {
                    if (S.periodic != 0) { cx = tx < 0 ? 1u : 2u; tx = tx < 0 ? nx - 1 : 0; }
                    else ok = false;
                }
                if (ok) {
                    r_lo = d.off[row + tx];
                    r_len = d.off[row + tx + 1] - r_lo;
                    r_code = cx | (cy << 2);
                }
            }
        }
    }
    uint32_t incl = r_len;
#pragma unroll
    for (int o = 1; o < 32; o <<= 1) {
        const uint32_t v = __shfl_up(incl, o, 64);
        if (lane >= (uint32_t)o) incl += v;
    }
    const uint32_t r_pre = incl - r_len;
    const uint32_t T = __shfl(incl, 26, 64);
    const uint64_t runs = __ballot(r_len != 0u);

    Cand cand[SEARCH_REG_CHUNKS];
#pragma unroll
    for (int j = 0; j < SEARCH_REG_CHUNKS; ++j)
        cand[j] = load_cand(d, 64u * j + lane, T, runs, r_lo, r_pre, r_len, r_code);

    for (uint32_t m = m0; m < m1; ++m) {
        const double4 xa = spos(d, S, m);
        const SlotRow slot = slot_row(d, m);
        MemberState st;
        st.mask = d.ro.cmask[d.perm[m]];
        st.fresh = 0; st.nc = 0; st.err = 0; st.stop = false; st.loaded = false;
        uint32_t w = 0;
        bool dirty = false;
#pragma unroll
        for (int j = 0; j < SEARCH_REG_CHUNKS; ++j)
            if (64u * j < T && !st.stop) member_chunk(cand[j], lane, m, xa, slot, w, dirty, st);
        for (uint32_t base = 64u * SEARCH_REG_CHUNKS; base < T && !st.stop; base += 64u) {
            const Cand cb = load_cand(d, base + lane, T, runs, r_lo, r_pre, r_len, r_code);
            member_chunk(cb, lane, m, xa, slot, w, dirty, st);
        }
        if (dirty) slot[(int)lane] = w;
        if (lane == 0) {
            d.tmask[m] = st.mask;
            d.tfresh[m] = st.fresh;
            if (st.err) atomicOr(d.flags, st.err);
        }
    }
}

// ------------------------------------------------------------ force kernel
// One thread per sorted particle: contact forces from the occupied slots in
// slot order, wall contacts, bond forces, leapfrog.
constexpr int FORCE_BATCH = 4;

template <int K>
__device__ __forceinline__ void quad_add_ft1(V3<double>& F, V3<double>& T, const Acc& c) {
    F.x += quad_bcast<K>(c.F.x); F.y += quad_bcast<K>(c.F.y); F.z += quad_bcast<K>(c.F.z);
    T.x += quad_bcast<K>(c.T.x); T.y += quad_bcast<K>(c.T.y); T.z += quad_bcast<K>(c.T.z);
}
__device__ __forceinline__ void quad_add_ft(V3<double>& F, V3<double>& T, const Acc& c) {
    quad_add_ft1<0>(F, T, c);
    quad_add_ft1<1>(F, T, c);
    quad_add_ft1<2>(F, T, c);
    quad_add_ft1<3>(F, T, c);
}
template <int K>
__device__ __forceinline__ void quad_add1(Acc& a, const Acc& c) {
    quad_add_ft1<K>(a.F, a.T, c);
    a.es_dot += quad_bcast<K>(c.es_dot);
    a.ev_dot += quad_bcast<K>(c.ev_dot);
    a.p += quad_bcast<K>(c.p);
}
// (A lane without a contribution adds +0, which leaves a sum that started at
// +0 as it is.)
__device__ __forceinline__ void quad_add(Acc& a, const Acc& c) {
    quad_add1<0>(a, c);
    quad_add1<1>(a, c);
    quad_add1<2>(a, c);
    quad_add1<3>(a, c);
}
__device__ __forceinline__ Acc zero_acc() {
    Acc c;
    c.F = c.T = mk(0.0, 0.0, 0.0);
    c.es_dot = c.ev_dot = c.p = 0.0;
    return c;
}
// ---- walls (src/contactsearch.cuh:587-663): wf receives the normal force on
// each (the floor keeps none).
__device__ __forceinline__ void wall_contacts(const DemDev& d, const Sys& S, Acc& acc, double4 xa, V3<double> va, V3<double> wa,
                                              double* wf) {
    const double ra = xa.w;
    wf[0] = wf[1] = wf[2] = wf[3] = wf[4] = 0.0;
    {
        const double4 w0 = d.wnx[S.wbase + 0];
        const double dw = w0.w - (xa.z + ra);
        if (dw < 0.0) wf[0] = contact_wall(S, acc, va, wa, ra, mk(w0.x, w0.y, w0.z), dw, d.wmvfd[S.wbase + 0].y);
    }
    {
        const double dw = xa.z - ra - S.origo[2];
        if (dw < 0.0) (void)contact_wall(S, acc, va, wa, ra, mk(0.0, 0.0, 1.0), dw, 0.0);
    }
    if (S.periodic == 0) {
        const double4 w1 = d.wnx[S.wbase + 1], w2 = d.wnx[S.wbase + 2];
        double dw = w1.w - (xa.x + ra);
        if (dw < 0.0) wf[1] = contact_wall(S, acc, va, wa, ra, mk(w1.x, w1.y, w1.z), dw, d.wmvfd[S.wbase + 1].y);
        dw = xa.x - ra - w2.w;
        if (dw < 0.0) wf[2] = contact_wall(S, acc, va, wa, ra, mk(w2.x, w2.y, w2.z), dw, d.wmvfd[S.wbase + 2].y);
    }
    if (S.periodic == 0 || S.periodic == 2) {
        const double4 w3 = d.wnx[S.wbase + 3], w4 = d.wnx[S.wbase + 4];
        double dw = w3.w - (xa.y + ra);
        if (dw < 0.0) wf[3] = contact_wall(S, acc, va, wa, ra, mk(w3.x, w3.y, w3.z), dw, d.wmvfd[S.wbase + 3].y);
        dw = xa.y - ra - w4.w;
        if (dw < 0.0) wf[4] = contact_wall(S, acc, va, wa, ra, mk(w4.x, w4.y, w4.z), dw, d.wmvfd[S.wbase + 4].y);
    }
}

// The rest of sorted particle s's step once its contacts are summed in acc:
// walls, outputs, bond forces, leapfrog, and what the next step needs.  `mask`:
// the contact slots that last; `ended`: some did not.  CHAIN: also what the
// chain's next step needs beyond the stages' (list of changed cells, positions
// by original index).
template <class T, bool B, bool CHAIN>
__device__ __forceinline__ void finish_particle(const DemDev& d, const Sys& S, Words wd, bool keep, uint32_t s, uint32_t o,
                                                uint32_t prev, double4 xa, double4 va4, double4 wa4, Acc& acc,
                                                uint32_t mask, bool ended) {
    const V3<double> va = xyz(va4), wa = xyz(wa4);
    const double ra = xa.w;
    const bool sorted = wd.sorted;
    double wf[5];
    wall_contacts(d, S, acc, xa, va, wa, wf);

    // ---- per-particle outputs (src/contactsearch.cuh:669-687)
    const double dt = S.dt;
    const double4 q0 = d.ro.pr0[prev], q1 = d.ro.pr1[prev], q2 = d.ro.pr2[prev];
    double4 ea = make_double4(q2.y, q2.z, q2.w, wa4.w);  // xysum.x, xysum.y, es, ev
    ea.z += acc.es_dot * dt;
    ea.w += acc.ev_dot * dt;
    // Kept where they can be read: pressure, force, torque and the forces on
    // walls that stand still by the last step of a call only (72 of the 530
    // bytes a contact-free sphere moves)
    const uint32_t wkeep = keep ? (1u << S.nw) - 1u : S.wmoving;
    if (keep) d.pres[s] = acc.p;
    if (wkeep & 1u) d.wall_pp[o] = wf[0];
    if (wkeep & 2u) d.wall_pp[(size_t)d.np + o] = wf[1];
    if (wkeep & 4u) d.wall_pp[2 * (size_t)d.np + o] = wf[2];
    if (wkeep & 8u) d.wall_pp[3 * (size_t)d.np + o] = wf[3];
    if (wkeep & 16u) d.wall_pp[4 * (size_t)d.np + o] = wf[4];

    // ---- bond forces in ascending bond index (src/cohesion.cuh:220-226)
    V3<double> force = acc.F, torque = acc.T;
    if (d.nb0) {
        const uint32_t e0 = d.bcsr_off[o], e1 = d.bcsr_off[o + 1];
        for (uint32_t e = e0; e < e1; ++e) {
            const uint32_t ent = d.bcsr_ent[e];
            const uint32_t k = ent >> 1;
            if (!(d.bonds[k].x < d.np)) continue;
            const V3<double> f = xyz(d.bond_f[k]), t = xyz(d.bond_t[k]);
            if ((ent & 1u) == 0u) { force = force + f; torque = torque - t; }
            else { force = force - f; torque = torque + t; }
        }
    }
    if (keep) {
        d.force[s] = make_double4(force.x, force.y, force.z, acc.es_dot);
        d.torque[s] = make_double4(torque.x, torque.y, torque.z, acc.ev_dot);
    }

    // ---- leapfrog (src/integration.cuh:20-185)
    const double radius = ra;
    const double m = 4.0 / 3.0 * PI_REF * radius * radius * radius * S.rho;
    double ax = force.x / m, ay = force.y / m, az = force.z / m;
    double bx = torque.x * 1.0 / (2.0 / 5.0 * m * radius * radius);
    double by = torque.y * 1.0 / (2.0 / 5.0 * m * radius * radius);
    double bz = torque.z * 1.0 / (2.0 / 5.0 * m * radius * radius);
    ax += S.g[0]; ay += S.g[1]; az += S.g[2];
    if (va4.w > 0.0) {
        ax = 0.0; ay = 0.0; az -= S.g[2];
        if (va4.w >= SPH_FIXVEL_HOLD_Z) az = 0.0;  // extension: the z velocity held as well
        bx = 0.0; by = 0.0; bz = 0.0;
    }
    double px = xa.x, py = xa.y, pz = xa.z;
    (void)wrap_xy(S, px, py);
    double4 v0 = make_double4(q0.x, q0.y, q0.z, 0.0), w0 = make_double4(q0.w, q1.x, q1.y, 0.0);
    double4 ap = make_double4(q1.z, q1.w, q2.x, 0.0);
    v0.x += ax * dt; v0.y += ay * dt; v0.z += az * dt;
    w0.x += bx * dt; w0.y += by * dt; w0.z += bz * dt;
    px += v0.x * dt; py += v0.y * dt; pz += v0.z * dt;
    ap.x += w0.x * dt; ap.y += w0.y * dt; ap.z += w0.z * dt;
    const double vx = v0.x + 0.5 * ax * dt, vy = v0.y + 0.5 * ay * dt, vz = v0.z + 0.5 * az * dt;
    const double wx = w0.x + 0.5 * bx * dt, wy = w0.y + 0.5 * by * dt, wz = w0.z + 0.5 * bz * dt;
    double sx = 0.0, sy = 0.0;
    sx += vx * dt;
    sy += vy * dt;
    ea.x += sx;
    ea.y += sy;
    put(d, d.wo.pr0 + s, make_double4(v0.x, v0.y, v0.z, w0.x));
    put(d, d.wo.pr1 + s, make_double4(w0.y, w0.z, ap.x, ap.y));
    put(d, d.wo.pr2 + s, make_double4(ap.z, ea.x, ea.y, ea.z));
    d.wo.angvel[s] = make_double4(wx, wy, wz, ea.w);
    d.wo.vel[s] = make_double4(vx, vy, vz, va4.w);
    if constexpr (sizeof(T) == 4) {
        d.wo.vf[s] = make_float4((float)vx, (float)vy, (float)vz, 0.0f);
        d.wo.wf[s] = make_float4((float)wx, (float)wy, (float)wz, 0.0f);
    }
    d.wo.x[s] = make_double4(px, py, pz, radius);
    d.wo.id[s] = o;
    d.wo.cmask[s] = mask;

    // cell id of the new position for the next step, which sorts if any
    // sphere changed its cell
    uint32_t cerr = 0;
    const uint32_t nkey = cell_key(S, px, py, pz, cerr), okey = d.skey[s];
    d.key[s] = nkey;
    if (cerr) atomicOr(&d.fw[FW_ERR], cerr);
    if (nkey != okey) {
        atomicSub(&d.count[okey], 1u);
        atomicAdd(&d.count[nkey], 1u);
        if constexpr (CHAIN) {
            const uint32_t k = atomicAdd(&d.fw[FW_CHANGED], 1u);
            if (k < PATCH_MAX) d.change_out[k] = make_uint4(s, okey, nkey, o);
        }
    }
    if (sorted && s == 0u) atomicOr(&d.fw[FW_SORT], SORT_PERM);
    raise(nkey != okey, &d.fw[FW_SORT], SORT_CELLS);
    if constexpr (CHAIN) d.pos_out[o] = s;
    double nx_ = px, ny_ = py;
    const bool wraps = wrap_xy(S, nx_, ny_);
    d.xfs_out[s] = make_float4((float)nx_, (float)ny_, (float)pz, (float)radius);

    // neighbour lists (search mode 5): the list index travels with the
    // particle; request a rebuild once it moved list_lim since the build
    if (d.search_mode == 5) {
        // the next step wraps the new position: the sphere crossed a periodic
        // face (the image through which its contacts meet may change)
        raise(wraps, &d.fw[FW_WRAP], 1u);
        const uint32_t li = d.slidx[s];
        d.wo.lidx[s] = li;
        if (CHAIN && ended) d.nfree[li] = 0.0f;
        const float4 xr = d.xref[li];
        float ddx = (float)px - xr.x, ddy = (float)py - xr.y;
        const float ddz = (float)pz - xr.z;
        if (S.periodic == 1 || S.periodic == 2) ddx -= S.Lf[0] * rintf(ddx / S.Lf[0]);
        if (S.periodic == 1) ddy -= S.Lf[1] * rintf(ddy / S.Lf[1]);
        const float dd2 = ddx * ddx + ddy * ddy + ddz * ddz;
        d.ldisp_out[li] = sqrtf(dd2);
        raise(dd2 > d.list_lim * d.list_lim, &d.fw[FW_REBUILD], 1u);
    }
}

// VW: the partners' velocity records are gathered with their positions, ahead
// of the slots' processing (more registers, fewer waves: faster with many
// contacts per sphere, slower with few; the host picks by timing).  M3:
// contact model 3's pair force (FP64, one system) instead of model 2's.  The
// one-system FP64 kernel without the gathers ahead is held to three waves per
// SIMD (168 VGPRs, no spills): with two it loses 4-8 % on both a contact-free
// packing and the dense crystal.
template <class T, bool B, bool VW, bool M3, bool CHAIN>
__device__ __forceinline__ void force_particle(const DemDev& d, Words wd, bool keep, uint32_t s, Slots sl) {
    const Sys& S = sys_at<B>(d, s);
    const uint32_t o = d.sid[s];
    const uint32_t prev = wd.sorted ? d.perm[s] : s;  // where this particle's records are stored
    double4 xa = d.ro.x[prev];
    (void)wrap_xy(S, xa.x, xa.y);
    const double ra = xa.w;

    // contact slots after the search kernel (contact model 1 keeps none)
    const bool viscous = S.contactmodel == 1;
    uint32_t mask = viscous ? 0u : sl.mask;
    const uint32_t had = mask;
    const uint32_t fresh = viscous ? 0u : sl.fresh;  // slots taken from empty this step: delta_t starts at 0
    const SlotRow slot{d.ro.cslot + prev, d.np};

    // ---- forces from the occupied slots in slot order (src/contactsearch.cuh:479-543)
    const double4 va4 = d.ro.vel[prev], wa4 = d.ro.angvel[prev];
    const V3<double> va = xyz(va4), wa = xyz(wa4);
    Acc acc;
    acc.F = mk(0.0, 0.0, 0.0);
    acc.T = mk(0.0, 0.0, 0.0);
    acc.es_dot = 0.0; acc.ev_dot = 0.0; acc.p = 0.0;
    // Slots in groups of FORCE_BATCH: the group's dependent gathers (slot
    // word -> where the partner's record is stored, pos_of still holding the
    // storage positions -> the record) are issued together, then the slots
    // are processed one by one in slot order.
    for (uint32_t m = mask; m;) {
        int si[FORCE_BATCH];
        uint32_t sw[FORCE_BATCH], pb[FORCE_BATCH];
        int cnt = 0;
#pragma unroll
        for (int k = 0; k < FORCE_BATCH; ++k) {
            si[k] = m ? __ffs(m) - 1 : -1;
            if (m) { m &= m - 1; ++cnt; }
        }
#pragma unroll
        for (int k = 0; k < FORCE_BATCH; ++k) sw[k] = k < cnt ? slot[si[k]] : 0u;
#pragma unroll
        for (int k = 0; k < FORCE_BATCH; ++k) pb[k] = k < cnt ? d.pos_of[sw[k] & SLOT_IDX_MASK] : 0u;
        using PV = PartnerVel<T>;
        double4 xbs[FORCE_BATCH];
        typename PV::type vbs[VW ? FORCE_BATCH : 1], wbs[VW ? FORCE_BATCH : 1];
#pragma unroll
        for (int k = 0; k < FORCE_BATCH; ++k) xbs[k] = k < cnt ? d.ro.x[pb[k]] : make_double4(0.0, 0.0, 0.0, 0.0);
        if constexpr (VW) {
#pragma unroll
            for (int k = 0; k < FORCE_BATCH; ++k) {
                vbs[k] = k < cnt ? PV::vel(d, pb[k]) : PV::zero();
                wbs[k] = k < cnt ? PV::angvel(d, pb[k]) : PV::zero();
            }
        }
#pragma unroll
        for (int k = 0; k < FORCE_BATCH; ++k) {
            if (k >= cnt) break;
            const int i = si[k];
            double4 xb = xbs[k];
            (void)wrap_xy(S, xb.x, xb.y);
            double dmx, dmy;
            decode_image(S, sw[k] >> 28, dmx, dmy);
            const V3<double> xab = mk((xa.x - xb.x) + dmx, (xa.y - xb.y) + dmy, (xa.z - xb.z) + 0.0);
            const double len = vlen(xab);
            const double delta_n = len - (ra + xb.w);
            if (delta_n < 0.0) {
                V3<T> dt0 = (fresh >> i) & 1u ? mk<T>(0, 0, 0) : SlotStore<T>::load(d, i, prev);
                const typename PV::type vb = VW ? vbs[VW ? k : 0] : PV::vel(d, pb[k]);
                const typename PV::type wb = VW ? wbs[VW ? k : 0] : PV::angvel(d, pb[k]);
                if constexpr (M3)
                    contact_hertz(S, acc, va, wa, PV::v3(vb), PV::v3(wb), ra, xb.w, xab, len, delta_n, dt0);
                else
                    contact_linear<T>(S, acc, cvt<T>(va), cvt<T>(wa), PV::v3(vb), PV::v3(wb), (T)ra,
                                      (T)xb.w, cvt<T>(xab), (T)len, (T)delta_n, dt0, keep);
                SlotStore<T>::store(d, i, s, dt0);
                d.wo.cslot[(size_t)i * d.np + s] = sw[k];  // the contact lasts: its slot word moves with it
            } else {
                mask &= ~(1u << i);  // contact ended: the slot is empty again
            }
        }
    }

    // ---- contact model 1: contacts found and processed at once over the 27
    // cells in z, y, x order, sorted order within a cell, with the capillary
    // bond for gaps below db (src/contactsearch.cuh:76-173,548-576)
    if (viscous) {
        const int nx = (int)S.num[0], ny = (int)S.num[1], nz = (int)S.num[2];
        const uint32_t key = d.skey[s] - S.cbase;
        const int gx = (int)(key % S.num[0]), gy = (int)((key / S.num[0]) % S.num[1]);
        const int gz = (int)(key / (S.num[0] * S.num[1]));
        for (int dz = -1; dz <= 1; ++dz) {
            const int tz = gz + dz;
            if (tz < 0 || tz == nz) continue;
            for (int dy = -1; dy <= 1; ++dy) {
                int ty = gy + dy;
                double dmy = 0.0;
                if (ty < 0 || ty == ny) {
                    if (S.periodic != 1) continue;
                    dmy = ty < 0 ? S.L[1] : -S.L[1];
                    ty = ty < 0 ? ny - 1 : 0;
                }
                for (int dx = -1; dx <= 1; ++dx) {
                    int tx = gx + dx;
                    double dmx = 0.0;
                    if (tx < 0 || tx == nx) {
                        if (S.periodic == 0) continue;
                        dmx = tx < 0 ? S.L[0] : -S.L[0];
                        tx = tx < 0 ? nx - 1 : 0;
                    }
                    const uint32_t c = S.cbase + (uint32_t)tx + (uint32_t)ty * S.num[0] + (S.num[0] * S.num[1]) * (uint32_t)tz;
                    const uint32_t hi = d.off[c + 1];
                    for (uint32_t sb = d.off[c]; sb < hi; ++sb) {
                        if (sb == s) continue;
                        const uint32_t pb = wd.sorted ? d.perm[sb] : sb;
                        double4 xb = d.ro.x[pb];
                        (void)wrap_xy(S, xb.x, xb.y);
                        const V3<double> xab = mk((xa.x - xb.x) + dmx, (xa.y - xb.y) + dmy, (xa.z - xb.z) + 0.0);
                        const double len = vlen(xab);
                        const double delta = len - (ra + xb.w);
                        if (delta < 0.0)
                            contact_viscous(S, acc, va, wa, xyz(d.ro.vel[pb]), xyz(d.ro.angvel[pb]), ra, xb.w, xab, len,
                                            delta);
                        else if (delta < S.db)
                            capillary(S, acc, ra, xb.w, delta, xab, len);
                    }
                }
            }
        }
    }

    finish_particle<T, B, CHAIN>(d, S, wd, keep, s, o, prev, xa, va4, wa4, acc, mask, mask != had);
}

template <class T, bool B, bool VW, bool M3 = false>
__global__ __launch_bounds__(BLOCK, (sizeof(T) == 8 && !B && !VW && !M3) ? 3 : 1) void k_force(DemDev d) {
    static_assert(!M3 || (sizeof(T) == 8 && !B), "contact model 3: FP64, one system");
    const uint32_t s = xcd_block() * blockDim.x + threadIdx.x;
    if (s >= d.np) return;
    Slots sl = {0u, 0u};
    if (B || d.sys.contactmodel != 1) sl = {d.tmask[s], d.tfresh[s]};
    force_particle<T, B, VW, M3, false>(d, words_of(d), d.outputs != 0u, s, sl);
}

// FP32 copies of the input set's velocity records (mixed mode), by storage
// position.
__global__ __launch_bounds__(BLOCK) void k_f32_copies(DemDev d) {
    const uint32_t q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= d.np) return;
    const double4 v = d.ro.vel[q], w = d.ro.angvel[q];
    d.ro.vf[q] = make_float4((float)v.x, (float)v.y, (float)v.z, 0.0f);
    d.ro.wf[q] = make_float4((float)w.x, (float)w.y, (float)w.z, 0.0f);
}

// ------------------------------------------------------------- quad steps
// Contact search and force of one sorted particle by the four lanes of a quad:
// each takes every fourth list entry and every fourth contact, so the serial
// chain of a particle -- its list's dependent loads and one contact's square
// roots and divisions after another's -- is a quarter as long.  That chain is
// what bounds a step of up to some ten thousand spheres, which leave most of
// the chip's SIMDs with a wavefront or none.  The sums keep the slot order:
// every lane adds the quad's four contributions lane by lane.
// LDS written by one lane of a wavefront and read by another.
__device__ __forceinline__ void quad_sync() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

constexpr int QUAD_N = BLOCK / 4;  // particles of a workgroup

// LDS columns of a quad's particle: stride QUAD_N.
struct QuadCols {
    uint32_t* sw;  // slot words of the occupied slots
    uint32_t* pb;  // where those slots' partners are stored
    uint64_t* nk;  // keys of new contacts; contact model 1: its candidates
};

// One list entry as a lane of the search loads it.
struct ListEntry {
    uint32_t lb, hb, lw;
    float g;
    bool in;
};
__device__ __forceinline__ ListEntry list_entry(const DemDev& d, uint32_t li, uint32_t nl, uint32_t e, bool slots, bool skip_held) {
    ListEntry r;
    r.in = e < nl;
    const size_t at = (size_t)(r.in ? e : 0u) * d.np + li;
    r.lb = r.in ? d.nlist[at] : li;
    r.g = r.in ? d.nlistg[at] : 1e30f;
    r.hb = r.in && slots ? d.nhint[at] : 0xffu;
    r.lw = r.in && slots && skip_held ? d.nlo[at] : 0xffffffffu;
    return r;
}

// The neighbour-list search (list_search) by a quad: QUAD_E entries a lane at
// a time, all loads of one kind in flight together, so the chain of dependent
// loads is gone through once for 4 QUAD_E entries.  The FP64 test follows the
// displacement test directly (the FP32 one would be another load in the
// chain).  sw and pb hold the particle's occupied slots, and those of new
// contacts afterwards.
constexpr int QUAD_E = 4;
__device__ __forceinline__ void quad_list_search(const DemDev& d, Words wd, uint32_t s, uint32_t j, double4 xa, uint32_t key,
                                                 uint32_t li, uint32_t nl, float disp, const ListEntry* first, bool skip_held,
                                                 QuadCols q, uint32_t& mask, uint32_t& fresh) {
    const Sys& S = d.sys;
    const uint32_t mask0 = mask;
    const uint32_t held_bits = wd.wrap ? 0xffffffffu : SLOT_IDX_MASK;  // with wraps: the word must carry no image
    int gx, gy, gz;
    cell_xyz(S, key - S.cbase, gx, gy, gz);
    const float da = disp + 3.0f * d.search_eps;
    const float dfar = da + d.list_lim + 3.0f * d.search_eps;
    uint32_t n = 0, nnew = 0;
    for (uint32_t i0 = 0; i0 < nl; i0 += 4 * QUAD_E) {
        ListEntry en[QUAD_E];
        bool near[QUAD_E], hinted[QUAD_E];
        uint32_t sb[QUAD_E];
#pragma unroll
        for (int k = 0; k < QUAD_E; ++k) {
            if (i0 == 0) en[k] = first[k];
            else en[k] = list_entry(d, li, nl, i0 + 4 * k + j, mask0 != 0u, skip_held);
        }
#pragma unroll
        for (int k = 0; k < QUAD_E; ++k) {
            hinted[k] = en[k].hb < 32u && ((mask0 >> (en[k].hb & 31u)) & 1u);
            const bool held = hinted[k] && (q.sw[(en[k].hb & 31u) * QUAD_N] & held_bits) == en[k].lw;
            near[k] = en[k].in && !held && en[k].g <= dfar;
        }
        if (!quad_ballot(near[0] || near[1] || near[2] || near[3])) continue;
        float db[QUAD_E];
        uint32_t kb[QUAD_E], bo[QUAD_E], pb[QUAD_E];
        double4 xb[QUAD_E];
#pragma unroll
        for (int k = 0; k < QUAD_E; ++k) {
            db[k] = near[k] ? d.ldisp[en[k].lb] : 0.0f;
            sb[k] = !near[k] ? s : wd.aligned ? en[k].lb : d.linv[en[k].lb];
        }
#pragma unroll
        for (int k = 0; k < QUAD_E; ++k) {
            if (near[k]) {
                pb[k] = wd.sorted ? d.perm[sb[k]] : sb[k];
                kb[k] = d.skey[sb[k]];
                bo[k] = d.sid[sb[k]];
            }
        }
#pragma unroll
        for (int k = 0; k < QUAD_E; ++k)
            if (near[k]) xb[k] = d.ro.x[pb[k]];
#pragma unroll
        for (int k = 0; k < QUAD_E; ++k) {
            uint64_t hit = 0;
            if (near[k] && en[k].g <= da + db[k]) hit = list_pair(S, sb[k], kb[k] - S.cbase, xb[k], xa, gx, gy, gz);
            bool fresh_one = false;
            if (hit != 0ull) {
                int cpos = -1;
                if (hinted[k] && (q.sw[(en[k].hb & 31u) * QUAD_N] & SLOT_IDX_MASK) == bo[k]) {
                    cpos = (int)en[k].hb;
                } else {
                    for (uint32_t m = mask0; m; m &= m - 1) {
                        const int i = __ffs(m) - 1;
                        if ((q.sw[i * QUAD_N] & SLOT_IDX_MASK) == bo[k]) { cpos = i; break; }
                    }
                    if (cpos >= 0) {  // the entry's hint and partner, written together
                        const size_t at = (size_t)(i0 + 4 * k + j) * d.np + li;
                        d.nhint[at] = (uint8_t)cpos;
                        d.nlo[at] = bo[k];
                    }
                }
                // kept: a partner occurs once, so no other lane touches this slot
                if (cpos >= 0) q.sw[cpos * QUAD_N] = bo[k] | ((uint32_t)(hit >> 32) & 15u) << 28;
                else fresh_one = true;
            }
            n += __popc(quad_ballot(hit != 0ull));
            const uint32_t fb = quad_ballot(fresh_one);
            if (fresh_one) {
                const uint32_t at = nnew + __popc(fb & ((1u << j) - 1u));
                if (at < (uint32_t)NC) q.nk[(size_t)at * QUAD_N] = hit;
            }
            nnew += __popc(fb);
        }
    }
    uint32_t err = n > (uint32_t)NC ? FLAG_CONTACT_OVERFLOW : 0u;
    if (nnew > (uint32_t)NC) nnew = NC;
    fresh = 0;
    if (nnew) {  // (the same in all four lanes)
        quad_sync();
        if (j == 0) {
            // empty slots in key order
            for (uint32_t i = 1; i < nnew; ++i) {
                const uint64_t v = q.nk[(size_t)i * QUAD_N];
                uint32_t k = i;
                while (k > 0 && q.nk[(size_t)(k - 1) * QUAD_N] > v) {
                    q.nk[(size_t)k * QUAD_N] = q.nk[(size_t)(k - 1) * QUAD_N];
                    --k;
                }
                q.nk[(size_t)k * QUAD_N] = v;
            }
            for (uint32_t h = 0; h < nnew; ++h) {
                const uint64_t v = q.nk[(size_t)h * QUAD_N];
                const uint32_t b = (uint32_t)(v & 0xffffffffu);
                const uint32_t empty = ~mask;
                if (empty == 0u) { err |= FLAG_CONTACT_OVERFLOW; break; }
                const int cpos = 31 - __clz(empty);
                fresh |= 1u << cpos;
                q.sw[cpos * QUAD_N] = d.sid[b] | ((uint32_t)(v >> 32) & 15u) << 28;
                q.pb[cpos * QUAD_N] = wd.sorted ? d.perm[b] : b;
                mask |= 1u << cpos;
            }
        }
        quad_sync();
        mask = quad_bcast<0>(mask);
        fresh = quad_bcast<0>(fresh);
    }
    // (the force phase carries the words of the contacts that last into the
    // output set; nothing reads the input set's afterwards)
    if (err) atomicOr(d.flags, err);
}

// Contact model 1 by a quad.  The FP32 copies of the candidates in each row of
// cells are read four at a time, the nine rows' first four ahead of their use;
// those within the reach of a contact or a capillary bond go to the LDS column
// list in the order of force_particle, and are worked off four at a time.
__device__ __forceinline__ void quad_viscous(const DemDev& d, Words wd, uint32_t s, uint32_t j, double4 xa, V3<double> va,
                                             V3<double> wa, uint64_t* list, Acc& acc) {
    const Sys& S = d.sys;
    const float4* xf = xf_sorted(d, wd);
    const float4 xaf = xf[s];
    const float reach = xaf.w + d.search_eps + fmaxf(0.0f, (float)S.db * 1.000001f);
    int gx, gy, gz;
    cell_xyz(S, d.skey[s] - S.cbase, gx, gy, gz);
    const int nx = (int)S.num[0], ny = (int)S.num[1], nz = (int)S.num[2];
    uint32_t n = 0, base = 0;  // candidates within reach so far; the first the list holds
    // candidate sb (its FP32 copy c) of a run that ends at h, image code
    auto test = [&](uint32_t sb, uint32_t h, float4 c, uint32_t code) {
        bool close = false;
        if (sb < h && sb != s) {
            const uint32_t cx = code & 3u, cyi = code >> 2;
            const float ex = (xaf.x - c.x) + (cx == 1u ? S.Lf[0] : (cx == 2u ? -S.Lf[0] : 0.0f));
            const float ey = (xaf.y - c.y) + (cyi == 1u ? S.Lf[1] : (cyi == 2u ? -S.Lf[1] : 0.0f)), ez = xaf.z - c.z;
            const float rs = reach + c.w;
            close = !(ex * ex + ey * ey + ez * ez > rs * rs);
        }
        const uint32_t m = quad_ballot(close), at = n + __popc(m & ((1u << j) - 1u)) - base;
        if (close && at < (uint32_t)NC) list[(size_t)at * QUAD_N] = ((uint64_t)code << 32) | sb;
        n += __popc(m);
    };
    auto run = [&](uint32_t l, uint32_t h, uint32_t code) {
        for (uint32_t sb = l + j; sb - j < h; sb += 4) test(sb, h, sb < h ? xf[sb] : xaf, code);
    };
    // A row of cells x - 1 .. x + 1 is one run of the sorted arrays, or two
    // where it passes through a periodic face: cells a0 .. a1 with image code
    // ca, then b0 .. b1 with cb.
    int a0 = gx > 0 ? gx - 1 : 0, a1 = gx + 1 < nx ? gx + 1 : nx - 1, b0 = 0, b1 = -1;
    uint32_t ca = 0, cb = 0;
    if (S.periodic != 0 && gx == 0) { b0 = 0; b1 = a1; a0 = a1 = nx - 1; ca = 1u; }
    else if (S.periodic != 0 && gx == nx - 1) { b0 = b1 = 0; cb = 2u; }
    for (;; base += NC) {  // (once, unless more than NC are within reach)
        n = 0;
        uint32_t lo[9], hi[9], lob[9], hib[9], cy[9];
        float4 c[9];
#pragma unroll
        for (int r = 0; r < 9; ++r) {  // rows in z, y order
            const int tz = gz + r / 3 - 1;
            int ty = gy + r % 3 - 1;
            bool ok = tz >= 0 && tz < nz;
            cy[r] = 0;
            if (ty < 0 || ty == ny) {
                ok = ok && S.periodic == 1;
                cy[r] = ty < 0 ? 4u : 8u;
                ty = ty < 0 ? ny - 1 : 0;
            }
            const uint32_t row = S.cbase + (uint32_t)ty * S.num[0] + (S.num[0] * S.num[1]) * (uint32_t)tz;
            lo[r] = ok ? d.off[row + a0] : 0u;
            hi[r] = ok ? d.off[row + a1 + 1] : 0u;
            lob[r] = ok && b1 >= b0 ? d.off[row + b0] : 0u;
            hib[r] = ok && b1 >= b0 ? d.off[row + b1 + 1] : 0u;
        }
#pragma unroll
        for (int r = 0; r < 9; ++r) c[r] = lo[r] + j < hi[r] ? xf[lo[r] + j] : xaf;
#pragma unroll
        for (int r = 0; r < 9; ++r) {
            if (lo[r] < hi[r]) {
                test(lo[r] + j, hi[r], c[r], cy[r] | ca);
                if (hi[r] - lo[r] > 4u) run(lo[r] + 4u, hi[r], cy[r] | ca);
            }
            if (lob[r] < hib[r]) run(lob[r], hib[r], cy[r] | cb);
        }
        quad_sync();
        for (uint32_t k0 = base; k0 < n && k0 < base + NC; k0 += 4) {
            Acc c = zero_acc();
            if (k0 + j < n) {
                const uint64_t v = list[(size_t)(k0 + j - base) * QUAD_N];
                const uint32_t sb = (uint32_t)v;
                double dmx, dmy;
                decode_image(S, (uint32_t)(v >> 32), dmx, dmy);
                const uint32_t pb = wd.sorted ? d.perm[sb] : sb;
                double4 xb = d.ro.x[pb];
                const double4 vb = d.ro.vel[pb], wb = d.ro.angvel[pb];
                (void)wrap_xy(S, xb.x, xb.y);
                const V3<double> xab = mk((xa.x - xb.x) + dmx, (xa.y - xb.y) + dmy, (xa.z - xb.z) + 0.0);
                const double len = vlen(xab);
                const double delta = len - (xa.w + xb.w);
                if (delta < 0.0) contact_viscous(S, c, va, wa, xyz(vb), xyz(wb), xa.w, xb.w, xab, len, delta);
                else if (delta < S.db) capillary(S, c, xa.w, xb.w, delta, xab, len);
            }
            quad_add(acc, c);
        }
        quad_sync();
        if (n <= base + NC) break;
    }
}

// x, y or z for lane 0, 1 or 2 and 3 (by value: a choice among elements in
// place would be one of addresses).
template <class V>
__device__ __forceinline__ V by_lane(uint32_t j, V x, V y, V z) { return j == 0u ? x : j == 1u ? y : z; }

// The rest of a quad's particle (finish_particle): lane j < 3 integrates
// component j and the four lanes of a record write its four doubles, so the
// divisions, the cell coordinates and the stores are a third to a quarter of
// one thread's.
// Returns (lane 0) the product of the objective's weights with the force, if
// the step records one.
template <class T>
__device__ __forceinline__ double quad_finish(const DemDev& d, Words wd, uint32_t s, uint32_t j, bool keep, uint32_t o, uint32_t okey,
                                            double4 xa, double4 va4, double4 wa4, double v0, double w0, double ap, double sum,
                                            uint32_t li, float xr, Acc& acc, uint32_t mask) {
    const Sys& S = d.sys;
    const V3<double> va = xyz(va4), wa = xyz(wa4);
    const double ra = xa.w, dt = S.dt;
    double wf[5];
    wall_contacts(d, S, acc, xa, va, wa, wf);
    const uint32_t wkeep = keep ? (1u << S.nw) - 1u : S.wmoving;
    if (keep && j == 0u) d.pres[s] = acc.p;
    if (j == 1u) {
#pragma unroll
        for (int w = 0; w < 5; ++w)
            if ((wkeep >> w) & 1u) d.wall_pp[(size_t)w * d.np + o] = wf[w];
    }
    V3<double> force = acc.F, torque = acc.T;
    if (d.nb0) {  // bond forces in ascending bond index, four at a time, added lane by lane
        const uint32_t e0 = d.bcsr_off[o], e1 = d.bcsr_off[o + 1];
        for (uint32_t e = e0; e < e1; e += 4) {
            Acc c;
            c.F = c.T = mk(0.0, 0.0, 0.0);
            if (e + j < e1) {
                const uint32_t ent = d.bcsr_ent[e + j], k = ent >> 1;
                if (d.bonds[k].x < d.np) {
                    const V3<double> f = xyz(d.bond_f[k]), t = xyz(d.bond_t[k]);
                    const bool own_side = (ent & 1u) == 0u;
                    c.F = own_side ? f : -f;
                    c.T = own_side ? -t : t;
                }
            }
            quad_add_ft(force, torque, c);
        }
    }
    double product = 0.0;
    if (d.rec.wobj && j == 0u) {
        const double4 w = d.rec.wobj[o];
        product = w.x * force.x + w.y * force.y + w.z * force.z;
    }
    if (keep && j == 2u) d.force[s] = make_double4(force.x, force.y, force.z, acc.es_dot);
    if (keep && j == 3u) d.torque[s] = make_double4(torque.x, torque.y, torque.z, acc.ev_dot);
    // component j (what lane 3 computes along is not used; it stores the rest)
    const bool x_ = j == 0u, y_ = j == 1u;
    const double m = 4.0 / 3.0 * PI_REF * ra * ra * ra * S.rho;
    double a = by_lane(j, force.x, force.y, force.z) / m;
    double b = by_lane(j, torque.x, torque.y, torque.z) * 1.0 / (2.0 / 5.0 * m * ra * ra);
    a += by_lane(j, S.g[0], S.g[1], S.g[2]);
    if (va4.w > 0.0) {
        a = x_ || y_ ? 0.0 : a - S.g[2];
        if (!x_ && !y_ && va4.w >= SPH_FIXVEL_HOLD_Z) a = 0.0;
        b = 0.0;
    }
    const bool per = x_ ? S.periodic == 1 || S.periodic == 2 : y_ && S.periodic == 1;
    const double lo = by_lane(j, S.origo[0], S.origo[1], S.origo[2]), len = by_lane(j, S.L[0], S.L[1], S.L[2]);
    auto wrap = [&](double& v) -> bool {
        bool changed = false;
        if (per) {
            if (v < lo) { v += len; changed = true; }
            if (v > len) { v -= len; changed = true; }
        }
        return changed;
    };
    double p = by_lane(j, xa.x, xa.y, xa.z);
    (void)wrap(p);
    v0 += a * dt;
    w0 += b * dt;
    p += v0 * dt;
    ap += w0 * dt;
    const double v = v0 + 0.5 * a * dt, w = w0 + 0.5 * b * dt;
    double sx = 0.0;
    sx += v * dt;
    const bool l3 = j == 3u;
    // sum: displacement sum of lanes 0 and 1, es of lane 3
    if (l3) sum += acc.es_dot * dt;
    else sum += sx;
    const size_t at = 4 * (size_t)s + j;
    double* const pr0 = reinterpret_cast<double*>(d.wo.pr0);
    double* const pr1 = reinterpret_cast<double*>(d.wo.pr1);
    double* const pr2 = reinterpret_cast<double*>(d.wo.pr2);
    reinterpret_cast<double*>(d.wo.x)[at] = l3 ? ra : p;
    reinterpret_cast<double*>(d.wo.vel)[at] = l3 ? va4.w : v;
    reinterpret_cast<double*>(d.wo.angvel)[at] = l3 ? wa4.w + acc.ev_dot * dt : w;
    if (!l3) {
        pr0[at] = v0;
        (x_ ? pr0 : pr1)[x_ ? at + 3 : at - 1] = w0;
        (x_ || y_ ? pr1 : pr2)[x_ || y_ ? at + 2 : at - 2] = ap;
    }
    if (x_ || y_) pr2[at + 1] = sum;
    if (l3) pr2[at] = sum;
    if constexpr (sizeof(T) == 4) {
        reinterpret_cast<float*>(d.wo.vf)[at] = l3 ? 0.0f : (float)v;
        reinterpret_cast<float*>(d.wo.wf)[at] = l3 ? 0.0f : (float)w;
    }
    if (x_) d.wo.id[s] = o;
    if (y_) d.wo.cmask[s] = mask;
    if (l3) d.pos_out[o] = s;

    // the next step's cell, FP32 copy and displacement
    const double pu = p;
    const bool wrapped = wrap(p);
    uint32_t cerr = 0;
    const uint32_t cj = (uint32_t)cell_coord(p, lo, by_lane(j, S.cell_len[0], S.cell_len[1], S.cell_len[2]),
                                             by_lane(j, S.num[0], S.num[1], S.num[2]), cerr);
    if (l3) cerr = 0u;  // (its p is no position)
    reinterpret_cast<float*>(d.xfs_out)[at] = (float)(l3 ? ra : p);
    const uint32_t nkey = S.cbase + ((quad_bcast<2>(cj) * S.num[1]) * S.num[0] + quad_bcast<1>(cj) * S.num[0] + quad_bcast<0>(cj));
    cerr = quad_or(cerr);
    const bool any_wrap = quad_or(wrapped ? 1u : 0u) != 0u;
    float dd = (float)pu - xr;
    const float lf = by_lane(j, S.Lf[0], S.Lf[1], 1.0f);
    if (per) dd -= lf * rintf(dd / lf);
    const float sq = dd * dd;
    const float dd2 = (__uint_as_float(quad_bcast<0>(__float_as_uint(sq))) + __uint_as_float(quad_bcast<1>(__float_as_uint(sq)))) +
                      __uint_as_float(quad_bcast<2>(__float_as_uint(sq)));
    if (j != 0u) return 0.0;
    d.key[s] = nkey;
    if (cerr) atomicOr(&d.fw[FW_ERR], cerr);
    if (nkey != okey) {
        atomicSub(&d.count[okey], 1u);
        atomicAdd(&d.count[nkey], 1u);
        const uint32_t k = atomicAdd(&d.fw[FW_CHANGED], 1u);
        if (k < PATCH_MAX) d.change_out[k] = make_uint4(s, okey, nkey, o);
    }
    if (wd.sorted && s == 0u) atomicOr(&d.fw[FW_SORT], SORT_PERM);
    raise(nkey != okey, &d.fw[FW_SORT], SORT_CELLS);
    if (d.search_mode == 5) {
        raise(any_wrap, &d.fw[FW_WRAP], 1u);
        d.wo.lidx[s] = li;
        d.ldisp_out[li] = sqrtf(dd2);
        raise(dd2 > d.list_lim * d.list_lim, &d.fw[FW_REBUILD], 1u);
    }
    return product;
}

// Search (unless a rebuild made it) and force of sorted particle s.  All that
// its own index leads to is loaded first.
template <class T, int MODEL>
__device__ __forceinline__ double quad_step(const DemDev& d, Words wd, uint32_t s, uint32_t j, uint32_t i, bool keep,
                                            QuadCols q) {
    const Sys& S = d.sys;
    const uint32_t prev = wd.sorted ? d.perm[s] : s;
    constexpr bool slots = MODEL != 1;
    const bool lists = slots && d.search_mode == 5;
    const uint32_t li = !lists ? s : wd.aligned ? s : d.slidx[s];
    uint32_t mask = !slots ? 0u : wd.rebuild ? d.tmask[s] : d.ro.cmask[prev];
    const uint32_t o = d.sid[s], okey = d.skey[s];
    double4 xa = d.ro.x[prev];
    const double4 va4 = d.ro.vel[prev], wa4 = d.ro.angvel[prev];
    uint32_t fresh = slots && wd.rebuild ? d.tfresh[s] : 0u;
    const bool search = slots && !wd.rebuild;
    const uint32_t nl = search ? d.ncnt[li] : 0u;
    const float disp = search ? d.ldisp[li] : 0.0f;
    const float xr = lists ? reinterpret_cast<const float*>(d.xref)[4 * (size_t)li + j] : 0.0f;
    const size_t at = 4 * (size_t)prev + j;
    const double* const pr0 = reinterpret_cast<const double*>(d.ro.pr0);
    const double* const pr1 = reinterpret_cast<const double*>(d.ro.pr1);
    const double* const pr2 = reinterpret_cast<const double*>(d.ro.pr2);
    const bool x_ = j == 0u, y_ = j == 1u;
    const double v0 = pr0[at];
    const double w0 = (x_ ? pr0 : pr1)[x_ ? at + 3 : at - 1];
    const double ap = (x_ || y_ ? pr1 : pr2)[x_ || y_ ? at + 2 : at & ~(size_t)3];
    const double sum = pr2[x_ || y_ ? at + 1 : at];
    // the first list entries, and the occupied slots' words and partners
    ListEntry first[QUAD_E];
    bool skip_held = !wd.wrap;
    if (search && wd.wrap) {
        int gx, gy, gz;
        cell_xyz(S, okey - S.cbase, gx, gy, gz);
        skip_held = (S.periodic == 0 || (gx > 0 && gx < (int)S.num[0] - 1)) &&
                    (S.periodic != 1 || (gy > 0 && gy < (int)S.num[1] - 1));
    }
#pragma unroll
    for (int k = 0; k < QUAD_E; ++k) first[k] = list_entry(d, li, nl, 4 * k + j, mask != 0u, skip_held);
    const SlotRow slot{d.ro.cslot + prev, d.np};
    for (uint32_t m = mask; m;) {
        int si[3];
        uint32_t w[3], pb[3];
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            si[r] = -1;
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                if (k == j && m) si[r] = __ffs(m) - 1;
                m &= m - 1;  // (0 stays 0)
            }
        }
#pragma unroll
        for (int r = 0; r < 3; ++r) w[r] = si[r] >= 0 ? slot[si[r]] : 0u;
#pragma unroll
        for (int r = 0; r < 3; ++r) pb[r] = si[r] >= 0 ? d.pos_of[w[r] & SLOT_IDX_MASK] : 0u;
#pragma unroll
        for (int r = 0; r < 3; ++r)
            if (si[r] >= 0) {
                q.sw[si[r] * QUAD_N] = w[r];
                q.pb[si[r] * QUAD_N] = pb[r];
            }
    }
    (void)wrap_xy(S, xa.x, xa.y);
    const V3<double> va = xyz(va4), wa = xyz(wa4);
    Acc acc = zero_acc();
    if constexpr (!slots) {
        quad_viscous(d, wd, s, j, xa, va, wa, q.nk, acc);
    } else {
        quad_sync();
        if (search) quad_list_search(d, wd, s, j, xa, okey, li, nl, disp, first, skip_held, q, mask, fresh);
        quad_sync();
        // (the tape keys slots and springs by original index; a fresh slot's
        // spring is not read)
        const size_t rec = (size_t)(d.rec.step0 + i) * d.np, rec_slot = (rec + o) * NC;
        if (d.rec.x) {
            if (j == 0u) {
                d.rec.x[rec + s] = xa;
                d.rec.id[rec + s] = o;
                d.rec.pos_of[rec + o] = s;
            } else if (j == 1u) {
                d.rec.vel[rec + s] = va4;
            } else if (j == 2u) {
                d.rec.angvel[rec + s] = wa4;
            } else {
                d.rec.tmask[rec + s] = mask;
                d.rec.tfresh[rec + s] = fresh;
            }
        }
        using PV = PartnerVel<T>;
        // one contact a lane; the next group's records are loaded while one is worked on
        struct Contact {
            int i;
            uint32_t w;
            double4 x;
            typename PV::type v, wv;
            V3<T> dt0;
        };
        uint32_t m = mask, ended = 0;
        auto next = [&]() -> Contact {
            Contact c;
            c.i = -1;
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                if (k == j && m) c.i = __ffs(m) - 1;
                m &= m - 1;
            }
            if (c.i >= 0) {
                const uint32_t pb = q.pb[c.i * QUAD_N];
                c.w = q.sw[c.i * QUAD_N];
                c.x = d.ro.x[pb];
                c.v = PV::vel(d, pb);
                c.wv = PV::angvel(d, pb);
                c.dt0 = (fresh >> c.i) & 1u ? mk<T>(0, 0, 0) : SlotStore<T>::load(d, c.i, prev);
            }
            return c;
        };
        bool more = m != 0u;
        Contact cur;
        cur.i = -1;
        if (more) cur = next();
        while (more) {
            more = m != 0u;
            Contact after;
            after.i = -1;
            if (more) after = next();
            Acc c = zero_acc();
            if (cur.i >= 0 && d.rec.x) {
                const size_t at = rec_slot + (size_t)cur.i;
                d.rec.cslot[at] = cur.w;
                if constexpr (sizeof(T) == 4) {
                    float* const p = d.rec.cdt32 + 3 * at;
                    p[0] = cur.dt0.x; p[1] = cur.dt0.y; p[2] = cur.dt0.z;
                } else {
                    double* const p = d.rec.cdt + 3 * at;
                    p[0] = cur.dt0.x; p[1] = cur.dt0.y; p[2] = cur.dt0.z;
                }
            }
            if (cur.i >= 0) {
                double4 xb = cur.x;
                (void)wrap_xy(S, xb.x, xb.y);
                double dmx, dmy;
                decode_image(S, cur.w >> 28, dmx, dmy);
                const V3<double> xab = mk((xa.x - xb.x) + dmx, (xa.y - xb.y) + dmy, (xa.z - xb.z) + 0.0);
                const double len = vlen(xab);
                const double delta_n = len - (xa.w + xb.w);
                if (delta_n < 0.0) {
                    V3<T> dt0 = cur.dt0;
                    if constexpr (MODEL == 3)
                        contact_hertz(S, c, va, wa, PV::v3(cur.v), PV::v3(cur.wv), xa.w, xb.w, xab, len, delta_n, dt0);
                    else
                        contact_linear<T>(S, c, cvt<T>(va), cvt<T>(wa), PV::v3(cur.v), PV::v3(cur.wv), (T)xa.w, (T)xb.w,
                                          cvt<T>(xab), (T)len, (T)delta_n, dt0, keep);
                    SlotStore<T>::store(d, cur.i, s, dt0);
                    d.wo.cslot[(size_t)cur.i * d.np + s] = cur.w;  // the contact lasts: its slot word moves with it
                } else {
                    ended |= 1u << cur.i;  // the slot is empty again
                }
            }
            quad_add(acc, c);
            cur = after;
        }
        mask &= ~quad_or(ended);
    }
    return quad_finish<T>(d, wd, s, j, keep, o, okey, xa, va4, wa4, v0, w0, ap, sum, li, xr, acc, mask);
}

// The sort of a step before which only n spheres (`list`) changed their cell,
// for the particle stored at i.  The others keep their order, so its sorted
// position follows from where the n left and where they arrive: their places
// among (cell, original index).  One launch, n comparisons a particle, instead
// of the counts, scan, placement and order of the full sort.
__device__ __forceinline__ void patch_order(const DemDev& d, const uint4* list, uint32_t n, uint32_t i) {
    const uint32_t id = d.ro.id[i], key = d.key[i];
    bool moved = false;
    for (uint32_t k = 0; k < n; ++k) moved = moved || list[k].x == i;
    uint32_t before = i;  // spheres stored before it in the order of (cell, index) of the last step
    if (moved) {
        const uint32_t e = d.off[key + 1];
        before = d.off[key];
        for (uint32_t m = before; m < e; ++m) before += d.ro.id[m] < id ? 1u : 0u;
    }
    uint32_t q = before;
    for (uint32_t k = 0; k < n; ++k) {
        const uint4 c = list[k];
        q -= c.x < before ? 1u : 0u;
        q += c.z < key || (c.z == key && c.w < id) ? 1u : 0u;
    }
    if (q >= d.np) return;  // (never: q is a permutation by construction)
    d.perm[q] = i;
    d.sid[q] = id;
    d.skey[q] = key;
    d.xf[q] = d.xfs[i];
    if (d.search_mode == 5) {
        const uint32_t li = d.ro.lidx[i];
        d.linv[li] = q;
        d.slidx[q] = li;
    }
}

// The cell offsets of that sort, those of block b.
__device__ __forceinline__ void patch_offsets(const DemDev& d, const uint4* change, uint32_t n, uint32_t b, uint4* list) {
    if (b * BLOCK >= d.K) return;
    if (threadIdx.x < n) list[threadIdx.x] = change[threadIdx.x];
    __syncthreads();
    const uint32_t c = b * BLOCK + threadIdx.x;
    if (c >= d.K) return;
    uint32_t off = d.off[c];
    const uint32_t was = off;
    for (uint32_t k = 0; k < n; ++k) off += (list[k].z < c ? 1u : 0u) - (list[k].y < c ? 1u : 0u);
    if (off != was) d.off[c] = off;
}

// A launch of a chain: the phase of a step that follows what the last launch
// did, as the step's words ask for it.  The launches of a call are all alike,
// so a step costs as many as it has work for -- one, when no sphere changed its
// cell, no list is due and no bond is there -- and the host need not know
// which: it issues about as many as the call will take and looks where the
// chain stands.
// The words a step raises go to the chain's sets in turn (step i reads set
// i % 3, raises i + 1 and clears i + 2, which nothing else touches meanwhile);
// a call's first step reads the handle's own and its last launch leaves them
// there.
__device__ __forceinline__ uint32_t next_phase(const DemDev& d, uint32_t phase, uint32_t steps_left, uint32_t sort, bool patch,
                                               bool rebuild) {
    rebuild = rebuild && d.search_mode == 5 && d.sys.contactmodel != 1;
    switch (phase) {
        case PH_FORCE:
            if (d.wall_launches) return d.wall_launches == 2u ? PH_WALL_SUMS : PH_WALLS;
            [[fallthrough]];
        case PH_WALLS:
        case PH_START:
            if (steps_left == 0u) return phase == PH_START ? PH_DONE : PH_TAIL;
            if (sort & SORT_CELLS) return patch ? PH_PATCH : PH_HEAD;
            break;
        case PH_PATCH:
            // the force phase patches the cell offsets itself where nothing reads them before
            if (rebuild || d.sys.contactmodel == 1) return PH_OFFSETS;
            break;
        case PH_WALL_SUMS: return PH_WALLS;
        case PH_HEAD: return PH_DOWN;
        case PH_DOWN: return PH_SCATTER;
        case PH_SCATTER: return PH_ORDER;
        case PH_TAIL:
        case PH_DONE: return PH_DONE;
        default: break;
    }
    if (phase != PH_REBUILD && phase != PH_BONDS && rebuild) return PH_REBUILD;
    if (phase != PH_BONDS && d.nb0) return PH_BONDS;
    return PH_FORCE;
}

// MODEL: the contact model.  QUAD: four lanes a sphere (one system); otherwise
// one, whose search and force then run in one thread: the slot masks, the
// particle's position and its slot words stay where the search left them, and
// the force of one block hides the search of another.  us a step as stages and
// as this chain: settling 990 spheres 47 and 16 (calls of 100 steps), 16,384 sheared 65 and 28,
// 32,000 bonded 84 and 48; one lane a sphere: 131,072-sphere crystal 69 and 50,
// 1,048,576 461 and 393 (mixed precision 363 and 293), loose packing of 131,071
// under a moving wall 53 and 35, contact model 1 of 262,144 80 and 53; a
// sheared box of 2,000,000, which sorts at most steps, 977 and 984.
// Bound by latency in the small systems (one dependent launch a step, then the
// loads that one sphere's index leads to), by HBM in the large: the force phase
// of the 1,048,576-sphere crystal moves 1.60 GB at 4.1 TB/s where a copy
// reaches 5.0.
// The step views lie in memory that no kernel writes and are read through the
// constant address space: like kernel arguments, but chosen by the step, and an
// argument list of 1.6 KB less to a launch.
template <class T, int MODEL, bool QUAD, bool B>
__global__ __launch_bounds__(BLOCK, QUAD ? 2 : 3) void k_chain(const DemDev* views, uint32_t* nstate, uint32_t own,
                                                               uint32_t steps, uint32_t launch) {
    static_assert(!B || (!QUAD && MODEL == 2), "ensembles: one lane a sphere, contact model 2");
    __shared__ uint32_t sw_all[NC * BLOCK];  // slot words; the scans' and sums' scratch in other phases
    using Const = const __attribute__((address_space(4))) DemDev*;
    uint32_t* const chain = nstate + NSTATE_CHAIN;
    uint32_t* const ctl = nstate + NSTATE_CTL;
    const uint32_t* const was = ctl + (launch & 1u) * CHAIN_WORDS;
    const uint32_t i = launch ? was[CHAIN_STEPS] : 0u;
    const DemDev& d = (const DemDev&)*((Const)(uintptr_t)views + (i ? 1u + i % 6u : 0u));
    uint32_t word[FW_WORDS];
    {
        const uint32_t* const from = i ? chain + (i % 3u) * FW_WORDS : nstate + own * FW_WORDS;
#pragma unroll
        for (uint32_t w = 0; w < FW_WORDS; ++w) word[w] = from[w];
    }
    const uint32_t sort = word[FW_SORT], changed = word[FW_CHANGED];
    const Words wd = {(sort & SORT_CELLS) != 0u, word[FW_REBUILD] != 0u, word[FW_WRAP] != 0u, nstate[NSTATE_ALIGNED] != 0u};
    const bool patch = wd.sorted && changed != 0u && changed <= PATCH_MAX;
    const uint32_t phase = next_phase(d, launch ? was[CHAIN_PHASE] : PH_START, steps - i, sort, patch, wd.rebuild);
    const uint32_t b = blockIdx.x, t = threadIdx.x;
    const bool first = b == 0u && t == 0u;
    if (first) {
        uint32_t* now = ctl + ((launch & 1u) ^ 1u) * CHAIN_WORDS;
        now[CHAIN_PHASE] = phase;
        now[CHAIN_STEPS] = i + (phase == PH_FORCE ? 1u : 0u);
        uint32_t used = launch ? was[CHAIN_USED] : 0u;  // launches with work
        if (phase == PH_FORCE) used = wd.sorted ? used | CHAIN_SORTED : used & ~CHAIN_SORTED;
        now[CHAIN_USED] = used + (phase < PH_TAIL ? 1u : 0u);
    }
    switch (phase) {
        case PH_HEAD:
            if (first) nstate[NSTATE_ALIGNED] = 0u;
            if (b < d.scan_blocks) scan_reduce(d, b, sw_all);
            break;
        case PH_DOWN:
            if (b < d.scan_blocks) scan_down(d, b, sw_all);
            break;
        case PH_SCATTER:
            if (const uint32_t q = xcd_item(d.np); q < d.np) place(d, q);
            break;
        case PH_ORDER: {
            const uint32_t nb = (d.K + BLOCK - 1) / BLOCK;
            if (b < nb) order_cells(d, xcd_block(nb));
            break;
        }
        case PH_PATCH: {
            if (first) nstate[NSTATE_ALIGNED] = 0u;
            uint4* list = reinterpret_cast<uint4*>(sw_all);
            if (b * BLOCK >= d.np) break;
            if (t < changed) list[t] = d.change_in[t];
            __syncthreads();
            if (b * BLOCK + t < d.np) patch_order(d, list, changed, b * BLOCK + t);
            break;
        }
        case PH_OFFSETS: patch_offsets(d, d.change_in, changed, b, reinterpret_cast<uint4*>(sw_all)); break;
        case PH_REBUILD: {
            if (first) {
                d.nstate[NSTATE_BUILDS] += 1u;
                d.nstate[NSTATE_ALIGNED] = 1u;
            }
            const uint32_t s = xcd_item(d.np);
            if (s < d.np) rows_search<true, B>(d, wd, s, sw_all + t, BLOCK);
            break;
        }
        case PH_BONDS:
            if (b * BLOCK + t < d.nb0) bond_force(d, b * BLOCK + t);
            break;
        case PH_FORCE: {
            if (first) {
                if (word[FW_ERR]) atomicOr(d.flags, word[FW_ERR]);
                uint32_t* clear = chain + ((i + 2u) % 3u) * FW_WORDS;
                for (uint32_t w = 0; w < FW_WORDS; ++w) clear[w] = 0u;
            }
            if (patch && !wd.rebuild && MODEL != 1) {
                patch_offsets(d, d.change_in, changed, b, reinterpret_cast<uint4*>(sw_all));
                __syncthreads();
            }
            if constexpr (!QUAD) {
                const uint32_t s = xcd_item(d.np);
                if (s < d.np) {
                    Slots sl = {0u, 0u};
                    if (MODEL != 1 && wd.rebuild) sl = {d.tmask[s], d.tfresh[s]};
                    else if (MODEL != 1) sl = list_search<B, BLOCK, true>(d, wd, s, sw_all + t);
                    force_particle<T, B, false, MODEL == 3, true>(d, wd, i + 1u == steps, s, sl);
                }
                if (b == 0u && !d.wall_launches)
                    for (uint32_t k = t; k < d.nsys; k += BLOCK) d.t_cur[k] += B ? d.systems[k].dt : d.sys.dt;
                break;
            }
            const uint32_t nq = (d.np + QUAD_N - 1) / QUAD_N;
            const uint32_t s = b < nq ? xcd_block(nq) * QUAD_N + (t >> 2) : d.np;
            double product = 0.0;
            if (s < d.np)
                product = quad_step<T, MODEL>(d, wd, s, t & 3u, i, i + 1u == steps,
                                              QuadCols{sw_all + (t >> 2), sw_all + NC * QUAD_N + (t >> 2),
                                                       reinterpret_cast<uint64_t*>(sw_all + 2 * NC * QUAD_N) + (t >> 2)});
            if (d.rec.wobj) {
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) product += __shfl_xor(product, o, 64);
                if ((t & 63u) == 0u && product != 0.0) unsafeAtomicAdd(d.rec.obj, product);
            }
            if (d.rec.x && b == 0u && t < 6u) {
                d.rec.wnx[6 * (d.rec.step0 + i) + t] = d.wnx[t];
                d.rec.wmvfd[6 * (d.rec.step0 + i) + t] = d.wmvfd[t];
            }
            if (first && !d.wall_launches) d.t_cur[0] += d.sys.dt;
            break;
        }
        case PH_WALL_SUMS: wall_partials<B>(d, b * (BLOCK / 64) + (t >> 6)); break;
        case PH_WALLS:
            if (b >= d.nsys) break;
            if (d.wall_launches == 2u) walls_update<B>(d, b);
            else walls_sum_update<B>(d, b, reinterpret_cast<double*>(sw_all));
            break;
        case PH_TAIL:
            if (b * BLOCK + t < d.np) {
                const uint32_t q = b * BLOCK + t;
                if (!(was[CHAIN_USED] & CHAIN_SORTED)) d.perm[q] = q;  // (the last step kept the order)
                if (i & 1u) d.pos_out[q] = d.pos_of[q];  // (the handle's array is that of even steps)
            }
            own ^= i & 1u;
            if (b == 0u && t < PATCH_MAX) d.changes[own * PATCH_MAX + t] = d.change_in[t];
            if (first) {
                for (uint32_t w = 0; w < FW_WORDS; ++w) nstate[own * FW_WORDS + w] = word[w];
                for (uint32_t w = 0; w < 3 * FW_WORDS; ++w) chain[w] = 0u;
            }
            break;
        default: break;
    }
}

// A per-particle field in the original order, for a read-back: one thread per
// stored particle.  The copy to the host then moves the finished field and
// nothing else.  (Bound by the scattered stores of nc doubles; the order of
// storage follows the cells, so they go to few lines when the input's order
// does too.)
__global__ __launch_bounds__(BLOCK) void k_gather_field(GatherField g, const uint32_t* __restrict__ id, uint32_t q0,
                                                        uint32_t n, uint32_t base, double* __restrict__ dst) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const size_t q = (size_t)q0 + i;
    double* out = dst + (size_t)g.nc * (id[q] - base);
#pragma unroll
    for (uint32_t c = 0; c < 4; ++c)
        if (c < g.nc) out[c] = g.src[c][g.stride * q];
}

// Every copy of a list, block row y the y-th: a state of some thousand spheres
// is thirty-odd arrays of a few KB to MB, and a copy call for each costs more
// than the bytes (the 16 bytes a lane moves are the widest there are).
__global__ __launch_bounds__(BLOCK) void k_copies(CopyList c) {
    const uint32_t r = blockIdx.y;
    const uint64_t n16 = c.bytes[r] >> 4, step = (uint64_t)gridDim.x * BLOCK;
    const uint4* const src = static_cast<const uint4*>(c.src[r]);
    uint4* const dst = static_cast<uint4*>(c.dst[r]);
    const uint64_t i0 = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
    for (uint64_t i = i0; i < n16; i += step) dst[i] = src[i];
    const uint32_t words = (uint32_t)(c.bytes[r] >> 2) & 3u;
    if (i0 < words) reinterpret_cast<uint32_t*>(dst + n16)[i0] = reinterpret_cast<const uint32_t*>(src + n16)[i0];
}

// Plain streaming copy used to calibrate bandwidth counters.
__global__ __launch_bounds__(BLOCK) void k_copy_probe(const double4* __restrict__ src, double4* __restrict__ dst,
                                                      uint64_t n) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

// Counter calibration: every thread runs `iters` rounds of 8 independent
// fused multiply-adds, i.e. exactly 16 * iters floating-point operations,
// and stores one value so that nothing is removed.
template <class T>
__global__ __launch_bounds__(BLOCK) void k_flops_probe(T* __restrict__ out, uint32_t iters, T a, T b) {
    T acc[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) acc[k] = (T)(threadIdx.x + k);
    for (uint32_t it = 0; it < iters; ++it) {
#pragma unroll
        for (int k = 0; k < 8; ++k) acc[k] = fma(acc[k], a, b);
    }
    T sum = acc[0];
#pragma unroll
    for (int k = 1; k < 8; ++k) sum += acc[k];  // (7 adds, outside the counted work's 16 * iters)
    out[(size_t)blockIdx.x * blockDim.x + threadIdx.x] = sum;
}

inline uint32_t nblk(uint64_t n, uint32_t b = BLOCK) { return (uint32_t)((n + b - 1) / b); }

}  // namespace

void launch_fill_u32(uint32_t* p, uint64_t n, uint32_t v, hipStream_t s) {
    if (n) k_fill_u32<<<nblk(n), BLOCK, 0, s>>>(p, n, v);
}
void launch_bonds(const DemDev& d, hipStream_t s) {
    if (d.nb0) k_bonds<<<nblk(d.nb0), BLOCK, 0, s>>>(d);
}
void launch_cellid(const DemDev& d, hipStream_t s) {
    if (d.systems) k_cellid<true><<<nblk(d.np), BLOCK, 0, s>>>(d);
    else k_cellid<false><<<nblk(d.np), BLOCK, 0, s>>>(d);
}
void launch_scan(const DemDev& d, bool lead, hipStream_t s) {
    const bool ens = d.systems != nullptr;
    if (lead) {
        const uint32_t nb = std::max(std::max(d.scan_blocks, nblk(d.np)), nblk(d.nwall_blocks, BLOCK / 64));
        if (ens) k_head<true, true><<<nb, BLOCK, 0, s>>>(d);
        else k_head<false, true><<<nb, BLOCK, 0, s>>>(d);
    } else {
        k_head<false, false><<<d.scan_blocks, BLOCK, 0, s>>>(d);
    }
    k_scan_down<<<d.scan_blocks, BLOCK, 0, s>>>(d);
}
void launch_scatter(const DemDev& d, hipStream_t s) { k_scatter<<<nblk(d.np), BLOCK, 0, s>>>(d); }
void launch_order(const DemDev& d, hipStream_t s) { k_order<<<nblk(d.K), BLOCK, 0, s>>>(d); }
void launch_walls(const DemDev& d, hipStream_t s) {
    if (d.systems) k_walls<true><<<d.nsys, BLOCK, 0, s>>>(d);
    else k_walls<false><<<1, BLOCK, 0, s>>>(d);
}
void launch_tail(const DemDev& d, hipStream_t s) {
    const uint32_t nb = std::max(nblk(d.np), nblk(d.nwall_blocks, BLOCK / 64));
    if (d.systems) k_tail<true><<<nb, BLOCK, 0, s>>>(d);
    else k_tail<false><<<nb, BLOCK, 0, s>>>(d);
    launch_walls(d, s);
}
template <bool B>
void topology(DemDev d, bool lead, hipStream_t s) {
    d.lead_blocks = lead ? (B ? d.nsys : 1u) : 0u;
    const uint32_t lb = d.lead_blocks;
    const bool slots = B || d.sys.contactmodel != 1;  // contact model 1 keeps no slots (src/device.cu:809)
    if (slots && d.search_mode == 5) {  // one of the two returns at once (FW_REBUILD)
        DemDev e = d;
        e.lead_blocks = 0;
        k_topo_rows<true, B><<<nblk(d.np, d.tpb_search), d.tpb_search, NC * 4 * d.tpb_search, s>>>(e);
        k_list_search<B><<<lb + nblk(d.np, APPLY_BLOCK), APPLY_BLOCK, 0, s>>>(d);
    } else if (slots && d.search_mode == 4) {  // hcnt starts at zero: k_topo_apply clears it
        k_topo_half<B><<<nblk(d.np, d.tpb_search), d.tpb_search, 0, s>>>(d);
        k_topo_apply<B><<<lb + nblk(d.np, APPLY_BLOCK), APPLY_BLOCK, 0, s>>>(d);
    } else if (slots && d.search_mode == 2) {
        k_topo_rows<false, B><<<lb + nblk(d.np, d.tpb_search), d.tpb_search, NC * 4 * d.tpb_search, s>>>(d);
    } else {
        if (lead) launch_walls(d, s);
        if (!slots || B) return;  // (modes 1 and 3 walk one grid; the host refuses them for ensembles)
        if (d.search_mode == 3) k_topo_wave<<<(d.K + BLOCK / 64 - 1) / (BLOCK / 64), BLOCK, 0, s>>>(d);
        else k_topo<<<d.tiles_x * d.tiles_y * d.sys.num[2], BLOCK, 0, s>>>(d);
    }
}
void launch_topology(const DemDev& d, bool lead, hipStream_t s) {
    if (d.systems) topology<true>(d, lead, s);
    else topology<false>(d, lead, s);
}
template <bool B, bool VW>
void forces(const DemDev& d, bool mixed, hipStream_t s) {
    if (mixed) k_force<float, B, VW><<<nblk(d.np, d.tpb_force), d.tpb_force, 0, s>>>(d);
    else if (!B && d.sys.contactmodel == 3) k_force<double, false, VW, true><<<nblk(d.np, d.tpb_force), d.tpb_force, 0, s>>>(d);
    else k_force<double, B, VW><<<nblk(d.np, d.tpb_force), d.tpb_force, 0, s>>>(d);
}
void launch_forces(const DemDev& d, int precision, hipStream_t s) {
    const bool mixed = precision == SPH_PREC_MIXED;
    if (d.systems) {
        if (d.force_vw) forces<true, true>(d, mixed, s);
        else forces<true, false>(d, mixed, s);
    } else {
        if (d.force_vw) forces<false, true>(d, mixed, s);
        else forces<false, false>(d, mixed, s);
    }
}
template <class T, int MODEL, bool QUAD, bool B>
void chain(const DemDev& d, const DemDev* views, uint32_t steps, uint32_t l, hipStream_t s) {
    const uint32_t nb = std::max({nblk((QUAD ? 4 : 1) * (uint64_t)d.np), nblk(d.K), d.scan_blocks, nblk(d.nb0), d.nsys});
    k_chain<T, MODEL, QUAD, B><<<nb, BLOCK, 0, s>>>(views, d.nstate, d.fr == d.nstate ? 0u : 1u, steps, l);
}
template <bool QUAD>
void chain_model(const DemDev& d, const DemDev* views, bool mixed, uint32_t steps, uint32_t l, hipStream_t s) {
    if (d.sys.contactmodel == 1) chain<double, 1, QUAD, false>(d, views, steps, l, s);
    else if (mixed) chain<float, 2, QUAD, false>(d, views, steps, l, s);
    else if (d.sys.contactmodel == 3) chain<double, 3, QUAD, false>(d, views, steps, l, s);
    else chain<double, 2, QUAD, false>(d, views, steps, l, s);
}
void launch_chain(const DemDev& d, const DemDev* views, int precision, uint32_t steps, uint32_t l, hipStream_t s) {
    const bool mixed = precision == SPH_PREC_MIXED;
    if (d.systems && mixed) chain<float, 2, false, true>(d, views, steps, l, s);
    else if (d.systems) chain<double, 2, false, true>(d, views, steps, l, s);
    else if (d.np <= QUAD_NP) chain_model<true>(d, views, mixed, steps, l, s);
    else chain_model<false>(d, views, mixed, steps, l, s);
}
void launch_copy_probe(const double4* src, double4* dst, uint64_t n, hipStream_t s) {
    k_copy_probe<<<2048, BLOCK, 0, s>>>(src, dst, n);
}
void launch_flops_probe(void* out, uint32_t blocks, uint32_t iters, bool fp64, hipStream_t s) {
    if (fp64) k_flops_probe<double><<<blocks, BLOCK, 0, s>>>(static_cast<double*>(out), iters, 0.999999, 1e-7);
    else k_flops_probe<float><<<blocks, BLOCK, 0, s>>>(static_cast<float*>(out), iters, 0.999999f, 1e-7f);
}
void launch_gather_field(const GatherField& g, const uint32_t* id, uint32_t q0, uint32_t n, uint32_t base, double* dst,
                         hipStream_t s) {
    if (n) k_gather_field<<<nblk(n), BLOCK, 0, s>>>(g, id, q0, n, base, dst);
}
void launch_copies(const CopyList& c, hipStream_t s) {
    uint64_t most = 0;
    for (uint32_t k = 0; k < c.n; ++k) most = std::max(most, c.bytes[k]);
    if (c.n && most) k_copies<<<dim3(std::min(nblk(most / 16 + 1), 1024u), c.n), BLOCK, 0, s>>>(c);
}
void launch_f32_copies(const DemDev& d, hipStream_t s) { k_f32_copies<<<nblk(d.np), BLOCK, 0, s>>>(d); }
}  // namespace sph
