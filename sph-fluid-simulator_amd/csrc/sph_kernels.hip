// sph_kernels.hip -- hand-written CDNA4 (gfx950) kernels of one SPH step.
//
// One step is, in launch order:
//   scan          exclusive scan of per-cell counts -> cstart, counts := 0,
//                 and the list of cells holding more than kSmallCell
//   scatter       perm[cstart[cell] + rank] = A index
//   sort_big      sorts the A indices inside each listed big cell
//   reorder       stable cell order (ties by A index), gather A -> B
//   plan          how every wave walks its candidates; short walks get their
//                 density and neighbour lists here
//   density       poly6 density + pressure        (src/sph.cpp:28-76)
//   force_integrate
//                 spiky pressure + viscosity force (src/sph.cpp:80-129),
//                 symplectic Euler + walls          (src/sph.cpp:133-181),
//                 then the next step's cell key and in-cell rank
// The hash / sort / table passes of the reference (src/sph.cpp:17-24,
// 184-192, src/neighborTable.cpp:19-37) are replaced by the dense-grid
// counting sort; the reference's 16-bit bucket semantics are kept through
// the multiplicity rule documented in sph_common.h.
//
// Floating-point contraction is off for the whole file: the squared
// distance must be fl(fl(fl(dx*dx) + fl(dy*dy)) + fl(dz*dz)) as glm forms it,
// and integration reproduces the reference's rounding step by step.  The
// force pass uses explicit fmaf() where the reference's rounding is not the
// contract (tolerance-checked sums).
#include "sph_kernels.h"

#include <algorithm>
#include <type_traits>

#pragma clang fp contract(off)

namespace sph {

// Blocks are dispatched round-robin over the 8 XCDs (block b -> XCD b % 8).
// Re-map so each XCD walks a contiguous range of particles: neighbouring
// cells then share one XCD's L2.
__device__ inline uint32_t xcd_block()
{
    uint32_t b = blockIdx.x, nb = gridDim.x;
    uint32_t per = nb >> 3, rem = nb & 7u;
    uint32_t xcd = b & 7u, k = b >> 3;
    return xcd * per + (xcd < rem ? xcd : rem) + k;
}

// The wave task of the calling wave: its scene (wave-uniform, so the
// scene's constants are scalar loads) and its slot.  Returns false for
// waves past the task list and lanes past the scene's last slot.
struct Lane {
    const StepParams *P;
    uint32_t slot;
    uint32_t first;  // first slot of the wave (wave-uniform)
    uint32_t task;   // index of the wave task (wave-uniform)
};

template <int BLOCK>
__device__ inline bool lane_of(const SceneSet &S, Lane &out)
{
    const uint32_t w = __builtin_amdgcn_readfirstlane(xcd_block() * (BLOCK / 64) + (threadIdx.x >> 6));
    if (w >= S.nwaves)
        return false;
    const WaveTask t = S.tasks[w];
    const uint32_t scene = __builtin_amdgcn_readfirstlane(t.scene);
    const uint32_t first = __builtin_amdgcn_readfirstlane(t.first);
    out.P = S.params + scene;
    out.first = first;
    out.slot = first + (threadIdx.x & 63u);
    return out.slot < out.P->p_end;
}

// Wave task w (wave-uniform) with every lane live: lanes past the scene's
// last slot mirror the wave's first slot (always a valid slot) and report
// active = false, so wave-wide votes and shuffles see defined data.
__device__ inline void wave_task(const SceneSet &S, uint32_t w, Lane &out, bool &active)
{
    const WaveTask t = S.tasks[w];
    const uint32_t scene = __builtin_amdgcn_readfirstlane(t.scene);
    const uint32_t first = __builtin_amdgcn_readfirstlane(t.first);
    out.P = S.params + scene;
    out.first = first;
    out.task = w;
    const uint32_t slot = first + (threadIdx.x & 63u);
    active = slot < out.P->p_end;
    out.slot = active ? slot : first;
}

inline uint32_t blocks_for_waves(uint32_t nwaves, int block) { return (nwaves + block / 64 - 1) / (block / 64); }

// Waves the device holds at once: CUs x 4 SIMDs x 8 wave slots.
uint32_t resident_waves()
{
    static uint32_t cached = 0;
    if (!cached) {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
            cus = 256;
        cached = 32u * (uint32_t)cus;
    }
    return cached;
}

// ---------------------------------------------------------------- utilities

__global__ void k_fill_u32(uint32_t *__restrict__ p, uint32_t value, size_t n)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride)
        p[i] = value;
}

void launch_fill_u32(hipStream_t st, uint32_t *p, uint32_t value, size_t n)
{
    if (n == 0)
        return;
    size_t nb = (n + kBlock - 1) / kBlock;
    if (nb > 4096)
        nb = 4096;
    hipLaunchKernelGGL(k_fill_u32, dim3((uint32_t)nb), dim3(kBlock), 0, st, p, value, n);
}

// Reference Particle AoS (60 bytes) -> posA/velA with id = input index.
__global__ void k_unpack_aos(const float *__restrict__ aos, uint32_t n, float4 *__restrict__ posA,
                             float4 *__restrict__ velA)
{
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n)
        return;
    const float *p = aos + (size_t)i * 15;
    posA[i] = make_float4(p[0], p[1], p[2], 0.0f);
    velA[i] = make_float4(p[3], p[4], p[5], __uint_as_float(i));
}

void launch_unpack_aos(hipStream_t st, const void *aos, uint32_t n, float4 *posA, float4 *velA)
{
    hipLaunchKernelGGL(k_unpack_aos, dim3(blocks_for(n)), dim3(kBlock), 0, st,
                       (const float *)aos, n, posA, velA);
}

// Order-preserving float <-> int map for atomic min/max.
__device__ inline int32_t ordered_int(float f)
{
    int32_t i = __float_as_int(f);
    return i >= 0 ? i : (int32_t)(i ^ 0x7FFFFFFF);
}

__device__ inline void widen(int32_t (&v)[6], float x, float y, float z)
{
    const float c[3] = {x, y, z};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        if (c[k] - c[k] == 0.0f) {  // finite
            const int32_t o = ordered_int(c[k]);
            v[k] = min(v[k], o);
            v[k + 3] = max(v[k + 3], o);
        }
    }
}

// Joins every thread's bounds into bbox6: six atomics a block.
__device__ inline void join_bounds(const int32_t (&v)[6], int32_t *__restrict__ bbox6)
{
    __shared__ int32_t red[6][kBlock / 64];
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        int32_t x = v[k];
        for (int d = 32; d >= 1; d >>= 1) {
            int32_t y = __shfl_xor(x, d, 64);
            x = (k < 3) ? min(x, y) : max(x, y);
        }
        if ((threadIdx.x & 63) == 0)
            red[k][threadIdx.x >> 6] = x;
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        int k = threadIdx.x;
        int32_t x = red[k][0];
        for (int w = 1; w < kBlock / 64; ++w)
            x = (k < 3) ? min(x, red[k][w]) : max(x, red[k][w]);
        if (k < 3)
            atomicMin(&bbox6[k], x);
        else
            atomicMax(&bbox6[k], x);
    }
}

// Bounding box of finite positions: bbox6 = {min x,y,z, max x,y,z} as
// ordered ints.  kBoundsBlocks blocks at most: what the pass costs is its
// atomics on six addresses (one block per 256 particles took 26 us at 262
// thousand of them).
constexpr uint32_t kBoundsBlocks = 128;

__global__ void k_bbox_init(int32_t *__restrict__ bbox6)
{
    if (threadIdx.x < 6u)
        bbox6[threadIdx.x] = threadIdx.x < 3u ? INT32_MAX : INT32_MIN;
}

__global__ __launch_bounds__(kBlock) void k_bbox(const float4 *__restrict__ pos, uint32_t n,
                                                int32_t *__restrict__ bbox6)
{
    int32_t v[6] = {INT32_MAX, INT32_MAX, INT32_MAX, INT32_MIN, INT32_MIN, INT32_MIN};
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        const float4 p = pos[i];
        widen(v, p.x, p.y, p.z);
    }
    join_bounds(v, bbox6);
}

void launch_bbox(hipStream_t st, const float4 *pos, uint32_t n, int32_t *bbox6)
{
    hipLaunchKernelGGL(k_bbox_init, dim3(1), dim3(64), 0, st, bbox6);
    hipLaunchKernelGGL(k_bbox, dim3(std::min(blocks_for(n), kBoundsBlocks)), dim3(kBlock), 0, st, pos, n, bbox6);
}

// A scene's state from the caller's arrays (three floats a particle; vel may
// be null) into slots [first, first + n): ids in order, everything a step
// has not yet computed cleared, and the bounds of the finite positions.
__global__ __launch_bounds__(kBlock) void k_load_state(const float *__restrict__ pos3, const float *__restrict__ vel3,
                                                      ParticleArrays a, float4 *__restrict__ force, uint32_t first,
                                                      uint32_t n, int32_t *__restrict__ bbox6)
{
    int32_t v[6] = {INT32_MAX, INT32_MAX, INT32_MAX, INT32_MIN, INT32_MIN, INT32_MIN};
    const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        const size_t k = 3 * (size_t)i, s = (size_t)first + i;
        const float x = pos3[k], y = pos3[k + 1], z = pos3[k + 2];
        widen(v, x, y, z);
        a.posA[s] = make_float4(x, y, z, 0.0f);
        a.velA[s] = vel3 ? make_float4(vel3[k], vel3[k + 1], vel3[k + 2], __uint_as_float(i))
                         : make_float4(0.0f, 0.0f, 0.0f, __uint_as_float(i));
        a.rhoB[s] = 0.0f;
        a.posB[s] = zero;
        a.posR[s] = zero;
        a.velR[s] = zero;
        if (force)
            force[s] = zero;
    }
    join_bounds(v, bbox6);
}

void launch_load_state(hipStream_t st, const float *pos3, const float *vel3, const ParticleArrays &a, float4 *force,
                       uint32_t first, uint32_t n, int32_t *bbox6)
{
    hipLaunchKernelGGL(k_bbox_init, dim3(1), dim3(64), 0, st, bbox6);
    hipLaunchKernelGGL(k_load_state, dim3(std::min(blocks_for(n), 4u * kBoundsBlocks)), dim3(kBlock), 0, st, pos3,
                       vel3, a, force, first, n, bbox6);
}

// The downloaded quantities of slots [first, first + n), each an array of its
// own (null: not wanted): positions, velocities, densities, pressures, ids.
__global__ __launch_bounds__(kBlock) void k_store_state(ParticleArrays a, uint32_t first, uint32_t n,
                                                       float *__restrict__ pos3, float *__restrict__ vel3,
                                                       float *__restrict__ rho, float *__restrict__ pressure,
                                                       uint32_t *__restrict__ ids)
{
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n)
        return;
    const size_t k = 3 * (size_t)i, s = (size_t)first + i;
    if (pos3) {
        const float4 x = a.posA[s];
        pos3[k] = x.x;
        pos3[k + 1] = x.y;
        pos3[k + 2] = x.z;
    }
    if (vel3 || ids) {
        const float4 v = a.velA[s];
        if (vel3) {
            vel3[k] = v.x;
            vel3[k + 1] = v.y;
            vel3[k + 2] = v.z;
        }
        if (ids)
            ids[i] = __float_as_uint(v.w);
    }
    if (rho)
        rho[i] = a.rhoB[s];
    if (pressure)
        pressure[i] = a.velR[s].w;
}

void launch_store_state(hipStream_t st, const ParticleArrays &a, uint32_t first, uint32_t n, float *pos3, float *vel3,
                        float *rho, float *pressure, uint32_t *ids)
{
    hipLaunchKernelGGL(k_store_state, dim3(blocks_for(n)), dim3(kBlock), 0, st, a, first, n, pos3, vel3, rho, pressure,
                       ids);
}

// Cell key and bucket of the positions in posA, counted into their cells
// (the count is not read back here: the scatter ranks the particles).
__global__ __launch_bounds__(kBlock) void k_init_keys(float4 *__restrict__ posA,
                                                     uint32_t *__restrict__ cellcA,
                                                     uint32_t *__restrict__ counts, SceneSet S)
{
    Lane L;
    if (!lane_of<kBlock>(S, L))
        return;
    const StepParams &P = *L.P;
    const uint32_t i = L.slot;
    float4 p = posA[i];
    Classified c = classify(p.x, p.y, p.z, P);
    posA[i].w = __uint_as_float(c.h16);
    cellcA[i] = c.cellc;
    atomicAdd(&counts[linear_cell(P, c.cellc)], 1u);
}

void launch_init_keys(hipStream_t st, const ParticleArrays &a, const CellArrays &c, const SceneSet &S)
{
    hipLaunchKernelGGL(k_init_keys, dim3(blocks_for_waves(S.nwaves, kBlock)), dim3(kBlock), 0, st,
                       a.posA, a.cellcA, c.counts, S);
}

// ------------------------------------------------------------- cell scan
// Three passes over the (padded) cell array: per-block totals, a one-block
// scan of the totals, then the block-local exclusive scan plus offset.  The
// last pass appends every cell above kSmallCell to the big-cell list and,
// when asked, clears the counts (the cell scan leaves them: the scatter
// counts them back down to zero while it ranks the particles).

__device__ inline uint32_t wave_inclusive_scan(uint32_t x)
{
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        uint32_t y = __shfl_up(x, d, 64);
        if (lane >= d)
            x += y;
    }
    return x;
}

// Exclusive scan across the block of one value per thread; returns the
// exclusive prefix and writes the block total.
__device__ inline uint32_t block_exclusive_scan(uint32_t x, uint32_t *total)
{
    __shared__ uint32_t wsum[kBlock / 64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t inc = wave_inclusive_scan(x);
    if (lane == 63)
        wsum[wave] = inc;
    __syncthreads();
    uint32_t off = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w) {
        uint32_t s = wsum[w];
        off += (w < wave) ? s : 0u;
        tot += s;
    }
    __syncthreads();
    *total = tot;
    return off + inc - x;
}

__global__ void k_scan_reduce(const uint32_t *__restrict__ counts, uint32_t *__restrict__ partials,
                              uint32_t *__restrict__ big)
{
    if (big && blockIdx.x == 0u && threadIdx.x == 0u)
        big[0] = 0u;  // the big-cell count
    const uint4 *src = (const uint4 *)(counts + (size_t)blockIdx.x * kScanChunk);
    uint32_t s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems / 4; ++k) {
        uint4 v = src[k * kBlock + threadIdx.x];
        s += v.x + v.y + v.z + v.w;
    }
    uint32_t tot;
    block_exclusive_scan(s, &tot);
    if (threadIdx.x == 0)
        partials[blockIdx.x] = tot;
}

// One block: exclusive scan of nparts block totals in place.
__global__ void k_scan_partials(uint32_t *__restrict__ partials, uint32_t nparts)
{
    uint32_t carry = 0;
    for (uint32_t base = 0; base < nparts; base += kBlock) {
        uint32_t i = base + threadIdx.x;
        uint32_t x = i < nparts ? partials[i] : 0u;
        uint32_t tot;
        uint32_t ex = block_exclusive_scan(x, &tot);
        if (i < nparts)
            partials[i] = carry + ex;
        carry += tot;
    }
}

// SUMS: partials holds the blocks' own totals, and each block adds up those
// before it; otherwise k_scan_partials has.
template <bool SUMS>
__global__ void k_scan_final(uint32_t *__restrict__ counts, const uint32_t *__restrict__ partials,
                             uint32_t *__restrict__ cstart, uint32_t *__restrict__ big, uint32_t big_cap,
                             bool clear)
{
    size_t base = (size_t)blockIdx.x * kScanChunk + (size_t)threadIdx.x * kScanItems;
    uint4 *src = (uint4 *)(counts + base);
    uint32_t before = 0;
    if (SUMS)
        for (uint32_t b = threadIdx.x; b < blockIdx.x; b += kBlock)
            before += partials[b];
    uint32_t v[kScanItems];
#pragma unroll
    for (int k = 0; k < kScanItems / 4; ++k) {
        uint4 q = src[k];
        v[4 * k + 0] = q.x;
        v[4 * k + 1] = q.y;
        v[4 * k + 2] = q.z;
        v[4 * k + 3] = q.w;
    }
    uint32_t local = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k)
        local += v[k];
    uint32_t tot;
    uint32_t run = block_exclusive_scan(local, &tot);
    if (SUMS) {
        block_exclusive_scan(before, &tot);
        run += tot;
    } else {
        run += partials[blockIdx.x];
    }
    uint4 *dst = (uint4 *)(cstart + base);
#pragma unroll
    for (int k = 0; k < kScanItems / 4; ++k) {
        uint4 q;
        q.x = run;
        run += v[4 * k + 0];
        q.y = run;
        run += v[4 * k + 1];
        q.z = run;
        run += v[4 * k + 2];
        q.w = run;
        run += v[4 * k + 3];
        dst[k] = q;
        if (clear)
            src[k] = make_uint4(0u, 0u, 0u, 0u);
    }
    if (blockIdx.x + 1u == gridDim.x && threadIdx.x + 1u == blockDim.x)
        cstart[base + kScanItems] = run;  // the grand total, behind the last cell
    if (big) {
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) {
            if (v[k] > kSmallCell) {
                const uint32_t at = atomicAdd(&big[0], 1u);
                if (at < big_cap)
                    big[1 + at] = (uint32_t)(base + k);
            }
        }
    }
}

// Up to so many blocks each adds up the totals before it (a load or two a
// thread): one launch fewer, which at a few cells is what a scan costs
// (8,000 particles: 9.1 -> 8.2 us).  Beyond, those sums would read more than
// the scan does.
constexpr uint32_t kScanSumsMax = 1024;

void launch_scan(hipStream_t st, const CellArrays &c, bool clear_counts)
{
    uint32_t nparts = c.ncells_padded / kScanChunk;
    hipLaunchKernelGGL(k_scan_reduce, dim3(nparts), dim3(kBlock), 0, st, c.counts, c.partials, c.big);
    if (nparts <= kScanSumsMax) {
        hipLaunchKernelGGL((k_scan_final<true>), dim3(nparts), dim3(kBlock), 0, st, c.counts, c.partials, c.cstart,
                           c.big, c.big_cap, clear_counts);
        return;
    }
    hipLaunchKernelGGL(k_scan_partials, dim3(1), dim3(kBlock), 0, st, c.partials, nparts);
    hipLaunchKernelGGL((k_scan_final<false>), dim3(nparts), dim3(kBlock), 0, st, c.counts, c.partials, c.cstart, c.big,
                       c.big_cap, clear_counts);
}

// ---------------------------------------------------------- scatter/reorder

// Each particle takes a distinct place in its cell's range by counting the
// cell's count down (the order within a cell is fixed afterwards by the
// reorder), which also leaves the counts at zero for the next step.  The
// one atomic whose result a thread waits on is here, in a kernel that does
// nothing else, rather than at the end of the force pass.  Neighbouring lanes
// that share a cell (A is in the previous step's cell order: nearly all that
// do) take their places with one atomic: the lowest lane of each run subtracts
// the run's size, and every lane of the run adds its position in it.  (Finding
// all lanes of a cell, one ballot per cell of the wave, took 23 us for a
// million particles in as many cells; runs take 7.8.)
__global__ __launch_bounds__(kBlock) void k_scatter(const uint32_t *__restrict__ cellcA,
                                                   uint32_t *__restrict__ counts,
                                                   const uint32_t *__restrict__ cstart,
                                                   uint32_t *__restrict__ perm, SceneSet S)
{
    Lane L;
    if (!lane_of<kBlock>(S, L))
        return;
    const uint32_t i = L.slot;
    const uint32_t lin = linear_cell(*L.P, cellcA[i]);
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t live = (uint32_t)__builtin_popcountll(__ballot(1));  // the lowest ones
    const uint32_t before = (uint32_t)__shfl_up((int)lin, 1, 64);
    const uint64_t heads = __ballot(lane == 0u || lin != before);
    const uint32_t leader = 63u - (uint32_t)__builtin_clzll(heads & ((2ull << lane) - 1ull));
    const uint64_t above = lane == 63u ? 0ull : heads >> (lane + 1u);
    const uint32_t end = above ? lane + 1u + (uint32_t)__builtin_ctzll(above) : live;
    const uint32_t size = end - leader, offset = lane - leader;
    uint32_t top = 0;
    if (lane == leader)
        top = atomicSub(&counts[lin], size);  // one instruction for every run of the wave
    top = (uint32_t)__shfl((int)top, (int)leader, 64);
    perm[cstart[lin] + top - size + offset] = i;
}

void launch_scatter(hipStream_t st, const ParticleArrays &a, const CellArrays &c, const SceneSet &S)
{
    hipLaunchKernelGGL(k_scatter, dim3(blocks_for_waves(S.nwaves, kBlock)), dim3(kBlock), 0, st,
                       a.cellcA, c.counts, c.cstart, a.perm, S);
}

// Big cells: one block sorts the A indices of one listed cell (bitonic,
// ascending), so slot order inside the cell is the stable order.  Thread t
// holds elements t + kBigSortBlock j in registers: compare-exchanges at
// strides >= kBigSortBlock stay in the thread, strides < 64 are wave
// shuffles, and only strides 64 .. kBigSortBlock / 2 go through LDS (22 of
// the 91 stages of an 8192-element sort).  Blocks walk the list with a
// stride; every block exits when the list ends.
constexpr int kBigSortRegs = (int)(kBigCellSortMax / kBigSortBlock);

// Stages at stride Q kBigSortBlock: element j pairs with j | Q in the same
// thread (Q and the element count RR compile-time, so the register indices
// are fixed).
template <int RR, uint32_t Q>
__device__ inline void sort_stage_in_thread(uint32_t (&x)[RR], uint32_t t, uint32_t size)
{
#pragma unroll
    for (int j = 0; j < RR; ++j) {
        if (((uint32_t)j & Q) == 0u && (j | (int)Q) < RR) {
            const int jj = j | (int)Q;
            const bool up = ((t + (uint32_t)kBigSortBlock * (uint32_t)j) & size) == 0u;
            const uint32_t lo = min(x[j], x[jj]), hi = max(x[j], x[jj]);
            x[j] = up ? lo : hi;
            x[jj] = up ? hi : lo;
        }
    }
}

// Sorts the len (<= RR kBigSortBlock, > 64) entries of perm at b; m is the
// power of two >= len.  Called by every thread of the block.
template <int RR>
__device__ inline void sort_cell(uint32_t *__restrict__ perm, uint32_t b, uint32_t len, uint32_t m,
                                 uint32_t *__restrict__ sh)
{
    constexpr uint32_t T = kBigSortBlock;
    const uint32_t t = threadIdx.x;
    // m >= 128 is a multiple of 64: a wave is wholly live or wholly idle
    const bool live = t < m;
    uint32_t x[RR];
#pragma unroll
    for (int j = 0; j < RR; ++j) {
        const uint32_t k = t + T * (uint32_t)j;
        x[j] = k < len ? perm[b + k] : 0xFFFFFFFFu;
    }
    for (uint32_t size = 2; size <= m; size <<= 1) {
        for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
            if (stride >= T) {
                switch (stride / T) {
                case 1: sort_stage_in_thread<RR, 1>(x, t, size); break;
                case 2: sort_stage_in_thread<RR, 2>(x, t, size); break;
                case 4: sort_stage_in_thread<RR, 4>(x, t, size); break;
                default: sort_stage_in_thread<RR, 8>(x, t, size); break;
                }
            } else if (stride < 64u) {
                if (live) {
#pragma unroll
                    for (int j = 0; j < RR; ++j) {
                        const uint32_t k = t + T * (uint32_t)j;
                        const uint32_t y = (uint32_t)__shfl_xor((int)x[j], (int)stride, 64);
                        const bool up = (k & size) == 0u, low = (k & stride) == 0u;
                        x[j] = (low == up) ? min(x[j], y) : max(x[j], y);
                    }
                }
            } else {
                if (live) {
#pragma unroll
                    for (int j = 0; j < RR; ++j)
                        sh[t + T * (uint32_t)j] = x[j];
                }
                __syncthreads();
                if (live) {
#pragma unroll
                    for (int j = 0; j < RR; ++j) {
                        const uint32_t k = t + T * (uint32_t)j;
                        const uint32_t y = sh[k ^ stride];
                        const bool up = (k & size) == 0u, low = (k & stride) == 0u;
                        x[j] = (low == up) ? min(x[j], y) : max(x[j], y);
                    }
                }
                __syncthreads();
            }
        }
    }
#pragma unroll
    for (int j = 0; j < RR; ++j) {
        const uint32_t k = t + T * (uint32_t)j;
        if (k < len)
            perm[b + k] = x[j];
    }
}

__global__ __launch_bounds__(kBigSortBlock) void k_sort_big_cells(
    uint32_t *__restrict__ perm, const uint32_t *__restrict__ cstart, const uint32_t *__restrict__ big,
    uint32_t big_cap, unsigned long long *__restrict__ unordered)
{
    static_assert(kBigSortRegs == 16 && kSmallCell >= 64, "sort layout");
    __shared__ uint32_t sh[kBigCellSortMax];
    const uint32_t nbig = min(big[0], big_cap);
    for (uint32_t e = blockIdx.x; e < nbig; e += gridDim.x) {
        const uint32_t cell = big[1 + e];
        const uint32_t b = cstart[cell], len = cstart[cell + 1] - b;
        if (len > kBigCellSortMax) {  // uniform: keeps arrival order, counted
            if (threadIdx.x == 0 && unordered)
                atomicAdd(unordered, 1ull);
            continue;
        }
        uint32_t m = 1;
        while (m < len)
            m <<= 1;
        switch (m > (uint32_t)kBigSortBlock ? m / kBigSortBlock : 1u) {  // elements per thread
        case 1: sort_cell<1>(perm, b, len, m, sh); break;
        case 2: sort_cell<2>(perm, b, len, m, sh); break;
        case 4: sort_cell<4>(perm, b, len, m, sh); break;
        case 8: sort_cell<8>(perm, b, len, m, sh); break;
        default: sort_cell<16>(perm, b, len, m, sh); break;
        }
    }
}

void launch_sort_big_cells(hipStream_t st, const ParticleArrays &a, const CellArrays &c)
{
    if (!c.big)
        return;
    hipLaunchKernelGGL(k_sort_big_cells, dim3(kBigSortBlocks), dim3(kBigSortBlock), 0, st, a.perm,
                       c.cstart, c.big, c.big_cap, c.unordered);
}

// Slot s holds A index i; its stable destination is the cell start plus the
// number of smaller A indices in the same cell.  Cells above kSmallCell
// were sorted by k_sort_big_cells, so their destination is s itself.
__global__ __launch_bounds__(kBlock) void k_reorder(
    const uint32_t *__restrict__ perm, const uint32_t *__restrict__ cellcA,
    const uint32_t *__restrict__ cstart, const float4 *__restrict__ posA,
    const float4 *__restrict__ velA, float4 *__restrict__ posB, float4 *__restrict__ velB,
    uint32_t *__restrict__ cellcB, SceneSet S)
{
    Lane L;
    if (!lane_of<kBlock>(S, L))
        return;
    const uint32_t s = L.slot;
    const uint32_t i = perm[s];
    const uint32_t c = cellcA[i];
    const uint32_t lin = linear_cell(*L.P, c);
    const uint32_t b = cstart[lin], e = cstart[lin + 1];
    uint32_t d;
    if (e - b <= kSmallCell) {
        uint32_t r = 0;
        for (uint32_t t = b; t < e; ++t)
            r += (perm[t] < i) ? 1u : 0u;
        d = b + r;
    } else {
        d = s;
    }
    posB[d] = posA[i];
    velB[d] = velA[i];
    cellcB[d] = c;
}

void launch_reorder(hipStream_t st, const ParticleArrays &a, const CellArrays &c, const SceneSet &S)
{
    hipLaunchKernelGGL(k_reorder, dim3(blocks_for_waves(S.nwaves, kBlock)), dim3(kBlock), 0, st,
                       a.perm, a.cellcA, c.cstart, a.posA, a.velA, a.posB, a.velB, a.cellcB, S);
}

// ------------------------------------------------------------ stencil walk

// fl(fl(fl(dx*dx) + fl(dy*dy)) + fl(dz*dz)), dx = x_j - x_i: glm::length2.
__device__ inline float dist2_ref(float4 pi, float4 q, float &dx, float &dy, float &dz)
{
    dx = q.x - pi.x;
    dy = q.y - pi.y;
    dz = q.z - pi.z;
    return dx * dx + dy * dy + dz * dz;
}

// Correctly rounded sqrt for x >= 2^-96 (any d2 a neighbour pair can have
// short of coincident points; x = 0 also comes out exact): v_sqrt_f32 is
// within 1 ulp, and the neighbouring value whose residual x - s * s' changes
// sign is the correctly rounded root.
__device__ inline float sqrt_rn(float x)
{
    const float s = __builtin_amdgcn_sqrtf(x);
    const float down = __uint_as_float(__float_as_uint(s) - 1u);
    const float up = __uint_as_float(__float_as_uint(s) + 1u);
    const float below = fmaf(-down, s, x) <= 0.0f ? down : s;
    return fmaf(-up, s, x) > 0.0f ? up : below;
}

// The same root r and y = 1 / sqrt(x) within an ulp, for
// x >= 2^-96 (any d2 a neighbour pair can have short of coincident points,
// where both come out NaN / inf as the reference's division by r = 0 does):
// one Newton step on v_rsq_f32, whose result equals the rounded root for
// every mantissa at every exponent from -62 to 23 (all 2^23 of each tried
// against the double root).  One transcendental and four multiplies or fmas
// in place of v_sqrt, v_rcp and two compare-and-select corrections: 18 against
// 41 issue cycles a wave, and 1 / r is nearer (1.6 against 2.0 half-ulps).
__device__ inline float root(float x, float &y)
{
    y = __builtin_amdgcn_rsqf(x);
    const float r0 = x * y;
    return fmaf(fmaf(-r0, r0, x), 0.5f * y, r0);
}

// max(x, 0).  UNIT: x is at most 1, so a clamp to [0, 1] will do, which comes
// free with the operation that made x (v_max is an instruction of its own, at
// half the rate of an add).  NaN gives 0 either way.
template <bool UNIT>
__device__ inline float positive(float x)
{
    return UNIT ? __builtin_amdgcn_fmed3f(x, 0.0f, 1.0f) : fmaxf(x, 0.0f);
}

// x in a vector register: an instruction with a scalar-register operand
// issues at half the rate of one without (measured: 4.4 against 2.3 cycles a
// wave for add and multiply).
__device__ inline float in_vgpr(float x)
{
    asm("" : "+v"(x));
    return x;
}

struct RefCell {
    int x, y, z;
};

__device__ inline RefCell ref_cell(float4 p, const StepParams &P)
{
    return RefCell{trunc_to_int(p.x / P.h), trunc_to_int(p.y / P.h), trunc_to_int(p.z / P.h)};
}

// The (2R + 1)^2 rows of the (2R + 1)^3 grid-cell stencil around packed
// cell cc (R = P.reach), clipped to the grid: for row (y, z) the x-run of
// cells [gx - R, gx + R] is one contiguous range [b, e) of the cell-ordered
// arrays.  Calls row(b, e) for each row, z-major then y, both ascending.
// The bounds of the next row are loaded while the current row runs.
template <class Row>
__device__ inline void for_each_row(const uint32_t *__restrict__ cstart, uint32_t cc,
                                    const StepParams &P, Row row)
{
    const int gx = cell_x(cc), gy = cell_y(cc), gz = cell_z(cc), R = P.reach;
    const int x0 = max(gx - R, 0), x1 = min(gx + R, P.nx - 1);
    const int y0 = max(gy - R, 0), y1 = min(gy + R, P.ny - 1);
    const int z0 = max(gz - R, 0), z1 = min(gz + R, P.nz - 1);
    const int nrows = (y1 - y0 + 1) * (z1 - z0 + 1);
    auto base = [&](int y, int z) {
        return P.cell_base + (uint32_t)P.nx * ((uint32_t)y + (uint32_t)P.ny * (uint32_t)z);
    };
    int y = y0, z = z0;
    uint32_t r0 = base(y, z);
    uint32_t b = cstart[r0 + (uint32_t)x0], e = cstart[r0 + (uint32_t)x1 + 1u];
    for (int k = 0; k < nrows; ++k) {
        if (++y > y1) {
            y = y0;
            ++z;
        }
        uint32_t bn = 0, en = 0;
        if (k + 1 < nrows) {
            r0 = base(y, z);
            bn = cstart[r0 + (uint32_t)x0];
            en = cstart[r0 + (uint32_t)x1 + 1u];
        }
        row(b, e);
        b = bn;
        e = en;
    }
}

// The lane's place in its grid cell, for cutting its stencil to the cells
// a neighbour can occupy.  A neighbour j of lane i has fl(d^2) < fl(h^2),
// so its true distance is below h (1 + 2^-21), i.e. below rho = h / H cell
// edges.  The cell offset d along an axis lies at least gap(d) cell edges
// away (d - f for d > 0, -d - 1 + f for d < 0, 0 for d = 0, f = the lane's
// fraction of its cell), so a cell whose squared gaps add up to rho^2 or
// more holds no neighbour.  f comes from the same double expression as the
// cell index, and the float work around it errs by far less than the slack
// taken off every gap (2^-12 edges) and added to the reach (2^-10 of
// rho^2): the cut drops only candidates whose float squared distance
// exceeds h^2.
struct LaneTrim {
    float fx, fy, fz;  // fraction of the cell, clamped to [0, 1]
    float r2;          // rho^2 (1 + 2^-10)
};

constexpr float kTrimSlack = 1.0f / 4096.0f;

__device__ inline LaneTrim lane_trim(float4 p, uint32_t cc, const StepParams &P)
{
    auto frac = [&](float x, double o, int g) {
        const double q = ((double)x - o) * P.grid_inv - (double)g;
        return fminf(fmaxf((float)q, 0.0f), 1.0f);  // NaN -> 0
    };
    LaneTrim t;
    t.fx = frac(p.x, P.grid_o[0], cell_x(cc));
    t.fy = frac(p.y, P.grid_o[1], cell_y(cc));
    t.fz = frac(p.z, P.grid_o[2], cell_z(cc));
    const double rh = (double)P.h * P.grid_inv;
    t.r2 = (float)(rh * rh * (1.0 + 1.0 / 1024.0));
    return t;
}

// gap(d) less the slack, at least 0
__device__ inline float trim_gap(int d, float f)
{
    const float g = d > 0 ? (float)d - f : (d < 0 ? (float)(-d - 1) + f : 0.0f);
    return fmaxf(g - kTrimSlack, 0.0f);
}

// for_each_row cut by the lane's trim: row (y, z) is skipped when its
// gaps alone reach rho, else its x-run is cut to the cells within the
// remaining chord.  Calls row(b, e) for every non-empty row, in
// for_each_row's order, so the passing candidates come in the same order
// as on the whole stencil.  The bounds of the next row are loaded while the
// current row runs.
template <class Row>
__device__ inline void for_each_cut_row(const uint32_t *__restrict__ cstart, uint32_t cc, const LaneTrim &T,
                                        const StepParams &P, Row row)
{
    const int gx = cell_x(cc), gy = cell_y(cc), gz = cell_z(cc), R = P.reach;
    const int y0 = max(gy - R, 0), y1 = min(gy + R, P.ny - 1);
    const int z0 = max(gz - R, 0), z1 = min(gz + R, P.nz - 1);
    const int nrows = (y1 - y0 + 1) * (z1 - z0 + 1);
    auto bounds = [&](int y, int z, uint32_t &b, uint32_t &e) {
        const float ay = trim_gap(y - gy, T.fy), az = trim_gap(z - gz, T.fz);
        const float rem = T.r2 - (ay * ay + az * az);
        b = e = 0u;
        if (rem > 0.0f) {
            const float w = __builtin_amdgcn_sqrtf(rem) + 2.0f * kTrimSlack;
            const int x0 = max(gx + max((int)floorf(T.fx - w), -R), 0);
            const int x1 = min(gx + min((int)floorf(T.fx + w), R), P.nx - 1);
            if (x0 <= x1) {
                const uint32_t r0 = P.cell_base + (uint32_t)P.nx * ((uint32_t)y + (uint32_t)P.ny * (uint32_t)z);
                b = cstart[r0 + (uint32_t)x0];
                e = cstart[r0 + (uint32_t)x1 + 1u];
            }
        }
    };
    int y = y0, z = z0;
    uint32_t b, e;
    bounds(y, z, b, e);
    for (int k = 0; k < nrows; ++k) {
        if (++y > y1) {
            y = y0;
            ++z;
        }
        uint32_t bn = 0, en = 0;
        if (k + 1 < nrows)
            bounds(y, z, bn, en);
        if (b < e)
            row(b, e);
        b = bn;
        e = en;
    }
}

// for_each_row restricted to the positions [lo, hi) of the lane's own
// candidate sequence (its rows in order, slots ascending).
template <class Row>
__device__ inline void for_each_row_span(const uint32_t *__restrict__ cstart, uint32_t cc, const StepParams &P,
                                         uint32_t lo, uint32_t hi, Row row)
{
    uint32_t off = 0;
    for_each_row(cstart, cc, P, [&](uint32_t b, uint32_t e) {
        const uint32_t len = e - b;
        const uint32_t s0 = max(lo, off), s1 = min(hi, off + len);
        if (s0 < s1)
            row(b + (s0 - off), b + (s1 - off));
        off += len;
    });
}

__device__ inline int wave_min_i(int x)
{
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1)
        x = min(x, __shfl_xor(x, d, 64));
    return __builtin_amdgcn_readfirstlane(x);
}

__device__ inline int wave_max_i(int x)
{
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1)
        x = max(x, __shfl_xor(x, d, 64));
    return __builtin_amdgcn_readfirstlane(x);
}

// Most cells a union walk's wave may span in y and in z: the union's
// (span + 2R)^2 rows fit the 64 lanes that stage them (R = 1: 4, 2: 4, 3: 2).
__device__ inline int union_span(int R) { return min(4, 8 - 2 * R); }

// What a wave walks together: a box of grid cells [x0, x1] x [y0, y1] x
// [z0, z1] (inside the grid), or the stencils of the wave's segments (runs
// of lanes in one x-row of cells), one after the other, each for its own
// lanes.
struct UnionRows {
    int x0, x1, y0, y1, z0, z1;
    bool segments;
};

__device__ inline uint32_t row_base(const StepParams &P, int y, int z)
{
    return P.cell_base + (uint32_t)P.nx * ((uint32_t)y + (uint32_t)P.ny * (uint32_t)z);
}

// Length of the lane's own (2R + 1)^3 stencil, the sum of its rows'
// lengths as for_each_row visits them; the bounds of one z-layer's rows are
// loaded together (all in flight at once) instead of a row ahead.
__device__ inline uint32_t stencil_length(const uint32_t *__restrict__ cstart, uint32_t cc, const StepParams &P)
{
    const int gx = cell_x(cc), gy = cell_y(cc), gz = cell_z(cc), R = P.reach;
    const int x0 = max(gx - R, 0), x1 = min(gx + R, P.nx - 1);
    const int y0 = max(gy - R, 0), y1 = min(gy + R, P.ny - 1);
    const int z0 = max(gz - R, 0), z1 = min(gz + R, P.nz - 1);
    uint32_t own = 0;
    for (int z = z0; z <= z1; ++z) {
        uint32_t b[2 * kMaxReach + 1], e[2 * kMaxReach + 1];
#pragma unroll
        for (int k = 0; k < 2 * kMaxReach + 1; ++k) {
            b[k] = e[k] = 0u;
            if (y0 + k <= y1) {  // 2R + 1 rows (fewer at the grid's border)
                const uint32_t r0 = P.cell_base + (uint32_t)P.nx * ((uint32_t)(y0 + k) + (uint32_t)P.ny * (uint32_t)z);
                b[k] = cstart[r0 + (uint32_t)x0];
                e[k] = cstart[r0 + (uint32_t)x1 + 1u];
            }
        }
#pragma unroll
        for (int k = 0; k < 2 * kMaxReach + 1; ++k)
            own += e[k] - b[k];
    }
    return own;
}

// The segments of a wave: the lanes are in cell order, so those of one (y, z)
// row of cells are consecutive and ascend in x.
__device__ inline uint64_t segment_heads(uint32_t cc, bool active)
{
    const uint32_t yz = cc & ~kSlowBit & ~2047u;
    const uint32_t before = (uint32_t)__shfl_up((int)yz, 1, 64);
    return __ballot(active && ((threadIdx.x & 63u) == 0u || yz != before));
}

// Row `lane` of the wave's segments' stencils ((2R + 1)^2 rows each, z-major
// then y): its first slot and length (0 where there is no such row).
__device__ inline void segment_row(const uint32_t *__restrict__ cstart, uint32_t cc, bool active, uint64_t heads,
                                   const StepParams &P, uint32_t &b, uint32_t &len)
{
    const int R = P.reach;
    const uint32_t W = 2u * (uint32_t)R + 1u, lane = threadIdx.x & 63u;
    const uint32_t nact = (uint32_t)__builtin_popcountll(__ballot(active));
    uint32_t first = 0, last = 0;  // cells of the ends of the lane's segment
    uint32_t k = 0;
    for (uint64_t h = heads; h != 0ull; ++k) {
        const uint32_t a = (uint32_t)__builtin_ctzll(h);
        h &= h - 1ull;
        const uint32_t e = h != 0ull ? (uint32_t)__builtin_ctzll(h) - 1u : nact - 1u;
        if (lane / (W * W) == k) {
            first = (uint32_t)__builtin_amdgcn_readlane((int)cc, (int)a);
            last = (uint32_t)__builtin_amdgcn_readlane((int)cc, (int)e);
        }
    }
    b = len = 0u;
    const int r = (int)(lane % (W * W));
    const int y = cell_y(first) + r % (int)W - R, z = cell_z(first) + r / (int)W - R;
    if (lane < k * W * W && y >= 0 && y < P.ny && z >= 0 && z < P.nz) {
        const uint32_t r0 = row_base(P, y, z);
        b = cstart[r0 + (uint32_t)max(cell_x(first) - R, 0)];
        len = cstart[r0 + (uint32_t)min(cell_x(last) + R, P.nx - 1) + 1u] - b;
    }
}

// own: the lane's own candidate count when this computed it (the
// comparison needs it unless all lanes share one cell), else kNoOwn.
constexpr uint32_t kNoOwn = 0xFFFFFFFFu;

// Chooses between the two ways a wave walks its candidates:
//  * per lane: each lane walks its own (2R + 1)^3 stencil (gathers);
//  * union: all lanes walk the union of their stencils together, read from
//    LDS with one broadcast for the wave.
// Union is taken when all lanes sit in one cell (the dense regime: one cell
// holds many waves), or when their cells span at most union_span(R) in y and
// z (so the union has at most 64 rows) and the union holds at most 3x the
// largest own stencil (a per-lane walk costs three times as much per
// candidate and more).  A wave whose cells lie further apart (the end of one
// clump and the start of the next) walks its segments' stencils, under the
// same limits: per lane such waves took 1.0 of the 1.9 ms of a density pass
// over a late state of a million particles, a tenth of its tasks.
// A candidate the union adds to a lane's own stencil lies in a cell R + 1 or
// more cells away, beyond R whole cells of edge >= h (1 + 2^-10) / R along
// some axis, so its float squared distance is above h^2 and it never passes
// (and a segment's candidates are met by its own lanes only): both walks
// visit a lane's passing candidates in the same order (rows z-major, then y,
// slots ascending) and give bit-identical sums.
__device__ inline bool plan_union(const uint32_t *__restrict__ cstart, uint32_t cc, bool active, const StepParams &P,
                                  UnionRows &U, uint32_t &count, uint32_t &own)
{
    U = UnionRows{0, 0, 0, 0, 0, 0, false};
    if (P.lane_walk)
        return false;
    const uint32_t cell = cc & ~kSlowBit;
    const uint32_t c0 = __builtin_amdgcn_readfirstlane(cell);
    int x0, x1, y0, y1, z0, z1;
    const bool one = __all(cell == c0);
    if (one) {
        x0 = x1 = cell_x(c0);
        y0 = y1 = cell_y(c0);
        z0 = z1 = cell_z(c0);
    } else {
        const int gx = cell_x(cell), gy = cell_y(cell), gz = cell_z(cell);
        x0 = wave_min_i(gx);
        x1 = wave_max_i(gx);
        y0 = wave_min_i(gy);
        y1 = wave_max_i(gy);
        z0 = wave_min_i(gz);
        z1 = wave_max_i(gz);
    }
    uint32_t own_max = 0;
    if (!one) {
        own = stencil_length(cstart, cc, P);
        own_max = (uint32_t)wave_max_i((int)own);
    }
    const int R = P.reach, span = union_span(R);
    if (y1 - y0 < span && z1 - z0 < span) {
        U.x0 = max(x0 - R, 0);
        U.x1 = min(x1 + R, P.nx - 1);
        U.y0 = max(y0 - R, 0);
        U.y1 = min(y1 + R, P.ny - 1);
        U.z0 = max(z0 - R, 0);
        U.z1 = min(z1 + R, P.nz - 1);
        uint32_t un = 0;
        for (int z = U.z0; z <= U.z1; ++z)
            for (int y = U.y0; y <= U.y1; ++y) {
                const uint32_t r0 = row_base(P, y, z);
                un += cstart[r0 + (uint32_t)U.x1 + 1u] - cstart[r0 + (uint32_t)U.x0];
            }
        count = __builtin_amdgcn_readfirstlane(un);
        if (one || count <= 3ull * own_max)
            return true;
    }
    const uint64_t heads = segment_heads(cc, active);
    const uint32_t W = 2u * (uint32_t)R + 1u;
    if ((uint32_t)__builtin_popcountll(heads) * W * W > 64u)
        return false;
    uint32_t b, len;
    segment_row(cstart, cc, active, heads, P, b, len);
    count = (uint32_t)__builtin_amdgcn_readlane((int)wave_inclusive_scan(len), 63);
    U.segments = true;
    return count <= 3ull * own_max;
}

// Whether a wave task takes the union walk, and then its box, from the
// step's part plan.
__device__ inline bool walk_of(const PartPlan &pp, uint32_t wt, UnionRows &U)
{
    const int4 a = pp.walk[2u * wt], b = pp.walk[2u * wt + 1u];
    U.x0 = __builtin_amdgcn_readfirstlane(a.x);
    U.x1 = __builtin_amdgcn_readfirstlane(a.y);
    U.y0 = __builtin_amdgcn_readfirstlane(a.z);
    U.y1 = __builtin_amdgcn_readfirstlane(a.w);
    U.z0 = __builtin_amdgcn_readfirstlane(b.x);
    U.z1 = __builtin_amdgcn_readfirstlane(b.y);
    const int w = __builtin_amdgcn_readfirstlane(b.w);
    U.segments = (w & (int)kWalkSegments) != 0;
    return (w & (int)kWalkBox) != 0;
}

// Length of the lane's own candidate sequence (its (2R + 1)^3 stencil).
__device__ inline uint32_t own_length(const PartPlan &pp, uint32_t s, const uint32_t *__restrict__ cstart, uint32_t cc,
                                      const StepParams &P)
{
    if (pp.own)
        return pp.own[s];
    return stencil_length(cstart, cc, P);
}

__device__ inline void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Union walk.  The wave's union candidates, flattened in row order (rows as
// for_each_row visits them, slots ascending, the rows of each z-layer
// starting at a multiple of 64), are fetched 64 at a time -- one coalesced
// load per lane and record array, a chunk ahead of their use -- into a
// per-wave LDS double buffer, then read back by all lanes together, so the
// candidate loop never waits on a global load, never pays per-row overhead,
// and its operands are vector registers (fed from scalar registers the same
// loop issues its three subtractions at half rate).  Places that hold no
// candidate stage a record with slot ~0 that passes no test, so chunks run in
// groups of four unchecked: at infinity, or, where products with its distance
// must stay finite (FINITE), far away from every wave that has none of its
// own near there (StepParams::zero_limit).
constexpr float kFarAway = 0x1p60f;  // its square is finite
constexpr uint32_t kNoSlot = 0xFFFFFFFFu;

// One record array (positions, w unused) is kept as three coordinate arrays:
// four candidates are three 16-byte reads instead of four (a read that all
// lanes share still returns 1 KB: 8 cycles of the LDS that four SIMDs share).
template <int NV>
struct ChunkRecords {
    float4 rec[NV][64];
};
template <>
struct ChunkRecords<1> {
    alignas(16) float x[64], y[64], z[64];
};

template <int NV>
struct UnionStage {
    ChunkRecords<NV> chunk[2];
    uint32_t slot[2][64];
    // rows: first flattened position, end, and slot less position
    uint32_t start[65], end[65], shift[65];
    uint32_t ny;           // rows of a z-layer
    uint32_t segment[64];  // of each lane, when segments are walked
};

// The row table of U in T; returns the length of the flattened sequence
// (layers padded).  Every lane of the wave calls it.
template <int NV>
__device__ inline uint32_t union_rows(const uint32_t *__restrict__ cstart, const UnionRows &U, uint32_t cc, bool active,
                                      const StepParams &P, UnionStage<NV> &T)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t W = 2u * (uint32_t)P.reach + 1u;
    uint32_t ny, nrows, b = 0, len = 0;
    if (U.segments) {
        const uint64_t heads = segment_heads(cc, active);
        ny = W;
        nrows = W * W * (uint32_t)__builtin_popcountll(heads);
        segment_row(cstart, cc, active, heads, P, b, len);
        const uint64_t upto = (2ull << lane) - 1ull;  // lanes 0 .. lane
        T.segment[lane] = active ? (uint32_t)__builtin_popcountll(heads & upto) - 1u : 0u;
    } else {
        ny = (uint32_t)(U.y1 - U.y0 + 1);
        nrows = ny * (uint32_t)(U.z1 - U.z0 + 1);  // at most (union_span + 2R)^2 <= 64 lanes
        if (lane < nrows) {
            const uint32_t r0 = row_base(P, U.y0 + (int)(lane % ny), U.z0 + (int)(lane / ny));
            b = cstart[r0 + (uint32_t)U.x0];
            len = cstart[r0 + (uint32_t)U.x1 + 1u] - b;
        }
    }
    const uint32_t sum = wave_inclusive_scan(len);
    const uint32_t before = (uint32_t)__shfl((int)sum, (int)(lane - ny) & 63, 64);
    uint32_t pad = 0;  // behind the last row of a layer
    if (lane < nrows && lane % ny == ny - 1u)
        pad = (0u - (sum - (lane >= ny ? before : 0u))) & 63u;
    const uint32_t end = wave_inclusive_scan(len + pad);
    const uint32_t start = end - len - pad;
    T.start[lane] = lane < nrows ? start : 0xFFFFFFFFu;
    T.end[lane] = start + len;
    T.shift[lane] = b - start;
    if (lane == 0u) {
        T.start[64] = 0xFFFFFFFFu;
        T.end[64] = 0u;
        T.shift[64] = 0u;
        T.ny = ny;
    }
    wave_lds_sync();
    return (uint32_t)__builtin_amdgcn_readlane((int)end, 63);
}

// Part `part` of `nparts` equal slices (whole chunks) of a flattened sequence.
__device__ inline void part_slice(uint32_t total, uint32_t part, uint32_t nparts, uint32_t &lo, uint32_t &hi)
{
    const uint64_t chunks = (total + 63u) >> 6;
    lo = (uint32_t)(chunks * part / nparts) << 6;
    hi = (uint32_t)(chunks * (part + 1u) / nparts) << 6;
}

// Walks the positions [lo, hi) (multiples of 64) of the table's sequence:
// chunk(records, slots, n, odd, layer) for each 64 of them, n candidates (a
// multiple of four with the ones far away), all of z-layer `layer` (2R + 1 to
// a segment).  odd: the
// chunk holds some of the wave's own slots [first, first + 64) or, with
// FINITE, a record with values beyond `limit` (or not finite).
template <int NV, bool FINITE, class Chunk>
__device__ inline void union_walk(uint32_t lo, uint32_t hi, uint32_t first, float limit,
                                  const float4 *const (&src)[NV], UnionStage<NV> &T, Chunk chunk)
{
    constexpr float far = FINITE ? kFarAway : __builtin_inff();
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t ny = __builtin_amdgcn_readfirstlane(T.ny);
    uint32_t row = 0, next = T.start[1];
    auto fetch = [&](uint32_t f0, float4(&r)[NV], uint32_t &slot) {
        const uint32_t f = f0 + lane;
        while (f >= next) {  // ends at the last row: the starts behind it are ~0
            ++row;
            next = T.start[row + 1u];
        }
        if (f < T.end[row]) {
            slot = f + T.shift[row];
#pragma unroll
            for (int v = 0; v < NV; ++v)
                r[v] = src[v][slot];
        } else {
            slot = kNoSlot;
            r[0] = make_float4(far, far, far, 0.0f);
#pragma unroll
            for (int v = 1; v < NV; ++v)
                r[v] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
    };
    float4 nr[NV];
    uint32_t ns = kNoSlot;
    if (lo < hi)
        fetch(lo, nr, ns);
    for (uint32_t f0 = lo, bs = 0; f0 < hi; f0 += 64u, bs ^= 1u) {
        const uint32_t layer = (uint32_t)__builtin_amdgcn_readfirstlane((int)row) / ny;
        bool odd = ns - first < 64u;
        if (FINITE) {
            float size = 0.0f;
#pragma unroll
            for (int v = 0; v < NV; ++v)
                size += fabsf(nr[v].x) + fabsf(nr[v].y) + fabsf(nr[v].z) + fabsf(nr[v].w);
            odd = odd || (ns != kNoSlot && !(size <= limit));
        }
        const bool any_odd = __any(odd);
        const uint32_t n = (uint32_t)__builtin_popcountll(__ballot(ns != kNoSlot));
        if constexpr (NV == 1) {
            T.chunk[bs].x[lane] = nr[0].x;
            T.chunk[bs].y[lane] = nr[0].y;
            T.chunk[bs].z[lane] = nr[0].z;
        } else {
#pragma unroll
            for (int v = 0; v < NV; ++v)
                T.chunk[bs].rec[v][lane] = nr[v];
        }
        T.slot[bs][lane] = ns;
        wave_lds_sync();
        if (f0 + 64u < hi)
            fetch(f0 + 64u, nr, ns);
        chunk(T.chunk[bs], T.slot[bs], (n + 3u) & ~3u, any_odd, layer);
    }
}

// ------------------------------------------------------------ part plan

// A wave task's staged candidates: the records of its lanes' stencil cells,
// z-layer after z-layer, row after row, and what finds them.
// Coordinates lie in three arrays, each row from a multiple of four on:
// four candidates are three 16-byte reads, and lanes of neighbouring cells
// read different banks (records of 16 bytes, eight to a cell, all met in the
// same banks: 58% of the LDS cycles were conflicts).
constexpr uint32_t kStageCap = 1296;  // candidates, every row rounded up to a multiple of four
constexpr uint32_t kStageSegs = 7;    // runs of lanes in one x-row of cells, 3 rows each per layer
constexpr uint32_t kStageWords = 3;   // a lane's row: at most 32 candidates per mask word
                                      // (a lattice of spacing h / 2.1 can line up 66)
// Room for the terms of one lane's neighbours in layers 1 and 2, the former
// from the first row up, the latter from the last row down; each side's next
// term is written wherever it will come to lie, so two rows more than terms.
// A lattice of spacing h / 2 has 32 at most.  (Six blocks fit a CU with this;
// with 52 rows, five: planning 64 scenes took 214 us instead of 195.)
constexpr uint32_t kStageTerms = 34;
struct StagedLayer {
    uint32_t shift[3 * kStageSegs];  // row -> LDS index less slot
    uint32_t x0[kStageSegs], x1[kStageSegs], yz[kStageSegs];
    uint32_t total, fits;
    uint32_t own[64], listed[64], counted[64];
};
struct Stage {
    alignas(16) float x[kStageCap + 4], y[kStageCap + 4], z[kStageCap + 4];  // four are read ahead
    StagedLayer layer[3];
    float term[kStageTerms][64];
};

// Coordinates of the records [first, first + n), first and n wave-uniform,
// into LDS, without registers in between; the caller waits for vmcnt.
// The lanes' offsets stay 32 bits beside a scalar address: one instruction
// a load (64-bit vector addresses were a quarter of k_plan_fine).
__device__ inline void load_to_lds(const float4 *__restrict__ pos, uint32_t first, uint32_t n, float *x, float *y,
                                   float *z)
{
    const uint32_t lane = threadIdx.x & 63u;
    for (uint32_t k = 0; k < n; k += 64u) {
        const char *base = reinterpret_cast<const char *>(pos + (first + k));
        if (lane < n - k) {
            auto load = [&](uint32_t at, float *dst) {
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(base + (lane * 16u + at)),
                                                 (__attribute__((address_space(3))) void *)(dst + k), 4, 0, 0);
            };
            load(0u, x);
            load(4u, y);
            load(8u, z);
        }
    }
}

struct __attribute__((packed, aligned(4))) Bounds4 {
    uint32_t v[4];
};

// The end of a staged task: its lanes' densities, and how the force pass
// walks it where the lists (`listed` entries, or kNoList for any) don't do.
__device__ inline void finish_staged(const uint32_t *__restrict__ cstart, uint32_t cc, bool active, bool any_slow,
                                     const StepParams &P, const PartPlan &pp, const NeighborLists &nl, uint32_t task,
                                     uint32_t s, float4 pi, const float4 *__restrict__ vel, float acc, uint32_t listed,
                                     float *__restrict__ rho, float4 *__restrict__ posR, float4 *__restrict__ velR)
{
    UnionRows U{0, 0, 0, 0, 0, 0, false};
    uint32_t ucount = 0, unused = kNoOwn, w = kWalkUnion | kWalkSummed;
    if (__any(listed == kNoList) && plan_union(cstart, cc, active, P, U, ucount, unused) && !any_slow)
        w |= kWalkBox | (U.segments ? kWalkSegments : 0u);
    if (active) {
        const float4 vs = vel[s];
        const float d = acc + P.self_dens;
        rho[s] = d;
        posR[s] = make_float4(pi.x, pi.y, pi.z, 0.5f / d);
        velR[s] = make_float4(vs.x, vs.y, vs.z, P.gas * (d - P.rho0));
        nl.count[s] = listed;
    }
    if ((threadIdx.x & 63u) == 0u) {
        pp.measure[task] = 0u;
        pp.walk[2u * task] = make_int4(U.x0, U.x1, U.y0, U.y1);
        pp.walk[2u * task + 1u] = make_int4(U.z0, U.z1, (int)ucount, (int)w);
    }
}

// The lane's cut rows in layer l (0 .. 4) of a grid of reach 2: first
// candidates, and behind the last ones (the same for a row that is out).  A
// cell whose squared gaps add up to the reach or more is out (see LaneTrim).
// Ten loads without a branch between them (a branch each, and the compiler
// waits in each): rows that are out read cell 0.
__device__ inline void cut_rows(const uint32_t *__restrict__ cstart, uint32_t cc, const LaneTrim &T,
                                const StepParams &P, int l, uint32_t (&from)[5], uint32_t (&to)[5])
{
    const int gx = cell_x(cc), gy = cell_y(cc), z = cell_z(cc) + l - 2;
    auto square = [](float g) { return g * g; };
    const float left1 = square(trim_gap(-1, T.fx)), left2 = square(trim_gap(-2, T.fx));
    const float right1 = square(trim_gap(1, T.fx)), right2 = square(trim_gap(2, T.fx));
    const uint32_t nx = (uint32_t)P.nx;
    const uint32_t row = P.cell_base + nx * ((uint32_t)(gy - 2) + (uint32_t)P.ny * (uint32_t)z);
    const bool layer = z >= 0 && z < P.nz;
#pragma unroll
    for (int r = 0; r < 5; ++r) {
        const int y = gy + r - 2;
        const float rem = T.r2 - (square(trim_gap(r - 2, T.fy)) + square(trim_gap(l - 2, T.fz)));
        const bool in = rem > 0.0f && layer && y >= 0 && y < P.ny;
        const int xa = max(gx - (left1 < rem ? 1 : 0) - (left2 < rem ? 1 : 0), 0);
        const int xb = min(gx + (right1 < rem ? 1 : 0) + (right2 < rem ? 1 : 0), P.nx - 1);
        const uint32_t r0 = row + nx * (uint32_t)r;
        from[r] = cstart[in ? r0 + (uint32_t)xa : 0u];
        to[r] = cstart[in ? r0 + (uint32_t)xb + 1u : 0u];
    }
}

// The walk, and its length, of a task left to k_density.  own: the lanes'
// own candidate counts, or kNoOwn.  longest: on a grid of reach 2, the
// largest count of a lane's cut rows, or kNoOwn.
// A task is left whole by the same count in every launch (k_plan_fine's tasks
// are planned here where scenes on other grids share the launch), so that a
// scene's sums don't depend on its company.
__device__ inline void plan_walk(const uint32_t *__restrict__ cstart, uint32_t cc, bool active, bool any_slow,
                                 const StepParams &P, const SceneSet &S, const PartPlan &pp, uint32_t task, uint32_t s,
                                 uint32_t own, const float4 *__restrict__ pos, uint32_t longest_cut)
{
    UnionRows U;
    uint32_t ucount = 0, len, fresh = kNoOwn;
    const bool use_union = plan_union(cstart, cc, active, P, U, ucount, fresh) && !any_slow;
    if (__builtin_amdgcn_readfirstlane(own) == kNoOwn)  // wave-uniform
        own = fresh;
    if (!use_union && __builtin_amdgcn_readfirstlane(own) == kNoOwn)
        own = stencil_length(cstart, cc, P);
    const uint32_t longest = (uint32_t)wave_max_i((int)own);  // kNoOwn (-1): all lanes in one cell
    uint32_t shortness = longest;
    if (fine_stageable(P)) {
        shortness = longest_cut;
        if (longest_cut == kNoOwn) {
            const LaneTrim T = lane_trim(pos[s], cc, P);
            uint32_t cut = 0;
#pragma unroll 1
            for (int l = 0; l < 5; ++l) {
                uint32_t from[5], to[5];
                cut_rows(cstart, cc, T, P, l, from, to);
#pragma unroll
                for (int r = 0; r < 5; ++r)
                    cut += to[r] - from[r];
            }
            shortness = (uint32_t)wave_max_i((int)cut);
        }
    }
    if (shortness <= kShortWalk) {
        len = 0;  // left whole: it records neighbour lists, which the force pass then visits
    } else if (use_union) {
        len = ucount;
    } else {
        // Per-lane walks cost several times as much per candidate as the
        // union walk (divergent gathers, no shared loads), so they count
        // several times toward the part size; with slow lanes (m_ij counted
        // from the 27 buckets per neighbour, the wave waiting on them) more
        // again.
        len = longest * (any_slow ? kSlowWalkWeight : kLaneWalkWeight);
    }
    if (!use_union && active)
        pp.own[s] = own;
    if ((threadIdx.x & 63u) == 0u) {
        pp.walk[2u * task] = make_int4(U.x0, U.x1, U.y0, U.y1);
        pp.walk[2u * task + 1u] = make_int4(
            U.z0, U.z1, (int)ucount, use_union ? (int)(kWalkUnion | kWalkBox | (U.segments ? kWalkSegments : 0u)) : 0);
        pp.measure[task] = len;
        // only walks that may be split count toward the scene's part size
        if (len > kPartCandidates)
            atomicAdd(&pp.total[kTotalSlots * S.tasks[task].scene + task % kTotalSlots], (unsigned long long)len);
    }
}

// Plans the walk of every wave task and, where all of its lanes' stencils
// are short, runs its density pass at once: one block of three waves per
// task, a wave for each z-layer of the stencil.
//
// Short walks (the largest own stencil at most kShortWalk candidates, cells
// of h or larger) are staged: each wave
// copies the three rows of its layer, for every segment of the task's lanes,
// to LDS with asynchronous loads, all in flight together, and its lanes walk
// their own cut stencil (for_each_cut_row's cells, in its order) from there.
// Walked from global memory the same pass is a chain of some fifty dependent
// round trips, each also waiting for the list entries stored before it; here
// it is three (cells, bounds, records), and a third as many candidates.
// The waves only find the neighbours of their layers; their terms are then
// added in the order of every other walk, and listed in it, so both are the
// per-lane walk's bit for bit: the first wave adds its own, then those the
// others left in LDS.
// Measured, planning and density of a step together, walked from memory and
// staged: 8,000 particles 65 and 23 us, 64 scenes of 1.06 million in all 263
// and 195 us.  What bounds those is arithmetic and waiting about equally (90 M
// vector instructions for a lattice of a million, finding neighbours and adding
// their terms in order about equal shares: 0.45 of the issue slots at two
// cycles each; three waves a SIMD that wait 40% of their time); below some
// thousand tasks, the latency of one wave.
// (Adding each layer's terms in its own wave takes 19 and 151 us, but then
// the sums are not the per-lane walk's, and over a run of steps the particles
// that meet a wall bounce a step apart.)
//
// All other tasks get a walk length (union count, or the largest own
// stencil weighted), which splits them into parts, and are left to
// k_density.
//
// Without STAGED (no scene of the launch can be staged) a task is one wave
// that only plans.
template <bool STAGED, bool COUNT>
__global__ __launch_bounds__(STAGED ? 192 : 64) void k_plan_list(
    const float4 *__restrict__ pos, const float4 *__restrict__ vel, const uint32_t *__restrict__ cellcB,
    const uint32_t *__restrict__ cstart, float *__restrict__ rho, float4 *__restrict__ posR,
    float4 *__restrict__ velR, SceneSet S, PartPlan pp, NeighborLists nl, uint32_t *__restrict__ count)
{
    const uint32_t lane = threadIdx.x & 63u;
    const int lz = STAGED ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) : 0;  // the wave's layer
    const uint32_t task = xcd_block();
    if (task >= S.nwaves)
        return;
    if (task == 0u && threadIdx.x < 3u)
        pp.queue[threadIdx.x] = 0u;  // parts taken by the density and force passes, parts queued
    Lane L;
    bool active;
    wave_task(S, task, L, active);
    const StepParams P = *L.P;
    const uint32_t s = L.slot;
    const uint32_t cc = cellcB[s];
    const bool slow = (cc & kSlowBit) != 0u;
    const bool any_slow = __any(slow);
    uint32_t own = kNoOwn;
    if (STAGED && stageable(P) && nl.list) {  // block-uniform
        __shared__ Stage stage;
        StagedLayer(&layers)[3] = stage.layer;
        const float4 pi = pos[s];
        StagedLayer &G = layers[lz];
        const int gx = cell_x(cc), gy = cell_y(cc), z = cell_z(cc) + lz - 1;
        // the four cell bounds of each of the lane's three rows
        // (cells gx - 1 .. gx + 1, moved inside at the grid's ends)
        const int xs = min(max(gx - 1, 0), P.nx - 3);
        Bounds4 v[3];
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            const int y = gy + r - 1;
            v[r] = Bounds4{{0u, 0u, 0u, 0u}};
            if (y >= 0 && y < P.ny && z >= 0 && z < P.nz)
                v[r] = *reinterpret_cast<const Bounds4 *>(cstart + row_base(P, y, z) + (uint32_t)xs);
        }
        const uint32_t yz = cc & ~kSlowBit & ~2047u;
        const uint64_t heads = segment_heads(cc, active);
        const bool head = (heads >> lane & 1ull) != 0ull;
        const uint32_t nact = (uint32_t)__builtin_popcountll(__ballot(active));
        const uint32_t nseg = (uint32_t)__builtin_popcountll(heads);
        const uint64_t upto = (2ull << lane) - 1ull;  // lanes 0 .. lane
        const uint32_t seg = active ? (uint32_t)__builtin_popcountll(heads & upto) - 1u : 0u;
        uint32_t b = 0, len = 0, gap = 0;
        if (nseg <= kStageSegs) {
            if (head) {
                G.x0[seg] = (uint32_t)gx;
                G.yz[seg] = yz;
            }
            if (active && (lane + 1u == nact || ((heads >> 1) >> lane & 1ull)))
                G.x1[seg] = (uint32_t)gx;
            wave_lds_sync();
            if (lane < 3u * nseg) {
                const uint32_t k = lane / 3u, c = G.yz[k];
                const int y = cell_y(c) + (int)(lane % 3u) - 1, zc = cell_z(c) + lz - 1;
                if (y >= 0 && y < P.ny && zc >= 0 && zc < P.nz) {
                    const uint32_t r0 = row_base(P, y, zc);
                    b = cstart[r0 + (uint32_t)max((int)G.x0[k] - 1, 0)];
                    len = cstart[r0 + (uint32_t)min((int)G.x1[k] + 1, P.nx - 1) + 1u] - b;
                    gap = (0u - len) & 3u;
                }
            }
        }
        const uint32_t end = wave_inclusive_scan(len + gap);
        if (lane == 63u)
            G.total = end;
        __syncthreads();
        const uint32_t t0 = layers[0].total, t1 = layers[1].total, t2 = layers[2].total;
        const bool room = __builtin_amdgcn_readfirstlane(nseg <= kStageSegs && t0 + t1 + t2 <= kStageCap ? 1 : 0) != 0;
        const uint32_t off = (lz == 0 ? 0u : lz == 1 ? t0 : t0 + t1) + end - len - gap;
        if (room) {
            if (lane < 3u * nseg)
                G.shift[lane] = off - b;
            for (uint32_t e = 0; e < 3u * nseg; ++e) {
                const uint32_t bs = (uint32_t)__builtin_amdgcn_readlane((int)b, (int)e);
                const uint32_t n = (uint32_t)__builtin_amdgcn_readlane((int)len, (int)e);
                const uint32_t o = (uint32_t)__builtin_amdgcn_readlane((int)off, (int)e);
                load_to_lds(pos, bs, n, &stage.x[o], &stage.y[o], &stage.z[o]);
            }
            for (uint32_t k = 0; k < gap; ++k)  // behind a row: candidates that never pass
                stage.x[off + len + k] = __builtin_inff();
        }
        // lanes at the ends of the grid's x axis: back to (start of the
        // cell below, own start, own end, end of the cell above)
        const int at = gx - xs;  // 1 except there
        if (!__all(at == 1)) {
#pragma unroll
            for (int r = 0; r < 3; ++r) {
                const uint32_t *q = v[r].v;
                v[r] = at == 1 ? v[r]
                               : at == 0 ? Bounds4{{q[0], q[0], q[1], q[2]}} : Bounds4{{q[1], q[2], q[3], q[3]}};
            }
        }
        // the lane's cut rows: LDS index of the first candidate, rounded down
        // to a multiple of four, and the count from there
        const LaneTrim T = lane_trim(pi, cc, P);
        const float az = trim_gap(lz - 1, T.fz);
        uint32_t l0[3], n[3], mine = 0;
        bool short_rows = true;
        wave_lds_sync();  // shift[]
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            mine += v[r].v[3] - v[r].v[0];
            // for_each_cut_row's cells at reach 1: the cell below is in
            // when fx < w, the one above when fx + w >= 1
            const float ay = trim_gap(r - 1, T.fy);
            const float rem = T.r2 - (ay * ay + az * az);
            const float w = __builtin_amdgcn_sqrtf(fmaxf(rem, 0.0f)) + 2.0f * kTrimSlack;
            const uint32_t from = T.fx < w ? v[r].v[0] : v[r].v[1];
            const uint32_t to = T.fx + w >= 1.0f ? v[r].v[3] : v[r].v[2];
            const uint32_t at0 = from + (room ? G.shift[3u * seg + (uint32_t)r] : 0u);
            l0[r] = at0 & ~3u;
            n[r] = rem > 0.0f && from < to ? to - from + (at0 & 3u) : 0u;
            short_rows = short_rows && n[r] <= 32u * kStageWords;
        }
        G.own[lane] = mine;
        const bool ok = room && __all(short_rows);
        if (lane == 0u)
            G.fits = ok ? 1u : 0u;
        // The staged records have landed (vmcnt 0), also where they go
        // unused.  As a builtin, so that the compiler knows: it would
        // otherwise wait for vmcnt before every read.
        __builtin_amdgcn_s_waitcnt(0x0F70);
        __syncthreads();
        own = layers[0].own[lane] + layers[1].own[lane] + layers[2].own[lane];
        const uint32_t longest = (uint32_t)wave_max_i((int)own);
        if (__builtin_amdgcn_readfirstlane(layers[0].fits & layers[1].fits & layers[2].fits) != 0u &&
            longest <= kShortWalk) {
            const float h2 = in_vgpr(P.h2);
            const float mp6 = P.mp6;
            float acc = 0.0f;
            uint32_t mask[3][kStageWords];
            const int term0 = (lz == 2 ? (int)kStageTerms - 1 : 0) * 64 + (int)lane, next_term = lz == 2 ? -64 : 64;
            const int term_lo = (lz == 2 ? 3 : 0) * 64 + (int)lane, term_hi = term_lo + ((int)kStageTerms - 4) * 64;
            int at_term = term0;
            float *const terms = &stage.term[0][0];
            auto test = [&](float x, float y, float z) {
                float dx, dy, dz;
                return h2 - dist2_ref(pi, make_float4(x, y, z, 0.0f), dx, dy, dz);
            };
            // Four candidates at a time, the next four read meanwhile.  What
            // lies before the row's first and behind its last candidate is
            // the rest of its x-row (beyond the cut or the stencil: it never
            // passes) or a sentinel.  The passing ones (h2 - d2 > 0: exactly
            // when d2 < h2, the float difference of unequal values being
            // nonzero) are collected in a mask, the first on top.
            auto walk = [&](auto first_tag, auto unit_tag) {
                constexpr bool first = decltype(first_tag)::value;  // layer 0
#pragma unroll
                for (int r = 0; r < 3; ++r) {
#pragma unroll
                    for (uint32_t c = 0; c < kStageWords; ++c) {
                        const uint32_t k0 = 32u * c, m = n[r] > k0 ? min(32u, n[r] - k0) : 0u;
                        const uint32_t from = l0[r] + k0;
                        // only row 1 of layer 1 holds the particle itself
                        const uint32_t self = r == 1 && lz == 1 ? s + G.shift[3u * seg + 1u] - from : ~0u;
                        uint32_t bits = 0;
                        if (m != 0u) {
                            float4 x = *reinterpret_cast<const float4 *>(&stage.x[from]);
                            float4 y = *reinterpret_cast<const float4 *>(&stage.y[from]);
                            float4 z = *reinterpret_cast<const float4 *>(&stage.z[from]);
                            for (uint32_t k = 0; k < m; k += 4u) {
                                const float u[4] = {test(x.x, y.x, z.x), test(x.y, y.y, z.y), test(x.z, y.z, z.z),
                                                    test(x.w, y.w, z.w)};
                                x = *reinterpret_cast<const float4 *>(&stage.x[from + k + 4u]);
                                y = *reinterpret_cast<const float4 *>(&stage.y[from + k + 4u]);
                                z = *reinterpret_cast<const float4 *>(&stage.z[from + k + 4u]);
#pragma unroll
                                for (int i = 0; i < 4; ++i) {
                                    float t = positive<decltype(unit_tag)::value>(u[i]);
                                    if (!first && r == 1)
                                        t = k + (uint32_t)i != self ? t : 0.0f;
                                    const uint32_t hit = (0u - __float_as_uint(t)) >> 31;
                                    bits = bits << 1 | hit;
                                    if (first) {
                                        acc = acc + mp6 * ((t * t) * t);
                                    } else {  // kept if it is one, else overwritten by the next
                                        terms[at_term] = t;
                                        at_term += __mul24((int)hit, next_term);
                                    }
                                }
                                // inside the array after four more, whatever it overwrites
                                if (!first)
                                    at_term = min(max(at_term, term_lo), term_hi);
                            }
                            bits <<= 32u - ((m + 3u) & ~3u);
                        }
                        mask[r][c] = bits;
                    }
                }
            };
            if (P.h2 <= 1.0f) {
                if (lz == 0)
                    walk(std::true_type{}, std::true_type{});
                else
                    walk(std::false_type{}, std::true_type{});
            } else {
                if (lz == 0)
                    walk(std::true_type{}, std::false_type{});
                else
                    walk(std::false_type{}, std::false_type{});
            }
            uint32_t nn = 0;
#pragma unroll
            for (int r = 0; r < 3; ++r)
#pragma unroll
                for (uint32_t c = 0; c < kStageWords; ++c)
                    nn += (uint32_t)__builtin_popcount(mask[r][c]);
            G.listed[lane] = nn;
            __syncthreads();
            const uint32_t n0 = layers[0].listed[lane], n1 = layers[1].listed[lane], n2 = layers[2].listed[lane];
            const uint32_t all = n0 + n1 + n2;
            const bool listing = !__any(all > kListMax),
                       parallel = !__any(n1 + n2 + 2u > kStageTerms || max(n1, n2) > kStageTerms - 4u);
            auto neighbours = [&](auto visit) {
#pragma unroll
                for (int r = 0; r < 3; ++r)
#pragma unroll
                    for (uint32_t c = 0; c < kStageWords; ++c)
                        for (uint32_t bits = mask[r][c]; bits != 0u;) {
                            const uint32_t k = (uint32_t)__builtin_clz(bits);
                            bits &= ~(0x80000000u >> k);
                            visit(l0[r] + 32u * c + k, G.shift[3u * seg + (uint32_t)r]);
                        }
            };
            if (listing) {
                uint32_t *lp = nl.list + list_at(lz == 0 ? 0u : lz == 1 ? n0 : n0 + n1, s, nl.stride);
                neighbours([&](uint32_t k, uint32_t shift) {
                    *lp = k - shift;
                    lp += nl.stride;
                });
            }
            uint32_t cnt = nn;
            if (parallel && !any_slow) {
                if (COUNT)
                    G.counted[lane] = cnt;
                if (COUNT)
                    __syncthreads();
            } else {
                // The terms again, neighbours only, each with its m_ij; one
                // layer after the other where they don't all fit.
                RefCell ci{0, 0, 0};
                if (slow)
                    ci = ref_cell(pi, P);
                auto again = [&](auto add) {
                    neighbours([&](uint32_t k, uint32_t shift) {
                        const float t = test(stage.x[k], stage.y[k], stage.z[k]);
                        float term = mp6 * ((t * t) * t);
                        if (slow) {
                            const uint32_t hash = __float_as_uint(pos[k - shift].w) & 0xFFFFu;
                            const int mult = bucket_multiplicity(ci.x, ci.y, ci.z, hash);
                            term = (float)mult * term;
                            cnt += (uint32_t)mult - 1u;
                        }
                        add(term);
                    });
                };
                acc = 0.0f;
                if (parallel) {
                    at_term = term0;
                    again([&](float term) {
                        if (lz == 0) {
                            acc += term;
                        } else {
                            terms[at_term] = term;
                            at_term += next_term;
                        }
                    });
                    G.counted[lane] = cnt;
                    __syncthreads();
                } else {
                    for (int turn = 0; turn < 3; ++turn) {
                        if (turn == lz) {
                            acc = turn != 0 ? stage.term[0][lane] : 0.0f;
                            again([&](float term) { acc += term; });
                            stage.term[0][lane] = acc;
                            G.counted[lane] = cnt;
                        }
                        __syncthreads();
                    }
                }
            }
            if (lz != 0)
                return;
            if (parallel) {
                const uint32_t rest = n1 + n2, most = (uint32_t)wave_max_i((int)rest);
                for (uint32_t k = 0; k < most; k += 4u) {
                    float v[4];
#pragma unroll
                    for (uint32_t i = 0; i < 4u; ++i) {
                        const uint32_t q = min(k + i, kStageTerms - 1u);
                        v[i] = stage.term[q < n1 ? q : kStageTerms - 1u - (q - n1)][lane];
                    }
#pragma unroll
                    for (uint32_t i = 0; i < 4u; ++i) {
                        const float term = any_slow ? v[i] : mp6 * ((v[i] * v[i]) * v[i]);
                        acc = k + i < rest ? acc + term : acc;
                    }
                }
            } else {
                acc = stage.term[0][lane];
            }
            if (COUNT && active)
                count[s] = layers[0].counted[lane] + layers[1].counted[lane] + layers[2].counted[lane];
            finish_staged(cstart, cc, active, any_slow, P, pp, nl, task, s, pi, vel, acc, listing ? all : kNoList, rho,
                          posR, velR);
            return;
        }
    }
    if (lz != 0)
        return;
    plan_walk(cstart, cc, active, any_slow, P, S, pp, task, s, own, pos, kNoOwn);
}

// The same for cells of h / 2 to h (reach 2), where a stencil is 25 rows of a
// few cells: one wave per task, which copies layer after layer of its lanes'
// rows to LDS, the next one while it walks one.  The bounds of the lanes' 25
// cut rows are read at once beforehand, and a layer's neighbours are listed
// after the next layer has arrived, so that no load waits for the list's
// stores.  Planned and walked here, against planned and walked from memory in
// k_density: 262 thousand particles 62 us and 26 + 86, a million 157 and
// 30 + 150.  What bounds it is waiting at low occupancy: 163 registers let
// three waves onto a SIMD, 2.2 are there on average, and they spend 44% of
// their time waiting for LDS and memory, 27% in vector instructions (58 M for
// a million particles: 0.29 of the issue slots at two cycles each).
// Tasks in many rows (a surface), whose layers don't fit the room, walk from
// memory here (in k_density, behind the others, the latency of a few hundred
// such waves was 40 us); those with a row of more than kFineRow candidates in a lane's
// stencil, or a longer walk, are left to k_density.
constexpr uint32_t kFineCap = 448;  // candidates of a layer (64 slots and 4 cells in each of 5 rows: about 350)
constexpr uint32_t kFineGap = 2;    // behind a row: three candidates are tested at a time
constexpr uint32_t kFineRow = 30, kFineRowBits = 5, kFineAtBits = 9;
constexpr uint32_t kFineSegs = 12;  // runs of lanes in one x-row of cells, 5 rows each per layer
struct FineStage {
    float x[2][kFineCap + 3], y[2][kFineCap + 3], z[2][kFineCap + 3];  // three are read ahead
    uint32_t slot[5][64], at[5][64];  // of a row's first candidate
    uint32_t x0[kFineSegs], x1[kFineSegs], yz[kFineSegs];
};
union FineShared {
    FineStage staged;
    uint32_t row[2][25][64];  // or each lane's rows: first slot, and count, then which are neighbours
};
static_assert(kFineCap <= 1u << kFineAtBits && kFineRow < 1u << kFineRowBits && kFineRowBits + kFineAtBits <= 16, "");

template <bool COUNT>
__global__ __launch_bounds__(64) void k_plan_fine(
    const float4 *__restrict__ pos, const float4 *__restrict__ vel, const uint32_t *__restrict__ cellcB,
    const uint32_t *__restrict__ cstart, float *__restrict__ rho, float4 *__restrict__ posR,
    float4 *__restrict__ velR, SceneSet S, PartPlan pp, NeighborLists nl, uint32_t *__restrict__ count)
{
    __shared__ FineShared shared;
    FineStage &stage = shared.staged;
    const uint32_t lane = threadIdx.x;
    const uint32_t task = xcd_block();
    if (task >= S.nwaves)
        return;
    if (task == 0u && lane < 3u)
        pp.queue[lane] = 0u;  // as in k_plan_list
    Lane L;
    bool active;
    wave_task(S, task, L, active);
    const StepParams P = *L.P;
    const uint32_t s = L.slot;
    const uint32_t cc = cellcB[s];
    const bool slow = (cc & kSlowBit) != 0u;
    const bool any_slow = __any(slow);
    const uint64_t heads = segment_heads(cc, active);
    const uint32_t nseg = (uint32_t)__builtin_popcountll(heads);
    uint32_t longest = kNoOwn;
    if (fine_stageable(P) && nl.list) {  // wave-uniform
        const float4 pi = pos[s];
        const int gx = cell_x(cc);
        const bool few = nseg <= kFineSegs;
        const uint32_t nact = (uint32_t)__builtin_popcountll(__ballot(active));
        const uint32_t seg = active && few ? (uint32_t)__builtin_popcountll(heads & ((2ull << lane) - 1ull)) - 1u : 0u;
        if (few) {
            if ((heads >> lane & 1ull) != 0ull) {
                stage.x0[seg] = (uint32_t)gx;
                stage.yz[seg] = cc & ~kSlowBit & ~2047u;
            }
            if (active && (lane + 1u == nact || ((heads >> 1) >> lane & 1ull)))
                stage.x1[seg] = (uint32_t)gx;
        }
        wave_lds_sync();
        // All the bounds, 60 loads in flight together
        const uint32_t nx = (uint32_t)P.nx, plane = nx * (uint32_t)P.ny;
        // lane: row lane % 5 of segment lane / 5, in each layer
        const bool owner = few && lane < 5u * nseg;
        uint32_t b[5], len[5];
        {
            const uint32_t k = owner ? lane / 5u : 0u, c = owner ? stage.yz[k] : 0u;
            const int y = cell_y(c) + (int)(lane % 5u) - 2, z0 = cell_z(c) - 2;
            const uint32_t row = P.cell_base + nx * (uint32_t)y + plane * (uint32_t)z0;
            const uint32_t xa = owner ? (uint32_t)max((int)stage.x0[k] - 2, 0) : 0u;
            const uint32_t xb = owner ? (uint32_t)min((int)stage.x1[k] + 2, P.nx - 1) + 1u : 0u;
            const bool in = owner && y >= 0 && y < P.ny;
#pragma unroll
            for (int l = 0; l < 5; ++l) {
                const bool at = in && z0 + l >= 0 && z0 + l < P.nz;
                const uint32_t r0 = row + plane * (uint32_t)l;
                b[l] = cstart[at ? r0 + xa : 0u];
                len[l] = cstart[at ? r0 + xb : 0u];
            }
        }
        uint32_t from[5][5], n[5][5];
        const LaneTrim T = lane_trim(pi, cc, P);
#pragma unroll
        for (int l = 0; l < 5; ++l)
            cut_rows(cstart, cc, T, P, l, from[l], n[l]);
        uint32_t own = 0;
#pragma unroll
        for (int l = 0; l < 5; ++l) {
            len[l] -= b[l];  // 0 for a row that is out
#pragma unroll
            for (int r = 0; r < 5; ++r) {
                n[l][r] -= from[l][r];
                own += n[l][r];
            }
        }
        longest = (uint32_t)wave_max_i((int)own);
        bool ok = few, short_rows = true;
#pragma unroll
        for (int l = 0; l < 5; ++l) {
            const uint32_t room = owner ? len[l] + kFineGap : 0u;
            const uint32_t end = wave_inclusive_scan(room);
            ok = ok && (uint32_t)__builtin_amdgcn_readlane((int)end, 63) <= kFineCap;
            stage.slot[l][lane] = b[l];
            stage.at[l][lane] = end - room;
        }
        wave_lds_sync();
        // each row in 16 bits: count, offset of its first candidate
        uint32_t rows[13] = {};
#pragma unroll
        for (int l = 0; l < 5; ++l)
#pragma unroll
            for (int r = 0; r < 5; ++r) {
                const uint32_t off = n[l][r] ? from[l][r] - stage.slot[l][5u * seg + (uint32_t)r] : 0u;
                short_rows = short_rows && n[l][r] <= kFineRow;
                rows[(5 * l + r) / 2] |= (n[l][r] | off << kFineRowBits) << (((5 * l + r) & 1) * 16);
            }
        if (__all(short_rows) && longest <= kShortWalk) {
            auto stage_layer = [&](int l) {
                const int buf = l & 1;
                const uint32_t at0 = stage.at[l][lane];
                for (uint32_t e = 0; e < 5u * nseg; ++e) {
                    const uint32_t first = (uint32_t)__builtin_amdgcn_readlane((int)b[l], (int)e);
                    const uint32_t m = (uint32_t)__builtin_amdgcn_readlane((int)len[l], (int)e);
                    const uint32_t o = (uint32_t)__builtin_amdgcn_readlane((int)at0, (int)e);
                    load_to_lds(pos, first, m, &stage.x[buf][o], &stage.y[buf][o], &stage.z[buf][o]);
                }
                if (owner)
#pragma unroll
                    for (uint32_t k = 0; k < kFineGap; ++k)  // candidates that never pass
                        stage.x[buf][at0 + len[l] + k] = __builtin_inff();
            };
            auto arrived = [] {
                __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt 0
                wave_lds_sync();
            };
            const float h2 = in_vgpr(P.h2), mp6 = in_vgpr(P.mp6);
            auto test = [&](float x, float y, float z) {  // h <= 1: clamping to 1 changes nothing
                float dx, dy, dz;
                return positive<true>(h2 - dist2_ref(pi, make_float4(x, y, z, 0.0f), dx, dy, dz));
            };
            RefCell ci{0, 0, 0};
            if (slow)
                ci = ref_cell(pi, P);
            float acc = 0.0f, slow_acc = 0.0f;
            uint32_t nn = 0, cnt = 0;
            uint32_t *lp = nl.list + s;
            // a neighbour, in order: listed; summed again with its m_ij where
            // the wave has slow lanes
            auto neighbour = [&](uint32_t j, auto record) {
                if (nn < kListMax) {
                    *lp = j;
                    lp += nl.stride;
                }
                ++nn;
                if (any_slow) {
                    const float4 q = record();
                    const float t = test(q.x, q.y, q.z);
                    int mult = 1;
                    if (slow)
                        mult = bucket_multiplicity(ci.x, ci.y, ci.z, __float_as_uint(pos[j].w) & 0xFFFFu);
                    slow_acc += (float)mult * (mp6 * ((t * t) * t));
                    cnt += (uint32_t)mult - 1u;
                }
            };
            if (__all(ok)) {
                stage_layer(0);
                arrived();
#pragma unroll
                for (int l = 0; l < 5; ++l) {
                    const int buf = l & 1;
                    if (l < 4)
                        stage_layer(l + 1);
                    uint32_t bits[5];
#pragma unroll
                    for (int r = 0; r < 5; ++r) {
                        const uint32_t row = rows[(5 * l + r) / 2] >> (((5 * l + r) & 1) * 16);
                        const uint32_t m = row & ((1u << kFineRowBits) - 1u);
                        const uint32_t off = row >> kFineRowBits & ((1u << kFineAtBits) - 1u);
                        bits[r] = 0u;
                        if (m == 0u)
                            continue;
                        const uint32_t at = stage.at[l][5u * seg + (uint32_t)r] + off;
                        const float *px = &stage.x[buf][at], *py = &stage.y[buf][at], *pz = &stage.z[buf][at];
                        // only the middle row holds the particle itself
                        const uint32_t self = l == 2 && r == 2 ? s - stage.slot[l][5u * seg + (uint32_t)r] - off : 0u;
                        float x[3], y[3], z[3];
#pragma unroll
                        for (int i = 0; i < 3; ++i) {
                            x[i] = px[i];
                            y[i] = py[i];
                            z[i] = pz[i];
                        }
                        uint32_t k = 0;
                        do {
                            float t[3];
#pragma unroll
                            for (int i = 0; i < 3; ++i) {
                                t[i] = test(x[i], y[i], z[i]);
                                if (l == 2 && r == 2)
                                    t[i] = k + (uint32_t)i != self ? t[i] : 0.0f;
                            }
#pragma unroll
                            for (int i = 0; i < 3; ++i) {  // the next three, meanwhile
                                x[i] = px[k + 3u + (uint32_t)i];
                                y[i] = py[k + 3u + (uint32_t)i];
                                z[i] = pz[k + 3u + (uint32_t)i];
                            }
#pragma unroll
                            for (int i = 0; i < 3; ++i) {
                                acc = acc + mp6 * ((t[i] * t[i]) * t[i]);
                                bits[r] = __builtin_amdgcn_alignbit(bits[r], 0u - __float_as_uint(t[i]), 31u);  // << 1 | (t > 0)
                            }
                            k += 3u;
                        } while (k < m);
                        bits[r] <<= 32u - k;  // the first on top (k <= 30)
                    }
                    if (l < 4)
                        arrived();
#pragma unroll
                    for (int r = 0; r < 5; ++r) {
                        if (bits[r] == 0u)
                            continue;
                        const uint32_t row = rows[(5 * l + r) / 2] >> (((5 * l + r) & 1) * 16);
                        const uint32_t off = row >> kFineRowBits & ((1u << kFineAtBits) - 1u);
                        const uint32_t j0 = stage.slot[l][5u * seg + (uint32_t)r] + off;
                        do {
                            const uint32_t k = (uint32_t)__builtin_clz(bits[r]);
                            bits[r] &= ~(0x80000000u >> k);
                            neighbour(j0 + k, [&] {
                                const uint32_t at = stage.at[l][5u * seg + (uint32_t)r] + off + k;
                                return make_float4(stage.x[buf][at], stage.y[buf][at], stage.z[buf][at], 0.0f);
                            });
                        } while (bits[r] != 0u);
                    }
                }
            } else {
                // The thin surface of a flow: a wave's lanes lie in many rows,
                // whose stencils don't fit.  Each lane walks its own rows from
                // memory, the next row's first four candidates on the way
                // meanwhile, and lists at the end.
                wave_lds_sync();  // at[], slot[]
#pragma unroll
                for (int l = 0; l < 5; ++l)
#pragma unroll
                    for (int r = 0; r < 5; ++r) {
                        shared.row[0][5 * l + r][lane] = from[l][r];
                        shared.row[1][5 * l + r][lane] = n[l][r];
                    }
                wave_lds_sync();
                auto four = [&](uint32_t first, uint32_t m, uint32_t k, float4 (&q)[4]) {
#pragma unroll
                    for (uint32_t i = 0; i < 4u; ++i)  // the last one again behind it
                        q[i] = pos[m != 0u ? first + min(k + i, m - 1u) : s];
                };
                uint32_t first = shared.row[0][0][lane], m = shared.row[1][0][lane];
                float4 q[4];
                four(first, m, 0u, q);
                for (uint32_t r = 0; r < 25u; ++r) {
                    const uint32_t next = min(r + 1u, 24u);
                    const uint32_t next_first = shared.row[0][next][lane], next_m = shared.row[1][next][lane];
                    float4 next_q[4];
                    four(next_first, next_m, 0u, next_q);
                    uint32_t bits = 0, k = 0;
                    for (;;) {
#pragma unroll
                        for (uint32_t i = 0; i < 4u; ++i) {
                            float t = test(q[i].x, q[i].y, q[i].z);
                            t = k + i < m && first + k + i != s ? t : 0.0f;
                            acc = acc + mp6 * ((t * t) * t);
                            bits = __builtin_amdgcn_alignbit(bits, 0u - __float_as_uint(t), 31u);
                        }
                        k += 4u;
                        if (k >= m)
                            break;
                        four(first, m, k, q);
                    }
                    shared.row[1][r][lane] = bits << (32u - k);  // k <= 32
                    first = next_first;
                    m = next_m;
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        q[i] = next_q[i];
                }
                for (uint32_t r = 0; r < 25u; ++r) {
                    const uint32_t j0 = shared.row[0][r][lane];
                    for (uint32_t bits = shared.row[1][r][lane]; bits != 0u;) {
                        const uint32_t k = (uint32_t)__builtin_clz(bits);
                        bits &= ~(0x80000000u >> k);
                        neighbour(j0 + k, [&] { return pos[j0 + k]; });
                    }
                }
            }
            if (any_slow)
                acc = slow_acc;
            if (COUNT && active)
                count[s] = nn + cnt;
            const bool listing = !__any(nn > kListMax);
            finish_staged(cstart, cc, active, any_slow, P, pp, nl, task, s, pi, vel, acc, listing ? nn : kNoList, rho,
                          posR, velR);
            return;
        }
    }
    plan_walk(cstart, cc, active, any_slow, P, S, pp, task, s, kNoOwn, pos, longest);
}

// Parts per wave task, queued: the part size grows beyond kPartCandidates
// when the scene's total walk over its part room would exceed it.  A wave's
// split tasks take their places in the queue with one atomic; their order
// there varies, the sums of a task don't depend on it.  (8,000 particles: 4.8 us;
// counting, a scan of
// the counts and writing them out in five launches took 16.3.)
__global__ __launch_bounds__(kBlock) void k_queue_parts(SceneSet S, PartPlan pp)
{
    const uint32_t g = blockIdx.x * kBlock + threadIdx.x;
    uint32_t np = 0;
    if (g < S.nwaves) {
        const uint32_t length = pp.measure[g];
        if (length > kPartCandidates) {
            const uint32_t scene = S.tasks[g].scene;
            const StepParams &P = S.params[scene];
            const unsigned long long waves = (P.p_end - P.p_begin + 63u) / 64u;
            const unsigned long long room = part_room(waves);
            unsigned long long sum = 0;
            for (uint32_t k = 0; k < kTotalSlots; ++k)
                sum += pp.total[kTotalSlots * scene + k];
            const unsigned long long size = max((unsigned long long)kPartCandidates, (sum + room - 1u) / room);
            const unsigned long long p = (length + size - 1u) / size;
            np = (uint32_t)min(p, (unsigned long long)kMaxParts);
            np = np > 1u ? np : 0u;  // an unsplit task is not queued
        }
        pp.nparts[g] = np;
    }
    if (!__any(np != 0u))
        return;
    const uint32_t end = wave_inclusive_scan(np);
    uint32_t base = 0;
    if ((threadIdx.x & 63u) == 63u)
        base = atomicAdd(&pp.queue[2], end);
    base = (uint32_t)__builtin_amdgcn_readlane((int)base, 63) + end - np;
    if (np != 0u)
        pp.off[g] = base;
    for (uint32_t p = 0; p < np; ++p)
        pp.tasks[base + p] = (g << kPartBits) | p;
}

void launch_plan_parts(hipStream_t st, const ParticleArrays &a, const CellArrays &c, const SceneSet &S,
                       const PartPlan &pp, const NeighborLists &nl, uint32_t *count)
{
    const dim3 grid(std::max(1u, S.nwaves));
#define SPH_LAUNCH_PLAN(STAGED, COUNT)                                                                             \
    hipLaunchKernelGGL((k_plan_list<STAGED, COUNT>), grid, dim3(STAGED ? 192 : 64), 0, st, a.posB, a.velB, a.cellcB, \
                       c.cstart, a.rhoB, a.posR, a.velR, S, pp, nl, count)
    if (S.staged && count)
        SPH_LAUNCH_PLAN(true, true);
    else if (S.staged)
        SPH_LAUNCH_PLAN(true, false);
    else if (!S.fine)
        SPH_LAUNCH_PLAN(false, false);  // counts nothing itself
#undef SPH_LAUNCH_PLAN
    else if (count)
        hipLaunchKernelGGL((k_plan_fine<true>), grid, dim3(64), 0, st, a.posB, a.velB, a.cellcB, c.cstart, a.rhoB,
                           a.posR, a.velR, S, pp, nl, count);
    else
        hipLaunchKernelGGL((k_plan_fine<false>), grid, dim3(64), 0, st, a.posB, a.velB, a.cellcB, c.cstart, a.rhoB,
                           a.posR, a.velR, S, pp, nl, count);
    hipLaunchKernelGGL(k_queue_parts, dim3(blocks_for(std::max(1u, S.nwaves))), dim3(kBlock), 0, st, S, pp);
}

// Runs task(w, part, nparts) for the work the calling wave takes.  Without
// a plan each wave runs wave task w of its own index, unsplit.  With one,
// each wave first runs its static share of the unsplit tasks, with no queue
// traffic, neighbouring tasks on one XCD sharing its L2, then parts of split
// tasks until there are none left (every wave exits then), which also evens
// out the static share.  All 64 lanes must be live on entry.
// skip_summed: leave out the tasks whose sums the planning pass made.
template <int BLOCK, bool skip_summed, class Task>
__device__ inline void for_each_part(const SceneSet &S, const PartPlan &pp, uint32_t *queue, Task task)
{
    const uint32_t first = __builtin_amdgcn_readfirstlane(xcd_block() * (BLOCK / 64) + (threadIdx.x >> 6));
    if (!queue) {
        if (first < S.nwaves)
            task(first, 0u, 1u);
        return;
    }
    const uint32_t total = __builtin_amdgcn_readfirstlane(pp.queue[2]);  // parts of split tasks
    constexpr uint32_t kWaves = BLOCK / 64;
    const uint32_t G = gridDim.x * kWaves;
    // G tasks at a time, each XCD a contiguous share of them in proportion to
    // its waves (blocks go round the XCDs).  Fewer tasks than waves are spread
    // over all XCDs so; dealt by wave index, contiguous on each XCD too, they
    // fell to the first of them, beside parts that are taken everywhere (97
    // thousand particles at spacing 0.4 h: density 152 and 80 us, force 212 and
    // 135).
    const uint32_t xcd = blockIdx.x & 7u, per = gridDim.x >> 3, rem = gridDim.x & 7u;
    const uint32_t below = (xcd * per + min(xcd, rem)) * kWaves;  // waves on lower XCDs
    const uint32_t here = (per + (xcd < rem ? 1u : 0u)) * kWaves;
    const uint32_t mine = __builtin_amdgcn_readfirstlane((blockIdx.x >> 3) * kWaves + (threadIdx.x >> 6));
    // Of n <= G tasks, this wave's, if `mine` of the XCD's share is below hi.
    // (Products below 2^32: G is at most the waves resident at once.)
    auto share = [&](uint32_t n, uint32_t &lo, uint32_t &hi) {
        lo = n * below / G;
        hi = n * (below + here) / G;
    };
    // Waves without a share take a part of their own first, as many on every
    // XCD (`spare`, what the XCD with the fewest has at least), without asking:
    // where these are all the parts, the counter is not touched (a few thousand
    // waves that ask once each to learn it cost a pass some 50 us).
    uint32_t t = kNoSlot, dealt = 0;
    if (total != 0u && S.nwaves < G) {
        uint32_t lo, hi;
        share(S.nwaves, lo, hi);
        const uint32_t spare = per * kWaves - (per * kWaves * S.nwaves + G - 1u) / G;
        const uint32_t k = mine - (hi - lo);  // huge for a wave with a share
        dealt = 8u * spare;
        if (k < spare)
            t = k * 8u + xcd;
    }
    for (uint32_t base = 0; base < S.nwaves; base += G) {
        uint32_t lo, hi;
        share(min(G, S.nwaves - base), lo, hi);
        const uint32_t w = base + lo + mine;
        if (lo + mine >= hi)
            continue;
        if (total == 0u || __builtin_amdgcn_readfirstlane(pp.nparts[w]) == 0u)
            if (!skip_summed || !(__builtin_amdgcn_readfirstlane(pp.walk[2u * w + 1u].w) & (int)kWalkSummed))
                task(w, 0u, 1u);
    }
    if (t == kNoSlot && total <= dealt)
        return;
    for (;;) {
        if (t == kNoSlot) {
            uint32_t asked = 0;
            if ((threadIdx.x & 63u) == 0u)
                asked = atomicAdd(queue, 1u);
            t = dealt + (uint32_t)__builtin_amdgcn_readfirstlane((int)asked);
        }
        if (t >= total)
            return;
        const uint32_t packed = __builtin_amdgcn_readfirstlane(pp.tasks[t]);
        const uint32_t w = packed >> kPartBits, part = packed & (kMaxParts - 1u);
        task(w, part, __builtin_amdgcn_readfirstlane(pp.nparts[w]));
        if (total <= dealt)
            return;
        t = kNoSlot;
    }
}

// Part `part` of wave task w stores its N partial sums; the last part to
// finish gets every part's sums added in part order in v and returns true
// (the others return false).  Every lane of the wave calls it.
//
// The parts of a task run on different XCDs, whose L2s do not see each
// other's lines.  The sums are stored and loaded at agent scope (past the
// L2), and each wave waits for its own stores before it counts itself
// finished, so the last one finds every sum in memory.  A device-wide fence
// would do the same by writing back the whole L2, once per part: with some
// 42,000 parts a step those fences took a quarter of a density pass.
template <int N>
__device__ inline bool combine_parts(const PartPlan &pp, uint32_t w, uint32_t part, uint32_t nparts, float (&v)[N])
{
    static_assert(N <= 4, "a part task has room for four sums per lane");
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t base = __builtin_amdgcn_readfirstlane(pp.off[w]);
    auto at = [&](uint32_t q, int k) {  // sum k of part q: the lanes side by side
        return reinterpret_cast<uint32_t *>(pp.buf) + (((size_t)base + q) * 4u + (uint32_t)k) * 64u + lane;
    };
#pragma unroll
    for (int k = 0; k < N; ++k)
        __hip_atomic_store(at(part, k), __float_as_uint(v[k]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");  // keeps the order in the program ...
    __builtin_amdgcn_s_waitcnt(0x0F70);                     // ... and vmcnt 0: the stores are done
    uint32_t prev = 0;
    if (lane == 0u)
        prev = __hip_atomic_fetch_add(&pp.done[w], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    prev = __builtin_amdgcn_readfirstlane(prev);
    if (prev + 1u != nparts)
        return false;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    for (uint32_t q0 = 0; q0 < nparts; q0 += 4u) {  // four parts' loads in flight
        float x[4][N];
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i)
#pragma unroll
            for (int k = 0; k < N; ++k)
                x[i][k] = __uint_as_float(__hip_atomic_load(at(min(q0 + i, nparts - 1u), k), __ATOMIC_RELAXED,
                                                            __HIP_MEMORY_SCOPE_AGENT));
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i)
            if (q0 + i < nparts)
#pragma unroll
                for (int k = 0; k < N; ++k)
                    v[k] = q0 + i == 0u ? x[i][k] : v[k] + x[i][k];
    }
    if (lane == 0u)
        pp.done[w] = 0u;  // ready for the next pass
    return true;
}

// --------------------------------------------------------------- density
// MODE 0: density + pressure.  MODE 1: also the neighbour count per
// particle.  MODE 2: also the neighbour ids (multiplicity-repeated).  MODE
// 3: MODE 0 plus the neighbour count (with multiplicity) of the production
// walks.  Writes rho, posR = (x, 0.5 / rho) and velR = (v, p) for the force
// pass, and in MODE 0 / 3 the neighbour lists of unsplit tasks.  With a plan
// it takes only the tasks the planning pass has not summed.
template <int MODE, int BLOCK>
__global__ __launch_bounds__(BLOCK, 6) void k_density(
    const float4 *__restrict__ pos, const float4 *__restrict__ vel,
    const uint32_t *__restrict__ cellc, const uint32_t *__restrict__ cstart,
    float *__restrict__ rho, float4 *__restrict__ posR, float4 *__restrict__ velR, SceneSet S,
    NeighborDump dump, PartPlan pp, NeighborLists nl)
{
    constexpr bool kCount = MODE >= 1;
    __shared__ UnionStage<1> stage[MODE == 0 || MODE == 3 ? BLOCK / 64 : 1];
    if (pp.queue && blockIdx.x == 0u)
        for (uint32_t k = threadIdx.x; k < kTotalSlots * pp.nscenes; k += BLOCK)
            pp.total[k] = 0ull;  // for the next step's plan
    for_each_part<BLOCK, true>(S, pp, pp.queue, [&](uint32_t wt, uint32_t part, uint32_t nparts) {
        Lane L;
        bool active;
        wave_task(S, wt, L, active);
        // a copy: read once (scalar loads) before the task's first store
        const StepParams P = *L.P;
        const uint32_t s = L.slot;
        const float4 pi = pos[s];
        const uint32_t cc = cellc[s];
        const bool slow = (cc & kSlowBit) != 0u;
        // the reference cell (three IEEE divisions) only matters for m_ij
        RefCell ci{0, 0, 0};
        if (slow)
            ci = ref_cell(pi, P);
        const float h2 = P.h2;
        const float mp6 = P.mp6;
        float acc = 0.0f;
        uint32_t cnt = 0;
        uint32_t listed = kNoList;
        uint64_t w = (MODE == 2 && active) ? dump.off[s] : 0;
        // true when q passes (and then adds its term)
        auto body = [&](uint32_t j, float4 q) -> bool {
            float dx, dy, dz;
            float d2 = dist2_ref(pi, q, dx, dy, dz);
            if (d2 < h2) {
                int m = 1;
                if (slow) {
                    int cx = ci.x, cy = ci.y, cz = ci.z;
                    asm volatile("" : "+v"(cx), "+v"(cy), "+v"(cz));
                    m = bucket_multiplicity(cx, cy, cz, __float_as_uint(q.w) & 0xFFFFu);
                }
                float t = h2 - d2;
                const float term = mp6 * ((t * t) * t);
                acc += (float)m * term;
                if (kCount)
                    cnt += (uint32_t)m;
                if (MODE == 2 && active) {
                    uint32_t id = __float_as_uint(vel[j].w);
                    for (int k = 0; k < m; ++k)
                        dump.out[w++] = id;
                }
                return true;
            }
            return false;
        };
        // Waves with a slow-multiplicity lane (rare where the union pays)
        // take the per-lane walk, so the union walk needs no m_ij.  A split
        // task walks its slice [part, part + 1) / nparts of the sequence.
        UnionRows U;
        if ((MODE == 0 || MODE == 3) && walk_of(pp, wt, U)) {
            UnionStage<1> &T = stage[threadIdx.x >> 6];
            uint32_t lo, hi;
            part_slice(union_rows(cstart, U, cc, active, P, T), part, nparts, lo, hi);
            const float4 *const src[1] = {pos};
            const float h2v = in_vgpr(h2);
            // An unsplit task records its lanes' neighbours here too (in
            // walk order, as the per-lane walk below), until one of them
            // has more than a list holds: the force pass then visits 30-odd
            // listed slots instead of the union's hundreds of candidates
            // (64 scenes of 1.06 million particles: 415 -> 169 us).
            bool listing = nl.list && nparts == 1u;
            uint32_t nn = 0, at_layer = kNoSlot;
            uint32_t *lp = nl.list + s;
            const uint32_t W = 2u * (uint32_t)P.reach + 1u;
            float4 me = pi;  // at infinity for the candidates of other lanes' segments
            // Unsplit sums are the per-lane walk's bit for bit.  Split ones
            // (added up part by part, so never quite those) leave the factor
            // to the end of the part: two operations a term instead of four.
            auto walk = [&](auto unit_tag, auto split_tag) {
                constexpr bool unit = decltype(unit_tag)::value, split = decltype(split_tag)::value;
                union_walk<1, false>(lo, hi, L.first, 0.0f, src, T, [&](const ChunkRecords<1> &c, const uint32_t *slots,
                                                                      uint32_t n, bool odd, uint32_t lz) {
                    if (U.segments && lz != at_layer) {
                        at_layer = lz;
                        me.x = T.segment[threadIdx.x & 63u] == lz / W ? pi.x : __builtin_inff();
                    }
                    // Branch-free: h2 - d2 > 0 exactly when d2 < h2 (the float
                    // difference of unequal values is nonzero), so clamping it
                    // at 0 turns a failing candidate into a +0 term, which
                    // leaves acc unchanged bit for bit.
                    auto term = [&](float x, float y, float z) {
                        float dx, dy, dz;
                        return positive<unit>(h2v - dist2_ref(me, make_float4(x, y, z, 0.0f), dx, dy, dz));
                    };
                    auto add = [&](float t) {
                        if (split)
                            acc = fmaf(t * t, t, acc);
                        else
                            acc = acc + mp6 * ((t * t) * t);
                    };
                    // candidates k .. k + 3, each given to visit in turn
                    auto four = [&](uint32_t k, auto self_tag, auto visit) {
                        const float4 x = *reinterpret_cast<const float4 *>(&c.x[k]);
                        const float4 y = *reinterpret_cast<const float4 *>(&c.y[k]);
                        const float4 z = *reinterpret_cast<const float4 *>(&c.z[k]);
                        float t[4] = {term(x.x, y.x, z.x), term(x.y, y.y, z.y), term(x.z, y.z, z.z),
                                      term(x.w, y.w, z.w)};
                        if (decltype(self_tag)::value) {
                            const uint4 j = *reinterpret_cast<const uint4 *>(&slots[k]);
                            t[0] = j.x != s ? t[0] : 0.0f;
                            t[1] = j.y != s ? t[1] : 0.0f;
                            t[2] = j.z != s ? t[2] : 0.0f;
                            t[3] = j.w != s ? t[3] : 0.0f;
                        }
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            add(t[i]);
                            visit(t[i]);
                        }
                    };
                    if (!split && listing) {
                        // Neighbours are marked as they pass (two operations a
                        // candidate) and appended 32 candidates at a time.
                        // (With a branch and a store for each: a lattice of
                        // spacing 0.4 h, 97 thousand particles, 173 us instead
                        // of 151, spacing h / 2 on cells of 1.7 h, 262
                        // thousand, 267 instead of 217.)
                        for (uint32_t k0 = 0; k0 < n; k0 += 32u) {
                            const uint32_t m = min(32u, n - k0);
                            uint32_t bits = 0;
                            auto mark = [&](float t) {  // << 1 | (t > 0)
                                bits = __builtin_amdgcn_alignbit(bits, 0u - __float_as_uint(t), 31u);
                            };
                            if (odd)
                                for (uint32_t k = 0; k < m; k += 4u)
                                    four(k0 + k, std::true_type{}, mark);
                            else
                                for (uint32_t k = 0; k < m; k += 4u)
                                    four(k0 + k, std::false_type{}, mark);
                            bits <<= 32u - m;  // the first on top
                            if (kCount)
                                cnt += (uint32_t)__builtin_popcount(bits);
                            for (; bits != 0u; ++nn) {
                                const uint32_t k = (uint32_t)__builtin_clz(bits);
                                bits &= ~(0x80000000u >> k);
                                if (nn < kListMax) {
                                    *lp = slots[k0 + k];
                                    lp += nl.stride;
                                }
                            }
                        }
                        listing = !__any(nn > kListMax);
                        return;
                    }
                    auto pass = [&](float t) {
                        if (kCount)
                            cnt += t > 0.0f ? 1u : 0u;
                    };
                    if (odd)
                        for (uint32_t k = 0; k < n; k += 4u)
                            four(k, std::true_type{}, pass);
                    else
                        for (uint32_t k = 0; k < n; k += 4u)
                            four(k, std::false_type{}, pass);
                });
            };
            if (nparts == 1u) {
                walk(std::false_type{}, std::false_type{});
            } else {
                if (h2 <= 1.0f)
                    walk(std::true_type{}, std::true_type{});
                else
                    walk(std::false_type{}, std::true_type{});
                acc = mp6 * acc;
            }
            if (listing)
                listed = nn;
        } else if ((MODE == 0 || MODE == 3) && nl.list && nparts == 1u) {
            // Per-lane walk that also records the lane's neighbours, in
            // walk order (rows in order, slots ascending).
            uint32_t nn = 0;
            // Without slow lanes every neighbour counts once, and the sum
            // runs branch-free: a failing candidate, or the particle
            // itself, adds +0, which leaves acc unchanged bit for bit (as
            // in the union walk), so both forms give the same sums.
            const bool any_slow = __any(slow);
            // On fine grids (R >= 2: rows of a few candidates) each
            // neighbour is appended as it passes; on cells of h (longer
            // rows, most candidates failing) a row's passes are collected
            // in a bitmask and appended afterwards, which issues fewer
            // stores.  The order is the same.
            const bool direct = P.reach >= 2;
            uint32_t *lp = nl.list + s;  // list entry nn (list_at's layout)
            auto fast = [&](float4 q) -> bool {
                float dx, dy, dz;
                const float d2 = dist2_ref(pi, q, dx, dy, dz);
                const float t = fmaxf(h2 - d2, 0.0f);
                acc = acc + mp6 * ((t * t) * t);
                if (kCount)
                    cnt += t > 0.0f ? 1u : 0u;
                return t > 0.0f;
            };
            auto append = [&](uint32_t j) {
                if (nn < kListMax) {
                    *lp = j;
                    lp += nl.stride;
                }
                ++nn;
            };
            // candidates [j0, j1), appended as they pass
            auto run_direct = [&](uint32_t j0, uint32_t j1) {
                uint32_t j = j0;
                for (; j + 4u <= j1; j += 4u) {  // four candidates in flight
                    const float4 q0 = pos[j], q1 = pos[j + 1u], q2 = pos[j + 2u], q3 = pos[j + 3u];
                    if (fast(q0))
                        append(j);
                    if (fast(q1))
                        append(j + 1u);
                    if (fast(q2))
                        append(j + 2u);
                    if (fast(q3))
                        append(j + 3u);
                }
                for (; j < j1; ++j)
                    if (fast(pos[j]))
                        append(j);
            };
            // candidates [j0, j1) of the segment starting at g, into its mask
            auto run_mask = [&](uint32_t j0, uint32_t j1, uint32_t g, uint64_t &mask) {
                uint32_t j = j0;
                for (; j + 4u <= j1; j += 4u) {
                    const float4 q0 = pos[j], q1 = pos[j + 1u], q2 = pos[j + 2u], q3 = pos[j + 3u];
                    mask |= fast(q0) ? 1ull << (j - g) : 0ull;
                    mask |= fast(q1) ? 2ull << (j - g) : 0ull;
                    mask |= fast(q2) ? 4ull << (j - g) : 0ull;
                    mask |= fast(q3) ? 8ull << (j - g) : 0ull;
                }
                for (; j < j1; ++j)
                    mask |= fast(pos[j]) ? 1ull << (j - g) : 0ull;
            };
            // Once a lane has more neighbours than a list holds, the force
            // pass walks this task anyway: the wave stops recording (and
            // only sums) for the rest of its rows.
            // The cut stencil: it drops only candidates that fail, each of
            // which adds +0 below, so the sums equal the whole stencil's.
            bool listing = true;
            const LaneTrim T = lane_trim(pi, cc, P);
            for_each_cut_row(cstart, cc, T, P, [&](uint32_t b, uint32_t e) {
                if (!any_slow && direct) {
                    // the row split at the lane's own slot (when it holds
                    // it), so no candidate needs a self test
                    const uint32_t m = (s >= b && s < e) ? s : e;
                    run_direct(b, m);
                    run_direct(min(m + 1u, e), e);
                    return;
                }
                for (uint32_t g = b; g < e; g += 64u) {
                    const uint32_t ge = min(g + 64u, e);
                    uint64_t mask = 0;
                    uint32_t j = g;
                    if (!any_slow) {
                        // the segment split at the lane's own slot
                        const uint32_t m = (s >= g && s < ge) ? s : ge;
                        run_mask(g, m, g, mask);
                        run_mask(min(m + 1u, ge), ge, g, mask);
                        j = ge;
                    }
                    for (; j + 1u < ge; j += 2u) {  // two candidates in flight
                        const float4 q0 = pos[j];
                        const float4 q1 = pos[j + 1u];
                        if (j != s && body(j, q0))
                            mask |= 1ull << (j - g);
                        if (j + 1u != s && body(j + 1u, q1))
                            mask |= 2ull << (j - g);
                    }
                    if (j < ge && j != s && body(j, pos[j]))
                        mask |= 1ull << (j - g);
                    if (!listing)
                        continue;
                    while (mask != 0ull) {
                        const uint32_t k = (uint32_t)__builtin_ctzll(mask);
                        mask &= mask - 1ull;
                        if (nn < kListMax)
                            nl.list[list_at(nn, s, nl.stride)] = g + k;
                        ++nn;
                    }
                    listing = !__any(nn > kListMax);
                }
            });
            if (!any_slow && direct)
                listing = !__any(nn > kListMax);
            listed = listing ? nn : kNoList;
        } else {
            uint32_t lo = 0, hi = 0xFFFFFFFFu;
            if (nparts > 1u) {
                const uint32_t own = own_length(pp, s, cstart, cc, P);
                lo = (uint32_t)((uint64_t)own * part / nparts);
                hi = (uint32_t)((uint64_t)own * (part + 1u) / nparts);
            }
            for_each_row_span(cstart, cc, P, lo, hi, [&](uint32_t b, uint32_t e) {
                uint32_t j = b;
                for (; j + 3u < e; j += 4u) {  // four candidates in flight
                    const float4 q[4] = {pos[j], pos[j + 1u], pos[j + 2u], pos[j + 3u]};
#pragma unroll
                    for (uint32_t i = 0; i < 4u; ++i)
                        if (j + i != s)
                            body(j + i, q[i]);
                }
                for (; j < e; ++j)
                    if (j != s)
                        body(j, pos[j]);
            });
        }
        if (nparts > 1u) {
            if constexpr (kCount) {
                float v[2] = {acc, (float)cnt};  // counts stay far below 2^24: exact
                if (!combine_parts<2>(pp, wt, part, nparts, v))
                    return;
                acc = v[0];
                cnt = (uint32_t)v[1];
            } else {
                float v[1] = {acc};
                if (!combine_parts<1>(pp, wt, part, nparts, v))
                    return;
                acc = v[0];
            }
        }
        if (!active)
            return;
        const float r = acc + P.self_dens;
        const float p = P.gas * (r - P.rho0);
        rho[s] = r;
        posR[s] = make_float4(pi.x, pi.y, pi.z, 0.5f / r);
        const float4 vs = vel[s];
        velR[s] = make_float4(vs.x, vs.y, vs.z, p);
        if (nl.count)
            nl.count[s] = listed;
        if (kCount)
            dump.count[s] = cnt;
    });
}

// Waves of `kernel` (at `block` threads) the device holds at once, from its
// register and LDS use.
static uint32_t occupancy_waves(const void *kernel, int block)
{
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, block, 0) != hipSuccess || nb <= 0)
        return resident_waves();
    return std::min<uint32_t>(resident_waves(), (uint32_t)nb * (uint32_t)(block / 64) * (resident_waves() / 32u));
}

// Waves of a stencil pass with a plan: a persistent grid of the waves the
// device holds at once for this kernel (a wave launched beyond them would
// start only as the first ones finish, with a full share of a static
// assignment), and at most 4 per wave task (more would only pull from an
// empty queue: a small scene splits into about as many parts as it has wave
// tasks).
inline uint32_t stencil_waves(const SceneSet &S, const PartPlan &pp, uint32_t resident)
{
    return std::min<uint32_t>(std::min<uint32_t>(pp.cap, resident), 4u * std::max(S.nwaves, 1u));
}

template <int MODE, int BLOCK>
static void launch_density_block(hipStream_t st, const ParticleArrays &a, const CellArrays &c,
                                 const SceneSet &S, const NeighborDump &d, const PartPlan &pp,
                                 const NeighborLists &nl)
{
    static const uint32_t resident = occupancy_waves(reinterpret_cast<const void *>(&k_density<MODE, BLOCK>), BLOCK);
    const uint32_t waves = pp.queue ? stencil_waves(S, pp, resident) : S.nwaves;
    hipLaunchKernelGGL((k_density<MODE, BLOCK>), dim3(std::max(1u, blocks_for_waves(waves, BLOCK))), dim3(BLOCK), 0, st,
                       a.posB, a.velB, a.cellcB, c.cstart, a.rhoB, a.posR, a.velR, S, d, pp, nl);
}

void launch_density(hipStream_t st, const ParticleArrays &a, const CellArrays &c, const SceneSet &S,
                    const PartPlan &parts, const NeighborLists &lists, int block, uint32_t *count)
{
    const NeighborDump d{count, nullptr, nullptr};
    if (count)
        return launch_density_block<3, kStencilBlock>(st, a, c, S, d, parts, lists);
    switch (block) {
    case 64:
        return launch_density_block<0, 64>(st, a, c, S, d, parts, lists);
    case 256:
        return launch_density_block<0, 256>(st, a, c, S, d, parts, lists);
    default:
        return launch_density_block<0, kStencilBlock>(st, a, c, S, d, parts, lists);
    }
}

void launch_neighbor_dump(hipStream_t st, const ParticleArrays &a, const CellArrays &c, const SceneSet &S,
                          const NeighborDump &dump)
{
    const NeighborLists none{nullptr, nullptr, 0u};
    if (dump.out)
        launch_density_block<2, kStencilBlock>(st, a, c, S, dump, PartPlan{}, none);
    else
        launch_density_block<1, kStencilBlock>(st, a, c, S, dump, PartPlan{}, none);
}

// ----------------------------------------------------- force + integrate
// Per neighbour (reference, src/sph.cpp:103-118):
//   pressure = -dir m (p_i + p_j) / (2 rho_j) spikyGrad (h - r)^2
//   visco    = mu m (v_j - v_i) / rho_j spikyLap (h - r)
// with dir = (x_j - x_i) / r.  Both are evaluated as one scalar coefficient
// times a vector, from 0.5 / rho_j precomputed by the density pass.
__device__ inline void integrate_and_walls(float4 &x, float4 &v, float fx, float fy, float fz,
                                           float rho, const StepParams &P)
{
    // src/sph.cpp:145-150: a = F / rho + (0, g, 0); v += a dt; x += v dt
    float ax = fx / rho + 0.0f;
    float ay = fy / rho + P.g;
    float az = fz / rho + 0.0f;
    v.x += ax * P.dt;
    v.y += ay * P.dt;
    v.z += az * P.dt;
    x.x += v.x * P.dt;
    x.y += v.y * P.dt;
    x.z += v.z * P.dt;
    // src/sph.cpp:153-176, planes L = lo + h, U = hi - h: floor, ceiling,
    // x-low, x-high, z-low, z-high.
    const float e = P.restitution, off = P.offset;
    if (x.y < P.wall_lo[1]) {
        x.y = -x.y + 2.0f * P.wall_lo[1] + off;
        v.y = -v.y * e;
    }
    if (x.y > P.wall_hi[1]) {
        x.y = -x.y + 2.0f * P.wall_hi[1] - off;
        v.y = -v.y * e;
    }
    if (x.x < P.wall_lo[0]) {
        x.x = -x.x + 2.0f * P.wall_lo[0] + off;
        v.x = -v.x * e;
    }
    if (x.x > P.wall_hi[0]) {
        x.x = -x.x + 2.0f * P.wall_hi[0] - off;
        v.x = -v.x * e;
    }
    if (x.z < P.wall_lo[2]) {
        x.z = -x.z + 2.0f * P.wall_lo[2] + off;
        v.z = -v.z * e;
    }
    if (x.z > P.wall_hi[2]) {
        x.z = -x.z + 2.0f * P.wall_hi[2] - off;
        v.z = -v.z * e;
    }
}

// The force of one candidate, accumulated into (fx, fy, fz):
//   cp = -m spikyGrad (p_i + p_j) m_ij (0.5 / rho_j) (h - r)^2 / r
//   cv = 2 mu m spikyLap (h - r) m_ij (0.5 / rho_j)
//   F += cp d + cv (v_j - v_i)
// q = (x_j, 0.5 / rho_j), w = (v_j, p_j), d = x_j - x_i, am = m_ij (0.5 / rho_j).
// r and h - r are the reference's values bit for bit (near the support edge
// h - r cancels, and an error in r would be amplified).
// CLAMP: also for candidates that are no neighbours, where h2 = fl(h h): they
// have d2 >= h2, so r >= h (the root of the rounded square is h itself) and
// h - r clamps to 0: they add zeros, without a test.  (With another h2 a
// neighbour may be farther than h, and h - r below zero.)  For split walks.
// SPLIT: the part of a split walk, whose sums depend on the parts' bounds
// anyway: the same product in an order that takes fewer operations and root()
// (28 against 49 issue cycles a wave before the six fmas).  Unsplit walks
// keep one order of operations in all their forms.
template <bool CLAMP, bool UNIT, bool SPLIT>
__device__ inline void force_pair(float d2, float dx, float dy, float dz, float am, float4 w, float4 vi,
                                  float p_i, float h, float neg_m_spg, float mu2_m_lap, float &fx,
                                  float &fy, float &fz)
{
    float cp, cv;
    if (SPLIT) {
        float rinv;
        const float r = root(d2, rinv);
        const float hr = CLAMP ? positive<UNIT>(h - r) : h - r;
        const float u = hr * am;
        cp = ((p_i + w.w) * neg_m_spg) * u * (hr * rinv);
        cv = u * mu2_m_lap;
    } else {
        const float r = sqrt_rn(d2);
        const float hr = CLAMP ? positive<UNIT>(h - r) : h - r;
        cp = neg_m_spg * (p_i + w.w) * am * (hr * hr) * __builtin_amdgcn_rcpf(r);
        cv = mu2_m_lap * hr * am;
    }
    fx = fmaf(cp, dx, fx);
    fy = fmaf(cp, dy, fy);
    fz = fmaf(cp, dz, fz);
    fx = fmaf(cv, w.x - vi.x, fx);
    fy = fmaf(cv, w.y - vi.y, fy);
    fz = fmaf(cv, w.z - vi.z, fz);
}

// Three walks.  Unsplit, they give the same sums bit for bit:
//  * lists, where every lane of an unsplit task has one: the listed slots,
//    four at a time.  Bound by the gathers: on cells of h / 2, where the k-th
//    neighbours of neighbouring lanes are neighbours, a million particles take
//    91 us, on cells of h 155;
//  * union: candidates shared by the wave, 64 at a time through LDS and
//    tested, or in split walks clamped to terms of zeros where they are none
//    of the lane's.  Bound by arithmetic: in a late state of a million particles (3,260 neighbours
//    each) 29 instructions, 79 cycles, a candidate: 0.70 of the issue slots at
//    two cycles each, and this mix takes 2.7;
//    4.0 ms with operands in scalar registers, a test and two
//    transcendentals a candidate, 3.55 now;
//  * per lane: candidates filtered kForceChunk at a time into a per-lane
//    bitmask, the terms then run only over the set bits, so a wave pays for
//    the most neighbours any of its lanes has in the chunk.
template <bool WRITE_FORCE, bool NEXT_KEYS, int BLOCK>
__global__ __launch_bounds__(BLOCK, 5) void k_force_integrate(
    const float4 *__restrict__ posB, const float4 *__restrict__ velB,
    const float4 *__restrict__ posR, const float4 *__restrict__ velR,
    const uint32_t *__restrict__ cellcB, const uint32_t *__restrict__ cstart,
    const float *__restrict__ rhoB, float4 *__restrict__ posA, float4 *__restrict__ velA,
    uint32_t *__restrict__ cellcA, uint32_t *__restrict__ counts,
    float4 *__restrict__ force_out, SceneSet S, PartPlan pp, NeighborLists nl)
{
    __shared__ UnionStage<2> stage[BLOCK / 64];
    for_each_part<BLOCK, false>(S, pp, pp.queue ? pp.queue + 1 : nullptr, [&](uint32_t wt, uint32_t part,
                                                                      uint32_t nparts) {
        Lane L;
        bool active;
        wave_task(S, wt, L, active);
        const StepParams &P = *L.P;
        const uint32_t s = L.slot;
        float4 pi = posR[s];        // w = 0.5 / rho_i
        const float4 vr = velR[s];  // w = p_i
        float4 vi = make_float4(vr.x, vr.y, vr.z, velB[s].w);  // w = particle id
        const uint32_t cc = cellcB[s];
        const bool slow = (cc & kSlowBit) != 0u;
        // the reference cell (three IEEE divisions) only matters for m_ij
        RefCell ci{0, 0, 0};
        if (slow)
            ci = ref_cell(pi, P);
        const float p_i = vr.w;
        const float h = in_vgpr(P.h), h2 = P.h2, neg_m_spg = in_vgpr(P.neg_m_spg);
        const float mu2_m_lap = in_vgpr(2.0f * P.mu_m_lap);
        float fx = 0.0f, fy = 0.0f, fz = 0.0f;

        // The term of neighbour j in the order the walks visit it.
        auto pair = [&](uint32_t j, float4 q, float4 w) {
            float dx, dy, dz;
            const float d2 = dist2_ref(pi, q, dx, dy, dz);
            float am = q.w;  // 0.5 / rho_j
            if (slow) {
                int cx = ci.x, cy = ci.y, cz = ci.z;
                asm volatile("" : "+v"(cx), "+v"(cy), "+v"(cz));
                am = q.w * (float)bucket_multiplicity(cx, cy, cz, __float_as_uint(posB[j].w) & 0xFFFFu);
            }
            force_pair<false, false, false>(d2, dx, dy, dz, am, w, vi, p_i, h, neg_m_spg, mu2_m_lap, fx, fy, fz);
        };
        // Every lane holds its neighbour list (the task is unsplit; the
        // planning pass or the density pass has recorded them): visit the
        // listed slots four at a time, the next group of four slots loaded
        // while the current one runs; entries past a lane's list stand for its
        // own slot and add nothing.
        const uint32_t listed = nparts == 1u ? nl.count[s] : kNoList;
        const bool use_list = nparts == 1u && __all(listed != kNoList);
        UnionRows U;
        if (use_list) {
            const uint32_t groups = ((uint32_t)wave_max_i((int)listed) + 3u) >> 2;
            const uint32_t *ent = nl.list + s;
            const size_t stride = nl.stride;
            // groups <= kListMax / 4, so every entry loaded lies inside the
            // list array; entries a lane has not written are never used
            auto group = [&](uint32_t g) {
                const uint32_t *e0 = ent + (size_t)(4u * g) * stride;
                return make_uint4(e0[0], e0[stride], e0[2 * stride], e0[3 * stride]);
            };
            uint4 next = group(0);
            for (uint32_t g = 0; g < groups; ++g) {
                const uint32_t k = 4u * g;
                const uint4 cur = next;
                if (g + 1u < groups)
                    next = group(g + 1u);
                const uint32_t j0 = k < listed ? cur.x : s, j1 = k + 1u < listed ? cur.y : s;
                const uint32_t j2 = k + 2u < listed ? cur.z : s, j3 = k + 3u < listed ? cur.w : s;
                const float4 q0 = posR[j0], w0 = velR[j0], q1 = posR[j1], w1 = velR[j1];
                const float4 q2 = posR[j2], w2 = velR[j2], q3 = posR[j3], w3 = velR[j3];
                if (k < listed)
                    pair(j0, q0, w0);
                if (k + 1u < listed)
                    pair(j1, q1, w1);
                if (k + 2u < listed)
                    pair(j2, q2, w2);
                if (k + 3u < listed)
                    pair(j3, q3, w3);
            }
        } else if (walk_of(pp, wt, U)) {  // as in k_density
            UnionStage<2> &T = stage[threadIdx.x >> 6];
            uint32_t lo, hi;
            part_slice(union_rows(cstart, U, cc, active, P, T), part, nparts, lo, hi);
            const float4 *const src[2] = {posR, velR};
            // Values that are not finite (or far beyond any scene's) would
            // reach a lane through a candidate that is no neighbour (0 x inf):
            // a chunk that holds some, and every chunk of a wave that does, is
            // walked with a test per candidate, as are the wave's own slots, and
            // every chunk of a scene whose h2 is not its h squared (force_pair).
            const float limit = P.zero_limit;
            const bool plain = __all(fabsf(pi.x) + fabsf(pi.y) + fabsf(pi.z) + fabsf(vi.x) + fabsf(vi.y) +
                                         fabsf(vi.z) + fabsf(p_i) <= limit);
            // A test also lets the wave skip a candidate that is no lane's
            // neighbour.  That pays in unsplit walks, whose pair terms are the
            // dearer ones (a lattice of spacing 0.4 h, 97 thousand particles:
            // 281 us without, 212 with), and on cells much larger than h, where
            // two thirds of the candidates are such (spacing h / 2 on cells of
            // 1.7 h, 262 thousand: 336 and 232).
            const bool tested = !plain || (P.reach == 1 && P.grid_inv * (double)P.h < 0.8);
            const uint32_t W = 2u * (uint32_t)P.reach + 1u;
            uint32_t at_layer = kNoSlot;
            bool mine = true;  // the chunk's candidates are those of the lane's segment
            auto walk = [&](auto unit_tag, auto split_tag) {
                constexpr bool unit = decltype(unit_tag)::value, split = decltype(split_tag)::value;
                union_walk<2, true>(lo, hi, L.first, limit, src, T, [&](const ChunkRecords<2> &c, const uint32_t *slots,
                                                                     uint32_t n, bool odd, uint32_t lz) {
                    const float4(&rec)[2][64] = c.rec;
                    float dx, dy, dz;
                    if (U.segments && lz != at_layer) {
                        at_layer = lz;
                        mine = T.segment[threadIdx.x & 63u] == lz / W;
                    }
                    if (!split || odd || tested) {
                        for (uint32_t k = 0; k < n; k += 4u) {
                            float4 q[4], w[4];  // (x_j, 0.5 / rho_j), (v_j, p_j)
#pragma unroll
                            for (uint32_t i = 0; i < 4u; ++i) {
                                q[i] = rec[0][k + i];
                                w[i] = rec[1][k + i];
                            }
                            const uint4 j = *reinterpret_cast<const uint4 *>(&slots[k]);
                            auto visit = [&](uint32_t slot, const float4 &qi, const float4 &wi) {
                                const float d2 = dist2_ref(pi, qi, dx, dy, dz);
                                if (d2 < h2 && mine && slot != s && slot != kNoSlot)
                                    force_pair<false, unit, split>(d2, dx, dy, dz, qi.w, wi, vi, p_i, h, neg_m_spg, mu2_m_lap,
                                                                   fx, fy, fz);
                            };
                            visit(j.x, q[0], w[0]);
                            visit(j.y, q[1], w[1]);
                            visit(j.z, q[2], w[2]);
                            visit(j.w, q[3], w[3]);
                        }
                        return;
                    }
                    const float4 me = make_float4(mine ? pi.x : kFarAway, pi.y, pi.z, 0.0f);
                    for (uint32_t k = 0; k < n; k += 2u) {
                        const float4 q0 = rec[0][k], w0 = rec[1][k], q1 = rec[0][k + 1u], w1 = rec[1][k + 1u];
                        float d2 = dist2_ref(me, q0, dx, dy, dz);
                        force_pair<true, unit, split>(d2, dx, dy, dz, q0.w, w0, vi, p_i, h, neg_m_spg, mu2_m_lap, fx, fy, fz);
                        d2 = dist2_ref(me, q1, dx, dy, dz);
                        force_pair<true, unit, split>(d2, dx, dy, dz, q1.w, w1, vi, p_i, h, neg_m_spg, mu2_m_lap, fx, fy, fz);
                    }
                });
            };
            if (nparts == 1u)
                walk(std::false_type{}, std::false_type{});
            else if (P.h <= 1.0f)
                walk(std::true_type{}, std::true_type{});
            else
                walk(std::false_type{}, std::true_type{});
        } else {
            uint32_t lo = 0, hi = 0xFFFFFFFFu;
            if (nparts > 1u) {
                const uint32_t own = own_length(pp, s, cstart, cc, P);
                lo = (uint32_t)((uint64_t)own * part / nparts);
                hi = (uint32_t)((uint64_t)own * (part + 1u) / nparts);
            }
            for_each_row_span(cstart, cc, P, lo, hi, [&](uint32_t b, uint32_t e) {
                for (uint32_t jj = b; jj < e; jj += kForceChunk) {
                    uint32_t mask = 0u;
#pragma unroll
                    for (int k = 0; k < kForceChunk; ++k) {
                        const uint32_t j = jj + (uint32_t)k;
                        const float4 q = posR[j < e ? j : e - 1u];
                        float dx, dy, dz;
                        const float d2 = dist2_ref(pi, q, dx, dy, dz);
                        const bool pass = (j < e) && (j != s) && (d2 < h2);
                        mask |= pass ? (1u << k) : 0u;
                    }
                    while (mask != 0u) {
                        const uint32_t k = (uint32_t)__builtin_ctz(mask);
                        mask &= mask - 1u;
                        const uint32_t j = jj + k;
                        pair(j, posR[j], velR[j]);  // (x_j, 0.5 / rho_j), (v_j, p_j)
                    }
                }
            });
        }
        if (nparts > 1u) {
            float v[3] = {fx, fy, fz};
            if (!combine_parts<3>(pp, wt, part, nparts, v))
                return;
            fx = v[0];
            fy = v[1];
            fz = v[2];
        }
        if (!active)
            return;
        if (WRITE_FORCE)
            force_out[s] = make_float4(fx, fy, fz, 0.0f);
        integrate_and_walls(pi, vi, fx, fy, fz, rhoB[s], P);
        if (NEXT_KEYS) {
            Classified c = classify(pi.x, pi.y, pi.z, P);
            pi.w = __uint_as_float(c.h16);
            cellcA[s] = c.cellc;
            atomicAdd(&counts[linear_cell(P, c.cellc)], 1u);  // no result: nothing waits on it
        } else {
            pi.w = 0.0f;
        }
        posA[s] = pi;
        velA[s] = vi;
    });
}

template <int BLOCK>
static void launch_force_block(hipStream_t st, const ParticleArrays &a, const CellArrays &c, const SceneSet &S,
                               float4 *force_out, bool next_keys, const PartPlan &pp, const NeighborLists &nl)
{
    static const uint32_t resident =
        occupancy_waves(reinterpret_cast<const void *>(&k_force_integrate<false, true, BLOCK>), BLOCK);
    dim3 g(std::max(1u, blocks_for_waves(stencil_waves(S, pp, resident), BLOCK))), b(BLOCK);
#define SPH_LAUNCH_FI(WF, NK)                                                                          \
    hipLaunchKernelGGL((k_force_integrate<WF, NK, BLOCK>), g, b, 0, st, a.posB, a.velB, a.posR, a.velR, \
                       a.cellcB, c.cstart, a.rhoB, a.posA, a.velA, a.cellcA, c.counts,         \
                       force_out, S, pp, nl)
    if (force_out && next_keys)
        SPH_LAUNCH_FI(true, true);
    else if (force_out)
        SPH_LAUNCH_FI(true, false);
    else if (next_keys)
        SPH_LAUNCH_FI(false, true);
    else
        SPH_LAUNCH_FI(false, false);
#undef SPH_LAUNCH_FI
}

void launch_force_integrate(hipStream_t st, const ParticleArrays &a, const CellArrays &c,
                            const SceneSet &S, float4 *force_out, bool next_keys, const PartPlan &parts,
                            const NeighborLists &lists, int block)
{
    switch (block) {
    case 64:
        return launch_force_block<64>(st, a, c, S, force_out, next_keys, parts, lists);
    case 256:
        return launch_force_block<256>(st, a, c, S, force_out, next_keys, parts, lists);
    default:
        return launch_force_block<kStencilBlock>(st, a, c, S, force_out, next_keys, parts, lists);
    }
}

// ------------------------------------------------------- grid statistic
// Candidates per neighbour of a sample of every scene: its wave tasks
// 0, kGridStatEvery, 2 kGridStatEvery, ... (counted from the scene's own
// first slot, so the sample is the same in any batch) walk their lanes' whole
// stencils over the current cell ranges and B order, counting the
// candidates and those within h (the particle itself excluded); each
// wave adds its sums to stat[2 scene] and stat[2 scene + 1].  The ratio
// tells a state uniform at the scale of h (a jittered lattice of spacing
// h / 2 reads 7.2 at cell scale 1, 4.2 at cell scale 1/2) from one clumped
// below it (near 1).  Lanes with more than kGridStatTests candidates (the
// clumps of a collapsed flow, thousands each) test an evenly strided subset
// and scale their count, so the sample costs a few hundred tests a lane
// however dense the state; the uniform states the choice turns on have
// fewer candidates and are counted exactly.
__global__ __launch_bounds__(kBlock) void k_grid_stat(const float4 *__restrict__ pos,
                                                     const uint32_t *__restrict__ cellc,
                                                     const uint32_t *__restrict__ cstart, SceneSet S,
                                                     unsigned long long *__restrict__ stat)
{
    const uint32_t w = __builtin_amdgcn_readfirstlane(blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6));
    if (w >= S.nwaves)
        return;
    Lane L;
    bool active;
    wave_task(S, w, L, active);
    const StepParams &P = *L.P;
    if (((L.first - P.p_begin) / 64u) % kGridStatEvery != 0u)
        return;  // the sample counts tasks from the scene's own first slot
    const uint32_t s = L.slot;
    uint32_t cand = 0, nbr = 0;
    if (active) {
        const float4 pi = pos[s];
        const float h2 = P.h2;
        const uint32_t cc = cellc[s];
        for_each_row(cstart, cc, P, [&](uint32_t b, uint32_t e) { cand += e - b; });
        const uint32_t stride = max((cand + kGridStatTests - 1u) / kGridStatTests, 1u);
        uint32_t q = 0;  // offset of the next tested candidate in the current row
        for_each_row(cstart, cc, P, [&](uint32_t b, uint32_t e) {
            for (; q < e - b; q += stride) {
                const uint32_t j = b + q;
                float dx, dy, dz;
                nbr += (j != s && dist2_ref(pi, pos[j], dx, dy, dz) < h2) ? 1u : 0u;
            }
            q -= e - b;
        });
        nbr *= stride;
    }
    unsigned long long c = cand, nb = nbr;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        c += __shfl_xor(c, d, 64);
        nb += __shfl_xor(nb, d, 64);
    }
    if ((threadIdx.x & 63u) == 0u) {
        const uint32_t scene = S.tasks[w].scene;
        atomicAdd(&stat[2u * scene], c);
        atomicAdd(&stat[2u * scene + 1u], nb);
    }
}

void launch_grid_stat(hipStream_t st, const ParticleArrays &a, const CellArrays &c, const SceneSet &S,
                      unsigned long long *stat, uint32_t nscenes)
{
    launch_fill_u32(st, (uint32_t *)stat, 0u, 4ull * nscenes);
    if (S.nwaves)
        hipLaunchKernelGGL(k_grid_stat, dim3(blocks_for_waves(S.nwaves, kBlock)), dim3(kBlock), 0, st, a.posB,
                           a.cellcB, c.cstart, S, stat);
}

// ------------------------------------------------------- drop-in output
// glm::translate(x) * glm::scale(vec3(s)) with glm's column arithmetic
// (src/sph.cpp:179-180): T[3] = I0 x + I1 y + I2 z + I3, then
// M[c] = T0 S[c][0] + T1 S[c][1] + T2 S[c][2] + T3 S[c][3].
__device__ inline void write_transform(float *__restrict__ xf, float x, float y, float z, float sc)
{
    const float pos[3] = {x, y, z};
    float T3[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        float a0 = (r == 0) ? 1.0f : 0.0f, a1 = (r == 1) ? 1.0f : 0.0f, a2 = (r == 2) ? 1.0f : 0.0f;
        float a3 = (r == 3) ? 1.0f : 0.0f;
        T3[r] = ((a0 * pos[0] + a1 * pos[1]) + a2 * pos[2]) + a3;
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const float s0 = (c == 0) ? sc : 0.0f, s1 = (c == 1) ? sc : 0.0f;
        const float s2 = (c == 2) ? sc : 0.0f, s3 = (c == 3) ? 1.0f : 0.0f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float t0 = (r == 0) ? 1.0f : 0.0f, t1 = (r == 1) ? 1.0f : 0.0f, t2 = (r == 2) ? 1.0f : 0.0f;
            xf[c * 4 + r] = ((t0 * s0 + t1 * s1) + t2 * s2) + T3[r] * s3;
        }
    }
}

__global__ void k_h16_rank(const float4 *__restrict__ posB, uint32_t *__restrict__ counts16,
                           uint32_t *__restrict__ rank16, uint32_t n)
{
    uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n)
        return;
    uint32_t h = __float_as_uint(posB[s].w) & 0xFFFFu;
    rank16[s] = atomicAdd(&counts16[h], 1u);
}

void launch_h16_rank(hipStream_t st, const ParticleArrays &a, const CellArrays &c16, uint32_t n)
{
    // rankA is free once the force pass ran without next keys
    hipLaunchKernelGGL(k_h16_rank, dim3(blocks_for(n)), dim3(kBlock), 0, st, a.posB, c16.counts,
                       a.rankA, n);
}

// perm16: the buckets' input indices, in arrival order; slot_of: where each is.
__global__ void k_h16_scatter(const float4 *__restrict__ posB, const float4 *__restrict__ velB,
                              const uint32_t *__restrict__ rank16, const uint32_t *__restrict__ cstart16,
                              uint32_t *__restrict__ perm16, uint32_t *__restrict__ slot_of, uint32_t n)
{
    uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n)
        return;
    const uint32_t h = __float_as_uint(posB[s].w) & 0xFFFFu, id = __float_as_uint(velB[s].w);
    perm16[cstart16[h] + rank16[s]] = id;
    slot_of[id] = s;
}

// Also sorts the buckets above kSmallCell by index, as the cells of the step
// are (those above kBigCellSortMax keep arrival order).
void launch_h16_scatter(hipStream_t st, const ParticleArrays &a, const CellArrays &c16, uint32_t n,
                        uint32_t *perm16)
{
    // cellcA is free once the force pass ran without next keys
    hipLaunchKernelGGL(k_h16_scatter, dim3(blocks_for(n)), dim3(kBlock), 0, st, a.posB, a.velB, a.rankA,
                       c16.cstart, perm16, a.cellcA, n);
    ParticleArrays sorted = a;
    sorted.perm = perm16;
    if (n > kSmallCell)
        launch_sort_big_cells(st, sorted, c16);
}

// Output slot o: particle perm16[o].  In a bucket of up to kSmallCell it
// lands at the bucket start plus the number of members with a smaller index
// (ties of std::sort resolved by input order); the others are sorted.
// (Counting in buckets of any size, 51 thousand particles with some in the
// thousands: 172 us; now the sort takes 12 and this 10.)
__global__ void k_pack_out(const uint32_t *__restrict__ perm16, const uint32_t *__restrict__ cstart16,
                           const uint32_t *__restrict__ slot_of, const float4 *__restrict__ posB,
                           const float *__restrict__ rhoB, const float4 *__restrict__ velR,
                           const float4 *__restrict__ force, const float4 *__restrict__ posA,
                           const float4 *__restrict__ velA, const float *__restrict__ aos_in,
                           float *__restrict__ aos_out, float *__restrict__ xf_out, uint32_t n,
                           float sc)
{
    uint32_t o = blockIdx.x * blockDim.x + threadIdx.x;
    if (o >= n)
        return;
    const uint32_t id = perm16[o], s = slot_of[id];
    const uint32_t h = __float_as_uint(posB[s].w) & 0xFFFFu;
    const uint32_t b = cstart16[h], e = cstart16[h + 1];
    uint32_t d = o;
    if (e - b <= kSmallCell) {
        uint32_t r = 0;
        for (uint32_t t = b; t < e; ++t)
            r += perm16[t] < id ? 1u : 0u;
        d = b + r;
    }
    const float4 x = posA[s], v = velA[s], f = force[s];
    const float *src = aos_in + (size_t)id * 15;
    float *dst = aos_out + (size_t)d * 15;
    dst[0] = x.x;
    dst[1] = x.y;
    dst[2] = x.z;
    dst[3] = v.x;
    dst[4] = v.y;
    dst[5] = v.z;
    dst[6] = src[6];
    dst[7] = src[7];
    dst[8] = src[8];
    dst[9] = f.x;
    dst[10] = f.y;
    dst[11] = f.z;
    dst[12] = rhoB[s];
    dst[13] = velR[s].w;
    dst[14] = __uint_as_float(h);  // uint16 hash + zero padding (little endian)
    if (xf_out)
        write_transform(xf_out + (size_t)d * 16, x.x, x.y, x.z, sc);
}

void launch_pack_out(hipStream_t st, const ParticleArrays &a, const CellArrays &c16,
                     const uint32_t *perm16, const float4 *force, const void *aos_in, uint32_t n,
                     float xf_scale, void *aos_out, float *xf_out)
{
    hipLaunchKernelGGL(k_pack_out, dim3(blocks_for(n)), dim3(kBlock), 0, st, perm16, c16.cstart,
                       a.cellcA, a.posB, a.rhoB, a.velR, force, a.posA, a.velA,
                       (const float *)aos_in, (float *)aos_out, xf_out, n, xf_scale);
}

// Resident download: slots [first, first + n) of the A arrays (device
// order).  Bucket, density and pressure belong to the last step (B slot s is
// the same particle).
__global__ void k_pack_state(const float4 *__restrict__ posA, const float4 *__restrict__ velA,
                             const float4 *__restrict__ posB, const uint32_t *__restrict__ kept,
                             const float *__restrict__ rhoB, const float4 *__restrict__ velR,
                             const float4 *__restrict__ force, float *__restrict__ aos_out,
                             float *__restrict__ xf_out, uint32_t first,
                             uint32_t n, float sc)
{
    uint32_t o = blockIdx.x * blockDim.x + threadIdx.x;
    if (o >= n)
        return;
    const uint32_t s = first + o;
    const float4 x = posA[s], v = velA[s];
    const float4 f = force ? force[s] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float *dst = aos_out + (size_t)o * 15;
    dst[0] = x.x;
    dst[1] = x.y;
    dst[2] = x.z;
    dst[3] = v.x;
    dst[4] = v.y;
    dst[5] = v.z;
    dst[6] = 0.0f;
    dst[7] = 0.0f;
    dst[8] = 0.0f;
    dst[9] = f.x;
    dst[10] = f.y;
    dst[11] = f.z;
    dst[12] = rhoB[s];
    dst[13] = velR[s].w;
    dst[14] = __uint_as_float(kept ? kept[s] : __float_as_uint(posB[s].w) & 0xFFFFu);
    if (xf_out)
        write_transform(xf_out + (size_t)o * 16, x.x, x.y, x.z, sc);
}

__global__ void k_keep_hashes(const float4 *__restrict__ posB, uint32_t *__restrict__ kept, uint32_t n)
{
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < n)
        kept[s] = __float_as_uint(posB[s].w) & 0xFFFFu;
}

void launch_keep_hashes(hipStream_t st, const ParticleArrays &a, uint32_t n)
{
    hipLaunchKernelGGL(k_keep_hashes, dim3(blocks_for(n)), dim3(kBlock), 0, st, a.posB, a.rankA, n);
}

void launch_pack_state(hipStream_t st, const ParticleArrays &a, bool kept, const float4 *force, uint32_t first,
                       uint32_t n, float xf_scale, void *aos_out, float *xf_out)
{
    hipLaunchKernelGGL(k_pack_state, dim3(blocks_for(n)), dim3(kBlock), 0, st, a.posA, a.velA,
                       a.posB, kept ? a.rankA : nullptr, a.rhoB, a.velR, force, (float *)aos_out, xf_out, first, n,
                       xf_scale);
}

// ------------------------------------------------------------------ copy

__global__ void k_copy(const uint4 *__restrict__ src, uint4 *__restrict__ dst, size_t n16)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n16; i += stride)
        dst[i] = src[i];
}

void launch_copy(hipStream_t st, const uint4 *src, uint4 *dst, size_t n16)
{
    size_t nb = (n16 + kBlock - 1) / kBlock;
    if (nb > 65536)
        nb = 65536;
    hipLaunchKernelGGL(k_copy, dim3((uint32_t)nb), dim3(kBlock), 0, st, src, dst, n16);
}

}  // namespace sph
