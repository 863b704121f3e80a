// pbf_kernels.hip -- the PBF step on gfx950, one thread per particle slot.
//
// Stage map (reference kernel -> kernel here):
//   kernel_predict_position + kernel_compute_hashes     -> k_predict_hash
//   thrust::sort of the records                         -> radix sort by hash (logical order),
//                                                          k_cell_keys, radix sort by super-cell
//                                                          (physical order), k_gather
//   table fill + kernel_build_hash_table                -> k_cell_keys (cell-table inserts)
//   kernel_find_neighbours                              -> k_neighbours_wave (k_neighbours for very
//                                                          long lists)
//   kernel_calculate_densities + kernel_calculate_lambdas   -> k_density_lambda (one sweep)
//   kernel_calculate_position_delta + kernel_correct_position -> k_delta_correct
//   ... last iteration also kernel_update_position_and_velocity
//       + kernel_apply_boundary_velocity_damping        -> k_delta_correct<final>
//   kernel_compute_vorticities                          -> k_vorticity
//   kernel_apply_vorticity_confinement                  -> k_confinement
//   kernel_apply_xsph_viscosity (Jacobi)                -> k_xsph
// Every kernel reads the previous kernel's complete output (Jacobi), like the reference's
// launch-then-synchronise sequence, except XSPH, which reads a copy of the velocities instead of
// racing on them.
//
// Kernels that walk neighbours map workgroups to XCDs by chunks of physical slots (xcd_block), so that
// each XCD's L2 serves spatially coherent ranges of the particles.
#include "pbf_kernels.h"

#include <algorithm>
#include <map>
#include <mutex>
#include <stdexcept>
#include <string>
#include <type_traits>
#include "boundary.h"
#include "pbf_math.h"

namespace akua {

namespace {

constexpr uint32_t kXcds = kXcdCount;

__device__ __forceinline__ const SceneDev& scene_of(const DeviceState& d, uint32_t i) {
    return d.scenes[d.chunkScene[i >> 8]];
}

// The neighbour list in chunks of four entries: chunk c (entries 4c..4c+3) of slot i is the
// uint4 at list_base(i) + c * 64, so the 64 lanes of a wave read chunk c of their lists as one
// 1 KB block (one 16-byte load per lane for four entries).
__device__ __forceinline__ uint32_t list_chunks(int maxN) { return ((uint32_t)maxN + 3u) >> 2; }
__device__ __forceinline__ size_t list_base(uint32_t i, int maxN) {
    return (size_t)(i >> 6) * (size_t)list_chunks(maxN) * 64u + (i & 63u);
}

// Visits the n entries of a neighbour list in order.  Memory requests are issued kListBatch at a
// time (the neighbours' data through load(j)), then body(value) runs for each entry in list order,
// so every per-particle sum keeps its reference order.  The list chunks of the next batch are
// loaded while the current batch's data is in flight, so a batch's gathers wait only for
// themselves, not for a list load before them.
constexpr int kListBatch = 4;
// per-kernel batch: 4 where the 8-entry batch's registers would cost occupancy
constexpr int kBatchDelta = 4, kBatchVort = 4, kBatchConf = 4, kBatchXsph = 8;

template <class T, int B = kListBatch, class Load, class Body>
__device__ __forceinline__ void walk_list(const uint4* __restrict__ lp, uint32_t n, Load load,
                                          Body body) {
    static_assert(B == 4 || B == 8, "one or two chunks per batch");
    if (n == 0u) return;
    uint4 a = lp[0];
    uint4 b = (B == 8 && n > 4u) ? lp[64] : a;
    for (uint32_t k0 = 0; k0 < n; k0 += B) {
        uint32_t j[8];
        j[0] = a.x; j[1] = a.y; j[2] = a.z; j[3] = a.w;
        if (B == 8) {
            j[4] = b.x; j[5] = b.y; j[6] = b.z; j[7] = b.w;
        }
        // entries past n are not list entries: load a valid one in their place (discarded)
#pragma unroll
        for (int u = 1; u < B; ++u) j[u] = k0 + u < n ? j[u] : j[0];
        T v[B];
#pragma unroll
        for (int u = 0; u < B; ++u) v[u] = load(j[u]);
        const uint32_t k1 = k0 + B;
        if (k1 < n) {
            a = lp[(size_t)(k1 >> 2) * 64u];
            if (B == 8) b = k1 + 4u < n ? lp[(size_t)((k1 >> 2) + 1u) * 64u] : a;
        }
#pragma unroll
        for (int u = 0; u < B; ++u)
            if (k0 + u < n) body(v[u]);
    }
}

struct XLam {
    float4 x;
    float lam;
};
struct XV {
    float4 x;
    float4 v;
};
struct XW {
    float4 x;
    float w;
};

// Element j of a per-slot array through a 32-bit byte offset from its base: slot counts stay
// below kMaxSlots (2^28), so j * sizeof(T) <= 16 j fits in 32 bits, and the gather then takes the
// base from scalar registers and one 32-bit lane offset instead of a 64-bit address per lane.
template <class T>
__device__ __forceinline__ T ld(const T* __restrict__ base, uint32_t j) {
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + (uint32_t)(j * (uint32_t)sizeof(T)));
}

// The work of workgroup b of nb (a multiple of 8), of `per` slots each: the hardware places b on XCD b % 8,
// which takes every eighth chunk of kXcdChunk slots, and of the rest a contiguous eighth.  A chunk's data
// and its surroundings stay in one XCD's L2; eighths of a whole scene differ in density, so that one XCD
// works longest (us per step by launch_tally, one eighth / chunks of 32,768 / 4,096: 8M two columns 14,596 /
// 11,370 / 11,213, sprayed 1M 1,394 / 1,257 / 1,281, learned 1M 959 / 942 / 938; 64 scenes 2,449 / 2,468 /
// 2,461).
constexpr uint32_t kXcdChunk = 32768u;
__device__ __forceinline__ uint32_t xcd_block(uint32_t b, uint32_t nb, uint32_t per) {
    const uint32_t x = b % kXcds, j = b / kXcds, mine = nb / kXcds;
    const uint32_t c = kXcdChunk / per, whole = mine / c * c;
    return j < whole ? (j / c * kXcds + x) * c + j % c : whole * kXcds + x * (mine - whole) + (j - whole);
}

// Physical slot of this thread (with L lanes per slot: its lane's index among all slots' lanes).
template <int BS, int L = 1>
__device__ __forceinline__ uint32_t xcd_slot() {
    return xcd_block(blockIdx.x, gridDim.x, BS / L) * BS + threadIdx.x;
}

// The same slot for virtual workgroup vb of nvb (a kernel that loops over virtual workgroups
// with a smaller grid).
template <int BS>
__device__ __forceinline__ uint32_t xcd_slot_of(uint32_t vb, uint32_t nvb) {
    return xcd_block(vb, nvb, BS) * BS + threadIdx.x;
}

__global__ void k_fill_u32(uint32_t* __restrict__ p, uint32_t n, uint32_t v) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

__global__ void k_fill_u4(uint4* __restrict__ p, uint32_t n, uint32_t v) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = make_uint4(v, v, v, v);
}

__device__ __forceinline__ uint32_t spread3(uint32_t x) {
    x &= 0x3FFu;
    x = (x | (x << 16)) & 0xFF0000FFu;
    x = (x | (x << 8)) & 0x0300F00Fu;
    x = (x | (x << 4)) & 0x030C30C3u;
    x = (x | (x << 2)) & 0x09249249u;
    return x;
}

// Morton code of the particle's super-cell (2^L cells per axis, L = layoutOrigin[3]), relative to
// the scene's layout origin and clamped to the key range.  It only decides where the particle's
// data is stored.
__device__ __forceinline__ uint32_t layout_key(int cx, int cy, int cz, const SceneDev& sc) {
    const int hi = (1 << sc.layoutBits) - 1;
    const int L = sc.layoutOrigin[3];
    int u = min(max((cx >> L) - sc.layoutOrigin[0], 0), hi);
    int v = min(max((cy >> L) - sc.layoutOrigin[1], 0), hi);
    int w = min(max((cz >> L) - sc.layoutOrigin[2], 0), hi);
    return spread3((uint32_t)u) | (spread3((uint32_t)v) << 1) | (spread3((uint32_t)w) << 2);
}

// kernel_predict_position (IntegrationCUDA.cu:27-36) + kernel_compute_hashes
// (NeighbourSearchCUDA.cu:36-44) with smoothRadius as the cell size (NeighbourSearchCUDA.cu:163).
// The hash, and the layout key with the particle's current physical slot, are stored at its
// previous logical index, the first sort's input order.
// layoutPrev: the layout sort runs over the previous logical order too, in the hash sort's
// launches (single-cell super-cells, where the previous and the new logical order agree within
// every layout key): its keys go straight into its input (keysM) and the record keeps only the
// slot, to which k_cell_keys adds the new logical index.
// Blocks from predictBlocks on clear the cell table instead (every record empty), the next kZeroBlocks
// zero the sorts' scratch spans and the last gathers what the import found in the masses: none of it is
// touched by the prediction, so one launch serves all four.
constexpr uint32_t kZeroBlocks = 8;

// Masses taken from device memory (SphParams::fast 2): massesDiffer becomes 0 where every 256 imported
// records had unit masses, else 1.  Every thread of one workgroup.
__device__ __forceinline__ void gather_masses(const DeviceState& d, const SphParams& P) {
    if (P.fast != 2) return;
    const uint32_t blocks = (d.nslots + 255u) / 256u;
    int differ = 0;
    for (uint32_t b = threadIdx.x; b < blocks; b += kBlock) differ |= d.blockMasses[b] != 0u;
    differ = __syncthreads_or(differ);
    if (threadIdx.x == 0) *d.massesDiffer = differ ? 1u : 0u;
}

__global__ __launch_bounds__(kBlock) void k_predict_hash(DeviceState d, SphParams P, StepParams S,
                                                         bool layoutPrev, uint32_t predictBlocks,
                                                         uint32_t clearBlocks, SortZeroSpans zero) {
    if (blockIdx.x == gridDim.x - 1u) {
        gather_masses(d, P);
        return;
    }
    if (blockIdx.x >= predictBlocks + clearBlocks) {
        const uint32_t i = (blockIdx.x - predictBlocks - clearBlocks) * kBlock + threadIdx.x;
#pragma unroll
        for (uint32_t s = 0; s < 6; ++s) {
            if (s >= zero.count) break;
            for (uint32_t k = i; k < zero.n[s]; k += kZeroBlocks * kBlock) zero.p[s][k] = 0u;
        }
        return;
    }
    if (blockIdx.x >= predictBlocks) {
        const uint32_t i = (blockIdx.x - predictBlocks) * kBlock + threadIdx.x;
        if (i < d.tableTotal) d.table[i] = make_uint4(kEmptyKey, kEmptyKey, kEmptyKey, kEmptyKey);
        return;
    }
    uint32_t p = blockIdx.x * kBlock + threadIdx.x;
    if (p >= d.nslots) return;
    const SceneDev& sc = scene_of(d, p);
    if (p >= sc.end) return;
    float4 x = d.X[p], v = d.V[p];
    f3 xs = predict_x(make3(x), make3(v), S);
    int cx, cy, cz;
    discretize(xs, P.cellHash, cx, cy, cz);
    const uint32_t k = d.lid[p];
    d.keysL[k] = P.searchCells == 2 ? cell_key_fine(cx, cy, cz) : cell_hash(cx, cy, cz, sc);
    if (layoutPrev) {
        d.keysM[k] = layout_key(cx, cy, cz, sc);
        d.layPhys[k] = make_uint2(0u, p);
    } else {
        d.layPhys[k] = make_uint2(layout_key(cx, cy, cz, sc), p);
    }
}

__device__ __forceinline__ uint32_t table_insert(uint4* table, const SceneDev& sc, uint32_t h) {
    const uint32_t mask = (1u << sc.tabLog2) - 1u;
    uint32_t s = table_slot(h, sc.tabLog2);
    // The table holds at least twice as many slots as the scene has particles, so an empty
    // slot is always found; the probe count is bounded all the same.
    for (uint32_t probe = 0; probe <= mask; ++probe) {
        uint32_t prev = atomicCAS(&table[sc.tabOffset + s].x, kEmptyKey, h);
        if (prev == kEmptyKey || prev == h) return sc.tabOffset + s;
        s = (s + 1u) & mask;
    }
    return kEmptyKey;
}

// Per logical index k: the layout key (second sort's input), the previous physical slot of the
// particle, and the cell-table entry of k's bucket (kernel_build_hash_table,
// NeighbourSearchCUDA.cu:52-65, plus the bucket end the reference finds by scanning).
// kKeep: the physical layout is kept this step (every particle stays in its slot), so instead of
// the layout key, the inverse map physical slot -> new logical index is written directly.
// layoutPrev (not with kKeep): the layout was sorted over the previous logical order, so the
// record at the previous logical index receives the new one instead (read back by k_gather).
template <bool kKeep>
__global__ __launch_bounds__(kBlock) void k_cell_keys(DeviceState d, SphParams P, StepParams S,
                                                      bool layoutPrev) {
    uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= d.nslots) return;
    const SceneDev& sc = scene_of(d, k);
    if (k >= sc.end) return;
    const uint32_t prevLogical = d.perm1[k];
    if (prevLogical >= d.nslots) return;  // a consistent sort never produces this
    if (!kKeep && layoutPrev) {
        reinterpret_cast<uint32_t*>(d.layPhys)[2u * prevLogical] = k;
    } else {
        const uint2 lp = d.layPhys[prevLogical];  // (layout key, previous physical slot)
        const uint32_t src = lp.y;
        if (kKeep) {
            if (src < d.nslots) d.perm2keep[src] = k;
        } else {
            d.keysM[k] = lp.x;
        }
        d.srcL[k] = src;
    }
    const uint32_t h = d.skeys[k];
    const bool first = (k == sc.begin) || (d.skeys[k - 1] != h);
    const bool last = (k + 1 == sc.end) || (d.skeys[k + 1] != h);
    if (first || last) {
        uint32_t slot = table_insert(d.table, sc, h);
        if (slot != kEmptyKey) {
            if (first) d.table[slot].y = k;
            if (last) d.table[slot].z = k + 1;
        }
        if (first) d.bslot[k] = slot;
    }
}

// Moves each particle to its new physical slot (the record move of the reference's thrust::sort).
// x* is recomputed from the gathered x and v with the same operations as k_predict_hash, so it is
// bit-identical to the value that was hashed.
// kCarry: also the previous density and lambda (read by a step without iterations and by the
// learned features; a step with iterations rewrites both before anything reads them).
// kCarryDelta: also the position delta (a step without iterations keeps the previous one).
// layoutPrev: the layout was sorted over the previous logical order, so perm2 gives the previous
// logical index, whose record holds the new logical index and the previous physical slot.
template <bool kCarry, bool kCarryDelta>
__global__ __launch_bounds__(kBlock) void k_gather(DeviceState d, SphParams P, StepParams S,
                                                   bool layoutPrev) {
    uint32_t p = blockIdx.x * kBlock + threadIdx.x;
    if (p >= d.nslots) return;
    const SceneDev& sc = scene_of(d, p);
    if (p >= sc.end) return;
    uint32_t k, src;
    if (layoutPrev) {
        const uint32_t prev = d.perm2[p];
        if (prev >= d.nslots) return;  // consistent sorts never produce these
        const uint2 r = d.layPhys[prev];
        k = r.x;
        src = r.y;
    } else {
        k = d.perm2[p];
        if (k >= d.nslots) return;
        src = d.srcL[k];
    }
    if (k >= d.nslots || src >= d.nslots) return;
    float4 x = d.X[src], v = d.V[src];
    f3 xs = predict_x(make3(x), make3(v), S);
    const float4 xs4 = make_float4(xs.x, xs.y, xs.z, x.w);
    d.X0[p] = x;
    d.XsA[p] = xs4;
    if (kCarry) {
        d.Tdens[p] = d.dens[src];
        d.Tlam[p] = d.lam[src];
    }
    if (kCarryDelta) d.TDP[p] = d.DP[src];
    d.Tid[p] = d.id[src];
    d.lidT[p] = k;
    d.physT[k] = p;
}

// Inclusive prefix sum over the wave's 64 lanes.
__device__ __forceinline__ uint32_t wave_prefix(uint32_t v) {
    int x = (int)v;
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false);  // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false);  // row_shr:2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false);  // row_shr:4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false);  // row_shr:8
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false);  // row_bcast:15 into rows 1 and 3
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false);  // row_bcast:31 into rows 2 and 3
    return (uint32_t)x;
}

// The largest value of this lane and those below it.
__device__ __forceinline__ uint32_t wave_prefix_max(uint32_t v) {
    int x = (int)v;
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false));  // row_shr:1
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false));  // row_shr:2
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false));  // row_shr:4
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false));  // row_shr:8
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false));  // row_bcast:15 into rows 1 and 3
    x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false));  // row_bcast:31 into rows 2 and 3
    return (uint32_t)x;
}

// LDS written by some lanes of a wave and read by others: LDS instructions of one wave complete in
// issue order, so only the compiler has to be kept from moving accesses across this point.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ uint32_t lanes_below(uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// ---- small scenes: both orders from one counting pass ----------------------------------------------
// Up to kOrderMaxSlots slots of a single scene take three launches where the two radix sorts, the cell
// table and the move take thirteen, each at the launch's own cost (27,000 particles: 85 us of a 235 us
// step before, 14 now; 1,000: 57 and 13).  The physical order is the logical order: the particles of a
// cell are still neighbours in memory, and the arrays of such a scene fit the caches.  Larger scenes gain
// more from the cell order than its two further launches cost (launch_tally; us per step so / there: 16,000
// particles 87 / 90, 27,000 106 / 108, 32,000 sprayed 126 / 119, 40,000 134 / 124, 130,000 260 / 232).
//   1. k_order_count: hashes; each particle takes a place in the group of its hash's upper bits;
//   2. k_order_place: the groups' prefix (each workgroup its own, in LDS), hashes to their groups;
//   3. k_order_rank: each particle's rank by (hash, previous logical index) among its group's few
//      members, which also gives its bucket's bounds: the move and the table entry.
constexpr uint32_t kOrderBlock = 1024;

// Groups are counted by runs: particles of one cell mostly lie side by side.  The last block gathers what
// the import found in the masses (gather_masses).
__global__ __launch_bounds__(kBlock) void k_order_count(DeviceState d, SphParams P, StepParams S, uint32_t countBlocks) {
    if (blockIdx.x == gridDim.x - 1u) {
        gather_masses(d, P);
        return;
    }
    if (blockIdx.x >= countBlocks) {
        const uint32_t i = (blockIdx.x - countBlocks) * kBlock + threadIdx.x;
        if (i < d.tableTotal) d.table[i] = make_uint4(kEmptyKey, kEmptyKey, kEmptyKey, kEmptyKey);
        return;
    }
    const uint32_t p = blockIdx.x * kBlock + threadIdx.x;
    const SceneDev& sc = d.scenes[0];
    const bool valid = p < d.nslots;
    uint32_t h = 0, k = 0, group = kEmptyKey;
    if (valid) {
        k = d.lid[p];
        const f3 xs = predict_x(make3(d.X[p]), make3(d.V[p]), S);
        int cx, cy, cz;
        discretize(xs, P.cellHash, cx, cy, cz);
        h = cell_hash(cx, cy, cz, sc);
        group = h >> d.groupShift;
    }
    const uint32_t lane = __lane_id();
    const uint32_t before = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)group, 0x138, 0xF, 0xF, false);  // wave_shr:1
    const uint64_t heads = __ballot(lane == 0u || before != group);
    const uint32_t head = 63u - (uint32_t)__builtin_clzll(heads & (~0ull >> (63u - lane)));
    uint32_t place = 0;
    if (valid && lane == head) {
        const uint64_t after = lane == 63u ? 0ull : heads & (~0ull << (lane + 1u));
        const uint32_t end = after ? (uint32_t)__builtin_ctzll(after) : 64u;
        place = atomicAdd(&d.groupCount[group], end - lane);  // the lanes past the last slot are a run of their own
    }
    place = (uint32_t)__shfl((int)place, (int)head, 64) + (lane - head);
    if (!valid || k >= d.nslots) return;  // a consistent order never produces k >= nslots
    d.keysL[k] = h;
    d.layPhys[k] = make_uint2(place, p);
}

__global__ __launch_bounds__(kOrderBlock) void k_order_place(DeviceState d) {
    __shared__ uint32_t base[kOrderMaxGroups];
    __shared__ uint32_t waveSum[kOrderBlock / 64];
    const uint32_t t = threadIdx.x;
    const uint32_t k = blockIdx.x * kOrderBlock + t;
    uint32_t h = 0;
    uint2 r = make_uint2(0u, 0u);
    if (k < d.nslots) {
        h = d.keysL[k];
        r = d.layPhys[k];
    }
    // eight consecutive counts per thread (groups is a multiple of 8, the rest of the array is zero)
    constexpr uint32_t kPer = kOrderMaxGroups / kOrderBlock;
    static_assert(kPer == 8, "two chunks of four");
    uint32_t c[kPer] = {};
    if (t * kPer < d.groups) {
        const uint4* const g = reinterpret_cast<const uint4*>(d.groupCount) + 2u * t;
        const uint4 a = g[0], b = g[1];
        c[0] = a.x; c[1] = a.y; c[2] = a.z; c[3] = a.w;
        c[4] = b.x; c[5] = b.y; c[6] = b.z; c[7] = b.w;
    }
    uint32_t sum = 0;
#pragma unroll
    for (uint32_t u = 0; u < kPer; ++u) sum += c[u];
    const uint32_t inclusive = wave_prefix(sum);
    if (__lane_id() == 63u) waveSum[t >> 6] = inclusive;
    __syncthreads();
    uint32_t run = inclusive - sum;
    for (uint32_t w = 0; w < (t >> 6); ++w) run += waveSum[w];
#pragma unroll
    for (uint32_t u = 0; u < kPer; ++u) {
        base[t * kPer + u] = run;
        run += c[u];
    }
    __syncthreads();
    if (blockIdx.x == 0) {
        for (uint32_t g = t; g < d.groups; g += kOrderBlock) d.groupBase[g] = base[g];
        if (t == 0) d.groupBase[d.groups] = d.nslots;
    }
    if (k >= d.nslots) return;
    const uint32_t q = base[(h >> d.groupShift) & (kOrderMaxGroups - 1u)] + r.x;
    if (q < d.nslots) d.placed[q] = make_uint4(h, k, r.y, 0u);
}

// ---- crowded groups of the orderings by counting -----------------------------------------------------
// k_order_rank and k_tally_rank rank a particle by going through its group, a handful of members where the
// particles spread over the cells.  In a group of more than kCrowd (thousands in one cell, or coincident, or
// not finite, which all hash to one cell) that would be quadratic; such a group is sorted instead, by one of
// the workgroups that the rank launch has in front for this: by digits of eight bits, stable, its 16-byte
// records going to and fro between placed and tallied, which is free then.  Passes in which all digits are
// equal fall away, so a group that is one crowded cell takes the two or three of the index.
// Measured: 1M with clumps of up to 4,800 in a cell, rank launch 474 us unsorted, and with groups sorted from
// 128 / 256 / 512 / 1,024 members on 286 / 208 / 208 / 216; 100,000 particles at one point 7.5 -> 0.44 ms a step
// (0.49 by radix sorts), a million, one workgroup's work, 20 ms (2.2 by radix sorts).  Scenes without crowds: 1M
// 110.5 us both ways, 27,000 particles 7.4 -> 7.7.
constexpr uint32_t kCrowd = 512;
constexpr uint32_t kCrowdPer = 4;  // records of a thread between the barriers of a pass
constexpr uint32_t kMaxCrowdBlocks = 256;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct CrowdLds {
    uint32_t first[kBlock];              // next place of each digit
    uint32_t wave[kBlock / 64][kBlock];  // digits of a tile by wave
    uint32_t sums[kBlock / 64];
    uint32_t crowds[kBlock], ncrowds;    // crowded groups of 256
};
// One for all the rank kernels: one in each would take its room in all of them.
__device__ __forceinline__ CrowdLds& crowd_lds() {
    __shared__ CrowdLds lds;
    return lds;
}

__device__ __forceinline__ uint32_t bits_below(uint32_t n) { return n > 1u ? 32u - (uint32_t)__builtin_clz(n - 1u) : 0u; }

// Sorts a[0, m) by the low bits of field kField, to and fro with b; a is where the records end up.  Every thread of
// the workgroup, with the same arguments.
template <char kField>
__device__ __forceinline__ void crowd_sort(u32x4*& a, u32x4*& b, uint32_t m, uint32_t bits, CrowdLds& L) {
    const auto key = [](u32x4 r) { return kField == 'x' ? r.x : kField == 'y' ? r.y : r.w; };
    static_assert(kBlock == 256, "a thread per digit");
    const uint32_t t = threadIdx.x, lane = __lane_id(), wave = t >> 6;
    for (uint32_t shift = 0; shift < bits; shift += 8u) {
        L.first[t] = 0u;
#pragma unroll
        for (uint32_t w = 0; w < kBlock / 64; ++w) L.wave[w][t] = 0u;
        __syncthreads();
        for (uint32_t i0 = 0; i0 < m; i0 += kBlock * 8u) {  // eight loads in flight
            uint32_t k[8];
#pragma unroll
            for (uint32_t u = 0; u < 8u; ++u) k[u] = key(a[min(i0 + u * kBlock + t, m - 1u)]);
#pragma unroll
            for (uint32_t u = 0; u < 8u; ++u)
                if (i0 + u * kBlock + t < m) atomicAdd(&L.first[(k[u] >> shift) & 255u], 1u);
        }
        __syncthreads();
        const uint32_t count = L.first[t];
        if (__syncthreads_or(count == m)) continue;  // one digit
        const uint32_t inclusive = wave_prefix(count);
        if (lane == 63u) L.sums[wave] = inclusive;
        __syncthreads();
        uint32_t before = inclusive - count;
        for (uint32_t w = 0; w < wave; ++w) before += L.sums[w];
        L.first[t] = before;
        __syncthreads();
        for (uint32_t t0 = 0; t0 < m; t0 += kBlock * kCrowdPer) {
            u32x4 r[kCrowdPer];
            uint32_t rank[kCrowdPer];
            const uint32_t mine = t0 + wave * (64u * kCrowdPer) + lane;
#pragma unroll
            for (uint32_t u = 0; u < kCrowdPer; ++u) r[u] = a[min(mine + 64u * u, m - 1u)];
#pragma unroll
            for (uint32_t u = 0; u < kCrowdPer; ++u) {
                const bool in = mine + 64u * u < m;
                const uint32_t digit = (key(r[u]) >> shift) & 255u;
                uint64_t peers = __ballot(in);
#pragma unroll
                for (uint32_t k = 0; k < 8u; ++k) {
                    const bool one = ((digit >> k) & 1u) != 0u;
                    const uint64_t ones = __ballot(one);
                    peers &= one ? ones : ~ones;
                }
                const uint32_t below = lanes_below(peers), prior = L.wave[wave][digit];
                wave_lds_order();
                if (in && below == 0u) L.wave[wave][digit] = prior + (uint32_t)__builtin_popcountll(peers);
                wave_lds_order();
                rank[u] = prior + below;
            }
            __syncthreads();
#pragma unroll
            for (uint32_t u = 0; u < kCrowdPer; ++u) {
                const uint32_t digit = (key(r[u]) >> shift) & 255u;
                uint32_t at = L.first[digit] + rank[u];
                for (uint32_t w = 0; w < wave; ++w) at += L.wave[w][digit];
                if (mine + 64u * u < m && at < m) b[at] = r[u];
            }
            __syncthreads();
            uint32_t sum = 0;
#pragma unroll
            for (uint32_t w = 0; w < kBlock / 64; ++w) {
                sum += L.wave[w][t];
                L.wave[w][t] = 0u;
            }
            L.first[t] += sum;
            __syncthreads();
        }
        u32x4* const x = a;
        a = b;
        b = x;
    }
}

// The move of a particle from slot src to slot p, logical index to.  kCarry, kCarryDelta: as in k_gather.
template <bool kCarry, bool kCarryDelta>
__device__ __forceinline__ void order_move(const DeviceState& d, const StepParams& S, uint32_t src, uint32_t to,
                                           uint32_t p, float4 x, float4 v, uint32_t id) {
    const f3 xs = predict_x(make3(x), make3(v), S);
    d.physT[to] = p;
    d.X0[p] = x;
    d.XsA[p] = make_float4(xs.x, xs.y, xs.z, x.w);
    if (kCarry) {
        d.Tdens[p] = d.dens[src];
        d.Tlam[p] = d.lam[src];
    }
    if (kCarryDelta) d.TDP[p] = d.DP[src];
    d.Tid[p] = id;
    d.lidT[p] = to;
}

// The group of records [b, e): orders, table entries and moves.  kBins: with bins (k_tally_rank); else the
// physical order is the logical order.  Records keep their hash in x throughout: the rank launch's other
// threads read it to see that their group is not theirs.
template <bool kCarry, bool kCarryDelta, bool kBins>
__device__ __forceinline__ void crowd_place(const DeviceState& d, const StepParams& S, uint32_t b, uint32_t e, CrowdLds& L) {
    const SceneDev& sc = d.scenes[0];
    const uint32_t t = threadIdx.x, lane = __lane_id(), wave = t >> 6, m = e - b;
    u32x4 *a = reinterpret_cast<u32x4*>(d.placed + b), *o = reinterpret_cast<u32x4*>(d.tallied + b);
    crowd_sort<'y'>(a, o, m, bits_below(d.nslots), L);
    crowd_sort<'x'>(a, o, m, kBins ? sc.groupShift : d.groupShift, L);
    // logical order: (hash, logical index and in the top bit whether the hash begins there, slot, bin)
    for (uint32_t i = t; i < m; i += kBlock) {
        const u32x4 r = a[i];
        const bool head = i == 0u || a[i - 1u].x != r.x;
        d.skeysOut[b + i] = r.x;
        d.perm1Out[b + i] = r.y;
        o[i] = u32x4{r.x, (b + i) | (head ? 0x80000000u : 0u), r.z, r.w};
    }
    __syncthreads();
    u32x4* const ordered = o;
    o = a;
    a = ordered;
    if (kBins) crowd_sort<'w'>(a, o, m, bits_below(d.tallyCount), L);
    uint32_t carry = 0;  // where the bin begins that the records before are in
    for (uint32_t t0 = 0; t0 < m; t0 += kBlock) {
        const uint32_t i = t0 + t;
        const u32x4 r = a[min(i, m - 1u)];
        const uint32_t h = r.x, to = r.y & 0x7FFFFFFFu, src = r.z, bin = r.w;
        uint32_t p = to;
        if (kBins) {
            const uint32_t begins = wave_prefix_max(i < m && i != 0u && a[i - 1u].w != bin ? i : 0u);
            if (lane == 63u) L.sums[wave] = begins;
            __syncthreads();
            uint32_t begin = max(carry, begins);
            for (uint32_t w = 0; w < kBlock / 64; ++w) {
                if (w < wave) begin = max(begin, L.sums[w]);
                carry = max(carry, L.sums[w]);
            }
            __syncthreads();
            if (d.tallyGroups + bin >= d.tallyCount) continue;  // consistent counts never produce this
            p = d.tallyBase[d.tallyGroups + bin] - d.nslots + (i - begin);
        }
        if (i >= m || src >= d.nslots || to >= sc.end || p >= sc.end) continue;
        if ((r.y >> 31) != 0u) {
            uint32_t last = to + 1u, end = e;  // the hash's end: the first place of another
            while (last < end) {
                const uint32_t mid = (last + end) >> 1;
                if (d.skeysOut[mid] == h) last = mid + 1u;
                else end = mid;
            }
            const uint32_t same = last - to;
            bool together = same <= 256u;  // as in k_bucket_phys
            if (kBins && together) {  // in one bin: its last member stands same - 1 records on
                together = same <= m - i;
                const u32x4 z = a[together ? i + same - 1u : i];
                together = together && z.w == bin && (z.y & 0x7FFFFFFFu) == to + same - 1u;
            }
            const uint32_t slot = table_insert(d.table, sc, h);
            if (slot != kEmptyKey) {
                d.table[slot].y = to;
                d.table[slot].z = to + same;
                d.table[slot].w = p | (together ? 0x80000000u : 0u);
            }
        }
        order_move<kCarry, kCarryDelta>(d, S, src, to, p, d.X[src], d.V[src], d.id[src]);
    }
    __syncthreads();
}

// The crowded ones of the groups, which begin at base[0, groups], by workgroup blockIdx.x of crowdBlocks.
template <bool kCarry, bool kCarryDelta, bool kBins>
__device__ __forceinline__ void crowd_groups(const DeviceState& d, const StepParams& S, const uint32_t* __restrict__ base,
                                             uint32_t groups, uint32_t end, uint32_t crowdBlocks, CrowdLds& L) {
    for (uint32_t g0 = blockIdx.x * kBlock; g0 < groups; g0 += crowdBlocks * kBlock) {
        const uint32_t g = g0 + threadIdx.x;
        const bool crowd = g < groups && min(base[g + 1u], end) - base[g] > kCrowd;
        if (!__syncthreads_or(crowd)) continue;
        if (threadIdx.x == 0) L.ncrowds = 0u;
        __syncthreads();
        if (crowd) L.crowds[atomicAdd(&L.ncrowds, 1u)] = g;
        __syncthreads();
        for (uint32_t k = 0; k < L.ncrowds; ++k) {
            const uint32_t c = L.crowds[k];
            crowd_place<kCarry, kCarryDelta, kBins>(d, S, base[c], min(base[c + 1u], end), L);
        }
        __syncthreads();
    }
}

// kCarry, kCarryDelta: as in k_gather.  The first crowdBlocks workgroups take the crowded groups.
template <bool kCarry, bool kCarryDelta>
__global__ __launch_bounds__(kBlock) void k_order_rank(DeviceState d, StepParams S, uint32_t crowdBlocks) {
    if (blockIdx.x < crowdBlocks) {
        crowd_groups<kCarry, kCarryDelta, false>(d, S, d.groupBase, d.groups, d.nslots, crowdBlocks, crowd_lds());
        return;
    }
    const uint32_t q = (blockIdx.x - crowdBlocks) * kBlock + threadIdx.x;
    // the counts were read by the launch before: empty for the next step
    for (uint32_t g = q; g < d.groups; g += (gridDim.x - crowdBlocks) * kBlock) d.groupCount[g] = 0u;
    if (q >= d.nslots) return;
    const SceneDev& sc = d.scenes[0];
    const uint4 me = d.placed[q];
    const uint32_t h = me.x, k = me.y, src = me.z, group = h >> d.groupShift;
    if (k >= d.nslots || src >= d.nslots || group >= d.groups) return;  // consistent counts never produce these
    const float4 x = d.X[src], v = d.V[src];
    const uint32_t id = d.id[src];
    const uint32_t b = d.groupBase[group], e = min(d.groupBase[group + 1u], d.nslots);
    if (e - b > kCrowd) return;
    uint32_t smaller = 0, same = 0, sameBefore = 0;
    constexpr uint32_t kBatch = 8;
    for (uint32_t m0 = b; m0 < e; m0 += kBatch) {
        uint2 o[kBatch];
#pragma unroll
        for (uint32_t u = 0; u < kBatch; ++u) o[u] = *reinterpret_cast<const uint2*>(&d.placed[min(m0 + u, e - 1u)]);
#pragma unroll
        for (uint32_t u = 0; u < kBatch; ++u) {
            const bool in = m0 + u < e;
            smaller += in && o[u].x < h ? 1u : 0u;
            same += in && o[u].x == h ? 1u : 0u;
            sameBefore += in && o[u].x == h && o[u].y < k ? 1u : 0u;
        }
    }
    const uint32_t first = b + smaller, to = first + sameBefore;
    if (to >= d.nslots) return;  // consistent counts never produce this
    if (sameBefore == 0u) {
        const uint32_t slot = table_insert(d.table, sc, h);
        if (slot != kEmptyKey) {
            d.table[slot].y = first;
            d.table[slot].z = first + same;
            // physical order is logical order: the bucket is one run (256 particles at most, as in k_bucket_phys)
            d.table[slot].w = first | (same <= 256u ? 0x80000000u : 0u);
        }
    }
    d.skeysOut[to] = h;
    d.perm1Out[to] = k;
    order_move<kCarry, kCarryDelta>(d, S, src, to, to, x, v, id);
}

// ---- larger scenes: both orders by counting, in five launches ----------------------------------------
// The same idea where the cell order in memory is worth having: besides its group of hashes a particle is
// counted in the bin of its cell, one prefix over groups and bins together gives the first place of each,
// and the rank among its group's members also gives its place in the bin (a cell has one hash, so all its
// particles are in one group).  Bins are the cells of the box and a few beyond, in cubes of 2^cubeLog2
// cells with the Morton order inside; cells farther out share one bin per group.
// Against the two radix sorts in shared launches, the cell table and the move (kernel time at 1M): 180 ->
// 112 us in a settled flow, 266 -> 237 sprayed, where particles of a cell seldom lie side by side and the
// counting (22 -> 92 us) and ranking (65 -> 110) slow down.

// Bin of a cell; outside the range the group's.  The groups' bins lie behind blocks of
// cells' bins, 2^binSpare to each: particles far out list slowly and sweep fast, so they are spread over
// the scene (behind all cells they are one XCD's: list build of 8M sprayed particles 2.35 -> 3.32 ms).
__device__ __forceinline__ uint32_t cell_bin(int cx, int cy, int cz, uint32_t group, const SceneDev& sc) {
    const uint32_t u = (uint32_t)cx - (uint32_t)sc.binOrigin[0], v = (uint32_t)cy - (uint32_t)sc.binOrigin[1],
                   w = (uint32_t)cz - (uint32_t)sc.binOrigin[2];
    if (u >= sc.binCells[0] || v >= sc.binCells[1] || w >= sc.binCells[2])
        return (((group >> sc.binSpare) + 1u) << sc.binBlock) + group;
    const uint32_t c = sc.cubeLog2, low = (1u << c) - 1u;
    const uint32_t cube = (u >> c) * sc.cubeStride[0] + (v >> c) * sc.cubeStride[1] + (w >> c) * sc.cubeStride[2];
    const uint32_t b = (cube << (3u * c)) | spread3(u & low) | (spread3(v & low) << 1) | (spread3(w & low) << 2);
    return b + ((b >> sc.binBlock) << sc.binSpare);
}

__global__ __launch_bounds__(kBlock) void k_tally_count(DeviceState d, SphParams P, StepParams S, uint32_t countBlocks) {
    if (blockIdx.x == gridDim.x - 1u) {
        gather_masses(d, P);
        return;
    }
    if (blockIdx.x >= countBlocks) {
        const uint32_t i = (blockIdx.x - countBlocks) * kBlock + threadIdx.x;
        if (i < d.tableTotal) d.table[i] = make_uint4(kEmptyKey, kEmptyKey, kEmptyKey, kEmptyKey);
        return;
    }
    const uint32_t p = blockIdx.x * kBlock + threadIdx.x;
    const SceneDev& sc = d.scenes[0];
    const bool valid = p < d.nslots;
    uint32_t h = 0, k = 0, group = 0, bin = kEmptyKey;
    if (valid) {
        k = d.lid[p];
        const f3 xs = predict_x(make3(d.X[p]), make3(d.V[p]), S);
        int cx, cy, cz;
        discretize(xs, P.cellHash, cx, cy, cz);
        h = cell_hash(cx, cy, cz, sc);
        group = h >> sc.groupShift;
        bin = cell_bin(cx, cy, cz, group, sc);
    }
    // by runs of one bin and group (particles of a cell mostly lie side by side)
    const uint32_t lane = __lane_id();
    const uint32_t bin1 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)bin, 0x138, 0xF, 0xF, false);  // wave_shr:1
    const uint64_t heads = __ballot(lane == 0u || bin1 != bin);
    const uint32_t head = 63u - (uint32_t)__builtin_clzll(heads & (~0ull >> (63u - lane)));
    uint32_t place = 0;
    if (valid && lane == head) {
        const uint64_t after = lane == 63u ? 0ull : heads & (~0ull << (lane + 1u));
        const uint32_t length = (after ? (uint32_t)__builtin_ctzll(after) : 64u) - lane;
        place = atomicAdd(&d.tally[group], length);
        atomicAdd(&d.tally[d.tallyGroups + bin], length);
    }
    place = (uint32_t)__shfl((int)place, (int)head, 64) + (lane - head);
    if (valid) d.tallied[p] = make_uint4(h, k, place, bin);
}

// The prefix, kTallyBlock counters per workgroup, eight per thread: each workgroup's sum, then its prefix
// behind the sums before it.  The counters are read for the last time there and are left empty.
constexpr uint32_t kTallyThreads = kTallyBlock / 8u;

__device__ __forceinline__ uint32_t block_sum(uint32_t v, uint32_t* waves) {
    const uint32_t inclusive = wave_prefix(v);
    if (__lane_id() == 63u) waves[threadIdx.x >> 6] = inclusive;
    __syncthreads();
    uint32_t sum = 0;
    for (uint32_t w = 0; w < kTallyThreads / 64u; ++w) sum += waves[w];
    __syncthreads();
    return sum;
}

__global__ __launch_bounds__(kTallyThreads) void k_tally_sum(DeviceState d) {
    __shared__ uint32_t waves[kTallyThreads / 64u];
    const uint4* const c = reinterpret_cast<const uint4*>(d.tally) + (size_t)blockIdx.x * (kTallyBlock / 4u) + 2u * threadIdx.x;
    const uint4 a = c[0], b = c[1];
    const uint32_t sum = block_sum(((a.x + a.y) + (a.z + a.w)) + ((b.x + b.y) + (b.z + b.w)), waves);
    if (threadIdx.x == 0) d.tallyPart[blockIdx.x] = sum;
}

__global__ __launch_bounds__(kTallyThreads) void k_tally_prefix(DeviceState d) {
    __shared__ uint32_t waves[kTallyThreads / 64u];
    uint4* const c = reinterpret_cast<uint4*>(d.tally) + (size_t)blockIdx.x * (kTallyBlock / 4u) + 2u * threadIdx.x;
    const uint4 a = c[0], b = c[1];
    uint32_t before = 0;
    for (uint32_t k = threadIdx.x; k < blockIdx.x; k += kTallyThreads) before += d.tallyPart[k];
    before = block_sum(before, waves);
    const uint32_t sum = ((a.x + a.y) + (a.z + a.w)) + ((b.x + b.y) + (b.z + b.w));
    const uint32_t inclusive = wave_prefix(sum);
    if (__lane_id() == 63u) waves[threadIdx.x >> 6] = inclusive;
    __syncthreads();
    uint32_t run = before + inclusive - sum;
    for (uint32_t w = 0; w < (threadIdx.x >> 6); ++w) run += waves[w];
    uint4 x, y;
    x.x = run;       x.y = x.x + a.x; x.z = x.y + a.y; x.w = x.z + a.z;
    y.x = x.w + a.w; y.y = y.x + b.x; y.z = y.y + b.y; y.w = y.z + b.z;
    uint4* const out = reinterpret_cast<uint4*>(d.tallyBase) + (size_t)blockIdx.x * (kTallyBlock / 4u) + 2u * threadIdx.x;
    out[0] = x;
    out[1] = y;
    c[0] = c[1] = make_uint4(0u, 0u, 0u, 0u);
}

__global__ __launch_bounds__(kBlock) void k_tally_place(DeviceState d) {
    const uint32_t p = blockIdx.x * kBlock + threadIdx.x;
    if (p >= d.nslots) return;
    const uint4 r = d.tallied[p];
    const uint32_t q = d.tallyBase[r.x >> d.scenes[0].groupShift] + r.z;
    if (q < d.nslots) d.placed[q] = make_uint4(r.x, r.y, p, r.w);
}

// kCarry, kCarryDelta: as in k_gather.  The first crowdBlocks workgroups take the crowded groups.
template <bool kCarry, bool kCarryDelta>
__global__ __launch_bounds__(kBlock) void k_tally_rank(DeviceState d, StepParams S, uint32_t crowdBlocks) {
    if (blockIdx.x < crowdBlocks) {
        crowd_groups<kCarry, kCarryDelta, true>(d, S, d.tallyBase, d.tallyGroups, d.nslots, crowdBlocks, crowd_lds());
        return;
    }
    const uint32_t q = (blockIdx.x - crowdBlocks) * kBlock + threadIdx.x;
    if (q >= d.nslots) return;
    const uint4 me = d.placed[q];
    const uint32_t h = me.x, k = me.y, src = me.z, bin = me.w;
    if (src >= d.nslots) return;  // consistent counts never produce this
    const SceneDev& sc = d.scenes[0];
    const uint32_t group = h >> sc.groupShift;
    if (group >= d.tallyGroups || d.tallyGroups + bin >= d.tallyCount) return;  // nor this
    const float4 x = d.X[src], v = d.V[src];
    const uint32_t id = d.id[src];
    const uint32_t b = d.tallyBase[group], e = min(d.tallyBase[group + 1u], d.nslots);
    if (e - b > kCrowd) return;
    const uint32_t binFirst = d.tallyBase[d.tallyGroups + bin] - d.nslots;
    // among the group: smaller hashes, the bucket, those of it before this particle, those of it in the same
    // bin, and those in the same bin before this particle by hash and index
    uint32_t smaller = 0, same = 0, sameBefore = 0, sameBin = 0, binBefore = 0;
    constexpr uint32_t kBatch = 4;
    for (uint32_t m0 = b; m0 < e; m0 += kBatch) {
        uint4 o[kBatch];
#pragma unroll
        for (uint32_t u = 0; u < kBatch; ++u) o[u] = d.placed[min(m0 + u, e - 1u)];
#pragma unroll
        for (uint32_t u = 0; u < kBatch; ++u) {
            const bool in = m0 + u < e, less = in && o[u].x < h, equal = in && o[u].x == h, mine = o[u].w == bin;
            const bool before = equal && o[u].y < k;
            smaller += less ? 1u : 0u;
            same += equal ? 1u : 0u;
            sameBefore += before ? 1u : 0u;
            sameBin += equal && mine ? 1u : 0u;
            binBefore += (less || before) && mine ? 1u : 0u;
        }
    }
    const uint32_t first = b + smaller, to = first + sameBefore, p = binFirst + binBefore;
    if (to >= sc.end || p >= sc.end) return;  // consistent counts never produce this
    if (sameBefore == 0u) {
        const uint32_t slot = table_insert(d.table, sc, h);
        if (slot != kEmptyKey) {
            d.table[slot].y = first;
            d.table[slot].z = first + same;
            // one bin: the bucket's particles lie side by side in logical order (256 at most, as in k_bucket_phys)
            d.table[slot].w = p | (sameBin == same && same <= 256u ? 0x80000000u : 0u);
        }
    }
    d.skeysOut[to] = h;
    d.perm1Out[to] = k;
    order_move<kCarry, kCarryDelta>(d, S, src, to, p, x, v, id);
}

// Per bucket: where it starts in physical order and whether its particles occupy consecutive
// physical slots in logical order (always true for a bucket of one cell, which lies inside one
// super-cell; buckets of more than 256 particles are not marked).  One thread per logical index k,
// all reads in logical order: the bucket's first index ANDs (first physical slot | run bit) into
// the record's w, which the table fill left all ones, and every index whose logical successor in
// the bucket is not in the next physical slot clears the run bit (ANDs commute, so the order of
// the two does not matter).  Only hash-collision buckets take that second path.
__device__ __forceinline__ uint32_t table_slot_of(const uint4* __restrict__ table, const SceneDev& sc,
                                                  uint32_t h) {
    const uint32_t mask = (1u << sc.tabLog2) - 1u;
    uint32_t s = table_slot(h, sc.tabLog2);
    for (uint32_t probe = 0; probe <= mask; ++probe) {
        const uint32_t key = table[sc.tabOffset + s].x;
        if (key == h) return sc.tabOffset + s;
        if (key == kEmptyKey) return kEmptyKey;
        s = (s + 1u) & mask;
    }
    return kEmptyKey;
}

__global__ __launch_bounds__(kBlock) void k_bucket_phys(DeviceState d) {
    const uint32_t k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= d.nslots) return;
    const SceneDev& sc = scene_of(d, k);
    if (k >= sc.end) return;
    const uint32_t h = d.skeys[k];
    const uint32_t p = d.physT[k];
    if (k == sc.begin || d.skeys[k - 1] != h) {
        const uint32_t slot = d.bslot[k];
        if (slot < d.tableTotal) {
            // at most 256 indices: the one 256 ahead is past the scene or in another bucket (the
            // sorted hashes, read nearby, instead of the record's end through the table)
            const bool small = k + 256u >= sc.end || d.skeys[k + 256u] != h;
            atomicAnd(&d.table[slot].w, p | (small ? 0x80000000u : 0u));
        }
    }
    if (k + 1u < sc.end && d.skeys[k + 1u] == h && d.physT[k + 1u] != p + 1u) {
        const uint32_t slot = table_slot_of(d.table, sc, h);
        if (slot != kEmptyKey) atomicAnd(&d.table[slot].w, 0x7FFFFFFFu);
    }
}

// A bucket's entry (first logical index, one past the last, first physical slot, contiguity)
// from its table record, with its ranges clamped to the scene (a consistent table never needs
// it, but no entry can then index outside the scene).
__device__ __forceinline__ uint4 clamp_entry(uint4 r, const SceneDev& sc) {
    uint4 e = make_uint4(r.y, r.z, r.w & 0x7FFFFFFFu, r.w >> 31);
    e.x = max(e.x, sc.begin);
    e.y = min(e.y, sc.end);
    if (e.y < e.x) e.y = e.x;
    if (e.w && (e.z < sc.begin || e.z + (e.y - e.x) > sc.end)) e.w = 0u;
    return e;
}

__device__ __forceinline__ bool table_find(const uint4* __restrict__ table, const SceneDev& sc,
                                           uint32_t h, uint4& entry) {
    const uint32_t mask = (1u << sc.tabLog2) - 1u;
    uint32_t s = table_slot(h, sc.tabLog2);
    for (uint32_t probe = 0; probe <= mask; ++probe) {
        const uint4 r = table[sc.tabOffset + s];
        if (r.x == h) {
            entry = clamp_entry(r, sc);
            return true;
        }
        if (r.x == kEmptyKey) return false;
        s = (s + 1u) & mask;
    }
    return false;
}

// kernel_find_neighbours (NeighbourSearchCUDA.cu:72-130), one thread per particle: for lists too long
// for k_neighbours_wave's rows.  Stencil cells in (dx, dy, dz) order, each bucket walked in logical
// order, self skipped, r^2 < h^2 kept, at most maxNeighbours.  A bucket reached from two stencil cells with equal hashes is walked twice, as in the reference.
// The list stores physical slots.
//
// The walk is latency-bound, so memory requests are issued in batches: the nine table probes of
// one dx slab together, then each bucket's candidates eight at a time (position and physical
// slot), after which the candidates are tested and appended strictly in order.
constexpr int kWalkBatch = 8;
constexpr int kProbeGroup = 3;

// Physical slots of bucket positions m0 .. m0 + N - 1 (clamped to the bucket's last, b - 1): by
// the bucket's offset when its slots are consecutive (run), else from physT.  The physT loads sit
// on a branch of their own, so the walks' position loads stay one batch of independent requests.
template <int N>
__device__ __forceinline__ void batch_slots(const DeviceState& d, bool run, uint32_t m0, uint32_t b,
                                            int32_t shift, uint32_t (&ph)[N]) {
    if (__builtin_expect(run, 1)) {
#pragma unroll
        for (int u = 0; u < N; ++u) ph[u] = (uint32_t)((int32_t)min(m0 + u, b - 1u) + shift);
    } else {
#pragma unroll
        for (int u = 0; u < N; ++u) ph[u] = ld(d.physT, min(m0 + u, b - 1u));
    }
}

__global__ __launch_bounds__(kBlock) void k_neighbours(DeviceState d, SphParams P) {
    const uint32_t p = xcd_slot<kBlock>();
    uint32_t count = 0;
    if (p < d.nslots) {
        const SceneDev& sc = scene_of(d, p);
        if (p < sc.end) {
            const f3 xi = make3(d.XsA[p]);
            int cx, cy, cz;
            discretize(xi, P.cellSearch, cx, cy, cz);
            // entry k of this list: element k % 4 of chunk k / 4, at byte offset
            // (p % 64) * 16 + (k / 4) * 1024 + (k % 4) * 4 from the wave's list block, whose
            // address is the same in every lane (the wave's 64 slots share p / 64)
            char* const waveOut = reinterpret_cast<char*>(
                d.nbr4 + (size_t)__builtin_amdgcn_readfirstlane(p >> 6) * list_chunks(P.maxN) * 64u);
            const uint32_t laneOff = (p & 63u) * 16u;
            const uint32_t maxN = (uint32_t)P.maxN;
            // stencil cells c = 0..26 in (dx, dy, dz) order, probed kProbeGroup at a time
            for (int g = 0; g < 27 / kProbeGroup && count < maxN; ++g) {
                uint32_t hq[kProbeGroup], sl[kProbeGroup];
                uint4 rq[kProbeGroup], e[kProbeGroup];
#pragma unroll
                for (int q = 0; q < kProbeGroup; ++q) {
                    const int c = g * kProbeGroup + q;
                    hq[q] = cell_hash((int)((uint32_t)cx + (uint32_t)(c / 9 - 1)),
                                      (int)((uint32_t)cy + (uint32_t)((c / 3) % 3 - 1)),
                                      (int)((uint32_t)cz + (uint32_t)(c % 3 - 1)), sc);
                    sl[q] = sc.tabOffset + table_slot(hq[q], sc.tabLog2);
                }
#pragma unroll
                for (int q = 0; q < kProbeGroup; ++q) rq[q] = d.table[sl[q]];
#pragma unroll
                for (int q = 0; q < kProbeGroup; ++q) {
                    e[q] = make_uint4(0u, 0u, 0u, 0u);
                    if (rq[q].x == hq[q]) {
                        e[q] = clamp_entry(rq[q], sc);
                    } else if (rq[q].x != kEmptyKey) {
                        if (!table_find(d.table, sc, hq[q], e[q])) e[q] = make_uint4(0u, 0u, 0u, 0u);
                    }
                }
#pragma unroll
                for (int q = 0; q < kProbeGroup; ++q) {
                    const uint32_t a = e[q].x, b = e[q].y;
                    // bucket of consecutive physical slots: read the cell-ordered positions
                    // directly; otherwise (hash collisions) find each slot through physT first
                    const bool run = e[q].w != 0u;
                    const int32_t shift = (int32_t)e[q].z - (int32_t)a;  // physical - logical
                    for (uint32_t m0 = a; m0 < b && count < maxN; m0 += kWalkBatch) {
                        float4 c[kWalkBatch];
                        uint32_t ph[kWalkBatch];
                        batch_slots<kWalkBatch>(d, run, m0, b, shift, ph);
#pragma unroll
                        for (int u = 0; u < kWalkBatch; ++u) c[u] = ld(d.XsA, ph[u]);
                        // test the whole batch without branches, then append in order
                        uint32_t acc = 0u;
#pragma unroll
                        for (int u = 0; u < kWalkBatch; ++u) {
                            const f3 sep = xi - make3(c[u]);
                            const bool ok = (dot3(sep, sep) < P.h2) & (ph[u] != p) & (m0 + u < b);
                            acc |= (uint32_t)ok << u;
                        }
                        const uint32_t room = maxN - count;
                        while ((uint32_t)__popc(acc) > room) acc &= ~(1u << (31 - __clz(acc)));
                        if (acc) {
                            // append in order: the u-th candidate goes to position count + (the
                            // accepted candidates before it)
#pragma unroll
                            for (int u = 0; u < kWalkBatch; ++u) {
                                if (acc & (1u << u)) {
                                    const uint32_t k = count + (uint32_t)__popc(acc & ((1u << u) - 1u));
                                    *reinterpret_cast<uint32_t*>(waveOut + (laneOff + ((k & ~3u) << 8) +
                                                                            ((k & 3u) << 2))) = ph[u];
                                }
                            }
                            count += (uint32_t)__popc(acc);
                        }
                    }
                }
            }
        }
        d.cnt[p] = count;
    }
}

// The same lists built by whole waves.  A wave owns S consecutive slots.  Neighbouring slots mostly
// lie in the same search cell (the layout is cell ordered), so its particles fall into runs of at most
// eight with one cell each, and kWaveRuns runs are taken at a time:
//   1. their 27 buckets each are probed one per lane, all at once; a prefix over the bucket lengths
//      makes them one stream of candidates, each run's in stencil order (a bucket reached from two
//      cells appears twice);
//   2. the stream passes 64 candidates at a time, one per lane (the next 64 are loaded meanwhile), and
//      each particle of the run (its position in scalar registers) is tested against all 64 at once:
//      the accepted lanes' ranks in the ballot are their positions behind the particle's entries so
//      far, in stream order;
//   3. entries gather in LDS, one row per particle, and leave as whole 16-byte chunks;
//   4. once all lists of a run are full, the stream goes on at the next run's first candidates.
// With one thread per particle a wave walks 27 buckets per lane, for as long as its lane with most
// candidates, and appends under eight masks per batch; here probes and candidate loads are made once
// per run, every lane of a test does work, and lists of uneven length cost no idle lanes.
// Measured against one thread per particle (kernel time): 1M settled column 359 -> 222 us, 1M dam
// break (sprayed: 29 cells per 64 particles) 448 -> 332, 64 scenes of 2.6M 892 -> 637, 27,000
// particles 66 -> 17, 1,000 particles 62 -> 11.  The tests bound it (168 of the 222 us, 14 vector
// instructions per 64 pairs); in sprayed scenes also the probes (129 of the 332 us).
// Candidates find their bucket by rank: bit t of the bitmap says that a bucket begins at t + 1, so the
// set bits below a lane count the non-empty buckets before its own, and those buckets' (slot offset,
// contiguity) sit in LDS in that order.
constexpr uint32_t kWaveRuns = 4;              // runs probed together
constexpr uint32_t kWaveWindow = 2048;         // stream positions per bitmap
constexpr int kWaveBuildBlock = 256;
// Longest lists that are built with eight, or two, rows per wave: 47 KB of LDS a workgroup at 320, so that
// three share a CU's 160 KB, and 63 of the 64 KB that a workgroup can have at 1,792.
constexpr int kWaveBuildMaxN8 = 320, kWaveBuildMaxN2 = 1792;

typedef __attribute__((address_space(3))) uint32_t lds_u32;

// Words of a list row in LDS: a stride of 4 modulo 32 banks, so the chunk reads of the eight rows fall
// on different banks.
__host__ __device__ __forceinline__ uint32_t wave_row_words(int maxN) {
    return (((uint32_t)maxN + 3u) / 4u * 4u + 27u) / 32u * 32u + 4u;
}
// Words per wave: the rows, the bitmap, the buckets' (offset, contiguity) and a spare word per lane.
template <uint32_t kWaveRows>
__host__ __device__ __forceinline__ uint32_t wave_build_words(int maxN) {
    return kWaveRows * wave_row_words(maxN) + kWaveWindow / 32u + (2u * kWaveRuns * 27u + 3u) / 4u * 4u + 64u;
}

__device__ __forceinline__ uint32_t lane_u(uint32_t v, uint32_t lane) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)lane);
}
__device__ __forceinline__ float lane_f(float v, uint32_t lane) {
    return __uint_as_float(lane_u(__float_as_uint(v), lane));
}

// a in the lanes of m, b in the others.  Written out: as an expression it becomes a branch.
__device__ __forceinline__ uint32_t select(uint64_t m, uint32_t a, uint32_t b) {
    uint32_t r;
    asm("v_cndmask_b32 %0, %1, %2, %3" : "=v"(r) : "v"(b), "v"(a), "s"(m));
    return r;
}

// kWaveRows: list rows in LDS, and the longest run.
template <int S, uint32_t kWaveRows>
__global__ __launch_bounds__(kWaveBuildBlock) void k_neighbours_wave(DeviceState d, SphParams P) {
    extern __shared__ uint4 waveLds[];
    constexpr uint32_t kWaves = kWaveBuildBlock / 64;
    const uint32_t lane = __lane_id();
    const uint32_t block = xcd_block(blockIdx.x, gridDim.x, kWaves * (uint32_t)S);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t base = (block * kWaves + wave) * (uint32_t)S;  // the wave's first slot
    if (base >= d.nslots) return;
    const SceneDev& sc = d.scenes[d.chunkScene[base >> 8]];  // S divides 256: one scene per wave
    const float4* __restrict__ const Xs = d.XsA;
    const uint32_t maxN = (uint32_t)P.maxN, rowWords = wave_row_words(P.maxN);
    const float h2 = P.h2;
    uint32_t* const lds = reinterpret_cast<uint32_t*>(waveLds) + wave * wave_build_words<kWaveRows>(P.maxN);
    const uint32_t ldsAt = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_u32*)lds);
    uint32_t* const bitmap = lds + kWaveRows * rowWords;
    uint2* const bucket = reinterpret_cast<uint2*>(bitmap + kWaveWindow / 32u);
    const uint32_t spare = ldsAt + 4u * (wave_build_words<kWaveRows>(P.maxN) - 64u + lane);
    uint4* const lists = d.nbr4 + (size_t)(base >> 6) * list_chunks(P.maxN) * 64u + (base & 63u);

    const uint32_t slot = base + lane;
    const bool mine = lane < (uint32_t)S && slot < d.nslots;
    const bool valid = mine && slot < sc.end;  // a scene's slots are consecutive: the first lanes
    const uint32_t nvalid = (uint32_t)__builtin_popcountll(__ballot(valid));
    f3 xi{0.0f, 0.0f, 0.0f};
    int cx = 0, cy = 0, cz = 0;
    if (valid) {
        xi = make3(Xs[slot]);
        discretize(xi, P.cellSearch, cx, cy, cz);
    }
    // first lanes of the runs: another cell than the lane before, or the ninth, 17th, ... of its cell
    const int px = __builtin_amdgcn_update_dpp(0, cx, 0x138, 0xF, 0xF, false);  // wave_shr:1
    const int py = __builtin_amdgcn_update_dpp(0, cy, 0x138, 0xF, 0xF, false);
    const int pz = __builtin_amdgcn_update_dpp(0, cz, 0x138, 0xF, 0xF, false);
    const uint64_t cells = __ballot(valid && (lane == 0u || px != cx || py != cy || pz != cz));
    const uint64_t upTo = cells & (~0ull >> (63u - lane));
    const uint32_t inCell = upTo ? lane - (63u - (uint32_t)__builtin_clzll(upTo)) : 1u;
    uint64_t heads = __ballot(valid && (inCell & (kWaveRows - 1u)) == 0u);

    uint32_t counts = 0;            // this lane's particle's list length
    uint32_t row0 = 0, rowEnd = 0;  // the rows hold the lists of lanes [row0, rowEnd)
    const auto flush = [&]() {
        wave_lds_order();
        const uint32_t r = lane & (kWaveRows - 1u), c0 = lane / kWaveRows;
        const uint32_t held = (uint32_t)__shfl((int)counts, (int)((row0 + r) & 63u), 64);
        const uint32_t n = row0 + r < rowEnd ? held : 0u;
        for (uint32_t c = c0; __ballot(4u * c < n); c += 64u / kWaveRows)
            if (4u * c < n)
                lists[(size_t)c * 64u + row0 + r] = *reinterpret_cast<const uint4*>(&lds[r * rowWords + 4u * c]);
        wave_lds_order();
        row0 = rowEnd;
    };

    while (heads) {
        // ---- the buckets of the next runs, entry 27 i + cell of run i in lane (entry % 64) ----
        uint64_t h4 = heads;
        uint32_t leader[kWaveRuns];
        uint32_t nruns = 0;
#pragma unroll
        for (uint32_t i = 0; i < kWaveRuns; ++i) {
            leader[i] = h4 ? (uint32_t)__builtin_ctzll(h4) : leader[i ? i - 1u : 0u];
            nruns += h4 ? 1u : 0u;
            h4 &= h4 - 1ull;
        }
        constexpr uint32_t kRounds = (kWaveRuns * 27u + 63u) / 64u;
        uint32_t key[kRounds], at[kRounds], start[kRounds], len[kRounds], incl[kRounds];
#pragma unroll
        for (uint32_t u = 0; u < kRounds; ++u) {
            const uint32_t entry = u * 64u + lane, i = entry / 27u, c = entry - 27u * i;
            uint32_t from = leader[0];
#pragma unroll
            for (uint32_t k = 1; k < kWaveRuns; ++k) from = i == k ? leader[k] : from;
            const uint32_t gx = (uint32_t)__shfl(cx, (int)from, 64), gy = (uint32_t)__shfl(cy, (int)from, 64),
                           gz = (uint32_t)__shfl(cz, (int)from, 64);
            const uint32_t h = cell_hash((int)(gx + (c / 9u - 1u)), (int)(gy + ((c / 3u) % 3u - 1u)),
                                         (int)(gz + (c % 3u - 1u)), sc);
            key[u] = i < nruns ? h : kEmptyKey;  // kEmptyKey: an idle lane
            at[u] = table_slot(h, sc.tabLog2);
        }
        // every lane's first two table slots at once; the rare longer probes one slot at a time
        const uint4* __restrict__ const table = d.table + sc.tabOffset;
        const uint32_t mask = (1u << sc.tabLog2) - 1u;
        uint4 e[kRounds], e1[kRounds];
#pragma unroll
        for (uint32_t u = 0; u < kRounds; ++u) {
            e[u] = table[at[u]];
            e1[u] = table[(at[u] + 1u) & mask];
        }
#pragma unroll
        for (uint32_t u = 0; u < kRounds; ++u) {
            const bool past = e[u].x != key[u] && e[u].x != kEmptyKey;
            if (past) e[u] = e1[u];
            at[u] += past ? 1u : 0u;
            for (uint32_t probe = 0; probe <= mask; ++probe) {
                const bool open = e[u].x != key[u] && e[u].x != kEmptyKey && key[u] != kEmptyKey;
                if (!__ballot(open)) break;
                at[u] += 1u;
                if (open) e[u] = table[at[u] & mask];
            }
            e[u] = key[u] != kEmptyKey && e[u].x == key[u] ? clamp_entry(e[u], sc) : make_uint4(0u, 0u, 0u, 0u);
        }
        uint32_t total = 0, filled = 0;
        bool logical = false;
        wave_lds_order();
#pragma unroll
        for (uint32_t u = 0; u < kRounds; ++u) {
            len[u] = e[u].y - e[u].x;
            incl[u] = total + wave_prefix(len[u]);
            start[u] = incl[u] - len[u];
            total = lane_u(incl[u], 63u);
            const uint64_t f = __ballot(len[u] != 0u);
            // buckets whose slots are not consecutive (hash collisions) are read through physT
            logical |= len[u] != 0u && e[u].w == 0u;
            if (len[u] != 0u)
                bucket[filled + lanes_below(f)] = make_uint2((e[u].w ? e[u].z : e[u].x) - start[u], e[u].w);
            filled += (uint32_t)__builtin_popcountll(f);
        }
        const bool anyLogical = __ballot(logical) != 0ull;
        wave_lds_order();

        // ---- the stream, one candidate per lane: position and slot ----
        uint32_t mark[kRounds];  // of a non-empty bucket but the first: its position - 1
#pragma unroll
        for (uint32_t u = 0; u < kRounds; ++u) mark[u] = len[u] != 0u ? start[u] - 1u : ~0u;
        constexpr uint32_t kSkipped = 0x80000000u;  // in ranked: the next load does not follow the last one
        uint32_t ranked = 0;  // non-empty buckets that begin before the next 64 positions, but for the first
        const auto load = [&](uint32_t t0, uint32_t& ph) {
            if (t0 >= total) return make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (t0 % kWaveWindow == 0u || (ranked & kSkipped) != 0u) {
                ranked &= ~kSkipped;
                wave_lds_order();
                bitmap[lane] = 0u;
                wave_lds_order();
#pragma unroll
                for (uint32_t u = 0; u < kRounds; ++u) {
                    const uint32_t bit = mark[u] - t0 / kWaveWindow * kWaveWindow;
                    if (bit < kWaveWindow) atomicOr(&bitmap[bit >> 5], 1u << (bit & 31u));
                }
                wave_lds_order();
            }
            const uint2 bits = *reinterpret_cast<const uint2*>(&bitmap[(t0 % kWaveWindow) >> 5]);
            const uint64_t begins = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)bits.y) << 32) |
                                    (uint32_t)__builtin_amdgcn_readfirstlane((int)bits.x);
            const uint2 of = bucket[ranked + lanes_below(begins)];
            ranked += (uint32_t)__builtin_popcountll(begins);
            const bool in = t0 + lane < total;
            ph = in ? t0 + lane + of.x : base;
            if (anyLogical) {
                if (in && of.y == 0u) ph = ld(d.physT, ph);
            }
            return ld(Xs, ph);
        };
        uint32_t t0 = 0, ph = base, phNext = base;
        float4 c = load(0u, ph), cNext = load(64u, phNext);
        const auto advance = [&]() {
            t0 += 64u;
            c = cNext;
            ph = phNext;
            cNext = load(t0 + 64u, phNext);
        };

        uint32_t begin = 0;
        for (uint32_t i = 0; i < nruns; ++i) {
            const uint32_t last = 27u * i + 26u;  // the run's last entry
            const uint32_t end = last < 64u ? lane_u(incl[0], last) : lane_u(incl[kRounds - 1u], last - 64u);
            const uint32_t first = (uint32_t)__builtin_ctzll(heads);
            heads &= heads - 1ull;
            const uint32_t np = (heads ? (uint32_t)__builtin_ctzll(heads) : nvalid) - first;
            if (rowEnd - row0 + np > kWaveRows) flush();
            const uint32_t row = ldsAt + 4u * (rowEnd - row0) * rowWords;  // LDS byte address of the run's first row
            rowEnd += np;
            if (begin == end) continue;  // no candidates: empty lists
            while (begin >= t0 + 64u) advance();
            // the run's particles against its stretch of the stream.  Each pass over them leaves at
            // np, compared anew after each particle (after the lists' growth, to the compiler):
            // hoisted out of the loop, the results of the compares take a scalar register pair each
            // and spill.
            const auto done = [&](uint32_t q, uint32_t after) {
                uint32_t n = np;
                asm("" : "+s"(n) : "s"(after));
                return q >= n;
            };
            float qx[kWaveRows], qy[kWaveRows], qz[kWaveRows];
            uint32_t put[kWaveRows];  // LDS byte address of the particle's next entry
#pragma unroll
            for (uint32_t q = 0; q < kWaveRows; ++q) {
                put[q] = row + 4u * q * rowWords;
                qx[q] = qy[q] = qz[q] = 0.0f;
            }
#pragma unroll
            for (uint32_t q = 0; q < kWaveRows; ++q) {
                if (q >= np) break;
                qx[q] = lane_f(xi.x, first + q);
                qy[q] = lane_f(xi.y, first + q);
                qz[q] = lane_f(xi.z, first + q);
            }
            for (;;) {
                const uint32_t t = t0 + lane;
                // other runs' candidates are never within h
                const float cx1 = (t >= begin) & (t < end) ? c.x : __builtin_inff();
                const auto within = [&](uint32_t q) {
                    const f3 sep{qx[q] - cx1, qy[q] - c.y, qz[q] - c.z};
                    return __builtin_amdgcn_ballot_w64(dot3(sep, sep) < h2) &
                           __builtin_amdgcn_ballot_w64(ph != base + first + q);
                };
                uint32_t row0At = row;  // its sums below are made anew: kept across the loop they spill
                asm("" : "+s"(row0At));
                bool room = t0 + 64u - begin <= maxN;  // no list can be longer than the stretch so far
                if (!room) {
                    uint32_t most = 0;
#pragma unroll
                    for (uint32_t q = 0; q < kWaveRows; ++q) {
                        if (q >= np) break;
                        most = max(most, put[q] - (row0At + 4u * q * rowWords));
                    }
                    room = most + 256u <= 4u * maxN;
                    if (most == 4u * maxN) {  // a list is full: perhaps every one
                        uint32_t least = most;
#pragma unroll
                        for (uint32_t q = 0; q < kWaveRows; ++q) {
                            if (q && done(q, least)) break;
                            least = min(least, put[q] - (row0At + 4u * q * rowWords));
                        }
                        if (least == most) {
                            // On at the next run's candidates, which two advances load.  Cells of thousands would
                            // else pass through whole (1M, 8 iterations, clumps at the cap of 128: 4.74 -> 2.19 ms).
                            if (end > t0 + 128u) {
                                uint32_t to = end & ~63u;
                                asm("" : "+s"(to));  // as in done: not in advance for every run
                                ranked = kSkipped;
#pragma unroll
                                for (uint32_t u = 0; u < kRounds; ++u)
                                    ranked += (uint32_t)__builtin_popcountll(__ballot(mark[u] < to));
                                t0 = to - 128u;
                            }
                            break;
                        }
                    }
                }
                uint32_t grown = 0;
                if (room) {
#pragma unroll
                    for (uint32_t q = 0; q < kWaveRows; ++q) {
                        if (q && done(q, grown)) break;
                        const uint64_t m = within(q);
                        grown = (uint32_t)__builtin_popcountll(m);
                        *(lds_u32*)select(m, put[q] + 4u * lanes_below(m), spare) = ph;
                        put[q] += 4u * grown;
                    }
                } else {  // lists near their cap
                    asm volatile("");  // the branches' first tests, merged, would pass through vector registers
#pragma unroll
                    for (uint32_t q = 0; q < kWaveRows; ++q) {
                        if (q && done(q, grown)) break;
                        const uint64_t m = within(q);
                        grown = (uint32_t)__builtin_popcountll(m);
                        const uint32_t left = maxN - ((put[q] - (row0At + 4u * q * rowWords)) >> 2);
                        const uint32_t k = lanes_below(m);
                        *(lds_u32*)select(m & __builtin_amdgcn_ballot_w64(k < left), put[q] + 4u * k, spare) = ph;
                        put[q] += 4u * min(grown, left);
                    }
                }
                if (end <= t0 + 64u) break;
                advance();
            }
#pragma unroll
            for (uint32_t q = 0; q < kWaveRows; ++q) {
                if (q >= np) break;
                counts = lane == first + q ? (put[q] - (row + 4u * q * rowWords)) >> 2 : counts;
            }
            begin = end;
        }
    }
    flush();
    if (mine) d.cnt[slot] = counts;
}

// The balanced work order (launch_balance): one workgroup per tile of T physical slots.  The
// slots are ranked by the key (scene rank within the tile, 254 - min(count, 254)), padding slots
// past a scene's end last within their scene; a slot's work position is the tile base plus its
// rank.  A scene owns whole 256-slot chunks, so its slots keep exactly the positions of its own
// chunks and every wave of work positions belongs to one scene.  Equal keys are ranked by LDS
// atomics, in no fixed order: the order only decides which lane handles which particle, never a
// result.  Then each lane copies the list of one work position into nbrW, one 16-byte chunk per
// four entries, so a wave writes each chunk row as one 1 KB block.
constexpr uint32_t kBalanceThreads = 256;
constexpr uint32_t kBalanceBins = (kBalanceMaxTile / 256) * 256;  // scene ranks x count classes

__global__ __launch_bounds__(kBalanceThreads) void k_balance(DeviceState d, SphParams P, uint32_t T,
                                                             uint32_t* __restrict__ work,
                                                             uint32_t* __restrict__ cntW,
                                                             uint4* __restrict__ nbrW) {
    __shared__ uint32_t bins[kBalanceBins];
    __shared__ uint32_t scan[kBalanceThreads];
    __shared__ uint16_t keyOf[kBalanceMaxTile];
    __shared__ uint16_t rankOf[kBalanceMaxTile];
    __shared__ uint32_t srcOf[kBalanceMaxTile];
    const uint32_t base = blockIdx.x * T;
    if (base >= d.nslots) return;
    const uint32_t n = min(T, d.nslots - base);
    const uint32_t tid = threadIdx.x;
    for (uint32_t b = tid; b < kBalanceBins; b += kBalanceThreads) bins[b] = 0u;
    __syncthreads();
    const uint32_t s0 = d.chunkScene[base >> 8];
    for (uint32_t e = tid; e < n; e += kBalanceThreads) {
        const uint32_t p = base + e;
        const uint32_t sc = d.chunkScene[p >> 8];
        const bool valid = p < d.scenes[sc].end;
        const uint32_t cls = valid ? 254u - min(d.cnt[p], 254u) : 255u;
        const uint32_t key = min(sc - s0, kBalanceMaxTile / 256 - 1) * 256u + cls;
        keyOf[e] = (uint16_t)key;
        rankOf[e] = (uint16_t)atomicAdd(&bins[key], 1u);
    }
    __syncthreads();
    // exclusive scan of the bins: each thread sums a run of kBalanceBins / kBalanceThreads bins
    constexpr uint32_t kRun = kBalanceBins / kBalanceThreads;
    uint32_t run = 0;
#pragma unroll
    for (uint32_t k = 0; k < kRun; ++k) run += bins[tid * kRun + k];
    scan[tid] = run;
    __syncthreads();
    for (uint32_t off = 1; off < kBalanceThreads; off <<= 1) {
        const uint32_t v = tid >= off ? scan[tid - off] : 0u;
        __syncthreads();
        scan[tid] += v;
        __syncthreads();
    }
    uint32_t acc = scan[tid] - run;
#pragma unroll
    for (uint32_t k = 0; k < kRun; ++k) {
        const uint32_t c = bins[tid * kRun + k];
        bins[tid * kRun + k] = acc;
        acc += c;
    }
    __syncthreads();
    for (uint32_t e = tid; e < n; e += kBalanceThreads) {
        const uint32_t r = bins[keyOf[e]] + rankOf[e];
        srcOf[r] = base + e;
    }
    __syncthreads();
    const uint32_t chunks = list_chunks(P.maxN);
    const uint32_t lane = tid & 63u, wave = tid >> 6;
    for (uint32_t w = wave; w * 64u < n; w += kBalanceThreads / 64u) {
        const uint32_t r = w * 64u + lane;
        if (r >= n) continue;
        const uint32_t t = base + r, p = srcOf[r];
        const uint32_t c = d.cnt[p];
        work[t] = p;
        cntW[t] = c;
        const uint4* src = d.nbr4 + list_base(p, P.maxN);
        uint4* dst = nbrW + list_base(t, P.maxN);
        const uint32_t nc = min((c + 3u) >> 2, chunks);
        for (uint32_t k = 0; k < nc; ++k) dst[(size_t)k * 64u] = src[(size_t)k * 64u];
    }
}

// Physical slot of work position t of a neighbour sweep (t itself without balancing).
__device__ __forceinline__ uint32_t work_slot(const DeviceState& d, uint32_t t) {
    return (d.work != nullptr && t < d.nslots) ? d.work[t] : t;
}

// The non-parity search (SphParams::searchCells == 2): cells of c = h / 2, keyed by their packed
// coordinates (cell_key_fine), so every bucket is one cell and none is walked twice.  A cell at
// offset (dx, dy, dz) from the particle's cell, |d| <= 2, can hold a particle within h only if its
// box comes within h of x_i: with f the particle's position in its cell (cell units), the box lies
// d - f away along an axis for d >= 1, f - d - 1 for d <= -1 and 0 for d = 0, and it is walked when
// the squared distances sum below (h / c)^2 = 4 (with a margin of 0.25% for the rounding of f).
// Walked cells go in (dx, dy, dz) order, each bucket in logical order, self skipped, r^2 < h^2
// kept, at most maxNeighbours: the list holds every particle within h (up to the cap).
__global__ __launch_bounds__(kBlock) void k_neighbours_fine(DeviceState d, SphParams P) {
    const uint32_t p = xcd_slot<kBlock>();
    uint32_t count = 0;
    if (p < d.nslots) {
        const SceneDev& sc = scene_of(d, p);
        if (p < sc.end) {
            const f3 xi = make3(d.XsA[p]);
            const float qx = xi.x / P.cellSearch, qy = xi.y / P.cellSearch, qz = xi.z / P.cellSearch;
            const int cx = to_int_sat(floorf(qx)), cy = to_int_sat(floorf(qy)), cz = to_int_sat(floorf(qz));
            const float fx = qx - floorf(qx), fy = qy - floorf(qy), fz = qz - floorf(qz);
            constexpr float kReach2 = 4.01f;
            uint32_t* out = reinterpret_cast<uint32_t*>(d.nbr4 + list_base(p, P.maxN));
            const uint32_t maxN = (uint32_t)P.maxN;
            auto gap = [](int dd, float f) {
                return dd > 0 ? (float)dd - f : dd < 0 ? f - (float)(dd + 1) : 0.0f;
            };
            for (int dx = -2; dx <= 2 && count < maxN; ++dx) {
                const float gx = gap(dx, fx), gx2 = gx * gx;
                if (gx2 >= kReach2) continue;
                for (int dy = -2; dy <= 2 && count < maxN; ++dy) {
                    const float gy = gap(dy, fy), gxy = gx2 + gy * gy;
                    if (gxy >= kReach2) continue;
                    for (int dz = -2; dz <= 2 && count < maxN; ++dz) {
                        const float gz = gap(dz, fz);
                        if (gxy + gz * gz >= kReach2) continue;
                        const uint32_t h = cell_key_fine(cx + dx, cy + dy, cz + dz);
                        uint4 e;
                        if (!table_find(d.table, sc, h, e)) continue;
                        const uint32_t a = e.x, b = e.y;
                        const bool run = e.w != 0u;
                        const int32_t shift = (int32_t)e.z - (int32_t)a;
                        for (uint32_t m0 = a; m0 < b && count < maxN; m0 += 4) {
                            float4 c[4];
                            uint32_t ph[4];
                            batch_slots<4>(d, run, m0, b, shift, ph);
#pragma unroll
                            for (int u = 0; u < 4; ++u) c[u] = ld(d.XsA, ph[u]);
#pragma unroll
                            for (int u = 0; u < 4; ++u) {
                                const f3 sep = xi - make3(c[u]);
                                if ((m0 + u < b) & (dot3(sep, sep) < P.h2) & (ph[u] != p) & (count < maxN)) {
                                    out[((size_t)(count >> 2) * 64u) * 4u + (count & 3u)] = ph[u];
                                    ++count;
                                }
                            }
                        }
                    }
                }
            }
        }
        d.cnt[p] = count;
    }
}

// Sum of the neighbour counts of every particle slot (statistics, on demand): one partial per
// workgroup, summed by the host.
__global__ __launch_bounds__(256) void k_count_sum(const DeviceState d, unsigned long long* part) {
    __shared__ unsigned long long sm[256];
    unsigned long long t = 0;
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < d.nslots; i += gridDim.x * 256)
        if (i < scene_of(d, i).end) t += d.cnt[i];
    sm[threadIdx.x] = t;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) sm[threadIdx.x] += sm[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sm[0];
}

// kernel_calculate_densities (ConstraintSolverCUDA.cu:16-42) and kernel_calculate_lambdas
// (ConstraintSolverCUDA.cu:51-97) in one neighbour sweep.  Each sum keeps the reference's order
// (the list order), so fusing the loops changes no rounding.
// Residual contribution of one particle: max(0, C), with a non-finite C counted as infinite.
__device__ __forceinline__ float positive_part(float C) {
    return C > 0.0f ? C : (C == C ? 0.0f : __builtin_inff());
}

// Residual statistics of one check: the wave's max and sum of non-negative values, written as
// the wave's partial (no atomics; k_resid_reduce combines the partials of each scene in a fixed
// order).  Every wave with a slot below nslots writes its partial.
__device__ __forceinline__ void wave_resid_partial(const DeviceState& d, int slot, uint32_t i,
                                                   float v) {
    float m = v, t = v;
    for (int off = 32; off > 0; off >>= 1) {
        m = fmaxf(m, __shfl_xor(m, off, 64));
        t += __shfl_xor(t, off, 64);
    }
    if (__lane_id() == 0) d.residPart[(size_t)slot * d.nWaves + (i >> 6)] = make_float2(m, t);
}

// A sweep's body by SphParams::fast: f(std::true_type) or f(std::false_type), chosen by the launch, or,
// where the masses came from device memory (2), by what the device found in them.  The branch is the same
// for a whole launch; with it a sweep of unit masses costs what it does where the host knows them, plus
// one scalar load.
template <int kFast, class F>
__device__ __forceinline__ void by_masses(const DeviceState& d, F f) {
    if constexpr (kFast == 2) {
        if (*d.massesDiffer == 0u)
            f(std::true_type{});
        else
            f(std::false_type{});
    } else {
        f(std::bool_constant<kFast == 1>{});
    }
}

// kFast (SphParams::fast): unit masses, range-tested quotients bounded in advance.
// kBnd: boundary samples (SphParams::bd): their density and gradient sums join rho and grad_i C
// after the neighbour sweep; the gradient sum is kept in Bg for the position-delta pass, which
// runs at the same x*.
template <int BS, bool kFast, bool kBnd>
__device__ __forceinline__ void density_lambda_slot(const DeviceState& d, const SphParams& P,
                                                    const float4* __restrict__ Xs, int residSlot,
                                                    int gated, uint32_t t) {
    const uint32_t t0 = t & ~63u;
    if (t0 >= d.nslots) return;  // the whole wave is past the last slot
    const uint32_t sIdx = d.chunkScene[t0 >> 8];  // a wave never spans two scenes
    if (gated && !d.gate[sIdx]) return;
    const uint32_t i = work_slot(d, t);
    const bool valid = t < d.nslots && i < d.scenes[sIdx].end;
    float C = 0.0f;
    if (valid) {
        const float4 xi4 = Xs[i];
        const f3 xi = make3(xi4);
        const uint32_t n = d.cntW[t];
        const uint4* lp = d.nbrW + list_base(t, P.maxN);
        float rho = xi4.w * P.w0;
        f3 gi{0.0f, 0.0f, 0.0f};
        float sum = 0.0f;
        const float negInv = -P.invRest;
        walk_list<float4>(
            lp, n, [&](uint32_t j) { return ld(Xs, j); },
            [&](const float4& xj4) {
                f3 sep = xi - make3(xj4);
                float d2 = dot3(sep, sep);
                // m_j == 1 under kFast: every product by m_j is the other factor itself
                const float w = poly6_of<kFast>(d2, P);
                rho = rho + (kFast ? w : xj4.w * w);
                // a zero gradient would add zeros to gi and sum, which change neither (both start
                // at +0, and x + (-x) rounds to +0, so neither is ever -0): it is skipped
                f3 g;
                if (grad_of<kFast>(sep, d2, P, g)) {
                    if (kFast) {
                        gi = gi + g;
                        f3 gj = negInv * g;
                        sum = sum + dot3(gj, gj);
                    } else {
                        gi = gi + xj4.w * g;
                        f3 gj = (negInv * xj4.w) * g;
                        sum = sum + dot3(gj, gj);
                    }
                }
            });
        if (kBnd) {
            float rb = 0.0f;
            f3 gb{0.0f, 0.0f, 0.0f};
            if (boundary_near(P.bd, xi.x, xi.y, xi.z, P.h2)) {
                boundary_visit(P.bd, xi.x, xi.y, xi.z, P.h, P.h2,
                               [&](uint32_t idx, float s0, float s1, float s2, float d2) {
                                   const float psi = P.bd.psi[idx];
                                   rb = rb + psi * poly6_of<kFast>(d2, P);
                                   gb = gb + psi * grad_or_zero<kFast>(f3{s0, s1, s2}, d2, P);
                               });
                d.Bg[i] = make_float4(gb.x, gb.y, gb.z, 0.0f);
            }
            rho = rho + rb;
            gi = gi + gb;
        }
        gi = gi * P.invRest;
        C = rho * P.invRest - 1.0f;
        d.dens[i] = rho;
        const float lam = -C / ((sum + dot3(gi, gi)) + P.relax);
        d.lam[i] = lam;
        // unit masses: (x*, lambda) side by side for the position-delta pass, in W (free until
        // the vorticity pass)
        if (kFast) d.W[i] = make_float4(xi.x, xi.y, xi.z, lam);
    }
    if (residSlot >= 0) wave_resid_partial(d, residSlot, t, valid ? positive_part(C) : 0.0f);
}

// One workgroup per virtual workgroup (the loop runs once); the loop form lets a launch use any
// grid size.
template <int BS, int kFast, bool kBnd>
__global__ __launch_bounds__(BS) void k_density_lambda(DeviceState d, SphParams P,
                                                           const float4* __restrict__ Xs,
                                                           int residSlot, int gated, uint32_t nvb) {
    by_masses<kFast>(d, [&](auto fast) {
        for (uint32_t vb = blockIdx.x; vb < nvb; vb += gridDim.x)
            density_lambda_slot<BS, decltype(fast)::value, kBnd>(d, P, Xs, residSlot, gated, xcd_slot_of<BS>(vb, nvb));
    });
}

// Features of the learned warm start at x*_pred, one neighbour sweep (list order):
//   0 C = rho / rho0 - 1 and 1 lambda, as the first Jacobi iteration computes them
//   2 neighbour count, 3 lambda of the previous step
//   4-6 (x*_pred - x) / h
//   7-9 2 lambda (1/rho0) sum_j m_j grad W_ij / h: the correction if every neighbour had this
//       particle's lambda
//   10-12 (1/rho0) sum_j m_j s_corr,ij grad W_ij / h: the artificial-pressure correction
//   13-15 wall proximity per axis, clamp((x - lo) / h, 0, 2) - clamp((hi - x) / h, 0, 2)
__device__ __forceinline__ void features_slot(const DeviceState& d, const SphParams& P, int record,
                                              uint32_t t) {
    const uint32_t t0 = t & ~63u;
    if (t0 >= d.nslots) return;
    const uint32_t sIdx = d.chunkScene[t0 >> 8];
    const SceneDev& sc = d.scenes[sIdx];
    const uint32_t i = work_slot(d, t);
    const bool valid = t < d.nslots && i < sc.end;
    float C = 0.0f;
    if (valid) {
        const float4 xi4 = d.XsA[i];
        const f3 xi = make3(xi4);
        const uint32_t n = d.cntW[t];
        const uint4* lp = d.nbrW + list_base(t, P.maxN);
        float rho = xi4.w * P.w0;
        f3 gi{0.0f, 0.0f, 0.0f}, ac{0.0f, 0.0f, 0.0f};
        float sum = 0.0f;
        const float negInv = -P.invRest;
        const Recip Rdq = recip(P.wdq);
        walk_list<float4>(
            lp, n, [&](uint32_t j) { return ld(d.XsA, j); },
            [&](const float4& xj4) {
                f3 sep = xi - make3(xj4);
                float d2 = dot3(sep, sep);
                const float w = poly6(d2, P);
                rho = rho + xj4.w * w;
                f3 g = grad_spiky(sep, P);
                gi = gi + xj4.w * g;
                f3 gj = (negInv * xj4.w) * g;
                sum = sum + dot3(gj, gj);
                if (P.corrOn) {
                    const float lc = P.negCorrK * corr_pow(div_rn(w, Rdq), P);
                    ac = ac + (lc * xj4.w) * g;
                }
            });
        gi = gi * P.invRest;
        C = rho * P.invRest - 1.0f;
        const float lam1 = -C / ((sum + dot3(gi, gi)) + P.relax);
        const float invH = 1.0f / P.h;
        const float4 x0 = d.X0[i];
        const f3 sg = gi * (2.0f * lam1 * invH);
        const f3 sa = ac * (P.invRest * invH);
        float wall[3];
        const float xa[3] = {xi.x, xi.y, xi.z};
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const float lo = fminf(fmaxf((xa[a] - sc.bmin[a]) * invH, 0.0f), 2.0f);
            const float hi = fminf(fmaxf((sc.bmax[a] - xa[a]) * invH, 0.0f), 2.0f);
            wall[a] = lo - hi;
        }
        float4* f = reinterpret_cast<float4*>(d.feat + (size_t)i * kMlpFeatures);
        f[0] = make_float4(C, lam1, (float)n, d.Tlam[i]);
        f[1] = make_float4((xi.x - x0.x) * invH, (xi.y - x0.y) * invH, (xi.z - x0.z) * invH, sg.x);
        f[2] = make_float4(sg.y, sg.z, sa.x, sa.y);
        f[3] = make_float4(sa.z, wall[0], wall[1], wall[2]);
        if (record) d.XsP[i] = xi4;
    }
    wave_resid_partial(d, 0, t, valid ? positive_part(C) : 0.0f);
}

template <int BS>
__global__ __launch_bounds__(BS) void k_features(DeviceState d, SphParams P, int record) {
    features_slot(d, P, record, xcd_slot<BS>());
}

// Residual statistics per scene in two fixed-order stages (deterministic sums, no atomics).
// Stage 1: workgroup (b, s) reduces up to kResidWavesPerBlock wave partials of scene s for each
// check in slotMask into one block partial.
constexpr int kReduceBlock = 256;
constexpr uint32_t kResidWavesPerBlock = 8u * kReduceBlock;

__device__ __forceinline__ void block_max_sum(float& m, float& t, float* sm, float* st) {
    for (int off = 32; off > 0; off >>= 1) {
        m = fmaxf(m, __shfl_xor(m, off, 64));
        t += __shfl_xor(t, off, 64);
    }
    const int w = threadIdx.x >> 6;
    if (__lane_id() == 0) {
        sm[w] = m;
        st[w] = t;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < kReduceBlock / 64; ++k) {
            sm[0] = fmaxf(sm[0], sm[k]);
            st[0] += st[k];
        }
    }
    __syncthreads();
    m = sm[0];
    t = st[0];
    __syncthreads();
}

__global__ __launch_bounds__(kReduceBlock) void k_resid_blocks(DeviceState d, int slotMask) {
    __shared__ float sm[kReduceBlock / 64], st[kReduceBlock / 64];
    const uint32_t b = blockIdx.x, s = blockIdx.y;
    const SceneDev& sc = d.scenes[s];
    const uint32_t w0 = (sc.begin >> 6) + b * kResidWavesPerBlock;
    const uint32_t w1 = min((sc.end + 63) >> 6, w0 + kResidWavesPerBlock);
    for (int k = 0; k < 3; ++k) {
        if (!((slotMask >> k) & 1)) continue;
        float m = 0.0f, t = 0.0f;
        const float2* part = d.residPart + (size_t)k * d.nWaves;
#pragma unroll
        for (uint32_t r = 0; r < kResidWavesPerBlock / kReduceBlock; ++r) {
            const uint32_t w = w0 + r * kReduceBlock + threadIdx.x;
            if (w < w1) {
                const float2 p = part[w];
                m = fmaxf(m, p.x);
                t += p.y;
            }
        }
        block_max_sum(m, t, sm, st);
        if (threadIdx.x == 0)
            d.residBlk[((size_t)s * d.residBlocks + b) * 3 + k] = make_float2(m, t);
    }
}

// Stage 2, one wave per scene: the scene's block partials into its record; with gate, also the
// fallback decision from checks 0 (x*_pred) and 1 (x*_w).
__global__ __launch_bounds__(64) void k_resid_reduce(DeviceState d, int slotMask, int gate,
                                                     int statistic, float ratio, float tolerance) {
    const uint32_t s = blockIdx.x;
    const SceneDev& sc = d.scenes[s];
    const uint32_t nb = ((((sc.end + 63) >> 6) - (sc.begin >> 6)) + kResidWavesPerBlock - 1) /
                        kResidWavesPerBlock;
    unsigned int* rec = d.resid + s * kResidStride;
    for (int k = 0; k < 3; ++k) {
        if (!((slotMask >> k) & 1)) continue;
        float m = 0.0f, t = 0.0f;
        for (uint32_t b = __lane_id(); b < nb; b += 64) {
            const float2 p = d.residBlk[((size_t)s * d.residBlocks + b) * 3 + k];
            m = fmaxf(m, p.x);
            t += p.y;
        }
        for (int off = 32; off > 0; off >>= 1) {
            m = fmaxf(m, __shfl_xor(m, off, 64));
            t += __shfl_xor(t, off, 64);
        }
        if (__lane_id() == 0) {
            rec[k] = __float_as_uint(m);
            rec[kResidSum + k] = __float_as_uint(t);
        }
    }
    if (gate && __lane_id() == 0) {
        float rp, rw;
        if (statistic == 0) {
            rp = __uint_as_float(rec[0]);
            rw = __uint_as_float(rec[1]);
        } else {
            const float inv = 1.0f / (float)max(1u, sc.end - sc.begin);
            rp = __uint_as_float(rec[kResidSum]) * inv;
            rw = __uint_as_float(rec[kResidSum + 1]) * inv;
        }
        const uint32_t g = (rw <= ratio * rp + tolerance) ? 0u : 1u;
        d.gate[s] = g;
        d.fallbacks[s] += g;
    }
}

// Targets: x* before the last Jacobi iteration (XsLast) relative to x*_pred, in units of h, and
// the last iteration's lambda.
__global__ void k_targets(DeviceState d, SphParams P, const float4* __restrict__ XsLast) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= d.nslots) return;
    if (i >= scene_of(d, i).end) return;
    const float invH = 1.0f / P.h;
    const float4 x = XsLast[i], p = d.XsP[i];
    reinterpret_cast<float4*>(d.targ)[i] =
        make_float4((x.x - p.x) * invH, (x.y - p.y) * invH, (x.z - p.z) * invH, d.lam[i]);
}

__global__ void k_sample(DeviceState d, uint64_t seed, uint32_t count, float* __restrict__ fo,
                         float* __restrict__ to) {
    const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= count) return;
    const SceneDev& sc = d.scenes[0];
    uint64_t z = seed + 0x9E3779B97F4A7C15ull * (uint64_t)(b + 1);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    const uint32_t slot = sc.begin + (uint32_t)(z % (uint64_t)(sc.end - sc.begin));
    const float4* f = reinterpret_cast<const float4*>(d.feat + (size_t)slot * kMlpFeatures);
    float4* g = reinterpret_cast<float4*>(fo + (size_t)b * kMlpFeatures);
#pragma unroll
    for (int k = 0; k < 4; ++k) g[k] = f[k];
    reinterpret_cast<float4*>(to)[b] = reinterpret_cast<const float4*>(d.targ)[slot];
}

// resolve_collision over the six walls in order (IntegrationCUDA.cu:51-102), restitution 0 and
// friction 0.95 (PBFSolver.cpp:64); vector form as written, so every rounding matches.
__device__ __forceinline__ f3 damp_walls(f3 x, f3 v, const SceneDev& sc) {
    const float minDist = 0.025f, restitution = 0.0f, friction = 0.95f;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        const int a = k >> 1;
        const float sgn = (k & 1) ? -1.0f : 1.0f;
        const float b = (k & 1) ? sc.bmax[a] : sc.bmin[a];
        f3 pt{a == 0 ? b : 0.0f, a == 1 ? b : 0.0f, a == 2 ? b : 0.0f};
        f3 nm{a == 0 ? sgn : 0.0f, a == 1 ? sgn : 0.0f, a == 2 ? sgn : 0.0f};
        float distance = dot3(x - pt, nm);
        float approaching = dot3(v, nm);
        if (distance < minDist) {
            f3 vn = approaching * nm;
            f3 vt = v - vn;
            if (approaching < 0.0f) {
                v = (-restitution) * vn + (1.0f - friction) * vt;
            } else if (fabsf(approaching) < 1e-5f) {
                v = (1.0f - friction) * vt;
            }
        }
    }
    return v;
}

// kernel_correct_position with handle_particle_collision (ConstraintSolverCUDA.cu:136-169) after
// the neighbour sum: dp becomes sum / rho0 and the corrected position is clamped to the walls.
__device__ __forceinline__ f3 correct_position(f3 xi, f3& dp, const SphParams& P, const SceneDev& sc) {
    dp = dp * P.invRest;
    f3 q = xi + dp;
    const float minDist = 0.025f, stiff = 0.5f;
    float qa[3] = {q.x, q.y, q.z};
    float c[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        if (qa[a] < sc.bmin[a] + minDist) c[a] = c[a] + stiff * (sc.bmin[a] + minDist - qa[a]);
        if (qa[a] > sc.bmax[a] - minDist) c[a] = c[a] + stiff * (sc.bmax[a] - minDist - qa[a]);
    }
    return q + f3{c[0], c[1], c[2]};
}

// kernel_update_position_and_velocity (IntegrationCUDA.cu:38-49) and the wall damping at the last
// iteration's corrected position q, and the step's writes of slot i.
struct FinishIn {
    float4 x0;
    uint32_t id, lid;
};
__device__ __forceinline__ FinishIn finish_in(const DeviceState& d, uint32_t i) {
    return {d.X0[i], d.Tid[i], d.lidT[i]};
}

template <bool kApplyDelta>
__device__ __forceinline__ void finish_step(const DeviceState& d, const StepParams& S, const SceneDev& sc,
                                            uint32_t i, float4 xi4, const FinishIn& in, f3 q, f3 dp) {
    f3 v = div3_rn(q - make3(in.x0), S.dt);
    d.VS[i] = make_float4(v.x, v.y, v.z, 0.0f);  // the record's new_velocity (IntegrationCUDA.cu:45)
    v = damp_walls(q, v, sc);
    d.X[i] = make_float4(q.x, q.y, q.z, xi4.w);
    d.V[i] = make_float4(v.x, v.y, v.z, 0.0f);
    d.id[i] = in.id;
    d.lid[i] = in.lid;
    if (kApplyDelta) {  // the record's position_delta (ConstraintSolverCUDA.cu:129)
        d.DP[i] = make_float4(dp.x, dp.y, dp.z, 0.0f);
    } else {  // no iteration ran: density, lambda and the position delta carry over
        d.dens[i] = d.Tdens[i];
        d.lam[i] = d.Tlam[i];
        d.DP[i] = d.TDP[i];
    }
}

// kernel_calculate_position_delta (ConstraintSolverCUDA.cu:99-130), then kernel_correct_position
// with handle_particle_collision (ConstraintSolverCUDA.cu:136-169).  x* is double-buffered: the
// kernel reads XsIn and writes XsOut, so every particle sees the positions of the same iteration.
// kFinal: also kernel_update_position_and_velocity (IntegrationCUDA.cu:38-49) and the wall
// damping, writing the step's positions X, velocities V, ids and the two order maps.
// gateMode 1: only scenes whose gate is set run; 2: scenes whose gate is clear read XsAlt.
template <int BS, bool kFinal, bool kApplyDelta, bool kFast, bool kBnd>
__device__ __forceinline__ void delta_correct_slot(const DeviceState& d, const SphParams& P,
                                                   const StepParams& S,
                                                   const float4* __restrict__ XsSet,
                                                   float4* __restrict__ XsOut,
                                                   const float4* __restrict__ XsAlt, int gateMode,
                                                   uint32_t t) {
    if (t >= d.nslots) return;
    const uint32_t i = work_slot(d, t);
    const uint32_t sIdx = d.chunkScene[i >> 8];
    const SceneDev& sc = d.scenes[sIdx];
    if (i >= sc.end) return;
    if (gateMode == 1 && !d.gate[sIdx]) return;
    const float4* __restrict__ XsIn = (gateMode == 2 && !d.gate[sIdx]) ? XsAlt : XsSet;
    const float4 xi4 = XsIn[i];
    const f3 xi = make3(xi4);
    f3 q = xi;
    f3 dp{0.0f, 0.0f, 0.0f};
    if (kApplyDelta) {
        const float li = d.lam[i];
        const uint32_t n = d.cntW[t];
        const uint4* lp = d.nbrW + list_base(t, P.maxN);
        const Recip Rdq = recip(P.wdq);
        // unit masses: x*_j and lambda_j from one float4 written by the density pass (W)
        const auto load = [&](uint32_t j) {
            if (kFast) {
                const float4 a = ld(d.W, j);
                return XLam{a, a.w};
            }
            return XLam{ld(XsIn, j), ld(d.lam, j)};
        };
        // the walk once with and once without the artificial pressure s_corr, chosen per launch
        const auto walk = [&](auto corrOn) {
            constexpr bool kCorr = decltype(corrOn)::value;
            walk_list<XLam, kBatchDelta>(lp, n, load, [&](const XLam& nb) {
                f3 sep = xi - make3(nb.x);
                float d2 = dot3(sep, sep);
                float coef = li + nb.lam;
                f3 g;
                bool some;  // a gradient that is not zero
                if constexpr (kFast) {
                    // the quotient of s_corr and the gradient's, with one test for the rare cases of all
                    const float w = kCorr ? poly6_bounded(d2, P) : 1.0f;
                    float q = kCorr ? div_by(w, Rdq.b, Rdq.r) : 0.0f;
                    GradTerm G;
                    some = grad_term(sep, d2, P, G);
                    if (__builtin_expect(some && (fminf(G.low, w) < kDivLowest || G.inexact), 0)) {
                        if (kCorr) q = corr_by_division(w, q, Rdq);
                        grad_by_division(G);
                    }
                    if (kCorr) coef = coef + P.negCorrK * corr_pow(q, P);
                    if (some) g = G.g;
                } else {
                    if (kCorr) coef = coef + P.negCorrK * corr_pow(div_rn(poly6(d2, P), Rdq), P);
                    some = grad_spiky_nonzero(sep, P, g);
                }
                const float c = kFast ? coef : coef * nb.x.w;  // m_j == 1 under kFast
                if (__builtin_expect(some, 1)) {
                    dp = dp + c * g;
                } else {  // the zero gradient's term c * 0: zeros, or NaN where c is not finite
                    const f3 z{0.0f, 0.0f, 0.0f};
                    dp = dp + c * z;
                }
            });
        };
        if (P.corrOn)
            walk(std::true_type{});
        else
            walk(std::false_type{});
        if (kBnd) {  // lambda_i times the boundary gradient sum of the density pass (same x*)
            f3 gb{0.0f, 0.0f, 0.0f};
            if (boundary_near(P.bd, xi.x, xi.y, xi.z, P.h2)) gb = make3(d.Bg[i]);
            dp = dp + li * gb;
        }
        q = correct_position(xi, dp, P, sc);
    }
    if (!kFinal) {
        XsOut[i] = make_float4(q.x, q.y, q.z, xi4.w);
        return;
    }
    finish_step<kApplyDelta>(d, S, sc, i, xi4, finish_in(d, i), q, dp);
}

// Unit masses: held to 8 waves per SIMD (its scalar registers, over the 8-wave budget, spill to
// vector lanes); the general kernels would spill vector registers there.
template <int BS, bool kFinal, bool kApplyDelta, int kFast, bool kBnd>
__global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(kFast == 1 && !kBnd ? 8 : 1)))
void k_delta_correct(DeviceState d, SphParams P, StepParams S,
                                                          const float4* __restrict__ XsSet,
                                                          float4* __restrict__ XsOut,
                                                          const float4* __restrict__ XsAlt,
                                                          int gateMode, uint32_t nvb) {
    by_masses<kFast>(d, [&](auto fast) {
        for (uint32_t vb = blockIdx.x; vb < nvb; vb += gridDim.x)
            delta_correct_slot<BS, kFinal, kApplyDelta, decltype(fast)::value, kBnd>(d, P, S, XsSet, XsOut, XsAlt,
                                                                                     gateMode, xcd_slot_of<BS>(vb, nvb));
    });
}

// kernel_compute_vorticities (IntegrationCUDA.cu:104-128).  W.w keeps |omega| for the next pass,
// which also finds it beside the position in XsB (free between the last Jacobi iteration and the
// next step's): (x, |omega|), one gather per neighbour there.
template <bool kFast>
__device__ __forceinline__ void vorticity_slot(const DeviceState& d, const SphParams& P, uint32_t t) {
    if (t >= d.nslots) return;
    const uint32_t i = work_slot(d, t);
    if (i >= scene_of(d, i).end) return;
    const f3 xi = make3(d.X[i]);
    const f3 vi = make3(d.V[i]);
    const uint32_t n = d.cntW[t];
    const uint4* lp = d.nbrW + list_base(t, P.maxN);
    f3 w{0.0f, 0.0f, 0.0f};
    walk_list<XV, kBatchVort>(
        lp, n, [&](uint32_t j) { return XV{ld(d.X, j), ld(d.V, j)}; },
        [&](const XV& nb) {
            f3 vij = make3(nb.v) - vi;
            f3 sep = xi - make3(nb.x);
            const float mj = kFast ? -1.0f : -nb.x.w;  // m_j == 1 under kFast
            f3 g;
            if (__builtin_expect(grad_of<kFast>(sep, dot3(sep, sep), P, g), 1))
                w = w + mj * cross3(vij, g);
            else  // the zero gradient's term: zeros, or NaN where v_ij is not finite
                w = w + mj * cross3(vij, f3{0.0f, 0.0f, 0.0f});
        });
    const float wl = length3(w);
    d.W[i] = make_float4(w.x, w.y, w.z, wl);
    d.XsB[i] = make_float4(xi.x, xi.y, xi.z, wl);
}

template <int BS, int kFast>
__global__ __launch_bounds__(BS) void k_vorticity(DeviceState d, SphParams P) {
    by_masses<kFast>(d, [&](auto fast) { vorticity_slot<decltype(fast)::value>(d, P, xcd_slot<BS>()); });
}

// The confinement force from the summed eta (IntegrationCUDA.cu:146-163) and the write of Vc.
__device__ __forceinline__ void confine_finish(const DeviceState& d, const SphParams& P,
                                               const StepParams& S, uint32_t i, float xi4w, float4 wi,
                                               float4 v, f3 eta, float rho) {
    eta = eta * (1.0f / rho);
    float el = length3(eta);
    if (!(el < 1e-5f)) {
        f3 N = div3_rn(eta, el);
        f3 f = P.vortEps * cross3(N, make3(wi));
        f3 vn = make3(v) + S.dt * f;
        v = make_float4(vn.x, vn.y, vn.z, 0.0f);
    }
    v.w = xi4w / rho;
    d.Vc[i] = v;
}

// kernel_apply_vorticity_confinement (IntegrationCUDA.cu:130-165), writing Vc: the confined
// velocity, with the particle's m / rho in .w for the XSPH pass (the quotient the reference
// forms per neighbour, IntegrationCUDA.cu:184, computed once per particle instead).
template <bool kFast>
__device__ __forceinline__ void confinement_slot(const DeviceState& d, const SphParams& P,
                                                 const StepParams& S, uint32_t t) {
    if (t >= d.nslots) return;
    const uint32_t i = work_slot(d, t);
    if (i >= scene_of(d, i).end) return;
    const float4 xi4 = d.X[i];
    const f3 xi = make3(xi4);
    const float xi4w = xi4.w;
    const float4 wi = d.W[i];
    const uint32_t n = d.cntW[t];
    const uint4* lp = d.nbrW + list_base(t, P.maxN);
    f3 eta{0.0f, 0.0f, 0.0f};
    // XW.x: (x_j, |omega_j|); XW.w: m_j (read only without unit masses)
    walk_list<XW, kBatchConf>(
        lp, n, [&](uint32_t j) { return XW{ld(d.XsB, j), kFast ? 1.0f : ld(d.X, j).w}; },
        [&](const XW& nb) {
            float diff = wi.w - nb.x.w;
            f3 sep = xi - make3(nb.x);
            const float c = kFast ? diff : nb.w * diff;  // m_j == 1 under kFast
            f3 g;
            if (__builtin_expect(grad_of<kFast>(sep, dot3(sep, sep), P, g), 1))
                eta = eta + c * g;
            else  // the zero gradient's term c * 0: zeros, or NaN where c is not finite
                eta = eta + c * f3{0.0f, 0.0f, 0.0f};
        });
    confine_finish(d, P, S, i, xi4w, wi, d.V[i], eta, d.dens[i]);
}

template <int BS, int kFast>
__global__ __launch_bounds__(BS) void k_confinement(DeviceState d, SphParams P, StepParams S) {
    by_masses<kFast>(d, [&](auto fast) { confinement_slot<decltype(fast)::value>(d, P, S, xcd_slot<BS>()); });
}

// kernel_apply_xsph_viscosity (IntegrationCUDA.cu:167-195), Jacobi: reads Vc, writes V.
__device__ __forceinline__ void xsph_slot(const DeviceState& d, const SphParams& P, uint32_t t) {
    if (t >= d.nslots) return;
    const uint32_t i = work_slot(d, t);
    if (i >= scene_of(d, i).end) return;
    const f3 xi = make3(d.X[i]);
    const f3 vi = make3(d.Vc[i]);
    const uint32_t n = d.cntW[t];
    const uint4* lp = d.nbrW + list_base(t, P.maxN);
    f3 dv{0.0f, 0.0f, 0.0f};
    walk_list<XV, kBatchXsph>(
        lp, n, [&](uint32_t j) { return XV{ld(d.X, j), ld(d.Vc, j)}; },
        [&](const XV& nb) {
            f3 vij = make3(nb.v) - vi;
            f3 sep = xi - make3(nb.x);
            float w = poly6(dot3(sep, sep), P);
            dv = dv + (nb.v.w * vij) * w;  // nb.v.w = m_j / rho_j
        });
    f3 vn = vi + P.visc * dv;
    d.V[i] = make_float4(vn.x, vn.y, vn.z, 0.0f);
}

template <int BS>
__global__ __launch_bounds__(BS) void k_xsph(DeviceState d, SphParams P) {
    xsph_slot(d, P, xcd_slot<BS>());
}

// ---- long lists shared by their wave -------------------------------------------------------------
// In a sprayed scene the lists of a wave differ: 16 entries on average, 54 the longest (1M dam break after
// 100 steps), and with one lane per list most lanes wait for a few.  Here each lane walks its list up to a
// little over the wave's average; the chunks of four entries that are left are dealt to all lanes, which
// compute their terms, and each list's own lane adds them from LDS in list order (a chunk's addition is
// some seven instructions against sixty per entry's terms).  The same terms in the same order: the same
// sums, with +0 in the place of entries past a list's end.
// Where no list is more than kTailMin entries over the average (settled scenes), nothing is dealt.
// Measured against one lane per list (the last delta: two): 50 steps of the 1M dam break 68 -> 61 us, the
// last 77 -> 75, a settled 1M 56 -> 55 and 82 -> 70, 64 scenes of 2.6M 136 -> 127 and 163 -> 158.  The density
// sweep, with five sums to pass through LDS and more waves per SIMD without them, gains nothing (55.9 us with
// one lane, 57.5 so) and keeps one lane.
constexpr uint32_t kTailMin = 8;

// The largest value of the wave's 64 lanes.
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
    for (int off = 32; off > 0; off >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, off, 64));
    return v;
}

// LDS of a wave: NA rows of 64 chunks' terms, and the lists' lanes by chunk.
template <int NA>
struct TailLds {
    float4 terms[NA][64];
    uint32_t owner[64];
};

// wave: chunk 0 of the list of the wave's lane 0; n: this lane's entries (0 without a particle);
// own: what the terms need of the particle, as floats.  Every lane of the wave takes part.
template <int NA, class T, int NO, class Load, class Term>
__device__ __forceinline__ void walk_shared(const uint4* __restrict__ wave, uint32_t n, const float (&own)[NO],
                                            Load load, Term term, float (&acc)[NA], TailLds<NA>& lds) {
    const uint32_t lane = __lane_id();
    const uint32_t longest = wave_max(n), mean = lane_u(wave_prefix(n), 63u) >> 6;
    uint32_t until = (mean + mean / 8u + 3u) & ~3u;
    if (longest <= until + kTailMin) until = longest;
    const auto one = [&](const float (&o)[NO], const T& v, float (&t)[NA]) { term(o, v, t); };
    walk_list<T>(wave + lane, min(n, until), load, [&](const T& v) {
        float t[NA];
        one(own, v, t);
#pragma unroll
        for (int c = 0; c < NA; ++c) acc[c] = acc[c] + t[c];
    });
    if (until == longest) return;
    const uint32_t chunks = n > until ? (n - until + 3u) >> 2 : 0u;
    const uint32_t end = wave_prefix(chunks), begin = end - chunks;
    const uint32_t total = lane_u(end, 63u);
    for (uint32_t q0 = 0; q0 < total; q0 += 64u) {
        // whose chunk is q0 + lane: the last list that begins at or before it
        wave_lds_order();
        lds.owner[lane] = 0u;
        wave_lds_order();
        if (chunks != 0u && begin < q0 + 64u && end > q0) lds.owner[begin > q0 ? begin - q0 : 0u] = lane;
        wave_lds_order();
        const int who = (int)wave_prefix_max(lds.owner[lane]);
        float o[NO];
#pragma unroll
        for (int k = 0; k < NO; ++k) o[k] = __shfl(own[k], who, 64);
        const uint32_t first = (uint32_t)__shfl((int)begin, who, 64), entries = (uint32_t)__shfl((int)n, who, 64);
        const bool in = q0 + lane < total;
        const uint32_t k = in ? until + 4u * (q0 + lane - first) : 0u;  // the chunk's first entry; 0: some list's
        float t[4][NA] = {};
        if (in) {
            const uint4 ch = wave[(size_t)(k >> 2) * 64u + (uint32_t)who];
            const uint32_t e[4] = {ch.x, ch.y, ch.z, ch.w};
            T v[4];
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) v[u] = load(k + u < entries ? e[u] : e[0]);
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {
                float r[NA];
                one(o, v[u], r);
#pragma unroll
                for (int c = 0; c < NA; ++c) t[u][c] = k + u < entries ? r[c] : 0.0f;
            }
        }
#pragma unroll
        for (int c = 0; c < NA; ++c) lds.terms[c][lane] = make_float4(t[0][c], t[1][c], t[2][c], t[3][c]);
        wave_lds_order();
        const uint32_t from = max(begin, q0), to = min(end, q0 + 64u);
        for (uint32_t q = from; q < to; ++q) {
#pragma unroll
            for (int c = 0; c < NA; ++c) {
                const float4 x = lds.terms[c][q - q0];
                acc[c] = (((acc[c] + x.x) + x.y) + x.z) + x.w;
            }
        }
    }
}

constexpr int kTailBlock = 256;

// The position delta and correction of a plain step (no work order, gate or wall samples).
template <bool kFinal, bool kFast>
__device__ __forceinline__ void delta_correct_tail(const DeviceState& d, const SphParams& P, const StepParams& S,
                                                   const float4* __restrict__ XsIn, float4* __restrict__ XsOut,
                                                   TailLds<3>* lds) {
    const uint32_t i = xcd_slot<kTailBlock>(), i0 = i & ~63u;
    if (i0 >= d.nslots) return;
    const SceneDev& sc = scene_of(d, i0);
    const bool valid = i < d.nslots && i < sc.end;
    const float4 xi4 = valid ? XsIn[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const f3 xi = make3(xi4);
    const float own[4] = {xi.x, xi.y, xi.z, valid ? d.lam[i] : 0.0f};
    const Recip Rdq = recip(P.wdq);
    float acc[3] = {0.0f, 0.0f, 0.0f};
    const auto walk = [&](auto corrOn) {
        constexpr bool kCorr = decltype(corrOn)::value;
        walk_shared<3, XLam>(
            d.nbr4 + list_base(i0, P.maxN), valid ? d.cnt[i] : 0u, own,
            [&](uint32_t j) {
                if (kFast) {
                    const float4 a = ld(d.W, j);
                    return XLam{a, a.w};
                }
                return XLam{ld(XsIn, j), ld(d.lam, j)};
            },
            [&](const float (&o)[4], const XLam& nb, float (&t)[3]) {
                const f3 sep = f3{o[0], o[1], o[2]} - make3(nb.x);
                const float d2 = dot3(sep, sep);
                float coef = o[3] + nb.lam;
                f3 g{0.0f, 0.0f, 0.0f};
                if constexpr (kFast) {
                    // the quotient of s_corr and the gradient's, with one test for the rare cases of all
                    const float w = kCorr ? poly6_bounded(d2, P) : 1.0f;
                    float q = kCorr ? div_by(w, Rdq.b, Rdq.r) : 0.0f;
                    GradTerm G;
                    const bool some = grad_term(sep, d2, P, G);
                    if (__builtin_expect(some && (fminf(G.low, w) < kDivLowest || G.inexact), 0)) {
                        if (kCorr) q = corr_by_division(w, q, Rdq);
                        grad_by_division(G);
                    }
                    if (kCorr) coef = coef + P.negCorrK * corr_pow(q, P);
                    if (some) g = G.g;
                } else {
                    if (kCorr) coef = coef + P.negCorrK * corr_pow(div_rn(poly6(d2, P), Rdq), P);
                    grad_spiky_nonzero(sep, P, g);
                }
                const f3 u = (kFast ? coef : coef * nb.x.w) * g;  // m_j == 1 under kFast
                t[0] = u.x; t[1] = u.y; t[2] = u.z;
            },
            acc, lds[threadIdx.x >> 6]);
    };
    if (P.corrOn)
        walk(std::true_type{});
    else
        walk(std::false_type{});
    if (!valid) return;
    f3 dp{acc[0], acc[1], acc[2]};
    const f3 q = correct_position(xi, dp, P, sc);
    if (!kFinal) {
        XsOut[i] = make_float4(q.x, q.y, q.z, xi4.w);
        return;
    }
    finish_step<true>(d, S, sc, i, xi4, finish_in(d, i), q, dp);
}

template <bool kFinal, int kFast>
__global__ __launch_bounds__(kTailBlock) void k_delta_correct_tail(DeviceState d, SphParams P, StepParams S,
                                                                   const float4* __restrict__ XsIn,
                                                                   float4* __restrict__ XsOut) {
    __shared__ TailLds<3> lds[kTailBlock / 64];
    by_masses<kFast>(d, [&](auto fast) { delta_correct_tail<kFinal, decltype(fast)::value>(d, P, S, XsIn, XsOut, lds); });
}

// ---- work queue: the sweeps as persistent kernels over 256-slot tiles, heaviest first -------
// A batch of uneven scenes (and the uneven lists of one scene) leave each sweep's last waves
// running on a few CUs.  With the work queue, each XCD has a contiguous eighth of the tiles, ordered by
// the sum of their neighbour counts, heaviest first, once per step after the list build; each sweep then runs a resident grid whose workgroups take tiles of
// their XCD's queue until it is empty: in the dynamic mode the next free position (through
// counters), in the static mode every R-th position from their own rank (R resident workgroups
// per XCD).  Which workgroup runs which tile decides nothing: every slot is computed as in the
// one-launch sweep.
constexpr uint32_t kQueueTile = kQueueTileSlots;
constexpr uint32_t kQueueBuckets = 512;
constexpr uint32_t kQueueThreads = 1024;

// Per tile: the sum of its slots' neighbour counts (one wave per tile).
__global__ __launch_bounds__(256) void k_tile_cost(DeviceState d, uint32_t ntiles,
                                                   uint32_t* __restrict__ cost) {
    const uint32_t tile = blockIdx.x * 4u + (threadIdx.x >> 6);
    if (tile >= ntiles) return;  // whole waves
    uint32_t c = 0;
    for (uint32_t k = __lane_id(); k < kQueueTile; k += 64u) {
        const uint32_t s = tile * kQueueTile + k;
        if (s < d.nslots) c += d.cntW[s];
    }
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, 64);
    if (__lane_id() == 0) cost[tile] = c;
}

// One workgroup per XCD x: its tiles [x * T8, min((x + 1) * T8, ntiles)) by cost class, heaviest
// first (a counting sort over kQueueBuckets classes of cost >> shift; the order within a class is
// whatever the LDS atomics give), their number, and the XCD's pass counters cleared.
__global__ __launch_bounds__(kQueueThreads) void k_tile_queue(const uint32_t* __restrict__ cost,
                                                             uint32_t ntiles, uint32_t T8,
                                                             uint32_t shift, uint32_t* __restrict__ queue,
                                                             uint32_t* __restrict__ qcount,
                                                             uint32_t* __restrict__ heads,
                                                             uint32_t passes) {
    __shared__ uint32_t start[kQueueBuckets];
    __shared__ uint32_t wsum[kQueueThreads / 64];
    const uint32_t x = blockIdx.x, tid = threadIdx.x, lane = __lane_id(), wave = tid >> 6;
    const uint32_t t0 = x * T8, t1 = min(t0 + T8, ntiles);
    for (uint32_t k = tid; k < kQueueBuckets; k += kQueueThreads) start[k] = 0u;
    for (uint32_t k = tid; k < passes * kQueueSubs; k += kQueueThreads)
        heads[(((size_t)(k / kQueueSubs) * kXcds + x) * kQueueSubs + k % kQueueSubs) * kQueueHeadStride] = 0u;
    __syncthreads();
    for (uint32_t t = t0 + tid; t < t1; t += kQueueThreads)
        atomicAdd(&start[min(cost[t] >> shift, kQueueBuckets - 1u)], 1u);
    __syncthreads();
    // exclusive prefix in descending class order: thread r < kQueueBuckets holds class B - 1 - r
    const uint32_t v = tid < kQueueBuckets ? start[kQueueBuckets - 1u - tid] : 0u;
    uint32_t inc = v;
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(inc, off, 64);
        if ((int)lane >= off) inc += y;
    }
    if (lane == 63u) wsum[wave] = inc;
    __syncthreads();
    uint32_t base = 0;
    for (uint32_t w = 0; w < wave; ++w) base += wsum[w];
    __syncthreads();
    if (tid < kQueueBuckets) start[kQueueBuckets - 1u - tid] = base + inc - v;
    __syncthreads();
    for (uint32_t t = t0 + tid; t < t1; t += kQueueThreads) {
        const uint32_t pos = atomicAdd(&start[min(cost[t] >> shift, kQueueBuckets - 1u)], 1u);
        queue[t0 + pos] = t;
    }
    if (tid == 0) qcount[x] = t1 > t0 ? t1 - t0 : 0u;
}

// Counter of sub-queue `sub` of XCD x in pass `pass` (the dynamic mode).
__device__ __forceinline__ uint32_t* queue_head(const DeviceState& d, uint32_t pass, uint32_t x, uint32_t sub) {
    return d.heads + (((size_t)pass * kXcds + x) * kQueueSubs + sub) * kQueueHeadStride;
}

// The persistent loop: workgroup b serves XCD b % 8 (where the hardware places it); f(slot) runs
// once per thread and tile.  Static: rank r = b / 8 of R takes positions r, r + R, ...  Dynamic:
// the positions sub + 8 m form eight sub-queues (one counter each, so that no single counter
// takes every request); the workgroup takes the next m of sub-queue (b / 8) % 8 until it is empty,
// then of the seven others in turn.  Every workgroup leaves once each sub-queue is empty.
template <class F>
__device__ __forceinline__ void queue_loop(const DeviceState& d, uint32_t pass, uint32_t& sq, F f) {
    const uint32_t x = blockIdx.x % kXcds;
    const uint32_t n = d.qcount[x];
    const uint32_t* q = d.queue + (size_t)x * d.queueT8;
    if (d.queueMode == 2) {
        const uint32_t R = gridDim.x / kXcds;
        for (uint32_t k = blockIdx.x / kXcds; k < n; k += R) f(q[k] * kQueueTile + threadIdx.x);
        return;
    }
    const uint32_t sub0 = (blockIdx.x / kXcds) % kQueueSubs;
    for (uint32_t u = 0; u < kQueueSubs; ++u) {
        const uint32_t sub = (sub0 + u) % kQueueSubs;
        const uint32_t len = n > sub ? (n - sub + kQueueSubs - 1u) / kQueueSubs : 0u;
        uint32_t* head = queue_head(d, pass, x, sub);
        for (;;) {
            if (threadIdx.x == 0) sq = atomicAdd(head, 1u);
            __syncthreads();
            const uint32_t m = sq;
            __syncthreads();  // every thread has read sq before thread 0 takes the next position
            if (m >= len) break;
            f(q[sub + kQueueSubs * m] * kQueueTile + threadIdx.x);
        }
    }
}

template <bool kFast, bool kBnd>
__global__ __launch_bounds__(kQueueTile) void k_density_lambda_queue(DeviceState d, SphParams P,
                                                                     const float4* __restrict__ Xs,
                                                                     uint32_t pass) {
    __shared__ uint32_t sq;
    queue_loop(d, pass, sq, [&](uint32_t t) { density_lambda_slot<kQueueTile, kFast, kBnd>(d, P, Xs, -1, 0, t); });
}

template <bool kFinal, bool kFast, bool kBnd>
__global__ __launch_bounds__(kQueueTile) __attribute__((amdgpu_waves_per_eu(8)))
void k_delta_correct_queue(DeviceState d, SphParams P, StepParams S,
                                                                    const float4* __restrict__ XsIn,
                                                                    float4* __restrict__ XsOut, uint32_t pass) {
    __shared__ uint32_t sq;
    queue_loop(d, pass, sq, [&](uint32_t t) {
        delta_correct_slot<kQueueTile, kFinal, true, kFast, kBnd>(d, P, S, XsIn, XsOut, nullptr, 0, t);
    });
}

template <bool kFast>
__global__ __launch_bounds__(kQueueTile) void k_vorticity_queue(DeviceState d, SphParams P, uint32_t pass) {
    __shared__ uint32_t sq;
    queue_loop(d, pass, sq, [&](uint32_t t) { vorticity_slot<kFast>(d, P, t); });
}

template <bool kFast>
__global__ __launch_bounds__(kQueueTile) void k_confinement_queue(DeviceState d, SphParams P, StepParams S,
                                                                  uint32_t pass) {
    __shared__ uint32_t sq;
    queue_loop(d, pass, sq, [&](uint32_t t) { confinement_slot<kFast>(d, P, S, t); });
}

__global__ __launch_bounds__(kQueueTile) void k_xsph_queue(DeviceState d, SphParams P, uint32_t pass) {
    __shared__ uint32_t sq;
    queue_loop(d, pass, sq, [&](uint32_t t) { xsph_slot(d, P, t); });
}

// ---- lane groups: L lanes per particle, for scenes too small to fill the chip ------------------
// Thread T of a lane-group launch works on particle T / L (physical order).  A round takes 4 L list
// entries (32 with 16 lanes): lane r loads its entries' chunk and gathers, computes their terms and
// stores them in its group's rows of LDS, one row per sum; then lane c alone adds row c in entry
// order.  Each sum is therefore the one-lane sweep's, term for term and in list order.  Entries past
// the list's end contribute +0: no sum here starts at or reaches -0 (each starts at +0 or a positive
// value, and x + (-x) rounds to +0), so adding +0 changes nothing.
// Bound by one chain of dependent loads (count and list chunk, then gathers), the 4 L adds of a round
// (4 cycles each, the sums side by side in different lanes) and the launch itself.
// Plain steps only (no learned gate, no residual check), in the physical order.
template <int L>
struct LaneGroup {
    static_assert(L >= 2 && L <= 16 && (L & (L - 1)) == 0, "2, 4, 8 or 16");
    static constexpr int kEntries = L == 16 ? 2 : 4;          // list entries per lane and round
    static constexpr uint32_t kRound = (uint32_t)(L * kEntries);
    // floats of a row: 4 more than a round, so that the rows read together start on different banks
    static constexpr uint32_t kRow = kRound + 4u;
    uint32_t i;     // particle slot
    uint32_t r;     // lane within the group
    uint32_t base;  // first lane of the group within the wave
};

constexpr int kGroupBlock = 256;

template <int L>
__device__ __forceinline__ LaneGroup<L> lane_group() {
    const uint32_t T = xcd_slot<kGroupBlock, L>();
    return {T / (uint32_t)L, T % (uint32_t)L, __lane_id() & ~(uint32_t)(L - 1)};
}

// NA sums of a group: lane r keeps sums r, r + L, ...
template <int L, int NA>
struct GroupSums {
    static constexpr int kMine = (NA + L - 1) / L;
    float s[kMine];
    float* rows;  // the group's NA rows

    // start: sum 0's first value (the others start at 0)
    __device__ __forceinline__ GroupSums(const LaneGroup<L>& g, float start, float* lds) {
        rows = lds + (threadIdx.x / (uint32_t)L) * (NA * LaneGroup<L>::kRow);
#pragma unroll
        for (int q = 0; q < kMine; ++q) s[q] = q == 0 && g.r == 0u ? start : 0.0f;
    }
    // t[u][c]: this lane's terms of sum c, entries r * kEntries + u of the round
    __device__ __forceinline__ void add(const LaneGroup<L>& g, const float (&t)[LaneGroup<L>::kEntries][NA]) {
        constexpr int E = LaneGroup<L>::kEntries;
        constexpr uint32_t kRow = LaneGroup<L>::kRow;
#pragma unroll
        for (int c = 0; c < NA; ++c) {
            float* const at = rows + (uint32_t)c * kRow + g.r * (uint32_t)E;
            if constexpr (E == 4)
                *reinterpret_cast<float4*>(at) = make_float4(t[0][c], t[1][c], t[2][c], t[3][c]);
            else
                *reinterpret_cast<float2*>(at) = make_float2(t[0][c], t[1][c]);
        }
        wave_lds_order();
#pragma unroll
        for (int q = 0; q < kMine; ++q) {
            const uint32_t c = g.r + (uint32_t)(q * L);
            const float4* const row = reinterpret_cast<const float4*>(rows + min(c, (uint32_t)NA - 1u) * kRow);
            float4 v[LaneGroup<L>::kRound / 4u];
#pragma unroll
            for (uint32_t m = 0; m < LaneGroup<L>::kRound / 4u; ++m) v[m] = row[m];
#pragma unroll
            for (uint32_t m = 0; m < LaneGroup<L>::kRound / 4u; ++m) s[q] = (((s[q] + v[m].x) + v[m].y) + v[m].z) + v[m].w;
        }
        wave_lds_order();
    }
    // sum c, in every lane of the group
    __device__ __forceinline__ float of(const LaneGroup<L>& g, int c) const {
        return __shfl(s[c / L], (int)(g.base + (uint32_t)(c % L)), 64);
    }
};

// A group's list: the particle's entry count and this lane's chunk of the first round, loaded without
// waiting for the count (the chunk lies inside the particle's row).
template <int L>
struct GroupList {
    const uint4* lp;
    uint32_t n;
    uint4 first;
};

template <int L>
__device__ __forceinline__ uint4 group_chunk(const uint4* __restrict__ lp, const LaneGroup<L>& g, uint32_t k0) {
    if constexpr (LaneGroup<L>::kEntries == 4) return lp[(size_t)((k0 >> 2) + g.r) * 64u];
    const uint2 e = *(reinterpret_cast<const uint2*>(lp + (size_t)((k0 >> 2) + (g.r >> 1)) * 64u) + (g.r & 1u));
    return make_uint4(e.x, e.y, 0u, 0u);
}

template <int L>
__device__ __forceinline__ GroupList<L> group_list(const DeviceState& d, const SphParams& P, const LaneGroup<L>& g) {
    GroupList<L> l;
    l.lp = d.nbr4 + list_base(g.i, P.maxN);
    l.n = d.cnt[g.i];  // 0 in the padding slots past a scene's end
    const uint32_t chunk = g.r * (uint32_t)LaneGroup<L>::kEntries / 4u;
    l.first = chunk < list_chunks(P.maxN) ? group_chunk(l.lp, g, 0u) : make_uint4(0u, 0u, 0u, 0u);
    return l;
}

// Adds the terms of every list entry to the sums.
template <int L, int NA, class T, class Load, class Term>
__device__ __forceinline__ void walk_split(const GroupList<L>& l, const LaneGroup<L>& g, GroupSums<L, NA>& sums,
                                           Load load, Term term) {
    constexpr int E = LaneGroup<L>::kEntries;
    uint4 ch = l.first;
    for (uint32_t k0 = 0; k0 < l.n; k0 += LaneGroup<L>::kRound) {
        const uint32_t k = k0 + g.r * (uint32_t)E;
        const uint32_t e[4] = {ch.x, ch.y, ch.z, ch.w};
        T v[E];
#pragma unroll
        for (int u = 0; u < E; ++u) v[u] = load(k + (uint32_t)u < l.n ? e[u] : g.i);  // past the end: discarded
        if (k + LaneGroup<L>::kRound < l.n) ch = group_chunk(l.lp, g, k0 + LaneGroup<L>::kRound);
        float t[E][NA];
#pragma unroll
        for (int u = 0; u < E; ++u) {
            term(v[u], t[u]);
            const bool in = k + (uint32_t)u < l.n;
#pragma unroll
            for (int c = 0; c < NA; ++c) t[u][c] = in ? t[u][c] : 0.0f;
        }
        sums.add(g, t);
    }
}

template <int L, int NA>
constexpr uint32_t group_lds_floats() {
    return (uint32_t)(kGroupBlock / L * NA) * LaneGroup<L>::kRow;
}

// The wall samples of the group's particle, in the order of boundary_visit: each plane's window is
// one row-major stream of candidates, a round of them at a time; a candidate that does not count adds
// +0.  sums: the samples' density and gradient.
template <int L, bool kFast>
__device__ __forceinline__ void boundary_split(const SphParams& P, f3 xi, const LaneGroup<L>& g, GroupSums<L, 4>& sums) {
    constexpr int E = LaneGroup<L>::kEntries;
    const BoundaryDev& B = P.bd;
    boundary_windows(B, xi.x, xi.y, xi.z, P.h, P.h2, [&](auto wall, int l, const BoundaryWindow& win) {
        const uint32_t nc = (uint32_t)(win.c1 - win.c0 + 1), total = (uint32_t)(win.b1 - win.b0 + 1) * nc;
        for (uint32_t k0 = 0; k0 < total; k0 += LaneGroup<L>::kRound) {
            float t[E][4];
#pragma unroll
            for (int u = 0; u < E; ++u) {
                const uint32_t k = k0 + g.r * (uint32_t)E + (uint32_t)u, row = k / nc;
                float sep[3], d2;
                t[u][0] = t[u][1] = t[u][2] = t[u][3] = 0.0f;
                if (k < total && boundary_sample<decltype(wall)::value>(B, xi.x, xi.y, xi.z, P.h2, l, win.b0 + (int)row,
                                                                        win.c0 + (int)(k - row * nc), sep, d2)) {
                    const float psi = B.psi[boundary_index<decltype(wall)::value>(B, l, win.b0 + (int)row,
                                                                                  win.c0 + (int)(k - row * nc))];
                    const f3 gr = psi * grad_or_zero<kFast>(f3{sep[0], sep[1], sep[2]}, d2, P);
                    t[u][0] = psi * poly6_of<kFast>(d2, P);
                    t[u][1] = gr.x; t[u][2] = gr.y; t[u][3] = gr.z;
                }
            }
            sums.add(g, t);
        }
    });
}

template <int L, bool kFast, bool kBnd>
__device__ __forceinline__ void density_lambda_group_slots(const DeviceState& d, const SphParams& P, const float4* __restrict__ Xs, float* lds) {
    const LaneGroup<L> g = lane_group<L>();
    if (g.i >= d.nslots) return;  // whole groups
    const GroupList<L> list = group_list<L>(d, P, g);
    const SceneDev& sc = scene_of(d, g.i);
    const float4 xi4 = Xs[g.i];
    const f3 xi = make3(xi4);
    const float negInv = -P.invRest;
    // rho, grad_i C (x, y, z), sum |grad_j C|^2
    GroupSums<L, 5> sums(g, xi4.w * P.w0, lds);
    walk_split<L, 5, float4>(
        list, g, sums, [&](uint32_t j) { return ld(Xs, j); },
        [&](const float4& xj4, float (&t)[5]) {
            f3 sep = xi - make3(xj4);
            float d2 = dot3(sep, sep);
            f3 gr = grad_or_zero<kFast>(sep, d2, P);
            if (kFast) {
                t[0] = poly6_bounded(d2, P);
                t[1] = gr.x; t[2] = gr.y; t[3] = gr.z;
                f3 gj = negInv * gr;
                t[4] = dot3(gj, gj);
            } else {
                t[0] = xj4.w * poly6(d2, P);
                f3 mg = xj4.w * gr;
                t[1] = mg.x; t[2] = mg.y; t[3] = mg.z;
                f3 gj = (negInv * xj4.w) * gr;
                t[4] = dot3(gj, gj);
            }
        });
    float rho = sums.of(g, 0);
    f3 gi{sums.of(g, 1), sums.of(g, 2), sums.of(g, 3)};
    const float sum = sums.of(g, 4);
    const bool writes = g.r == 0u && g.i < sc.end;
    if (kBnd) {
        const bool near = g.i < sc.end && boundary_near(P.bd, xi.x, xi.y, xi.z, P.h2);
        float rb = 0.0f;
        f3 gb{0.0f, 0.0f, 0.0f};
        if (near) {
            GroupSums<L, 4> wall(g, 0.0f, lds);
            // the rows of its own group again: a group's rows of four sums lie inside its rows of five
            wall.rows = sums.rows;
            boundary_split<L, kFast>(P, xi, g, wall);
            rb = wall.of(g, 0);
            gb = f3{wall.of(g, 1), wall.of(g, 2), wall.of(g, 3)};
            if (writes) d.Bg[g.i] = make_float4(gb.x, gb.y, gb.z, 0.0f);
        }
        rho = rho + rb;
        gi = gi + gb;
    }
    if (!writes) return;
    gi = gi * P.invRest;
    const float C = rho * P.invRest - 1.0f;
    d.dens[g.i] = rho;
    const float lam = -C / ((sum + dot3(gi, gi)) + P.relax);
    d.lam[g.i] = lam;
    if (kFast) d.W[g.i] = make_float4(xi.x, xi.y, xi.z, lam);
}

template <int L, int kFast, bool kBnd>
__global__ __launch_bounds__(kGroupBlock) void k_density_lambda_group(DeviceState d, SphParams P, const float4* __restrict__ Xs) {
    __shared__ float4 lds[group_lds_floats<L, 5>() / 4u];
    by_masses<kFast>(d, [&](auto fast) {
        density_lambda_group_slots<L, decltype(fast)::value, kBnd>(d, P, Xs, reinterpret_cast<float*>(lds));
    });
}

template <int L, bool kFinal, bool kFast, bool kBnd>
__device__ __forceinline__ void delta_correct_group_slots(const DeviceState& d, const SphParams& P, const StepParams& S,
    const float4* __restrict__ XsIn, float4* __restrict__ XsOut, float* lds) {
    const LaneGroup<L> g = lane_group<L>();
    if (g.i >= d.nslots) return;
    const GroupList<L> list = group_list<L>(d, P, g);
    const SceneDev& sc = scene_of(d, g.i);
    const float4 xi4 = XsIn[g.i];
    const f3 xi = make3(xi4);
    const float li = d.lam[g.i];
    FinishIn in{};
    if (kFinal) in = finish_in(d, g.i);
    const Recip Rdq = recip(P.wdq);
    GroupSums<L, 3> sums(g, 0.0f, lds);
    walk_split<L, 3, XLam>(
        list, g, sums,
        [&](uint32_t j) {
            if (kFast) {
                const float4 a = ld(d.W, j);
                return XLam{a, a.w};
            }
            return XLam{ld(XsIn, j), ld(d.lam, j)};
        },
        [&](const XLam& nb, float (&t)[3]) {
            f3 sep = xi - make3(nb.x);
            float d2 = dot3(sep, sep);
            float coef = li + nb.lam;
            if (P.corrOn) {
                const float w = poly6_of<kFast>(d2, P);
                const float q = kFast ? corr_by_division(w, div_by(w, Rdq.b, Rdq.r), Rdq) : div_rn(w, Rdq);
                coef = coef + P.negCorrK * corr_pow(q, P);
            }
            f3 gr = grad_or_zero<kFast>(sep, d2, P);
            const f3 u = kFast ? coef * gr : (coef * nb.x.w) * gr;
            t[0] = u.x; t[1] = u.y; t[2] = u.z;
        });
    f3 dp{sums.of(g, 0), sums.of(g, 1), sums.of(g, 2)};
    if (g.r != 0u || g.i >= sc.end) return;
    if (kBnd) {  // lambda_i times the boundary gradient sum of the density pass (same x*)
        f3 gb{0.0f, 0.0f, 0.0f};
        if (boundary_near(P.bd, xi.x, xi.y, xi.z, P.h2)) gb = make3(d.Bg[g.i]);
        dp = dp + li * gb;
    }
    const f3 q = correct_position(xi, dp, P, sc);
    if (!kFinal) {
        XsOut[g.i] = make_float4(q.x, q.y, q.z, xi4.w);
        return;
    }
    finish_step<true>(d, S, sc, g.i, xi4, in, q, dp);
}

template <int L, bool kFinal, int kFast, bool kBnd>
__global__ __launch_bounds__(kGroupBlock) void k_delta_correct_group(DeviceState d, SphParams P, StepParams S,
    const float4* __restrict__ XsIn, float4* __restrict__ XsOut) {
    __shared__ float4 lds[group_lds_floats<L, 3>() / 4u];
    by_masses<kFast>(d, [&](auto fast) {
        delta_correct_group_slots<L, kFinal, decltype(fast)::value, kBnd>(d, P, S, XsIn, XsOut, reinterpret_cast<float*>(lds));
    });
}

template <int L, bool kFast>
__device__ __forceinline__ void vorticity_group_slots(const DeviceState& d, const SphParams& P, float* lds) {
    const LaneGroup<L> g = lane_group<L>();
    if (g.i >= d.nslots) return;
    const GroupList<L> list = group_list<L>(d, P, g);
    const SceneDev& sc = scene_of(d, g.i);
    const f3 xi = make3(d.X[g.i]);
    const f3 vi = make3(d.V[g.i]);
    GroupSums<L, 3> sums(g, 0.0f, lds);
    walk_split<L, 3, XV>(
        list, g, sums, [&](uint32_t j) { return XV{ld(d.X, j), ld(d.V, j)}; },
        [&](const XV& nb, float (&t)[3]) {
            f3 vij = make3(nb.v) - vi;
            f3 sep = xi - make3(nb.x);
            const f3 c = cross3(vij, grad_or_zero<kFast>(sep, dot3(sep, sep), P));
            const f3 u = (kFast ? -1.0f : -nb.x.w) * c;
            t[0] = u.x; t[1] = u.y; t[2] = u.z;
        });
    const f3 w{sums.of(g, 0), sums.of(g, 1), sums.of(g, 2)};
    if (g.r != 0u || g.i >= sc.end) return;
    const float wl = length3(w);
    d.W[g.i] = make_float4(w.x, w.y, w.z, wl);
    d.XsB[g.i] = make_float4(xi.x, xi.y, xi.z, wl);
}

template <int L, int kFast>
__global__ __launch_bounds__(kGroupBlock) void k_vorticity_group(DeviceState d, SphParams P) {
    __shared__ float4 lds[group_lds_floats<L, 3>() / 4u];
    by_masses<kFast>(d, [&](auto fast) {
        vorticity_group_slots<L, decltype(fast)::value>(d, P, reinterpret_cast<float*>(lds));
    });
}

template <int L, bool kFast>
__device__ __forceinline__ void confinement_group_slots(const DeviceState& d, const SphParams& P, const StepParams& S, float* lds) {
    const LaneGroup<L> g = lane_group<L>();
    if (g.i >= d.nslots) return;
    const GroupList<L> list = group_list<L>(d, P, g);
    const SceneDev& sc = scene_of(d, g.i);
    const float4 xi4 = d.X[g.i];
    const f3 xi = make3(xi4);
    const float4 wi = d.W[g.i], vi = d.V[g.i];
    const float rho = d.dens[g.i];
    GroupSums<L, 3> sums(g, 0.0f, lds);
    walk_split<L, 3, XW>(
        list, g, sums, [&](uint32_t j) { return XW{ld(d.XsB, j), kFast ? 1.0f : ld(d.X, j).w}; },
        [&](const XW& nb, float (&t)[3]) {
            float diff = wi.w - nb.x.w;
            f3 sep = xi - make3(nb.x);
            const f3 gr = grad_or_zero<kFast>(sep, dot3(sep, sep), P);
            const f3 u = (kFast ? diff : nb.w * diff) * gr;
            t[0] = u.x; t[1] = u.y; t[2] = u.z;
        });
    const f3 eta{sums.of(g, 0), sums.of(g, 1), sums.of(g, 2)};
    if (g.r != 0u || g.i >= sc.end) return;
    confine_finish(d, P, S, g.i, xi4.w, wi, vi, eta, rho);
}

template <int L, int kFast>
__global__ __launch_bounds__(kGroupBlock) void k_confinement_group(DeviceState d, SphParams P, StepParams S) {
    __shared__ float4 lds[group_lds_floats<L, 3>() / 4u];
    by_masses<kFast>(d, [&](auto fast) {
        confinement_group_slots<L, decltype(fast)::value>(d, P, S, reinterpret_cast<float*>(lds));
    });
}

template <int L>
__global__ __launch_bounds__(kGroupBlock) void k_xsph_group(DeviceState d, SphParams P) {
    __shared__ float4 lds[group_lds_floats<L, 3>() / 4u];
    const LaneGroup<L> g = lane_group<L>();
    if (g.i >= d.nslots) return;
    const GroupList<L> list = group_list<L>(d, P, g);
    const SceneDev& sc = scene_of(d, g.i);
    const f3 xi = make3(d.X[g.i]);
    const f3 vi = make3(d.Vc[g.i]);
    GroupSums<L, 3> sums(g, 0.0f, reinterpret_cast<float*>(lds));
    walk_split<L, 3, XV>(
        list, g, sums, [&](uint32_t j) { return XV{ld(d.X, j), ld(d.Vc, j)}; },
        [&](const XV& nb, float (&t)[3]) {
            f3 vij = make3(nb.v) - vi;
            f3 sep = xi - make3(nb.x);
            float w = poly6(dot3(sep, sep), P);
            const f3 u = (nb.v.w * vij) * w;
            t[0] = u.x; t[1] = u.y; t[2] = u.z;
        });
    const f3 dv{sums.of(g, 0), sums.of(g, 1), sums.of(g, 2)};
    if (g.r != 0u || g.i >= sc.end) return;
    f3 vn = vi + P.visc * dv;
    d.V[g.i] = make_float4(vn.x, vn.y, vn.z, 0.0f);
}

// Density at the current positions over every particle within h, each counted once: the walk of
// k_neighbours with the hashing cell size, each distinct bucket of the stencil visited once (no
// duplicates from stencil hash collisions) and no neighbour cap.  Accumulates, per scene, the
// maximum and the sum of max(0, rho / rho0 - 1) (the density-constraint error).
template <int BS>
__global__ __launch_bounds__(BS) void k_density_probe(DeviceState d, SphParams P,
                                                          float* __restrict__ rhoOut,
                                                          unsigned int* __restrict__ errMaxBits,
                                                          double* __restrict__ errSum) {
    const uint32_t i = xcd_slot<BS>();
    float err = 0.0f;
    uint32_t scene = 0;
    bool active = false;
    if (i < d.nslots) {
        scene = d.chunkScene[i >> 8];
        const SceneDev& sc = d.scenes[scene];
        if (i < sc.end) {
            active = true;
            const uint32_t self = d.lidT[i];
            const float4 xi4 = d.XsA[i];
            const f3 xi = make3(xi4);
            int cx, cy, cz;
            discretize(xi, P.cellHash, cx, cy, cz);
            float rho = xi4.w * P.w0;
            uint32_t hs[27];
#pragma unroll
            for (int q = 0; q < 27; ++q)
                hs[q] = cell_hash((int)((uint32_t)cx + (uint32_t)(q / 9 - 1)),
                                  (int)((uint32_t)cy + (uint32_t)((q / 3) % 3 - 1)),
                                  (int)((uint32_t)cz + (uint32_t)(q % 3 - 1)), sc);
#pragma unroll
            for (int q = 0; q < 27; ++q) {
                bool dup = false;
#pragma unroll
                for (int r = 0; r < q; ++r) dup |= hs[r] == hs[q];
                uint4 e;
                if (dup || !table_find(d.table, sc, hs[q], e)) continue;
                const int32_t shift = (int32_t)e.z - (int32_t)e.x;
                for (uint32_t m = e.x; m < e.y; ++m) {
                    if (m == self) continue;
                    float4 xk = ld(d.XsA, e.w ? (uint32_t)((int32_t)m + shift) : ld(d.physT, m));
                    f3 sep = xi - make3(xk);
                    float d2 = dot3(sep, sep);
                    if (d2 < P.h2) rho = rho + xk.w * poly6(d2, P);
                }
            }
            if (rhoOut) rhoOut[self] = rho;
            err = fmaxf(0.0f, rho * P.invRest - 1.0f);
        }
    }
    // one atomic per wave (a wave never spans two scenes: scenes start 256-aligned)
    float m = err;
    double sum = err;
    for (int off = 32; off > 0; off >>= 1) {
        m = fmaxf(m, __shfl_down(m, off, 64));
        sum += __shfl_down(sum, off, 64);
    }
    const uint64_t any = __ballot(active);
    const uint32_t s0 = __shfl(scene, 0, 64);
    if (__lane_id() == 0 && any) {
        atomicMax(&errMaxBits[s0], __float_as_uint(m));  // non-negative floats order as integers
        atomicAdd(&errSum[s0], sum);
    }
}

inline unsigned grid(uint32_t n) { return (n + kBlock - 1) / kBlock; }
// Neighbour kernels: a whole number of workgroups of bs threads per XCD.
inline unsigned grid_xcd(uint32_t n, int bs) {
    const unsigned g = (n + (unsigned)bs - 1) / (unsigned)bs;
    return (g + kXcds - 1) / kXcds * kXcds;
}

#define AKUA_BY_BLOCK(bs, CALL)         \
    do {                                \
        if ((bs) == 128) {              \
            constexpr int BS = 128;     \
            CALL;                       \
        } else if ((bs) == 512) {       \
            constexpr int BS = 512;     \
            CALL;                       \
        } else {                        \
            constexpr int BS = 256;     \
            CALL;                       \
        }                               \
    } while (0)

// Lane-group launches: L in {2, 4, 8, 16}, nslots * L threads.
#define AKUA_BY_LANES(lanes, CALL)      \
    do {                                \
        if ((lanes) == 2) {             \
            constexpr int L = 2;        \
            CALL;                       \
        } else if ((lanes) == 4) {      \
            constexpr int L = 4;        \
            CALL;                       \
        } else if ((lanes) == 8) {      \
            constexpr int L = 8;        \
            CALL;                       \
        } else {                        \
            constexpr int L = 16;       \
            CALL;                       \
        }                               \
    } while (0)

// The masses' form: K is P.fast.
#define AKUA_BY_FAST(CALL)       \
    do {                         \
        if (P.fast == 2) {       \
            constexpr int K = 2; \
            CALL;                \
        } else if (P.fast) {     \
            constexpr int K = 1; \
            CALL;                \
        } else {                 \
            constexpr int K = 0; \
            CALL;                \
        }                        \
    } while (0)

inline unsigned grid_lanes(uint32_t nslots, int lanes) {
    return grid_xcd(nslots * (uint32_t)lanes, kGroupBlock);
}

}  // namespace

void launch_fill_u32(hipStream_t st, uint32_t* p, uint32_t n, uint32_t v) {
    if (n) k_fill_u32<<<grid(n), kBlock, 0, st>>>(p, n, v);
}
void launch_clear_table(hipStream_t st, uint4* table, uint32_t n) {
    if (n) k_fill_u4<<<grid(n), kBlock, 0, st>>>(table, n, kEmptyKey);
}
void launch_predict_hash(hipStream_t st, const DeviceState& d, const SphParams& P,
                         const StepParams& S, bool layoutPrev, bool clearTable, const SortZeroSpans* zero) {
    const uint32_t predict = grid(d.nslots);
    const uint32_t clear = clearTable && d.tableTotal ? grid(d.tableTotal) : 0u;
    SortZeroSpans z{};
    if (zero) z = *zero;
    const uint32_t zeroBlocks = z.count ? kZeroBlocks : 0u;
    k_predict_hash<<<predict + clear + zeroBlocks + 1u, kBlock, 0, st>>>(d, P, S, layoutPrev, predict, clear, z);
}
void launch_cell_keys(hipStream_t st, const DeviceState& d, const SphParams& P,
                      const StepParams& S, bool keepLayout, bool layoutPrev) {
    if (keepLayout)
        k_cell_keys<true><<<grid(d.nslots), kBlock, 0, st>>>(d, P, S, false);
    else
        k_cell_keys<false><<<grid(d.nslots), kBlock, 0, st>>>(d, P, S, layoutPrev);
}
void launch_gather(hipStream_t st, const DeviceState& d, const SphParams& P, const StepParams& S,
                   bool carry, bool carryDelta, bool layoutPrev) {
    if (carryDelta)
        k_gather<true, true><<<grid(d.nslots), kBlock, 0, st>>>(d, P, S, layoutPrev);
    else if (carry)
        k_gather<true, false><<<grid(d.nslots), kBlock, 0, st>>>(d, P, S, layoutPrev);
    else
        k_gather<false, false><<<grid(d.nslots), kBlock, 0, st>>>(d, P, S, layoutPrev);
}
namespace {
// Workgroups for the crowded groups: each looks at 256 groups at least.
inline uint32_t crowd_blocks(uint32_t groups) { return std::min((groups + kBlock - 1u) / kBlock, kMaxCrowdBlocks); }
}  // namespace
void launch_order(hipStream_t st, const DeviceState& d, const SphParams& P, const StepParams& S, bool carry,
                  bool carryDelta) {
    const uint32_t count = grid(d.nslots);
    k_order_count<<<count + grid(d.tableTotal) + 1u, kBlock, 0, st>>>(d, P, S, count);
    k_order_place<<<(d.nslots + kOrderBlock - 1) / kOrderBlock, kOrderBlock, 0, st>>>(d);
    const uint32_t crowd = crowd_blocks(d.groups);
    if (carryDelta)
        k_order_rank<true, true><<<crowd + count, kBlock, 0, st>>>(d, S, crowd);
    else if (carry)
        k_order_rank<true, false><<<crowd + count, kBlock, 0, st>>>(d, S, crowd);
    else
        k_order_rank<false, false><<<crowd + count, kBlock, 0, st>>>(d, S, crowd);
}
void launch_tally(hipStream_t st, const DeviceState& d, const SphParams& P, const StepParams& S, bool carry,
                  bool carryDelta) {
    const uint32_t count = grid(d.nslots), prefix = d.tallyCount / kTallyBlock;
    k_tally_count<<<count + grid(d.tableTotal) + 1u, kBlock, 0, st>>>(d, P, S, count);
    k_tally_sum<<<prefix, kTallyThreads, 0, st>>>(d);
    k_tally_prefix<<<prefix, kTallyThreads, 0, st>>>(d);
    k_tally_place<<<count, kBlock, 0, st>>>(d);
    const uint32_t crowd = crowd_blocks(d.tallyGroups);
    if (carryDelta)
        k_tally_rank<true, true><<<crowd + count, kBlock, 0, st>>>(d, S, crowd);
    else if (carry)
        k_tally_rank<true, false><<<crowd + count, kBlock, 0, st>>>(d, S, crowd);
    else
        k_tally_rank<false, false><<<crowd + count, kBlock, 0, st>>>(d, S, crowd);
}
void launch_bucket_phys(hipStream_t st, const DeviceState& d) {
    k_bucket_phys<<<grid(d.nslots), kBlock, 0, st>>>(d);
}
namespace {
// Slots per wave of the list build: 64, or fewer in scenes that would leave the chip's 1,024 SIMDs
// without waves (a wave's runs are worked through one after another): us with 4 / 8 / 16 / 32 slots,
// 1,000 particles 9.0 / 11.5 / - / 25, 27,000 18.8 / 17.3 / - / 33, 100,000 - / 37 / 39 / 44.
template <int S, uint32_t kWaveRows>
void neighbours_wave_of(hipStream_t st, const DeviceState& d, const SphParams& P) {
    constexpr uint32_t kWaves = kWaveBuildBlock / 64;
    const unsigned lds = kWaves * wave_build_words<kWaveRows>(P.maxN) * (unsigned)sizeof(uint32_t);
    k_neighbours_wave<S, kWaveRows><<<grid_xcd(d.nslots, (int)kWaves * S), kWaveBuildBlock, lds, st>>>(d, P);
}
template <uint32_t kWaveRows>
void neighbours_wave(hipStream_t st, const DeviceState& d, const SphParams& P) {
    if (d.nslots >= (1u << 19))
        neighbours_wave_of<64, kWaveRows>(st, d, P);
    else if (d.nslots >= (1u << 17))
        neighbours_wave_of<32, kWaveRows>(st, d, P);
    else if (d.nslots >= (1u << 13))
        neighbours_wave_of<8, kWaveRows>(st, d, P);
    else
        neighbours_wave_of<4, kWaveRows>(st, d, P);
}
}  // namespace
void launch_neighbours(hipStream_t st, const DeviceState& d, const SphParams& P) {
    if (P.searchCells == 2)
        k_neighbours_fine<<<grid_xcd(d.nslots, kBlock), kBlock, 0, st>>>(d, P);
    else if (P.maxN <= kWaveBuildMaxN8)
        neighbours_wave<8>(st, d, P);
    else if (P.maxN <= kWaveBuildMaxN2)
        neighbours_wave<2>(st, d, P);
    else
        k_neighbours<<<grid_xcd(d.nslots, kBlock), kBlock, 0, st>>>(d, P);
}
template <int BS>
void density_lambda_bs(hipStream_t st, const DeviceState& d, const SphParams& P, const float4* Xs,
                       int residSlot, bool gated) {
    const unsigned nvb = grid_xcd(d.nslots, BS);
    const int g = gated ? 1 : 0;
    if (P.bd.on) {
        AKUA_BY_FAST((k_density_lambda<BS, K, true><<<nvb, BS, 0, st>>>(d, P, Xs, residSlot, g, nvb)));
    } else {
        AKUA_BY_FAST((k_density_lambda<BS, K, false><<<nvb, BS, 0, st>>>(d, P, Xs, residSlot, g, nvb)));
    }
}
void launch_density_lambda(hipStream_t st, const DeviceState& d, const SphParams& P,
                           const float4* Xs, int bs, int residSlot, bool gated, int lanes) {
    if (lanes > 1) {
        const unsigned g = grid_lanes(d.nslots, lanes);
#define AKUA_DLG(B) \
    AKUA_BY_FAST(AKUA_BY_LANES(lanes, (k_density_lambda_group<L, K, B><<<g, kGroupBlock, 0, st>>>(d, P, Xs))))
        if (P.bd.on) AKUA_DLG(true); else AKUA_DLG(false);
#undef AKUA_DLG
        return;
    }
    AKUA_BY_BLOCK(bs, (density_lambda_bs<BS>(st, d, P, Xs, residSlot, gated)));
}
void launch_balance(hipStream_t st, const DeviceState& d, const SphParams& P, uint32_t tile,
                    uint32_t* work, uint32_t* cntW, uint4* nbrW) {
    if (!d.nslots) return;
    const uint32_t blocks = (d.nslots + tile - 1) / tile;
    k_balance<<<blocks, kBalanceThreads, 0, st>>>(d, P, tile, work, cntW, nbrW);
}
void launch_count_sum(hipStream_t st, const DeviceState& d, unsigned long long* part, uint32_t blocks) {
    k_count_sum<<<blocks, 256, 0, st>>>(d, part);
}
void launch_features(hipStream_t st, const DeviceState& d, const SphParams& P, bool record, int bs) {
    AKUA_BY_BLOCK(bs, (k_features<BS><<<grid_xcd(d.nslots, BS), BS, 0, st>>>(d, P, record ? 1 : 0)));
}
void launch_gate(hipStream_t st, const DeviceState& d, uint32_t nscenes, int statistic,
                 float ratio, float tolerance) {
    k_resid_blocks<<<dim3(d.residBlocks, nscenes), kReduceBlock, 0, st>>>(d, 3);
    k_resid_reduce<<<nscenes, 64, 0, st>>>(d, 3, 1, statistic, ratio, tolerance);
}
void launch_resid_reduce(hipStream_t st, const DeviceState& d, uint32_t nscenes, int slotMask) {
    k_resid_blocks<<<dim3(d.residBlocks, nscenes), kReduceBlock, 0, st>>>(d, slotMask);
    k_resid_reduce<<<nscenes, 64, 0, st>>>(d, slotMask, 0, 0, 0.0f, 0.0f);
}
uint32_t resid_blocks_for(uint32_t maxSceneSlots) {
    const uint32_t waves = (maxSceneSlots + 63) / 64 + 1;  // +1: a scene may start mid-wave-row
    return std::max(1u, (waves + kResidWavesPerBlock - 1) / kResidWavesPerBlock);
}
void launch_targets(hipStream_t st, const DeviceState& d, const SphParams& P, const float4* XsLast) {
    k_targets<<<grid(d.nslots), kBlock, 0, st>>>(d, P, XsLast);
}
void launch_sample(hipStream_t st, const DeviceState& d, uint64_t seed, uint32_t count,
                   float* featOut, float* targOut) {
    if (count) k_sample<<<(count + 255) / 256, 256, 0, st>>>(d, seed, count, featOut, targOut);
}
template <int BS>
void delta_correct_bs(hipStream_t st, const DeviceState& d, const SphParams& P,
                      const StepParams& S, const float4* XsIn, float4* XsOut, bool final,
                      bool applyDelta, int gate, const float4* XsAlt) {
    const unsigned nvb = grid_xcd(d.nslots, BS);
    const unsigned g = nvb;
#define AKUA_DC(F, A, K, B) \
    k_delta_correct<BS, F, A, K, B><<<g, BS, 0, st>>>(d, P, S, XsIn, XsOut, XsAlt, gate, nvb)
    if (final && !applyDelta) {
        AKUA_DC(true, false, 0, false);  // a step without iterations
    } else if (P.bd.on) {
        if (final) AKUA_BY_FAST(AKUA_DC(true, true, K, true)); else AKUA_BY_FAST(AKUA_DC(false, true, K, true));
    } else if (final) {
        AKUA_BY_FAST(AKUA_DC(true, true, K, false));
    } else {
        AKUA_BY_FAST(AKUA_DC(false, true, K, false));
    }
#undef AKUA_DC
}
void launch_delta_correct(hipStream_t st, const DeviceState& d, const SphParams& P,
                          const StepParams& S, const float4* XsIn, float4* XsOut, bool final,
                          bool applyDelta, int bs, int gate, const float4* XsAlt, int lanes) {
    if (lanes > 1 && applyDelta) {
        const unsigned g = grid_lanes(d.nslots, lanes);
#define AKUA_DCG(F, B) \
    AKUA_BY_FAST(      \
        AKUA_BY_LANES(lanes, (k_delta_correct_group<L, F, K, B><<<g, kGroupBlock, 0, st>>>(d, P, S, XsIn, XsOut))))
        if (P.bd.on) {
            if (final) AKUA_DCG(true, true); else AKUA_DCG(false, true);
        } else {
            if (final) AKUA_DCG(true, false); else AKUA_DCG(false, false);
        }
#undef AKUA_DCG
        return;
    }
    if (lanes == kLanesShared && applyDelta) {
        const unsigned g = grid_xcd(d.nslots, kTailBlock);
        if (final)
            AKUA_BY_FAST((k_delta_correct_tail<true, K><<<g, kTailBlock, 0, st>>>(d, P, S, XsIn, XsOut)));
        else
            AKUA_BY_FAST((k_delta_correct_tail<false, K><<<g, kTailBlock, 0, st>>>(d, P, S, XsIn, XsOut)));
        return;
    }
    AKUA_BY_BLOCK(bs, (delta_correct_bs<BS>(st, d, P, S, XsIn, XsOut, final, applyDelta, gate,
                                            XsAlt)));
}
void launch_vorticity(hipStream_t st, const DeviceState& d, const SphParams& P, int bs, int lanes) {
    if (lanes > 1) {
        const unsigned g = grid_lanes(d.nslots, lanes);
        AKUA_BY_FAST(AKUA_BY_LANES(lanes, (k_vorticity_group<L, K><<<g, kGroupBlock, 0, st>>>(d, P))));
        return;
    }
    AKUA_BY_FAST(AKUA_BY_BLOCK(bs, (k_vorticity<BS, K><<<grid_xcd(d.nslots, BS), BS, 0, st>>>(d, P))));
}
void launch_confinement(hipStream_t st, const DeviceState& d, const SphParams& P,
                        const StepParams& S, int bs, int lanes) {
    if (lanes > 1) {
        const unsigned g = grid_lanes(d.nslots, lanes);
        AKUA_BY_FAST(AKUA_BY_LANES(lanes, (k_confinement_group<L, K><<<g, kGroupBlock, 0, st>>>(d, P, S))));
        return;
    }
    AKUA_BY_FAST(AKUA_BY_BLOCK(bs, (k_confinement<BS, K><<<grid_xcd(d.nslots, BS), BS, 0, st>>>(d, P, S))));
}
void launch_xsph(hipStream_t st, const DeviceState& d, const SphParams& P, int bs, int lanes) {
    if (lanes > 1) {
        const unsigned g = grid_lanes(d.nslots, lanes);
        AKUA_BY_LANES(lanes, (k_xsph_group<L><<<g, kGroupBlock, 0, st>>>(d, P)));
        return;
    }
    AKUA_BY_BLOCK(bs, (k_xsph<BS><<<grid_xcd(d.nslots, BS), BS, 0, st>>>(d, P)));
}
namespace {
// Workgroups of 256 threads that the device holds at once for `kernel`, per XCD (cached per
// kernel and device).
unsigned resident_per_xcd(const void* kernel) {
    static std::mutex mu;
    static std::map<std::pair<const void*, int>, unsigned> cache;
    auto check = [](hipError_t e, const char* what) {
        if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
    };
    int dev = 0;
    check(hipGetDevice(&dev), "hipGetDevice");
    std::lock_guard<std::mutex> lock(mu);
    const auto key = std::make_pair(kernel, dev);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    int perCu = 0, cus = 0;
    check(hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCu, kernel, (int)kQueueTile, 0),
          "hipOccupancyMaxActiveBlocksPerMultiprocessor");
    check(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev), "hipDeviceGetAttribute");
    const unsigned v = std::max(1u, (unsigned)std::max(perCu, 1) * (unsigned)std::max(cus, 1) / kXcds);
    cache.emplace(key, v);
    return v;
}
// The grid of a queued sweep: a multiple of 8 workgroups, no more per XCD than its queue holds.
template <class K>
unsigned queue_grid(K kernel, const DeviceState& d) {
    return kXcds * std::max(1u, std::min(resident_per_xcd(reinterpret_cast<const void*>(kernel)), d.queueT8));
}
}  // namespace

void launch_tile_queue(hipStream_t st, const DeviceState& d, const SphParams& P, uint32_t* cost,
                       uint32_t* queue, uint32_t* qcount, uint32_t* heads, uint32_t passes) {
    const uint32_t ntiles = (d.nslots + kQueueTile - 1) / kQueueTile;
    if (ntiles) k_tile_cost<<<(ntiles + 3) / 4, 256, 0, st>>>(d, ntiles, cost);
    // cost classes: the largest possible tile cost (256 full lists) spans kQueueBuckets classes
    const uint64_t maxCost = (uint64_t)kQueueTile * (uint64_t)std::max(P.maxN, 1);
    uint32_t shift = 0;
    while ((maxCost >> shift) >= kQueueBuckets) ++shift;
    k_tile_queue<<<kXcds, kQueueThreads, 0, st>>>(cost, ntiles, d.queueT8, shift, queue, qcount, heads, passes);
}
void launch_density_lambda_queue(hipStream_t st, const DeviceState& d, const SphParams& P,
                                 const float4* Xs, uint32_t pass) {
#define AKUA_DLQ(K, B) \
    k_density_lambda_queue<K, B><<<queue_grid(k_density_lambda_queue<K, B>, d), kQueueTile, 0, st>>>(d, P, Xs, pass)
    if (P.bd.on) {
        if (P.fast == 1) AKUA_DLQ(true, true); else AKUA_DLQ(false, true);
    } else {
        if (P.fast == 1) AKUA_DLQ(true, false); else AKUA_DLQ(false, false);
    }
#undef AKUA_DLQ
}
void launch_delta_correct_queue(hipStream_t st, const DeviceState& d, const SphParams& P,
                                const StepParams& S, const float4* XsIn, float4* XsOut, bool final,
                                uint32_t pass) {
#define AKUA_DCQ(F, K, B)                                                                             \
    k_delta_correct_queue<F, K, B><<<queue_grid(k_delta_correct_queue<F, K, B>, d), kQueueTile, 0, st>>>( \
        d, P, S, XsIn, XsOut, pass)
    if (P.bd.on) {
        if (final) {
            if (P.fast == 1) AKUA_DCQ(true, true, true); else AKUA_DCQ(true, false, true);
        } else {
            if (P.fast == 1) AKUA_DCQ(false, true, true); else AKUA_DCQ(false, false, true);
        }
    } else if (final) {
        if (P.fast == 1) AKUA_DCQ(true, true, false); else AKUA_DCQ(true, false, false);
    } else {
        if (P.fast == 1) AKUA_DCQ(false, true, false); else AKUA_DCQ(false, false, false);
    }
#undef AKUA_DCQ
}
void launch_vorticity_queue(hipStream_t st, const DeviceState& d, const SphParams& P, uint32_t pass) {
    if (P.fast == 1)
        k_vorticity_queue<true><<<queue_grid(k_vorticity_queue<true>, d), kQueueTile, 0, st>>>(d, P, pass);
    else
        k_vorticity_queue<false><<<queue_grid(k_vorticity_queue<false>, d), kQueueTile, 0, st>>>(d, P, pass);
}
void launch_confinement_queue(hipStream_t st, const DeviceState& d, const SphParams& P,
                              const StepParams& S, uint32_t pass) {
    if (P.fast == 1)
        k_confinement_queue<true><<<queue_grid(k_confinement_queue<true>, d), kQueueTile, 0, st>>>(d, P, S, pass);
    else
        k_confinement_queue<false><<<queue_grid(k_confinement_queue<false>, d), kQueueTile, 0, st>>>(d, P, S, pass);
}
void launch_xsph_queue(hipStream_t st, const DeviceState& d, const SphParams& P, uint32_t pass) {
    k_xsph_queue<<<queue_grid(k_xsph_queue, d), kQueueTile, 0, st>>>(d, P, pass);
}
void launch_density_probe(hipStream_t st, const DeviceState& d, const SphParams& P, float* rho,
                          unsigned int* errMaxBits, double* errSum) {
    k_density_probe<256><<<grid_xcd(d.nslots, 256), 256, 0, st>>>(d, P, rho, errMaxBits, errSum);
}

}  // namespace akua
