// The CWBVH traversal kernel (gfx950, wave64), its team tail and its launch
// templates.  trace.hip and trace_prefetch.hip instantiate them: the latter the
// launches with node prefetch, which are compiled with other flags.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <tuple>

#include "aogen.h"
#include "device_common.h"
#include "internal.h"

namespace cwk {

using namespace cwd;

static_assert(kStackCapacity == CWBVH_STACK_CAPACITY, "device and public stack capacities agree");


constexpr int kMaxBlock = 256;
constexpr int kWorkSlices = cw::kWorkSlices;
constexpr int kWorkStride = cw::kWorkStride;
constexpr int kWorkExited = cw::kWorkExited;
constexpr int kWorkOverflow = cw::kWorkOverflow;
constexpr int kWorkProfile = cw::kWorkProfile;
constexpr int kWorkDrained = cw::kWorkDrained;
constexpr int kWorkGroupExit = cw::kWorkGroupExit;

// Work distribution of the persistent grids (cwbvh_trace, bvh2_trace_persistent).
// The items (rays; in a batch, chunk indices) are split into `slices` contiguous
// ranges with one claim counter each.  Blocks are dispatched round-robin over the
// XCDs, so block b takes slice b % slices (its home) first, then the others.
//  * First claim without an atomic: wave i of the W_s waves whose home is
//    slice s owns [i * amount, (i + 1) * amount) of it outright, and the
//    counter hands out the slice from W_s * amount on.  Otherwise every wave
//    of the grid claims at once when the launch starts, and the claims queue
//    on eight counter lines.
//  * Drained mask: the first wave to find a slice dry sets its bit in one
//    word.  A wave that has run out of its home slice reads the word once and
//    skips the drained slices, instead of probing every counter with an
//    atomic at the end of the launch.
//  * Exit: blocks count their exits per home slice; the last block of a home
//    group counts on one word, and the last group resets everything, so no
//    line takes an atomic from every block.
//  * Splits: the host passes n = item_q * slices + item_r and the grid's
//    blocks = block_q * slices + block_r, so the claims divide nothing (a
//    64-bit division by a run-time value costs about 40 VALU instructions).
// Blocks whose home is slice s (blocks b with b mod slices = s).
__device__ __forceinline__ unsigned home_blocks(int s, unsigned block_q, unsigned block_r) {
    return block_q + ((unsigned)s < block_r ? 1u : 0u);
}

// First item of slice s: the first item_r slices hold item_q + 1 items, the
// others item_q.
__device__ __forceinline__ unsigned slice_begin(int s, unsigned item_q, unsigned item_r) {
    return (unsigned)s * item_q + min((unsigned)s, item_r);
}

// Slice-relative base of the wave's next claim of `amount` items from slice
// `sl` (>= the slice size when it has run dry).  `first`: the wave's first
// claim, from its home slice, with index `first_index` among that slice's
// waves.  The wave's first active lane does the memory work; the result is
// wave-uniform (scalar registers).
__device__ __forceinline__ unsigned slice_claim(unsigned* work, int sl, unsigned amount, bool first,
                                                unsigned first_index, unsigned block_q, unsigned block_r, int lane) {
    // 64-bit sums, saturated: a value past 2^32 - 1 reads as a dry slice
    if (first) return (unsigned)min((unsigned long long)first_index * amount, 0xFFFFFFFFull);
    unsigned base = 0;
    if (lane == __builtin_amdgcn_readfirstlane(lane)) base = atomicAdd(&work[sl * kWorkStride], amount);
    base = __builtin_amdgcn_readfirstlane(base);
    const unsigned long long static_items =
        (unsigned long long)home_blocks(sl, block_q, block_r) * (blockDim.x >> 6) * amount;
    return (unsigned)min(static_items + base, 0xFFFFFFFFull);
}

// Whether the first claims of slice sl's waves cover all its `size` items, so
// that nothing is left to claim from its counter.
__device__ __forceinline__ bool static_only(int sl, unsigned size, unsigned amount, unsigned block_q, unsigned block_r) {
    return (unsigned long long)home_blocks(sl, block_q, block_r) * (blockDim.x >> 6) * amount >= size;
}

// Marks slice `sl` drained and returns the drained mask as now known: one
// load, and an atomic only when the slice is not marked yet.
__device__ __forceinline__ unsigned mark_drained(unsigned* work, int sl, int lane) {
    unsigned m = 0;
    if (lane == __builtin_amdgcn_readfirstlane(lane)) {
        m = __hip_atomic_load(&work[kWorkDrained], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (!((m >> sl) & 1u)) m = atomicOr(&work[kWorkDrained], 1u << sl);
    }
    return __builtin_amdgcn_readfirstlane(m) | (1u << sl);
}

// Exit of a persistent block (all threads call it).  Every wave has consumed
// the result of its last claim before the barrier, so the claims are
// complete when the exit is counted; the last block out resets the counters
// for the next launch on the stream.
__device__ __forceinline__ void block_exit(unsigned* work, int total_blocks, int slices, unsigned block_q,
                                           unsigned block_r) {
    __syncthreads();
    if (threadIdx.x == 0) {
        const int g = (int)(blockIdx.x % (unsigned)slices);
        const unsigned prev = atomicAdd(&work[kWorkGroupExit + g * kWorkStride], 1u);
        if (prev == home_blocks(g, block_q, block_r) - 1u) {
            const unsigned groups = (unsigned)min(slices, total_blocks);
            const unsigned gprev = atomicAdd(&work[kWorkExited], 1u);
            if (gprev == groups - 1u) {
                for (int k = 0; k < kWorkSlices; ++k) {
                    atomicExch(&work[k * kWorkStride], 0u);
                    atomicExch(&work[kWorkGroupExit + k * kWorkStride], 0u);
                }
                atomicExch(&work[kWorkDrained], 0u);
                atomicExch(&work[kWorkExited], 0u);
            }
        }
    }
}

struct CwbvhParams {
    const float4* __restrict__ nodes;
    const float4* __restrict__ tris;
    const int* __restrict__ prim_map;
    const Ray4* __restrict__ rays;
    const int* __restrict__ order;
    float4* __restrict__ hits;
    const cw::BatchJob* __restrict__ jobs;
    unsigned* work;                 // fetch counters, exited waves, overflow (kWork*)
    unsigned long long* stats;      // {nodes, triangles}
    int n;                          // rays (single) or total chunks (multi)
    int slices;                     // single scene: contiguous ray ranges, one per XCD
    int persistent;                 // 0: each wave traces rays_per_wave rays, no refill
    int rays_per_wave;              // persistent 0: rays given to a wave, 1..64
    int num_jobs;
    int job_step;                   // batches: jobs per lane of the chunk search, ceil(num_jobs / 64)
    int stride;                     // float4 per node: 5 or 8
    int spread;                     // host side: nodes are spread nodes (SPREAD kernels)
    int lds_depth;
    int chunk;
    int idle_lanes;
    int idle_budget;
    int postpone_pct;
    int prim_id;
    int total_waves;
    int total_blocks;
    unsigned item_q, item_r;        // n = item_q * slices + item_r
    unsigned block_q, block_r;      // total_blocks = block_q * slices + block_r
    int spec_limit;                 // single scene: speculation_limit of its tree
    int lds_only;                   // host side: the tree's stack need fits lds_depth (LDS-only kernels)
    // SRC = kRaysFromSurfels: generate ray r from surfel r / rays_per_texel
    const float4* __restrict__ surf_pos;
    const float4* __restrict__ surf_nrm;
    const float* __restrict__ surf_rad;
    int rays_per_texel;
    float gen_tmin, gen_tmax;
    unsigned long long seed;
    unsigned* texel_hits;           // non-null: count hits per surfel instead of writing hits
    int streams;                    // host side: the scene is larger than the Infinity Cache
};

constexpr int kRaysFromBuffer = 0;
constexpr int kRaysFromSurfels = 1;

// Keeps an address in its registers until the first load from it has returned, so
// that the last load does not write its result over them.  Batches read their nodes
// and triangles through per-lane 64-bit pointers; where the compiler let the last
// load of a visit overwrite its own address, batches whose scenes stream from memory
// ran 5-7% slower with otherwise the same loop (32 scenes of 100 M triangles in all, 1
// M rays each, closest / any hit: 7.67 / 6.68 ms, with the address kept 7.20 / 6.22;
// the served requests of such scenes at saturation 3.77 and 4.0 Grays/s), and the
// more waves the more so.  It costs no register.
__device__ __forceinline__ void keep_address(const float4* p, float loaded) { asm volatile("" ::"v"(p), "v"(loaded)); }

__device__ __forceinline__ const float4* node_at(const float4* nodes, unsigned i, unsigned stride_sh) {
    return nodes + ((i << 2) + (i << stride_sh));
}

// Spread nodes (internal.h): the 128 B node's 16-byte slots exchanged by the
// node's index.  Slot s of node i sits at slot s XOR (i mod 8).  A load
// instruction of 64 lanes reads one slot of 64 nodes; at a 128 B stride all of
// them would sit in the same 16-byte column of their cache lines, and the L1
// serves such a load in 64 cycles, against 34 when the columns differ
// (measured with the lines in L1).
__device__ __forceinline__ unsigned spread_offset(unsigned i) { return (i << 7) | ((i & 7u) << 4); }

__device__ __forceinline__ const char* spread_at(const float4* nodes, unsigned offset, unsigned byte) {
    return reinterpret_cast<const char*>(nodes) + (offset ^ byte);
}

__device__ __forceinline__ float4 spread_slot(const float4* nodes, unsigned offset, unsigned slot) {
    return *reinterpret_cast<const float4*>(spread_at(nodes, offset, slot << 4));
}

// Quantized slab test of 4 children (one meta dword, one byte per child).
__device__ __forceinline__ unsigned child_hits4(unsigned meta4, unsigned lox, unsigned loy, unsigned loz,
                                                unsigned hix, unsigned hiy, unsigned hiz, float adjx, float adjy,
                                                float adjz, float origx, float origy, float origz, float tmin,
                                                float tmax, unsigned octinv4) {
    const unsigned is_inner4 = (meta4 & (meta4 << 1)) & 0x10101010u;
    const unsigned ones = is_inner4 >> 4;                 // 0x01 per inner child byte
    const unsigned inner_mask4 = (ones << 8) - ones;      // 0xFF per inner child byte
    const unsigned bit_index4 = (meta4 ^ (octinv4 & inner_mask4)) & 0x1F1F1F1Fu;
    const unsigned child_bits4 = (meta4 >> 5) & 0x07070707u;
    unsigned hitmask = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int sh = 8 * j;
        const float tnx = __builtin_fmaf((float)((lox >> sh) & 0xFFu), adjx, origx);
        const float tny = __builtin_fmaf((float)((loy >> sh) & 0xFFu), adjy, origy);
        const float tnz = __builtin_fmaf((float)((loz >> sh) & 0xFFu), adjz, origz);
        const float tfx = __builtin_fmaf((float)((hix >> sh) & 0xFFu), adjx, origx);
        const float tfy = __builtin_fmaf((float)((hiy >> sh) & 0xFFu), adjy, origy);
        const float tfz = __builtin_fmaf((float)((hiz >> sh) & 0xFFu), adjz, origz);
        // int-ordered combine with tmin/tmax as well: equal to fmaxf/fminf for
        // tmin, tmax >= +0 and non-NaN slabs, without NaN canonicalization ops
        const float cmin = imax2(imax3(tnx, tny, tnz), tmin);
        const float cmax = imin2(imin3(tfx, tfy, tfz), tmax);
        const unsigned bits = (child_bits4 >> sh) & 0xFFu;
        const unsigned idx = (bit_index4 >> sh) & 0xFFu;
        hitmask |= (cmin <= cmax) ? (bits << idx) : 0u;
    }
    return hitmask;
}

// Inner-loop schedules (cwbvh_trace_config.loop_mode).
//  kLoopGroup: per iteration one node visit, then every triangle of the
//    group it produced (the reference's order, :93-340), with optional
//    postponing of the triangle group.
//  kLoopInterleave: per iteration a lane either visits a node (when it holds
//    no triangles) or tests ONE triangle; the per-ray sequence of visits and
//    tests is the same as kLoopGroup, but a lane with a long triangle group no
//    longer holds the other 63 lanes in a triangle loop.
//  kLoopSpeculate: as kLoopInterleave, and a lane that holds triangles still
//    visits a node in the same iteration; the new node's triangle group is
//    pushed on the stack and tested later, so node visits keep every lane
//    with inner children busy.  With postpone_pct > 0 the wave also holds
//    back its triangle step until that share of its lanes hold triangles and
//    have no node to visit (or no lane can visit a node), so the step runs
//    with more lanes on.
//    A lane speculates only while its stack holds fewer than spec_limit
//    entries (capacity minus the tree's stack need), so the parked groups
//    never push the stack past its capacity.
//  loop_mode 3 (a per-wave queue of triangle tests run 64 at a time) is
//    refused by validate_config: its first GPU run faulted the device
//    together with another untested path, and the cause was not shown, so the
//    schedule was taken out.
//  kLoopInterleave lets a lane with a long triangle group stall less, in one of
//    three ways; all keep each ray's sequence of visits and tests, so hits are
//    those of kLoopGroup to the bit, ties included:
//    - any hit (kTwoGroups): a lane holds up to two triangle groups, so it
//      visits its next node while the first group waits.  Until its first
//      accepted triangle an any-hit ray's interval is constant, so a visit made
//      early finds what it would find later, and the groups are tested in the
//      order they were found.  33 M AO rays 1.92 -> 1.84 ms.
//    - closest hit, prefetch kernels (kLookAhead): one visit ahead, undone and
//      made again when the waiting group shortens the ray.  Node loads bound
//      these kernels, and a lane that waits has none in flight.  5 M-triangle
//      soup, 16.8 M rays: 11.18 -> 11.00 ms.  (Elsewhere a visit made twice
//      costs more than the wait: 33 M AO rays 2.11 -> 2.24 ms, batch 325 -> 358
//      us.  Not undone, visits ahead gave 2.03 ms, but a grazing ray whose
//      triangles tie could then report another one than in the other schedules,
//      depending on the rays it shares a wave with.)
//    - closest hit otherwise (kRepeatTriangles): the triangle step repeats while
//      kTriangleAgain lanes hold triangles.  1 M AO rays on a heightfield 146 us
//      without, 139.6 at 12 lanes, 139.7 at 9, 143 at 6, 154 at 3; 1920x1080
//      camera rays 332 / 328 / 329 / 336 / 356; 33 M AO rays 2.15 / 2.15 / 2.16
//      / 2.19 / 2.33 ms.
//    The prefetch kernels, whose scenes have the most triangle tests per visit,
//    also hold the triangle step back until kTriangleLanes lanes hold triangles
//    (with two groups, 5 M-triangle soup: 10.83 ms at 8 lanes, 11.10 at 1, 11.54
//    at 24; at 4 with look-ahead 1.6% slower than at 8).  The others do not (33 M
//    AO rays: 2.06 ms at 8, 2.05 at 1, 2.16 at 24).
constexpr int kTriangleLanes = 8;
constexpr int kTriangleAgain = 12;
constexpr int kLoopGroup = 0;
constexpr int kLoopInterleave = 1;
constexpr int kLoopSpeculate = 2;
constexpr int kLoopQueue = 3;

// Register budget (cwbvh_trace_config.occupancy).  The plain interleaved
// kernels (one scene, no counters, no prefetch) that read rays from a buffer are
// held to 6 waves: team_trace's code would lift them from 76 to 83 VGPRs, i.e. to
// 5; held, they take 77-78 and spill nothing.  Those that make rays from surfels
// take 84-89 (5 waves).  Both are also built for 7 waves (72 VGPRs; up to 1 and 7
// registers of cold state spilled), which traces launches of tens of millions of
// AO rays 3-5% faster and launches of a million rays 6-7% slower (more waves,
// each slower, lengthen the tail of a short launch).  The batch kernels (85-94) and
// the prefetch kernels (90-96), 5 waves both, stay unconstrained: at 7 waves they
// would spill 10 registers or more.
// The grouped kernel is built for 6 waves (76 VGPRs, nothing spilled) beside the
// free build (83: 5 waves): the former serves scenes that the cache holds, the
// latter those that stream from memory, where a sixth wave evicts more than it
// hides.  us, free / 6 waves: 1 M-triangle spheres, AO rays, closest hit, 1 M 254 /
// 242, 8 M 1449 / 1323; 5 M-triangle soup, 0.3 M rays 719 / 751, 16 M 14370 / 14773.
constexpr int kOccupancyAuto = 0;
constexpr int kOccupancyFree = 1;
constexpr int kOccupancy7 = 7;
// Launches that make their rays from surfels run 5 waves otherwise (same scene,
// any hit, 5 / 7 waves: 2.9 M rays 349 / 347 us, 4 M 470 / 459, 8.3 M 804 / 766;
// a 200 k-triangle heightfield 330 / 344, 438 / 444, 854 / 822).
constexpr long long kOccupancy7MinSurfelRays = 1ll << 22;

#ifndef CWBVH_TRACE_ATTR
#define CWBVH_TRACE_ATTR                        \
    __attribute__((amdgpu_waves_per_eu(TIGHT ? (LOOP == kLoopGroup ? 6 : 7) : \
                                       LOOP == kLoopInterleave && !STATS && !PREFETCH && SRC == 0 && !MULTI ? 6 : 1)))
#endif

// A wave whose pool is dry traces its last kLastRays rays with teams of lanes
// (team_trace): 4 lanes per ray, and 8 once 8 rays are left.
constexpr int kLastRays = 16;

// A value of the other lane of each pair, the other pair of each quad, and the
// other quad of each 8 lanes (DPP quad_perm [1,0,3,2], quad_perm [2,3,0,1],
// row_half_mirror): two (teams of 4) or three (teams of 8) steps of an
// associative, commutative operation leave its result over the team in all of
// its lanes.
constexpr int kDppPair = 0xB1, kDppQuad = 0x4E, kDppHalf = 0x141;
template <int CTRL>
__device__ __forceinline__ int team_swap(int v) {
    return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xF, 0xF, false);
}

template <int TEAM>
__device__ __forceinline__ unsigned team_or(unsigned v) {
    v |= (unsigned)team_swap<kDppPair>((int)v);
    v |= (unsigned)team_swap<kDppQuad>((int)v);
    if (TEAM == 8) v |= (unsigned)team_swap<kDppHalf>((int)v);
    return v;
}

// The lower (t, address) of two candidates.
template <int CTRL>
__device__ __forceinline__ void team_min_step(float& t, int& a) {
    const float ot = i2f(team_swap<CTRL>(f2i(t)));
    const int oa = team_swap<CTRL>(a);
    const bool take = ot < t || (ot == t && oa < a);
    t = take ? ot : t;
    a = take ? oa : a;
}

// One ray's traversal state, as cwbvh_trace holds it per lane.
struct RayState {
    float3 o, d;
    float tmin, tmax, idx, idy, idz;
    unsigned octinv;
    uint2 ng, tg, tg2;
    int sp, col, hit_addr, out_idx;   // col: the ray's stack column in LDS
    unsigned out_texel;
    float hu, hv;
    const float4* nodes;
    const float4* tris;
    float4* hits;
    const int* prim_map;
    unsigned stride_sh;
};

template <class T>
__device__ __forceinline__ T* shfl_ptr(T* p, int src) {
    return (T*)__shfl((unsigned long long)p, src);
}

template <int SRC, bool MULTI>
__device__ __forceinline__ void shfl_state(RayState& r, int src) {
    r.o.x = __shfl(r.o.x, src); r.o.y = __shfl(r.o.y, src); r.o.z = __shfl(r.o.z, src);
    r.d.x = __shfl(r.d.x, src); r.d.y = __shfl(r.d.y, src); r.d.z = __shfl(r.d.z, src);
    r.tmin = __shfl(r.tmin, src); r.tmax = __shfl(r.tmax, src);
    r.idx = __shfl(r.idx, src); r.idy = __shfl(r.idy, src); r.idz = __shfl(r.idz, src);
    r.octinv = __shfl(r.octinv, src);
    r.ng.x = __shfl(r.ng.x, src); r.ng.y = __shfl(r.ng.y, src);
    r.tg.x = __shfl(r.tg.x, src); r.tg.y = __shfl(r.tg.y, src);
    r.tg2.x = __shfl(r.tg2.x, src); r.tg2.y = __shfl(r.tg2.y, src);
    r.sp = __shfl(r.sp, src); r.col = __shfl(r.col, src);
    r.hit_addr = __shfl(r.hit_addr, src); r.out_idx = __shfl(r.out_idx, src);
    r.hu = __shfl(r.hu, src); r.hv = __shfl(r.hv, src);
    if constexpr (SRC == kRaysFromSurfels) r.out_texel = __shfl(r.out_texel, src);
    if constexpr (MULTI) {
        r.nodes = shfl_ptr(r.nodes, src);
        r.tris = shfl_ptr(r.tris, src);
        r.hits = shfl_ptr(r.hits, src);
        r.prim_map = shfl_ptr(r.prim_map, src);
        r.stride_sh = __shfl(r.stride_sh, src);
    }
}

// Writes a finished ray's hit, or counts it on its surfel.
template <int SRC>
__device__ __forceinline__ void write_hit(const CwbvhParams& P, const RayState& r) {
    if (SRC == kRaysFromSurfels && P.texel_hits) {
        if (r.hit_addr >= 0) atomicAdd(&P.texel_hits[r.out_texel], 1u);
    } else {
        const int out_id = (r.hit_addr >= 0 && P.prim_id) ? r.prim_map[r.hit_addr] : r.hit_addr;
        nt_store4(make_float4(r.tmax, i2f(out_id), r.hu, r.hv), &r.hits[r.out_idx]);
    }
}

// Traces a wave's remaining rays (lanes `live`, at most 64 / TEAM of them)
// with a team of TEAM lanes per ray until at most `leave` are left; returns
// the lanes that hold those (the first lane of each team).  All 64 lanes call
// it, each with its own ray state in `r`.
//
// The last rays of a wave are chains of dependent node loads and of the ~320
// instructions between them, issued for a few lanes: about 1 us per visit, so a
// launch lasts as long as its slowest rays however few they are.  Here lane j of
// a team tests 8 / TEAM children of the node and one triangle of the group,
// which cuts the chain per visit to the load and about 90 instructions.
// The visits, the tests and their arithmetic are those of the one-lane
// schedule, so the hits are too: a triangle group's closest hit is its lowest
// (t, address) under the same tie rule, its any hit the accepted triangle with
// the highest bit.  The stack stays in the LDS column of the ray's first lane.
// Entries beyond lds_depth (two-level stacks) go to every lane's own `spill`:
// the lanes of a team push and pop alike, so each holds the same copy.  Rays
// come in and leave with none there.
template <bool ANY, int SRC, bool MULTI, bool LDSO, bool SPREAD, int TEAM>
__device__ __forceinline__ unsigned long long team_trace(const CwbvhParams& P, CWD_LDS unsigned long long* lds_stack,
                                                         unsigned long long (&spill)[kStackCapacity],
                                                         unsigned long long live, int leave, int lane, RayState& r) {
    constexpr int kChildren = 8 / TEAM;   // children per lane: j and, teams of 4, j + 4
    const int team = (int)((unsigned)lane / TEAM), j = (int)((unsigned)lane % TEAM);
    int src = 0;
    const int count = __popcll(live);
    for (int k = 0; k < count; ++k) {
        const int s = __ffsll((long long)live) - 1;
        live &= live - 1ull;
        if (team == k) src = s;
    }
    shfl_state<SRC, MULTI>(r, src);
    bool busy = team < count;
    if (busy) {
        const int tx = r.idx < 0.f ? 24 : 0, ty = r.idy < 0.f ? 24 : 0, tz = r.idz < 0.f ? 24 : 0;
        while (true) {
            if (r.tg.y == 0u && r.ng.y > 0x00FFFFFFu) {
                const unsigned imask = r.ng.y;
                const int bit = 31 - __clz((int)r.ng.y);
                const unsigned slot = (unsigned)(bit - 24) ^ r.octinv;
                const unsigned rel = (unsigned)__popc(imask & ~(0xFFFFFFFFu << slot));
                // this lane's planes: bytes lo x, y, z, hi x, y, z of 8 children each
                float4 n0, n1;
                unsigned near[kChildren][3], far[kChildren][3];
                if constexpr (SPREAD) {
                    const unsigned off = spread_offset(r.ng.x + rel);
                    n0 = spread_slot(r.nodes, off, 0);
                    n1 = spread_slot(r.nodes, off, 1);
                    auto plane = [&](int at) { return *(const unsigned char*)spread_at(r.nodes, off, (unsigned)(32 + at)); };
#pragma unroll
                    for (int c = 0; c < kChildren; ++c) {
                        near[c][0] = plane(j + tx + 4 * c);
                        near[c][1] = plane(j + 8 + ty + 4 * c);
                        near[c][2] = plane(j + 16 + tz + 4 * c);
                        far[c][0] = plane(j + 24 - tx + 4 * c);
                        far[c][1] = plane(j + 32 - ty + 4 * c);
                        far[c][2] = plane(j + 40 - tz + 4 * c);
                    }
                } else {
                    const float4* np = node_at(r.nodes, r.ng.x + rel, r.stride_sh);
                    const unsigned char* q = reinterpret_cast<const unsigned char*>(np + 2) + j;
                    n0 = np[0];
                    n1 = np[1];
#pragma unroll
                    for (int c = 0; c < kChildren; ++c) {
                        near[c][0] = q[tx + 4 * c];
                        near[c][1] = q[8 + ty + 4 * c];
                        near[c][2] = q[16 + tz + 4 * c];
                        far[c][0] = q[24 - tx + 4 * c];
                        far[c][1] = q[32 - ty + 4 * c];
                        far[c][2] = q[40 - tz + 4 * c];
                    }
                }
                r.ng.y &= ~(1u << bit);
                if (r.ng.y > 0x00FFFFFFu) {
                    if (r.sp < (LDSO ? P.lds_depth : kStackCapacity)) {
                        if (LDSO || r.sp < P.lds_depth) lds_stack[(r.sp << 6) + r.col] = pack2(r.ng);
                        else spill[r.sp - P.lds_depth] = pack2(r.ng);
                        ++r.sp;
                    } else {
                        P.work[kWorkOverflow] = 1u;
                    }
                }
                const unsigned eb = f2u(n0.w);
                const int ex = (int)(signed char)(eb & 0xFFu);
                const int ey = (int)(signed char)((eb >> 8) & 0xFFu);
                const int ez = (int)(signed char)((eb >> 16) & 0xFFu);
                const float adjx = u2f((unsigned)(ex + 127) << 23) * r.idx;
                const float adjy = u2f((unsigned)(ey + 127) << 23) * r.idy;
                const float adjz = u2f((unsigned)(ez + 127) << 23) * r.idz;
                const float origx = -(r.o.x - n0.x) * r.idx;
                const float origy = -(r.o.y - n0.y) * r.idy;
                const float origz = -(r.o.z - n0.z) * r.idz;
                unsigned hitmask = 0;
#pragma unroll
                for (int c = 0; c < kChildren; ++c) {
                    const float tnx = __builtin_fmaf((float)near[c][0], adjx, origx);
                    const float tny = __builtin_fmaf((float)near[c][1], adjy, origy);
                    const float tnz = __builtin_fmaf((float)near[c][2], adjz, origz);
                    const float tfx = __builtin_fmaf((float)far[c][0], adjx, origx);
                    const float tfy = __builtin_fmaf((float)far[c][1], adjy, origy);
                    const float tfz = __builtin_fmaf((float)far[c][2], adjz, origz);
                    const float cmin = imax2(imax3(tnx, tny, tnz), r.tmin);
                    const float cmax = imin2(imin3(tfx, tfy, tfz), r.tmax);
                    const unsigned meta4 = (TEAM == 8 ? j < 4 : c == 0) ? f2u(n1.z) : f2u(n1.w);
                    const unsigned meta = (meta4 >> (8 * (j & 3))) & 0xFFu;
                    const bool inner = (meta & (meta << 1) & 0x10u) != 0u;
                    const unsigned at = (meta ^ (inner ? r.octinv : 0u)) & 0x1Fu;
                    hitmask |= cmin <= cmax ? (meta >> 5) << at : 0u;
                }
                hitmask = team_or<TEAM>(hitmask);
                r.ng = make_uint2(f2u(n1.x), (hitmask & 0xFF000000u) | (eb >> 24));
                r.tg = make_uint2(f2u(n1.y), hitmask & 0x00FFFFFFu);
            }
            bool finished = false;
            while (r.tg.y != 0u) {
                // lane j takes the (j + 1)-th highest triangle of the group
                int mine = -1;
                for (int k = 0; k < TEAM && r.tg.y != 0u; ++k) {
                    const int h = 31 - __clz((int)r.tg.y);
                    mine = j == k ? h : mine;
                    r.tg.y &= ~(1u << h);
                }
                bool ok = false;
                int addr = 0;
                float t = 0.f, u = 0.f, v = 0.f;
                if (mine >= 0) {
                    addr = (int)(r.tg.x * 3u + (unsigned)mine * 3u);
                    const float4 v0 = r.tris[addr], v1 = r.tris[addr + 1], v2 = r.tris[addr + 2];
                    ok = woop_test<ANY>(v0, v1, v2, r.o, r.d, r.tmin, r.tmax, addr, r.hit_addr, t, u, v);
                }
                if constexpr (ANY) {
                    // the first accepted triangle in the group's order
                    const unsigned m = (unsigned)(__ballot(ok) >> (team * TEAM)) & ((1u << TEAM) - 1u);
                    if (m != 0u) {
                        const int w = team * TEAM + __ffs((int)m) - 1;
                        r.tmax = __shfl(t, w);
                        r.hit_addr = __shfl(addr, w);
                        r.hu = __shfl(u, w);
                        r.hv = __shfl(v, w);
                        finished = true;
                        break;
                    }
                } else {
                    float bt = ok ? t : INFINITY;
                    int ba = ok ? addr : 0x7FFFFFFF;
                    team_min_step<kDppPair>(bt, ba);
                    team_min_step<kDppQuad>(bt, ba);
                    if (TEAM == 8) team_min_step<kDppHalf>(bt, ba);
                    if (ba != 0x7FFFFFFF) {
                        const bool won = ok && addr == ba;
                        r.tmax = bt;
                        r.hit_addr = ba;
                        r.hu = u2f(team_or<TEAM>(won ? f2u(u) : 0u));
                        r.hv = u2f(team_or<TEAM>(won ? f2u(v) : 0u));
                    }
                }
                if (r.tg.y == 0u) {   // the ray's second group, held when its wave's pool ran dry
                    r.tg = r.tg2;
                    r.tg2.y = 0u;
                }
            }
            if (!finished && r.ng.y <= 0x00FFFFFFu) {
                if (r.sp > 0) {
                    --r.sp;
                    if (LDSO || r.sp < P.lds_depth) r.ng = unpack2(lds_stack[(r.sp << 6) + r.col]);
                    else r.ng = unpack2(spill[r.sp - P.lds_depth]);
                } else {
                    finished = true;
                }
            }
            if (finished) {
                if (j == 0) write_hit<SRC>(P, r);
                busy = false;
                break;
            }
            if (__popcll(__ballot(j == 0)) <= leave && (LDSO || !__any(r.sp > P.lds_depth))) break;
        }
    }
    return __ballot(busy && j == 0);
}

template <bool ANY, bool STATS, bool MULTI, bool PREFETCH, int LOOP, int SRC = kRaysFromBuffer, bool TIGHT = false,
          bool LDSO = false, bool SPREAD = false>
__global__ __launch_bounds__(kMaxBlock) CWBVH_TRACE_ATTR void cwbvh_trace(CwbvhParams P) {
    static_assert(!TIGHT || (LOOP != kLoopSpeculate && !MULTI && !STATS && !PREFETCH),
                  "the tight builds are made for the plain interleaved and grouped kernels only");
    // LDSO: the launch's trees (a batch: every job's tree) need at most
    // lds_depth stack entries, so the stack lives in LDS only (interleaved
    // schedule: only node groups are pushed, one per level of the tree)
    static_assert(!LDSO || (LOOP == kLoopInterleave && !STATS), "LDS-only stacks serve the interleaved schedule");
    static_assert(!SPREAD || (LDSO && !MULTI), "spread nodes serve the LDS-only single-scene kernels");
    // The last rays of a wave go to teams of lanes (team_trace), with a two-level
    // stack once none of them has entries in scratch.  The 7-wave builds serve launches of 3 x 2^21 rays and more, whose
    // tail is 3% of their time; with team_trace their node loop spills scalars
    // and they run 2.3% slower (33 M AO rays: 2.19 against 2.14 ms).
    constexpr bool kTwoGroups = ANY && LOOP == kLoopInterleave && !STATS;
    constexpr bool kRepeatTriangles = !ANY && !PREFETCH && LOOP == kLoopInterleave && !STATS;
    constexpr bool kLookAhead = !ANY && PREFETCH && LOOP == kLoopInterleave && !STATS;
    constexpr bool kTeams = LOOP == kLoopInterleave && !STATS && !TIGHT;
    extern __shared__ unsigned long long lds_stack_raw[];
    CWD_LDS unsigned long long* lds_stack = lds_ptr(lds_stack_raw);
    unsigned long long spill[kStackCapacity];
    const StackIndex sx((int)threadIdx.x, P.lds_depth);
    const int lane = lane_id();

    // per-lane ray state
    int out_idx = -1;
    unsigned out_texel = 0;
    const float4* nodes = P.nodes;
    const float4* tris = P.tris;
    float4* hits = P.hits;
    const int* prim_map = P.prim_map;
    // node i starts at float4 (i << 2) + (i << stride_sh): stride 5 or 8
    // without a quarter-rate integer multiply
    unsigned stride_sh = P.stride == 8 ? 2u : 0u;
    int spec_limit = P.spec_limit;
    float3 o = make_float3(0.f, 0.f, 0.f), d = o;
    float tmin = 0.f, tmax = 0.f, idx = 0.f, idy = 0.f, idz = 0.f;
    unsigned octinv = 0, octinv4 = 0;
    // tg2.x with kLookAhead: kNoGroup unless a node was visited while tg waits
    constexpr unsigned kNoGroup = kLookAhead ? 0xFFFFFFFFu : 0u;
    uint2 ng = make_uint2(0u, 0u), tg = make_uint2(0u, 0u), tg2 = make_uint2(kNoGroup, 0u);
    int sp = 0;
    int hit_addr = -1;
    float hu = 0.f, hv = 0.f;
    unsigned long long st_nodes = 0, st_tris = 0;
    // STATS only: {slots, uses} of the loop iteration, the node code and the
    // triangle code; a slot is one lane of a wave instruction stream that ran
    // the code (64 per wave pass), a use is a lane that needed it
    unsigned long long pr_it = 0, pr_act = 0, pr_nd = 0, pr_ndu = 0, pr_tr = 0, pr_tru = 0;
    auto prof = [&](bool used, unsigned long long& slots, unsigned long long& uses) {
        if (STATS) {
            const unsigned long long act = __ballot(1);
            if (__any(used) && lane == __ffsll((long long)act) - 1) slots += 64;
            uses += used ? 1 : 0;
        }
    };
    bool have_pf = false;
    float4 pf0, pf1, pf2, pf3, pf4;
    // A lane is busy from loading a ray until writing its hit.  (Deriving
    // "terminated" from an empty stack and empty groups, as the reference
    // does at src/TraversalKernelCWBVH.cu:60, misreads a lane whose last
    // stack entry was a postponed triangle group just popped into ng.)
    bool busy = false;

    // wave-uniform work pool; single-scene launches split the rays into
    // `slices` contiguous ranges and a wave drains the range of its XCD
    // (workgroups are dispatched round-robin over the XCDs) before stealing
    unsigned pool_next = 0, pool_end = 0;
    int pool_job = 0;
    bool exhausted = false;
    const int home = (int)(blockIdx.x % (unsigned)P.slices);
    int slice_k = 0;
    const unsigned first_index =
        (blockIdx.x / (unsigned)P.slices) * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    // Batches: lane k holds the first chunk of job k * job_step, so a claimed
    // chunk's job is found by one ballot (job_step 1: up to 64 jobs) and a search
    // among job_step jobs, not by log2(jobs) dependent loads per claim.
    unsigned seg_begin = 0xFFFFFFFFu;
    if constexpr (MULTI && kTeams) {
        if (lane * P.job_step < P.num_jobs) seg_begin = P.jobs[lane * P.job_step].chunk_begin;
    }

    while (true) {
        const bool terminated = !busy;
        unsigned long long need = __ballot(terminated);
        bool got = false;
        unsigned my = 0;
        int my_job = 0;
        while (need != 0ull) {
            if (pool_next >= pool_end) {
                if (exhausted) break;
                const int leader = __ffsll((long long)need) - 1;
                if (!MULTI && !P.persistent) {
                    // no work fetching: the only "pool" is this wave's own rays_per_wave indices
                    exhausted = true;
                    const unsigned share = kTeams ? (unsigned)P.rays_per_wave : 64u;
                    const unsigned first = (blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * share;
                    pool_next = min(first, (unsigned)P.n);
                    pool_end = min(first + share, (unsigned)P.n);
                    if (pool_next >= pool_end) break;
                } else if (MULTI) {
                    // claim one chunk index from the home slice of the chunk
                    // range, then from the others
                    bool found = false;
                    unsigned base = 0;
                    const bool first_claim = slice_k == 0 && pool_end == 0u;
                    unsigned drained = 0;
                    while (slice_k < P.slices) {
                        const int sl = home + slice_k - (home + slice_k >= P.slices ? P.slices : 0);
                        if (slice_k > 0 && ((drained >> sl) & 1u)) {
                            ++slice_k;
                            continue;
                        }
                        const unsigned lo = slice_begin(sl, P.item_q, P.item_r);
                        const unsigned hi = slice_begin(sl + 1, P.item_q, P.item_r);
                        const bool static_claim = first_claim && slice_k == 0;
                        if (!static_claim && static_only(sl, hi - lo, 1u, P.block_q, P.block_r)) {
                            ++slice_k;
                            continue;
                        }
                        const unsigned claim = slice_claim(P.work, sl, 1u, static_claim, first_index,
                                                           P.block_q, P.block_r, lane);
                        if (claim < hi - lo) {
                            base = lo + claim;
                            found = true;
                            break;
                        }
                        if (!static_claim) drained = mark_drained(P.work, sl, lane);
                        ++slice_k;
                    }
                    if (!found) {
                        exhausted = true;
                        break;
                    }
                    // job j owns chunks [jobs[j].chunk_begin, jobs[j+1].chunk_begin)
                    int lo = 0, hi = P.num_jobs - 1;
                    if constexpr (kTeams) {
                        // all 64 lanes are here: the segment whose first job starts at or before the chunk
                        const int seg = __popcll(__ballot(seg_begin <= base)) - 1;
                        lo = seg * P.job_step;
                        hi = min(lo + P.job_step, P.num_jobs) - 1;
                    }
                    while (lo < hi) {
                        const int mid = (lo + hi + 1) >> 1;
                        if (P.jobs[mid].chunk_begin <= base) lo = mid;
                        else hi = mid - 1;
                    }
                    pool_job = lo;
                    const unsigned first = (base - P.jobs[lo].chunk_begin) * (unsigned)P.chunk;
                    pool_next = first;
                    pool_end = min(first + (unsigned)P.chunk, (unsigned)P.jobs[lo].n);
                } else {
                    bool found = false;
                    // the wave's first claim: nothing claimed yet; slices found dry in this refill
                    const bool first_claim = slice_k == 0 && pool_end == 0u;
                    unsigned drained = 0;
                    while (slice_k < P.slices) {
                        const int sl = home + slice_k - (home + slice_k >= P.slices ? P.slices : 0);
                        if (slice_k > 0 && ((drained >> sl) & 1u)) {
                            ++slice_k;
                            continue;
                        }
                        const unsigned lo = slice_begin(sl, P.item_q, P.item_r);
                        const unsigned hi = slice_begin(sl + 1, P.item_q, P.item_r);
                        const unsigned base = slice_claim(P.work, sl, (unsigned)P.chunk, first_claim && slice_k == 0, first_index,
                                                          P.block_q, P.block_r, lane);
                        if (base < hi - lo) {
                            pool_next = lo + base;
                            pool_end = lo + min(base + (unsigned)P.chunk, hi - lo);
                            found = true;
                            break;
                        }
                        drained = mark_drained(P.work, sl, lane);
                        ++slice_k;
                    }
                    if (!found) {
                        exhausted = true;
                        break;
                    }
                }
            }
            const unsigned avail = pool_end - pool_next;
            const unsigned rank = (unsigned)__popcll(need & lanemask_lt());
            if (((need >> lane) & 1ull) && rank < avail) {
                my = pool_next + rank;
                my_job = pool_job;
                got = true;
            }
            pool_next += min((unsigned)__popcll(need), avail);
            need = __ballot(terminated && !got);
        }

        if (got) {
            const Ray4* rays = P.rays;
            const int* order = P.order;
            unsigned ray_count = (unsigned)P.n;
            if (MULTI) {
                const cw::BatchJob& J = P.jobs[my_job];
                nodes = (const float4*)J.nodes;
                tris = (const float4*)J.woop;
                hits = (float4*)J.hits;
                prim_map = J.prim_idx;
                stride_sh = J.node_stride == 8 ? 2u : 0u;
                spec_limit = J.spec_limit;
                rays = (const Ray4*)J.rays;
                order = J.order;
                ray_count = (unsigned)J.n;
            }
            if constexpr (SRC == kRaysFromSurfels) {
                // the ray is made here from its surfel instead of read back
                const int ri = (int)my;
                out_idx = ri;
                out_texel = (unsigned)ri / (unsigned)P.rays_per_texel;
                const float4 sp = P.surf_pos[out_texel], sn = P.surf_nrm[out_texel];
                cwao::F3 go, gd;
                cwao::surfel_ray(cwao::F3{sp.x, sp.y, sp.z}, cwao::F3{sn.x, sn.y, sn.z}, P.surf_rad[out_texel],
                                 P.seed, (unsigned long long)ri, go, gd);
                o = make_float3(go.x, go.y, go.z);
                d = make_float3(gd.x, gd.y, gd.z);
                tmin = P.gen_tmin;
                tmax = P.gen_tmax;
            } else {
                int ri = order ? order[my] : (int)my;
                // an order entry outside the launch's rays traces ray `my`
                // itself, so a malformed order cannot read or write out of bounds
                if ((unsigned)ri >= ray_count) ri = (int)my;
                out_idx = ri;
                // rays are read once: keep them out of the caches the BVH lives in
                const float4 ro = nt_load4(&rays[ri].o);
                const float4 rd = nt_load4(&rays[ri].d);
                o = make_float3(ro.x, ro.y, ro.z);
                d = make_float3(rd.x, rd.y, rd.z);
                tmin = ro.w;
                tmax = rd.w;
            }
            safe_rcp3(d, idx, idy, idz);
            const unsigned oct = ((d.x < 0.f ? 1u : 0u) << 2) | ((d.y < 0.f ? 1u : 0u) << 1) | (d.z < 0.f ? 1u : 0u);
            octinv = 7u - oct;
            octinv4 = octinv * 0x01010101u;
            ng = make_uint2(0u, 0x80000000u);
            tg = make_uint2(0u, 0u);
            tg2 = make_uint2(kNoGroup, 0u);
            sp = 0;
            hit_addr = -1;
            hu = hv = 0.f;
            have_pf = false;
            busy = true;
        }

        if constexpr (kTeams) {
            if (exhausted && __popcll(__ballot(busy)) <= kLastRays && (LDSO || !__any(busy && sp > P.lds_depth))) break;
            if (!busy) continue;  // idle until the wave ends
        } else {
            if (terminated && !got) break;  // no work left for this lane
        }

        // stack push of a node or triangle group (overflow is flagged, not written)
        auto push = [&](uint2 e) {
            if constexpr (LDSO) {
                if (sp < P.lds_depth) {
                    lds_stack[(sp << 6) + sx.col] = pack2(e);
                    ++sp;
                } else {
                    P.work[kWorkOverflow] = 1u;
                }
            } else {
                if (sp < kStackCapacity) {
                    stack_put(lds_stack, spill, sx, sp, pack2(e));
                    ++sp;
                } else {
                    P.work[kWorkOverflow] = 1u;
                }
            }
        };
        auto stack_at = [&](int i) -> unsigned long long {
            if constexpr (LDSO) return lds_stack[(i << 6) + sx.col];
            else return stack_get(lds_stack, spill, sx, i);
        };
        // Visit the highest-priority child of ng: the remainder of ng goes on
        // the stack, ng becomes the child's inner children, the child's leaf
        // triangles are returned.  A visit ahead leaves the child, as a group of
        // its own, in the free slot above the stack's top.
        auto visit_node = [&](bool ahead = false) -> uint2 {
            const unsigned imask = ng.y;
            const int bit = 31 - __clz((int)ng.y);
            const unsigned base = ng.x;
            ng.y &= ~(1u << bit);
            if (ng.y > 0x00FFFFFFu) push(ng);
            const unsigned slot = (unsigned)(bit - 24) ^ octinv;
            const unsigned visited = base + (unsigned)__popc(imask & ~(0xFFFFFFFFu << slot));
            if (ahead) lds_stack[(sp << 6) + sx.col] = pack2(make_uint2(visited, 0x80000000u));
            float4 n0, n1, n2, n3, n4;
            if (PREFETCH && have_pf) {
                n0 = pf0; n1 = pf1; n2 = pf2; n3 = pf3; n4 = pf4;
                have_pf = false;
            } else {
                if constexpr (SPREAD) {
                    const unsigned off = spread_offset(visited);
                    n0 = spread_slot(nodes, off, 0); n1 = spread_slot(nodes, off, 1); n2 = spread_slot(nodes, off, 2);
                    n3 = spread_slot(nodes, off, 3); n4 = spread_slot(nodes, off, 4);
                } else {
                    const float4* np = node_at(nodes, visited, stride_sh);
                    n0 = np[0]; n1 = np[1]; n2 = np[2]; n3 = np[3]; n4 = np[4];
                    if constexpr (MULTI) keep_address(np, n0.x);
                }
            }
            if (STATS) ++st_nodes;
            const unsigned eb = f2u(n0.w);
            const int ex = (int)(signed char)(eb & 0xFFu);
            const int ey = (int)(signed char)((eb >> 8) & 0xFFu);
            const int ez = (int)(signed char)((eb >> 16) & 0xFFu);
            const float adjx = u2f((unsigned)(ex + 127) << 23) * idx;
            const float adjy = u2f((unsigned)(ey + 127) << 23) * idy;
            const float adjz = u2f((unsigned)(ez + 127) << 23) * idz;
            const float origx = -(o.x - n0.x) * idx;
            const float origy = -(o.y - n0.y) * idy;
            const float origz = -(o.z - n0.z) * idz;
            const bool sgx = idx < 0.f, sgy = idy < 0.f, sgz = idz < 0.f;
            unsigned hitmask;
            {
                const unsigned qlx = f2u(n2.x), qly = f2u(n2.z), qlz = f2u(n3.x);
                const unsigned qhx = f2u(n3.z), qhy = f2u(n4.x), qhz = f2u(n4.z);
                hitmask = child_hits4(f2u(n1.z), sgx ? qhx : qlx, sgy ? qhy : qly, sgz ? qhz : qlz,
                                      sgx ? qlx : qhx, sgy ? qly : qhy, sgz ? qlz : qhz, adjx, adjy, adjz,
                                      origx, origy, origz, tmin, tmax, octinv4);
            }
            {
                const unsigned qlx = f2u(n2.y), qly = f2u(n2.w), qlz = f2u(n3.y);
                const unsigned qhx = f2u(n3.w), qhy = f2u(n4.y), qhz = f2u(n4.w);
                hitmask |= child_hits4(f2u(n1.w), sgx ? qhx : qlx, sgy ? qhy : qly, sgz ? qhz : qlz,
                                       sgx ? qlx : qhx, sgy ? qly : qhy, sgz ? qlz : qhz, adjx, adjy, adjz,
                                       origx, origy, origz, tmin, tmax, octinv4);
            }
            ng.x = f2u(n1.x);
            ng.y = (hitmask & 0xFF000000u) | (eb >> 24);
            if (PREFETCH && ng.y > 0x00FFFFFFu) {
                // the next node visit takes the highest hit child: start its
                // loads now so they overlap the triangle tests in between
                const int nb = 31 - __clz((int)ng.y);
                const unsigned nslot = (unsigned)(nb - 24) ^ octinv;
                const unsigned nrel = (unsigned)__popc(ng.y & ~(0xFFFFFFFFu << nslot));
                if constexpr (SPREAD) {
                    const unsigned off = spread_offset(ng.x + nrel);
                    pf0 = spread_slot(nodes, off, 0); pf1 = spread_slot(nodes, off, 1); pf2 = spread_slot(nodes, off, 2);
                    pf3 = spread_slot(nodes, off, 3); pf4 = spread_slot(nodes, off, 4);
                } else {
                    const float4* np = node_at(nodes, ng.x + nrel, stride_sh);
                    pf0 = np[0]; pf1 = np[1]; pf2 = np[2]; pf3 = np[3]; pf4 = np[4];
                }
                have_pf = true;
            }
            return make_uint2(f2u(n1.y), hitmask & 0x00FFFFFFu);
        };
        // Test the highest triangle of tg; true when it is accepted.
        auto test_triangle = [&]() -> bool {
            const int ti = 31 - __clz((int)tg.y);
            const int addr = (int)(tg.x * 3u + (unsigned)ti * 3u);
            const float4* tp = tris + addr;
            const float4 v0 = tp[0], v1 = tp[1], v2 = tp[2];
            if constexpr (MULTI) keep_address(tp, v0.x);
            if (STATS) ++st_tris;
            tg.y &= ~(1u << ti);
            float t, u, v;
            if (woop_test<ANY>(v0, v1, v2, o, d, tmin, tmax, addr, hit_addr, t, u, v)) {
                tmax = t;
                hit_addr = addr;
                hu = u;
                hv = v;
                return true;
            }
            return false;
        };

        int lost = 0;
        while (true) {
            bool finished = false;
            prof(true, pr_it, pr_act);
            if constexpr (LOOP == kLoopGroup) {
                prof(ng.y > 0x00FFFFFFu, pr_nd, pr_ndu);
                if (ng.y > 0x00FFFFFFu) {
                    tg = visit_node();
                } else {
                    // a postponed triangle group came off the stack
                    tg = ng;
                    ng = make_uint2(0u, 0u);
                }
                const int total = P.postpone_pct > 0 ? __popcll(__ballot(1)) : 0;
                while (tg.y != 0u) {
                    if (P.postpone_pct > 0) {
                        const int active = __popcll(__ballot(1));
                        if (active * 100 < total * P.postpone_pct) {
                            push(tg);
                            tg.y = 0u;
                            break;
                        }
                    }
                    prof(true, pr_tr, pr_tru);
                    if (test_triangle() && ANY) {
                        finished = true;
                        break;
                    }
                }
                if (!finished && ng.y <= 0x00FFFFFFu) {
                    if (sp > 0) {
                        --sp;
                        ng = unpack2(stack_at(sp));
                    } else {
                        finished = true;
                    }
                }
            } else {
                if constexpr (kTwoGroups) {
                    if (tg2.y == 0u && ng.y > 0x00FFFFFFu) {
                        const uint2 ntg = visit_node();
                        if (tg.y == 0u) tg = ntg;
                        else tg2 = ntg;
                    }
                    if (ng.y <= 0x00FFFFFFu && sp > 0) {
                        --sp;
                        ng = unpack2(stack_at(sp));
                    }
                    bool run_tri = true;
                    if constexpr (PREFETCH) {
                        const bool can_visit = tg2.y == 0u && ng.y > 0x00FFFFFFu;
                        run_tri = __popcll(__ballot(tg.y != 0u)) >= kTriangleLanes || !__any(can_visit);
                    }
                    if (run_tri && tg.y != 0u) {
                        finished = test_triangle();
                        if (tg.y == 0u) {
                            tg = tg2;
                            tg2.y = 0u;
                        }
                    }
                    if (tg.y == 0u && ng.y <= 0x00FFFFFFu) finished = true;
                } else if constexpr (kLookAhead) {
                    auto can_visit = [&]() {
                        return ng.y > 0x00FFFFFFu && (tg.y == 0u || (tg2.x == kNoGroup && sp + 1 < P.lds_depth));
                    };
                    if (can_visit()) {
                        const uint2 ntg = visit_node(tg.y != 0u);
                        if (tg.y == 0u) tg = ntg;
                        else tg2 = ntg;
                    }
                    const bool run_tri = __popcll(__ballot(tg.y != 0u)) >= kTriangleLanes || !__any(can_visit());
                    if (run_tri && tg.y != 0u) {
                        if (test_triangle() && tg2.x != kNoGroup) {
                            ng = unpack2(lds_stack[(sp << 6) + sx.col]);
                            tg2 = make_uint2(kNoGroup, 0u);
                            have_pf = false;
                        }
                        if (tg.y == 0u) {
                            tg = tg2;
                            tg2 = make_uint2(kNoGroup, 0u);
                        }
                    }
                    if (ng.y <= 0x00FFFFFFu && tg2.x == kNoGroup) {
                        if (sp > 0) {
                            --sp;
                            ng = unpack2(stack_at(sp));
                        } else if (tg.y == 0u) {
                            finished = true;
                        }
                    }
                } else {
                    // node step: lanes without triangles (and, speculating, every
                    // lane with inner children left) visit one node
                    const bool spec_ok = LOOP == kLoopSpeculate && sp < spec_limit;
                    const bool node_step = (spec_ok || tg.y == 0u) && ng.y > 0x00FFFFFFu;
                    prof(node_step, pr_nd, pr_ndu);
                    if (node_step) {
                        const uint2 ntg = visit_node();
                        if (tg.y != 0u) {
                            if (ntg.y != 0u) push(ntg);
                        } else {
                            tg = ntg;
                        }
                    }
                    // triangle step: one test (speculating with postpone_pct, only
                    // once enough lanes hold triangles or a lane holds nothing else)
                    bool run_tri = true;
                    if (LOOP == kLoopSpeculate && P.postpone_pct > 0) {
                        // lanes that hold triangles and cannot visit a node next
                        // iteration idle until the triangle step runs
                        const bool can_visit = ng.y > 0x00FFFFFFu && (tg.y == 0u || sp < spec_limit);
                        const int stuck = __popcll(__ballot(tg.y != 0u && !can_visit));
                        run_tri = !__any(can_visit) || stuck * 100 >= P.postpone_pct * __popcll(__ballot(1));
                    }
                    prof(run_tri && tg.y != 0u, pr_tr, pr_tru);
                    if constexpr (kRepeatTriangles) {
                        do {
                            if (tg.y != 0u) test_triangle();
                        } while (__popcll(__ballot(tg.y != 0u)) >= kTriangleAgain);
                    } else {
                        if (run_tri && tg.y != 0u) finished = test_triangle() && ANY;
                    }
                    // out of inner children: take the next group off the stack
                    if (!finished && ng.y <= 0x00FFFFFFu) {
                        if (tg.y == 0u) {
                            if (sp > 0) {
                                --sp;
                                const uint2 e = unpack2(stack_at(sp));
                                if (e.y > 0x00FFFFFFu) {
                                    ng = e;
                                } else {
                                    tg = e;
                                    ng = make_uint2(0u, 0u);
                                }
                            } else {
                                finished = true;
                            }
                        } else if (LOOP == kLoopSpeculate && sp > 0) {
                            const uint2 e = unpack2(stack_at(sp - 1));
                            if (e.y > 0x00FFFFFFu) {
                                --sp;
                                ng = e;
                            }
                        }
                    }
                }
            }
            if (finished) {
                if (SRC == kRaysFromSurfels && P.texel_hits) {
                    if (hit_addr >= 0) atomicAdd(&P.texel_hits[out_texel], 1u);
                } else {
                    const int out_id = (hit_addr >= 0 && P.prim_id) ? prim_map[hit_addr] : hit_addr;
                    nt_store4(make_float4(tmax, i2f(out_id), hu, hv), &hits[out_idx]);
                }
                sp = 0;
                ng = make_uint2(0u, 0u);
                tg = make_uint2(0u, 0u);
                tg2 = make_uint2(kNoGroup, 0u);
                have_pf = false;
                busy = false;
                break;
            }
            const int idle = __popcll(~__ballot(1));
            lost += idle - P.idle_lanes;
            if constexpr (kTeams) {
                if (exhausted ? idle >= 64 - kLastRays : lost >= P.idle_budget) break;
            } else {
                if (lost >= P.idle_budget) break;
            }
        }
    }

    if constexpr (kTeams) {
        // the last rays of the wave, with teams of lanes
        unsigned long long live = __ballot(busy);
        if (live != 0ull) {
            if (kLookAhead && tg2.x != kNoGroup) {   // teams do not look ahead
                ng = unpack2(lds_stack[(sp << 6) + sx.col]);
                tg2.y = 0u;
            }
            RayState r{o, d, tmin, tmax, idx, idy, idz, octinv, ng, tg, tg2, sp, sx.col, hit_addr, out_idx,
                       out_texel, hu, hv, nodes, tris, hits, prim_map, stride_sh};
            if (__popcll(live) > 8) live = team_trace<ANY, SRC, MULTI, LDSO, SPREAD, 4>(P, lds_stack, spill, live, 8, lane, r);
            team_trace<ANY, SRC, MULTI, LDSO, SPREAD, 8>(P, lds_stack, spill, live, 0, lane, r);
        }
    }
    if (STATS) {
        atomicAdd(&P.stats[0], st_nodes);
        atomicAdd(&P.stats[1], st_tris);
        unsigned long long* pr = reinterpret_cast<unsigned long long*>(P.work + kWorkProfile);
        atomicAdd(&pr[0], pr_it);
        atomicAdd(&pr[1], pr_act);
        atomicAdd(&pr[2], pr_nd);
        atomicAdd(&pr[3], pr_ndu);
        atomicAdd(&pr[4], pr_tr);
        atomicAdd(&pr[5], pr_tru);
    }
    // one-ray-per-thread launches claim nothing and skip the exit count
    if (!MULTI && !P.persistent) return;
    block_exit(P.work, P.total_blocks, P.slices, P.block_q, P.block_r);
}

// ------------------------------------------------------------ occupancy

template <class K>
int resident_blocks(K kernel, int block, size_t lds) {
    static std::mutex mu;
    static std::map<std::tuple<const void*, int, size_t>, int> cache;
    std::lock_guard<std::mutex> g(mu);
    auto key = std::make_tuple((const void*)kernel, block, lds);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, block, lds) != hipSuccess) {
        (void)hipGetLastError();  // tolerated: one block per unit
        nb = 1;
    }
    if (nb < 1) nb = 1;
    cache[key] = nb;
    return nb;
}

// Items (rays or chunks) and grid blocks split over the work slices.
template <class Params>
void set_splits(Params& p) {
    const unsigned sl = (unsigned)std::max(1, p.slices);
    p.item_q = (unsigned)p.n / sl;
    p.item_r = (unsigned)p.n % sl;
    p.block_q = (unsigned)p.total_blocks / sl;
    p.block_r = (unsigned)p.total_blocks % sl;
}

template <bool ANY, bool STATS, bool MULTI, bool PREFETCH, int LOOP, int SRC = kRaysFromBuffer, bool TIGHT = false,
          bool LDSO = false, bool SPREAD = false>
int32_t launch_cwbvh_t(CwbvhParams& p, const cwbvh_trace_config& cfg, hipStream_t stream) {
    const int block = cfg.block_size;
    const size_t lds = (size_t)block * (size_t)cfg.lds_depth * sizeof(unsigned long long);
    auto kernel = cwbvh_trace<ANY, STATS, MULTI, PREFETCH, LOOP, SRC, TIGHT, LDSO, SPREAD>;
    long long grid = cfg.grid_blocks;
    if (!MULTI && !p.persistent) {
        p.rays_per_wave = LOOP == kLoopInterleave && !STATS && !TIGHT
                              ? cw::team_rays_per_wave(p.n, cw::device_compute_units())
                              : 64;
        const long long per_block = (long long)p.rays_per_wave * (block / 64);
        grid = ((long long)p.n + per_block - 1) / per_block;
        p.idle_budget = 0x7FFFFFFF;  // nothing to refill from
    } else if (grid <= 0) {
        grid = resident_blocks(kernel, block, lds);
        const int waves = cw::grid_waves(!MULTI && PREFETCH, p.order != nullptr, p.streams != 0);
        if (waves > 0) grid = std::min(grid, (long long)waves * 4 * 64 / block);
        grid *= cw::device_compute_units();
    }
    p.total_waves = (int)(grid * (block / 64));
    if (MULTI && cfg.grid_blocks <= 0) {
        // a batch of fewer chunks than waves: one chunk per wave, no idle blocks
        const long long slices = std::max(1, p.slices), waves = block / 64;
        const long long per_slice = ((long long)p.n + slices - 1) / slices;
        grid = std::min(grid, slices * ((per_slice + waves - 1) / waves));
    }
    p.total_blocks = (int)grid;
    set_splits(p);
    if (p.chunk <= 0) {
        // automatic: about 32 claims per wave over the launch, a multiple of 64
        // rays, at most 512.  At least 128 once the launch averages 1024 rays
        // per wave; below that one ray per lane per claim balances the short
        // launch better (1-3 M AO rays: 2-5% faster than 128; from 8 M rays
        // on, 64 is slower, by 9% at 33 M)
        const long long per_wave = (long long)p.n / p.total_waves;
        long long c = (long long)p.n / ((long long)p.total_waves * 32);
        c = std::min<long long>(512, std::max<long long>(per_wave < 1024 ? 64 : 128, (c + 63) / 64 * 64));
        p.chunk = (int)c;
        // The smaller the claims, the closer together the rays in flight, and the
        // more of the nodes they share are in L2.  Rays traced in an order (as a
        // launch that sorts them does) gain from that, and so do the prefetch
        // kernels, whose scenes stream from memory; their visits also hide more
        // claims.  ms at claims of 32 / 64 / 128 / 512 rays, sorted: 5 M-triangle
        // soup (prefetch) 16.8 M rays 10.60 / 10.64 / 10.91 / 12.42, 2 M rays 1.75 /
        // 1.81 / 2.02 / 2.75; 1 M-triangle spheres 16 M AO rays 1.96 / 1.89 / 1.91 /
        // 2.10, 2 M 0.332 / 0.310 / 0.325 / 0.463.
        if (!MULTI && PREFETCH) p.chunk = 32;
        else if (!MULTI && p.order) p.chunk = 64;
    }
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(block), lds, stream, p);
    CW_HIP(hipGetLastError());
    return CWBVH_OK;
}

template <bool ANY, bool STATS, bool MULTI, bool PREFETCH>
int32_t dispatch_loop(CwbvhParams& p, const cwbvh_trace_config& cfg, hipStream_t st) {
    switch (cfg.loop_mode) {
        case kLoopInterleave:
            if constexpr (!STATS && !MULTI) {
                const bool w7 = !PREFETCH && (cfg.occupancy == kOccupancy7 ||
                                              (cfg.occupancy == kOccupancyAuto && p.n >= cw::seven_wave_rays(ANY, p.lds_only != 0)));
                if (p.lds_only) {
                    if (w7) return launch_cwbvh_t<ANY, false, false, false, kLoopInterleave, kRaysFromBuffer, true, true>(p, cfg, st);
                    if (p.spread) return launch_cwbvh_t<ANY, false, false, PREFETCH, kLoopInterleave, kRaysFromBuffer, false, true, true>(p, cfg, st);
                    return launch_cwbvh_t<ANY, false, false, PREFETCH, kLoopInterleave, kRaysFromBuffer, false, true>(p, cfg, st);
                }
                if (w7) return launch_cwbvh_t<ANY, false, false, false, kLoopInterleave, kRaysFromBuffer, true>(p, cfg, st);
            }
            if constexpr (!STATS && MULTI) {
                if (p.lds_only)
                    return launch_cwbvh_t<ANY, false, true, PREFETCH, kLoopInterleave, kRaysFromBuffer, false, true>(p, cfg, st);
            }
            return launch_cwbvh_t<ANY, STATS, MULTI, PREFETCH, kLoopInterleave>(p, cfg, st);
        case kLoopSpeculate: return launch_cwbvh_t<ANY, STATS, MULTI, PREFETCH, kLoopSpeculate>(p, cfg, st);
        default:
            if constexpr (!STATS && !MULTI && !PREFETCH) {
                if (!p.streams) return launch_cwbvh_t<ANY, false, false, false, kLoopGroup, kRaysFromBuffer, true>(p, cfg, st);
            }
            return launch_cwbvh_t<ANY, STATS, MULTI, PREFETCH, kLoopGroup>(p, cfg, st);
    }
}

}  // namespace cwk
