// Traversal kernels for gfx950 (wave64) and their launchers.
//
//  * cwbvh_trace (cwbvh_kernel.h): persistent CWBVH traversal with wave-level work fetching.
//    Follows the reference kernel src/TraversalKernelCWBVH.cu:24-375:
//      - ray fetch: terminated lanes of a wave are refilled together; one
//        lane claims `fetch_chunk` rays with a single atomic and the wave
//        hands them out by prefix rank (ballot + popcount), instead of one
//        atomic per refill as in the reference (:60-72);
//      - node group / triangle group state machine, highest-bit-first child
//        order with octant XOR, 8-child quantized slab test (:93-295);
//      - optional triangle postponing (:297-311) and the dynamic-fetch exit
//        when idle lanes accumulate (:365-371), both tunable for 64 lanes;
//      - traversal stack: first `lds_depth` entries in LDS (interleaved by
//        lane), the rest in per-lane scratch, capacity 64 entries with an
//        overflow flag (the reference has 8 shared + 32 local entries and
//        no check).
//    One template serves a single scene (uniform scene pointers) and the
//    multi-scene batch (per-lane scene pointers from a job table).
//  * bvh2_trace: one lane per ray, Aila-Laine while-while traversal with one
//    postponed leaf and a wave-wide "any lane wants nodes" exit, Woop leaves
//    closed by a 0x80000000 terminator (src/TraversalKernelBVH2.cu:26-178).
//
// Both kernels use the arithmetic contract of device_common.h, so results are
// bit-identical between kernel variants and to the scalar CPU restatement
// used by the tests.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "cwbvh_kernel.h"

using namespace cwd;

// instantiated in trace_prefetch.hip
#define CWBVH_PREFETCH_LAUNCHES(ANY, STATS)                                                              \
    extern template int32_t cwk::dispatch_loop<ANY, STATS, false, true>(cwk::CwbvhParams&,               \
                                                                        const cwbvh_trace_config&, hipStream_t); \
    extern template int32_t cwk::dispatch_loop<ANY, STATS, true, true>(cwk::CwbvhParams&,                \
                                                                       const cwbvh_trace_config&, hipStream_t);
CWBVH_PREFETCH_LAUNCHES(false, false)
CWBVH_PREFETCH_LAUNCHES(false, true)
CWBVH_PREFETCH_LAUNCHES(true, false)
CWBVH_PREFETCH_LAUNCHES(true, true)
#undef CWBVH_PREFETCH_LAUNCHES

namespace {

using namespace cwk;

struct Bvh2Params {
    const float4* __restrict__ nodes;
    const float4* __restrict__ tris;
    const int* __restrict__ prim_map;
    const Ray4* __restrict__ rays;
    const int* __restrict__ order;
    float4* __restrict__ hits;
    unsigned* work;
    unsigned long long* stats;
    int n;
    int lds_depth;
    int woop_last;   // last valid float4 index of tris (loads past a leaf terminator clamp here)
    int prim_id;
    // persistent launches (bvh2_trace_persistent) only
    int slices;
    int chunk;
    int idle_lanes;
    int idle_budget;
    int total_blocks;
    unsigned item_q, item_r;   // n = item_q * slices + item_r
    unsigned block_q, block_r; // total_blocks = block_q * slices + block_r
    // not read by the persistent kernel, so behind its fields: before them they moved
    // those into one more 64-byte line of arguments, which its short launches, most of
    // whose time is their waves' start, paid with 20 us (3,000 rays 223 us, 206 so)
    int share;       // bvh2_trace: rays per wave
    int in_l2;       // host side: the scene fits one XCD's L2
};

// Slab test of one BVH2 child box (reference src/TraversalKernelBVH2.cu:14-24).
__device__ __forceinline__ bool box2(float lox, float hix, float loy, float hiy, float loz, float hiz, float idx,
                                     float idy, float idz, float oodx, float oody, float oodz, float tmin, float tmax,
                                     float& dist) {
    const float lx = __builtin_fmaf(lox, idx, -oodx), hx = __builtin_fmaf(hix, idx, -oodx);
    const float ly = __builtin_fmaf(loy, idy, -oody), hy = __builtin_fmaf(hiy, idy, -oody);
    const float lz = __builtin_fmaf(loz, idz, -oodz), hz = __builtin_fmaf(hiz, idz, -oodz);
    const float smin = imax2(imax3(imin2(lx, hx), imin2(ly, hy), imin2(lz, hz)), tmin);
    const float smax = imin2(imin3(imax2(lx, hx), imax2(ly, hy), imax2(lz, hz)), tmax);
    dist = smin;
    return smin <= smax;
}

// Bound by its 16-byte load instructions: each takes 16 cycles of the unit's
// address path however few lanes are on, and a third are (33 M AO rays: TA busy
// 91%, VALU 49%).  Tried and slower or within 7%: loads shared by node visits and
// triangle tests with refilled lanes (8.2 M rays 1.08 ms, but slower below 2 M),
// nodes staged in LDS by four lanes each (1.28 ms).
template <bool ANY, bool STATS>
__global__ __launch_bounds__(kMaxBlock) void bvh2_trace(Bvh2Params P) {
    constexpr int SENTINEL = 0x76543210;
    extern __shared__ int lds_stack_raw_i[];
    CWD_LDS int* lds_stack_i = lds_ptr(lds_stack_raw_i);
    // `share` rays per wave
    const int slot = (int)(threadIdx.x & 63u);
    const int i = (int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * P.share + slot;
    if (slot >= P.share || i >= P.n) return;
    int spill[kBvh2StackCapacity];
    const StackIndex sx((int)threadIdx.x, P.lds_depth);

    int ri = P.order ? P.order[i] : i;
    if ((unsigned)ri >= (unsigned)P.n) ri = i;  // malformed order: stay in bounds
    const float4 ro = nt_load4(&P.rays[ri].o);
    const float4 rd = nt_load4(&P.rays[ri].d);
    const float3 o = make_float3(ro.x, ro.y, ro.z), d = make_float3(rd.x, rd.y, rd.z);
    const float tmin = ro.w;
    float hitT = rd.w;
    float idx, idy, idz;
    safe_rcp3(d, idx, idy, idz);
    const float oodx = o.x * idx, oody = o.y * idy, oodz = o.z * idz;
    unsigned long long st_nodes = 0, st_tris = 0;

    int sp = 0;
    stack_put(lds_stack_i, spill, sx, 0, SENTINEL);
    int node = 0, leaf = 0, hit_addr = -1;
    float hu = 0.f, hv = 0.f;
    bool done = false;
    while (node != SENTINEL) {
        leaf = 0;
        while (node != SENTINEL && node >= 0) {
            const float4* np = P.nodes + node;
            const float4 n0 = np[0], n1 = np[1], n2 = np[2], n3 = np[3];
            if (STATS) ++st_nodes;
            float d0, d1;
            const bool t0 = box2(n0.x, n0.y, n0.z, n0.w, n2.x, n2.y, idx, idy, idz, oodx, oody, oodz, tmin, hitT, d0);
            const bool t1 = box2(n1.x, n1.y, n1.z, n1.w, n2.z, n2.w, idx, idy, idz, oodx, oody, oodz, tmin, hitT, d1);
            const int c0 = f2i(n3.x), c1 = f2i(n3.y);
            if (!t0 && !t1) {
                node = stack_get(lds_stack_i, spill, sx, sp);
                --sp;
            } else {
                node = t0 ? c0 : c1;
                if (t0 && t1) {
                    int far = c1;
                    if (d1 < d0) {
                        far = node;
                        node = c1;
                    }
                    if (sp + 1 < kBvh2StackCapacity) {
                        ++sp;
                        stack_put(lds_stack_i, spill, sx, sp, far);
                    } else {
                        P.work[kWorkOverflow] = 1u;
                    }
                }
            }
            if (node < 0 && leaf >= 0) {
                leaf = node;
                node = stack_get(lds_stack_i, spill, sx, sp);
                --sp;
            }
            if (!__any(leaf >= 0)) break;
        }
        while (leaf < 0) {
            for (int a = ~leaf;; a += 3) {
                const float4 v0 = P.tris[a];
                const float4 v1 = P.tris[min(a + 1, P.woop_last)];
                const float4 v2 = P.tris[min(a + 2, P.woop_last)];
                if (f2u(v0.x) == 0x80000000u) break;
                if (STATS) ++st_tris;
                float t, u, v;
                if (woop_test<ANY>(v0, v1, v2, o, d, tmin, hitT, a, hit_addr, t, u, v)) {
                    hitT = t;
                    hit_addr = a;
                    hu = u;
                    hv = v;
                    if (ANY) {
                        done = true;
                        break;
                    }
                }
            }
            if (done) break;
            leaf = node;
            if (node < 0) {
                node = stack_get(lds_stack_i, spill, sx, sp);
                --sp;
            }
        }
        if (done) break;
    }
    const int out_id = (hit_addr >= 0 && P.prim_id) ? P.prim_map[hit_addr] : hit_addr;
    nt_store4(make_float4(hitT, i2f(out_id), hu, hv), &P.hits[ri]);
    if (STATS) {
        atomicAdd(&P.stats[0], st_nodes);
        atomicAdd(&P.stats[1], st_tris);
    }
}

// Persistent BVH2 traversal.  One thread per ray leaves a lane idle from the
// moment its ray ends until the slowest ray of its wave ends (33 M AO rays on
// a 1 M-triangle scene of icospheres: 34% VALU lane use).  Here a grid sized to the device keeps its waves and
// hands rays to idle lanes: rays are claimed `chunk` at a time from `slices`
// contiguous ranges (a wave starts with the range of its XCD) and given to the
// idle lanes by ballot rank.  Each lane runs the while-while rounds of
// bvh2_trace on its ray unchanged (a round: node steps until every lane of the
// wave holds a leaf, then the leaves), so each ray's visits and tests, and its
// hit, are the same.  After each round a wave counts its idle lanes; once it
// has lost `idle_budget` lane-rounds beyond `idle_lanes` per round, it leaves
// the rounds to refill.  The last block to exit resets the claim counters.
template <bool ANY, bool STATS>
__global__ __launch_bounds__(kMaxBlock) void bvh2_trace_persistent(Bvh2Params P) {
    constexpr int SENTINEL = 0x76543210;
    extern __shared__ int lds_stack_raw_i[];
    CWD_LDS int* lds_stack_i = lds_ptr(lds_stack_raw_i);
    int spill[kBvh2StackCapacity];
    const StackIndex sx((int)threadIdx.x, P.lds_depth);
    const int lane = lane_id();

    int out_idx = 0;
    float3 o = make_float3(0.f, 0.f, 0.f), d = o;
    float tmin = 0.f, hitT = 0.f, idx = 0.f, idy = 0.f, idz = 0.f, oodx = 0.f, oody = 0.f, oodz = 0.f;
    int sp = 0, node = SENTINEL, leaf = 0, hit_addr = -1;
    float hu = 0.f, hv = 0.f;
    bool busy = false;
    unsigned long long st_nodes = 0, st_tris = 0;

    // wave-uniform claim state
    unsigned pool_next = 0, pool_end = 0;
    bool exhausted = false;
    const int home = (int)(blockIdx.x % (unsigned)P.slices);
    int slice_k = 0;
    const unsigned first_index =
        (blockIdx.x / (unsigned)P.slices) * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    while (true) {
        const bool idle = !busy;
        unsigned long long need = __ballot(idle);
        bool got = false;
        unsigned my = 0;
        while (need != 0ull) {
            if (pool_next >= pool_end) {
                if (exhausted) break;
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
            const unsigned avail = pool_end - pool_next;
            const unsigned rank = (unsigned)__popcll(need & lanemask_lt());
            if (((need >> lane) & 1ull) && rank < avail) {
                my = pool_next + rank;
                got = true;
            }
            pool_next += min((unsigned)__popcll(need), avail);
            need = __ballot(idle && !got);
        }
        if (idle && !got) break;  // no rays left for this lane

        if (got) {
            int ri = P.order ? P.order[my] : (int)my;
            if ((unsigned)ri >= (unsigned)P.n) ri = (int)my;  // malformed order: stay in bounds
            out_idx = ri;
            const float4 ro = nt_load4(&P.rays[ri].o);
            const float4 rd = nt_load4(&P.rays[ri].d);
            o = make_float3(ro.x, ro.y, ro.z);
            d = make_float3(rd.x, rd.y, rd.z);
            tmin = ro.w;
            hitT = rd.w;
            safe_rcp3(d, idx, idy, idz);
            oodx = o.x * idx;
            oody = o.y * idy;
            oodz = o.z * idz;
            sp = 0;
            stack_put(lds_stack_i, spill, sx, 0, SENTINEL);
            node = 0;
            hit_addr = -1;
            hu = hv = 0.f;
            busy = true;
        }

        int lost = 0;
        while (true) {
            bool done = false;
            leaf = 0;
            while (node != SENTINEL && node >= 0) {
                const float4* np = P.nodes + node;
                const float4 n0 = np[0], n1 = np[1], n2 = np[2], n3 = np[3];
                if (STATS) ++st_nodes;
                float d0, d1;
                const bool t0 = box2(n0.x, n0.y, n0.z, n0.w, n2.x, n2.y, idx, idy, idz, oodx, oody, oodz, tmin, hitT, d0);
                const bool t1 = box2(n1.x, n1.y, n1.z, n1.w, n2.z, n2.w, idx, idy, idz, oodx, oody, oodz, tmin, hitT, d1);
                const int c0 = f2i(n3.x), c1 = f2i(n3.y);
                if (!t0 && !t1) {
                    node = stack_get(lds_stack_i, spill, sx, sp);
                    --sp;
                } else {
                    node = t0 ? c0 : c1;
                    if (t0 && t1) {
                        int far = c1;
                        if (d1 < d0) {
                            far = node;
                            node = c1;
                        }
                        if (sp + 1 < kBvh2StackCapacity) {
                            ++sp;
                            stack_put(lds_stack_i, spill, sx, sp, far);
                        } else {
                            P.work[kWorkOverflow] = 1u;
                        }
                    }
                }
                if (node < 0 && leaf >= 0) {
                    leaf = node;
                    node = stack_get(lds_stack_i, spill, sx, sp);
                    --sp;
                }
                if (!__any(leaf >= 0)) break;
            }
            while (leaf < 0) {
                for (int a = ~leaf;; a += 3) {
                    const float4 v0 = P.tris[a];
                    const float4 v1 = P.tris[min(a + 1, P.woop_last)];
                    const float4 v2 = P.tris[min(a + 2, P.woop_last)];
                    if (f2u(v0.x) == 0x80000000u) break;
                    if (STATS) ++st_tris;
                    float t, u, v;
                    if (woop_test<ANY>(v0, v1, v2, o, d, tmin, hitT, a, hit_addr, t, u, v)) {
                        hitT = t;
                        hit_addr = a;
                        hu = u;
                        hv = v;
                        if (ANY) {
                            done = true;
                            break;
                        }
                    }
                }
                if (done) break;
                leaf = node;
                if (node < 0) {
                    node = stack_get(lds_stack_i, spill, sx, sp);
                    --sp;
                }
            }
            if (done || node == SENTINEL) {
                const int out_id = (hit_addr >= 0 && P.prim_id) ? P.prim_map[hit_addr] : hit_addr;
                nt_store4(make_float4(hitT, i2f(out_id), hu, hv), &P.hits[out_idx]);
                node = SENTINEL;
                busy = false;
                break;
            }
            lost += __popcll(~__ballot(1)) - P.idle_lanes;
            if (lost >= P.idle_budget) break;
        }
    }
    if (STATS) {
        atomicAdd(&P.stats[0], st_nodes);
        atomicAdd(&P.stats[1], st_tris);
    }
    block_exit(P.work, P.total_blocks, P.slices, P.block_q, P.block_r);
}

__global__ void copy_u4_kernel(uint4* __restrict__ dst, const uint4* __restrict__ src, long long n) {
    long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long step = (long long)gridDim.x * blockDim.x;
    for (; i < n; i += step) dst[i] = src[i];
}

// VALU issue-rate probes: `iters` iterations of a fixed vector body on
// independent chains, no memory access but one store per lane at the end, so
// a full grid keeps every SIMD issuing vector instructions back to back.
// Timing one launch against its SQ_INSTS_VALU count gives the issue ceiling
// of that instruction mix:
//   kValuProbeFma   8 chains of FP32 fma;
//   kValuProbeInt   8 chains of 32-bit integer add / xor / min3 / max3;
//   kValuProbeSlab  two 4-child quantized slab tests per iteration (the
//                   node-visit body of cwbvh_trace: byte->float conversions,
//                   fma, integer-ordered min3/max3, mask logic) on operands
//                   that change every iteration.
constexpr int kValuProbeFma = 0;
constexpr int kValuProbeInt = 1;
constexpr int kValuProbeSlab = 2;

// Every binary32 pattern x, by magnitude: counts[0] += |x| in [2^-125, 2^125]
// and rcp_refined(x) differs from 1.0f / x; counts[1] += |x| in that range;
// counts[2] += |x| outside it and the two differ.
__global__ __launch_bounds__(256) void rcp_check_kernel(unsigned long long* __restrict__ counts) {
    const unsigned long long total = 1ull << 32;
    const unsigned long long stride = (unsigned long long)gridDim.x * blockDim.x;
    unsigned long long bad_in = 0, n_in = 0, bad_out = 0;
    for (unsigned long long i = (unsigned long long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        const float x = u2f((unsigned)i);
        const bool in_range = fabsf(x) >= 0x1p-125f && fabsf(x) <= 0x1p125f;
        const bool differ = f2u(rcp_refined(x)) != f2u(1.0f / x);
        bad_in += (in_range && differ) ? 1 : 0;
        n_in += in_range ? 1 : 0;
        bad_out += (!in_range && differ) ? 1 : 0;
    }
    atomicAdd(&counts[0], bad_in);
    atomicAdd(&counts[1], n_in);
    atomicAdd(&counts[2], bad_out);
}

template <int MODE>
__global__ __launch_bounds__(256) void valu_probe_kernel(float* __restrict__ out, long long iters, float a, float b) {
    const unsigned tid = blockIdx.x * blockDim.x + threadIdx.x;
    float f[8];
    unsigned u[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        f[k] = (float)(tid + k) * 1e-7f;
        u[k] = tid * 2654435761u + (unsigned)k * 40503u;
    }
    for (long long i = 0; i < iters; ++i) {
        if constexpr (MODE == kValuProbeFma) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int k = 0; k < 8; ++k) f[k] = __builtin_fmaf(f[k], a, b);
        } else if constexpr (MODE == kValuProbeInt) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const int x = (int)(u[k] + (unsigned)r), y = (int)(u[(k + 1) & 7] ^ 0x5bd1e995u);
                    u[k] = (unsigned)max(max(x, y), (int)u[(k + 3) & 7]) ^ (unsigned)min(min(x, y), (int)u[(k + 5) & 7]);
                }
        } else {
            const unsigned s = (unsigned)i;
            const unsigned h0 = child_hits4(u[0] ^ s, u[1] + s, u[2] ^ s, u[3] + s, u[4] ^ s, u[5] + s, u[6] ^ s, f[0], f[1],
                                            f[2], f[3], f[4], f[5], a, b, u[7]);
            const unsigned h1 = child_hits4(u[7] ^ s, u[6] + s, u[5] ^ s, u[4] + s, u[3] ^ s, u[2] + s, u[1] ^ s, f[2], f[0],
                                            f[1], f[5], f[3], f[4], a, b, u[0]);
            u[0] ^= h0;
            u[7] += h1;
            f[0] = __builtin_fmaf(f[0], a, b);
            f[3] = __builtin_fmaf(f[3], a, b);
        }
    }
    float acc = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) acc += f[k] + (float)u[k];
    out[tid] = acc;
}

template <bool ANY, bool STATS>
int32_t launch_bvh2_t(Bvh2Params& p, const cwbvh_trace_config& cfg, bool persistent, hipStream_t stream) {
    const int block = cfg.block_size;
    const size_t lds = (size_t)block * (size_t)cfg.lds_depth * sizeof(int);
    if (!persistent) {
        // One wave per block, whatever block_size says: the waves share nothing,
        // and a block of several keeps the registers and LDS of those that ended
        // until its last one ends.  1 M-triangle spheres, AO rays, closest hit, us
        // for blocks of 256 / 128 / 64 threads: 4,000 rays 79 / 74 / 73, 150 k 118 /
        // 110 / 107, 780 k 214 / 211 / 199, 8.2 M 1156 / 1159 / 1103.
        // Not so for a million rays and more in a scene that fits one XCD's 4 MB of L2: its
        // waves are short and end together, and dispatching them one by one costs
        // 1-4% (heightfields, us for blocks of 256 / 64: 0.5 MB 2 M rays 236 / 241, 8 M
        // 876 / 913; 3.1 MB 1 M 196 / 195, 2 M 357 / 361, 8 M 1298 / 1333; but 6.1 MB 2 M
        // 445 / 431, 8 M 1631 / 1571).
        // Elsewhere what a block per wave saves at the end of a launch outweighs the
        // dispatching until about 25 M rays (1 M-triangle spheres, any hit, us for
        // blocks of 256 / 64: 8.2 M 1231 / 1187, 14.5 M 2139 / 2105, 20 M 2881 / 2856,
        // 33 M 3973 / 3984).
        const int one_block = p.n >= (p.in_l2 ? 1 << 20 : 3 << 23) ? block : 64;
        // A launch too small to fill the device gives each wave fewer rays: a wave
        // lasts as long as the visits that its rays make in turn.  The smallest
        // share that needs at most 4 waves per SIMD, up to 16 rays (us for 64 / 16 /
        // 8 / 4 / 1 rays per wave: 1,000 rays 44 / 40 / 35 / 35 / 29; 8,000 rays 63
        // / 56 / 57 / 52 / 56; 32,000 rays 71 / 64 / 64 / 64 / 136; 64,000 rays 74 /
        // 72 / 80 / 112; 100,000 rays 80 / 87, and 81 for 32)
        const long long waves = 16ll * cw::device_compute_units();
        p.share = 1;
        while (p.share < 64 && ((long long)p.n + p.share - 1) / p.share > waves) p.share *= p.share < 16 ? 2 : 4;
        const long long per_block = (long long)p.share * (one_block / 64);
        const long long grid = ((long long)p.n + per_block - 1) / per_block;
        const size_t block_lds = (size_t)one_block * (size_t)cfg.lds_depth * sizeof(int);
        hipLaunchKernelGGL((bvh2_trace<ANY, STATS>), dim3((unsigned)grid), dim3(one_block), block_lds, stream, p);
        CW_HIP(hipGetLastError());
        return CWBVH_OK;
    }
    auto kernel = bvh2_trace_persistent<ANY, STATS>;
    long long grid = cfg.grid_blocks;
    if (grid <= 0) grid = (long long)resident_blocks(kernel, block, lds) * cw::device_compute_units();
    p.total_blocks = (int)grid;
    p.slices = cfg.work_slices;
    p.idle_lanes = cfg.refill_idle;
    p.idle_budget = cfg.refill_budget;
    p.chunk = cfg.fetch_chunk;
    set_splits(p);
    if (p.chunk <= 0) {
        // automatic: about 32 claims per wave over the launch, 128..512 rays each
        const long long waves = grid * (block / 64);
        long long c = (long long)p.n / (waves * 32);
        c = std::min<long long>(512, std::max<long long>(128, (c + 63) / 64 * 64));
        p.chunk = (int)c;
    }
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(block), lds, stream, p);
    CW_HIP(hipGetLastError());
    return CWBVH_OK;
}

template <bool ANY, bool STATS, bool MULTI>
int32_t dispatch_prefetch(CwbvhParams& p, const cwbvh_trace_config& cfg, hipStream_t st) {
    return cfg.prefetch ? dispatch_loop<ANY, STATS, MULTI, true>(p, cfg, st)
                        : dispatch_loop<ANY, STATS, MULTI, false>(p, cfg, st);
}

template <bool MULTI>
int32_t dispatch_cwbvh(CwbvhParams& p, uint32_t flags, const cwbvh_trace_config& cfg, hipStream_t st) {
    const bool any = (flags & CWBVH_TRACE_ANY) != 0, stats = (flags & CWBVH_TRACE_STATS) != 0;
    if (any) return stats ? dispatch_prefetch<true, true, MULTI>(p, cfg, st) : dispatch_prefetch<true, false, MULTI>(p, cfg, st);
    return stats ? dispatch_prefetch<false, true, MULTI>(p, cfg, st) : dispatch_prefetch<false, false, MULTI>(p, cfg, st);
}

template <bool ANY, bool STATS>
int32_t dispatch_surfels(CwbvhParams& p, const cwbvh_trace_config& cfg, hipStream_t st) {
    switch (cfg.loop_mode) {
        case kLoopInterleave:
            if constexpr (!STATS) {
                const bool w7 = cfg.occupancy == kOccupancy7 ||
                                (cfg.occupancy == kOccupancyAuto && (long long)p.n >= kOccupancy7MinSurfelRays);
                if (p.lds_only) {
                    if (w7) return launch_cwbvh_t<ANY, false, false, false, kLoopInterleave, kRaysFromSurfels, true, true>(p, cfg, st);
                    return launch_cwbvh_t<ANY, false, false, false, kLoopInterleave, kRaysFromSurfels, false, true>(p, cfg, st);
                }
                if (w7) return launch_cwbvh_t<ANY, false, false, false, kLoopInterleave, kRaysFromSurfels, true>(p, cfg, st);
            }
            return launch_cwbvh_t<ANY, STATS, false, false, kLoopInterleave, kRaysFromSurfels>(p, cfg, st);
        case kLoopSpeculate: return launch_cwbvh_t<ANY, STATS, false, false, kLoopSpeculate, kRaysFromSurfels>(p, cfg, st);
        default: return launch_cwbvh_t<ANY, STATS, false, false, kLoopGroup, kRaysFromSurfels>(p, cfg, st);
    }
}

// Spread nodes from 80 B or 128 B ones: one thread per 16-byte slot.
__global__ __launch_bounds__(256) void spread_nodes_kernel(const float4* __restrict__ nodes, long long num_nodes, int stride,
                                                           float4* __restrict__ out) {
    const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= num_nodes * 8) return;
    const long long i = t >> 3;
    const int slot = (int)(t & 7) ^ (int)(i & 7);   // the slot stored at place t mod 8 of node i
    out[t] = slot < 5 ? nodes[i * stride + slot] : make_float4(0.f, 0.f, 0.f, 0.f);
}

// One thread per ray: the unfused generator (same arithmetic as the fused one).
__global__ void surfel_rays_kernel(const float4* __restrict__ pos, const float4* __restrict__ nrm,
                                   const float* __restrict__ rad, long long n_rays, int rays_per_texel, float tmin,
                                   float tmax, unsigned long long seed, Ray4* __restrict__ out) {
    const long long r = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n_rays) return;
    const long long t = r / rays_per_texel;
    const float4 p = pos[t], n = nrm[t];
    cwao::F3 o, d;
    cwao::surfel_ray(cwao::F3{p.x, p.y, p.z}, cwao::F3{n.x, n.y, n.z}, rad[t], seed, (unsigned long long)r, o, d);
    nt_store4(make_float4(o.x, o.y, o.z, tmin), &out[r].o);
    nt_store4(make_float4(d.x, d.y, d.z, tmax), &out[r].d);
}

}  // namespace

namespace cw {

using namespace cwk;

int32_t validate_config(int32_t kind, const cwbvh_trace_config& c) {
    if (!(c.block_size == 64 || c.block_size == 128 || c.block_size == 256)) {
        set_error("block_size must be 64, 128 or 256");
        return CWBVH_ERR_INVALID_ARGUMENT;
    }
    const int cap = kind == CWBVH_KIND_CWBVH ? kStackCapacity : kBvh2StackCapacity;
    if (c.lds_depth < 1 || c.lds_depth > cap) {
        set_error("lds_depth must be in [1, stack capacity]");
        return CWBVH_ERR_INVALID_ARGUMENT;
    }
    const size_t lds = (size_t)c.block_size * c.lds_depth * (kind == CWBVH_KIND_CWBVH ? 8 : 4);
    if (lds > 160 * 1024) {
        set_error("LDS stack exceeds 160 KiB per block");
        return CWBVH_ERR_INVALID_ARGUMENT;
    }
    if (c.ray_order < 0 || c.ray_order > 1) {
        set_error("ray_order must be 0 or 1");
        return CWBVH_ERR_INVALID_ARGUMENT;
    }
    if (kind == CWBVH_KIND_CWBVH) {
        if (c.fetch_chunk < 0 || c.fetch_chunk > (1 << 20) || c.grid_blocks < 0 || c.refill_budget < 1 ||
            c.persistent < 0 || c.persistent > 2 ||
            c.refill_idle < 0 || c.refill_idle > 64 || c.postpone_pct < 0 || c.postpone_pct > 100 ||
            c.prefetch < 0 || c.prefetch > 1 || c.work_slices < 1 || c.work_slices > kWorkSlices ||
            c.loop_mode < kLoopGroup || c.loop_mode > kLoopQueue ||
            !(c.occupancy == kOccupancyAuto || c.occupancy == kOccupancyFree || c.occupancy == kOccupancy7)) {
            set_error("invalid CWBVH trace configuration");
            return CWBVH_ERR_INVALID_ARGUMENT;
        }
        if (c.loop_mode == kLoopQueue) {
            set_error("loop_mode 3 (triangle queue) is switched off: use 0, 1 or 2");
            return CWBVH_ERR_INVALID_ARGUMENT;
        }
        if (c.postpone_pct > 0 && c.loop_mode == kLoopInterleave) {
            set_error("postpone_pct applies to loop_mode 0 and 2");
            return CWBVH_ERR_INVALID_ARGUMENT;
        }
    } else {
        // BVH2: one ray per thread (persistent 0) or the persistent grid
        // (1, or 2 = automatic by ray count), whose claim and refill fields
        // then apply; the CWBVH-only fields must stay 0
        if (c.persistent < 0 || c.persistent > 2 || c.loop_mode != 0 || c.prefetch != 0 || c.postpone_pct != 0 ||
            c.occupancy != 0) {
            set_error("invalid BVH2 trace configuration: persistent is 0, 1 or 2; loop_mode, prefetch, "
                      "postpone_pct and occupancy are 0");
            return CWBVH_ERR_INVALID_ARGUMENT;
        }
        if (c.persistent != 0 && (c.fetch_chunk < 0 || c.fetch_chunk > (1 << 20) || c.grid_blocks < 0 ||
                                  c.refill_budget < 1 || c.refill_idle < 0 || c.refill_idle > 64 ||
                                  c.work_slices < 1 || c.work_slices > kWorkSlices)) {
            set_error("invalid BVH2 persistent configuration (refill_budget >= 1, refill_idle in [0, 64], "
                      "work_slices in [1, 8])");
            return CWBVH_ERR_INVALID_ARGUMENT;
        }
    }
    return CWBVH_OK;
}

// A tree whose stack need (known from its layout, or declared when caller
// arrays are wrapped) fits the LDS part of the stack is traversed by kernels
// without the scratch part.
static bool lds_only(const cwbvh_scene* s, const cwbvh_trace_config& c) {
    return s->stack_need > 0 && s->stack_need <= c.lds_depth && c.lds_depth <= kStackCapacity;
}

// Persistent grid or one ray per lane; configuration value 2 = automatic: below
// the line the grid's fixed start-up and exit cost outweighs its load balancing.
static int persistent_grid(const TraceLaunch& L, bool surfels) {
    if (L.cfg.persistent != 2) return L.cfg.persistent;
    const bool teams = L.cfg.loop_mode == kLoopInterleave && !(L.flags & CWBVH_TRACE_STATS) && L.cfg.occupancy != kOccupancy7;
    return L.n >= auto_persistent_rays((L.flags & CWBVH_TRACE_ANY) != 0, surfels, teams, L.scene->bytes > kCacheResidentBytes);
}

// The spread nodes of a scene serve its LDS-only interleaved launches (no
// counters, rays from a buffer, the build for 6 or fewer waves).
static void choose_nodes(CwbvhParams& p, const TraceLaunch& L) {
    const cwbvh_trace_config& c = L.cfg;
    const bool w7 = !c.prefetch && (c.occupancy == kOccupancy7 ||
                                    (c.occupancy == kOccupancyAuto && L.n >= seven_wave_rays((L.flags & CWBVH_TRACE_ANY) != 0, true)));
    p.spread = p.lds_only && L.scene->spread_nodes && c.loop_mode == kLoopInterleave && !w7 && !(L.flags & CWBVH_TRACE_STATS);
    if (p.spread) p.nodes = (const float4*)L.scene->spread_nodes;
}

int32_t launch_cwbvh(const TraceLaunch& L) {
    const cwbvh_scene* s = L.scene;
    CwbvhParams p{};
    p.nodes = (const float4*)s->nodes;
    p.tris = (const float4*)s->woop;
    p.prim_map = s->prim_idx;
    p.rays = (const Ray4*)L.rays;
    p.order = L.order;
    p.hits = (float4*)L.hits;
    p.jobs = nullptr;
    p.work = L.counters;
    p.stats = (unsigned long long*)L.stats;
    p.n = (int)L.n;
    p.num_jobs = 0;
    p.stride = s->node_stride;
    p.lds_depth = L.cfg.lds_depth;
    p.chunk = L.cfg.fetch_chunk;
    p.idle_lanes = L.cfg.refill_idle;
    p.idle_budget = L.cfg.refill_budget;
    p.postpone_pct = L.cfg.postpone_pct;
    p.prim_id = (L.flags & CWBVH_TRACE_PRIM_ID) ? 1 : 0;
    p.slices = L.cfg.work_slices;
    p.persistent = persistent_grid(L, false);
    p.spec_limit = cw::speculation_limit(s->stack_need);
    p.lds_only = lds_only(s, L.cfg) ? 1 : 0;
    p.streams = s->bytes > kCacheResidentBytes ? 1 : 0;
    choose_nodes(p, L);
    return dispatch_cwbvh<false>(p, L.flags, L.cfg, L.stream);
}

int32_t launch_spread_nodes(const void* nodes, int64_t num_nodes, int32_t stride, void* out, hipStream_t stream) {
    const long long threads = (long long)num_nodes * 8;
    if (threads == 0) return CWBVH_OK;
    hipLaunchKernelGGL(spread_nodes_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream,
                       (const float4*)nodes, (long long)num_nodes, stride, (float4*)out);
    CW_HIP(hipGetLastError());
    return CWBVH_OK;
}

int32_t launch_cwbvh_surfels(const TraceLaunch& L) {
    if (L.cfg.prefetch != 0) {
        set_error("surfel traces do not use node prefetch");
        return CWBVH_ERR_INVALID_ARGUMENT;
    }
    const cwbvh_scene* s = L.scene;
    CwbvhParams p{};
    p.nodes = (const float4*)s->nodes;
    p.tris = (const float4*)s->woop;
    p.prim_map = s->prim_idx;
    p.rays = nullptr;
    p.order = nullptr;
    p.hits = (float4*)L.hits;
    p.work = L.counters;
    p.stats = (unsigned long long*)L.stats;
    p.n = (int)L.n;
    p.stride = s->node_stride;
    p.lds_depth = L.cfg.lds_depth;
    p.chunk = L.cfg.fetch_chunk;
    p.idle_lanes = L.cfg.refill_idle;
    p.idle_budget = L.cfg.refill_budget;
    p.postpone_pct = L.cfg.postpone_pct;
    p.prim_id = (L.flags & CWBVH_TRACE_PRIM_ID) ? 1 : 0;
    p.slices = L.cfg.work_slices;
    p.persistent = persistent_grid(L, true);
    p.spec_limit = cw::speculation_limit(s->stack_need);
    p.lds_only = lds_only(s, L.cfg) ? 1 : 0;
    p.surf_pos = (const float4*)L.surf_pos;
    p.surf_nrm = (const float4*)L.surf_nrm;
    p.surf_rad = L.surf_rad;
    p.rays_per_texel = L.rays_per_texel;
    p.gen_tmin = L.gen_tmin;
    p.gen_tmax = L.gen_tmax;
    p.seed = L.seed;
    p.texel_hits = L.texel_hits;
    const bool any = (L.flags & CWBVH_TRACE_ANY) != 0, stats = (L.flags & CWBVH_TRACE_STATS) != 0;
    if (any) return stats ? dispatch_surfels<true, true>(p, L.cfg, L.stream) : dispatch_surfels<true, false>(p, L.cfg, L.stream);
    return stats ? dispatch_surfels<false, true>(p, L.cfg, L.stream) : dispatch_surfels<false, false>(p, L.cfg, L.stream);
}

int32_t launch_surfel_rays(const cwbvh_float4* pos, const cwbvh_float4* nrm, const float* rad, int64_t num_texels,
                           int32_t rays_per_texel, float tmin, float tmax, uint64_t seed, cwbvh_ray* out,
                           hipStream_t stream) {
    const long long n = (long long)num_texels * rays_per_texel;
    if (n == 0) return CWBVH_OK;
    const int block = 256;
    hipLaunchKernelGGL(surfel_rays_kernel, dim3((unsigned)((n + block - 1) / block)), dim3(block), 0, stream,
                       (const float4*)pos, (const float4*)nrm, rad, n, rays_per_texel, tmin, tmax,
                       (unsigned long long)seed, (Ray4*)out);
    CW_HIP(hipGetLastError());
    return CWBVH_OK;
}

// About 4 claims per resident wave (5 per SIMD), 64 to 256 rays each: fewer
// leave the waves unevenly loaded at the end, more cost claims (MI355X, us at
// 64 / 128 / 192 / 256 rays: 136 k rays in 12 jobs 94 / 113 / 133 / 150; 4.6 M
// rays in 40 jobs 410 / 378 / 389 / 395, and 348 / 326 / 321 / 323 with batches of
// other streams overlapping; 27 M rays in 32 jobs 2139 / 1882 / 1823 / 1815).
// Launches that give each wave one chunk of 8 or 16 rays, traced by teams of
// lanes from the start, do so up to 4 waves per SIMD, as single-scene launches do.
int32_t batch_chunk(int64_t total_rays) {
    const int64_t simds = 4ll * device_compute_units();
    if (total_rays <= 8 * 4 * simds) return 8;
    if (total_rays <= 16 * 4 * simds) return 16;
    const int64_t c = total_rays / (5 * simds * 4) / 64 * 64;
    return (int32_t)std::min<int64_t>(256, std::max<int64_t>(64, c));
}

int32_t launch_cwbvh_batch(const BatchLaunch& L) {
    if (L.cfg.fetch_chunk <= 0) {
        set_error("batch launch needs the chunk size its job table was planned with");
        return CWBVH_ERR_INVALID_ARGUMENT;
    }
    CwbvhParams p{};
    p.jobs = L.d_jobs;
    p.num_jobs = L.num_jobs;
    p.job_step = (L.num_jobs + 63) / 64;
    p.n = (int)L.total_chunks;
    p.work = L.counters;
    p.stats = (unsigned long long*)L.stats;
    p.lds_depth = L.cfg.lds_depth;
    p.chunk = L.cfg.fetch_chunk;
    p.idle_lanes = L.cfg.refill_idle;
    p.idle_budget = L.cfg.refill_budget;
    p.postpone_pct = L.cfg.postpone_pct;
    p.prim_id = (L.flags & CWBVH_TRACE_PRIM_ID) ? 1 : 0;
    p.slices = L.cfg.work_slices;
    p.persistent = 1;
    p.lds_only = L.lds_only;
    return dispatch_cwbvh<true>(p, L.flags, L.cfg, L.stream);
}

int32_t launch_bvh2(const TraceLaunch& L) {
    const cwbvh_scene* s = L.scene;
    Bvh2Params p{};
    p.nodes = (const float4*)s->nodes;
    p.tris = (const float4*)s->woop;
    p.prim_map = s->prim_idx;
    p.rays = (const Ray4*)L.rays;
    p.order = L.order;
    p.hits = (float4*)L.hits;
    p.work = L.counters;
    p.stats = (unsigned long long*)L.stats;
    p.n = (int)L.n;
    p.lds_depth = L.cfg.lds_depth;
    p.woop_last = s->woop_f4 > 0 ? (int)(s->woop_f4 - 1) : 0x7FFFFFFF;
    p.prim_id = (L.flags & CWBVH_TRACE_PRIM_ID) ? 1 : 0;
    p.in_l2 = s->bytes > 0 && s->bytes <= (4ll << 20);
    // persistent 2 = automatic: the persistent grid from kAutoPersistentRays up
    const bool pers = L.cfg.persistent == 2 ? L.n >= cw::kAutoPersistentRays : L.cfg.persistent == 1;
    const bool any = (L.flags & CWBVH_TRACE_ANY) != 0, stats = (L.flags & CWBVH_TRACE_STATS) != 0;
    if (any) return stats ? launch_bvh2_t<true, true>(p, L.cfg, pers, L.stream) : launch_bvh2_t<true, false>(p, L.cfg, pers, L.stream);
    return stats ? launch_bvh2_t<false, true>(p, L.cfg, pers, L.stream) : launch_bvh2_t<false, false>(p, L.cfg, pers, L.stream);
}

}  // namespace cw

extern "C" int32_t cwbvh_copy_u4(void* dst, const void* src, int64_t n_u4, void* stream) {
    CW_CHECK_ARG(n_u4 >= 0 && (n_u4 == 0 || (dst && src)), "bad copy arguments");
    if (n_u4 == 0) return CWBVH_OK;
    const int block = 256;
    long long grid = (n_u4 + block - 1) / block;
    if (grid > 65536) grid = 65536;
    hipLaunchKernelGGL(copy_u4_kernel, dim3((unsigned)grid), dim3(block), 0, (hipStream_t)stream, (uint4*)dst,
                       (const uint4*)src, (long long)n_u4);
    CW_HIP(hipGetLastError());
    return CWBVH_OK;
}

extern "C" int32_t cwbvh_rcp_check(uint64_t* d_counts, void* stream) {
    CW_CHECK_ARG(d_counts != nullptr, "d_counts is null");
    hipStream_t st = (hipStream_t)stream;
    CW_HIP(hipMemsetAsync(d_counts, 0, 3 * sizeof(uint64_t), st));
    hipLaunchKernelGGL(rcp_check_kernel, dim3(8192), dim3(256), 0, st, (unsigned long long*)d_counts);
    CW_HIP(hipGetLastError());
    return CWBVH_OK;
}

extern "C" int32_t cwbvh_valu_probe(int32_t mode, int64_t iters, int32_t blocks, float* d_out, void* stream) {
    CW_CHECK_ARG(mode >= kValuProbeFma && mode <= kValuProbeSlab, "mode must be 0, 1 or 2");
    CW_CHECK_ARG(iters >= 1 && blocks >= 1 && blocks <= (1 << 20) && d_out != nullptr, "bad probe arguments");
    const dim3 grid((unsigned)blocks), block(256);
    hipStream_t st = (hipStream_t)stream;
    if (mode == kValuProbeFma)
        hipLaunchKernelGGL(valu_probe_kernel<kValuProbeFma>, grid, block, 0, st, d_out, (long long)iters, 0.999f, 1e-7f);
    else if (mode == kValuProbeInt)
        hipLaunchKernelGGL(valu_probe_kernel<kValuProbeInt>, grid, block, 0, st, d_out, (long long)iters, 0.999f, 1e-7f);
    else
        hipLaunchKernelGGL(valu_probe_kernel<kValuProbeSlab>, grid, block, 0, st, d_out, (long long)iters, 0.999f, 1e-7f);
    CW_HIP(hipGetLastError());
    return CWBVH_OK;
}
