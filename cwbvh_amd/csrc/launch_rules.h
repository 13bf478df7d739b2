// How launches are laid out by their size: host code without HIP.  Ray counts
// reach 2^31 - 1, so sums with them are 64-bit.
#pragma once

#include <cstdint>

namespace cw {

// cwbvh_trace_config.persistent == 2: persistent grid from this many rays up
// (MI355X, AO rays on a 65 k-triangle heightfield: one ray per thread 0.142
// against 0.164 ms at 2^19 rays, 0.230 against 0.200 ms at 2^20).
constexpr int64_t kAutoPersistentRays = 3ll << 18;
// CWBVH any hit: its shorter rays end with teams of lanes in every wave of a
// one-ray-per-lane launch, and a persistent grid of short rays queues on its
// claims.  us one ray per lane / persistent, at 1.05 M rays: AO on 1 M-triangle
// spheres 110 / 127, on 65 k- and 400 k-triangle heightfields 123 / 126 and 165 /
// 149, diffuse rays in a 300 k-triangle soup 420 / 429, camera rays 22 / 59; at
// 1.6 M: 142 / 161, 174 / 167, 229 / 200, 597 / 581, 27 / 68.
constexpr int64_t kAutoPersistentAnyRays = 5ll << 18;
// Rays made from surfels: a refill also makes its rays, for few lanes.  us one
// ray per lane / persistent, any hit, 1 M-triangle spheres and a 200 k-triangle
// heightfield: 0.8 M rays 113 / 121 and 113 / 127, 1.9 M 234 / 255 and 234 / 237,
// 2.9 M 339 / 349 and 340 / 330, 4 M 463 / 470 and 467 / 438.
constexpr int64_t kAutoPersistentSurfelRays = 1ll << 21;

// The line of a launch.  Only kernels with teams of lanes gain from the later
// lines: without them a wave lasts as long as its slowest ray (400 k-triangle
// heightfield, us one ray per lane / persistent, any hit, 1 M AO rays: grouped 278 /
// 229, speculative 247 / 208; 2 M surfel rays, closest hit: 454 / 415, 450 / 342).  Nor
// does any hit in a scene that streams from memory, where a wave's last rays wait on
// loads that teams do not shorten (diffuse rays, 1.3 M: 5 M-triangle soup 1584 / 1358,
// 20 M-triangle soup 1957 / 1578; rays made from surfels in the former at 1.06 M 324 /
// 331, 2 M 585 / 571).
constexpr int64_t auto_persistent_rays(bool any, bool surfels, bool teams, bool streams) {
    if (!teams) return kAutoPersistentRays;
    if (surfels) return kAutoPersistentSurfelRays;
    return any && !streams ? kAutoPersistentAnyRays : kAutoPersistentRays;
}

// Rays per wave of a CWBVH launch without work fetching, for kernels whose waves
// trace their last 16 rays with 4 or 8 lanes each (team_trace): a launch too
// small to fill the device gives each wave only 8 or 16 rays, so that one latency
// chain per ray shrinks from the start.  The limit is 4 waves per SIMD; with more,
// the teams' waves queue behind one another (MI355X, AO rays on a 65 k-triangle
// heightfield, closest hit, us for 64 / 16 / 8 rays per wave: 1,000 rays 37 / 32 /
// 21; 32,000 rays 36 / 32 / 28; 48,000 rays 35 / 32 / 43; 96,000 rays 40 / 69 / 63).
// Up to half a wave per SIMD, 4 rays per wave: the teams of a wave wait for one
// another's loads (same scene, closest hit, us for 8 / 4 / 2 rays per wave: 500 rays
// 20.1 / 17.6 / 17.1, 1,000 20.4 / 18.8 / 18.7, 2,000 20.3 / 20.0 / 19.7; 300
// k-triangle soup, 1,000 rays 50.3 / 49.2 / 52.6, 2,000 50.1 / 48.9 / 48.4, 4,000 50.7
// / 51.1 / 55.6).
constexpr int32_t team_rays_per_wave(int64_t n, int32_t compute_units) {
    const int64_t waves = 16ll * compute_units;
    if ((n + 3) / 4 <= waves / 8) return 4;
    if ((n + 7) / 8 <= waves) return 8;
    if ((n + 15) / 16 <= waves) return 16;
    return 64;
}

// Rays from which launches of the plain interleaved kernels run the 7-wave builds
// (1 M-triangle spheres, AO rays, closest hit, 6 / 7 waves: 4 M rays 381 / 394 us, 5 M
// 472 / 478, 6 M 548 / 547, 8 M 721 / 708, 16 M 1285 / 1240; any hit 5 M 415 / 416, 6 M
// 481 / 477, 8 M 621 / 609).  Any hit with a two-level stack, whose 6-wave build is the
// slower of the two kinds, earlier (4.3 M rays 487 / 467, 5.5 M 605 / 576; heightfields of
// 65 k and 2 M triangles 399 / 400 and 589 / 602, 498 / 487 and 732 / 746; closest hit 567 /
// 567, 698 / 703, 455 / 477, 660 / 713).
constexpr int64_t seven_wave_rays(bool any, bool lds_only) { return any && !lds_only ? 1ll << 22 : 3ll << 21; }

// Waves per SIMD of an automatic persistent grid, 0 = all that fit.  A prefetch
// launch on rays in the caller's order in a scene that streams from memory runs 4: the
// rays in flight share few nodes, and those of a fifth wave evict more from the
// caches than it hides.  (Rays sorted by the launch share many, and from 16 M up 5
// waves are faster.)  5 / 4 / 3 waves, ms: diffuse rays, 20 M-triangle soup, closest hit,
// 16 M 16.41 / 15.72 / 15.67, 4 M 4.39 / 4.20 / 4.20, 1 M 1.44 / 1.36 / 1.38; 5 M triangles
// 13.84 / 13.69 / 13.74, 3.69 / 3.63 / 3.66, 1.18 / 1.14 / 1.17; AO rays in the former 9.90 /
// 9.69 / 10.51, 2.60 / 2.54 / 2.75, 0.79 / 0.78 / 0.83; any hit alike.
constexpr int32_t grid_waves(bool prefetch, bool ordered, bool streams) { return prefetch && !ordered && streams ? 4 : 0; }

}  // namespace cw
