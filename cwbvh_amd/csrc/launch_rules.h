// How launches are laid out by their size: host code without HIP.  Ray counts
// reach 2^31 - 1, so sums with them are 64-bit.
#pragma once

#include <cstdint>

namespace cw {

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

}  // namespace cw
