// The CWBVH launches with node prefetch (the default of scenes larger than the
// Infinity Cache).  They are compiled without SLP vectorization (build.py): it
// groups the 8 children's slab tests into vector operations that keep all
// planes in registers at once, 106 VGPRs (4 waves per SIMD) for the LDS-only
// kernel; without it 93-96 (5 waves).  These launches wait on memory, so waves
// matter most: 5 M-triangle soup, 16.8 M shuffled rays, closest hit: 11.94 ms
// with it, 11.40 ms without.  The kernels without prefetch keep it: they are
// bound by instruction issue, and its grouping is 1-4% faster there (1 M AO
// rays 146 us with it, 151 us without; 33 M AO rays 2.14 and 2.16 ms).
#include "cwbvh_kernel.h"

namespace cwk {

#define CWBVH_PREFETCH_LAUNCHES(ANY, STATS)                                                                           \
    template int32_t dispatch_loop<ANY, STATS, false, true>(CwbvhParams&, const cwbvh_trace_config&, hipStream_t);    \
    template int32_t dispatch_loop<ANY, STATS, true, true>(CwbvhParams&, const cwbvh_trace_config&, hipStream_t);
CWBVH_PREFETCH_LAUNCHES(false, false)
CWBVH_PREFETCH_LAUNCHES(false, true)
CWBVH_PREFETCH_LAUNCHES(true, false)
CWBVH_PREFETCH_LAUNCHES(true, true)
#undef CWBVH_PREFETCH_LAUNCHES

}  // namespace cwk
