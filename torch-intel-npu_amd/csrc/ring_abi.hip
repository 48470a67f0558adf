// Launches of the few-tile GEMM of lb_ring.h (a translation unit of its own, so the library's
// sources compile in parallel).
#include <hip/hip_runtime.h>

#include "lb_ring.h"

namespace lb {

template <int FMT, int SCALE_KB, bool POST, bool RANKED>
void launch_ring_t(const RingParams &p, int rt, int tiles, hipStream_t s) {
  const dim3 grid((unsigned)tiles, (unsigned)((p.M + 16 * rt - 1) / (16 * rt)));
  switch (rt) {
    case 1: hipLaunchKernelGGL((ring_gemm_kernel<FMT, SCALE_KB, POST, RANKED, 1, RING_PLAIN>), grid, dim3(kRingThreads), 0, s, p); break;
    case 2: hipLaunchKernelGGL((ring_gemm_kernel<FMT, SCALE_KB, POST, RANKED, 2, RING_PLAIN>), grid, dim3(kRingThreads), 0, s, p); break;
    default:
      if constexpr (!RANKED) hipLaunchKernelGGL((ring_gemm_kernel<FMT, SCALE_KB, POST, RANKED, 4, RING_PLAIN>), grid, dim3(kRingThreads), 0, s, p);
      break;
  }
}

template <int FMT, bool RANKED>
void launch_ring_scaled(const RingParams &p, int rt, int tiles, hipStream_t s) {
  if (p.group_shift == 5) {
    if (ring_scale_kb(p.G) == 8) launch_ring_t<FMT, 8, false, RANKED>(p, rt, tiles, s);
    else launch_ring_t<FMT, 28, false, RANKED>(p, rt, tiles, s);
  } else {
    if (ring_scale_kb(p.G) == 8) launch_ring_t<FMT, 8, true, RANKED>(p, rt, tiles, s);
    else launch_ring_t<FMT, 28, true, RANKED>(p, rt, tiles, s);
  }
}

void launch_ring(const RingParams &p, int format, bool scaled, bool ranked, int rt, int tiles, hipStream_t s) {
  switch (format) {
    case FMT_INT8:
      if (scaled) ranked ? launch_ring_scaled<FMT_INT8, true>(p, rt, tiles, s) : launch_ring_scaled<FMT_INT8, false>(p, rt, tiles, s);
      else ranked ? launch_ring_t<FMT_INT8, 0, false, true>(p, rt, tiles, s) : launch_ring_t<FMT_INT8, 0, false, false>(p, rt, tiles, s);
      break;
    case FMT_INT4: ranked ? launch_ring_scaled<FMT_INT4, true>(p, rt, tiles, s) : launch_ring_scaled<FMT_INT4, false>(p, rt, tiles, s); break;
    case FMT_NF4: ranked ? launch_ring_scaled<FMT_NF4, true>(p, rt, tiles, s) : launch_ring_scaled<FMT_NF4, false>(p, rt, tiles, s); break;
    default: ranked ? launch_ring_t<FMT_FP16, 0, false, true>(p, rt, tiles, s) : launch_ring_t<FMT_FP16, 0, false, false>(p, rt, tiles, s); break;
  }
}

template <int FMT, int SCALE_KB>
void launch_ring_slices_t(const RingParams &p, int rt, const dim3 &grid, hipStream_t s) {
  if (rt == 1) hipLaunchKernelGGL((ring_gemm_kernel<FMT, SCALE_KB, SCALE_KB != 0, false, 1, RING_SLICE>), grid, dim3(kRingThreads), 0, s, p);
  else if (rt == 2) hipLaunchKernelGGL((ring_gemm_kernel<FMT, SCALE_KB, SCALE_KB != 0, false, 2, RING_SLICE>), grid, dim3(kRingThreads), 0, s, p);
  else hipLaunchKernelGGL((ring_gemm_kernel<FMT, SCALE_KB, SCALE_KB != 0, false, 4, RING_SLICE>), grid, dim3(kRingThreads), 0, s, p);
}

void launch_ring_slices(const RingParams &p, int format, int rt, int tiles, int slices, hipStream_t s) {
  const dim3 grid((unsigned)tiles, (unsigned)((p.M + 16 * rt - 1) / (16 * rt)), (unsigned)slices);
  switch (format) {
    case FMT_INT8: launch_ring_slices_t<FMT_INT8, 0>(p, rt, grid, s); break;
    case FMT_INT4: launch_ring_slices_t<FMT_INT4, 28>(p, rt, grid, s); break;
    default: launch_ring_slices_t<FMT_NF4, 28>(p, rt, grid, s); break;
  }
}

}  // namespace lb
