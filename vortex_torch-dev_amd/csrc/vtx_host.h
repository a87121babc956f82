// Host-side helpers of the C ABI: per-thread error message, launch checks.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cstdarg>

#include "../../include/vortex_hip.h"

namespace vtx {

// Records a printf-style message as this thread's last error; returns `code`.
int fail(int code, const char* fmt, ...);

// Clears this thread's last error.
void clear_error();

// Checks the launch that was just issued; returns VTX_OK or VTX_E_LAUNCH.
int check_launch(const char* what);

// Compute units of the current device (cached per device).
int device_cu_count();

inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

// log2(d) when d is a power of two, else -1 (the `shift` of vtx::div_c).
inline int log2_exact(int d) { return d > 0 && (d & (d - 1)) == 0 ? __builtin_ctz((unsigned)d) : -1; }

inline bool aligned16(const void* p) {
  return (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
}

// Threads per workgroup of the fused indexer kernels with one workgroup per
// segment (of at most max_pages pages): 4 or 8 waves for up to 256 or 512
// pages, and past that 16 only where no CU has two workgroups.  Two of 8 waves
// per CU do one's select while the other's rows arrive; alone on a CU, 16 waves
// are faster.  Measured per layer, 8 / 16 waves: block-sparse, 512 segments of
// up to 2048 pages 33.0 / 37.9 us, 256 of up to 1024 pages 16.6 / 14.9; GQA,
// 320 of up to 1024 pages 23.5 / 28.5, 128 of up to 1024 18.7 / 16.6; Quest,
// 384 of up to 2048 pages 60.3 / 63.8, 128 of up to 1024 26.4 / 23.8.
inline int segment_threads(long long segments, long long max_pages, int cus) {
  if (max_pages <= 256) return 256;
  return max_pages <= 512 || segments > cus ? 512 : 1024;
}

}  // namespace vtx
