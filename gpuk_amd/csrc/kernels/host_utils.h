// Host-side helpers shared by the C-ABI launchers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../../include/gpuk_amd.h"

namespace gpuk {

inline bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
inline bool aligned8(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 7u) == 0; }
inline int round_up(int v, int m) { return (v + m - 1) / m * m; }
inline int hip_status(hipError_t e) { return e == hipSuccess ? GPUK_OK : GPUK_ERR_LAUNCH; }

// Launches a kernel.  A small call is bound by what its launch costs the host, and that grows with the number of kernel
// parameters (each is copied into the argument segment by itself) and where the segment exceeds 112 bytes: us per launch of
// an empty kernel from C, on a machine in its fast / its slow state, 16 scalar parameters of 88 bytes 2.64 / 4.05, ten and a
// struct of 184 bytes 2.64 / 3.8, three vectors and a struct 2.46 / 3.03 at 88 bytes, 2.50 / 3.06 at 112, 2.58 / 3.28 at 120, 2.58 /
// 3.6 from 160 on; the same three vectors and struct launched in this way and not by <<<>>> 2.29 / 2.80 at 88, 2.35 / 2.82 at 112.
template <typename T> struct Undeduced { typedef T type; };
template <typename... P>
int launch_kernel(void (*kernel)(P...), dim3 grid, uint32_t threads, uint32_t lds_bytes, hipStream_t stream, typename Undeduced<P>::type... params) {
    void *at[] = {&params...};
    const hipError_t e = hipLaunchKernel(reinterpret_cast<const void *>(kernel), grid, dim3(threads), at, lds_bytes, stream);
    if (e != hipSuccess) (void)hipGetLastError();  // (reported by the status, and not once more by the caller's next check)
    return hip_status(e);
}
inline uint32_t low_half(const void *p) { return (uint32_t)reinterpret_cast<uintptr_t>(p); }
inline uint32_t high_half(const void *p) { return (uint32_t)(reinterpret_cast<uintptr_t>(p) >> 32); }

void set_norm_quant_tuning(int key, int value);  // add_rmsnorm_quant.hip
void set_rope_tuning(int key, int value);  // rope_rms.hip

}  // namespace gpuk
