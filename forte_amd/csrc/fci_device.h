// fci_device.h -- device helpers that several kernels share.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

// global-memory pointers, said so: a pointer picked from an item table is otherwise taken as flat, and
// a flat load waits with the LDS counter
#define GLOBAL_MEM __attribute__((address_space(1)))

namespace fci {

// Hardware dispatches workgroup b to XCD (b % 8); give each XCD a contiguous range of work.
__device__ __forceinline__ int64_t xcd_remap(int64_t b, int64_t nwork) {
    const int64_t per = (nwork + 7) / 8;
    return (b % 8) * per + b / 8;
}
inline unsigned xcd_grid(int64_t nwork) { return unsigned(((nwork + 7) / 8) * 8); }

__device__ __forceinline__ void split_bf16(float x, __bf16& hi, __bf16& lo) {
    hi = __bf16(x);
    lo = __bf16(x - float(hi));
}

}  // namespace fci
