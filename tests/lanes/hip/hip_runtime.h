// The HIP names that the react kernel's headers use, for lanes emulated on the host (lanes.h).
#pragma once
#include <math.h>
#include <stdint.h>
#include <string.h>

#define __device__
#define __host__
#define __global__
#define __shared__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __align__(n) __attribute__((aligned(n)))
#define threadIdx emu::thread_idx()
#define blockDim emu::block_dim()
#define gridDim emu::one()
#define blockIdx emu::zero()

struct uint4 {
  uint32_t x, y, z, w;
};

#include "../lanes.h"
