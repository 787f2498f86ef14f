// The modulus constants of a launch's planes, read by the kernels from a
// constant table in device memory (one per source file, built at compile
// time).
//
// They used to be passed by value, 44 bytes per plane in the kernel
// arguments. Arguments are written by the host for every launch, so each
// launch read them cold, one cache line after another as a kernel went through
// its planes; the table stays in the L2.
#pragma once

#include <hip/hip_runtime.h>

#include "tables.hpp"

namespace rns8x {

static __device__ const ModulusTable kModulusTable = make_modulus_table();

__device__ __forceinline__ const ModulusConsts& plane_mod(PlaneConsts pc, uint32_t plane) {
  return kModulusTable.entry[modulus_table_index(pc, plane)];
}

}  // namespace rns8x
