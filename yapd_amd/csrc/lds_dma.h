// Direct global -> LDS loads (device code).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace yapd {

// 16 bytes per lane from src into LDS at lds_run + 16 * lane (lds_run must be
// the same for the whole wave: it is the M0 base of global_load_lds_dwordx4).
__device__ __forceinline__ void load_lds16(const uint16_t* src, char* lds_run) {
  __builtin_amdgcn_global_load_lds(
      src, reinterpret_cast<__attribute__((address_space(3))) void*>(reinterpret_cast<uintptr_t>(lds_run)), 16, 0, 0);
}

// 16 bytes per lane into LDS at lds_run + 16 * lane (uniform: the M0 base)
// through a buffer descriptor: bytes [ofs + sofs, +16) per lane from its base
// (ofs per lane, sofs uniform).  A buffer load is no FLAT instruction, so the
// compiler's waits for LDS reads stay counted ones; with global_load_lds in
// flight it waits for every LDS read outstanding (lgkmcnt(0)) before each use
// of a fragment.  kStream: a non-temporal load, for bytes read once.
template <bool kStream = false>
__device__ __forceinline__ void load_lds16(__amdgpu_buffer_rsrc_t rsrc, uint32_t ofs, uint32_t sofs, char* lds_run) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(
      rsrc, reinterpret_cast<__attribute__((address_space(3))) void*>(reinterpret_cast<uintptr_t>(lds_run)), 16, ofs,
      sofs, 0, kStream ? 2 : 0);
}

// Descriptor over the 4 GiB from p on (word 3: raw 32-bit elements, no swizzle).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_from(const uint16_t* p) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p), 0, -1, 0x00020000);
}

}  // namespace yapd
