// What the walks over tiles of edges share (internal).
#ifndef APC_SCORE_TILES_H_
#define APC_SCORE_TILES_H_
#include "apc_device.h"

namespace apc_tiles {

constexpr int kTileDoubles = 5120;  // 40 KB: one of the two buffers
constexpr int kRows = 16;           // rows of choices a tile reads
constexpr int kTileSteps = 64;      // of a tile: a lane each

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;

// Global memory to LDS without registers in between: lane i's 16 (4) bytes to lds + i * 16 (4).
// Written by hand, and waited for by hand, so that the loads stay in flight while the lanes draw
// from the other buffer; m0 is put back because the compiler keeps it for its own uses.
__device__ __forceinline__ void load16_lds(const void* g, uint32_t lds) {
  uint32_t saved;
  lds = __builtin_amdgcn_readfirstlane(lds);
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %2, off\n\ts_mov_b32 m0, %0"
               : "=&s"(saved) : "s"(lds), "v"(g) : "memory");
}
// 4 KB: an instruction's offset counts for both addresses
__device__ __forceinline__ void load16x4_lds(const void* g, uint32_t lds) {
  uint32_t saved;
  lds = __builtin_amdgcn_readfirstlane(lds);
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %2, off\n\t"
               "global_load_lds_dwordx4 %2, off offset:1024\n\tglobal_load_lds_dwordx4 %2, off offset:2048\n\t"
               "global_load_lds_dwordx4 %2, off offset:3072\n\ts_mov_b32 m0, %0"
               : "=&s"(saved) : "s"(lds), "v"(g) : "memory");
}
__device__ __forceinline__ void load4_lds(const void* g, uint32_t lds) {
  uint32_t saved;
  lds = __builtin_amdgcn_readfirstlane(lds);
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 3\n\tglobal_load_lds_dword %2, off\n\ts_mov_b32 m0, %0"
               : "=&s"(saved) : "s"(lds), "v"(g) : "memory");
}

// The words of an image name places in LDS counted from 0, so that a read needs no addition: right while a kernel that
// reads them has nothing in front of its dynamic part, neither a __shared__ variable nor an array that the compiler
// moved there.  Asked of the built kernel before every launch.
inline int check_lds_from_0(const void* kernel, const char* name) {
  hipFuncAttributes a;
  hipError_t e = hipFuncGetAttributes(&a, kernel);
  if (e != hipSuccess) return fail(APC_ERR_LAUNCH, "hipFuncGetAttributes: %s", hipGetErrorString(e));
  if (a.sharedSizeBytes != 0) return fail(APC_ERR_UNSUPPORTED, "%s: the dynamic part of its LDS does not begin at 0", name);
  return 0;
}

}  // namespace apc_tiles
#endif  // APC_SCORE_TILES_H_
