// tfgfa_device.h - device helpers shared by the kernels that stage tiles in LDS by direct
// buffer -> LDS loads.
#ifndef TFGFA_DEVICE_H
#define TFGFA_DEVICE_H

#include <hip/hip_runtime.h>

#include <stdint.h>

namespace tfgfa {

typedef __attribute__((address_space(3))) void lds_void;

// Swizzle of tiles of 128-B rows (8 chunks of 16 B): chunk c of row r is stored at chunk
// c ^ swz_k(r), so any 8 (or 16) consecutive rows of one chunk hit distinct banks; rows r and
// r + 32 share it.
__device__ __forceinline__ int swz_k(int row) { return (row ^ ((row >> 3) & 3)) & 7; }

// Buffer descriptor over one head's N rows (row r at byte r * row_bytes; row_bytes = 2 * D for
// a contiguous head), as four SGPRs for the loads issued from inline assembly: base address,
// stride 0, num_records = N * row_bytes, format word 0x20000 (the layout
// __builtin_amdgcn_make_buffer_rsrc builds for the Q loads).  A raw buffer load whose byte
// offset is at or past num_records returns zero: that is the zero-fill of tiles and query
// blocks past the sequence end (row N starts exactly at num_records: rows are at least 2D
// bytes apart and a lane never reads past byte 2D of a row).  The whole offset is kept in the
// VGPR operand so the range check covers all of it.
typedef int i32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ i32x4 head_desc(const void* base, int N, int row_bytes) {
  const uint64_t b = reinterpret_cast<uint64_t>(base);
  i32x4 d;
  d[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)b);
  d[1] = __builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32));
  d[2] = N * row_bytes;
  d[3] = 0x00020000;
  return d;
}

// One 1-KiB HBM -> LDS transfer: lane i's 16 B (global byte offset `voff` in the buffer) land at
// LDS byte address lds_base + 16*i.  Issued from inline assembly so that the compiler does not
// track it: it would otherwise wait for every outstanding transfer before LDS reads it cannot
// prove disjoint (it loses that proof at control-flow joins).  The only waits on these
// transfers are the explicit vmcnt waits of the pipeline.
// The transfer takes its LDS address from M0, a register the compiler reserves (a clobber of it
// is not honoured).  So the statement saves M0 in a scalar register of its own, sets it, issues
// the load and puts the saved value back: whatever the compiler keeps in M0 is unchanged after
// the statement.  The s_nop is the one wait state GFX9 needs between an SALU write of M0 and an
// LDS DMA that reads it.
__device__ __forceinline__ void lds_transfer(i32x4 desc, uint32_t lds_base, int voff) {
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %1\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %2, %3, 0 offen lds\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved)
      : "s"(lds_base), "v"(voff), "s"(desc)
      : "memory");
}

__device__ __forceinline__ uint32_t lds_addr(const unsigned char* p) {
  return (uint32_t)(uintptr_t)(const lds_void*)p;
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

}  // namespace tfgfa

#endif  // TFGFA_DEVICE_H
