// Loads from global memory straight into LDS, the waits that count them, and rows of operands that come in whole lines.
#pragma once
#include "common.h"
#include "mma.h"
#include "vec.h"

#define KC 512                        // elements per chunk of the reduction axis

// 16 bytes per lane from global memory into LDS at lds_addr + 16 * lane, the address in two parts: a base held in scalar registers, the same for every lane, and a
// 32-bit offset per lane.  The compiler's own form of it adds base and offset in vector registers before every
// load (it moves what does not change along K out of the loop and is left with a vector sum); written out, the
// advancing base costs two scalar additions per K tile for all loads together.  lds_addr: the wave's 1 KB
// block, anywhere in LDS (the grouped product's third stage starts at 96 KB).
__device__ __forceinline__ void pipe_load_to_lds16_sv(const unsigned char* sbase, unsigned voff, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(voff), "s"(sbase), "s"(lds_addr) : "memory");     // m0 is the compiler's scratch: it sets it anew before every use of its own
}
// The same for bytes that one workgroup reads once: they pass through the caches without taking the place of what stays.
__device__ __forceinline__ void pipe_load_to_lds16_once(const unsigned char* sbase, unsigned voff, unsigned lds_addr) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt" : : "v"(voff), "s"(sbase), "s"(lds_addr) : "memory");
}
__device__ __forceinline__ unsigned lds_offset_of(const unsigned char* p) {
  return (unsigned)(unsigned long)((__attribute__((address_space(3))) const void*)p);
}

template <int N_>
__device__ __forceinline__ void wait_vmcnt_n() {             // vmcnt(N_), N_ below 64; the other counters at their maxima
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N_ & 0xF) | ((N_ >> 4) << 14));
}

#ifdef VK_BF16
#define LINE_SLOTS 6                    // of a wave's ring, at most
// Rows of one chunk in LDS, a kilobyte each, the 16-byte piece j of row r at piece j ^ turn(r): the fragments of no two rows lie on the same banks, and
// a load brings one row whole.
template <int ROWS>
struct LineRows {
  static constexpr int ROW_BYTES = KC * (int)sizeof(elem_t);
  static_assert(ROW_BYTES == 1024, "a load brings a row of a chunk");
  __device__ static __forceinline__ int turn(int r) { return ROWS == 1 ? 0 : r * (16 / ROWS); }
  // Asks for the rows from `first` on, `stride` elements apart; beyond the first `count` the last one again.
  // pieces: how many of a row's 64 pieces exist (the last one is read again instead of those beyond).
  template <bool ONCE>
  __device__ static __forceinline__ void ask(const elem_t* first, int64_t stride, int count, int lane, unsigned lds_addr, int pieces = 64) {
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      const unsigned char* row = reinterpret_cast<const unsigned char*>(first + (int64_t)min(r, count - 1) * stride);
      const unsigned at = __builtin_amdgcn_readfirstlane(lds_addr + r * ROW_BYTES), piece = (unsigned)(min(lane ^ turn(r), pieces - 1) * 16);
      if (ONCE) pipe_load_to_lds16_once(row, piece, at);
      else pipe_load_to_lds16_sv(row, piece, at);
    }
  }
  __device__ static __forceinline__ frag_t fragment(const unsigned char* rows, int slab, int r16, int kg) {      // rows beyond ROWS repeat them
    const int r = r16 & (ROWS - 1);
    return *reinterpret_cast<const frag_t*>(rows + r * ROW_BYTES + ((slab * 4 + kg) ^ turn(r)) * 16);
  }
};
#endif
