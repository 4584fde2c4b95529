// skl_kcstream.hpp - the product of a decode batch against weights whose columns are contiguous in K, for the kernels of
// skl_gemv_kcrows.hip and skl_gemv_f4.hip (not installed).
//
// A workgroup owns 16 to 64 columns and all of K, so the sums of its columns never leave it: no scratch memory, no second
// launch, the same bits on every run. Its waves take the 128-byte lines of the columns in turn; a line of every column, and
// the same k of up to 96 rows of A, is a unit. A wave's units go from memory to LDS without passing through registers
// (buffer_load ... lds) into a ring that only that wave writes and reads: no barrier before the end, the wave waits for its own
// oldest unit while the others are under way.
//
// What bounds it: the stream over B, and next to it what the loads cost a compute unit. A load of 16-byte pieces of 16
// columns straight into the matrix cores' operand layout touches 16 lines for 1024 bytes; here an instruction fetches
// eight whole lines, and the operand layout is made by the reads from LDS (a lane's 16 bytes of one column or row, pieces of
// a line exchanged by the column's low bits so that no two lanes of a read meet in a bank). Every workgroup reads all of A,
// from its die's L2: the more columns share that the better, as long as the columns fill the chip - their number is the
// smallest of 1 to 4 groups of 16 that needs no second round of workgroups.
// Loads are never guarded: an offset outside the descriptor's range writes zeros to LDS. That is what rows beyond M, k
// beyond K and the requests behind the last unit get, so that every wave counts the same loads.
#pragma once

#include "skl_device.hpp"

namespace skl_kcstream {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));

constexpr unsigned kLine = 128;            // bytes of a column in a unit
constexpr unsigned kRange = 0x7FFFFFF0u;   // of a buffer descriptor; offsets are checked to stay below it on the host
constexpr unsigned kOutside = 0x7FFFFFF0u; // loads zeros
constexpr int kMaxLds = 160 * 1024;

// Groups of 16 columns per workgroup: as few as give every workgroup a compute unit at once.
inline int column_groups(size_t n) {
  const size_t groups = (n + 15) / 16, cg = (groups + 255) / 256;
  return cg < 4 ? (int)cg : 4;
}

// The ring's shape for RG groups of 16 rows, CG groups of 16 columns, and A_LINES lines of A per row and unit: eight waves
// with at least two units each where 160 KiB hold that, else four, else two.
template <int RG, int CG, int A_LINES>
struct Shape {
  static constexpr int kUnitBytes = 16 * (int)kLine * (CG + RG * A_LINES);
  static constexpr int kLoads = 2 * (CG + RG * A_LINES);  // per unit and wave
  static constexpr int kSpace = A_LINES == 1 ? kMaxLds : kMaxLds - 32 * 1024;  // 4-bit weights keep their scales next to the ring
  static constexpr int kWaves = A_LINES == 1 && 16 * kUnitBytes <= kSpace ? 8 : 8 * kUnitBytes <= kSpace ? 4 : 2;
  static constexpr int kFit = kSpace / (kWaves * kUnitBytes);
  static constexpr int kUnits = kFit < 4 ? kFit : 4;
  static constexpr int kRingBytes = kWaves * kUnits * kUnitBytes;
  static constexpr int kPitch = 16 * CG + 1;
  static_assert(kUnits >= 2 && (kUnits - 1) * kLoads < 63);
  static_assert(kWaves * RG * 16 * kPitch * 4 <= kRingBytes, "the sums meet in the ring's place");
};

// Both operands of one instruction for CG column groups and M row groups (or pieces of A), 2048 bytes apart in LDS. The waits
// are the kernel's own, in the block of the reads: the compiler would make every read of LDS wait for all loads under way.
#define SKL_RD(name, addr, off) "ds_read_b128 %[" #name "], %[" #addr "] offset:" #off "\n"
#define SKL_B1 SKL_RD(b0, pb, 0)
#define SKL_B2 SKL_B1 SKL_RD(b1, pb, 2048)
#define SKL_B3 SKL_B2 SKL_RD(b2, pb, 4096)
#define SKL_B4 SKL_B3 SKL_RD(b3, pb, 6144)
#define SKL_A1 SKL_RD(a0, pa, 0)
#define SKL_A2 SKL_A1 SKL_RD(a1, pa, 2048)
#define SKL_A3 SKL_A2 SKL_RD(a2, pa, 4096)
#define SKL_A4 SKL_A3 SKL_RD(a3, pa, 6144)
#define SKL_A5 SKL_A4 SKL_RD(a4, pa, 8192)
#define SKL_A6 SKL_A5 SKL_RD(a5, pa, 10240)
#define SKL_BO1 [b0] "=&v"(b[0])
#define SKL_BO2 SKL_BO1, [b1] "=&v"(b[1])
#define SKL_BO3 SKL_BO2, [b2] "=&v"(b[2])
#define SKL_BO4 SKL_BO3, [b3] "=&v"(b[3])
#define SKL_AO1 [a0] "=&v"(a[0])
#define SKL_AO2 SKL_AO1, [a1] "=&v"(a[1])
#define SKL_AO3 SKL_AO2, [a2] "=&v"(a[2])
#define SKL_AO4 SKL_AO3, [a3] "=&v"(a[3])
#define SKL_AO5 SKL_AO4, [a4] "=&v"(a[4])
#define SKL_AO6 SKL_AO5, [a5] "=&v"(a[5])
#define SKL_READ(N, MM)                                                                                                   \
  if constexpr (CG == N && M == MM)                                                                                       \
    asm volatile(SKL_B##N SKL_A##MM "s_waitcnt lgkmcnt(0)" : SKL_BO##N, SKL_AO##MM : [pb] "v"(pb), [pa] "v"(pa) : "memory");
#define SKL_READ_ROW(MM) SKL_READ(1, MM) SKL_READ(2, MM) SKL_READ(3, MM) SKL_READ(4, MM)
template <int CG, int M>
__device__ __forceinline__ void read_operands(v4i (&b)[CG], v4i (&a)[M], unsigned pb, unsigned pa) {
  static_assert(CG >= 1 && CG <= 4 && M >= 1 && M <= 6);
  SKL_READ_ROW(1) SKL_READ_ROW(2) SKL_READ_ROW(3) SKL_READ_ROW(4) SKL_READ_ROW(5) SKL_READ_ROW(6)
}
#undef SKL_READ_ROW
#undef SKL_READ

// The eight scales of a unit for each of CG column groups (128 bytes apart): 8 bytes per lane.
template <int CG>
__device__ __forceinline__ void read_scales(v2i (&s)[CG], unsigned p) {
  if constexpr (CG == 1)
    asm volatile("ds_read_b64 %0, %1\ns_waitcnt lgkmcnt(0)" : "=&v"(s[0]) : "v"(p) : "memory");
  else if constexpr (CG == 2)
    asm volatile("ds_read_b64 %0, %2\nds_read_b64 %1, %2 offset:128\ns_waitcnt lgkmcnt(0)" : "=&v"(s[0]), "=&v"(s[1]) : "v"(p) : "memory");
  else if constexpr (CG == 3)
    asm volatile("ds_read_b64 %0, %3\nds_read_b64 %1, %3 offset:128\nds_read_b64 %2, %3 offset:256\ns_waitcnt lgkmcnt(0)"
                 : "=&v"(s[0]), "=&v"(s[1]), "=&v"(s[2]) : "v"(p) : "memory");
  else
    asm volatile("ds_read_b64 %0, %4\nds_read_b64 %1, %4 offset:128\nds_read_b64 %2, %4 offset:256\nds_read_b64 %3, %4 offset:384\ns_waitcnt lgkmcnt(0)"
                 : "=&v"(s[0]), "=&v"(s[1]), "=&v"(s[2]), "=&v"(s[3]) : "v"(p) : "memory");
}

// What a wave requests of one operand per unit: LINES * 16 * GROUPS lines, eight per instruction. Lane l fetches piece
// (l % 8) ^ (l / 8) of line l / 8 into slot l % 8: the reader of line r finds piece x in slot x ^ (r % 8).
template <int GROUPS, int LINES>
struct Requests {
  static constexpr int kEach = 2 * GROUPS;  // instructions per line of the unit
  const char *base;                         // the operand's first row or column of this workgroup
  unsigned off[kEach];                      // the lane's offset for instruction i, less the unit's: row * pitch + piece * 16
  unsigned piece;                           // the lane's first byte in a line
  unsigned total;                           // bytes of a row: k beyond it loads zeros

  // Rows from `rows` on: zeros, or (CLAMP) the last row again, for columns that are computed and not written.
  template <bool CLAMP>
  __device__ __forceinline__ void set(const char *first, size_t pitch, size_t rows, unsigned bytes, int lane) {
    base = first;
    total = bytes;
    piece = (unsigned)((lane & 7) ^ (lane >> 3)) * 16u;
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
      const unsigned row = (unsigned)i * 8u + (unsigned)(lane >> 3);
      const bool in = row < rows;
      const unsigned at = in ? row : (unsigned)rows - 1u;
      off[i] = CLAMP || in ? at * (unsigned)pitch + piece : kOutside;
    }
  }

  template <int CACHE>
  __device__ __forceinline__ void issue(__attribute__((address_space(3))) char *to, unsigned unit) const {
#pragma unroll
    for (int l = 0; l < LINES; ++l) {
      const unsigned k0 = (unit * LINES + (unsigned)l) * kLine;
      const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(base + k0), 0, (int)kRange, 0x00027000);
      const bool in = k0 + piece < total;
#pragma unroll
      for (int i = 0; i < kEach; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void *)(to + (l * kEach + i) * 1024), 16,
                                                 (int)(in ? off[i] : kOutside), 0, 0, CACHE);
    }
  }
};

// Every product of a matrix-core instruction rounds at the size of the sum it is added to, so one chain over a wave's share of a
// long K loses what short chains keep. The products of a few units are a block of their own; here it is added to the running
// sums and starts again from zero.
template <typename V, int RG, int CG>
__device__ __forceinline__ void settle(V (&sum)[RG][CG], V (&block)[RG][CG]) {
#pragma unroll
  for (int rg = 0; rg < RG; ++rg)
#pragma unroll
    for (int cg = 0; cg < CG; ++cg) {
#pragma unroll
      for (int r = 0; r < 4; ++r) sum[rg][cg][r] = __fadd_rn(sum[rg][cg][r], block[rg][cg][r]);
      block[rg][cg] = V{0, 0, 0, 0};
    }
}

// Waits until at most N of the wave's loads are under way.
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

}  // namespace skl_kcstream
