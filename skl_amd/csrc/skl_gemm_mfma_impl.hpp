// skl_gemm_mfma_impl.hpp - the dense contractions on the gfx950 matrix cores (kernel templates and their
// launchers; included by one translation unit per operand kind, skl_gemm_mfma_<kind>.hip, and by the dispatch in
// skl_gemm_mfma.hip):
// int8 x int8 -> int32 (v_mfma_i32_32x32x32_i8), bf16 / f16 -> f32
// (v_mfma_f32_32x32x16_{bf16,f16}) and OCP fp8 E4M3 / E5M2, in any pairing,
// -> f32 (v_mfma_f32_32x32x64_f8f6f4).
//
// Semantics: C = alpha*A*B + beta*C of ref/gemm/gemm_i8rcprc_i8rcprc_i32rcprc.c:10-37
// and its typed twins, for the layouts the optimized SKL entry points use
// (src/gemm/gemm_i8_i8_i32_zve32x.h:38-48 row-major, src/gemm/gemm_i8c_i8_i32_xsfmm32a8i.h:38-48
// column-major A, :85-95 TE x 1 / 1 x TE panels with TE x TE blocks of C). The
// integer result is exact; the fp result accumulates exact products in fp32
// in an order that differs from the reference's k-ascending loop.
//
// One kernel template serves every layout pair. Each operand is either
// "K-contiguous" (row-major A, column-major B) or "MN-contiguous" (column-major
// A, row-major B, and both panel formats); blocks of 64 along M / N may sit
// anywhere (block stride), which is what the panel formats need. A workgroup
// owns a BM x BN tile of C (128 x 128 on eight waves or 64 x 64 on four; the streaming kernel below has larger ones); per
// slice of K (128 or 256 bytes) it copies the A and B tiles global -> registers -> LDS in their native orientation with
// 128-bit accesses (up to two slices under way in registers, two in LDS) and the waves read MFMA operands straight from
// LDS: ds_read_b128 for a K-contiguous tile (row pitch padded to 144 bytes),
// ds_read_b64_tr_b8 / _tr_b16 - the LDS transpose loads - for an
// MN-contiguous one (row pitch padded so the eight/four rows of one transpose
// land in distinct banks). No data is transposed by VALU work. The k order
// inside an MFMA is the same for both operands whichever way they were read, so
// any layout pair multiplies matching k. alpha / beta are applied per wave on
// the accumulator registers in the epilogue.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>

#include <cstdlib>
#include <utility>

#include "skl_device.hpp"
#include "skl_fp8.hpp"

// The arguments of a launch, shared by the translation units of the operand kinds and the dispatch.
struct MfmaArgs {
  const char *a;
  const char *b;
  char *c;
  size_t m, n, k;
  size_t a_s1, a_s0, a_sk;  // elements
  size_t b_s1, b_s0, b_sk;
  size_t rsc0, csc0, rsc1, csc1;
  unsigned crs, ccs;  // log2 of C's block rows / columns (6 unless C comes in smaller power-of-two blocks; crs >= 2)
  skl_scalar alpha, beta;
  const char *bias;  // fused epilogue: per-column addend and running maximum of C's type, or null
  char *max;
  skl_requant rq;    // ... activation and requantised int8 copy
  unsigned tiles_m, tiles_n;
  unsigned by_group = 0, by_rest = 0;  // tile_of_block's divisions as multiplications (set_tiles), 0: too many tiles for that
  // Split along K (bounds-checked kernel only): workgroup (b, split) works on tile b and on the
  // slices [split * slices_per_split, ...); splits > 1 stores the raw
  // sums to partial[split][m][n] (row-major, 4-byte elements) for gemm_split_reduce_kernel.
  unsigned splits, slices_per_split;
  char *partial;
  bool a_loose = false, b_loose = false;  // bounds-checked kernel: the operand is off the 16-byte rule (Loader)
  bool blocked_sums = false;              // 64 x 64 tiles: K is added up in blocks (see the kernel)
};

namespace {

typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

#define LDS_PTR(T, p) ((__attribute__((address_space(3))) T *)(p))

// Bytes of K per LDS stage and operand row in the bounds-checked kernels. The 64 x 64 tiles serve problems too small to fill the
// chip, whose time is a chain - LDS stores, a barrier, fragment reads, products - per slice, most of it latency: 256 bytes to
// a slice halve the chain. (The 128 x 128 tiles keep two workgroups on a compute unit with 128.)
constexpr int slice_bytes(int tile) { return tile == 64 ? 256 : 128; }


// A block of sums, fetched from its accumulation (IN_A) or vector registers here: left to itself the compiler copies all of a wave's
// 256 to vector registers ahead of the first use, and spills.
template <bool IN_A, typename Acc>
__device__ __forceinline__ Acc fetched(Acc acc) {
  if constexpr (IN_A) asm volatile("" : "+a"(acc)); else asm volatile("" : "+v"(acc));
  return acc;
}

// A row-major copy on 4-byte boundaries with no activation beyond ReLU, in the format that goes with C's type (int8 behind an int32
// C, OCP fp8 behind a floating-point one): steps of a few instructions per element.
template <typename T>
__host__ __device__ inline bool dword_copy(const skl_requant &r) {
  return r.q && r.act <= 1 && (r.q_fmt != 0) == !std::is_same<T, int>::value && r.csq == 1 && (r.rsq & 3) == 0 && ((uintptr_t)r.q & 3) == 0;
}

// The steps behind the alpha/beta step that need no more than a lane's column: its bias, and the running maximum.
template <typename T>
struct FusedSteps {
  const T *bias;
  T *max;
  T bias_j, running;
  __device__ explicit FusedSteps(const MfmaArgs &p)
      : bias(reinterpret_cast<const T *>(p.bias)), max(reinterpret_cast<T *>(p.max)), bias_j(0), running(skl_lowest<T>()) {}
  // What the steps need to know about column c, fetched ahead of the stores (a load issued behind a store has to
  // wait for that store's acknowledgement before its value can be used) ...
  __device__ __forceinline__ T fetch(size_t c) const { return bias ? bias[c] : T(0); }
  // ... and made current.
  __device__ __forceinline__ void column(T k) { bias_j = k; }
  // An element of the current column: the steps, then C (written once and not read again: a non-temporal store keeps it out of
  // the operands' caches).
  __device__ __forceinline__ void put(T v, T *dst) {
    if (bias) v = skl_add_bias(v, bias_j);
    if (max && v > running) running = v;
    __builtin_nontemporal_store(v, dst);
  }
  // Every lane of the wave calls this once, after its last element.
  __device__ __forceinline__ void finish() {
    if (!max) return;
    const T best = skl_wave_max(running);
    if ((threadIdx.x & 63) == 0 && best > skl_lowest<T>()) skl_atomic_max(max, best);
  }
};

// Operand kinds of the MFMA: element size, accumulator type, k per instruction.
template <int DT>
struct Kind;
template <>
struct Kind<SKL_DT_I8> {
  static constexpr int ES = 1, KB = 32;  // KB: bytes of K consumed per MFMA per operand row
  using Acc = v16i;
};
template <>
struct Kind<SKL_DT_BF16> {
  static constexpr int ES = 2, KB = 32;
  using Acc = v16f;
};
template <>
struct Kind<SKL_DT_F16> {
  static constexpr int ES = 2, KB = 32;
  using Acc = v16f;
};
template <>
struct Kind<SKL_DT_F8E4M3> {
  static constexpr int ES = 1, KB = 64;
  using Acc = v16f;
};
template <>
struct Kind<SKL_DT_F8E5M2> {
  static constexpr int ES = 1, KB = 64;
  using Acc = v16f;
};

// One MFMA: FR = bytes per lane / 4 registers of each operand fragment.
template <int TA, int TB>
struct Mma;
template <>
struct Mma<SKL_DT_I8, SKL_DT_I8> {
  using Frag = v4i;
  __device__ static v16i run(v4i a, v4i b, v16i c) { return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, c, 0, 0, 0); }
};
template <>
struct Mma<SKL_DT_BF16, SKL_DT_BF16> {
  using Frag = v4i;
  __device__ static v16f run(v4i a, v4i b, v16f c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
  }
};
template <>
struct Mma<SKL_DT_F16, SKL_DT_F16> {
  using Frag = v4i;
  __device__ static v16f run(v4i a, v4i b, v16f c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
  }
};
// f8f6f4 format codes: 0 = E4M3, 1 = E5M2. Scales 0/0 select the unscaled instruction.
#define SKL_F8_MMA(TA_, TB_, FA_, FB_)                                                                   \
  template <>                                                                                            \
  struct Mma<TA_, TB_> {                                                                                 \
    using Frag = v8i;                                                                                    \
    __device__ static v16f run(v8i a, v8i b, v16f c) {                                                   \
      return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, FA_, FB_, 0, 0, 0, 0);             \
    }                                                                                                    \
  };
SKL_F8_MMA(SKL_DT_F8E4M3, SKL_DT_F8E4M3, 0, 0)
SKL_F8_MMA(SKL_DT_F8E5M2, SKL_DT_F8E5M2, 1, 1)
SKL_F8_MMA(SKL_DT_F8E4M3, SKL_DT_F8E5M2, 0, 1)
SKL_F8_MMA(SKL_DT_F8E5M2, SKL_DT_F8E4M3, 1, 0)

// OCP fp8 operands multiplied exactly: the bytes are widened to f16 in registers (every E4M3 / E5M2 value is an
// f16 value) and two f16 instructions take 32 bytes of K - exact products, fp32 sums, which is what the reference's
// error bound assumes. The fp8 instructions above align the products of one instruction to a common exponent and
// keep about 12 bits below the largest; that is inside the bound only once K is a few thousand (the bound grows
// with K, the instruction's error does not), so short K runs here, at the f16 rate.
template <int TA, int TB>
struct MmaF8Exact {
  static constexpr int KB = 32;  // bytes of K per step: a 16-byte fragment per lane, like int8
  using Frag = v4i;
  struct Ready {
    v8h lo, hi;
  };
  template <int DT>
  __device__ static Ready widen(v4i f) {
    constexpr bool e5m2 = DT == SKL_DT_F8E5M2;
    return Ready{skl_fp8::widen8_to_f16<e5m2>((unsigned)f.x, (unsigned)f.y), skl_fp8::widen8_to_f16<e5m2>((unsigned)f.z, (unsigned)f.w)};
  }
  __device__ static Ready prep_a(v4i f) { return widen<TA>(f); }
  __device__ static Ready prep_b(v4i f) { return widen<TB>(f); }
  __device__ static v16f run(const Ready &a, const Ready &b, v16f c) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_f16(a.lo, b.lo, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a.hi, b.hi, c, 0, 0, 0);
  }
};
// K up to which the fp8 kinds run on MmaF8Exact: the reference's bound 2((1 + 2^-24)^(K+2) - 1) passes the fp8
// instructions' 2^-11.9 at K = 2193.
constexpr size_t kF8ExactMaxK = 2304;

// What the streaming kernel multiplies with: blocks of SIDE x SIDE, 64 bytes of K. The instructions take B's columns as their
// first operand, A's rows as their second, so that a lane holds four consecutive columns of a row of C: 16 bytes of a row-major C.
// 16 x 16 blocks run no slower by themselves than 32 x 32 ones (instructions alone on random operands, P/s for 32 x 32 / 16 x 16: bf16
// 1.75 / 1.75, f16 1.62 / 1.66, int8 3.32 / 3.49), their sums are there after half as many passes, and the error against 64 bits is the same.
// Written in assembly for the registers' sake: a wave's operands are vector registers that LDS reads under way will write, its sums
// accumulation registers, and left to itself the compiler moves both about. Of the 256 sums per lane of a 256 x 256 tile a few are
// vector registers (IN_A false): where all accumulation registers are taken the compiler copies a block out and back around a
// product, which it does not know to be under way.
// run() with a load: also 16 bytes per lane from g + off to LDS at `lds` + AT (a load to LDS takes its place there from M0, which is
// to be written an instruction ahead; the compiler takes no clobber of M0, so every other load of such a kernel is load_to_lds).
#define SKL_RING_PRODUCT(IN_, INSN, MODS) asm volatile("v_mfma_" INSN " %0, %1, %2, %0" MODS : "+" IN_(c) : "v"(b), "v"(a))
#define SKL_RING_PRODUCT_LOAD(IN_, INSN, MODS)                                                                       \
  asm volatile("s_add_u32 m0, %3, %6\n\tv_mfma_" INSN " %0, %1, %2, %0" MODS "\n\tglobal_load_lds_dwordx4 %4, %5"   \
               : "+" IN_(c) : "v"(b), "v"(a), "s"(lds), "v"(off), "s"(g), "n"(AT) : "memory", "scc")
#define SKL_RING_MMA(INSN, MODS, FRAG)                                                                                            \
  template <bool IN_A>                                                                                                            \
  __device__ static __forceinline__ void run(FRAG a, FRAG b, Acc &c) {                                                            \
    if constexpr (IN_A) SKL_RING_PRODUCT("a", INSN, MODS); else SKL_RING_PRODUCT("v", INSN, MODS);                                \
  }                                                                                                                               \
  template <bool IN_A, unsigned AT>                                                                                               \
  __device__ static __forceinline__ void run(FRAG a, FRAG b, Acc &c, unsigned lds, const char *g, unsigned off) {                 \
    if constexpr (IN_A) SKL_RING_PRODUCT_LOAD("a", INSN, MODS); else SKL_RING_PRODUCT_LOAD("v", INSN, MODS);                      \
  }
template <int TA, int TB, bool EXACT>
struct RingMma;
#define SKL_RING_F8(TA_, TB_, MODS)                   \
  template <>                                         \
  struct RingMma<TA_, TB_, false> {                   \
    using Frag = v8i;                                 \
    static constexpr int kSide = 32, kFrag = 32;      \
    using Acc = v16f;                                 \
    SKL_RING_MMA("f32_32x32x64_f8f6f4", MODS, v8i)    \
  };
SKL_RING_F8(SKL_DT_F8E4M3, SKL_DT_F8E4M3, "")
SKL_RING_F8(SKL_DT_F8E4M3, SKL_DT_F8E5M2, " cbsz:1")
SKL_RING_F8(SKL_DT_F8E5M2, SKL_DT_F8E4M3, " blgp:1")
SKL_RING_F8(SKL_DT_F8E5M2, SKL_DT_F8E5M2, " cbsz:1 blgp:1")
#undef SKL_RING_F8
template <>
struct RingMma<SKL_DT_I8, SKL_DT_I8, false> {
  using Frag = v4i;
  static constexpr int kSide = 16, kFrag = 16;
  using Acc = v4i;
  SKL_RING_MMA("i32_16x16x64_i8", "", v4i)
};
struct RingMmaI8Large {  // 32 x 32 blocks, a fragment's halves one behind the other; see ring_few_issue_slots
  using Frag = v8i;
  static constexpr int kSide = 32, kFrag = 32;
  using Acc = v16i;
  SKL_RING_MMA("i32_32x32x32_i8", "", v4i)
};
template <>
struct RingMma<SKL_DT_BF16, SKL_DT_BF16, false> {
  using Frag = v4i;
  static constexpr int kSide = 16, kFrag = 16;
  using Acc = v4f;
  SKL_RING_MMA("f32_16x16x32_bf16", "", v4i)
};
template <>
struct RingMma<SKL_DT_F16, SKL_DT_F16, false> {
  using Frag = v4i;
  static constexpr int kSide = 16, kFrag = 16;
  using Acc = v4f;
  SKL_RING_MMA("f32_16x16x32_f16", "", v4i)
};
template <int TA, int TB>
struct RingMma<TA, TB, true> {  // a lane's 16 bytes of K are two products' worth (see FragReader): its first eight, its last eight
  using Frag = v4i;
  static constexpr int kSide = 16, kFrag = 16;
  using Acc = v4f;
  template <int DT>
  __device__ static v8h widen(v4i f, int half) {
    return half ? skl_fp8::widen8_to_f16<DT == SKL_DT_F8E5M2>((unsigned)f.z, (unsigned)f.w) : skl_fp8::widen8_to_f16<DT == SKL_DT_F8E5M2>((unsigned)f.x, (unsigned)f.y);
  }
  __device__ static v8h widen_a(v4i f, int half) { return widen<TA>(f, half); }
  __device__ static v8h widen_b(v4i f, int half) { return widen<TB>(f, half); }
  SKL_RING_MMA("f32_16x16x32_f16", "", v8h)
};
#undef SKL_RING_MMA
#undef SKL_RING_PRODUCT
#undef SKL_RING_PRODUCT_LOAD
// Whether block (i, j) of a wave's MI x NI lies in accumulation registers: all but half a row of blocks where there are 256 sums.
template <int MI, int NI, typename Acc>
constexpr bool ring_sum_in_a(int i, int j) { return MI * NI * sizeof(Acc) < 1024 || i < MI - 1 || j < NI / 2; }

// A fragment as the multiply wants it: widened where the operand kind asks for that, else as it was read.
template <typename M, typename F>
__device__ __forceinline__ auto prep_a(F f) {
  if constexpr (requires { M::prep_a(f); }) return M::prep_a(f); else return f;
}
template <typename M, typename F>
__device__ __forceinline__ auto prep_b(F f) {
  if constexpr (requires { M::prep_b(f); }) return M::prep_b(f); else return f;
}

// ---------------------------------------------------------------------------
// LDS tile geometry of one operand: ROWS along M or N, a slice of K.
// ---------------------------------------------------------------------------
template <int ES, int ROWS, bool KC, int NT>
struct Tile {
  static constexpr int kSlice = slice_bytes(ROWS);
  static constexpr int kRowChunks = kSlice / 16;
  static constexpr int CE = 16 / ES;                 // elements per 16-byte chunk
  static constexpr int KE = kSlice / ES;             // k elements per slice
  static constexpr int kPitchKC = kSlice + 16;       // 16 rows of 16 bytes fill the 64 banks once
  // MN-contiguous tile: KE rows of ROWS*ES bytes. A transpose load is served 32
  // lanes at a time: 8 rows x 32 B (8-bit) or 4 rows x 64 B (16-bit). Skewing
  // consecutive rows by that width spreads them over all 64 banks (measured:
  // zero bank conflicts with 32 / 64 bytes of padding, conflicts with 16 / 32).
  // The tiles of 64 rows do it without padding - four (two) rows fill the banks, the next ones swap their halves -,
  // which lets two workgroups share a compute unit.
  static constexpr bool kSwizzled = ROWS == 64;
  static constexpr int kPitchMC = ROWS * ES + (kSwizzled ? 0 : ES == 1 ? 32 : 64);
  __device__ static __forceinline__ int mc(int r, int byte) {  // byte `byte` of k-row r
    if constexpr (!kSwizzled) return r * kPitchMC + byte;
    return r * kPitchMC + (ES == 1 ? byte ^ ((r >> 2 & 1) << 5) : byte ^ ((r >> 1 & 1) << 6));
  }
  static constexpr int kBytes = KC ? ROWS * kPitchKC : KE * kPitchMC;
  static constexpr int kChunks = ROWS * kRowChunks;  // 16-byte chunks per slice
  static constexpr int kPerThread = kChunks / NT;    // chunks each of the NT threads moves
  static constexpr int kMnChunks = ROWS * ES / 16;   // chunks along MN of an MN-contiguous row
};

// The low bytes of a 16-byte chunk moved down by `bytes` (0 to 15, its own for every lane), zeros above.
__device__ __forceinline__ v4i chunk_shift_down(v4i v, unsigned bytes) {
  const bool two = bytes & 8, one = bytes & 4;
  int w0 = two ? v.z : v.x, w1 = two ? v.w : v.y, w2 = two ? 0 : v.z, w3 = two ? 0 : v.w;
  w0 = one ? w1 : w0, w1 = one ? w2 : w1, w2 = one ? w3 : w2, w3 = one ? 0 : w3;
  return v4i{(int)__builtin_amdgcn_alignbyte((unsigned)w1, (unsigned)w0, bytes), (int)__builtin_amdgcn_alignbyte((unsigned)w2, (unsigned)w1, bytes),
             (int)__builtin_amdgcn_alignbyte((unsigned)w3, (unsigned)w2, bytes), (int)__builtin_amdgcn_alignbyte(0u, (unsigned)w3, bytes)};
}
// A chunk's first `bytes` (0 to 16) bytes, zeros above.
__device__ __forceinline__ v4i chunk_keep(v4i v, int bytes) {
  const auto keep = [&](int w, int b) { return b >= 4 ? w : b <= 0 ? 0 : (int)((unsigned)w & ((1u << (8 * b)) - 1u)); };
  return v4i{keep(v.x, bytes), keep(v.y, bytes - 4), keep(v.z, bytes - 8), keep(v.w, bytes - 12)};
}

// One thread's share of the global loads of an operand, without a branch: a guard is a branch, and at a branch that is not
// uniform every load in flight is waited for (guarded chunk by chunk, a slice of the 64 x 64 kernel cost four memory
// latencies one after another: 2.2 us of it, 128 bytes of K). Chunks go through a buffer descriptor whose base follows K as a
// scalar; a chunk that does not exist (rows or columns beyond the matrix, k beyond its end) gets an offset beyond the
// descriptor's range, for which the load returns zeros and touches no memory.
// `loose`: the operand is off the 16-byte rule, and what is loaded must not reach beyond it. Then a chunk of which only the
// first elements exist is loaded from further down, so that it ends with the last of them, and its bytes are moved into place
// on the way to LDS. (An operand on the rule has no such chunk in a 16-byte unit of its own: whatever follows the last element
// there is cut off along K, and along M / N reaches rows and columns that do not exist.)
template <int ES, int ROWS, bool KC, int NT>
struct Loader {
  using T = Tile<ES, ROWS, KC, NT>;
  static constexpr unsigned kRange = 0xC0000000u, kOutside = 0xE0000000u;  // (offsets inside a tile stay below 0xA8000000, see operand_ok)
  static constexpr unsigned kBias = 16;  // the base lies 16 bytes ahead of the tile, so that no offset is negative
  static constexpr int kRowsPerPass = KC ? NT / T::kRowChunks : NT / T::kMnChunks;
  static_assert(KC || kRowsPerPass % 8 == 0, "the swizzle of a thread's chunks is that of its first");
  const char *base;              // uniform
  size_t k_step;                 // bytes between consecutive slices
  unsigned off[T::kPerThread];   // byte offset of each chunk
  unsigned lds_off;              // of the first chunk; the others follow kRowsPerPass rows apart
  int k_first;                   // KC: k element of the chunks in the slice; MC: k row of the first chunk
  unsigned back;                 // MC: bytes by which the chunks are loaded too low
  bool loose, mn_shift;          // uniform

  // A thread's chunks lie kRowsPerPass rows (or k-rows) apart: their offsets are that of its first one plus scalars. (All in 32
  // bits: instructions ahead of the first load are time that a small problem has nothing to hide under.)
  __device__ __forceinline__ void init(const char *operand, size_t mn0, size_t mn_dim, size_t s1, size_t s0, size_t sk, bool is_loose) {
    const unsigned t = threadIdx.x, extent = mn_dim - mn0 < (size_t)ROWS ? (unsigned)(mn_dim - mn0) : (unsigned)ROWS;
    loose = is_loose;
    base = operand + (mn0 >> 6) * s1 * ES - kBias;  // mn0 is a multiple of 64
    back = 0;
    mn_shift = false;
    if constexpr (KC) {
      static_assert(64 % kRowsPerPass == 0, "a pass lies in one block of 64 rows");
      const unsigned c = t % T::kRowChunks, first_row = t / T::kRowChunks, mine = first_row * (unsigned)(s0 * ES) + c * 16 + kBias;
      k_first = (int)(c * T::CE);
      lds_off = first_row * T::kPitchKC + c * 16;
#pragma unroll
      for (int i = 0; i < T::kPerThread; ++i) {
        constexpr int R = kRowsPerPass;
        off[i] = first_row + i * R < extent ? mine + (unsigned)(((size_t)(i * R >> 6) * s1 + (size_t)(i * R & 63) * s0) * ES) : kOutside;
      }
    } else {
      const unsigned mc = t % T::kMnChunks, r = mc * T::CE, row = t / T::kMnChunks;
      k_first = (int)row;
      lds_off = T::mc((int)row, (int)mc * 16);
      const int there = (int)extent - (int)r;  // elements from the chunk's first on
      if (loose && there > 0 && there < T::CE) back = (unsigned)((T::CE - there) * ES);
      mn_shift = loose && extent < (unsigned)ROWS && extent % T::CE != 0;
      const unsigned mine = (ROWS > 64 ? (r >> 6) * (unsigned)(s1 * ES) : 0u) + (r & 63) * ES + row * (unsigned)(sk * ES) + kBias - back;
#pragma unroll
      for (int i = 0; i < T::kPerThread; ++i) off[i] = there > 0 ? mine + (unsigned)((size_t)(i * kRowsPerPass) * sk * ES) : kOutside;
    }
    k_step = KC ? (size_t)T::kSlice : (size_t)T::KE * sk * ES;
  }

  // `left`: elements of K from the slice's first on, none or fewer beyond the last slice.
  __device__ __forceinline__ void fetch(v4i (&regs)[T::kPerThread], size_t slice, int left) const {
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(base + slice * k_step), 0, (int)kRange, 0x00027000);
    unsigned tail = 0;
    if (KC && loose) {
      const int over = k_first + T::CE - left;  // elements of the chunk beyond K
      tail = over > 0 ? (unsigned)(over * ES) : 0u;
    }
#pragma unroll
    for (int i = 0; i < T::kPerThread; ++i) {
      const bool there = (KC ? k_first : k_first + i * kRowsPerPass) < left;
      const unsigned o = there ? off[i] - tail : kOutside;
      regs[i] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)o, 0, 0));
    }
  }

  // Into LDS, the chunks that end inside 16 bytes put right first (along K: LAST, the share's last slice may be among them).
  template <bool LAST>
  __device__ __forceinline__ void stash(char *tile, v4i (&regs)[T::kPerThread], int left) const {
    if constexpr (KC) {
      if (LAST && left < T::KE && left % T::CE != 0) {  // uniform: the last slice of a K that ends inside a chunk
        const int bytes = (left - k_first) * ES;
#pragma unroll
        for (int i = 0; i < T::kPerThread; ++i)
          regs[i] = loose ? chunk_shift_down(regs[i], bytes > 0 && bytes < 16 ? 16u - (unsigned)bytes : 0u) : chunk_keep(regs[i], bytes);
      }
    } else {
      if (mn_shift) {
#pragma unroll
        for (int i = 0; i < T::kPerThread; ++i) regs[i] = chunk_shift_down(regs[i], back);
      }
    }
#pragma unroll
    for (int i = 0; i < T::kPerThread; ++i) *reinterpret_cast<v4i *>(tile + lds_off + i * kRowsPerPass * (KC ? T::kPitchKC : T::kPitchMC)) = regs[i];
  }
};

// Reads the MFMA operand fragment of 32 rows starting at `row0` for the k-step
// that starts `kb` bytes into the slice. FRB = bytes per lane (16 or 32).
template <int ES, int ROWS, bool KC, int FRB>
__device__ __forceinline__ auto read_frag(const char *tile, int row0, int kb) {
  using T = Tile<ES, ROWS, KC, 64>;
  const int lane = threadIdx.x & 63;
  const int h = lane >> 5;  // which half of the k-step this lane feeds
  if constexpr (KC) {
    const char *p = tile + (row0 + (lane & 31)) * T::kPitchKC + kb + h * FRB;
    if constexpr (FRB == 16) {
      return *reinterpret_cast<const v4i *>(p);
    } else {
      const v4i lo = *reinterpret_cast<const v4i *>(p), hi = *reinterpret_cast<const v4i *>(p + 16);
      return v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    }
  } else if constexpr (ES == 1) {
    // ds_read_b64_tr_b8: 16 lanes read an 8 (k) x 16 (mn) byte block; lane j receives column j.
    const int g16 = (lane >> 4) & 1, j = lane & 15;
    const int kfirst = kb + h * FRB + (j >> 1);
    const char *p = tile + T::mc(kfirst, row0 + g16 * 16 + (j & 1) * 8);
    v2i r[FRB / 8];
#pragma unroll
    for (int s = 0; s < FRB / 8; ++s) r[s] = __builtin_amdgcn_ds_read_tr8_b64_v2i32(LDS_PTR(v2i, p + s * 8 * T::kPitchMC));
    if constexpr (FRB == 16) {
      return v4i{r[0].x, r[0].y, r[1].x, r[1].y};
    } else {
      return v8i{r[0].x, r[0].y, r[1].x, r[1].y, r[2].x, r[2].y, r[3].x, r[3].y};
    }
  } else {
    // ds_read_b64_tr_b16: 16 lanes read a 4 (k) x 16 (mn) block of 16-bit elements.
    static_assert(FRB == 16, "16-bit fragments are 16 bytes");
    const int g16 = (lane >> 4) & 1, j = lane & 15;
    const int kfirst = kb / 2 + h * 8 + (j >> 2);
    const char *p = tile + T::mc(kfirst, (row0 + g16 * 16 + (j & 3) * 4) * 2);
    const v4s r0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(v4s, p));
    const v4s r1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(v4s, p + 4 * T::kPitchMC));
    const v2i a = __builtin_bit_cast(v2i, r0), b = __builtin_bit_cast(v2i, r1);
    return v4i{a.x, a.y, b.x, b.y};
  }
}

// ---------------------------------------------------------------------------
// The epilogue of the bounds-checked kernels: one wave writes its MI x NI blocks of 32 x 32, lane l of a block holding column
// l % 32 and rows 8 * (r / 4) + 4 * (l / 32) + r % 4 in register r, as C = beta*C + alpha*acc followed by the fused
// steps. C is written once and not read again: non-temporal stores keep it out of the operands' caches.
//
// What decides the time is how the wave's loads and stores follow each other. On this target one counter covers
// both, in issue order, so the value of a load cannot be used before every store issued in front of it has been
// acknowledged - and under the write burst of a whole chip ending its tiles together that takes microseconds.
// Hence: (1) when C is not read (beta == 0, and no element is the one case below) the 16 * MI * NI stores of a
// lane go out with no load between them - the columns' bias values and scales are fetched first; (2) when C is
// read, the old values of block b + kAhead are requested before block b is stored, so a wait only ever covers
// loads that were issued in front of the stores still in flight.
// beta == 0 in floating point reads C only where alpha*acc is the negative zero (skl_initialise_needs_c); whether
// any element of the wave's tile is one is decided once, for the whole wave, before the first store.
// CHECK: rows / columns beyond p.m / p.n are left alone.
// ---------------------------------------------------------------------------
template <int MI, int NI, bool CHECK, typename Acc>
__device__ __forceinline__ void write_wave_tile(const MfmaArgs &p, const Acc (&acc)[MI][NI], size_t row0, size_t col0) {
  using AccElem = decltype(Acc{}.x);
  constexpr int kBlocks = MI * NI;            // block b: j = b / MI, i = b % MI (a column strip at a time)
  constexpr int kAhead = (kBlocks < 2 || CHECK) ? 1 : 2;  // the bounds-checked kernels run four waves per SIMD: 128 registers
  // The lane index from the execution mask rather than from threadIdx: nothing the epilogue needs is then computed
  // in front of the main loop and held in a vector register across it (the loop uses every one of them).
  const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  AccElem *c = reinterpret_cast<AccElem *>(p.c);
  const size_t rmask = (size_t(1) << p.crs) - 1, cmask = (size_t(1) << p.ccs) - 1;
  const bool init = skl_beta_is_zero<AccElem>(p.beta);  // C is initialised, not updated
  bool read_c = !init;
  if constexpr (!std::is_same<AccElem, int>::value) {
    if (init) {
      // alpha through a copy the compiler cannot identify with p.alpha: the products of this test are then not
      // kept (all 16 * MI * NI of them, spilled) for the stores below, which multiply again.
      skl_scalar alpha = p.alpha;
      asm volatile("" : "+s"(alpha.i));
      bool need = false;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) need |= skl_initialise_needs_c(acc[i][j][r], alpha, p.beta);
      read_c = __builtin_amdgcn_ballot_w64(need) != 0;
    }
  }
  auto col_of = [&](int j) { return col0 + (size_t)j * 32 + (lane & 31); };
  // first of the four consecutive rows of register group g (all in one block of C: blocks have a multiple of 4 rows)
  auto first_row = [&](int i, int g) { return row0 + (size_t)i * 32 + g * 8 + (lane >> 5) * 4; };
  auto inside = [&](int j, int i, int r) { return !CHECK || (col_of(j) < p.n && first_row(i, r >> 2) + (r & 3) < p.m); };
  // The four row groups of block (i, j): where the first row of each starts.
  struct Where {
    AccElem *out[4];
  };
  auto where = [&](int j, int i) {
    // A zero the compiler cannot see through, new at every use: the addresses of a block are then computed where
    // the block is written and not, all 16 * MI * NI of them, ahead of the first block (which spills half of them).
    unsigned opaque = 0;
    asm volatile("" : "+s"(opaque));
    const size_t col = col_of(j) + opaque, col_off = (col >> p.ccs) * p.csc1 + (col & cmask) * p.csc0;
    Where w;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const size_t row = first_row(i, g);
      w.out[g] = c + (row >> p.crs) * p.rsc1 + (row & rmask) * p.rsc0 + col_off;
    }
    return w;
  };
  FusedSteps<AccElem> fused(p);
  AccElem columns[NI];
#pragma unroll
  for (int j = 0; j < NI; ++j) columns[j] = (!CHECK || col_of(j) < p.n) ? fused.fetch(col_of(j)) : AccElem(0);

  // Block B. MODE 0: C is not read; 1: with the old values `old` (C is updated, or beta == 0 and they decide the sign of
  // zeros); 2: C is not read and there is no fused step (no bias, no maximum, no copy).
  // (Block numbers are compile-time constants throughout, so that the buffers of old values stay in registers.)
  auto write_block = [&](auto mode, auto bc, const AccElem (&old)[16]) {
    constexpr int MODE = decltype(mode)::value, B = decltype(bc)::value;
    constexpr int j = B / MI, i = B % MI;
    fused.column(columns[j]);
    const Where w = where(j, i);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int r = 4 * g + q;
        if (inside(j, i, r)) {
          AccElem v;
          if constexpr (MODE == 0 || MODE == 2) v = skl_initialise_plain(acc[i][j][r], p.alpha, p.beta);
          if constexpr (MODE == 1) {  // one path for both ways of using the old value: a select per element
            const AccElem vi = skl_initialise_with(acc[i][j][r], old[r], p.alpha, p.beta), vc = skl_combine(acc[i][j][r], old[r], p.alpha, p.beta);
            v = init ? vi : vc;
          }
          if constexpr (MODE == 2)  // no fused step at all: the value as it is
            __builtin_nontemporal_store(v, w.out[g] + q * p.rsc0);
          else
            fused.put(v, w.out[g] + q * p.rsc0);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // a block at a time: the addresses of later blocks are not computed (and held) early
  };
  // The blocks in order, block B + kAhead requested before block B is written.
  auto update_blocks = [&](auto mode) {
    AccElem old[kAhead + 1][16];
    auto request = [&](auto bc) {
      constexpr int B = decltype(bc)::value;
      if constexpr (B < kBlocks) {
        constexpr int j = B / MI, i = B % MI;
        const Where w = where(j, i);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          // beyond the edge the first element of C is read in place of one that does not exist: a guard would be a branch, at
          // which the loads in flight are waited for (int8 3584 x 1266 x 768 reading C: 33.4 -> 21.2 us)
          const AccElem *from = w.out[r >> 2] + (r & 3) * p.rsc0;
          if (CHECK) from = inside(j, i, r) ? from : c;
          old[B % (kAhead + 1)][r] = *from;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    [&]<int... Bs>(std::integer_sequence<int, Bs...>) { (request(std::integral_constant<int, Bs>{}), ...); }(std::make_integer_sequence<int, kAhead>{});
    [&]<int... Bs>(std::integer_sequence<int, Bs...>) {
      ((request(std::integral_constant<int, Bs + kAhead>{}), write_block(mode, std::integral_constant<int, Bs>{}, old[Bs % (kAhead + 1)])), ...);
    }(std::make_integer_sequence<int, kBlocks>{});
  };
  if (!read_c) {
    const AccElem none[16] = {};
    if (!p.bias && !p.max) {  // the plain product: two or three instructions and a store per element
      [&]<int... Bs>(std::integer_sequence<int, Bs...>) {
        (write_block(std::integral_constant<int, 2>{}, std::integral_constant<int, Bs>{}, none), ...);
      }(std::make_integer_sequence<int, kBlocks>{});
    } else {
      [&]<int... Bs>(std::integer_sequence<int, Bs...>) {
        (write_block(std::integral_constant<int, 0>{}, std::integral_constant<int, Bs>{}, none), ...);
      }(std::make_integer_sequence<int, kBlocks>{});
    }
  } else {
    update_blocks(std::integral_constant<int, 1>{});
  }
  fused.finish();
}

// ---------------------------------------------------------------------------
// The bounds-checked kernels' epilogue for fused calls with any activation and any 8-bit copy. Such steps - a GELU is some
// forty instructions - cannot be written out for each of a lane's 128 accumulators (spilled registers, code beyond the
// instruction cache), and accumulators cannot be indexed by a loop counter. So a wave puts 32 rows of its tile at a time
// into LDS, the operands' stages being over, and loops over them: a lane takes four neighbouring columns of a row, the
// same columns every time, so their biases, scales and offsets are fetched once, and C and the copy go out 16 and 4
// bytes per lane where the layout has them side by side. Every element goes through the same operations in the same
// order as in the other epilogues. `stage`: this wave's 32 x (32 NI + 8) elements; eight elements of padding put the
// two halves of a wave's writes, four rows apart, into different banks.
// alpha, beta and the old C are applied as a strip of 32 rows goes into LDS, and the old values of the next strip are
// requested ahead of this one's stores: a load inside the loop waits for the stores of the pass before, every pass
// (see write_wave_tile; C read, us, loads in the loop / ahead: E5M2 1024 x 14080 x 6272 with ReLU into int8 102 / 91, E4M3
// 7424 x 8576 x 2048 with GELU into int8 433 / 389, bf16 2816^2 x 3584 with SiLU 85 / 81).
// ---------------------------------------------------------------------------
template <int NI>
constexpr int staged_pitch() { return 32 * NI + 8; }
template <int MI, int NI, bool CHECK, typename Acc>
__device__ __forceinline__ void write_wave_tile_staged(const MfmaArgs &p, const Acc (&acc)[MI][NI], size_t row0, size_t col0, char *stage_bytes) {
  using T = decltype(Acc{}.x);
  typedef T V4 __attribute__((ext_vector_type(4)));
  constexpr int P = staged_pitch<NI>(), kLanesPerRow = 8 * NI, kRowsPerPass = 64 / kLanesPerRow;
  const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
  T *const stage = reinterpret_cast<T *>(stage_bytes);
  T *const stage_in = stage + (lane >> 5) * 4 * P + (lane & 31);
  const int r_first = lane / kLanesPerRow, c_first = lane % kLanesPerRow * 4;
  const T *const stage_out = stage + r_first * P + c_first;
  const size_t col = col0 + c_first;
  const int cols = !CHECK ? 4 : col >= p.n ? 0 : p.n - col < 4 ? (int)(p.n - col) : 4;
  const size_t rmask = (size_t(1) << p.crs) - 1, cmask = (size_t(1) << p.ccs) - 1;
  const T *const bias = reinterpret_cast<const T *>(p.bias);
  size_t c_off[4];
  T bias_of[4];
  float scale_of[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const size_t j = e < cols ? col + e : 0;
    c_off[e] = (j >> p.ccs) * p.csc1 + (j & cmask) * p.csc0;
    bias_of[e] = bias && e < cols ? bias[j] : T(0);
    scale_of[e] = p.rq.q && e < cols ? p.rq.q_scale[p.rq.q_per_column ? j : 0] : 0.0f;
  }
  // C's four columns side by side on a 16-byte boundary (columns come in blocks of 2^ccs, col is a multiple of four), and
  // the copy's four bytes on a dword
  const bool c_run = cols == 4 && p.csc0 == 1 && p.ccs >= 2 && (((uintptr_t)p.c | (p.csc1 * 4) | (p.rsc0 * 4) | (p.rsc1 * 4)) & 15) == 0;
  const bool q_run = cols == 4 && p.rq.csq == 1 && (p.rq.rsq & 3) == 0 && ((uintptr_t)p.rq.q & 3) == 0;
  // A pass covers four (eight) rows from a multiple of four (eight) on, whole blocks of C or part of one: where they start is
  // the same for the whole wave (scalar arithmetic), the lane's row among them a constant.
  static_assert(kRowsPerPass == 4 || kRowsPerPass == 8, "blocks of C have a power of two of rows, at least four");
  T *const c_lane = reinterpret_cast<T *>(p.c) + ((size_t)r_first >> p.crs) * p.rsc1 + ((size_t)r_first & rmask) * p.rsc0;
  int8_t *const q_lane = reinterpret_cast<int8_t *>(p.rq.q) + (size_t)r_first * p.rq.rsq + col * p.rq.csq;
  const skl_fp8::Ofp8Format f8(p.rq.q_fmt);
  T running = skl_lowest<T>();
  const bool init = skl_beta_is_zero<T>(p.beta);
  typedef T Rows4 __attribute__((ext_vector_type(4), aligned(4)));  // C by columns: a lane's four rows, on any element boundary
  T old[NI][16];
  // The old values of strip i, if it needs any.
  auto request = [&](int i) {
    bool need = !init;
    skl_scalar alpha = p.alpha;  // a copy the compiler cannot identify with it: the products below are not kept
    unsigned opaque = 0;         // and addresses are worked out here, not all of them ahead of the first strip
    asm volatile("" : "+s"(alpha.i), "+s"(opaque));
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) need |= init && skl_initialise_needs_c(acc[i][j][r], alpha, p.beta);
    const bool any = __builtin_amdgcn_ballot_w64(need) != 0;
    if (!any) return any;
    const auto fetch = [&](auto by_rows) {
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        const size_t jc = col0 + (size_t)j * 32 + (lane & 31) + opaque;
        const T *const c = reinterpret_cast<const T *>(p.c) + ((jc >> p.ccs) * p.csc1 + (jc & cmask) * p.csc0);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const size_t row = row0 + (size_t)i * 32 + g * 8 + (lane >> 5) * 4;  // four rows, in one block of C
          const T *const from = c + ((row >> p.crs) * p.rsc1 + (row & rmask) * p.rsc0);
          if constexpr (decltype(by_rows)::value) {
            const Rows4 four = *reinterpret_cast<const Rows4 *>(from);
#pragma unroll
            for (int q = 0; q < 4; ++q) old[j][4 * g + q] = four[q];
          } else {
#pragma unroll
            for (int q = 0; q < 4; ++q) {  // (no guard, see write_wave_tile)
              const T *at = from + q * p.rsc0;
              if (CHECK) at = jc < p.n && row + q < p.m ? at : reinterpret_cast<const T *>(p.c);
              old[j][4 * g + q] = *at;
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    if (!CHECK && p.rsc0 == 1)
      fetch(std::true_type{});
    else
      fetch(std::false_type{});
    return any;
  };
  const auto put_strip = [&](int i, auto value) {
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) stage_in[((r >> 2) * 8 + (r & 3)) * P + j * 32] = value(acc[i][j][r], j, r);
  };
  bool read_c = request(0);
#pragma unroll
  for (int i = 0; i < MI; ++i) {
    if (!read_c)
      put_strip(i, [&](T sum, int, int) { return skl_initialise_plain(sum, p.alpha, p.beta); });
    else if (init)
      put_strip(i, [&](T sum, int j, int r) { return skl_initialise_with(sum, old[j][r], p.alpha, p.beta); });
    else
      put_strip(i, [&](T sum, int j, int r) { return skl_combine(sum, old[j][r], p.alpha, p.beta); });
    if (i + 1 < MI) read_c = request(i + 1);
    // the wave's own LDS accesses complete in order; the compiler must not move them across each other
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll 2
    for (int pass = 0; pass < 32 / kRowsPerPass; ++pass) {
      const V4 sum = *reinterpret_cast<const V4 *>(stage_out + pass * kRowsPerPass * P);
      const size_t four = row0 + (size_t)(i * 32 + pass * kRowsPerPass);  // the first of them: a scalar
      if (CHECK && (four + r_first >= p.m || cols == 0)) continue;
      T *const c_row = c_lane + ((four >> p.crs) * p.rsc1 + (four & rmask) * p.rsc0);
      V4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        T x = sum[e];
        if (bias) x = skl_add_bias(x, bias_of[e]);
        v[e] = skl_activate(x, p.rq.act);
        if (p.max && e < cols && v[e] > running) running = v[e];
      }
      if (!p.rq.q_only) {
        if (c_run) {
          __builtin_nontemporal_store(v, reinterpret_cast<V4 *>(c_row + c_off[0]));
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (e < cols) c_row[c_off[e]] = v[e];
        }
      }
      if (p.rq.q) {
        unsigned packed = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const unsigned byte = p.rq.q_fmt == 0 ? (unsigned)skl_requantise_int((float)v[e], scale_of[e], p.rq.q_zero) & 0xFFu
                                                : skl_fp8::encode_ofp8_hw(__fmul_rn((float)v[e], scale_of[e]), f8) & 0xFFu;
          packed |= byte << (8 * e);
        }
        int8_t *const q = q_lane + four * p.rq.rsq;
        if (q_run) {
          *reinterpret_cast<unsigned *>(q) = packed;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (e < cols) q[e * p.rq.csq] = (int8_t)(packed >> (8 * e));
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  if (p.max) {
    const T best = skl_wave_max(running);
    if (lane == 0 && best > skl_lowest<T>()) skl_atomic_max(reinterpret_cast<T *>(p.max), best);
  }
}

// ---------------------------------------------------------------------------
// 16 bytes per lane of sums to LDS from the accumulation (IN_A) or vector registers that hold them: the compiler copies them first.
template <bool IN_A, int AT, typename V4>
__device__ __forceinline__ void lds_write_b128(unsigned to, V4 four) {
  if constexpr (IN_A) asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(to), "a"(four), "n"(AT) : "memory");
  else asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(to), "v"(four), "n"(AT) : "memory");
}

// The streaming kernel's epilogue: one wave writes its MI x NI blocks, of which a lane holds four consecutive columns of a row at a
// time (acc[i][j][4 g + e]: row S i + lane % S, column S j + 8 g + 4 (lane / S) + e). The operands' ring being over, the rows of one row
// of blocks at a time go to LDS as they are, and a loop takes them from there in the order that C wants: a wave's rows of 128 (64)
// columns in whole lines, 16 bytes per lane. A loop, because what is behind it - a GELU is some forty instructions - cannot be written
// out for each of a lane's 256 sums: eight copies of the loop, one behind every row of blocks, are 250 KB of code and were three times
// as slow (E4M3 2048 x 8192 x 2048 with GELU into E4M3, all of it 137 us). And whole lines, because the sums as they lie make pieces of 64
// bytes (32 x 32 blocks: 32 bytes), which took 17.5 us for the 64 MiB of 4096^2 (with 32 x 32 blocks 35).
// C by columns is written from LDS by columns, 16 bytes of a column per lane.
// The old values of C are requested a batch ahead: one counter covers loads and stores, in issue order, so that a value used
// right behind its load has waited for every store in front of it. beta == 0 in floating point reads C only where alpha * acc is the
// negative zero (skl_initialise_needs_c), decided for a batch at a time.
// CHECK: rows and columns beyond p.m / p.n are left alone; a lane at the edge reads its old values from the last four columns.
// `stage`: this wave's S x (COLS + 4) elements.
// ---------------------------------------------------------------------------
template <int COLS>
constexpr int wave_rows_pitch() { return COLS + 4; }
template <int MI, int NI, int ES, int MOST, bool CHECK, bool STEPS, typename Acc>
__device__ __forceinline__ void write_wave_rows(const MfmaArgs &p, const Acc (&acc)[MI][NI], size_t row0, size_t col0, char *stage_bytes) {
  using T = decltype(Acc{}.x);
  typedef T V4 __attribute__((ext_vector_type(4)));
  typedef T Run4 __attribute__((ext_vector_type(4), aligned(4)));
  constexpr int S = sizeof(Acc) == 64 ? 32 : 16, G = S == 32 ? 4 : 1, COLS = NI * S, P = wave_rows_pitch<COLS>();
  // A pass: 256 elements, as many whole rows as that is; by columns: S rows by 256 / S columns. A chunk: up to MOST passes. Under way are the
  // old values of one chunk of eight passes, or of two of four where eight waves write (4096 x 8192 x 512, us, one / two: bf16 81 / 74,
  // int8 73 / 62; four waves with two or four of eight: int8 4096 x 8192 x 2048 3 and 13 us more than with one).
  constexpr int kPasses = S * COLS / 256, kMost = MOST, kChunk = kPasses < kMost ? kPasses : kMost, kDown = 256 / COLS, kColsDown = 256 / S;
  constexpr int kChunks = MI * kPasses / kChunk;
  static_assert(kPasses % kChunk == 0);
  const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));  // (not from threadIdx, see write_wave_tile)
  T *const stage = reinterpret_cast<T *>(stage_bytes);
  T *const c = reinterpret_cast<T *>(p.c);
  const size_t rmask = (size_t(1) << p.crs) - 1, cmask = (size_t(1) << p.ccs) - 1;
  const auto row_at = [&](size_t row) { return (row >> p.crs) * p.rsc1 + (row & rmask) * p.rsc0; };
  const auto col_at = [&](size_t col) { return (col >> p.ccs) * p.csc1 + (col & cmask) * p.csc0; };
  const T *const bias = reinterpret_cast<const T *>(p.bias);
  const skl_fp8::Ofp8Format f8(p.rq.q_fmt);
  // Which way the stores go. Through the caches they are the faster ones (us, through / past: 4096 x 8192 x 512 bf16 48.4 / 59.1, int8 of
  // 8192^2 x 2048 134 / 147, E4M3 212 / 227, one round of 64 MiB, 2048 x 8192 x 512, 27.0 / 30.6), as long as the 256 MiB behind them
  // hold all that is written (8192 x 8448 x 2048 bf16 253 / 235, int8 149 / 142; 8192 x 12288 x 512 148 / 130) and A and B, which are
  // read again and again, are no more than half of that (E4M3 of 8192^2 by 4096, 6144 and 8192: 223 / 228, 310 / 312, 396 / 392; 4096 x 14336
  // by 8192, 144 MiB: 359 / 347, int8 361 / 345). Little is better past them: it would still lie in the L2s, which are written back when the kernel
  // ends (4352 x 1024 x 512 int8 9.6 / 8.5, bf16 12.8 / 11.3; 2048 x 4096 x 512 16.5 / 15.1). A C that is read meets its stores there
  // when there are several rounds (8192^2 x 512 bf16 178 / 154), not in one (2048 x 8192 x 512 39 / 42).
  const bool one_round = p.tiles_m * p.tiles_n <= 256;
  const size_t written = p.m * p.n * ((p.rq.q_only ? 0 : 4) + (p.rq.q ? 1 : 0));
  const bool fits = written > (size_t(48) << 20) && written <= (size_t(256) << 20) && (p.m + p.n) * p.k * ES <= (size_t(128) << 20);

  // Row of blocks i's sums to LDS (accumulators cannot be indexed: a branch for each).
  const auto put = [&](unsigned i) __attribute__((always_inline)) {
    [[maybe_unused]] const unsigned to = (unsigned)(size_t)LDS_PTR(char, stage_bytes) + (lane % S * P + lane / S * 4) * (unsigned)sizeof(T);
    [&]<int... Is>(std::integer_sequence<int, Is...>) __attribute__((always_inline)) {
      (
          [&](auto ic) __attribute__((always_inline)) {
            constexpr int I = decltype(ic)::value;
            if (i == I) {
              if constexpr (G == 1) {
                [&]<int... Js>(std::integer_sequence<int, Js...>) __attribute__((always_inline)) {
                  (lds_write_b128<ring_sum_in_a<MI, NI, Acc>(I, Js), Js * S * (int)sizeof(T)>(to, acc[I][Js]), ...);
                }(std::make_integer_sequence<int, NI>{});
              } else {
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                  const Acc sums = j < NI / 2 ? fetched<ring_sum_in_a<MI, NI, Acc>(I, 0)>(acc[I][j]) : fetched<ring_sum_in_a<MI, NI, Acc>(I, NI - 1)>(acc[I][j]);
#pragma unroll
                  for (int g = 0; g < G; ++g)
                    *reinterpret_cast<V4 *>(stage + lane % S * P + lane / S * 4 + j * S + g * 8) = V4{sums[4 * g], sums[4 * g + 1], sums[4 * g + 2], sums[4 * g + 3]};
                }
              }
            }
          }(std::integral_constant<int, Is>{}),
          ...);
    }(std::make_integer_sequence<int, MI>{});
  };

  // RUN: four columns lie side by side in C. Otherwise, `down`, a lane's four elements are four rows of a column: side by side in a C by
  // columns, and in any other C as good as four columns. UPDATE: C is read (not only where a zero's sign asks for it). FUSED: there are
  // steps behind the alpha/beta step.
  const auto write = [&](auto run, auto update, auto fused, auto ones, auto through) __attribute__((always_inline)) {
    constexpr bool RUN = decltype(run)::value, UPDATE = decltype(update)::value, FUSED = decltype(fused)::value, ONES = decltype(ones)::value;
    // the lane's first row and column in a pass, from those of the pass
    const int r_lane = RUN ? lane / (COLS / 4) : lane % (S / 4) * 4, c_lane = RUN ? lane % (COLS / 4) * 4 : lane / (S / 4);
    // Where in C the lane's elements of pass y of a row of blocks are: that of the row of blocks, a scalar, and this (passes begin at
    // multiples of their rows and columns, rows of blocks at multiples of theirs, and blocks of C are powers of two)
    T *const c_lane_at = c + row_at(r_lane) + col_at(col0) + col_at(c_lane);
    size_t step[kChunk];  // from a chunk's first pass to its others
#pragma unroll
    for (int t = 0; t < kChunk; ++t) step[t] = RUN ? row_at(t * kDown) : col_at(t * kColsDown);
    const auto cols_in = [&](size_t col) -> int {  // of four columns from `col` on
      if constexpr (!CHECK) return 4;
      return col >= p.n ? 0 : p.n - col < 4 ? (int)(p.n - col) : 4;
    };
    const auto column_at = [&](size_t k) { return !CHECK || k < p.n ? k : 0; };
    T bias_of[4];
    float scale_of[4];
    if constexpr (RUN && FUSED) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const size_t k = column_at(col0 + c_lane + e);
        bias_of[e] = bias ? bias[k] : T(0);
        scale_of[e] = STEPS && p.rq.q ? p.rq.q_scale[p.rq.q_per_column ? k : 0] : 0.0f;
      }
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): in the loop they would be waited for with every chunk, and its stores with them
    }
    int8_t *const q_lane_at = p.rq.q + (row0 + r_lane) * p.rq.rsq + (col0 + c_lane) * p.rq.csq;  // as c_lane_at: the rest are scalars
    const bool q_run = STEPS && RUN && p.rq.csq == 1 && (p.rq.rsq & 3) == 0 && ((uintptr_t)p.rq.q & 3) == 0;
    T running = skl_lowest<T>();

    // Chunk x: its first row and column, and, from those on, the lane's first row and column of its pass t.
    constexpr unsigned kOfRow = kPasses / kChunk;  // chunks of a row of blocks
    constexpr int kAhead = UPDATE && !STEPS && !CHECK && MOST == 4 ? 2 : 1;  // chunks whose old values are under way
    static_assert(kChunks % kAhead == 0);
    const auto top_of = [&](unsigned x) { return row0 + (RUN ? x * (kChunk * kDown) : x / kOfRow * S); };
    const auto left_of = [&](unsigned x) { return RUN ? size_t(0) : (size_t)(x % kOfRow * (kChunk * kColsDown)); };
    const auto row_of = [&](size_t top, int t) { return top + (RUN ? t * kDown : 0) + r_lane; };
    const auto col_of = [&](size_t left, int t) { return col0 + left + (RUN ? 0 : t * kColsDown) + c_lane; };
    const auto request = [&](unsigned x, V4 (&old)[kChunk]) __attribute__((always_inline)) {
      const size_t top = top_of(x), left = left_of(x);
      const T *const at = c_lane_at + row_at(top) + col_at(left);
#pragma unroll
      for (int t = 0; t < kChunk; ++t) {
        const size_t row = row_of(top, t), k = col_of(left, t);
        if constexpr (RUN && !CHECK) {
          old[t] = *reinterpret_cast<const Run4 *>(at + step[t]);
        } else if constexpr (RUN) {  // (rows and columns that do not exist: some that do)
          old[t] = *reinterpret_cast<const Run4 *>(c + row_at(row < p.m ? row : p.m - 1) + col_at(k + 4 > p.n ? p.n - 4 : k));
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) old[t][e] = c[!CHECK || (row + e < p.m && k < p.n) ? row_at(row) + e * p.rsc0 + col_at(k) : 0];
        }
      }
    };
    const auto moved = [&](size_t k, V4 o) __attribute__((always_inline)) {  // the last four columns, moved down to the lane's own
      if constexpr (CHECK && RUN) {
        const int by = cols_in(k) > 0 ? 4 - cols_in(k) : 0;
        if (by & 1) o = V4{o.y, o.z, o.w, o.w};
        if (by & 2) o = V4{o.z, o.w, o.w, o.w};
      }
      return o;
    };

    // `next`: the old values of chunk x, then those of the next but kAhead - 1.
    const auto chunk = [&](unsigned x, V4 (&next)[kChunk]) __attribute__((always_inline)) {
      const size_t top = top_of(x), left = left_of(x);
      const unsigned in_row = x % kOfRow;
      const T *const stage_x = stage + (RUN ? (in_row * (kChunk * kDown) + r_lane) * P + c_lane : r_lane * P + in_row * (kChunk * kColsDown) + c_lane);
      V4 v[kChunk];
#pragma unroll
      for (int t = 0; t < kChunk; ++t) {
        if constexpr (RUN) {
          v[t] = *reinterpret_cast<const V4 *>(stage_x + t * kDown * P);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[t][e] = stage_x[e * P + t * kColsDown];
        }
      }
      // The wave's own LDS accesses complete in order; the compiler must not move them across each other. The next row of blocks goes to
      // LDS under what follows.
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (in_row == kOfRow - 1) put(x / kOfRow + 1);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if constexpr (UPDATE) {
#pragma unroll
        for (int t = 0; t < kChunk; ++t) {
          const V4 old = moved(col_of(left, t), next[t]);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if constexpr (ONES) v[t][e] = skl_add_bias(v[t][e], old[e]);
            else v[t][e] = skl_combine(v[t][e], old[e], p.alpha, p.beta);
          }
        }
        __builtin_amdgcn_sched_barrier(0);  // the values to come take these registers
        request(x + kAhead < (unsigned)kChunks ? x + kAhead : x, next);  // (beyond the end: some, not used)
      } else if constexpr (!ONES) {
        bool need = false;
#pragma unroll
        for (int t = 0; t < kChunk; ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e) need |= skl_initialise_needs_c(v[t][e], p.alpha, p.beta);
        if (!std::is_same<T, int>::value && __builtin_amdgcn_ballot_w64(need) != 0) {  // the old values decide the sign of some zeros
          V4 signs[kChunk];
          request(x, signs);
#pragma unroll
          for (int t = 0; t < kChunk; ++t) {
            const V4 o = moved(col_of(left, t), signs[t]);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[t][e] = skl_initialise_with(v[t][e], o[e], p.alpha, p.beta);
          }
        } else {
#pragma unroll
          for (int t = 0; t < kChunk; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[t][e] = skl_initialise_plain(v[t][e], p.alpha, p.beta);
        }
      }
      if constexpr (FUSED) {
        if (bias) {
#pragma unroll
          for (int t = 0; t < kChunk; ++t) {
            const T by_column = RUN ? T(0) : bias[column_at(col_of(left, t))];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[t][e] = skl_add_bias(v[t][e], RUN ? bias_of[e] : by_column);
          }
        }
        if constexpr (STEPS) {  // (the choice outside of the elements: chains of instructions then run side by side)
          const auto activate = [&](auto act) __attribute__((always_inline)) {
#pragma unroll
            for (int t = 0; t < kChunk; ++t)
#pragma unroll
              for (int e = 0; e < 4; ++e) v[t][e] = skl_activate(v[t][e], decltype(act)::value);
          };
          if (p.rq.act == 1) activate(std::integral_constant<int, 1>{});
          if constexpr (!std::is_same<T, int>::value) {
            if (p.rq.act == 2) activate(std::integral_constant<int, 2>{});
            if (p.rq.act >= 3) activate(std::integral_constant<int, 3>{});
          }
        }
        if (p.max) {
#pragma unroll
          for (int t = 0; t < kChunk; ++t) {
            const size_t row = row_of(top, t), k = col_of(left, t);
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if ((!CHECK || (row + (RUN ? 0 : e) < p.m && k + (RUN ? e : 0) < p.n)) && v[t][e] > running) running = v[t][e];
          }
        }
      }
      T *const at = c_lane_at + row_at(top) + col_at(left);
      if (!STEPS || !p.rq.q_only) {
        // (the two ways with an empty instruction of each one's own around them: the compiler takes the stores for the same and makes
        // one of them otherwise)
        const auto store = [&](auto kept_c) __attribute__((always_inline)) {
          constexpr bool KEPT = decltype(kept_c)::value;
          if constexpr (RUN) asm volatile("; %0" ::"n"(KEPT));
#pragma unroll
          for (int t = 0; t < kChunk; ++t) {
            const size_t row = row_of(top, t), k = col_of(left, t);
            T *const to = at + step[t];
            if constexpr (RUN) {
              if (!CHECK || (row < p.m && cols_in(k) == 4)) {
                if constexpr (KEPT) *reinterpret_cast<Run4 *>(to) = v[t];
                else __builtin_nontemporal_store((Run4)v[t], reinterpret_cast<Run4 *>(to));
              } else if (row < p.m) {
#pragma unroll
                for (int e = 0; e < 3; ++e)
                  if (k + e < p.n) c[row_at(row) + col_at(k + e)] = v[t][e];
              }
            } else {
              if (p.rsc0 == 1 && (!CHECK || (row + 4 <= p.m && k < p.n))) {
                *reinterpret_cast<Run4 *>(to) = v[t];
              } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                  if (!CHECK || (row + e < p.m && k < p.n)) to[e * p.rsc0] = v[t][e];
              }
            }
          }
          if constexpr (RUN) asm volatile("; %0" ::"n"(KEPT));
        };
        if constexpr (!RUN) store(std::true_type{});
        else if constexpr (UPDATE) store(through);  // (no branch: what waits for old values would wait for the stores that might have been left out)
        else if (fits) store(std::true_type{});
        else store(std::false_type{});
      }
      if constexpr (STEPS) {
        if (p.rq.q) {
          // The copy's four bytes of each pass. OCP fp8: where no value of the chunk leaves the format's finite range the instruction's
          // codes are the rule's, two values at a time.
          float w[kChunk][4];
          unsigned packed[kChunk];
#pragma unroll
          for (int t = 0; t < kChunk; ++t) {
            const float by_column = RUN ? 0.0f : p.rq.q_scale[p.rq.q_per_column ? column_at(col_of(left, t)) : 0];
#pragma unroll
            for (int e = 0; e < 4; ++e) w[t][e] = (float)v[t][e], w[t][e] = p.rq.q_fmt == 0 ? w[t][e] : __fmul_rn(w[t][e], RUN ? scale_of[e] : by_column);
          }
          if (p.rq.q_fmt == 0) {
#pragma unroll
            for (int t = 0; t < kChunk; ++t) {
              const float by_column = RUN ? 0.0f : p.rq.q_scale[p.rq.q_per_column ? column_at(col_of(left, t)) : 0];
              packed[t] = 0;
#pragma unroll
              for (int e = 0; e < 4; ++e)
                packed[t] |= ((unsigned)skl_requantise_int(w[t][e], RUN ? scale_of[e] : by_column, p.rq.q_zero) & 0xFFu) << (8 * e);
            }
          } else {
            unsigned largest = 0;
#pragma unroll
            for (int t = 0; t < kChunk; ++t)
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const unsigned bits = __float_as_uint(w[t][e]) & 0x7FFFFFFFu;
                largest = bits > largest ? bits : largest;
              }
            const float limit = f8.e5m2 ? 57344.0f : 448.0f;
            if (__builtin_amdgcn_ballot_w64(largest > __float_as_uint(limit)) != 0) {
#pragma unroll
              for (int t = 0; t < kChunk; ++t) {
                packed[t] = 0;
#pragma unroll
                for (int e = 0; e < 4; ++e) packed[t] |= (skl_fp8::encode_ofp8_hw(w[t][e], f8) & 0xFFu) << (8 * e);
              }
            } else if (f8.e5m2) {
#pragma unroll
              for (int t = 0; t < kChunk; ++t)
                packed[t] = (unsigned)__builtin_amdgcn_cvt_pk_bf8_f32(w[t][2], w[t][3], __builtin_amdgcn_cvt_pk_bf8_f32(w[t][0], w[t][1], 0, false), true);
            } else {
#pragma unroll
              for (int t = 0; t < kChunk; ++t)
                packed[t] = (unsigned)__builtin_amdgcn_cvt_pk_fp8_f32(w[t][2], w[t][3], __builtin_amdgcn_cvt_pk_fp8_f32(w[t][0], w[t][1], 0, false), true);
            }
          }
#pragma unroll
          for (int t = 0; t < kChunk; ++t) {
            const size_t row = row_of(top, t), k = col_of(left, t);
            int8_t *const q = q_lane_at + (RUN ? (top - row0 + t * kDown) * p.rq.rsq : (top - row0) * p.rq.rsq + (left + t * kColsDown) * p.rq.csq);
            if (q_run && (!CHECK || (row < p.m && cols_in(k) == 4))) {
              *reinterpret_cast<unsigned *>(q) = packed[t];
            } else {
#pragma unroll
              for (int e = 0; e < 4; ++e)
                if (!CHECK || (row + (RUN ? 0 : e) < p.m && k + (RUN ? e : 0) < p.n)) q[e * (RUN ? p.rq.csq : p.rq.rsq)] = (int8_t)(packed[t] >> (8 * e));
            }
          }
        }
      }
    };

    put(0);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    V4 next[kAhead][kChunk];
    if constexpr (UPDATE) {
#pragma unroll
      for (int a = 0; a < kAhead; ++a) request(a, next[a]);
    }
    if constexpr (kAhead > 1) {  // written out: a loop waits for what its first turn would have to wait for, which has fewer stores in front
      [&]<int... Xs>(std::integer_sequence<int, Xs...>) __attribute__((always_inline)) {
        (chunk(Xs, next[Xs % kAhead]), ...);
      }(std::make_integer_sequence<int, kChunks>{});
    } else {
#pragma clang loop unroll(disable)
      for (unsigned x = 0; x < (unsigned)kChunks; ++x) chunk(x, next[0]);
    }
    if (FUSED && p.max) {
      const T best = skl_wave_max(running);
      if (lane == 0 && best > skl_lowest<T>()) skl_atomic_max(reinterpret_cast<T *>(p.max), best);
    }
  };
  // int8 copies in dwords of whole numbers with no activation but ReLU, of a C that is not read: the loop with nothing but their steps.
  // (The general loop decides at every turn what there is to be done, and its branches cost such a copy more than its arithmetic: us, the
  // general loop / this, each with eight waves: 7424 x 7040 x 512 with ReLU 76 / 71, 4352 x 1024 x 128 9.4 / 8.6.)
  const auto write_int8 = [&]() __attribute__((always_inline)) {
    const int r_lane = lane / (COLS / 4), c_lane = lane % (COLS / 4) * 4;
    const auto column_at = [&](size_t k) { return !CHECK || k < p.n ? k : 0; };
    T *const c_at = c + row_at(r_lane) + row_at(row0) + col_at(col0) + col_at(c_lane);
    int8_t *const q_at = reinterpret_cast<int8_t *>(p.rq.q) + (row0 + r_lane) * p.rq.rsq + col0 + c_lane;
    T bias_of[4];
    float scale_of[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const size_t k = column_at(col0 + c_lane + e);
      bias_of[e] = bias ? bias[k] : T(0);
      scale_of[e] = p.rq.q_scale[p.rq.q_per_column ? k : 0];
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0), as above
    const T floor = p.rq.act == 1 ? T(0) : skl_lowest<T>();
    const bool there = !CHECK || col0 + c_lane + 4 <= p.n;
    constexpr unsigned kOfRow = kPasses / kChunk;
    put(0);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma clang loop unroll(disable)
    for (unsigned x = 0; x < (unsigned)kChunks; ++x) {
      const size_t top = x * (kChunk * kDown);
      const T *const stage_x = stage + (x % kOfRow * (kChunk * kDown) + r_lane) * P + c_lane;
      V4 v[kChunk];
#pragma unroll
      for (int t = 0; t < kChunk; ++t) v[t] = *reinterpret_cast<const V4 *>(stage_x + t * kDown * P);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (x % kOfRow == kOfRow - 1) put(x / kOfRow + 1);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (p.alpha.i != 1) {
#pragma unroll
        for (int t = 0; t < kChunk; ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e) v[t][e] = skl_initialise_plain(v[t][e], p.alpha, p.beta);
      }
#pragma unroll
      for (int t = 0; t < kChunk; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const T w = skl_add_bias(v[t][e], bias_of[e]);
          v[t][e] = w < floor ? floor : w;
        }
      const auto store = [&](auto kept_c) __attribute__((always_inline)) {
        constexpr bool KEPT = decltype(kept_c)::value;
        asm volatile("; %0" ::"n"(KEPT));
#pragma unroll
        for (int t = 0; t < kChunk; ++t) {
          Run4 *const to = reinterpret_cast<Run4 *>(c_at + row_at(top) + row_at(t * kDown));
          if (there && (!CHECK || row0 + top + t * kDown + r_lane < p.m)) {
            if constexpr (KEPT) *to = v[t];
            else __builtin_nontemporal_store((Run4)v[t], to);
          }
        }
        asm volatile("; %0" ::"n"(KEPT));
      };
      if (!p.rq.q_only) {
        if (fits) store(std::true_type{});
        else store(std::false_type{});
      }
#pragma unroll
      for (int t = 0; t < kChunk; ++t) {
        unsigned packed = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) packed |= ((unsigned)skl_requantise_int((float)v[t][e], scale_of[e], p.rq.q_zero) & 0xFFu) << (8 * e);
        if (there && (!CHECK || row0 + top + t * kDown + r_lane < p.m)) *reinterpret_cast<unsigned *>(q_at + (top + t * kDown) * p.rq.rsq) = packed;
      }
    }
  };
  // any row-major C, blocks of four columns and more (a lane at the edge reads its old values from the last four columns)
  const bool run = p.csc0 == 1 && p.ccs >= 2 && (!CHECK || (p.n >= 4 && (p.n % 4 == 0 || p.csc1 == (size_t(1) << p.ccs))));
  const bool update = !skl_beta_is_zero<T>(p.beta);
  constexpr std::true_type yes;
  constexpr std::false_type no;
  if (!run) {
    if (update) write(no, yes, yes, no, yes);
    else write(no, no, yes, no, yes);
    return;
  }
  const auto write_run = [&](auto fused, auto ones) __attribute__((always_inline)) {
    if (!update) write(yes, no, fused, ones, yes);
    else if (one_round) write(yes, yes, fused, ones, yes);
    else write(yes, yes, fused, ones, no);
  };
  const auto write_scaled = [&](auto fused) __attribute__((always_inline)) {
    if constexpr (std::is_same<T, int>::value && !(CHECK && STEPS)) {  // multiplications of whole numbers take four times as long as anything else here
      if (p.alpha.i == 1 && (p.beta.i == 0 || p.beta.i == 1)) {
        write_run(fused, yes);
        return;
      }
    }
    write_run(fused, no);
  };
  if constexpr (STEPS) {
    if constexpr (std::is_same<T, int>::value) {
      if (!update && !p.max && dword_copy<T>(p.rq) && (!CHECK || p.n % 4 == 0)) {
        write_int8();
        return;
      }
    }
    write_scaled(yes);
  } else {
    if (p.bias || p.max) write_scaled(yes);
    else write_scaled(no);
  }
}

// The raw sums of one share of K, held as in write_wave_rows, to the share's M x N plane.
template <int MI, int NI, bool CHECK, typename Acc>
__device__ __forceinline__ void write_wave_plane(const MfmaArgs &p, const Acc (&acc)[MI][NI], size_t row0, size_t col0, unsigned split) {
  using T = decltype(Acc{}.x);
  typedef T Run4 __attribute__((ext_vector_type(4), aligned(4)));
  constexpr int S = sizeof(Acc) == 64 ? 32 : 16, G = S == 32 ? 4 : 1;
  const int lane = threadIdx.x & 63;
  T *const plane = reinterpret_cast<T *>(p.partial) + (size_t)split * p.m * p.n;
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const Acc sums = i < MI - 1 || j < NI / 2 ? fetched<true>(acc[i][j]) : fetched<ring_sum_in_a<MI, NI, Acc>(MI - 1, NI - 1)>(acc[i][j]);
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const size_t row = row0 + i * S + lane % S, col = col0 + j * S + g * 8 + lane / S * 4;
        const Run4 v = {sums[4 * g], sums[4 * g + 1], sums[4 * g + 2], sums[4 * g + 3]};
        T *const to = plane + row * p.n + col;
        if (!CHECK || (row < p.m && col + 4 <= p.n)) {
          *reinterpret_cast<Run4 *>(to) = v;
        } else if (row < p.m) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (col + e < p.n) to[e] = v[e];
        }
      }
    }
}

// Tile index of a workgroup. Consecutive workgroup ids go to different XCDs
// (eight of them, each with its own L2), so ids are first regrouped per XCD into
// contiguous ranges, then walked in column-major groups of kGroupM tile rows so
// that the tiles resident on one XCD at a time share A and B panels.
// ANY: also when the tiles are not a multiple of eight. The bounds-checked kernels gain by it (bf16 6409 x 14591 x 1344 on
// 5814 tiles of 128 x 128: 458 -> 398 us); the streaming kernel with its larger tiles does not (int8 5169 x 15488 x 704 on
// 1281 tiles: 362 -> 389 us): its eight XCDs then read eight tile rows of the same columns.
template <bool ANY>
__device__ __forceinline__ void tile_of_block(unsigned bid, const MfmaArgs &p, unsigned &tm, unsigned &tn) {
  constexpr unsigned kXcd = 8, kGroupM = 8;
  const unsigned tiles_m = p.tiles_m, tiles_n = p.tiles_n;
  const unsigned total = tiles_m * tiles_n, xcd = bid % kXcd, longer = total % kXcd;  // the first `longer` ranges hold one tile more
  unsigned t = bid;
  if (ANY || longer == 0) t = xcd * (total / kXcd) + (xcd < longer ? xcd : longer) + bid / kXcd;
  const unsigned per_group = kGroupM * tiles_n;
  const unsigned group = p.by_group ? __umulhi(t, p.by_group) : t / per_group, first_m = group * kGroupM;
  const unsigned in_group = t - group * per_group;
  const bool full = tiles_m - first_m >= kGroupM;
  const unsigned rows = full ? kGroupM : tiles_m - first_m;  // of the last group: tiles_m % 8
  const unsigned column = full ? in_group / kGroupM : rows == 1 ? in_group : p.by_group ? __umulhi(in_group, p.by_rest) : in_group / rows;
  tm = first_m + in_group - column * rows;
  tn = column;
}

enum Few { kFewRows = 1, kFewest = 2 };  // gemm_mfma_kernel's FEW

// The kernel for ragged and small problems: any M, N and K, operands on any boundary. A problem of few tiles is bound by the
// time from one slice to the next (requests, their memory latency, LDS, barrier), so several slices of loads are under way, and
// the loads are never guarded (Loader). Guarded loads, a slice ahead -> this, us: int8 512^3 5.9 -> 5.0, bf16 16 x 11008 x 4096
// 28.4 -> 23.7 with its second pass, int8 136 x 704 x 2207 51 -> 12.4 (no copy of A in front), f16 427 x 5901 x 1805 93 -> 33;
// over 120 random problems 0.70.
template <int TA, int TB, bool A_KC, bool B_KC, int BM, int BN, int WAVES_M, int WAVES_N, bool EXACT = false, bool EXTRA = false, int FEW = 0>
__global__ void __launch_bounds__(WAVES_M *WAVES_N * 64, (BM == 64 ? 2 : 4)) gemm_mfma_kernel(MfmaArgs p) {
  constexpr int NT = WAVES_M * WAVES_N * 64;
  using KA = Kind<TA>;
  using M = typename std::conditional<EXACT, MmaF8Exact<TA, TB>, Mma<TA, TB>>::type;
  using Acc = typename KA::Acc;
  using AccElem = decltype(Acc{}.x);
  constexpr int ES = KA::ES;
  constexpr int KB = EXACT ? 32 : KA::KB;       // bytes of K per MFMA step
  constexpr int FRB = KB / 2;                   // fragment bytes per lane
  constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;  // wave tile
  constexpr int MI = WM / 32, NI = WN / 32;     // MFMA blocks per wave
  using TileA = Tile<ES, BM, A_KC, NT>;
  using TileB = Tile<ES, BN, B_KC, NT>;
  constexpr int kStage = TileA::kBytes + TileB::kBytes;
  // Slices under way: 16 registers each, of the 128 a thread has (the 32-byte fragments of the fp8 kinds take twice the room);
  // 64 x 64: 32 of 256.
  constexpr int kAhead = BM == 128 ? (FRB == 32 ? 1 : 2) : 2;

  extern __shared__ __attribute__((aligned(16))) char smem[];

  unsigned tm, tn;
  const unsigned split = blockIdx.y;
  tile_of_block<true>(blockIdx.x, p, tm, tn);
  const size_t m0 = (size_t)tm * BM, n0 = (size_t)tn * BN;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;  // the wave index as a scalar: nothing derived from it occupies a vector register across the main loop
  const int wm = (wave / WAVES_N) * WM, wn = (wave % WAVES_N) * WN;

  Loader<ES, BM, A_KC, NT> la;
  Loader<ES, BN, B_KC, NT> lb;
  la.init(p.a, m0, p.m, p.a_s1, p.a_s0, p.a_sk, p.a_loose);
  lb.init(p.b, n0, p.n, p.b_s1, p.b_s0, p.b_sk, p.b_loose);

  Acc acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;

  // This workgroup's share of K: whole slices, and the elements from slice s on that belong to it (as a number of at most 31
  // bits; negative beyond the end).
  constexpr int KE = TileA::KE;
  const size_t all_slices = (p.k + KE - 1) / KE;
  const size_t s_begin = (size_t)split * p.slices_per_split;  // the host makes every split non-empty
  const size_t s_end = all_slices - s_begin < p.slices_per_split ? all_slices : s_begin + p.slices_per_split;
  const unsigned count = (unsigned)(s_end - s_begin);
  const int last_left = (int)((s_end == all_slices ? p.k : s_end * KE) - (s_end - 1) * KE);  // elements in the last slice
  const auto left = [&](unsigned s) __attribute__((always_inline)) { return s + 1 < count ? KE : s + 1 == count ? last_left : 0; };

  // Slices s + 1 to s + kAhead are on their way, global -> registers, while slice s is multiplied from LDS.
  v4i ra[kAhead][TileA::kPerThread], rb[kAhead][TileB::kPerThread];
#pragma unroll
  for (int d = 0; d < kAhead; ++d) {
    la.fetch(ra[d], s_begin + d, left(d));
    lb.fetch(rb[d], s_begin + d, left(d));
  }
  la.template stash<true>(smem, ra[0], left(0));
  lb.template stash<true>(smem + TileA::kBytes, rb[0], left(0));
  la.fetch(ra[0], s_begin + kAhead, left(kAhead));
  lb.fetch(rb[0], s_begin + kAhead, left(kAhead));
  __builtin_amdgcn_sched_barrier(0);
  __syncthreads();

  constexpr int kSteps = TileA::kSlice / KB;  // MFMA k-steps per slice
  // Operand fragments: read a k-step ahead of their use, or, 64 x 64, all of a slice at once.
  constexpr bool kAllAtOnce = BM == 64;
  constexpr int kSets = kAllAtOnce ? kSteps : 2;
  typename M::Frag fa[kSets][MI], fb[kSets][NI];
  const auto read_step = [&](unsigned s, int ks, int set) __attribute__((always_inline)) {
    const char *ta = smem + (s & 1) * kStage;
    const char *tb = ta + TileA::kBytes;
#pragma unroll
    for (int i = 0; i < MI; ++i) fa[set][i] = read_frag<ES, BM, A_KC, FRB>(ta, wm + i * 32, ks * KB);
#pragma unroll
    for (int j = 0; j < NI; ++j) fb[set][j] = read_frag<ES, BN, B_KC, FRB>(tb, wn + j * 32, ks * KB);
  };
  const auto products = [&](int set) __attribute__((always_inline)) {
    decltype(prep_a<M>(fa[set][0])) wa[MI];
    decltype(prep_b<M>(fb[set][0])) wb[NI];
#pragma unroll
    for (int i = 0; i < MI; ++i) wa[i] = prep_a<M>(fa[set][i]);
#pragma unroll
    for (int j = 0; j < NI; ++j) wb[j] = prep_b<M>(fb[set][j]);
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) acc[i][j] = M::run(wa[i], wb[j], acc[i][j]);
  };
  // Slice s, whose loads have been under way for kAhead slices, into LDS; slice s + kAhead requested in its registers (not
  // by the last slices: LAST).
  const auto advance = [&](auto last, unsigned s, v4i (&next_a)[TileA::kPerThread], v4i (&next_b)[TileB::kPerThread]) __attribute__((always_inline)) {
    constexpr bool LAST = decltype(last)::value;
    char *na = smem + (s & 1) * kStage;
    la.template stash<LAST>(na, next_a, left(s));
    lb.template stash<LAST>(na + TileA::kBytes, next_b, left(s));
    if constexpr (!LAST) {
      la.fetch(next_a, s_begin + s + kAhead, left(s + kAhead));
      lb.fetch(next_b, s_begin + s + kAhead, left(s + kAhead));
      __builtin_amdgcn_sched_barrier(0);  // the loads stay up here, not next to the stores that use them
    }
  };
  // How the products of a floating-point kind are added up on the 64 x 64 tiles. Every product of the chain in `acc` rounds at the
  // size of the sum so far, so one chain over a long K loses what short ones keep.
  // blocked_sums, a K that the larger tile would share between workgroups: the products of two slices, 512 bytes of K as in the
  // shortest share there is, are a sum of their own, and `sum` adds those (bf16 1024 x 1024 x 2048, error against 64 bits: one chain
  // 2.7e-7, eight shares 1.0e-7, blocks 1.0e-7).
  // FEW, a few rows in place of a streaming kernel, with sums as exact as its many short ones: half a slice is a block and, kFewest,
  // what its addition to `sum` loses is carried along in `lost`: seven instructions per element and four products, for the rows
  // that exist.
  // (Not for the fp8 instructions: what they lose in aligning products, 1.3e-5, does not depend on the sums.)
  constexpr bool kSums = BM == 64 && (EXACT || ES == 2);
  static_assert(kSums || !FEW);
  [[maybe_unused]] Acc sum[kSums ? MI : 1][kSums ? NI : 1], lost[FEW == kFewest ? MI : 1][FEW == kFewest ? NI : 1];
  [[maybe_unused]] const auto settle = [&]() __attribute__((always_inline)) {
    if constexpr (kSums) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            sum[i][j][r] = __fadd_rn(sum[i][j][r], acc[i][j][r]);
            acc[i][j][r] = 0;
          }
    }
  };
  [[maybe_unused]] const auto settle_rows = [&](auto from, auto to) __attribute__((always_inline)) {
    if constexpr (FEW) {
      static_assert(MI == 1 && NI == 1);
#pragma unroll
      for (int r = decltype(from)::value; r < decltype(to)::value; ++r) {
        if constexpr (FEW == kFewest) {
          float l = lost[0][0][r];
          sum[0][0][r] = skl_add_keeping_loss(sum[0][0][r], acc[0][0][r], l);
          lost[0][0][r] = l;
        } else {
          sum[0][0][r] = __fadd_rn(sum[0][0][r], acc[0][0][r]);
        }
        acc[0][0][r] = 0;
      }
    }
  };
  [[maybe_unused]] const auto settle_existing = [&]() __attribute__((always_inline)) {  // registers 0 to 3 hold rows 0 to 7 of the wave's, 4 to 7 rows 8 to 15
    if (m0 + wm >= p.m) return;
    settle_rows(std::integral_constant<int, 0>{}, std::integral_constant<int, 4>{});
    if (p.m > 8) settle_rows(std::integral_constant<int, 4>{}, std::integral_constant<int, 8>{});
    if (p.m > 16) settle_rows(std::integral_constant<int, 8>{}, std::integral_constant<int, 16>{});
  };
  if constexpr (kSums) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) {
        sum[i][j] = acc[i][j];
        if constexpr (FEW == kFewest) lost[i][j] = acc[i][j];
      }
  }
  // Slice s is multiplied and, if there are `more`, the next one put into the other half of LDS, which every wave has left.
  const auto slice = [&](auto last, bool more, unsigned s, v4i (&next_a)[TileA::kPerThread], v4i (&next_b)[TileB::kPerThread]) __attribute__((always_inline)) {
    read_step(s, 0, 0);
    if constexpr (kAllAtOnce) {  // the next slice's stores land under this one's products
#pragma unroll
      for (int ks = 1; ks < kSteps; ++ks) read_step(s, ks, ks);
      if (more) advance(last, s + 1, next_a, next_b);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < kSteps; ++ks) {
        products(ks);
        if (FEW && ks % (kSteps / 2) == kSteps / 2 - 1) settle_existing();
      }
    } else {
#pragma unroll
      for (int ks = 0; ks < kSteps; ++ks) {
        // The next k-step's LDS reads are all issued before the first MFMA below and are not needed until then: the scheduler
        // must not pull them down next to their uses.
        if (ks + 1 < kSteps) read_step(s, ks + 1, (ks + 1) & 1);
        __builtin_amdgcn_sched_barrier(0);
        products(ks & 1);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (more) advance(last, s + 1, next_a, next_b);
    }
    if (more) __syncthreads();
  };
  // The compiler counts the loads in flight along every path into a block: a loop with a way out after each slice, or around
  // one, makes it wait for the youngest of them. So the loop runs whole rounds of kAhead slices, up to the last kAhead + 1.
  static_assert(!kSums || kAhead == 2, "a round is a block");
  unsigned s = 0;
  for (; s + kAhead + 1 < count; s += kAhead) {
    [&]<int... Us>(std::integer_sequence<int, Us...>) __attribute__((always_inline)) {
      (slice(std::false_type{}, true, s + Us, ra[(Us + 1) % kAhead], rb[(Us + 1) % kAhead]), ...);
    }(std::make_integer_sequence<int, kAhead>{});
    if (kSums && !FEW && p.blocked_sums) settle();
  }
  [&]<int... Us>(std::integer_sequence<int, Us...>) __attribute__((always_inline)) {
    (void)((slice(std::true_type{}, s + 1 < count, s, ra[(Us + 1) % kAhead], rb[(Us + 1) % kAhead]), ++s < count) && ...);
  }(std::make_integer_sequence<int, kAhead>{});
  if (s < count) {
    if (kSums && !FEW && p.blocked_sums) settle();
    slice(std::true_type{}, false, s, ra[0], rb[0]);
  }
  if constexpr (kSums) {
    if (!FEW && p.blocked_sums) settle();
    if (FEW || p.blocked_sums) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = sum[i][j];
    }
  }

  // Lane l of a 32x32 block holds column l%32 and rows 8*(r/4) + 4*(l/32) + r%4.
  if (p.splits > 1) {  // a share of K: the raw sums go to this split's M x N plane
    AccElem *plane = reinterpret_cast<AccElem *>(p.partial) + (size_t)split * p.m * p.n;
#pragma unroll
    for (int j = 0; j < NI; ++j) {
      const size_t col = n0 + wn + j * 32 + (lane & 31);
      if (col >= p.n) continue;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const size_t row = m0 + wm + i * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
          if (row < p.m) plane[row * p.n + col] = acc[i][j][r];
        }
    }
    return;
  }
  if constexpr (EXTRA) {
    __syncthreads();  // the last slice has been read by every wave
    write_wave_tile_staged<MI, NI, true>(p, acc, m0 + wm, n0 + wn, smem + wave * 32 * staged_pitch<NI>() * 4);
  } else {
    if constexpr (BM == 64) {  // a tile that lies inside C is written without a test per element
      if (m0 + BM <= p.m && n0 + BN <= p.n) {
        write_wave_tile<MI, NI, false>(p, acc, m0 + wm, n0 + wn);
        return;
      }
    }
    write_wave_tile<MI, NI, true>(p, acc, m0 + wm, n0 + wn);
  }
}

// ===========================================================================
// Streaming kernel for whole tiles (256 x 256 or 256 x 128): global -> LDS
// without passing through registers (global_load_lds_dwordx4), K in slices of
// 64 bytes held in a ring of four or six LDS stages. Each wave-level load deposits
// 64 x 16 bytes as one contiguous KiB of LDS, so tiles are stored without
// padding and bank conflicts are avoided by an XOR swizzle of the 16-byte
// chunk index instead; the swizzle is applied on the global side (which chunk
// a lane fetches) and again by the fragment reads. Four waves, one per
// SIMD, a quarter of the tile each, so that every byte in LDS is read by two
// waves (eight waves of a quarter of the columns read a half more; bf16 with K
// contiguous, us, eight waves of 32 x 32 products / this: 8192^3 843 / 721,
// 4096^3 115 / 97.5), or eight, two per SIMD (ring_waves).
//
// An MN-contiguous operand (k-rows of ROWS elements) is loaded a slice at a
// time: a load covers whole k-rows, i.e. whole 128-byte lines. A K-contiguous
// operand is different: a 64-byte slice is HALF a line of each row, and loads
// made of half lines run at less than half the rate of loads made of whole
// ones. So its loads cover 8 rows x 128 bytes - two slices at once - and the
// stages of such an operand are interleaved in LDS at 512-byte granularity
// (8 rows x 64 bytes of stage 0, then of stage 1, ...), which puts the two
// halves of such a load next to each other: one KiB, as the load writes it.
// ===========================================================================
constexpr int kRingSlice = 64;   // bytes of K per stage
// Waves. Four, one per SIMD, each a quarter of the tile, so that as little as possible is read twice: the fastest main loop. Eight, two
// per SIMD, where what is around the loop counts: one wave's start, old C, steps and stores lie under the other's. Eight over four waves,
// geometric means over 600 random problems, by K in bytes from 512 / 1024 / 2048 / 4096 / 8192:
//                            256 x 256 tiles                          256 x 128 tiles
//   ragged, 16 bits, plain   0.79 0.90 0.91 0.89 0.89                 0.82 0.87 0.90 0.91 0.97
//           int8, plain       -   0.93 0.93  -    -                   0.87 0.93 0.94  -   0.94    fp8, beyond the exact K  0.94 0.96 0.98
//           with steps       0.77 to 0.87 (int8 0.81 to 0.87)         0.78 to 0.93 (int8 0.83 to 0.96, fp8 0.88 to 0.96)
//   whole, with steps        16 bits 0.80 0.83 0.89 0.93 0.92         0.82 0.84 0.88 0.93 0.96
//                            exact fp8 0.86 0.90 0.82, int8 0.89 to 0.96   0.81 0.87 0.85, int8 0.90 0.94 0.96 1.01 1.04, fp8 0.85 0.91 0.94
//          exact fp8, plain  0.96 0.95                                0.89 0.92 0.94    fp8 beyond it, plain or C read, 0.96 to 0.99
//          16 bits, C read   1.02 1.02 1.00 0.98 1.03                 0.92 0.93 0.98 0.98 0.99     plain  -   0.94 0.94 0.96 0.99
//          int8, C read       -   1.02 1.00  -    -                    -   0.97 0.98 1.00 1.02     plain 0.93 0.99 1.02 0.99
// fp8 beyond the exact K keeps four on 256 x 256 tiles: fragments of 32 x 32 products leave eight no registers. So do the calls whose old C
// is looked through (SCAN): its slots would not fit beside the stages.
constexpr bool ring_few_issue_slots(int es, bool a_kc, bool b_kc, int bn) { return es == 1 && !a_kc && !b_kc && bn == 128; }
template <int TA, bool A_KC, bool B_KC, int BN, bool EDGE, bool STEPS, bool SCAN, bool EXACT>
constexpr int ring_waves() {  // 0: ring_waves_by_size
  constexpr bool fp8 = TA == SKL_DT_F8E4M3 || TA == SKL_DT_F8E5M2;
  if (fp8 && !EXACT && BN == 256) return 4;
  if (SCAN) return fp8 && ring_few_issue_slots(1, A_KC, B_KC, BN) ? 8 : 4;
  if (EXACT && BN == 256 && !EDGE && !STEPS) return 0;
  return fp8 || EDGE || STEPS ? 8 : 0;
}
// Of them side by side: two; eight of 256 x 256 tiles four where that holds fewer widened fragments (EXACT; the other way 34 registers
// are spilled) and where C is read (us, two / four: int8 8192^2 x 1024 162 / 149, 4096 x 8192 x 2048 103 / 102, bf16 the same).
constexpr int ring_waves_n(int waves, int bn, bool edge, bool steps, bool exact) { return waves == 8 && bn == 256 && (exact || !(edge || steps)) ? 4 : 2; }
// Stages of an operand's ring: four, or six of an operand with K contiguous where 160 KiB of LDS hold them (see the kernel's loads).
constexpr int ring_stages_a(bool a_kc, bool b_kc, int bn, bool scan) { return !a_kc || (bn == 256 && (b_kc || scan)) ? 4 : 6; }
constexpr int ring_stages_b(bool, bool b_kc, int bn, bool scan) { return !b_kc || (bn == 256 && scan) ? 4 : 6; }
template <int ES, bool KC, int ROWS, int NS, int SIDE>
struct STile {
  static constexpr int kStages = NS;
  static constexpr int kBytes = ROWS * kRingSlice;            // one stage
  static constexpr int kRegion = kBytes * NS;                 // all stages of the operand
  static constexpr int kRowBytes = ROWS * ES;                 // a k-row of an MN-contiguous tile
  static constexpr int kStageStep = KC ? 512 : kBytes;        // from one stage to the next
  static constexpr int kGroup = NS * 512;                     // K-contiguous: from 8 rows to the next 8
  // K-contiguous: a b128 read is served 16 lanes at a time - 0-3, 12-15 and 20-27, then 4-11, 16-19 and 28-31, and so in the upper
  // half (found from the conflicts of other arrangements) -, which in 16 x 4 chunks are the 16 rows, eight of them with the next chunk.
  __device__ static constexpr int turn(int r) { return (r >> 2 & 3) ^ (r >> 1 & 2); }
  // Byte offset (inside stage 0) of 16-byte chunk `c` of line `r`. A line is an M/N row
  // holding 64 bytes of K (KC), or a k-row holding ROWS elements along M/N (MC).
  __device__ static __forceinline__ int chunk(int r, int c) {
    if constexpr (KC)  // 4 chunks: rows r and r+4 share banks, the XOR parts them; 16 rows fill the banks once
      return (r >> 3) * kGroup + (r & 7) * 64 + ((c ^ turn(r)) << 4);
    else if constexpr (ES == 2)  // 32 or 16 chunks; 32 lanes of a tr16 read take k-rows r .. r + 3 and r + 8 .. r + 11, 32 B of each
      return r * kRowBytes + ((c ^ ((r & 3) << 1 | (r & 8))) << 4);
    else if constexpr (SIDE == 32 && kRowBytes == 256)
      return r * 256 + ((c ^ ((r & 7) << 1)) << 4);   // 16 chunks; tr8 reads take 8 k-rows x 32 B
    else if constexpr (SIDE == 32)
      return r * 128 + ((c ^ (((r >> 1) & 3) << 1)) << 4);  // 8 chunks: two k-rows fill the banks once
    else if constexpr (kRowBytes == 256)  // 32 lanes of a tr8 read take k-rows r .. r + 7 and r + 16 .. r + 23, 16 B of each
      return r * 256 + ((c ^ ((r & 7) | (r >> 1 & 8))) << 4);
    else
      return r * 128 + ((c ^ ((r >> 1 & 3) | (r >> 2 & 4))) << 4);
  }
};

// 16 bytes per lane from g + off to LDS at `lds`, where the wave's KiB begins. (In assembly, like the loads that go out with a product
// (RingMma): those write M0 without the compiler's knowing, so no load beside them may be one for which it keeps M0.)
__device__ __forceinline__ void load_to_lds(unsigned lds, const char *g, unsigned off) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(g) : "memory");
}

// Global -> LDS loads of one operand, this wave's share. `unit` below is a slice
// for an MN-contiguous operand and a pair of slices for a K-contiguous one.
// EDGE: the operand ends inside the tile, along M / N or along K. Its loads go through a buffer descriptor whose base follows K
// as a scalar; a lane whose 16 bytes do not exist holds an offset beyond the descriptor's range, for which the load writes zeros
// to LDS and touches no memory. The offsets of rows beyond M / N are so from the start; those of k beyond the end are chosen
// with every load (offset()).
template <int ES, bool KC, int WAVES, int ROWS, int NS, int SIDE, bool EDGE>
struct SLoader {
  using T = STile<ES, KC, ROWS, NS, SIDE>;
  static constexpr unsigned kRange = 0xC0000000u, kOutside = 0xE0000000u;  // (the host checks that offsets stay below kRange)
  static constexpr int kUnitBytes = KC ? 2 * T::kBytes : T::kBytes;
  static constexpr int kBlocks = kUnitBytes / 1024 / WAVES;  // KiB blocks per wave and unit
  static_assert(kBlocks >= 1, "every wave loads at least one block per unit");
  const char *tile_base;
  size_t k_step;           // bytes from one unit to the next
  unsigned off[kBlocks];   // global byte offsets of this lane
  unsigned lds;            // LDS byte offset (inside the operand's region, stage 0) of block 0
  static constexpr unsigned kBlockStep = KC ? T::kGroup : 1024;  // ... and from one block to the next
  unsigned k_lane;         // EDGE: where along K the lane's 16 bytes of block 0 lie in a unit - KC: bytes, MC: k rows
  unsigned k_total;        // EDGE: bytes / k rows of K

  __device__ __forceinline__ void init(const char *base, size_t mn0, size_t mn_dim, size_t k, size_t s1, size_t s0, size_t sk) {
    // The wave index as a scalar: the LDS address of a block (which goes into M0) is then scalar arithmetic, not a
    // vector add and a v_readfirstlane per load, and lds[] lives in scalar registers.
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    tile_base = base + (mn0 >> 6) * s1 * ES;
    lds = wave * kBlocks * kBlockStep;
    // spelled out as scalars, like the step below: the loads take their base as one (EDGE: a descriptor in vector registers costs a
    // loop over the lanes per load)
    const uintptr_t at = (uintptr_t)tile_base;
    tile_base = (const char *)(((uintptr_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(at >> 32)) << 32) | (unsigned)__builtin_amdgcn_readfirstlane((int)at));
#pragma unroll
    for (int i = 0; i < kBlocks; ++i) {
      const int b = wave * kBlocks + i;
      if constexpr (KC) {  // block = 8 rows x (64 bytes of the even slice, then 64 bytes of the odd one)
        const int half = lane >> 5, row = 8 * b + ((lane & 31) >> 2), pos = lane & 3;
        const int c = pos ^ T::turn(row);
        off[i] = (unsigned)(((size_t)(row >> 6) * s1 + (size_t)(row & 63) * s0) * ES + half * 64 + c * 16);
        if constexpr (EDGE) {
          static_assert(kBlocks % 2 == 0, "c of block i is that of block 0 with its second bit turned for odd i");
          if (i == 0) k_lane = half * 64 + c * 16;
          if (mn0 + row >= mn_dim) off[i] = kOutside;
        }
      } else {
        constexpr int kLanesPerRow = T::kRowBytes / 16, kRowsPerBlock = 1024 / T::kRowBytes;
        const int kr = kRowsPerBlock * b + lane / kLanesPerRow, pos = lane % kLanesPerRow;
        const int mn = ((T::chunk(kr, pos) - kr * T::kRowBytes) >> 4) * (16 / ES);  // the chunk stored at position `pos`
        off[i] = (unsigned)(((size_t)(mn >> 6) * s1 + (size_t)(mn & 63) + (size_t)kr * sk) * ES);
        if constexpr (EDGE) {
          if (i == 0) k_lane = kr;
          if (mn0 + mn >= mn_dim) off[i] = kOutside;
        }
      }
    }
    if constexpr (EDGE) k_total = (unsigned)(KC ? k * ES : k);
    // (spelled out as a scalar: as a member next to per-lane offsets it otherwise ends up in a vector register, and
    // every load of an MN-contiguous operand pays a 64-bit vector multiply-add for its address)
    const size_t step = KC ? (size_t)(2 * kRingSlice) : (size_t)(kRingSlice / ES) * sk * ES;
    k_step = ((size_t)(unsigned)__builtin_amdgcn_readfirstlane((int)(step >> 32)) << 32) | (unsigned)__builtin_amdgcn_readfirstlane((int)step);
  }

  // EDGE: how much of K (bytes / k rows) is left from the start of `unit` on, and the offset of the lane's 16 bytes of block i of a
  // unit of which so much exists. (Chosen for every load: a branch for the last units, in a loop whose sums are all of the accumulation
  // registers, has the compiler move a block of sums about behind a product that is still under way.)
  static constexpr unsigned kUnitK = KC ? 2 * kRingSlice : kRingSlice / ES;
  __device__ __forceinline__ unsigned left_of(unsigned unit) const { return k_total > unit * kUnitK ? k_total - unit * kUnitK : 0; }
  __device__ __forceinline__ unsigned offset(unsigned left, int i) const {
    if constexpr (!EDGE) return off[i];
    if constexpr (KC) return (k_lane ^ (unsigned)(i & 1) * 32u) < left ? off[i] : kOutside;
    const unsigned rows_above = (unsigned)i * (1024 / T::kRowBytes);
    return k_lane < (left > rows_above ? left - rows_above : 0) ? off[i] : kOutside;
  }

  // Requests block `i` of `unit`; it lands in stage `stage` (the even one of the pair for KC) of `region`.
  __device__ __forceinline__ void issue_one(char *region, int stage, size_t unit, unsigned left, int i) const {
    const char *g = tile_base + unit * k_step;
    if constexpr (EDGE) {
      // The lane's offset through a copy the compiler cannot follow: it otherwise widens every offset to 64 bits ahead
      // of the loop, two registers each.
      unsigned o = offset(left, i);
      asm volatile("" : "+v"(o));
      __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void *)g, 0, (int)kRange, 0x00027000),
                                               (__attribute__((address_space(3))) void *)(region + stage * T::kStageStep + lds + i * kBlockStep), 16, (int)o, 0, 0, 0);
    } else {
      load_to_lds((unsigned)(size_t)LDS_PTR(char, region) + stage * T::kStageStep + lds + i * kBlockStep, g, off[i]);
    }
  }
};

// ---------------------------------------------------------------------------
// The software pipeline is written out by hand:
//   * Fragment reads are inline assembly. The compiler cannot tell an LDS read
//     from the LDS writes of outstanding global->LDS loads apart and makes every
//     ds_read_tr wait for ALL loads in flight (vmcnt(0)), and it waits for reads
//     it has only just issued (lgkmcnt(0) in front of every step) - either
//     one exposes a memory latency per step. Here the kernel does its own
//     counting: one lgkmcnt(0) at the top of a step, when the only reads in
//     flight are the ones issued during the previous step; one vmcnt(n) per
//     slice in front of the barrier.
//   * Reads and loads are dealt out one at a time behind the MFMAs instead of
//     going out in bursts: a wave issues in order, and a burst that finds the
//     LDS or the load path busy is a stretch in which it issues no MFMA. The
//     reads sit behind the first three quarters of a step's MFMAs, which leaves
//     the last quarter for them to land.
// ---------------------------------------------------------------------------
template <int N>
__device__ __forceinline__ void wait_loads_upto() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <int OFF>
__device__ __forceinline__ v4i lds_read_b128(unsigned addr) {
  v4i r;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(OFF) : "memory");
  return r;
}
template <int OFF>
__device__ __forceinline__ v2i lds_read_b64(unsigned addr) {
  v2i r;
  asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(OFF) : "memory");
  return r;
}
template <int OFF>
__device__ __forceinline__ v2i lds_read_tr8(unsigned addr) {
  v2i r;
  asm volatile("ds_read_b64_tr_b8 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(OFF) : "memory");
  return r;
}
template <int OFF>
__device__ __forceinline__ v2i lds_read_tr16(unsigned addr) {
  v2i r;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(OFF) : "memory");
  return r;
}

// The fragments of one operand for one wave: NFRAG blocks of SIDE rows with the 64 bytes of K of a stage, read in pieces of
// one LDS instruction each. Lane l holds row l % SIDE; its FRB bytes of K are the (l / SIDE)-th of the stage. Offsets inside the
// stage are per lane and computed once; what changes from fragment to fragment is, wherever the swizzle allows, an immediate
// offset, else an exclusive or.
// EXACT: two pieces of eight bytes, one for each of two products of 32 bytes of K. Lane groups 0 to 3 hold the first, third, second and
// fourth eight bytes of the 32: the products are then added up in the order of the bounds-checked kernels, which take a 16-byte
// fragment's low halves first, so that a call's sums are the same on both.
template <int ES, bool KC, int FRB, int ROWS, int NS, int SIDE, bool EXACT>
struct FragReader {
  using T = STile<ES, KC, ROWS, NS, SIDE>;
  static constexpr int RB = T::kRowBytes;
  static constexpr int kPieceBytes = KC && !EXACT ? 16 : 8;
  using Piece = typename std::conditional<kPieceBytes == 16, v4i, v2i>::type;
  static constexpr int kPieces = FRB / kPieceBytes;  // LDS instructions per fragment
  static constexpr int kBases = KC ? kPieces : 1;
  static constexpr int kTurn = SIDE * ES;            // fragment f: its columns' chunks are those of fragment 0 with f * kTurn turned
  static_assert(FRB * (64 / SIDE) == kRingSlice, "a fragment takes the whole stage");
  static_assert(!EXACT || (ES == 1 && SIDE == 16));
  unsigned base[kBases];

  __device__ void init(int row0) {
    const int lane = threadIdx.x & 63, g = lane / SIDE;
    [[maybe_unused]] const int eighth = (g & 1) * 2 + (g >> 1);  // EXACT: which eight bytes of 32
    if constexpr (KC) {
#pragma unroll
      for (int pc = 0; pc < kPieces; ++pc)
        base[pc] = EXACT ? (unsigned)(T::chunk(row0 + lane % SIDE, 2 * pc + (eighth >> 1)) + (eighth & 1) * 8) : (unsigned)T::chunk(row0 + lane % SIDE, ((g * FRB) >> 4) + pc);
    } else {
      // 16 lanes read 8 k-rows x 16 bytes (16-bit: 4 k-rows x 16 elements), lane j receives column j
      const int g16 = SIDE == 32 ? (lane >> 4) & 1 : 0, j = lane & 15;
      if constexpr (ES == 1)
        base[0] = (unsigned)(T::chunk((EXACT ? eighth * 8 : g * FRB) + (j >> 1), (row0 >> 4) + g16) + (j & 1) * 8);
      else
        base[0] = (unsigned)(T::chunk(g * (FRB / 2) + (j >> 2), (row0 >> 3) + g16 * 2 + ((j & 3) >> 1)) + (j & 1) * 8);
    }
  }
  // Piece PC of fragment F of the stage at LDS address `stage`.
  template <int F, int PC>
  __device__ __forceinline__ Piece read(unsigned stage) const {
    if constexpr (KC && EXACT)
      return lds_read_b64<F * (SIDE / 8) * T::kGroup>(stage + base[PC]);
    else if constexpr (KC)
      return lds_read_b128<F * (SIDE / 8) * T::kGroup>(stage + base[PC]);
    else if constexpr (ES == 1)
      return lds_read_tr8<PC * (EXACT ? 32 : 8) * RB>(stage + (base[0] ^ (unsigned)(F * kTurn)));
    else
      return lds_read_tr16<PC * 4 * RB>(stage + (base[0] ^ (unsigned)(F * kTurn)));
  }
};

template <typename Frag, typename Piece, int N>
__device__ __forceinline__ Frag join_pieces(const Piece (&pc)[N]) {
  if constexpr (sizeof(Piece) == sizeof(Frag)) {
    return pc[0];
  } else if constexpr (sizeof(Piece) == 16) {  // two 128-bit pieces
    return Frag{pc[0].x, pc[0].y, pc[0].z, pc[0].w, pc[1].x, pc[1].y, pc[1].z, pc[1].w};
  } else if constexpr (N == 2) {
    return Frag{pc[0].x, pc[0].y, pc[1].x, pc[1].y};
  } else {
    return Frag{pc[0].x, pc[0].y, pc[1].x, pc[1].y, pc[2].x, pc[2].y, pc[3].x, pc[3].y};
  }
}

template <int X>
__device__ __forceinline__ v4i half_of(v8i f) { return v4i{f[4 * X], f[4 * X + 1], f[4 * X + 2], f[4 * X + 3]}; }

constexpr int ceil_div(int a, int b) { return (a + b - 1) / b; }

// EDGE: problems that are not whole tiles, or whole pairs of slices along K: the loads take nothing from beyond the operands
// (SLoader), and the epilogue touches no row or column beyond p.m / p.n.
// SCAN (floating-point row-major C, beta == 0 evaluated like the reference's loops, whole tiles, K of at least 64
// slices on the wide tile and 32 on the narrow one): whether 0 * c is a zero for every old c of the tile - i.e. no NaN,
// no infinity - is found out while the tile is multiplied. Every slice each wave requests 1 KiB of the tile's
// old C (a row of the wide tile, two rows of the narrow one; wave w takes every fourth, or eighth) into one of four slots of LDS
// behind the operand stages; three slices later it reads them back, 16 bytes per lane (its own
// loads, its own counter: no barrier), and tests the exponents. After the loop the waves put their findings together.
// A tile without such a value is then written as an initialised one (the sign of exact zeros is still taken from the
// old c, see write_wave_rows); a tile with one takes the path that reads all of C. Either way the bits are those of
// 0 * c + alpha * acc.
// (Measured on fp8 8192^3, old C in memory: a first version - every wave its own block, lane addresses for any
// layout of C, 64-bit block arithmetic per load - cost 62-70 us of 415 whether it loaded 4 bytes per lane every slice
// or 16 every other one, 25-43 us of that with the rows already in cache: the instructions between two MFMAs, not the
// loads. Hence contiguous rows, whose address is a scalar product and a shift of the lane index.)
// EXACT: OCP fp8 operands multiplied exactly (MmaF8Exact). The bytes travel like int8's; a fragment is widened behind the
// products in front of its first use, for each half of its bytes anew, A's a row of blocks ahead, B's half a step. A wave widens
// MI + NI fragments for MI x NI products - on the 128 x 128 kernels, with 64 x 32 per wave, three for two, which is
// more vector work than the matrix cores take for the products; here twelve for 32 (256 columns) or eight for 16 (128).
// E4M3 2048 x 8192 x 2048: 77 us there, 62 with eight waves of 32 x 32 products here; with a bias, into E4M3, 73 so and now 56.
template <int TA, int TB, bool A_KC, bool B_KC, int BN, bool EDGE, bool STEPS, bool SCAN, bool EXACT, int WAVES>
__global__ void __launch_bounds__((WAVES * 64)) gemm_mfma_ring_kernel(MfmaArgs p) {
  constexpr bool kLarge = TA == SKL_DT_I8 && ring_few_issue_slots(1, A_KC, B_KC, BN);
  using M = typename std::conditional<kLarge, RingMmaI8Large, RingMma<TA, TB, EXACT>>::type;
  using Frag = typename M::Frag;
  using Acc = typename M::Acc;
  using AccElem = decltype(Acc{}.x);
  constexpr int SB = kRingSlice, NSA = ring_stages_a(A_KC, B_KC, BN, SCAN), NSB = ring_stages_b(A_KC, B_KC, BN, SCAN);
  constexpr int ES = Kind<TA>::ES, S = M::kSide, FRB = M::kFrag;
  constexpr int BM = 256, WAVES_N = ring_waves_n(WAVES, BN, EDGE, STEPS, EXACT), WAVES_M = WAVES / WAVES_N;
  constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N, MI = WM / S, NI = WN / S;
  // A step is a slice: the products of the wave's blocks, once, or EXACT with each half of the fragments' bytes.
  constexpr int kProducts = MI * NI, kSlots = (EXACT || kLarge ? 2 : 1) * kProducts;
  using LA = SLoader<ES, A_KC, WAVES, BM, NSA, S, EDGE>;
  using LB = SLoader<ES, B_KC, WAVES, BN, NSB, S, EDGE>;
  using TileA = STile<ES, A_KC, BM, NSA, S>;
  using TileB = STile<ES, B_KC, BN, NSB, S>;
  using RA = FragReader<ES, A_KC, FRB, BM, NSA, S, EXACT>;
  using RB = FragReader<ES, B_KC, FRB, BN, NSB, S, EXACT>;
  constexpr int PA = RA::kPieces, PB = RB::kPieces;
  constexpr int kReadsB = NI * PB, kReads = kReadsB + MI * PA;  // LDS instructions per step
  constexpr int kReadSlots = (EXACT ? kProducts : kSlots) * 3 / 4;  // ... behind the first of its products, the rest is time to land
  // Item r of n that are spread over m slots goes out in slot r * m / n.
  constexpr auto first_in_slot = [](int q, int n, int m) { return q >= m ? n : (q * n + m - 1) / m; };
  // ... and a load, so as not to meet a read, half of the way on to the next one's.
  constexpr auto first_load = [](int q, int n, int m) { return q >= m ? n : q * 2 * n <= m ? 0 : (2 * q * n - m + 2 * m - 1) / (2 * m); };
  // The loads of step s, in this order (U: parity of s):
  //   an operand with K contiguous and four stages: behind the barrier of an odd slice the pair s + 3, s + 4, whose stages it frees;
  //   with six stages: in odd steps the first blocks of the pair s + 5, s + 6, in even steps the rest of the pair s + 4, s + 5 -
  //   half each, or, next to an operand of four stages, all of them in even steps;
  //   an operand read across K: slice s + 4.
  // What counts is that they are evenly spread: a load keeps the compute unit's address path for 16 cycles, four waves request at
  // the same time, and a wave that has to wait for the path does not issue products either (bf16 8192^3 with K contiguous, epilogue
  // left out: 64 loads within 512 / 768 / 1024 cycles of a step of 1024 761 / 738 / 728 us; in two steps another 1.6 per cent less).
  constexpr auto blocks_of = [](int u, bool kc, int ns, int blocks, bool beside_four) {
    if (!kc) return 0;
    if (ns == 4) return u == 1 ? blocks : 0;
    return beside_four ? (u == 0 ? blocks : 0) : blocks / 2;
  };
  constexpr bool kBesideFour = A_KC && B_KC && (NSA == 4) != (NSB == 4);
  constexpr int kPairA[2] = {blocks_of(0, A_KC, NSA, LA::kBlocks, kBesideFour), blocks_of(1, A_KC, NSA, LA::kBlocks, kBesideFour)};
  constexpr int kPairB[2] = {blocks_of(0, B_KC, NSB, LB::kBlocks, kBesideFour), blocks_of(1, B_KC, NSB, LB::kBlocks, kBesideFour)};
  constexpr int kEachA = A_KC ? 0 : LA::kBlocks, kEachB = B_KC ? 0 : LB::kBlocks, kEach = kEachA + kEachB;
  constexpr int kLoadsOfU[2] = {kPairA[0] + kPairB[0] + kEach, kPairA[1] + kPairB[1] + kEach};
  static_assert(!kBesideFour || NSA == 4, "loads of four-stage operands come first");
  constexpr int kScanSlots = 4, kScanSlot = WAVES * 1024;
  static_assert(!SCAN || (std::is_same<AccElem, float>::value && !EDGE && !STEPS), "a plain floating-point product on whole tiles");
  // Loads that may be in flight at the barrier of slice s (of parity U), where slice s + 1 has to have landed: what has been requested
  // behind the last load that brings any of it. SCAN: one more load in front of each step's.
  constexpr auto in_flight = [=](int u) {
    constexpr int sc = SCAN ? 1 : 0, n[2] = {kLoadsOfU[0] + sc, kLoadsOfU[1] + sc};
    constexpr bool four = (A_KC && NSA == 4) || (B_KC && NSB == 4), six = (A_KC && NSA == 6) || (B_KC && NSB == 6);
    constexpr int c4 = (A_KC && NSA == 4 ? LA::kBlocks : 0) + (B_KC && NSB == 4 ? LB::kBlocks : 0);
    int most = 63;
    const auto at_most = [&](int x) { most = x < most ? x : most; };
    if (four) at_most(kLoadsOfU[1] - c4 + n[0] + (u == 0 ? n[1] : 0));  // step s - 2, or s - 3, then what followed
    if (six && u == 1) at_most(kEach + n[1] + n[0]);                    // step s - 3
    if (kEach) at_most(n[u] + n[u ^ 1]);                                // step s - 3, whose last loads these are
    if (SCAN) at_most(kLoadsOfU[u ^ 1] + n[u] + n[u ^ 1]);              // the rows requested in step s - 3 are read in step s
    return most;
  };
  constexpr int kInFlightOfU[2] = {in_flight(0), in_flight(1)};
  static_assert(kInFlightOfU[1] + kLoadsOfU[1] < 64, "vmcnt is a 6-bit counter");

  extern __shared__ __attribute__((aligned(16))) char smem[];
  char *region_a = smem, *region_b = smem + TileA::kRegion;
  const unsigned addr_a = (unsigned)(size_t)LDS_PTR(char, smem), addr_b = addr_a + TileA::kRegion;

  // K may be shared between `splits` workgroups per tile: p.k is then one share (whole slice pairs), split s
  // starts s shares into K and leaves its raw sums in plane s of the workspace.
  unsigned tm, tn;
  const unsigned tiles = p.tiles_m * p.tiles_n, split = blockIdx.x / tiles;
  tile_of_block<false>(blockIdx.x % tiles, p, tm, tn);
  const size_t m0 = (size_t)tm * BM, n0 = (size_t)tn * BN;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // as a scalar: nothing derived from it occupies a vector register across the main loop
  const int wm = (wave / WAVES_N) * WM, wn = (wave % WAVES_N) * WN;

  LA la;
  LB lb;
  la.init(p.a + (size_t)split * p.k * p.a_sk * ES, m0, p.m, p.k, p.a_s1, p.a_s0, p.a_sk);
  lb.init(p.b + (size_t)split * p.k * p.b_sk * ES, n0, p.n, p.k, p.b_s1, p.b_s0, p.b_sk);
  RA ra;
  RB rb;
  ra.init(wm);
  rb.init(wn);

  Acc acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int r = 0; r < (int)(sizeof(Acc) / 4); ++r) acc[i][j][r] = 0;

  // K is a whole number of slice pairs (EDGE: what is missing is zeros). Units beyond the end are requested as the last unit
  // again: in range, and the stage they land in is never read, which keeps the load counts static.
  // (32-bit counters - the host refuses a K of 2^31 slices or more: a 64-bit "less than" of two scalars is a vector
  // compare and two vector registers)
  const unsigned slices = EDGE ? (unsigned)((p.k * ES + 2 * SB - 1) / (2 * SB)) * 2 : (unsigned)(p.k * ES / SB), pairs = slices / 2;

  // SCAN: the tile's old C, 1 KiB per wave and slice (the host has checked that K has the slices for it and
  // that C is row-major with 16-byte aligned rows).
  unsigned long long scan_bad = 0;   // lanes that have seen a NaN or an infinity
  v4i scan_pend = {0, 0, 0, 0};      // the 16 bytes read back during the step before
  char *const scan_region = smem + TileA::kRegion + TileB::kRegion + wave * 1024;
  const unsigned scan_addr = addr_b + TileB::kRegion + wave * 1024;
  // (row of this wave's first load, and the bytes from one load's rows to the next: scalars, 64 x rsc0 fits 32 bits)
  constexpr unsigned kScanRowsPerLoad = BN == 256 ? 1 : 2, kScanLoadsPerWave = BM / (WAVES * kScanRowsPerLoad);
  // C in panels of 64 x 64 contiguous values (rsc0 == 64): 1 KiB is four rows of a panel; the tile's panels row by
  // row, 16 such pieces each, piece WAVES * q + w is wave w's load q.
  const bool scan_panels = p.rsc0 == 64 && p.rsc1 != 64 * 64;
  const char *const scan_rows = scan_panels ? reinterpret_cast<const char *>(p.c) + ((m0 >> 6) * p.rsc1 + (n0 >> 6) * p.csc1) * 4
                                            : reinterpret_cast<const char *>(p.c) + ((m0 + (size_t)wave * kScanRowsPerLoad) * p.rsc0 + n0) * 4;
  // (each layout's own steps, the other's are zero: a choice inside the loop would be a branch, see SLoader::offset)
  const unsigned scan_step = scan_panels ? 0u : (unsigned)p.rsc0 * (WAVES * kScanRowsPerLoad * 4u), scan_piece = scan_panels ? 1024u : 0u;
  const size_t scan_panel_row = scan_panels ? p.rsc1 * 4 : 0, scan_panel_col = scan_panels ? p.csc1 * 4 : 0;
  [[maybe_unused]] auto scan_issue = [&](unsigned s) {  // load s of this wave (the last one again beyond the tile)
    const unsigned q = s < kScanLoadsPerWave ? s : kScanLoadsPerWave - 1;  // uniform
    const unsigned piece = q * WAVES + wave, panel = piece >> 4, pi = panel / (BN / 64), pj = panel % (BN / 64);
    const char *rows = scan_rows + (pi * scan_panel_row + pj * scan_panel_col + (piece & 15u) * scan_piece + (size_t)q * scan_step);
    // The lane's own part of the address is computed anew for every load, from a lane index the compiler cannot
    // follow: held across the loop it would be a register that the loop does not have.
    unsigned l = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(l));
    unsigned mine;
    if constexpr (BN == 256)
      mine = l * 16u;                                                                // 64 lanes x 16 bytes: one row of 256 columns
    else
      mine = (l & 31u) * 16u + ((unsigned)((int)(l << 26) >> 31) & (scan_panels ? 512u : (unsigned)p.rsc0 * 4u));  // lanes 32-63: the row below (panels: the next 512 bytes)
    load_to_lds(scan_addr + s % kScanSlots * kScanSlot, rows, mine);
  };
  [[maybe_unused]] auto scan_read = [&](unsigned slot) {  // this wave's 1024 bytes in `slot`; the value counts from the next lgkmcnt(0) on
    unsigned l = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(l));
    const unsigned addr = scan_addr + slot * kScanSlot + l * 16;
    asm volatile("ds_read_b128 %0, %1" : "=v"(scan_pend) : "v"(addr) : "memory");
  };
  [[maybe_unused]] auto scan_check = [&]() {  // behind an lgkmcnt(0): NaN or infinity, either sign, in any dword
    asm volatile("" : "+v"(scan_pend));
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      unsigned long long x;
      const int word = scan_pend[e];
      asm volatile("v_cmp_class_f32_e64 %0, %1, %2" : "=s"(x) : "v"(word), "s"(0x207));
      scan_bad |= x;
    }
  };

  // What the steps before the first would have requested, in their order, so that the counts of the main loop hold from its start.
  // (Units beyond the end are requested as the last one again; so are they in the main loop.)
  const auto request_a = [&](int unit, int first, int last) __attribute__((always_inline)) {
    const unsigned u = (unsigned)unit < (A_KC ? pairs : slices) ? (unsigned)unit : (A_KC ? pairs : slices) - 1;
#pragma unroll
    for (int i = first; i < last; ++i) la.issue_one(region_a, (A_KC ? 2 : 1) * unit, u, EDGE ? la.left_of(u) : 0, i);
  };
  const auto request_b = [&](int unit, int first, int last) __attribute__((always_inline)) {
    const unsigned u = (unsigned)unit < (B_KC ? pairs : slices) ? (unsigned)unit : (B_KC ? pairs : slices) - 1;
#pragma unroll
    for (int i = first; i < last; ++i) lb.issue_one(region_b, (B_KC ? 2 : 1) * unit, u, EDGE ? lb.left_of(u) : 0, i);
  };
#pragma unroll
  for (int step = -5; step < 0; ++step) {
    const int u = step & 1;
    if (A_KC && NSA == 4 && u == 1 && step + 3 >= 0) request_a((step + 3) / 2, 0, LA::kBlocks);
    if (B_KC && NSB == 4 && u == 1 && step + 3 >= 0) request_b((step + 3) / 2, 0, LB::kBlocks);
    if (A_KC && NSA == 6 && u == 1) request_a((step + 5) / 2, 0, kPairA[1]);
    if (A_KC && NSA == 6 && u == 0) request_a((step + 4) / 2, kPairA[1], LA::kBlocks);
    if (B_KC && NSB == 6 && u == 1) request_b((step + 5) / 2, 0, kPairB[1]);
    if (B_KC && NSB == 6 && u == 0) request_b((step + 4) / 2, kPairB[1], LB::kBlocks);
    if (!A_KC && step + 4 >= 0) request_a(step + 4, 0, LA::kBlocks);
    if (!B_KC && step + 4 >= 0) request_b(step + 4, 0, LB::kBlocks);
  }
  if constexpr (SCAN) {  // the slots start as zeros: the first slices read slots that no load has filled yet
#pragma unroll
    for (int slot = 0; slot < kScanSlots; ++slot)
#pragma unroll
      for (int quarter = 0; quarter < 4; ++quarter)
        *reinterpret_cast<float *>(scan_region + slot * kScanSlot + quarter * 256 + (threadIdx.x & 63) * 4) = 0.0f;
  }
  wait_loads_upto<(SCAN ? 0 : kInFlightOfU[1] + kLoadsOfU[1])>();  // slice 0
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();

  typename RA::Piece pa[2][MI][PA];
  typename RB::Piece pb[2][NI][PB];
  // LDS read R of a step, into the registers of buffer `buf`: B's fragments, then A's in the order of their use.
  const auto read_item = [&](auto rc, auto bufc, unsigned stage_a, unsigned stage_b) __attribute__((always_inline)) {
    constexpr int R = decltype(rc)::value, BUF = decltype(bufc)::value;
    if constexpr (R < kReadsB)
      pb[BUF][R / PB][R % PB] = rb.template read<R / PB, R % PB>(stage_b);
    else
      pa[BUF][(R - kReadsB) / PA][(R - kReadsB) % PA] = ra.template read<(R - kReadsB) / PA, (R - kReadsB) % PA>(stage_a);
  };
  // All reads in flight have landed; from here on the compiler may use buffer `buf`.
  const auto landed = [&](int buf) __attribute__((always_inline)) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int w = 0; w < PA; ++w) asm volatile("" : "+v"(pa[buf][i][w]));
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int w = 0; w < PB; ++w) asm volatile("" : "+v"(pb[buf][j][w]));
  };

  [&]<int... Rs>(std::integer_sequence<int, Rs...>) __attribute__((always_inline)) {
    (read_item(std::integral_constant<int, Rs>{}, std::integral_constant<int, 0>{}, addr_a, addr_b), ...);
  }(std::make_integer_sequence<int, kReads>{});

  // EXACT: the operands as they are multiplied. A's fragments are widened a row of blocks ahead, B's half a step ahead.
  [[maybe_unused]] v8h wide_a[2], wide_b[EXACT ? 2 : 1][NI];
  if constexpr (EXACT) {
    landed(0);
    wide_a[0] = M::widen_a(join_pieces<Frag>(pa[0][0]), 0);
#pragma unroll
    for (int j = 0; j < NI; ++j) wide_b[0][j] = M::widen_b(join_pieces<Frag>(pb[0][j]), 0);
  }

  // Two slices per trip: the parity of the slice decides which loads follow its barrier and which registers hold its fragments.
  [[maybe_unused]] unsigned six = 0;  // s0 % 6
  unsigned s0 = 0;
  do {  // (K is not empty)
    [[maybe_unused]] const unsigned six_next = six == 4 ? 0 : six + 2;
    [&]<int... Us>(std::integer_sequence<int, Us...>) __attribute__((always_inline)) {
      (
          [&](auto uc) __attribute__((always_inline)) {
            constexpr int U = decltype(uc)::value;
            constexpr int kLoads = kLoadsOfU[U];
            const unsigned s = s0 + U;
            unsigned unit_a, unit_b, next_a, next_b;
            [[maybe_unused]] unsigned left_a = 0, left_b = 0;  // of K, from these units on (EDGE)
            int fill_a, fill_b;
            [[maybe_unused]] unsigned lds_a, lds_b;
            [[maybe_unused]] const char *from_a, *from_b;
            // The reads below are of the next slice: its data must have landed for every wave. Own reads first: the stage refilled
            // behind the barrier is the one that everybody has read.
            wait_loads_upto<kInFlightOfU[U]>();
            landed(U);
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            [&]<int... Qs>(std::integer_sequence<int, Qs...>) __attribute__((always_inline)) {
              (
                  [&](auto qc) __attribute__((always_inline)) {
                    constexpr int Q = decltype(qc)::value, X = Q / kProducts, i = Q % kProducts / NI, j = Q % NI;  // X: half of the fragments' bytes (EXACT)
                    const auto fragment_a = [&]() __attribute__((always_inline)) { if constexpr (EXACT) return wide_a[i & 1]; else if constexpr (kLarge) return half_of<X>(join_pieces<Frag>(pa[U][i])); else return join_pieces<Frag>(pa[U][i]); };
                    const auto fragment_b = [&]() __attribute__((always_inline)) { if constexpr (EXACT) return wide_b[X][j]; else if constexpr (kLarge) return half_of<X>(join_pieces<Frag>(pb[U][j])); else return join_pieces<Frag>(pb[U][j]); };
                    // this slot's load, if it has one
                    constexpr int L = first_load(Q, kLoads, kSlots), kLoadsHere = first_load(Q + 1, kLoads, kSlots) - L;
                    constexpr bool kHasLoad = kLoadsHere > 0 && !EDGE && Q > 0;  // with the product (what it needs is worked out behind the first)
                    // load l is block block_of(l) of A's unit or (not of_a(l)) of B's; of six stages, odd steps load the first blocks, even ones the rest
                    constexpr auto of_a = [](int l) { return l < kPairA[U] || (l >= kPairA[U] + kPairB[U] && l - kPairA[U] - kPairB[U] < kEachA); };
                    constexpr auto block_of = [](int l) {
                      constexpr int six_a = A_KC && NSA == 6 && U == 0 ? kPairA[1] : 0, six_b = B_KC && NSB == 6 && U == 0 ? kPairB[1] : 0;
                      if (l < kPairA[U]) return l + six_a;
                      if (l < kPairA[U] + kPairB[U]) return l - kPairA[U] + six_b;
                      const int each = l - kPairA[U] - kPairB[U];
                      return each < kEachA ? each : each - kEachA;
                    };
                    constexpr bool kOfA = of_a(L);
                    constexpr int kBlock = kHasLoad ? block_of(L) : 0;
                    constexpr bool kInA = ring_sum_in_a<MI, NI, Acc>(i, j);
                    if constexpr (!kHasLoad)
                      M::template run<kInA>(fragment_a(), fragment_b(), acc[i][j]);
                    else if constexpr (kOfA)
                      M::template run<kInA, (kBlock * LA::kBlockStep)>(fragment_a(), fragment_b(), acc[i][j], lds_a, from_a, la.off[kBlock]);
                    else
                      M::template run<kInA, (kBlock * LB::kBlockStep)>(fragment_a(), fragment_b(), acc[i][j], lds_b, from_b, lb.off[kBlock]);
                    // The MFMA first, what belongs to its slot in its shadow. Left to itself the compiler moves a slot's address
                    // arithmetic, reads and loads in front of the MFMA - and behind a barrier, which the waves leave together,
                    // instructions in front of the first MFMA are a gap in every SIMD's matrix core at once.
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (Q == 0) {
                      // The stage of the next slice, the unit to load and the stage it goes to, of an operand with `stages` stages.
                      const auto next_stage = [&](int stages) { return stages == 6 ? (U == 0 ? six + 1 : six_next) : (s + 1) % 4; };
                      const auto unit = [&](bool kc, int stages) {
                        const unsigned x = kc ? (stages == 6 ? s0 + 4 + 2 * U : s + 3) / 2 : s + 4, most = (kc ? pairs : slices) - 1;
                        return x < most ? x : most;
                      };
                      const auto fill_stage = [&](bool kc, int stages) { return stages == 6 ? (U == 1 ? six : six == 0 ? 4 : six - 2) : (s + (kc ? 3 : 4)) % 4; };
                      unit_a = unit(A_KC, NSA), unit_b = unit(B_KC, NSB);
                      if constexpr (EDGE) left_a = la.left_of(unit_a), left_b = lb.left_of(unit_b);
                      fill_a = (int)fill_stage(A_KC, NSA), fill_b = (int)fill_stage(B_KC, NSB);
                      next_a = addr_a + next_stage(NSA) * TileA::kStageStep, next_b = addr_b + next_stage(NSB) * TileB::kStageStep;
                      lds_a = addr_a + fill_a * TileA::kStageStep + la.lds, lds_b = addr_b + fill_b * TileB::kStageStep + lb.lds;
                      from_a = la.tile_base + (size_t)unit_a * la.k_step;
                      from_b = lb.tile_base + (size_t)unit_b * lb.k_step;
                    }
                    if constexpr (EXACT) {
                      static_assert(MI % 2 == 0);
                      if constexpr (X == 1 && Q == kProducts) landed(U ^ 1);
                      if constexpr (j == 0) {
                        if constexpr (i + 1 < MI) wide_a[(i + 1) & 1] = M::widen_a(join_pieces<Frag>(pa[U][i + 1]), X);
                        else wide_a[0] = M::widen_a(join_pieces<Frag>(pa[X ? U ^ 1 : U][0]), X ^ 1);
                      }
                      if constexpr (j == NI / 2 && i < NI) wide_b[X ^ 1][i] = M::widen_b(join_pieces<Frag>(pb[X ? U ^ 1 : U][i]), X ^ 1);
                    }
                    if constexpr (SCAN && Q == 0) scan_issue(s);
                    if constexpr (SCAN && Q == 1) scan_check();  // what the last read of the step before has brought, behind this step's wait
                    // this slot's share of the next step's reads
                    [&]<int... Rs>(std::integer_sequence<int, Rs...>) __attribute__((always_inline)) {
                      (read_item(std::integral_constant<int, first_in_slot(Q, kReads, kReadSlots) + Rs>{}, std::integral_constant<int, U ^ 1>{}, next_a, next_b), ...);
                    }(std::make_integer_sequence<int, first_in_slot(Q + 1, kReads, kReadSlots) - first_in_slot(Q, kReads, kReadSlots)>{});
                    if constexpr (SCAN && Q == kReadSlots) scan_read((s + 1) % kScanSlots);  // the rows of three slices before (the first slices find zeros)
#pragma unroll
                    for (int l = L + (kHasLoad ? 1 : 0); l < L + kLoadsHere; ++l) {
                      if (of_a(l))
                        la.issue_one(region_a, fill_a, unit_a, left_a, block_of(l));
                      else
                        lb.issue_one(region_b, fill_b, unit_b, left_b, block_of(l));
                    }
                    __builtin_amdgcn_sched_barrier(0);
                  }(std::integral_constant<int, Qs>{}),
                  ...);
            }(std::make_integer_sequence<int, kSlots>{});
          }(std::integral_constant<int, Us>{}),
          ...);
    }(std::make_integer_sequence<int, 2>{});
    // The sums' registers are not to be touched before the last product has written them, and the compiler, to which these are no matrix
    // instructions, may copy one as soon as the loop is left: the product's passes (16 x 16: 4, fp8 32 x 32: 16) and four states.
    asm volatile("s_nop %0" ::"n"(S == 32 ? 15 : 7));
    if constexpr (S == 32) asm volatile("s_nop 3");
    six = six_next;
    s0 += 2;
  } while (s0 < slices);
  __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0), as the compiler understands it: it takes the loads to LDS above for pending with every read of LDS below
  landed(0);  // the last step's reads, of a slice that does not exist: their registers are theirs up to here
  asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");  // the last products' results (the compiler does not see that these are matrix instructions)
  [&]<int... Bs>(std::integer_sequence<int, Bs...>) __attribute__((always_inline)) {
    ((acc[Bs / NI][Bs % NI] = fetched<ring_sum_in_a<MI, NI, Acc>(Bs / NI, Bs % NI)>(acc[Bs / NI][Bs % NI])), ...);
  }(std::make_integer_sequence<int, MI * NI>{});
  if constexpr (SCAN) {
    // The last rows requested have not been read back: all slots once more (a row tested twice changes nothing).
    scan_check();
#pragma unroll
    for (int slot = 0; slot < kScanSlots; ++slot) {
      scan_read(slot);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      scan_check();
    }
  }

  if (p.splits > 1) {  // a share of K: the raw sums go to this split's M x N plane
    write_wave_plane<MI, NI, EDGE>(p, acc, m0 + wm, n0 + wn, split);
    return;
  }
  constexpr int kStageBytes = S * wave_rows_pitch<WN>() * 4;
  constexpr int kPassesAtOnce = WAVES == 8 && BN == 256 && STEPS && (EXACT || EDGE) ? 2 : WAVES == 8 || STEPS ? 4 : 8;  // (more are spilled registers)
  static_assert(WAVES * kStageBytes <= TileA::kRegion + TileB::kRegion, "the waves' rows take the place of the operand stages");
  if constexpr (SCAN) {
    // What the waves have found, put together: each wave's word where its first slot began (its own reads of
    // the slots are over), a barrier, and everybody reads all of them.
    unsigned *const found = reinterpret_cast<unsigned *>(smem + TileA::kRegion + TileB::kRegion);
    found[wave * 256] = scan_bad != 0;
    __syncthreads();
    unsigned any = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) any |= found[w * 256];
    MfmaArgs q = p;
    if (any == 0) q.beta.fz.skip_c_read = 1;  // 0 * c is a zero everywhere in this tile
    write_wave_rows<MI, NI, ES, kPassesAtOnce, EDGE, STEPS>(q, acc, m0 + wm, n0 + wn, smem + wave * kStageBytes);
  } else {
    __syncthreads();  // every wave's reads of the stages and loads into them are over
    write_wave_rows<MI, NI, ES, kPassesAtOnce, EDGE, STEPS>(p, acc, m0 + wm, n0 + wn, smem + wave * kStageBytes);
  }
}

// C = beta*C + alpha * (sum of the splits' planes, in split order), then the fused steps: the second
// half of a GEMM whose K range was shared out between workgroups. A thread takes V neighbouring columns of a row; what the
// pass costs is its launch and one trip to memory, so everything it needs is requested at once and the row is found with one
// 32-bit division (one element per thread and 64-bit divisions: 4.7 us for 3 planes of 16 x 11008, now 3.0).
template <typename T, int V>
__global__ void __launch_bounds__(256) gemm_split_reduce_kernel(MfmaArgs p) {
  typedef T Run __attribute__((ext_vector_type(4)));
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x, per_row = p.n / V;
  if (idx >= p.m * per_row) return;
  const size_t row = p.m * per_row >> 32 ? idx / per_row : (size_t)((unsigned)idx / (unsigned)per_row), col = (idx - row * per_row) * V;
  const size_t mn = p.m * p.n;
  const T *plane = reinterpret_cast<const T *>(p.partial) + row * p.n + col;
  const auto load = [](const T *at, T (&v)[V]) __attribute__((always_inline)) {
    if constexpr (V == 4) {
      const Run r = *reinterpret_cast<const Run *>(at);
#pragma unroll
      for (int e = 0; e < V; ++e) v[e] = r[e];
    } else {
      v[0] = *at;
    }
  };
  // V columns of C: they lie in one block of C if its columns come in multiples of V, else each is found by itself.
  T *const c_row = reinterpret_cast<T *>(p.c) + (row >> p.crs) * p.rsc1 + (row & ((size_t(1) << p.crs) - 1)) * p.rsc0;
  T *c[V];
  T bias[V], old[V];
  const bool init = skl_beta_is_zero<T>(p.beta);
#pragma unroll
  for (int e = 0; e < V; ++e) {
    c[e] = c_row + ((col + e) >> p.ccs) * p.csc1 + ((col + e) & ((size_t(1) << p.ccs) - 1)) * p.csc0;
    bias[e] = p.bias ? reinterpret_cast<const T *>(p.bias)[col + e] : T(0);
    old[e] = init ? T(0) : *c[e];
  }
  // Eight planes are requested before the first is used (one memory round trip per eight, not per plane); they are added in
  // order, the first nine to each other, then each eight by themselves: shorter chains of roundings than one over all planes.
  T sum[V];
  load(plane, sum);
  for (unsigned q0 = 1; q0 < p.splits; q0 += 8) {
    T v[8][V];
#pragma unroll
    for (unsigned u = 0; u < 8; ++u)
      if (q0 + u < p.splits) load(plane + (size_t)(q0 + u) * mn, v[u]);
    const auto add = [](T (&to)[V], const T (&by)[V]) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 0; e < V; ++e) {
        if constexpr (std::is_same<T, int>::value) to[e] = (int)((unsigned)to[e] + (unsigned)by[e]);
        else to[e] = __fadd_rn(to[e], by[e]);
      }
    };
    if (q0 == 1) add(sum, v[0]);
#pragma unroll
    for (unsigned u = 1; u < 8; ++u) {
      if (q0 + u >= p.splits) continue;
      if (q0 == 1) add(sum, v[u]);
      else add(v[0], v[u]);
    }
    if (q0 != 1) add(sum, v[0]);
  }
  T best = skl_lowest<T>();
  Run out;
#pragma unroll
  for (int e = 0; e < V; ++e) {
    T v = init ? skl_initialise(sum[e], c[e], p.alpha, p.beta) : skl_combine(sum[e], old[e], p.alpha, p.beta);
    if (p.bias) v = skl_add_bias(v, bias[e]);
    v = skl_activate(v, p.rq.act);
    out[e] = v;
    if (v > best) best = v;
  }
  if (!p.rq.q_only) {
    if (V == 4 && p.csc0 == 1 && p.ccs >= 2 && ((uintptr_t)c[0] & 15) == 0) {
      *reinterpret_cast<Run *>(c[0]) = out;
    } else {
#pragma unroll
      for (int e = 0; e < V; ++e) *c[e] = out[e];
    }
  }
#pragma unroll
  for (int e = 0; e < V; ++e) skl_emit_requantised(p.rq, (T)out[e], row, col + e);
  if (p.max && best > skl_lowest<T>()) skl_atomic_max(reinterpret_cast<T *>(p.max), best);
}

// The tiles of a launch. t / d is the high word of t * (2^32 / d + 1) as long as t * d < 2^32 (the remainder of 2^32 / d, at
// most d, times t stays below 2^32).
inline void set_tiles(MfmaArgs &p, unsigned tiles_m, unsigned tiles_n) {
  p.tiles_m = tiles_m, p.tiles_n = tiles_n;
  p.by_group = p.by_rest = 0;
  const size_t total = (size_t)tiles_m * tiles_n, per_group = (size_t)8 * tiles_n, rest = tiles_m % 8 ? tiles_m % 8 : 8;
  if (total < (size_t(1) << 31) && (total + 8) * per_group < (size_t(1) << 32)) {
    p.by_group = (unsigned)((size_t(1) << 32) / per_group + 1);
    p.by_rest = rest == 1 ? 0 : (unsigned)((size_t(1) << 32) / rest + 1);
  }
}

template <typename T>
int launch_split_reduce(const MfmaArgs &p, const char *who) {
  const int v = p.n % 4 == 0 && ((uintptr_t)p.partial & 15) == 0 ? 4 : 1;
  const size_t blocks = (p.m * (p.n / v) + 255) / 256;
  if (blocks > 0x7FFFFFFFu) {
    skl_hip_record_error(-2, "gemm_mfma: grid too large");
    return -2;
  }
  if (v == 4)
    gemm_split_reduce_kernel<T, 4><<<(unsigned)blocks, 256, 0, skl_current_stream()>>>(p);
  else
    gemm_split_reduce_kernel<T, 1><<<(unsigned)blocks, 256, 0, skl_current_stream()>>>(p);
  return skl_check_launch(who);
}

struct SequenceGuard {
  const bool held;
  explicit SequenceGuard(bool hold) : held(hold) { if (held) skl_hip_sequence_begin(); }
  ~SequenceGuard() { if (held) skl_hip_sequence_end(); }
};

constexpr size_t kRingMinSlicesPerSplit = 64;  // below 8 KiB of K per row the pass over the planes costs what the split saves

// The streaming kernels also exist with the activation and requantisation steps (STEPS).
template <int TA, int TB>
constexpr bool kRingCarriesExtraSteps = TA == TB;   // every kind but the mixed fp8 pairings, which have no fused entry point

// An int32 C in blocks of 4 to 16 columns (the 4 x 4 blocks of src/gemm/packed-gemm.md:270-298) that the streaming kernel writes 16
// bytes per lane like a row-major one: contiguous rows, a multiple of four per block, on 16-byte boundaries, no fused steps.
inline bool c_in_row_quads(const MfmaArgs &p) {
  return !p.bias && !p.max && !p.rq.act && !p.rq.q && p.csc0 == 1 && p.ccs >= 2 && p.ccs <= 4 && p.crs >= 2 &&
         (((uintptr_t)p.c | (p.rsc0 * 4) | (p.rsc1 * 4) | (p.csc1 * 4)) & 15) == 0;
}

// The waves of plain products on whole tiles, int8, 16 bits or exact fp8 (see ring_waves): 256 x 256 tiles of exact fp8 take four only for C
// that is read in one round (E4M3 4096^2 x 512 34 / 36 us, x 2048 63 / 67), those of the others eight only for C that is read over
// two rounds, or more with a short K (us, four / eight: 4096 x 8192 x 512 int8 73 / 62, bf16 84 / 74, x 2048 104 / 97, 148 / 144; 8192^2 x 1024 int8
// 162 / 156, but x 2048 198 / 204; one round, 4096^2 x 512, 29 / 33); 256 x 128 tiles below the K from which the main loop is what counts - except
// int8 read across K on both sides, whose 32 x 32 products are four waves' (2048 x 4096^2 36.2 / 37.9 us).
template <typename AccElem, bool A_KC, bool B_KC, int BN, bool EXACT>
int ring_waves_by_size(const MfmaArgs &p) {
  constexpr bool kInt = std::is_same<AccElem, int>::value;
  const bool reads_c = kInt ? p.beta.i != 0 : !(p.beta.fz.skip_c_read && p.beta.f == 0.0f);
  if (BN == 256) {
    const size_t tiles = (p.m / 256) * (p.n / 256);
    if (EXACT) return reads_c && tiles <= 256 ? 4 : 8;
    return reads_c && tiles > 256 && (tiles <= 512 || p.k * (kInt ? 1 : 2) < 2048) ? 8 : 4;
  }
  if (kInt) return !A_KC && !B_KC ? 4 : p.k < (reads_c ? 4096 : 2048) ? 8 : 4;
  return p.k * 2 < 8192 ? 8 : 4;
}

template <int TA, int TB, bool A_KC, bool B_KC, int BN, bool EDGE = false, bool STEPS = false, bool SCAN = false, bool EXACT = false, int WAVES = 0>
int launch_ring(const MfmaArgs &args) {
  if constexpr (!STEPS && !SCAN && kRingCarriesExtraSteps<TA, TB>) {
    if (args.rq.act || args.rq.q) return launch_ring<TA, TB, A_KC, B_KC, BN, EDGE, true, false, EXACT>(args);
  }
  constexpr int ES = Kind<TA>::ES;
  using AccElem = decltype(typename Kind<TA>::Acc{}.x);
  if constexpr (std::is_same<AccElem, float>::value && !EDGE && !STEPS && !SCAN && !EXACT && WAVES == 0) {
    // beta == 0 evaluated as the reference's loops do (0 * c: a NaN or an infinity in C stays a NaN): the old C is
    // looked through while the tile is multiplied, a KiB of it per wave and slice - needs 64 slices on the wide tile, 32
    // on the narrow one, a tile to itself (no shared K) and a row-major C.
    const size_t scan_slices = args.k * ES / kRingSlice, scan_tiles = (args.m / 256) * (args.n / BN);
    const bool shared_k = scan_tiles <= 128 && scan_slices % 4 == 0 && scan_slices / 2 >= kRingMinSlicesPerSplit;
    // C row-major: rows and columns at one stride each across the blocks, rows of 16-byte aligned starts ...
    const bool row_major = args.csc0 == 1 && args.csc1 == (size_t(1) << args.ccs) && args.rsc1 == (args.rsc0 << args.crs) &&
                           (((uintptr_t)args.c | (args.rsc0 * 4)) & 15) == 0 && args.rsc0 < (size_t(1) << 26) &&
                           !(args.rsc0 == 64 && args.rsc1 != 64 * 64);
    // ... or in panels of 64 x 64 contiguous values on 16-byte boundaries
    const bool panels = args.csc0 == 1 && args.rsc0 == 64 && args.crs == 6 && args.ccs == 6 && args.rsc1 != 64 * 64 &&
                        (((uintptr_t)args.c | (args.rsc1 * 4) | (args.csc1 * 4)) & 15) == 0;
    if (args.beta.f == 0.0f && args.beta.fz.skip_c_read == 0 && !shared_k && (row_major || panels) && scan_slices >= (BN == 256 ? 64 : 32))
      return launch_ring<TA, TB, A_KC, B_KC, BN, EDGE, false, true>(args);
  }
  if constexpr (WAVES == 0) {
    constexpr int waves = ring_waves<TA, A_KC, B_KC, BN, EDGE, STEPS, SCAN, EXACT>();
    if constexpr (waves != 0) return launch_ring<TA, TB, A_KC, B_KC, BN, EDGE, STEPS, SCAN, EXACT, waves>(args);
    else if (ring_waves_by_size<AccElem, A_KC, B_KC, BN, EXACT>(args) == 8) return launch_ring<TA, TB, A_KC, B_KC, BN, EDGE, STEPS, SCAN, EXACT, 8>(args);
    else return launch_ring<TA, TB, A_KC, B_KC, BN, EDGE, STEPS, SCAN, EXACT, 4>(args);
  } else {
  constexpr int lds = (ring_stages_a(A_KC, B_KC, BN, SCAN) * 256 + ring_stages_b(A_KC, B_KC, BN, SCAN) * BN) * kRingSlice + (SCAN ? 4 * WAVES * 1024 : 0);
  static_assert(lds <= 160 * 1024);
  auto kernel = gemm_mfma_ring_kernel<TA, TB, A_KC, B_KC, BN, EDGE, STEPS, SCAN, EXACT, WAVES>;
  static std::atomic<bool> configured{false};  // per instantiation; racing threads set the same value
  if (!configured.load(std::memory_order_acquire)) {
    int rc = skl_check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, lds),
                           "gemm_mfma_ring: LDS size");
    if (rc != 0) return rc;
    configured.store(true, std::memory_order_release);
  }
  MfmaArgs p = args;
  p.tiles_m = (unsigned)((p.m + (EDGE ? 255 : 0)) / 256);
  p.tiles_n = (unsigned)((p.n + (EDGE ? BN - 1 : 0)) / BN);
  const size_t tiles = (size_t)p.tiles_m * p.tiles_n;
  // Tiles for at most half of the 256 compute units: K is shared between two workgroups per tile (each at least
  // kRingMinSlicesPerSplit slices long) and a second pass adds the two planes and applies alpha / beta.
  const size_t slices = p.k * ES / kRingSlice;
  if (slices >= (size_t(1) << 31)) {
    skl_hip_record_error(-2, "gemm_mfma: K too long");
    return -2;
  }
  p.splits = (tiles <= 128 && p.k * ES % (4 * kRingSlice) == 0 && slices / 2 >= kRingMinSlicesPerSplit) ? 2 : 1;
  SequenceGuard sequence(p.splits > 1);
  if (p.splits > 1) {
    p.partial = (char *)skl_workspace((size_t)p.splits * p.m * p.n * 4);
    if (!p.partial) return -4;
    p.k /= p.splits;  // one share; whole slice pairs
  }
  const size_t grid = tiles * p.splits;
  if (grid > 0x7FFFFFFFu) {
    skl_hip_record_error(-2, "gemm_mfma: grid too large");
    return -2;
  }
  kernel<<<(unsigned)grid, WAVES * 64, lds, skl_current_stream()>>>(p);
  int rc = skl_check_launch("gemm_mfma_ring");
  if (rc != 0 || p.splits == 1) return rc;
  return launch_split_reduce<AccElem>(p, "gemm_split_reduce");
  }
}

constexpr size_t kMinBytesPerSplit = 512, kSplitFromBytes = 4096, kSplitEarlyTiles = 96, kSplitPlaneLimit = size_t(64) << 20;
inline size_t bytes_in_lines(size_t k_bytes) { return (k_bytes + 127) / 128 * 128; }

// A few rows of A, or columns of B, off the 16-byte rule, of a floating-point kind. Copied into aligned rows contiguous in K they
// would be the streaming kernels' - fp8 also a decode batch, with K up to 4096 or against a wide B -, whose sums are many and short
// and whose fp8 products are exact for any K. Read in place they keep both, on the 64 x 64 tiles: exact products, and sums
// compensated up to four rows (or few columns), beyond that in blocks (us and error against 64 bits, copies / one chain of the fp8
// instructions or of 16-bit products in place / this: E4M3 2 x 1755 x 3408 27.9, 7.4, 8.3 and 2.7e-8, 1.3e-5, 3.0e-8; E5M2 89 x 7045 x 3440
// 100, 19.9, 25.3 and 4.7e-8, 9.0e-6, 4.5e-8; bf16 4 x 6614 x 1400 30.6, 10.7, 13.0 and 5.0e-8, 1.3e-7, 4.2e-8).
template <int ES>
bool few_off_rule(const MfmaArgs &p) {
  if (!p.a_loose && !p.b_loose) return false;
  if (p.n <= 8 && p.n < p.m) return true;
  if (ES == 2) return p.m <= 4 || (p.m <= 16 && p.b_sk != 1);
  return p.m <= 4 || (p.m <= 96 && p.n * p.k >= (size_t(1) << 20) && (p.k <= 4096 || p.n >= 8192));
}
// Decode batches of the 16-bit kinds with a short K, from 1 MiB of B on: what the streaming kernel for operands with K contiguous
// leaves to the tiles. Their sums are as short chains there: half slices up to 2816 bytes of K, where those become more than two
// slices to a block are, then blocks.
constexpr size_t kHalfSlicesBelow = 2816;
inline bool short_decode_batch(const MfmaArgs &p, size_t k_bytes) {
  return p.a_sk == 1 && p.b_sk == 1 && p.m > 4 && p.m <= 96 && k_bytes * p.n >= (size_t(1) << 20) && bytes_in_lines(k_bytes) < kSplitFromBytes;
}

// How many ways K is shared out when a problem has too few tiles for the chip: each share at least kMinBytesPerSplit of K per
// row, planes within 64 MiB. (512 bytes: the reference's benchmark shapes of one 128 x 128 tile - 8192 k of int8, 4096 k of
// bf16 - 10.2 -> 8.9 us and 10.0 -> 9.0 us against twice that; half of it measures the same.) The pass over the planes costs
// 3.5 us, so K is shared from 4 KiB on, and where few workgroups leave a slice's chain of latencies uncovered from 2 KiB, or
// 1 KiB where fp8 is widened for exact products (us, whole / shared: bf16 32 x 320 x 1920 11.9 / 9.1, E4M3 97 x 1920 x 1280
// 12.3 / 10.3; with more tiles the other way, f16 105 x 3712 x 1216 9.5 / 15.4), as are exact products of a longer K.
// 512 workgroups run at a time: a few more than that would be a round of their own, and of larger problems' fewer are enough,
// with fewer planes. But a sum of rounded products is the more exact the more parts it is made of: `many`, the 16-bit kinds on the
// 128 x 128 tiles, take the next number above 512 workgroups (bf16 300 x 4096 x 4096, six shares instead of four: error against
// 64 bits 1.9e-7 -> 1.6e-7, 28 -> 31 us; 3648 x 320 x 13056 59 -> 73), and two shares also at 256 tiles, from 8 KiB of K on
// (2001 x 2001 x 8192: 5.7e-7 -> 4.0e-7, 85 -> 97 us).
inline unsigned splits_for(size_t tiles, size_t slices, size_t m, size_t n, size_t k_bytes, int slice, bool exact, bool many) {
  const bool early = tiles <= kSplitEarlyTiles || (exact && k_bytes > kF8ExactMaxK);
  const size_t from = !early ? kSplitFromBytes : exact ? kSplitFromBytes / 4 : kSplitFromBytes / 2;
  if (tiles >= 256 || slices * slice < from) return many && tiles == 256 && k_bytes >= 8192 ? 2 : 1;
  size_t want = 512 / tiles;
  if (many) want = (512 + tiles - 1) / tiles;
  else if (!(slice == 256 && tiles < kSplitEarlyTiles) && want > (384 + tiles - 1) / tiles) want = (384 + tiles - 1) / tiles;
  const size_t most = slices * slice / kMinBytesPerSplit;
  if (want > most) want = most;
  while (want > 1 && want * m * n * 4 > kSplitPlaneLimit) --want;
  return (unsigned)(want < 1 ? 1 : want);
}

template <int TA, int TB, bool A_KC, bool B_KC, int BM, int BN, int WAVES_M, int WAVES_N, bool EXACT = false, bool EXTRA = false, int FEW = 0>
int launch_one(const MfmaArgs &args) {
  if constexpr (!EXTRA) {  // calls with an activation or a requantised copy take the kernels that carry those steps
    if (args.rq.act || args.rq.q) return launch_one<TA, TB, A_KC, B_KC, BM, BN, WAVES_M, WAVES_N, EXACT, true>(args);
  }
  if constexpr (!FEW && BM == 64 && (EXACT || Kind<TA>::ES == 2)) {
    if (few_off_rule<Kind<TA>::ES>(args) && (args.m <= 4 || args.n <= 8))
      return launch_one<TA, TB, A_KC, B_KC, BM, BN, WAVES_M, WAVES_N, EXACT, EXTRA, kFewest>(args);
    if constexpr (Kind<TA>::ES == 2) {
      if (few_off_rule<2>(args) || (args.k * 2 < kHalfSlicesBelow && short_decode_batch(args, args.k * 2)))
        return launch_one<TA, TB, A_KC, B_KC, BM, BN, WAVES_M, WAVES_N, EXACT, EXTRA, kFewRows>(args);
    }
  }
  using AccElem = decltype(typename Kind<TA>::Acc{}.x);
  constexpr int ES = Kind<TA>::ES;
  constexpr int NT = WAVES_M * WAVES_N * 64;
  constexpr int lds = 2 * (Tile<ES, BM, A_KC, NT>::kBytes + Tile<ES, BN, B_KC, NT>::kBytes);
  auto kernel = gemm_mfma_kernel<TA, TB, A_KC, B_KC, BM, BN, WAVES_M, WAVES_N, EXACT, EXTRA, FEW>;
  static std::atomic<bool> configured{false};  // per instantiation; racing threads set the same value
  if (!configured.load(std::memory_order_acquire)) {
    int rc = skl_check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, lds),
                           "gemm_mfma: LDS size");
    if (rc != 0) return rc;
    configured.store(true, std::memory_order_release);
  }
  MfmaArgs p = args;
  set_tiles(p, skl_div_up(p.m, BM), skl_div_up(p.n, BN));
  const size_t tiles = (size_t)p.tiles_m * p.tiles_n;
  constexpr int kSlice = slice_bytes(BM);
  const size_t slices = (p.k * ES + kSlice - 1) / kSlice;
  p.splits = splits_for(tiles, slices, p.m, p.n, p.k * ES, kSlice, EXACT, ES == 2 && BM == 128);
  p.blocked_sums = few_off_rule<ES>(p) || short_decode_batch(p, p.k * ES) || bytes_in_lines(p.k * ES) >= kSplitFromBytes;
  p.slices_per_split = (unsigned)((slices + p.splits - 1) / p.splits);
  p.splits = (unsigned)((slices + p.slices_per_split - 1) / p.slices_per_split);  // no empty share
  SequenceGuard sequence(p.splits > 1);  // the partial sums travel from this kernel to the next through the workspace
  if (p.splits > 1) {
    // A K below kSplitFromBytes is shared for speed alone: without scratch memory one workgroup per tile takes all of it.
    const bool optional = bytes_in_lines(p.k * ES) < kSplitFromBytes;
    p.partial = (char *)skl_workspace((size_t)p.splits * p.m * p.n * 4, optional);
    if (!p.partial && !optional) return -4;
    if (!p.partial) p.splits = 1, p.slices_per_split = (unsigned)slices;
  }
  if (tiles > 0x7FFFFFFFu || p.splits > 0xFFFFu) {
    skl_hip_record_error(-2, "gemm_mfma: grid too large");
    return -2;
  }
  kernel<<<dim3((unsigned)tiles, p.splits), NT, lds, skl_current_stream()>>>(p);
  int rc = skl_check_launch("gemm_mfma");
  if (rc != 0 || p.splits == 1) return rc;
  return launch_split_reduce<AccElem>(p, "gemm_split_reduce");
}

// What the lines below depend on besides the problem: C's type, whether fp8 is multiplied exactly, which operands have K contiguous,
// whether the fp8 instructions multiply (FP8), whether the kind has kernels with steps.
struct RingKind {
  bool is_int, exact, fp8, a_kc, b_kc, carries_steps;
  size_t es;
};
inline bool reads_old_c(const MfmaArgs &p, bool is_int) { return is_int ? p.beta.i != 0 : !(p.beta.fz.skip_c_read && p.beta.f == 0.0f); }

// Whether the streaming kernel beats the bounds-checked ones on whole tiles: those have several workgroups on a compute unit, whose
// starts and ends overlap with others' products, it has one. What decides is how full its last round is, how much K there is to gain
// on, and whether C is read, which it requests earlier than the others do; an activation of some twenty or forty instructions (SiLU,
// GELU) is covered by less there. Its time over theirs, geometric means over 720 random problems, by K in bytes; more than one round, by
// `filled` (50-60 / 60-70 / 70-80 / 80-90 / 90-100 per cent); "-": none drawn:
//   16 bits, plain        from  512  1.17  -   1.01 1.07 1.07   from 1024  1.16 1.11 0.89 0.99 0.94   from 2048   -   1.00 0.84 0.85 0.91   from 4096  -   0.93 -  0.83 0.80
//     C read              from  512  1.04 1.13 1.02  -   0.95   from 1024   -   0.95  -   0.95 0.93   from 2048   -    -   0.88 0.87 0.79
//     ReLU                from  512   -   0.94  -   0.94 0.82   from 1024   -    -   0.81 0.89 0.89   from 2048  0.93  -   0.90  -   0.86
//     a copy              0.67 to 0.90 at any K
//     SiLU or GELU        from  512  1.03 1.04 0.96 0.94 0.95   from 1024  1.13 1.05 1.00 1.03 0.90   from 2048   -   0.89 0.91 0.92 0.83   from 4096  0.97 - 0.89 0.74 -
//   fp8, plain            from 2305  0.99  -   1.07 0.96  -     from 4096  0.92  -   0.86 0.78 0.85
//     C read, ReLU, a copy  from 2305  0.89 0.96 0.92  -  0.84  from 4096  0.96 0.89 0.87 0.83 0.78
//     SiLU or GELU        from 2305   -   1.12  -   0.95 0.85   from 4096  1.13 0.93 1.07 0.99  -     from 8192  0.90 0.87 0.83 0.74 -
//   short fp8, plain      from  512  1.27 1.28 1.11 0.99 0.99   from 1024  1.18  -   1.05 0.93 1.01
//     C read              from  512  1.07 1.02 0.92 1.00 0.99   from 1024  1.09 1.05 0.93 0.92 0.94
//     ReLU                from  512  1.07  -    -   0.99 0.92   from 1024   -   1.08  -   0.92 0.84
//     a copy              from  512  1.07  -    -   0.83 0.78   from 1024  1.00 0.94 0.83 0.84 0.83
//     SiLU or GELU        from  512  1.14  -   1.09 0.99 0.93   from 1024   -   1.06 1.02 0.93 0.98   from 2048   -   1.14  -    -    -
//   int8, plain           from  512  1.12  -   1.13  -   1.07   from 1024  1.17 1.12 0.92 1.13 1.08   from 2048  0.98 0.98 0.83  -   0.76
//     C read              0.67 to 0.84 at any K
//     ReLU                from  512   -    -   1.00  -   1.01   from 1024   -   1.01  -   1.14 0.96   from 2048   -   0.84  -    -    -
//     a copy              from  512   -    -    -   0.94 0.89   from 1024  0.97 0.87 0.90 0.91 0.93   from 2048   -   0.96 0.89 0.85  -
// A single round of 200 to 256 tiles: 16 bits plain 1.07 below 1024, short fp8 1.01, all others 0.65 to 0.97. 129 to 199 tiles: 0.64 to 0.98,
// everything. 96 to 128 tiles, half of the chip: plain 1.09 (16 bits), 1.06 (fp8), 1.33 (short fp8) and 1.06 to 1.10 (int8) below 4096, from there on
// 0.78 to 0.81, C read 0.76 to 0.93, a copy 0.72 to 0.90, short fp8 with SiLU or GELU 1.07. With a K of 8 KiB and more also 65 to 128 tiles with steps,
// which share K, 0.78; exactly 64 are 128 bounds-checked tiles, which share it four ways: 1.12 to 1.24. Several rounds of 256 x 128 tiles (N no
// multiple of 256) below 2 KiB of K: plain 1.08 (16 bits), 1.05 to 1.15 (short fp8), 1.11 (int8), int8 with ReLU 1.09, SiLU or GELU
// 0.99 (80 to 90 per cent 1.02), with a copy there 0.84 to 0.94.
inline bool ring_pays(const MfmaArgs &p, const RingKind &kind, bool wide, size_t tiles, bool long_k, unsigned filled) {
  const bool slow_others = kind.fp8 && !kind.exact && !(kind.a_kc && kind.b_kc);  // transposed fragments of 32 bytes: they take two to four times as long
  constexpr unsigned kNever = 101;
  const size_t k_bytes = p.k * kind.es;
  const bool reads_c = reads_old_c(p, kind.is_int), steps = p.rq.act || p.rq.q, many_steps = p.rq.act >= 2;
  const bool dwords = kind.is_int ? dword_copy<int>(p.rq) : dword_copy<float>(p.rq);
  const bool in_rows = p.csc0 == 1 && (p.ccs >= 6 || p.csc1 == (size_t(1) << p.ccs));  // a C that is not: the others take three to four times as long
  if (tiles < 200) {
    if (long_k) return tiles > 64 || !steps || slow_others;
    if (tiles > 128) return true;
    if (kind.exact) return dwords;
    if (steps) return dwords;
    return reads_c || k_bytes >= 4096 || slow_others || !in_rows;
  }
  if (tiles <= 256) return reads_c || steps || kind.is_int || k_bytes >= 1024;
  if (slow_others || (!in_rows && (!kind.exact || steps) && !p.rq.q_only)) return true;
  if (!wide && k_bytes < 2048 && !reads_c && !p.rq.q && !(steps && !kind.is_int)) return false;
  if (many_steps) {
    if (reads_c) return filled >= (k_bytes >= 4096 ? 0 : k_bytes >= 2048 ? 70 : k_bytes >= 1024 ? 80 : kNever);
    return filled >= (k_bytes >= 8192 ? 0 : k_bytes >= 4096 || (k_bytes >= 2048 && kind.es == 2) ? 60 : wide || k_bytes >= 2048 || p.rq.q ? 80 : 90);
  }
  if (kind.exact) return filled >= (reads_c || p.rq.q ? 70 : 80);
  if (kind.is_int) return reads_c || steps || filled >= (k_bytes >= 2048 ? 0 : k_bytes >= 1024 ? 70 : kNever);
  return steps || filled >= (k_bytes >= 2048 ? 0 : k_bytes >= 1024 ? reads_c ? 60 : 70 : reads_c ? 80 : kNever);
}

// How well `tiles` workgroups, one at a time on each of the 256 compute units, fill the rounds they take, in per cent.
// `tail`: the last round runs as 256 x 128 tiles, half as long.
inline unsigned rounds_filled(size_t tiles, bool tail = false) {
  const size_t half_rounds = tail ? tiles / 256 * 2 + 1 : (tiles + 255) / 256 * 2;
  return (unsigned)(tiles * 200 / (256 * half_rounds));
}

// How the streaming kernel takes a problem that its tiles divide evenly (operands on the 16-byte rule): 256 x 256 tiles when those can
// fill the 256 compute units, 256 x 128 tiles for the sizes below that, from 96 tiles on, or from 64 when K is long enough to be shared
// between two workgroups per tile. No columns: the tiles don't divide it, or the bounds-checked kernels are faster.
struct WholeTiles {
  int cols;
  size_t tail_tiles;  // 256 x 256 tiles of a last round that runs as 256 x 128 ones
};
inline WholeTiles whole_tiles(const MfmaArgs &p, const RingKind &kind) {
  if (p.m % 256 != 0 || p.n % 128 != 0 || (p.k * kind.es) % 128 != 0) return {0, 0};
  if ((p.rq.act || p.rq.q) && !kind.carries_steps) return {0, 0};
  const size_t tiles_m = p.m / 256, slices = p.k * kind.es / kRingSlice;
  const size_t tiles = p.n % 256 == 0 ? tiles_m * (p.n / 256) : 0, tiles128 = tiles_m * (p.n / 128);
  // A last round of 256 x 256 tiles that would fill at most half of the 256 compute units is run as 256 x 128 tiles
  // instead (a second launch on the trailing columns): twice the workgroups at half the length.
  const size_t rest = tiles % 256;
  const bool wide = tiles >= 200, tail_round = rest != 0 && rest <= 128 && rest % tiles_m == 0;
  const bool long_k = slices % 4 == 0 && slices / 2 >= kRingMinSlicesPerSplit;
  if (!wide && tiles128 < 96 && !(tiles128 >= 64 && long_k)) return {0, 0};
  if (!ring_pays(p, kind, wide, wide ? tiles : tiles128, long_k, wide ? rounds_filled(tiles, tail_round) : rounds_filled(tiles128))) return {0, 0};
  return {wide ? 256 : 128, wide && tail_round ? rest : 0};
}

template <int TA, int TB, bool A_KC, bool B_KC, bool EXACT>
constexpr RingKind ring_kind() {
  constexpr bool fp8 = TA == SKL_DT_F8E4M3 || TA == SKL_DT_F8E5M2;
  return {TA == SKL_DT_I8, EXACT, fp8, A_KC, B_KC, kRingCarriesExtraSteps<TA, TB>, (size_t)Kind<TA>::ES};
}
constexpr int kNotWholeTiles = 0x7FFFFFFF;
template <int TA, int TB, bool A_KC, bool B_KC, bool EXACT>
int launch_whole_tiles(const MfmaArgs &p) {
  constexpr int ES = Kind<TA>::ES;
  const auto wide = [](const MfmaArgs &q) { return launch_ring<TA, TB, A_KC, B_KC, 256, false, false, false, EXACT>(q); };
  const auto narrow = [](const MfmaArgs &q) { return launch_ring<TA, TB, A_KC, B_KC, 128, false, false, false, EXACT>(q); };
  if (p.a_loose || p.b_loose) return kNotWholeTiles;
  const WholeTiles how = whole_tiles(p, ring_kind<TA, TB, A_KC, B_KC, EXACT>());
  if (how.cols == 0) return kNotWholeTiles;
  if (how.cols == 128) return narrow(p);
  if (how.tail_tiles == 0) return wide(p);
  const size_t tiles_m = p.m / 256, tail_cols = how.tail_tiles / tiles_m * 256, head_cols = p.n - tail_cols, slices = p.k * ES / kRingSlice;
  MfmaArgs head = p, tail = p;
  head.n = head_cols;
  tail.n = tail_cols;
  tail.b = p.b + (head_cols / 64) * p.b_s1 * ES;
  tail.c = p.c + (head_cols >> p.ccs) * p.csc1 * sizeof(float);  // whole blocks; C elements are 4 bytes for every kind
  if (p.bias) tail.bias = p.bias + head_cols * sizeof(float);
  if (p.rq.q) tail.rq.q = p.rq.q + head_cols * p.rq.csq;
  if (p.rq.q && p.rq.q_per_column) tail.rq.q_scale = p.rq.q_scale + head_cols;
  // The tail may be tiles few enough to share K (launch_ring): what it needs for that is there before the head has written
  // its columns of C, which no other kernel could then start from.
  const bool long_k = slices % 4 == 0 && slices / 2 >= kRingMinSlicesPerSplit;
  if (tiles_m * (tail_cols / 128) <= 128 && long_k && !skl_workspace((size_t)2 * p.m * tail_cols * 4)) return -4;
  const int rc = wide(head);
  return rc != 0 ? rc : narrow(tail);
}

// The streaming kernel on problems that are not whole tiles (EDGE): the tile's columns, or 0 where the bounds-checked kernels
// are as good. Those have 512 tiles of 128 x 128 on the chip at a time and waste little of a last round, so what counts is how much
// of the larger tiles' rounds the 128 x 128 ones that exist would fill (per cent), then K, and as in ring_pays whether C is read
// and what is behind the product. Streaming over bounds-checked, geometric means over 4829 random problems, 256 columns from the line on
// to ten per cent beyond it: int8 reading C 0.77 to 0.83, else 0.79 to 0.93; other kinds 0.90 to 0.98, from 8 KiB of K 0.81, with SiLU or GELU
// 0.94 and 0.90; below the line 1.00 to 1.35. 128 columns 0.82 to 0.95. The problems that the rule moves take 0.73 (int8 reading C) to
// 0.95 (16 bits reading C, 128 columns) of the time.
// Floating point only beyond 256 tiles of 128 x 128: fewer share K, and sums of several parts are the more exact ones.
inline int ragged_tile_cols(const MfmaArgs &p, const RingKind &kind) {
  constexpr size_t limit = 0xB0000000u;
  const size_t es = kind.es;
  if (p.a_loose || p.b_loose || ((p.rq.act || p.rq.q) && !kind.carries_steps)) return 0;
  if (p.m % 256 == 0 && p.n % 128 == 0 && p.k * es % 128 == 0) return 0;  // whole tiles: launch_whole_tiles has decided
  // 16 bytes along K that K ends in would need zeros behind it; the offsets inside a tile stay in the descriptor's range
  if (p.k * es % 16 != 0 && (kind.a_kc || kind.b_kc)) return 0;
  if ((3 * p.a_s1 + (kind.a_kc ? 63 * p.a_s0 : 64 * p.a_sk)) * es >= limit || (3 * p.b_s1 + (kind.b_kc ? 63 * p.b_s0 : 64 * p.b_sk)) * es >= limit) return 0;
  const size_t tiles_m = (p.m + 255) / 256, wide = tiles_m * ((p.n + 255) / 256), narrow = tiles_m * ((p.n + 127) / 128);
  const size_t small = (size_t)skl_div_up(p.m, 128) * skl_div_up(p.n, 128), k_bytes = p.k * es;
  constexpr unsigned kNever = 101;
  const bool reads_c = reads_old_c(p, kind.is_int);
  const unsigned of_wide = (unsigned)(small * 100 / ((wide + 255) / 256 * 1024)), of_narrow = (unsigned)(small * 100 / ((narrow + 255) / 256 * 512));
  const auto by_k = [&](unsigned from_512, unsigned from_1k, unsigned from_2k, unsigned from_4k, unsigned from_8k) {
    return k_bytes >= 8192 ? from_8k : k_bytes >= 4096 ? from_4k : k_bytes >= 2048 ? from_2k : k_bytes >= 1024 ? from_1k : k_bytes >= 512 ? from_512 : kNever;
  };
  if (!kind.is_int && small <= 256) return 0;
  unsigned from_wide, from_narrow;
  if (kind.is_int) {
    from_wide = reads_c ? by_k(65, 65, 55, 55, 55) : by_k(kNever, kNever, 80, 55, 55);
    from_narrow = reads_c ? by_k(55, 55, 55, 55, 55) : by_k(kNever, kNever, kNever, 55, 55);
  } else if (p.rq.act >= 2) {
    from_wide = by_k(kNever, kNever, kNever, 70, 52);
    from_narrow = by_k(kNever, kNever, kNever, kNever, 55);
  } else {
    from_wide = by_k(kNever, reads_c ? 80 : kNever, 70, 60, 52);
    from_narrow = by_k(kNever, kNever, reads_c ? 70 : kNever, 70, 52);
  }
  return of_wide >= from_wide ? 256 : of_narrow >= from_narrow ? 128 : 0;
}
template <int TA, int TB, bool A_KC, bool B_KC>
int launch_ragged(const MfmaArgs &p, int tile_cols) {
  return tile_cols == 256 ? launch_ring<TA, TB, A_KC, B_KC, 256, true>(p) : launch_ring<TA, TB, A_KC, B_KC, 128, true>(p);
}

// Whether the 64 x 64 tiles take a problem: where 128 x 128 ones are few - fewer than 128 as long as K is short and they are
// not to be shared, fewer than 256 where C is read or there are steps behind the product, which one workgroup to a compute unit
// leaves uncovered - and for the 16-bit kinds up to 64 rows of A, of which the larger tile would fetch and multiply as many
// again that do not exist. Where C and the steps decide, floating point has a K that neither tile shares (kSplitFromBytes), so that
// the sums, which both then make in the same order, are the same with and without fused steps. Us, 128 x 128 / 64 x 64 tiles: int8
// 64 tiles of 128 x 128, 256 x 4096 x 1344 with GELU 24.8 / 13.2, f16 448 x 1932 x 1024 reading C 20.0 / 11.1, int8 1664 x 1536 x 832
// reading C 21.4 / 13.0; the other way, int8 256 x 11520 x 896 8.9 / 11.2, E5M2 128 x 10240 x 12608 53 / 96.
// (Their slices are up to 256 rows of an operand read across K: offsets inside a tile stay in 32 bits.)
template <int ES, bool INT, bool A_KC, bool B_KC>
bool small_tiles(const MfmaArgs &p) {
  constexpr size_t limit = size_t(1) << 31;
  if ((!A_KC && p.a_sk * ES * 256 >= limit) || (!B_KC && p.b_sk * ES * 256 >= limit)) return false;
  const size_t large = skl_div_up(p.m, 128) * (size_t)skl_div_up(p.n, 128), k_bytes = p.k * ES;
  if ((ES == 2 && p.m <= 64) || large < 64 || (!INT && few_off_rule<ES>(p))) return true;
  const bool reads_c = INT ? p.beta.i != 0 : !(p.beta.fz.skip_c_read && p.beta.f == 0.0f);
  if (!INT && large >= 128 && bytes_in_lines(k_bytes) >= kSplitFromBytes) return false;
  return k_bytes < (large < 128 ? 5120 : large < 256 && (reads_c || p.rq.act || p.rq.q) ? 4096 : 0);
}

template <int TA, int TB, bool A_KC, bool B_KC>
int launch_tile(const MfmaArgs &p) {
  constexpr int ES = Kind<TA>::ES;
  constexpr bool kFp8 = TA == SKL_DT_F8E4M3 || TA == SKL_DT_F8E5M2;
  if constexpr (kFp8) {
    // short K: exact products (see MmaF8Exact), on the streaming kernel when its tiles fill the chip and ring_pays() (us,
    // bounds-checked 128 x 128 / streaming: 2048 x 8192 x 2048 77 / 56, 2048 x 4096 x 2048 42 / 33; on 128 tiles,
    // 512 x 8192 x 2048, 25.4 / 26.2)
    if (p.k <= kF8ExactMaxK || few_off_rule<ES>(p)) {
      const int rc = launch_whole_tiles<TA, TB, A_KC, B_KC, true>(p);  // (not of operands off the 16-byte rule)
      if (rc != kNotWholeTiles) return rc;
      if (small_tiles<ES, TA == SKL_DT_I8, A_KC, B_KC>(p))
        return launch_one<TA, TB, A_KC, B_KC, 64, 64, 2, 2, true>(p);
      return launch_one<TA, TB, A_KC, B_KC, 128, 128, 2, 4, true>(p);
    }
  }
  const int rc = launch_whole_tiles<TA, TB, A_KC, B_KC, false>(p);
  if (rc != kNotWholeTiles) return rc;
  if (const int cols = ragged_tile_cols(p, ring_kind<TA, TB, A_KC, B_KC, false>())) return launch_ragged<TA, TB, A_KC, B_KC>(p, cols);
  if (small_tiles<ES, TA == SKL_DT_I8, A_KC, B_KC>(p))
    return launch_one<TA, TB, A_KC, B_KC, 64, 64, 2, 2>(p);
  return launch_one<TA, TB, A_KC, B_KC, 128, 128, 2, 4>(p);
}

template <int TA, int TB>
int launch_layout(const MfmaArgs &p) {
  const bool a_kc = p.a_sk == 1, b_kc = p.b_sk == 1;
  if (a_kc && b_kc) return launch_tile<TA, TB, true, true>(p);
  if (a_kc) return launch_tile<TA, TB, true, false>(p);
  if (b_kc) return launch_tile<TA, TB, false, true>(p);
  return launch_tile<TA, TB, false, false>(p);
}

inline bool mult16(size_t bytes) { return (bytes & 15) == 0; }

// One operand: exactly one unit stride; the other strides and the base 16-byte aligned.
inline bool operand_ok(const void *base, size_t es, size_t s1, size_t s0, size_t sk, size_t mn, size_t k) {
  if (((uintptr_t)base & 15) != 0) return false;
  // Offsets inside one tile (up to four 64-blocks, 64 rows, 128 k-rows) are kept in 32 bits.
  const size_t limit = size_t(1) << 31;
  if (sk == 1) {  // K-contiguous: rows anywhere on 16-byte boundaries
    if (s1 * es * 4 >= limit || s0 * es * 64 >= limit) return false;
    return (mn <= 1 || mult16(s0 * es)) && (mn <= 64 || mult16(s1 * es));
  }
  if (s0 == 1) {  // MN-contiguous in runs of 64 elements
    if (s1 * es * 4 >= limit || sk * es * 128 >= limit) return false;
    return (k <= 1 || mult16(sk * es)) && (mn <= 64 || mult16(s1 * es));
  }
  return false;
}

// What the bounds-checked kernels read besides: an operand off the 16-byte rule whose rows (K-contiguous), or whose runs along
// M / N, hold at least one chunk that can be loaded in a place further down (Loader).
inline bool operand_loose_ok(size_t es, size_t s1, size_t s0, size_t sk, size_t mn, size_t k) {
  const size_t limit = size_t(1) << 31, chunk = 16 / es;
  if (sk == 1) return s1 * es * 4 < limit && s0 * es * 64 < limit && k >= chunk;
  if (s0 == 1) return s1 * es * 4 < limit && sk * es * 128 < limit && (mn % chunk == 0 || (mn >= chunk && (mn <= 64 || s1 == 64)));
  return false;
}

template <int TA, int TB>
int launch_padded(const MfmaArgs &p, size_t tile_cols) {
  return tile_cols == 256 ? launch_ring<TA, TB, true, true, 256, true>(p) : launch_ring<TA, TB, true, true, 128, true>(p);
}

}  // namespace

// One translation unit per operand kind defines these two (SKL_MFMA_DEFINE_KIND below); the dispatch calls them.
#define SKL_MFMA_DECLARE_KIND(NAME)                 \
  int skl_mfma_launch_##NAME(const MfmaArgs &p);    \
  int skl_mfma_launch_padded_##NAME(const MfmaArgs &p, size_t tile_cols);
#define SKL_MFMA_DEFINE_KIND(NAME, TA, TB)                                                                   \
  int skl_mfma_launch_##NAME(const MfmaArgs &p) { return launch_layout<TA, TB>(p); }                         \
  int skl_mfma_launch_padded_##NAME(const MfmaArgs &p, size_t tile_cols) { return launch_padded<TA, TB>(p, tile_cols); }
