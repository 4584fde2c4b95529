// skl_gemv_kcrows.hip - decode batches against weights stored column by column: 2 to 96 rows of A (K contiguous)
// times a B whose columns are contiguous in K - a linear layer's [out][in] weight -, int8, the OCP fp8 kinds, bf16 and f16.
// The reference's generic kernels take any strides (ref/gemm/gemm_i8rc_i8rc_i32rc.c:9-24, ref/gemm/gemm_f8rc_f8rc_f32rc.c,
// ref/gemm/gemm_bf16rc_bf16rc_f32rc.c); one row, and up to four against a small B, skl_gemv.hip's gemv_kc_kernel streams such a B with dot products.
//
// With K contiguous in both operands 16 bytes of a column, or of a row, ARE a matrix-core operand. How they get there is
// skl_kcstream.hpp's: a workgroup of four or eight waves owns 16 to 64 columns and all of K, every wave streams its own lines
// of them through LDS. Which k meet in which instruction is free as long as A's and B's lanes hold the same ones: lane
// group g takes bytes 16 g to 16 g + 15 of each half line. The sums of the waves meet in LDS in wave order, C is
// written once, with the alpha / beta step and the fused steps of a fused call applied in place.
// int8: v_mfma_i32_16x16x64_i8; bf16, f16: v_mfma_f32_16x16x32. fp8: every E4M3 / E5M2 value is an f16 value, so the bytes are
// widened in registers and multiplied by v_mfma_f32_16x16x32_f16 - exact products, fp32 sums, inside the reference's
// bound for any K (the fp8 instructions align the products of an instruction and drop low bits, which short K would show).
//
// Measured against the kernel that loaded operands straight into registers (int8, fp8: 64 columns and 4096 k per launch) and the
// tile kernels with a pass over planes of sums (bf16, f16), us before / now: 4096 x 11008 bf16, 16 / 64 / 96 rows 28.0 / 16.3,
// 31.3 / 24.2, 41.3 / 30.6 (90 MB of weights: 5.5 TB/s at 16 rows); int8, 8 / 64 rows 13.3 / 9.5, 22.3 / 15.2; 14336 x 8192
// E5M2, 96 rows 137 / 40.
#include <hip/hip_runtime.h>

#include <atomic>
#include <type_traits>

#include "skl_device.hpp"
#include "skl_fp8.hpp"
#include "skl_kcstream.hpp"

namespace {

using skl_kcstream::v4i;
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

constexpr int kMaxRowGroups = 6, kMinRows = 2;  // one row: dot products, level for 16 bits (15.6 us against 16.0) and ahead for int8 (8.1 against 10.1)
enum { kI8 = 0, kE4M3 = 1, kE5M2 = 2, kMixed = 3, kBF16 = 4, kF16 = 5 };  // kMixed: E4M3 A with E5M2 B

struct KcRowsArgs {
  const char *a;  // row i at a + i * a_row (bytes), K contiguous
  size_t a_row;
  const char *b;  // column j at b + j * b_col (bytes), K contiguous
  size_t b_col;
  void *c;        // element (i, j) at i * c_row + j * c_col (elements)
  size_t c_row, c_col;
  size_t m, n;
  unsigned k_bytes;
  skl_scalar alpha, beta;
  const void *bias;  // fused steps behind alpha / beta (bias and maximum of C's type, or null) ...
  void *max;
  skl_requant rq;    // ... activation and 8-bit copy
};

template <int KIND, int RG, int CG>
__global__ void __launch_bounds__((skl_kcstream::Shape<RG, CG, 1>::kWaves * 64)) gemv_kc_rows_kernel(KcRowsArgs p) {
  using Shape = skl_kcstream::Shape<RG, CG, 1>;
  constexpr int kWaves = Shape::kWaves, kCols = 16 * CG, kPitch = Shape::kPitch;
  using Acc = typename std::conditional<KIND == kI8, int, float>::type;
  typedef Acc v4acc __attribute__((ext_vector_type(4)));
  extern __shared__ __attribute__((aligned(1024))) char kc_ring[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int jl = lane & 15, g = lane >> 4;
  const size_t col0 = (size_t)blockIdx.x * kCols;
  skl_kcstream::Requests<RG, 1> ra;
  skl_kcstream::Requests<CG, 1> rb;
  ra.template set<false>(p.a, p.a_row, p.m, p.k_bytes, lane);
  rb.template set<true>(p.b + col0 * p.b_col, p.b_col, p.n - col0, p.k_bytes, lane);
  __attribute__((address_space(3))) char *mine = (__attribute__((address_space(3))) char *)kc_ring + wave * Shape::kUnits * Shape::kUnitBytes;
  const unsigned at0 = (unsigned)(uintptr_t)mine + (unsigned)jl * skl_kcstream::kLine + (unsigned)(g ^ (jl & 7)) * 16u;
  const unsigned units = (p.k_bytes + skl_kcstream::kLine - 1) / skl_kcstream::kLine, steps = (units + kWaves - 1) / kWaves;
  auto request = [&](unsigned step) {  // the step's unit into its place in the ring
    __attribute__((address_space(3))) char *to = mine + (step % Shape::kUnits) * Shape::kUnitBytes;
    rb.template issue<2>(to, step * kWaves + (unsigned)wave);  // non-temporal: B is read once
    ra.template issue<0>(to + 2048 * CG, step * kWaves + (unsigned)wave);
  };
#pragma unroll
  for (unsigned s = 0; s < (unsigned)Shape::kUnits; ++s) request(s);
  // Floating point: the units of a block of products (settle()). Up to 16 rows every unit is one, and what the sum over the waves
  // loses is carried along, so that few rows are as exact as by the dot products of skl_gemv.hip; beyond that every four, or, with half
  // as many waves, every eight in two sums (error against 64 bits, one chain per wave / blocks: bf16 2 x 4096 x 14336 2.5e-7 / 1.1e-7,
  // 16 x 11008 x 4096 1.4e-7 / 7.8e-8, 96 x 11008 x 4096 1.3e-7 / 1.0e-7, E4M3 16 x 11008 x 14336 5.8e-8 / 3.7e-8; 29.3 -> 31.0 us for the 96
  // rows, nothing for 16).
  constexpr int kChains = KIND != kI8 && RG > 1 && kWaves < 8 && RG * CG < 24 ? 2 : 1;  // (6 x 4 groups leave no registers for two)
  constexpr unsigned kBlock = RG == 1 ? 1 : 4 * kChains;
  v4acc acc2[kChains][RG][CG];
  [[maybe_unused]] v4acc sums[KIND == kI8 ? 1 : RG][CG];
#pragma unroll
  for (int rg = 0; rg < RG; ++rg)
#pragma unroll
    for (int cg = 0; cg < CG; ++cg) {
      acc2[0][rg][cg] = acc2[kChains - 1][rg][cg] = v4acc{0, 0, 0, 0};
      if constexpr (KIND != kI8) sums[rg][cg] = acc2[0][rg][cg];
    }
  [[maybe_unused]] const auto settle_all = [&]() __attribute__((always_inline)) {
    if constexpr (KIND != kI8) {
#pragma unroll
      for (int c = 0; c < kChains; ++c) skl_kcstream::settle(sums, acc2[c]);
    }
  };
  for (unsigned step = 0; step < steps; ++step) {
    skl_kcstream::wait_loads<(Shape::kUnits - 1) * Shape::kLoads>();
    const unsigned at = at0 + (step % Shape::kUnits) * Shape::kUnitBytes;
    v4i a[2][RG], b[2][CG];
    skl_kcstream::read_operands<CG, RG>(b[0], a[0], at, at + 2048 * CG);
    skl_kcstream::read_operands<CG, RG>(b[1], a[1], at ^ 64u, (at ^ 64u) + 2048 * CG);
    request(step + Shape::kUnits);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      auto &acc = acc2[h % kChains];
      if constexpr (KIND == kI8 || KIND == kBF16 || KIND == kF16) {
#pragma unroll
        for (int rg = 0; rg < RG; ++rg)
#pragma unroll
          for (int cg = 0; cg < CG; ++cg) {
            if constexpr (KIND == kI8) acc[rg][cg] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[h][rg], b[h][cg], acc[rg][cg], 0, 0, 0);
            else if constexpr (KIND == kBF16)
              acc[rg][cg] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a[h][rg]), __builtin_bit_cast(v8bf, b[h][cg]), acc[rg][cg], 0, 0, 0);
            else
              acc[rg][cg] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a[h][rg]), __builtin_bit_cast(v8h, b[h][cg]), acc[rg][cg], 0, 0, 0);
          }
      } else {
        constexpr bool a_e5m2 = KIND == kE5M2, b_e5m2 = KIND != kE4M3;
        v8h bw[CG][2];
#pragma unroll
        for (int cg = 0; cg < CG; ++cg) {
          bw[cg][0] = skl_fp8::widen8_to_f16<b_e5m2>((unsigned)b[h][cg].x, (unsigned)b[h][cg].y);
          bw[cg][1] = skl_fp8::widen8_to_f16<b_e5m2>((unsigned)b[h][cg].z, (unsigned)b[h][cg].w);
        }
#pragma unroll
        for (int rg = 0; rg < RG; ++rg) {
          const auto a0 = skl_fp8::widen8_to_f16<a_e5m2>((unsigned)a[h][rg].x, (unsigned)a[h][rg].y);
          const auto a1 = skl_fp8::widen8_to_f16<a_e5m2>((unsigned)a[h][rg].z, (unsigned)a[h][rg].w);
#pragma unroll
          for (int cg = 0; cg < CG; ++cg) {
            acc[rg][cg] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, bw[cg][0], acc[rg][cg], 0, 0, 0);
            acc[rg][cg] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, bw[cg][1], acc[rg][cg], 0, 0, 0);
          }
        }
      }
    }
    if constexpr (KIND != kI8) {
      if (step % kBlock == kBlock - 1) settle_all();
    }
  }
  if constexpr (KIND != kI8 && kBlock != 1) settle_all();
  skl_kcstream::wait_loads<0>();  // the requests behind the last unit write zeros into the ring
  __syncthreads();
  // acc2[0][rg][cg][r], or sums[rg][cg][r], is row 16 rg + 4 g + r of C, column 16 cg + jl of the workgroup's.
  Acc(*red)[RG * 16][kPitch] = reinterpret_cast<Acc(*)[RG * 16][kPitch]>(kc_ring);
#pragma unroll
  for (int rg = 0; rg < RG; ++rg)
#pragma unroll
    for (int cg = 0; cg < CG; ++cg)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if constexpr (KIND == kI8) red[wave][16 * rg + 4 * g + r][cg * 16 + jl] = acc2[0][rg][cg][r];
        else red[wave][16 * rg + 4 * g + r][cg * 16 + jl] = sums[rg][cg][r];
      }
  __syncthreads();
  const bool fused = p.bias || p.max || p.rq.act || p.rq.q;  // the same for every thread
  Acc largest = skl_lowest<Acc>();                           // what this thread wrote, for the maximum
  Acc *cbase = reinterpret_cast<Acc *>(p.c);
  const unsigned rows = p.m < (size_t)(16 * RG) ? (unsigned)p.m : (unsigned)(16 * RG);
  for (unsigned at = threadIdx.x; at < rows * kCols; at += kWaves * 64) {
    const unsigned i = at / kCols, tc = at % kCols;
    const size_t j = col0 + tc;
    if (j >= p.n) continue;
    Acc sum = red[0][i][tc];
    [[maybe_unused]] Acc loss = 0;
#pragma unroll
    for (int w = 1; w < kWaves; ++w) {
      if constexpr (KIND == kI8) sum = (int)((unsigned)sum + (unsigned)red[w][i][tc]);
      else if constexpr (RG == 1) sum = skl_add_keeping_loss(sum, red[w][i][tc], loss);
      else sum = __fadd_rn(sum, red[w][i][tc]);
    }
    Acc *c = cbase + (size_t)i * p.c_row + j * p.c_col;
    Acc v = skl_beta_is_zero<Acc>(p.beta) ? skl_initialise(sum, c, p.alpha, p.beta) : skl_combine(sum, *c, p.alpha, p.beta);
    if (fused) {  // the steps of include/skl-gfx950.h's fused calls on the same sums: a fused call gives the plain call's bits plus the steps
      if (p.bias) v = skl_add_bias(v, reinterpret_cast<const Acc *>(p.bias)[j]);
      v = skl_activate(v, p.rq.act);
      skl_emit_requantised(p.rq, v, i, j);
      if (v > largest) largest = v;
    }
    if (!fused || !p.rq.q_only) *c = v;
  }
  if (fused && p.max) {  // one atomic per wave that wrote something
    const Acc best = skl_wave_max(largest);
    if ((threadIdx.x & 63) == 0 && best > skl_lowest<Acc>()) skl_atomic_max(reinterpret_cast<Acc *>(p.max), best);
  }
}

template <int KIND, int RG, int CG>
int launch_groups(const KcRowsArgs &p, unsigned grid, hipStream_t st) {
  using Shape = skl_kcstream::Shape<RG, CG, 1>;
  static std::atomic<bool> configured{false};  // per instantiation; racing threads set the same value
  if (!configured.load(std::memory_order_acquire)) {
    int rc = skl_check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(gemv_kc_rows_kernel<KIND, RG, CG>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, Shape::kRingBytes), "gemv_kc_rows: LDS size");
    if (rc != 0) return rc;
    configured.store(true, std::memory_order_release);
  }
  gemv_kc_rows_kernel<KIND, RG, CG><<<grid, Shape::kWaves * 64, Shape::kRingBytes, st>>>(p);
  return skl_check_launch("gemv_kc_rows");
}

template <int KIND, int CG>
int launch_width(const KcRowsArgs &p, unsigned grid, hipStream_t st) {
  switch ((p.m + 15) / 16) {
    case 1: return launch_groups<KIND, 1, CG>(p, grid, st);
    case 2: return launch_groups<KIND, 2, CG>(p, grid, st);
    case 3: return launch_groups<KIND, 3, CG>(p, grid, st);
    case 4: return launch_groups<KIND, 4, CG>(p, grid, st);
    case 5: return launch_groups<KIND, 5, CG>(p, grid, st);
    default: return launch_groups<KIND, 6, CG>(p, grid, st);
  }
}

template <int KIND>
int launch_kind(const KcRowsArgs &p) {
  hipStream_t st = skl_current_stream();
  const int cg = skl_kcstream::column_groups(p.n);
  const unsigned grid = (unsigned)((p.n + 16 * (size_t)cg - 1) / (16 * (size_t)cg));
  switch (cg) {
    case 1: return launch_width<KIND, 1>(p, grid, st);
    case 2: return launch_width<KIND, 2>(p, grid, st);
    case 3: return launch_width<KIND, 3>(p, grid, st);
    default: return launch_width<KIND, 4>(p, grid, st);
  }
}

int kind_of(const skl_gemm_canon *g) {
  if (g->ta == SKL_DT_I8 && g->tb == SKL_DT_I8) return kI8;
  if (g->ta == SKL_DT_F8E4M3 && g->tb == SKL_DT_F8E4M3) return kE4M3;
  if (g->ta == SKL_DT_F8E5M2 && g->tb == SKL_DT_F8E5M2) return kE5M2;
  if (g->ta == SKL_DT_F8E4M3 && g->tb == SKL_DT_F8E5M2) return kMixed;
  if (g->ta == SKL_DT_BF16 && g->tb == SKL_DT_BF16) return kBF16;
  if (g->ta == SKL_DT_F16 && g->tb == SKL_DT_F16) return kF16;
  return -1;
}

inline bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

// Whether another kernel is the better one: the tile kernels, which share K or have more rows and columns to a workgroup, or up to
// three rows the dot products of skl_gemv.hip. Not for fp8 with K up to 4096, or a B of 8192 columns and more: beyond K = 2304 the
// tile kernels multiply fp8 with instructions that align the products (error 1.3e-5 against 5e-8 here).
// A workgroup streams its columns and all of A at 60 to 70 KB per microsecond, at two thirds of that if the columns start inside
// lines. With fewer workgroups than compute units a long K is better shared out (us here / there: int8 48 x 2048 x 8192 on 128
// workgroups, 512 KiB each, 11.1 / 9.4; int8 96 x 1024 x 8192, 896 KiB, 16.0 / 12.2; f16 64 x 448 x 2688, 420 KiB, 10.3 / 8.8; int8
// 28 x 153 x 11312, 486 KiB and columns inside lines, 13.0 / 9.6; the other way, with a ring of four units, int8 16 x 128 x 14336,
// 448 KiB, 5.9 / 9.1). Medians over some 2000 random problems, by KiB per workgroup, here over there: up to 80 workgroups 0.69 at
// 128, 0.90 at 256, 1.07 at 384, inside lines 0.78, 1.05 and 1.28; 129 to 191 workgroups 0.62, 0.77, 0.88 and 0.72, 0.90, 1.02.
// On a full chip the 16-bit kinds' ring gets short as rows and columns are many: bf16 96 x 8192 x 14336 75 / 49, 48 x 4096 x 14336
// 35 / 28, 64 x 4096 x 8192 22.5 / 20.6; with a short K the sums' way through LDS is what takes the time: bf16 64 x 11008 x 512
// 1.5 times theirs, 48 x 8192 x 256 1.08. More than 16384 columns are more than one round of workgroups, each with its own start and
// end: 32 rows of bf16 at K = 1024 / 2048 / 4096 / 8192 take 1.35 / 1.33 / 1.27 / 1.05 of the tile kernels' time at 32000 columns, 16 rows 1.04,
// 1.06, 1.13 and 0.89; two rows 1.0 to 1.2 of the dot products' up to 24576 columns. From 65 rows on the tile kernels' sums would be
// longer chains than the ones here (they are the faster ones there too: bf16 96 x 50257 x 2048 85 / 43).
bool others_are_faster(int kind, size_t m, size_t n, size_t k, size_t k_bytes, size_t b_pitch) {
  constexpr size_t kib = 1024;
  const size_t cg = (size_t)skl_kcstream::column_groups(n), groups = (n + 16 * cg - 1) / (16 * cg);
  const bool half = kind >= kBF16, fp8 = kind != kI8 && !half, lines = b_pitch % skl_kcstream::kLine == 0;
  size_t bytes = (16 * cg + m) * k_bytes;
  if (m <= 4) {
    if (n <= 16384 || k < (half ? lines ? 2048u : 1024u : 4096u)) return false;
    return lines ? !fp8 && m == 2 && n <= 24576 : m <= (kind == kI8 ? 3u : 2u);
  }
  const bool starved = (groups < 192 && bytes > 512 * kib) || (groups < 224 && bytes > 1280 * kib);
  if (fp8) return k > 4096 && n < 8192 && starved;
  if (starved || (half && m > 64 && n > 8192)) return starved;
  if (!lines) bytes = bytes / 2 * 3;  // what they take the time of
  if (kind == kI8 && k <= 4096) return false;
  if (groups < 224 && (m > 16 || !lines) && bytes >= (groups <= 80 && (half || !lines) ? 384 : groups < 192 ? 512 : 960) * kib) return true;
  if (!half) return n <= 4096 && k > 4096 && bytes > 800 * kib;
  if (cg == 1) return bytes > 960 * kib;
  if (cg == 2) return m > 32 && (bytes > 1416 * kib || (m > 48 && m <= 64 && k < 768));
  if (m > 64) return false;
  if (cg == 3) return m > 32 && k < 1024;
  if (n <= 14336) return m > 16 && k < (m > 48 ? 2048u : 640u);
  if (n <= 16384) return m > 16 && k < (m > 48 ? 12288u : m > 32 ? 2048u : 1024u);
  return k < (m > 16 ? 8192u : 2048u);
}

}  // namespace

// 2 to 96 rows of A and a B of at least 1 MiB, both with K contiguous (16-byte aligned rows and columns a fixed
// distance apart, K a multiple of 16 bytes), C flat or in blocks of 64; fused steps in the last stage. A workgroup's rows and
// columns lie within the 31 bits of a load's offset.
extern "C" int skl_hip_gemv_kc_rows_supported(const skl_gemm_canon *g) {
  const int kind = kind_of(g);
  if (kind < 0) return 0;
  if (g->c_row_shift != 6 || g->c_col_shift != 6) return 0;
  if (g->m < (size_t)kMinRows || g->m > (size_t)(16 * kMaxRowGroups) || g->n == 0 || g->k == 0) return 0;
  const size_t es = kind >= kBF16 ? 2 : 1, most = (size_t(1) << 31) - 4096;
  if (((g->k * es) % 16) != 0 || g->k * es > most || g->k * es * g->n < (size_t(1) << 20)) return 0;
  if (g->a_sk != 1 || g->b_sk != 1 || others_are_faster(kind, g->m, g->n, g->k, g->k * es, g->b_s0 * es)) return 0;
  if (!aligned16(g->a) || ((g->a_s0 * es) % 16) != 0 || (g->m > 64 && g->a_s1 != 64 * g->a_s0)) return 0;
  if (!aligned16(g->b) || ((g->b_s0 * es) % 16) != 0 || (g->n > 64 && g->b_s1 != 64 * g->b_s0)) return 0;
  if (g->a_s0 * es > most / 96 || g->b_s0 * es > most / 64) return 0;
  if ((g->m > 64 && g->rsc1 != 64 * g->rsc0) || (g->n > 64 && g->csc1 != 64 * g->csc0)) return 0;
  return 1;
}

extern "C" int skl_hip_launch_gemv_kc_rows(const skl_gemm_canon *g) {
  if (!skl_hip_gemv_kc_rows_supported(g)) {
    skl_hip_record_error(-2, "gemv_kc_rows: unsupported problem");
    return -2;
  }
  const size_t grid = (g->n + 15) / 16;  // at most: one group of 16 columns per workgroup
  if (grid > 0x7FFFFFFFu) {
    skl_hip_record_error(-2, "gemv_kc_rows: grid too large");
    return -2;
  }
  const int kind = kind_of(g);
  const size_t es = kind >= kBF16 ? 2 : 1;
  const KcRowsArgs p = {(const char *)g->a, g->a_s0 * es, (const char *)g->b, g->b_s0 * es, g->c, g->rsc0, g->csc0,
                        g->m, g->n, (unsigned)(g->k * es), g->alpha, g->beta, g->bias, g->max, g->rq};
  switch (kind) {
    case kI8: return launch_kind<kI8>(p);
    case kE4M3: return launch_kind<kE4M3>(p);
    case kE5M2: return launch_kind<kE5M2>(p);
    case kMixed: return launch_kind<kMixed>(p);
    case kBF16: return launch_kind<kBF16>(p);
    default: return launch_kind<kF16>(p);
  }
}
