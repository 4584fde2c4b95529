// skl_gemm_tiled.hip - register-tiled GEMM for the contractions that have no matrix-core path here because
// their results are defined operation by operation: f32 x f32 -> f32 (ref/gemm/gemm_f32rc_f32rc_f32rc.c:9-24),
// f64 x f64 -> f64 (ref/gemm/gemm_f64rc_f64rc_f64rc.c:9-24), f16 x f16 -> f16 with an f16 accumulator
// (ref/gemm/gemm_f16rc_f16rc_f16rc.c:9-24) and their blocked twins in the canonical layouts.
//
// Every element of C is accumulated exactly as the reference's loop does it - k ascending, a separately rounded
// multiply and add per step (f16: the sum rounded to half per step) - so results equal the reference's bit for
// bit for finite data, like the any-stride kernel's; what changes is where the operands come from: a workgroup
// keeps a tile of C in registers and walks K in slabs of 16 or 32 staged through LDS (two stages, the next slab's
// global loads issued before the current slab's arithmetic, four elements per load along the operand's unit stride).
// A thread's rows and columns are runs of up to four, a share of the tile apart, so that the lanes of a wave
// read consecutive 16-byte pieces of the LDS rows. The last slab is filled past K with +0 in A and B: adding the product
// +0 leaves an f32 or f64 accumulator unchanged, which started at +0 and is never -0. An f16 one can be: a negative sum
// underflows when it is rounded to half, and C's sign shows it if beta*C is a -0 too. There B's fill is -0, and adding
// the product -0 leaves every accumulator as it is.
//
// What bounds it: the order of the sum is fixed, so K cannot be shared out, and a wave alone on its SIMD issues one
// vector instruction in five to six cycles where several waves together issue one in three. So a tile is split over
// as many waves as its LDS reads allow: 8 x 4 per thread on the 128 x 128 tile (8 x 8, one wave per SIMD at
// 2048^3: 600 us; 8 x 4: 345), and fewer elements per thread, on smaller tiles, the fewer tiles there are - which
// also shortens the chain of K steps that every thread goes through (f32 512 x 512 x 2048: 64 x 64 tiles of 4 x 4
// per thread 182 us, 4 x 2 121, 32 x 32 tiles of 2 x 2 78, 16 x 32 tiles of 2 x 1 70).
// f32 2048^3: 427 us with 64 x 64 tiles, one element per load and bounds checks on each -> 345 us, 50 T
// vector operations per second (a multiply and an add per step); 4096 x 4096 x 2048 1381 -> 1243 us, 55 T.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "skl_device.hpp"

namespace {

// Whether the beta == 0 case needs the old C at all (kinds that cannot tell say yes).
__device__ __forceinline__ bool tiled_needs_c(float acc, skl_scalar alpha, skl_scalar beta) { return skl_initialise_needs_c(acc, alpha, beta); }
__device__ __forceinline__ bool tiled_needs_c(double, skl_scalar, skl_scalar) { return true; }

template <int DT>
struct Kind;
template <>
struct Kind<SKL_DT_F32> {
  using In = float;     // element type in memory
  using Stage = float;  // element type in LDS
  using Acc = float;
  using C = float;
  __device__ static Stage stage(In v) { return v; }
  __device__ static Acc step(Acc acc, Stage a, Stage b) { return __fadd_rn(acc, __fmul_rn(a, b)); }
};
template <>
struct Kind<SKL_DT_F64> {
  using In = double;
  using Stage = double;
  using Acc = double;
  using C = double;
  __device__ static Stage stage(In v) { return v; }
  __device__ static Acc step(Acc acc, Stage a, Stage b) { return __dadd_rn(acc, __dmul_rn(a, b)); }
};
// `_Float16` arithmetic as a C compiler evaluates it without half-precision instructions: operands promoted to
// float (the product of two halves is exact there), the sum rounded to float and then to half on assignment.
template <>
struct Kind<SKL_DT_F16H> {
  using In = _Float16;
  using Stage = float;
  using Acc = _Float16;
  using C = _Float16;
  __device__ static Stage stage(In v) { return (float)v; }
  __device__ static Acc step(Acc acc, Stage a, Stage b) { return (_Float16)__fadd_rn((float)acc, __fmul_rn(a, b)); }
};

struct TiledArgs {
  const void *a, *b;
  void *c;
  size_t m, n, k;
  size_t a_s1, a_s0, a_sk, b_s1, b_s0, b_sk;
  size_t rsc0, csc0, rsc1, csc1;
  skl_scalar alpha, beta;
  unsigned tiles_n;
};

// N values that lie side by side, at the alignment of one of them: the memory unit takes 16-byte accesses on any
// element boundary, so no layout needs a copy or a path of its own for its alignment.
template <typename T, int N>
struct Run {
  typedef T Vec __attribute__((ext_vector_type(N)));
  typedef Vec Type __attribute__((aligned(sizeof(T))));
};

// One operand's share of a slab: BT rows (columns) x kSlab k, in groups of four elements along the operand's unit
// stride (K if KC, else its rows / columns); kGroups groups per thread. A thread's groups keep their place from slab to
// slab, so the addresses are worked out once.
template <int DT, int BT, int kSlab, int kThreads, bool KC>
struct Fetch {
  static constexpr int kTotal = BT * kSlab / 4, kGroups = (kTotal + kThreads - 1) / kThreads;
  using In = typename Kind<DT>::In;
  using Stage = typename Kind<DT>::Stage;
  using Four = typename Run<In, 4>::Type;
  const In *at[kGroups];  // the group's first element in the first slab (clamped into the operand)
  int inside[kGroups];    // elements along the rows / columns in range: 4 or fewer (KC: 1 or 0)
  size_t s0, sk;
  bool unit;              // the stride groups run along is 1

  __device__ static int group(int e) { return e * kThreads + (int)threadIdx.x; }
  __device__ static bool whole(int e) { return kTotal % kThreads == 0 || group(e) < kTotal; }
  __device__ static int x_of(int e) { return KC ? group(e) / (kSlab / 4) : group(e) % (BT / 4) * 4; }
  __device__ static int p_of(int e) { return KC ? group(e) % (kSlab / 4) * 4 : group(e) / (BT / 4); }

  __device__ void init(const In *base, size_t s1, size_t s0_, size_t sk_, size_t x0, size_t xn) {
    s0 = s0_, sk = sk_;
    unit = (KC ? sk : s0) == 1;
#pragma unroll
    for (int e = 0; e < kGroups; ++e) {
      const size_t x = x0 + (whole(e) ? x_of(e) : 0);
      const size_t left = x < xn ? xn - x : 0;
      inside[e] = KC ? left != 0 : left < 4 ? (int)left : 4;
      const size_t y = left ? x : 0;
      at[e] = base + (y / 64) * s1 + (y % 64) * s0 + (whole(e) ? p_of(e) : 0) * sk;
    }
  }

  // The slab that starts `p0` k into the operand and has `left` of them (kSlab or more: whole); `past`: what stands
  // for elements outside the operand.
  __device__ __forceinline__ void load(Stage (&r)[kGroups][4], size_t p0, size_t left, Stage past) const {
#pragma unroll
    for (int e = 0; e < kGroups; ++e) {
      const In *g = at[e] + p0 * sk;
      if (!whole(e)) continue;
      if (left >= (size_t)kSlab && unit && inside[e] == (KC ? 1 : 4)) {
        const Four v = *reinterpret_cast<const Four *>(g);
#pragma unroll
        for (int i = 0; i < 4; ++i) r[e][i] = Kind<DT>::stage(v[i]);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const bool in = KC ? inside[e] != 0 && (size_t)(p_of(e) + i) < left : i < inside[e] && (size_t)p_of(e) < left;
          r[e][i] = in ? Kind<DT>::stage(g[i * (KC ? sk : s0)]) : past;
        }
      }
    }
  }

  __device__ __forceinline__ void store(const Stage (&r)[kGroups][4], Stage (*tile)[BT + 4]) const {
#pragma unroll
    for (int e = 0; e < kGroups; ++e) {
      if (!whole(e)) continue;
      const int x = x_of(e), p = p_of(e);
      if constexpr (KC) {
#pragma unroll
        for (int i = 0; i < 4; ++i) tile[p + i][x] = r[e][i];
      } else {
        typedef Stage V4 __attribute__((ext_vector_type(4)));
        *reinterpret_cast<V4 *>(&tile[p][x]) = V4{r[e][0], r[e][1], r[e][2], r[e][3]};
      }
    }
  }
};

// A thread's rows (columns): T of them in runs of up to four, the runs a share of the tile apart.
template <int BT, int T>
__device__ constexpr int tiled_index(int t, int i) {
  constexpr int W = T < 4 ? T : 4;
  return (i / W) * (BT / (T / W)) + t * W + i % W;
}
template <int T, typename Stage, int BT>
__device__ __forceinline__ void tiled_read(Stage (&v)[T], const Stage (&row)[BT], int t, int edge) {
  constexpr int W = T < 4 ? T : 4;
  typedef Stage V __attribute__((ext_vector_type(W)));
#pragma unroll
  for (int q = 0; q < T / W; ++q) {
    const V x = *reinterpret_cast<const V *>(&row[q * (edge / (T / W)) + t * W]);
#pragma unroll
    for (int i = 0; i < W; ++i) v[q * W + i] = x[i];
  }
}

template <int DT, int BM, int BN, int TR, int TC, int kSlab, bool A_KC, bool B_KC>
__global__ void __launch_bounds__((BM / TR) * (BN / TC)) gemm_tiled_kernel(TiledArgs g) {
  using K = Kind<DT>;
  using Stage = typename K::Stage;
  using Acc = typename K::Acc;
  constexpr int kThreads = (BM / TR) * (BN / TC);
  using FA = Fetch<DT, BM, kSlab, kThreads, A_KC>;
  using FB = Fetch<DT, BN, kSlab, kThreads, B_KC>;
  constexpr int kUnrollK = TR * TC >= 64 ? 2 : 4;
  constexpr Stage kPastB = DT == SKL_DT_F16H ? Stage(-0.0) : Stage(0.0);
  __shared__ __attribute__((aligned(16))) Stage As[2][kSlab][BM + 4];
  __shared__ __attribute__((aligned(16))) Stage Bs[2][kSlab][BN + 4];

  const int tid = threadIdx.x, ty = tid / (BN / TC), tx = tid % (BN / TC);
  const size_t row0 = (size_t)(blockIdx.x / g.tiles_n) * BM, col0 = (size_t)(blockIdx.x % g.tiles_n) * BN;

  Acc acc[TR][TC];
#pragma unroll
  for (int r = 0; r < TR; ++r)
#pragma unroll
    for (int c = 0; c < TC; ++c) acc[r][c] = Acc(0);

  FA fa;
  FB fb;
  fa.init((const typename K::In *)g.a, g.a_s1, g.a_s0, g.a_sk, row0, g.m);
  fb.init((const typename K::In *)g.b, g.b_s1, g.b_s0, g.b_sk, col0, g.n);
  Stage ra[FA::kGroups][4], rb[FB::kGroups][4];
  fa.load(ra, 0, g.k, Stage(0.0));
  fb.load(rb, 0, g.k, kPastB);
  fa.store(ra, As[0]);
  fb.store(rb, Bs[0]);
  __syncthreads();
  int cur = 0;
  for (size_t p0 = 0; p0 < g.k; p0 += kSlab, cur ^= 1) {
    const size_t next = p0 + kSlab;
    if (next < g.k) {
      fa.load(ra, next, g.k - next, Stage(0.0));
      fb.load(rb, next, g.k - next, kPastB);
    }
#pragma unroll kUnrollK  // a full unroll makes the compiler fetch a whole slab into registers (256 + AGPRs)
    for (int kk = 0; kk < kSlab; ++kk) {
      Stage av[TR], bv[TC];
      tiled_read(av, As[cur][kk], ty, BM);
      tiled_read(bv, Bs[cur][kk], tx, BN);
#pragma unroll
      for (int r = 0; r < TR; ++r)
#pragma unroll
        for (int c = 0; c < TC; ++c) acc[r][c] = K::step(acc[r][c], av[r], bv[c]);
    }
    if (next < g.k) {
      fa.store(ra, As[cur ^ 1]);
      fb.store(rb, Bs[cur ^ 1]);
    }
    __syncthreads();
  }

  using Out = typename K::C;
  using Wide = typename std::conditional<DT == SKL_DT_F16H, float, Out>::type;  // what alpha and beta are applied in
  Out *cbase = (Out *)g.c;
  const bool init = skl_beta_is_zero<Wide>(g.beta);
  constexpr int W = TC < 4 ? TC : 4, kRuns = TC / W;
  using CRun = typename Run<Out, W>::Type;
#pragma unroll
  for (int r = 0; r < TR; ++r) {
    const size_t i = row0 + tiled_index<BM, TR>(ty, r);
    if (i >= g.m) continue;
    Out *crow = cbase + (i / 64) * g.rsc1 + (i % 64) * g.rsc0;
    // A row's old values are requested together, ahead of its first store. Where C's columns lie side by side a run of
    // them is one access: dword by dword every store of a wave covers a quarter of each cache line (f32 2406 x 2003 x 16
    // 21.5 -> 17.6 us, 13.7 with slabs of 16; 2048 x 2048 x 2048 unchanged).
    Out *cp[kRuns];
    Wide old[TC];
#pragma unroll
    for (int q = 0; q < kRuns; ++q) {
      const size_t j = col0 + tiled_index<BN, TC>(tx, q * W);
      cp[q] = crow + (j / 64) * g.csc1 + (j % 64) * g.csc0;
      bool need[W], any = false;
#pragma unroll
      for (int e = 0; e < W; ++e) {
        old[q * W + e] = Wide(0);
        need[e] = j + e < g.n && (!init || tiled_needs_c((Wide)acc[r][q * W + e], g.alpha, g.beta));
        any |= need[e];
      }
      if (g.csc0 == 1 && j + W <= g.n) {
        if (any) {
          const CRun v = *reinterpret_cast<const CRun *>(cp[q]);
#pragma unroll
          for (int e = 0; e < W; ++e) old[q * W + e] = need[e] ? (Wide)v[e] : Wide(0);
        }
      } else {
#pragma unroll
        for (int e = 0; e < W; ++e)
          if (need[e]) old[q * W + e] = (Wide)cp[q][e * g.csc0];
      }
    }
#pragma unroll
    for (int q = 0; q < kRuns; ++q) {
      const size_t j = col0 + tiled_index<BN, TC>(tx, q * W);
      CRun v;
#pragma unroll
      for (int e = 0; e < W; ++e) {
        const Wide sum = (Wide)acc[r][q * W + e];
        v[e] = (Out)(init ? skl_initialise(sum, &old[q * W + e], g.alpha, g.beta) : skl_combine(sum, old[q * W + e], g.alpha, g.beta));
      }
      if (g.csc0 == 1 && j + W <= g.n) {
        *reinterpret_cast<CRun *>(cp[q]) = v;
      } else {
#pragma unroll
        for (int e = 0; e < W; ++e)
          if (j + e < g.n) cp[q][e * g.csc0] = v[e];
      }
    }
  }
}

template <int DT, int BM, int BN, int TR, int TC, int kSlab, bool A_KC, bool B_KC>
int launch_layout(const skl_gemm_canon *g) {
  TiledArgs p;
  p.a = g->a, p.b = g->b, p.c = g->c;
  p.m = g->m, p.n = g->n, p.k = g->k;
  p.a_s1 = g->a_s1, p.a_s0 = g->a_s0, p.a_sk = g->a_sk;
  p.b_s1 = g->b_s1, p.b_s0 = g->b_s0, p.b_sk = g->b_sk;
  p.rsc0 = g->rsc0, p.csc0 = g->csc0, p.rsc1 = g->rsc1, p.csc1 = g->csc1;
  p.alpha = g->alpha, p.beta = g->beta;
  const size_t tm = (g->m + BM - 1) / BM, tn = (g->n + BN - 1) / BN;
  if (tm * tn > 0x7FFFFFFFu) {
    skl_hip_record_error(-2, "gemm_tiled: too many tiles for one launch");
    return -2;
  }
  p.tiles_n = (unsigned)tn;
  gemm_tiled_kernel<DT, BM, BN, TR, TC, kSlab, A_KC, B_KC><<<(unsigned)(tm * tn), (BM / TR) * (BN / TC), 0, skl_current_stream()>>>(p);
  return skl_check_launch("gemm_tiled");
}

template <int DT, int BM, int BN, int TR, int TC, int kSlab>
int launch(const skl_gemm_canon *g) {
  const bool a_kc = g->a_sk <= g->a_s0, b_kc = g->b_sk <= g->b_s0;
  if (a_kc && b_kc) return launch_layout<DT, BM, BN, TR, TC, kSlab, true, true>(g);
  if (a_kc) return launch_layout<DT, BM, BN, TR, TC, kSlab, true, false>(g);
  if (b_kc) return launch_layout<DT, BM, BN, TR, TC, kSlab, false, true>(g);
  return launch_layout<DT, BM, BN, TR, TC, kSlab, false, false>(g);
}

// The tile by the number of 64 x 64 and 32 x 32 tiles there are: the largest that still gives every SIMD several waves.
// f32, us, at K = 2048 (128 x 128 / 64 x 64 of 4 x 4 / 64 x 64 of 4 x 2 / 32 x 32 / 16 x 32 tiles):
//   4096^2: 1243 / 1275 / 1356 / 2110 / 3066    2048^2: 347 / 349 / 364 / 532 / 779
//   1024^2: 349 / 180 / 132 / 159 / 220          512^2: 338 / 170 / 121 / 78 / 70     256^2: 337 / 169 / 121 / 76 / 61
// The same limits serve f64 and f16: over 500 random problems the median time over that of 64 x 64 and 128 x 128 tiles alone
// is, on the tiles from 64 x 64 of 4 x 2 down, f32 0.71 / 0.45 / 0.30, f64 0.81 / 0.56 / 0.40, f16 0.72 / 0.48 / 0.27.
//
// Floats are staged in slabs of 32 from K = 512 on, of 16 below on the two larger tiles: half the LDS puts more
// workgroups on a compute unit, which is what a short K lives on, and a K of 16 fills its slab (f32, over the time with
// slabs of 32, K up to 16 / 32 / 64 / 128 / 256: 64 x 64 tiles 0.78 / 0.96 / 0.95 / 0.96 / 0.94, 128 x 128
// 0.67 / 0.86 / 0.87 / 0.95 / 0.95; 2048^3 361 us with 32 and 367 with 16, f16 with A by columns 4096 x 4096 x 2048 2291 and 2404).
template <int DT>
int launch_sized(const skl_gemm_canon *g) {
  constexpr bool kDoubles = sizeof(typename Kind<DT>::Stage) == 8;
  constexpr int kSlab = kDoubles ? 16 : 32;  // 66 KiB of LDS for the largest tile of floats
  const auto tiles = [&](size_t bm, size_t bn) { return ((g->m + bm - 1) / bm) * ((g->n + bn - 1) / bn); };
  if (tiles(128, 128) >= 512) {
    // doubles: twice the bytes of LDS per step, so 8 x 8 per thread (4096 x 4096 x 2048: 8 x 4 2517 us, 8 x 8
    // 2203 us)
    if constexpr (kDoubles) return launch<DT, 128, 128, 8, 8, 8>(g);
    else return g->k < 512 ? launch<DT, 128, 128, 8, 4, 16>(g) : launch<DT, 128, 128, 8, 4, kSlab>(g);
  }
  if (tiles(64, 64) >= 768) return g->k < 512 ? launch<DT, 64, 64, 4, 4, 16>(g) : launch<DT, 64, 64, 4, 4, kSlab>(g);
  if (tiles(64, 64) >= 176) return launch<DT, 64, 64, 4, 2, 16>(g);
  if (tiles(32, 32) > 256) return launch<DT, 32, 32, 2, 2, kSlab>(g);
  return launch<DT, 16, 32, 2, 1, kSlab>(g);
}

}  // namespace

extern "C" int skl_hip_gemm_tiled_supported(const skl_gemm_canon *g) {
  if (g->ta != g->tb || g->bias || g->max || g->rq.act || g->rq.q || g->c_row_shift != 6 || g->c_col_shift != 6) return 0;
  if (g->ta != SKL_DT_F32 && g->ta != SKL_DT_F64 && g->ta != SKL_DT_F16H) return 0;
  return g->m != 0 && g->n != 0 && g->k != 0;
}

extern "C" int skl_hip_launch_gemm_tiled(const skl_gemm_canon *g) {
  if (!skl_hip_gemm_tiled_supported(g)) {
    skl_hip_record_error(-2, "gemm_tiled: unsupported problem");
    return -2;
  }
  switch (g->ta) {
    case SKL_DT_F32: return launch_sized<SKL_DT_F32>(g);
    case SKL_DT_F64: return launch_sized<SKL_DT_F64>(g);
    default: return launch_sized<SKL_DT_F16H>(g);
  }
}
