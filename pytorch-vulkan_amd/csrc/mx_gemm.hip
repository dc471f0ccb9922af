// FP32 strided / batched GEMM with fused alpha, beta*bias epilogue on gfx950
// MFMA (FP32 operands as three bf16 pieces, mfma_core.hpp).
//
// Covers the reference's matmul_strided{,_reg}{,_bias}.comp and
// bmm_strided.comp (mm_impl csrc/ops/mm.cpp:244-343, addmm_bias_vulkan
// csrc/ops/mm.cpp:835-879, bmm_impl csrc/ops/bmm.cpp:16-68): A and B are read
// straight from arbitrary strided views (a transposed weight costs no copy),
// and the bias add of nn.Linear happens in the store.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <string>
#include <type_traits>

#include "mfma_core.hpp"
#include "mx_internal.hpp"

namespace mx {
namespace {

using namespace mfma;

struct GemmArgs {
  const float* a;
  const float* b;
  const float* bias;
  float* c;
  int64_t a_sb, a_sm, a_sk;
  int64_t b_sb, b_sk, b_sn;
  int64_t c_sb, ldc;
  int64_t bias_sb, bias_sm, bias_sn;
  int M, N, K, batch, batch0;
  int tiles_m, tiles_n;
  float alpha, beta;
  int bias_kind;
  // K split (splits > 1): split i takes k in [i * kps, (i + 1) * kps) and
  // writes its partial product to ws[i][batch][M][N].
  int splits, kps;
  float* ws;
};

template <class C, Mode MA, Mode MB>
MX_TILE_KERNEL(C) void gemm_kernel(GemmArgs p) {
  __shared__ __attribute__((aligned(16))) float smem[C::SMEM_FLOATS];
  int tm, tn;
  tile_coords(xcd_remap(blockIdx.x, p.tiles_m * p.tiles_n), p.tiles_m, p.tiles_n, tm, tn);
  const int row0 = tm * C::BM, col0 = tn * C::BN;
  const int64_t bz = int64_t(p.batch0) + blockIdx.z;
  const int split = blockIdx.y;
  const int k0 = split * p.kps, k1 = min(p.K, k0 + p.kps);
  StridedLoader<C::BM, C::BK, MA> la;
  StridedLoader<C::BN, C::BK, MB> lb;
  Acc<C> acc;
  const float scale = tile_product<C, true>(acc, la, lb, (k1 - k0 + C::BK - 1) / C::BK, smem, [&](auto& a, auto& b) {
    a.init(p.a + bz * p.a_sb, p.a_sm, p.a_sk, row0, p.M, k0, k1);
    b.init(p.b + bz * p.b_sb, p.b_sn, p.b_sk, col0, p.N, k0, k1);
  });
  if (p.splits > 1) {
    uint32_t col[C::FN];
#pragma unroll
    for (int j = 0; j < C::FN; ++j) {
      const int n = acc_col<C>(j);
      col[j] = col0 + n < p.N ? uint32_t(n) * 4u : kOffNone;
    }
    float* const part = p.ws + ((int64_t(split) * p.batch + bz) * p.M + row0) * p.N + col0;
    store_tile<C>(buffer_rsrc(part, kBufMaxBytes), col, uint32_t(p.N) * 4u, 0, p.M - row0,
                  [&](int i, int j, int v) { return acc.v[i][j][v] * scale; });
    return;
  }
  float* __restrict__ cb = p.c + bz * p.c_sb;
  const float* __restrict__ bias = p.bias ? p.bias + bz * p.bias_sb : nullptr;
  const float alpha = p.alpha, beta = p.beta;
  const int kind = (p.bias_kind == MX_BIAS_NONE || beta == 0.f) ? MX_BIAS_NONE : p.bias_kind;
  int ccol[C::FN];
  float bcol[C::FN];
#pragma unroll
  for (int j = 0; j < C::FN; ++j) {
    ccol[j] = col0 + acc_col<C>(j);
    // Column bias (nn.Linear): one value per fragment column, loaded once.
    bcol[j] = (kind == MX_BIAS_COL && ccol[j] < p.N) ? beta * bias[int64_t(ccol[j]) * p.bias_sn] : 0.f;
  }
  // Two separate walks: stores and loads share the vector-memory counter, so
  // a bias load between stores makes every later store wait for the earlier
  // ones; only the matrix-bias walk (baddbmm) reads memory between stores.
  if (kind == MX_BIAS_MATRIX) {
    for_each_acc_row<C>([&](int r, int i, int v) {
      const int row = row0 + r;
      if (row >= p.M) return;
      float* __restrict__ crow = cb + int64_t(row) * p.ldc;
      const float* __restrict__ brow = bias + int64_t(row) * p.bias_sm;
#pragma unroll
      for (int j = 0; j < C::FN; ++j)
        if (ccol[j] < p.N) crow[ccol[j]] = alpha * (acc.v[i][j][v] * scale) + beta * brow[int64_t(ccol[j]) * p.bias_sn];
    });
    return;
  }
  if (p.ldc >= 0 && p.ldc <= kVecStrideMax) {
    // Offsets from the tile's corner, below 2^31 bytes at this row stride.
    uint32_t col[C::FN];
#pragma unroll
    for (int j = 0; j < C::FN; ++j) col[j] = ccol[j] < p.N ? uint32_t(ccol[j] - col0) * 4u : kOffNone;
    store_tile<C>(buffer_rsrc(cb + int64_t(row0) * p.ldc + col0, kBufMaxBytes), col, uint32_t(p.ldc) * 4u, 0,
                  p.M - row0, [&](int i, int j, int v) { return alpha * (acc.v[i][j][v] * scale) + bcol[j]; });
    return;
  }
  for_each_acc_row<C>([&](int r, int i, int v) {
    const int row = row0 + r;
    if (row >= p.M) return;
    float* __restrict__ crow = cb + int64_t(row) * p.ldc;
#pragma unroll
    for (int j = 0; j < C::FN; ++j)
      if (ccol[j] < p.N) crow[ccol[j]] = alpha * (acc.v[i][j][v] * scale) + bcol[j];
  });
}

// C = alpha * (sum of the K splits' partial products, in split order) +
// beta * bias.  VEC: four columns per thread (N and C's strides multiples of
// four, C 16-byte aligned).
template <bool VEC>
__global__ __launch_bounds__(256) void gemm_sum_kernel(GemmArgs p) {
  constexpr int W = VEC ? 4 : 1;
  typedef float vec __attribute__((ext_vector_type(W)));
  const int64_t plane = int64_t(p.M) * p.N, total = plane * p.batch;
  const int kind = p.beta == 0.f ? int(MX_BIAS_NONE) : p.bias_kind;
  for (int64_t i = (int64_t(blockIdx.x) * 256 + threadIdx.x) * W; i < total; i += int64_t(gridDim.x) * 256 * W) {
    const float* src = p.ws + i;
    vec s = *reinterpret_cast<const vec*>(src);
#pragma unroll 8
    for (int q = 1; q < p.splits; ++q) s += *reinterpret_cast<const vec*>(src + q * total);
    const int64_t bz = i / plane;
    const uint32_t at = uint32_t(i - bz * plane), row = at / uint32_t(p.N), n = at - row * uint32_t(p.N);
    vec o;
    if constexpr (VEC) {
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = p.alpha * s[e];
    } else {
      o = p.alpha * s;
    }
    if (kind != MX_BIAS_NONE) {
      const float* b = p.bias + bz * p.bias_sb + n * p.bias_sn + (kind == MX_BIAS_COL ? 0 : row * p.bias_sm);
      if constexpr (VEC) {
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] += p.beta * b[e * p.bias_sn];
      } else {
        o += p.beta * b[0];
      }
    }
    *reinterpret_cast<vec*>(p.c + bz * p.c_sb + int64_t(row) * p.ldc + n) = o;
  }
}

// k == 0: C = beta * bias (or zeros when beta == 0 / no bias).
__global__ void gemm_k0_kernel(GemmArgs p) {
  const int64_t total = int64_t(p.batch) * p.M * p.N;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
       i += int64_t(gridDim.x) * blockDim.x) {
    const int col = int(i % p.N);
    const int64_t rest = i / p.N;
    const int row = int(rest % p.M);
    const int bz = int(rest / p.M);
    float out = 0.f;
    if (p.bias_kind != MX_BIAS_NONE && p.beta != 0.f) {
      const float* bias = p.bias + int64_t(bz) * p.bias_sb;
      const float bv = p.bias_kind == MX_BIAS_COL ? bias[int64_t(col) * p.bias_sn]
                                                  : bias[int64_t(row) * p.bias_sm + int64_t(col) * p.bias_sn];
      out = p.beta * bv;
    }
    p.c[int64_t(bz) * p.c_sb + int64_t(row) * p.ldc + col] = out;
  }
}

bool aligned16(const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15u) == 0; }

// Operand layout -> loader mode.  rows = m for A, n for B.
Mode pick_mode(const float* base, int64_t s_row, int64_t s_k, int64_t s_batch, int64_t batch, int64_t R,
               int64_t K) {
  const bool batch_ok = batch <= 1 || s_batch % 4 == 0;
  const auto vec_stride = [](int64_t s) { return s >= 0 && s <= kVecStrideMax && s % 4 == 0; };
  if (s_k == 1 && aligned16(base) && vec_stride(s_row) && batch_ok && K % 4 == 0) return Mode::KVEC;
  if (s_row == 1 && aligned16(base) && vec_stride(s_k) && batch_ok && R % 4 == 0) return Mode::RVEC;
  if (s_k == 1) return Mode::KSCALAR;
  if (s_row == 1) return Mode::RSCALAR;
  return std::llabs(s_k) <= std::llabs(s_row) ? Mode::KSCALAR : Mode::RSCALAR;
}

template <class C, Mode MA, Mode MB>
int launch3(GemmArgs p, hipStream_t s) {
  // A 128x128 tile has the registers for two slabs of each operand in flight
  // when both are read 16 bytes at a time, and for the second accumulator set
  // unless both are row-scalar.
  constexpr bool sq = C::BM * C::BN == 128 * 128;
  constexpr bool vec = (MA == Mode::KVEC || MA == Mode::RVEC) && (MB == Mode::KVEC || MB == Mode::RVEC);
  constexpr bool dual = !(sq && MA == Mode::RSCALAR && MB == Mode::RSCALAR);
  using D = std::conditional_t<sq, Cfg<C::BM, C::BN, C::BK, C::WAVES_M, C::OCC, dual, vec>, C>;
  const int ntiles = p.tiles_m * p.tiles_n;
  for (int b0 = 0; b0 < p.batch; b0 += 65535) {
    p.batch0 = b0;
    const dim3 grid(ntiles, p.splits, std::min(p.batch - b0, 65535));
    hipLaunchKernelGGL((gemm_kernel<D, MA, MB>), grid, dim3(kThreads), 0, s, p);
    MX_HIP(hipGetLastError());
  }
  return MX_OK;
}

template <class C, Mode MA>
int launch2(const GemmArgs& p, Mode mb, hipStream_t s) {
  switch (mb) {
    case Mode::KVEC: return launch3<C, MA, Mode::KVEC>(p, s);
    case Mode::RVEC: return launch3<C, MA, Mode::RVEC>(p, s);
    case Mode::KSCALAR: return launch3<C, MA, Mode::KSCALAR>(p, s);
    default: return launch3<C, MA, Mode::RSCALAR>(p, s);
  }
}

template <class C>
int launch1(GemmArgs p, Mode ma, Mode mb, hipStream_t s) {
  p.tiles_m = (p.M + C::BM - 1) / C::BM;
  p.tiles_n = (p.N + C::BN - 1) / C::BN;
  switch (ma) {
    case Mode::KVEC: return launch2<C, Mode::KVEC>(p, mb, s);
    case Mode::RVEC: return launch2<C, Mode::RVEC>(p, mb, s);
    case Mode::KSCALAR: return launch2<C, Mode::KSCALAR>(p, mb, s);
    default: return launch2<C, Mode::RSCALAR>(p, mb, s);
  }
}

// 256-row tiles are built for the 16-byte operand modes only (scalar modes
// would need a register per row pass).
template <class C>
int launch1_vec(GemmArgs p, Mode ma, Mode mb, hipStream_t s) {
  p.tiles_m = (p.M + C::BM - 1) / C::BM;
  p.tiles_n = (p.N + C::BN - 1) / C::BN;
  if (ma == Mode::KVEC)
    return mb == Mode::KVEC ? launch3<C, Mode::KVEC, Mode::KVEC>(p, s) : launch3<C, Mode::KVEC, Mode::RVEC>(p, s);
  return mb == Mode::KVEC ? launch3<C, Mode::RVEC, Mode::KVEC>(p, s) : launch3<C, Mode::RVEC, Mode::RVEC>(p, s);
}

bool is_vec(Mode m) { return m == Mode::KVEC || m == Mode::RVEC; }

// Tile menu (BM x BN x BK, wave grid, waves per SIMD).  All keep two or more
// workgroups resident per CU.
using TileTall = Cfg<256, 128, 16, 2, 2>;  // 4 waves of 128 x 64
using TileWide = Cfg<128, 256, 16, 2, 2>;  // 4 waves of 64 x 128
using TileSq = Cfg<128, 128, 16, 2, 2>;    // 4 waves of 64 x 64
using TileSmall = Cfg<64, 64, 16, 2, 4>;   // 4 waves of 32 x 32

struct TileChoice {
  int bm, bn, per_cu;
  double rate;  // throughput of a CU full of such tiles, relative to 85% of its FP32 MFMA peak
};
constexpr TileChoice kTiles[] = {{256, 128, 2, 1.81}, {128, 256, 2, 1.75}, {128, 128, 2, 1.70}, {64, 64, 4, 1.36}};

constexpr int64_t kMaxSplitBytes = int64_t(64) << 20;  // partial products of one call (a caller's budget may hold less)
constexpr int kSplitBK = 32;                           // K granularity of a split
constexpr int kMinSplitSpan = 64;                      // shortest K range worth a split

// Estimated time: a CU holding n tiles runs at rate * occ(n), occ rising from
// 0.71 with one resident tile to 1 with per_cu; a tile's first loads and its
// stores cost as much as 41 more k; the sum of the partials moves
// (splits + 1) outputs at 3.6 TB/s after a launch.  The figures are the
// convolution planner's, whose tiles run the same product.
// `tiles` without splits; `cu` the CU count, a runtime query made once a call.
double tile_cost(const TileChoice& t, int64_t tiles, int64_t cu, int64_t m, int64_t n, int64_t batch, int64_t splits,
                 int64_t kps) {
  const double per_cu = double((tiles * splits + cu - 1) / cu);
  const double occ = std::min(1.0, 0.71 + 0.29 * (per_cu - 1) / double(t.per_cu - 1));
  double s = per_cu * 2.0 * t.bm * t.bn * (double(kps) + 41.0) / (0.85 * 157.3e12 / 256.0 * t.rate * occ) + 2e-6;
  if (splits > 1) s += double(splits + 1) * double(m * n * batch) * 4.0 / 3.6e12 + 3e-6;
  return s;
}

// Cheapest (tile, K split).  Few tiles over a long K leave most of the chip
// idle (8 x 2048 x 1000: 16 workgroups walking 128 slabs each, 38 us), so K is
// split where the model finds it faster, the partials summed by a second
// launch.  That launch and the partials' block cost the host 2.5 us (4.8 -> 7.3
// a call), lost wherever a program issues its calls no faster than they run, so
// a product that takes less than kMinSplitTime in one pass keeps it: about what
// a training loop takes to issue one of its calls.  Training passes of a linear
// layer, split / one pass: 8 x 573 x 466 56.9 / 49.1 us, 256 x 512 x 512 57.8 /
// 52.6, 8 x 1024 x 1024 54.7 / 56.6, 8 x 2048 x 1000 54.1 / 78.7; forward calls
// on their own: 8 x 512 x 512 10.0 / 13.5, 8 x 768 x 768 10.0 / 18.9, 8 x 2048 x
// 1000 11.1 / 45.3.  Operands read as scalars take longer than the model has it:
// 10 x 694 x 378, 13.9 us of it, runs for 23.5 us in one pass, 9.3 split.
// `partials`: bytes they may take.  MX_GEMM_TILE=<index into kTiles> forces a
// tile in one pass over K (tests and diagnosis; the 256-wide tiles only for
// 16-byte operand modes).  `kernel` (mx_gemm_kernel) forces the 64x64 tile or
// keeps the choice among the large ones.
constexpr double kMinSplitTime = 14e-6;

void pick_gemm_tile(int64_t m, int64_t n, int64_t k, int64_t batch, bool vec, int kernel, int64_t partials, int* tile,
                    int* splits, int* kps) {
  int first = vec ? 0 : 2, last = 3;
  if (kernel == MX_GEMM_KERNEL_TILED) first = 3;
  if (kernel == MX_GEMM_KERNEL_REGISTER) last = 2;
  if (const char* e = std::getenv("MX_GEMM_TILE")) {
    const int t = std::atoi(e);
    if (t >= (vec ? 0 : 2) && t < 4) {
      first = last = t;
      partials = 0;
    }
  }
  const int64_t cu = cu_count();
  const auto tiles_of = [&](int i) {
    return ((m + kTiles[i].bm - 1) / kTiles[i].bm) * ((n + kTiles[i].bn - 1) / kTiles[i].bn) * batch;
  };
  double best = -1;
  *splits = 1;
  *kps = int(k);
  for (int i = first; i <= last; ++i) {
    const double cost = tile_cost(kTiles[i], tiles_of(i), cu, m, n, batch, 1, k);
    if (best < 0 || cost < best) {
      best = cost;
      *tile = i;
    }
  }
  if (partials <= 0 || best * (vec ? 1.0 : 1.1) < kMinSplitTime) return;
  static const int kSplits[] = {2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64};
  for (int i = first; i <= last; ++i) {
    const int64_t tiles = tiles_of(i);
    for (const int want : kSplits) {
      const int64_t span = ((k + want - 1) / want + kSplitBK - 1) / kSplitBK * kSplitBK, s = (k + span - 1) / span;
      if (s < 2) continue;
      if (span < kMinSplitSpan || s * m * n * batch * 4 > partials) break;
      const double cost = tile_cost(kTiles[i], tiles, cu, m, n, batch, s, span);
      if (cost < best) {
        best = cost;
        *tile = i;
        *splits = int(s);
        *kps = int(span);
      }
    }
  }
}

}  // namespace
}  // namespace mx

using namespace mx;

namespace mx {
namespace {

const char* mode_name(Mode m) {
  switch (m) {
    case Mode::KVEC: return "KVEC";
    case Mode::RVEC: return "RVEC";
    case Mode::KSCALAR: return "KSCALAR";
    default: return "RSCALAR";
  }
}

// Validated arguments, operand modes and tile of one mx_gemm_f32 call (the
// pointers only decide alignment; nothing is read).  Returns MX_OK with
// *empty set when the call writes nothing.
struct GemmPlan {
  GemmArgs p{};
  Mode ma = Mode::KVEC, mb = Mode::KVEC;
  int tile = 2;
  bool empty = false;
};

int plan_gemm(const mx_gemm_desc* d, const float* a, const float* b, const float* bias, float* c, int64_t partials,
              GemmPlan* g) {
  MX_REQUIRE(d, MX_ERR_INVALID, "mx_gemm_f32: null descriptor");
  MX_REQUIRE(d->batch >= 0 && d->m >= 0 && d->n >= 0 && d->k >= 0, MX_ERR_INVALID,
             "mx_gemm_f32: negative dimension");
  MX_REQUIRE(d->m <= INT32_MAX && d->n <= INT32_MAX && d->k <= INT32_MAX && d->batch <= INT32_MAX,
             MX_ERR_INVALID, "mx_gemm_f32: dimension exceeds int32");
  MX_REQUIRE(d->bias_kind >= MX_BIAS_NONE && d->bias_kind <= MX_BIAS_MATRIX, MX_ERR_INVALID,
             "mx_gemm_f32: bad bias kind");
  MX_REQUIRE(d->kernel >= MX_GEMM_KERNEL_AUTO && d->kernel <= MX_GEMM_KERNEL_REGISTER, MX_ERR_INVALID,
             "mx_gemm: unknown kernel class ", d->kernel);
  g->empty = d->batch == 0 || d->m == 0 || d->n == 0;
  if (g->empty) return MX_OK;
  GemmArgs& p = g->p;
  p.a = a ? a + d->a_offset : nullptr;
  p.b = b ? b + d->b_offset : nullptr;
  p.bias = bias ? bias + d->bias_offset : nullptr;
  p.c = c ? c + d->c_offset : nullptr;
  p.a_sb = d->a_stride_b;
  p.a_sm = d->a_stride_m;
  p.a_sk = d->a_stride_k;
  p.b_sb = d->b_stride_b;
  p.b_sk = d->b_stride_k;
  p.b_sn = d->b_stride_n;
  p.c_sb = d->c_stride_b;
  p.ldc = d->ldc;
  p.bias_sb = d->bias_stride_b;
  p.bias_sm = d->bias_stride_m;
  p.bias_sn = d->bias_stride_n;
  p.M = int(d->m);
  p.N = int(d->n);
  p.K = int(d->k);
  p.batch = int(d->batch);
  p.alpha = d->alpha;
  p.beta = d->beta;
  p.bias_kind = d->bias_kind;
  if (d->k == 0) return MX_OK;
  MX_REQUIRE(((d->m + 63) / 64) * ((d->n + 63) / 64) <= INT32_MAX, MX_ERR_INVALID, "mx_gemm_f32: too many tiles");
  g->ma = pick_mode(p.a, p.a_sm, p.a_sk, p.a_sb, p.batch, p.M, p.K);
  g->mb = pick_mode(p.b, p.b_sn, p.b_sk, p.b_sb, p.batch, p.N, p.K);
  pick_gemm_tile(d->m, d->n, d->k, d->batch, is_vec(g->ma) && is_vec(g->mb), d->kernel,
                 d->n <= kVecStrideMax && d->m * d->n <= INT32_MAX ? partials : 0, &g->tile, &p.splits, &p.kps);
  return MX_OK;
}

// A call whose stream is being captured into a graph must not take scratch
// from the allocator: the block would return to the cache while replays of the
// graph still use it.
bool may_allocate(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &st) == hipSuccess) return st == hipStreamCaptureStatusNone;
  (void)hipGetLastError();
  return false;
}

int launch_sum(const GemmArgs& p, hipStream_t s) {
  const bool vec = p.N % 4 == 0 && p.ldc % 4 == 0 && p.c_sb % 4 == 0 && aligned16(p.c) && aligned16(p.ws);
  const int64_t items = int64_t(p.batch) * p.M * p.N / (vec ? 4 : 1);
  const int blocks = int(std::min<int64_t>((items + 255) / 256, 65535));
  if (vec)
    hipLaunchKernelGGL(gemm_sum_kernel<true>, dim3(blocks), dim3(256), 0, s, p);
  else
    hipLaunchKernelGGL(gemm_sum_kernel<false>, dim3(blocks), dim3(256), 0, s, p);
  MX_HIP(hipGetLastError());
  return MX_OK;
}

constexpr const char* kTileNames[] = {"256x128x16", "128x256x16", "128x128x16", "64x64x16"};

int64_t partial_bytes(const GemmArgs& p) { return p.splits > 1 ? int64_t(p.splits) * p.batch * p.M * p.N * 4 : 0; }

}  // namespace

int gemm_within(const mx_gemm_desc* d, const float* a, const float* b, const float* bias, float* c, int64_t partials,
                hipStream_t s) {
  GemmPlan g;
  MX_TRY(plan_gemm(d, a, b, bias, c, std::min(partials, kMaxSplitBytes), &g));
  if (g.empty) return MX_OK;
  if (g.p.splits > 1 && !may_allocate(s)) MX_TRY(plan_gemm(d, a, b, bias, c, 0, &g));
  MX_REQUIRE(c, MX_ERR_INVALID, "mx_gemm_f32: null output");
  MX_REQUIRE(d->bias_kind == MX_BIAS_NONE || bias, MX_ERR_INVALID, "mx_gemm_f32: null bias");
  GemmArgs& p = g.p;
  if (d->k == 0) {
    const int64_t total = d->batch * d->m * d->n;
    const int blocks = int(std::min<int64_t>((total + 255) / 256, 65535));
    hipLaunchKernelGGL(gemm_k0_kernel, dim3(blocks), dim3(256), 0, s, p);
    MX_HIP(hipGetLastError());
    return MX_OK;
  }
  MX_REQUIRE(a && b, MX_ERR_INVALID, "mx_gemm_f32: null operand");
  Scratch ws;
  if (p.splits > 1) {
    if (ws.alloc(size_t(partial_bytes(p)), s) == MX_OK) {
      p.ws = ws.as<float>();
    } else {  // no room for partials: one pass over K
      clear_error();
      MX_TRY(plan_gemm(d, a, b, bias, c, 0, &g));
    }
  }
  switch (g.tile) {
    case 0: MX_TRY(launch1_vec<TileTall>(p, g.ma, g.mb, s)); break;
    case 1: MX_TRY(launch1_vec<TileWide>(p, g.ma, g.mb, s)); break;
    case 2: MX_TRY(launch1<TileSq>(p, g.ma, g.mb, s)); break;
    default: MX_TRY(launch1<TileSmall>(p, g.ma, g.mb, s));
  }
  return p.splits > 1 ? launch_sum(p, s) : MX_OK;
}

int gemm_describe(const mx_gemm_desc* d, const float* a, const float* b, int64_t partials, std::string* name,
                  int64_t* bytes) {
  GemmPlan g;
  MX_TRY(plan_gemm(d, a, b, nullptr, nullptr, std::min(partials, kMaxSplitBytes), &g));
  *bytes = g.empty ? 0 : partial_bytes(g.p);
  if (g.empty) {
    *name = "none";
  } else if (d->k == 0) {
    *name = "gemm_k0_kernel";
  } else {
    const int kind = (d->bias_kind == MX_BIAS_NONE || d->beta == 0.f) ? MX_BIAS_NONE : d->bias_kind;
    *name = cat("gemm_kernel<", kTileNames[g.tile], ",", mode_name(g.ma), ",", mode_name(g.mb), ">", g.p.splits > 1 ? "+split" : "",
               kind == MX_BIAS_COL ? "+bias_col" : kind == MX_BIAS_MATRIX ? "+bias_matrix" : "",
               d->batch > 65535 ? "+batch_chunks" : "");
  }
  return MX_OK;
}

}  // namespace mx

extern "C" int mx_gemm_f32(const mx_gemm_desc* d, const float* a, const float* b, const float* bias,
                           float* c, void* stream) {
  MX_ABI_BEGIN
  return gemm_within(d, a, b, bias, c, kMaxSplitBytes, resolve_stream(stream));
  MX_ABI_END
}

extern "C" int mx_gemm_variant(const mx_gemm_desc* d, const float* a, const float* b, char* buf, size_t len) {
  MX_ABI_BEGIN
  MX_REQUIRE(buf || !len, MX_ERR_INVALID, "mx_gemm_variant: null buffer");
  std::string name;
  int64_t bytes = 0;
  MX_TRY(gemm_describe(d, a, b, kMaxSplitBytes, &name, &bytes));
  if (len) {
    std::strncpy(buf, name.c_str(), len - 1);
    buf[len - 1] = 0;
  }
  return MX_OK;
  MX_ABI_END
}
