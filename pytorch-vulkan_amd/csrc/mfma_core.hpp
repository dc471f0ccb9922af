// MFMA tile machinery for gfx950 (CDNA4), shared by the GEMM and the
// implicit-GEMM convolution kernels.
//
// A 256-thread workgroup (4 wave64) computes a BM x BN tile of C = A x B in
// FP32 accuracy.  Operands are staged through LDS in double-buffered BK slabs.
// On the way into LDS each FP32 value is split into three bf16 pieces, and the
// product runs as six bf16 MFMAs per 16 k (SplitStage, mma_slab_split); tiles
// whose result is not finite run again on FP32 MFMA (tile_product).  Each
// operand loader chooses its LDS layout: row-major with k contiguous or k-major
// with rows contiguous, whichever its global reads can fill with wide LDS
// stores (a row-contiguous operand written row-major would be a strided
// transpose).  Each wave owns a (BM/WAVES_M) x (BN/WAVES_N) sub-tile built from
// 32x32 blocks.  Inside a slab lane half h (lane / 32) handles k in [h*BK/2,
// (h+1)*BK/2) for both operands.
//
// Cfg::OCC is the register budget in waves per SIMD the kernels are compiled
// for (amdgpu_waves_per_eu): 2 keeps a 128 x 128 tile in 256 registers so two
// workgroups share a CU and hide each other's slab-load latency.
//
// Measured (MI355X), FP32 MFMA -> split: 8192 x 4096 x 4096 GEMM 2100-2195 ->
// 1275-1345 us (131 -> 211 TFLOP/s; a register-only loop of the bf16
// instruction sustains 1300-1870 TFLOP/s on random data, a sixth of which is
// 217-310), 1x1 conv 128 -> 512 at 64x28x28 forward + backward 213 -> 171 us.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mx {
namespace mfma {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;

template <int BM_, int BN_, int BK_, int WAVES_M_, int OCC_ = 2, bool DUAL_ = true,
          bool DEEP_ = BM_ * BN_ <= 64 * 64 && BK_ == 16>
struct Cfg {
  static constexpr int BM = BM_, BN = BN_, BK = BK_, OCC = OCC_;
  static constexpr int WAVES_M = WAVES_M_, WAVES_N = 4 / WAVES_M_;
  static constexpr int WTM = BM / WAVES_M, WTN = BN / WAVES_N;
  static constexpr int FM = WTM / 32, FN = WTN / 32;
  static constexpr int PAD = 4;
  static constexpr int LDK = BK + PAD;
  static constexpr int KH = BK / 2;
  // A stage holds either layout: [rows][BK + PAD] or [BK][rows + PAD].
  static constexpr int A_STAGE = (BM * LDK > BK * (BM + PAD)) ? BM * LDK : BK * (BM + PAD);
  static constexpr int B_STAGE = (BN * LDK > BK * (BN + PAD)) ? BN * LDK : BK * (BN + PAD);
  // The split product's stages: three bf16 planes per operand, no padding.
  static constexpr int A_SPLIT = 3 * BM * BK / 2, B_SPLIT = 3 * BN * BK / 2;
  static constexpr int SMEM_FLOATS = 2 * (A_STAGE + B_STAGE > A_SPLIT + B_SPLIT ? A_STAGE + B_STAGE : A_SPLIT + B_SPLIT);
  static constexpr bool DEEP = DEEP_;  // two register sets of operand slabs
  static constexpr bool DUAL = DUAL_ && FM * FN <= 4;  // small piece products in their own accumulators
  static_assert(WAVES_M * WAVES_N == 4, "4 waves per workgroup");
  static_assert(WTM % 32 == 0 && WTN % 32 == 0, "wave tile must be a multiple of 32");
  static_assert(BK % 8 == 0, "BK must be a multiple of 8");
};

// Qualifiers of a tile kernel compiled for configuration C.
#define MX_TILE_KERNEL(C) \
  __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(C::OCC, C::OCC)))

template <class C>
struct Acc {
  f32x16 v[C::FM][C::FN];
};

// Branch-free guarded loads: a masked element reads a zero from kZeroPage
// instead of its own address, so the loop has no control flow and no
// instruction touches a loaded value before it is stored to LDS one slab
// later.  (A branch or a select right after the load makes the compiler wait
// for every load in flight, prefetched slabs included.)
static __device__ float kZeroPage[1];  // zero-initialised, never written

__device__ __forceinline__ float load_or_zero(const float* p, bool ok) { return *(ok ? p : kZeroPage); }

// Raw buffer loads.  An operand tensor becomes one buffer resource (base,
// byte extent) held in scalar registers; a lane supplies a 32-bit byte offset
// and the per-element stride goes in the scalar offset, so a run of loads
// costs no vector ALU work beyond its first offset.  The hardware range check
// returns zero for an offset at or past the extent: a masked lane uses
// kOffNone, which needs every operand to end below 2^31 bytes (kBufMaxBytes,
// enforced by the host, which splits larger batches).
typedef int i32x4 __attribute__((ext_vector_type(4)));
extern "C" __device__ float mx_raw_buffer_load_f32(i32x4 rsrc, int voffset, int soffset, int aux) __asm(
    "llvm.amdgcn.raw.buffer.load.f32");
extern "C" __device__ f32x4 mx_raw_buffer_load_v4f32(i32x4 rsrc, int voffset, int soffset, int aux) __asm(
    "llvm.amdgcn.raw.buffer.load.v4f32");
typedef float f32x2 __attribute__((ext_vector_type(2)));
extern "C" __device__ f32x2 mx_raw_buffer_load_v2f32(i32x4 rsrc, int voffset, int soffset, int aux) __asm(
    "llvm.amdgcn.raw.buffer.load.v2f32");
// Vector-memory store through the same resource: a store at an offset past
// the extent (kOffNone) is dropped by the range check.
extern "C" __device__ void mx_raw_buffer_store_f32(float v, i32x4 rsrc, int voffset, int soffset, int aux) __asm(
    "llvm.amdgcn.raw.buffer.store.f32");

extern "C" __device__ void mx_raw_buffer_store_v2f32(f32x2 v, i32x4 rsrc, int voffset, int soffset, int aux) __asm(
    "llvm.amdgcn.raw.buffer.store.v2f32");

constexpr uint32_t kOffNone = 0x80000000u;
constexpr int64_t kBufMaxBytes = 0x7FFF0000;

// Word 3 = 0x00020000: 32-bit data format, raw (stride 0) addressing.
__device__ __forceinline__ i32x4 buffer_rsrc(const void* base, int64_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  i32x4 r;
  r.x = __builtin_amdgcn_readfirstlane(int(uint32_t(a)));
  r.y = __builtin_amdgcn_readfirstlane(int(uint32_t(a >> 32) & 0xFFFFu));
  r.z = __builtin_amdgcn_readfirstlane(int(uint32_t(bytes)));
  r.w = 0x00020000;
  return r;
}
__device__ __forceinline__ float bload(const i32x4& r, uint32_t voff, uint32_t soff) {
  return mx_raw_buffer_load_f32(r, int(voff), int(soff), 0);
}
__device__ __forceinline__ f32x4 bload4(const i32x4& r, uint32_t voff, uint32_t soff) {
  return mx_raw_buffer_load_v4f32(r, int(voff), int(soff), 0);
}
__device__ __forceinline__ f32x2 bload2(const i32x4& r, uint32_t voff, uint32_t soff) {
  return mx_raw_buffer_load_v2f32(r, int(voff), int(soff), 0);
}
__device__ __forceinline__ void bstore(float v, const i32x4& r, uint32_t voff, uint32_t soff) {
  mx_raw_buffer_store_f32(v, r, int(voff), int(soff), 0);
}

__device__ __forceinline__ void bstore2(f32x2 v, const i32x4& r, uint32_t voff, uint32_t soff) {
  mx_raw_buffer_store_v2f32(v, r, int(voff), int(soff), 0);
}

// n / d for n < 2^31 by multiply-high (m, l from fast_div(d) on the host):
// (umulhi(n, m) + n) >> l with l = ceil(log2 d), m = 2^32 (2^l - d) / d + 1.
struct FastDiv {
  uint32_t m;
  uint32_t l;
};
inline FastDiv fast_div(uint32_t d) {
  uint32_t l = 0;
  while ((uint64_t(1) << l) < d) ++l;
  const uint64_t m = ((uint64_t(1) << 32) * ((uint64_t(1) << l) - d)) / d + 1;
  return FastDiv{uint32_t(m), l};
}
__device__ __forceinline__ uint32_t fdiv(uint32_t n, FastDiv f) { return (__umulhi(n, f.m) + n) >> f.l; }

// ------------------------------------------------------------------ stages
// A stage is one operand's BK slab in LDS.  Loaders write it through one of
// four calls: row4 / run (consecutive k of one row), rows1 (one k of several
// rows, the lanes of a wave along k) or col4 (four consecutive rows of one k).

// FP32 stage: row-major [row][BK + 4], or k-major [k][ROWS + 4] for col4.
template <int ROWS, int BK>
struct F32Stage {
  static constexpr int LDK = BK + 4, LDR = ROWS + 4;
  float* p;
  __device__ __forceinline__ void row4(int row, int k, f32x4 v) const {
    *reinterpret_cast<f32x4*>(p + row * LDK + k) = v;
  }
  __device__ __forceinline__ void col4(int k, int row, f32x4 v) const {
    *reinterpret_cast<f32x4*>(p + k * LDR + row) = v;
  }
  template <int N>
  __device__ __forceinline__ void run(int row, int k, const float (&v)[N]) const {
    static_assert(N % 4 == 0, "runs are whole 16-byte chunks");
#pragma unroll
    for (int e = 0; e < N; e += 4) row4(row, k + e, f32x4{v[e], v[e + 1], v[e + 2], v[e + 3]});
  }
  template <int N>
  __device__ __forceinline__ void rows1(int row0, int step, int k, const float (&v)[N]) const {
#pragma unroll
    for (int q = 0; q < N; ++q) p[(row0 + q * step) * LDK + k] = v[q];
  }
};

// Split stage: each FP32 value as three bf16 pieces, 2^16 x = hi + mid + lo,
// every piece the round-to-nearest bf16 of what the pieces before it leave (3 x
// 8 significant bits: the sum is exact), in three planes.  bf16 ends at 2^-133
// and FP32 at 2^-149; the factor puts FP32's last bit on bf16's (conversions
// and both matrix instructions keep denormals), without it a value below 2^-110
// loses bits whatever the factor it meets.  It costs a multiplication per value
// (1x1 conv 128 -> 512 at 64x28x28 forward + backward 170 -> 173 us, linear
// 8192 x 4096 x 4096 4144 -> 4119; noting such values instead, three
// operations a pair, 178 and 4342); the sums carry 2^32 until they are stored.
// The split happens here, on the way into LDS, so each operand value is split
// once per workgroup and the product loop reads ready bf16 fragments; splitting
// the fragments after the LDS read costs every wave of a tile row or column the
// same work again (256x128 tile, 8192 x 4096 x 4096: 179 TFLOP/s that way).
// Row-major planes are [k / 8][row][8]: a lane's fragment (8 k of one row) is
// one 16-byte read and consecutive rows are contiguous; the row index of the
// later k groups has bits exchanged, so that 16 lanes writing 8 bytes each,
// BK / 4 lanes to a row, meet every bank once.  K-major planes are [k][ROWS]
// with the 32-byte quarters of a line rotated by k, so that the transposing
// read ds_read_b64_tr_b16, which takes 4 k x 16 rows per 16 lanes, does too.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

// What pieces are scaled by, and back from a product of two.
constexpr float kPieceScale = 0x1p16f, kProductScale = 0x1p-32f;

// hi / mid / lo pairs of two (scaled) values.  The residuals x - piece come from
// v_dot2c_f32_bf16 (x + piece0 * -1 + piece1 * 0), which reads the packed pair
// in place and is exact here; its constants stay in scalar registers because
// the compiler folds them to an inline constant that the packed operand reads
// differently.
struct Pieces2 {
  uint32_t hi, mid, lo;
};
__device__ __forceinline__ Pieces2 split2(float x0, float x1) {
  uint32_t sel0, sel1;  // (-1, 0) and (0, -1) as bf16 pairs
  asm("s_mov_b32 %0, 0xbf80" : "=s"(sel0));
  asm("s_mov_b32 %0, 0xbf800000" : "=s"(sel1));
  const bf16x2 d0 = __builtin_bit_cast(bf16x2, sel0), d1 = __builtin_bit_cast(bf16x2, sel1);
  const bf16x2 h = __builtin_convertvector((f32x2{x0, x1}), bf16x2);
  const float r0 = __builtin_amdgcn_fdot2_f32_bf16(h, d0, x0, false);
  const float r1 = __builtin_amdgcn_fdot2_f32_bf16(h, d1, x1, false);
  const bf16x2 m = __builtin_convertvector((f32x2{r0, r1}), bf16x2);
  const float q0 = __builtin_amdgcn_fdot2_f32_bf16(m, d0, r0, false);
  const float q1 = __builtin_amdgcn_fdot2_f32_bf16(m, d1, r1, false);
  const bf16x2 l = __builtin_convertvector((f32x2{q0, q1}), bf16x2);
  return {__builtin_bit_cast(uint32_t, h), __builtin_bit_cast(uint32_t, m), __builtin_bit_cast(uint32_t, l)};
}

template <int ROWS, int BK>
struct SplitStage {
  static constexpr int PLANE = ROWS * BK;  // bf16 elements of one plane
  static constexpr int FLOATS = 3 * PLANE / 2;
  float* p;
  float scale = kPieceScale;  // negative: the slab is summed negated
  __device__ __forceinline__ uint16_t* at(int elem) const { return reinterpret_cast<uint16_t*>(p) + elem; }
  __device__ __forceinline__ void put4(int elem, f32x4 v) const {
    v *= scale;
    const Pieces2 a = split2(v[0], v[1]), b = split2(v[2], v[3]);
    *reinterpret_cast<u32x2*>(at(elem)) = u32x2{a.hi, b.hi};
    *reinterpret_cast<u32x2*>(at(elem + PLANE)) = u32x2{a.mid, b.mid};
    *reinterpret_cast<u32x2*>(at(elem + 2 * PLANE)) = u32x2{a.lo, b.lo};
  }
  static __device__ __forceinline__ int row_elem(int row, int k) {
    return ((k >> 3) * ROWS + (row ^ ((k >> 3) * (64 / BK)))) * 8 + (k & 7);
  }
  static __device__ __forceinline__ int col_elem(int k, int row) { return k * ROWS + (row ^ ((k & 3) << 4)); }
  __device__ __forceinline__ void row4(int row, int k, f32x4 v) const { put4(row_elem(row, k), v); }
  __device__ __forceinline__ void col4(int k, int row, f32x4 v) const { put4(col_elem(k, row), v); }
  template <int N>
  __device__ __forceinline__ void run(int row, int k, const float (&v)[N]) const {
    if constexpr (N % 8 == 0) {
#pragma unroll
      for (int e = 0; e < N; e += 8) {
        u32x4 w[3];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const Pieces2 s = split2(v[e + 2 * q] * scale, v[e + 2 * q + 1] * scale);
          w[0][q] = s.hi, w[1][q] = s.mid, w[2][q] = s.lo;
        }
        const int elem = row_elem(row, k + e);
#pragma unroll
        for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x4*>(at(elem + q * PLANE)) = w[q];
      }
    } else {
#pragma unroll
      for (int e = 0; e < N; e += 4) row4(row, k + e, f32x4{v[e], v[e + 1], v[e + 2], v[e + 3]});
    }
  }
  // Lanes 2i and 2i + 1 hold k and k + 1 of the same rows: they trade values
  // so that each holds both k of every other row and writes whole pairs.
  template <int N>
  __device__ __forceinline__ void rows1(int row0, int step, int k, const float (&v)[N]) const {
    static_assert(N % 2 == 0, "rows are traded in pairs");
    const bool odd = k & 1;
#pragma unroll
    for (int q = 0; q < N; q += 2) {
      const float mine = odd ? v[q + 1] : v[q], give = odd ? v[q] : v[q + 1];
      const float got = __builtin_bit_cast(
          float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, give), 0xB1, 0xF, 0xF, true));  // lane ^ 1
      const Pieces2 s = split2((odd ? got : mine) * scale, (odd ? mine : got) * scale);
      const int elem = row_elem(row0 + (q + (odd ? 1 : 0)) * step, k & ~1);
      *reinterpret_cast<uint32_t*>(at(elem)) = s.hi;
      *reinterpret_cast<uint32_t*>(at(elem + PLANE)) = s.mid;
      *reinterpret_cast<uint32_t*>(at(elem + 2 * PLANE)) = s.lo;
    }
  }
};

struct Frag3 {
  bf16x8 hi, mid, lo;
};

// k0 .. k0 + 7 (k0 % 8 == 0, the same for a lane half) of rows row0 .. row0 +
// 31 of a split stage, row row0 + lane % 32 to each lane.
template <int ROWS, int BK, bool KMAJOR>
__device__ __forceinline__ Frag3 load_frag3(const float* stage, int row0, int k0, int lane) {
  using St = SplitStage<ROWS, BK>;
  const uint16_t* const base = reinterpret_cast<const uint16_t*>(stage);
  bf16x8 f[3];
#pragma unroll
  for (int pl = 0; pl < 3; ++pl) {
    if constexpr (KMAJOR) {
      // Each group of 16 lanes reads 4 k x 16 rows (8 bytes a lane: k c / 4,
      // rows 4 (c % 4)) and gets them transposed, 4 k of one row per lane.
      const int c = lane & 15, k = k0 + (c >> 2), row = row0 + (lane & 16) + 4 * (c & 3);
      s16x4 half[2];
#pragma unroll
      for (int q = 0; q < 2; ++q)
        half[q] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4*)(base + pl * St::PLANE + St::col_elem(k + 4 * q, row)));
      f[pl] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(half[0], half[1], 0, 1, 2, 3, 4, 5, 6, 7));
    } else {
      f[pl] = *reinterpret_cast<const bf16x8*>(base + pl * St::PLANE + St::row_elem(row0 + (lane & 31), k0));
    }
  }
  return {f[0], f[1], f[2]};
}

// The pieces of eight values already in registers.
__device__ __forceinline__ Frag3 split8(const f32x4& a, const f32x4& b) {
  u32x4 w[3];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const Pieces2 s = q < 2 ? split2(a[2 * q], a[2 * q + 1]) : split2(b[2 * q - 4], b[2 * q - 3]);
    w[0][q] = s.hi, w[1][q] = s.mid, w[2][q] = s.lo;
  }
  return {__builtin_bit_cast(bf16x8, w[0]), __builtin_bit_cast(bf16x8, w[1]), __builtin_bit_cast(bf16x8, w[2])};
}

template <class C>
__device__ __forceinline__ void acc_zero(Acc<C>& acc) {
#pragma unroll
  for (int i = 0; i < C::FM; ++i)
#pragma unroll
    for (int j = 0; j < C::FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc.v[i][j][r] = 0.f;
}

// Operand fragment for one 32-row block: the KH k values (this lane's half of
// the slab) of row `row` of a stage in either layout.
template <class C, int ROWS, bool KMAJOR>
__device__ __forceinline__ void load_frag(float (&f)[C::KH], const float* stage, int row, int h) {
  if constexpr (KMAJOR) {
    constexpr int LDR = ROWS + C::PAD;
    const float* src = stage + h * C::KH * LDR + row;
#pragma unroll
    for (int q = 0; q < C::KH; ++q) f[q] = src[q * LDR];
  } else {
    const float* src = stage + row * C::LDK + h * C::KH;
#pragma unroll
    for (int q = 0; q < C::KH; q += 4) {
      const f32x4 t = *reinterpret_cast<const f32x4*>(src + q);
      f[q + 0] = t[0];
      f[q + 1] = t[1];
      f[q + 2] = t[2];
      f[q + 3] = t[3];
    }
  }
}

// One BK slab: fragments from LDS, BK/2 MFMA steps per 32x32 block.
template <class C, bool KMA, bool KMB>
__device__ __forceinline__ void mma_slab(Acc<C>& acc, const float* As, const float* Bs, int wm,
                                         int wn, int lane) {
  const int r = lane & 31, h = lane >> 5;
  float a[C::FM][C::KH];
  float b[C::FN][C::KH];
#pragma unroll
  for (int i = 0; i < C::FM; ++i) load_frag<C, C::BM, KMA>(a[i], As, wm * C::WTM + i * 32 + r, h);
#pragma unroll
  for (int j = 0; j < C::FN; ++j) load_frag<C, C::BN, KMB>(b[j], Bs, wn * C::WTN + j * 32 + r, h);
  // All fragment reads are in flight before the first MFMA; the MFMAs then
  // wait only on their own operands (LDS returns in order).
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int s = 0; s < C::KH; ++s)
#pragma unroll
    for (int i = 0; i < C::FM; ++i)
#pragma unroll
      for (int j = 0; j < C::FN; ++j)
        acc.v[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][s], b[j][s], acc.v[i][j], 0, 0, 0);
}

// FP32 main loop over nk slabs: the products on v_mfma_f32_32x32x2f32.  It
// runs where the split loop's result is not finite (tile_product).
// Loaders expose load() (global -> registers, advancing their k cursor by
// one slab), skip() (one slab on without
// loading), store(stage) and KMAJOR (whether store() calls col4).  Two LDS
// stages; the loads past the last slab read zeros (the loaders mask k >= kmax)
// into a stage nobody reads.
template <class C, class LA, class LB>
__device__ __forceinline__ void mainloop_f32(Acc<C>& acc, LA& la, LB& lb, int nk, float* smem) {
  float* As = smem;
  float* Bs = smem + 2 * C::A_STAGE;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / C::WAVES_N, wn = wave % C::WAVES_N;
  acc_zero<C>(acc);
  if (nk <= 0) return;
  la.load();
  lb.load();
  la.store(F32Stage<C::BM, C::BK>{As});
  lb.store(F32Stage<C::BN, C::BK>{Bs});
  __syncthreads();
  for (int t = 0; t < nk; ++t) {
    const int cur = t & 1;
    la.load();
    lb.load();
    mma_slab<C, LA::KMAJOR, LB::KMAJOR>(acc, As + cur * C::A_STAGE, Bs + cur * C::B_STAGE, wm, wn, lane);
    la.store(F32Stage<C::BM, C::BK>{As + (cur ^ 1) * C::A_STAGE});
    lb.store(F32Stage<C::BN, C::BK>{Bs + (cur ^ 1) * C::B_STAGE});
    __syncthreads();
  }
}

// One slab of the split product: six of the nine piece products, smallest
// first (the dropped mid*lo, lo*mid and lo*lo are below 2^-24 of the
// product), on v_mfma_f32_32x32x16_bf16, which accumulates in FP32.
//
// Why: six bf16 MFMAs take 16 k of a 32x32 block through the matrix pipe in
// 6 x 32 cycles; eight v_mfma_f32_32x32x2f32 take 8 x 64.  The error is
// smaller as well, since 16 products enter one rounding: relative 2-norm
// against float64 on normal operands, K = 64 / 4096: 1.1e-7 / 0.98e-6 in one
// accumulator, 0.5e-7 / 0.40e-6 with the five small products in their own,
// 1.4e-7 / 1.15e-6 on the FP32 instruction.  The bf16 instruction rounds
// towards minus infinity below the accumulator's last bit.  Tiles with the
// registers for it (DUAL) keep the small products, which lie there, in their
// own accumulator: no bias.  In one accumulator it is -2.1e-7 of the result at
// K = 4096 and -8.4e-6 at 2^18, and the partial sums of a K split add it up
// (-6.4e-7 of a dW over 16 splits); there the middle half of the slabs is
// summed negated (mainloop_split): 0.1e-7, 3.8e-7 and 0.4e-7, and the error
// against float64 at K = 2^18 goes from 1.1e-5 to 0.64e-5 (FP32: 0.92e-5).
template <class C, bool KMA, bool KMB>
__device__ __forceinline__ void mma_slab_split(Acc<C>& acc, Acc<C>& small, const float* As, const float* Bs, int wm,
                                               int wn, int lane) {
  static_assert(C::KH % 8 == 0, "a lane half holds whole groups of 8 k");
  const int h = lane >> 5;
#pragma unroll
  for (int s = 0; s < C::KH; s += 8) {
    const int k0 = h * C::KH + s;
    Frag3 b[C::FN], a[C::FM];
    // The shorter side's fragments stay in registers while the longer side's
    // go by, each piece product over all blocks of one of those before the
    // next: consecutive MFMAs write different accumulators.
    Acc<C>& sm = C::DUAL ? small : acc;
#define MX_BLOCK(ACC, P, Q, I, J) \
  ACC.v[I][J] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[I].P, b[J].Q, ACC.v[I][J], 0, 0, 0);
#define MX_SPLIT_PRODUCT(ACC, P, Q)                                                             \
  if constexpr (C::FN <= C::FM) {                                                               \
    _Pragma("unroll") for (int j = 0; j < C::FN; ++j) MX_BLOCK(ACC, P, Q, o, j)                 \
  } else {                                                                                      \
    _Pragma("unroll") for (int i = 0; i < C::FM; ++i) MX_BLOCK(ACC, P, Q, i, o)                 \
  }
#pragma unroll
    for (int j = 0; j < C::FN; ++j) b[j] = load_frag3<C::BN, C::BK, KMB>(Bs, wn * C::WTN + j * 32, k0, lane);
#pragma unroll
    for (int i = 0; i < C::FM; ++i) a[i] = load_frag3<C::BM, C::BK, KMA>(As, wm * C::WTM + i * 32, k0, lane);
#pragma unroll
    for (int o = 0; o < (C::FN <= C::FM ? C::FM : C::FN); ++o) {
      MX_SPLIT_PRODUCT(sm, lo, hi)
      MX_SPLIT_PRODUCT(sm, hi, lo)
      MX_SPLIT_PRODUCT(sm, mid, mid)
      MX_SPLIT_PRODUCT(sm, mid, hi)
      MX_SPLIT_PRODUCT(sm, hi, mid)
      MX_SPLIT_PRODUCT(acc, hi, hi)
    }
#undef MX_BLOCK
#undef MX_SPLIT_PRODUCT
  }
}

// Instruction order of one slab of the split loop: the fragment reads of the
// first block row, then the products with the other rows' reads, the next
// slab's split and its LDS writes dealt between them, so the vector unit works
// under the matrix pipe instead of before and after it.
template <class C, bool KMA, bool KMB>
__device__ __forceinline__ void split_schedule() {
  constexpr int kMfma = 0x8, kValu = 0x2, kRead = 0x100, kWrite = 0x200;
  constexpr bool ROWS_GO_BY = C::FN <= C::FM;
  constexpr int IN = ROWS_GO_BY ? C::FN : C::FM, OUT = ROWS_GO_BY ? C::FM : C::FN;
  constexpr int RI = (ROWS_GO_BY ? KMB : KMA) ? 6 : 3, RO = (ROWS_GO_BY ? KMA : KMB) ? 6 : 3;  // LDS reads of a fragment
  constexpr int V = C::FM * C::FN >= 8 ? 3 : C::FM * C::FN >= 4 ? 4 : 8;
  __builtin_amdgcn_sched_group_barrier(kRead, RO + IN * RI, 0);
#pragma unroll
  for (int o = 0; o < OUT; ++o)
#pragma unroll
    for (int m = 0; m < 6 * IN; ++m) {
      __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
      if (m < RO && o + 1 < OUT) __builtin_amdgcn_sched_group_barrier(kRead, 1, 0);
      __builtin_amdgcn_sched_group_barrier(kValu, V, 0);
      __builtin_amdgcn_sched_group_barrier(kWrite, 1, 0);
    }
}

// Loaders that keep per-thread row sums (dBias) add those of a second copy.
template <class L>
__device__ __forceinline__ auto merge_row_sums(L& a, const L& b, int) -> decltype(a.bsum[0], void()) {
#pragma unroll
  for (int q = 0; q < int(sizeof(a.bsum) / sizeof(a.bsum[0])); ++q) a.bsum[q] += b.bsum[q];
}
template <class L>
__device__ __forceinline__ void merge_row_sums(L&, const L&, long) {}

// Split main loop over nk slabs, one barrier per slab: slab t + 1 is split and
// written to the other stage among slab t's products.  DEEP tiles (64x64x16;
// 128x128 in the convolution forward and input gradient, and in GEMMs that read
// both operands 16 bytes at a time) keep two register sets, even slabs in one
// and odd slabs in the other, so a load has two slabs of products to land; the
// others have registers for one set, or slabs long enough to cover a load.  The
// DEEP loop runs whole pairs of slabs (one exit keeps the accumulators in
// place): an odd count runs one more, of zeros, since loads past the last slab
// read zeros.
template <class C, bool PARTED, class LA, class LB>
__device__ __forceinline__ void mainloop_split(Acc<C>& acc, LA& la, LB& lb, int nk, float* smem) {
  float* const As = smem;
  float* const Bs = smem + 2 * C::A_SPLIT;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / C::WAVES_N, wn = wave % C::WAVES_N;
  acc_zero<C>(acc);
  if (nk <= 0) return;
  Acc<C> small;
  if constexpr (C::DUAL) acc_zero<C>(small);
  // Slab in stage `cur`; `na` / `nb` hold the next one and take the one `ahead`.
  const auto slab = [&](int cur, LA& na, LB& nb, float scale = kPieceScale) {
    mma_slab_split<C, LA::KMAJOR, LB::KMAJOR>(acc, small, As + cur * C::A_SPLIT, Bs + cur * C::B_SPLIT, wm, wn, lane);
    na.store(SplitStage<C::BM, C::BK>{As + (cur ^ 1) * C::A_SPLIT, C::BM < C::BN ? scale : kPieceScale});
    nb.store(SplitStage<C::BN, C::BK>{Bs + (cur ^ 1) * C::B_SPLIT, C::BM < C::BN ? kPieceScale : scale});
    if constexpr (C::KH == 8) split_schedule<C, LA::KMAJOR, LB::KMAJOR>();
    na.load();
    nb.load();
    __syncthreads();
  };
  la.load();
  lb.load();
  if constexpr (C::DEEP) {
    LA la1 = la;
    LB lb1 = lb;
    la1.load();
    lb1.load();
    la.store(SplitStage<C::BM, C::BK>{As});
    lb.store(SplitStage<C::BN, C::BK>{Bs});
    la.skip();
    lb.skip();
    la.load();
    lb.load();
    la.skip();
    lb.skip();
    la1.skip();
    lb1.skip();
    __syncthreads();
    for (int t = 0; t < nk; t += 2) {
      slab(0, la1, lb1);
      la1.skip();
      lb1.skip();
      slab(1, la, lb);
      la.skip();
      lb.skip();
    }
    merge_row_sums(la, la1, 0);
  } else {
    la.store(SplitStage<C::BM, C::BK>{As});
    lb.store(SplitStage<C::BN, C::BK>{Bs});
    la.load();
    lb.load();
    __syncthreads();
    if constexpr (C::DUAL) {
      for (int t = 0; t < nk; ++t) slab(t & 1, la, lb);
    } else {
      // The middle half of the slabs enters one operand negated and the
      // accumulators change sign at both ends, so the rounding bias of these
      // slabs meets that of the others.  A slab's bias goes as the sum's last
      // place: as the square root of the slabs so far for operands of both signs
      // (5% of the bias is left), as their number for operands of one (none).
      // Below 16 slabs it is 1e-8 of the result.
      const auto negate = [&]() {
#pragma unroll
        for (int i = 0; i < C::FM; ++i)
#pragma unroll
          for (int j = 0; j < C::FN; ++j) acc.v[i][j] = -acc.v[i][j];
      };
      if constexpr (PARTED) {
        // A loop for each part (the sign of slab t goes into its pieces one step
        // ahead): linear 8192 x 4096 x 4096 training 4252 -> 4156 us, 7886 x 3071
        // x 1753 1936 -> 1905.
        float sign = kPieceScale;
        for (int part = 0, t = 0, end = nk >= 16 ? nk / 4 : nk; part < 3; ++part) {
          for (; t < end; ++t) slab(t & 1, la, lb, t + 1 < end ? sign : -sign);
          if (part < 2) negate();
          sign = -sign;
          end = 2 * end < nk ? nk - end : nk;
        }
      } else {
        const int from = nk >= 16 ? nk / 4 : -1, to = nk - from;
        for (int t = 0; t < nk; ++t) {
          if (t == from || (t == to && from >= 0)) negate();
          slab(t & 1, la, lb, t + 1 >= from && t + 1 < to && from >= 0 ? -kPieceScale : kPieceScale);
        }
      }
    }
  }
  if constexpr (C::DUAL) {
#pragma unroll
    for (int i = 0; i < C::FM; ++i)
#pragma unroll
      for (int j = 0; j < C::FN; ++j) acc.v[i][j] += small.v[i][j];
  }
}

// True, for the whole workgroup, when some accumulator of a split product is
// not finite: an infinite operand, or one that the piece scale takes there
// (from 2^112 up), has no finite pieces, and neither inf - inf nor inf * 0 of
// pieces is what FP32 gives; sums from 2^96 up overflow with the scale.  Uses
// the first four words of smem, free after the main loop's last barrier.
template <class C>
__device__ __forceinline__ bool acc_not_finite(const Acc<C>& acc, float* smem) {
  uint32_t top = 0;
#pragma unroll
  for (int i = 0; i < C::FM; ++i)
#pragma unroll
    for (int j = 0; j < C::FN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) top = max(top, __float_as_uint(acc.v[i][j][v]) << 1);
  int* flags = reinterpret_cast<int*>(smem);
  const bool any = __any(top >= 0xFF000000u);
  if ((threadIdx.x & 63) == 0) flags[threadIdx.x >> 6] = any;
  __syncthreads();
  return (flags[0] | flags[1] | flags[2] | flags[3]) != 0;
}

// The tile's product over nk slabs: the split loop, and again in FP32 where
// its result is not finite.  init(la, lb) sets up fresh loaders; la ends as the
// loader of the loop that counted (its row sums are whole).  Returns what the
// caller multiplies the accumulators by as it stores them (a pass of its own
// over them spills).  PARTED: tiles in one accumulator walk the parts of their
// slabs in a loop each, for kernels with registers for it.
template <class C, bool PARTED = false, class LA, class LB, class Init>
__device__ __forceinline__ float tile_product(Acc<C>& acc, LA& la, LB& lb, int nk, float* smem, Init&& init) {
  init(la, lb);
  mainloop_split<C, PARTED>(acc, la, lb, nk, smem);
  float scale = kProductScale;
  if (acc_not_finite<C>(acc, smem)) {
    __syncthreads();  // every wave has read the flags before the stages are written
    init(la, lb);
    mainloop_f32<C>(acc, la, lb, nk, smem);
    scale = 1.f;
  }
  return scale;
}

// 32x32 output layout: lane l, register v -> row 8 * (v / 4) + 4 * (l / 32) + v % 4,
// column l % 32.
// This lane's column inside the tile for fragment column j.
template <class C>
__device__ __forceinline__ int acc_col(int j) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  return (wave % C::WAVES_N) * C::WTN + j * 32 + (lane & 31);
}

// This lane's row inside the tile for accumulator (i, v).
template <class C>
__device__ __forceinline__ int acc_row(int i, int v) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  return (wave / C::WAVES_N) * C::WTM + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
}

// Epilogue walk by rows: f(row, i, v) once per accumulator row of this lane;
// the callee loops over the FN fragment columns (acc.v[i][j][v]) with column
// data it computed once (acc_col).
template <class C, class F>
__device__ __forceinline__ void for_each_acc_row(F&& f) {
#pragma unroll
  for (int i = 0; i < C::FM; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) f(acc_row<C>(i, v), i, v);
}

// Rows of this lane's accumulators as a wave-uniform part (block_row, in
// scalar registers) plus 4 * (lane / 32).
template <class C>
__device__ __forceinline__ int wave_row0() {
  return __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6) / C::WAVES_N * C::WTM);
}
__device__ __forceinline__ int lane_row() { return 4 * int((threadIdx.x & 63) >> 5); }
__device__ __forceinline__ constexpr int block_row(int i, int v) { return i * 32 + 8 * (v >> 2) + (v & 3); }

// Stores a tile through a buffer resource: element (row, fragment column j)
// at byte offset row * pitch4 + col[j], rows counted from row0 and valid below
// `rows`.  The row's offset is wave-uniform but for the lane half, so it goes
// in the store's scalar offset and an element costs its value and the store;
// whole tiles skip the row test.  col[j] is kOffNone for a masked column (the
// range check drops the store); a masked row also takes a scalar offset
// inside the buffer.  value(i, j, v) gives the element.
template <class C, class F>
__device__ __forceinline__ void store_tile(const i32x4& ro, const uint32_t (&col)[C::FN], uint32_t pitch4, int row0,
                                           int rows, F&& value) {
  const int first = row0 + wave_row0<C>();
  uint32_t at[C::FN];
#pragma unroll
  for (int j = 0; j < C::FN; ++j)
    at[j] = col[j] == kOffNone ? kOffNone : col[j] + uint32_t(lane_row()) * pitch4;
  if (row0 + C::BM <= rows) {
#pragma unroll
    for (int i = 0; i < C::FM; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v)
#pragma unroll
        for (int j = 0; j < C::FN; ++j) {
          bstore(value(i, j, v), ro, at[j], uint32_t(first + block_row(i, v)) * pitch4);
          if (j + 1 == C::FN) __builtin_amdgcn_sched_barrier(0);  // keeps few values live
        }
  } else {
#pragma unroll
    for (int i = 0; i < C::FM; ++i)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int r = first + block_row(i, v);
        const bool ok = r + lane_row() < rows;
#pragma unroll
        for (int j = 0; j < C::FN; ++j)
          bstore(value(i, j, v), ro, ok ? at[j] : kOffNone, uint32_t(min(r, rows - 1)) * pitch4);
        __builtin_amdgcn_sched_barrier(0);
      }
  }
}

// ---------------------------------------------------------------- loaders
// Operand element (row, k) = base[row * s_row + k * s_k] for rows
// [row0, row0 + ROWS) clipped to R and k < kmax (zero outside).
enum class Mode : int {
  KVEC = 0,     // k contiguous, 16-byte aligned: float4 along k
  RVEC = 1,     // rows contiguous, 16-byte aligned: float4 along rows
  KSCALAR = 2,  // consecutive lanes -> consecutive k
  RSCALAR = 3   // consecutive lanes -> consecutive rows
};

template <int ROWS, int BK, Mode MODE>
struct StridedLoader;

// The 16-byte modes read through a buffer resource whose base follows the k
// cursor (a scalar add per slab), so a lane keeps one 32-bit byte offset per
// row pass and needs no address arithmetic.  Strides are in [0, kVecStrideMax]:
// the offsets of one tile's slab stay below 2^31 whatever the operand's size.
constexpr int64_t kVecStrideMax = (int64_t(1) << 31) / 4 / 256 - 16;

struct SlabBase {
  uint64_t at;
  __device__ __forceinline__ i32x4 rsrc() const {
    return buffer_rsrc(reinterpret_cast<const void*>(at), kBufMaxBytes);
  }
};

template <int ROWS, int BK>
struct StridedLoader<ROWS, BK, Mode::KVEC> {
  static constexpr bool KMAJOR = false;
  static constexpr int TPR = BK / 4;                 // threads per row
  static constexpr int RPP = kThreads / TPR;         // rows per pass
  static constexpr int PASSES = ROWS / RPP;
  static_assert(PASSES >= 1 && ROWS % RPP == 0, "KVEC tiling");
  f32x4 v[PASSES];
  SlabBase base;
  uint32_t off[PASSES];
  int k, kmax, kq;
  __device__ __forceinline__ void init(const float* p0, int64_t s_row, int64_t /*s_k*/, int row0, int R, int k0,
                                       int kmax_) {
    const int tid = threadIdx.x;
    kq = tid % TPR;
    k = k0;
    kmax = kmax_;
    base.at = reinterpret_cast<uint64_t>(p0 + int64_t(row0) * s_row + k0);
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
      const int r = tid / TPR + p * RPP;
      off[p] = row0 + r < R ? (uint32_t(r) * uint32_t(s_row) + 4 * kq) * 4u : kOffNone;
    }
  }
  __device__ __forceinline__ void load() {
    const bool kin = k + 4 * kq < kmax;
    const i32x4 rs = base.rsrc();
#pragma unroll
    for (int p = 0; p < PASSES; ++p) v[p] = bload4(rs, kin ? off[p] : kOffNone, 0);
    skip();
  }
  __device__ __forceinline__ void skip() {
    k += BK;
    base.at += BK * 4;
  }
  template <class S>
  __device__ __forceinline__ void store(S st) const {
#pragma unroll
    for (int p = 0; p < PASSES; ++p) st.row4(threadIdx.x / TPR + p * RPP, 4 * kq, v[p]);
  }
};

template <int ROWS, int BK>
struct StridedLoader<ROWS, BK, Mode::RVEC> {
  // Rows are contiguous in memory: each thread reads 4 rows at one k with a
  // 16-byte load and writes them unchanged into the k-major stage.
  static constexpr bool KMAJOR = true;
  static constexpr int TPK = ROWS / 4;               // threads per k
  static constexpr int KPP = kThreads / TPK;         // k per pass
  static constexpr int PASSES = BK / KPP;
  static_assert(PASSES >= 1 && BK % KPP == 0, "RVEC tiling");
  f32x4 v[PASSES];
  SlabBase base;
  uint64_t slab;        // bytes from one slab to the next
  uint32_t off, pass4;  // lane's byte offset, bytes between passes
  int k, kmax, kk;
  __device__ __forceinline__ void init(const float* p0, int64_t /*s_row*/, int64_t s_k, int row0, int R, int k0,
                                       int kmax_) {
    const int tid = threadIdx.x;
    const int rq = tid % TPK;
    kk = tid / TPK;
    base.at = reinterpret_cast<uint64_t>(p0 + row0 + int64_t(k0) * s_k);
    off = row0 + 4 * rq < R ? (uint32_t(kk) * uint32_t(s_k) + 4 * rq) * 4u : kOffNone;
    pass4 = uint32_t(KPP) * uint32_t(s_k) * 4u;
    slab = uint64_t(s_k) * (BK * 4);
    k = k0;
    kmax = kmax_;
  }
  __device__ __forceinline__ void load() {
    const i32x4 rs = base.rsrc();
#pragma unroll
    for (int p = 0; p < PASSES; ++p)
      v[p] = bload4(rs, k + kk + p * KPP < kmax ? off : kOffNone, uint32_t(p) * pass4);
    skip();
  }
  __device__ __forceinline__ void skip() {
    k += BK;
    base.at += slab;
  }
  template <class S>
  __device__ __forceinline__ void store(S st) const {
#pragma unroll
    for (int p = 0; p < PASSES; ++p) st.col4(kk + p * KPP, 4 * (threadIdx.x % TPK), v[p]);
  }
};

template <int ROWS, int BK>
struct StridedLoader<ROWS, BK, Mode::KSCALAR> {
  static constexpr bool KMAJOR = false;
  static constexpr int RPP = kThreads / BK;
  static constexpr int PASSES = ROWS / RPP;
  static_assert(PASSES >= 1 && ROWS % RPP == 0, "KSCALAR tiling");
  float v[PASSES];
  const float* ptr[PASSES];
  bool ok[PASSES];
  int64_t s_k;
  int k, kmax, kk;
  __device__ __forceinline__ void init(const float* base, int64_t s_row, int64_t s_k_, int row0, int R, int k0, int kmax_) {
    const int tid = threadIdx.x;
    kk = tid % BK;
    s_k = s_k_;
    k = k0;
    kmax = kmax_;
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
      const int row = row0 + tid / BK + p * RPP;
      ok[p] = row < R;
      ptr[p] = base + (ok[p] ? int64_t(row) * s_row : 0);
    }
  }
  __device__ __forceinline__ void load() {
    const int kx = k + kk;
    const bool kin = kx < kmax;
    const int64_t off = int64_t(kx) * s_k;
#pragma unroll
    for (int p = 0; p < PASSES; ++p) v[p] = load_or_zero(ptr[p] + off, ok[p] && kin);
    skip();
  }
  __device__ __forceinline__ void skip() { k += BK; }
  template <class S>
  __device__ __forceinline__ void store(S st) const {
    st.template rows1<PASSES>(threadIdx.x / BK, RPP, kk, v);
  }
};

template <int ROWS, int BK>
struct StridedLoader<ROWS, BK, Mode::RSCALAR> {
  static constexpr bool KMAJOR = false;
  static_assert(kThreads % ROWS == 0 || ROWS % kThreads == 0, "RSCALAR tiling");
  static constexpr int EPT = ROWS * BK / kThreads;   // consecutive k per thread
  static_assert(ROWS <= kThreads, "RSCALAR expects ROWS <= 256");
  float v[EPT];
  const float* ptr;
  int64_t s_k;
  bool ok;
  int k, kmax, ks;
  __device__ __forceinline__ void init(const float* base, int64_t s_row, int64_t s_k_, int row0, int R, int k0, int kmax_) {
    const int tid = threadIdx.x;
    const int r = tid % ROWS;
    ks = (tid / ROWS) * EPT;
    const int row = row0 + r;
    ok = row < R;
    ptr = base + (ok ? int64_t(row) * s_row : 0);
    s_k = s_k_;
    k = k0;
    kmax = kmax_;
  }
  __device__ __forceinline__ void load() {
#pragma unroll
    for (int e = 0; e < EPT; ++e) {
      const int kx = k + ks + e;
      v[e] = load_or_zero(ptr + int64_t(kx) * s_k, ok && kx < kmax);
    }
    skip();
  }
  __device__ __forceinline__ void skip() { k += BK; }
  template <class S>
  __device__ __forceinline__ void store(S st) const {
    st.template run<EPT>(threadIdx.x % ROWS, ks, v);
  }
};

// The same operand views through a buffer resource over [base, base + bytes)
// (bytes < kBufMaxBytes, 32-bit element strides): per-lane byte offsets are
// fixed at init, the k cursor moves the scalar offset, and masked elements
// read zero through the range check.  Used for convolution weights; the
// general GEMM keeps StridedLoader (its operands may exceed the 2^31 range).
template <int ROWS, int BK, Mode MODE>
struct BufStridedLoader;

template <int ROWS, int BK>
struct BufStridedLoader<ROWS, BK, Mode::KVEC> {
  static constexpr bool KMAJOR = false;
  static constexpr int TPR = BK / 4;
  static constexpr int RPP = kThreads / TPR;
  static constexpr int PASSES = ROWS / RPP;
  static_assert(PASSES >= 1 && ROWS % RPP == 0, "KVEC tiling");
  f32x4 v[PASSES];
  i32x4 rs;
  uint32_t off[PASSES];
  int k, kmax, kq;
  __device__ __forceinline__ void init(const float* base, int64_t bytes, int s_row, int /*s_k*/, int row0, int R,
                                       int k0, int kmax_) {
    const int tid = threadIdx.x;
    kq = tid % TPR;
    rs = buffer_rsrc(base, bytes);
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
      const int row = row0 + tid / TPR + p * RPP;
      off[p] = row < R ? uint32_t(row * s_row + 4 * kq) * 4u : kOffNone;
    }
    k = k0;
    kmax = kmax_;
  }
  __device__ __forceinline__ void load() {
    const bool kin = k + 4 * kq < kmax;
#pragma unroll
    for (int p = 0; p < PASSES; ++p) v[p] = bload4(rs, kin ? off[p] : kOffNone, uint32_t(k) * 4u);
    skip();
  }
  __device__ __forceinline__ void skip() { k += BK; }
  template <class S>
  __device__ __forceinline__ void store(S st) const {
#pragma unroll
    for (int p = 0; p < PASSES; ++p) st.row4(threadIdx.x / TPR + p * RPP, 4 * kq, v[p]);
  }
};

template <int ROWS, int BK>
struct BufStridedLoader<ROWS, BK, Mode::RVEC> {
  static constexpr bool KMAJOR = true;
  static constexpr int TPK = ROWS / 4;
  static constexpr int KPP = kThreads / TPK;
  static constexpr int PASSES = BK / KPP;
  static_assert(PASSES >= 1 && BK % KPP == 0, "RVEC tiling");
  f32x4 v[PASSES];
  i32x4 rs;
  uint32_t off, sk4;
  int k, kmax, kk;
  __device__ __forceinline__ void init(const float* base, int64_t bytes, int /*s_row*/, int s_k, int row0, int R,
                                       int k0, int kmax_) {
    const int tid = threadIdx.x;
    kk = tid / TPK;
    const int row = row0 + 4 * (tid % TPK);
    rs = buffer_rsrc(base, bytes);
    off = row < R ? uint32_t(row + kk * s_k) * 4u : kOffNone;
    sk4 = uint32_t(s_k) * 4u;
    k = k0;
    kmax = kmax_;
  }
  __device__ __forceinline__ void load() {
#pragma unroll
    for (int p = 0; p < PASSES; ++p)
      v[p] = bload4(rs, k + kk + p * KPP < kmax ? off : kOffNone, uint32_t(k + p * KPP) * sk4);
    skip();
  }
  __device__ __forceinline__ void skip() { k += BK; }
  template <class S>
  __device__ __forceinline__ void store(S st) const {
#pragma unroll
    for (int p = 0; p < PASSES; ++p) st.col4(kk + p * KPP, 4 * (threadIdx.x % TPK), v[p]);
  }
};

template <int ROWS, int BK>
struct BufStridedLoader<ROWS, BK, Mode::RSCALAR> {
  static constexpr bool KMAJOR = false;
  static_assert(ROWS % 64 == 0 && ROWS <= kThreads, "RSCALAR tiling");
  static constexpr int EPT = ROWS * BK / kThreads;  // consecutive k per thread (wave-uniform run)
  float v[EPT];
  i32x4 rs;
  uint32_t off, sk4;
  int k, kmax, ks;
  __device__ __forceinline__ void init(const float* base, int64_t bytes, int s_row, int s_k, int row0, int R, int k0,
                                       int kmax_) {
    const int tid = threadIdx.x;
    ks = __builtin_amdgcn_readfirstlane((tid / ROWS) * EPT);
    const int row = row0 + tid % ROWS;
    rs = buffer_rsrc(base, bytes);
    off = row < R ? uint32_t(row * s_row) * 4u : kOffNone;
    sk4 = uint32_t(s_k) * 4u;
    k = k0;
    kmax = kmax_;
  }
  __device__ __forceinline__ void load() {
#pragma unroll
    for (int e = 0; e < EPT; ++e) {
      const int kx = k + ks + e;  // wave-uniform
      v[e] = bload(rs, kx < kmax ? off : kOffNone, uint32_t(kx) * sk4);
    }
    skip();
  }
  __device__ __forceinline__ void skip() { k += BK; }
  template <class S>
  __device__ __forceinline__ void store(S st) const {
    st.template run<EPT>(threadIdx.x % ROWS, ks, v);
  }
};

// Bijective block remap so that consecutive logical tiles land on the same
// XCD (hardware dispatches workgroup b to XCD b % 8): tiles that share an
// operand panel then share that XCD's L2.
__device__ __forceinline__ int xcd_remap(int b, int n) {
  constexpr int X = 8;
  if (n < 2 * X) return b;
  const int per = n / X, rem = n % X;
  const int xcd = b % X, idx = b / X;
  return xcd < rem ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
}

// Logical tile id -> (tile_m, tile_n) in GROUP_M-row bands (raster order
// within a band) so a wave of resident tiles reuses A and B panels.
__device__ __forceinline__ void tile_coords(int t, int tiles_m, int tiles_n, int& tm, int& tn) {
  constexpr int GROUP_M = 8;
  const int band = GROUP_M * tiles_n;
  const int g = t / band;
  const int first_m = g * GROUP_M;
  const int gm = min(tiles_m - first_m, GROUP_M);
  const int in = t % band;
  tm = first_m + in % gm;
  tn = in / gm;
}

}  // namespace mfma
}  // namespace mx
