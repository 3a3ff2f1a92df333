// fp32 contractions on the bf16 matrix cores: C[m][n] = epi(sum_k A[m][k] B[n][k])
// for the executor's fp32 ops (matmul wgsl-ops.js:477-556, gemm :821-897, convMM
// :584-698) and the fp32 linears.
//
// Every fp32 operand value is scaled by 2^16 and split, as its tile is staged,
// into three bf16 parts x = h + m + l (each the rounding of what the parts
// before it left; bf16 reaches down to 2^-133, the scaled value's last bit to
// 2^-133 or above, so the sum is exact, subnormals included; the method is
// Henry, Tang and Heinecke's, ARITH 2019), and a product is the six MFMA products of parts whose
// weight is above 2^-24: h h, h m, m h, m m, h l, l h.  The three products
// left out are below the rounding of one fp32 product.  The matrix cores do
// bf16 at 16 times the fp32 MFMA rate, so six products still leave 2.7 times
// the fp32 MFMA's peak, and one bf16 MFMA sums 32 products where the fp32 one
// sums 4: fewer roundings of the running sum, a smaller error.  The sums are
// scaled back, exactly, before the epilogue.
//
// Infinities and NaNs have no such split (inf - inf).  They, and values and
// sums that overflow scaled (from 2^112 and 2^96 on), leave a non-finite sum in
// every output they reach; a workgroup that finds one in its tile computes the tile
// again with the fp32 MFMA on the unsplit values, so those results are the
// fp32 instruction's own.
//
// Measured against the fp32 MFMA kernel it replaces (one tile of 128 x 128 or
// 64 x 64, no split-K, gathered conv loads with divisions per element):
// conv 3x3 1280 -> 1280 at 16 x 16 969 -> 56 us, linear 2048 x 5120 x 1280
// 460 -> 165 us and 2048 x 1280 x 5120 470 -> 155 us (170 TFLOP/s of fp32
// work, a PFLOP/s of bf16; the fp32 MFMA's peak is 157), batched 5 x 2304 x
// 2304 x 64 90 -> 53 us.  Error against 64 bits (relative 2-norm): 1.4e-6 ->
// 2.5e-7, 8.0e-7 -> 4.9e-7 over both linears, and between 0.3 and 0.9 times the
// old kernel's on every shape tried.  The linears' times are those before the
// scaling, which costs 1 to 3 % (2048 x 5120 x 1280 168.1 -> 171.5 us, 2048 x
// 1280 x 5120 154.4 -> 157.5, 512 -> 512 at 64 x 64 113.7 -> 117.0 in turn on one
// card) and without which operands below 2^-110 lost bits: a relative error of
// 2e-6 at 2^-116, 2e-3 at 2^-126 and 1 at 2^-135, now 1e-7 throughout.  What
// bounds it is the split-and-store phase (6.5 VALU operations per staged fp32
// value, 8.9 VALU instructions with addresses and epilogue) that one workgroup's
// MFMAs hide from another only in part: the MFMAs are busy 41 to 49 % of the
// clocks, the LDS 37 to 48 %.
#include <cstdlib>
#include <type_traits>

#include "k_gemm_families.h"
#include "k_gemm_kernel.h"

namespace di {

namespace {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kOut = 0x80000000u;  // a buffer offset past every extent: reads 0

// fp32 operands are split times 2^16: the last bit of the smallest subnormal,
// 2^-149, is then bf16's own smallest step, 2^-133, and every part of every
// fp32 value is held.  (fp16-resident B: two parts hold a value of any size.)
template <typename T>
constexpr float kScale = sizeof(T) == 4 ? 0x1p16f : 1.0f;

// Two values of a T operand, scaled -> their h, m and l parts, each a packed bf16 pair.
template <typename T>
__device__ __forceinline__ void split2(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
  a *= kScale<T>;
  b *= kScale<T>;
  h = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
  const float ra = a - __uint_as_float(h << 16), rb = b - __uint_as_float(h & 0xffff0000u);
  m = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{ra, rb}, bf16x2));
  const float sa = ra - __uint_as_float(m << 16), sb = rb - __uint_as_float(m & 0xffff0000u);
  l = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{sa, sb}, bf16x2));
}

// One operand tile of ROWS rows x 32 k as a thread holds it between its
// global loads and its LDS stores: ROWS / 8 values.
//  * row-major sources (k contiguous): eight lanes read one row's 128 bytes,
//    four values each, rows 32 apart;
//  * k-major sources (rows contiguous: a [K][N] matrix, an NCHW image's
//    pixels): a lane keeps one row, a wavefront reads 64 neighbouring rows
//    of one k, KC consecutive k per thread.
template <int ROWS>
struct F32Tile {
  static constexpr int V = ROWS / 8;    // values per thread
  static constexpr int NR = ROWS / 32;  // rows per thread, row-major
  static constexpr int KC = V;          // k per thread, k-major
  float v[V];
};

// Byte offset of 16-byte chunk c (8 k) of a row in one part's plane of 64-byte
// rows: the chunk position is XORed with (row >> 2) & 3, which spreads sixteen
// rows of one chunk (a fragment read, a k-major store) over all 64 banks.  (A
// third of the LDS's active clocks are bank conflicts all the same.)
__device__ __forceinline__ uint32_t plane_at(uint32_t row, uint32_t c) {
  return row * 64 + ((c ^ ((row >> 2) & 3)) << 4);
}

template <typename T, int ROWS>
__device__ __forceinline__ void store_split(char* s, const F32Tile<ROWS>& t, bool kmajor) {
  constexpr uint32_t P = ROWS * 64;  // bytes of one plane
  const uint32_t tid = threadIdx.x;
  if (!kmajor) {
#pragma unroll
    for (int i = 0; i < F32Tile<ROWS>::NR; i++) {
      const uint32_t row = (tid >> 3) + 32 * i, kq = tid & 7;
      const uint32_t at = plane_at(row, kq >> 1) + (kq & 1) * 8;
      u32x2 h, m, l;
#pragma unroll
      for (int j = 0; j < 2; j++) {
        uint32_t a, b, c;
        split2<T>(t.v[4 * i + 2 * j], t.v[4 * i + 2 * j + 1], a, b, c);
        h[j] = a;
        m[j] = b;
        l[j] = c;
      }
      *(u32x2*)(s + at) = h;
      *(u32x2*)(s + P + at) = m;
      *(u32x2*)(s + 2 * P + at) = l;
    }
  } else {
    const uint32_t row = tid % ROWS, kg = tid / ROWS;
#pragma unroll
    for (int i = 0; i < F32Tile<ROWS>::KC / 8; i++) {
      const uint32_t at = plane_at(row, kg * (F32Tile<ROWS>::KC / 8) + i);
      u32x4 h, m, l;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        uint32_t a, b, c;
        split2<T>(t.v[8 * i + 2 * j], t.v[8 * i + 2 * j + 1], a, b, c);
        h[j] = a;
        m[j] = b;
        l[j] = c;
      }
      *(u32x4*)(s + at) = h;
      *(u32x4*)(s + P + at) = m;
      *(u32x4*)(s + 2 * P + at) = l;
    }
  }
}

// The unsplit tile for the fp32 MFMA: rows of 36 floats.
constexpr uint32_t kRawLd = 36;
template <int ROWS>
__device__ __forceinline__ void store_raw(float* s, const F32Tile<ROWS>& t, bool kmajor) {
  const uint32_t tid = threadIdx.x;
  if (!kmajor) {
#pragma unroll
    for (int i = 0; i < F32Tile<ROWS>::NR; i++)
#pragma unroll
      for (int j = 0; j < 4; j++)
        s[((tid >> 3) + 32 * i) * kRawLd + (tid & 7) * 4 + j] = t.v[4 * i + j];
  } else {
#pragma unroll
    for (int j = 0; j < F32Tile<ROWS>::KC; j++)
      s[(tid % ROWS) * kRawLd + (tid / ROWS) * F32Tile<ROWS>::KC + j] = t.v[j];
  }
}

__device__ __forceinline__ float buf_f32(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t soff = 0) {
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off, soff, 0));
}
template <typename TB>
__device__ __forceinline__ float buf_elem(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t soff) {
  if constexpr (sizeof(TB) == 4) {
    return buf_f32(r, off, soff);
  } else {
    const uint16_t u = __builtin_amdgcn_raw_buffer_load_b16(r, off, soff, 0);
    return (float)__builtin_bit_cast(f16, u);
  }
}

// Bytes from element offset `at` to the end of an operand of n elements, as a
// buffer extent.
__device__ __forceinline__ uint32_t extent_from(uint64_t n, uint64_t at, uint32_t es) {
  const uint64_t b = (n - at) * es;
  return b < 0x7fff0000ull ? (uint32_t)b : 0x7fff0000u;
}

// Row-major operand: ROWS rows from row r0 of [R][ld], k in [k_begin, k_end).
template <int ROWS, typename TB>
struct RowMajor {
  __amdgpu_buffer_rsrc_t rs;
  uint32_t off[F32Tile<ROWS>::NR];
  bool vec;
  uint32_t k_end;
  __device__ RowMajor(const void* p, uint64_t ld, uint32_t R, uint32_t K, uint32_t r0, bool vec_,
                      uint32_t k_end_)
      : vec(vec_), k_end(k_end_) {
    const uint64_t total = (uint64_t)(R - 1) * ld + K, at = (uint64_t)r0 * ld;
    rs = make_rsrc((const TB*)p + at, extent_from(total, at, sizeof(TB)));
#pragma unroll
    for (int i = 0; i < F32Tile<ROWS>::NR; i++) {
      const uint32_t row = (threadIdx.x >> 3) + 32 * i;
      off[i] = r0 + row < R ? row * (uint32_t)ld * (uint32_t)sizeof(TB) : kOut;
    }
  }
  __device__ __forceinline__ void load(uint32_t kb, F32Tile<ROWS>& t) {
    const uint32_t k = kb + (threadIdx.x & 7) * 4;
    if (vec && kb + 32 <= k_end) {  // uniform
#pragma unroll
      for (int i = 0; i < F32Tile<ROWS>::NR; i++) {
        if constexpr (sizeof(TB) == 4) {
          const f32x4 x = buf_load16s<f32x4>(rs, off[i] + (threadIdx.x & 7) * 16, kb * 4);
#pragma unroll
          for (int j = 0; j < 4; j++) t.v[4 * i + j] = x[j];
        } else {
          const f16x4 x = __builtin_bit_cast(
              f16x4, __builtin_amdgcn_raw_buffer_load_b64(rs, off[i] + (threadIdx.x & 7) * 8,
                                                          kb * 2, 0));
#pragma unroll
          for (int j = 0; j < 4; j++) t.v[4 * i + j] = (float)x[j];
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < F32Tile<ROWS>::NR; i++)
#pragma unroll
        for (int j = 0; j < 4; j++)
          t.v[4 * i + j] = buf_elem<TB>(
              rs, k + j < k_end ? off[i] + (k + j) * (uint32_t)sizeof(TB) : kOut, 0);
    }
  }
};

// [K][N] operand (n contiguous): columns n0 + lane.
template <int ROWS, typename TB>
struct KMajor {
  const TB* base;
  uint64_t ld, total;
  uint32_t off, k_end, kg;
  __device__ KMajor(const void* p, uint64_t ld_, uint32_t N, uint32_t K, uint32_t n0,
                    uint32_t k_end_)
      : base((const TB*)p), ld(ld_), total((uint64_t)(K - 1) * ld_ + N), k_end(k_end_) {
    const uint32_t n = n0 + threadIdx.x % ROWS;
    off = n < N ? n * (uint32_t)sizeof(TB) : kOut;
    kg = __builtin_amdgcn_readfirstlane(threadIdx.x / ROWS);
  }
  __device__ __forceinline__ void load(uint32_t kb, F32Tile<ROWS>& t) {
    const uint32_t k0 = min(kb + kg * F32Tile<ROWS>::KC, k_end - 1);
    const uint64_t at = (uint64_t)k0 * ld;
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(base + at, extent_from(total, at, sizeof(TB)));
    const uint32_t left = k_end - kb > kg * F32Tile<ROWS>::KC ? k_end - kb - kg * F32Tile<ROWS>::KC : 0;
    if (left >= (uint32_t)F32Tile<ROWS>::KC) {
#pragma unroll
      for (int j = 0; j < F32Tile<ROWS>::KC; j++)
        t.v[j] = buf_elem<TB>(rs, off, j * (uint32_t)ld * (uint32_t)sizeof(TB));
    } else {
#pragma unroll
      for (int j = 0; j < F32Tile<ROWS>::KC; j++)
        t.v[j] = (uint32_t)j < left
                     ? buf_elem<TB>(rs, off, j * (uint32_t)ld * (uint32_t)sizeof(TB))
                     : 0.0f;
    }
  }
};

// Implicit im2col of an NCHW image, k = (ci, ky, kx): output pixels m0 + lane.
// The window of a k is uniform over the lanes, so a load needs no arithmetic
// where the lane's offset of each tap (out of range outside the image) is kept
// in a register and the channel goes into the scalar offset: 3x3 kernels,
// where a run's first tap selects one of nine bodies with compile-time taps,
// and 1x1 kernels.  Other kernels, upsampled inputs and the ragged last
// stage compute each offset.
template <int ROWS>
struct ConvNchw {
  static constexpr int KC = F32Tile<ROWS>::KC;
  __amdgpu_buffer_rsrc_t rs;
  uint32_t tap[9];         // lane: byte offset of each tap of a 3x3 (tap[0]: 1x1) window
  int32_t base, iy0, ix0;  // lane: its image's element offset, its window's corner
  uint32_t Hi, Wi, W, HW, ks, upsh, k_end;
  int mode;  // 3: 3x3, 1: 1x1, 0: computed
  bool ok;
  uint32_t k;  // uniform: first k of this thread's next run
  __device__ ConvNchw(const GemmArgs& g, uint32_t m0, uint32_t k_begin, uint32_t k_end_) {
    const uint32_t hw = g.Ho * g.Wo, img0 = m0 / hw;
    const uint32_t m = m0 + threadIdx.x % ROWS;
    ok = m < g.M;
    const uint32_t img = m / hw, p = m % hw, oy = p / g.Wo, ox = p % g.Wo;
    W = g.W;
    HW = g.H * g.W;
    ks = g.ks;
    upsh = g.up == 2 ? 1 : 0;
    Hi = g.H << upsh;
    Wi = g.W << upsh;
    k_end = k_end_;
    iy0 = (int32_t)(oy * g.stride) - (int32_t)g.pad;
    ix0 = (int32_t)(ox * g.stride) - (int32_t)g.pad;
    const uint64_t total = (uint64_t)(g.M / hw) * g.Cin * HW, at = (uint64_t)img0 * g.Cin * HW;
    rs = make_rsrc((const float*)g.a + at, extent_from(total, at, 4));
    base = (int32_t)((img - img0) * g.Cin * HW);
    mode = upsh ? 0 : ks == 3 ? 3 : ks == 1 ? 1 : 0;
#pragma unroll
    for (int t = 0; t < 9; t++)
      tap[t] = mode && t < (mode == 3 ? 9 : 1) ? at_tap(t / 3, t % 3) : kOut;
    k = k_begin + __builtin_amdgcn_readfirstlane(threadIdx.x / ROWS) * KC;
  }
  // byte offset of window position (y, x) in channel 0, kOut outside the image
  __device__ __forceinline__ uint32_t at_tap(uint32_t y, uint32_t x) const {
    const uint32_t iy = (uint32_t)(iy0 + (int32_t)y), ix = (uint32_t)(ix0 + (int32_t)x);
    return ok && iy < Hi && ix < Wi
               ? ((uint32_t)base + (iy >> upsh) * W + (ix >> upsh)) * 4u
               : kOut;
  }
  template <int P>  // a 3x3 run that starts at tap P of channel c
  __device__ __forceinline__ void run3(uint32_t c, F32Tile<ROWS>& t) const {
#pragma unroll
    for (int j = 0; j < KC; j++)
      t.v[j] = buf_f32(rs, tap[(P + j) % 9], (c + (P + j) / 9) * HW * 4u);
  }
  // the run of the next 32-deep stage (stages are visited in order)
  __device__ __forceinline__ void load(uint32_t kb, F32Tile<ROWS>& t) {
    if (mode == 3 && kb + 32 <= k_end) {
      const uint32_t c = k / 9;
      switch (k - c * 9) {
        case 0: run3<0>(c, t); break;
        case 1: run3<1>(c, t); break;
        case 2: run3<2>(c, t); break;
        case 3: run3<3>(c, t); break;
        case 4: run3<4>(c, t); break;
        case 5: run3<5>(c, t); break;
        case 6: run3<6>(c, t); break;
        case 7: run3<7>(c, t); break;
        default: run3<8>(c, t); break;
      }
    } else if (mode == 1 && kb + 32 <= k_end) {
#pragma unroll
      for (int j = 0; j < KC; j++) t.v[j] = buf_f32(rs, tap[0], (k + j) * HW * 4u);
    } else {
      const uint32_t taps = ks * ks;
      uint32_t c = k / taps, y = (k - c * taps) / ks, x = k % ks;
#pragma unroll
      for (int j = 0; j < KC; j++) {
        uint32_t off = kOut;
        if (k + j < k_end) {
          off = at_tap(y, x);
          if (off != kOut) off += c * HW * 4u;
        }
        t.v[j] = buf_f32(rs, off);
        if (++x == ks) {
          x = 0;
          if (++y == ks) {
            y = 0;
            c++;
          }
        }
      }
    }
    k += 32;
  }
};

// BM x BN tile, four wavefronts as 2 x 2 wave tiles, 32 k per stage.  One LDS
// buffer (48 KiB at 128 x 128): the next stage's global loads are in flight in
// registers while this one is computed, and two workgroups per CU overlap one's
// split-and-store phase with the other's MFMAs.
template <int BM, int BN, int AM, int BMD, typename TB>
__global__ __launch_bounds__(256, 2) void k_gemm_f32(GemmArgs g) {
  constexpr int TM = BM / 32, TN = BN / 32;  // 16-row fragments of a wave tile
  constexpr uint32_t PA = BM * 64, PB = BN * 64;
  constexpr bool A_KMAJ = AM == A_CONV_NCHW, B_KMAJ = BMD == B_KN;
  static_assert((BM + BN) * kRawLd * 4 <= 3 * (PA + PB), "unsplit tiles fit the parts' planes");
  __shared__ __attribute__((aligned(16))) char smem[3 * (PA + PB)];
  char *sA = smem, *sB = smem + 3 * PA;

  args_warm(g);
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t wm0 = (wave >> 1) * (BM / 2), wn0 = (wave & 1) * (BN / 2);
  const uint32_t fr = lane & 15, fq = lane >> 4;
  // tile order: N fastest, a contiguous run of tiles per XCD
  const uint32_t n_tiles = (g.N + BN - 1) / BN;
  uint32_t tile = blockIdx.x;
  {
    const uint32_t per = gridDim.x / 8, rem = gridDim.x % 8, xcd = tile % 8, slot = tile / 8;
    tile = xcd < rem ? xcd * (per + 1) + slot : rem * (per + 1) + (xcd - rem) * per + slot;
  }
  const uint32_t m0 = (tile / n_tiles) * BM, n0 = (tile % n_tiles) * BN;
  const uint32_t bz = blockIdx.z / g.splits, split = blockIdx.z % g.splits;
  const uint32_t k_begin = split * g.k_split, k_end = min(g.K, k_begin + g.k_split);
  // (a trailing split may start past K: it contributes zeros)
  const uint32_t n_stages = k_end > k_begin ? (k_end - k_begin + 31) / 32 : 0;

  auto make_a = [&]() {
    if constexpr (A_KMAJ) return ConvNchw<BM>(g, m0, k_begin, k_end);
    else
      return RowMajor<BM, float>((const float*)g.a + (uint64_t)bz * g.sa, g.lda, g.M, g.K, m0,
                                 g.a_vec_ok, k_end);
  };
  auto make_b = [&]() {
    const TB* b = (const TB*)g.b + (uint64_t)bz * g.sb;
    if constexpr (B_KMAJ) return KMajor<BN, TB>(b, g.ldb, g.N, g.K, n0, k_end);
    else return RowMajor<BN, TB>(b, g.ldb, g.N, g.K, n0, g.b_vec_ok, k_end);
  };

  f32x4 acc[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; a++)
#pragma unroll
    for (int b = 0; b < TN; b++) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

  // D = mma(X, Y): a lane holds four consecutive X rows of one Y row, so X is
  // the operand whose index is contiguous in the output: A (pixels) for an
  // NCHW image, B (columns) otherwise.
  auto mma = [](bf16x8 a, bf16x8 b, f32x4 c) {
    return A_KMAJ ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0)
                  : __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a, c, 0, 0, 0);
  };

  {
    auto LA = make_a();
    auto LB = make_b();
    F32Tile<BM> ta;
    F32Tile<BN> tb;
    if (n_stages > 0) {
      LA.load(k_begin, ta);
      LB.load(k_begin, tb);
    }
    for (uint32_t s = 0; s < n_stages; s++) {
      store_split<float>(sA, ta, A_KMAJ);
      store_split<TB>(sB, tb, B_KMAJ);
      if (s + 1 < n_stages) {  // on its way while this stage is computed
        LA.load(k_begin + (s + 1) * 32, ta);
        LB.load(k_begin + (s + 1) * 32, tb);
      }
      lds_barrier();
      bf16x8 bf[TN][3];
#pragma unroll
      for (int b = 0; b < TN; b++)
#pragma unroll
        for (int p = 0; p < 3; p++)
          bf[b][p] = *(const bf16x8*)(sB + p * PB + plane_at(wn0 + b * 16 + fr, fq));
#pragma unroll
      for (int a = 0; a < TM; a++) {
        bf16x8 af[3];
#pragma unroll
        for (int p = 0; p < 3; p++)
          af[p] = *(const bf16x8*)(sA + p * PA + plane_at(wm0 + a * 16 + fr, fq));
        // parts (A, B) from the smallest products up
        constexpr int PI[6] = {2, 0, 1, 1, 0, 0}, PJ[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
        for (int q = 0; q < 6; q++)
#pragma unroll
          for (int b = 0; b < TN; b++) acc[a][b] = mma(af[PI[q]], bf[b][PJ[q]], acc[a][b]);
      }
      lds_barrier();  // the stage has been read
    }
  }

  // non-finite sums: again with the fp32 MFMA on the unsplit values
  float z = 0.0f;
#pragma unroll
  for (int a = 0; a < TM; a++)
#pragma unroll
    for (int b = 0; b < TN; b++)
#pragma unroll
      for (int i = 0; i < 4; i++) z = fmaf(acc[a][b][i], 0.0f, z);
  if (__syncthreads_or(z != 0.0f)) {
    auto LA = make_a();
    auto LB = make_b();
    float *fA = (float*)smem, *fB = fA + BM * kRawLd;
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
      for (int b = 0; b < TN; b++) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (uint32_t s = 0; s < n_stages; s++) {
      F32Tile<BM> ta;
      F32Tile<BN> tb;
      LA.load(k_begin + s * 32, ta);
      LB.load(k_begin + s * 32, tb);
      __syncthreads();
      store_raw(fA, ta, A_KMAJ);
      store_raw(fB, tb, B_KMAJ);
      __syncthreads();
#pragma unroll 1
      for (int k = 0; k < 32; k += 4) {
        float bf[TN];
#pragma unroll
        for (int b = 0; b < TN; b++) bf[b] = fB[(wn0 + b * 16 + fr) * kRawLd + k + fq];
#pragma unroll
        for (int a = 0; a < TM; a++) {
          const float af = fA[(wm0 + a * 16 + fr) * kRawLd + k + fq];
#pragma unroll
          for (int b = 0; b < TN; b++)
            acc[a][b] = A_KMAJ ? __builtin_amdgcn_mfma_f32_16x16x4f32(af, bf[b], acc[a][b], 0, 0, 0)
                               : __builtin_amdgcn_mfma_f32_16x16x4f32(bf[b], af, acc[a][b], 0, 0, 0);
        }
      }
    }
    __syncthreads();  // read before the strips below take the memory
  } else {
    constexpr float unscale = 1.0f / (kScale<float> * kScale<TB>);
#pragma unroll
    for (int a = 0; a < TM; a++)
#pragma unroll
      for (int b = 0; b < TN; b++) acc[a][b] *= unscale;
  }

  // ---- store ----
  // Each wavefront passes 16 rows of the non-contiguous index (Y) at a time
  // through its own strip of LDS, so that it writes whole 128- or 256-byte
  // runs, and the epilogue is one loop over vectors instead of one copy per
  // accumulator.
  constexpr int TX = A_KMAJ ? TM : TN, TY = A_KMAJ ? TN : TM, WX = TX * 16;
  constexpr uint32_t LDS_X = WX + 4;
  static_assert(4 * 16 * LDS_X * 4 <= sizeof(smem), "strips fit");
  float* strip = (float*)smem + wave * 16 * LDS_X;
  const bool part = g.splits > 1;
  float* P = part ? g.part + ((uint64_t)split * g.batch + bz) * (uint64_t)g.M * g.N : nullptr;
  const bool geglu = g.act == ACT_GEGLU && !part;
  // four values of every vector are contiguous and aligned in every tensor
  const bool v4 = A_KMAJ ? g.c_hw % 4 == 0
                         : g.N % 4 == 0 && (part || (g.ldc % 4 == 0 && g.ldr % 4 == 0));
#pragma unroll
  for (int y = 0; y < TY; y++) {
#pragma unroll
    for (int x = 0; x < TX; x++)
      *(f32x4*)(strip + fr * LDS_X + x * 16 + fq * 4) = A_KMAJ ? acc[x][y] : acc[y][x];
    for (uint32_t i = lane; i < 16 * WX / 4; i += 64) {
      const uint32_t yr = i / (WX / 4), x4 = (i % (WX / 4)) * 4;
      f32x4 v = *(const f32x4*)(strip + yr * LDS_X + x4);
      const uint32_t m = m0 + wm0 + (A_KMAJ ? x4 : y * 16 + yr);
      const uint32_t n = n0 + wn0 + (A_KMAJ ? y * 16 + yr : x4);
      if (m >= g.M || n >= g.N) continue;
      if (geglu) {  // 32-column groups of 16 hidden, 16 gate; N % 32 == 0
        if (x4 & 16) continue;
        const f32x4 t = *(const f32x4*)(strip + yr * LDS_X + x4 + 16);
#pragma unroll
        for (int j = 0; j < 4; j++)
          store_out(g, bz, m, (n / 32) * 16 + n % 16 + j, g.N / 2,
                    epi_value<float>(g, bz, m, n + j, v[j]) *
                        gelu_erf_f(epi_value<float>(g, bz, m, n + 16 + j, t[j])));
        continue;
      }
      uint64_t at, rat;
      uint32_t left = 4;  // pixels of m's image from m on
      if (A_KMAJ) {  // partials in the output's layout
        const uint32_t img = m / g.c_hw;
        rat = at = ((uint64_t)img * g.N + n) * g.c_hw + (m - img * g.c_hw);
        left = g.c_hw - (m - img * g.c_hw);
      } else if (part) {
        rat = at = (uint64_t)m * g.N + n;
      } else {
        at = (uint64_t)bz * g.sc + (uint64_t)m * g.ldc + n;
        rat = (uint64_t)bz * g.sr + (uint64_t)m * g.ldr + n;
      }
      if (v4) {
        if (part) {
          *(f32x4*)(P + at) = v;
          continue;
        }
        f32x4 bias = {0.f, 0.f, 0.f, 0.f};
        if (g.bias) {
          if (A_KMAJ) bias[0] = bias[1] = bias[2] = bias[3] = g.bias[n];
          else bias = *(const f32x4*)(g.bias + n);
        }
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] = apply_act(g.act, v[j] * g.alpha + bias[j]);
        if (g.res) v += *(const f32x4*)((const float*)g.res + rat);
        *(f32x4*)((float*)g.c + at) = v;
        continue;
      }
      // Rows or images of no multiple of four: one by one, in straight-line code
      // (137 x 562 x 18 8.6 us with a loop of one value a turn, 6.1 so; one value
      // a lane, or 16 bytes wherever a row has them and single values at its end,
      // took 7.0 and 6.1, but 6.7 and 6.0 against 5.6 for 1499 x 10 x 1).
      uint64_t off[4], o = 0;
      bool ok[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        off[j] = o++;
        ok[j] = A_KMAJ ? m + j < g.M : n + j < g.N;
        if (A_KMAJ && --left == 0) {  // the next image's first pixel of this channel
          o += (uint64_t)(g.N - 1) * g.c_hw;
          left = g.c_hw;
        }
      }
      if (!part) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const float bias = g.bias && ok[j] ? g.bias[A_KMAJ ? n : n + j] : 0.0f;
          v[j] = apply_act(g.act, v[j] * g.alpha + bias);
        }
        if (g.res) {
#pragma unroll
          for (int j = 0; j < 4; j++)
            if (ok[j]) v[j] += ((const float*)g.res + rat)[off[j]];
        }
      }
      float* c = (part ? P : (float*)g.c) + at;
#pragma unroll
      for (int j = 0; j < 4; j++)
        if (ok[j]) c[off[j]] = v[j];
    }
  }
}

// Sum of the split partials, then the epilogue: one element of the output's
// own layout per thread (four where rows allow), partials loaded eight at once.
template <int V>
__global__ __launch_bounds__(256) void k_f32_reduce(GemmArgs g) {
  args_warm(g);
  typedef float vec __attribute__((ext_vector_type(V)));
  const uint64_t mn = (uint64_t)g.M * g.N, step = mn * g.batch;
  const bool geglu = g.act == ACT_GEGLU;
  const uint32_t ncols = geglu ? g.N / 2 : g.N;
  const uint64_t total = (uint64_t)g.batch * g.M * ncols / V;
  auto sum_at = [&](uint64_t e) {
    vec s = {};
    for (uint32_t s0 = 0; s0 < g.splits; s0 += 8) {
      vec t[8];
#pragma unroll
      for (int u = 0; u < 8; u++)
        t[u] = *(const vec*)(g.part + (s0 + u < g.splits ? s0 + u : s0) * step + e);
#pragma unroll
      for (int u = 0; u < 8; u++)
        if (s0 + u < g.splits) s += t[u];
    }
    return s;
  };
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < total;
       i += (uint64_t)gridDim.x * 256) {
    const uint64_t e = i * V;
    if (g.c_nchw) {  // the partials are laid out as the output
      const float bias = g.bias ? g.bias[(e / g.c_hw) % g.N] : 0.0f;
      vec v = sum_at(e);
#pragma unroll
      for (int j = 0; j < V; j++) v[j] = apply_act(g.act, v[j] * g.alpha + bias);
      if (g.res) v += *(const vec*)((const float*)g.res + e);
      *(vec*)((float*)g.c + e) = v;
      continue;
    }
    const uint32_t n = (uint32_t)(e % ncols);
    const uint64_t row = e / ncols;
    const uint32_t m = (uint32_t)(row % g.M), bz = (uint32_t)(row / g.M);
    const uint64_t pr = (uint64_t)bz * mn + (uint64_t)m * g.N;
    vec v;
    if (geglu) {
      const uint32_t nh = (n / 16) * 32 + n % 16;
      const vec h = sum_at(pr + nh), t = sum_at(pr + nh + 16);
#pragma unroll
      for (int j = 0; j < V; j++)
        v[j] = epi_value<float>(g, bz, m, nh + j, h[j]) *
               gelu_erf_f(epi_value<float>(g, bz, m, nh + 16 + j, t[j]));
    } else {
      v = sum_at(pr + n);
#pragma unroll
      for (int j = 0; j < V; j++) v[j] = apply_act(g.act, epi_value<float>(g, bz, m, n + j, v[j]));
    }
    if (g.res) v += *(const vec*)((const float*)g.res + (uint64_t)bz * g.sr + (uint64_t)m * g.ldr + n);
    *(vec*)((float*)g.c + (uint64_t)bz * g.sc + (uint64_t)m * g.ldc + n) = v;
  }
}

template <int BM, int BN, int AM, int BMD, typename TB>
void launch_f32_tile(const GemmArgs& g, hipStream_t s) {
  const dim3 grid(((g.M + BM - 1) / BM) * ((g.N + BN - 1) / BN), 1, g.batch * g.splits);
  k_gemm_f32<BM, BN, AM, BMD, TB><<<grid, 256, 0, s>>>(g);
}

template <int AM, int BMD, typename TB>
void launch_f32(const GemmArgs& g, int tile, hipStream_t s) {
  if (tile == TILE_128x128) launch_f32_tile<128, 128, AM, BMD, TB>(g, s);
  else if (tile == TILE_128x64) launch_f32_tile<128, 64, AM, BMD, TB>(g, s);
  else launch_f32_tile<64, 64, AM, BMD, TB>(g, s);
}

}  // namespace

bool gemm_f32_ok(const GemmArgs& g, int a_mode, int b_mode) {
  // a tile's part of an operand is addressed with 31-bit byte offsets from
  // its first row (its first image; its stage's first k)
  const uint64_t lim = 0x7fff0000ull;
  if (!g.c_f32 || (g.res && !g.res_f32) || g.bias2) return false;
  // Narrow shallow products whose rows are no multiple of four stay with the
  // fp32 MFMA, which stores such rows straight from its accumulators: up to 15
  // columns and K of 31 (B k-major) or 64, M of 64 to 8192, its time is 0.88 to
  // 0.98 of this kernel's; even at K = 32 and 96 and from there on, and from 17
  // columns on, this one is the faster (1.1 to 3.5).
  if (a_mode == A_DENSE && g.N < 16 && g.N % 4 != 0 && g.K <= (b_mode == B_KN ? 31u : 64u))
    return false;
  if (a_mode == A_CONV_NCHW) {
    const uint64_t hw = (uint64_t)g.Ho * g.Wo, img = (uint64_t)g.Cin * g.H * g.W * 4;
    if ((127 / hw + 2) * img > lim || (g.up != 1 && g.up != 2)) return false;
  } else if (128ull * g.lda * 4 + 4ull * g.K > lim) {
    return false;
  }
  if (b_mode == B_KN) return 32ull * g.ldb * 4 <= lim;
  return 128ull * g.ldb * 4 + 4ull * g.K <= lim;
}

void gemm_f32(const GemmArgs& g, int a_mode, int b_mode, int tile, hipStream_t s) {
  if (a_mode == A_CONV_NCHW) {
    if (g.b_f16) launch_f32<A_CONV_NCHW, B_NK, f16>(g, tile, s);
    else launch_f32<A_CONV_NCHW, B_NK, float>(g, tile, s);
  } else if (b_mode == B_NK) {
    if (g.b_f16) launch_f32<A_DENSE, B_NK, f16>(g, tile, s);
    else launch_f32<A_DENSE, B_NK, float>(g, tile, s);
  } else {
    if (g.b_f16) launch_f32<A_DENSE, B_KN, f16>(g, tile, s);
    else launch_f32<A_DENSE, B_KN, float>(g, tile, s);
  }
  if (g.splits <= 1) return;
  const uint32_t ncols = g.act == ACT_GEGLU ? g.N / 2 : g.N;
  const bool v4 = g.c_nchw ? g.c_hw % 4 == 0
                           : g.N % 4 == 0 && ncols % 4 == 0 && g.ldc % 4 == 0 && g.ldr % 4 == 0;
  const uint64_t total = (uint64_t)g.batch * g.M * ncols / (v4 ? 4 : 1);
  const unsigned blocks = (unsigned)(total < 256ull * 65535 ? (total + 255) / 256 : 65535);
  if (v4) k_f32_reduce<4><<<blocks, 256, 0, s>>>(g);
  else k_f32_reduce<1><<<blocks, 256, 0, s>>>(g);
}

}  // namespace di
