// 3x3 stride-1 NHWC fp16 convolution for large images: 256 output pixels x
// 128 output channels per workgroup (gfx950).
//
// The 128 x 64 halo kernel (k_conv3.hip) and the 128 x 128 implicit GEMM reach
// 570-600 TFLOP/s on the decoder's convolutions: a wave there runs 8-16 MFMAs
// between barriers, and the implicit GEMM reads every input pixel nine times.
// Here a workgroup owns a 16 x 16 block of output pixels and 128 channels, and
// a wave 128 x 64 of them on one of two k halves, 32 MFMAs per stage.  The
// (18 x 18)-pixel patch of a 64-channel chunk is loaded once and serves the
// chunk's nine taps (one stage of 256 x 128 x 64 each); a stage loads 16 KB of
// weights and a ninth of the next 41 KB patch, 20 bytes per clock of MFMA time
// where a CU's load path takes 30-40.  Fragments are 12 reads for 32 MFMAs:
// 96 KB of LDS reads per 1024 MFMA clocks, under the LDS's 128 bytes per
// clock, which the 64 x 64 wave tiles of eight undivided waves would use up.
// Square blocks keep the halo at 27 % for any image width; blocks past the
// right or bottom edge compute pixels that are not stored.
//
// Loads go straight to LDS (buffer_load ... lds, lane l at base + 16 l): four
// weight buffers, two patch buffers.  Stage s issues the weights of stage s + 3
// and, at taps 0-5, one of six pieces of the next chunk's patch, computes,
// waits until the weights of stage s + 1 have landed (loads retire in order,
// and the patch's last piece is older than they are) and meets the barrier.
// Weight buffer s % 4 is refilled from stage s + 1 on, after that barrier.
// LDS rows are 64 channels (128 bytes) with the 16-byte chunk position XORed by
// half the pixel column (of the patch) or row (of the weights): sixteen
// neighbouring pixels from any start column, or sixteen weight rows, cover all
// banks once.
//
// A workgroup runs its tiles as one stream of chunks: the last chunk's stages
// issue the next tile's first patch and weights, so that they land during the
// epilogue and its stores during the next tile's first stages (one workgroup
// owns the CU, so nothing else would overlap them; a tile of 128 input channels
// has 18 stages, and its epilogue and first loads took as long as they did).
// Loads past the last tile read zeros into buffers that no stage reads; they
// keep every wait count a constant.
//
// At a tile's end the two k halves swap half of their sums through the patch
// buffer just consumed, four vectors a round, so that each wave finishes 64
// pixels (four image rows of sixteen) x 64 channels in registers: bias, temb
// bias, activation, residual, store, and the GroupNorm statistics of the stored
// values.
//
// Measured in turn against the kernels that had these sizes (halo and implicit
// GEMM): 512 -> 512 at 96 x 96 90 -> 58 us, at 192 x 192 251 -> 182 (955 TFLOP/s),
// 512 -> 512 upsampled to 384 x 384 781 -> 599 (1.16 PFLOP/s), 256 -> 256 at 384 x
// 384 250 -> 181, 128 -> 128 at 768 x 768 298 -> 212.  What bounds it: over the
// clocks of the CUs that hold a tile the MFMAs are busy 67 % (512 channels) and
// 48 % (128: a tile's end, 7 us that no other workgroup of the CU covers), at the
// 1.8 GHz that the card runs at here; LDS 38 and 31 %, bank conflicts 11 and 8;
// waves wait 34 % of theirs, on barriers and the loads behind them.
#include <type_traits>

#include "di_kernels.h"
#include "k_gemm_kernel.h"

namespace di {

namespace {

typedef __attribute__((address_space(3))) void* lds_ptr;

constexpr int BG_PW = 18;                      // patch width and height
constexpr int BG_PIECES = 6;                   // patch pieces (64 rows each, the last 8)
constexpr int BG_PBUF = 328 * 128;             // patch buffer: 324 pixels in whole 8-row loads
constexpr int BG_WBUF = 128 * 128;             // weight buffer
constexpr int BG_NW = 4;
constexpr int BG_PTAB = BG_PIECES * 512 * 4;   // the threads' patch pixels
constexpr int BG_SMEM = 2 * BG_PBUF + BG_NW * BG_WBUF + BG_PTAB;
static_assert(BG_PBUF >= 8 * 4 * 1024, "a round of the k halves' swap fits a patch buffer");

template <int VM>
__device__ __forceinline__ void wait_vm() {  // vmcnt only
  __builtin_amdgcn_s_waitcnt((VM & 15) | ((VM >> 4) << 14) | (7 << 4) | (15 << 8));
}

// The value again, as one the compiler cannot derive: what is computed from it
// stays where it is used.  (Hoisted out of the tile loop, the per-lane constants
// of the patch and the epilogue spilled 81 registers of the stages.)
__device__ __forceinline__ int here(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// Sum over the 16 lanes of a row (every lane gets it).
__device__ __forceinline__ float row_sum16(float v) {
#define DI_ROR(n)                                                                               \
  v += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x120 + n, 0xf, 0xf, \
                                                   false));
  DI_ROR(8)
  DI_ROR(4)
  DI_ROR(2)
  DI_ROR(1)
#undef DI_ROR
  return v;
}

__global__ __launch_bounds__(512, 2) void k_conv3_big(GemmArgs g) {
  __shared__ __attribute__((aligned(1024))) char smem[BG_SMEM];
  args_warm(g);
  char* const patch = smem;
  char* const wbuf = smem + 2 * BG_PBUF;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kh = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;

  // tiles: channels fastest (they share the patch), then blocks row by row.
  // Workgroup b (on XCD b % 8) takes run (b % 8) * ceil(grid / 8) + b / 8 of
  // the list, so neighbouring runs share an XCD's L2.
  const uint32_t nbn = (g.N + 127) / 128, nbx = (g.Wo + 15) / 16, nby = (g.Ho + 15) / 16;
  const uint32_t n_tiles = g.M / (g.Ho * g.Wo) * nby * nbx * nbn;
  uint32_t t0, t1;
  {
    const uint32_t n_wg = gridDim.x, per = n_wg / 8, rem = n_wg % 8, xcd = blockIdx.x % 8,
                   slot = blockIdx.x / 8;
    const uint32_t run =
        xcd < rem ? xcd * (per + 1) + slot : rem * (per + 1) + (xcd - rem) * per + slot;
    const uint32_t len = n_tiles / n_wg, more = n_tiles % n_wg;
    t0 = run * len + min(run, more);
    t1 = t0 + len + (run < more ? 1 : 0);
  }
  struct Tile {
    uint32_t n0, img, bin, y0, x0;
  };
  auto tile_at = [&](uint32_t t) {
    Tile T;
    const uint32_t blk = t / nbn;
    T.n0 = (t - blk * nbn) * 128;
    T.img = blk / (nby * nbx);
    T.bin = blk - T.img * (nby * nbx);
    const uint32_t by = T.bin / nbx;
    T.y0 = by * 16;
    T.x0 = (T.bin - by * nbx) * 16;
    return T;
  };
  const uint32_t ush = g.up == 2 ? 1u : 0u;
  const int nch = (int)(g.Cin / 64);

  constexpr uint32_t kInv = 0x80000000u;
  const __amdgpu_buffer_rsrc_t rA = make_rsrc(g.a, g.a_bytes), rA2 = make_rsrc(g.a2, g.a2_bytes),
                               rB = make_rsrc(g.b, g.b_bytes);

  // ---- this lane's DMA slots: row lane / 8 of an 8-row load, chunk lane % 8 ----
  uint32_t fw[2];  // weights: rows wave * 16 + i * 8 + lrow
  auto set_weights = [&](uint32_t n0, bool live) {
    const int l = here(lane), lrow = l >> 3, lpos = l & 7;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const uint32_t row = wave * 16 + i * 8 + lrow;
      fw[i] = live && n0 + row < g.N
                  ? (n0 + row) * (uint32_t)g.ldb * 2u + (lpos ^ ((row >> 1) & 7u)) * 16u
                  : kInv;
    }
  };
  // patch piece i: rows i * 64 + wave * 8 + lrow; the last piece is eight rows,
  // which every wave loads alike.  Each thread keeps its pieces' (source pixel
  // << 3) | chunk, or kInv outside the image, in its own column of LDS: six
  // registers that the accumulators need.
  uint32_t* const ptab = (uint32_t*)(smem + 2 * BG_PBUF + BG_NW * BG_WBUF) + tid;
  auto set_patch = [&](const Tile& T, bool live) {
    const int l = here(lane), lrow = l >> 3, lpos = l & 7;
#pragma unroll
    for (int i = 0; i < BG_PIECES; i++) {
      const uint32_t pr = i + 1 < BG_PIECES ? i * 64 + wave * 8 + lrow : i * 64 + lrow;
      const uint32_t py = pr / BG_PW, px = pr % BG_PW;
      const int iy = (int)(T.y0 + py) - 1, ix = (int)(T.x0 + px) - 1;
      const bool ok = live & (pr < BG_PW * BG_PW) & ((uint32_t)iy < g.Ho) & ((uint32_t)ix < g.Wo);
      ptab[i * 512] =
          ok ? (((T.img * g.H + ((uint32_t)iy >> ush)) * g.W + ((uint32_t)ix >> ush)) << 3 |
                (lpos ^ ((px >> 1) & 7u)))
             : kInv;
    }
  };
  auto dma_weights = [&](int chunk, int tap, int buf) {
    const uint32_t koff = ((uint32_t)tap * g.Cin + (uint32_t)chunk * 64u) * 2u;
#pragma unroll
    for (int i = 0; i < 2; i++)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rB, (lds_ptr)(wbuf + buf * BG_WBUF + (wave * 16 + i * 8) * 128), 16, fw[i], koff, 0, 0);
  };
  // the source of the patch pieces being issued: one of the two tensors, its
  // pixel stride and the chunk's first channel, in bytes
  __amdgpu_buffer_rsrc_t rP = rA;
  uint32_t pld = 0, pch = 0;
  auto set_source = [&](int chunk) {
    const uint32_t cb = (uint32_t)chunk * 64u;
    const bool s2 = cb >= g.c1;
    rP = s2 ? rA2 : rA;
    pld = (uint32_t)(s2 ? g.lda2 : g.lda) * 2u;
    pch = (s2 ? cb - g.c1 : cb) * 2u;
  };
  // p: the piece's entry of ptab
  auto dma_patch = [&](uint32_t p, int buf, int piece) {
    const uint32_t off = (p >> 3) * pld + (p & 7u) * 16u;
    const int row = piece + 1 < BG_PIECES ? piece * 64 + wave * 8 : piece * 64;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rP, (lds_ptr)(patch + buf * BG_PBUF + row * 128), 16,
                                             p == kInv ? kInv : off, pch, 0, 0);
  };

  // ---- fragments (16x16x32: lane row lane % 16, k (lane / 16) * 8) ----
  f32x4 acc[8][4];
  auto clear = [&]() {
#pragma unroll
    for (int a = 0; a < 8; a++)
#pragma unroll
      for (int b = 0; b < 4; b++) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  };

  // ---- prologue: the first tile's patch and stages 0-2 ----
  Tile T = tile_at(t0);
  set_patch(T, true);
  set_weights(T.n0, true);
  set_source(0);
#pragma unroll
  for (int i = 0; i < BG_PIECES; i++) dma_patch(ptab[i * 512], 0, i);
#pragma unroll
  for (int s = 0; s < 3; s++) dma_weights(0, s, s);
  wait_vm<0>();
  __builtin_amdgcn_s_barrier();

  int s = 0, pbuf = 0;  // stage (mod 4) and patch buffer of the whole run
  // cn: the chunk after this one (0 of the next tile after the last).  landed:
  // a tile's first chunk, whose stages 1 and 2 arrived before its stage 0
  auto stage = [&](auto tap_c, int chunk, int cn, bool landed) {
    constexpr int tap = decltype(tap_c)::value, ky = tap / 3, kx = tap % 3;
    // acc[0..3] are the rows this k half finishes (4 kh + a of the wave tile),
    // acc[4..7] the other's
    const int r = lane & 15, kc = kh * 4 + (lane >> 4), x = kx + r;  // kc: 16-byte k chunk
    const char* pp = patch + pbuf * BG_PBUF + ((wm * 8 + ky) * BG_PW + x) * 128 +
                     ((kc ^ ((x >> 1) & 7)) << 4);
    const char* p0 = pp + kh * 4 * BG_PW * 128;
    const char* p1 = pp - kh * 4 * BG_PW * 128;
    const char* wb =
        wbuf + (s & 3) * BG_WBUF + (wn * 64 + r) * 128 + ((kc ^ ((r >> 1) & 7)) << 4);
    f16x8 bf[4], af[4];
#pragma unroll
    for (int b = 0; b < 4; b++) bf[b] = *(const f16x8*)(wb + b * 16 * 128);
#pragma unroll
    for (int a = 0; a < 2; a++) af[a] = *(const f16x8*)(p0 + a * BG_PW * 128);
    const uint32_t pp_next = ky < 2 ? ptab[(ky * 3 + kx) * 512] : 0;
    // two pixel rows at a time, the next two on their way; a fence after half
    // of them keeps the scheduler from reading every fragment first
#pragma unroll
    for (int a0 = 0; a0 < 8; a0 += 2) {
      if (a0 == 4) __builtin_amdgcn_sched_barrier(0);
      if (a0 < 6) {
#pragma unroll
        for (int a = a0 + 2; a < a0 + 4; a++)
          af[a & 3] = *(const f16x8*)((a < 4 ? p0 : p1) + a * BG_PW * 128);
      }
      // D = mma(weights, pixels): a lane holds four consecutive channels of
      // pixel column lane % 16
#pragma unroll
      for (int a = a0; a < a0 + 2; a++)
#pragma unroll
        for (int b = 0; b < 4; b++)
          acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bf[b], af[a & 3], acc[a][b], 0, 0, 0);
      if (a0 == 0) {  // behind the first MFMAs: they need none of this
        dma_weights(ky < 2 ? chunk : cn, ky < 2 ? ky * 3 + 3 + kx : kx, (s + 3) & 3);
        if (ky < 2) dma_patch(pp_next, pbuf ^ 1, ky * 3 + kx);
      }
    }
    // stage s + 1's weights were issued at stage s - 2, before that stage's
    // patch piece: younger are stages s - 1's and s's weights and the pieces of
    // taps s - 2 to s that are among the first six
    if (ky == 0) {
      if (kx == 2 || !landed) wait_vm<5 + kx>();
    } else if (ky == 1) {
      wait_vm<7>();
    } else {
      wait_vm<6 - kx>();
    }
    lds_barrier();
    s = (s + 1) & 3;
  };
  // ---- epilogue of a tile: rows y0 + wm * 8 + kh * 4 + a, column x0 + lane % 16,
  // channels n0 + wn * 64 + b * 16 + (lane / 16) * 4 .. + 3 ----
  auto finish = [&](const Tile& T) {
    const int l = here(lane), r = l & 15, q = l >> 4;
    const uint32_t ox = T.x0 + r, oy0 = T.y0 + wm * 8 + kh * 4, nb = T.n0 + wn * 64 + q * 4;
    const bool silu = g.act == ACT_SILU;
    char* const xb = patch + (pbuf ^ 1) * BG_PBUF;  // the last chunk's patch: consumed
    f32x4* const mine = (f32x4*)(xb + wave * 4 * 1024) + l;
    const f32x4* const other = (const f32x4*)(xb + (wave ^ 4) * 4 * 1024) + l;
    f32x4 bias[4], sm[4], sq[4];
#pragma unroll
    for (int b = 0; b < 4; b++) {
      sm[b] = sq[b] = bias[b] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (nb + b * 16 < g.N) {
        if (g.bias) bias[b] = ld4(g.bias + nb + b * 16);
        // the temb bias is per image (rows_b2 = Ho * Wo)
        if (g.bias2) bias[b] += ld4(g.bias2 + (uint64_t)T.img * g.ld_b2 + nb + b * 16);
      }
    }
    // every residual row at once, with the biases and whatever is left of the
    // next tile's first patch and stages 0-2 (this wave's are waited for here,
    // every wave's by the barriers below)
    f16x4 res[4][4];
    uint32_t m[4];
    bool ok[4];
#pragma unroll
    for (int a = 0; a < 4; a++) {
      ok[a] = ox < g.Wo && oy0 + a < g.Ho;
      m[a] = ok[a] ? (T.img * g.Ho + oy0 + a) * g.Wo + ox : T.img * g.Ho * g.Wo;
    }
    if (g.res) {
#pragma unroll
      for (int a = 0; a < 4; a++) {
        const f16* R = (const f16*)g.res + (uint64_t)m[a] * g.ldr + nb;
#pragma unroll
        for (int b = 0; b < 4; b++)
          if (nb + b * 16 < g.N) res[a][b] = *(const f16x4*)(R + b * 16);
      }
    }
    wait_vm<0>();
    // swap halves row by row: k half h finishes rows 4 h .. 4 h + 3 of its tile
#pragma unroll
    for (int a = 0; a < 4; a++) {
#pragma unroll
      for (int b = 0; b < 4; b++) mine[b * 64] = acc[a + 4][b];
      lds_barrier();
      f16* C = (f16*)g.c + (uint64_t)m[a] * g.ldc + nb;
#pragma unroll
      for (int b = 0; b < 4; b++) {
        const f32x4 v = acc[a][b] + other[b * 64];
        f16x4 o;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          float t = v[i] * g.alpha + bias[b][i];
          if (silu) t = silu_f(t);
          if (g.res) t += (float)res[a][b][i];
          o[i] = (f16)t;
          const float u = ok[a] ? (float)o[i] : 0.0f;
          sm[b][i] += u;
          sq[b][i] += u * u;
        }
        if (ok[a] && nb + b * 16 < g.N) *(f16x4*)(C + b * 16) = o;
      }
      lds_barrier();
    }
    if (!g.stats) return;

    // ---- statistics: this wave's 64 pixels per channel ----
#pragma unroll
    for (int b = 0; b < 4; b++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        sm[b][i] = row_sum16(sm[b][i]);
        sq[b][i] = row_sum16(sq[b][i]);
      }
    const uint32_t slots = (g.Ho * g.Wo + 63) / 64, nblk = nby * nbx;
    float* st = g.stats + (uint64_t)T.img * slots * g.N * 2;
    if (slots == 4 * nblk) {  // whole blocks: one slot per wave
      if (r == 0) {
        float* p = st + ((uint64_t)(T.bin * 4 + wm * 2 + kh) * g.N + nb) * 2;
#pragma unroll
        for (int b = 0; b < 4; b++)
          if (nb + b * 16 < g.N) {
            *(f32x4*)(p + b * 32) = f32x4{sm[b][0], sq[b][0], sm[b][1], sq[b][1]};
            *(f32x4*)(p + b * 32 + 4) = f32x4{sm[b][2], sq[b][2], sm[b][3], sq[b][3]};
          }
      }
      return;
    }
    // ragged edges: the block's sums go to slot bin, and the slots past the
    // last block are cleared (conv3_big_stats_ok: at least one slot per block)
    float* sp = (float*)xb;  // [wm * 2 + kh][128 channels][2]
    if (r == 0) {
#pragma unroll
      for (int b = 0; b < 4; b++)
#pragma unroll
        for (int i = 0; i < 4; i++)
          *(float2*)(sp + ((wm * 2 + kh) * 128 + wn * 64 + b * 16 + q * 4 + i) * 2) =
              float2{sm[b][i], sq[b][i]};
    }
    lds_barrier();
    if (tid < 128 && T.n0 + tid < g.N) {
      float2 t = *(const float2*)(sp + tid * 2);
#pragma unroll
      for (int w = 1; w < 4; w++) {
        const float2 u = *(const float2*)(sp + (w * 128 + tid) * 2);
        t.x += u.x;
        t.y += u.y;
      }
      for (uint32_t k = T.bin; k < slots; k += nblk) {
        *(float2*)(st + ((uint64_t)k * g.N + T.n0 + tid) * 2) = t;
        t = float2{0.0f, 0.0f};
      }
    }
    lds_barrier();  // read before the next tile's patches take the buffer
  };

  for (uint32_t t = t0; t < t1; t++) {
    clear();
    Tile Tn = T;
    for (int c = 0; c < nch; c++) {
      const bool last = c + 1 == nch, first = c == 0;
      const int cn = last ? 0 : c + 1;
      set_source(cn);
      if (last && t + 1 < t1) Tn = tile_at(t + 1);
      if (last) set_patch(Tn, t + 1 < t1);  // (this tile's patches are all on their way)
      stage(std::integral_constant<int, 0>{}, c, cn, first);
      stage(std::integral_constant<int, 1>{}, c, cn, first);
      stage(std::integral_constant<int, 2>{}, c, cn, first);
      stage(std::integral_constant<int, 3>{}, c, cn, first);
      stage(std::integral_constant<int, 4>{}, c, cn, first);
      stage(std::integral_constant<int, 5>{}, c, cn, first);
      if (last) set_weights(Tn.n0, t + 1 < t1);  // issued by the next three stages
      stage(std::integral_constant<int, 6>{}, c, cn, first);
      stage(std::integral_constant<int, 7>{}, c, cn, first);
      stage(std::integral_constant<int, 8>{}, c, cn, first);
      pbuf ^= 1;
    }

    finish(T);
    T = Tn;
  }
}

}  // namespace

bool conv3_big_ok(const GemmArgs& g) {
  const bool single = g.a2 == nullptr || g.a2 == g.a || g.c1 == 0 || g.c1 == 0xffffffffu;
  const uint64_t hw = (uint64_t)g.Ho * g.Wo;
  return g.Cin > 0 && g.ks == 3 && g.stride == 1 && g.pad == 1 && (g.up == 1 || g.up == 2) &&
         g.Cin % 64 == 0 && (single || g.c1 % 64 == 0) && g.N % 64 == 0 && g.Ho == g.H * g.up &&
         g.Wo == g.W * g.up && g.M % hw == 0 && g.batch == 1 && g.splits <= 1 &&
         (g.act == ACT_NONE || g.act == ACT_SILU) && (!g.bias2 || g.rows_b2 == hw) && g.b_vec_ok && !g.part_slots &&
         g.a_bytes > 0 && g.b_bytes > 0 && (single || g.a2_bytes > 0) && g.K == 9 * g.Cin &&
         (uint64_t)g.N * g.ldb * 2 < (1ull << 31) &&
         (uint64_t)g.M / (g.up * g.up) < (1ull << 28);
}

bool conv3_big_stats_ok(const GemmArgs& g) {
  const uint64_t hw = (uint64_t)g.Ho * g.Wo;
  return (hw % 64 == 0 || g.M == hw) &&
         (uint64_t)((g.Ho + 15) / 16) * ((g.Wo + 15) / 16) <= (hw + 63) / 64;
}

uint32_t conv3_big_tiles(const GemmArgs& g) {
  return g.M / (g.Ho * g.Wo) * ((g.Ho + 15) / 16) * ((g.Wo + 15) / 16) * ((g.N + 127) / 128);
}

void launch_conv3_big(const GemmArgs& g, hipStream_t s) {
  // one workgroup per CU of a whole MI355X, each with a run of tiles; a partition
  // of fewer CUs takes the same runs in turn
  const uint32_t tiles = conv3_big_tiles(g);
  k_conv3_big<<<tiles < 256 ? tiles : 256, 512, 0, s>>>(g);
}

}  // namespace di
