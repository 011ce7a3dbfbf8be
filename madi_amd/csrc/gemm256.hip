// gemm256.hip -- the Q8 GEMM for many rows (long recordings, many windows):
// 256 x 256 tiles on a weight dequantised once per call.
//
// Under a sustained MFMA load the card holds its power, not its clock: over a
// long recording the fused kernels of gemm.hip run at 1.5 - 1.7 GHz with the
// matrix pipes 61 - 66 % busy (5120 -> 1280), so what pays is less energy per
// product.  Three things do that here.  The panel-layout weight is written once per call as F16 [N][K]
// rows into an array of the library (the exact fp16_rne(q * s) of every other
// kernel, 6.4 us for 5120 x 1280) instead of being dequantised once per 128-row
// tile beside the MFMAs.  The MFMA is 16x16x32: a register-only loop on random
// operands sustains 1.91 PFLOP/s with it and 1.58-1.68 with 32x32x16 (both
// 2.4 on zeros), because each product updates half as many accumulators.  And
// a 256 x 256 tile brings a third less through L2 and LDS per product than a
// 128 x 256 one.  At M = 24000, 5120 -> 1280 the clock is 1.90 - 1.94 GHz, the
// matrix pipes 62 % busy, 251-283 us against 265-315 over boxes (alternating
// on one, 257 / 268); without any operand loads (results discarded) the same
// loop took 239 where it took 268.  1280 -> 5120 + bias + GELU: 336 / 343 on
// one box, 336 / 321 on another, 331-377 in all: GELU runs with nothing under
// it (pipes 44 % busy).
//
// Rows past M load as zeros; results differ from the fused kernels' only by
// the order of the fp32 sums.
#include "common.h"
#include "gemm256.h"
#include "vmem.h"

namespace madi {
namespace {

typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) u32x2 lds_u32x2;

constexpr uint32_t kBM = 256, kBN = 256;
// The LDS is a ring of five units: one operand's 256 rows x 64 k (128 bytes a
// row) of one chunk, in the order A0 W0 A1 W1 A2 W2 ..
constexpr uint32_t kUnit = 256 * 128, kUnits = 5;
constexpr int kSc1 = 16;                    // buffer cache policy: write through the L2

__device__ inline f16x8 frag(uint32_t addr) {
  return __builtin_bit_cast(f16x8, *(const lds_u32x4 *)(uintptr_t)addr);
}
// 16-byte piece p of a 128-byte LDS row is kept at p ^ swz(row): the 32 rows
// of a fragment read spread over all banks
__device__ inline uint32_t swz(uint32_t row) { return (row >> 1) & 7; }

// Panel layout -> F16 [N][K] rows.  One wave per (panel, chunk): lane (h, r)
// dequantises its quantisation block of row r, the wave's 32 x 128-byte tile
// goes through LDS and leaves as whole 128-byte row segments.  N % 32 == 0.
__global__ __launch_bounds__(256) void q8_rows_f16_kernel(f16 *__restrict__ out,
                                                          const uint8_t *__restrict__ qs,
                                                          const f16 *__restrict__ sc, uint32_t K,
                                                          uint32_t units) {
  __shared__ __attribute__((aligned(16))) uint8_t tile[4][32 * 128];
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t u = blockIdx.x * 4 + wave;  // panel * chunks + chunk
  if (u >= units) return;
  const uint32_t chunks = K / kChunkK, p = u / chunks, c = u - p * chunks;
  const uint32_t r = lane & 31, h = lane >> 5;
  const uint8_t *q = qs + (size_t)u * (kPanelRows * kChunkK);
  const f16 s = sc[(size_t)u * 64 + lane];
  uint8_t *row = tile[wave] + r * 128;
#pragma unroll
  for (uint32_t j = 0; j < 2; ++j) {
    f16x8 lo, hi;
    dequant16(*reinterpret_cast<const u32x4 *>(q + ((2 * j + h) * 32 + r) * 16), s, lo, hi);
    *reinterpret_cast<f16x8 *>(row + 16 * ((4 * h + 2 * j) ^ swz(r))) = lo;
    *reinterpret_cast<f16x8 *>(row + 16 * ((4 * h + 2 * j + 1) ^ swz(r))) = hi;
  }
  __builtin_amdgcn_wave_barrier();
  uint8_t *dst = reinterpret_cast<uint8_t *>(out + (size_t)p * kPanelRows * K + c * kChunkK);
#pragma unroll
  for (uint32_t j = 0; j < 4; ++j) {
    const uint32_t t = 8 * j + (lane >> 3), piece = lane & 7;
    *reinterpret_cast<u32x4 *>(dst + (size_t)t * K * 2 + 16 * piece) =
        *reinterpret_cast<const u32x4 *>(tile[wave] + t * 128 + 16 * (piece ^ swz(t)));
  }
}

// Tile t of round j for workgroup b: the 32 workgroups of an XCD (b % 8) take
// a contiguous run of the round's tiles, so their operands meet in one L2.
struct Walk {
  uint32_t tiles, tiles_m, tiles_n, group_m;
  __device__ inline bool at(uint32_t round, uint32_t b, uint32_t grid, uint32_t &m0, uint32_t &n0) const {
    const uint32_t base = round * grid;
    if (base >= tiles) return false;
    const uint32_t left = tiles - base < grid ? tiles - base : grid;
    const uint32_t x = b & 7, slot = b >> 3, per = left >> 3, extra = left & 7;
    if (slot >= per + (x < extra ? 1u : 0u)) return false;
    const uint32_t t = base + x * per + (x < extra ? x : extra) + slot;
    const uint32_t per_group = group_m * tiles_n, gi = t / per_group, first = gi * group_m;
    const uint32_t gm = tiles_m - first < group_m ? tiles_m - first : group_m;
    const uint32_t in = t - gi * per_group;
    m0 = (first + in % gm) * kBM;
    n0 = (in / gm) * kBN;
    return true;
  }
};

// Persistent: the chunks of a workgroup's tiles form one stream, so a tile's
// first loads run under the tile before it.  Wave (wm, wn) = (wave / 4, wave %
// 4) owns 128 rows x 64 columns as 8 x 4 accumulators of 16 x 16, the weight
// the MFMA's first operand.
//
// The two waves of a SIMD, one of each wm, take turns: while one issues a
// step's 32 MFMAs the other issues the DMAs and reads the fragments of its
// next step, a barrier between the phases, wm = 1 one phase behind (all eight
// waves in step measured 290 us where the turns take 268, 5120 -> 1280 at M =
// 24000).  With phase t = 4c + .. of chunk c, wm = 0 reads in 4c and 4c + 2,
// wm = 1 in 4c + 1 and 4c + 3, so the chunk's units are free from 4c + 4 on
// and the DMAs into them are issued in the next chunk's reading phases.
template <int EPI>
__global__ __launch_bounds__(512) void q8_gemm256_kernel(const f16 *__restrict__ A,
                                                         const f16 *__restrict__ W, uint32_t M,
                                                         uint32_t N, uint32_t K, Walk walk,
                                                         f16 *__restrict__ C,
                                                         const float *__restrict__ bias) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[kUnits * kUnit];
  const uint32_t lane = threadIdx.x & 63, wave = sgpr(threadIdx.x >> 6);
  const uint32_t wm = wave >> 2, wn = wave & 3;
  const uint32_t nk = K / kChunkK, grid = gridDim.x;
  const uint32_t lds = lds_addr(smem);
  const desc_t dw = make_desc(W, N * K * 2);

  // Load cursors: the next chunk of each operand in the stream.  A DMA i of
  // this wave copies rows 32 wave + 8 i + lane / 8.  The A descriptor spans
  // the tile's rows that exist; rows past M lie outside it (zeros, for
  // output rows that are never stored).
  struct Cursor {
    uint32_t round, c, m, n;
    bool live;
  };
  uint32_t m0, n0;
  if (!walk.at(0, blockIdx.x, grid, m0, n0)) return;
  Cursor ca = {0, 0, m0, n0, true}, cw = {0, 0, m0, n0, true};
  auto advance = [&](Cursor &cur) {
    if (cur.live && ++cur.c == nk) {
      cur.c = 0;
      cur.live = walk.at(++cur.round, blockIdx.x, grid, cur.m, cur.n);
    }
  };
  uint32_t va[4], vw[2];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t row = 32 * wave + 8 * i + (lane >> 3), x = (lane & 7) ^ swz(row);
    const uint32_t q = 16 * ((x & 3) * 2 + (x >> 2));
    va[i] = row * K * 2 + q;
    if (i < 2) vw[i] = (lane >> 3) * K * 2 + q;
  }
  auto dma_a = [&](uint32_t slot) {
    const uint32_t left = M - ca.m < kBM ? M - ca.m : kBM;
    const desc_t da = make_desc(A + (size_t)ca.m * K, left * K * 2);
    const uint32_t at = lds + slot * kUnit + wave * 4096;
#pragma unroll
    for (int i = 0; i < 4; ++i) dma16<0, true>(da, va[i], ca.c * 128, at + 1024 * i);
  };
  auto dma_w = [&](uint32_t slot) {
    const uint32_t at = lds + slot * kUnit + wave * 4096;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      dma16<0, true>(dw, vw[i & 1], (cw.n + 32 * wave + 8 * i) * K * 2 + cw.c * 128, at + 1024 * i);
  };

  // fragments: lane (g, c) of step e holds k = 16g + 8e .. + 8 of row c of a
  // 16-row tile, piece 2g + e of the row
  uint32_t fo[2];
  {
    const uint32_t g = lane >> 4, c16 = lane & 15;
#pragma unroll
    for (int e = 0; e < 2; ++e) fo[e] = c16 * 128 + 16 * ((4 * e + g) ^ swz(c16));
  }
  f16x8 af[8], wf[4];
  auto read = [&](int e, uint32_t a_slot, uint32_t w_slot) {
    const uint32_t aw = lds + w_slot * kUnit + wn * (64 * 128) + fo[e];
    const uint32_t aa = lds + a_slot * kUnit + wm * (128 * 128) + fo[e];
#pragma unroll
    for (int t = 0; t < 4; ++t) wf[t] = frag(aw + t * 2048);
#pragma unroll
    for (int i = 0; i < 8; ++i) af[i] = frag(aa + i * 2048);
  };
  auto wrap = [](uint32_t slot) { return slot >= kUnits ? slot - kUnits : slot; };
  auto landed = [](bool ahead) {
    if (ahead)
      asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  };
  auto meet = [] {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  // prologue: units A0 W0 A1 W1 A2 into slots 0 .. 4
  uint32_t issued_a = 0;
#pragma unroll
  for (uint32_t u = 0; u < kUnits; ++u) {
    Cursor &cur = u & 1 ? cw : ca;
    if (cur.live) {
      if (u & 1) {
        dma_w(u);
      } else {
        dma_a(u);
        ++issued_a;
      }
    }
    advance(cur);
  }
  // (a stream of fewer than three chunks has issued less)
  bool ahead = issued_a == 3;  // the A of two chunks on was issued
  if (ahead)
    wait_then_barrier<12>();
  else
    wait_then_barrier<0>();
  uint32_t sa = 0;  // this chunk's A slot; its W is in the next
  bool first = true;
  if (wm == 1) meet();

  for (uint32_t round = 0;;) {
    f32x4 acc[8][4];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[i][t] = (f32x4){};
    auto mfmas = [&] {
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int t = 0; t < 4; ++t)
          acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[t], af[i], acc[i][t], 0, 0, 0);
      __builtin_amdgcn_s_setprio(0);
    };
#pragma unroll 1
    for (uint32_t c = 0; c < nk; ++c) {
      const uint32_t sw = wrap(sa + 1);
      if (cw.live && !first) dma_w(wrap(sa + 3));
      read(0, sa, sw);
      if (!first) advance(cw);
      meet();
      mfmas();
      meet();
      if (ca.live && !first) dma_a(wrap(sa + 4));
      read(1, sa, sw);
      if (!first) {
        ahead = ca.live;
        advance(ca);
      }
      first = false;
      if (wm == 1) landed(ahead);
      meet();
      mfmas();
      if (wm == 0) landed(ahead);
      meet();
      sa = wrap(sa + 2);
    }

    // Epilogue, one 32-row m-tile at a time through the wave's own 4 KiB of
    // the last chunk's W slot (refilled, by this wave's own DMAs, only from
    // the next chunk's quarter 1 on).  The lane is made opaque so that these
    // addresses are not kept in registers over the loop.
    uint32_t ln = lane;
    asm volatile("" : "+v"(ln));
    const uint32_t g = ln >> 4, c16 = ln & 15;
    const uint32_t stg = lds + wrap(sa + 4) * kUnit + wave * 4096;
    const uint32_t rows = M - m0 < kBM ? M - m0 : kBM;
    const __amdgpu_buffer_rsrc_t cr = __builtin_amdgcn_make_buffer_rsrc(
        C + (size_t)m0 * N, 0, (int)(rows * N * 2), 0x00020000);
    f32x4 bv[4];
    if constexpr (EPI != MADI_EPI_NONE) {
#pragma unroll
      for (int t = 0; t < 4; ++t)
        bv[t] = *reinterpret_cast<const f32x4 *>(bias + n0 + 64 * wn + 16 * t + 4 * g);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const uint32_t row = 16 * u + c16;
          f16x4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float v = acc[2 * i + u][t][e];
            if constexpr (EPI != MADI_EPI_NONE) v += bv[t][e];
            if constexpr (EPI == MADI_EPI_BIAS_GELU) v = gelu_erf_fast(v);
            o[e] = (f16)v;
          }
          *(lds_u32x2 *)(uintptr_t)(stg + row * 128 + 16 * ((2 * t + (g >> 1)) ^ swz(row)) + 8 * (g & 1)) =
              __builtin_bit_cast(u32x2, o);
        }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t row = 8 * j + (ln >> 3), m = 128 * wm + 32 * i + row;
        const u32x4 v = *(const lds_u32x4 *)(uintptr_t)(stg + row * 128 + 16 * ((ln & 7) ^ swz(row)));
        if (m < rows)
          __builtin_amdgcn_raw_buffer_store_b128(v, cr, (m * N + n0 + 64 * wn) * 2 + 16 * (ln & 7), 0, kSc1);
      }
    }
    if (!walk.at(++round, blockIdx.x, grid, m0, n0)) break;
  }
  if (wm == 0) meet();
}

template <int EPI>
int launch(const void *a, const f16 *w, void *c, const float *bias, uint32_t m, uint32_t n, uint32_t k) {
  Walk walk;
  walk.tiles_m = (m + kBM - 1) / kBM;
  walk.tiles_n = n / kBN;
  walk.tiles = walk.tiles_m * walk.tiles_n;
  walk.group_m = walk.tiles_m < 8 ? walk.tiles_m : 8;
  const uint32_t cus = (uint32_t)cu_count() / 8 * 8, up = (walk.tiles + 7) & ~7u;
  hipLaunchKernelGGL((q8_gemm256_kernel<EPI>), dim3(up < cus ? up : cus), dim3(512), 0, stream(),
                     static_cast<const f16 *>(a), w, m, n, k, walk, static_cast<f16 *>(c), bias);
  return check_launch("madi_q8_gemm");
}

// The dequantised weight of the call in progress, one array per device.
constexpr size_t kWeightBytes = size_t(16) << 20;
static __device__ __align__(256) uint8_t weight_rows[kWeightBytes];
constexpr int kMaxDevices = 64;
f16 *g_weight[kMaxDevices];
}  // namespace

f16 *gemm256_weight() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
  if (!g_weight[dev]) {
    void *ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(weight_rows)) != hipSuccess) {
      (void)hipGetLastError();  // the launch that follows takes another kernel
      return nullptr;
    }
    g_weight[dev] = static_cast<f16 *>(ptr);
  }
  return g_weight[dev];
}

// Whole 256-column groups (a weight that fits its array, byte offsets inside
// 2 GiB) whose tiles fill their rounds of one tile per CU to at least nine
// tenths, where the kernels of gemm.hip are the slower ones (us, theirs /
// these, back to back; the pass that writes the weight counts here):
// - In rounds, a tile stands for two of their 128 x 256 ones, which it takes
//   0.91 to 0.98 of, so up to a fifteenth more rounds than theirs (1280 ->
//   5120 + bias: equal rounds M = 9200 114 / 107, 15000 186 / 171, 22000 264 /
//   248; a fifteenth more M = 23600 278 / 275, 299 / 287, + GELU 348 / 343,
//   319 / 324; a thirteenth more M = 21000 243 / 246, + GELU 277 / 288; a
//   ninth more M = 14600 169 / 173, + GELU 194 / 205).
// - At two rounds or more the weight's pass needs 5120 rows to be worth it
//   (n x k = 8192 x 768, M = 3840 53.8 / 58.1, 6400 x 1280, M = 5120 81.1 /
//   81.1, 5120 x 1280, M = 6000 80.9 / 77.4).
// - One round is short: M = 3072 of 5120 x 1280 37.9 / 44.1, 12288 of 1280 x
//   1280 38.7 / 40.8, 12288 of 1280 x 2048 56.8 / 57.4, 6144 of 2560 x 3072
//   82.5 / 85.9; 12000 of 1280 x 5120 133 / 130, 10240 of 1536 x 5120 135 /
//   130, 20480 of 768 x 3072 85.4 / 82.5.
bool gemm256_suits(uint32_t m, uint32_t n, uint32_t k) {
  const uint64_t cus = (uint64_t)cu_count() / 8 * 8;
  if (n % kBN || cus == 0 || (uint64_t)n * k * 2 >= kWeightBytes || (uint64_t)n * 512 >= (1ull << 31))
    return false;
  const uint64_t tiles = (uint64_t)((m + kBM - 1) / kBM) * (n / kBN), rounds = (tiles + cus - 1) / cus;
  const uint64_t fused = (uint64_t)((m + 127) / 128) * (n / kBN), fused_rounds = (fused + cus - 1) / cus;
  if (tiles * 10 < rounds * cus * 9 || rounds * 2 * 15 > fused_rounds * 16) return false;
  return rounds >= 2 ? m >= 5120 : m >= 10240 && k >= 3072;
}

int gemm256(const void *a, const uint8_t *qs, const f16 *sc, void *c, const float *bias, uint32_t m,
            uint32_t n, uint32_t k, int epilogue, f16 *w) {
  const uint32_t units = n / kPanelRows * (k / kChunkK);
  hipLaunchKernelGGL(q8_rows_f16_kernel, dim3((units + 3) / 4), dim3(256), 0, stream(), w, qs, sc, k,
                     units);
  if (int rc = check_launch("madi_q8_gemm(rows)")) return rc;
  switch (epilogue) {
  case MADI_EPI_NONE: return launch<MADI_EPI_NONE>(a, w, c, bias, m, n, k);
  case MADI_EPI_BIAS: return launch<MADI_EPI_BIAS>(a, w, c, bias, m, n, k);
  case MADI_EPI_BIAS_GELU: return launch<MADI_EPI_BIAS_GELU>(a, w, c, bias, m, n, k);
  default: return fail(MADI_ERR_ARG, "madi_q8_gemm: unknown epilogue %d", epilogue);
  }
}

}  // namespace madi
