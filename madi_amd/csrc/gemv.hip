// gemv.hip -- decoder Q8 GEMV family (M = 1).
//
// Replaces gemv_q8 / _bias / _bias_gelu / _bias_res / _qkv and logit_gemv_q8
// (engine/metal/kernels/graph_helpers.metal:320-558).  The reference runs one
// 32-lane simdgroup per output row reading char4 + float4; here two kernels
// share the arithmetic and the epilogues.
//
// q8_gemv_kernel, the vocab matrix and other wide ones (HBM-bound): a
// workgroup of four waves (sixteen for 128 to 255 panels of a long K) owns one
// 32-row panel of the panel layout and its waves split K.  Every wave64 load instruction moves one contiguous KiB (16
// bytes per lane, lane (h, r) receiving 16 weights of row r in quantisation
// block h), issued as a buffer load with the panel/chunk offset in an SGPR.
// Each wave streams its K range through a two-chunk window (use chunk c,
// refill with chunk c+2).  Four waves: 62 - 71 VGPRs (seven waves per SIMD
// allow 72), so every workgroup of the 51866-row vocab matrix (1621 panels,
// seven per CU) is resident from the start.
//
// q8_gemv_rows_kernel, the decoder's projections (latency-bound): a workgroup
// owns 8 or 16 rows and all of K (below).
//
// The activation vector is loaded next to the first weights (after them for
// the wide matrices, before them for the narrow ones), staged once per
// workgroup in LDS and read back as broadcast 128-bit LDS loads, ahead of
// the weights they meet.  v_perm_b32 turns two stored bytes u = q + 128 into
// the fp16 pair 1024 + u and one packed subtract of 1152 leaves the exact
// fp16 pair (q0, q1); fp16 activations accumulate x * q with v_dot2_f32_f16
// (exact products, fp32 sums), fp32 activations with FMA.  Each lane's
// partial over (its half of) a quantisation block is multiplied by the
// block's scale, the (partial * scale) structure of the reference's kernels;
// lanes meet by cross-lane operations and waves through LDS.  (Accumulating
// x * (1024 + u) and subtracting 1152 * sum(x) per block saves the subtract
// but cancels two large sums: an all-zero block, whose scale is 1.0, then
// leaks ~1e-2 of rounding noise into its row.)
//
// Kernel arguments: pointers travel as integers and only what a kernel uses
// is passed.  Host cost of a launch (one box, an empty kernel of 40 x 1024
// threads, no argument 1.2 us): ten pointers 3.7 us, the same ten as 64-bit
// integers 2.8 us (the runtime looks every pointer argument up), 64 bytes
// 2.7, 128 bytes 3.4.  At 2.5 - 3.5 us a kernel the decoder's projections
// were bound by that.
#include "common.h"

using namespace madi;

namespace {

// Waves per panel of the wide kernel (seven workgroups per CU), which takes
// matrices of at least kWidePanels panels; and of its form for fewer panels
// of a long K, at most one workgroup per CU.
constexpr int kWaves = 4, kLongWaves = 16;
constexpr uint32_t kWidePanels = 256;
// Chunks in flight per wave, a sliding window: two keeps ~26 MB of the vocab
// matrix in flight across the GPU, enough to cover HBM latency, while the
// texture queues stay short enough that the activation vector (loaded first)
// is not stuck behind a flood of weight requests; deeper windows measured
// slower (the waves then sit blocked on issue and compute in one late burst).
constexpr int kWin = 2;
constexpr uint32_t kMaxK = 12288;


enum GemvMode { kPlain = 0, kBias = 1, kBiasGelu = 2, kBiasRes = 3, kQkv = 4 };

struct GemvArgs {
  float *out;
  const void *x;
  const uint8_t *qs;
  const f16 *sc;
  const float *bias;
  uint32_t n, k;
  // QKV epilogue (graph_helpers.metal:527-558)
  const float *qb, *vb;
  float *kc, *vc;
  const uint32_t *pos;
};

typedef __attribute__((address_space(1))) float gfloat;
typedef __attribute__((address_space(1))) uint32_t guint;
inline uint64_t addr(const void *p) { return reinterpret_cast<uint64_t>(p); }

// LDS bytes of the wide kernel: x (K elements of XT), the KW waves' partials
template <typename XT, int KW>
constexpr size_t lds_bytes(uint32_t k) {
  return (size_t)k * sizeof(XT) + KW * 32 * 4;
}

// One chunk's loads for a lane: its two 16-byte units and its block's scale.
struct ChunkW {
  u32x4 w[2];
  uint32_t s;
};

typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ inline rsrc_t make_rsrc(const void *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)bytes, 0x00020000);
}

// Issue chunk c of panel p (R rows) with buffer loads: the panel and chunk
// offsets are uniform (SGPR) and the lane offsets fixed, so the loads need no
// per-load address arithmetic.
__device__ inline void load_chunk(ChunkW &b, rsrc_t wq, rsrc_t ws, uint32_t K, uint32_t c,
                                  uint32_t p, uint32_t R, uint32_t w_voff, uint32_t s_voff) {
  const uint32_t so = (uint32_t)panel_chunk_qs(K, p, R, c);
  b.w[0] = __builtin_amdgcn_raw_buffer_load_b128(wq, w_voff, so, 0);
  b.w[1] = __builtin_amdgcn_raw_buffer_load_b128(wq, w_voff + 2 * R * 16, so, 0);
  b.s = __builtin_amdgcn_raw_buffer_load_b16(ws, s_voff, (uint32_t)panel_chunk_sc(K, p, R, c) * 2, 0);
}

// sum_i x[i] * q[i] over one 16-byte unit, fp16 activations: v_dot2_f32_f16
// multiplies two exact fp16 pairs (exact products) and adds them in fp32.
__device__ inline float unit_dot(const u32x4 &w, const f16 *x16, float part) {
  const f16x8 xa = *reinterpret_cast<const f16x8 *>(x16);
  const f16x8 xb = *reinterpret_cast<const f16x8 *>(x16 + 8);
  const uint32_t wd[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const f16x8 &xv = d < 2 ? xa : xb;
    const int e = (d & 1) * 4;
    part = __builtin_amdgcn_fdot2(q_pair(wd[d], kSelLo), (f16x2){xv[e], xv[e + 1]}, part, false);
    part = __builtin_amdgcn_fdot2(q_pair(wd[d], kSelHi), (f16x2){xv[e + 2], xv[e + 3]}, part, false);
  }
  return part;
}

// The same sum for fp32 activations: FMA of the fp32 x with the exact q.
__device__ inline float unit_dot(const u32x4 &w, const float *x32, float part) {
  const uint32_t wd[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const f32x4 xv = *reinterpret_cast<const f32x4 *>(x32 + 4 * d);
    const f16x2 q01 = q_pair(wd[d], kSelLo), q23 = q_pair(wd[d], kSelHi);
    part = __builtin_fmaf(xv.x, (float)q01.x, part);
    part = __builtin_fmaf(xv.y, (float)q01.y, part);
    part = __builtin_fmaf(xv.z, (float)q23.x, part);
    part = __builtin_fmaf(xv.w, (float)q23.y, part);
  }
  return part;
}

// One 16-weight unit's fp32 activations in registers, and its sum against
// them (the same FMA order as unit_dot).
struct XUnit {
  f32x4 v[4];
};
__device__ inline XUnit read_unit(const float *x32) {
  XUnit u;
#pragma unroll
  for (int d = 0; d < 4; ++d) u.v[d] = *reinterpret_cast<const f32x4 *>(x32 + 4 * d);
  return u;
}
__device__ inline float unit_dot(const u32x4 &w, const XUnit &x, float part) {
  const uint32_t wd[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const f16x2 q01 = q_pair(wd[d], kSelLo), q23 = q_pair(wd[d], kSelHi);
    part = __builtin_fmaf(x.v[d].x, (float)q01.x, part);
    part = __builtin_fmaf(x.v[d].y, (float)q01.y, part);
    part = __builtin_fmaf(x.v[d].z, (float)q23.x, part);
    part = __builtin_fmaf(x.v[d].w, (float)q23.y, part);
  }
  return part;
}

// acc += scale * (sum_k x[k] q[k]) over the lane's quantisation block, its
// 32 activations at xp (LDS, or registers)
template <typename XT>
__device__ inline void accumulate_x(const ChunkW &b, const XT *xp, float &acc) {
  float part = unit_dot(b.w[0], xp, 0.0f);
  part = unit_dot(b.w[1], xp + 16, part);
  acc = __builtin_fmaf(part, (float)__builtin_bit_cast(f16, (uint16_t)b.s), acc);
}
// the same over the lane's block of chunk c, x in LDS
template <typename XT>
__device__ inline void accumulate(const ChunkW &b, uint32_t c, const XT *xs, uint32_t h,
                                  float &acc) {
  accumulate_x(b, xs + c * kChunkK + h * 32, acc);
}

// The epilogue's operands of one output row, loaded behind the first weights
// so their latency passes during the K loop, and its store.
struct RowEpi {
  float bias = 0.0f, res = 0.0f;
  uint32_t pos = 0;
};
template <int MODE>
__device__ inline RowEpi epi_load(bool mine, uint32_t row, uint32_t K, const gfloat *out,
                                  const gfloat *bias, const gfloat *vb, const guint *pos) {
  RowEpi e;
  if (mine) {
    if constexpr (MODE == kBias || MODE == kBiasGelu) {
      e.bias = bias[row];
    } else if constexpr (MODE == kBiasRes) {
      e.bias = bias[row];
      e.res = out[row];
    } else if constexpr (MODE == kQkv) {  // bias: q's
      if (row < K) e.bias = bias[row];
      else if (row >= 2 * K) e.bias = vb[row - 2 * K];
    }
  }
  if constexpr (MODE == kQkv) e.pos = pos[0];
  return e;
}
template <int MODE>
__device__ inline void epi_store(float v, const RowEpi &e, uint32_t row, uint32_t K, gfloat *out,
                                 gfloat *kc, gfloat *vc) {
  if constexpr (MODE == kPlain) {
    out[row] = v;
  } else if constexpr (MODE == kBias) {
    out[row] = v + e.bias;
  } else if constexpr (MODE == kBiasGelu) {
    out[row] = gelu_erf(v + e.bias);
  } else if constexpr (MODE == kBiasRes) {
    out[row] = e.res + v + e.bias;
  } else {  // kQkv: n = 3 D, K = D
    if (row < K)
      out[row] = v + e.bias;
    else if (row < 2 * K)
      kc[(size_t)e.pos * K + (row - K)] = v;
    else
      vc[(size_t)e.pos * K + (row - 2 * K)] = v + e.bias;
  }
}

template <typename XT>
constexpr bool kBlockF32 = sizeof(XT) == 4;

// Grid: one workgroup of KW waves per panel.  bias is q's for the QKV mode.
template <typename XT, int MODE, int KW>
__global__ __launch_bounds__(KW * 64) __attribute__((amdgpu_waves_per_eu(KW == kWaves ? 7 : 4))) void q8_gemv_kernel(
    uint64_t qs_, uint64_t sc_, uint64_t x_, uint32_t n, uint32_t K, uint64_t out_, uint64_t bias_,
    uint64_t vb_, uint64_t kc_, uint64_t vc_, uint64_t pos_) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  XT *xs = reinterpret_cast<XT *>(smem);                        // [K]
  float *red = reinterpret_cast<float *>(smem + (size_t)K * sizeof(XT));  // [KW][32]

  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t h = lane >> 5, r = lane & 31;
  const uint32_t p = blockIdx.x;
  const uint32_t R = panel_rows(n, p);
  const bool live = r < R;
  const uint32_t chunks = K / kChunkK;
  const uint32_t c0 = (wave * chunks) / KW, c1 = ((wave + 1) * chunks) / KW;

  // ---- Four waves: the first weight window, then x (16 bytes per thread and
  // piece), so the HBM requests leave before the L2-resident vector's
  // (alternating runs in one process: 12.16 -> 11.92 us with f16 x, 12.66 ->
  // 12.35 us with f32 x).  Sixteen: x first, whose staging barrier is then the
  // longer wait.  Lanes past a partial panel's last row read row R-1 (in
  // bounds; their sums are never stored).
  constexpr bool kWeightsFirst = KW == kWaves;
  const uint32_t pieces = K * sizeof(XT) / 16;
  const rsrc_t xr = make_rsrc((const void *)x_, K * sizeof(XT));
  u32x4 xv0 = {}, xv1 = {};
  const uint32_t i0 = threadIdx.x, i1 = threadIdx.x + KW * 64;
  if constexpr (!kWeightsFirst) {
    if (i0 < pieces) xv0 = __builtin_amdgcn_raw_buffer_load_b128(xr, i0 * 16, 0, 0);
    if (i1 < pieces) xv1 = __builtin_amdgcn_raw_buffer_load_b128(xr, i1 * 16, 0, 0);
  }
  const rsrc_t wq = make_rsrc((const void *)qs_, n * K), ws = make_rsrc((const void *)sc_, n * (K / 32) * 2);
  // chunks past the wave's range load through an empty resource: no memory
  // access, zeros returned, so their scale is 0 and they add exactly nothing.
  // Every window load is then unconditional, which keeps each window slot in
  // the same registers from trip to trip (a conditional load makes the
  // compiler copy the slot at the loop back edge, and a copy must first wait
  // for the load that was just issued, collapsing the window).
  const rsrc_t wz = make_rsrc((const void *)qs_, 0);
  const uint32_t rr = live ? r : R - 1;
  const uint32_t w_voff = (h * R + rr) * 16, s_voff = (h * R + rr) * 2;
  // the first kWin chunks of this wave's range
  ChunkW win[kWin];
#pragma unroll
  for (int k = 0; k < kWin; ++k) {
    const bool in = c0 + k < c1;
    load_chunk(win[k], in ? wq : wz, in ? ws : wz, K, c0 + k, p, R, w_voff, s_voff);
  }
  if constexpr (kWeightsFirst) {
    if (i0 < pieces) xv0 = __builtin_amdgcn_raw_buffer_load_b128(xr, i0 * 16, 0, 0);
    if (i1 < pieces) xv1 = __builtin_amdgcn_raw_buffer_load_b128(xr, i1 * 16, 0, 0);
  }

  // lanes 0..R-1 of wave 0 own the panel's rows
  const uint32_t erow = p * kPanelRows + threadIdx.x;
  const RowEpi epi = epi_load<MODE>(threadIdx.x < R, erow, K, (const gfloat *)out_, (const gfloat *)bias_,
                                    (const gfloat *)vb_, (const guint *)pos_);

  // stage x
  for (uint32_t i = threadIdx.x; i < pieces; i += KW * 64) {
    const u32x4 v =
        i == i0 ? xv0 : (i == i1 ? xv1 : __builtin_amdgcn_raw_buffer_load_b128(xr, i * 16, 0, 0));
    reinterpret_cast<u32x4 *>(xs)[i] = v;
  }
  __syncthreads();

  // stream the range through the kWin-chunk window: use chunk c, refill its
  // registers with chunk c + kWin
  float acc = 0.0f;
  uint32_t cfirst = c0;
  if constexpr (KW == kLongWaves) {
    // Sixteen waves: the first window's activations are read from LDS now,
    // while its weights are still in flight, instead of after they land, when
    // all the waves would queue at the LDS at once.
    if (c0 < c1) {
      XT xf[kWin][32];
#pragma unroll
      for (int k = 0; k < kWin; ++k) {
        const uint32_t cc = c0 + k < c1 ? c0 + k : c1 - 1;
#pragma unroll
        for (int i = 0; i < 32; ++i) xf[k][i] = xs[cc * kChunkK + h * 32 + i];
      }
      // the reads stay ahead of the first wait for the weights
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < kWin; ++k) {
        // (a chunk past the range adds nothing where x is infinite either)
        const float before = acc;
        accumulate_x<XT>(win[k], xf[k], acc);
        acc = c0 + k < c1 ? acc : before;
        const uint32_t cn = c0 + k + kWin;
        const bool in = cn < c1;
        load_chunk(win[k], in ? wq : wz, in ? ws : wz, K, cn, p, R, w_voff, s_voff);
        __builtin_amdgcn_sched_barrier(0);
      }
      cfirst = c0 + kWin < c1 ? c0 + kWin : c1;
    }
  }
  if constexpr (KW == kWaves && kBlockF32<XT>) {
    // The vocab matrix with fp32 activations: each unit's activations are
    // read from LDS one unit ahead of their use (the next chunk's first unit
    // during this chunk's second), so the LDS latency passes under the
    // arithmetic; a whole chunk ahead would not fit the 72 VGPRs that keep
    // seven waves per SIMD.
    const float *xf = reinterpret_cast<const float *>(xs) + h * 32;
    XUnit xa = read_unit(xf + (c0 < c1 ? c0 : 0) * kChunkK);
#pragma unroll 1
    for (uint32_t c = c0; c < c1; c += kWin) {
#pragma unroll
      for (int k = 0; k < kWin; ++k) {
        const uint32_t cc = c + k < c1 ? c + k : c1 - 1;
        const uint32_t cx = c + k + 1 < c1 ? c + k + 1 : c1 - 1;  // the next slot's chunk
        // each read is issued before the arithmetic that precedes its use
        const XUnit xb = read_unit(xf + cc * kChunkK + 16);
        __builtin_amdgcn_sched_barrier(0);
        float part = unit_dot(win[k].w[0], xa, 0.0f);
        __builtin_amdgcn_sched_barrier(0);
        xa = read_unit(xf + cx * kChunkK);
        __builtin_amdgcn_sched_barrier(0);
        part = unit_dot(win[k].w[1], xb, part);
        acc = __builtin_fmaf(part, (float)__builtin_bit_cast(f16, (uint16_t)win[k].s), acc);
        const uint32_t cn = c + k + kWin;
        const bool in = cn < c1;
        load_chunk(win[k], in ? wq : wz, in ? ws : wz, K, cn, p, R, w_voff, s_voff);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    cfirst = c1;
  }
  // whole windows, then (sixteen waves) the last one's chunks by themselves:
  // a slot past the range adds nothing there even where x is infinite
  const uint32_t cend = KW == kLongWaves ? c1 - (c1 - cfirst) % kWin : c1;
#pragma unroll 1
  for (uint32_t c = cfirst; c < cend; c += kWin) {
#pragma unroll
    for (int k = 0; k < kWin; ++k) {
      // a chunk past the range (zeros, scale 0) reads the x of the range's
      // last chunk, so its partial stays finite and 0 * partial is exact
      const uint32_t cc = c + k < c1 ? c + k : c1 - 1;
      accumulate<XT>(win[k], cc, xs, h, acc);
      const uint32_t cn = c + k + kWin;
      const bool in = cn < c1;
      load_chunk(win[k], in ? wq : wz, in ? ws : wz, K, cn, p, R, w_voff, s_voff);
      // keep the next slot's math behind this reload: interleaved, both
      // slots would have to land before either is reissued
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if constexpr (KW == kLongWaves) {
#pragma unroll
    for (int k = 0; k < kWin - 1; ++k)
      if (cend + k < c1) accumulate<XT>(win[k], cend + k, xs, h, acc);
  }

  acc += __shfl_xor(acc, 32);
  if (h == 0) red[wave * 32 + r] = acc;
  __syncthreads();
  const uint32_t t = threadIdx.x;
  if (t >= R) return;
  float v = red[t];  // the waves' partials in wave order
#pragma unroll
  for (int w = 1; w < KW; ++w) v += red[w * 32 + t];
  epi_store<MODE>(v, epi, erow, K, (gfloat *)out_, (gfloat *)kc_, (gfloat *)vc_);
}

// ---- narrow matrices (fewer than kWidePanels panels: the decoder's
// projections), one workgroup per 8 NR rows.
//
// These are 1.7 - 7 MB each, so a launch is latency and, per CU, arithmetic:
// a workgroup per 32-row panel left a 1280-row projection on 40 of the 256
// CUs with four waves per SIMD of dequantisation and FMAs, and a K of 5120
// had to be split over workgroups that met through memory.  Here a wave's
// load takes 8 rows x 2 chunks (eight whole 128-byte lines of the panel
// layout: lane (u, row) gets unit u % 4 of chunk u / 4), so a workgroup can
// own as few as 8 rows with all of K, and its waves meet in LDS only.
constexpr int kRowWaves = 16;

// One pair of chunks: NR row groups' units and scales.
template <int NR>
struct PairW {
  u32x4 w[NR];
  uint32_t s[NR];
};

__device__ inline float xunit_dot(const u32x4 &w, const f32x4 (&x)[4]) {
  const uint32_t wd[4] = {w.x, w.y, w.z, w.w};
  float part = 0.0f;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const f16x2 q01 = q_pair(wd[d], kSelLo), q23 = q_pair(wd[d], kSelHi);
    part = __builtin_fmaf(x[d].x, (float)q01.x, part);
    part = __builtin_fmaf(x[d].y, (float)q01.y, part);
    part = __builtin_fmaf(x[d].z, (float)q23.x, part);
    part = __builtin_fmaf(x[d].w, (float)q23.y, part);
  }
  return part;
}
__device__ inline float xunit_dot(const u32x4 &w, const f16x8 (&x)[2]) {
  const uint32_t wd[4] = {w.x, w.y, w.z, w.w};
  float part = 0.0f;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const f16x8 &xv = x[d / 2];
    const int e = (d & 1) * 4;
    part = __builtin_amdgcn_fdot2(q_pair(wd[d], kSelLo), (f16x2){xv[e], xv[e + 1]}, part, false);
    part = __builtin_amdgcn_fdot2(q_pair(wd[d], kSelHi), (f16x2){xv[e + 2], xv[e + 3]}, part, false);
  }
  return part;
}
template <typename XT>
struct XUnitOf;
template <>
struct XUnitOf<float> {
  f32x4 v[4];
};
template <>
struct XUnitOf<f16> {
  f16x8 v[2];
};
__device__ inline void read_x(XUnitOf<float> &u, const float *x) {
#pragma unroll
  for (int i = 0; i < 4; ++i) u.v[i] = *reinterpret_cast<const f32x4 *>(x + 4 * i);
}
__device__ inline void read_x(XUnitOf<f16> &u, const f16 *x) {
#pragma unroll
  for (int i = 0; i < 2; ++i) u.v[i] = *reinterpret_cast<const f16x8 *>(x + 8 * i);
}

// the sum over the lanes with the same lane % 8
__device__ inline float sum_units(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x128, 0xf,
                                                             0xf, true));  // row_ror:8
  const uint32_t a = __builtin_bit_cast(uint32_t, v);
  const auto s16 = __builtin_amdgcn_permlane16_swap(a, a, false, false);
  v = __builtin_bit_cast(float, (uint32_t)s16[0]) + __builtin_bit_cast(float, (uint32_t)s16[1]);
  const uint32_t b = __builtin_bit_cast(uint32_t, v);
  const auto s32 = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  return __builtin_bit_cast(float, (uint32_t)s32[0]) + __builtin_bit_cast(float, (uint32_t)s32[1]);
}

constexpr uint32_t kNowhere = 0x80000000u;  // past every buffer (operands stay below 2 GiB)

template <typename XT, int MODE, int NR, int WIN, bool ONE>
__device__ inline void gemv_rows(uint64_t x_, uint64_t qs_, uint32_t n, uint32_t K, uint64_t sc_,
                                 uint64_t out_, uint64_t bias_, uint64_t vb_, uint64_t kc_, uint64_t vc_,
                                 uint64_t pos_) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  XT *xs = reinterpret_cast<XT *>(smem);                                  // [K]
  float *red = reinterpret_cast<float *>(smem + (size_t)K * sizeof(XT));  // [waves][8 NR]
  constexpr uint32_t kRows = 8 * NR;
  const uint32_t chunks = K / kChunkK, pairs = (chunks + 1) / 2;
  const uint32_t waves = ONE ? (pairs + WIN - 1) / WIN : kRowWaves, threads = waves * 64;
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t row0 = blockIdx.x * kRows;  // of 32-row panel p
  const uint32_t p = row0 / kPanelRows, R = panel_rows(n, p);

  // x first: its staging barrier is the longer wait
  const uint32_t pieces = K * sizeof(XT) / 16;
  const rsrc_t xr = make_rsrc((const void *)x_, K * sizeof(XT));
  u32x4 xv0 = {}, xv1 = {};
  const uint32_t i0 = threadIdx.x, i1 = threadIdx.x + threads;
  if (i0 < pieces) xv0 = __builtin_amdgcn_raw_buffer_load_b128(xr, i0 * 16, 0, 0);
  if (i1 < pieces) xv1 = __builtin_amdgcn_raw_buffer_load_b128(xr, i1 * 16, 0, 0);

  // lane (u, r8): unit (j, h) = (u / 2 % 2, u % 2) of chunk 2 pair + u / 4,
  // row r8 of each group.  Rows past a partial panel's last read row R - 1
  // (never stored).
  const uint32_t u = lane >> 3, cp = u >> 2, j = (u >> 1) & 1, h = u & 1;
  const rsrc_t wq = make_rsrc((const void *)qs_, n * K), ws = make_rsrc((const void *)sc_, n * (K / 32) * 2);
  const rsrc_t wz = make_rsrc((const void *)qs_, 0);
  uint32_t w_voff[NR], s_voff[NR];
#pragma unroll
  for (int g = 0; g < NR; ++g) {
    const uint32_t want = row0 % kPanelRows + 8 * g + (lane & 7), r = want < R ? want : R - 1;
    w_voff[g] = cp * R * kChunkK + ((2 * j + h) * R + r) * 16;
    s_voff[g] = cp * R * 4 + (h * R + r) * 2;
  }
  // Pairs past the range load through an empty resource and the missing
  // second chunk of an odd last pair at an offset outside the range.
  PairW<NR> win[WIN];
  auto load = [&](PairW<NR> &b, uint32_t pr) {
    const bool in = pr < pairs, none = 2 * pr + cp >= chunks;
    const uint32_t so = (uint32_t)panel_chunk_qs(K, p, R, 2 * pr);
    const uint32_t ss = (uint32_t)panel_chunk_sc(K, p, R, 2 * pr) * 2;
#pragma unroll
    for (int g = 0; g < NR; ++g) {
      b.w[g] = __builtin_amdgcn_raw_buffer_load_b128(in ? wq : wz, none ? kNowhere : w_voff[g], so, 0);
      b.s[g] = __builtin_amdgcn_raw_buffer_load_b16(in ? ws : wz, none ? kNowhere : s_voff[g], ss, 0);
    }
  };
#pragma unroll
  for (int k = 0; k < WIN; ++k) load(win[k], wave + k * waves);

  const uint32_t erow = row0 + threadIdx.x;
  const bool mine = threadIdx.x < kRows && erow < n;
  const RowEpi epi = epi_load<MODE>(mine, erow, K, (const gfloat *)out_, (const gfloat *)bias_,
                                    (const gfloat *)vb_, (const guint *)pos_);

  for (uint32_t i = threadIdx.x; i < pieces; i += threads) {
    const u32x4 v =
        i == i0 ? xv0 : (i == i1 ? xv1 : __builtin_amdgcn_raw_buffer_load_b128(xr, i * 16, 0, 0));
    reinterpret_cast<u32x4 *>(xs)[i] = v;
  }
  __syncthreads();

  float acc[NR];
#pragma unroll
  for (int g = 0; g < NR; ++g) acc[g] = 0.0f;
#pragma unroll 1
  for (uint32_t base = wave;;) {
    // the window's x is read while its weights are in flight (a missing chunk
    // reads the last one's, and its sum is dropped)
    XUnitOf<XT> xu[WIN];
#pragma unroll
    for (int k = 0; k < WIN; ++k) {
      const uint32_t want = 2 * (base + k * waves) + cp, c = want < chunks ? want : chunks - 1;
      read_x(xu[k], xs + c * kChunkK + h * 32 + j * 16);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < WIN; ++k) {
      const bool real = 2 * (base + k * waves) + cp < chunks;
#pragma unroll
      for (int g = 0; g < NR; ++g) {
        const float sum = __builtin_fmaf(xunit_dot(win[k].w[g], xu[k].v),
                                         (float)__builtin_bit_cast(f16, (uint16_t)win[k].s[g]), acc[g]);
        acc[g] = real ? sum : acc[g];
      }
      if constexpr (!ONE) {
        load(win[k], base + (k + WIN) * waves);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if constexpr (ONE) break;
    base += WIN * waves;
    if (base >= pairs) break;
  }
#pragma unroll
  for (int g = 0; g < NR; ++g) {
    const float v = sum_units(acc[g]);
    if (lane < 8) red[wave * kRows + 8 * g + lane] = v;
  }
  __syncthreads();
  if (!mine) return;
  float v = red[threadIdx.x];  // the waves' partials in wave order
  for (uint32_t w = 1; w < waves; ++w) v += red[w * kRows + threadIdx.x];
  epi_store<MODE>(v, epi, erow, K, (gfloat *)out_, (gfloat *)kc_, (gfloat *)vc_);
}

// 48 bytes of arguments; the QKV mode's four more in a kernel of its own.
template <typename XT, int MODE, int NR, int WIN, bool ONE>
__global__ __launch_bounds__(kRowWaves * 64) void q8_gemv_rows_kernel(uint64_t x, uint64_t qs, uint32_t n,
                                                                      uint32_t K, uint64_t sc, uint64_t out,
                                                                      uint64_t bias) {
  gemv_rows<XT, MODE, NR, WIN, ONE>(x, qs, n, K, sc, out, bias, 0, 0, 0, 0);
}
template <typename XT, int NR, int WIN, bool ONE>
__global__ __launch_bounds__(kRowWaves * 64) void q8_gemv_rows_qkv_kernel(
    uint64_t x, uint64_t qs, uint32_t n, uint32_t K, uint64_t sc, uint64_t out, uint64_t qb, uint64_t vb,
    uint64_t kc, uint64_t vc, uint64_t pos) {
  gemv_rows<XT, kQkv, NR, WIN, ONE>(x, qs, n, K, sc, out, qb, vb, kc, vc, pos);
}

template <typename XT, int MODE, int NR, int WIN, bool ONE>
void launch_rows(const GemvArgs &a) {
  const uint32_t pairs = (a.k / kChunkK + 1) / 2, waves = ONE ? (pairs + WIN - 1) / WIN : kRowWaves;
  const dim3 grid((a.n + 8 * NR - 1) / (8 * NR)), block(waves * 64);
  const size_t lds = a.k * sizeof(XT) + waves * 8 * NR * 4;
  if constexpr (MODE == kQkv)
    hipLaunchKernelGGL((q8_gemv_rows_qkv_kernel<XT, NR, WIN, ONE>), grid, block, lds, stream(), addr(a.x),
                       addr(a.qs), a.n, a.k, addr(a.sc), addr(a.out), addr(a.qb), addr(a.vb), addr(a.kc),
                       addr(a.vc), addr(a.pos));
  else
    hipLaunchKernelGGL((q8_gemv_rows_kernel<XT, MODE, NR, WIN, ONE>), grid, block, lds, stream(), addr(a.x),
                       addr(a.qs), a.n, a.k, addr(a.sc), addr(a.out), addr(a.bias));
}

// Rows per workgroup: 8 while that is at most one workgroup per CU or so,
// else 16, which halve the x staged per weight (issued from C, us, 8 / 16 /
// 32 rows: 1280 x 1280 2.5 / 2.7 / -, 3840 x 1280 4.1 / 2.7 / 3.1, 5120 x
// 1280 5.5 / 3.0 / 3.3, 1280 x 5120 3.6 / 4.5 / -).  The line is that of K =
// 1280: past K = 4096, where a workgroup holds its CU, 16 rows lead from 2049
// on (2304 x 5120 with 8 7.2, 2305 x 5120 with 16 5.7).  One pair of chunks per
// wave up to K = 2048; three, all in flight at once, above (1280 x 1280 with
// two or three per wave 2.8); past 6144 sixteen waves go round.
constexpr uint32_t kRows8 = 2304;
template <typename XT, int MODE, int NR>
void pick_rows(const GemvArgs &a) {
  const uint32_t pairs = (a.k / kChunkK + 1) / 2;
  if (pairs <= kRowWaves) launch_rows<XT, MODE, NR, 1, true>(a);
  else if (pairs <= 3 * kRowWaves) launch_rows<XT, MODE, NR, 3, true>(a);
  else launch_rows<XT, MODE, NR, 3, false>(a);
}

template <typename XT, int MODE, int KW>
void launch_panels(const GemvArgs &a, uint32_t np) {
  hipLaunchKernelGGL((q8_gemv_kernel<XT, MODE, KW>), dim3(np), dim3(KW * 64), (lds_bytes<XT, KW>(a.k)),
                     stream(), addr(a.qs), addr(a.sc), addr(a.x), a.n, a.k, addr(a.out),
                     addr(MODE == kQkv ? a.qb : a.bias), addr(a.vb), addr(a.kc), addr(a.vc), addr(a.pos));
}

// From 128 panels of a K past 1536 sixteen waves per panel are the faster
// form: 16 rows per workgroup would be 256 workgroups and more, which hold a
// CU each at the registers and waves of a long K, in two rounds, each staging
// all of x.  (Issued from C, us, 16 waves per panel / 16 rows: 4608 x 1536
// 3.6 / 3.5, x 1920 3.8 / 4.0, x 3072 5.4 / 6.1, x 4096 5.8 / 9.4, 5120 x 5120
// 7.3 / 11.1, 8160 x 1280 4.0 / 3.9, x 2048 5.2 / 5.5, x 6144 10.9 / 14.6;
// 4064 x 4096, in four splits then, 10.3 / 6.3.)
constexpr uint32_t kLongPanels = 128, kLongK = 1536;

template <typename XT, int MODE>
int launch(const char *what, const GemvArgs &a) {
  if (!a.out || !a.x || !a.qs || !a.sc) return fail(MADI_ERR_NULL, "%s: null pointer", what);
  if ((MODE == kBias || MODE == kBiasGelu || MODE == kBiasRes) && !a.bias)
    return fail(MADI_ERR_NULL, "%s: null bias", what);
  if (a.n == 0 || a.k == 0 || a.k % kChunkK)
    return fail(MADI_ERR_SHAPE, "%s: n=%u k=%u (need n > 0, k a positive multiple of 64)", what, a.n, a.k);
  if (a.k > kMaxK) return fail(MADI_ERR_SHAPE, "%s: k=%u exceeds %u", what, a.k, kMaxK);
  // buffer ranges and offsets are 32-bit: the weight (n*k bytes) must stay
  // below 2 GiB, as for the GEMM and the batched projection
  if ((uint64_t)a.n * a.k >= (1ull << 31))
    return fail(MADI_ERR_SHAPE, "%s: n=%u k=%u exceeds the 2 GiB operand limit", what, a.n, a.k);
  if (!aligned(a.qs, 16) || !aligned(a.sc, 2) || !aligned(a.x, 16))
    return fail(MADI_ERR_ALIGN, "%s: qs and x need 16-byte alignment", what);
  if (!initialized()) return fail(MADI_ERR_NOT_INIT, "%s: madi_init has not succeeded", what);
  if (int rc = deferred_before_read(a.x, (size_t)a.k * sizeof(XT))) return rc;
  if (MODE == kQkv) {
    // q_out [D], and one row of each cache at a position only the device
    // knows: somewhere in the allocation from kc (vc) on, if the library
    // allocated it, else at least the first row
    const size_t row = (size_t)(a.n / 3) * 4;
    const size_t kext = alloc_extent(a.kc), vext = alloc_extent(a.vc);
    if (int rc = deferred_before_write(a.out, row)) return rc;
    if (int rc = deferred_before_write(a.kc, kext > row ? kext : row)) return rc;
    if (int rc = deferred_before_write(a.vc, vext > row ? vext : row)) return rc;
  } else if (int rc = deferred_before_write(a.out, (size_t)a.n * 4)) {
    return rc;
  }
  const uint32_t np = (a.n + kPanelRows - 1) / kPanelRows;
  if (np >= kWidePanels)
    launch_panels<XT, MODE, kWaves>(a, np);
  else if (np >= kLongPanels && a.k > kLongK)
    launch_panels<XT, MODE, kLongWaves>(a, np);
  else if (a.n > kRows8)
    pick_rows<XT, MODE, 2>(a);
  else
    pick_rows<XT, MODE, 1>(a);
  return check_launch(what);
}

GemvArgs args(float *out, const void *x, const void *qs, const void *scales, const float *bias,
              uint32_t n, uint32_t k) {
  GemvArgs a{};
  a.out = out;
  a.x = x;
  a.qs = static_cast<const uint8_t *>(qs);
  a.sc = static_cast<const f16 *>(scales);
  a.bias = bias;
  a.n = n;
  a.k = k;
  return a;
}

}  // namespace

extern "C" int madi_q8_gemv(float *out, const float *x, const void *qs, const void *scales,
                            uint32_t n, uint32_t k) {
  return launch<float, kPlain>("madi_q8_gemv", args(out, x, qs, scales, nullptr, n, k));
}

extern "C" int madi_q8_gemv_bias(float *out, const float *x, const void *qs, const void *scales,
                                 const float *bias, uint32_t n, uint32_t k) {
  return launch<float, kBias>("madi_q8_gemv_bias", args(out, x, qs, scales, bias, n, k));
}

extern "C" int madi_q8_gemv_bias_gelu(float *out, const float *x, const void *qs,
                                      const void *scales, const float *bias, uint32_t n,
                                      uint32_t k) {
  return launch<float, kBiasGelu>("madi_q8_gemv_bias_gelu", args(out, x, qs, scales, bias, n, k));
}

extern "C" int madi_q8_gemv_bias_res(float *out, const float *x, const void *qs,
                                     const void *scales, const float *bias, uint32_t n,
                                     uint32_t k) {
  return launch<float, kBiasRes>("madi_q8_gemv_bias_res", args(out, x, qs, scales, bias, n, k));
}

extern "C" int madi_q8_gemv_qkv(float *q_out, const float *x, const void *qs, const void *scales,
                                const float *qb, const float *vb, float *kc, float *vc,
                                const uint32_t *pos, uint32_t d) {
  if (!qb || !vb || !kc || !vc || !pos) return fail(MADI_ERR_NULL, "madi_q8_gemv_qkv: null pointer");
  if (d == 0 || d % kChunkK) return fail(MADI_ERR_SHAPE, "madi_q8_gemv_qkv: d=%u must be a positive multiple of 64", d);
  GemvArgs a = args(q_out, x, qs, scales, nullptr, 3 * d, d);
  a.qb = qb;
  a.vb = vb;
  a.kc = kc;
  a.vc = vc;
  a.pos = pos;
  return launch<float, kQkv>("madi_q8_gemv_qkv", a);
}

extern "C" int madi_q8_logit_gemv(float *logits, const void *qs, const void *scales,
                                  const float *x, uint32_t vocab, uint32_t dim) {
  return launch<float, kPlain>("madi_q8_logit_gemv", args(logits, x, qs, scales, nullptr, vocab, dim));
}

extern "C" int madi_q8_gemv_f16x(float *out, const void *x_f16, const void *qs,
                                 const void *scales, const float *bias, uint32_t n, uint32_t k,
                                 int epilogue) {
  const GemvArgs a = args(out, x_f16, qs, scales, bias, n, k);
  switch (epilogue) {
  case MADI_EPI_NONE: return launch<f16, kPlain>("madi_q8_gemv_f16x", a);
  case MADI_EPI_BIAS: return launch<f16, kBias>("madi_q8_gemv_f16x", a);
  case MADI_EPI_BIAS_GELU: return launch<f16, kBiasGelu>("madi_q8_gemv_f16x", a);
  case MADI_EPI_BIAS_RES: return launch<f16, kBiasRes>("madi_q8_gemv_f16x", a);
  default: return fail(MADI_ERR_ARG, "madi_q8_gemv_f16x: unknown epilogue %d", epilogue);
  }
}
