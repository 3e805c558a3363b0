// Backbone decode GEMVs for gfx950 (include/bz_gemv.h): the reference's flash_bb_fused (flash/csrc/bb_fused.cu).
//
// y[m, n] = epilogue(sum_k xin[m, k] * W[n, k]) for the decode step's M <= 4 rows: weight-streaming and HBM-bound
// (each weight byte is used M times, 2 FLOPs each). The work is laid out for the weights:
//   - a wave owns R output rows (2 R weight rows for the SiLU * up epilogue: gate and up of the same outputs) and
//     streams them whole; lane l reads the 16 bytes at k = 8 l + 512 c of every chunk c, so one wave load instruction
//     covers 1 KiB of one weight row. Rows are raw buffer resources cut at k (and empty past the last output row), so
//     every load is unconditional, nothing past a row is read, and the compiler's vmcnt accounting stays exact.
//   - two tiles of R x U chunks are in flight (ping-pong); the first two are issued before the x prologue, after x's
//     own loads, so the prologue waits for x alone.
//   - x (RMSNorm'ed at the eager rounding points when asked) is held in registers when it fits (k <= 1024, or
//     k <= 2048 with M <= 2: every lane keeps its own 16 bytes of each chunk, and the norm's sum of squares is reduced
//     over the wave, so there is no LDS and no barrier); otherwise it is staged once per workgroup in LDS,
//     zero-padded to a multiple of the tile, and read with one ds_read_b128 per chunk and row of x.
//   - products: four v_dot2c_f32_bf16 per 16 bytes (bf16 x bf16 exact, fp32 accumulation); the R * M (2 R * M)
//     accumulators are summed over the wave with DPP inside 16-lane rows and transposed permlane swaps across rows,
//     so each lane of a row ends with one finished output, written with the epilogue by that row's first lane.
// The weight loads carry the non-temporal hint: 2.8 GB of weights stream through per decode step.
// Where it measured faster (4096 < k <= 6144 at any M, the backbone's down projection; 1024 < k <= 2048 at M >= 3)
// a block-ordered kernel runs instead: a workgroup streams its rows as one contiguous block, every thread holding one
// x vector for all of its rows, and the sums are reduced over the workgroup once, at the end (gemv_block_kernel).
// A third kernel works the products out on the 4x4x4 MFMA, four weight rows per load (gemv_mfma_kernel): for
// 2048 < k <= 4096, most of SiLU * up and plain at M >= 3 (mfma_route).
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>

#include "bz_gemv.h"
#include "device_common.cuh"

namespace bz {
int device_cu_count(int* cus);  // gqa_decode.hip: the current device's CU count, cached per device
}  // namespace bz

namespace {

constexpr int kGemvThreads = 256;              // 4 waves per workgroup (x in registers; rmsnorm)
constexpr int kGemvWaves = kGemvThreads / kWave;
// Threads of a workgroup that stages x in LDS: eight waves share one copy of x (down: 6.47 against 6.9 us with
// four); with x in registers every wave loads its own, and four waves per workgroup measured fastest.
constexpr int kGemvLdsThreads = 512;
template <int KC>
constexpr int gemv_threads() { return KC > 0 ? kGemvThreads : kGemvLdsThreads; }
constexpr int kChunk = 8 * kWave;              // k elements per wave load instruction
constexpr int kU = 2;                          // chunks per tile
constexpr int kTileK = kChunk * kU;            // k elements per tile
constexpr int kMaxLds = 64 * 1024;             // bytes of LDS for x
// With x in registers every wave issues all its weight loads at once; spacing them by s_sleep(kIssueGap) (about
// 64 * kIssueGap clocks) measured faster where the loads queue: q|k|v 5.06 against 5.19 us, gate/up 10.0 against
// 10.3-10.5. Gaps of 1, 3, 4 and 6 were tried; 2 was best or within noise of best. A small grid just waits longer for
// its last load (gate/up, M = 2, k = 2048: 12 workgroups 3.43 against 2.89 us, 32 workgroups 4.05 against 3.92, 128
// workgroups 4.25 against 4.43), and so does a grid of one workgroup per CU whose waves issue few loads (o_proj, 256
// workgroups of eight 1 KiB loads per wave: 3.31 us unpaced against 3.64 paced; q|k|v at two workgroups per CU 4.89
// either way; gate/up, 16 loads per wave, 9.68 paced against 9.96). So the host picks the paced variant (GAP =
// kIssueGap) for grids of at least kPaceMinGrid workgroups whose waves issue at least kPaceMinLoads weight loads each
// or that hold more workgroups than the device has CUs. The gap is a template parameter, not a runtime flag: a branch
// around each s_sleep split the loads over basic blocks, and the compiler's wait counts then went pessimistic (the
// prologue waited for three more weight loads than it needs).
constexpr int kIssueGap = 2;
constexpr int kPaceMinGrid = 64;
constexpr int kPaceMinLoads = 16;

struct GemvParams {
  const uint16_t* x;
  int64_t ldx;
  const uint16_t* nw;
  float eps;
  const uint16_t* w0;
  const uint16_t* w1;
  const uint16_t* w2;
  int n0, n1, ntot;  // rows of segments 0 and 1; output rows
  int k, kp;         // k, and k rounded up to kTileK (the LDS row pitch of x)
  uint16_t* y;
  int64_t ldy;
  const uint16_t* res;
  int64_t ldr;
};

// x is staged in two steps. x_issue loads the first kXr 16-byte vectors per thread into registers before the weight
// tiles are issued, so the prologue waits for x alone (loads complete in issue order). stage_x writes them to LDS,
// loads any rest directly, and with NORM rewrites LDS as bf16(w * bf16(x * rsqrt(mean(x^2) + eps))), the mean over
// the k real elements (bb_fused.cu:95-140). One resource covers the x matrix; elements past k in a row (the row
// padding, or past the last row) read as 0, so LDS holds x zero-padded to kp.
constexpr int kXr = 4;

template <int M>
__device__ __forceinline__ uint4 x_vector(const GemvParams& p, const Rsrc& rx, int idx) {
  const int kv = p.kp / 8;
  const int m = idx / kv, j = idx - m * kv;
  const bool in = idx < M * kv && j * 8 < p.k;
  const uint32_t off = in ? (uint32_t)(m * p.ldx + j * 8) * 2 : 0xfffffff0u;  // out of range: reads 0
  return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rx, off, 0, 0));
}

template <int M, int NT>
__device__ __forceinline__ void x_issue(const GemvParams& p, const Rsrc& rx, uint4 (&xr)[kXr]) {
#pragma unroll
  for (int i = 0; i < kXr; ++i) xr[i] = x_vector<M>(p, rx, threadIdx.x + i * NT);
}

template <int M, bool NORM, int NT>
__device__ __forceinline__ void stage_x(const GemvParams& p, const Rsrc& rx, const uint4 (&xr)[kXr], uint16_t* xs) {
  const int tid = threadIdx.x;
  const int kv = p.kp / 8, total = M * kv;
  float ss[M];
#pragma unroll
  for (int m = 0; m < M; ++m) ss[m] = 0.f;
  auto put = [&](int idx, const uint4& v) {
    reinterpret_cast<uint4*>(xs)[idx] = v;  // LDS row pitch kp: vector idx of the [M][kp] array
    if (NORM) {
      float f[8];
      unpack8(v, f);
      float s2 = 0.f;
#pragma unroll
      for (int t = 0; t < 8; ++t) s2 = fmaf(f[t], f[t], s2);
      const int m = idx / kv;
#pragma unroll
      for (int mm = 0; mm < M; ++mm)
        if (mm == m) ss[mm] += s2;
    }
  };
#pragma unroll
  for (int i = 0; i < kXr; ++i) {
    const int idx = tid + i * NT;
    if (idx < total) put(idx, xr[i]);
  }
  for (int idx = tid + kXr * NT; idx < total; idx += NT) put(idx, x_vector<M>(p, rx, idx));
  if (!NORM) return;
  __shared__ float red[NT / kWave][M];
  const int lane = tid % kWave, wave = tid / kWave;
#pragma unroll
  for (int m = 0; m < M; ++m) {
    const float s2 = wave_sum(ss[m]);
    if (lane == 0) red[wave][m] = s2;
  }
  __syncthreads();
  const Rsrc rw = span_rsrc(p.nw, p.k * 2);
#pragma unroll
  for (int m = 0; m < M; ++m) {
    float tot = 0.f;
#pragma unroll
    for (int w = 0; w < NT / kWave; ++w) tot += red[w][m];
    const float r = rsqrtf(tot * (1.f / (float)p.k) + p.eps);
    for (int j = tid; j < kv; j += NT) {
      float f[8], w[8];
      unpack8(reinterpret_cast<const uint4*>(xs + m * p.kp)[j], f);
      unpack8(__builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rw, j * 16, 0, 0)), w);
#pragma unroll
      for (int t = 0; t < 8; ++t) f[t] *= r;
      round8(f);
#pragma unroll
      for (int t = 0; t < 8; ++t) f[t] *= w[t];
      reinterpret_cast<uint4*>(xs + m * p.kp)[j] =
          make_uint4(pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]), pack_bf16x2(f[4], f[5]), pack_bf16x2(f[6], f[7]));
    }
  }
}

// x of one lane in registers: row m, chunk c (k = 512 c + 8 lane), zero past k.
__device__ __forceinline__ uint4 x_chunk(const GemvParams& p, const Rsrc& rx, int m, int c, int lane) {
  const int k0 = c * kChunk + lane * 8;
  const uint32_t off = k0 < p.k ? (uint32_t)(m * p.ldx + k0) * 2 : 0xfffffff0u;
  return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rx, off, 0, 0));
}

// The residual values the writing lanes of a wave need (lane 16 q writes flat value 4 g + q of each group g, i.e.
// output row r = f / M of batch row m = f % M), loaded with the first weight tiles so that the epilogue waits for
// nothing: one 2-byte buffer load per group and lane. Values past the output rows are never used; loads past the
// residual matrix read 0 without a memory access.
template <int M, int R>
__device__ __forceinline__ void load_residual(const GemvParams& p, int row0, int lane, float (&res)[(R * M + 3) / 4]) {
  const Rsrc rr = span_rsrc(p.res, (int)(((int64_t)(M - 1) * p.ldr + p.ntot) * 2));
  const int q = lane / 16;
#pragma unroll
  for (int g = 0; g < (R * M + 3) / 4; ++g) {
    const int f = 4 * g + q, r = f / M, m = f % M;
    const uint32_t off = (uint32_t)(((int64_t)m * p.ldr + row0 + r) * 2);
    res[g] = bf16_to_f32(__builtin_amdgcn_raw_buffer_load_b16(rr, off, 0, 0));
  }
}

// KC > 0: x held in registers, KC chunks per lane (k <= 512 KC <= 2 tiles): no LDS, and the RMSNorm's sum of squares
// is reduced over the wave, so the prologue needs no barrier. KC == 0: x staged in LDS (any k).
// What the first loads need (the weight segments, their row counts, k, x and its stride) comes as leading scalar
// arguments, 56 bytes, which kernel-argument preloading (-mllvm -amdgpu-kernarg-preload-count) puts in SGPRs when the
// wave starts, so the weight and x loads go out at once rather than after a load of the argument buffer; they are
// the block's fields again, which the kernel then reads from these arguments.
template <int M, int R, bool NORM, int EPI, int KC, int GAP>
__global__ void __launch_bounds__(gemv_threads<KC>())
    gemv_kernel(const uint16_t* w0, const uint16_t* w1, const uint16_t* w2, int n0, int n1, int ntot, int k,
                const uint16_t* x, int64_t ldx, const GemvParams args) {
  GemvParams p = args;
  p.w0 = w0;
  p.w1 = w1;
  p.w2 = w2;
  p.n0 = n0;
  p.n1 = n1;
  p.ntot = ntot;
  p.k = k;
  p.x = x;
  p.ldx = ldx;
  static_assert(GAP == 0 || KC > 0, "issue pacing on the x-in-registers path only");
  constexpr int NT = gemv_threads<KC>(), NW = NT / kWave;
  constexpr int NR = EPI == BZ_GEMV_SILU_MUL ? 2 * R : R;  // weight rows per wave
  extern __shared__ __align__(16) uint16_t xs[];            // [M][kp] bf16
  // The paced variant takes the wave index through a scalar register, so the weight resources are scalar and each
  // load is one instruction, spaced by s_sleep. The unpaced variants (x in LDS; small grids) leave it in a VGPR, where
  // the compiler issues every load from a one-iteration loop over the wave's distinct resources. That measured faster
  // than scalar resources without pacing, for reasons not pinned down (down: 6.03 against 6.36 us, paced or not;
  // gate/up on 12 and 32 workgroups: 2.93 and 3.93 against 3.23 and 4.45 us).
  const int tid = threadIdx.x, lane = tid % kWave, wave = GAP > 0 ? wave_uniform(tid / kWave) : tid / kWave;
  const int row0 = (blockIdx.x * NW + wave) * R;

  // this wave's weight rows (a row past the last output: an empty resource, whose loads read 0)
  Rsrc wr[NR];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int n = row0 + r;
    const int bytes = n < p.ntot ? p.k * 2 : 0;
    if (EPI == BZ_GEMV_SILU_MUL) {
      wr[r] = span_rsrc(p.w0 + (int64_t)n * p.k, bytes);
      wr[R + r] = span_rsrc(p.w1 + (int64_t)n * p.k, bytes);
    } else {
      const uint16_t* base = n < p.n0 ? p.w0 + (int64_t)n * p.k
                           : n < p.n0 + p.n1 ? p.w1 + (int64_t)(n - p.n0) * p.k
                                             : p.w2 + (int64_t)(n - p.n0 - p.n1) * p.k;
      wr[r] = span_rsrc(base, bytes);
    }
  }

  uint4 ta[NR][kU], tb[NR][kU];
  const uint32_t lane_off = lane * 16;
  auto load = [&](uint4 (&t)[NR][kU], int it) {
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const uint32_t off = (uint32_t)(it * kTileK + u * kChunk) * 2 + lane_off;
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        t[r][u] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(wr[r], off, 0, kStream));
        if constexpr (GAP > 0) __builtin_amdgcn_s_sleep(GAP);
      }
    }
  };
  const Rsrc rx = span_rsrc(p.x, (int)(((int64_t)(M - 1) * p.ldx + p.k) * 2));
  [[maybe_unused]] float resv[(R * M + 3) / 4];
  float acc[NR][M];
#pragma unroll
  for (int r = 0; r < NR; ++r)
#pragma unroll
    for (int m = 0; m < M; ++m) acc[r][m] = 0.f;
  auto dot16 = [](const uint4& w, const uint4& xv, float a) {
    a = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w.x), __builtin_bit_cast(bf16x2_t, xv.x), a, false);
    a = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w.y), __builtin_bit_cast(bf16x2_t, xv.y), a, false);
    a = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w.z), __builtin_bit_cast(bf16x2_t, xv.z), a, false);
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w.w), __builtin_bit_cast(bf16x2_t, xv.w), a, false);
  };

  if constexpr (KC > 0) {
    static_assert(KC <= 2 * kU, "x in registers: the row fits the first two tiles");
    // x (and the norm weight) first, then both weight tiles; the prologue waits for x alone
    uint4 xv[M][KC], nwv[KC];
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int c = 0; c < KC; ++c) xv[m][c] = x_chunk(p, rx, m, c, lane);
    if (NORM) {
      const Rsrc rw = span_rsrc(p.nw, p.k * 2);
#pragma unroll
      for (int c = 0; c < KC; ++c)
        nwv[c] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rw, (c * kChunk + lane * 8) * 2, 0, 0));
    }
    load(ta, 0);
    load(tb, 1);
    if (EPI == BZ_GEMV_RESIDUAL) load_residual<M, R>(p, row0, lane, resv);
    __builtin_amdgcn_sched_barrier(0);
    if (NORM) {
#pragma unroll
      for (int m = 0; m < M; ++m) {
        float ss = 0.f;
#pragma unroll
        for (int c = 0; c < KC; ++c) {
          float f[8];
          unpack8(xv[m][c], f);
#pragma unroll
          for (int t = 0; t < 8; ++t) ss = fmaf(f[t], f[t], ss);
        }
        const float rs = rsqrtf(wave_sum(ss) * (1.f / (float)p.k) + p.eps);
#pragma unroll
        for (int c = 0; c < KC; ++c) {
          float f[8], w[8];
          unpack8(xv[m][c], f);
          unpack8(nwv[c], w);
#pragma unroll
          for (int t = 0; t < 8; ++t) f[t] *= rs;
          round8(f);
#pragma unroll
          for (int t = 0; t < 8; ++t) f[t] *= w[t];
          xv[m][c] = make_uint4(pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]), pack_bf16x2(f[4], f[5]),
                                pack_bf16x2(f[6], f[7]));
        }
      }
    }
#pragma unroll
    for (int c = 0; c < KC; ++c)
#pragma unroll
      for (int m = 0; m < M; ++m)
#pragma unroll
        for (int r = 0; r < NR; ++r)
          acc[r][m] = dot16(c < kU ? ta[r][c % kU] : tb[r][c % kU], xv[m][c], acc[r][m]);
  } else {
    // x first (the prologue then waits for x alone), then the first two weight tiles, all before the prologue
    uint4 xr[kXr];
    x_issue<M, NT>(p, rx, xr);
    load(ta, 0);
    load(tb, 1);
    if (EPI == BZ_GEMV_RESIDUAL) load_residual<M, R>(p, row0, lane, resv);
    __builtin_amdgcn_sched_barrier(0);

    stage_x<M, NORM, NT>(p, rx, xr, xs);
    __syncthreads();

    auto consume = [&](const uint4 (&t)[NR][kU], int it) {
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int kk = it * kTileK + u * kChunk + lane * 8;
#pragma unroll
        for (int m = 0; m < M; ++m) {
          const uint4 xv = *reinterpret_cast<const uint4*>(xs + m * p.kp + kk);
#pragma unroll
          for (int r = 0; r < NR; ++r) acc[r][m] = dot16(t[r][u], xv, acc[r][m]);
        }
      }
    };
    const int nit = p.kp / kTileK;
    for (int it = 0; it < nit; it += 2) {
      consume(ta, it);
      load(ta, it + 2);  // past k: reads 0 without a memory access
      if (it + 1 < nit) consume(tb, it + 1);
      load(tb, it + 3);
    }
  }

  // sum the accumulators over the wave: DPP inside each 16-lane row, then transposed swaps across the 4 rows, so
  // row q of red[g] holds the total of flat value 4 g + q. Flat order: (r, m) -> r * M + m for the R output rows,
  // padded to a multiple of 4 (NG); the up rows of SILU_MUL follow at NG + r * M + m, in the same row as their gate.
  constexpr int NG = (R * M + 3) / 4 * 4;
  constexpr int NV = EPI == BZ_GEMV_SILU_MUL ? 2 * NG : NG;
  float flat[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) flat[v] = 0.f;
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int m = 0; m < M; ++m) {
      flat[r * M + m] = row_sum<16>(acc[r][m]);
      if (EPI == BZ_GEMV_SILU_MUL) flat[NG + r * M + m] = row_sum<16>(acc[R + r][m]);
    }
  float red[NV / 4];
#pragma unroll
  for (int g = 0; g < NV / 4; ++g) red[g] = rows_sum4(flat[4 * g], flat[4 * g + 1], flat[4 * g + 2], flat[4 * g + 3]);

  if (lane % 16 != 0) return;
  const int q = lane / 16;
#pragma unroll
  for (int g = 0; g < NG / 4; ++g) {
    const int f = 4 * g + q;
    if (f >= R * M) continue;
    const int r = f / M, m = f % M, n = row0 + r;
    if (n >= p.ntot) continue;
    float v;
    if (EPI == BZ_GEMV_PLAIN) {
      v = red[g];
    } else if (EPI == BZ_GEMV_RESIDUAL) {
      v = resv[g] + bf16_to_f32(f32_to_bf16(red[g]));
    } else {
      const float gt = bf16_to_f32(f32_to_bf16(red[g]));
      const float up = bf16_to_f32(f32_to_bf16(red[NG / 4 + g]));
      v = bf16_to_f32(f32_to_bf16(gt / (1.f + expf(-gt)))) * up;
    }
    p.y[(int64_t)m * p.ldy + n] = f32_to_bf16(v);
  }
}

// Block-ordered GEMV: a workgroup of NT threads owns R output rows (2 R weight rows for the SiLU * up epilogue: the gate
// rows, then the up rows) and streams them as one contiguous block. Load i of thread t reads the 16 bytes at k = 8 t of
// row i (k <= 8 NT; past k it reads 0), so every thread needs one x vector per row of x for all of its rows, and all NS
// loads per thread go out at once. Against the wave-per-row kernel above this keeps the workgroup's bytes in flight
// contiguous (the wave-per-row kernel with x in LDS holds a third of each of eight rows 12 KB apart at k = 6144) and
// each workgroup reads x once (with x in registers there every wave reads its own: 32 MB of L2 traffic for q | k | v at
// M = 4). The sums are reduced once, at the end: DPP and transposed swaps inside each wave, then the waves through LDS
// in wave order. Where a row has no more vectors than a workgroup of 256 threads, four waves finish alone: with 512
// threads and two rows per load instruction (the same order of sums) a workgroup held 16 rows, its norm, reductions and
// barriers left eight waves idle together, and two such workgroups fitted on a CU (84 VGPRs) against five of four
// waves: gate / up at k = 2048, 6144 outputs, M = 3 / 4 11.0 / 11.8 -> 10.4 / 10.3 us (4.9 TB/s), q | k | v 5.0 / 5.4 ->
// 4.8 / 5.0, o_proj 3.5 -> 3.4.
template <int M, int NT, int R, bool NORM, int EPI>
__global__ void __launch_bounds__(NT)
    gemv_block_kernel(const uint16_t* w0, const uint16_t* w1, const uint16_t* w2, int n0, int n1, int ntot, int k,
                      const uint16_t* x, int64_t ldx, const GemvParams args) {
  GemvParams p = args;
  p.w0 = w0;
  p.w1 = w1;
  p.w2 = w2;
  p.n0 = n0;
  p.n1 = n1;
  p.ntot = ntot;
  p.k = k;
  p.x = x;
  p.ldx = ldx;
  constexpr int NW = NT / kWave;
  constexpr bool SILU = EPI == BZ_GEMV_SILU_MUL;
  constexpr int NS = SILU ? 2 * R : R;  // weight-row slots per thread (SiLU: the gate slots, then the up slots)
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int row0 = blockIdx.x * R;

  // x (and the norm weight) first, then every weight load; the prologue waits for x alone
  const Rsrc rx = span_rsrc(p.x, (int)(((int64_t)(M - 1) * p.ldx + p.k) * 2));
  uint4 xv[M], nwv = make_uint4(0, 0, 0, 0);
#pragma unroll
  for (int m = 0; m < M; ++m) {
    const uint32_t off = 8 * tid < p.k ? (uint32_t)(m * p.ldx + 8 * tid) * 2 : 0xfffffff0u;  // past k: reads 0
    xv[m] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rx, off, 0, 0));
  }
  if (NORM)
    nwv = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(span_rsrc(p.nw, p.k * 2), 16 * tid, 0, 0));
  uint4 wt[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const bool up = SILU && s >= R;
    const int n = row0 + (up ? s - R : s);
    const int bytes = n < p.ntot ? p.k * 2 : 0;  // a row past the last output: an empty resource, its loads read 0
    const uint16_t* base;
    if (SILU) {
      base = (up ? p.w1 : p.w0) + (int64_t)n * p.k;
    } else {
      base = n < p.n0 ? p.w0 + (int64_t)n * p.k
           : n < p.n0 + p.n1 ? p.w1 + (int64_t)(n - p.n0) * p.k
                             : p.w2 + (int64_t)(n - p.n0 - p.n1) * p.k;
    }
    wt[s] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(span_rsrc(base, bytes), 16 * tid, 0, kStream));
  }
  // the residual value of the output this thread writes (thread f < R * M: row f / M, batch row f % M); loads past
  // the residual matrix read 0 without a memory access, and values past the output rows are never used
  float resv = 0.f;
  if (EPI == BZ_GEMV_RESIDUAL) {
    const Rsrc rr = span_rsrc(p.res, (int)(((int64_t)(M - 1) * p.ldr + p.ntot) * 2));
    const int f = tid % (R * M), n = row0 + f / M, m = f % M;
    resv = bf16_to_f32(__builtin_amdgcn_raw_buffer_load_b16(rr, (uint32_t)(((int64_t)m * p.ldr + n) * 2), 0, 0));
  }
  __builtin_amdgcn_sched_barrier(0);

  if (NORM) {
    __shared__ float s_ss[NW][M];
#pragma unroll
    for (int m = 0; m < M; ++m) {
      float f[8], ss = 0.f;
      unpack8(xv[m], f);
#pragma unroll
      for (int t = 0; t < 8; ++t) ss = fmaf(f[t], f[t], ss);
      ss = wave_sum(ss);
      if (lane == 0) s_ss[wave][m] = ss;
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < M; ++m) {
      float tot = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) tot += s_ss[w][m];
      const float rs = rsqrtf(tot * (1.f / (float)p.k) + p.eps);
      float f[8], w[8];
      unpack8(xv[m], f);
      unpack8(nwv, w);
#pragma unroll
      for (int t = 0; t < 8; ++t) f[t] *= rs;
      round8(f);
#pragma unroll
      for (int t = 0; t < 8; ++t) f[t] *= w[t];
      xv[m] = make_uint4(pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]), pack_bf16x2(f[4], f[5]),
                         pack_bf16x2(f[6], f[7]));
    }
  }

  // flat value s * M + m (zero-padded to a power of two), summed over the wave by the transposed sum: one total per
  // value, written to LDS by the first lane that holds it
  constexpr int NV = NS * M, NP = NV <= 4 ? 4 : NV <= 8 ? 8 : NV <= 16 ? 16 : NV <= 32 ? 32 : 64;
  float flat[NP];
#pragma unroll
  for (int v = 0; v < NP; ++v) flat[v] = 0.f;
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const uint4& w = wt[s];
      float a = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w.x), __builtin_bit_cast(bf16x2_t, xv[m].x),
                                                0.f, false);
      a = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w.y), __builtin_bit_cast(bf16x2_t, xv[m].y), a,
                                          false);
      a = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w.z), __builtin_bit_cast(bf16x2_t, xv[m].z), a,
                                          false);
      a = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w.w), __builtin_bit_cast(bf16x2_t, xv[m].w), a,
                                          false);
      flat[s * M + m] = a;
    }
  const float tot = transposed_sum<NP>(flat, lane);
  __shared__ float s_red[NW][NP];
  if (transposed_writer<NP>(lane)) s_red[wave][transposed_index<NP>(lane)] = tot;
  __syncthreads();
  // thread f < R * M writes row row0 + f / M of batch row f % M
  if (tid >= R * M) return;
  const int r = tid / M, m = tid % M, n = row0 + r;
  if (n >= p.ntot) return;
  float red = 0.f, upv = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    red += s_red[w][r * M + m];
    if (SILU) upv += s_red[w][(R + r) * M + m];
  }
  float v;
  if (EPI == BZ_GEMV_PLAIN) {
    v = red;
  } else if (EPI == BZ_GEMV_RESIDUAL) {
    v = resv + bf16_to_f32(f32_to_bf16(red));
  } else {
    const float gt = bf16_to_f32(f32_to_bf16(red));
    const float u = bf16_to_f32(f32_to_bf16(upv));
    v = bf16_to_f32(f32_to_bf16(gt / (1.f + expf(-gt)))) * u;
  }
  p.y[(int64_t)m * p.ldy + n] = f32_to_bf16(v);
}

// GEMV on the 4x4x4 MFMA (16 blocks). A wave load covers four rows of weights, 256 bytes each: lane 4 b + i holds row i,
// the 8 k-values 128 c + 8 b .. of chunk c, which are the A operands of two MFMAs (block b: 4 rows x 4 k); lane 4 b + j
// holds the same 8 k-values of x's row j, their B operands (4 k x up to 4 rows of x). So a block sums its own k-values of
// all 4 x 4 products into four registers, x costs one 16-byte vector per chunk and lane whatever the number of its rows,
// its RMSNorm is worked out once per element, and a wave ends with 4 sums per four rows to add over its 16 blocks.
// Against four dot2 per vector and row of x on the vector unit (the kernels above) that is an eighth of the instructions
// at four rows of x, where they bound the tail of every workgroup.
//
// A workgroup of eight waves owns Q such groups of four rows ("quads"; with the SiLU * up epilogue the first half are gate
// quads, the second the up quads of the same outputs) and splits k over its waves: wave w takes the TR chunks w, w + 8,
// ..., so that the workgroup reads 2048 consecutive bytes of every row at a time, x once, and every load goes out at
// once. Each weight segment starts a quad of its own, so a quad has one resource, cut at its last row; lanes past k take
// an offset outside of it (their loads read 0: a neighbouring row's Inf or NaN must not meet x's padding). The sums meet
// in LDS.
constexpr int kMfmaWaves = 8;

template <int Q, int TR, bool NORM, int EPI>
__global__ void __launch_bounds__(kMfmaWaves* kWave)
    gemv_mfma_kernel(const uint16_t* w0, const uint16_t* w1, const uint16_t* w2, int n0, int n1, int ntot, int km,
                     const uint16_t* x, int64_t ldx, const GemvParams p) {
  constexpr bool SILU = EPI == BZ_GEMV_SILU_MUL;
  constexpr int QO = SILU ? Q / 2 : Q;  // quads of outputs
  constexpr int NW = kMfmaWaves;
  static_assert(EPI != BZ_GEMV_RESIDUAL, "the residual epilogue stays on the other kernels");
  constexpr uint32_t kOut = 0x40000000u;  // past every quad (4 k * 2 bytes)
  const int k = km & 0xffffff, M = km >> 24;  // one preloaded argument
  const int tid = threadIdx.x, lane = tid % kWave, wave = wave_uniform(tid / kWave);
  const int j = lane % 4, b = lane / 4;

  // the quads: resource and first output row; segment s has ceil(n_s / 4) of them
  const int c0 = (n0 + 3) / 4, c1 = (n1 + 3) / 4;
  auto quad = [&](int qo, bool up, int& row, int& rows) {
    const int q = blockIdx.x * QO + qo;
    const uint16_t* base = SILU && up ? w1 : w0;
    int first = 4 * q, n = n0;
    row = first;
    if (!SILU && q >= c0) {
      const bool third = q >= c0 + c1;
      base = third ? w2 : w1;
      first = 4 * (q - c0 - (third ? c1 : 0));
      n = third ? ntot - n0 - n1 : n1;
      row = first + n0 + (third ? n1 : 0);
    }
    rows = min(4, n - first);  // <= 0 past the last quad: an empty resource
    return span_rsrc(base + (int64_t)first * k, rows > 0 ? rows * k * 2 : 0);
  };
  Rsrc wr[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    int row, rows;
    wr[q] = quad(SILU ? q % QO : q, SILU && q >= QO, row, rows);
  }
  const Rsrc rx = span_rsrc(x, (int)(((int64_t)(M - 1) * ldx + k) * 2));
  const uint32_t xrow = (uint32_t)(j * ldx) * 2;

  // x first, then every weight load; the prologue waits for x alone
  uint4 xv[TR], nwv[TR], wt[TR][Q];
#pragma unroll
  for (int r = 0; r < TR; ++r) {
    const int k0 = 128 * (r * NW + wave) + 8 * b;
    const uint32_t off = k0 < k && j < M ? xrow + 2 * k0 : 0xfffffff0u;
    xv[r] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rx, off, 0, 0));
    if (NORM)
      nwv[r] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(span_rsrc(p.nw, k * 2), 2 * k0, 0, 0));
  }
#pragma unroll
  for (int r = 0; r < TR; ++r) {
    const int k0 = 128 * (r * NW + wave) + 8 * b;
    const uint32_t off = k0 < k ? 2 * (j * k + k0) : kOut;
#pragma unroll
    for (int q = 0; q < Q; ++q)
      wt[r][q] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(wr[q], off, 0, kStream));
  }
  // thread t < 16 Q (the lanes of wave 0 after the sums) writes value v = 4 q + row of row j of x
  constexpr int NV = 4 * Q;
  const int v = transposed_index<NV>(tid), vq = v / 4, vr = v % 4;
  const bool writes = tid < kWave && (Q == 4 || (tid & (Q == 2 ? 4 : 12)) == 0) && vq < QO && j < M;
  int row = 0, rows = 0;
  if (tid < kWave) (void)quad(vq, false, row, rows);
  __builtin_amdgcn_sched_barrier(0);

  if (NORM) {
    __shared__ float s_ss[NW][4];
    float ss = 0.f;
#pragma unroll
    for (int r = 0; r < TR; ++r) {
      float f[8];
      unpack8(xv[r], f);
#pragma unroll
      for (int i = 0; i < 8; ++i) ss = fmaf(f[i], f[i], ss);
    }
    ss += dpp<0x124>(ss);  // row_ror:4 and :8: over the 4 blocks of a 16-lane row (same j)
    ss += dpp<0x128>(ss);
    float y = ss;
    swap16(ss, y);
    ss += y;
    y = ss;
    swap32(ss, y);
    ss += y;
    if (lane < 4) s_ss[wave][lane] = ss;
    __syncthreads();
    float tot = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) tot += s_ss[w][j];
    const float rs = rsqrtf(tot * (1.f / (float)k) + p.eps);
#pragma unroll
    for (int r = 0; r < TR; ++r) {
      float f[8], w[8];
      unpack8(xv[r], f);
      unpack8(nwv[r], w);
#pragma unroll
      for (int i = 0; i < 8; ++i) f[i] *= rs;
      round8(f);
#pragma unroll
      for (int i = 0; i < 8; ++i) f[i] *= w[i];
      xv[r] = make_uint4(pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]), pack_bf16x2(f[4], f[5]),
                         pack_bf16x2(f[6], f[7]));
    }
  }

  f32x4_t acc[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) acc[q] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto half = [](uint32_t lo, uint32_t hi) { return __builtin_bit_cast(s16x4_t, make_uint2(lo, hi)); };
#pragma unroll
  for (int r = 0; r < TR; ++r)
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const uint4 &w = wt[r][q], &u = xv[r];
      acc[q] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(half(w.x, w.y), half(u.x, u.y), acc[q], 0, 0, 0);
      acc[q] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(half(w.z, w.w), half(u.z, u.w), acc[q], 0, 0, 0);
    }

  // the 4 Q sums of a lane over the 16 blocks, transposed over lane bits 5, 4, 3, 2 (transposed_sum's levels; the lanes
  // of one j stay apart), then over the waves
  float flat[NV];
#pragma unroll
  for (int q = 0; q < Q; ++q)
#pragma unroll
    for (int r = 0; r < 4; ++r) flat[4 * q + r] = acc[q][r];
  swap_level<NV / 2>(flat, true);
  swap_level<NV / 4>(flat, false);
  if constexpr (NV >= 8) dpp_level<NV / 8, 0x128>(flat, lane & 8);
  else flat[0] += dpp<0x128>(flat[0]);
  auto xor4 = [](float f) {  // lane ^ 4: row_ror:12 for the lanes with bit 2 clear, row_ror:4 for the others
    const int up = __builtin_amdgcn_update_dpp(0, __float_as_int(f), 0x12c, 0xf, 0xf, true);
    return __int_as_float(__builtin_amdgcn_update_dpp(up, __float_as_int(f), 0x124, 0xf, 0xa, false));
  };
  if constexpr (NV >= 16) {
    const bool hi = lane & 4;
    flat[0] = (hi ? flat[1] : flat[0]) + xor4(hi ? flat[0] : flat[1]);
  } else {
    flat[0] += xor4(flat[0]);
  }
  __shared__ float s_red[NW][kWave];
  s_red[wave][lane] = flat[0];
  __syncthreads();
  if (!writes || vr >= rows) return;
  float red = 0.f, upv = 0.f;
  // the lane of the up value: its quad's bit of the value index is lane bit 5
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    red += s_red[w][tid];
    if (SILU) upv += s_red[w][tid + 32];
  }
  float out;
  if (EPI == BZ_GEMV_PLAIN) {
    out = red;
  } else {
    const float gt = bf16_to_f32(f32_to_bf16(red));
    const float u = bf16_to_f32(f32_to_bf16(upv));
    out = bf16_to_f32(f32_to_bf16(gt / (1.f + expf(-gt)))) * u;
  }
  p.y[(int64_t)j * p.ldy + row + vr] = f32_to_bf16(out);
}

// Standalone row RMSNorm, one workgroup per row (bb_fused.cu:219-248).
__global__ void __launch_bounds__(kGemvThreads) rmsnorm_kernel(const uint16_t* x, int64_t ldx, const uint16_t* w,
                                                               float eps, uint16_t* y, int64_t ldy, int k) {
  const int m = blockIdx.x, tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const uint16_t* xr = x + (int64_t)m * ldx;
  float ss = 0.f;
  for (int j = tid * 8; j < k; j += kGemvThreads * 8) {
    float f[8];
    unpack8(*reinterpret_cast<const uint4*>(xr + j), f);
#pragma unroll
    for (int t = 0; t < 8; ++t) ss = fmaf(f[t], f[t], ss);
  }
  __shared__ float red[kGemvWaves];
  ss = wave_sum(ss);
  if (lane == 0) red[wave] = ss;
  __syncthreads();
  float tot = 0.f;
#pragma unroll
  for (int i = 0; i < kGemvWaves; ++i) tot += red[i];
  const float r = rsqrtf(tot * (1.f / (float)k) + eps);
  for (int j = tid * 8; j < k; j += kGemvThreads * 8) {
    float f[8], ww[8];
    unpack8(*reinterpret_cast<const uint4*>(xr + j), f);
    unpack8(*reinterpret_cast<const uint4*>(w + j), ww);
#pragma unroll
    for (int t = 0; t < 8; ++t) f[t] *= r;
    round8(f);
#pragma unroll
    for (int t = 0; t < 8; ++t) f[t] *= ww[t];
    *reinterpret_cast<uint4*>(y + (int64_t)m * ldy + j) =
        make_uint4(pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]), pack_bf16x2(f[4], f[5]), pack_bf16x2(f[6], f[7]));
  }
}

// ---------------------------------------------------------------------------------------------- host side

using GemvFn = void (*)(const uint16_t*, const uint16_t*, const uint16_t*, int, int, int, int, const uint16_t*,
                        int64_t, const GemvParams);

template <int M, int R, int KC, int GAP>
GemvFn pick_epi(int epi, bool norm) {
  if (epi == BZ_GEMV_PLAIN)
    return norm ? gemv_kernel<M, R, true, BZ_GEMV_PLAIN, KC, GAP> : gemv_kernel<M, R, false, BZ_GEMV_PLAIN, KC, GAP>;
  if (epi == BZ_GEMV_RESIDUAL) return norm ? nullptr : gemv_kernel<M, R, false, BZ_GEMV_RESIDUAL, KC, GAP>;
  if (epi == BZ_GEMV_SILU_MUL)
    return norm ? gemv_kernel<M, R, true, BZ_GEMV_SILU_MUL, KC, GAP>
                : gemv_kernel<M, R, false, BZ_GEMV_SILU_MUL, KC, GAP>;
  return nullptr;
}

// With x in LDS: R = 1, 2 or 4 rows per wave, no pacing. With x in registers: R = 2, paced or not.
template <int M, int KC>
GemvFn pick_r(int r, int epi, bool norm, bool pace) {
  if constexpr (KC > 0) {
    if (r != 2) return nullptr;
    return pace ? pick_epi<M, 2, KC, kIssueGap>(epi, norm) : pick_epi<M, 2, KC, 0>(epi, norm);
  } else {
    switch (r) {
      case 1: return pick_epi<M, 1, KC, 0>(epi, norm);
      case 2: return pick_epi<M, 2, KC, 0>(epi, norm);
      default: return pick_epi<M, 4, KC, 0>(epi, norm);
    }
  }
}

// x in registers for k <= 2048 (KC = 2: k <= 1024, KC = 4: k <= 2048); LDS otherwise.
template <int M>
GemvFn pick_kc(int kc, int r, int epi, bool norm, bool pace) {
  if (kc == 4) return pick_r<M, 4>(r, epi, norm, pace);
  if (kc == 2) return pick_r<M, 2>(r, epi, norm, pace);
  return pick_r<M, 0>(r, epi, norm, pace);
}

// Chunks of x per lane held in registers (0: x in LDS).
int kc_for(int m, int k) {
  (void)m;
  const int chunks = (k + kChunk - 1) / kChunk;
  return chunks <= 2 ? 2 : (chunks <= 4 ? 4 : 0);
}

GemvFn pick_gemv(int m, int kc, int r, int epi, bool norm, bool pace) {
  switch (m) {
    case 1: return pick_kc<1>(kc, r, epi, norm, pace);
    case 2: return pick_kc<2>(kc, r, epi, norm, pace);
    case 3: return pick_kc<3>(kc, r, epi, norm, pace);
    case 4: return pick_kc<4>(kc, r, epi, norm, pace);
    default: return nullptr;
  }
}

// The block-ordered kernel where it measured faster than the wave-per-row kernel (us per call, wave-per-row -> block):
//   4096 < k <= 6144, any M: 768 threads (down at k = 6144, M = 1 / 2 / 4: 6.71 / 6.77 / 7.50 -> 5.93 / 6.01 / 6.30);
//   1024 < k <= 2048 and M >= 3: 256 threads (M = 4: q | k | v 7.04 -> 5.0, gate / up 12.75 -> 10.3, o_proj 3.85 -> 3.4).
//     At M <= 2 the wave-per-row kernel with x in registers stays faster there (the backbone step at M = 2 on one box:
//     gate / up 9.70 against 9.92 us, the step 852 against 861 us).
// Eight rows per workgroup: with four, x is read twice as often (256 threads: q | k | v 5.6 against 5.0, 8000 rows of
// k = 1056 8.0 against 6.5, o_proj 3.6 against 3.4; 768 threads, k 6144, M = 4: 2048 rows 6.3 against 6.15, 4096 rows 10.3
// against 9.7). Four of them with 768 threads where eight leave half of the CUs without a workgroup, or a second round
// at most half full (M = 1 / 2 / 4, eight -> four: k 6144, 1024 rows 4.50 / 4.43 / 4.88 -> 3.96 / 4.06 / 4.25; 2560 rows
// 7.71 / 7.84 / 8.45 -> 7.03 / 7.08 / 7.90; k 4960, 2976 rows 7.30 / 7.20 / 7.85 -> 6.65 / 6.71 / 7.49; k 5120, 1536 rows,
// 192 workgroups of eight: 4.67 / 4.56 / 4.95 against 4.71 / 4.87 / 5.37; two rows: 8.9 at k 6144, 2560 rows, M = 4).
// Four of each kind for the SiLU * up epilogue. There 256 threads take eight gate and eight up rows where that gives
// every CU two or three workgroups, all that fit at once (133 VGPRs): k 2048, M = 4, four / eight rows: 6144 outputs (768
// workgroups of eight) 10.6 / 10.3, k 1536, 4096 (512) 7.0 / 6.6, but k 1280, 2560 (320) 5.6 / 5.9, 1024 (128) 3.7 / 4.2 and
// k 1888, 7112 (889) 11.3 / 11.4.
template <int M, int NT, int R>
GemvFn pick_block_rows(int epi, bool norm) {
  if (epi == BZ_GEMV_SILU_MUL) {
    if constexpr (R == 4 || NT == 256)
      return norm ? gemv_block_kernel<M, NT, R, true, BZ_GEMV_SILU_MUL>
                  : gemv_block_kernel<M, NT, R, false, BZ_GEMV_SILU_MUL>;
    return nullptr;
  }
  if constexpr (R == 8 || NT == 768) {
    if (epi == BZ_GEMV_PLAIN)
      return norm ? gemv_block_kernel<M, NT, R, true, BZ_GEMV_PLAIN> : gemv_block_kernel<M, NT, R, false, BZ_GEMV_PLAIN>;
    return norm ? nullptr : gemv_block_kernel<M, NT, R, false, BZ_GEMV_RESIDUAL>;
  }
  return nullptr;
}
template <int M, int NT>
GemvFn pick_block_m(bool eight, int epi, bool norm) {
  return eight ? pick_block_rows<M, NT, 8>(epi, norm) : pick_block_rows<M, NT, 4>(epi, norm);
}
// The block kernel for this call, its workgroup size and grid; nullptr where the wave-per-row kernel is taken.
GemvFn pick_block(int m, int k, int ntot, int epi, bool norm, int cus, int* threads, int* grid) {
  const bool silu = epi == BZ_GEMV_SILU_MUL;
  auto groups = [&](int rows) { return ntot / rows + (ntot % rows != 0); };
  const int g8 = groups(8);
  if (k > 4096 && k <= 6144) {
    const bool eight = !silu && (g8 > cus / 2 && (g8 <= cus || g8 > cus + cus / 2));
    *threads = 768;
    *grid = eight ? g8 : groups(4);
    switch (m) {
      case 1: return pick_block_m<1, 768>(eight, epi, norm);
      case 2: return pick_block_m<2, 768>(eight, epi, norm);
      case 3: return pick_block_m<3, 768>(eight, epi, norm);
      default: return pick_block_m<4, 768>(eight, epi, norm);
    }
  }
  if (k <= 1024 || k > 2048 || m < 3) return nullptr;
  const bool eight = !silu || (g8 >= 2 * cus && g8 <= 3 * cus);
  *threads = 256;
  *grid = eight ? g8 : groups(4);
  return m == 3 ? pick_block_m<3, 256>(eight, epi, norm) : pick_block_m<4, 256>(eight, epi, norm);
}

// Workgroups of q quads (outputs of SiLU * up: q / 2) over the CUs. g is even where its last round is 90% full; where it is
// one round that twice as many, smaller workgroups would exceed; or from four rounds on, past k = 3072 (four chunks a wave,
// where two quads cost more) one and a half with the last 75% full.
struct Quads {
  int quads, cus, k;
  bool silu;
  int groups(int q) const { return (quads + (silu ? q / 2 : q) - 1) / (silu ? q / 2 : q); }
  int rounds(int g) const { return (g + cus - 1) / cus; }
  bool full(int g, int tenths) const { return 10 * (int64_t)g >= (int64_t)tenths * cus * rounds(g); }
  bool even(int g) const {
    if (full(g, 9) || (g <= cus && 2 * g > cus)) return true;
    return k > 3072 ? 2 * (int64_t)g > 3 * (int64_t)cus && 4 * (int64_t)g >= 3 * (int64_t)cus * rounds(g) : g >= 4 * cus;
  }
};
Quads quads_of(int k, int n0, int n1, int n2, bool silu, int cus) {
  return {(n0 + 3) / 4 + (silu ? 0 : (n1 + 3) / 4 + (n2 + 3) / 4), cus, k, silu};
}

// Where the 4x4x4 MFMA kernel is taken (graph of calls on their own weights, us per call, the other kernels -> this one):
//   SiLU * up for 2048 < k <= 4096 (x in LDS before), M = 1 / 2 / 4: k 4096, 12288 outputs 41.1 / 42.2 / 47.1 -> 31.8 / 30.8 /
//     32.9 (6.5 TB/s); 3072, 8192: 19.6 / 20.6 / 23.1 -> 17.8 / 17.7 / 18.2; 2976, 4960: 16.8 / 16.8 / 19.2 -> 12.7 / 12.5 /
//     13.7; 2560, 6912: 16.1 / 16.2 / 19.0 -> 14.6 / 15.1 / 16.8. Past k = 3072 not at M <= 2 where this kernel's second or
//     fourth round is 75 to 90% full, as the LDS kernel's last round is too (its workgroup has as many outputs or twice as
//     many): k 3840, 6912 outputs, M = 1 / 2: 19.6 / 20.1, here 20.9 / 21.5; and at M = 1 not where a single round is between
//     half and three quarters full: k 3840, 1152 outputs 6.1, here 6.8;
//   plain there at M >= 3: k 4096, 6144 rows 11.8 / 13.0 -> 11.5 / 12.0 at M = 3 / 4 (M = 1 / 2: 10.7 / 11.1 against 12.4 /
//     12.6);
// Up to k = 2048 it measured faster at four rows too (SiLU * up at k 1024, 3072 outputs 6.0 -> 4.6; 568, 2272 5.9 -> 3.8; level
// with the block kernel at 2048, 6144). Every M keeps the other kernels there: a backbone step of such a hidden size is held
// to 1% of its earlier outputs, and another order of the sums in one layer, no less exact, moves them by up to 1.5% after 12
// layers (use_mfma in gqa_kernels.cuh has the figures). A step of a hidden size above 2048 does change: its MLP gains a
// quarter. The residual epilogue gains 12% at k 4096, 1024 rows and loses 7% at k 3072, 1536: it stays on the other kernels.
bool mfma_route(int m, int k, int epi, const Quads& t) {
  if (k <= 2048 || k > 4096) return false;
  if (epi == BZ_GEMV_PLAIN) return m >= 3;
  if (epi != BZ_GEMV_SILU_MUL) return false;
  const int g = t.groups(4), rounds = t.rounds(g);
  if (m <= 2 && k > 3072 && (rounds == 2 || rounds == 4) && !t.full(g, 9) && 4 * g >= 3 * t.cus * rounds) return false;
  return !(m == 1 && k > 3072 && 2 * g > t.cus && 4 * g < 3 * t.cus);
}

template <int TR, int Q>
GemvFn pick_mfma_epi(bool silu, bool norm) {
  if (!silu) return norm ? gemv_mfma_kernel<Q, TR, true, BZ_GEMV_PLAIN> : gemv_mfma_kernel<Q, TR, false, BZ_GEMV_PLAIN>;
  if constexpr (Q > 1)
    return norm ? gemv_mfma_kernel<Q, TR, true, BZ_GEMV_SILU_MUL> : gemv_mfma_kernel<Q, TR, false, BZ_GEMV_SILU_MUL>;
  return nullptr;
}
template <int TR>
GemvFn pick_mfma_q(int q, bool silu, bool norm) {
  if (q == 4) return pick_mfma_epi<TR, 4>(silu, norm);
  if (q == 2) return pick_mfma_epi<TR, 2>(silu, norm);
  return pick_mfma_epi<TR, 1>(silu, norm);
}

// Quads per workgroup: four where their grid is even, else two, or one where all of those fit one round (us per call, 4 / 2
// quads: plain at k 4096, 384 / 768 workgroups 12.9 / 12.0, k 3584, 640 / 1280 16.0 / 17.6; gate / up at k 2976, 620 / 1240
// 13.5 / 12.6, k 3328, 864 / 1728 19.7 / 22.8, 608 / 1216 14.7 / 16.6, k 2560, 144 / 288 5.8 / 6.3; 2 / 1 quads, plain at k
// 3072, M = 3: 128 / 256 workgroups 4.7 / 4.2, 144 / 288 4.7 / 5.3).
GemvFn pick_mfma(const Quads& t, bool norm, int* grid) {
  int q = 4;
  if (!t.even(t.groups(4))) q = t.silu || t.groups(1) > t.cus ? 2 : 1;
  *grid = t.groups(q);
  return t.k <= 3072 ? pick_mfma_q<3>(q, t.silu, norm) : pick_mfma_q<4>(q, t.silu, norm);  // chunks per wave
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// Output rows per wave. With x in registers every wave loads its own x, so two rows per wave halve that L2 traffic
// (measured at the backbone shapes: q|k|v 6.6 -> 5.3 us, o_proj 3.7 -> 3.55 us); with x in LDS, one row per wave
// keeps more waves streaming until the rows are many (down: 7.2 us with two rows, 6.9 with one).
int rows_per_wave(int ntot, int epi, int kc) {
  const int rows = epi == BZ_GEMV_SILU_MUL ? 2 * ntot : ntot;
  if (kc > 0) return 2;
  if (rows >= 16384) return 4;
  if (rows >= 8192) return 2;
  return 1;
}

}  // namespace

extern "C" {

__attribute__((visibility("default"))) int bz_gemv(const bz_gemv_args* a, hipStream_t stream) {
  if (a == nullptr || a->x == nullptr || a->y == nullptr || a->w[0] == nullptr) return BZ_ERR_NULL;
  if (a->m < 1 || a->m > 4 || a->k <= 0 || (a->k & 7)) return BZ_ERR_SHAPE;
  if (a->epilogue < BZ_GEMV_PLAIN || a->epilogue > BZ_GEMV_SILU_MUL) return BZ_ERR_UNSUPPORTED;
  for (int i = 0; i < 3; ++i)
    if (a->n[i] < 0) return BZ_ERR_SHAPE;
  int ntot;
  if (a->epilogue == BZ_GEMV_SILU_MUL) {
    if (a->w[1] == nullptr) return BZ_ERR_NULL;
    if (a->n[0] != a->n[1] || a->n[2] != 0) return BZ_ERR_SHAPE;
    ntot = a->n[0];
  } else {
    if ((a->n[1] > 0 && a->w[1] == nullptr) || (a->n[2] > 0 && a->w[2] == nullptr)) return BZ_ERR_NULL;
    if ((int64_t)a->n[0] + a->n[1] + a->n[2] > INT32_MAX) return BZ_ERR_SHAPE;
    ntot = a->n[0] + a->n[1] + a->n[2];
  }
  if (ntot <= 0) return BZ_ERR_SHAPE;
  if (a->epilogue == BZ_GEMV_RESIDUAL) {
    if (a->res == nullptr) return BZ_ERR_NULL;
    if (a->norm_weight != nullptr) return BZ_ERR_UNSUPPORTED;  // the reference's gemv_resid takes no norm
  }
  if (a->x_stride < a->k || a->y_stride < ntot || (a->epilogue == BZ_GEMV_RESIDUAL && a->res_stride < ntot))
    return BZ_ERR_SHAPE;
  if (!aligned16(a->x) || (a->x_stride & 7) || (a->norm_weight && !aligned16(a->norm_weight))) return BZ_ERR_ALIGNMENT;
  for (int i = 0; i < 3; ++i)
    if (a->w[i] && !aligned16(a->w[i])) return BZ_ERR_ALIGNMENT;
  const int kp = (a->k + kTileK - 1) / kTileK * kTileK;
  const size_t lds = (size_t)a->m * kp * 2;
  if (lds > (size_t)kMaxLds || (int64_t)a->k * 2 > INT32_MAX) return BZ_ERR_UNSUPPORTED;
  if (((int64_t)(a->m - 1) * a->x_stride + a->k) * 2 > INT32_MAX) return BZ_ERR_SHAPE;  // x: 32-bit byte offsets
  if (a->epilogue == BZ_GEMV_RESIDUAL && ((int64_t)(a->m - 1) * a->res_stride + ntot) * 2 > INT32_MAX)
    return BZ_ERR_SHAPE;  // the residual: 32-bit byte offsets

  GemvParams p;
  p.x = static_cast<const uint16_t*>(a->x);
  p.ldx = a->x_stride;
  p.nw = static_cast<const uint16_t*>(a->norm_weight);
  p.eps = a->eps;
  p.w0 = static_cast<const uint16_t*>(a->w[0]);
  p.w1 = static_cast<const uint16_t*>(a->w[1] ? a->w[1] : a->w[0]);
  p.w2 = static_cast<const uint16_t*>(a->w[2] ? a->w[2] : a->w[0]);
  p.n0 = a->n[0];
  p.n1 = a->epilogue == BZ_GEMV_SILU_MUL ? 0 : a->n[1];
  p.ntot = ntot;
  p.k = a->k;
  p.kp = kp;
  p.y = static_cast<uint16_t*>(a->y);
  p.ldy = a->y_stride;
  p.res = static_cast<const uint16_t*>(a->res);
  p.ldr = a->res_stride;
  int bthreads = 0, bgrid = 0;
  int cus = 0;
  const int rc = bz::device_cu_count(&cus);
  if (rc != BZ_OK) return rc;
  const Quads quads = quads_of(a->k, p.n0, p.n1, ntot - p.n0 - p.n1, a->epilogue == BZ_GEMV_SILU_MUL, cus);
  if (mfma_route(a->m, a->k, a->epilogue, quads)) {
    GemvFn mf = pick_mfma(quads, a->norm_weight != nullptr, &bgrid);
    if (mf == nullptr) return BZ_ERR_UNSUPPORTED;
    hipLaunchKernelGGL(mf, dim3(bgrid), dim3(kMfmaWaves * kWave), 0, stream, p.w0, p.w1, p.w2, p.n0, p.n1, p.ntot,
                       p.k | a->m << 24, p.x, p.ldx, p);
    return hipGetLastError() == hipSuccess ? BZ_OK : BZ_ERR_LAUNCH;
  }
  if (GemvFn bf = pick_block(a->m, a->k, ntot, a->epilogue, a->norm_weight != nullptr, cus, &bthreads, &bgrid)) {
    hipLaunchKernelGGL(bf, dim3(bgrid), dim3(bthreads), 0, stream, p.w0, p.w1, p.w2, p.n0, p.n1, p.ntot, p.k, p.x,
                       p.ldx, p);
    return hipGetLastError() == hipSuccess ? BZ_OK : BZ_ERR_LAUNCH;
  }
  const int kc = kc_for(a->m, a->k);
  const int r = rows_per_wave(ntot, a->epilogue, kc);
  const int threads = kc > 0 ? kGemvThreads : kGemvLdsThreads;
  const int rows_per_block = threads / kWave * r;
  const int grid = (ntot + rows_per_block - 1) / rows_per_block;
  bool pace = kc > 0 && grid >= kPaceMinGrid;
  if (pace && (a->epilogue == BZ_GEMV_SILU_MUL ? 2 * r : r) * kc < kPaceMinLoads) pace = grid > cus;
  GemvFn fn = pick_gemv(a->m, kc, r, a->epilogue, a->norm_weight != nullptr, pace);
  if (fn == nullptr) return BZ_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(fn, dim3(grid), dim3(threads), kc > 0 ? 0 : lds, stream, p.w0, p.w1, p.w2, p.n0, p.n1, p.ntot,
                     p.k, p.x, p.ldx, p);
  return hipGetLastError() == hipSuccess ? BZ_OK : BZ_ERR_LAUNCH;
}

__attribute__((visibility("default"))) int bz_rmsnorm(const void* x, int64_t x_stride, const void* w, float eps,
                                                       void* y, int64_t y_stride, int32_t m, int32_t k,
                                                       hipStream_t stream) {
  if (x == nullptr || w == nullptr || y == nullptr) return BZ_ERR_NULL;
  if (m <= 0 || m > 65535 || k <= 0 || (k & 7) || x_stride < k || y_stride < k) return BZ_ERR_SHAPE;
  if (!aligned16(x) || !aligned16(w) || !aligned16(y) || (x_stride & 7) || (y_stride & 7)) return BZ_ERR_ALIGNMENT;
  hipLaunchKernelGGL(rmsnorm_kernel, dim3(m), dim3(kGemvThreads), 0, stream, static_cast<const uint16_t*>(x), x_stride,
                     static_cast<const uint16_t*>(w), eps, static_cast<uint16_t*>(y), y_stride, k);
  return hipGetLastError() == hipSuccess ? BZ_OK : BZ_ERR_LAUNCH;
}

}  // extern "C"
