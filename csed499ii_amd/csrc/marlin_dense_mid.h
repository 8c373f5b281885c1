// Decode- and mid-sized batches (1 to 2048 rows) of the dense INT4 x FP16 GEMM for gfx950
// (the dense Marlin layout: see marlin_dense.hip).
//
// Work decomposition as the 2:4 mid-batch kernel (sm24_mid.h): a workgroup of 8 waves
// owns a tile of 64 NCH output columns x 16 RB batch rows over the whole K or one K
// split; wave w computes every 8th 64-deep k-step from the w-th on, for the whole tile,
// as v_mfma_f32_16x16x32_f16 accumulators, and the 8 sums are added in LDS at the end, in
// wave order.  No barrier runs in the main loop.
//
// What bounds it: the latency of the one stage that a wave has in flight.  At 4 rows of the
// 7B shapes (the codes, K N / 2 bytes from HBM) the waves wait half of their life, over 700
// clocks a read; at 200 rows (the activation rows, 128 bytes per row and k-step against 34
// per column) 28-30 %, with the matrix cores busy 34-43 % and the path from L2 into a compute
// unit at 17-29 of its 64 bytes per clock (counters over the life of a wave).  All operands
// come by LDS-DMA (codes 1 KiB to an instruction, activation rows in whole 128-byte
// lines) into one stage buffer per wave, refilled as soon as the stage is in registers
// (buffers for more stages were no faster: see sm24_mid.h).  The kernel this replaces
// loaded 8 bytes per lane straight into operand order, through the same path 64 lanes at
// a time, and re-read the codes for every 64 rows.
//
// us per call, the kernels before -> this one (one box): 7B at M = 4 qkv 12.4 -> 9.0, o
// 8.6 -> 6.8, gate_up 22.4 -> 13.3, down 11.8 -> 9.6; M = 64 38.3 -> 15.6, 22.1 -> 8.3,
// 69.3 -> 23.1, 36.7 -> 15.0; against the large-M kernel at M = 131 48.6 -> 29.3, 42.5 ->
// 10.4, 65.6 -> 46.5, 61.5 -> 24.0, at M = 512 4096x4096 45.9 -> 22.0, 2048x2048 35.1 ->
// 8.7; 70B down 28672x8192 at M = 1 37.2 -> 25.9.
#pragma once
#include "marlin_dense_prefill.h"
#include "sm24_decode_dma.h"

namespace sm24 {

constexpr int kDmWaves = 8;

// One wave's stage buffer (its activation rows, codes and scales of one k-step); the
// workgroup's reduction buffer lies in the same space.
template <int NCH, int RB, bool GROUPED>
struct DmLds {
  static constexpr int TC = 64 * NCH;
  static constexpr int act_b = 16 * RB * 128;       // activation rows of one 64-deep k-step
  static constexpr int stage_b = act_b + NCH * (2048 + (GROUPED ? 128 : 0));
  static constexpr int redp = TC + 4;               // floats of one reduction row
  static constexpr int red_row = kDmWaves * 16 * redp * 4;  // 16 rows of every wave
  // 16-row blocks reduced at a time: half the LDS where the registers let two workgroups
  // share a compute unit
  static constexpr int RC = cmin(RB, (4 * NCH * RB <= 12 ? 80 : 160) * 1024 / red_row);
  static constexpr int bytes = cmax(kDmWaves * stage_b, RC * red_row);
};

template <int NCH, int RB, int AI, bool GROUPED>
__global__ __launch_bounds__(64 * kDmWaves) void marlin_dense_mid_kernel(const void* A_, const uint32_t* B_,
                                                                         const void* s_, int M_, int N_, int K_,
                                                                         int splits_, void* C_, float* partial_,
                                                                         uint32_t* counters_) {
  // scalar arguments, preloaded into SGPRs (built with -amdgpu-kernarg-preload-count=14);
  // the fp16 pointers travel as void pointers, which keeps the kernel's name demangleable
  const DensePreArgs a{static_cast<const _Float16*>(A_), B_, static_cast<const _Float16*>(s_),
                       static_cast<_Float16*>(C_), M_, N_, K_, splits_, partial_, counters_};
  using T = DmLds<NCH, RB, GROUPED>;
  constexpr int MB = 16 * RB, TC = T::TC, KG = kDmWaves, NT = 4 * NCH;
  constexpr int WOFF = T::act_b, SOFF = WOFF + 2048 * NCH;
  static_assert(AI == 2 * RB || (RB == 1 && AI == 1), "AI: activation DMAs per stage, 8 rows each");
  __shared__ __attribute__((aligned(16))) uint8_t lds[T::bytes];
  typedef __attribute__((address_space(3))) uint8_t lds_u8;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int N = a.N, K = a.K, M = a.M, S = a.splits;

  // ---- tile of this workgroup: each XCD (block b on XCD b % 8) works through a
  // contiguous range, rows fastest, then splits, then columns ----
  const int ntm = (M + MB - 1) / MB;
  const int G = gridDim.x;
  int t = blockIdx.x;
  if ((G & 7) == 0) t = (t & 7) * (G >> 3) + (t >> 3);
  const int tm = (int)((unsigned)t % (unsigned)ntm);
  const int tz = (int)((unsigned)t / (unsigned)ntm);
  const int z = (int)((unsigned)tz % (unsigned)S), tn = (int)((unsigned)tz / (unsigned)S);
  const int m0 = tm * MB, n0 = tn * TC;
  // 64-deep k-steps [p0, p1) of the split; this wave takes p0 + wave, p0 + wave + 8, ...
  const int np = K >> 6;
  const int p0 = (int)((unsigned)(np * z) / (unsigned)S), p1 = (int)((unsigned)(np * (z + 1)) / (unsigned)S);
  const int mine = (p1 - p0 - wave + KG - 1) / KG;  // stages of this wave
  const int q0 = p0 + wave;                         // its first k-step

  // ---- DMA sources ----
  // activations: instruction u moves rows 8 u .. 8 u + 7 of the tile, 8 pieces per row,
  // swizzled as in sm24_mid.h; rows past M repeat row M - 1 (never stored)
  auto swz = [](int row) {
    const int p = (row >> 1) & 7;
    return (p & 5) | ((p & 4) >> 1);
  };
  uint32_t act_v[AI];
#pragma unroll
  for (int u = 0; u < AI; u++) {
    const int row = 8 * u + (lane >> 3);
    const int m = m0 + row < M ? m0 + row : M - 1;
    act_v[u] = ((uint32_t)m * (uint32_t)K + 8 * ((lane & 7) ^ swz(row))) * 2;
  }
  const char* gA = reinterpret_cast<const char*>(a.A) + 128 * (size_t)q0;
  // codes: instruction u moves k-tiles 2 (u % 2), + 1 of chunk u / 2; slot s of k-tile t
  // holds the 16-byte piece (ci, rq) with 8 rq + ci = s ^ 8 (t & 1), so that the reads of
  // one rq over all ci and two k-tiles fall on distinct banks
  const int ws = (lane & 31) ^ (8 * (lane >> 5));
  const uint32_t rowB = 8 * (uint32_t)N;
  const uint32_t wv = (uint32_t)(lane >> 5) * rowB + 8 * (uint32_t)n0 + 16 * (4 * (ws & 7) + (ws >> 3));
  const char* gB = reinterpret_cast<const char*>(a.B) + (size_t)q0 * 4 * rowB;
  // grouped scales of the tile's columns, 8 pieces per chunk
  const char* gS =
      reinterpret_cast<const char*>(a.s) + ((size_t)(q0 >> 1) * (uint32_t)N + n0) * 2 + 16 * cmin(lane, 8 * NCH - 1);
  uint8_t* const wlds = lds + wave * T::stage_b;  // this wave's buffer
  const uint32_t lb = (uint32_t)(size_t)(lds_u8*)lds + (uint32_t)(wave * T::stage_b);
  // DMAs of this wave's next stage
  auto issue = [&] {
#pragma unroll
    for (int u = 0; u < 2 * NCH; u++)
      dma16x1(lb + WOFF + 1024 * u, wv + (uint32_t)(u & 1) * 2 * rowB + 512 * (u >> 1), gB);
    if constexpr (GROUPED) {
      dma_lanes_v<8 * NCH>(lb + SOFF, gS);
      gS += (size_t)(KG / 2) * 2 * (uint32_t)N;
    }
#pragma unroll
    for (int u = 0; u < AI; u++) dma16x1(lb + 1024 * u, act_v[u], gA);
    gA += 128 * KG;
    gB += (size_t)(KG * 4) * rowB;
  };

  if (mine > 0) issue();  // uniform

  // ---- MFMA lane roles.  The weight is the A operand of v_mfma_f32_16x16x32_f16 (rows =
  // output columns), the activations the B operand.  Lane (rho, h) holds column
  // 16 jt + rho of a chunk (ci = rho & 7, byte half b = rho >> 3) and the 16 k of k-tile
  // h of the k-step: the first MFMA takes the low nibbles of its words rq = 0..3 (k 0..7
  // of the k-tile, in order), the second the high ones (k 8..15) ----
  const int h = lane >> 4, rho = lane & 15;
  const int ci = rho & 7, bh = rho >> 3;
  const uint32_t nsh = 8u * bh, ssh = 16u * bh;
  const uint32_t o_act0 = rho * 128 + 16 * ((2 * h) ^ swz(rho));
  const uint32_t o_act1 = rho * 128 + 16 * ((2 * h + 1) ^ swz(rho));
  // pieces (ci, rq) of k-tile h: slots 8 rq + ci, the 8-slot halves of odd k-tiles swapped
  const uint32_t o_w0 = WOFF + 512 * h + 16 * ci + 128 * (h & 1), o_w1 = WOFF + 512 * h + 16 * ci - 128 * (h & 1);
  uint32_t kMask, kMaskHi, kMagic;
  asm volatile("v_mov_b32 %0, 0x000f000f" : "=v"(kMask));
  asm volatile("v_mov_b32 %0, 0x00f000f0" : "=v"(kMaskHi));
  asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(kMagic));

  float4_t acc[NT][RB];
#pragma unroll
  for (int c = 0; c < NT; c++)
#pragma unroll
    for (int rb = 0; rb < RB; rb++) acc[c][rb] = (float4_t){0.f, 0.f, 0.f, 0.f};

  auto compute = [&](const uint8_t* st, auto refill) {
    // every LDS operand of the stage first, then the dequantisation and MFMAs
    u32x4 w[NCH][4], sc[NCH];
    half8_t act[RB][2];
#pragma unroll
    for (int ch = 0; ch < NCH; ch++) {
#pragma unroll
      for (int rq = 0; rq < 4; rq++)
        w[ch][rq] = *reinterpret_cast<const u32x4*>(st + (rq & 1 ? o_w1 : o_w0) + 2048 * ch + 128 * rq);
      if constexpr (GROUPED) sc[ch] = *reinterpret_cast<const u32x4*>(st + SOFF + 128 * ch + 16 * ci);
    }
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
      act[rb][0] = *reinterpret_cast<const half8_t*>(st + o_act0 + 2048 * rb);
      act[rb][1] = *reinterpret_cast<const half8_t*>(st + o_act1 + 2048 * rb);
    }
    // the stage is in registers: its buffer is free for the next one
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    refill();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < NT; c++) {
      const int ch = c >> 2, jt = c & 3;
      const half2_t kz = {(_Float16)1032.0f, (_Float16)1032.0f};
      const half2_t k16 = {(_Float16)0.0625f, (_Float16)0.0625f};
      const half2_t kzh = {(_Float16)-72.0f, (_Float16)-72.0f};
      half2_t lo[4], hi[4];
#pragma unroll
      for (int rq = 0; rq < 4; rq++) {
        const uint32_t x = w[ch][rq][jt] >> nsh;
        lo[rq] = __builtin_bit_cast(half2_t, (x & kMask) | kMagic) - kz;
        hi[rq] = __builtin_bit_cast(half2_t, (x & kMaskHi) | kMagic) * k16 + kzh;
      }
      half8_t a0 = {lo[0].x, lo[0].y, lo[1].x, lo[1].y, lo[2].x, lo[2].y, lo[3].x, lo[3].y};
      half8_t a1 = {hi[0].x, hi[0].y, hi[1].x, hi[1].y, hi[2].x, hi[2].y, hi[3].x, hi[3].y};
      if constexpr (GROUPED) {
        const _Float16 s = __builtin_bit_cast(half2_t, sc[ch][jt] >> ssh).x;
        const half8_t sv = {s, s, s, s, s, s, s, s};
        a0 = a0 * sv;
        a1 = a1 * sv;
      }
#pragma unroll
      for (int rb = 0; rb < RB; rb++) {
        acc[c][rb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, act[rb][0], acc[c][rb], 0, 0, 0);
        asm volatile("" : "+v"(acc[c][rb]));
      }
#pragma unroll
      for (int rb = 0; rb < RB; rb++) {
        acc[c][rb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, act[rb][1], acc[c][rb], 0, 0, 0);
        asm volatile("" : "+v"(acc[c][rb]));
      }
    }
  };

  // ---- main loop: a wave waits for its own DMAs of stage s, reads the stage into
  // registers, sends for the next one and computes ----
  for (int s = 0; s < mine; s++) {
    wait_vm<0>();
    compute(wlds, [&] {
      if (s + 1 < mine) issue();
    });
    __builtin_amdgcn_sched_barrier(0);
  }

  // ---- reduction: the 8 waves' sums, RC 16-row blocks at a time, in wave order; thread
  // e of the pass takes 4 columns of one row ----
  float* const red = reinterpret_cast<float*>(lds);
  constexpr int RP = T::redp, RC = T::RC, CQ = TC / 4;
  const int tile = tn * ntm + tm;
  auto part = [&](int zz, int row, int col) -> float* {
    return a.partial + (((size_t)tile * S + zz) * MB + row) * TC + col;
  };
  auto write_c = [&](int row, int col, float4_t v) {
    const int n = n0 + col;
    half4_t o;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      o[i] = (_Float16)v[i];
      if constexpr (!GROUPED) {
        // per-column scale of the fp16-rounded sum: within 32 columns, column c sits at
        // slot 8 ((c >> 1) & 3) + 2 ((c >> 3) & 3) + (c & 1)
        const int c = (n + i) & 31;
        o[i] = o[i] * a.s[((n + i) & ~31) + 8 * ((c >> 1) & 3) + 2 * ((c >> 3) & 3) + (c & 1)];
      }
    }
    *reinterpret_cast<half4_t*>(a.C + (size_t)(m0 + row) * N + n) = o;
  };
#pragma unroll
  for (int r0 = 0; r0 < RB; r0 += RC) {
    __syncthreads();
#pragma unroll
    for (int rb = r0; rb < cmin(r0 + RC, RB); rb++)
#pragma unroll
      for (int c = 0; c < NT; c++)
        *reinterpret_cast<float4_t*>(red + ((wave * RC + rb - r0) * 16 + rho) * RP + 16 * c + 4 * h) = acc[c][rb];
    __syncthreads();
    for (int e = tid; e < 16 * cmin(RC, RB - r0) * CQ; e += 64 * kDmWaves) {
      const int row = e / CQ, col = 4 * (e % CQ);
      if (m0 + 16 * r0 + row >= M) break;  // rows ascend with e
      const float* p = red + row * RP + col;
      float4_t v = *reinterpret_cast<const float4_t*>(p);
#pragma unroll
      for (int k = 1; k < KG; k++) v += *reinterpret_cast<const float4_t*>(p + k * RC * 16 * RP);
      if (S == 1) write_c(16 * r0 + row, col, v);
      else *reinterpret_cast<float4_t*>(part(z, 16 * r0 + row, col)) = v;
    }
  }
  if (S == 1) return;

  // ---- split-K hand-off through the uncached scratch: the last split to arrive adds all
  // partials in split order and writes C ----
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0);
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __syncthreads();
  uint32_t* const arrived = reinterpret_cast<uint32_t*>(lds);  // the reduction's reads are done
  if (tid == 0) *arrived = __hip_atomic_fetch_add(a.counters + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u;
  __syncthreads();
  if (*arrived != (uint32_t)S) return;
  if (tid == 0) __hip_atomic_store(a.counters + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (int e = tid; e < MB * CQ; e += 64 * kDmWaves) {
    const int row = e / CQ, col = 4 * (e % CQ);
    if (m0 + row >= M) break;
    float4_t v = {};
    for (int z0 = 0; z0 < S; z0 += 4) {
      float4_t q[4];
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (z0 + i < S) q[i] = *reinterpret_cast<const float4_t*>(part(z0 + i, row, col));
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (z0 + i < S) v = z0 + i == 0 ? q[0] : v + q[i];
    }
    write_c(row, col, v);
  }
}

// Tile (64 nch columns x 16 rb rows) and K splits of one call.
struct DenseMidShape {
  int nch, rb, splits;
};
hipError_t launch_dense_mid(const DensePreArgs& a, const DenseMidShape& d, bool grouped, hipStream_t stream);

}  // namespace sm24
