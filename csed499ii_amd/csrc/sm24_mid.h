// Mid-sized batches (17 to 192 rows, narrow N up to 1024) of the 2:4 INT4 x FP16 GEMM for gfx950, where one
// workgroup per tile and K split covers the call in one round over the compute units.
//
// Work decomposition: a workgroup of 8 waves owns a tile of 16 NCB output columns (64 or
// 128) x 16 RB batch rows over the whole K or one K split.  Wave w computes every 8th
// 64-deep k-pair from the w-th on, for the whole tile, as NCB x RB
// v_smfmac_f32_16x16x64_f16 accumulators; the 8 waves' sums are added in LDS at the end,
// in wave order.  Nothing is shared before that, so no barrier runs in the main loop and
// the waves of a SIMD fall out of step: one reads LDS or waits while the other computes.
//
// What bounds it: the latency of the one stage that a wave has in flight, no unit's rate.
// On 7B qkv and o at 64 and 131 rows the waves wait 43-48 % of their life; the matrix cores
// are busy 9-18 % of it, LDS 29-40 %, and the path from L2 into a compute unit carries 20-28
// of its 64 bytes per clock, at 320-370 clocks per read (counters over the life of a wave).
// The activation rows are most of that traffic: 128 bytes per row and k-pair against 26 per
// column.  So they come by LDS-DMA in whole 128-byte lines, 8 rows to an instruction (every
// CU reading the same 64 rows of K = 4096: 5.8 us with the launch, against 7.2 in 64-byte
// pieces and 17 by loads into registers in operand order).  A wave has one stage buffer: it
// reads the due stage into registers in one go, sends for the next one into the same buffer
// and computes meanwhile.  Buffers for more stages were slower on every call (1 / 2 / 4
// stages, us: 7B qkv at M = 64 12.3 / 13.8 / 13.8, o at M = 131 8.6 / 9.6 / 9.8, 70B o at
// M = 64 15.3 / 15.9 / 16.8): the LDS they take goes from the tile (four 16-row blocks of
// one stage are 136 KiB over the 8 waves) or from a second workgroup on the compute unit.
// 4, 12 and 16 waves were slower than 8.
//
// us per call on one box, against the decode launches of up to 32 rows or the large-M
// kernel: M = 64 7B qkv 18.9 -> 12.4, o 14.6 -> 6.6, gate_up 21.3 -> 19.0,
// down 20.2 -> 12.9, 70B o 24.3 -> 15.2, down 56.7 -> 33.7; M = 131 7B o 15.9 -> 8.6, 70B
// qkv 35.9 -> 24.0; 2048x2048 at M = 96 17.4 -> 5.2.
#pragma once
#include "sm24_decode_dma.h"
#include "sm24_host.h"

namespace sm24 {

constexpr int kMidWaves = 8;

// One wave's stage buffer (its activation rows and weight side of one k-pair); the
// workgroup's reduction buffer lies in the same space.
template <int NCB, int RB, bool GROUPED, int VF, int MF>
struct MidLds {
  static constexpr int TC = 16 * NCB;
  static constexpr int act_b = 16 * RB * 128;                  // activation rows of one k-pair
  static constexpr int bpk = VF == VAL4 ? TC / 2 : 3 * TC / 8;  // 16-byte value pieces per k-block
  static constexpr int mpk = MF == META4 ? TC / 4 : 3 * TC / 16;
  static constexpr int sc_n = GROUPED ? TC / 8 : 0;
  static constexpr int nms = 2 * mpk + sc_n;                   // metadata and scale pieces of a stage
  static constexpr int stage_b = act_b + 16 * (2 * bpk + nms);
  static constexpr int vdma = (2 * bpk + 63) / 64, msdma = (nms + 63) / 64;  // weight DMAs
  static constexpr int redp = TC + 4;                          // floats of one reduction row
  static constexpr int red_row = kMidWaves * 16 * redp * 4;    // 16 rows of every wave
  // 16-row blocks reduced at a time: half the LDS where the registers let two workgroups
  // share a compute unit
  static constexpr int RC = cmin(RB, (NCB * RB <= 12 ? 80 : 160) * 1024 / red_row);
  static constexpr int bytes = cmax(kMidWaves * stage_b, RC * red_row);
};

template <int NCB, int RB, bool GROUPED, int VF, int MF>
__global__ __launch_bounds__(64 * kMidWaves) void sm24_mid_kernel(const void* B_, const void* meta_, const void* s_,
                                                                  const void* A_, const void* zeros_, int M_, int N_,
                                                                  int K_, int splits_, GemmArgs a_) {
  const GemmArgs a = with_lead(a_, B_, meta_, s_, A_, zeros_, M_, N_, K_, splits_);
  using T = MidLds<NCB, RB, GROUPED, VF, MF>;
  constexpr int MB = 16 * RB, TC = T::TC, KG = kMidWaves;
  constexpr int BPK = T::bpk, MPK = T::mpk, NMS = T::nms;
  constexpr int VOFF = T::act_b, MOFF = VOFF + 32 * BPK, SOFF = MOFF + 32 * MPK;
  static_assert(T::bytes <= 160 * 1024 && BPK <= 64, "one k-block of values per instruction");
  __shared__ __attribute__((aligned(16))) uint8_t lds[T::bytes];
  typedef __attribute__((address_space(3))) uint8_t lds_u8;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int N = a.N, K = a.K, M = a.M, S = a.splits;

  // ---- tile of this workgroup.  Each XCD (block b on XCD b % 8) works through a
  // contiguous range, rows fastest, then splits, then columns: the row tiles of a
  // column tile share its weight in that XCD's L2. ----
  const int ntm = (M + MB - 1) / MB;
  const int G = gridDim.x;
  int t = blockIdx.x;
  if ((G & 7) == 0) t = (t & 7) * (G >> 3) + (t >> 3);
  const int tm = (int)((unsigned)t % (unsigned)ntm);
  const int tz = (int)((unsigned)t / (unsigned)ntm);
  const int z = (int)((unsigned)tz % (unsigned)S), tn = (int)((unsigned)tz / (unsigned)S);
  const int m0 = tm * MB, n0 = tn * TC;
  // k-pairs [p0, p1) of the split; this wave takes p0 + wave, p0 + wave + 8, ...
  const int np = K >> 6;
  const int p0 = (int)((unsigned)(np * z) / (unsigned)S), p1 = (int)((unsigned)(np * (z + 1)) / (unsigned)S);
  const int mine = (p1 - p0 - wave + KG - 1) / KG;  // stages of this wave
  const int q0 = p0 + wave;                         // its first k-pair

  // ---- DMA sources ----
  // activations: instruction u moves rows 8 u .. 8 u + 7 of the tile, 8 pieces per row;
  // physical slot s of row r holds the logical 16-byte slot s ^ swz(r).  A ds_read_b128
  // serves lanes {0-3, 12-15, 20-27} and {4-11, 16-19, 28-31} of each half-wave together:
  // with this swz the rows and slots of the B-fragment reads below fall on distinct
  // banks.  Rows past M repeat row M - 1 (never stored); the host keeps 2 M K below 2^32.
  auto swz = [](int row) {
    const int p = (row >> 1) & 7;
    return (p & 5) | ((p & 4) >> 1);
  };
  uint32_t act_v[2 * RB];
#pragma unroll
  for (int u = 0; u < 2 * RB; u++) {
    const int row = 8 * u + (lane >> 3);
    const int m = m0 + row < M ? m0 + row : M - 1;
    act_v[u] = ((uint32_t)m * (uint32_t)K + 8 * ((lane & 7) ^ swz(row))) * 2;
  }
  const char* gA = reinterpret_cast<const char*>(a.A) + 128 * (size_t)q0;
  // packed values of both k-blocks, piece i of k-block i / BPK; 4-bit pieces of the odd
  // k-block swap 8-piece halves so that the two k-blocks a read touches lie on other banks
  constexpr int bpc = VF == VAL4 ? 8 : 6;  // packed bytes per column and k-block
  constexpr int VN = 2 * BPK <= 64 ? 2 * BPK : BPK;  // value pieces per instruction
  uint32_t val_v[T::vdma];
#pragma unroll
  for (int u = 0; u < T::vdma; u++) {
    const int i = VN * u + cmin(lane, VN - 1), kb = i / BPK, p = i % BPK;
    val_v[u] = (uint32_t)kb * bpc * (uint32_t)N + (uint32_t)bpc * n0 + 16u * (VF == VAL4 ? p ^ (8 * kb) : p);
  }
  const char* gB = static_cast<const char*>(a.B) + (size_t)q0 * (2 * bpc) * (uint32_t)N;
  // metadata of both k-blocks, then the scales of the k-pair's group
  constexpr int mpc = MF == META4 ? 4 : 3;  // metadata bytes per column and k-block
  const char* ms_p[T::msdma];
  uint32_t ms_inc[T::msdma];
#pragma unroll
  for (int u = 0; u < T::msdma; u++) {
    const int i = cmin(64 * u + lane, NMS - 1);
    if (i < 2 * MPK) {
      ms_p[u] = static_cast<const char*>(a.meta) + ((size_t)(2 * q0 + i / MPK) * mpc) * (uint32_t)N +
                (size_t)mpc * n0 + 16 * (i % MPK);
      ms_inc[u] = KG * 2 * mpc * (uint32_t)N;
    } else {
      ms_p[u] = reinterpret_cast<const char*>(a.s) + ((size_t)(q0 >> 1) * (uint32_t)N + n0) * 2 + 16 * (i - 2 * MPK);
      ms_inc[u] = KG / 2 * 2 * (uint32_t)N;
    }
  }
  uint8_t* const wlds = lds + wave * T::stage_b;  // this wave's buffer
  const uint32_t lb = (uint32_t)(size_t)(lds_u8*)lds + (uint32_t)(wave * T::stage_b);
  // DMAs of this wave's next stage
  auto issue = [&] {
    static_for<0, T::vdma>([&](auto ui) {
      constexpr int u = decltype(ui)::value;
      if constexpr (VN == 64) dma16x1(lb + VOFF + 16 * VN * u, val_v[u], gB);
      else dma_lanes_v<VN>(lb + VOFF + 16 * VN * u, gB + val_v[u]);
    });
    static_for<0, T::msdma>([&](auto ui) {
      constexpr int u = decltype(ui)::value;
      dma_lanes_v<cmin(64, NMS - 64 * u)>(lb + MOFF + 1024 * u, ms_p[u]);
      ms_p[u] += ms_inc[u];
    });
#pragma unroll
    for (int u = 0; u < 2 * RB; u++) dma16x1(lb + 1024 * u, act_v[u], gA);
    gA += 128 * KG;
    gB += (size_t)(KG * 2 * bpc) * (uint32_t)N;
  };

  if (mine > 0) issue();  // uniform

  // ---- MFMA lane roles (as in sm24_decode_kernel) ----
  const int h = lane >> 4, rho = lane & 15;
  const int gl = rho >> 3, blk = (rho >> 2) & 1, j = rho & 3;
  const int jb = j >> 1, jj = j & 1;
  const int t0 = 2 * (h & 1), kh = h >> 1;
  const int au = kh | ((h & 1) << 1);
  const uint32_t nsh = 8u * blk;
  const uint32_t msel = (uint32_t)(2 * blk + (h & 1)) | ((uint32_t)(4 + 2 * blk + (h & 1)) << 8) | 0x0c0c0000u;
  const uint32_t m3pos = 3u * (4u * blk + 2u * (h & 1));
  const uint32_t m3s0 = (jb ? 24u : 0u) + m3pos, m3s1 = (jb ? 40u : 16u) + m3pos;
  const uint32_t m3tlo = jb ? kTabLowLo : kTabHighLo, m3thi = jb ? kTabLowHi : kTabHighHi;
  const int wi_lane = 16 * gl + 4 * t0 + j;
  // logical slots au and 4 + au of row 16 rb + rho
  const uint32_t o_act0 = rho * 128 + 16 * (au ^ swz(rho));
  const uint32_t o_act1 = rho * 128 + 16 * ((4 + au) ^ swz(rho));
  // 4-bit words (2 cb + gl, t0, j): piece 8 cb + 4 gl + t0 of k-block kh, halves swapped for kh = 1
  const uint32_t o_val = VOFF + 16 * BPK * kh + (VF == VAL4 ? 4 * wi_lane : 0);
  const uint32_t o_val2[2] = {o_val + 128 * kh, o_val - 128 * kh};  // even, odd cb
  const uint32_t o_meta = MOFF + 16 * MPK * kh + jb * 128 + 8 * (2 * gl + jj);
  const uint32_t o_mrow = MOFF + 16 * MPK * kh;
  const uint32_t o_scale = SOFF + 2 * (8 * gl + 2 * j + blk);
  uint32_t kMask, kMaskHi, kMagic;
  if constexpr (VF == VAL4) {
    asm volatile("v_mov_b32 %0, 0x000f000f" : "=v"(kMask));
    asm volatile("v_mov_b32 %0, 0x00f000f0" : "=v"(kMaskHi));
  } else {
    asm volatile("v_mov_b32 %0, 0x00070007" : "=v"(kMask));
    asm volatile("v_mov_b32 %0, 0x00380038" : "=v"(kMaskHi));
  }
  asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(kMagic));

  float4_t acc[NCB][RB];
#pragma unroll
  for (int cb = 0; cb < NCB; cb++)
#pragma unroll
    for (int rb = 0; rb < RB; rb++) acc[cb][rb] = (float4_t){0.f, 0.f, 0.f, 0.f};

  auto compute = [&](const uint8_t* st, auto refill) {
    // every LDS operand of the stage first, then the dequantisation and MFMAs; the raw
    // 3-bit operands of 128 columns take more registers and come in two halves
    constexpr int HB = NCB == 8 && (VF != VAL4 || MF != META4) ? 4 : NCB;
    half16_t act[RB];
    uint32_t xr[HB][VF == VAL4 ? 2 : 4];
    u32x2 mr[HB];
    uint32_t m3y[HB][2], m3l[HB][2];
    _Float16 sr[HB];
#pragma unroll
    for (int c0 = 0; c0 < NCB; c0 += HB) {
#pragma unroll
      for (int cb = c0; cb < c0 + HB; cb++) {
        if constexpr (VF == VAL4) {
          const uint8_t* vp4 = st + o_val2[cb & 1] + 128 * cb;
          xr[cb - c0][0] = *reinterpret_cast<const uint32_t*>(vp4);
          xr[cb - c0][1] = *reinterpret_cast<const uint32_t*>(vp4 + 16);
        } else {
          const uint8_t* rowp = st + o_val;
          const int b0 = 3 * (wi_lane + 32 * cb), b1 = b0 + 12;
          const uint32_t* w0 = reinterpret_cast<const uint32_t*>(rowp + (b0 & ~3));
          const uint32_t* w1 = reinterpret_cast<const uint32_t*>(rowp + (b1 & ~3));
          xr[cb - c0][0] = w0[0];
          xr[cb - c0][1] = w0[1];
          xr[cb - c0][2] = w1[0];
          xr[cb - c0][3] = w1[1];
        }
        if constexpr (MF == META4) {
          mr[cb - c0] = *reinterpret_cast<const u32x2*>(st + o_meta + 256 * (cb >> 2) + 32 * (cb & 3));
        } else {
          const uint32_t* mrow = reinterpret_cast<const uint32_t*>(st + o_mrow + 192 * (cb >> 2));
          const int gt = 2 * (cb & 3) + gl;
#pragma unroll
          for (int e = 0; e < 2; e++) {
            const int ix = 16 * (gt >> 2) + ((4 * gt + 2 * jj + e) & 15), iy = ix + 16;
            m3y[cb - c0][e] = mrow[iy];
            m3l[cb - c0][e] = mrow[((gt >> 2) == 0 ? m3s0 : m3s1) >= 32u ? iy : ix];
          }
        }
        if constexpr (GROUPED) sr[cb - c0] = *reinterpret_cast<const _Float16*>(st + o_scale + 32 * cb);
      }
      if (c0 == 0) {
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
          const half8_t lo = *reinterpret_cast<const half8_t*>(st + o_act0 + 2048 * rb);
          const half8_t hi = *reinterpret_cast<const half8_t*>(st + o_act1 + 2048 * rb);
          act[rb] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
        }
      }
      // the stage is in registers: its buffer is free for the next one
      if (c0 + HB == NCB) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        refill();
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int cb = c0; cb < c0 + HB; cb++) {
        uint32_t x0, x1;
        if constexpr (VF == VAL4) {
          x0 = xr[cb - c0][0] >> nsh;
          x1 = xr[cb - c0][1] >> nsh;
        } else {
          const int b0 = 3 * (wi_lane + 32 * cb), b1 = b0 + 12;
          const uint32_t y0 = __builtin_amdgcn_alignbit(xr[cb - c0][1], xr[cb - c0][0], 8 * (b0 & 3) + 6 * blk);
          const uint32_t y1 = __builtin_amdgcn_alignbit(xr[cb - c0][3], xr[cb - c0][2], 8 * (b1 & 3) + 6 * blk);
          x0 = (y0 & 0x0000FFFFu) | ((y0 << 4) & 0xFFFF0000u);
          x1 = (y1 & 0x0000FFFFu) | ((y1 << 4) & 0xFFFF0000u);
        }
        const uint32_t lo0 = (x0 & kMask) | kMagic, lo1 = (x1 & kMask) | kMagic;
        const uint32_t hi0 = (x0 & kMaskHi) | kMagic, hi1 = (x1 & kMaskHi) | kMagic;
        constexpr float zp = VF == VAL4 ? 1032.0f : 1028.0f;
        constexpr float hs = VF == VAL4 ? 0.0625f : 0.125f;
        constexpr float zh = (zp - 1024.0f) + 1024.0f * hs;
        const half2_t kz = {(_Float16)zp, (_Float16)zp};
        const half2_t k16 = {(_Float16)hs, (_Float16)hs};
        const half2_t kzh = {(_Float16)-zh, (_Float16)-zh};
        const half2_t l0 = __builtin_bit_cast(half2_t, lo0) - kz, l1 = __builtin_bit_cast(half2_t, lo1) - kz;
        const half2_t u0 = __builtin_bit_cast(half2_t, hi0) * k16 + kzh;
        const half2_t u1 = __builtin_bit_cast(half2_t, hi1) * k16 + kzh;
        half8_t aop = (half8_t){l0.x, l0.y, l1.x, l1.y, u0.x, u0.y, u1.x, u1.y};
        uint32_t idx;
        if constexpr (MF == META4) {
          idx = __builtin_amdgcn_perm(mr[cb - c0].y, mr[cb - c0].x, msel);
        } else {
          uint32_t v[2];
#pragma unroll
          for (int e = 0; e < 2; e++)
            v[e] = __builtin_amdgcn_alignbit(m3y[cb - c0][e], m3l[cb - c0][e],
                                             ((2 * (cb & 3) + gl) >> 2 == 0 ? m3s0 : m3s1) & 31u);
          const uint32_t s2 = __builtin_amdgcn_perm(v[1], v[0], 0x0c0c0400u);
          const uint32_t sel = (s2 | (s2 << 13)) & 0x07070707u;
          const uint32_t nib = __builtin_amdgcn_perm(m3thi, m3tlo, sel);
          idx = (nib & 0x0f0fu) | ((nib >> 12) & 0xf0f0u);
        }
        if constexpr (GROUPED) {
          const _Float16 sc = sr[cb - c0];
          aop = aop * (half8_t){sc, sc, sc, sc, sc, sc, sc, sc};
        }
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
          acc[cb][rb] = smfmac64<0>(aop, act[rb], acc[cb][rb], idx);
          asm volatile("" : "+v"(acc[cb][rb]));
        }
      }
      __builtin_amdgcn_sched_barrier(0);
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
      if constexpr (!GROUPED) o[i] = o[i] * a.s[n + i];
    }
    *reinterpret_cast<half4_t*>(a.C + (size_t)(m0 + row) * N + n) = o;
  };
#pragma unroll
  for (int r0 = 0; r0 < RB; r0 += RC) {
    __syncthreads();
#pragma unroll
    for (int rb = r0; rb < cmin(r0 + RC, RB); rb++)
#pragma unroll
      for (int cb = 0; cb < NCB; cb++)
        *reinterpret_cast<float4_t*>(red + ((wave * RC + rb - r0) * 16 + rho) * RP + 16 * cb + 4 * h) = acc[cb][rb];
    __syncthreads();
    for (int e = tid; e < 16 * cmin(RC, RB - r0) * CQ; e += 64 * kMidWaves) {
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

  // ---- split-K hand-off through the uncached scratch, as in the decode kernels: the last
  // split to arrive adds all partials in split order and writes C.  It ends inside the
  // launch: the calls of a stream share the scratch, and a launch of another host thread
  // may lie between two of a call ----
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __builtin_amdgcn_s_waitcnt(0);
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
  __syncthreads();
  uint32_t* const arrived = reinterpret_cast<uint32_t*>(lds);  // the reduction's reads are done
  if (tid == 0) *arrived = __hip_atomic_fetch_add(a.counters + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u;
  __syncthreads();
  if (*arrived != (uint32_t)S) return;
  if (tid == 0) __hip_atomic_store(a.counters + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (int e = tid; e < MB * CQ; e += 64 * kMidWaves) {
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

// Launch of one operand format (sm24_mid.hip, sm24_mid_w3.hip, sm24_mid_m3.hip).
template <int VF, int MF>
hipError_t launch_mid_t(const GemmArgs& a, const MidShape& d, bool grouped, hipStream_t stream);

template <int NCB, int RB, int VF, int MF>
void launch_mid_v(const GemmArgs& a, bool grouped, dim3 grid, hipStream_t stream) {
  const dim3 block(64 * kMidWaves);
  if (grouped)
    hipLaunchKernelGGL((sm24_mid_kernel<NCB, RB, true, VF, MF>), grid, block, 0, stream, a.B, a.meta, a.s, a.A,
                       a.zeros, a.M, a.N, a.K, a.splits, a);
  else
    hipLaunchKernelGGL((sm24_mid_kernel<NCB, RB, false, VF, MF>), grid, block, 0, stream, a.B, a.meta, a.s, a.A,
                       a.zeros, a.M, a.N, a.K, a.splits, a);
}

#define SM24_MID_INSTANTIATE(VF, MF)                                                                     \
  template <>                                                                                            \
  hipError_t launch_mid_t<VF, MF>(const GemmArgs& a, const MidShape& d, bool grouped, hipStream_t stream) { \
    const dim3 grid(a.N / (16 * d.ncb) * ((a.M + 16 * d.rb - 1) / (16 * d.rb)) * a.splits);               \
    if (d.ncb == 4) {                                                                                    \
      if (d.rb == 1) launch_mid_v<4, 1, VF, MF>(a, grouped, grid, stream);                               \
      else if (d.rb == 2) launch_mid_v<4, 2, VF, MF>(a, grouped, grid, stream);                          \
      else if (d.rb == 3) launch_mid_v<4, 3, VF, MF>(a, grouped, grid, stream);                          \
      else if (d.rb == 4) launch_mid_v<4, 4, VF, MF>(a, grouped, grid, stream);                          \
      else launch_mid_v<4, 5, VF, MF>(a, grouped, grid, stream);                                         \
    } else {                                                                                             \
      if (d.rb == 2) launch_mid_v<8, 2, VF, MF>(a, grouped, grid, stream);                               \
      else if (d.rb == 3) launch_mid_v<8, 3, VF, MF>(a, grouped, grid, stream);                          \
      else launch_mid_v<8, 4, VF, MF>(a, grouped, grid, stream);                                         \
    }                                                                                                    \
    return hipGetLastError();                                                                            \
  }

}  // namespace sm24
