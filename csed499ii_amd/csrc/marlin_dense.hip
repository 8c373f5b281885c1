// Dense INT4 x FP16 GEMM on gfx950 (the reference's dense Marlin `mul`):
// C[M,N] = A[M,K] * W[K,N], W = (q - 8) * s with 4-bit codes q and fp16 scales.
//
// W is read in the dense Marlin pack() layout (reference
// kernel_experiments/sparse_marlin/src/marlin/__init__.py:78-99, 177-226):
//   * B  int32 [K/16][2N]: row r holds k-tile r (16 K).  Within a 64-column chunk c
//        (128 words) word w = 16*ci + 4*rq + jt holds, for the two columns
//        n = 64c + 16*jt + ci (bytes 0, 2) and n + 8 (bytes 1, 3), the codes of
//        k = 16r + {2rq, 2rq+8} (low / high nibble of byte 0 or 1) and
//        k = 16r + {2rq+1, 2rq+9} (low / high nibble of byte 2 or 3).
//   * s  fp16 [K/128][N] grouped: within 64 columns, slot 8i + j holds column i + 8j;
//        or [1][N] per column: within 32 columns, slot 8i + t holds column
//        2i + {0,1,8,9,16,17,24,25}[t] (applied to the fp16-rounded sum).
//
// The weight is the A operand of v_mfma_f32_16x16x32_f16 (rows = output columns),
// activations the B operand (columns = batch rows).  Lane (rho, h) = (l % 16, l / 16)
// of the MFMA for column tile jt holds column 64c + 16*jt + rho (ci = rho & 7, byte
// b = rho >> 3) and 8 k of k-tile kt = h >> 1 of the 32-deep k-step: k = 4(h&1) + 0..3
// (low nibbles of words rq = 2(h&1), 2(h&1)+1) and 8 + 4(h&1) + 0..3 (their high
// nibbles).  So one lane loads the two 16-byte word groups (ci, rq, jt = 0..3) and
// feeds the four column tiles of the chunk from them.
//
// Three kernels.  Up to 2048 rows mostly marlin_dense_mid.h, above that (and for much
// work) marlin_dense_prefill.h.  The kernel here takes what neither covers: activations of 4 GiB
// and more (their kernels address them by 32-bit offsets).  Its work decomposition: grid.x
// 64-column chunk, grid.z batch tile of 64 rows; NW waves take contiguous ranges of the
// k-steps through a ring of U in-flight fragments and are reduced in LDS in a fixed order.
//
// Reference: marlin_cuda_kernel.cu (Marlin at 90-605, host dispatch marlin_cuda at
// 655-736) and marlin_cuda.cpp:38-64 (the binding's checks).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdlib.h>

#include "marlin_dense_mid.h"
#include "marlin_dense_prefill.h"
#include "sm24_device.h"
#include "sm24_host.h"
#include "../../include/marlin_hip.h"

namespace sm24 {

struct DenseArgs {
  const _Float16* A;
  const uint32_t* B;
  const _Float16* s;
  _Float16* C;
  const _Float16* zeros;  // >= 64 zero bytes (rows past M)
  int M, N, K;
};

constexpr int BB = 4;  // 16-row blocks per batch tile

template <bool GROUPED>
struct DenseFrag {
  u32x4 w0, w1;      // word groups (ci, rq0, jt = 0..3) and (ci, rq0 + 1, jt = 0..3)
  half8_t sc;        // grouped: scale slots 8*ci .. 8*ci + 7 (columns ci + 8j)
  half8_t act[BB];   // activation B operands
};

// The fields the prologue needs first come as leading scalar arguments, preloaded
// into SGPRs (this translation unit is built with -mllvm
// -amdgpu-kernarg-preload-count=14), ahead of the whole DenseArgs; the fp16
// pointers travel as void pointers, which keeps the kernel's name demangleable.
template <int NW, bool GROUPED>
__global__ __launch_bounds__(64 * NW) void marlin_dense_kernel(const void* A_, const uint32_t* B_, const void* s_,
                                                               const void* zeros_, int M_, int N_, int K_, int nks_,
                                                               DenseArgs a_) {
  DenseArgs a = a_;
  a.A = static_cast<const _Float16*>(A_);
  a.B = B_;
  a.s = static_cast<const _Float16*>(s_);
  a.zeros = static_cast<const _Float16*>(zeros_);
  a.M = M_;
  a.N = N_;
  a.K = K_;
  constexpr int NT = 64 * NW;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int chunk = blockIdx.x, bt = blockIdx.z;
  const int N = a.N, K = a.K, M = a.M;
  const int h = lane >> 4, rho = lane & 15;
  const int ci = rho & 7, b = rho >> 3;
  const int kt = h >> 1, rq0 = 2 * (h & 1);
  const uint32_t sh = 8u * (uint32_t)b;

  // k-step ks reads B rows 2ks + kt: words (ci, rq0, 0..3) and (ci, rq0 + 1, 0..3)
  const uint32_t* bw = a.B + 128 * (size_t)chunk + 16 * ci + 4 * rq0 + 2 * (size_t)N * kt;
  const size_t bstep = 4 * (size_t)N;  // words per k-step (two rows)
  const _Float16* sp = a.s + 64 * (size_t)chunk + 8 * ci;
  const int row0 = 16 * BB * bt + rho;
  const int koff = 16 * kt + 4 * (h & 1);

  auto fetch = [&](int ks, bool live, DenseFrag<GROUPED>& f) {
    const uint32_t* p = bw + (size_t)ks * bstep;
    f.w0 = *reinterpret_cast<const u32x4*>(p);
    f.w1 = *reinterpret_cast<const u32x4*>(p + 4);
    if constexpr (GROUPED) f.sc = *reinterpret_cast<const half8_t*>(sp + (size_t)(ks >> 2) * N);
#pragma unroll
    for (int bb = 0; bb < BB; bb++) {
      // rows past M (and ring slots past the range) read the zero block: only the
      // address is selected, so the ring keeps a fixed shape
      const int m = row0 + 16 * bb;
      const _Float16* ap = (live && m < M) ? a.A + (size_t)m * K + 32 * ks + koff : a.zeros;
      const u32x2 lo = *reinterpret_cast<const u32x2*>(ap);
      const u32x2 hi = *reinterpret_cast<const u32x2*>(ap + 8);
      f.act[bb] = __builtin_bit_cast(half8_t, (u32x4){lo.x, lo.y, hi.x, hi.y});
    }
  };

  float4_t acc[BB][4];
#pragma unroll
  for (int bb = 0; bb < BB; bb++)
#pragma unroll
    for (int jt = 0; jt < 4; jt++) acc[bb][jt] = (float4_t){0.f, 0.f, 0.f, 0.f};

  // Dequant constants held in VGPRs, so that mask-and-or is one v_and_or_b32.
  uint32_t kMask, kMaskHi, kMagic;
  asm volatile("v_mov_b32 %0, 0x000f000f" : "=v"(kMask));
  asm volatile("v_mov_b32 %0, 0x00f000f0" : "=v"(kMaskHi));
  asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(kMagic));
  const uint32_t ssh = 16u * (uint32_t)b;  // the lane's scale: half b of scale word jt
  auto compute = [&](const DenseFrag<GROUPED>& f) {
#pragma unroll
    for (int jt = 0; jt < 4; jt++) {
      // column 16 jt + rho: byte b of words rq0 (k 4(h&1) + 0, 1 | 8 + ...) and rq0 + 1;
      // magic-exponent conversion as in dequant4 ({k, k+1 | k+8, k+9} of each word)
      const uint32_t x0 = f.w0[jt] >> sh, x1 = f.w1[jt] >> sh;
      const half2_t kz = {(_Float16)1032.0f, (_Float16)1032.0f};
      const half2_t k16 = {(_Float16)0.0625f, (_Float16)0.0625f};
      const half2_t kzh = {(_Float16)-72.0f, (_Float16)-72.0f};
      const half2_t l0 = __builtin_bit_cast(half2_t, (x0 & kMask) | kMagic) - kz;
      const half2_t l1 = __builtin_bit_cast(half2_t, (x1 & kMask) | kMagic) - kz;
      const half2_t u0 = __builtin_bit_cast(half2_t, (x0 & kMaskHi) | kMagic) * k16 + kzh;
      const half2_t u1 = __builtin_bit_cast(half2_t, (x1 & kMaskHi) | kMagic) * k16 + kzh;
      half8_t aop = (half8_t){l0.x, l0.y, l1.x, l1.y, u0.x, u0.y, u1.x, u1.y};
      if constexpr (GROUPED) {
        // scale slot 2 jt + b: one shift of word jt (a variable element index would
        // compile to a select over all eight halves)
        const uint32_t sw = __builtin_bit_cast(u32x4, f.sc)[jt] >> ssh;
        const _Float16 sc = __builtin_bit_cast(half2_t, sw).x;
        aop = aop * (half8_t){sc, sc, sc, sc, sc, sc, sc, sc};
      }
#pragma unroll
      for (int bb = 0; bb < BB; bb++)
        acc[bb][jt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(aop, f.act[bb], acc[bb][jt], 0, 0, 0);
    }
  };

  // Each wave streams a contiguous share of the split's k-steps through a ring of U
  // fragments; slots past the end re-read the last k-step with zero activations.
  constexpr int U = 4;
  const int r0 = nks_ * wave / NW, r1 = nks_ * (wave + 1) / NW;  // 32-deep k-steps
  if (r1 > r0) {
    const int rlast = r1 - 1;
    DenseFrag<GROUPED> ring[U];
#pragma unroll
    for (int i = 0; i < U; i++) {
      fetch(r0 + i < r1 ? r0 + i : rlast, r0 + i < r1, ring[i]);
      __builtin_amdgcn_sched_barrier(0);
    }
    for (int base = r0; base < r1; base += U) {
#pragma unroll
      for (int i = 0; i < U; i++) {
        compute(ring[i]);
        __builtin_amdgcn_sched_barrier(0);
        const int rn = base + i + U;
        fetch(rn < r1 ? rn : rlast, rn < r1, ring[i]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }

  // ---- reduce the NW waves in LDS: red[wave][row][col], col = column in the chunk ----
  constexpr int RS = 65;  // padded row stride (floats)
  __shared__ float red[NW][16 * BB][RS];
#pragma unroll
  for (int bb = 0; bb < BB; bb++)
#pragma unroll
    for (int jt = 0; jt < 4; jt++)
#pragma unroll
      for (int i = 0; i < 4; i++) red[wave][16 * bb + rho][16 * jt + 4 * h + i] = acc[bb][jt][i];
  __syncthreads();

  const int ntile = 16 * BB * 64;
  const int ncol0 = 64 * chunk;
  // per-column scale of chunk column nl (per-column quantization): slot 8 ((nl % 8) / 2)
  // + 2 (nl / 8) + nl % 2 of the 32-column half the column lies in
  auto col_scale = [&](int nl) -> _Float16 {
    const int c = nl & 31;
    return a.s[ncol0 + (nl & 32) + 8 * ((c & 7) >> 1) + 2 * (c >> 3) + (c & 1)];
  };
  for (int e = threadIdx.x; e < ntile; e += NT) {
    const int ml = e >> 6, nl = e & 63;
    const int m = 16 * BB * bt + ml;
    if (m >= M) continue;
    float v = red[0][ml][nl];
#pragma unroll
    for (int w = 1; w < NW; w++) v += red[w][ml][nl];
    _Float16 o = (_Float16)v;
    if constexpr (!GROUPED) o = o * col_scale(nl);
    a.C[(size_t)m * N + ncol0 + nl] = o;
  }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------

// The reference binding's and dispatch's shape rules (marlin_cuda.cpp:43-49,
// marlin_cuda_kernel.cu:660-683, 711-721): default tiles (thread_k, thread_n) =
// (128, 128) for at most 16 batch rows, else (64, 256); N % thread_n, K % thread_k
// and K % (groupsize / 16) (the reference's own test) or code 1; instantiated tiles
// (128, 128) for one 16-row block and (64, 256), with groupsize -1 or 128, or code 2.
int dense_validate(int prob_m, int prob_n, int prob_k, int groupsize, int thread_k, int thread_n) {
  if (thread_k == -1 || thread_n == -1) {
    if (prob_m <= 16) {
      thread_k = 128;
      thread_n = 128;
    } else {
      thread_k = 64;
      thread_n = 256;
    }
  }
  if (thread_k <= 0 || thread_n <= 0) return MARLIN_HIP_ERR_KERN_SHAPE;
  const int group_blocks = groupsize == -1 ? -1 : groupsize / 16;
  if (prob_n % thread_n != 0 || prob_k % thread_k != 0 || (group_blocks > 0 && prob_k % group_blocks != 0))
    return MARLIN_HIP_ERR_PROB_SHAPE;
  if (prob_m == 0 || prob_n == 0 || prob_k == 0) return MARLIN_HIP_OK;
  const bool tile_ok = (thread_n == 128 && thread_k == 128 && prob_m <= 16) || (thread_n == 256 && thread_k == 64);
  if (!tile_ok || !(group_blocks == -1 || group_blocks == 8)) return MARLIN_HIP_ERR_KERN_SHAPE;
  return MARLIN_HIP_OK;
}

template <bool G>
hipError_t launch_dense_t(const DenseArgs& a, dim3 grid, hipStream_t stream) {
  constexpr int NW = 4;
  hipLaunchKernelGGL((marlin_dense_kernel<NW, G>), grid, dim3(64 * NW), 0, stream, a.A, a.B, a.s, a.zeros, a.M, a.N,
                     a.K, a.K / 32, a);
  return hipGetLastError();
}

// Large-M path (marlin_dense_prefill_kernel): K a multiple of 128 (whole scale groups, an
// even number of 64-deep k-steps), N of its 512-column tile or of half of it (the last tile
// is then half empty).  32-bit operand offsets; from 65 rows.
// MARLIN_HIP_DENSE_PREFILL_MIN_M (>= 1) replaces the threshold, and then every call from it
// on runs this kernel, whatever dense_mid_fits estimates.
int dense_prefill_forced_min_m() {
  static const int v = [] {
    const char* e = getenv("MARLIN_HIP_DENSE_PREFILL_MIN_M");
    const int x = e ? atoi(e) : 0;
    return x >= 1 ? x : 0;
  }();
  return v;
}
bool dense_prefill_fits(int M, int N, int K) {
  const int min_m = dense_prefill_forced_min_m() ? dense_prefill_forced_min_m() : 65;
  return M >= min_m && N % (kDpTileCols / 2) == 0 && K % 128 == 0 && (long long)M * K < (1LL << 31) - 2048 &&
         (long long)K * N < (1LL << 33);
}

// K splits of the dense large-M kernel, by the 2:4 prefill planner's model: rounds of
// one workgroup per CU times the k-steps per split, plus the partial exchange (each
// split stores a 256 KiB fp32 tile), at ~1.3 us per 64-deep k-step of a tile (32
// MFMAs per wave) and ~2.5 TB/s for the exchange.  MARLIN_HIP_DENSE_PREFILL_SPLITS
// forces a count.  *estimate: the model's time of its own choice, us, forced or not.
int dense_prefill_splits(int tiles, int nks, int cus, double* estimate = nullptr) {
  static const int forced = [] {
    const char* e = getenv("MARLIN_HIP_DENSE_PREFILL_SPLITS");
    const int x = e ? atoi(e) : 0;
    return x >= 1 && x <= 16 ? x : 0;
  }();
  const int max_s = nks / 8 > 0 ? nks / 8 : 1;  // at least eight k-steps per split
  const double step_us = 1.3, exchange_bytes_per_us = 2.5e6;
  int best_s = 1;
  double best = 1e30;
  for (int s = 1; s <= 8 && s <= max_s; s++) {
    const long long rounds = ((long long)tiles * s + cus - 1) / cus;
    const double traffic = s > 1 ? 2.0 * tiles * s * (double)kDpSplitBytes : 0.0;
    const double cost = (double)rounds * step_us * nks / s + traffic / exchange_bytes_per_us;
    if (cost < 0.97 * best) {
      best = cost;
      best_s = s;
    }
  }
  if (estimate) *estimate = best;
  if (forced) best_s = forced < max_s ? forced : max_s;
  if ((size_t)tiles * sizeof(uint32_t) > kCounterBytes) best_s = 1;
  return best_s;
}

int run_dense_prefill(const void* A, const void* B, void* C, const void* s, int M, int N, int K, bool grouped,
                      int dev, hipStream_t stream, int sms) {
  DensePreArgs p{};
  p.A = static_cast<const _Float16*>(A);
  p.B = static_cast<const uint32_t*>(B);
  p.s = static_cast<const _Float16*>(s);
  p.C = static_cast<_Float16*>(C);
  p.M = M;
  p.N = N;
  p.K = K;
  const int tiles = ((N + kDpTileCols - 1) / kDpTileCols) * ((M + kDpRows - 1) / kDpRows);
  p.splits = dense_prefill_splits(tiles, K / 64, sms);
  if (p.splits > 1) {
    const int err = get_scratch(dev, stream, (size_t)tiles * p.splits * kDpSplitBytes, &p.counters, &p.partial);
    if (err != MARLIN_HIP_OK) return err;
    if (!p.counters) p.splits = 1;  // capturing, and this stream has no scratch yet
  }
  return launch_error(launch_dense_prefill(p, grouped, stream));
}

// Tile and K splits of the decode- and mid-batch kernel (marlin_dense_mid.h), from a cost
// model fitted to 2000 forced plans (every tile x splits 1-8 on eleven K x N, 1024x5120 to
// 8192x57344, M from 1 to 512, one box; mean error 5 %, the model's choices 0.6 % from the
// best of each call): a fixed cost, the stages of a wave at the tile's measured stage time
// per round of workgroups over the CUs (less for the small tiles, two of which share a CU),
// the reduction in LDS, the codes' bytes, and for a split the exchange of the fp32 partials
// (only up to one workgroup per CU).  *cost: the model's time of its own choice, us.
// MARLIN_HIP_DENSE_SPLITS (1-16, at most K / 256) forces the K splits, on the tile that the
// model then has the fastest.
DenseMidShape dense_mid_plan(int M, int N, int K, int cus, bool nosplit, double* cost) {
  static const int forced = [] {
    const char* e = getenv("MARLIN_HIP_DENSE_SPLITS");
    const int x = e ? atoi(e) : 0;
    return x >= 1 && x <= 16 ? x : 0;
  }();
  struct Cand {
    int nch, rb;
    double stage_us;
  };
  static const Cand cands[] = {{1, 1, 0.60}, {1, 2, 0.72}, {1, 3, 0.92}, {1, 4, 1.06}, {1, 5, 1.26},
                               {2, 1, 1.07}, {2, 2, 1.27}, {2, 3, 1.51}, {2, 4, 1.73}};
  DenseMidShape best{1, 1, 1}, fbest{0, 0, 0};
  double best_cost = 1e30, fbest_cost = 1e30;
  for (const Cand& c : cands) {
    if (N % (64 * c.nch) != 0) continue;
    const long long tiles = (long long)(N / (64 * c.nch)) * ((M + 16 * c.rb - 1) / (16 * c.rb));
    const bool counted = (size_t)tiles * sizeof(uint32_t) <= kCounterBytes;  // one arrival counter per tile
    auto us = [&](int s) {
      const double x = (double)(tiles * s) / cus;
      const double rounds = x <= 1 ? 1 : (double)((tiles * s + cus - 1) / cus);
      const double share = x > 1 && c.nch * c.rb <= 2 ? 0.89 : 1.0;
      const double f = share * rounds * (1 + 0.295 * (x / rounds - 0.75));
      double t = 2.7 + (K / 64 / s + 7) / 8 * c.stage_us * f + 0.50 * c.nch * c.rb * rounds + 2.8e-8 * K * (double)N;
      if (s > 1) t += 1.44 + 8.0 * s * M * (double)N / 7.5e6;
      return t;
    };
    for (int s = 1; s <= (nosplit ? 1 : 8); s++) {
      if (s > 1 && (tiles * s > cus || K / 64 < 8 * s || !counted)) break;
      const double t = us(s);
      if (t < best_cost) {
        best_cost = t;
        best = DenseMidShape{c.nch, c.rb, s};
      }
    }
    if (forced && !nosplit) {
      const int smax = K / 256 > 0 && counted ? K / 256 : 1, s = forced < smax ? forced : smax;
      const double t = us(s);
      if (t < fbest_cost) {
        fbest_cost = t;
        fbest = DenseMidShape{c.nch, c.rb, s};
      }
    }
  }
  if (cost) *cost = best_cost;
  return fbest.splits > 0 ? fbest : best;
}

// Whether a call runs the decode- and mid-batch kernel: up to 64 rows always, up to 2048
// where the large-M kernel does not take the shape or its own planner's estimate is not
// clearly lower.  Over the sweep above and 90 random shapes at 400-4096 rows this keeps
// the faster of the two or one within a few per cent of it up to 2048 rows (large-M ->
// this kernel, us: 943x1792x3584 43.7 -> 28.0, 768x11008x1536 68.1 -> 36.9, 1168x1280x1280
// 34.3 -> 12.2); beyond, two calls lost (3257x10752x2560 201.9 -> 224.3).  Below K = 512 the
// large-M kernel's fixed cost is most of its time, and the estimate has none of it: both
// kernels on 90 calls of K 128-384, N 1024-57344 and 65-2048 rows, one box (us, mid /
// large-M: 128x4096 at 512 rows 6.7 / 12.3, at 2048 22.2 / 14.4; 384x22016 at 131 15.4 /
// 19.1, at 512 42.1 / 21.6; 256x57344 at 2048 302 / 144); the rule takes the slower of the
// pair once (384x57344 at 65 rows, 20.8 / 16.4).  32-bit activation offsets.
constexpr int kDenseMidMaxM = 2048;
bool dense_mid_fits(int M, int N, int K, int cus) {
  if (M > kDenseMidMaxM || (long long)M * K >= (1LL << 31)) return false;
  if (!dense_prefill_fits(M, N, K)) return true;
  if (dense_prefill_forced_min_m()) return false;
  const int tiles = ((N + kDpTileCols - 1) / kDpTileCols) * ((M + kDpRows - 1) / kDpRows);
  double mid = 0.0, pre = 0.0;
  dense_mid_plan(M, N, K, cus, false, &mid);
  dense_prefill_splits(tiles, K / 64, cus, &pre);
  return mid < 0.82 * (pre + (K < 512 ? 15.5 : 6.0));
}

int run_dense_mid(const void* A, const void* B, void* C, const void* s, int M, int N, int K, bool grouped, int dev,
                  hipStream_t stream, int sms) {
  DensePreArgs p{};
  p.A = static_cast<const _Float16*>(A);
  p.B = static_cast<const uint32_t*>(B);
  p.s = static_cast<const _Float16*>(s);
  p.C = static_cast<_Float16*>(C);
  p.M = M;
  p.N = N;
  p.K = K;
  DenseMidShape d = dense_mid_plan(M, N, K, sms, false, nullptr);
  if (d.splits > 1) {
    const size_t tiles = (size_t)(N / (64 * d.nch)) * ((M + 16 * d.rb - 1) / (16 * d.rb));
    const int err =
        get_scratch(dev, stream, tiles * d.splits * 1024 * d.nch * d.rb * sizeof(float), &p.counters, &p.partial);
    if (err != MARLIN_HIP_OK) return err;
    if (!p.counters) d = dense_mid_plan(M, N, K, sms, true, nullptr);  // capturing, no scratch yet
  }
  p.splits = d.splits;
  return launch_error(launch_dense_mid(p, d, grouped, stream));
}

int run_dense(const void* A, const void* B, void* C, const void* s, int prob_m, int prob_n, int prob_k,
              int groupsize, int dev, hipStream_t stream, int thread_k, int thread_n, int sms) {
  int err = dense_validate(prob_m, prob_n, prob_k, groupsize, thread_k, thread_n);
  if (err != MARLIN_HIP_OK) return err;
  if (prob_m == 0 || prob_n == 0 || prob_k == 0) return MARLIN_HIP_OK;
  const int M = prob_m, N = prob_n, K = prob_k;
  if (N % 64 != 0 || K % 128 != 0) {  // implied by the tiles above; the kernel's own units
    set_error("marlin_hip: dense N must be a multiple of 64 and K of 128");
    return MARLIN_HIP_ERR_PROB_SHAPE;
  }
  DeviceScope scope(dev);
  if (!scope.ok) return MARLIN_HIP_ERR_LAUNCH;
  if (sms <= 0) {
    if (hipDeviceGetAttribute(&sms, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || sms <= 0)
      sms = 256;
  }
  if (dense_mid_fits(M, N, K, sms)) return run_dense_mid(A, B, C, s, M, N, K, groupsize != -1, dev, stream, sms);
  if (dense_prefill_fits(M, N, K)) return run_dense_prefill(A, B, C, s, M, N, K, groupsize != -1, dev, stream, sms);
  const int ztiles = (M + 16 * BB - 1) / (16 * BB);
  const int chunks = N / 64;
  DenseArgs a{};
  a.A = static_cast<const _Float16*>(A);
  a.B = static_cast<const uint32_t*>(B);
  a.s = static_cast<const _Float16*>(s);
  a.C = static_cast<_Float16*>(C);
  a.M = M;
  a.N = N;
  a.K = K;
  err = get_zeros(dev, stream, &a.zeros);
  if (err != MARLIN_HIP_OK) return err;
  const dim3 grid(chunks, 1, ztiles);
  return launch_error(groupsize != -1 ? launch_dense_t<true>(a, grid, stream) : launch_dense_t<false>(a, grid, stream));
}

}  // namespace sm24

extern "C" int marlin_hip_mul(const void* A, const void* B, void* C, void* s, int prob_m, int prob_n, int prob_k,
                              void* workspace, int groupsize, int dev, hipStream_t stream, int thread_k,
                              int thread_n, int sms, int max_par) {
  (void)workspace;
  (void)max_par;
  return sm24::run_dense(A, B, C, s, prob_m, prob_n, prob_k, groupsize, dev, stream, thread_k, thread_n, sms);
}
