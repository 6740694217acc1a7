// pz_lmhead.hip -- the LM head producing the sampler's logits on the device,
// and the same product with greedy argmax fused into its epilogue.
//
// Reference: src/transformer/forward.c:102-168 runs the classifier
// parallel_matmul_bf16 (src/math/parallel_matmul.c:283-414):
//   logits[i] = sum_j bf16(W[i, j]) * x[j]
// with W [V, n] row-major bf16 (the upper half of an fp32; widening is a
// 16-bit shift), x the fp32 final-norm activations and fp32 accumulation.
// Here B activation rows are done at once: logits[b, i] = W[i, :] . x[b, :].
//
// Batch 4 and up run on the matrix cores (k_lmhead_mfma, below).  Batches of
// 1 to 3 use the vector kernel.
//
// Vector kernel layout and schedule (HBM-bound: W is read once per batch
// tile, 2 bytes per weight):
//   * a workgroup of 4 waves owns 64 consecutive rows of W; the batch tile of
//     x (BT rows x n fp32) is staged in LDS once per workgroup;
//   * a wave takes 4 rows of W at a time; lane l covers elements
//     512 c + 8 l .. +7 of every row (one 16-byte load per row per c), the
//     next chunk's (or the next rows') loads on their way during a chunk's
//     multiply-adds: 6.7 TB/s at 128256 x 2560, batch 1 (5.7 with the loads
//     of a chunk waited for at once and cached);
//   * each lane accumulates with fused multiply-adds in a fixed order (c,
//     then the 8 elements), and a DPP tree sums the 64 lanes.
// The order differs from the reference's AVX-512 accumulators, so logits
// agree with an exact product to fp32 rounding, not bit for bit; the fused
// argmax sees exactly the values the unfused kernel writes, because both are
// the same template.
//
// Fused epilogue (greedy, src/sampling/argmax.c:3-13): the first maximum by
// strict '>' is the largest value with the lowest id among equals, NaN never
// winning, and a NaN logit at id 0 returns 0.  Each workgroup reduces its
// rows to one 64-bit key per batch row -- the order key of the value above,
// ~id below -- and takes the atomic maximum in global memory; the workgroup
// that owns id 0 records whether logit 0 is NaN.  A finishing kernel turns
// keys into ids and clears them for the next call.
#include <hip/hip_runtime.h>

#include "../../include/pz_sampler.h"
#include "pz_device.h"
#include "pz_lmtile.h"
#include "pz_sampler_impl.h"

namespace {

constexpr int LM_WAVES = 4;
constexpr int LM_RW = 4;                        // rows per wave step
constexpr int LM_ROWS = 64;                     // rows per workgroup
constexpr int LM_STEPS = LM_ROWS / (LM_WAVES * LM_RW);
constexpr size_t LM_LDS_MAX = 96 * 1024;        // x tile budget

// The 8 weights of one 16-byte load (little-endian: element 2k is the low
// half of word k).
typedef uint32_t lm_u32x4 __attribute__((ext_vector_type(4)));
typedef float lm_f32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void widen8(const lm_u32x4 q, float (&w)[8]) {
#pragma unroll
  for (int i = 0; i < 4; i++) {
    w[2 * i] = __uint_as_float(q[i] << 16);
    w[2 * i + 1] = __uint_as_float(q[i] & 0xffff0000u);
  }
}

__device__ __forceinline__ uint64_t argmax_key(float v, int id) {
  return ((uint64_t)pz_key(v) << 32) | (uint64_t)(0xffffffffu - (uint32_t)id);
}

// MODE 0: write logits.  MODE 1: argmax keys.  VEC: n % 8 == 0 and W 16-byte
// aligned (one 16-byte load per 8 weights), else element loads.
template <int BT, int MODE, bool VEC, bool NT>
__global__ __launch_bounds__(64 * LM_WAVES) void k_lmhead(
    const uint16_t* __restrict__ W, int V, int n, const float* __restrict__ X, long ldx, int nb,
    float* __restrict__ logits, long ld, unsigned long long* __restrict__ keys,
    uint8_t* __restrict__ nan0) {
  extern __shared__ __align__(16) float xs[];  // [BT][n rounded up to 512]
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nchunk = (n + 511) >> 9;
  // the wave's weights, one chunk of its 4 rows ahead of the multiply-adds
  // (the first before the activations are staged)
  const int wrow0 = blockIdx.x * LM_ROWS + w * LM_RW;
  lm_u32x4 q[LM_RW];
  auto fetch = [&](int r0, int c) {
    const int k = c * 512 + lane * 8;
#pragma unroll
    for (int r = 0; r < LM_RW; r++) {
      const int row = r0 + r < V ? r0 + r : V - 1;  // rows past V: a valid row, result unused
      const uint16_t* wr = W + (size_t)row * n;
      q[r] = lm_u32x4{0u, 0u, 0u, 0u};
      if (VEC) {
        const lm_u32x4* p = reinterpret_cast<const lm_u32x4*>(wr + k);
        if (k < n) q[r] = NT ? __builtin_nontemporal_load(p) : *p;
      } else {
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const uint32_t h = k + e < n ? wr[k + e] : 0u;
          q[r][e >> 1] |= h << (16 * (e & 1));
        }
      }
    }
  };
  if (wrow0 < V) fetch(wrow0, 0);
  const int ns = nchunk * 512;  // a staged row: zeros past n
  for (int b = 0; b < BT; b++)
    for (int j = tid; j < ns; j += 64 * LM_WAVES)
      xs[b * ns + j] = b < nb && j < n ? X[(size_t)b * ldx + j] : 0.0f;
  __syncthreads();
  unsigned long long best[BT];
#pragma unroll
  for (int b = 0; b < BT; b++) best[b] = 0ull;
  for (int step = 0; step < LM_STEPS; step++) {
    const int r0 = wrow0 + step * LM_WAVES * LM_RW;
    if (r0 >= V) break;  // whole wave
    float acc[LM_RW][BT];
#pragma unroll
    for (int r = 0; r < LM_RW; r++)
#pragma unroll
      for (int b = 0; b < BT; b++) acc[r][b] = 0.0f;
    for (int c = 0; c < nchunk; c++) {
      const int k = c * 512 + lane * 8;
      float wv[LM_RW][8];
#pragma unroll
      for (int r = 0; r < LM_RW; r++) widen8(q[r], wv[r]);
      {
        // the next chunk, or the next rows' first
        const bool more = c + 1 < nchunk;
        const int rn = more ? r0 : r0 + LM_WAVES * LM_RW;
        if (more || (step + 1 < LM_STEPS && rn < V)) fetch(rn, more ? c + 1 : 0);
      }
#pragma unroll
      for (int b = 0; b < BT; b++) {
        const lm_f32x4 x0 = *reinterpret_cast<const lm_f32x4*>(&xs[b * ns + k]);
        const lm_f32x4 x1 = *reinterpret_cast<const lm_f32x4*>(&xs[b * ns + k + 4]);
        const float xv[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
#pragma unroll
        for (int r = 0; r < LM_RW; r++)
#pragma unroll
          for (int e = 0; e < 8; e++) acc[r][b] = __builtin_fmaf(wv[r][e], xv[e], acc[r][b]);
      }
    }
#pragma unroll
    for (int r = 0; r < LM_RW; r++) {
      const int row = r0 + r;
#pragma unroll
      for (int b = 0; b < BT; b++) {
        const float v = pz_wave_sum(acc[r][b]);  // uniform
        if (row < V && b < nb) {
          if (MODE == 0) {
            if (lane == 0) logits[(size_t)b * ld + row] = v;
          } else {
            if (row == 0 && lane == 0) nan0[b] = v != v ? 1 : 0;
            if (!(v != v)) {
              const unsigned long long kk = argmax_key(v, row);
              best[b] = kk > best[b] ? kk : best[b];
            }
          }
        }
      }
    }
  }
  if (MODE == 1) {
    // the waves' keys meet where the activations were: LDS of their own would
    // leave room for one workgroup per CU less where the activations take a
    // half or a quarter of it (8 batch rows of 2049 weights x 50257: 370 us
    // with it, 238 without; 4 of 5001 x 32000: 412 and 277)
    unsigned long long* best_sh = reinterpret_cast<unsigned long long*>(xs);  // [LM_WAVES][BT]
    __syncthreads();
    if (lane == 0)
#pragma unroll
      for (int b = 0; b < BT; b++) best_sh[w * BT + b] = best[b];
    __syncthreads();
    if (tid < BT && tid < nb) {
      unsigned long long m = best_sh[tid];
      for (int i = 1; i < LM_WAVES; i++) m = best_sh[i * BT + tid] > m ? best_sh[i * BT + tid] : m;
      if (m) atomicMax(&keys[tid], m);
    }
  }
}

// ---- batch >= 4: bf16 MFMA ---------------------------------------------------
// logits[b, i] = W[i, :] . x[b, :] as a GEMM on the matrix cores.  Each fp32
// activation is split into three bf16 parts, x = x0 + x1 + x2 (its 24
// significant bits in three 8-bit pieces, by truncation: exact for finite x;
// an infinite or NaN x keeps x0 = x and zero parts), so every bf16 x bf16
// product is exact in fp32 and the sum of the three part-products per weight
// is the fp32-accumulated product the reference forms -- the order of the
// fp32 additions differs (as it does in the VALU kernel), inside the same
// summation bound.  A weight of +-inf would meet a zero part (inf * 0 = NaN
// where the reference has +-inf): a workgroup that saw one recomputes those
// rows with fp32 fused multiply-adds before its epilogue.
//
//   * k_lmx_split writes the parts once per call into the sampler's
//     workspace, in the order the matrix cores read them ("fragments": 16
//     batch rows x 32 k of one part, lane l's 8 values at 16 l), so the GEMM
//     moves them to LDS and reads them back without conversions or bank
//     conflicts.  Converting inside the GEMM instead cost every workgroup
//     the whole conversion again, and LDS writes of 2 bytes per lane.
//   * v_mfma_f32_16x16x32_bf16: A = 16 rows of W x 32 k, B = 32 k x 16 batch
//     rows of one part, D = 16 rows x 16 batch rows (lane l: batch row l %
//     16, rows 4 (l / 16) .. +3).  The smallest part goes first.
//   * A workgroup owns WR TR x 16 rows of W and WC TC x 16 batch rows; wave
//     (wr, wc) TR x TC tiles of it.  k advances in stages of KS x 32, NS
//     stages of LDS in a ring: W and parts come by LDS-direct 16-byte loads
//     (global_load_lds_dwordx4) NS - 1 stages ahead, one barrier per stage,
//     the loads spread between the stage's MFMAs.
//   * KS = 2: one load instruction takes 8 rows x 128 bytes of W, whole
//     cache lines (64-byte pieces, KS = 1, reach 4.2 TB/s at 16 batch rows
//     where KS = 2 reaches 5.6); the 16-byte pieces of a row are rotated by
//     XOR with the row in the source address so that the fragment reads do
//     not meet in the banks.  The 256 x 256 tile's stage only fits with
//     KS = 1; it is bound by the matrix cores, not by that.
//   * NS = 0: no workspace and no ring -- every workgroup makes its batch
//     rows' parts itself, KS k-steps at a time, W straight into registers --
//     for rows longer than the workspace serves (16 batch rows at 4000 x
//     131080: 2.7 ms, 3.7 before there was a workspace) and for short ones
//     (lm_own_parts).  KS = 2 leaves room for several workgroups per CU, which
//     cover each other's waits: KS = 4 took 29.4 us where 2 takes 25.1 (32 x
//     512 x 128256).
//   * 128256 x 2560: 16 batch rows 112 us, 32 124, 64 167, 128 237, 256 405
//     (one launch per 32 rows that split the activations in every workgroup
//     took 143, 152, 301, 601 and 1203).
//   * Bounds: above about 64 batch rows the three parts' 6 V n B operations
//     (1.3 PFLOP/s at 256 rows, against 1.65 for a large library bf16 product
//     on the same card), below that one read of W.
//   * Every tile adds up k in the same order (32 k at a time from 0, the
//     smallest part first), so a logit depends on its row of W and its
//     activations alone: equal rows of W tie wherever they lie, and a batch
//     row's logits are the same in any batch.  (Row tiles that each start k
//     at another stage spread rows a multiple of 4 KiB apart over the memory
//     channels, 16 batch rows at 160000 x 2048 in 126 us instead of 166, but
//     give equal rows different sums.)
// Workgroups of one row tile (its batch blocks) are consecutive on one XCD,
// so its L2 serves W to all but the first.
// MODE 1 (argmax keys) as in k_lmhead.
typedef __bf16 lm_bf16x8 __attribute__((ext_vector_type(8)));
typedef uint16_t lm_u16x2 __attribute__((ext_vector_type(2)));
constexpr int LMX_FRAG = 512;  // bf16 of one fragment (16 x 32)

__device__ __forceinline__ float lm_bf16_f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

// Keys of the fused argmax spread over LMM_SLOTS slots per batch row (one
// per workgroup index modulo LMM_SLOTS, each on its own cache line), so the
// workgroups' atomics do not all meet on the batch's few words.
constexpr int LMM_SLOTS = 16;

// The three bf16 parts of 8 activations, two to a word.
__device__ __forceinline__ void lm_split8(const float (&x)[8], lm_u32x4 (&h)[3]) {
#pragma unroll
  for (int e = 0; e < 8; e++) {
    const uint32_t ux = __float_as_uint(x[e]);
    const bool fin = (ux & 0x7f800000u) != 0x7f800000u;
    // (a NaN whose payload sits in the low bits stays a NaN)
    const uint32_t h0 = fin || !(ux & 0x7fffffu) ? ux >> 16 : 0x7fc0u;
    const float r0 = fin ? x[e] - __uint_as_float(h0 << 16) : 0.0f;  // exact: the low 16 bits
    const uint32_t h1 = __float_as_uint(r0) >> 16;
    const float r1 = r0 - __uint_as_float(h1 << 16);  // exact: at most 8 significant bits left
    const uint32_t h2 = __float_as_uint(r1) >> 16;
    const uint32_t hs[3] = {h0, h1, h2};
#pragma unroll
    for (int p = 0; p < 3; p++) h[p][e >> 1] = e & 1 ? h[p][e >> 1] | hs[p] << 16 : hs[p];
  }
}

// The activations' three bf16 parts as fragments: part p of batch rows 16 ct
// .. +15 and k 32 ks .. +31 at xp[((ks * ctt + ct) * 3 + p) * LMX_FRAG]
// (zeros past nb and past n).  One wave per (ks, ct).
__global__ __launch_bounds__(64) void k_lmx_split(const float* __restrict__ X, long ldx, int nb,
                                                  int n, int ctt, uint16_t* __restrict__ xp) {
  const int ks = blockIdx.x, ct = blockIdx.y, lane = threadIdx.x;
  const int b = ct * 16 + (lane & 15), k0 = ks * 32 + 8 * (lane >> 4);
  float x[8];
#pragma unroll
  for (int e = 0; e < 8; e++) x[e] = b < nb && k0 + e < n ? X[(size_t)b * ldx + k0 + e] : 0.0f;
  lm_u32x4 h[3];
  lm_split8(x, h);
  uint16_t* o = xp + ((size_t)ks * ctt + ct) * 3 * LMX_FRAG + lane * 8;
#pragma unroll
  for (int p = 0; p < 3; p++)
    *reinterpret_cast<lm_u32x4*>(o + p * LMX_FRAG) = h[p];
}

// 16 bytes per lane from base + off to LDS at byte address lds + 16 lane.
// (Written as asm because for the builtin the compiler orders every later
// LDS read of the workgroup behind all such loads; the stage loop below
// waits for exactly the loads that it needs.  M0, the LDS base, is a clobber:
// a value that the compiler keeps there is not taken for one that survived.)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // (M0 is a reserved register)
template <bool NT>
__device__ __forceinline__ void lm_lds_load16(const void* base, uint32_t off, uint32_t lds) {
  if (NT)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt"
                 :
                 : "s"(lds), "v"(off), "s"(base)
                 : "m0", "memory");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds), "v"(off), "s"(base)
                 : "m0", "memory");
}
#pragma clang diagnostic pop
// At most N of this wave's vector memory operations, and none of its LDS
// operations, still outstanding.
template <int N>
__device__ __forceinline__ void lm_wait() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(N) : "memory");
}

template <int WR, int WC, int TR, int TC, int KS, int NS, int MODE, bool NT>
__global__ __launch_bounds__(64 * WR * WC) __attribute__((amdgpu_waves_per_eu(NS ? 2 : 4, 8))) void
k_lmhead_mfma(const uint16_t* __restrict__ W, int V, int n, const uint16_t* __restrict__ xp,
              int ctt, int ncb, int nrt, const float* __restrict__ X, long ldx, int nb,
              float* __restrict__ logits, long ld, unsigned long long* __restrict__ keys,
              int kstride, uint8_t* __restrict__ nan0) {
  constexpr int NW = WR * WC;                    // waves
  constexpr int RF = WR * TR, CF = WC * TC;      // 16-row and 16-batch-row tiles
  constexpr int WI = RF * KS, XF = CF * 3 * KS;  // 1 KiB loads of a stage: weights, parts
  constexpr int WPW = WI / NW, XPW = (XF + NW - 1) / NW, PER = WPW + XPW;  // of a wave
  constexpr int STG = (WI + XF) * LMX_FRAG;
  static_assert(NS == 0 || (WI % NW == 0 && (KS == 1 || KS == 2) && NS >= 2), "");
  static_assert(TR % WC == 0 || WC % TR == 0, "");
  constexpr int SH = NS ? NS * STG : XF * LMX_FRAG;
  static_assert((size_t)SH * 2 >= NW * CF * 16 * 8, "the epilogue's keys reuse the ring");
  __shared__ __align__(16) uint16_t sh[SH];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 15, g = lane >> 4;
  const int wr = w % WR, wc = w / WR;
  // row tile rt and batch block cb: the batch blocks of a tile on one XCD
  // (workgroups go to the eight XCDs in turn), one after the other
  const int slot = blockIdx.x >> 3;
  const int rt = (slot / ncb) * 8 + (blockIdx.x & 7), cb = slot % ncb;
  if (rt >= nrt) return;
  const int row0 = rt * RF * 16;
  lm_f32x4 acc[TR][TC];
#pragma unroll
  for (int t = 0; t < TR; t++)
#pragma unroll
    for (int j = 0; j < TC; j++) acc[t][j] = lm_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // largest |weight| bits seen, two halves; the waves that share rows take
  // their tiles in turn
  lm_u16x2 wmax = {0, 0};
  if constexpr (NS == 0) {
    // no workspace: the workgroup makes its batch rows' parts itself, KS
    // k-steps at a time (in LDS as fragments, one per wave), W straight into
    // registers
    static_assert(NS > 0 || (WC == 1 && KS * CF <= NW), "");
    constexpr int KC = 32 * KS;
    const uint16_t* wp[TR];
#pragma unroll
    for (int t = 0; t < TR; t++) {
      const int r = row0 + (wr * TR + t) * 16 + m;
      wp[t] = W + (size_t)(r < V ? r : V - 1) * n;  // rows past V: a valid row, result unused
    }
    const int xb = (cb * CF + w % CF) * 16 + m, xk = (w / CF) * 32 + 8 * g;
    float xv[8];
    auto xload = [&](int k0) {  // (zeros past n, a multiple of 8, and past nb)
#pragma unroll
      for (int e = 0; e < 8; e++) xv[e] = 0.0f;
      if (w < KS * CF && xb < nb && k0 + xk < n) {
        const float* xr = X + (size_t)xb * ldx + k0 + xk;
        const pz_f4u u = *reinterpret_cast<const pz_f4u*>(xr);
        const pz_f4u v = *reinterpret_cast<const pz_f4u*>(xr + 4);
#pragma unroll
        for (int e = 0; e < 4; e++) {
          xv[e] = u[e];
          xv[e + 4] = v[e];
        }
      }
    };
    auto xstore = [&]() {
      if (w >= KS * CF) return;
      lm_u32x4 h[3];
      lm_split8(xv, h);
#pragma unroll
      for (int p = 0; p < 3; p++)
        *reinterpret_cast<lm_u32x4*>(sh + (w * 3 + p) * LMX_FRAG + lane * 8) = h[p];
    };
    auto wload = [&](lm_u32x4 (&a)[TR][KS], int k0) {
#pragma unroll
      for (int t = 0; t < TR; t++)
#pragma unroll
        for (int q = 0; q < KS; q++) {
          const int k = k0 + 32 * q + 8 * g;
          a[t][q] = lm_u32x4{0u, 0u, 0u, 0u};
          if (k < n) a[t][q] = *reinterpret_cast<const lm_u32x4*>(wp[t] + k);
        }
    };
    auto mma = [&](const lm_u32x4 (&a)[TR][KS]) {
#pragma unroll
      for (int q = 0; q < KS; q++) {
        lm_bf16x8 b[3][TC];
#pragma unroll
        for (int p = 0; p < 3; p++)
#pragma unroll
          for (int j = 0; j < TC; j++)
            b[p][j] = *reinterpret_cast<const lm_bf16x8*>(
                sh + ((q * CF + j) * 3 + p) * LMX_FRAG + lane * 8);
#pragma unroll
        for (int t = 0; t < TR; t++) {
#pragma unroll
          for (int e = 0; e < 4; e++)
            wmax = __builtin_elementwise_max(
                wmax, __builtin_bit_cast(lm_u16x2, a[t][q][e] & 0x7fff7fffu));
#pragma unroll
          for (int j = 0; j < TC; j++)
#pragma unroll
            for (int p = 2; p >= 0; p--)
              acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  __builtin_bit_cast(lm_bf16x8, a[t][q]), b[p][j], acc[t][j], 0, 0, 0);
        }
      }
    };
    // every load of a chunk in flight at once; several workgroups per CU
    // cover the waits
    for (int k0 = 0; k0 < n; k0 += KC) {
      lm_u32x4 a[TR][KS];
      xload(k0);
      wload(a, k0);
      __syncthreads();  // the chunk before is done with the LDS
      xstore();
      __syncthreads();
      mma(a);
    }
  } else {
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint16_t*)sh;
    const uint16_t* wbase = W + (size_t)row0 * n;
    const int nst = (n + 32 * KS - 1) / (32 * KS);
    // this wave's loads of W: row and 16-byte piece per lane.  Rows past V read
    // row V - 1 (values unused); pieces past n read the row's last piece, which
    // meets zero parts (and is non-finite only in a row flagged anyway).
    uint32_t woff[WPW];
    const int piece = KS == 1 ? g : (lane & 7) ^ (lane >> 3);
#pragma unroll
    for (int i = 0; i < WPW; i++) {
      const int q = w * WPW + i;
      const int r = KS == 1 ? q * 16 + m : q * 8 + (lane >> 3);
      const int last = V - 1 - row0;
      woff[i] = ((uint32_t)(r < last ? r : last) * (uint32_t)n + 8u * piece) * 2u;
    }
    const int klast = (nst - 1) * 32 * KS + 8 * piece;
    const uint32_t wadj = klast < n ? 0u : (uint32_t)(klast - (n - 8)) * 2u;
    const uint32_t xoff = (uint32_t)lane * 16u;
    auto issue = [&](int c, int buf, int i) {  // load i of stage c into ring slot buf
      const uint32_t l0 = lds0 + (uint32_t)buf * STG * 2;
      if (i < WPW) {
        const uint32_t off = woff[i] - (c == nst - 1 ? wadj : 0u), to = l0 + (w * WPW + i) * 1024;
        lm_lds_load16<NT>(wbase + c * 32 * KS, off, to);
      } else {
        int q = w * XPW + i - WPW;
        if (XF % NW) q = q < XF ? q : XF - 1;  // (the same bytes to the same place again)
        const int s = q / (CF * 3), e = q - s * CF * 3;
        lm_lds_load16<false>(xp + (((size_t)(c * KS + s) * ctt + cb * CF) * 3 + e) * LMX_FRAG, xoff,
                      l0 + (WI + q) * 1024);
      }
    };
#pragma unroll
    for (int i = 0; i < NS - 1; i++)
#pragma unroll
      for (int q = 0; q < PER; q++) issue(i < nst ? i : nst - 1, i, q);
    int buf = 0, nbuf = NS - 1;
#pragma clang loop unroll(disable)
    for (int c = 0; c < nst; c++) {
      // stage c has arrived (the NS - 2 after it may be on their way), in every
      // wave; and every wave is done reading the slot that is filled next
      lm_wait<(NS - 2) * PER>();
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      const uint16_t* sw = sh + buf * STG;
      const uint16_t* sx = sw + WI * LMX_FRAG;
      const int cn = c + NS - 1 < nst ? c + NS - 1 : nst - 1;  // (past the end: reloaded, unused)
#pragma unroll
      for (int s = 0; s < KS; s++) {
        lm_bf16x8 a[TR], b[3][TC];
        const uint16_t* sxs = sx + (s * CF + wc * TC) * 3 * LMX_FRAG + lane * 8;
#pragma unroll
        for (int j = 0; j < TC; j++)
          b[2][j] = *reinterpret_cast<const lm_bf16x8*>(sxs + (j * 3 + 2) * LMX_FRAG);
#pragma unroll
        for (int t = 0; t < TR; t++)
          a[t] = *reinterpret_cast<const lm_bf16x8*>(
              KS == 1 ? sw + (wr * TR + t) * LMX_FRAG + lane * 8
                      : sw + (wr * TR + t) * 2 * LMX_FRAG + m * 64 + ((s * 4 + g) ^ (m & 7)) * 8);
#pragma unroll
        for (int p = 1; p >= 0; p--)
#pragma unroll
          for (int j = 0; j < TC; j++)
            b[p][j] = *reinterpret_cast<const lm_bf16x8*>(sxs + (j * 3 + p) * LMX_FRAG);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int p = 2; p >= 0; p--)
#pragma unroll
          for (int j = 0; j < TC; j++)
#pragma unroll
            for (int t = 0; t < TR; t++) {
              acc[t][j] =
                  __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], b[p][j], acc[t][j], 0, 0, 0);
              // the next stage's loads, one every few MFMAs of the first k-step
              constexpr int SP = 3 * TR * TC / PER >= 4 ? 4 : 3 * TR * TC / PER;
              static_assert(SP >= 1, "");
              const int q = ((2 - p) * TC + j) * TR + t;
              if (s == 0 && q % SP == SP - 1 && q / SP < PER) {
                issue(cn, nbuf, q / SP);
                __builtin_amdgcn_sched_barrier(0);
              }
            }
#pragma unroll
        for (int t = 0; t < TR; t++)
          if (WC == 1 || t % WC == wc % TR) {
            const lm_u32x4 q = __builtin_bit_cast(lm_u32x4, a[t]);
#pragma unroll
            for (int e = 0; e < 4; e++)
              wmax = __builtin_elementwise_max(wmax,
                                               __builtin_bit_cast(lm_u16x2, q[e] & 0x7fff7fffu));
          }
      }
      asm volatile("" ::: "memory");
      buf = buf + 1 == NS ? 0 : buf + 1;
      nbuf = nbuf + 1 == NS ? 0 : nbuf + 1;
    }
    lm_wait<0>();
  }
  __syncthreads();  // the ring is free
  // an infinite or NaN weight anywhere in the workgroup's rows: those rows
  // again with fp32 fused multiply-adds over k (lanes), into the lanes that
  // hold them (rare: a loop per row)
  int* flag = reinterpret_cast<int*>(sh);
  if (tid == 0) *flag = 0;
  __syncthreads();
  if (__ballot(wmax[0] >= 0x7f80u || wmax[1] >= 0x7f80u) && lane == 0) atomicOr(flag, 1);
  __syncthreads();
  const bool fix = *flag != 0;
  __syncthreads();
  if (fix) {
#pragma unroll
    for (int t = 0; t < TR; t++)
      for (int r16 = 0; r16 < 16; r16++) {
        const int row = row0 + (wr * TR + t) * 16 + r16;
        if (row >= V) break;
        const uint16_t* wrow = W + (size_t)row * n;
        bool nf = false;
        for (int k = lane; k < n; k += 64) nf |= (wrow[k] & 0x7f80u) == 0x7f80u;
        if (!__ballot(nf)) continue;
        for (int bl = 0; bl < 16 * TC; bl++) {
          const int b = (cb * CF + wc * TC) * 16 + bl;
          if (b >= nb) break;
          float d = 0.0f;
          for (int k = lane; k < n; k += 64)
            d = __builtin_fmaf(lm_bf16_f(wrow[k]), X[(size_t)b * ldx + k], d);
          d = pz_wave_sum(d);
          if (g == (r16 >> 2) && m == (bl & 15))
#pragma unroll
            for (int j = 0; j < TC; j++)
              if (j == (bl >> 4))
#pragma unroll
                for (int i = 0; i < 4; i++)
                  if (i == (r16 & 3)) acc[t][j][i] = d;
        }
      }
  }
  // epilogue: lane l holds batch row l % 16 of each tile, rows 4 (l / 16) + i
  if (MODE == 0) {
    const bool vec = (ld & 3) == 0 && ((uintptr_t)logits & 15) == 0;
#pragma unroll
    for (int j = 0; j < TC; j++) {
      const int b = (cb * CF + wc * TC + j) * 16 + m;
      if (b >= nb) continue;
#pragma unroll
      for (int t = 0; t < TR; t++) {
        const int row = row0 + (wr * TR + t) * 16 + 4 * g;
        float* o = logits + (size_t)b * ld + row;
        if (vec && row + 3 < V) {
          *reinterpret_cast<lm_f32x4*>(o) = acc[t][j];
        } else {
#pragma unroll
          for (int i = 0; i < 4; i++)
            if (row + i < V) o[i] = acc[t][j][i];
        }
      }
    }
  } else {
    unsigned long long* best_sh = reinterpret_cast<unsigned long long*>(sh);  // [WR][CF * 16]
#pragma unroll
    for (int j = 0; j < TC; j++) {
      const int bl = (wc * TC + j) * 16 + m, b = cb * CF * 16 + bl;
      unsigned long long best = 0ull;
#pragma unroll
      for (int t = 0; t < TR; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int row = row0 + (wr * TR + t) * 16 + 4 * g + i;
          const float v = acc[t][j][i];
          if (row < V) {
            if (row == 0 && b < nb) nan0[b] = v != v ? 1 : 0;
            if (!(v != v)) {
              const unsigned long long kk = argmax_key(v, row);
              best = kk > best ? kk : best;
            }
          }
        }
      // the maximum over the four lane groups, then over the row waves
#pragma unroll
      for (int off = 16; off < 64; off <<= 1) {
        const unsigned long long o = __shfl_xor(best, off, 64);
        best = o > best ? o : best;
      }
      if (g == 0) best_sh[wr * CF * 16 + bl] = best;
    }
    __syncthreads();
    for (int bl = tid; bl < CF * 16; bl += 64 * NW) {
      const int b = cb * CF * 16 + bl;
      if (b >= nb) break;
      unsigned long long mx = best_sh[bl];
#pragma unroll
      for (int i = 1; i < WR; i++) {
        const unsigned long long o = best_sh[i * CF * 16 + bl];
        mx = o > mx ? o : mx;
      }
      if (mx) atomicMax(&keys[(size_t)(blockIdx.x % LMM_SLOTS) * kstride + b], mx);
    }
  }
}

template <int WR, int WC, int TR, int TC, int KS, int NS, int MODE>
int launch_mfma(pz_sampler* s, const uint16_t* d_w, int V, int n, const float* x, long ldx,
                int nb, float* out, long ld, unsigned long long* keys, uint8_t* nan0) {
  constexpr int rows = WR * TR * 16, cols = WC * TC * 16;
  const int ncb = (nb + cols - 1) / cols, nrt = (V + rows - 1) / rows;
  const unsigned grid = (unsigned)((nrt + 7) / 8 * 8) * ncb;
  if constexpr (NS == 0) {
    hipLaunchKernelGGL((k_lmhead_mfma<WR, WC, TR, TC, KS, NS, MODE, false>), dim3(grid),
                       dim3(64 * WR * WC), 0, s->stream, d_w, V, n, nullptr, 0, ncb, nrt, x, ldx,
                       nb, out, ld, keys, s->max_batch, nan0);
  } else {
    const int ctt = ncb * cols / 16, ksteps = (n + 63) / 64 * 2;
    hipLaunchKernelGGL(k_lmx_split, dim3(ksteps, ctt), dim3(64), 0, s->stream, x, ldx, nb, n, ctt,
                       s->d_lmh_x);
    PZ_HIP(s, hipGetLastError());
    // (the 256-row tile is bound by the matrix cores: plain loads)
    auto k = lm_once(V, n) && cols <= 128
                 ? k_lmhead_mfma<WR, WC, TR, TC, KS, NS, MODE, (cols <= 128)>
                 : k_lmhead_mfma<WR, WC, TR, TC, KS, NS, MODE, false>;
    hipLaunchKernelGGL(k, dim3(grid), dim3(64 * WR * WC), 0, s->stream, d_w, V, n, s->d_lmh_x,
                       ctt, ncb, nrt, x, ldx, nb, out, ld, keys, s->max_batch, nan0);
  }
  PZ_HIP(s, hipGetLastError());
  return PZ_OK;
}

// Keys to ids (argmax.c:3-13); clears the keys for the next call.  The
// matrix-core kernel spreads each row's key over LMM_SLOTS slots (stride
// kstride); the others use slot 0 only (the rest stay zero).
__global__ void k_lmhead_finish(int B, unsigned long long* keys, int kstride, const uint8_t* nan0,
                                int32_t* ids) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= B) return;
  unsigned long long k = 0ull;
  for (int sl = 0; sl < LMM_SLOTS; sl++) {
    const unsigned long long o = keys[(size_t)sl * kstride + b];
    k = o > k ? o : k;
    if (sl) keys[(size_t)sl * kstride + b] = 0ull;
  }
  // logit 0 NaN: argmax.c returns 0; no key at all means every logit was NaN,
  // logit 0 among them
  ids[b] = nan0[b] || !k ? 0 : (int32_t)(0xffffffffu - (uint32_t)(k & 0xffffffffull));
  keys[b] = 0ull;
}

// LDS of the vector kernel: bt activation rows of n rounded up to 512.
size_t lm_x_bytes(int bt, int n) { return (size_t)bt * ((n + 511) / 512) * 512 * sizeof(float); }

template <int BT, int MODE>
int launch_tile(pz_sampler* s, const uint16_t* d_w, int V, int n, const float* x, long ldx, int nb,
                float* out, long ld, unsigned long long* keys, uint8_t* nan0) {
  const bool vec = n % 8 == 0 && ((uintptr_t)d_w & 15) == 0;
  auto k = !vec ? k_lmhead<BT, MODE, false, false>
                : (lm_once(V, n) ? k_lmhead<BT, MODE, true, true> : k_lmhead<BT, MODE, true, false>);
  const size_t lds = lm_x_bytes(BT, n);
  if (lds > 65536)
    PZ_HIP(s, hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)lds));
  const int grid = (V + LM_ROWS - 1) / LM_ROWS;
  hipLaunchKernelGGL(k, dim3(grid), dim3(64 * LM_WAVES), lds, s->stream, d_w, V, n, x, ldx, nb,
                     out, ld, keys, nan0);
  PZ_HIP(s, hipGetLastError());
  return PZ_OK;
}

// Batch tile: the smallest of 1, 2, 4, 8 that holds B rows (so three rows are
// one read of W, not two), or the largest whose x tile fits the LDS budget
// (0: n too large even for one row).
int tile_for(int B, int n) {
  int bt = B <= 1 ? 1 : (B <= 2 ? 2 : (B <= 4 ? 4 : 8));
  while (bt >= 1 && lm_x_bytes(bt, n) > LM_LDS_MAX) bt >>= 1;
  return bt;
}

template <int MODE>
int run(pz_sampler* s, const uint16_t* d_w, int V, int n, const float* d_x, int B, long ldx,
        float* d_logits, long ld) {
  // batch 4 and up: the matrix cores, W 16-byte aligned with rows of a
  // multiple of 8 weights; as many batch rows at a time as the parts'
  // workspace holds (PZ_LMX_ROWS rows of n = 8192, 16 of n = 131072), at most
  // PZ_LMX_ROWS; longer rows without it, since a call that only queues work
  // neither allocates nor waits
  if (B >= 4 && n % 8 == 0 && ((uintptr_t)d_w & 15) == 0) {
    const size_t fit = s->lmh_x_elems / ((size_t)((n + 63) / 64) * 64 * 3) / 16 * 16;
    if (fit == 0 || lm_own_parts(V, n, B, s->n_cu))
      return B <= 16 ? launch_mfma<8, 1, 2, 1, 2, 0, MODE>(s, d_w, V, n, d_x, ldx, B, d_logits, ld,
                                                           s->d_lmh_keys, s->d_lmh_nan)
                     : launch_mfma<8, 1, 2, 2, 2, 0, MODE>(s, d_w, V, n, d_x, ldx, B, d_logits, ld,
                                                           s->d_lmh_keys, s->d_lmh_nan);
    const int most = fit < (size_t)PZ_LMX_ROWS ? (int)fit : PZ_LMX_ROWS;
    for (int b0 = 0; b0 < B; b0 += most) {
      const int nb = B - b0 < most ? B - b0 : most;
      const float* x = d_x + (size_t)b0 * ldx;
      float* out = MODE == 0 ? d_logits + (size_t)b0 * ld : nullptr;
      unsigned long long* keys = s->d_lmh_keys + b0;
      uint8_t* nan0 = s->d_lmh_nan + b0;
      int r;
      switch (lm_tile_for(V, nb, most, s->n_cu)) {
#define PZ_LM_CASE(I, ...) \
  case I: r = launch_mfma<__VA_ARGS__, MODE>(s, d_w, V, n, x, ldx, nb, out, ld, keys, nan0); break
        PZ_LM_CASE(0, 2, 4, 8, 4, 1, 2);
        PZ_LM_CASE(1, 4, 2, 4, 4, 2, 2);
        PZ_LM_CASE(2, 4, 2, 4, 2, 2, 2);
        PZ_LM_CASE(3, 8, 1, 2, 2, 2, 3);
        default: r = launch_mfma<8, 1, 2, 1, 2, 4, MODE>(s, d_w, V, n, x, ldx, nb, out, ld, keys, nan0);
#undef PZ_LM_CASE
      }
      if (r != PZ_OK) return r;
    }
    return PZ_OK;
  }
  const int bt = tile_for(B, n);
  if (!bt) return fail(s, PZ_ENOTSUP, "n=%d: the activation row does not fit in LDS", n);
  for (int b0 = 0; b0 < B; b0 += bt) {
    const int nb = B - b0 < bt ? B - b0 : bt;
    const float* x = d_x + (size_t)b0 * ldx;
    float* out = MODE == 0 ? d_logits + (size_t)b0 * ld : nullptr;
    unsigned long long* keys = s->d_lmh_keys + b0;
    uint8_t* nan0 = s->d_lmh_nan + b0;
    int rc;
    switch (bt) {
      case 8: rc = launch_tile<8, MODE>(s, d_w, V, n, x, ldx, nb, out, ld, keys, nan0); break;
      case 4: rc = launch_tile<4, MODE>(s, d_w, V, n, x, ldx, nb, out, ld, keys, nan0); break;
      case 2: rc = launch_tile<2, MODE>(s, d_w, V, n, x, ldx, nb, out, ld, keys, nan0); break;
      default: rc = launch_tile<1, MODE>(s, d_w, V, n, x, ldx, nb, out, ld, keys, nan0); break;
    }
    if (rc != PZ_OK) return rc;
  }
  return PZ_OK;
}

int check(pz_sampler* s, const uint16_t* d_w, int V, int n, const float* d_x, int B, long ldx) {
  if (!d_w || !d_x || V <= 0 || n <= 0 || B < 0 || ldx < n)
    return fail(s, PZ_EINVAL, "bad LM head shape");
  if (B > s->max_batch) return fail(s, PZ_ERANGE, "B=%d > max_batch=%d", B, s->max_batch);
  return PZ_OK;
}

}  // namespace

extern "C" int pz_lm_head_bf16(pz_sampler* s, const uint16_t* d_w, int V, int n, const float* d_x,
                               int B, long ldx, float* d_logits, long ld) {
  if (!s) return PZ_EINVAL;
  const int rc = check(s, d_w, V, n, d_x, B, ldx);
  if (rc != PZ_OK) return rc;
  if (!d_logits || ld < V) return fail(s, PZ_EINVAL, "bad logits buffer");
  if (B == 0) return PZ_OK;
  PZ_HIP(s, hipSetDevice(s->device));
  return run<0>(s, d_w, V, n, d_x, B, ldx, d_logits, ld);
}

extern "C" int pz_lm_head_argmax_bf16(pz_sampler* s, const uint16_t* d_w, int V, int n,
                                      const float* d_x, int B, long ldx, int32_t* d_ids) {
  if (!s) return PZ_EINVAL;
  const int rc = check(s, d_w, V, n, d_x, B, ldx);
  if (rc != PZ_OK) return rc;
  if (!d_ids) return fail(s, PZ_EINVAL, "null ids");
  if (B == 0) return PZ_OK;
  PZ_HIP(s, hipSetDevice(s->device));
  const int r = run<1>(s, d_w, V, n, d_x, B, ldx, nullptr, 0);
  if (r != PZ_OK) return r;
  hipLaunchKernelGGL(k_lmhead_finish, dim3((B + 255) / 256), dim3(256), 0, s->stream, B,
                     s->d_lmh_keys, s->max_batch, s->d_lmh_nan, d_ids);
  PZ_HIP(s, hipGetLastError());
  return PZ_OK;
}
