// pz_softmax.hip -- batched apply_temperature and softmax on device rows,
// bit-exact with the reference.
//
//   apply_temperature (src/sampling/temperature.c:8-25): T < 1e-6 -> 1e-6,
//     x *= 1/T (AVX-512 build) or x /= T (scalar build), in place.
//   softmax (src/math/softmax.c:4-23, the tn_softmax slot of
//     include/math/simd_dispatch.h:23,47): max by strict '>', e = expf(x -
//     max) with a sequential fp32 sum in ascending order, x *= 1/sum.  Any
//     NaN, or an infinite maximum, makes the sum NaN and every output NaN.
// Rows of more than SM_SPLIT_MIN entries are split over workgroups (k_sm_*,
// below); shorter ones, and rows the workspace does not hold, run one
// 1024-thread workgroup per row: pass 1 (max), the exact-sum records and walk
// (pz_rowpass.h), then one write pass.  Rows may have their own lengths
// (attention scores, pz_attn.hip).
#include "pz_device.h"
#include "pz_exact.h"
#include "pz_launch.h"
#include "pz_rowpass.h"
#include "pz_sampler_impl.h"
#include "pz_split.h"

namespace {

__global__ void k_temperature(float* __restrict__ x, long ld, int V, int B, PzTemp T) {
  const long n = (long)B * V;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n;
       i += (long)gridDim.x * blockDim.x) {
    const long r = i / V, c = i - r * V;
    float* p = x + r * ld + c;
    *p = T.apply(*p);
  }
}

struct SoftmaxShared {
  PzPass1Shared p1;
  PzRecShared r;
};

template <bool VEC>
__global__ __launch_bounds__(PZ_RB) void k_softmax(const float* in, long ld_in, float* out,
                                                   long ld_out, int Vmax, PzTemp T,
                                                   const int32_t* lens) {
  extern __shared__ __align__(16) char lds[];
  __shared__ SoftmaxShared S;
  __shared__ uint64_t etab[32];
  const pz_lds_u64* et = (const pz_lds_u64*)etab;
  pz_etab_fill((pz_lds_u64*)etab);  // ordered by pz_pass1's barriers
  const int row = blockIdx.x, tid = threadIdx.x;
  // the row's length: every thread reads the same value, so the early return
  // below is uniform over the workgroup
  const int V = lens ? (lens[row] < Vmax ? lens[row] : Vmax) : Vmax;
  if (V <= 0) return;
  PzTempRow<VEC> R;
  R.x = in + (long)row * ld_in;
  R.V = V;
  R.T = T;
  const int ntiles = pz_tiles(V);
  const PzRec REC = pz_rec_at(lds, ntiles * PZ_SEGS_PER_TILE);
  float* o = out + (long)row * ld_out;

  const float M = pz_pass1<8>(R, ntiles, S.p1);
  if (S.p1.any_nan || !(M > -__builtin_inff() && M < __builtin_inff())) {
    for (int i = tid; i < V; i += PZ_RB) o[i] = __builtin_nanf("");
    return;
  }
  PzExpTerms<PzTempRow<VEC>> X;
  X.R = R;
  X.M = M;
  X.thr = -__builtin_inff();
  X.inv = 1.0f;
  X.as_p = false;
  X.et = et;
  const float inv = 1.0f / pz_exact_sum(X, ntiles, REC, S.r);
  // every read of the row is done: the write pass may overwrite it (in == out)
  for (int t = 0; t < ntiles; t++) {
    float y[4];
    const int e0 = pz_tile_e0(t);
    const int n = R.get(e0, y);
#pragma unroll
    for (int c = 0; c < 4; c++)
      if (c < n) o[e0 + c] = pz_expf_tab(y[c] - M, et) * inv;
  }
}

// ---- rows split over workgroups -------------------------------------------------
// The row-split passes of pz_split.h over the rows' own lengths -- slice
// maxima and segment estimates (k_sm_stat), the integer increment records at
// the predicted grids (k_sm_rec), one workgroup per row for the exact sum
// (k_sm_walk), then every probability (k_sm_write) -- so the per-element work
// runs on every CU rather than one workgroup per row.  Each pass reads the
// row again (L2 / Infinity Cache).
// Shorter rows (pz_softmax_batch) take one workgroup each: four launches cost
// more than they spread (one workgroup / split, B = 64, T 0.7: V = 3000 22.0 /
// 23.4 us, 5000 26.3 / 24.8, 8192 28.2 / 24.9, 32768 56 / 35, 128256 146 /
// 55; B = 256: 5000 29 / 30, 8192 39 / 33, 128256 153 / 127; B = 1024 at
// 128256 601 / 528).
constexpr int SM_SPLIT_MIN = 6144;

struct SmSplit {
  const float* in;
  long ld_in;
  float* out;
  long ld_out;
  int n;
  PzTemp T;
  const int32_t* lens;
  PzSplitWs ws;
  int nseg, spw, S, nc;
};

__device__ __forceinline__ int sm_len(const SmSplit& A, int row) {
  const int len = A.lens ? A.lens[row] : A.n;
  return len < A.n ? len : A.n;  // (<= 0: the row is left alone)
}

template <bool VI>
__device__ __forceinline__ PzTempRow<VI> sm_row(const SmSplit& A, int row, int len) {
  PzTempRow<VI> R;
  R.x = A.in + (size_t)row * A.ld_in;
  R.V = len;
  R.T = A.T;
  return R;
}

__device__ __forceinline__ bool sm_bad(uint32_t flags) {
  return (flags & (PZ_RS_NAN | PZ_RS_NONFIN)) != 0;  // softmax.c:6-9: NaN everywhere
}

template <bool VI>
__global__ __launch_bounds__(PZ_SP_BLOCK) PZ_SP_TWO_PER_CU void k_sm_stat(SmSplit A) {
  __shared__ PzSpShared SS;
  const int row = blockIdx.y, len = sm_len(A, row);
  if (len <= 0) return;
  if (threadIdx.x == 0) SS.any = 0u;
  __syncthreads();
  pz_sp_stat_slice(sm_row<VI>(A, row, len), row, pz_sp_slice(A.nseg, A.spw), A.ws, SS, true);
}

template <bool VI>
__global__ __launch_bounds__(PZ_SP_BLOCK) PZ_SP_TWO_PER_CU void k_sm_rec(SmSplit A) {
  __shared__ PzSpShared SS;
  __shared__ uint64_t etab[32];
  pz_etab_fill((pz_lds_u64*)etab);
  const int row = blockIdx.y, len = sm_len(A, row);
  if (len <= 0) return;
  pz_sp_row_stat(row, A.S, A.ws, SS);
  if (sm_bad(SS.any)) return;
  const PzSlice sl = pz_sp_slice(A.nseg, A.spw);
  const PzEstRel est{A.ws.seg_m + (size_t)row * A.ws.nsc, A.ws.seg_s + (size_t)row * A.ws.nsc,
                     SS.M};
  const float carry = pz_sp_prefix(est, sl.k0, SS);
  pz_sp_predict(est, carry, row, sl, A.ws, SS);
  PzExpTerms<PzTempRow<VI>> X;
  X.R = sm_row<VI>(A, row, len);
  X.M = SS.M;
  X.thr = -__builtin_inff();
  X.inv = 1.0f;
  X.as_p = false;
  X.et = (const pz_lds_u64*)etab;
  pz_sp_records(X, row, sl, A.ws, nullptr, true);
  if (sl.k0 == 0 && threadIdx.x < 64) {
    // the row's first segment summed from zero (the DPP chain of real adds),
    // for the walk to start from instead of waiting for a producer
    float v[4];
    X.seg(0, v);
    PzAcc z;
    z.n = 0u;
    z.g = 1u;
    pz_sp_chain<PZ_STOP_NONE>(z, v, 0.0f);
    if (threadIdx.x == 0) A.ws.rs[row].s0 = __float_as_uint(pz_acc_value(z));
  }
}

// One workgroup per row: wave 0 walks, waves 1..15 pre-evaluate its specials.
template <bool VI>
__global__ __launch_bounds__(PZ_SP_BLOCK) void k_sm_walk(SmSplit A) {
  extern __shared__ __align__(16) char lds[];
  __shared__ PzSpShared SS;
  __shared__ uint64_t etab[32];
  __shared__ float sum_sh;
  pz_etab_fill((pz_lds_u64*)etab);
  const int row = blockIdx.x, len = sm_len(A, row);
  if (len <= 0) return;
  const PzRecAhead ra = pz_sp_rec_ahead(A.ws, row, A.nseg);  // in flight beside the maxima
  const uint32_t s0 = A.ws.rs[row].s0;  // segment 0's sum (k_sm_rec)
  pz_sp_row_stat(row, A.S, A.ws, SS);
  PzRowState& rs = A.ws.rs[row];
  if (sm_bad(SS.any)) {
    if (threadIdx.x == 0) {
      rs.M = SS.M;
      rs.flags = SS.any;
    }
    return;
  }
  PzExpTerms<PzTempRow<VI>> X;
  X.R = sm_row<VI>(A, row, len);
  X.M = SS.M;
  X.thr = -__builtin_inff();
  X.inv = 1.0f;
  X.as_p = false;
  X.et = (const pz_lds_u64*)etab;
  const PzWalk W = pz_sp_walk_setup(X, row, A.nseg, A.nc, A.ws, lds, SS, -1, s0, &ra);
  if (threadIdx.x < 64) {
    PzAcc st;
    pz_sp_walk<PZ_STOP_NONE>(st, W, 0.0f, X);
    if (threadIdx.x == 0) sum_sh = pz_acc_value(st);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    rs.M = SS.M;
    rs.flags = SS.any;
    rs.sum = sum_sh;
    rs.inv = 1.0f / sum_sh;  // softmax.c:19-22
  }
}

// p = e * (1 / sum) for every score of the slice (NaN on degenerate rows).
template <bool VI>
__global__ __launch_bounds__(PZ_SP_BLOCK) PZ_SP_TWO_PER_CU void k_sm_write(SmSplit A) {
  __shared__ uint64_t etab[32];
  pz_etab_fill((pz_lds_u64*)etab);
  const int row = blockIdx.y, len = sm_len(A, row);
  if (len <= 0) return;
  const PzRowState rs = A.ws.rs[row];
  const bool bad = sm_bad(rs.flags);
  PzExpTerms<PzTempRow<VI>> X;
  X.R = sm_row<VI>(A, row, len);
  X.M = rs.M;
  X.thr = -__builtin_inff();
  X.inv = 1.0f;
  X.as_p = false;
  X.et = (const pz_lds_u64*)etab;
  __syncthreads();  // the expf table
  float* o = A.out + (size_t)row * A.ld_out;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const PzSlice sl = pz_sp_slice(A.nseg, A.spw);
  for (int kb = sl.k0 + w; kb < sl.k1; kb += PZ_SP_U * PZ_SP_WAVES) {
    float y[PZ_SP_U][4];
#pragma unroll
    for (int u = 0; u < PZ_SP_U; u++)  // every load of the step in flight first
      X.R.load((kb + u * PZ_SP_WAVES) * PZ_SP_SEG + 4 * lane, y[u]);
#pragma unroll
    for (int u = 0; u < PZ_SP_U; u++) {
      const int k = kb + u * PZ_SP_WAVES, i0 = k * PZ_SP_SEG + 4 * lane;
      if (k >= sl.k1) break;
      if (i0 >= len) continue;
      X.R.apply(i0, 4, y[u]);
      float v[4];
#pragma unroll
      for (int c = 0; c < 4; c++)
        v[c] = bad ? __builtin_nanf("") : pz_expf_tab(y[u][c] - rs.M, X.et) * rs.inv;
      if (i0 + 3 < len) {
        pz_f4u q;
        q.x = v[0];
        q.y = v[1];
        q.z = v[2];
        q.w = v[3];
        *reinterpret_cast<pz_f4u*>(o + i0) = q;
      } else {
#pragma unroll
        for (int c = 0; c < 4; c++)
          if (i0 + c < len) o[i0 + c] = v[c];
      }
    }
  }
}

template <bool VI>
int launch_split_t(pz_sampler* s, const SmSplit& A, int n_rows, size_t walk_lds) {
  auto kw = k_sm_walk<VI>;
  if (walk_lds > 65536 && hipFuncSetAttribute((const void*)kw,
                                              hipFuncAttributeMaxDynamicSharedMemorySize,
                                              (int)walk_lds) != hipSuccess)
    return -1;
  const dim3 grid(A.S, n_rows), block(PZ_SP_BLOCK);
  hipLaunchKernelGGL(k_sm_stat<VI>, grid, block, 0, s->stream, A);
  hipLaunchKernelGGL(k_sm_rec<VI>, grid, block, 0, s->stream, A);
  hipLaunchKernelGGL(kw, dim3(n_rows), block, walk_lds, s->stream, A);
  hipLaunchKernelGGL(k_sm_write<VI>, grid, block, 0, s->stream, A);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

PzTemp temp_of(pz_sampler* s, float temperature) {
  float T = temperature;
  if (T < 1e-6f) T = 1e-6f;  // temperature.c:10 (a NaN temperature stays NaN)
  PzTemp t;
  t.t = T;
  t.inv = 1.0f / T;
  t.div = s->temp_mode == PZ_TEMP_DIV;
  return t;
}

}  // namespace

int pz_launch_softmax_split(pz_sampler* s, const PzSplitWs& ws, const float* d_in, long ld_in,
                            float* d_out, long ld_out, int n_rows, int n, PzTemp T,
                            const int32_t* d_len) {
  SmSplit A;
  A.in = d_in;
  A.ld_in = ld_in;
  A.out = d_out;
  A.ld_out = ld_out;
  A.n = n;
  A.T = T;
  A.lens = d_len;
  A.ws = ws;
  const PzSplitPlan pl = pz_split_plan(n, n_rows, ws.smax);
  if (pl.nseg > ws.nsc || pl.S > ws.smax || n_rows > 65535) return -2;
  A.nseg = pl.nseg;
  A.spw = pl.spw;
  A.S = pl.S;
  const size_t fixed = 4096;
  int nc = pz_sp_walk_nc(pl.nseg, (size_t)s->max_lds / 2 - fixed);
  if (nc < 12) nc = pz_sp_walk_nc(pl.nseg, (size_t)s->max_lds - fixed);
  if (nc < 2) return -2;
  A.nc = nc;
  const size_t walk_lds = pz_sp_walk_lds(pl.nseg, nc);
  const bool vi = (ld_in % 4 == 0) && (((uintptr_t)d_in & 15) == 0);
  return vi ? launch_split_t<true>(s, A, n_rows, walk_lds)
            : launch_split_t<false>(s, A, n_rows, walk_lds);
}

int pz_launch_softmax_rows(pz_sampler* s, const float* d_in, long ld_in, float* d_out,
                           long ld_out, int B, int V, PzTemp T, const int32_t* d_len) {
  const size_t lds = pz_rec_bytes(V);
  if (lds + sizeof(SoftmaxShared) + 64 > (size_t)s->max_lds)
    return fail(s, PZ_ENOTSUP, "V=%d needs more LDS than the device has", V);
  const bool vec = (ld_in % 4 == 0) && (((uintptr_t)d_in & 15) == 0);
  auto kern = vec ? k_softmax<true> : k_softmax<false>;
  if (lds > 65536)
    PZ_HIP(s, hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)lds));
  hipLaunchKernelGGL(kern, dim3(B), dim3(PZ_RB), lds, s->stream, d_in, ld_in, d_out, ld_out, V,
                     T, d_len);
  PZ_HIP(s, hipGetLastError());
  return PZ_OK;
}

extern "C" int pz_temperature_batch(pz_sampler* s, float* d_x, long ld, int B, int V,
                                    float temperature) {
  if (!s) return PZ_EINVAL;
  if (!d_x || B < 0 || V < 0 || ld < V) return fail(s, PZ_EINVAL, "bad temperature shape");
  if ((long)B * V == 0) return PZ_OK;
  PZ_HIP(s, hipSetDevice(s->device));
  const long n = (long)B * V;
  const int blocks = (int)((n + 255) / 256 < 65536 ? (n + 255) / 256 : 65536);
  hipLaunchKernelGGL(k_temperature, dim3(blocks), dim3(256), 0, s->stream, d_x, ld, V, B,
                     temp_of(s, temperature));
  PZ_HIP(s, hipGetLastError());
  return PZ_OK;
}

extern "C" int pz_softmax_batch(pz_sampler* s, const float* d_in, long ld_in, float* d_out,
                                long ld_out, int B, int V, float temperature) {
  if (!s) return PZ_EINVAL;
  if (!d_in || !d_out || B < 0 || V <= 0 || ld_in < V || ld_out < V)
    return fail(s, PZ_EINVAL, "bad softmax shape");
  if (B == 0) return PZ_OK;
  PZ_HIP(s, hipSetDevice(s->device));
  const PzTemp T = temp_of(s, temperature);
  if (V > SM_SPLIT_MIN && B <= s->max_batch && V <= s->max_vocab) {
    const int rc = pz_launch_softmax_split(s, s->ws, d_in, ld_in, d_out, ld_out, B, V, T, nullptr);
    if (rc == 0) return PZ_OK;
    if (rc != -2) return fail(s, PZ_EDEVICE, "softmax launch failed");
  }
  return pz_launch_softmax_rows(s, d_in, ld_in, d_out, ld_out, B, V, T, nullptr);
}
