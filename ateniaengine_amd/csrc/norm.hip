// RMSNorm(x) * gamma for the decoder layer's FFN block: the step that precedes the MoE layer in
// src/moe/full_forward.rs:239-243 (graph: RmsNorm node + BroadcastMul node) and in
// src/moe/mla.rs:442, src/moe/decoder_layer.rs:97-107 (imperative, f64 accumulation).
//
// The normalised rows feed the router, so the arithmetic of the reference is kept, not just its
// value:
//   policy 0 (graph, src/nn/normalization.rs:8-37): sum of squares folded left to right in f32
//     (multiply and add rounded separately), mean = sum / max(cols, 1), inv = 1 / sqrt(mean + eps),
//     y = (x * inv) * gamma with both products rounded to f32.  The fold is a dependent chain of
//     `cols` additions per row.  Two forms: rmsnorm_fold_kernel (a workgroup per row, the fold as a
//     scan that gives the same bits; rows of 256 to 8192 columns in whole eights) and, for other
//     widths and many narrow rows, rmsnorm_gamma_kernel: the whole workgroup fetches a column chunk and stores the
//     (rounded) squares in LDS, then one lane per row adds them in order while the next chunk is in
//     flight; 4 rows per workgroup.
//   policy 1 (f64): sum of squares in f64 (the squares of f32 values are exact in f64), mean and
//     inverse root in f64, y = (float)(x * inv) * gamma.  The reference adds left to right; here 64
//     lanes per row add interleaved columns and the partial sums are added in lane order.  The two
//     orders differ by at most a few units of the f64 sum's last place, which the rounding of
//     x * inv to f32 hides except for values within ~1e-9 (relative) of a rounding boundary.
// HBM-bound at large T (8 bytes of algorithmic traffic per element); at few rows it is latency.
#include "../../include/atenia_moe_hip.h"
#include "moe_internal.h"

// This file is compiled with -ffp-contract=off (see the Makefile): the reference rounds every
// product and every sum on its own, and hipcc would otherwise fuse `a * b + c` into one FMA
// (its default is -ffp-contract=fast, under which __fmul_rn / __fadd_rn are plain `*` and `+`
// and the fp-contract pragma is ignored).  sqrtf and `/` are hipcc's correctly rounded f32 forms;
// __fsqrt_rn is not.

namespace atenia_moe {

namespace {

constexpr int kRows = 4;           // rows (tokens) per workgroup: small, so several workgroups share a CU
constexpr int kChunk = 512;        // columns staged per step
constexpr int kPitch = kChunk + 4; // floats; 516 % 64 == 4: the walking lanes read disjoint banks
constexpr int kThreads = 256;
constexpr int kLanes = kThreads / kRows;  // f64 policy: lanes that share one row's sum
constexpr int kLoads = kRows * kChunk / 4 / kThreads;  // float4 per thread per chunk (2)

// Four consecutive floats of row `row` from column `col`; zero outside [0, T) x [0, d).
// VEC (d % 4 == 0, col % 4 == 0): one aligned 16-byte load from a clamped address, no branch.
template <bool VEC>
__device__ inline float4 load_x4(const float* __restrict__ x, int T, int d, int row, int col) {
  const bool ok = row < T && col < d;
  if (VEC) {
    const float4 v = *(const float4*)(x + (ok ? (size_t)row * d + col : 0));
    return ok ? v : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
  if (!ok) return v;
  const float* p = x + (size_t)row * d + col;
  v.x = p[0];
  if (col + 1 < d) v.y = p[1];
  if (col + 2 < d) v.z = p[2];
  if (col + 3 < d) v.w = p[3];
  return v;
}

template <int POLICY, bool VEC>
__global__ __launch_bounds__(kThreads) void rmsnorm_gamma_kernel(const float* __restrict__ x,
                                                                  const float* __restrict__ gamma,
                                                                  float eps, int T, int d,
                                                                  float* __restrict__ y) {
  __shared__ __attribute__((aligned(16))) float S[kRows * kPitch];
  __shared__ double part[kRows][kThreads / kRows];
  __shared__ double inv64[kRows];
  __shared__ float inv32[kRows];
  const int tid = threadIdx.x;
  const int t0 = blockIdx.x * kRows;
  const int n_chunks = (d + kChunk - 1) / kChunk;

  float4 pre[kLoads];
  auto fetch = [&](int chunk) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int flat = i * kThreads + tid;
      pre[i] = load_x4<VEC>(x, T, d, t0 + flat / (kChunk / 4), chunk * kChunk + (flat % (kChunk / 4)) * 4);
    }
  };
  auto stash = [&]() {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int flat = i * kThreads + tid;
      float4 v = pre[i];
      if (POLICY == 0) {  // the walking lane only adds: every thread squares what it fetched
        v.x = v.x * v.x; v.y = v.y * v.y; v.z = v.z * v.z; v.w = v.w * v.w;
      }
      *(float4*)&S[(flat / (kChunk / 4)) * kPitch + (flat % (kChunk / 4)) * 4] = v;
    }
  };

  float s32 = 0.f;   // policy 0: the row's running sum (lanes 0..15 of wave 0)
  double s64 = 0.0;  // policy 1: this lane's share of row tid / kLanes
  fetch(0);
  for (int chunk = 0; chunk < n_chunks; ++chunk) {
    __syncthreads();  // the previous chunk has been consumed
    stash();
    __syncthreads();
    if (chunk + 1 < n_chunks) fetch(chunk + 1);  // in flight while the sums advance
    // Columns past d are zero in LDS and add +0 to a non-negative sum: no effect on any bit.
    const int width = min(kChunk, d - chunk * kChunk);
    if (POLICY == 0) {
      if (tid < kRows) {
        // Sixteen squares are added while the next sixteen are on their way from LDS (two
        // register sets, so nothing is copied).  Columns past `width` hold zeros.
        const float* row = S + tid * kPitch;
        float4 a0 = *(const float4*)(row), a1 = *(const float4*)(row + 4),
               a2 = *(const float4*)(row + 8), a3 = *(const float4*)(row + 12);
        for (int c = 0; c < width; c += 32) {
          const float4 b0 = *(const float4*)(row + c + 16), b1 = *(const float4*)(row + c + 20),
                       b2 = *(const float4*)(row + c + 24), b3 = *(const float4*)(row + c + 28);
          __builtin_amdgcn_sched_barrier(0);
          s32 += a0.x; s32 += a0.y; s32 += a0.z; s32 += a0.w;
          s32 += a1.x; s32 += a1.y; s32 += a1.z; s32 += a1.w;
          s32 += a2.x; s32 += a2.y; s32 += a2.z; s32 += a2.w;
          s32 += a3.x; s32 += a3.y; s32 += a3.z; s32 += a3.w;
          __builtin_amdgcn_sched_barrier(0);
          const int nc = (c + 32) & (kChunk - 1);  // past the chunk: a harmless re-read of column 0
          a0 = *(const float4*)(row + nc); a1 = *(const float4*)(row + nc + 4);
          a2 = *(const float4*)(row + nc + 8); a3 = *(const float4*)(row + nc + 12);
          __builtin_amdgcn_sched_barrier(0);
          s32 += b0.x; s32 += b0.y; s32 += b0.z; s32 += b0.w;
          s32 += b1.x; s32 += b1.y; s32 += b1.z; s32 += b1.w;
          s32 += b2.x; s32 += b2.y; s32 += b2.z; s32 += b2.w;
          s32 += b3.x; s32 += b3.y; s32 += b3.z; s32 += b3.w;
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    } else {
      const float* row = S + (tid / kLanes) * kPitch;
      for (int c = tid % kLanes; c < width; c += kLanes) {
        const double v = (double)row[c];
        s64 = fma(v, v, s64);  // v * v is exact in f64, so this is the separately rounded sum
      }
    }
  }

  if (POLICY == 0) {
    if (tid < kRows) {
      const float cols = (float)d;
      const float mean = s32 / (cols > 1.0f ? cols : 1.0f);
      inv32[tid] = 1.0f / sqrtf(mean + eps);
    }
  } else {
    part[tid / kLanes][tid % kLanes] = s64;
    __syncthreads();
    if (tid < kRows) {
      double ms = 0.0;
      for (int p = 0; p < kLanes; ++p) ms += part[tid][p];
      ms /= (double)d;
      inv64[tid] = 1.0 / sqrt(ms + (double)eps);
    }
  }
  __syncthreads();

  // y = (x * inv) * gamma, every product rounded on its own.  The rows of the group are
  // independent loads of one column block, so several are in flight per thread.
  const int d4 = (d + 3) / 4;
  for (int q = tid; q < d4; q += kThreads) {
    const int c = q * 4;
    const float4 g = load_x4<VEC>(gamma, 1, d, 0, c);
    float4 v[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) v[r] = load_x4<VEC>(x, T, d, t0 + r, c);
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      if (t0 + r >= T) break;
      float4 o;
      if (POLICY == 0) {
        const float i32 = inv32[r];
        o.x = (v[r].x * i32) * g.x; o.y = (v[r].y * i32) * g.y;
        o.z = (v[r].z * i32) * g.z; o.w = (v[r].w * i32) * g.w;
      } else {
        const double i64 = inv64[r];
        o.x = (float)((double)v[r].x * i64) * g.x; o.y = (float)((double)v[r].y * i64) * g.y;
        o.z = (float)((double)v[r].z * i64) * g.z; o.w = (float)((double)v[r].w * i64) * g.w;
      }
      float* out = y + (size_t)(t0 + r) * d + c;
      if (VEC) {
        *(float4*)out = o;
      } else {
        out[0] = o.x;
        if (c + 1 < d) out[1] = o.y;
        if (c + 2 < d) out[2] = o.z;
        if (c + 3 < d) out[3] = o.w;
      }
    }
  }
}

// ---- policy 0 as a scan ----------------------------------------------------------------------
// The fold s <- RN(s + q) of squares q >= 0 rounds at each step, but while s stays in one binade
// [2^e, 2^(e+1)) it moves on the grid of u = 2^(e-23), and RN(s + q) = s + u RN(q / u), where only a
// q / u halfway between two integers looks at s at all: at the parity of s / u.  So a run of squares
// inside a binade is two numbers, the steps it adds from an even and from an odd s / u; runs compose
// (the first's result has the parity that picks the second's number), i.e. they scan; and adding n
// steps to s is adding n to its bit pattern.
//  * A thread holds eight squares.  Prefix sums in another order say which binade s is in when it gets
//    there: they are within (n + 256) 2^-24 of the fold's, relatively (the fold's own roundings
//    are n 2^-24 at most, theirs a few tens).
//  * A thread whose eight may take s across a power of two (and one that finds s = 0 or a denormal)
//    leaves its squares in a list, behind the composed run since the entry before it: some
//    log2(n) entries per row.  Where the sum is not finite every thread does.
//  * One wave walks the entries: s gets the run's steps, then the eight squares by plain addition.
// The same bits as the left-to-right fold, ties, zeros and outliers included (tests/test_gpu_block.py).
// What bounds it: a memory round trip in, the walk (some twenty entries of 0.1 us) and a trip out,
// against `cols` dependent additions of 9 clocks.  rmsnorm_gamma_kernel / this one, us: d = 2048, 48 rows
// 11.8 / 4.6, 12288 rows 50.5 / 43.2; d = 4096, 1 row 20.6 / 4.9, 16 rows 24.7 / 5.8, 400 rows 31.1 / 10.2,
// 3800 rows 42.5 / 33.8 (3.7 TB/s); d = 7168, 64 rows 38.6 / 8.1.
constexpr int kFoldCols = 8;  // per thread
constexpr int kFoldMaxCols = 1024 * kFoldCols;

struct Run {
  int flag;    // an entry of the list lies inside: d0, d1 are the run since then
  int d0, d1;  // steps added to an even and to an odd s
};
__device__ inline Run then(const Run& a, const Run& b) {
  const int c0 = a.d0 + ((a.d0 & 1) ? b.d1 : b.d0);
  const int c1 = a.d1 + ((a.d1 & 1) ? b.d0 : b.d1);
  return Run{a.flag | b.flag, b.flag ? b.d0 : c0, b.flag ? b.d1 : c1};
}
// the value of the lane CTRL names; `none` where there is no such lane or ROWS leaves the row out
template <int CTRL, int ROWS>
__device__ inline int dpp(int v, int none) {
  return __builtin_amdgcn_update_dpp(none, v, CTRL, ROWS, 0xf, false);
}
template <int CTRL, int ROWS>
__device__ inline float scan_step(float v) {
  return v + __int_as_float(dpp<CTRL, ROWS>(__float_as_int(v), 0));
}
template <int CTRL, int ROWS>
__device__ inline Run scan_step(const Run& v) {
  return then(Run{dpp<CTRL, ROWS>(v.flag, 0), dpp<CTRL, ROWS>(v.d0, 0), dpp<CTRL, ROWS>(v.d1, 0)}, v);
}
// inclusive scan over the wave: shifts by 1, 2, 4, 8 in rows of 16 lanes, then the rows' last lanes
template <typename V>
__device__ inline V wave_scan(V v) {
  v = scan_step<0x111, 0xf>(v);
  v = scan_step<0x112, 0xf>(v);
  v = scan_step<0x114, 0xf>(v);
  v = scan_step<0x118, 0xf>(v);
  v = scan_step<0x142, 0xa>(v);
  return scan_step<0x143, 0xc>(v);
}

__global__ __launch_bounds__(1024) void rmsnorm_fold_kernel(const float* __restrict__ x,
                                                             const float* __restrict__ gamma, float eps,
                                                             int d, float* __restrict__ y) {
  struct Entry {
    float4 lo, hi;  // the eight squares
    int d0, d1, pad0, pad1;
  };
  extern __shared__ Entry fold_list[];  // 65 per wave: its entries, then the run behind the last
  __shared__ float wave_sum[16], inv_shared;
  __shared__ int wave_entries[16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), n_waves = blockDim.x >> 6;
  const int col = tid * kFoldCols;
  const bool in = col < d;  // (d is a multiple of eight)
  const float4* px = (const float4*)(x + (size_t)blockIdx.x * d + (in ? col : 0));
  const float4* pg = (const float4*)(gamma + (in ? col : 0));
  const float4 xl = px[0], xh = px[1], gl = pg[0], gh = pg[1];
  const float xs[8] = {xl.x, xl.y, xl.z, xl.w, xh.x, xh.y, xh.z, xh.w};
  const float gs[8] = {gl.x, gl.y, gl.z, gl.w, gh.x, gh.y, gh.z, gh.w};
  float q[8], mine = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    q[i] = in ? xs[i] * xs[i] : 0.f;
    mine += q[i];
  }
  const float incl = wave_scan(mine);
  if (lane == 63) wave_sum[wave] = incl;
  __syncthreads();
  float before = 0.f, total = 0.f;
  for (int w = 0; w < n_waves; ++w) {
    if (w == wave) before = total;
    total += wave_sum[w];
  }
  // the sum in front of this thread's first square: the wave's scan of the lane before
  before += __int_as_float(dpp<0x138, 0xf>(__float_as_int(incl), 0));

  const float margin = (float)(blockDim.x * kFoldCols + 256) * 0x1p-24f;
  const float after = before + mine;
  const float lo = before - before * margin, hi = after + after * margin;
  const int e_lo = (int)(__float_as_uint(lo) >> 23), e_hi = (int)(__float_as_uint(hi) >> 23);
  bool listed = mine != 0.f && (e_lo != e_hi || e_lo == 0);
  if (!(total < 3e38f)) listed = true;  // an infinity, a NaN, or close to the largest number
  int v0 = 0, v1 = 1;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float s = listed ? 0.f : ldexpf(q[i], 150 - e_lo), fl = floorf(s), frac = s - fl;  // all exact
    const int whole = (int)fl;
    const bool up = frac > 0.5f, tie = frac == 0.5f;
    v0 += whole;
    v1 += whole;
    v0 += up ? 1 : tie ? v0 & 1 : 0;
    v1 += up ? 1 : tie ? v1 & 1 : 0;
  }
  const bool none = listed || mine == 0.f;
  const Run run = wave_scan(Run{listed ? 1 : 0, none ? 0 : v0, none ? 0 : v1 - 1});
  const unsigned long long entries = __ballot(listed);
  const int prev0 = dpp<0x138, 0xf>(run.d0, 0), prev1 = dpp<0x138, 0xf>(run.d1, 0);
  Entry* list = fold_list + wave * 65;
  if (listed) {
    Entry& en = list[__popcll(entries & ((1ull << lane) - 1))];
    en.lo = float4{q[0], q[1], q[2], q[3]};
    en.hi = float4{q[4], q[5], q[6], q[7]};
    en.d0 = prev0;
    en.d1 = prev1;
  }
  if (lane == 63) {
    Entry& en = list[__popcll(entries)];  // the run behind the last entry; +0 leaves s as it is
    en.lo = en.hi = float4{0.f, 0.f, 0.f, 0.f};
    en.d0 = run.d0;
    en.d1 = run.d1;
    wave_entries[wave] = __popcll(entries);
  }
  __syncthreads();
  if (wave == 0) {  // (all lanes alike)
    float s = 0.f;
    for (int w = 0; w < n_waves; ++w) {
      const Entry* at = fold_list + w * 65;
      const int n = __builtin_amdgcn_readfirstlane(wave_entries[w]);
      Entry en = at[0];
      for (int j = 0; j <= n; ++j) {
        const Entry next = at[min(j + 1, n)];
        const int b = __float_as_int(s);
        s = __int_as_float(b + ((b & 1) ? en.d1 : en.d0));
        s += en.lo.x; s += en.lo.y; s += en.lo.z; s += en.lo.w;
        s += en.hi.x; s += en.hi.y; s += en.hi.z; s += en.hi.w;
        en = next;
      }
    }
    if (lane == 0) {
      const float cols = (float)d;
      const float mean = s / (cols > 1.0f ? cols : 1.0f);
      inv_shared = 1.0f / sqrtf(mean + eps);
    }
  }
  __syncthreads();
  if (!in) return;
  const float inv = inv_shared;
  float o[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = (xs[i] * inv) * gs[i];
  float4* py = (float4*)(y + (size_t)blockIdx.x * d + col);
  py[0] = float4{o[0], o[1], o[2], o[3]};
  py[1] = float4{o[4], o[5], o[6], o[7]};
}

}  // namespace

hipError_t launch_rmsnorm_gamma(const NormArgs& a, hipStream_t s) {
  if (a.T <= 0 || a.d <= 0) return hipSuccess;
  const bool aligned = (((uintptr_t)a.x | (uintptr_t)a.gamma | (uintptr_t)a.y) & 15) == 0;
  // The scan takes a wave per 512 columns.  Rows of less than half a wave, and several thousand rows of less than
  // two and a half waves with a part of the last one empty, are faster four to a workgroup (that / the scan, us:
  // d = 128, 64 rows 3.2 / 3.6, 16384 7.3 / 12.9; d = 256, 64 3.8 / 3.6, 4096 5.1 / 6.1; d = 384, 2048 5.1 / 4.5, 4096 6.4 /
  // 6.8, 16384 11.8 / 14.0; d = 640, 6000 8.7 / 11.1; d = 1032, 3000 10.8 / 9.9, 6000 13.4 / 15.3; whole waves and longer
  // rows: d = 512, 4096 7.4 / 6.6, 16384 14.8 / 14.9; d = 1024, 16384 30.0 / 23.7; d = 1280, 6000 15.4 / 15.5, 16384 38.5 /
  // 32.1).
  const bool scan = a.d >= 256 && (a.T < 4096 || a.d >= 1280 || a.d % 512 == 0);
  if (a.policy != ATENIA_MOE_NORM_F64 && a.d % kFoldCols == 0 && a.d <= kFoldMaxCols && aligned && scan) {
    const int threads = (a.d / kFoldCols + 63) / 64 * 64;
    rmsnorm_fold_kernel<<<(unsigned)a.T, threads, threads / 64 * 65 * 48, s>>>(a.x, a.gamma, a.eps, a.d, a.y);
    return hipGetLastError();
  }
  const unsigned grid = (unsigned)((a.T + kRows - 1) / kRows);
  const bool vec = (a.d & 3) == 0;
#define ATENIA_NORM_LAUNCH(P, V) \
  rmsnorm_gamma_kernel<P, V><<<grid, kThreads, 0, s>>>(a.x, a.gamma, a.eps, a.T, a.d, a.y)
  if (a.policy == ATENIA_MOE_NORM_F64) {
    if (vec) ATENIA_NORM_LAUNCH(1, true); else ATENIA_NORM_LAUNCH(1, false);
  } else {
    if (vec) ATENIA_NORM_LAUNCH(0, true); else ATENIA_NORM_LAUNCH(0, false);
  }
#undef ATENIA_NORM_LAUNCH
  return hipGetLastError();
}

}  // namespace atenia_moe
