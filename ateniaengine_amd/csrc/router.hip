// Kernel 1: router GEMV/GEMM + softmax + top-k, bit-exact with the reference's CPU router.
//
// Follows, operation for operation and cast for cast:
//   logits  = matvec(W_r, x)            src/moe/dense.rs:97-115, 325-337
//             one sequential, c-ascending f64 sum per (token, expert), rounded to f32 once
//   weights = softmax(logits)           src/moe/dense.rs:172-187
//             f32 max, f32 subtraction, f64 exp, sequential f64 sum, (f32)(e * (1/sum))
//   top-k                               src/moe/sparse.rs:142-191
//             order (f32 weight desc, index asc); selected indices emitted ascending;
//             f64 renormalisation over the selected weights in ascending order
//   shared-expert gate                  src/moe/layer.rs:436-443  sigmoid(f64 dot)
//
// Products of two f32 values are exact in f64, so fma(w, x, acc) rounds exactly like the
// reference's separate multiply and add.  Two kernels compute the dot products:
//
//  * router_tile_kernel (any batch): each (token, row) pair is owned by one thread that walks
//    c = 0..d-1 in order, so the f64 sum IS the reference's sum.
//  * router_token_kernel (small batches, where that serial chain would dominate the layer):
//    one workgroup per token, every row split over a wavefront and reduced with shuffles.
//    A different summation order is only allowed when it provably cannot change the result: a
//    bound on the rounding of either order leaves one f32 (one sigmoid for the gate row) that both
//    can round to -- a crude bound for every sum, one from the partial sums for those it flags
//    (pieces_bound below).  A row that fails both is recomputed in the reference's order.
//  * router_mfma_kernel (larger batches): the same on the f64 matrix cores.
#include <algorithm>
#include <climits>
#include <cstdlib>

#include "moe_internal.h"

#include <mutex>

namespace atenia_moe {

namespace {

constexpr int kRouterThreads = 256;
constexpr int kKc = 32;            // columns staged per step
constexpr int kLd = kKc + 1;       // padded LDS row stride (words)
constexpr int kTokenThreads = 1024;
// Work (tokens x rows x columns) up to which the per-token kernel, which reads the whole stacked matrix
// for every token, takes batches of more than 64 rows.
constexpr long long kTokenMaxWork = 16ll << 20;

__device__ inline float load_x(const float* x, size_t i) { return x[i]; }
__device__ inline float load_x(const uint16_t* x, size_t i) {
  return __uint_as_float(((uint32_t)x[i]) << 16);
}

// f32 -> bf16 bits, round to nearest even (NaN kept quiet).
__device__ inline uint16_t f32_to_bf16_rne(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

// Two f32 -> two bf16 (round to nearest even), low half = a.
typedef __attribute__((ext_vector_type(2))) float router_f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 router_bf16x2;
__device__ inline uint32_t bf16_pair(float a, float b) {
  const router_f32x2 v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, router_bf16x2));
}

// Last-bit exponent of an exact zero.
constexpr int kNoLsb = 32767;

// Inclusive scan of f64 values over the lanes of a wave, on DPP moves.
template <int CTRL, int ROWS>
__device__ inline double add_dpp(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, ROWS, 0xf, false);
  const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, ROWS, 0xf, false);
  return v + __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);  // + 0.0 where a lane has no source
}
__device__ inline double wave_scan_f64(double v) {
  v = add_dpp<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8: scans of 16 lanes
  v = add_dpp<0x112, 0xf>(v);
  v = add_dpp<0x114, 0xf>(v);
  v = add_dpp<0x118, 0xf>(v);
  v = add_dpp<0x142, 0xa>(v);  // lane 15 of rows 0, 2 -> rows 1, 3
  v = add_dpp<0x143, 0xc>(v);  // lane 31 -> rows 2, 3
  return v;
}
__device__ inline double last_lane_f64(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_readlane((int)(uint32_t)b, 63);
  const uint32_t hi = __builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), 63);
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}

template <int CTRL, int ROWS>
__device__ inline double max_dpp(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_update_dpp((int)(uint32_t)b, (int)(uint32_t)b, CTRL, ROWS, 0xf, false);
  const uint32_t hi =
      __builtin_amdgcn_update_dpp((int)(uint32_t)(b >> 32), (int)(uint32_t)(b >> 32), CTRL, ROWS, 0xf, false);
  return fmax(v, __builtin_bit_cast(double, (uint64_t)hi << 32 | lo));
}
__device__ inline double wave_max_f64(double v) {  // of finite values; the same in all lanes
  v = max_dpp<0x111, 0xf>(v);
  v = max_dpp<0x112, 0xf>(v);
  v = max_dpp<0x114, 0xf>(v);
  v = max_dpp<0x118, 0xf>(v);
  v = max_dpp<0x142, 0xa>(v);
  return last_lane_f64(max_dpp<0x143, 0xc>(v));
}

// How far the reference's c-ascending f64 sum of one row is from a sum in another order, from what
// the partial sums amount to.  The interval the kernels test first allows every addition a rounding
// of sum|p| (2 d u sum|p| in all, u = 2^-53) and flags about one sum in a thousand; nearly all of those
// pass here, where the alternative is one thread walking the reference's order (2048 dependent steps of
// 15 ns).
// A row is cut into pieces of 512 columns, lane l of a wave holding the columns 8 l .. 8 l + 7 of a
// piece, so the partial sums in the reference's order are P + x + c_j (P: the pieces before, x: the
// lanes before, c_j: the lane's own first j products): none is larger than peak = max(|P| + |x| + |c_j|),
// and no sum of consecutive products, the difference of two, larger than 2 peak.  Two bounds:
//  * by size: d additions in the reference's order round by u peak at most, and the 14 d / 8 + pieces
//    of this one (8 per lane, six levels of the scan, the pieces) by 2 u peak.
//  * by steps, because most additions do not round at all: let 2 peak < 2^(g + 53).  Products that
//    are multiples of 2^g add up exactly in either order.  In the reference's order a product with
//    bits below 2^g leaves a sum that rounds again only when it grows past a power of two, each time
//    to the next coarser unit, by 2^(g - 1) at most: less than 2^g in all until the next such product.  In
//    this order its bits pass through 14 + pieces additions, each rounding by 2^(g - 1) at most.
//    bf16 times f32 products of like size have 32 bits, so of 2048 about one is that small (2^-21 of the
//    sum); bf16 times bf16 hardly ever.
// g has to be known before the products are counted: it comes from a generous guess of peak, which the
// counted sums confirm or not.  A row that fails is counted once more with the g of its counted peak: a few
// large products that cancel (a channel of large activations, say) make peak many times the guess.
// The work is dealt to all waves of the workgroup in one short pass: it is code that runs once per
// launch, and fetching its instructions and serial chains of f64 (15 ns a step) are most of its time.
constexpr int kPiece = 512;
struct PieceSums {
  double total, peak;  // its sum, its largest |x| + |c_j|
  double coarse;       // products that are not multiples of 2^g
};
// -g for a peak: 2 peak < 2^(ilogb + 1) = 2^(g + 53)
__device__ inline int units_of(double peak) { return 52 - ilogb(fmax(2.0 * peak, 0x1p-297)); }
// -g for a guess of what peak may be: eight times the random walk's step sum and twice the sum itself.
__device__ inline int guess_units(double sum, double sum_abs, int d) {
  return units_of(8.0 * sum_abs * (double)rsqrtf((float)d) + 2.0 * fabs(sum));
}
__device__ inline void visit_piece(const float (&w)[8], const float (&x)[8], int units, PieceSums* out) {
  double c = 0.0, cmax = 0.0;
  int coarse = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const double pr = (double)w[k] * (double)x[k];  // exact
    c += pr;
    cmax = fmax(cmax, fabs(c));
    const double of_g = ldexp(pr, units);
    coarse += __popcll(__ballot(rint(of_g) != of_g));  // (what is not a number counts)
  }
  const double incl = wave_scan_f64(c);
  const double peak = wave_max_f64(fabs(incl - c) + cmax);
  if ((threadIdx.x & 63) == 63) {
    out->total = incl;
    out->peak = peak;
    out->coarse = (double)coarse;
  }
}
// The row's sum and |a - reference| <= e from its pieces, by one wave; the same in all lanes.  The
// factors 1.001 cover the roundings of what was summed here and of the bounds, the 4 u |a| those of
// a -/+ e.  e = 0: both sums are exact.  counted: units of the counted peak (units where that is no number).
__device__ inline void pieces_bound(const PieceSums* piece, int pieces, int units, double& a, double& e,
                                    int& counted) {
  const int lane = threadIdx.x & 63;
  double peak = 0.0, coarse = 0.0;
  a = 0.0;
#pragma clang loop unroll(disable)
  for (int p = lane; p - lane < pieces; p += 64) {  // (once for rows of up to 32768 columns)
    const bool on = p < pieces;
    const double total = on ? piece[p].total : 0.0, top = on ? piece[p].peak : 0.0;
    const double incl = wave_scan_f64(total);
    peak = fmax(peak, wave_max_f64(fabs(a + (incl - total)) + top));
    coarse += last_lane_f64(wave_scan_f64(on ? piece[p].coarse : 0.0));
    a += last_lane_f64(incl);
  }
  peak *= 1.001;
  constexpr double u = 1.1102230246251565e-16;
  const double n = (double)kPiece * pieces;  // (the zeros past d count)
  const double by_size = (n + 2.0 * (1.75 * n + pieces)) * peak * (u * 1.001);
  const double unit = ldexp(1.0, -units);  // 2^g
  e = by_size;
  if (2.0 * peak < unit * 0x1p53) e = fmin(e, coarse * (1.0 + 0.5 * (14 + pieces)) * unit * 1.001);
  if (e > 0.0) e += 4.0 * u * fabs(a);
  counted = units_of(peak);
  if (!isfinite(a) || !(by_size < INFINITY)) {
    e = INFINITY;
    counted = units;
  }
}
// Every value of [a - e, a + e] rounds to the same f32 (the same f32 sigmoid for the gate row).
__device__ inline bool rounds_alike(double a, double e, bool gate_row) {
  const double lo = a - e, hi = a + e;
  if (gate_row) return (float)(1.0 / (1.0 + exp(-lo))) == (float)(1.0 / (1.0 + exp(-hi)));
  const float flo = (float)lo;
  return flo == (float)hi && isfinite(flo);
}

// Softmax + top-k + renormalisation of ONE token by the threads r = 0..E-1 that call with
// `on`; every thread of the workgroup must call (barriers inside).  lg: [E] f32 logits,
// ex: [E] f64, wt: [E] f32, sel: [E] i32 scratch of this token.
__device__ inline void softmax_topk(bool on, int r, int E, int k, int renorm, int token,
                                    const float* lg, double* ex, float* wt, int32_t* sel,
                                    int32_t* __restrict__ idx_out, float* __restrict__ w_out,
                                    int32_t* __restrict__ status) {
  float my_logit = 0.f;
  if (on) {
    float mx = -INFINITY;
#pragma unroll 8
    for (int e = 0; e < E; ++e) mx = fmaxf(mx, lg[e]);  // skips NaN like f32::max
    my_logit = lg[r];
    ex[r] = exp((double)(my_logit - mx));                // f32 subtraction, then f64 exp
  }
  __syncthreads();
  float my_w = 0.f;
  if (on) {
    double sum = 0.0;
#pragma unroll 8
    for (int e = 0; e < E; ++e) sum += ex[e];            // sequential fold, e ascending
    double inv = sum > 0.0 ? 1.0 / sum : 0.0;
    my_w = (float)(ex[r] * inv);
    wt[r] = my_w;
    if (!isfinite(my_w) || my_w < 0.f) {
      atomicMin(&status[0], -3);
      atomicMin(&status[1], (token << 10) | r);
    }
  }
  __syncthreads();
  bool selected = false;
  if (on) {
    int rank = 0;  // experts that sort before me under (weight desc, index asc)
#pragma unroll 8
    for (int e = 0; e < E; ++e) {
      float we = wt[e];
      rank += (we > my_w) || (we == my_w && e < r);
    }
    selected = rank < k;
    sel[r] = selected ? 1 : 0;
  }
  __syncthreads();
  if (on && selected) {
    int slot = 0;
    double sum = 0.0;
    for (int e = 0; e < E; ++e) {
      if (sel[e]) {
        slot += e < r;
        sum += (double)wt[e];  // ascending e, as the reference sums the sorted selection
      }
    }
    double scale = renorm ? 1.0 / sum : 1.0;
    if (slot < k) {
      size_t o = (size_t)token * k + slot;
      idx_out[o] = r;
      w_out[o] = (float)((double)my_w * scale);
    }
  }
}

template <typename XT>
__global__ __launch_bounds__(kRouterThreads) void router_tile_kernel(
    const XT* __restrict__ x, int T, int d, int E, int k, int renorm,
    const float* __restrict__ w_router, const float* __restrict__ bias,
    const float* __restrict__ gate_vec, int32_t* __restrict__ idx_out,
    float* __restrict__ w_out, float* __restrict__ sgate_out, uint16_t* __restrict__ xb,
    int d_pad, int32_t* __restrict__ status, float* __restrict__ logits_out, int tokens_per_block) {
  const int R = E + (gate_vec ? 1 : 0);  // rows of the stacked [W_r ; gate] matrix
  const int TT = tokens_per_block;
  const int t0 = blockIdx.x * TT;
  const int tid = threadIdx.x;

  extern __shared__ float smem[];
  float* sW = smem;                       // [R][kLd]
  float* sX = sW + (size_t)R * kLd;       // [TT][kLd]
  // after the dot products the same memory is reused:
  //   sLogit [TT][R] f32, sExp [TT][E] f64, sWt [TT][E] f32, sSel [TT][E] i32

  const int tl = tid / R;  // local token
  const int r = tid - tl * R;
  const bool owner = tl < TT && (t0 + tl) < T;
  double acc = 0.0;

  const int c_end = xb ? (d_pad > d ? d_pad : d) : d;
  for (int c0 = 0; c0 < c_end; c0 += kKc) {
    __syncthreads();
    for (int j = tid; j < R * kKc; j += kRouterThreads) {
      int row = j / kKc, col = j - row * kKc;
      int c = c0 + col;
      float v = 0.f;
      if (c < d) v = row < E ? w_router[(size_t)row * d + c] : gate_vec[c];
      sW[row * kLd + col] = v;
    }
    for (int j = tid; j < TT * kKc; j += kRouterThreads) {
      int row = j / kKc, col = j - row * kKc;
      int c = c0 + col, t = t0 + row;
      float v = 0.f;
      if (t < T && c < d) v = load_x(x, (size_t)t * d + c);
      sX[row * kLd + col] = v;
      if (xb && t < T && c < d_pad) xb[(size_t)t * d_pad + c] = f32_to_bf16_rne(v);
    }
    __syncthreads();
    if (owner && c0 < d) {
      const float* wr = sW + r * kLd;
      const float* xr = sX + tl * kLd;
      // Columns past d hold zeros in both tiles: adding +0.0 leaves the sum unchanged.
#pragma unroll
      for (int c = 0; c < kKc; ++c) acc = fma((double)wr[c], (double)xr[c], acc);
    }
  }
  __syncthreads();

  float* sLogit = smem;                                   // [TT][R]
  double* sExp = (double*)(smem + ((TT * R + 1) & ~1));   // [TT][E]
  float* sWt = (float*)(sExp + (size_t)TT * E);           // [TT][E]
  int32_t* sSel = (int32_t*)(sWt + (size_t)TT * E);       // [TT][E]

  if (owner) {
    float logit = (float)acc;
    if (r < E) {
      if (bias) logit = logit + bias[r];
      sLogit[tl * R + r] = logit;
      if (logits_out) logits_out[(size_t)(t0 + tl) * E + r] = logit;
    } else {
      sgate_out[t0 + tl] = (float)(1.0 / (1.0 + exp(-acc)));
    }
  }
  __syncthreads();
  if (logits_out) return;  // routing is decided by another kernel from the raw logits
  const int tls = owner ? tl : 0;
  softmax_topk(owner && r < E, r, E, k, renorm, t0 + tls, sLogit + tls * R, sExp + tls * E,
               sWt + tls * E, sSel + tls * E, idx_out, w_out, status);
}

// Softmax + top-k + renormalisation of a block of TT tokens at once, same arithmetic and order
// as softmax_topk.  The steps that the reference does as sequential folds over the experts
// (f64 sum of the exponentials, f64 sum of the selected weights) are dependent chains, so one
// thread per token runs them for all tokens of the block side by side; the element-wise steps
// (exp, weight, rank) are spread over all threads.  lg: [TT][R] f32 logits in LDS; scratch:
// ex [TT][E] f64, wt [TT][E] f32, sel [TT][E] u8, tok [TT] f64 (max, then 1/sum).
__device__ inline void softmax_topk_block(int TT, int R, int E, int k, int renorm, int t0, int T,
                                          const float* lg, double* ex, float* wt, uint8_t* sel,
                                          double* tok, int32_t* __restrict__ idx_out,
                                          float* __restrict__ w_out,
                                          int32_t* __restrict__ status) {
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int pairs = TT * E;
  if (tid < TT) {
    const float* l = lg + tid * R;
    float mx = -INFINITY;
#pragma unroll 8
    for (int e = 0; e < E; ++e) mx = fmaxf(mx, l[e]);  // skips NaN like f32::max
    tok[tid] = (double)mx;
  }
  __syncthreads();
  for (int pr = tid; pr < pairs; pr += nthr) {
    const int t = pr / E, e = pr - t * E;
    ex[pr] = exp((double)(lg[t * R + e] - (float)tok[t]));  // f32 subtraction, then f64 exp
  }
  __syncthreads();
  if (tid < TT) {
    const double* x = ex + tid * E;
    double sum = 0.0;
#pragma unroll 8
    for (int e = 0; e < E; ++e) sum += x[e];  // sequential fold, e ascending
    tok[tid] = sum > 0.0 ? 1.0 / sum : 0.0;
  }
  __syncthreads();
  for (int pr = tid; pr < pairs; pr += nthr) {
    const int t = pr / E, e = pr - t * E;
    const float w = (float)(ex[pr] * tok[t]);
    wt[pr] = w;
    if ((!isfinite(w) || w < 0.f) && t0 + t < T) {
      atomicMin(&status[0], -3);
      atomicMin(&status[1], ((t0 + t) << 10) | e);
    }
  }
  __syncthreads();
  for (int pr = tid; pr < pairs; pr += nthr) {
    const int t = pr / E, e = pr - t * E;
    const float* w = wt + t * E;
    const float my_w = w[e];
    int rank = 0;  // experts that sort before me under (weight desc, index asc)
#pragma unroll 8
    for (int o = 0; o < E; ++o) {
      const float wo = w[o];
      rank += (wo > my_w) || (wo == my_w && o < e);
    }
    sel[pr] = rank < k ? 1 : 0;
  }
  __syncthreads();
  if (tid < TT && t0 + tid < T) {
    const float* w = wt + tid * E;
    const uint8_t* sl = sel + tid * E;
    double sum = 0.0;
#pragma unroll 8
    for (int e = 0; e < E; ++e)
      if (sl[e]) sum += (double)w[e];  // ascending e, as the reference sums the sorted selection
    const double scale = renorm ? 1.0 / sum : 1.0;
    size_t o = (size_t)(t0 + tid) * k;
    int slot = 0;
    for (int e = 0; e < E && slot < k; ++e) {
      if (sl[e]) {
        idx_out[o + slot] = e;
        w_out[o + slot] = (float)((double)w[e] * scale);
        ++slot;
      }
    }
  }
}

// Batched form of the sequential kernel for up to 64 rows.  Same arithmetic and order as
// router_tile_kernel (one c-ascending f64 fma chain per (token, row)); what changes is how the
// chains are fed:
//   * a thread owns TPT tokens and RPT rows (rows rg, rg + RG, ...), so a value read from
//     LDS serves several chains and the chains of one thread hide each other's fma latency;
//   * tiles of KC columns are converted to f64 once while they are stored to LDS, so the
//     inner loop is ds_read_b128 (two consecutive columns) + fma only;
//   * the global loads of tile s+2 are issued into registers before tile s is multiplied.
template <typename XT> struct XVec;
template <> struct XVec<float> {
  typedef float4 type;
  static __device__ inline float4 load(const float* p) { return *(const float4*)p; }
  static __device__ inline void unpack(float4 v, float (&f)[4]) { f[0] = v.x; f[1] = v.y; f[2] = v.z; f[3] = v.w; }
  static __device__ inline float4 zero() { return make_float4(0.f, 0.f, 0.f, 0.f); }
};
template <> struct XVec<uint16_t> {
  typedef uint2 type;
  static __device__ inline uint2 load(const uint16_t* p) { return *(const uint2*)p; }
  static __device__ inline void unpack(uint2 v, float (&f)[4]) {
    f[0] = __uint_as_float(v.x << 16); f[1] = __uint_as_float(v.x & 0xffff0000u);
    f[2] = __uint_as_float(v.y << 16); f[3] = __uint_as_float(v.y & 0xffff0000u);
  }
  static __device__ inline uint2 zero() { return make_uint2(0u, 0u); }
};

template <typename XT, int RPT, int TPT, int KC>
__global__ __launch_bounds__(kRouterThreads) void router_batch_kernel(
    const XT* __restrict__ x, int T, int d, int E, int k, int renorm,
    const float* __restrict__ w_router, const float* __restrict__ bias,
    const float* __restrict__ gate_vec, int32_t* __restrict__ idx_out,
    float* __restrict__ w_out, float* __restrict__ sgate_out, uint16_t* __restrict__ xb,
    int d_pad, int32_t* __restrict__ status, float* __restrict__ logits_out) {
  constexpr int RG = 16;                   // row groups = threads per token
  constexpr int TG = kRouterThreads / RG;  // 16 token groups = threads per row group
  constexpr int TT = TG * TPT;             // tokens per block: a thread owns tokens tg, tg + TG, ...
  constexpr int RW = RG * RPT;             // rows of the staged weight tile (>= R)
  constexpr int LD = KC + 2;               // f64 row stride: rows 4 banks apart, 16-byte aligned
  constexpr int KV = KC / 4;               // 4-column vectors per tile row
  constexpr int NX = (TT * KV + kRouterThreads - 1) / kRouterThreads;
  constexpr int NW = (RW * KV + kRouterThreads - 1) / kRouterThreads;
  typedef XVec<XT> XV;
  const int R = E + (gate_vec ? 1 : 0);
  const int t0 = blockIdx.x * TT;
  // More than RW rows: blockIdx.y picks the block of RW rows (only when the logits go to
  // `logits_out`, since the softmax below needs all rows of a token in one workgroup).
  const int r_lo = blockIdx.y * RW;
  const int tid = threadIdx.x;
  const int tg = tid / RG, rg = tid - tg * RG;

  extern __shared__ double smem_b[];
  double* sX = smem_b;            // [TT][LD]
  double* sW = sX + TT * LD;      // [RW][LD]

  typedef typename XV::type xvec_t;
  auto load_tile = [&](xvec_t (&xr)[NX], float4 (&wr)[NW], int c0) {
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int j = tid + i * kRouterThreads;
      const int row = j / KV, c = c0 + (j - row * KV) * 4;
      xr[i] = XV::zero();
      if (j < TT * KV && t0 + row < T && c < d) xr[i] = XV::load(x + (size_t)(t0 + row) * d + c);
    }
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const int j = tid + i * kRouterThreads;
      const int row = j / KV, c = c0 + (j - row * KV) * 4;
      wr[i] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (j < RW * KV && r_lo + row < R && c < d)
        wr[i] = *(const float4*)((r_lo + row < E ? w_router + (size_t)(r_lo + row) * d : gate_vec) + c);
    }
  };
  auto store_tile = [&](const xvec_t (&xr)[NX], const float4 (&wr)[NW], int c0) {
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int j = tid + i * kRouterThreads;
      if (j < TT * KV) {
        const int row = j / KV, cl = (j - row * KV) * 4;
        float f[4];
        XV::unpack(xr[i], f);
        double* dst = sX + row * LD + cl;
        *(double2*)dst = make_double2((double)f[0], (double)f[1]);
        *(double2*)(dst + 2) = make_double2((double)f[2], (double)f[3]);
        const int c = c0 + cl;
        if (xb && blockIdx.y == 0 && t0 + row < T && c < d_pad) {
          uint2 b;
          b.x = f32_to_bf16_rne(f[0]) | ((uint32_t)f32_to_bf16_rne(f[1]) << 16);
          b.y = f32_to_bf16_rne(f[2]) | ((uint32_t)f32_to_bf16_rne(f[3]) << 16);
          *(uint2*)(xb + (size_t)(t0 + row) * d_pad + c) = b;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const int j = tid + i * kRouterThreads;
      if (j < RW * KV) {
        const int row = j / KV, cl = (j - row * KV) * 4;
        double* dst = sW + row * LD + cl;
        *(double2*)dst = make_double2((double)wr[i].x, (double)wr[i].y);
        *(double2*)(dst + 2) = make_double2((double)wr[i].z, (double)wr[i].w);
      }
    }
  };

  double acc[TPT][RPT];
#pragma unroll
  for (int j = 0; j < TPT; ++j)
#pragma unroll
    for (int i = 0; i < RPT; ++i) acc[j][i] = 0.0;
  // Columns from d up to c_end exist only to zero-fill the padding of xb; both staged tiles
  // hold +0.0 there, which leaves every sum unchanged.
  const int c_end = xb ? (d_pad > d ? d_pad : d) : d;
  // Two register sets: the loads of tile s+2 are issued while tile s is multiplied, so a
  // load has two multiply phases to land before its tile is stored to LDS.
  xvec_t xr0[NX], xr1[NX];
  float4 wr0[NW], wr1[NW];
  // Workgroup barrier that orders LDS traffic only.  __syncthreads() would also wait for
  // every outstanding global load, which is exactly the latency the prefetch is there to hide.
  auto lds_barrier = [] {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  auto step = [&](xvec_t (&xr)[NX], float4 (&wr)[NW], int c0) {
    lds_barrier();  // everyone is done reading the previous tile
    store_tile(xr, wr, c0);
    lds_barrier();
    if (c0 + 2 * KC < c_end) load_tile(xr, wr, c0 + 2 * KC);
    // Columns are taken in groups of CG: the LDS reads of group g+1 are issued before the
    // fma chain steps of group g (two register sets), so no read latency sits between them.
    const double* xs = sX + tg * LD;
    const double* ws = sW + rg * LD;
    constexpr int CG = TPT * RPT <= 4 ? 8 : 4, NV = CG / 2;
    double2 xa[TPT][NV], wa[RPT][NV], xb2[TPT][NV], wb2[RPT][NV];
    auto rd = [&](double2 (&xv)[TPT][NV], double2 (&wv)[RPT][NV], int c) {
#pragma unroll
      for (int u = 0; u < NV; ++u) {
#pragma unroll
        for (int j = 0; j < TPT; ++j) xv[j][u] = *(const double2*)(xs + j * TG * LD + c + 2 * u);
#pragma unroll
        for (int i = 0; i < RPT; ++i) wv[i][u] = *(const double2*)(ws + i * RG * LD + c + 2 * u);
      }
    };
    auto mul = [&](const double2 (&xv)[TPT][NV], const double2 (&wv)[RPT][NV]) {
#pragma unroll
      for (int u = 0; u < NV; ++u)
#pragma unroll
        for (int i = 0; i < RPT; ++i)
#pragma unroll
          for (int j = 0; j < TPT; ++j) {
            acc[j][i] = fma(wv[i][u].x, xv[j][u].x, acc[j][i]);
            acc[j][i] = fma(wv[i][u].y, xv[j][u].y, acc[j][i]);
          }
    };
    static_assert(KC % (2 * CG) == 0, "tile width must hold whole pairs of column groups");
    rd(xa, wa, 0);
    for (int c = 0; c < KC; c += 2 * CG) {
      rd(xb2, wb2, c + CG);
      __builtin_amdgcn_sched_barrier(0);
      mul(xa, wa);
      __builtin_amdgcn_sched_barrier(0);
      if (c + 2 * CG < KC) rd(xa, wa, c + 2 * CG);
      __builtin_amdgcn_sched_barrier(0);
      mul(xb2, wb2);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  load_tile(xr0, wr0, 0);
  if (KC < c_end) load_tile(xr1, wr1, KC);
  for (int c0 = 0; c0 < c_end; c0 += 2 * KC) {
    step(xr0, wr0, c0);
    if (c0 + KC < c_end) step(xr1, wr1, c0 + KC);
  }
  __syncthreads();

  // reuse of the tile memory: logits of the block, then the softmax scratch
  float* sLogit = (float*)smem_b;                          // [TT][R]
  double* sExp = smem_b + ((TT * R + 1) / 2);              // [TT][E]
  double* sTok = sExp + TT * E;                            // [TT]
  float* sWt = (float*)(sTok + TT);                        // [TT][E]
  uint8_t* sSel = (uint8_t*)(sWt + TT * E);                // [TT][E]
#pragma unroll
  for (int j = 0; j < TPT; ++j) {
    const int tl = tg + j * TG;
    if (t0 + tl >= T) continue;
#pragma unroll
    for (int i = 0; i < RPT; ++i) {
      const int r = r_lo + rg + i * RG;
      if (r < E) {
        float logit = (float)acc[j][i];
        if (bias) logit = logit + bias[r];
        sLogit[tl * R + r] = logit;
        if (logits_out) logits_out[(size_t)(t0 + tl) * E + r] = logit;
      } else if (r < R) {
        sgate_out[t0 + tl] = (float)(1.0 / (1.0 + exp(-acc[j][i])));
      }
    }
  }
  __syncthreads();
  if (logits_out) return;  // routing is decided by another kernel from the raw logits
  softmax_topk_block(TT, R, E, k, renorm, t0, T, sLogit, sExp, sWt, sSel, sTok, idx_out, w_out,
                     status);
}

template <typename XT, int RPT, int TPT, int KC>
hipError_t launch_router_batch(const RouterArgs& a, hipStream_t s) {
  constexpr int TT = kRouterThreads / 16 * TPT, RW = 16 * RPT, LD = KC + 2;
  const int R = a.E + (a.shared_gate ? 1 : 0);
  size_t dot_bytes = (size_t)(TT + RW) * LD * 8;
  size_t post_bytes = (((size_t)TT * R + 1) / 2) * 8 + (size_t)TT * a.E * (8 + 4 + 1) + TT * 8 + 16;
  size_t smem = dot_bytes > post_bytes ? dot_bytes : post_bytes;
  if (smem > 64 * 1024) {
    // per instantiation: largest size the attribute was set for (layers may launch from
    // several host threads)
    static std::mutex attr_mu;
    static size_t attr_bytes = 0;
    std::lock_guard<std::mutex> lock(attr_mu);
    if (smem > attr_bytes) {
      hipError_t e = hipFuncSetAttribute((const void*)router_batch_kernel<XT, RPT, TPT, KC>,
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
      if (e != hipSuccess) return e;
      attr_bytes = smem;
    }
  }
  const int blocks = (a.T + TT - 1) / TT;
  const int row_blocks = (R + RW - 1) / RW;
  if (row_blocks > 1 && !a.logits_out) return hipErrorInvalidValue;
  router_batch_kernel<XT, RPT, TPT, KC><<<dim3(blocks, row_blocks), kRouterThreads, smem, s>>>(
      (const XT*)a.x, a.T, a.d, a.E, a.k, a.renorm, a.w_router, a.router_bias, a.shared_gate,
      a.idx, a.w, a.sgate, a.xb, a.d_pad, a.status, a.logits_out);
  return hipGetLastError();
}

// ---- batches on the f64 matrix cores, any summation order made safe by a certificate ---------
// v_mfma_f64_16x16x4_f64 (operand layout: see ffn_f32.hip): A = 16 rows of [W_r ; gate], B = 16
// tokens, so lane l holds D[4 r + l / 16][l % 16] = rows 4 r + l / 16 of token l % 16.  A
// workgroup owns 16 tokens and all rows (RB blocks of 16); its four waves split k and add their
// partial sums in wave order.  f32 operands widen exactly and their products are exact in f64,
// so the result differs from the reference's c-ascending sum only by the order of the f64
// additions.  That is accepted only under the same two certificates as in router_token_kernel:
//   interval : every addition rounds by 2^-53 of what the sum then is.  A wave's share of k is a
//              contiguous segment s of it; the sums of either order are at most |P_s| + N_s inside it,
//              P_s the sum of the segments before (at hand when the waves' parts are added up) and
//              N_s = |w_s| |x_s| >= sum|p| over the segment (Cauchy-Schwarz; |x_s|^2 is accumulated next
//              to the matrix instructions, |w_s| comes with the layer).  With eight segments this
//              is some seven times narrower than d 2^-53 |w| |x|.  If all of [acc - e, acc + e] rounds
//              to one f32 (one f32 sigmoid for the gate row) that value is the reference's;
//   exact    : bf16 operands only: where all those sums stay below 2^53 times the lowest bit that a product
//              can have, nothing rounds in either order.  Passes most of what the interval flags;
//   steps    : the few sums that are left are looked at again with the bound of pieces_bound above;
// and a sum that fails these is recomputed in the reference's order by one lane.  (Launch, one norm over
// the whole of k and exactness followed only with several row blocks / as it is, us: 256 rows of
// d = 7168, 256 tokens 53.5 / 34.3, 1000 tokens 141 / 112; 61 rows, d = 2048, 300 tokens 13.0 / 11.0, 997
// 15.4 / 11.8; 8 rows, d = 4096, 4096 tokens 29.4 / 28.6.  Without any second look the first took 28.)
// Against one sequential chain per (token, row) this is 3-4x faster at 4096 tokens.
typedef __attribute__((__vector_size__(4 * sizeof(double)))) double f64x4_t;

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
template <typename XT> struct XChunk;
template <> struct XChunk<float> {
  float4 lo, hi;
  __device__ inline void load(const float* p) { lo = *(const float4*)p; hi = *(const float4*)(p + 4); }
  __device__ inline void keep(bool k) {  // selects, no branch
    lo.x = k ? lo.x : 0.f; lo.y = k ? lo.y : 0.f; lo.z = k ? lo.z : 0.f; lo.w = k ? lo.w : 0.f;
    hi.x = k ? hi.x : 0.f; hi.y = k ? hi.y : 0.f; hi.z = k ? hi.z : 0.f; hi.w = k ? hi.w : 0.f;
  }
  __device__ inline void get(float (&f)[8]) const {
    f[0] = lo.x; f[1] = lo.y; f[2] = lo.z; f[3] = lo.w; f[4] = hi.x; f[5] = hi.y; f[6] = hi.z; f[7] = hi.w;
  }
};
template <> struct XChunk<uint16_t> {
  uint4 v;
  __device__ inline void load(const uint16_t* p) { v = *(const uint4*)p; }
  __device__ inline void keep(bool k) {
    v.x = k ? v.x : 0u; v.y = k ? v.y : 0u; v.z = k ? v.z : 0u; v.w = k ? v.w : 0u;
  }
  __device__ inline void get(float (&f)[8]) const {
    const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f[2 * i] = __uint_as_float(u[i] << 16);
      f[2 * i + 1] = __uint_as_float(u[i] & 0xffff0000u);
    }
  }
  // min(key, |bits| - 1 of each of the eight values) as unsigned 16-bit numbers, two side by side:
  // magnitudes order like their bit patterns, and a zero wraps to the largest key, so the result names
  // the smallest non-zero magnitude seen (bf16_key_lsb below turns it into a last-bit exponent).
  __device__ inline u16x2 min_key(u16x2 key) const {
    const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i)
      key = __builtin_elementwise_min(key, (u16x2)(__builtin_bit_cast(u16x2, u[i] & 0x7fff7fffu) - (u16x2)1));
    return key;
  }
};
// A bf16 value with exponent field e is a multiple of 2^(e - 134) (2^-133 for a denormal), so
// the exponent field of the smallest non-zero magnitude among some values bounds the last-bit
// exponent of every one of them from below: cheaper to follow than the exact last set bit, and
// the exactness test it feeds has bits to spare.  kNoLsb: every value was zero.  (An inf or a
// NaN is not seen here; it makes the norm that the same test compares infinite or NaN.)
constexpr uint32_t kNoKey = 0xffffu;
__device__ inline int bf16_key_lsb(uint32_t key) {
  return key == kNoKey ? kNoLsb : (int)((key + 1u) >> 7) - 134;
}

// Softmax + top-k from logits that another launch left in HBM, one wavefront per token (up to 64
// experts; wave_select_token in select_wave.h).
constexpr int kWaveSelectThreads = 256;
__global__ __launch_bounds__(kWaveSelectThreads) void wave_select_kernel(
    const float* __restrict__ logits, int T, int E, int k, int renorm,
    int32_t* __restrict__ idx_out, float* __restrict__ w_out, int32_t* __restrict__ status) {
  const int lane = threadIdx.x & 63;
  const int t = blockIdx.x * (kWaveSelectThreads / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (t >= T) return;
  wave_select_token(logits + (size_t)t * E, E, k, renorm, t, lane, idx_out, w_out, status);
}

// PAIR (up to eight rows): eight tokens to a workgroup.  Rows and tokens take half of a matrix instruction each, and
// the other halves are the same rows and tokens at other k: of the wave's steps lanes with bit 3 clear take the first
// half, those with it set the second, and the two diagonal blocks of the result are the two sums.  (Sixteen tokens
// and half of every instruction zeros / this, 8 rows, d = 4096, launch, us: T = 512 to 1537 20 / 13-14, 2048 20.5 / 14.3, 4096
// 24.8 / 24.4, 8192 40.3 / 40.0; inside the layer T = 1000 29.0 / 19.0.)
template <typename XT, int RB, int NBUF, int NWV, bool PAIR>
__global__ __launch_bounds__(64 * NWV) void router_mfma_kernel(
    const XT* __restrict__ x, int T, int d, int E, int k, int renorm,
    const float* __restrict__ w_router, const float* __restrict__ bias,
    const float* __restrict__ gate_vec, int32_t* __restrict__ idx_out,
    float* __restrict__ w_out, float* __restrict__ sgate_out, int32_t* __restrict__ status,
    float* __restrict__ logits_out, const int32_t* __restrict__ w_lsb,
    const uint16_t* __restrict__ w_t8, int Rp, const double* __restrict__ w_norm2,
    uint16_t* __restrict__ xb, int d_pad) {
  // gridDim.y > 1 (only with logits_out): this workgroup owns the rows row0 .. row0 + R - 1 of
  // the stacked matrix [W_r ; gate] and leaves the logits to another launch; otherwise all rows.
  constexpr int TT = PAIR ? 8 : 16;
  static_assert(!PAIR || RB == 1, "eight rows");
  const int R_all = E + (gate_vec ? 1 : 0);
  constexpr int kRows = PAIR ? 8 : 16 * RB;
  const int row0 = blockIdx.y * kRows;
  const int R = min(kRows, R_all - row0);
  const int t0 = blockIdx.x * TT;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int r16 = lane & 15, q = lane >> 4;

  extern __shared__ double smem_m[];
  constexpr int NT = 64 * NWV;                    // NWV waves split k
  double* sPart = smem_m;                         // [NWV][RB][4][64] partial sums
  double* sXsq = sPart + NWV * RB * 4 * 64;       // [NWV][16]  partial |x_t|^2
  double* sAcc = sXsq + NWV * 16;                 // [16][R]
  double* sXn2 = sAcc + 16 * R;                   // [16]
  double* sWn2 = sXn2 + 16;                       // [R]
  double* sXseg = sWn2 + R;                       // [NWV][16]  |x_t| over each wave's share of k
  double* sWseg = sXseg + NWV * 16;               // [NWV][16 RB]  |w_r| over the same
  float* sLogit = (float*)(sWseg + NWV * 16 * RB);  // [16][R]
  uint32_t* sXq = (uint32_t*)(sLogit + 16 * R);   // [NWV][16] key of the smallest |x_t| (partial)
  uint8_t* sFlag = (uint8_t*)(sXq + NWV * 16);    // [16][R] 1 = the interval certificate failed
  // A lower bound of the last-bit exponent of the token's activations is followed beside the matrix
  // instructions: f64 matrix instructions and vector instructions do not overlap on this chip (a step
  // costs the sum of both), hence two values to an instruction.  (f32 activations: nearly no sum is exact
  // in every order, so nothing is followed.)
  constexpr bool kBf16X = sizeof(XT) == 2;
  u16x2 xq = (u16x2)(uint16_t)kNoKey;

  const int half = PAIR ? r16 >> 3 : 0;
  const int tok = min(t0 + (r16 & (TT - 1)), T - 1);  // rows past T repeat the last token; never written out
  const XT* px = x + (size_t)tok * d + 8 * q;
  // The stacked matrix comes from its bf16 copy in chunk-major order [d / 8][Rp][8] (made when
  // the layer is created; rows past the last one and chunks past d are zeros): the 16 rows of a
  // block lie side by side, so a load instruction reads 4 x 256 contiguous bytes instead of 64
  // bytes from each of 16 rows -- the row-major f32 matrix cost the load path a fifth of the
  // loop -- and neither a clamp nor a select is needed.
  const uint16_t* pw[RB];
#pragma unroll
  for (int b = 0; b < RB; ++b) pw[b] = w_t8 + ((size_t)q * Rp + row0 + 16 * b + (r16 & (TT - 1))) * 8;
  const size_t w_step = (size_t)32 * Rp;  // four chunks
  if (tid < R) sWn2[tid] = w_norm2[row0 + tid];  // |w_r|^2, read after the barriers below
  constexpr int kSegLoads = (NWV * 16 * RB + NT - 1) / NT;
  double w_seg[kSegLoads];  // stored below, behind the loop
#pragma unroll
  for (int i = 0; i < kSegLoads; ++i) {
    const int at = min(tid + i * NT, NWV * 16 * RB - 1);
    w_seg[i] = w_norm2[(size_t)((NWV == 8 ? kNormEighths : kNormQuarters) + at / (16 * RB)) * Rp + row0 + at % (16 * RB) % kRows];
  }
  static_assert(NWV == 8 || NWV == 4, "the layer has the norms of eighths and of quarters");
  // k in steps of 32 (8 per lane), the steps dealt to the four waves in contiguous runs
  const int nsteps = (d + 31) / 32;
  const int per = (nsteps + NWV - 1) / NWV;
  const int s0 = wave * per, s1 = min(nsteps, s0 + per);
  // PAIR: `n_half` steps for either half of the lanes, the second half's the last ones.  An odd number's middle step
  // is the first half's: the other lanes multiply zeros there.
  const int n_half = PAIR ? (s1 - s0 + 1) >> 1 : s1 - s0;
  const int lane_s0 = half ? max(s1 - n_half, 0) : s0;  // this lane's first step
  const bool skips_first = half && ((s1 - s0) & 1);
#pragma unroll
  for (int b = 0; b < RB; ++b) pw[b] += (size_t)lane_s0 * w_step;

  // One row block: two accumulators in turn, so that consecutive matrix instructions do not
  // wait for each other's result (summed once at the end; any order is as good).  With more
  // blocks their instructions interleave anyway and the registers are better spent on a second
  // workgroup per compute unit.
  constexpr int NACC = RB == 1 ? 2 : 1;
  f64x4_t acc[RB][NACC];
#pragma unroll
  for (int b = 0; b < RB; ++b)
#pragma unroll
    for (int n = 0; n < NACC; ++n) acc[b][n] = f64x4_t{0.0, 0.0, 0.0, 0.0};
  double xsq = 0.0;

  XChunk<XT> xc[NBUF];
  XChunk<uint16_t> wc[NBUF][RB];
  // Every step issues the same loads whatever the lane or the step: a chunk past d is fetched
  // from the row's first columns and zeroed with selects, a step past the wave's range repeats
  // its last one.  With a branch around a load the compiler can no longer count the loads in
  // flight and waits for all of them (s_waitcnt vmcnt(0)) before every use.  The selects stand
  // where the chunk is used: next to the load they made the loop wait for the chunk just requested,
  // once per NBUF steps (64 against 66 us for the launch on 256 rows of d = 7168, 256 tokens).
  // (st: steps from the lane's first one)
  auto load_step = [&](int buf, int st) {
    st = min(st, n_half - 1);
    const int c = (lane_s0 + st) * 32;
    xc[buf].load(px + (c + 8 * q < d ? c : 0));
#pragma unroll
    for (int b = 0; b < RB; ++b) wc[buf][b].load(pw[b] + (size_t)st * w_step);
  };
  // f32 activations: the workgroups of the first row block leave the bf16 copy the experts read
  const bool stores_xb = !kBf16X && xb && blockIdx.y == 0 && t0 + (r16 & (TT - 1)) < T;
  auto multiply = [&](int buf, int st) {
    const int c = (lane_s0 + st) * 32 + 8 * q;
    const bool mine = !(PAIR && st == 0 && skips_first);
    xc[buf].keep(c < d && mine);  // d is a multiple of 8: a chunk is whole or absent
    float xf[8];
    xc[buf].get(xf);
    if constexpr (!kBf16X) {
      if (stores_xb && c < d_pad && mine)
        *(uint4*)(xb + (size_t)tok * d_pad + c) = uint4{bf16_pair(xf[0], xf[1]), bf16_pair(xf[2], xf[3]),
                                                       bf16_pair(xf[4], xf[5]), bf16_pair(xf[6], xf[7])};
    }
    if constexpr (kBf16X) xq = xc[buf].min_key(xq);
    double xd[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      xd[t] = (double)xf[t];
      xsq = fma(xd[t], xd[t], xsq);
    }
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      float wf[8];
      wc[buf][b].get(wf);
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const double wd = (double)wf[t];
        acc[b][t % NACC] = __builtin_amdgcn_mfma_f64_16x16x4f64(wd, xd[t], acc[b][t % NACC], 0, 0, 0);
      }
    }
  };
  if (s0 < s1) {
#pragma unroll
    for (int i = 0; i < NBUF - 1; ++i) load_step(i, i);
    int st = 0;
    for (; st + NBUF <= n_half; st += NBUF) {
#pragma unroll
      for (int i = 0; i < NBUF; ++i) {
        load_step((i + NBUF - 1) % NBUF, st + i + NBUF - 1);
        // (left to itself the scheduler gathers the loads of several steps behind their arithmetic)
        __builtin_amdgcn_sched_barrier(0);
        multiply(i, st + i);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int i = 0; i < NBUF - 1; ++i)
      if (st + i < n_half) multiply(i, st + i);  // scalar branch around matrix instructions only
  }

  // partial sums and norms of this wave -> LDS
#pragma unroll
  for (int b = 0; b < RB; ++b) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      sPart[((wave * RB + b) * 4 + r) * 64 + lane] = NACC == 2 ? acc[b][0][r] + acc[b][NACC - 1][r] : acc[b][0][r];
  }
  {
    double v = xsq;
    if (PAIR) v += __shfl_xor(v, 8);
    v += __shfl_xor(v, 16);
    v += __shfl_xor(v, 32);
    const double root = sqrt(v);
    if (q == 0) {
      sXsq[wave * 16 + r16] = v;
      sXseg[wave * 16 + r16] = root;
    }
    if constexpr (kBf16X) {
      uint32_t key = min((uint32_t)xq.x, (uint32_t)xq.y);
      if (PAIR) key = min(key, __shfl_xor(key, 8));
      key = min(key, __shfl_xor(key, 16));
      key = min(key, __shfl_xor(key, 32));
      if (q == 0) sXq[wave * 16 + r16] = key;
    }
#pragma unroll
    for (int i = 0; i < kSegLoads; ++i)
      if (tid + i * NT < NWV * 16 * RB) sWseg[tid + i * NT] = w_seg[i];
  }
  __syncthreads();

  // thread (token t, row class rr) finishes rows rr, rr + 16, ...
  const int t = tid & 15, rr = tid >> 4;
  double xn2 = 0.0;
#pragma unroll
  for (int w = 0; w < NWV; ++w) xn2 += sXsq[w * 16 + t];
  if (rr == 0) sXn2[t] = xn2;
  int xq_t = kNoLsb;
  if constexpr (kBf16X) {
    uint32_t key = kNoKey;
#pragma unroll
    for (int w = 0; w < NWV; ++w) key = min(key, sXq[w * 16 + t]);
    xq_t = bf16_key_lsb(key);
  }
  constexpr double u53 = 1.1102230246251565e-16;
  // (the reference's additions and these in a segment, the two that join accumulators and segments; PAIR: the halves)
  const double by_segment = (double)(32 * per + (PAIR ? 5 : 4)) * u53 * 1.001;
  // what the sums differ by from the ones without roundings that the bound is made of
  const double second_order = ((double)d * u53) * ((double)d * u53) * 4.0;
  for (int r = rr; r < R && (!PAIR || t < TT); r += NT / 16) {
    const int b = r >> 4, rho = r & 15, reg = rho >> 2, qq = rho & 3;
    double a = 0.0, sums = 0.0, largest = 0.0;  // sum of |P_s| + 2 N_s (one N_s per order), largest |P_s| + N_s
#pragma unroll
    for (int w = 0; w < NWV; ++w) {
      const double n = sXseg[w * 16 + t] * sWseg[w * 16 * RB + r];
      const double p = fabs(a) + n;
      largest = fmax(largest, p);
      sums += p + n;
      double p_w = sPart[((w * RB + b) * 4 + reg) * 64 + qq * 16 + t];
      if (PAIR) p_w += sPart[(w * 4 + reg + 2) * 64 + qq * 16 + t + 8];
      a += p_w;
    }
    // the factors 1.001 cover the roundings of the norms and of the bound
    const double e = sums * by_segment + sqrt(xn2 * sWn2[r]) * second_order;
    const double lo = a - e, hi = a + e;
    bool ok;
    if (row0 + r < E) {
      const float flo = (float)lo, fhi = (float)hi;
      ok = flo == fhi && isfinite(flo);
    } else {
      const float glo = (float)(1.0 / (1.0 + exp(-lo))), ghi = (float)(1.0 / (1.0 + exp(-hi)));
      ok = glo == ghi;
    }
    if (kBf16X && !ok && w_lsb) {
      // Every product of the pair is a multiple of 2^(q_x + q_w), so with all sums below
      // 2^(q_x + q_w + 53) none rounds, segment after segment (all zeros on one side: the sum is
      // exactly 0).  (`sums` is no finite number if an operand is none.)
      const int wq = w_lsb[min(row0 + r, E)];
      if (xq_t == kNoLsb || wq == kNoLsb) {
        ok = true;
      } else {
        const int ql = xq_t + wq;
        ok = ql > -2000 && sums < INFINITY && largest * 1.001 < ldexp(1.0, ql + 53);
      }
    }
    sAcc[t * R + r] = a;
    sFlag[t * R + r] = ok ? 0 : 1;
  }
  __syncthreads();

  // Second look at the flagged sums (about one in a thousand, so about one per workgroup and
  // five in the unluckiest): the bound from their partial sums.  A sum that passes is replaced by the
  // one the bound belongs to; the others go on the other list and are looked at once more with the
  // counted unit.  The partial-sum area is free now and
  // holds the lists.  Launch, 256 rows of d = 7168, 256 bf16 tokens: 134 -> 48 us, 26 of them without
  // this look; 997 f32 tokens of a 61-row layer, d = 2048, route stage 120 -> 22 us.
  int* sList = (int*)sPart;          // [<= 16 R] flagged entries; those that want the reference's own order
  int* sList2 = sList + 16 * R;      // [<= 16 R] entries that failed the first look
  int* sUnits = sList2 + 16 * R;     // [16 R] the bound's unit, by entry
  int* sCount = sUnits + 16 * R;     // [0] flagged, [1] failed the first look, [2] the second
  constexpr int kSeqChunk = 512;     // 8 KiB: with the lists it fits the smallest partial-sum area
  double2* sSeq = (double2*)(((uintptr_t)(sCount + 3) + 15) & ~(uintptr_t)15);
  PieceSums* sPiece = (PieceSums*)sSeq;
  constexpr int kPieces = kSeqChunk * 16 / (int)sizeof(PieceSums);
  static_assert(3 * 16 * 16 * RB * 4 + 12 + 16 + kSeqChunk * 16 <= NWV * RB * 4 * 64 * 8,
                "lists and staging area must fit the partial-sum area");
  if (tid < 3) sCount[tid] = 0;
  __syncthreads();
  for (int ent = tid; ent < TT * R; ent += NT)
    if (sFlag[ent]) {
      const int ft = ent / R, fr = ent - ft * R;
      sList[atomicAdd(sCount, 1)] = ent;
      sUnits[ent] = guess_units(sAcc[ent], sqrt(sXn2[ft] * sWn2[fr]), d);
    }
  __syncthreads();
  const int pieces = (d + kPiece - 1) / kPiece;
  const int per_pass = kPieces / pieces;  // sums whose pieces the area holds
#pragma clang loop unroll(disable)
  for (int look = 0; look < 2; ++look) {
    const int* from = look ? sList2 : sList;
    int* left = look ? sList : sList2;  // (the second look's leavings go where the first one's list was)
    const int n_from = sCount[look];
    for (int i0 = 0; i0 < n_from;) {
      const int n_here = min(max(per_pass, 1), n_from - i0);
      const int n_items = per_pass ? n_here * pieces : 0;  // (0: rows of more than 170 000 columns)
#pragma clang loop unroll(disable)
      for (int it = wave; it < n_items; it += NWV) {
        const int i = it / pieces, piece = it - i * pieces;
        const int ei = from[i0 + i];
        const int ft = ei / R, fr = ei - ft * R;
        const int c = piece * kPiece + lane * 8;  // d is a multiple of 8: a chunk is whole or absent
        const bool in = c < d;
        const int cc = in ? c : 0;
        XChunk<XT> xn;
        XChunk<uint16_t> wn;  // (the bf16 copy, which the loop above has just read)
        xn.load(x + (size_t)min(t0 + ft, T - 1) * d + cc);
        wn.load(w_t8 + ((size_t)(cc >> 3) * Rp + row0 + fr) * 8);
        xn.keep(in);
        wn.keep(in);
        float xf[8], wf[8];
        xn.get(xf);
        wn.get(wf);
        visit_piece(wf, xf, sUnits[ei], sPiece + it);
      }
      __syncthreads();
      for (int i = wave; i < n_here; i += NWV) {
        const int ei = from[i0 + i];
        double a = 0.0, e = INFINITY;
        int units = sUnits[ei];
        if (n_items) pieces_bound(sPiece + i * pieces, pieces, units, a, e, units);
        const bool ok = rounds_alike(a, e, row0 + ei % R >= E);
        if (lane == 0) {
          if (ok) sAcc[ei] = a;
          else left[atomicAdd(sCount + 1 + look, 1)] = ei;
          sUnits[ei] = units;
        }
      }
      __syncthreads();
      i0 += n_here;
    }
  }
  const int n_chain = sCount[2];
  // The reference's own order for the rest: one sequential c-ascending f64 sum.  The workgroup
  // widens kSeqChunk columns at a time into LDS and one thread walks them, so each step of the
  // chain waits for an LDS read instead of two trips to L2 (d = 2048: ~10 us instead of ~115).
  for (int i = 0; i < n_chain; ++i) {
    const int ei = sList[i];
    const int ft = ei / R, fr = ei - ft * R;
    const XT* xr = x + (size_t)min(t0 + ft, T - 1) * d;
    const float* wr = row0 + fr < E ? w_router + (size_t)(row0 + fr) * d : gate_vec;
    double a = 0.0;
    for (int c0 = 0; c0 < d; c0 += kSeqChunk) {
      const int n = min(kSeqChunk, d - c0);
      for (int c = tid; c < n; c += NT)
        sSeq[c] = double2{(double)wr[c0 + c], (double)load_x(xr, c0 + c)};
      __syncthreads();
      if (tid == 0) {
#pragma unroll 8
        for (int c = 0; c < n; ++c) a = fma(sSeq[c].x, sSeq[c].y, a);
      }
      __syncthreads();
    }
    if (tid == 0) sAcc[ei] = a;
  }
  if (n_chain) __syncthreads();

  for (int ent = tid; ent < TT * R; ent += NT) {
    const int ft = ent / R, fr = ent - ft * R;
    const double a = sAcc[ent];
    if (row0 + fr < E) {
      float logit = (float)a;
      if (bias) logit = logit + bias[row0 + fr];
      sLogit[ent] = logit;
      if (logits_out && t0 + ft < T) logits_out[(size_t)(t0 + ft) * E + row0 + fr] = logit;
    } else if (t0 + ft < T) {
      sgate_out[t0 + ft] = (float)(1.0 / (1.0 + exp(-a)));
    }
  }
  if (logits_out) return;  // routing is decided by another launch from the logits
  __syncthreads();
  if (E <= 64) {
    // Softmax and top-k with lane r = expert r, a wave taking the tokens wave, wave + NWV, ...
    // Same arithmetic, casts and order as softmax_topk (and wave_softmax_topk in select_wave.h);
    // what is laid out for speed is the two loops of 64 steps: the reference's sequential fold
    // of the exponentials is run for all 16 tokens at once by 16 lanes reading LDS, and the
    // selection takes k maxima over the wave instead of ranking every expert against every
    // other.
    constexpr int TPW = TT / NWV;
    double* sExp = smem_m;            // [16][64]: the partial-sum area again
    double* sInv = sExp + TT * 64;    // [16]
    static_assert((TT * 64 + TT) * 8 <= NWV * RB * 4 * 64 * 8, "softmax scratch must fit");
    const bool on = lane < E;
    double ex[TPW];
#pragma unroll
    for (int j = 0; j < TPW; ++j) {
      const int tk = wave + j * NWV;
      const float my = on ? sLogit[tk * R + lane] : -INFINITY;
      // a NaN logit is skipped, as f32::max skips it
      const float mx = wave_max_f32(fmaxf(-INFINITY, my));
      ex[j] = on ? exp((double)(my - mx)) : 0.0;  // f32 subtraction, then f64 exp
      sExp[tk * 64 + lane] = ex[j];
    }
    __syncthreads();
    if (tid < TT) {
      const double* xe = sExp + tid * 64;
      double sum = 0.0;
      for (int e0 = 0; e0 < E; e0 += 8) {  // sequential fold, e ascending; the padding adds +0
#pragma unroll
        for (int u = 0; u < 8; ++u) sum += xe[e0 + u];
      }
      sInv[tid] = sum > 0.0 ? 1.0 / sum : 0.0;
    }
    __syncthreads();
    float wt[TPW];
    int token[TPW];
    bool valid[TPW];
#pragma unroll
    for (int j = 0; j < TPW; ++j) {
      const int tk = wave + j * NWV;
      token[j] = t0 + tk;
      valid[j] = token[j] < T;  // wave-uniform
      wt[j] = (float)(ex[j] * sInv[tk]);
      if (valid[j] && on && (!isfinite(wt[j]) || wt[j] < 0.f)) {
        atomicMin(&status[0], -3);
        atomicMin(&status[1], (token[j] << 10) | lane);
      }
    }
    wave_topk_write_n<TPW>(wt, on, lane, k, renorm, token, valid, idx_out, w_out);
    return;
  }
  // the partial-sum area is free now: softmax scratch
  double* sExp = smem_m;                          // [16][E]
  double* sTok = sExp + 16 * E;                   // [16]
  float* sWt = (float*)(sTok + 16);               // [16][E]
  uint8_t* sSel = (uint8_t*)(sWt + 16 * E);       // [16][E]
  softmax_topk_block(TT, R, E, k, renorm, t0, T, sLogit, sExp, sWt, sSel, sTok, idx_out, w_out,
                     status);
}

template <typename XT, int RB, int NBUF, int NWV, bool PAIR = false>
hipError_t launch_router_mfma_rb(const RouterArgs& a, int R, hipStream_t s) {
  const size_t smem = ((size_t)NWV * RB * 4 * 64 + NWV * 16 + (size_t)16 * R + 16 + R + NWV * 16 + NWV * 16 * RB) * 8 +
                      (size_t)16 * R * 4 + (size_t)NWV * 16 * 4 + (size_t)16 * R + 16;
  if (smem > 64 * 1024 || 16 * RB > a.w_rows_pad) return hipErrorInvalidValue;
  // (The selection stays inside this kernel, four tokens per wave: with the logits in HBM and a
  // second launch that gives every token a wave of its own the route stage measured 3-8 us
  // longer at 8192-16384 tokens.)
  constexpr int TT = PAIR ? 8 : 16;
  router_mfma_kernel<XT, RB, NBUF, NWV, PAIR><<<(a.T + TT - 1) / TT, 64 * NWV, smem, s>>>(
      (const XT*)a.x, a.T, a.d, a.E, a.k, a.renorm, a.w_router, a.router_bias, a.shared_gate,
      a.idx, a.w, a.sgate, a.status, nullptr, a.w_lsb_min, a.w_t8, a.w_rows_pad, a.w_norm2, a.xb, a.d_pad);
  return hipGetLastError();
}

// (defined further down: selection from logits in HBM with one thread per expert, up to 256 experts)
constexpr int kSelectThreads = 256;
__global__ __launch_bounds__(kSelectThreads) void softmax_select_kernel(
    const float* __restrict__ logits, int T, int E, int k, int renorm,
    int32_t* __restrict__ idx_out, float* __restrict__ w_out, int32_t* __restrict__ status,
    FusedGrouping fg);

// The same kernel with the rows dealt to workgroups in blocks of 16 (eight waves split k), the
// logits left in HBM and the routing decided by a second launch, one wave per token: with many
// rows and a batch that gives fewer workgroups of 16 tokens than the chip has compute units,
// four times as many workgroups of a quarter of the length.
template <typename XT, bool PAIR>
hipError_t launch_router_mfma_rows(const RouterArgs& a, int R, hipStream_t s) {
  constexpr int NWV = 8, RB = 1, RL = 16, TT = PAIR ? 8 : 16;
  const size_t smem = ((size_t)NWV * RB * 4 * 64 + NWV * 16 + (size_t)16 * RL + 16 + RL + NWV * 16 + NWV * 16 * RB) * 8 +
                      (size_t)16 * RL * 4 + (size_t)NWV * 16 * 4 + (size_t)16 * RL + 16;
  if ((R + 15) / 16 * 16 > a.w_rows_pad) return hipErrorInvalidValue;
  router_mfma_kernel<XT, RB, 4, NWV, PAIR><<<dim3((a.T + TT - 1) / TT, (R + TT - 1) / TT), 64 * NWV, smem, s>>>(
      (const XT*)a.x, a.T, a.d, a.E, a.k, a.renorm, a.w_router, a.router_bias, a.shared_gate,
      a.idx, a.w, a.sgate, a.status, a.logits_out ? a.logits_out : a.logits_tmp, a.w_lsb_min,
      a.w_t8, a.w_rows_pad, a.w_norm2, a.xb, a.d_pad);
  return hipGetLastError();
}
// Eight rows by eight tokens while the launch has one such workgroup to a compute unit or less: four times as
// many of half the length.  16 x 16 / 8 x 8, launch, caches cold, us: 61 rows, d = 2048, T = 33 12.0 / 9.6, 128 12.1 / 8.7,
// 256 11.8 / 9.0, 300 12.1 / 13.3; f32 activations T = 48 14.3 / 11.8, 256 15.2 / 12.7; 256 rows, d = 7168, T = 16 30.0 / 19.5, 64
// 33.9 / 22.3, 100 36.0 / 35.1; 33 rows, d = 4096, T = 256 18.1 / 12.2; 32 rows, with the selection, T = 192 to 500: d = 2048 14.0 / 11.3,
// f32 16.5 / 13.2, d = 4096 20.0 / 14.3, d = 7168 32.3 / 21.3.
bool router_split_by_eight(const RouterArgs& a, int R) {
  constexpr int n_cus = 256;
  return (long long)((a.T + 7) / 8) * ((R + 7) / 8) <= n_cus;
}
template <typename XT>
hipError_t launch_router_mfma_split(const RouterArgs& a, int R, bool by_eight, hipStream_t s) {
  const hipError_t e = by_eight ? launch_router_mfma_rows<XT, true>(a, R, s) : launch_router_mfma_rows<XT, false>(a, R, s);
  if (e != hipSuccess || a.logits_out) return e;  // the caller's own launch routes from the logits
  if (a.E <= 64) {
    constexpr int per = kWaveSelectThreads / 64;
    wave_select_kernel<<<(a.T + per - 1) / per, kWaveSelectThreads, 0, s>>>(
        a.logits_tmp, a.T, a.E, a.k, a.renorm, a.idx, a.w, a.status);
  } else {
    const int TT = kSelectThreads / a.E;
    softmax_select_kernel<<<(a.T + TT - 1) / TT, kSelectThreads, 0, s>>>(
        a.logits_tmp, a.T, a.E, a.k, a.renorm, a.idx, a.w, a.status, FusedGrouping{});
  }
  return hipGetLastError();
}

// Up to 80 rows, d a multiple of 8, routing decided in the same launch, no bf16 copy of x to
// write (bf16 activations of unpadded width: the store would sit in the loop).
bool router_mfma_ok(const RouterArgs& a, int R) {
  static const bool off = [] {
    const char* e = getenv("ATENIA_MOE_ROUTER_MFMA");  // tuning knob: 0 = sequential chains
    return e && atoi(e) == 0;
  }();
  // Against the sequential kernel (route stage, us): 8 rows, d = 4096: T = 4096 32 / 57-75,
  // 8192 48 / 89, 16384 89 / 160; 61-64 rows, d = 2048: T = 4096 59 / 92-97, 8192 86 / 87,
  // 12288 127 / 178, 16384 155 / 180: at every batch size.
  // Only with router rows whose f32 values fit bf16: of the products of two f32 values nearly every
  // one rounds, and the sums that the second look then leaves cost a sequential chain each.
  // f32 activations (the block and host entry points of bf16 and int8 layers) take it with the bf16
  // copy of x stored on the way, if the steps of 32 columns cover the copy's padding.
  const bool rows = a.x_is_bf16 ? !a.xb : a.xb && a.d_pad <= (a.d + 31) / 32 * 32;
  const bool operands = !off && a.d % 8 == 0 && rows &&
                        a.w_fits_bf16 && a.w_t8 && a.w_norm2 && a.E >= a.k;
  if (R < 0) return operands;  // the form that deals the rows to workgroups takes any row count
  return operands && R <= 80 && !a.logits_out;
}

// When the rows are dealt to workgroups.  Measured on MI355X, d = 2048, route stage in us,
// split / one workgroup per 16 tokens: 64 rows T = 600 26 / 54, 1024 25 / 54, 2048 36 / 57,
// 3072 57 / 58, 4096 64 / 59, 8192 116 / 87; 32 rows T = 1024 24 / 29, 2048 25 / (29-32),
// 4096 37 / 32; 48 rows, d = 4096, T = 2048 54 / 81.  Against the per-token kernel, 32 rows: T = 128 23 / 20, 512 23 / 35.
// More than 32 rows: where the per-token kernel's workgroups (four rows of one token) stand two to a compute unit, or
// some way into that where the matrix cores' launch is the longer one (f32 activations, the longest rows).  Launch and selection,
// caches cold, us, per-token / eight rows by eight tokens (T, workgroups of the former):
//   bf16  61 rows, d = 2048 T = 17 (272) 13.6 / 11.5; 34, d = 3072 29 (261) 13.7 / 12.7; 48, d = 4096 20 (240) 13.4 / 14.1, 22 (264) 14.7 /
//         14.1, 50 22.3 / 14.3; 60, d = 5120 18 (270) 17.1 / 15.9; 36, d = 6144 29 (261) 17.0 / 17.2; 64, d = 7168 15 (240) 18.8 / 20.3, 17
//         (272) 21.2 / 20.2; 40, d = 8192 26 (260) 20.0 / 21.5, 28 (280) 21.5 / 22.7, 29 (290) 22.9 / 21.9; 256, d = 7168 T = 4 19.9 / 18.4
//   f32   61 rows, d = 2048 T = 17 (272) 13.8 / 12.7; 34, d = 3072 30 (270) 13.9 / 14.2, 34 (306) 15.6 / 14.3; 48, d = 4096 22 (264) 15.1 /
//         16.1, 24 (288) 15.9 / 16.3, 29 (348) 16.5 / 16.2; 60, d = 5120 18 (270) 17.5 / 17.9, 22 (330) 18.5 / 18.4; 36, d = 6144 29 (261) 16.7 /
//         19.1, 34 (306) 20.0 / 19.9; 40, d = 7168 26 (260) 17.2 / 21.1, 30 (300) 22.0 / 21.2; 64, d = 7168 17 (272) 20.5 / 22.6, 19 (304) 23.1 / 21.4;
//         40, d = 8192 26 (260) 20.1 / 26.0, 30 (300) 22.5 / 24.6, 34 (340) 23.7 / 24.1, 37 24.7 / 24.2; 200, d = 4096 6 (300) 31.2 / 33.8
bool router_mfma_split_wanted(const RouterArgs& a, int R) {
  constexpr int max_t = 2048;
  // (with many rows the per-token kernel serves a few tokens only, launch_router: 256 rows,
  // d = 7168, 16 tokens: 36 us / 230 for the sequential-order kernel)
  constexpr int n_cus = 256;
  const int line = n_cus + (a.d > 2048 && !a.x_is_bf16 ? 48 : 0) + (a.d > 7168 ? 32 : 0);
  const bool two_each = a.token_max_is_set ? a.T > std::min(a.token_kernel_max_tokens, 51)  // (the line it had beside that one)
                                           : (long long)a.T * ((R + 3) / 4) > line;
  const int lo = R > 64 && (long long)a.T * R * a.d > kTokenMaxWork ? 1 : R > 32 ? (two_each ? 1 : INT_MAX) : 192;
  if (R <= 16 || a.T < lo || !router_mfma_ok(a, -1)) return false;
  // The raw logits are wanted (another launch routes), or more rows than one workgroup holds:
  // no other form on the matrix cores, so at every batch size (256 rows, d = 7168, logits for the
  // group-limited selection, T = 2048: 354 us / 316 for the sequential-order kernel, 4096 626 / 645,
  // 8192 1172 / 1302, before the second look at flagged sums became cheaper: T = 1500 352 -> 160).
  // Several blocks of 16 tokens per workgroup, to read the 7 MB matrix less often, and two or
  // four row blocks per workgroup, to read the tokens less often, both measured no faster.
  if (a.logits_out) return true;
  if (!a.logits_tmp || a.E > kSelectThreads) return false;
  return R > 80 || a.T <= max_t;
}

// Up to eight rows: the form of eight tokens against the per-token kernel, from where that has a second workgroup on some
// compute units.  8 rows, per-token / this, launch inside the layer, us: d = 4096, T = 10 8.4 / 13.2, 64 11.6 / 13.2, 333 24.6 /
// 16.5; launch alone, caches cold, bf16 and f32 activations: d = 2048 T = 257 10.9 / 8.7, 12.2 / 11.0; d = 4096 257 13.4 / 11.6, 15.0 / 14.1, 288 15.9 /
// 11.5, 18.2 / 14.3; d = 6144 257 16.5 / 15.5, 19.0 / 19.5, 264 17.7 / 15.4, 20.1 / 18.5; 4 rows, d = 8192 257 17.4 / 18.5, 20.1 / 21.5, 264 19.4 / 18.5,
// 21.4 / 21.4, 288 21.5 / 18.5, 23.3 / 21.5.
bool router_eight_from(const RouterArgs& a) {
  constexpr int more_than_one_each = 256 + 8;
  return a.T >= more_than_one_each;
}
// ... and against the one of 16 tokens, which has half as many workgroups and takes 1.1 (d = 256), 1.7 (d = 1024) to 1.9 times (d =
// 4096) as long for a round of 256 of them: in its first round, and where one more of the others gives less than half a round to it.
// Launch alone, caches cold, us, 16 tokens / 8:
//   bf16  d = 1024 T = 1024 9.3 / 7.1, 2100 9.3 / 9.5, 6000 13.9 / 12.1, 8192 14.0 / 15.5, 10240 18.9 / 18.7, 13500 23.3 / 24.2; d = 2048 2000 12.2 / 8.8,
//         2100 12.2 / 12.5, 6000 19.9 / 16.9, 8192 19.9 / 21.2, 10240 29.1 / 27.8; d = 4096 2000 19.8 / 13.5, 2100 19.8 / 18.7, 4000 19.8 / 19.1, 6000 32.8 /
//         27.7, 8192 33.7 / 34.5, 10240 46.6 / 41.4, 13500 58.7 / 54.7, 16384 57.6 / 60.5; d = 256 1024 7.0 / 6.4, 6000 9.1 / 10.3
//   f32   d = 1024 T = 1024 11.8 / 8.9, 2100 12.1 / 13.2, 6000 21.3 / 21.8, 8192 22.9 / 28.5; d = 2048 2000 17.1 / 13.6, 6000 29.6 / 30.6, 8192 32.8 / 40.2; d = 4096 2000
//         23.2 / 16.9, 2100 23.4 / 25.4, 6144 49.9 / 47.3, 8192 48.1 / 54.8, 8500 69.8 / 67.3, 10240 72.6 / 73.0; d = 6144 6000 62.0 / 53.3, 8500 97.7 / 93.4,
//         13500 136.9 / 133.7, 16384 149 / 158
bool router_eight_pays(const RouterArgs& a) {
  const int rounds = (a.T + 8 * 256 - 1) / (8 * 256);
  const int most = a.d >= (a.x_is_bf16 ? 4096 : 6144) ? 7 : a.d >= (a.x_is_bf16 ? 1024 : 4096) ? 5 : 1;
  return rounds == 1 || ((rounds & 1) && rounds <= most);
}

template <typename XT>
hipError_t launch_router_mfma(const RouterArgs& a, int R, bool by_eight, hipStream_t s) {
  // few rows: eight waves split k, so that a batch of 4096 tokens (256 workgroups, one per
  // compute unit) still puts two waves on every SIMD
  if (by_eight) return launch_router_mfma_rb<XT, 1, 4, 8, true>(a, R, s);
  if (R <= 16) return launch_router_mfma_rb<XT, 1, 4, 8>(a, R, s);
  if (R <= 32) return launch_router_mfma_rb<XT, 2, 3, 8>(a, R, s);
  if (R <= 48) return launch_router_mfma_rb<XT, 3, 3, 4>(a, R, s);
  if (R <= 64) return launch_router_mfma_rb<XT, 4, 3, 4>(a, R, s);
  return launch_router_mfma_rb<XT, 5, 3, 4>(a, R, s);
}

template <typename XT>
hipError_t dispatch_router_batch(const RouterArgs& a, int R, hipStream_t s) {
  if (R <= 16) return launch_router_batch<XT, 1, 1, 128>(a, s);
  if (R <= 32) return launch_router_batch<XT, 2, 1, 64>(a, s);
  // Many rows and many tokens: a thread takes two tokens as well (each w value read from LDS
  // serves two chains, eight independent f64 chains per thread) while the grid still covers
  // the chip.
  // measured on MI355X at 64 rows, d = 2048: two tokens per thread pay from 8192 tokens on
  const long long work = (long long)a.T * ((R + 63) / 64);  // row blocks count like more tokens
  const int tpt = work >= 8192 ? 2 : 1;
  if (tpt >= 2) return launch_router_batch<XT, 4, 2, 64>(a, s);
  return launch_router_batch<XT, 4, 1, 64>(a, s);
}

// The expert grouping of ONE token from its selection flags (what kernel 2 would produce).
// Called by the threads e = 0..E-1 of the workgroup (sel in LDS, already synchronised): thread e
// counts the selected experts before it and writes its own entries.
__device__ inline void write_single_token_grouping(const FusedGrouping& fg, const int32_t* sel,
                                                   int e, int E, int k) {
  if (e >= E) return;
  int run = 0, total = 0;
#pragma unroll 8
  for (int o = 0; o < E; ++o) {
    const int c = sel[o] ? 1 : 0;
    run += o < e ? c : 0;
    total += c;
  }
  const int c = sel[e] ? 1 : 0;
  fg.counts[e] = c;
  fg.offsets[e] = run;
  if (c && run < k) {
    fg.active[run] = e;
    fg.perm[run] = run;
    fg.inv[run] = run;
    int32_t* tile = fg.tiles + 4 * run;
    tile[0] = e;
    tile[1] = run;
    tile[2] = 1;
    tile[3] = 0;
  }
  if (e == 0) {
    fg.offsets[E] = total;
    *fg.n_active = total;
    *fg.n_tiles = total;
    fg.shared_offsets[0] = 0;
    fg.shared_offsets[1] = 1;
  }
}

// Softmax + top-k from logits that another launch left in HBM: used when the rows of the
// router matrix were spread over several workgroups per token (many experts, few tokens), so
// no single workgroup holds all logits of a token.  256 / E tokens per workgroup.
__global__ __launch_bounds__(kSelectThreads) void softmax_select_kernel(
    const float* __restrict__ logits, int T, int E, int k, int renorm,
    int32_t* __restrict__ idx_out, float* __restrict__ w_out, int32_t* __restrict__ status,
    FusedGrouping fg) {
  __shared__ double sExp[kSelectThreads];
  __shared__ float sWt[kSelectThreads], sLg[kSelectThreads];
  __shared__ int32_t sSel[kSelectThreads];
  const int TT = kSelectThreads / E;
  const int tid = threadIdx.x;
  const int tl = tid / E, r = tid - tl * E;
  const int t = blockIdx.x * TT + tl;
  const bool on = tl < TT && t < T;
  const int ts = on ? t : 0, ls = on ? tl : 0;
  sLg[tid] = on ? logits[(size_t)t * E + r] : 0.f;  // one coalesced read; the folds walk LDS
  __syncthreads();
  softmax_topk(on, r, E, k, renorm, ts, sLg + ls * E, sExp + ls * E, sWt + ls * E, sSel + ls * E,
               idx_out, w_out, status);
  if (fg.counts) {  // T == 1: the workgroup holds token 0 only
    __syncthreads();
    write_single_token_grouping(fg, sSel, tid, E, k);
  }
}

// What the per-token kernel needs after its sums are settled.  Its first argument, read from the argument
// segment when the sums are there: read with the rest at the kernel's start these registers were put aside
// (37 of them, in lanes of a vector register) past the second look (8 rows, d = 4096, one token:
// 9.7 -> 9.4 us).
struct RouterLate {
  const float* bias;
  int32_t* idx;
  float* w;
  float* sgate;
  int32_t* status;
  float* logits;
  int k, renorm;
  FusedGrouping fg;
};
typedef const __attribute__((address_space(4))) RouterLate* RouterLatePtr;

template <typename XT>
__global__ __launch_bounds__(kTokenThreads) void router_token_kernel(
    RouterLate, const XT* __restrict__ x, int T, int d, int E, const float* __restrict__ w_router,
    const float* __restrict__ gate_vec, uint16_t* __restrict__ xb, int d_pad) {
  // gridDim.y > 1 (only when the logits go to `logits_out`): this workgroup computes rows
  // row_lo .. row_lo + R - 1 of the stacked matrix; otherwise all of them.
  const int R_all = E + (gate_vec ? 1 : 0);
  const int rows_per_block = (R_all + gridDim.y - 1) / gridDim.y;
  const int row_lo = blockIdx.y * rows_per_block;
  const int R = min(rows_per_block, R_all - row_lo);
  const int t = blockIdx.x;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  constexpr int NW = kTokenThreads / 64;

  // (the token first: its place is then 16-byte aligned whatever R and E are, and four values are one read:
  // 9.4 -> 8.5 us for that launch)
  extern __shared__ float4 smem_f4[];
  float* sX = (float*)smem_f4;                 // [d]
  double* sAcc = (double*)(smem_f4 + (d + 3) / 4);  // [R]
  double* sExp = sAcc + R;                     // [E]
  double* sPart = sExp + E;                    // [max(R, NW)]
  double* sPartA = sPart + (R > NW ? R : NW);  // [max(R, NW)]
  PieceSums* sPiece = (PieceSums*)(sPartA + (R > NW ? R : NW));  // [pieces of a row]
  float* sLogit = (float*)(sPiece + (d + kPiece - 1) / kPiece);  // [E]
  float* sWt = sLogit + E;                     // [E]
  int32_t* sSel = (int32_t*)(sWt + E);         // [E]
  int32_t* sBad = sSel + E;                    // [3]: second look wanted, sequential order wanted, -g
  int32_t* sNeed = sBad + 3;                   // [R]

  if (tid < 2) sBad[tid] = 0;
  // Work items: (row, k slice).  With few rows each row is split over several waves so that
  // all 16 waves stream the router matrix.  Partial results meet in LDS; under the interval
  // certificate below their order of addition cannot change what the sum rounds to.
  const int KS = R >= NW ? 1 : NW / R;              // k slices per row
  const int slice = ((d + KS - 1) / KS + 3) & ~3;   // multiple of 4 for float4 loads
  const bool vec_ok = (d & 3) == 0;
  const int c_end = xb ? (d_pad > d ? d_pad : d) : d;
  for (int c = tid; c < c_end; c += kTokenThreads) {
    float v = c < d ? load_x(x, (size_t)t * d + c) : 0.f;
    if (c < d) sX[c] = v;
    if (xb && blockIdx.y == 0 && c < d_pad) xb[(size_t)t * d_pad + c] = f32_to_bf16_rne(v);
  }
  __syncthreads();

  for (int item = wave; item < R * KS; item += NW) {
    const int r = item / KS, ksl = item - r * KS;
    const float* wr = row_lo + r < E ? w_router + (size_t)(row_lo + r) * d : gate_vec;
    const int c_lo = ksl * slice, c_hi = min(d, c_lo + slice);
    double acc = 0.0, asum = 0.0;
    auto one = [&](float wv, float xv) {
      double wd = (double)wv, xd = (double)xv;
      acc = fma(wd, xd, acc);
      asum = fma(fabs(wd), fabs(xd), asum);
    };
    if (vec_ok) {
#pragma unroll 4
      for (int c = c_lo + lane * 4; c < c_hi; c += 256) {
        float4 w4 = *(const float4*)(wr + c);
        const float4 x4 = *(const float4*)(sX + c);
        one(w4.x, x4.x);
        one(w4.y, x4.y);
        one(w4.z, x4.z);
        one(w4.w, x4.w);
      }
    } else {
      for (int c = c_lo + lane; c < c_hi; c += 64) one(wr[c], sX[c]);
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      acc += __shfl_xor(acc, off);
      asum += __shfl_xor(asum, off);
    }
    if (lane == 0) {
      sPart[item] = acc;
      sPartA[item] = asum;
    }
  }
  __syncthreads();
  if (tid < R) {
    double acc = 0.0, asum = 0.0;
    for (int ksl = 0; ksl < KS; ++ksl) {
      acc += sPart[tid * KS + ksl];
      asum += sPartA[tid * KS + ksl];
    }
    bool exact;
    {
      // The certificate: any order of d exact products summed in f64 lands within
      // g = d * 2^-53 * sum|p| of the true sum (standard bound, 1 / (1 - d u) absorbed by the
      // margin; asum's own relative error of d * 2^-53 likewise), so this sum and the
      // reference's sequential one differ by at most 2 g.  If both ends of [acc - 2g, acc + 2g]
      // round to the same f32 (the same f32 sigmoid for the gate row), the reference's result is
      // that value, whatever its order.  Rounding is monotone; the two extra units of 2^-53
      // cover the roundings of acc -/+ e themselves.  About one sum in a thousand sits close
      // enough to an f32 rounding boundary to fail this; those rows get the second look below.
      const double e = asum * ((double)(2 * d + 4) * 1.1102230246251565e-16) * 1.0001;
      const double lo = acc - e, hi = acc + e;
      if (row_lo + tid < E) {
        const float flo = (float)lo, fhi = (float)hi;
        exact = flo == fhi && isfinite(flo);
      } else {
        const float glo = (float)(1.0 / (1.0 + exp(-lo))), ghi = (float)(1.0 / (1.0 + exp(-hi)));
        exact = glo == ghi;
      }
    }
    sAcc[tid] = acc;
    sNeed[tid] = exact ? 0 : 1;
    if (!exact) {
      sPartA[tid * KS] = asum;  // this thread's own entries: nobody else reads them
      sBad[0] = 1;
    }
  }
  __syncthreads();
  if (sBad[0]) {
    // Second look, for the flagged rows only: the bound from their partial sums.  (48 f32 rows of the
    // 65-row router, d = 2048: 42.5 -> 17.5 us for the launch, against asking only whether a row's sum
    // is exact in every order.)
    const int pieces = (d + kPiece - 1) / kPiece;
#pragma clang loop unroll(disable)
    for (int r = 0; r < R; ++r) {
      if (!sNeed[r]) continue;  // the same for every thread
      const float* wr = row_lo + r < E ? w_router + (size_t)(row_lo + r) * d : gate_vec;
      int units = guess_units(sAcc[r], sPartA[r * KS], d);
#pragma clang loop unroll(disable)
      for (int look = 0; look < 2; ++look) {
#pragma clang loop unroll(disable)
        for (int piece = wave; piece < pieces; piece += NW) {
          const int c = piece * kPiece + lane * 8;
          float w[8], xv[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const bool in = c + i < d;
            w[i] = wr[in ? c + i : 0];
            xv[i] = sX[in ? c + i : 0];
            w[i] = in ? w[i] : 0.f;
            xv[i] = in ? xv[i] : 0.f;
          }
          visit_piece(w, xv, units, sPiece + piece);
        }
        __syncthreads();
        if (wave == 0) {
          double a, e;
          int counted;
          pieces_bound(sPiece, pieces, units, a, e, counted);
          const bool ok = rounds_alike(a, e, row_lo + r >= E);
          if (lane == 0) {
            if (ok) {
              sAcc[r] = a;
              sNeed[r] = 0;
            } else if (look) {
              sBad[1] = 1;
            }
            sBad[2] = counted;
          }
        }
        __syncthreads();
        if (!sNeed[r]) break;
        units = sBad[2];
      }
    }
  }
  if (sBad[1]) {
    // The reference's own order: one sequential c-ascending f64 sum per row.
    for (int r = tid; r < R; r += kTokenThreads) {
      const float* wr = row_lo + r < E ? w_router + (size_t)(row_lo + r) * d : gate_vec;
      double acc = 0.0;
      for (int c = 0; c < d; ++c) acc = fma((double)wr[c], (double)sX[c], acc);
      sAcc[r] = acc;
    }
    __syncthreads();
  }
  RouterLatePtr late = (RouterLatePtr)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(late));  // (not before this point)
  const float* bias = late->bias;
  float* logits_out = late->logits;
  if (tid < R) {
    double acc = sAcc[tid];
    const int gr = row_lo + tid;
    if (gr < E) {
      float logit = (float)acc;
      if (bias) logit = logit + bias[gr];
      sLogit[tid] = logit;  // indexed by expert when the workgroup holds all rows (row_lo == 0)
      if (logits_out) logits_out[(size_t)t * E + gr] = logit;
    } else {
      late->sgate[t] = (float)(1.0 / (1.0 + exp(-acc)));
    }
  }
  __syncthreads();
  if (logits_out) return;  // routing is decided by another kernel from the raw logits
  const int k = late->k;
  softmax_topk(tid < E, tid, E, k, late->renorm, t, sLogit, sExp, sWt, sSel, late->idx, late->w, late->status);
  FusedGrouping fg;
  fg.counts = late->fg.counts;
  if (fg.counts) {  // T == 1: the grouping of a single token follows from its top-k
    __syncthreads();
    fg.offsets = late->fg.offsets; fg.perm = late->fg.perm; fg.inv = late->fg.inv;
    fg.active = late->fg.active; fg.n_active = late->fg.n_active;
    fg.shared_offsets = late->fg.shared_offsets; fg.tiles = late->fg.tiles; fg.n_tiles = late->fg.n_tiles;
    write_single_token_grouping(fg, sSel, tid, E, k);
  }
}

}  // namespace

static size_t token_smem(const RouterArgs& a, int R) {
  const size_t np = R > kTokenThreads / 64 ? R : kTokenThreads / 64;
  return ((size_t)R + a.E + 2 * np) * 8 + (size_t)((a.d + kPiece - 1) / kPiece) * sizeof(PieceSums) +
         (size_t)((a.d + 3) / 4) * 16 + (size_t)a.E * 12 + 12 + (size_t)R * 4 + 16;
}

RouterForm router_form(const RouterArgs& a) {
  const int R = a.E + (a.shared_gate ? 1 : 0);
  // The per-token kernel re-reads the whole stacked matrix for every token; with many rows
  // (row blocks, logits mode) that only pays for a handful of tokens.
  if (router_mfma_split_wanted(a, R)) return router_split_by_eight(a, R) ? kRouterSplit8 : kRouterSplit;
  const bool mfma = router_mfma_ok(a, R), eight = mfma && R <= 8;
  if (a.T <= a.token_kernel_max_tokens && (a.token_max_is_set || !(eight && router_eight_from(a))) &&
      (R <= 64 || (long long)a.T * R * a.d <= kTokenMaxWork) && token_smem(a, R) <= 64 * 1024)
    return kRouterToken;
  return !mfma ? kRouterChains : eight && router_eight_pays(a) ? kRouterMfma8 : kRouterMfma;
}

hipError_t launch_router(const RouterArgs& a, hipStream_t s, int* fused_permute) {
  const int R = a.E + (a.shared_gate ? 1 : 0);
  if (fused_permute) *fused_permute = 0;
  if (R > kMaxRouterRows || a.T <= 0) return hipErrorInvalidValue;
  const RouterForm form = router_form(a);
  if (form == kRouterSplit || form == kRouterSplit8)
    return a.x_is_bf16 ? launch_router_mfma_split<uint16_t>(a, R, form == kRouterSplit8, s)
                       : launch_router_mfma_split<float>(a, R, form == kRouterSplit8, s);
  if (form == kRouterToken) {
    const size_t smem = token_smem(a, R);
    // Many rows, few tokens: one workgroup per token would stream the whole stacked matrix
    // through a single CU.  The rows are spread over workgroups instead (four rows each, a
    // row split over four waves), the logits go to HBM, and the selection runs as a second,
    // tiny launch -- the caller's own one (logits_out) or softmax_select_kernel here.
    // Measured (61-65 rows, d = 2048): spread 29 / 30 / 35 / 46 us at T = 33 / 48 / 64 / 96
    // against 40-43 us for one workgroup per token, so the rows are spread up to 64 tokens.
    const bool spread = R > 32 && (a.logits_out || (a.logits_tmp && a.T <= 64 &&
                                                    a.E <= kSelectThreads));
    float* lg = a.logits_out ? a.logits_out : (spread ? a.logits_tmp : nullptr);
    FusedGrouping fg{};
    if (a.T == 1 && a.fuse_permute && !a.logits_out) {
      const PermuteArgs& pa = *a.fuse_permute;
      fg = FusedGrouping{pa.counts, pa.offsets, pa.perm, pa.inv, pa.active, pa.n_active,
                         pa.shared_offsets, (int32_t*)pa.tiles, pa.n_tiles};
      if (fused_permute) *fused_permute = 1;
    }
    const FusedGrouping fg_token = spread ? FusedGrouping{} : fg;
    const int row_blocks = spread ? (R + 3) / 4 : 1;
    const dim3 grid(a.T, row_blocks);
    const RouterLate late{a.router_bias, a.idx, a.w, a.sgate, a.status, lg, a.k, a.renorm, fg_token};
    if (a.x_is_bf16)
      router_token_kernel<uint16_t><<<grid, kTokenThreads, smem, s>>>(
          late, (const uint16_t*)a.x, a.T, a.d, a.E, a.w_router, a.shared_gate, a.xb, a.d_pad);
    else
      router_token_kernel<float><<<grid, kTokenThreads, smem, s>>>(
          late, (const float*)a.x, a.T, a.d, a.E, a.w_router, a.shared_gate, a.xb, a.d_pad);
    if (spread && !a.logits_out && a.defer_select && a.T == 1 && a.E <= 64 && fg.counts) {
      // the caller's next launch routes the token itself from the logits (select_wave.h)
      if (fused_permute) *fused_permute = 2;
      return hipGetLastError();
    }
    if (spread && !a.logits_out) {
      hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
      if (a.E <= 64 && !fg.counts) {  // one wave per token
        constexpr int per = kWaveSelectThreads / 64;
        wave_select_kernel<<<(a.T + per - 1) / per, kWaveSelectThreads, 0, s>>>(
            lg, a.T, a.E, a.k, a.renorm, a.idx, a.w, a.status);
        return hipGetLastError();
      }
      const int TT = kSelectThreads / a.E;
      softmax_select_kernel<<<(a.T + TT - 1) / TT, kSelectThreads, 0, s>>>(
          lg, a.T, a.E, a.k, a.renorm, a.idx, a.w, a.status, fg);
    }
    return hipGetLastError();
  }
  if (form == kRouterMfma || form == kRouterMfma8)
    return a.x_is_bf16 ? launch_router_mfma<uint16_t>(a, R, form == kRouterMfma8, s)
                       : launch_router_mfma<float>(a, R, form == kRouterMfma8, s);
  // Up to 64 rows per workgroup; more rows only when the logits leave the kernel (row blocks).
  if ((R <= 64 || a.logits_out) && a.d % 4 == 0 && (!a.xb || a.d_pad % 4 == 0)) {
    return a.x_is_bf16 ? dispatch_router_batch<uint16_t>(a, R, s)
                       : dispatch_router_batch<float>(a, R, s);
  }
  // More than 64 rows with softmax routing: the same row-block launch into the scratch logits,
  // then the selection as a second launch.
  if (a.logits_tmp && a.E <= kSelectThreads && a.d % 4 == 0 && (!a.xb || a.d_pad % 4 == 0)) {
    RouterArgs b = a;
    b.logits_out = a.logits_tmp;
    hipError_t e = a.x_is_bf16 ? dispatch_router_batch<uint16_t>(b, R, s)
                               : dispatch_router_batch<float>(b, R, s);
    if (e != hipSuccess) return e;
    const int TT = kSelectThreads / a.E;
    softmax_select_kernel<<<(a.T + TT - 1) / TT, kSelectThreads, 0, s>>>(
        a.logits_tmp, a.T, a.E, a.k, a.renorm, a.idx, a.w, a.status, FusedGrouping{});
    return hipGetLastError();
  }
  int TT = kRouterThreads / R;
  if (TT < 1) TT = 1;
  // Keep enough blocks in flight for small batches.
  while (TT > 1 && (a.T + TT - 1) / TT < 256 && TT * R > 64) TT = (TT + 1) / 2;
  const int blocks = (a.T + TT - 1) / TT;
  size_t dot_bytes = ((size_t)R + TT) * kLd * sizeof(float);
  size_t post_bytes = (((size_t)TT * R + 1) & ~(size_t)1) * 4 + (size_t)TT * a.E * (8 + 4 + 4);
  size_t smem = dot_bytes > post_bytes ? dot_bytes : post_bytes;
  if (a.x_is_bf16) {
    router_tile_kernel<uint16_t><<<blocks, kRouterThreads, smem, s>>>(
        (const uint16_t*)a.x, a.T, a.d, a.E, a.k, a.renorm, a.w_router, a.router_bias,
        a.shared_gate, a.idx, a.w, a.sgate, a.xb, a.d_pad, a.status, a.logits_out, TT);
  } else {
    router_tile_kernel<float><<<blocks, kRouterThreads, smem, s>>>(
        (const float*)a.x, a.T, a.d, a.E, a.k, a.renorm, a.w_router, a.router_bias,
        a.shared_gate, a.idx, a.w, a.sgate, a.xb, a.d_pad, a.status, a.logits_out, TT);
  }
  return hipGetLastError();
}

}  // namespace atenia_moe
