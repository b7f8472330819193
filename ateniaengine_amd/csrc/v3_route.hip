// DeepSeek-V3 routing: sigmoid scores, bias-corrected selection, group-limited top-k, scaled
// combine weights (src/moe/v3_router.rs:206-309), from the raw f32 logits the router kernels
// leave in HBM.  All arithmetic in f64 as in the reference:
//   score_e  = 1 / (1 + exp(-logit_e));  choice_e = score_e + bias_e
//   group score = sum of the group's two largest choices; the topk_group best groups stay
//   (ties: lower group), experts of other groups are masked to -inf; the top_k best remaining
//   experts are selected (ties: lower index) and emitted ascending;
//   weight = score (not choice), / (sum of selected scores, ascending, + 1e-20) when
//   norm_topk_prob, * routed_scaling_factor, rounded to f32.
// "The k best under (value desc, index asc)" is computed as a rank count per element, which is
// what the reference's stable sort yields, or as the largest remaining choice k times, the lowest index
// among equals.  A non-finite logit is reported through the status words like a non-finite
// routing weight of the softmax router (the reference fails with NonFinite{router_logits, index}).
#include "moe_internal.h"
#include "select_wave.h"

namespace atenia_moe {

namespace {

constexpr int kV3Threads = 256;

// One wavefront per token: lane l holds the J consecutive experts J l .. J l + J - 1, a group is an aligned
// power of two of lanes (v3_wave_groups).  Bound by latency: exponentials, then chains of cross-lane steps with no
// barrier and no LDS between them.  One thread per expert (below), seven barriers and a count against every expert
// of the kept groups / this, launch, us: 256 experts in 8 groups,
// T = 256 15.0 / 6.7; whole forward (d = 7168, f = 256) T = 1 60.1 / 52.9, 16 219 / 212, 256 424 / 417, 2000 946 / 929.
template <int CTRL>
__device__ inline double lane_from(double v) {  // of every lane's DPP partner
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)b, hi = (uint32_t)(b >> 32);
  const uint32_t l = __builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xf, 0xf, false);
  const uint32_t h = __builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xf, 0xf, false);
  return __builtin_bit_cast(double, (uint64_t)h << 32 | l);
}
constexpr int kSwapOne = 0xB1, kSwapTwo = 0x4E, kMirrorEight = 0x141, kMirrorSixteen = 0x140;
__device__ inline double wave_max_f64(double v) {  // no NaN
  v = fmax(v, lane_from<kSwapOne>(v));
  v = fmax(v, lane_from<kSwapTwo>(v));
  v = fmax(v, lane_from<kMirrorEight>(v));
  v = fmax(v, lane_from<kMirrorSixteen>(v));
  return fmax(fmax(readlane_f64(v, 0), readlane_f64(v, 16)), fmax(readlane_f64(v, 32), readlane_f64(v, 48)));
}

template <int J>
__global__ __launch_bounds__(kV3Threads) void v3_route_wave_kernel(
    const float* __restrict__ logits, const float* __restrict__ bias, int T, int k, int n_group, int topk_group,
    int norm_topk_prob, double scale, int32_t* __restrict__ idx_out, float* __restrict__ w_out,
    int32_t* __restrict__ status) {
  constexpr int E = 64 * J;
  const int lane = threadIdx.x & 63;
  const int t = blockIdx.x * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (t >= T) return;
  const int e0 = lane * J;
  double score[J], choice[J];
  float lg[J], bs[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    lg[j] = logits[(size_t)t * E + e0 + j];
    bs[j] = bias[e0 + j];
  }
#pragma unroll
  for (int j = 0; j < J; ++j) {
    if (!isfinite(lg[j])) {
      atomicMin(&status[0], -3);
      atomicMin(&status[1], (t << 10) | (e0 + j));
    }
    score[j] = 1.0 / (1.0 + exp(-(double)lg[j]));
    const double c = score[j] + (double)bs[j];
    choice[j] = isnan(c) ? -INFINITY : c;  // (of a token that is reported: its indices must still be indices)
  }
  // the group's two largest choices, over this lane's experts and then over its lanes: every step meets the
  // other half of a block of lanes that already agree
  double m1 = -INFINITY, m2 = -INFINITY;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    m2 = fmax(m2, fmin(m1, choice[j]));
    m1 = fmax(m1, choice[j]);
  }
  auto merge = [&](double o1, double o2) {
    m2 = fmax(fmin(m1, o1), fmax(m2, o2));
    m1 = fmax(m1, o1);
  };
  const int lanes = 64 / n_group;  // of a group
  if (lanes >= 2) merge(lane_from<kSwapOne>(m1), lane_from<kSwapOne>(m2));
  if (lanes >= 4) merge(lane_from<kSwapTwo>(m1), lane_from<kSwapTwo>(m2));
  if (lanes >= 8) merge(lane_from<kMirrorEight>(m1), lane_from<kMirrorEight>(m2));
  if (lanes >= 16) merge(lane_from<kMirrorSixteen>(m1), lane_from<kMirrorSixteen>(m2));
  if (lanes >= 32) merge(__shfl_xor(m1, 16), __shfl_xor(m2, 16));
  if (lanes >= 64) merge(__shfl_xor(m1, 32), __shfl_xor(m2, 32));
  const double mine = m1 + m2;
  const int my_group = lane / lanes;
  int before = 0;  // groups that sort before this one under (score desc, index asc)
  for (int g = 0; g < n_group; ++g) {
    const double o = readlane_f64(mine, g * lanes);
    before += (o > mine) || (o == mine && g < my_group);
  }
  unsigned open = before < topk_group ? (1u << J) - 1u : 0u;  // this lane's experts that are still to be had
  unsigned sel = 0;
  for (int r = 0; r < k; ++r) {
    double best = -INFINITY;
#pragma unroll
    for (int j = 0; j < J; ++j) best = (open >> j) & 1 ? fmax(best, choice[j]) : best;
    const double top = wave_max_f64(best);
    const unsigned long long cand = __ballot(open && best == top);
    if (!cand) break;  // wave-uniform; top_k <= experts of the kept groups makes it unreachable
    if (lane == __ffsll((long long)cand) - 1) {  // the lowest lane, its lowest expert
      unsigned at = 0;
#pragma unroll
      for (int j = J - 1; j >= 0; --j) at = ((open >> j) & 1) && choice[j] == top ? 1u << j : at;
      sel |= at;
      open &= ~at;
    }
  }
  // slots and the sum of the selected scores, indices ascending
  const unsigned long long chosen = __ballot(sel != 0);
  int slot = 0;
  double denom = 0.0;
  for (unsigned long long m = chosen; m; m &= m - 1) {
    const int l = __ffsll((long long)m) - 1;
    const unsigned s = (unsigned)__builtin_amdgcn_readlane((int)sel, l);
    slot += l < lane ? __popc(s) : 0;
#pragma unroll
    for (int j = 0; j < J; ++j)
      if ((s >> j) & 1) denom += readlane_f64(score[j], l);
  }
  denom += 1e-20;
#pragma unroll
  for (int j = 0; j < J; ++j)
    if ((sel >> j) & 1) {
      double w = score[j];
      if (norm_topk_prob) w /= denom;
      w *= scale;
      idx_out[(size_t)t * k + slot] = e0 + j;
      w_out[(size_t)t * k + slot] = (float)w;
      ++slot;
    }
}
// Experts in whole 64s and groups of whole lanes, a power of two of them (n_group divides 64).
bool v3_wave_groups(int E, int n_group) { return E % 64 == 0 && n_group <= 64 && 64 % n_group == 0; }

// Any number of experts up to 256: one thread per (token, expert), 256 / E tokens to a workgroup.

__global__ __launch_bounds__(kV3Threads) void v3_route_kernel(
    const float* __restrict__ logits, const float* __restrict__ bias, int T, int E, int k,
    int n_group, int topk_group, int norm_topk_prob, double scale, int32_t* __restrict__ idx_out,
    float* __restrict__ w_out, int32_t* __restrict__ status) {
  __shared__ double sScore[kV3Threads];   // [TT][E]
  __shared__ double sChoice[kV3Threads];  // [TT][E]
  __shared__ double sGroup[kV3Threads / 2];    // [TT][n_group]
  __shared__ uint8_t sGroupSel[kV3Threads / 2];
  __shared__ uint8_t sSel[kV3Threads];      // slot of a selected thread
  __shared__ double sList[kV3Threads];      // [TT][k] scores of the selected experts, ascending
  __shared__ unsigned long long sWaveVote[kV3Threads / 64];
  const int TT = kV3Threads / E;  // >= 1: the launcher refuses E > 256
  const int tid = threadIdx.x;
  const int tl = tid / E, r = tid - tl * E;
  const int t = blockIdx.x * TT + tl;
  const bool on = tl < TT && t < T;
  const int epg = E / n_group;
  const int base = tl * E, gbase = tl * n_group;

  if (on) {
    const float lg = logits[(size_t)t * E + r];
    if (!isfinite(lg)) {
      atomicMin(&status[0], -3);
      atomicMin(&status[1], (t << 10) | r);
    }
    const double sc = 1.0 / (1.0 + exp(-(double)lg));
    sScore[base + r] = sc;
    sChoice[base + r] = sc + (double)bias[r];
  }
  __syncthreads();
  if (on && r < n_group) {  // the two largest choices of group r
    const double* c = sChoice + base + r * epg;
    double m1 = -INFINITY, m2 = -INFINITY;
#pragma unroll 8
    for (int j = 0; j < epg; ++j) {
      const double v = c[j];  // finite: fmax / fmin are plain comparisons here
      m2 = fmax(m2, fmin(m1, v));
      m1 = fmax(m1, v);
    }
    sGroup[gbase + r] = m1 + m2;
  }
  __syncthreads();
  if (on && r < n_group) {
    const double mine = sGroup[gbase + r];
    int rank = 0;  // groups that sort before this one under (score desc, index asc)
    for (int g = 0; g < n_group; ++g) {
      const double o = sGroup[gbase + g];
      rank += (o > mine) || (o == mine && g < r);
    }
    sGroupSel[gbase + r] = rank < topk_group;
  }
  __syncthreads();
  // Only experts of the kept groups compete; an expert's rank counts those that sort before it
  // under (choice desc, index asc).  Masked experts never enter: top_k <= experts in the kept
  // groups (checked when the router is configured).
  bool selected = false;
  double my_score = 0.0;
  if (on && sGroupSel[gbase + r / epg]) {
    const double mine = sChoice[base + r];
    int rank = 0;
    for (int g = 0; g < n_group; ++g) {
      if (!sGroupSel[gbase + g]) continue;  // uniform across the workgroup when it holds one token
      const double* c = sChoice + base + g * epg;
      const int e0 = g * epg;
#pragma unroll 8
      for (int j = 0; j < epg; ++j) {
        const double o = c[j];
        rank += (o > mine) || (o == mine && e0 + j < r);
      }
    }
    selected = rank < k;
    my_score = sScore[base + r];
  }
  // Ascending slots: selected lanes before this one in its wave (ballot) plus the selected
  // lanes of the earlier waves that belong to the same token.
  const unsigned long long vote = __ballot(selected);
  const int lane = tid & 63, wave = tid >> 6;
  if (lane == 0) sWaveVote[wave] = vote;
  __syncthreads();
  if (selected) {
    int slot = 0;
    const int first = base, last = base + r;  // thread ids of this token before this expert
    for (int w = first >> 6; w <= wave; ++w) {
      unsigned long long m = sWaveVote[w];
      const int lo = w * 64;
      if (first > lo) m &= ~0ull << (first - lo);
      if (last < lo + 64) m &= (last - lo) >= 64 ? ~0ull : ((1ull << (last - lo)) - 1ull);
      slot += __popcll(m);
    }
    if (slot < k) {
      sList[tl * k + slot] = my_score;
      idx_out[(size_t)t * k + slot] = r;
    }
    sSel[tid] = (uint8_t)slot;
  }
  __syncthreads();
  if (selected) {
    const int slot = sSel[tid];
    double denom = 0.0;
    for (int j = 0; j < k; ++j) denom += sList[tl * k + j];  // ascending index, as the sorted selection is summed
    denom += 1e-20;
    double w = my_score;
    if (norm_topk_prob) w /= denom;
    w *= scale;
    if (slot < k) w_out[(size_t)t * k + slot] = (float)w;
  }
}

}  // namespace

hipError_t launch_v3_route(const V3RouteArgs& a, hipStream_t s) {
  if (a.T <= 0) return hipSuccess;
  if (a.E <= 0 || a.E > kV3Threads || a.n_group <= 0 || a.E % a.n_group != 0 ||
      a.n_group > kV3Threads / 2)
    return hipErrorInvalidValue;
  if (v3_wave_groups(a.E, a.n_group)) {
    // few tokens: a compute unit each
    const int threads = a.T <= 1024 ? 64 : kV3Threads, per = threads / 64;
    auto go = [&](auto kernel) {
      kernel<<<(a.T + per - 1) / per, threads, 0, s>>>(a.logits, a.bias, a.T, a.k, a.n_group, a.topk_group,
                                                       a.norm_topk_prob, a.routed_scaling_factor, a.idx, a.w, a.status);
      return hipGetLastError();
    };
    return a.E == 64 ? go(v3_route_wave_kernel<1>) : a.E == 128 ? go(v3_route_wave_kernel<2>)
         : a.E == 192 ? go(v3_route_wave_kernel<3>) : go(v3_route_wave_kernel<4>);
  }
  const int TT = kV3Threads / a.E;
  const unsigned grid = (unsigned)((a.T + TT - 1) / TT);
  v3_route_kernel<<<grid, kV3Threads, 0, s>>>(a.logits, a.bias, a.T, a.E, a.k, a.n_group,
                                              a.topk_group, a.norm_topk_prob,
                                              a.routed_scaling_factor, a.idx, a.w, a.status);
  return hipGetLastError();
}

}  // namespace atenia_moe
