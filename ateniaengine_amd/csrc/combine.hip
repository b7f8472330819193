// Kernel 4: weighted combine back to token order.
//
// out[t] = sum over the token's slots (ascending expert id) of w[t,slot] * y[t,slot], then
// += scale[t] * y_shared[t]      (src/moe/sparse.rs:226-233, src/moe/layer.rs:415-429), and,
// for the decoder layer's FFN block, out[t] = residual[t] + that (src/moe/full_forward.rs:251).
// The reference multiplies and adds in f32 with two roundings and a fixed order; the same
// sequence is kept here (no fused multiply-add, no atomics), so given equal expert outputs
// the combine is bit-identical.  Expert outputs are stored by pair id t*k+slot, so a token's
// k rows are adjacent and every read and write is coalesced.  When the down phase
// split the k range of some tiles, an expert output there is the f32 sum of its partial
// buffers, added in buffer order.  The bf16 tiled down kernels may leave the expert outputs as
// bf16 (half the bytes both ways); they are widened here, exactly, before the same arithmetic.
#include "moe_internal.h"

// This file is compiled with -ffp-contract=off (see the Makefile): the reference rounds every
// product and every sum on its own, and hipcc would otherwise fuse `a * b + c` into one FMA
// (its default is -ffp-contract=fast, under which __fmul_rn / __fadd_rn are plain `*` and `+`
// and the fp-contract pragma is ignored).

namespace atenia_moe {

namespace {

constexpr int kCombineSharedParts = 4;  // ranges of the shared expert's rows held at once

// CPT consecutive expert-output values as they are stored: f32 (CPT = 4) or bf16 (CPT = 4 or 8).
// Expert outputs are read exactly once: a streaming (non-temporal) load leaves the caches to the
// kernels around this one.  The launch alone is the faster one with ordinary loads while the outputs, just written,
// lie in the last-level cache (d = 7168, 256 tokens of 8 slots 12.0 / 11.0 us; d = 2048, 2048 of 10 20.3 / 17.2), but what
// it then leaves there costs the launches around it more (whole forward, streaming / ordinary, us: 256 experts
// of width 256, T = 256 561 / 577, 2048 986 / 1026; Qwen1.5-MoE shape T = 600 239 / 245, 997 265 / 270; 128 experts of width 1536,
// d = 4096, T = 600 827 / 868; Mixtral shape T = 333, ordinary for the second range on, 493 / 500).
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
template <bool BF16, int CPT> struct RawOf { typedef f32x4_t type; };
template <> struct RawOf<true, 4> { typedef u32x2_t type; };
template <> struct RawOf<true, 8> { typedef u32x4_t type; };
template <bool BF16, int CPT> using Raw = typename RawOf<BF16, CPT>::type;

template <bool BF16, int CPT>
__device__ inline Raw<BF16, CPT> load_raw(const void* base, size_t elem) {
  return __builtin_nontemporal_load((const Raw<BF16, CPT>*)((const char*)base + elem * (BF16 ? 2 : 4)));
}
template <bool BF16, int CPT>
__device__ inline void widen(const Raw<BF16, CPT>& q, float (&v)[CPT]) {
  if constexpr (BF16) {
#pragma unroll
    for (int j = 0; j < CPT / 2; ++j) {
      v[2 * j] = __uint_as_float(q[j] << 16);
      v[2 * j + 1] = __uint_as_float(q[j] & 0xffff0000u);
    }
  } else {
#pragma unroll
    for (int j = 0; j < CPT; ++j) v[j] = q[j];
  }
}
template <bool BF16>
__device__ inline float load1(const void* base, size_t elem) {
  if (BF16) return __uint_as_float((uint32_t)((const uint16_t*)base)[elem] << 16);
  return ((const float*)base)[elem];
}

// Partial buffers of the routed rows: none; as many everywhere (y_parts); by tile (part_flags: a few tiles).
enum { kRangesNone, kRangesAlike, kRangesByTile };

// Rows of whole CPT columns (8 only when both y and y_shared -- if any -- are bf16).
// What bounds it: HBM bytes at large batches, one memory round trip in and one out at small ones.
// All of a token's loads are therefore requested before the first is used: up to S slots, the shared
// expert's ranges, the residual; where every tile was cut into ranges (f32 rows), then one range of all
// slots at a time.  (A slot past k is not requested.  Where it repeated the last one's request, ten slots cost
// what sixteen do: d = 2048, 4096 tokens of 10 39.1 / 32.8 us, 2048 of 10 24.9 / 20.3.)
// Slot by slot / this way, us: d = 2048, 16384 tokens of 6 slots and a shared expert 111.9 / 90.6 (0.60 GB, 6.7
// TB/s), 12288 of 4 61.9 / 58.1, 600 of 6 (f32 rows) 9.5 / 7.6, 48 of 6 4.4 / 4.0; d = 7168, 256 of 8 15.9 / 11.9, 4096 of 10
// 155 / 109; d = 4096, 4096 of 2 28.1 / 27.2, 333 of 2 in four ranges 8.6 / 8.7.
template <bool YB, bool SB, int CPT, int S, int RANGES>
__global__ __launch_bounds__(256) void combine_kernel(CombineArgs a, FastDiv chunk_div, int chunks) {
  copy_status(a.status);
  const int t = div_by(blockIdx.x, chunk_div);
  const int c = ((blockIdx.x - t * chunks) * 256 + threadIdx.x) * CPT;
  if (c >= a.d) return;
  Raw<SB, CPT> ys[kCombineSharedParts];
  float sc = 1.0f;
  const size_t ys_at = (size_t)t * a.y_stride + c;
  if (a.y_shared) {
    if (a.sgate) sc = a.sgate[t];
    ys[0] = load_raw<SB, CPT>(a.y_shared, ys_at);
#pragma unroll
    for (int part = 1; part < kCombineSharedParts; ++part)
      if (part < a.ys_parts) ys[part] = load_raw<SB, CPT>(a.y_shared, ys_at + part * a.ys_part_stride);
  }
  f32x4_t res[CPT / 4];
  if (a.residual) {  // may alias `out`: each element is read and written by this thread only
#pragma unroll
    for (int i = 0; i < CPT / 4; ++i) res[i] = *(const f32x4_t*)(a.residual + (size_t)t * a.d + c + 4 * i);
  }
  float o[CPT];
#pragma unroll
  for (int j = 0; j < CPT; ++j) o[j] = 0.f;
  for (int s0 = 0; s0 < a.k; s0 += S) {
    const auto pair_of = [&](int i) { return (size_t)t * a.k + s0 + i; };
    const auto load_y = [&](int i, int part) {
      return load_raw<YB, CPT>(a.y, pair_of(i) * a.y_stride + c + part * a.y_part_stride);
    };
    Raw<YB, CPT> q[S];
    float ws[S];
    int n_parts[S];
#pragma unroll
    for (int i = 0; i < S; ++i) {
      if (s0 + i >= a.k) continue;
      q[i] = load_y(i, 0);
      ws[i] = a.w[pair_of(i)];
      if (RANGES == kRangesByTile) n_parts[i] = a.part_flags[pair_of(i) * a.flag_cols + c / 256];
    }
    if constexpr (RANGES == kRangesAlike) {
      for (int part = 1; part < a.y_parts; ++part) {  // (three at a time measured no faster)
        Raw<YB, CPT> p[S];
#pragma unroll
        for (int i = 0; i < S; ++i)
          if (s0 + i < a.k) p[i] = load_y(i, part);
#pragma unroll
        for (int i = 0; i < S; ++i)
#pragma unroll
          for (int j = 0; j < CPT; ++j)
            if (s0 + i < a.k) q[i][j] = __fadd_rn(q[i][j], p[i][j]);
      }
    }
#pragma unroll
    for (int i = 0; i < S; ++i) {
      if (s0 + i < a.k) {
        float v[CPT];
        widen<YB, CPT>(q[i], v);
        if constexpr (RANGES == kRangesByTile) {
          for (int part = 1; part < n_parts[i]; ++part) {
            float p[CPT];
            widen<YB, CPT>(load_y(i, part), p);
#pragma unroll
            for (int j = 0; j < CPT; ++j) v[j] = __fadd_rn(v[j], p[j]);
          }
        }
#pragma unroll
        for (int j = 0; j < CPT; ++j) o[j] = __fadd_rn(o[j], __fmul_rn(ws[i], v[j]));
      }
    }
  }
  if (a.y_shared) {
    float v[CPT];
    widen<SB, CPT>(ys[0], v);
#pragma unroll
    for (int part = 1; part < kCombineSharedParts; ++part)
      if (part < a.ys_parts) {
        float p[CPT];
        widen<SB, CPT>(ys[part], p);
#pragma unroll
        for (int j = 0; j < CPT; ++j) v[j] = __fadd_rn(v[j], p[j]);
      }
#pragma unroll
    for (int j = 0; j < CPT; ++j) o[j] = __fadd_rn(o[j], __fmul_rn(sc, v[j]));
  }
#pragma unroll
  for (int i = 0; i < CPT / 4; ++i) {
    f32x4_t r;
#pragma unroll
    for (int j = 0; j < 4; ++j) r[j] = a.residual ? __fadd_rn(res[i][j], o[4 * i + j]) : o[4 * i + j];
    *(f32x4_t*)(a.out + (size_t)t * a.d + c + 4 * i) = r;
  }
}

// Any other width: one column at a time.
template <bool YB, bool SB>
__global__ __launch_bounds__(256) void combine_odd_kernel(CombineArgs a, FastDiv chunk_div, int chunks) {
  copy_status(a.status);
  const int t = div_by(blockIdx.x, chunk_div);
  const int c = (blockIdx.x - t * chunks) * 256 + threadIdx.x;
  if (c >= a.d) return;
  float o = 0.f;
  for (int slot = 0; slot < a.k; ++slot) {
    const size_t pair = (size_t)t * a.k + slot, at = pair * a.y_stride + c;
    const int n_parts = a.part_flags ? a.part_flags[pair * a.flag_cols + c / 256] : a.y_parts;
    float v = load1<YB>(a.y, at);
    for (int part = 1; part < n_parts; ++part) v = __fadd_rn(v, load1<YB>(a.y, at + part * a.y_part_stride));
    o = __fadd_rn(o, __fmul_rn(a.w[pair], v));
  }
  if (a.y_shared) {
    const size_t at = (size_t)t * a.y_stride + c;
    float v = load1<SB>(a.y_shared, at);
    for (int part = 1; part < a.ys_parts; ++part) v = __fadd_rn(v, load1<SB>(a.y_shared, at + part * a.ys_part_stride));
    o = __fadd_rn(o, __fmul_rn(a.sgate ? a.sgate[t] : 1.0f, v));
  }
  const size_t at = (size_t)t * a.d + c;
  a.out[at] = a.residual ? __fadd_rn(a.residual[at], o) : o;
}

template <bool YB, bool SB, int CPT, int RANGES>
void launch_rows(const CombineArgs& a, hipStream_t s) {
  const int chunks = (a.d + 256 * CPT - 1) / (256 * CPT);
  const unsigned grid = (unsigned)chunks * (unsigned)a.T;
  const FastDiv div = fast_div(chunks);
  if (a.k <= 2) combine_kernel<YB, SB, CPT, 2, RANGES><<<grid, 256, 0, s>>>(a, div, chunks);
  else if (a.k <= 4) combine_kernel<YB, SB, CPT, 4, RANGES><<<grid, 256, 0, s>>>(a, div, chunks);
  else if (a.k <= 6) combine_kernel<YB, SB, CPT, 6, RANGES><<<grid, 256, 0, s>>>(a, div, chunks);
  else combine_kernel<YB, SB, CPT, 8, RANGES><<<grid, 256, 0, s>>>(a, div, chunks);
}

template <bool YB, bool SB>
void launch_types(const CombineArgs& a, hipStream_t s) {
  const bool alike = !a.part_flags && a.y_parts > 1;
  const int both = a.d | a.y_stride;
  if (both % 4 != 0 || (YB && alike) || (a.y_shared && a.ys_parts > kCombineSharedParts)) {
    const int chunks = (a.d + 255) / 256;
    combine_odd_kernel<YB, SB><<<(unsigned)chunks * (unsigned)a.T, 256, 0, s>>>(a, fast_div(chunks), chunks);
    return;
  }
  if constexpr (YB) {  // bf16 expert outputs: 8 columns (16 bytes of each row) per thread
    if ((SB || !a.y_shared) && both % 8 == 0)
      return a.part_flags ? launch_rows<true, true, 8, kRangesByTile>(a, s)
                          : launch_rows<true, true, 8, kRangesNone>(a, s);
  } else if (alike) {
    return launch_rows<YB, SB, 4, kRangesAlike>(a, s);
  }
  a.part_flags ? launch_rows<YB, SB, 4, kRangesByTile>(a, s) : launch_rows<YB, SB, 4, kRangesNone>(a, s);
}

}  // namespace

hipError_t launch_combine(const CombineArgs& a, hipStream_t s) {
  if (a.y_bf16 && a.ys_bf16) launch_types<true, true>(a, s);
  else if (a.y_bf16) launch_types<true, false>(a, s);
  else if (a.ys_bf16) launch_types<false, true>(a, s);
  else launch_types<false, false>(a, s);
  return hipGetLastError();
}

}  // namespace atenia_moe
