// Shared by the MFMA-tiled expert kernels (ffn_tiled.hip, ffn_tiled_duo.hip): operand types,
// the launch parameters, which tile a workgroup computes, and the global -> LDS load helper.
// gfx950 only.  Everything here sits in an unnamed namespace: each translation unit gets its own copy.
#pragma once

#include <type_traits>

#include "moe_internal.h"

namespace atenia_moe {

struct TiledParams {
  const uint4* wa;      // gate (up phase) or down blocks
  const uint4* wb;      // up blocks
  const float* sa;      // int8 row scales [G, n_rows]
  const float* sb;
  int64_t w_stride_u4;
  int n_rows;           // unpadded N
  int n_blocks;         // n_pad / 16
  int nkb;              // K blocks per strip (32 k each for bf16, 64 k for int8)
  int k_pad;
  const uint16_t* a;    // bf16 rows
  int a_stride;
  void* out;
  int out_stride;
  int out_bf16;         // down phase: y is stored as bf16 (nearest even) instead of f32
  const int32_t* perm;  // pair id of each grouped row
  const RowTile* tiles;       // [n_tiles], or null: one expert of rows_fixed rows in 256-row tiles
  const int32_t* n_tiles;     // [1]
  int max_groups;             // 32-row groups a row tile may hold: 8, or 9 (bf16 pipelined kernel only)
  int rows_fixed;
  FastDiv pair_div;           // token = pair id / pair_div
  uint32_t fixed_inv;         // tiles == null: tile_inv of the number of tiles
  FastDiv col_div, rest_div;  // by n_col_tiles, by its rest past whole patches
  int n_col_tiles;
  // k split of the tail tiles (pipelined down kernels; max_parts <= 1: off).  Workgroup ids
  // below wg_upper are the tiles themselves, ids from wg_upper on the extra k ranges of the
  // tiles in the last, partly filled round over the n_cus compute units.
  int max_parts;
  int wg_upper;
  int n_cus;
  FastDiv cu_div;             // by n_cus
  size_t out_part_stride;     // elements between the partial output buffers
  uint8_t* part_flags;        // [pairs, n_col_tiles] partial buffers written per (row, column tile)
};

// The form of the bf16 tiled kernels that runs two workgroups per compute unit (ffn_tiled_duo.hip).
bool tiled_duo_supported(const TiledParams& p);
hipError_t launch_tiled_duo_up(const TiledParams& p, int max_row_tiles, hipStream_t s);
hipError_t launch_tiled_duo_down(const TiledParams& p, int max_row_tiles, hipStream_t s);

namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

constexpr int kThreads = 256;
constexpr int TM = kTileM;   // 256 token rows
constexpr int TNB = 256;     // B rows per tile (gate/up: 128 + 128)
constexpr int TK = 64;       // k per LDS stage
constexpr int kChunk = 1024; // bytes
constexpr int kAStage = (TM / 16) * (TK / 32) * kChunk;   // 32 KiB
constexpr int kBStage = (TNB / 16) * (TK / 32) * kChunk;  // 32 KiB
constexpr int kStage = kAStage + kBStage;
constexpr int kLdsBytes = 2 * kStage;                     // 128 KiB


__device__ inline uint16_t bf16_rne(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

// Two f32 -> two bf16 (round to nearest even) in one v_cvt_pk_bf16_f32; low half = a.
typedef __attribute__((ext_vector_type(2))) float f32x2_t;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
__device__ inline uint32_t bf16_rne_pair(float a, float b) {
  f32x2_t v = {a, b};
  bf16x2_t h = __builtin_convertvector(v, bf16x2_t);
  return *(uint32_t*)&h;
}

// silu(g) * u with the hardware exp2 / rcp (1 ulp each; the result is rounded to bf16 next).
__device__ inline float swiglu_fast(float g, float u) {
  const float t = __builtin_amdgcn_exp2f(g * -1.4426950408889634f);
  return g * __builtin_amdgcn_rcpf(1.f + t) * u;
}

__device__ inline uint32_t pack_i8_pair(uint32_t w, int sh) {
  float f0 = (float)(int8_t)((w >> sh) & 0xff);
  float f1 = (float)(int8_t)((w >> (sh + 8)) & 0xff);
  // |q| <= 128 is exact in bf16, so dropping the low 16 bits loses nothing: one byte permute
  // takes the high halves of both floats (bytes 2, 3 of f0 below bytes 2, 3 of f1).
  return __builtin_amdgcn_perm(__float_as_uint(f1), __float_as_uint(f0), 0x07060302u);
}
__device__ inline void widen_i8x16(uint4 q, uint4& lo, uint4& hi) {
  lo.x = pack_i8_pair(q.x, 0);
  lo.y = pack_i8_pair(q.x, 16);
  lo.z = pack_i8_pair(q.y, 0);
  lo.w = pack_i8_pair(q.y, 16);
  hi.x = pack_i8_pair(q.z, 0);
  hi.y = pack_i8_pair(q.z, 16);
  hi.z = pack_i8_pair(q.w, 0);
  hi.w = pack_i8_pair(q.w, 16);
}

__device__ inline f32x4 mfma(uint4 a, uint4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(bf16x8*)&a, *(bf16x8*)&b, c, 0, 0, 0);
}

// A value that no running kernel writes, at an address the whole wave shares: one scalar load.
__device__ inline int uniform_load(const int32_t* p) { return *(const __attribute__((address_space(4))) int32_t*)p; }
__device__ inline RowTile uniform_load(const RowTile* p) {
  typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
  const i32x4 v = *(const __attribute__((address_space(4))) i32x4*)p;
  return RowTile{(uint32_t)v[0], v[1], v[2], (uint32_t)v[3]};
}

// Which (row tile, column tile) a workgroup computes.
//
// XCD-aware order: hardware deals consecutive workgroup ids round-robin to the 8 XCDs, each
// with its own L2, so XCD x is given the contiguous run [x*per_xcd, (x+1)*per_xcd) of the
// logical tile order.  In that order an expert's tiles are contiguous and walked in patches of
// (all row tiles of the expert) x (8 column tiles): the ~32 workgroups an XCD runs at a time
// share ~4 activation tiles and 8 weight tiles instead of streaming 64 different ones.
constexpr int kColGroup = 8;
struct TileAt {
  int e, base, m0, rows, ct;  // expert, its first grouped row, the tile's first row inside it and rows, column tile
};
__device__ inline int row_tiles(const TiledParams& p) {
  return p.tiles ? uniform_load(p.n_tiles) : (p.rows_fixed + TM - 1) / TM;
}
// NS > 1: for kernels whose workgroups take a slice of NS-th of a row tile's height (rows
// t.m0 = sub * TM / NS ..): every row tile counts as NS consecutive ones, so the slices of a tile
// and the column tiles of a patch stay neighbours in an XCD's run.
template <int NS = 1>
__device__ inline bool tile_of_workgroup(const TiledParams& p, int n_row_tiles, int wid, TileAt& t) {
  const int nct = p.n_col_tiles;
  const int total = n_row_tiles * NS * nct;
  const int per_xcd = (total + 7) >> 3;
  const int slot = wid >> 3;
  const int logical = (wid & 7) * per_xcd + slot;
  if (slot >= per_xcd || logical >= total) return false;
  // Row tiles are sorted by expert, so the expert owning this logical id is the expert of
  // row tile logical / nct; its entry tells where the expert's tiles start and how many they are.
  RowTile r{0, 0, p.rows_fixed, 0};
  int first = 0, n_expert_tiles = n_row_tiles;
  if (p.tiles) {
    const int rt_any = div_by(logical, p.col_div) / NS;
    r = uniform_load(p.tiles + rt_any);
    first = rt_any - (int)(r.e_i >> 16);
    n_expert_tiles = expert_tiles(r.rows, p.max_groups);
  } else {
    r.inv = p.fixed_inv;
  }
  // patches of (all row tiles) x kColGroup column tiles; the last patch may be narrower
  static_assert(kColGroup == 8, "shifts below");
  const int nt = n_expert_tiles * NS;
  int local = logical - first * NS * nct, cg = 0, rl, c;
  const int full = nct >> 3;
  if (local < full * 8 * nt) {
    cg = div_tiles(local >> 3, n_expert_tiles, r.inv) / NS;
    local -= cg * 8 * nt;
    rl = local >> 3;
    c = local & 7;
  } else {
    cg = full;
    local -= full * 8 * nt;
    rl = div_by(local, p.rest_div);
    c = local - rl * (nct - full * 8);
  }
  const int i = rl / NS;
  t.e = (int)(r.e_i & 0xffff);
  t.base = r.base;
  t.ct = cg * kColGroup + c;
  expert_tile(r.rows, p.max_groups, n_expert_tiles, r.inv, i, t.m0, t.rows);
  if (NS > 1) {
    const int sub = rl - i * NS;
    t.m0 += sub * (TM / NS);
    t.rows = min(TM / NS, t.rows - sub * (TM / NS));
  }
  return true;
}

// Tail split of the down phase.  With one workgroup per CU at a time, tiles run in rounds of
// n_cus; when the last round is at most half full, each of its tiles is cut into S k ranges
// (S <= max_parts) so that the round fills the chip and lasts 1/S as long.  Range 0 is
// computed by the tile's own workgroup, ranges 1..S-1 by workgroups with ids from wg_upper on;
// range i writes its partial sums to buffer i, and range 0 records S per (row, column tile) so
// that the combine adds up exactly the buffers that were written.  Sets wid (the tile's
// workgroup id for tile_of_workgroup), S and part; false = nothing to do.
// bid: the workgroup's id within its launch (blockIdx.x, or the id inside its own part of a launch
// that carries two parameter sets).
__device__ inline bool split_of_workgroup(const TiledParams& p, int n_row_tiles, int bid, int n_stages, int& wid,
                                          int& S, int& part) {
  wid = bid;
  S = 1;
  part = 0;
  if (p.max_parts <= 1) return true;
  const int total = n_row_tiles * p.n_col_tiles;
  const int per_xcd = (total + 7) >> 3;
  const int full_slots = div_by(total, p.cu_div) * (p.n_cus >> 3);  // slots per XCD in the full rounds
  const int tail = 8 * (per_xcd - full_slots);               // tile slots of the last round
  int s_tail = 1;
  if (tail > 0 && 2 * tail <= p.n_cus) s_tail = min(min(p.max_parts, p.n_cus / tail), n_stages / 2);
  if (s_tail < 1) s_tail = 1;
  if (bid >= p.wg_upper) {
    const int x = bid - p.wg_upper;
    if (s_tail == 1 || x >= tail * (s_tail - 1)) return false;
    part = 1 + x / tail;
    const int j = x - (part - 1) * tail;
    wid = (full_slots + j / 8) * 8 + (j & 7);
    S = s_tail;
    return true;
  }
  if ((wid >> 3) >= full_slots) S = s_tail;
  return true;
}

typedef __attribute__((address_space(3))) void* lptr_t;

// One wave-wide 16-byte-per-lane load from global memory straight into LDS: lane l's bytes
// land at lds_addr + 16*l.  Written as inline assembly so that the compiler's wait-count
// insertion does not tie later LDS reads to these loads (it would drain all stages); the
// kernel waits for exactly the stage it needs with an explicit s_waitcnt before its barrier.
__device__ inline void dma16(const void* gaddr, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off"
               :
               : "v"(gaddr), "s"(lds_addr)
               : "memory", "m0");
}

// The same with a wave-uniform base and a 32-bit byte offset per lane.
__device__ inline void dma16_at(const void* base, uint32_t off, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(off), "s"(base), "s"(lds_addr)
               : "memory", "m0");
}

// Four bytes per lane: lane l's land at lds_addr + 4*l.
__device__ inline void dma4_at(const void* base, uint32_t off, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dword %0, %1"
               :
               : "v"(off), "s"(base), "s"(lds_addr)
               : "memory", "m0");
}

typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;

// v_mfma_f32_32x32x16_bf16 operand layout: A lane l holds row l%32, k = 8*(l/32)..+7 of a
// 32 x 16 fragment; B the same with columns; D register r of lane l is element
// (row 8*(r/4) + 4*(l/32) + r%4, column l%32).  Measured on MI355X the 32x32x16 form sustains
// about 1.35x the rate of 16x16x32 in this kind of loop, so the tiled kernel uses it: an LDS
// chunk (1 KiB) is one 32 x 16 fragment.
__device__ inline f32x16 mfma32(uint4 a, uint4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(bf16x8*)&a, *(bf16x8*)&b, c, 0, 0, 0);
}

// Sixteen neighbouring entries of the pair list by one scalar load: scalar loads do not wait behind the
// vector loads in flight, so the row list is looked up while the first weights are on their way.  (The list
// is not written while the kernels that read it run.)  A wave's window of up to 64 entries starts inside its
// tile; what lies past the tile is not used, and past the list's end it is the next piece of the workspace.
typedef int32_t i32x16 __attribute__((ext_vector_type(16), aligned(4)));
__device__ inline i32x16 pairs16(const int32_t* perm, int at) {
  return *(const __attribute__((address_space(4))) i32x16*)(perm + __builtin_amdgcn_readfirstlane(at));
}
template <int AT>
__device__ inline int pick8(i32x16 v, int j) {  // v[AT + j], 0 <= j < 8
  const int a = j & 1 ? v[AT + 1] : v[AT], b = j & 1 ? v[AT + 3] : v[AT + 2];
  const int c = j & 1 ? v[AT + 5] : v[AT + 4], d = j & 1 ? v[AT + 7] : v[AT + 6];
  const int ab = j & 2 ? b : a, cd = j & 2 ? d : c;
  return j & 4 ? cd : ab;
}
// Grouped rows at + 8 q + j of NQ chunks of a wave (j per lane) -> row of the activations: the token of the
// pair where the rows are gathered, the grouped row itself otherwise.  Rows from `end` on: the first of the
// wave (or, where it has none, of the tile) again -- computed, never stored.
template <bool GATHER, int NQ>
__device__ __forceinline__ void source_rows(const int32_t* perm, FastDiv pair_div, int tile0, int at, int end, int j,
                                            int (&src)[NQ]) {
  int w0 = __builtin_amdgcn_readfirstlane(at < end ? at : tile0);
  const bool none = w0 != at;
  if (!GATHER) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) src[q] = none || at + 8 * q + j >= end ? w0 : at + 8 * q + j;
    return;
  }
#pragma unroll
  for (int q = 0; q < NQ; q += 4) {  // four chunks at a time: all eight would spill scalar registers
    const i32x16 lo = pairs16(perm, w0 + 8 * q);
    const i32x16 hi = q + 2 < NQ ? pairs16(perm, w0 + 8 * q + 16) : lo;
    const int first = q == 0 ? lo[0] : src[0];
#pragma unroll
    for (int c = 0; c < 4 && q + c < NQ; ++c) {
      const int v = c == 0 ? pick8<0>(lo, j) : c == 1 ? pick8<8>(lo, j) : c == 2 ? pick8<0>(hi, j) : pick8<8>(hi, j);
      src[q + c] = none || at + 8 * (q + c) + j >= end ? first : v;
    }
    if (q + 4 < NQ)
      asm volatile("" : "+s"(w0) : "v"(src[q]), "v"(src[q + 1]), "v"(src[q + 2]), "v"(src[q + 3]));
  }
#pragma unroll
  for (int q = 0; q < NQ; ++q) src[q] = div_by(src[q], pair_div);
}

// s_waitcnt vmcnt(N) lgkmcnt(0): vmcnt[3:0] in bits 3:0, vmcnt[5:4] in bits 15:14, expcnt
// (bits 6:4) left at "no wait".  lgkmcnt(0) makes sure the wave's own LDS reads have returned
// before it passes the barrier behind which other waves refill the buffers it read.
template <int N>
__device__ inline void wait_vm_lgkm0() {
  __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | ((N >> 4) << 14));
}

}  // namespace

}  // namespace atenia_moe
