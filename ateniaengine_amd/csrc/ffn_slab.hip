// Kernel 3, slab form: grouped SwiGLU expert GEMMs for batches whose experts see a few rows up to a
// little over a hundred on bf16 layers (short prompts, large decode batches), up to several hundred on
// W8A16 ones (slab_max_avg, moe_abi.hip).
//
//   gate/up : H[rows of e, f] = silu(X_e W_g^T) * (X_e W_u^T)     (src/moe/dense.rs:253-266)
//   down    : Y[rows of e, d] = H_e W_d^T                         (src/moe/dense.rs:267-269)
// on bf16 MFMA with f32 accumulation.  Here the weight stream and the matrix work are of the same
// order: every weight byte is read from HBM once (per 128 rows of its expert), and the kernel has
// to keep enough of that stream in flight while it multiplies.
//
// A workgroup of four waves owns a tile of up to 128 rows of one expert by 256 weight rows; two
// workgroups share a compute unit, so one's prologue and epilogue run under the other's stream.
// A wave owns 64 weight rows (gate/up: 32 gate rows and the same 32 up rows, so silu(g) * u is
// formed in registers) over the whole K range and all rows of the tile: 4 x 2 tiles of
// v_mfma_f32_32x32x16_bf16.
//   * Weights go from HBM straight into B-operand registers (no LDS): 64 k of the wave's 64 rows
//     are eight 16-byte registers per lane, and two such stages are in flight -- 16 KiB per wave,
//     128 KiB per compute unit, what HBM's latency times its rate asks for with room to spare.  (int8:
//     four registers, three stages, four where a tile has one or two row groups.)
//   * Token rows are shared by the four waves through LDS: a ring of four 64-k stages (16 KiB
//     each, 1 KiB chunks of 8 rows x 128 bytes, swizzled as in ffn_tiled.hip) that the waves fill
//     with global_load_lds, three stages ahead; one barrier per stage.
//   * Only the 32-row groups that hold rows are loaded and multiplied (RG = 1 .. 4 of them, one
//     code path each): a tile costs what its rows cost.
// What bounds it: the weight stream, and what a tile does after it.  Without its matrix instructions the
// launch takes nearly the same time (by stage timers, us, with / without: Mixtral shape, gate/up, T = 64 294 / 295 for
// 1.88 GB, T = 333 337 / 330; Qwen1.5-MoE shape T = 997 163 / 155), with twice the weight loads in flight the same, and
// neither the width of a load, the number of strips of a tile nor the K a tile starts from moves it.  With an
// epilogue of single values from the accumulators, it took 303 of 337 us without it (Mixtral T = 333,
// gate/up) and 76 of 115 (Qwen T = 997, down): all tiles reach theirs together, so its latency is the launch's.
// Hence pair ids that are in LDS by then, stores of whole rows and h rows that do not wait in L2 (medians
// of kernel traces, us, that epilogue / this one: Mixtral T = 64 295 / 294 gate/up, 148 / 147 down, T = 333 328 / 320, 166 / 155;
// Qwen T = 600 146 / 147, 100 / 83, T = 997 152 / 149, 110 / 91).  A streaming load policy helps (T = 64 with the default
// policy: 323 us), as long as one tile reads the weights -- where an expert has several row tiles they find them in L2
// with the default policy only (T = 600, whole forward: 989 us streaming, 730 default).
// Tiled or register-resident kernels | mid-batch kernel | this one, gate/up and down phase, the same traces: Mixtral
// T = 64 308, 157 | 315, 144 | 294, 147; T = 128 330, 157 | 327, 151 | 302, 150; T = 333 347, 163 | 357, 213 | 320, 155
// (the down phase writes four f32 ranges here: combine 5.5 | 5.4 | 8.7); Qwen T = 600 171, 128 | 174, 111 | 147, 83;
// T = 997 180, 131 | -, 126 | 149, 91.
// Narrow tiles (NWV = 2: two waves, 128 weight rows by up to 64 token rows, four workgroups to a compute unit) for
// launches of wide ones whose last round is half empty (slab_widths, moe_abi.hip): DeepSeek-V2-Lite
// shape T = 48, down launch 45 us register-resident, 40 wide, 32 narrow; 256 experts of width 256 T = 64, gate/up 217 / 188.
// W8A16 layers (I8): the int8 blocks go into registers as they are stored, sixteen consecutive k to a lane, and
// the token fragments are read in the k order that gives; each unit's operands are widened to bf16 (exact) between
// the matrix instructions of the unit before, and the row scales multiply the f32 sums.  Half the bytes, so it is the
// widening beside the matrix instructions that shows where tiles are full: Mixtral shape, whole forward, us, widened
// right in front of their own unit / one unit ahead, T = 200 281 / 268, 1000 763 / 735, Qwen1.5-MoE shape T = 997
// 222 / 217; mid-batch and tiled kernels / this one (moe_abi.hip has the whole list): Mixtral T = 128 300 / 261, 300 420 / 317,
// Qwen T = 997 340 / 215.
// A fragment read of LDS feeds two matrix instructions of 32 clocks here, where the
// mid-batch kernel (ffn_stream.hip) reads the same KiB for two of 16 clocks, and a 256-row tile
// (ffn_tiled.hip) that holds 80 rows leaves two of the four SIMDs without matrix work.
#include <algorithm>

#include "ffn_tiled_common.h"

#include "../../include/atenia_moe_hip.h"

namespace atenia_moe {

namespace {

constexpr int kSlabRing = 4;           // A stages in LDS
// A workgroup of NWV waves: 64 NWV weight rows by up to 32 NWV token rows.
template <int NWV>
struct Slab {
  static constexpr int kRows = 32 * NWV;
  static constexpr int kStage = kRows * 64 * 2 / 16;      // uint4 per A stage
  // LDS of a workgroup: the A ring, reused by the epilogue of a bf16 down phase (NWV waves x
  // kRows rows x 144 bytes); in the down phase the pair ids of the tile's rows follow
  static constexpr int kEpilogue = NWV * kRows * 144;
  static constexpr int kRing = kSlabRing * kStage * 16;
  static constexpr int kLdsBytes = kRing > kEpilogue ? kRing : kEpilogue;
  static_assert(kLdsBytes >= NWV * 32 * 288 && kLdsBytes >= kRows * (64 * NWV + 16), "the other epilogues");
};
static_assert(Slab<4>::kRows == kSlabTileM && Slab<2>::kRows == kSlabNarrowM, "tiles of kernel 2's list");

struct SlabParams {
  const uint4* wa;       // gate (up phase) or down blocks
  const uint4* wb;       // up blocks
  const float* sa;       // int8: scales of the output rows [E, n_rows] of wa, wb
  const float* sb;
  int64_t w_stride_u4;   // between experts
  int n_rows;            // unpadded N
  int n_blocks;          // n_pad / 16
  int nkb;               // blocks per strip (32 k, int8: 64 k)
  int nst;               // 64-k stages (even)
  const uint16_t* a;     // bf16 rows
  int a_stride;
  void* out;
  int out_stride;
  const int32_t* perm;
  FastDiv pair_div;
  const RowTile* tiles;        // kernel 2's list (tiles of up to kSlabRows rows), or null: one group of
  const int32_t* n_tiles;      // rows_fixed rows (shared expert)
  int max_groups;              // 32-row groups a tile of the list may hold: 4, or 2
  int rows_fixed;
  uint32_t fixed_inv;          // tiles == null: tile_inv of the number of tiles
  int nct;                     // column tiles
  int parts;                   // k ranges per tile (down phase)
  FastDiv part_div, col_div, row_tile_div, rot_div;  // by parts, by nct, by nct * parts, by nst_min
  int nst_min;                 // stages of the shortest k range
  int out_bf16;                // down phase in one k range: y leaves as bf16 (nearest even) instead of f32
  size_t out_part_stride;      // elements between the partial output buffers
};

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// (vector types all the way: through the uint4 struct each operand became four 32-bit values that
// the register allocator put together again with copies and spills)
__device__ inline f32x16 mfma32v(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                 c, 0, 0, 0);
}
constexpr int kRsrcWord3 = 0x00020000;  // buffer resource: raw, 32-bit data format
constexpr int kNonTemporal = 2;         // cache policy of buffer loads: weights are read once
constexpr int kWriteThrough = 16;       // cache policy of buffer stores: agent scope

// Eight int8 values -> eight bf16 (exact).
__device__ inline u32x4 widen_i8x8(uint32_t lo, uint32_t hi) {
  return u32x4{pack_i8_pair(lo, 0), pack_i8_pair(lo, 16), pack_i8_pair(hi, 0), pack_i8_pair(hi, 16)};
}

template <bool UP, bool I8, int NWV>
__device__ __forceinline__ void slab_tile(const SlabParams& p, int wid, u32x4* S) {
  // ---- which tile ------------------------------------------------------------------------
  // Workgroup ids are dealt round-robin to the eight XCDs; XCD x takes a contiguous run of the
  // logical order expert > k range > column tile > row tile, so the row tiles that read the same
  // weights are neighbours on one XCD's L2, and an expert's token rows stay in few L2s: of the shared expert,
  // whose rows are the whole batch's, an XCD reads the columns of one k range.  (Column tile > k range, where every XCD
  // reads all of them, whole forward, us: Qwen1.5-MoE shape T = 200 213.0 / 211.6, 600 254.1 / 251.2, int8 T = 200 138.3 / 136.7.)
  typedef Slab<NWV> L;
  constexpr int kSlabRows = L::kRows, kSlabStage = L::kStage, kSlabLdsBytes = L::kLdsBytes;
  const bool fixed = p.tiles == nullptr;
  const int n_row_tiles = fixed ? (p.rows_fixed + kSlabRows - 1) / kSlabRows : uniform_load(p.n_tiles);
  const int per_row_tile = p.nct * p.parts;
  const int total = n_row_tiles * per_row_tile;
  const int per_xcd = (total + 7) >> 3;
  const int slot = wid >> 3;
  const int logical = (wid & 7) * per_xcd + slot;
  if (slot >= per_xcd || logical >= total) return;
  int first = 0, nt = n_row_tiles;
  RowTile of{0, 0, p.rows_fixed, p.fixed_inv};
  if (!fixed) {
    const int rt_any = div_by(logical, p.row_tile_div);
    of = uniform_load(p.tiles + rt_any);
    first = rt_any - (int)(of.e_i >> 16);
    nt = expert_tiles(of.rows, p.max_groups);
  }
  const int in_expert = logical - first * per_row_tile, col = div_tiles(in_expert, nt, of.inv);
  const int rl = in_expert - col * nt;
  const int part = div_by(col, p.col_div), ct = col - part * p.nct;
  const int e = (int)(of.e_i & 0xffff), base = of.base;
  int tm0, rows_here;
  if (fixed) {
    tm0 = rl * kSlabRows;
    rows_here = min(kSlabRows, p.rows_fixed - tm0);
  } else {
    expert_tile(of.rows, p.max_groups, nt, of.inv, rl, tm0, rows_here);
  }

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kh = lane >> 5, l32 = lane & 31;
  const int st_lo = div_by(p.nst / 2 * part, p.part_div) * 2, st_hi = div_by(p.nst / 2 * (part + 1), p.part_div) * 2;
  const int nst = st_hi - st_lo;

  // ---- weights ---------------------------------------------------------------------------
  // column group c of this wave: 32 weight rows = two 16-row strips.  The loads are buffer loads
  // bounded by the expert's matrix: a stage past the end of K is requested at an offset outside of
  // it, which reads zeros and costs no memory traffic, so that the loop has one form and every
  // stage the same number of loads in flight.
  constexpr int kTileStrips = UP ? 2 * NWV : 4 * NWV;  // 16-row strips of wa per tile
  const int nb0 = ct * kTileStrips;
  const uint32_t w_bytes = (uint32_t)p.n_blocks * p.nkb * kChunk;
  const __amdgpu_buffer_rsrc_t wr[2] = {
      __builtin_amdgcn_make_buffer_rsrc((void*)(p.wa + (size_t)e * p.w_stride_u4), 0, w_bytes, kRsrcWord3),
      __builtin_amdgcn_make_buffer_rsrc((void*)((UP ? p.wb : p.wa) + (size_t)e * p.w_stride_u4), 0, w_bytes,
                                        kRsrcWord3)};
  uint32_t wv[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    // (strips past N read zeros and are never stored)
    const int nb = nb0 + (UP ? wave * 2 : wave * 4 + c * 2) + (l32 >> 4);
    wv[c] = nb >= p.n_blocks ? 0x80000000u : (uint32_t)(nb * p.nkb) * kChunk + (kh * 16 + (l32 & 15)) * 16;
    asm volatile("" : "+v"(wv[c]));
  }
  // k16 unit u of stage st (a stage index of the whole K; dead: reads zeros).  int8: a lane's 16 bytes are
  // sixteen consecutive k, the operands of two units, so unit u < 2 loads those of units 2 u and 2 u + 1.
  constexpr int LW = I8 ? 4 : 8;  // weight registers (of 16 bytes) per stage
  auto load_w = [&](auto once_c, u32x4 (&w)[LW], int st, uint32_t dead, int u) {
    constexpr int kPolicy = decltype(once_c)::value ? kNonTemporal : 0;
    const int soff = st * (I8 ? kChunk : 2 * kChunk);
#pragma unroll
    for (int c = 0; c < 2; ++c)
      w[2 * u + c] = __builtin_amdgcn_raw_buffer_load_b128(
          wr[c], (wv[c] | dead) + (I8 ? 0 : (u >> 1) * kChunk) + (I8 ? u : u & 1) * (kChunk / 2), soff, kPolicy);
  };
  // Tiles walk K from different first stages and wrap around: paced by one memory system they
  // would otherwise all read the same offset of strips that lie a power of two apart, i.e. few
  // memory channels.  The first stage depends on the column tile and the expert only, so a row's
  // sums do not depend on the rest of the batch.
  // (Nor on the tile's width: the column tiles of half the width count in pairs.)
  const int spread = (NWV == 4 ? ct : ct >> 1) * 13 + e * 29, rot = spread - div_by(spread, p.rot_div) * p.nst_min;
  auto at = [&](int st) {
    const int sc = min(st, nst - 1) + rot;
    return st_lo + (sc >= nst ? sc - nst : sc);
  };
  auto dead = [&](int st) { return st < nst ? 0u : 0x80000000u; };

  // ---- token rows ------------------------------------------------------------------------
  const int rg = (rows_here + 31) >> 5;

  // RG: 32-row groups of the tile; once_c: no other tile of the expert reads these weights
  auto run = [&](auto rg_c, auto once_c) {
    constexpr int RG = decltype(rg_c)::value;
    // Stages of weights in flight.  (16 KiB per wave; int8 tiles of four row groups have the registers
    // for three stages of 4 KiB.)
    constexpr int NS = I8 ? (RG <= 2 ? 4 : 3) : 2;
    float scale[2] = {1.f, 1.f};  // of this lane's columns
    if (I8) {
      const int n = nb0 * 16 + (UP ? wave * 32 : wave * 64) + l32;
      scale[0] = p.sa[(size_t)e * p.n_rows + min(n, p.n_rows - 1)];
      scale[1] = UP ? p.sb[(size_t)e * p.n_rows + min(n, p.n_rows - 1)]
                    : p.sa[(size_t)e * p.n_rows + min(n + 32, p.n_rows - 1)];
    }
    f32x16 acc[RG][2];
#pragma unroll
    for (int i = 0; i < RG; ++i)
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][c][r] = 0.f;
    // 4 RG chunks of 8 rows per stage, CW per wave.  Row r, 16-byte segment s of chunk q sits at
    // slot 8 r + (s ^ r ^ (q & 1)).
    constexpr int CW = 4 * RG / NWV;
    uint32_t arow[CW];  // byte offset of this lane's 16 bytes from p.a
    {
      const int r8 = lane >> 3, pslot = lane & 7, row0 = base + tm0;
      int src[CW];
      source_rows<UP>(p.perm, p.pair_div, row0, row0 + wave * CW * 8, row0 + rows_here, r8, src);
#pragma unroll
      for (int q = 0; q < CW; ++q) {
        arow[q] = (uint32_t)src[q] * (uint32_t)(p.a_stride * 2) + (pslot ^ r8 ^ ((wave * CW + q) & 1)) * 16;
        asm volatile("" : "+v"(arow[q]));  // (a register of its own, not half of a 64-bit product)
      }
    }
    if (!UP) {
      // the pair ids of the tile's rows, for the epilogue
      if (wave * 64 < rows_here)
        dma4_at(p.perm + base + tm0, min(wave * 64 + lane, rows_here - 1) * 4,
                (uint32_t)(uintptr_t)(lptr_t)S + kSlabLdsBytes + wave * 256);
    }
    const uint32_t fill = (uint32_t)(uintptr_t)(lptr_t)S + wave * CW * kChunk;
    auto dma_a = [&](int buf, int st) {
#pragma unroll
      for (int q = 0; q < CW; ++q)
        dma16_at((const char*)p.a + (size_t)st * 128, arow[q], fill + buf * (kSlabStage * 16) + q * kChunk);
    };
    // fragment of row group 0, unit 0; unit u flips bits of the segment, group i is 4 KiB on.  The eight k
    // that a half wave multiplies in unit u are segment 2 u + kh of the stage; int8, whose lanes hold sixteen
    // consecutive k, segment 4 (u / 2) + 2 kh + u % 2.
    const int aoff0 = (l32 >> 3) * 64 + (l32 & 7) * 8 + ((I8 ? 2 * kh : kh) ^ (l32 & 7) ^ ((l32 >> 3) & 1));
    auto unit_seg = [](int u) { return I8 ? 4 * (u >> 1) + (u & 1) : 2 * u; };
    auto fence = [&]() {
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
    };
    // One stage: four k16 units.  Stage st + NS of the weights is requested into the registers
    // each unit frees, stage st + 3 of the token rows into the LDS stage freed by the barrier.
    // int8: the operands of a unit are widened while the unit before multiplies (w_next: the registers
    // of the next stage).
    u32x4 b[2][2];
    auto widen = [&](u32x4 (&w)[LW], int u) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const u32x4 v = w[2 * (u >> 1) + c];
        b[u & 1][c] = u & 1 ? widen_i8x8(v[2], v[3]) : widen_i8x8(v[0], v[1]);
      }
    };
    auto stage = [&](u32x4 (&w)[LW], u32x4 (&w_next)[LW], int st) {
      wait_vm_lgkm0<2 * CW + (I8 ? 12 : 8)>();
      fence();
      const int a_st = aoff0 + (st & (kSlabRing - 1)) * kSlabStage;
      dma_a((st + 3) & (kSlabRing - 1), at(st + 3));
      const int nxt = at(st + NS);
      const uint32_t past = dead(st + NS);
      u32x4 fa[2][RG];
#pragma unroll
      for (int i = 0; i < RG; ++i) fa[0][i] = S[a_st + i * 256];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (u < 3) {  // the next unit's fragments are read while this one multiplies
#pragma unroll
          for (int i = 0; i < RG; ++i) fa[(u + 1) & 1][i] = S[(a_st ^ unit_seg(u + 1)) + i * 256];
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int i = 0; i < RG; ++i) {
          acc[i][0] = mfma32v(fa[u & 1][i], I8 ? b[u & 1][0] : w[2 * u], acc[i][0]);
          acc[i][1] = mfma32v(fa[u & 1][i], I8 ? b[u & 1][1] : w[2 * u + 1], acc[i][1]);
        }
        if (I8) {
          widen(u < 3 ? w : w_next, (u + 1) & 3);
#pragma unroll
          for (int i = 0; i < 2 * RG; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);                        // one matrix instruction,
            __builtin_amdgcn_sched_group_barrier(0x2, (24 + 2 * RG - 1) / (2 * RG), 0);  // its share of the widening
          }
        }
        if (!I8) load_w(once_c, w, nxt, past, u);
        else if (u == 0 || u == 2) load_w(once_c, w, nxt, past, u >> 1);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // Loads complete in issue order.  A stage issues CW row loads and then LW weight loads, and
    // needs its own row loads, which went out three stages ago: behind them are the row loads of
    // the next two stages and the weight loads of three, int8 (LW = 4) 2 CW + 12 in all; the first stages have
    // their row loads in front of the loop and NS LW weight loads behind them, which is no fewer.  bf16 (LW = 8) waits
    // further, for all but the eight of one: its own weights, which go out one stage later than its rows, are due then anyway.
    // (The first weight loads stand right in front of the loop: with a branch in between, the
    // allocator gives them registers of their own and copies -- that is, waits for -- them.)
#pragma unroll
    for (int t = 0; t < 3; ++t) dma_a(t, at(t));
    u32x4 w[NS][LW];
#pragma unroll
    for (int t = 0; t < NS; ++t)
#pragma unroll
      for (int u = 0; u < LW / 2; ++u) load_w(once_c, w[t], at(t), dead(t), u);
    if (I8) widen(w[0], 0);
    int st = 0;
#pragma clang loop unroll(disable)
    do {  // K comes in pairs of stages (slab_supported)
      stage(w[0], w[1], st);
      if (NS == 3 && st + 1 == nst) break;
      stage(w[1], w[NS > 2 ? 2 : 0], st + 1);
      if (NS > 2 && st + 2 == nst) break;
      if (NS > 2) stage(w[NS > 2 ? 2 : 0], w[NS > 3 ? 3 : 0], st + 2);
      if (NS > 3) stage(w[NS > 3 ? 3 : 0], w[0], st + 3);
      st += NS;
    } while (st < nst);
    wait_vm_lgkm0<0>();

    // ---- epilogue --------------------------------------------------------------------------
    // D register r of lane l: row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32.
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();  // every wave's loads have landed and its reads are done
    asm volatile("" ::: "memory");
    char* lds = (char*)S;
    const int32_t* pair_of = (const int32_t*)(lds + kSlabLdsBytes);
    if (UP) {
      // h = silu(g) * u as bf16; the waves' 32 columns each are put side by side in LDS so
      // that a row leaves as full 128-byte lines
      constexpr int kPitch = 64 * NWV + 16;
  #pragma unroll
      for (int i = 0; i < RG; ++i) {
        {
  #pragma unroll
          for (int r = 0; r < 16; r += 2) {
            const int m = i * 32 + 8 * (r >> 2) + 4 * kh + (r & 3);
            const uint32_t hh =
                I8 ? bf16_rne_pair(swiglu_fast(acc[i][0][r] * scale[0], acc[i][1][r] * scale[1]),
                                   swiglu_fast(acc[i][0][r + 1] * scale[0], acc[i][1][r + 1] * scale[1]))
                   : bf16_rne_pair(swiglu_fast(acc[i][0][r], acc[i][1][r]),
                                   swiglu_fast(acc[i][0][r + 1], acc[i][1][r + 1]));
            char* dst = lds + m * kPitch + (wave * 32 + l32) * 2;
            *(uint16_t*)dst = (uint16_t)hh;
            *(uint16_t*)(dst + kPitch) = (uint16_t)(hh >> 16);
          }
        }
      }
      __syncthreads();
      // Written through to memory where there are many rows: left dirty in L2, the rows of every tile would
      // go there together when the launch ends (launch, Mixtral shape T = 333 329 / 320 us, Qwen1.5-MoE shape
      // T = 997 151 / 149; with one row group the stores' way to memory is the longer one, Mixtral T = 64
      // 294 / 297).
      constexpr int kPolicy = RG >= 2 ? kWriteThrough : 0;
      const __amdgpu_buffer_rsrc_t hr = __builtin_amdgcn_make_buffer_rsrc(
          (uint16_t*)p.out + (size_t)(base + tm0) * p.out_stride, 0, rows_here * p.out_stride * 2, kRsrcWord3);
      const int c16 = tid & (4 * NWV - 1), n = nb0 * 16 + c16 * 8;
      if (n < p.n_blocks * 16)
        for (int m = tid / (4 * NWV); m < rows_here; m += 16)
          __builtin_amdgcn_raw_buffer_store_b128(*(const u32x4*)(lds + m * kPitch + c16 * 16), hr,
                                                 (m * p.out_stride + n) * 2, 0, kPolicy);
    } else if (!I8 && p.out_bf16) {
      // y as bf16: each wave's 64 columns are one full line per row, staged in its own region
      constexpr int kPitch = 144;
      char* mine = lds + wave * (kSlabRows * kPitch);
  #pragma unroll
      for (int i = 0; i < RG; ++i) {
        {
  #pragma unroll
          for (int c = 0; c < 2; ++c)
  #pragma unroll
            for (int r = 0; r < 16; r += 2) {
              const int m = i * 32 + 8 * (r >> 2) + 4 * kh + (r & 3);
              const uint32_t hh = bf16_rne_pair(acc[i][c][r], acc[i][c][r + 1]);
              char* dst = mine + m * kPitch + (c * 32 + l32) * 2;
              *(uint16_t*)dst = (uint16_t)hh;
              *(uint16_t*)(dst + kPitch) = (uint16_t)(hh >> 16);
            }
        }
      }
      uint16_t* y = (uint16_t*)p.out;
      const int c8 = lane & 7, n = nb0 * 16 + wave * 64 + c8 * 8;
      for (int m = lane >> 3; m < rows_here; m += 8) {
        const int pair = pair_of[m];
        if (n < p.n_rows)
          *(uint4*)(y + (size_t)pair * p.out_stride + n) = *(const uint4*)(mine + m * kPitch + c8 * 16);
      }
    } else {
      // y (or the sums of a k range) as f32, a row group at a time: each wave's 64 columns of 32 rows go to
      // its own region (a pitch of 72 values keeps the two half waves on different banks) and leave 16 bytes
      // per lane, four rows a store.  Straight from the accumulators it was four times the stores, each
      // behind a pair id fetched from memory there and then.
      constexpr int kPitch = 288;
      char* mine = lds + wave * (32 * kPitch);
      float* y = (float*)p.out + (size_t)part * p.out_part_stride;
      const int c16 = lane & 15, n = nb0 * 16 + wave * 64 + c16 * 4;
  #pragma unroll
      for (int i = 0; i < RG; ++i) {
  #pragma unroll
        for (int c = 0; c < 2; ++c)
  #pragma unroll
          for (int r = 0; r < 16; ++r)
            *(float*)(mine + (8 * (r >> 2) + 4 * kh + (r & 3)) * kPitch + (c * 32 + l32) * 4) =
                I8 ? acc[i][c][r] * scale[c] : acc[i][c][r];
  #pragma unroll
        for (int it = 0; it < 8; ++it) {
          const int m = it * 4 + (lane >> 4);
          const u32x4 v = *(const u32x4*)(mine + m * kPitch + c16 * 16);
          if (i * 32 + m < rows_here && n < p.n_rows)
            *(u32x4*)(y + (size_t)pair_of[i * 32 + m] * p.out_stride + n) = v;
        }
      }
    }
  };
  auto pick = [&](auto once_c) {
    if (rg <= 1) run(std::integral_constant<int, 1>{}, once_c);
    else if (rg == 2 || NWV == 2) run(std::integral_constant<int, 2>{}, once_c);
    else if (rg == 3) run(std::integral_constant<int, NWV == 4 ? 3 : 2>{}, once_c);
    else run(std::integral_constant<int, NWV>{}, once_c);
    static_assert(NWV == 4 || NWV == 2, "row groups of a tile");
  };
  if (nt == 1) pick(std::integral_constant<bool, true>{});
  else pick(std::integral_constant<bool, false>{});
}

// Tiles of p1 and of p2: the routed experts' and the shared expert's, or one of the two alone.  In eights of
// workgroups (one per XCD): n1 of p1 and the others of p2, or, turns > 0, one of each in turn as long as there are of p2 (`turns`
// eights, fewer than n1) and what is left of p1.
template <bool UP, bool I8, int NWV>
__global__ __launch_bounds__(64 * NWV, 2) void ffn_slab_kernel(SlabParams p1, SlabParams p2, int n1, int turns) {
  __shared__ u32x4 S[(Slab<NWV>::kLdsBytes + (UP ? 0 : Slab<NWV>::kRows * 4)) / 16];
  const int eight = blockIdx.x >> 3;
  const bool second = turns > 0 ? eight < 2 * turns && eight & 1 : eight >= n1;
  const int wid = (int)(blockIdx.x & 7) +
                  8 * (turns > 0 ? (eight < 2 * turns ? eight >> 1 : eight - turns) : eight - (second ? n1 : 0));
  SlabParams p;
  // (field by field: selecting between two by-value arguments by reference would copy them to the stack)
#define ATENIA_PICK(f) p.f = second ? p2.f : p1.f
  ATENIA_PICK(wa); ATENIA_PICK(wb); ATENIA_PICK(sa); ATENIA_PICK(sb); ATENIA_PICK(w_stride_u4); ATENIA_PICK(n_rows); ATENIA_PICK(n_blocks);
  ATENIA_PICK(nkb); ATENIA_PICK(nst); ATENIA_PICK(a); ATENIA_PICK(a_stride); ATENIA_PICK(out);
  ATENIA_PICK(out_stride); ATENIA_PICK(perm); ATENIA_PICK(pair_div.mul); ATENIA_PICK(pair_div.shift);
  ATENIA_PICK(tiles); ATENIA_PICK(n_tiles); ATENIA_PICK(max_groups); ATENIA_PICK(rows_fixed); ATENIA_PICK(nct); ATENIA_PICK(out_bf16); ATENIA_PICK(parts);
  ATENIA_PICK(out_part_stride); ATENIA_PICK(fixed_inv); ATENIA_PICK(nst_min);
  ATENIA_PICK(part_div.mul); ATENIA_PICK(part_div.shift); ATENIA_PICK(col_div.mul); ATENIA_PICK(col_div.shift); ATENIA_PICK(row_tile_div.mul);
  ATENIA_PICK(row_tile_div.shift); ATENIA_PICK(rot_div.mul); ATENIA_PICK(rot_div.shift);
#undef ATENIA_PICK
  slab_tile<UP, I8, NWV>(p, wid, S);
}

// The row-tile list is one whose tiles the launch can hold.
bool slab_list(const FfnArgs& a) {
  return a.tiles && (a.max_tile_groups == 2 || (a.max_tile_groups == 4 && !a.slab_narrow));
}
int slab_rows(const FfnArgs& a) { return a.slab_narrow ? kSlabNarrowM : kSlabTileM; }
SlabParams slab_params(const FfnArgs& a, const WeightSet& w, bool shared) {
  SlabParams p{};
  p.w_stride_u4 = w.expert_stride / 16;
  p.n_rows = w.n_rows;
  p.n_blocks = w.n_pad / 16;
  p.nkb = w.k_pad / (a.wdtype == ATENIA_MOE_WEIGHT_BF16 ? kKbBf16 : kKbInt8);
  p.nst = w.k_pad / 64;
  p.perm = a.g.perm;
  p.pair_div = fast_div(a.g.pair_div);
  if (!shared) {
    p.tiles = a.tiles;
    p.n_tiles = a.n_tiles;
    p.max_groups = a.max_tile_groups;
  }
  p.rows_fixed = a.rows_max;
  p.fixed_inv = tile_inv((a.rows_max + slab_rows(a) - 1) / slab_rows(a));
  p.parts = 1;
  return p;
}
void slab_divisions(SlabParams& p) {
  p.part_div = fast_div(p.parts);
  p.col_div = fast_div(p.nct);
  p.row_tile_div = fast_div(p.nct * p.parts);
  p.nst_min = p.nst / 2 / p.parts * 2;
  p.rot_div = fast_div(p.nst_min);
}
SlabParams slab_up_params(const FfnArgs& a, bool shared) {
  SlabParams p = slab_params(a, a.gate, shared);
  p.wa = (const uint4*)a.gate.w;
  p.wb = (const uint4*)a.up.w;
  p.sa = a.gate.scale;
  p.sb = a.up.scale;
  p.a = (const uint16_t*)a.x;
  p.a_stride = a.x_stride;
  p.out = a.h;
  p.out_stride = a.h_stride;
  p.nct = (p.n_blocks * 16 + slab_rows(a) - 1) / slab_rows(a);  // as many gate rows as token rows
  slab_divisions(p);
  return p;
}
SlabParams slab_down_params(const FfnArgs& a, bool shared) {
  SlabParams p = slab_params(a, a.down, shared);
  p.wa = (const uint4*)a.down.w;
  p.sa = a.down.scale;
  p.a = (const uint16_t*)a.h;
  p.a_stride = a.h_stride;
  p.out = a.y;
  p.out_stride = a.y_stride;
  p.nct = (p.n_blocks * 16 + 2 * slab_rows(a) - 1) / (2 * slab_rows(a));
  p.out_bf16 = a.y_bf16;
  if (a.y_parts > 1) {  // (every tile has as many: the combine is told by the host)
    p.parts = a.y_parts;
    p.out_part_stride = a.y_part_stride;
  }
  slab_divisions(p);
  return p;
}
// Workgroups without a tile leave at once, but where all others find a place at once (two to a compute unit) each takes a
// turn of the round-robin that deals those out: units that it passes over have none while others have three.  Such launches
// have no more row tiles than the list can hold.  (Two more, whole forward, us, with / without: 16 experts of width 1536, shared
// one of 3072, d = 5120, T = 54 190 / 167, 100 225 / 194.  Beyond that the workgroups wait for places and their number is a matter of
// luck: DeepSeek-V2-Lite shape T = 48 127 / 129, 300 190 / 195, 256 experts of width 256, d = 7168, T = 36 326 / 310.)
int slab_grid(const FfnArgs& a, const SlabParams& p) {
  constexpr int places = 2 * 256;
  const int per = p.nct * p.parts;
  const int tiles = !p.tiles ? (p.rows_fixed + slab_rows(a) - 1) / slab_rows(a)
                             : (long long)a.list_row_tiles * per <= places ? a.list_row_tiles : a.max_row_tiles;
  return (tiles * per + 7) / 8 * 8;
}
template <bool UP>
hipError_t launch_slab(const FfnArgs& a, const SlabParams& p1, int grid1, const SlabParams& p2, int grid2, hipStream_t s) {
  const bool i8 = a.wdtype != ATENIA_MOE_WEIGHT_BF16;
  // int8 batches of 65 to 640 tokens whose shared tiles are no more than two fifths of the routed ones: in turn.  The shared
  // expert's tiles, full of rows, wait for the matrix cores and the routed ones for their weights; smaller and larger batches
  // keep one after the other: the first have few such tiles, the last several row tiles that find each other's weights in
  // L2.  Whole forward, shared gate/up tiles as a share of the routed ones: in turn / one after the other, T = 66 to 640:
  //   up to 0.10  0.92-1.02 (128 experts of width 768, d = 2048 T = 100 0.92; 32 of width 2048, d = 4096 T = 128 0.88, 640 0.93;
  //               DeepSeek-V2-Lite shape T = 66 0.98, 128 0.97, 420 0.94), T = 48 0.94-1.00
  //   0.10-0.40   0.84-1.02, once 1.06 (Qwen1.5-MoE shape T = 200 0.97, 300 0.91, 640 0.96; 16 of width 1408, d = 2048, 0.88-0.89)
  //   0.50-2.0    0.98-1.10, once 0.87 (16 of width 4096 beside one of 16384 T = 420 1.08; 8 and one of width 8192, d = 5120 T = 420 1.05)
  // and from T = 800 on 0.96-1.11 (Qwen1.5-MoE shape 800 1.02, 2500 1.05).  bf16 layers, which wait for weights longer:
  // Qwen1.5-MoE shape T = 80 203 / 207 us one after the other / in turn, 600 252.6 / 254.5, 997 280.7 / 276.2, 1700 373 / 378.
  const int n1 = grid1 / 8;
  const int turns = i8 && a.rows_max > 64 && a.rows_max <= 640 && 5 * (long long)grid2 <= 2 * (long long)grid1 ? grid2 / 8 : 0;
  const int grid = grid1 + grid2;
  if (a.slab_narrow) {
    if (i8) ffn_slab_kernel<UP, true, 2><<<grid, 128, 0, s>>>(p1, p2, n1, turns);
    else ffn_slab_kernel<UP, false, 2><<<grid, 128, 0, s>>>(p1, p2, n1, turns);
  } else {
    if (i8) ffn_slab_kernel<UP, true, 4><<<grid, 256, 0, s>>>(p1, p2, n1, turns);
    else ffn_slab_kernel<UP, false, 4><<<grid, 256, 0, s>>>(p1, p2, n1, turns);
  }
  return hipGetLastError();
}
}  // namespace

bool slab_supported(const WeightSet& w, int wdtype) {
  const bool type_ok = wdtype == ATENIA_MOE_WEIGHT_BF16 ? !w.scale : wdtype == ATENIA_MOE_WEIGHT_INT8_W8A16;
  return type_ok && w.group_blocks == 0 && w.k_pad % 128 == 0 &&
         w.n_pad >= 16 && (int64_t)w.n_pad * w.k_pad * 2 < ((int64_t)1 << 31);  // offsets in one expert's matrix
}

// Until every compute unit has two tiles (a constant: whatever the device; tiles_per_expert: 1, and more for
// W8A16 batches whose experts see more than a tile's rows).
int slab_down_parts(const WeightSet& down, int n_experts, int tiles_per_expert) {
  constexpr int n_cus = 256;
  const int tiles = n_experts * ((down.n_pad + 255) / 256) * tiles_per_expert;
  const int nst = down.k_pad / 64;
  int parts = 1;
  while (parts < 4 && tiles * parts * 2 <= 2 * n_cus && nst / (parts * 2) >= 8) parts *= 2;
  return parts;
}

// The shared expert's tiles as long as a routed expert's, whatever the batch: a row's sums must not depend
// on the rows beside it.  (Half as many ranges are slower while their tiles are few and faster from some 500
// rows on, where the partial sums cost more than the longer tiles: as long / twice as long, whole forward, us,
// Qwen1.5-MoE shape T = 64 204 / 218, 130 218 / 230, 400 241 / 247, 600 265 / 254, 997 298 / 291, 1700 393 / 383;
// DeepSeek-V2-Lite shape T = 64 156 / 170, 200 197 / 210, 700 246 / 241, 1000 313 / 308.)
// row_tiles (W8A16 batches of more than 640 tokens, where the kernels they took before depended on the batch
// too; 0 otherwise): until the shared expert has 128 tiles (as long as a routed one / until 256 / until 128:
// Qwen1.5-MoE shape, T = 997 223 / 222 / 215, 2000 378 / 366 / 359, 4500 707 / 672 / 670, 12288 1753 / 1646 / 1648).
// down_parts (W8A16 batches of up to that many tokens; 1 otherwise): the ranges that a routed expert's tiles are cut into, so
// that the shared expert's are as long as those and not as the whole K (whole / as long, whole forward, us: 8 experts and a
// shared one of width 8192, d = 5120, T = 36 240 / 213, 64 252 / 224, 200 277 / 247, 600 381 / 385; of width 2048, d = 2048,
// T = 24 57 / 50, 64 65 / 55, 300 82 / 69, 640 107 / 100; 16 of width 4096, d = 4096, T = 70 198 / 185, 640 271 / 274, 1500 500 / 506).
int slab_shared_down_parts(const WeightSet& shared_down, const WeightSet& down, int down_parts, int row_tiles) {
  int parts = std::max(1, std::min(4, shared_down.k_pad * down_parts / std::max(down.k_pad, 512)));
  while (parts > 1 && row_tiles * ((shared_down.n_pad + 255) / 256) * parts > kSlabSharedTiles) parts /= 2;
  return parts;
}

hipError_t launch_slab_up(const FfnArgs& a, const FfnArgs* shared, hipStream_t s) {
  if (!slab_supported(a.gate, a.wdtype) || !slab_list(a)) return hipErrorInvalidValue;
  const SlabParams p = slab_up_params(a, false);
  const int n1 = slab_grid(a, p);
  SlabParams ps = p;
  int n2 = 0;
  if (shared) {
    if (!slab_supported(shared->gate, shared->wdtype)) return hipErrorInvalidValue;
    ps = slab_up_params(*shared, true);
    n2 = slab_grid(*shared, ps);
  }
  return launch_slab<true>(a, p, n1, ps, n2, s);
}

hipError_t launch_slab_down(const FfnArgs& a, const FfnArgs* shared, hipStream_t s) {
  if (!slab_supported(a.down, a.wdtype) || !slab_list(a)) return hipErrorInvalidValue;
  if (a.down.n_rows % 4 || (shared && shared->down.n_rows % 4)) return hipErrorInvalidValue;  // 16 bytes per lane
  // bf16: a lane stores 8 columns at once; the sums of k ranges are f32
  if (a.y_bf16 && (a.down.n_rows % 8 || a.y_parts > 1)) return hipErrorInvalidValue;
  if (shared && shared->y_bf16 && (shared->down.n_rows % 8 || shared->y_parts > 1)) return hipErrorInvalidValue;
  const SlabParams p = slab_down_params(a, false);
  const int n1 = slab_grid(a, p);
  SlabParams ps = p;
  int n2 = 0;
  if (shared) {
    if (!slab_supported(shared->down, shared->wdtype)) return hipErrorInvalidValue;
    ps = slab_down_params(*shared, true);
    n2 = slab_grid(*shared, ps);
  }
  // the shared expert's tiles (the longer K) first
  return shared ? launch_slab<false>(a, ps, n2, p, n1, s) : launch_slab<false>(a, p, n1, p, 0, s);
}

}  // namespace atenia_moe
