// Recompute path: the SwiGLU expert MLP of the slots that are not reused,
// grouped over experts, on bf16/fp16 matrix cores.
//
// Replaces the reference's per-expert loop (models/qwen3_vl_moe/
// cached_layers.py:431-437: index_select the expert's tokens, run the expert,
// scatter into collected[token, slot]) and its CUTLASS expert MLP
// (ops/csrc/fp16_fused_expert/fp16_fused_moe_mlp.cu:107-274 with the SiLU-mul
// epilogue of fp16_epilogue_utils.h:51-125):
//   g = dtype(x W1^T)                      (fp32 accumulation, one rounding)
//   f = dtype(silu(g) * (x W3^T))          (up projection unrounded, silu in fp32)
//   y = dtype(f W2^T)
//
// tm_group_slots (one workgroup) buckets the recomputed (token, slot) pairs
// by expert: per-expert counts in LDS, offsets, one row per pair (token and
// the element offset of its output row in the slot layout), and the list of
// BM-row tiles of every expert.  The order of rows inside an expert is that
// of LDS atomics; every output row is computed the same way wherever its row
// sits in a tile, so results do not depend on it.
//
// The two GEMMs of a tile run in one of two kernels, with the same bits:
// skinny_gemm_kernel (few rows: one wave per column group, bound by the stream
// of weights) and tile_gemm_kernel (eight waves per 256-row tile).  Both move K
// in BK-wide stages global -> LDS by direct loads (16-byte chunks XOR-swizzled
// by row, so the operand reads of 32 rows spread over the banks).  The up GEMM
// multiplies W1 and W3 against the same activation operands and applies the
// SiLU-mul; the down GEMM writes each row to its slot of the output.
//
// Packed path (tm_expert_pack_weights, tm_grouped_swiglu_packed,
// tm_expert_swiglu_packed): each weight tile is stored stage by stage in the
// LDS slot order, so a stage's weight tile is one contiguous read; the up
// GEMM then writes the intermediate in the same stage order (whole 256-row
// tiles) and the down GEMM reads its A stages contiguously.  Same arithmetic,
// same bits.
#include "tm_internal.h"
#include "tm_dma.h"
#include "tm_mfma.h"

namespace {

constexpr int BM = 256, BK = 32, kThreads = 256;
constexpr int kMinBN = 128;                  // column tile of the up GEMM (and of narrow down GEMMs)
constexpr int kCPR = BK / 8;                 // 16-byte chunks per tile row and stage

enum { kModeUp = 0, kModeDown = 1 };

// Slot of (row, 16-byte chunk kc) in a stage.  A row is 64 bytes, so four
// rows share one 256-byte line of the 64 banks, which a 16-byte read serves
// 16 lanes at a time; XOR-ing the chunk with (row / 4) % 4 puts 16
// consecutive rows on 16 distinct 16-byte bank groups, and an operand read
// (one chunk of 32 consecutive rows) is conflict-free.
__device__ __forceinline__ int swz_chunk(int row, int kc) { return kc ^ ((row >> 2) & (kCPR - 1)); }

// Tile source: the grouped tile list (tiles != nullptr: [0] rows, [1] tiles,
// then tile_expert[t_max], tile_row0[t_max]) or one dense expert of `rows`.
struct TileSrc {
  const int32_t *tiles;
  const int32_t *expert_offsets;
  int64_t t_max;
  int32_t rows;
};

// Few rows per expert (a decode batch, a short prompt, one token through one
// expert): the MLP is a stream of the experts' weights, and 256-row tiles put
// it on few workgroups (6 for one expert of 768 intermediate columns) that
// each wait for a stage at every barrier.  Here one wave is a workgroup: it
// owns CW output columns of one expert's tile and streams their weight rows
// and up to RBMAX activation rows through an LDS ring of its own (direct
// global -> LDS loads, no barrier anywhere), LDS bytes deep, so a CU's waves
// keep it filled and even a single expert spreads over one wave per CW
// columns.  16 KiB rings (10 waves per CU) measured 30 + 17 us (up + down) on
// a decode batch of 28 experts, 40 KiB ones 36 + 20 (the last round of waves
// is then less even).  Where waves are few, stages of two sub-stages halve the
// LDS round trips per column (one expert, one row: up 8.5 -> 6.9 us).
//
// A = weight rows (up: the gate and up rows of the same columns, so a lane
// ends with both and the SiLU-mul needs no exchange), B = the activation rows.
// Each result is the same chain of 32x32x16 products over K as in the tile
// kernel, so the rows are the same bit for bit, whichever kernel runs a tile.
//
// Bound by HBM: at 2 rows per expert (128 experts, hidden 2048, inter 768) the
// up GEMM streams its 0.8 GB at 6.9 TB/s.  us per call before (256-row tiles
// of 4 waves) -> now: one expert and one row 56 -> 11 (device), 32 slots of 28
// experts 74 -> 47, 256 slots of 110 experts 233 -> 138.
//
// A ring stage is SUB sub-stages of BK columns.
template <int MODE_, int CW_, int SUB_, int LDS_, int RBMAX_>
struct SkinnyCfg {
  static constexpr int MODE = MODE_, CW = CW_, SUB = SUB_, LDS = LDS_, RBMAX = RBMAX_;
  static constexpr int kWRows = MODE == kModeUp ? 2 * CW : CW;  // weight rows per stage
  static constexpr int kWDma = kWRows / 16;                     // loads of 16 rows x 64 bytes
  static constexpr int kNA = kWRows > 32 ? kWRows / 32 : 1;     // 32-row A operands (16 rows: read twice)
};

template <class Cfg, int RB>
struct SkinnyShape {
  static constexpr int kXDma = RB / 16;
  static constexpr int kNB = RB > 32 ? RB / 32 : 1;
  static constexpr int kDma = Cfg::SUB * (Cfg::kWDma + kXDma);
  static constexpr int kSubBytes = (Cfg::kWDma + kXDma) * 1024;
  static constexpr int kStageBytes = Cfg::SUB * kSubBytes;
  static constexpr int kFit = Cfg::LDS / kStageBytes;
  static constexpr int kDeep = (kFit * kDma < 62 ? kFit : 62 / kDma) & ~1;  // stages in flight (even; vmcnt holds 63)
  static constexpr int kShallow = Cfg::SUB == 1 && kDeep >= 4 ? 4 : 2;      // for K of 128 columns
};

template <int DT, class Cfg, int RB, int D, bool ONCE>
__device__ __forceinline__ void skinny_block(const typename Elem<DT>::T *const (&w_src)[4], int64_t w_step,
                                             const typename Elem<DT>::T *const (&x_src)[4], int64_t x_step, int KT,
                                             const uint32_t (&a_off)[2], uint32_t lds0, const char *lds,
                                             tm_f32x16 (&acc)[Cfg::kNA][Cfg::RBMAX > 32 ? Cfg::RBMAX / 32 : 1]) {
  using S = SkinnyShape<Cfg, RB>;
  constexpr int SUB = Cfg::SUB, NA = Cfg::kNA, NB = S::kNB, kWDma = Cfg::kWDma;
  static_assert(D >= 2 && D % 2 == 0 && D * S::kStageBytes <= Cfg::LDS && D * S::kDma < 63, "ring shape");
  const int lane = threadIdx.x & 63;
  const int tr = lane & (RB < 32 ? RB - 1 : 31);
  uint32_t b_off[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
    b_off[ks] = (uint32_t)(kWDma * 1024 + tr * 64 + swz_chunk(tr, 2 * ks + (lane >> 5)) * 16);
  auto issue = [&](int st, uint32_t slot) {
    tm_static_for<SUB>([&](auto u_c) {
      constexpr int u = decltype(u_c)::value;
      const int64_t kt = (int64_t)st * SUB + u;
      const uint32_t dst = lds0 + slot + u * S::kSubBytes;
      tm_static_for<kWDma>([&](auto j_c) {
        constexpr int j = decltype(j_c)::value;
        tm_dma16_s<ONCE>(w_src[j] + kt * w_step, dst + j * 1024);
      });
      tm_static_for<S::kXDma>([&](auto j_c) {
        constexpr int j = decltype(j_c)::value;
        tm_dma16_s(x_src[j] + kt * x_step, dst + (kWDma + j) * 1024);
      });
    });
  };
  uint4 fa[2][2 * SUB][NA], fb[2][2 * SUB][NB];  // [stage parity][k-step]
  auto read = [&](auto p_c, uint32_t slot) {
    constexpr int p = decltype(p_c)::value;
#pragma unroll
    for (int ks = 0; ks < 2 * SUB; ++ks) {
      const char *const sub = lds + slot + (ks >> 1) * S::kSubBytes;
#pragma unroll
      for (int a = 0; a < NA; ++a) fa[p][ks][a] = *reinterpret_cast<const uint4 *>(sub + a_off[ks & 1] + a * 2048);
#pragma unroll
      for (int b = 0; b < NB; ++b) fb[p][ks][b] = *reinterpret_cast<const uint4 *>(sub + b_off[ks & 1] + b * 2048);
    }
  };
  auto mul = [&](auto p_c) {
    constexpr int p = decltype(p_c)::value;
#pragma unroll
    for (int ks = 0; ks < 2 * SUB; ++ks)
#pragma unroll
      for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[a][b] = tm_mfma32x32x16<DT>(fa[p][ks][a], fb[p][ks][b], acc[a][b]);
  };
  constexpr uint32_t kRing = (uint32_t)(D * S::kStageBytes);
  for (int i = 0; i < D; ++i) issue(i, (uint32_t)(i * S::kStageBytes));
  tm_wait_vm_lgkm0_mem<(D - 1) * S::kDma>();
  uint32_t slot = 0;
  read(std::integral_constant<int, 0>{}, slot);
  // stage i is in registers (parity p) or on its way there; its slot takes
  // stage i + D, then stage i + 1 is read while stage i is multiplied
  auto step = [&](auto p_c, int i) {
    constexpr int p = decltype(p_c)::value;
    tm_wait_vm_lgkm0_mem<63>();  // stage i is read: its slot is free
    issue(i + D, slot);
    slot = slot + S::kStageBytes == kRing ? 0u : slot + S::kStageBytes;
    tm_wait_vm_lgkm0_mem<(D - 1) * S::kDma>();  // stage i + 1 landed
    read(std::integral_constant<int, 1 - p>{}, slot);
    mul(p_c);
  };
  for (int i = 0; i < KT / SUB - D; i += 2) {  // KT is a multiple of 4; KT / SUB and D are even
    step(std::integral_constant<int, 0>{}, i);
    step(std::integral_constant<int, 1>{}, i + 1);
  }
  tm_static_for<D>([&](auto t_c) {
    constexpr int t = decltype(t_c)::value;
    if constexpr (t < D - 1) {
      slot = slot + S::kStageBytes == kRing ? 0u : slot + S::kStageBytes;
      tm_wait_vm_lgkm0_mem<(D - 2 - t) * S::kDma>();
      read(std::integral_constant<int, (t + 1) & 1>{}, slot);
    }
    mul(std::integral_constant<int, t & 1>{});
  });
  tm_wait_vm_lgkm0_mem<0>();  // every read is done before the next block's loads
}

// A workgroup takes one RBMAX-row block of a tile.  Grouped rows: the first
// `slots` blocks of workgroups take the tiles' first row blocks, so a call whose
// experts have few rows each runs as if there were no others; the blocks past
// them look for the tile of their further row block (a scan of the tile list)
// and find none where routing is even.  One workgroup for all rows of a tile,
// one block after the other, made uneven routing slow (us, 2048 x 768: 192 rows
// on each of 8 experts 124, 63 now and 74 with tiles of four waves before; 1536
// rows on one expert 135, 61 now and 76).
// Packed weights of an expert of one row block are read by no other workgroup:
// they are loaded non-temporally and leave the L2 to the activation rows.
template <int DT, class Cfg, bool PB>
__global__ __launch_bounds__(64) void skinny_gemm_kernel(
    const typename Elem<DT>::T *__restrict__ A, int64_t lda, const int32_t *__restrict__ a_rows,
    const typename Elem<DT>::T *__restrict__ B0, const typename Elem<DT>::T *__restrict__ B1, int64_t b_expert,
    int K, int n_groups, int pack_bn, int slots, TileSrc ts, typename Elem<DT>::T *__restrict__ C, int64_t ldc,
    const int64_t *__restrict__ c_rows, const typename Elem<DT>::T *__restrict__ addend, int64_t ld_add) {
  using T = typename Elem<DT>::T;
  constexpr int MODE = Cfg::MODE, CW = Cfg::CW, SUB = Cfg::SUB;
  __shared__ uint4 ring[Cfg::LDS / 16];
  const int lane = threadIdx.x & 63;
  const int64_t blk = blockIdx.x / n_groups;
  const int n0 = (int)(blockIdx.x % n_groups) * CW;
  int64_t y = blk;
  int e, r0, r_end, rb = 0;  // expert, the tile's rows [r0, r_end), this block's first row in it
  bool once = false;
  if (ts.tiles != nullptr) {
    const int64_t nt = ts.tiles[1] < ts.t_max ? ts.tiles[1] : ts.t_max;
    if (blk >= slots) {
      int u = (int)(blk - slots);  // this is further row block u
      if (u >= (ts.tiles[0] - nt) / Cfg::RBMAX) return;  // uniform: more than the rows can have past their tiles' first
      for (int64_t t0 = 0;; t0 += 256) {  // four tiles per lane
        if (t0 >= nt) return;  // uniform: there are fewer
        const int64_t t = t0 + 4 * lane;
        int ex[4], at[4], more[4], sum = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int64_t tj = t + j < nt ? t + j : nt - 1;
          ex[j] = ts.tiles[2 + tj];
          at[j] = ts.tiles[2 + ts.t_max + tj];
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) ex[j] = ts.expert_offsets[ex[j] + 1] - at[j];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          more[j] = t + j < nt ? ((ex[j] < BM ? ex[j] : BM) - 1) / Cfg::RBMAX : 0;
          sum += more[j];
        }
        const int upto = (int)tm_wave_incl_scan((uint32_t)sum);
        const int total = __builtin_amdgcn_readlane(upto, 63);
        if (u < total) {  // uniform
          const int l = __builtin_ctzll(__ballot(u < upto));
          u -= __builtin_amdgcn_readlane(upto - sum, l);
          int j = 0;
          for (int m = __builtin_amdgcn_readlane(more[0], l); j < 3 && u >= m;) {
            u -= m;
            ++j;
            m = __builtin_amdgcn_readlane(j == 1 ? more[1] : j == 2 ? more[2] : more[3], l);
          }
          y = t0 + 4 * l + j;
          rb = (u + 1) * Cfg::RBMAX;
          break;
        }
        u -= total;
      }
    }
    if (y >= nt) return;  // uniform: past the last tile
    e = ts.tiles[2 + y];
    r0 = ts.tiles[2 + ts.t_max + y];
    r_end = ts.expert_offsets[e + 1];
    once = r_end - ts.expert_offsets[e] <= Cfg::RBMAX;
  } else {
    constexpr int kBlocks = BM / Cfg::RBMAX;
    y = blk / kBlocks;
    rb = (int)(blk % kBlocks) * Cfg::RBMAX;
    e = 0;
    r0 = (int)y * BM;
    if (r0 >= ts.rows) return;
    r_end = ts.rows;
  }
  r_end = r_end < r0 + BM ? r_end : r0 + BM;  // this tile's rows
  const int rows = r_end - r0 - rb < Cfg::RBMAX ? r_end - r0 - rb : Cfg::RBMAX;
  if (rows <= 0) return;  // uniform
  const int KT = K / BK;
  const uint32_t lds0 = (uint32_t)(uintptr_t)ring;
  const char *const lds = reinterpret_cast<const char *>(ring);

  // Weight loads: lane l fills 16-byte slot l % 4 of LDS row 16 j + l / 4;
  // row r holds chunk swz_chunk(r in its 128- or 256-row tile, slot), the
  // order of the packed layout, so the packed loads are contiguous.
  const T *w_src[4] = {nullptr, nullptr, nullptr, nullptr};
  const int64_t w_step = PB ? (int64_t)pack_bn * BK : BK;
  auto w_addr = [&](const T *B, int col) {  // column `col` (a weight row), slot lane % 4
    const T *we = B + (int64_t)e * b_expert;
    if constexpr (PB)
      return we + (int64_t)(col / pack_bn) * pack_bn * K + (col % pack_bn) * BK + (lane & 3) * 8;
    else
      return we + (int64_t)col * K + swz_chunk(col, lane & 3) * 8;
  };
  const int lr = lane >> 2;
  uint32_t a_off[2];
  const int ar = lane & 31;  // operand row of this lane
  int a_lds, a_col;          // its LDS row and weight row (for the swizzle)
  if constexpr (MODE == kModeUp && CW == 32) {  // operands: 32 gate rows, 32 up rows
    w_src[0] = w_addr(B0, n0 + lr);
    w_src[1] = w_addr(B0, n0 + 16 + lr);
    w_src[2] = w_addr(B1, n0 + lr);
    w_src[3] = w_addr(B1, n0 + 16 + lr);
    a_lds = ar;
    a_col = n0 + ar;
  } else if constexpr (MODE == kModeUp && CW == 16) {  // one operand: 16 gate rows, 16 up rows
    w_src[0] = w_addr(B0, n0 + lr);
    w_src[1] = w_addr(B1, n0 + lr);
    a_lds = ar;
    a_col = n0 + (ar & 15);
  } else if constexpr (MODE == kModeUp) {  // CW == 8: gate rows 0-7, up rows 8-15 of one load, read twice
    static_assert(CW == 8, "column counts");
    w_src[0] = w_addr(lr < 8 ? B0 : B1, n0 + (lr & 7));
    a_lds = ar & 15;
    a_col = n0 + (ar & 7);
  } else {
#pragma unroll
    for (int j = 0; j < Cfg::kWDma; ++j) w_src[j] = w_addr(B0, n0 + 16 * j + lr);
    a_lds = CW < 32 ? ar & (CW - 1) : ar;
    a_col = n0 + a_lds;
  }
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
    a_off[ks] = (uint32_t)(a_lds * 64 + swz_chunk(a_col, 2 * ks + (lane >> 5)) * 16);

  constexpr bool kTiledA = PB && MODE == kModeDown;
  constexpr int kNBMax = Cfg::RBMAX > 32 ? Cfg::RBMAX / 32 : 1;
  const int64_t x_step = kTiledA ? (int64_t)BM * BK : BK;
  const T *x_src[4] = {};
#pragma unroll
  for (int j = 0; j < Cfg::RBMAX / 16; ++j) {
    const int tr = 16 * j + lr;
    if constexpr (kTiledA) {
      x_src[j] = A + y * (int64_t)BM * lda + (int64_t)(rb + tr) * BK + (lane & 3) * 8;
    } else {
      int gr = r0 + rb + tr;
      gr = gr < r_end ? gr : r_end - 1;  // rows past the expert re-read its last row; their results are dropped
      const int64_t xr = a_rows ? (int64_t)a_rows[gr] : (int64_t)gr;
      x_src[j] = A + xr * lda + swz_chunk(tr, lane & 3) * 8;
    }
  }
  tm_f32x16 acc[Cfg::kNA][kNBMax];
#pragma unroll
  for (int a = 0; a < Cfg::kNA; ++a)
#pragma unroll
    for (int b = 0; b < kNBMax; ++b) acc[a][b] = tm_f32x16{};
  auto run = [&](auto rb_c) {
    constexpr int RB = decltype(rb_c)::value;
    using S = SkinnyShape<Cfg, RB>;
    auto stream = [&](auto once_c) {
      constexpr bool kOnce = decltype(once_c)::value;
      if (KT / SUB >= S::kDeep)
        skinny_block<DT, Cfg, RB, S::kDeep, kOnce>(w_src, w_step, x_src, x_step, KT, a_off, lds0, lds, acc);
      else
        skinny_block<DT, Cfg, RB, S::kShallow, kOnce>(w_src, w_step, x_src, x_step, KT, a_off, lds0, lds, acc);
    };
    if (PB && once) stream(std::integral_constant<bool, PB>{});
    else stream(std::false_type{});
  };
  if (rows <= 16) run(std::integral_constant<int, 16>{});
  else if (Cfg::RBMAX == 32 || rows <= 32) run(std::integral_constant<int, 32>{});
  else run(std::integral_constant<int, Cfg::RBMAX>{});
  // lane: activation row lane % 32 of each B operand, weight rows 8 (i / 4)
  // + 4 (lane / 32) + i % 4 of each A operand: runs of 4 consecutive columns
#pragma unroll
  for (int b = 0; b < kNBMax; ++b) {
    const int tr = 32 * b + (lane & 31);
    if (tr < rows && (rows > 16 || tr < 16)) {
      const int gr = r0 + rb + tr;
#pragma unroll
      for (int u = 0; u < CW / 8; ++u) {
        const int col = n0 + 8 * u + 4 * (lane >> 5);
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (MODE == kModeUp) {
            const float g = tm_round<DT>(acc[0][b][4 * u + i]);
            const float up = CW == 32 ? acc[Cfg::kNA - 1][b][4 * u + i] : acc[0][b][(CW / 2 + 4 * u + i) & 15];
            v[i] = g * __builtin_amdgcn_rcpf(1.f + __expf(-g)) * up;
          } else {
            v[i] = acc[u / 4][b][(4 * u + i) & 15];
          }
        }
        if constexpr (MODE == kModeDown) {
          if (addend != nullptr) {  // dense rows only
            const uint2 a = *reinterpret_cast<const uint2 *>(addend + (int64_t)gr * ld_add + col);
            const T *ae = reinterpret_cast<const T *>(&a);
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] += Elem<DT>::to_f(ae[i]);
          }
        }
        uint2 r;
        T *re = reinterpret_cast<T *>(&r);
#pragma unroll
        for (int i = 0; i < 4; ++i) re[i] = Elem<DT>::from_f(v[i]);
        T *dst;
        if constexpr (PB && MODE == kModeUp)  // tile y of the intermediate in the down GEMM's stage order
          dst = C + y * (int64_t)BM * ldc + (col / BK) * (BM * BK) +
                ((rb + tr) * kCPR + swz_chunk(rb + tr, (col % BK) / 8)) * 8 + col % 8;
        else
          dst = C + (c_rows ? c_rows[gr] + col : (int64_t)gr * ldc + col);
        *reinterpret_cast<uint2 *>(dst) = r;
      }
    }
  }
}

// One tile of one expert, up to BM rows x BN columns, operands as in the wave
// kernel (A = weight rows, B = activation rows), eight waves that share both:
// wave w owns the columns of group w % 4 (up: gate and up rows of 32 columns
// of the 128; down: BN / 4 columns) and the row blocks of half w / 4.  Only the
// 32-row blocks that the tile has rows in are loaded and multiplied, NB = 1 ..
// 4 per half, and the LDS ring is cut into as many stages as fit: few rows
// leave room for a deeper ring, which is what a tile that only streams its
// weights needs.  One barrier per stage, between its two k-steps: it publishes
// the next stage and frees the slot that the stage after the ring goes to.
// Every result is the same chain of products as in the wave kernel.
//
// Bound by the bytes that a CU has on their way from HBM (three 32 KiB stages
// of 4 waves before; with 8 waves and 5 to 8 stages now), by activation rows
// that miss L2 behind the stream of weights (so weights that one workgroup
// alone reads are loaded non-temporally: 5280 rows of 128 experts 272 -> 253
// us; weights that several row tiles read are not: 510 against 594 us at 14.4k
// rows of 64 experts).  With many rows per expert neither HBM nor the matrix
// cores are at their limit (230 rows of 64 experts, hidden 2560, inter 1536: up
// 797 TFLOP/s, weights at 3.5 TB/s, waves waiting half of the time, no bank
// conflicts; 4096 dense rows 982 TFLOP/s): 6 operand reads per 8 products and a
// barrier per stage on one workgroup per CU.  us per call before (4 waves, one per SIMD, always 256 rows) -> now: hidden 2048,
// inter 768, 128 experts: 960 rows 287 -> 205, 5280 rows 310 -> 253, 19.2k rows
// 409 -> 366; hidden 2560, inter 1536, 64 experts: 1800 rows 358 -> 287, 14.4k
// rows 556 -> 510.
constexpr int kTileThreads = 512;
constexpr int kTileLds = 163840;

// Wait until at most `left` stages of kDma loads are outstanding (and LDS
// reads are done).
template <int kDma, int kMost>
__device__ __forceinline__ void wait_stages(int left) {
  if constexpr (kMost <= 0) {
    tm_wait_vm_lgkm0_mem<0>();
  } else {
    if (left >= kMost) tm_wait_vm_lgkm0_mem<kMost * kDma>();
    else wait_stages<kDma, kMost - 1>(left);
  }
}

template <int DT, int MODE, int BN, bool PB>
__global__ __launch_bounds__(kTileThreads, 2) void tile_gemm_kernel(
    const typename Elem<DT>::T *__restrict__ A, int64_t lda, const int32_t *__restrict__ a_rows,
    const typename Elem<DT>::T *__restrict__ B0, const typename Elem<DT>::T *__restrict__ B1, int64_t b_expert,
    int K, int n_tiles, TileSrc ts, typename Elem<DT>::T *__restrict__ C, int64_t ldc,
    const int64_t *__restrict__ c_rows, const typename Elem<DT>::T *__restrict__ addend, int64_t ld_add) {
  using T = typename Elem<DT>::T;
  constexpr int kMats = MODE == kModeUp ? 2 : 1;
  constexpr int kWLoads = kMats * BN / 16;   // 1 KiB loads of a stage's weight rows
  constexpr int kWDma = kWLoads / 8;         // ... per wave
  constexpr int kWBytes = kWLoads * 1024;
  constexpr int NA = MODE == kModeUp ? 2 : BN / 128;  // 32-row weight operands per wave
  __shared__ uint4 ring[kTileLds / 16];

  // Work items: (row tile, column tile), n_tiles per row tile.  Item b of the
  // whole groups of 8 row tiles is row tile 8 (b / 8 / n_tiles) + b % 8, so a
  // row tile's items run on one XCD (the dispatcher's round robin) and share
  // its L2 copy of the activation rows; the last row tiles follow in order.
  // The items past the last whole round of 256 are cut into 2 or 4 row
  // ranges where that still fits the CUs (a range's parts on one XCD): 8192
  // dense rows of hidden 2560, inter 1536 (384 items) 239 -> 214 us.
  const int64_t row_tiles = ts.tiles != nullptr ? (ts.tiles[1] < ts.t_max ? ts.tiles[1] : ts.t_max)
                                                : ((int64_t)ts.rows + BM - 1) / BM;
  const int64_t total = row_tiles * n_tiles, full = row_tiles / 8 * 8 * n_tiles, rounds = total / 256 * 256;
  int64_t b = blockIdx.x;
  int h0 = 0, wg_rows = BM;  // this workgroup's row range of the row tile
  if (b >= rounds) {
    const int rem = (int)(total - rounds), id = (int)(b - rounds);
    const int sh = rem <= 64 ? 2 : rem <= 128 ? 1 : 0;
    wg_rows = BM >> sh;
    h0 = ((id >> 3) & ((1 << sh) - 1)) * wg_rows;
    b = rounds + (id >> (3 + sh)) * 8 + (id & 7);
  }
  if (b >= total) return;
  int64_t y, col_tile;
  if (b < full) {
    y = (b >> 3) / n_tiles * 8 + (b & 7);
    col_tile = (b >> 3) % n_tiles;
  } else {
    y = full / n_tiles + (b - full) / n_tiles;
    col_tile = (b - full) % n_tiles;
  }
  const int n0 = (int)col_tile * BN;
  int e, r0, r_end;
  bool once = false;
  if (ts.tiles != nullptr) {
    e = ts.tiles[2 + y];
    r0 = ts.tiles[2 + ts.t_max + y] + h0;
    r_end = ts.expert_offsets[e + 1];
    once = r_end - ts.expert_offsets[e] <= BM;
  } else {
    e = 0;
    r0 = (int)y * BM + h0;
    r_end = ts.rows;
  }
  if (r0 >= r_end) return;
  const int rows = r_end - r0 < wg_rows ? r_end - r0 : wg_rows;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cg = wave & 3, half = wave >> 2;
  const int KT = K / BK;  // a multiple of 4
  const uint32_t lds0 = (uint32_t)(uintptr_t)ring;
  const char *const lds = reinterpret_cast<const char *>(ring);

  // Weight loads wave * kWDma + j (16 rows of 64 bytes each, the slot order of
  // the packed layout), through a buffer whose scalar offset walks K.
  tm_rsrc_t w_rs[kMats];
  w_rs[0] = tm_make_rsrc(B0 + (int64_t)e * b_expert + (int64_t)n0 * K, (uint64_t)BN * K * sizeof(T));
  if constexpr (kMats > 1)
    w_rs[1] = tm_make_rsrc(B1 + (int64_t)e * b_expert + (int64_t)n0 * K, (uint64_t)BN * K * sizeof(T));
  const tm_rsrc_t w_mine = kMats > 1 && wave >= 4 ? w_rs[kMats - 1] : w_rs[0];  // up: waves 0-3 W1, waves 4-7 W3
  uint32_t w_off[kWDma];
#pragma unroll
  for (int j = 0; j < kWDma; ++j) {
    const int p = (((kMats > 1 ? wave & 3 : wave) * kWDma + j) * 64) + lane;  // 16-byte slot in the matrix's stage
    const int row = p / kCPR, kc = swz_chunk(row, p % kCPR);
    w_off[j] = PB ? (uint32_t)p * 16u : (uint32_t)row * (uint32_t)K * (uint32_t)sizeof(T) + (uint32_t)kc * 16u;
  }
  constexpr uint32_t kWStep = PB ? BN * 64 : BK * sizeof(T);
  constexpr bool kTiledA = PB && MODE == kModeDown;
  constexpr int64_t kXStep = kTiledA ? BM * BK : BK;

  // operand offsets in a slot: weight rows of this wave, activation rows
  uint32_t a_off[2], b_off[2];
  const int ar = lane & 31;
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const uint32_t in_rows = (uint32_t)(ar * 64 + swz_chunk(ar, 2 * ks + (lane >> 5)) * 16);
    a_off[ks] = in_rows + (uint32_t)cg * (MODE == kModeUp ? 2048u : NA * 2048u);
    b_off[ks] = in_rows + kWBytes;
    asm volatile("" : "+v"(a_off[ks]), "+v"(b_off[ks]));
  }

  tm_f32x16 acc[NA][4];
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[a][q] = tm_f32x16{};

  auto run = [&](auto nb_c, auto once_c) {
    constexpr int NB = decltype(nb_c)::value;
    constexpr int kXDma = (NB + 1) / 2;  // loads of 16 activation rows per wave (4 NB in all)
    constexpr int kDma = kWDma + kXDma;
    constexpr int kStageBytes = kWBytes + NB * 4096;
    constexpr int kSlots = kTileLds / kStageBytes < 8 ? kTileLds / kStageBytes : 8;
    const uint32_t b_half = (uint32_t)(half * NB * 2048);
    constexpr int kFrag = NA + NB, kMfma = NA * NB;
    const T *x_src[kXDma];
    uint32_t x_dst[kXDma];
#pragma unroll
    for (int j = 0; j < kXDma; ++j) {
      const int q = (wave * kXDma + j) % (4 * NB);  // (spare waves repeat a load)
      const int tr = q * 16 + (lane >> 2);
      x_dst[j] = (uint32_t)(kWBytes + q * 1024);
      if constexpr (kTiledA) {
        x_src[j] = A + y * (int64_t)BM * lda + (int64_t)(h0 + tr) * BK + (lane & 3) * 8;
      } else {
        int gr = r0 + tr;
        gr = gr < r_end ? gr : r_end - 1;  // rows past the expert re-read its last row; their results are dropped
        const int64_t xr = a_rows ? (int64_t)a_rows[gr] : (int64_t)gr;
        x_src[j] = A + xr * lda + swz_chunk(tr, lane & 3) * 8;
      }
    }
    // load j of stage kt into the slot at byte `slot`
    auto issue_one = [&](auto j_c, uint32_t slot, int kt) {
      constexpr int j = decltype(j_c)::value;
      if constexpr (j < kWDma)
        tm_dma16_buf_so<decltype(once_c)::value>(w_mine, w_off[j], (uint32_t)kt * kWStep,
                                                 lds0 + slot + (uint32_t)(wave * kWDma + j) * 1024u);
      else
        tm_dma16_s(x_src[j - kWDma] + (int64_t)kt * kXStep, lds0 + slot + x_dst[j - kWDma]);
    };
    uint4 fr[2][kFrag];
    auto read_one = [&](auto g_c, uint4 (&f)[kFrag], uint32_t slot, int ks) {
      constexpr int g = decltype(g_c)::value;
      if constexpr (g < NA)
        f[g] = *reinterpret_cast<const uint4 *>(lds + slot + a_off[ks] + g * (MODE == kModeUp ? BN * 64 : 2048));
      else
        f[g] = *reinterpret_cast<const uint4 *>(lds + slot + b_half + b_off[ks] + (g - NA) * 2048);
    };
    // one k-step: its products, and spread between them the operand reads of
    // the next one and (with DMA) the loads of a stage
    auto kstep = [&](auto dma_c, const uint4 (&f)[kFrag], uint4 (&next)[kFrag], uint32_t rd, int ks, uint32_t dst,
                     int st) {
      tm_static_for<kMfma>([&](auto m_c) {
        constexpr int m = decltype(m_c)::value;
        constexpr int a = m / NB, q = m % NB;
        acc[a][q] = tm_mfma32x32x16<DT>(f[a], f[NA + q], acc[a][q]);
        constexpr int g0 = m * kFrag / kMfma, g1 = (m + 1) * kFrag / kMfma;
        tm_static_for<g1 - g0>(
            [&](auto g_c) { read_one(std::integral_constant<int, g0 + decltype(g_c)::value>{}, next, rd, ks); });
        if constexpr (decltype(dma_c)::value) {
          constexpr int d0 = m * kDma / kMfma, d1 = (m + 1) * kDma / kMfma;
          tm_static_for<d1 - d0>(
              [&](auto d_c) { issue_one(std::integral_constant<int, d0 + decltype(d_c)::value>{}, dst, st); });
        }
        __builtin_amdgcn_sched_barrier(0);
      });
    };
    const int first = KT < kSlots ? KT : kSlots;
    for (int st = 0; st < first; ++st)
      tm_static_for<kDma>([&](auto j_c) { issue_one(j_c, (uint32_t)(st * kStageBytes), st); });
    wait_stages<kDma, kSlots - 1>(first - 1);  // stage 0 of this wave landed
    __builtin_amdgcn_s_barrier();
    tm_static_for<kFrag>([&](auto g_c) { read_one(g_c, fr[0], 0u, 0); });
    uint32_t cur = 0;
    int i = 0;
    for (; i < KT - kSlots; ++i) {
      const uint32_t nxt = cur == (kSlots - 1) * kStageBytes ? 0u : cur + kStageBytes;
      kstep(std::false_type{}, fr[0], fr[1], cur, 1, 0u, 0);
      tm_wait_vm_lgkm0_mem<(kSlots - 2) * kDma>();  // stage i + 1 of this wave landed; its reads are done
      __builtin_amdgcn_s_barrier();                 // ... in every wave; no wave reads slot `cur` any more
      kstep(std::true_type{}, fr[1], fr[0], nxt, 0, cur, i + kSlots);
      cur = nxt;
    }
    for (; i < KT; ++i) {  // the last stages: nothing more to load
      const uint32_t nxt = cur == (kSlots - 1) * kStageBytes ? 0u : cur + kStageBytes;
      kstep(std::false_type{}, fr[0], fr[1], cur, 1, 0u, 0);
      wait_stages<kDma, kSlots - 2>(KT - 2 - i);
      __builtin_amdgcn_s_barrier();
      kstep(std::false_type{}, fr[1], fr[0], nxt, 0, 0u, 0);
      cur = nxt;
    }
  };
  const int nb = (rows + 63) / 64;  // 32-row blocks per half
  const int first_row = half * nb * 32;
  auto run_nb = [&](auto once_c) {
    if (nb == 1) run(std::integral_constant<int, 1>{}, once_c);
    else if (nb == 2) run(std::integral_constant<int, 2>{}, once_c);
    else if (nb == 3) run(std::integral_constant<int, 3>{}, once_c);
    else run(std::integral_constant<int, 4>{}, once_c);
  };
  // Packed weights that no other row tile reads are loaded non-temporally (the
  // row ranges of a tile that is cut do read the same ones, at the same time).
  if (PB && once) run_nb(std::integral_constant<bool, PB>{});
  else run_nb(std::false_type{});

  // lane: activation row lane % 32 of each block, weight rows 8 (i / 4) + 4
  // (lane / 32) + i % 4 of each operand: runs of 4 consecutive columns
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int tr = first_row + 32 * q + (lane & 31);
    if (q < nb && tr < rows) {
      const int gr = r0 + tr;
#pragma unroll
      for (int u = 0; u < (MODE == kModeUp ? 4 : 4 * NA); ++u) {
        const int col = n0 + cg * (MODE == kModeUp ? 32 : NA * 32) + 8 * u + 4 * (lane >> 5);
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if constexpr (MODE == kModeUp) {
            const float g = tm_round<DT>(acc[0][q][4 * u + i]);
            v[i] = g * __builtin_amdgcn_rcpf(1.f + __expf(-g)) * acc[NA - 1][q][4 * u + i];
          } else {
            v[i] = acc[u / 4][q][(4 * u + i) & 15];
          }
        }
        if constexpr (MODE == kModeDown) {
          if (addend != nullptr) {  // dense rows only
            const uint2 ad = *reinterpret_cast<const uint2 *>(addend + (int64_t)gr * ld_add + col);
            const T *ae = reinterpret_cast<const T *>(&ad);
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] += Elem<DT>::to_f(ae[i]);
          }
        }
        uint2 r;
        T *re = reinterpret_cast<T *>(&r);
#pragma unroll
        for (int i = 0; i < 4; ++i) re[i] = Elem<DT>::from_f(v[i]);
        T *dst;
        if constexpr (PB && MODE == kModeUp)  // tile y of the intermediate in the down GEMM's stage order
          dst = C + y * (int64_t)BM * ldc + (col / BK) * (BM * BK) +
                ((h0 + tr) * kCPR + swz_chunk(tr, (col % BK) / 8)) * 8 + col % 8;
        else
          dst = C + (c_rows ? c_rows[gr] + col : (int64_t)gr * ldc + col);
        *reinterpret_cast<uint2 *>(dst) = r;
      }
    }
  }
}

// One workgroup of kGroupThreads: bucket the recomputed (token, slot) pairs
// by expert.  mask[b * ms_b + s * ms_s] != 0 selects a pair (ms_s = 0: a
// per-token flag); ids outside [0, n_experts) are skipped.
constexpr int kGroupThreads = 1024;
constexpr int kMaxExperts = 1024;  // one scanning thread per expert
static_assert(kMaxExperts <= kGroupThreads, "one expert per thread");
constexpr int kGroupTok = 4;    // tokens per thread on the register path (n <= 4096)
constexpr int kGroupSlots = 8;  // slots per token on the register path (top_k <= 8)
static_assert(kGroupTok * kGroupThreads * 8 <= 65536, "a placed row (token << 3 | slot) fits 16 bits");

__global__ __launch_bounds__(kGroupThreads) void group_slots_kernel(
    const int64_t *__restrict__ ids, int64_t n, int top_k, int64_t ld_ids, const uint8_t *__restrict__ mask,
    int64_t ms_b, int64_t ms_s, int n_experts, int64_t so_b, int64_t so_s, int32_t *__restrict__ offsets,
    int32_t *__restrict__ row_token, int64_t *__restrict__ row_out, int32_t *__restrict__ tiles, int64_t t_max) {
  __shared__ int32_t hist[kMaxExperts];
  __shared__ int32_t cursor[kMaxExperts];
  __shared__ int32_t tile_base[kMaxExperts + 1];
  // register path: each placed row as (token << 3 | slot), written out in row
  // order afterwards (scattered 4- and 8-byte stores cost ~10 us; in row
  // order they are a few coalesced passes)
  __shared__ uint16_t placed[kGroupTok * kGroupThreads * kGroupSlots];
  __shared__ int32_t s_rows;
  __shared__ int32_t wave_rows[kGroupThreads / 64], wave_tiles[kGroupThreads / 64];
  const int tid = threadIdx.x;
  for (int e = tid; e < n_experts; e += kGroupThreads) hist[e] = 0;
  // Each thread keeps the experts of its tokens (b = tid + 1024 j, j < kGroupTok)
  // in registers: all of their loads are issued before the first count.
  // (Reading the id array as consecutive elements per wave load instead
  // measured slower: 16.4 / 24.9 us against 15.2 / 21.7 us hot / cold.)
  int32_t ex[kGroupTok][kGroupSlots];
  // n == 0 takes the loop path, whose loops run no iteration: the register
  // path clamps to token n - 1 and would read below `ids` and `mask`.
  const bool fast = n > 0 && n <= (int64_t)kGroupTok * kGroupThreads && top_k <= kGroupSlots;  // uniform
  if (fast) {
#pragma unroll
    for (int j = 0; j < kGroupTok; ++j) {
      const int64_t b = tid + (int64_t)kGroupThreads * j;
      const int64_t bb = b < n ? b : n - 1;
#pragma unroll
      for (int s = 0; s < kGroupSlots; ++s) {
        const int ss = s < top_k ? s : top_k - 1;
        const int64_t e = ids[bb * ld_ids + ss];
        const bool use = b < n && s < top_k && mask[bb * ms_b + ss * ms_s] && e >= 0 && e < n_experts;
        ex[j][s] = use ? (int32_t)e : -1;
      }
    }
  }
  __syncthreads();
  if (fast) {
#pragma unroll
    for (int j = 0; j < kGroupTok; ++j)
#pragma unroll
      for (int s = 0; s < kGroupSlots; ++s)
        if (ex[j][s] >= 0) atomicAdd(&hist[ex[j][s]], 1);
  } else {
    for (int64_t b = tid; b < n; b += kGroupThreads)  // a token per thread, its slots in order
      for (int s = 0; s < top_k; ++s) {
        const int64_t e = ids[b * ld_ids + s];
        if (mask[b * ms_b + s * ms_s] && e >= 0 && e < n_experts) atomicAdd(&hist[e], 1);
      }
  }
  __syncthreads();
  {
    // offsets and tile bases: exclusive scans over the experts, thread e
    // owning expert e (n_experts <= kGroupThreads): wave scans, then the
    // waves' totals in wave order (a serial loop over the experts cost ~4 us)
    const int lane = tid & 63, wave = tid >> 6;
    const int32_t h = tid < n_experts ? hist[tid] : 0;
    const int32_t tc = (h + BM - 1) / BM;
    int32_t ih = h, it = tc;  // inclusive within the wave
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int32_t oh = __shfl_up(ih, d, 64), ot = __shfl_up(it, d, 64);
      if (lane >= d) {
        ih += oh;
        it += ot;
      }
    }
    if (lane == 63) {
      wave_rows[wave] = ih;
      wave_tiles[wave] = it;
    }
    __syncthreads();
    int32_t bh = 0, bt = 0;
    for (int w = 0; w < wave; ++w) {
      bh += wave_rows[w];
      bt += wave_tiles[w];
    }
    const int32_t eh = bh + ih - h, et = bt + it - tc;  // exclusive
    if (tid < n_experts) {
      offsets[tid] = eh;
      cursor[tid] = eh;
      tile_base[tid] = et;
    }
    if (tid == n_experts - 1) {
      offsets[n_experts] = eh + h;
      tile_base[n_experts] = et + tc;
      tiles[0] = eh + h;
      tiles[1] = et + tc;
      s_rows = eh + h;
    }
  }
  __syncthreads();
  for (int e = tid; e < n_experts; e += kGroupThreads) {
    const int32_t t0 = tile_base[e], t1 = tile_base[e + 1];
    int32_t r = cursor[e];
    for (int32_t t = t0; t < t1; ++t, r += BM) {
      tiles[2 + t] = e;
      tiles[2 + t_max + t] = r;
    }
  }
  __syncthreads();  // cursor[] is read above before the placement below advances it
  if (fast) {
#pragma unroll
    for (int j = 0; j < kGroupTok; ++j)
#pragma unroll
      for (int s = 0; s < kGroupSlots; ++s)
        if (ex[j][s] >= 0) {
          const int b = tid + kGroupThreads * j;  // < 4096
          const int32_t pos = atomicAdd(&cursor[ex[j][s]], 1);
          placed[pos] = (uint16_t)((b << 3) | s);
        }
    __syncthreads();
    const int32_t rows = s_rows;
    for (int32_t i = tid; i < rows; i += kGroupThreads) {
      const int v = placed[i];
      const int64_t b = v >> 3;
      row_token[i] = (int32_t)b;
      row_out[i] = b * so_b + (int64_t)(v & 7) * so_s;
    }
  } else {
    for (int64_t b = tid; b < n; b += kGroupThreads)
      for (int s = 0; s < top_k; ++s) {
        const int64_t e = ids[b * ld_ids + s];
        if (mask[b * ms_b + s * ms_s] && e >= 0 && e < n_experts) {
          const int32_t pos = atomicAdd(&cursor[e], 1);
          row_token[pos] = (int32_t)b;
          row_out[pos] = b * so_b + (int64_t)s * so_s;
        }
      }
  }
}

// Multi-workgroup grouping (tm_group_slots_ws): kGrpTok tokens per
// workgroup, in two launches (one workgroup counts for itself: up to 64 tokens
// take one launch).  group_count_kernel loads its tokens' ids and
// mask bytes and writes the workgroup's per-expert counts to a row of the
// workspace; group_place_kernel loads them again, sums every workgroup's row
// for each expert (and the rows of the workgroups before it), scans the
// experts for the offsets and tile bases (workgroup 0 writes them and the
// tile list) and places its rows at offset + rows of earlier workgroups +
// an LDS cursor.  Each CU then loads 1/G of the ids instead of one CU all
// of them.
constexpr int kGrpThreads = 256;
constexpr int kGrpTok = 64;            // tokens per workgroup: 4 threads per token, 2 slots each
constexpr int kGrpMaxSlots = 8;        // top_k
constexpr int kGrpMaxExperts = 256;    // one expert per thread in the scan
constexpr int kGrpMaxWgs = 128;        // n_tokens <= 8192
constexpr int kGrpBatch = 16;          // count rows loaded per round trip

// The two (token, slot) entries of this thread: expert id, or -1 when the
// pair is not recomputed.  Clamped addresses (no load is conditional).
__device__ __forceinline__ void grp_entries(const int64_t *__restrict__ ids, int64_t n, int top_k, int64_t ld_ids,
                                            const uint8_t *__restrict__ mask, int64_t ms_b, int64_t ms_s,
                                            int n_experts, int64_t b, int s0, int (&ex)[2]) {
  const int64_t bb = b < n ? b : n - 1;
  int64_t e[2];
  uint8_t m[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int s = s0 + u;
    const int ss = s < top_k ? s : top_k - 1;
    e[u] = ids[bb * ld_ids + ss];
    m[u] = mask[bb * ms_b + ss * ms_s];
  }
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const bool use = b < n && s0 + u < top_k && m[u] && e[u] >= 0 && e[u] < n_experts;
    ex[u] = use ? (int)e[u] : -1;
  }
}

__global__ __launch_bounds__(kGrpThreads) void group_count_kernel(const int64_t *__restrict__ ids, int64_t n,
                                                                  int top_k, int64_t ld_ids,
                                                                  const uint8_t *__restrict__ mask, int64_t ms_b,
                                                                  int64_t ms_s, int n_experts,
                                                                  int32_t *__restrict__ counts) {
  __shared__ int32_t h[kGrpMaxExperts];
  const int tid = threadIdx.x;
  int ex[2];
  grp_entries(ids, n, top_k, ld_ids, mask, ms_b, ms_s, n_experts, (int64_t)blockIdx.x * kGrpTok + tid / 4,
              2 * (tid % 4), ex);
  for (int e = tid; e < n_experts; e += kGrpThreads) h[e] = 0;
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 2; ++u)
    if (ex[u] >= 0) atomicAdd(&h[ex[u]], 1);
  __syncthreads();
  for (int e = tid; e < n_experts; e += kGrpThreads) counts[(int64_t)blockIdx.x * n_experts + e] = h[e];
}

// ONE: the batch fits one workgroup, which counts its rows itself (no
// group_count_kernel launch before it).
template <bool ONE>
__global__ __launch_bounds__(kGrpThreads) void group_place_kernel(
    const int64_t *__restrict__ ids, int64_t n, int top_k, int64_t ld_ids, const uint8_t *__restrict__ mask,
    int64_t ms_b, int64_t ms_s, int n_experts, int64_t so_b, int64_t so_s, const int32_t *__restrict__ counts,
    int32_t *__restrict__ offsets, int32_t *__restrict__ row_token, int64_t *__restrict__ row_out,
    int32_t *__restrict__ tiles, int64_t t_max) {
  __shared__ int32_t part_tot[kGrpThreads], part_bef[kGrpThreads];
  __shared__ int32_t cur[kGrpMaxExperts];
  __shared__ int32_t wave_rows[kGrpThreads / 64], wave_tiles[kGrpThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int G = (int)gridDim.x, g0 = (int)blockIdx.x;
  const int64_t b = (int64_t)g0 * kGrpTok + tid / 4;
  const int s0 = 2 * (tid % 4);
  int ex[2];
  grp_entries(ids, n, top_k, ld_ids, mask, ms_b, ms_s, n_experts, b, s0, ex);
  // thread x owns expert x: its total and the rows of the earlier workgroups
  int32_t h = 0, hb = 0;
  if constexpr (ONE) {
    part_tot[tid] = 0;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 2; ++u)
      if (ex[u] >= 0) atomicAdd(&part_tot[ex[u]], 1);
    __syncthreads();
    h = part_tot[tid];
  } else {
    // Thread (e, p) of ep = pow2 >= n_experts columns sums the count rows
    // g = p, p + P, .. (P = 256 / ep) of expert e: kGrpBatch rows per round
    // trip (clamped rows, masked by a select).
    int ep = 1;
    while (ep < n_experts) ep <<= 1;
    const int P = kGrpThreads / ep;
    const int e = tid % ep, p = tid / ep;
    const int ec = e < n_experts ? e : n_experts - 1;
    int32_t tot = 0, bef = 0;
    for (int g = p; g < G; g += P * kGrpBatch) {
      int32_t v[kGrpBatch];
#pragma unroll
      for (int j = 0; j < kGrpBatch; ++j) {
        const int gj = g + P * j;
        v[j] = counts[(int64_t)(gj < G ? gj : G - 1) * n_experts + ec];
      }
#pragma unroll
      for (int j = 0; j < kGrpBatch; ++j) {
        const int gj = g + P * j;
        const int32_t c = (gj < G && e < n_experts) ? v[j] : 0;
        tot += c;
        bef += gj < g0 ? c : 0;
      }
    }
    part_tot[tid] = tot;
    part_bef[tid] = bef;
    __syncthreads();
    if (tid < n_experts)
      for (int q = 0; q < P; ++q) {
        h += part_tot[q * ep + tid];
        hb += part_bef[q * ep + tid];
      }
  }
  // exclusive scans over the experts (rows and 256-row tiles): wave scans,
  // then the waves' totals in wave order
  const int32_t tc = (h + BM - 1) / BM;
  int32_t ih = h, it = tc;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int32_t oh = __shfl_up(ih, d, 64), ot = __shfl_up(it, d, 64);
    if (lane >= d) {
      ih += oh;
      it += ot;
    }
  }
  if (lane == 63) {
    wave_rows[wave] = ih;
    wave_tiles[wave] = it;
  }
  __syncthreads();
  int32_t bh = 0, bt = 0;
  for (int w = 0; w < wave; ++w) {
    bh += wave_rows[w];
    bt += wave_tiles[w];
  }
  const int32_t eh = bh + ih - h, et = bt + it - tc;  // exclusive
  if (tid < n_experts) {
    cur[tid] = eh + hb;
    if (g0 == 0) {
      offsets[tid] = eh;
      for (int32_t t = 0; t < tc; ++t) {
        tiles[2 + et + t] = tid;
        tiles[2 + t_max + et + t] = eh + t * BM;
      }
      if (tid == n_experts - 1) {
        offsets[n_experts] = eh + h;
        tiles[0] = eh + h;
        tiles[1] = et + tc;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 2; ++u)
    if (ex[u] >= 0) {
      const int32_t pos = atomicAdd(&cur[ex[u]], 1);
      row_token[pos] = (int32_t)b;
      row_out[pos] = b * so_b + (int64_t)(s0 + u) * so_s;
    }
}

// Column tile of the down GEMM: 256 columns when hidden allows (half the LDS
// reads per MFMA of 128-column tiles).
inline int down_bn(int32_t hidden) { return hidden % (2 * kMinBN) == 0 ? 2 * kMinBN : kMinBN; }

// Which kernel runs the two GEMMs; every one gives the same bits.
enum { kPlanTile = 0, kPlanWave, kPlanWave64 };

// Few waves: 8 (16) columns per wave, 64-column stages and a deep ring; else
// twice the columns and a ring that leaves room for 10 waves per CU.
using SkUpFew = SkinnyCfg<kModeUp, 8, 2, 49152, 32>;
using SkDownFew = SkinnyCfg<kModeDown, 16, 2, 49152, 32>;
using SkUpMany = SkinnyCfg<kModeUp, 16, 1, 16384, 32>;
using SkDownMany = SkinnyCfg<kModeDown, 32, 1, 16384, 32>;
using SkUp64 = SkinnyCfg<kModeUp, 32, 1, 32768, 64>;
using SkDown64 = SkinnyCfg<kModeDown, 64, 1, 32768, 64>;
constexpr int kSkManyWaves = 512;

template <int DT, class Cfg, bool PB>
void launch_skinny(const void *A, int64_t lda, const int32_t *a_rows, const void *B0, const void *B1, int64_t b_expert,
                   int K, int N, const TileSrc &ts, int64_t tiles, void *C, int64_t ldc, const int64_t *c_rows,
                   const void *addend, int64_t ld_add, hipStream_t s) {
  using T = typename Elem<DT>::T;
  const int pack_bn = Cfg::MODE == kModeUp ? kMinBN : down_bn(N);
  const bool grouped = ts.tiles != nullptr;
  // grouped: a row block per tile, and as many more as the rows can have past them
  const int64_t blocks = grouped ? tiles + (ts.rows - 1) / Cfg::RBMAX : tm_cdiv(ts.rows, Cfg::RBMAX);
  hipLaunchKernelGGL((skinny_gemm_kernel<DT, Cfg, PB>), dim3((unsigned)(blocks * (N / Cfg::CW))), dim3(64), 0, s,
                     static_cast<const T *>(A), lda, a_rows, static_cast<const T *>(B0), static_cast<const T *>(B1),
                     b_expert, K, N / Cfg::CW, pack_bn, (int)tiles, ts, static_cast<T *>(C), ldc, c_rows,
                     static_cast<const T *>(addend), ld_add);
}

template <int DT, int MODE, int BN, bool PB>
void launch_tile(const void *A, int64_t lda, const int32_t *a_rows, const void *B0, const void *B1, int64_t b_expert,
                 int K, int N, const TileSrc &ts, int64_t tiles, void *C, int64_t ldc, const int64_t *c_rows,
                 const void *addend, int64_t ld_add, hipStream_t s) {
  using T = typename Elem<DT>::T;
  const int n_tiles = N / BN;
  hipLaunchKernelGGL((tile_gemm_kernel<DT, MODE, BN, PB>), dim3((unsigned)(tm_cdiv(tiles * n_tiles, 256) * 256)),
                     dim3(kTileThreads), 0, s, static_cast<const T *>(A), lda, a_rows, static_cast<const T *>(B0),
                     static_cast<const T *>(B1), b_expert, K, n_tiles, ts, static_cast<T *>(C), ldc, c_rows,
                     static_cast<const T *>(addend), ld_add);
}

template <int DT, bool PB>
void swiglu_launch(const void *x, int64_t ld_x, const int32_t *row_token, int32_t hidden, int32_t inter,
                   const void *w1, const void *w3, const void *w2, const TileSrc &ts, int64_t tiles, void *out,
                   int64_t ld_out, const int64_t *row_out, void *fused, const void *addend, int64_t ld_add,
                   int plan, hipStream_t s) {
  const int64_t bw = (int64_t)inter * hidden;
  auto up = [&](auto cfg) {
    launch_skinny<DT, decltype(cfg), PB>(x, ld_x, row_token, w1, w3, bw, hidden, inter, ts, tiles, fused, inter,
                                         nullptr, nullptr, 0, s);
  };
  auto down = [&](auto cfg) {
    launch_skinny<DT, decltype(cfg), PB>(fused, inter, nullptr, w2, nullptr, bw, inter, hidden, ts, tiles, out, ld_out,
                                         row_out, addend, ld_add, s);
  };
  if (plan == kPlanWave) {
    const int64_t blocks = ts.tiles == nullptr ? tm_cdiv(ts.rows, 32) : tiles;
    if (blocks * (inter / 16) >= kSkManyWaves) up(SkUpMany{});
    else up(SkUpFew{});
    if (blocks * (hidden / 32) >= kSkManyWaves) down(SkDownMany{});
    else down(SkDownFew{});
  } else if (plan == kPlanWave64) {
    up(SkUp64{});
    down(SkDown64{});
  } else {
    launch_tile<DT, kModeUp, kMinBN, PB>(x, ld_x, row_token, w1, w3, bw, hidden, inter, ts, tiles, fused, inter,
                                         nullptr, nullptr, 0, s);
    if (down_bn(hidden) == 2 * kMinBN)
      launch_tile<DT, kModeDown, 2 * kMinBN, PB>(fused, inter, nullptr, w2, nullptr, bw, inter, hidden, ts, tiles, out,
                                                 ld_out, row_out, addend, ld_add, s);
    else
      launch_tile<DT, kModeDown, kMinBN, PB>(fused, inter, nullptr, w2, nullptr, bw, inter, hidden, ts, tiles, out,
                                             ld_out, row_out, addend, ld_add, s);
  }
}

// The plan of a dense call.  One wave per column group needs no LDS exchange
// and spreads a single expert over the chip, but re-reads its operands per 32
// (64) rows; measured crossovers (hidden x inter 2048 x 768 | 2560 x 1536, us
// per call): 128 rows 14 | 21 against 26 | 34 with 64-row waves and 44 | 64
// with tiles; 512 rows 22 | 54, 27 | 37, 41 | 65; 2048 rows 81 | 192, 53 | 132,
// 43 | 68.  Small weights: from 32 tiles of many rows on, tiles fill the chip and
// read the weights less often: 128 x 128 4096 rows 8.9 | 12.4 | 11.5, 16384 17.7 |
// 16.3 | 13.0, 65536 44 | 41 | 26; 256 x 512 2048 rows 14.7 | 17.2 | 17.3, 4096 22 | 21 |
// 18.6, 16384 61 | 47 | 32.
int dense_plan(int64_t rows, int32_t hidden, int32_t inter) {
  if (rows > 2048 && tm_cdiv(rows, BM) * (inter / kMinBN) >= 32) return kPlanTile;
  const double work = (double)rows * hidden * inter;
  return work <= 1.1e9 ? kPlanWave : work <= 3e9 ? kPlanWave64 : kPlanTile;
}

// The plan of a grouped call, from the most rows per expert that it can have
// on average (the counts are on the device): measured us per call, waves |
// tiles, at 12.5 (128 experts, 2048 x 768): 205 | 203, at 18.8 (64 experts,
// 2560 x 1536): 292 | 264, at 9.4: 235 | 243, at 0.5: 51 | 55.  Rows need not be
// even for it: the wave kernel spreads an expert's rows in blocks of 32, up to
// the work of one expert with all of them that the dense waves are good for: even
// routing | all rows on one expert, waves against tiles, 768 rows of 64 experts,
// 2560 x 1536: 262 | 70 against 260 | 53; 1536 rows of 128, 2560 x 1536: 543 | 124
// against 502 | 62; 3072 rows of 1024, 1024 x 256: 275 | 50 against 302 | 40.  Plain
// weights, which a wave reads in rows of 64 bytes, up to half of that: 512 rows of
// 128, 2048 x 768: 233 | 37 (on eight) against 248 | 50; 1536 rows: 281 | 77 against
// 262 | 53; 512 rows of 64, 2560 x 1536: 351 | 81 against 317 | 68.
int grouped_plan(int64_t max_rows, int32_t n_experts, int32_t hidden, int32_t inter, bool packed) {
  return max_rows <= 12 * (int64_t)n_experts && (double)max_rows * hidden * inter <= (packed ? 3.1e9 : 1.6e9)
             ? kPlanWave
             : kPlanTile;
}

// The two GEMMs of the MLP over the rows the tile source names; `addend`
// (dense rows only, nullable) is added to the down projection before its
// rounding; `packed`: the weights are in tm_expert_pack_weights's layout.
int swiglu_impl(int32_t dtype, const void *x, int64_t ld_x, const int32_t *row_token, int32_t hidden,
                int32_t inter, const void *w1, const void *w3, const void *w2, const TileSrc &ts, int64_t tiles,
                void *out, int64_t ld_out, const int64_t *row_out, void *fused, const void *addend, int64_t ld_add,
                bool packed, int plan, hipStream_t s) {
  return TM_DISPATCH_DTYPE(dtype, DT, [&] {
    if constexpr (DT == TM_DT_F32) {
      return tm_fail(TM_EINVAL_DTYPE, "tm_grouped_swiglu: dtype must be F16 or BF16");
    } else {
      if (packed)
        swiglu_launch<DT, true>(x, ld_x, row_token, hidden, inter, w1, w3, w2, ts, tiles, out, ld_out, row_out,
                                fused, addend, ld_add, plan, s);
      else
        swiglu_launch<DT, false>(x, ld_x, row_token, hidden, inter, w1, w3, w2, ts, tiles, out, ld_out, row_out,
                                 fused, addend, ld_add, plan, s);
      TM_LAUNCH_CHECK("tm_grouped_swiglu");
      return TM_OK;
    }
  });
}

// Packed weights: tile t of BN rows of expert e (rows n0 = t BN ..) keeps
// its place [e][n0 .. n0 + BN) x K of the nn.Linear layout, reordered by
// stage: stage kt (columns kt BK .. + BK) is one contiguous block of BN x BK
// elements holding slot p = 16 bytes (row p / kCPR, chunk swz_chunk(row,
// p % kCPR)) at element 8 p -- the order the GEMM's LDS ring holds a stage
// in, so a stage's weight tile is one contiguous read.  One workgroup per
// stage of one tile.
template <typename T, int BN>
__global__ __launch_bounds__(kThreads) void pack_weights_kernel(const T *__restrict__ w, int64_t K, int64_t KT,
                                                                 T *__restrict__ out) {
  const int64_t b = blockIdx.x;  // (tile of every expert) * KT + kt
  const int64_t tile = b / KT, kt = b % KT;
  const T *src = w + tile * BN * K + kt * BK;
  T *dst = out + tile * BN * K + kt * (BN * BK);
#pragma unroll
  for (int j = 0; j < BN * kCPR / kThreads; ++j) {
    const int p = threadIdx.x + kThreads * j;
    const int row = p / kCPR, kc = swz_chunk(row, p % kCPR);
    *reinterpret_cast<uint4 *>(dst + (int64_t)p * 8) =
        *reinterpret_cast<const uint4 *>(src + (int64_t)row * K + kc * 8);
  }
}

bool shapes_ok(int32_t hidden, int32_t inter) {
  // multiples of 128: whole column tiles, and K an even number of two-stage steps (the wave kernel's rings)
  return hidden > 0 && inter > 0 && hidden % kMinBN == 0 && inter % kMinBN == 0 && (int64_t)inter * hidden <
         ((int64_t)1 << 30);
}

}  // namespace

extern "C" int64_t tm_group_slots_tiles(int64_t max_rows, int32_t n_experts) {
  if (max_rows < 0 || n_experts <= 0) return 0;
  return tm_cdiv(max_rows, BM) + n_experts;
}

extern "C" int tm_group_slots(const int64_t *ids, int64_t n_tokens, int32_t top_k, int64_t ld_ids,
                              const uint8_t *mask, int64_t ms_b, int64_t ms_s, int32_t n_experts, int64_t so_b,
                              int64_t so_s, int32_t *expert_offsets, int32_t *row_token, int64_t *row_out,
                              int32_t *tiles, tm_stream_t stream) {
  TM_REQUIRE(n_tokens >= 0 && top_k >= 1 && ld_ids >= top_k && n_experts >= 1 && n_experts <= kMaxExperts,
             TM_EINVAL_SHAPE, "tm_group_slots: bad sizes (n_experts must be in [1, %d])", kMaxExperts);
  TM_REQUIRE(n_tokens * top_k < ((int64_t)1 << 31), TM_EINVAL_SHAPE, "tm_group_slots: too many slots");
  TM_REQUIRE(expert_offsets && tiles && (n_tokens == 0 || (ids && mask && row_token && row_out)), TM_EINVAL_ARG,
             "tm_group_slots: null pointer");
  // tm_grouped_swiglu's contract: rows at 16-byte offsets of row_out (it writes them in 8-byte pieces)
  TM_REQUIRE(so_b % 8 == 0 && so_s % 8 == 0, TM_EINVAL_SHAPE,
             "tm_group_slots: output strides (%lld, %lld) must be multiples of 8 elements", (long long)so_b,
             (long long)so_s);
  const int64_t t_max = tm_group_slots_tiles(n_tokens * top_k, n_experts);
  hipLaunchKernelGGL(group_slots_kernel, dim3(1), dim3(kGroupThreads), 0, tm_hip_stream(stream), ids, n_tokens,
                     top_k, ld_ids, mask, ms_b, ms_s, n_experts, so_b, so_s, expert_offsets, row_token, row_out,
                     tiles, t_max);
  TM_LAUNCH_CHECK("tm_group_slots");
  return TM_OK;
}

namespace {
bool group_multi_ok(int64_t n_tokens, int32_t top_k, int32_t n_experts) {
  return n_tokens > 0 && n_tokens <= (int64_t)kGrpTok * kGrpMaxWgs && top_k >= 1 && top_k <= kGrpMaxSlots &&
         n_experts >= 1 && n_experts <= kGrpMaxExperts;
}
}  // namespace

extern "C" size_t tm_group_slots_workspace_size(int64_t n_tokens, int32_t top_k, int32_t n_experts) {
  if (!group_multi_ok(n_tokens, top_k, n_experts)) return 0;
  return (size_t)tm_cdiv(n_tokens, kGrpTok) * (size_t)n_experts * sizeof(int32_t);
}

extern "C" int tm_group_slots_ws(const int64_t *ids, int64_t n_tokens, int32_t top_k, int64_t ld_ids,
                                 const uint8_t *mask, int64_t ms_b, int64_t ms_s, int32_t n_experts, int64_t so_b,
                                 int64_t so_s, int32_t *expert_offsets, int32_t *row_token, int64_t *row_out,
                                 int32_t *tiles, void *workspace, size_t workspace_bytes, tm_stream_t stream) {
  const size_t need = tm_group_slots_workspace_size(n_tokens, top_k, n_experts);
  if (need == 0)  // outside the multi-workgroup shapes: the one-workgroup grouping
    return tm_group_slots(ids, n_tokens, top_k, ld_ids, mask, ms_b, ms_s, n_experts, so_b, so_s, expert_offsets,
                          row_token, row_out, tiles, stream);
  TM_REQUIRE(ld_ids >= top_k && top_k >= 1, TM_EINVAL_SHAPE, "tm_group_slots_ws: bad sizes");
  TM_REQUIRE(ids && mask && expert_offsets && row_token && row_out && tiles, TM_EINVAL_ARG,
             "tm_group_slots_ws: null pointer");
  TM_REQUIRE(so_b % 8 == 0 && so_s % 8 == 0, TM_EINVAL_SHAPE,
             "tm_group_slots_ws: output strides (%lld, %lld) must be multiples of 8 elements", (long long)so_b,
             (long long)so_s);
  TM_REQUIRE(workspace != nullptr && workspace_bytes >= need && tm_aligned16(workspace), TM_EWORKSPACE,
             "tm_group_slots_ws: workspace %zu bytes < %zu", workspace_bytes, need);
  const int64_t t_max = tm_group_slots_tiles(n_tokens * top_k, n_experts);
  const unsigned G = (unsigned)tm_cdiv(n_tokens, kGrpTok);
  hipStream_t s = tm_hip_stream(stream);
  int32_t *counts = static_cast<int32_t *>(workspace);
  if (G == 1) {  // up to kGrpTok tokens: one launch
    hipLaunchKernelGGL(group_place_kernel<true>, dim3(1), dim3(kGrpThreads), 0, s, ids, n_tokens, top_k, ld_ids, mask,
                       ms_b, ms_s, n_experts, so_b, so_s, counts, expert_offsets, row_token, row_out, tiles, t_max);
  } else {
    hipLaunchKernelGGL(group_count_kernel, dim3(G), dim3(kGrpThreads), 0, s, ids, n_tokens, top_k, ld_ids, mask, ms_b,
                       ms_s, n_experts, counts);
    hipLaunchKernelGGL(group_place_kernel<false>, dim3(G), dim3(kGrpThreads), 0, s, ids, n_tokens, top_k, ld_ids, mask,
                       ms_b, ms_s, n_experts, so_b, so_s, counts, expert_offsets, row_token, row_out, tiles, t_max);
  }
  TM_LAUNCH_CHECK("tm_group_slots_ws");
  return TM_OK;
}

extern "C" size_t tm_swiglu_workspace_size(int64_t max_rows, int32_t inter, int32_t dtype) {
  if (max_rows <= 0 || inter <= 0) return 0;
  return (size_t)max_rows * (size_t)inter * (dtype == TM_DT_F32 ? 4 : 2);
}

// The packed path keeps the intermediate as whole 256-row tiles (one per
// entry of the tile list).
extern "C" size_t tm_grouped_swiglu_packed_workspace_size(int64_t max_rows, int32_t inter, int32_t n_experts,
                                                          int32_t dtype) {
  if (max_rows <= 0 || inter <= 0 || n_experts <= 0) return 0;
  return (size_t)tm_group_slots_tiles(max_rows, n_experts) * BM * (size_t)inter * (dtype == TM_DT_F32 ? 4 : 2);
}

namespace {

int grouped_swiglu_impl(int32_t dtype, const void *x, int64_t ld_x, int32_t hidden, int32_t inter,
                        int32_t n_experts, const void *w1, const void *w3, const void *w2, int64_t max_rows,
                        const int32_t *expert_offsets, const int32_t *row_token, const int64_t *row_out,
                        const int32_t *tiles, void *out, void *workspace, size_t workspace_bytes, bool packed,
                        tm_stream_t stream) {
  TM_REQUIRE(shapes_ok(hidden, inter), TM_EINVAL_SHAPE,
             "tm_grouped_swiglu: hidden and inter must be positive multiples of %d", kMinBN);
  TM_REQUIRE(n_experts >= 1 && max_rows >= 0 && max_rows < ((int64_t)1 << 31) && ld_x >= hidden, TM_EINVAL_SHAPE,
             "tm_grouped_swiglu: bad sizes");
  if (max_rows == 0) return TM_OK;
  TM_REQUIRE(x && w1 && w3 && w2 && expert_offsets && row_token && row_out && tiles && out, TM_EINVAL_ARG,
             "tm_grouped_swiglu: null pointer");
  TM_REQUIRE(tm_aligned16(x) && (ld_x * 2) % 16 == 0 && tm_aligned16(w1) && tm_aligned16(w3) && tm_aligned16(w2) &&
                 tm_aligned16(out),
             TM_EINVAL_SHAPE, "tm_grouped_swiglu: x rows, weights and out must be 16-byte aligned");
  const size_t need = packed ? tm_grouped_swiglu_packed_workspace_size(max_rows, inter, n_experts, dtype)
                              : tm_swiglu_workspace_size(max_rows, inter, dtype);
  TM_REQUIRE(workspace != nullptr && workspace_bytes >= need && tm_aligned16(workspace), TM_EWORKSPACE,
             "tm_grouped_swiglu: workspace %zu bytes < %zu", workspace_bytes, need);
  const int64_t t_max = tm_group_slots_tiles(max_rows, n_experts);
  const TileSrc ts{tiles, expert_offsets, t_max, (int32_t)max_rows};
  return swiglu_impl(dtype, x, ld_x, row_token, hidden, inter, w1, w3, w2, ts, max_rows < t_max ? max_rows : t_max,
                     out, 0, row_out, workspace, nullptr, 0, packed, grouped_plan(max_rows, n_experts, hidden, inter, packed),
                     tm_hip_stream(stream));  // (a tile holds at least one row)
}

}  // namespace

extern "C" int tm_grouped_swiglu(int32_t dtype, const void *x, int64_t ld_x, int32_t hidden, int32_t inter,
                                 int32_t n_experts, const void *w1, const void *w3, const void *w2, int64_t max_rows,
                                 const int32_t *expert_offsets, const int32_t *row_token, const int64_t *row_out,
                                 const int32_t *tiles, void *out, void *workspace, size_t workspace_bytes,
                                 tm_stream_t stream) {
  return grouped_swiglu_impl(dtype, x, ld_x, hidden, inter, n_experts, w1, w3, w2, max_rows, expert_offsets,
                             row_token, row_out, tiles, out, workspace, workspace_bytes, false, stream);
}

extern "C" int tm_grouped_swiglu_packed(int32_t dtype, const void *x, int64_t ld_x, int32_t hidden, int32_t inter,
                                        int32_t n_experts, const void *w1p, const void *w3p, const void *w2p,
                                        int64_t max_rows, const int32_t *expert_offsets, const int32_t *row_token,
                                        const int64_t *row_out, const int32_t *tiles, void *out, void *workspace,
                                        size_t workspace_bytes, tm_stream_t stream) {
  return grouped_swiglu_impl(dtype, x, ld_x, hidden, inter, n_experts, w1p, w3p, w2p, max_rows, expert_offsets,
                             row_token, row_out, tiles, out, workspace, workspace_bytes, true, stream);
}

extern "C" int tm_expert_pack_weights(int32_t dtype, const void *w, int32_t n_experts, int32_t hidden, int32_t inter,
                                      int32_t role, void *out, tm_stream_t stream) {
  TM_REQUIRE(shapes_ok(hidden, inter) && n_experts >= 1, TM_EINVAL_SHAPE,
             "tm_expert_pack_weights: hidden and inter must be positive multiples of %d", kMinBN);
  TM_REQUIRE(role == TM_PACK_GATE_UP || role == TM_PACK_DOWN, TM_EINVAL_ARG, "tm_expert_pack_weights: bad role");
  TM_REQUIRE(w && out, TM_EINVAL_ARG, "tm_expert_pack_weights: null pointer");
  TM_REQUIRE(tm_aligned16(w) && tm_aligned16(out), TM_EINVAL_SHAPE,
             "tm_expert_pack_weights: weights must be 16-byte aligned");
  // W1 / W3: [n_experts, inter, hidden] in 128-row tiles; W2: [n_experts, hidden, inter] in down_bn rows
  const int64_t rows = role == TM_PACK_GATE_UP ? inter : hidden;
  const int64_t K = role == TM_PACK_GATE_UP ? hidden : inter;
  const int bn = role == TM_PACK_GATE_UP ? kMinBN : down_bn(hidden);
  const int64_t esz = dtype == TM_DT_F32 ? 4 : 2;
  const char *wb = static_cast<const char *>(w);
  char *ob = static_cast<char *>(out);
  const int64_t bytes = (int64_t)n_experts * rows * K * esz;
  TM_REQUIRE(ob + bytes <= wb || wb + bytes <= ob, TM_EINVAL_ARG, "tm_expert_pack_weights: out overlaps the weights");
  const int64_t KT = K / BK;
  const int64_t blocks = (int64_t)n_experts * (rows / bn) * KT;
  hipStream_t s = tm_hip_stream(stream);
  return TM_DISPATCH_DTYPE(dtype, DT, [&] {
    if constexpr (DT == TM_DT_F32) {
      return tm_fail(TM_EINVAL_DTYPE, "tm_expert_pack_weights: dtype must be F16 or BF16");
    } else {
      using T = typename Elem<DT>::T;
      if (bn == kMinBN)
        hipLaunchKernelGGL((pack_weights_kernel<T, kMinBN>), dim3((unsigned)blocks), dim3(kThreads), 0, s,
                           static_cast<const T *>(w), K, KT, static_cast<T *>(out));
      else
        hipLaunchKernelGGL((pack_weights_kernel<T, 2 * kMinBN>), dim3((unsigned)blocks), dim3(kThreads), 0, s,
                           static_cast<const T *>(w), K, KT, static_cast<T *>(out));
      TM_LAUNCH_CHECK("tm_expert_pack_weights");
      return TM_OK;
    }
  });
}

namespace {

int expert_swiglu_impl(const char *name, int32_t dtype, const void *x, int64_t n_rows, int32_t hidden, int64_t ld_x,
                       const void *w1, const void *w3, const void *w2, int32_t inter, const void *addend,
                       int64_t ld_add, void *out, int64_t ld_out, void *workspace, size_t workspace_bytes,
                       bool packed, tm_stream_t stream) {
  TM_REQUIRE(shapes_ok(hidden, inter), TM_EINVAL_SHAPE, "%s: hidden and inter must be positive multiples of %d",
             name, kMinBN);
  TM_REQUIRE(n_rows >= 0 && n_rows < ((int64_t)1 << 31) && ld_x >= hidden && ld_out >= hidden &&
                 (addend == nullptr || ld_add >= hidden),
             TM_EINVAL_SHAPE, "%s: bad sizes", name);
  if (n_rows == 0) return TM_OK;
  TM_REQUIRE(x && w1 && w3 && w2 && out, TM_EINVAL_ARG, "%s: null pointer", name);
  TM_REQUIRE(tm_aligned16(x) && (ld_x * 2) % 16 == 0 && tm_aligned16(w1) && tm_aligned16(w3) && tm_aligned16(w2) &&
                 tm_aligned16(out) && (ld_out * 2) % 16 == 0 &&
                 (addend == nullptr || (tm_aligned16(addend) && (ld_add * 2) % 16 == 0)),
             TM_EINVAL_SHAPE, "%s: x, out and addend rows and the weights must be 16-byte aligned", name);
  const size_t need = packed ? tm_grouped_swiglu_packed_workspace_size(n_rows, inter, 1, dtype)
                              : tm_swiglu_workspace_size(n_rows, inter, dtype);
  TM_REQUIRE(workspace != nullptr && workspace_bytes >= need && tm_aligned16(workspace), TM_EWORKSPACE,
             "%s: workspace %zu bytes < %zu", name, workspace_bytes, need);
  const TileSrc ts{nullptr, nullptr, 0, (int32_t)n_rows};
  return swiglu_impl(dtype, x, ld_x, nullptr, hidden, inter, w1, w3, w2, ts, tm_cdiv(n_rows, BM), out, ld_out,
                     nullptr, workspace, addend, ld_add, packed, dense_plan(n_rows, hidden, inter),
                     tm_hip_stream(stream));
}

}  // namespace

extern "C" int tm_expert_swiglu(int32_t dtype, const void *x, int64_t n_rows, int32_t hidden, int64_t ld_x,
                                const void *w1, const void *w3, const void *w2, int32_t inter, void *out,
                                int64_t ld_out, void *workspace, size_t workspace_bytes, tm_stream_t stream) {
  return expert_swiglu_impl("tm_expert_swiglu", dtype, x, n_rows, hidden, ld_x, w1, w3, w2, inter, nullptr, 0, out,
                            ld_out, workspace, workspace_bytes, false, stream);
}

extern "C" int tm_expert_swiglu_add(int32_t dtype, const void *x, int64_t n_rows, int32_t hidden, int64_t ld_x,
                                    const void *w1, const void *w3, const void *w2, int32_t inter,
                                    const void *addend, int64_t ld_add, void *out, int64_t ld_out, void *workspace,
                                    size_t workspace_bytes, tm_stream_t stream) {
  TM_REQUIRE(addend != nullptr, TM_EINVAL_ARG, "tm_expert_swiglu_add: null addend");
  return expert_swiglu_impl("tm_expert_swiglu_add", dtype, x, n_rows, hidden, ld_x, w1, w3, w2, inter, addend, ld_add,
                            out, ld_out, workspace, workspace_bytes, false, stream);
}

extern "C" int tm_expert_swiglu_packed(int32_t dtype, const void *x, int64_t n_rows, int32_t hidden, int64_t ld_x,
                                       const void *w1p, const void *w3p, const void *w2p, int32_t inter,
                                       const void *addend, int64_t ld_add, void *out, int64_t ld_out,
                                       void *workspace, size_t workspace_bytes, tm_stream_t stream) {
  return expert_swiglu_impl("tm_expert_swiglu_packed", dtype, x, n_rows, hidden, ld_x, w1p, w3p, w2p, inter, addend,
                            ld_add, out, ld_out, workspace, workspace_bytes, true, stream);
}
