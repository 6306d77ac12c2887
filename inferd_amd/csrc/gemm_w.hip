// Prefill GEMM on T64 weights (M > 128): C (mode) = A . W^T with every weight dequantized to bf16(s q + b) (MLX qmm
// rounding, quantized.h:528-535) and fp32 accumulation (reference affine_qmm_t_nax,
// third_party/mlx/.../quantized_nax.h:938-1076, 1206-1267); in the SwiGLU mode also the gemm -> silu_mul pair of the
// MLP (engine/src/qwen35.h:2868-2878).
//
// What bounds it: the matrix cores at the clock the chip holds under their load (1.5 to 1.7 GHz on random data, by
// s_memtime against s_memrealtime), so the design spends as little else per MFMA as it can.
// - Tile 32 MT rows x 8 bands (256 columns), MT = 4 .. 8 by M, on 4 waves, one per SIMD, with a whole tile's sums in
//   the AGPRs: wave w owns two bands over all MT row tiles. So a weight is dequantized once per tile (17 VALU per 8
//   codes for 8 MT MFMAs) and an activation fragment read from LDS feeds two MFMAs. A single wave issues one
//   instruction per about 5 cycles and an MFMA takes 32, so the 3.4 others per MFMA (MT = 8) fit in its shadow.
//   Measured per 64-group step: 2280 cycles at MT = 8 (its MFMAs alone 2048), 1650 at MT = 5 (1280). The kernel before
//   it (8 waves on 256 x 256, each band dequantized by two of them, fragments read in the step that used them) took
//   about 3200.
// - A step is four sub-steps of 2 MT MFMAs (k slots 8 t .. of the fragments). Sub-step t reads the next one's
//   fragments, dequantizes in place the weight words whose MFMAs have just been issued, and carries its share of the
//   DMAs, in MT groups of two MFMAs each closed by a scheduling barrier. The block's barrier stands before sub-step 3,
//   whose operands are in registers by then.
// - Blocks are persistent (one per CU): the DMA streams run on through the end of a tile into the next one, so a
//   tile's stores overlap the next tile's first loads. Where the last round's tiles would leave CUs idle their groups
//   are shared out evenly among S blocks per tile or among all CUs: a block then sums its one or two pieces first (fp32,
//   to slots), and k_gemm_w_fixup adds a tile's pieces in K order. w_plan picks MT and the split by estimated time; over
//   twelve swept shapes no forced choice beat it by more than 4%.
// - Weights are the MFMA's A operand, so a lane holds four neighbouring columns of one row: with v_permlane32_swap
//   bf16 rows leave as 16-byte stores straight from the registers.
// Columns: where N % 256 == 0 a tile is bands 4 t .. + 3 of the left half of the columns and the same bands of the
// right half, wave w owning one of each, for the plain modes too: the SwiGLU mode pairs gate and up in one lane, and
// both modes cut the same columns at the same K, so the fused call gives the bits of the two calls it replaces.
// Measured (whole call, both on one box, before -> after): 4096 x 17408 x 5120 626 -> 573 us (other boxes 647 -> 590, 664 ->
// 614); gate and up with SwiGLU, 777 x 34816 x 5120, 341 -> 267 us (the product is not stored any more); 2048 x 5120 x 5120
// 132 -> 101 us; drawn shapes of 129 to 1500 rows 1.02 to 1.6 times faster. The matrix cores are busy for 70% of the cycles
// at MT = 8 and 55% at MT = 5 (counters).
// LDS: kWRA activation slabs [32 MT][64 bf16] (16-byte columns XOR-swizzled by row pair) and kWRW weight stages (8 code
// tiles, 8 (s, b) rows), filled by direct global -> LDS DMA; every DMA is issued by a whole wave under wave-uniform
// control flow (the LDS base goes to M0).
#include <algorithm>
#include <cmath>

#include "common.h"
#include "dma.h"
#include "host.h"
#include "kernels.h"
#include "share.h"
#include "t64.h"
#include "t64_dev.h"

namespace ifd {

constexpr int kWRA = 3;    // activation slabs in the LDS ring
constexpr int kWRW = 6;    // weight stages (their loads come from HBM: three steps ahead of the activations)
constexpr int kWBand = 4;  // M tiles per band of the tile order
constexpr int kWStage = 8 * kT64Tile;
__host__ __device__ constexpr int w_abytes(int MT) { return MT * 32 * 128; }
__host__ __device__ constexpr int w_lds(int MT) { return kWRA * w_abytes(MT) + kWRW * kWStage; }
__host__ __device__ constexpr size_t w_slot_bytes(int MT) { return (size_t)8 * MT * 16 * 64 * sizeof(float); }

struct GemmWArgs {
  const uint16_t* A;
  int lda;
  const uint8_t* wt;
  uint32_t w_bytes;  // bytes of the T64 weights (buffer bound)
  int N, K;
  void* C;
  int ldc, M, mode;
  float* part;  // piece slots [][8 bands][MT][4][64] float4
  int tiles_m, tiles_n;
  int half;           // bands per half of the columns (N % 256 == 0), or 0: a tile is 8 neighbouring bands
  int full;           // tiles 0 .. full - 1 are summed whole, block b taking b, b + gridDim.x, ..
  int rem, nsk;       // the rem other tiles' groups are shared evenly among blocks 0 .. nsk - 1 (rem < nsk)
};

// tile order: bands of kWBand M tiles, M fastest, so that neighbouring blocks (one XCD) share weight tiles in L2
__host__ __device__ inline void w_tile(int L, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int per_band = kWBand * tiles_n;
  const int bandi = L / per_band, within = L % per_band;
  const int bm = tiles_m - bandi * kWBand < kWBand ? tiles_m - bandi * kWBand : kWBand;
  tm = bandi * kWBand + within % bm;
  tn = within / bm;
}

// One wave-wide 16 (4)-byte-per-lane DMA through a buffer resource: lane l's bytes at voff(l) + soff land at
// lds + 16 l (4 l) (LDS base in M0, wave-uniform control flow only).
__device__ __forceinline__ void w_dma(__amdgpu_buffer_rsrc_t r, void* lds, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void_t*)lds, 16, (int)voff, (int)soff, 0, 0);
}
__device__ __forceinline__ void w_dma4(__amdgpu_buffer_rsrc_t r, void* lds, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void_t*)lds, 4, (int)voff, (int)soff, 0, 0);
}

// physical band of wave w's band nb of column tile tn (may lie past the last one when half == 0)
__device__ __forceinline__ int w_band(const GemmWArgs& p, int tn, int w, int nb) {
  return p.half ? nb * p.half + 4 * tn + w : 8 * tn + 2 * w + nb;
}

// Two dwords of neighbouring 8-column groups (u: columns .. + 3 by half h of the wave): afterwards half h holds, in lo
// and hi, the dwords of group h for columns 0 .. 3 and 4 .. 7.
__device__ __forceinline__ void w_swap32(uint32_t& lo, uint32_t& hi) {
  const auto r = __builtin_amdgcn_permlane32_swap(lo, hi, false, false);
  lo = r[0], hi = r[1];
}

// How the sums are stored: as the modes 0 - 3 with 16-byte accesses (C and its rows 16-byte aligned, N % 16 == 0), or
// one value at a time by the runtime mode, with the MFMA's operands exchanged so that a lane holds one column of 16 rows
// and a store's lanes neighbouring columns. A template parameter: with all of them in one kernel the epilogue's registers
// spill the sums.
enum WStore { kWBf16 = 0, kWAdd = 1, kWF32 = 2, kWSwiglu = kModeSwiglu, kWScalar = 4 };

// Sixteen bf16 values of one row in a band (this lane: columns 8 q + 4 h + e, value v[4 q + e]) to `row` (the band's
// first column, of n more columns), 16 bytes per store; lanes that are not live only take part in the swaps.
__device__ __forceinline__ void w_store_bf16(uint16_t* row, int n, int h, bool live, const float (&v)[16]) {
  uint32_t d[4][2];
#pragma unroll
  for (int q = 0; q < 4; q++) d[q][0] = pack_bf2(v[4 * q], v[4 * q + 1]), d[q][1] = pack_bf2(v[4 * q + 2], v[4 * q + 3]);
#pragma unroll
  for (int u = 0; u < 2; u++) {
    w_swap32(d[2 * u][0], d[2 * u + 1][0]);
    w_swap32(d[2 * u][1], d[2 * u + 1][1]);
    if (live && 16 * u < n)
      *(u32x4*)(row + 16 * u + 8 * h) = u32x4{d[2 * u][0], d[2 * u][1], d[2 * u + 1][0], d[2 * u + 1][1]};
  }
}

// The old values (mode 1) under a wave's two bands, of one row tile: this lane's 16 of each, as bf16 pairs (past M
// or N those of the last row or columns, which nothing uses). row: this lane's row, 32 a + j in its tile.
struct WOld {
  u32x2 c[2][4];
};
template <int ST>
__device__ __forceinline__ void w_load_old(const GemmWArgs& p, int row, int tn, int w, int j, int h, WOld& old) {
#pragma unroll
  for (int nb = 0; nb < 2; nb++) {
    const int col = w_band(p, tn, w, nb) * 32;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      if constexpr (ST == kWAdd) {
        const size_t o = (size_t)min(row, p.M - 1) * p.ldc + min(col + 8 * q, p.N - 8) + 4 * h;
        old.c[nb][q] = *(const u32x2*)((const uint16_t*)p.C + o);
      } else {
        uint32_t v[4];
#pragma unroll
        for (int e = 0; e < 4; e++)
          v[e] = ((const uint16_t*)p.C)[(size_t)min(row - j + 8 * q + 4 * h + e, p.M - 1) * p.ldc + min(col + j, p.N - 1)];
        old.c[nb][q] = u32x2{v[0] | v[1] << 16, v[2] | v[3] << 16};
      }
    }
  }
}

// The sums of wave w's two bands in one row tile of column tile tn, stored (old: the values that mode 1 adds to).
template <int ST>
__device__ __forceinline__ void w_emit(const GemmWArgs& p, int row, int tn, int w, int j, int h, const f32x16& x0,
                                       const f32x16& x1, const WOld& old) {
  const bool live = row < p.M;
  float v[2][16];
#pragma unroll
  for (int e = 0; e < 16; e++) v[0][e] = x0[e], v[1][e] = x1[e];
  if constexpr (ST == kWSwiglu) {
    float hv[16];
#pragma unroll
    for (int e = 0; e < 16; e++) hv[e] = swiglu_f(bf2f(f2bf(v[0][e])), bf2f(f2bf(v[1][e])));
    w_store_bf16((uint16_t*)p.C + (size_t)row * p.ldc + (4 * tn + w) * 32, 32, h, live, hv);
    return;
  }
#pragma unroll
  for (int nb = 0; nb < 2; nb++) {
    const int col = w_band(p, tn, w, nb) * 32, n = p.N - col;
    if (n <= 0) continue;  // wave-uniform
    const size_t o = (size_t)row * p.ldc + col;
    if (ST == kWAdd || (ST == kWScalar && p.mode == 1))
#pragma unroll
      for (int e = 0; e < 16; e++) v[nb][e] += bf2f((uint16_t)(old.c[nb][e / 4][e % 4 / 2] >> (16 * (e % 2))));
    if constexpr (ST == kWScalar) {
#pragma unroll
      for (int e = 0; e < 16; e++) {
        const int r = row - j + 8 * (e / 4) + 4 * h + e % 4;
        if (j < n && r < p.M) store_mode(p.C, (size_t)r * p.ldc + col + j, v[nb][e], p.mode & 2);
      }
    } else if constexpr (ST == kWF32) {
#pragma unroll
      for (int q = 0; q < 4; q++)
        if (live && 8 * q < n)
          *(float4*)((float*)p.C + o + 8 * q + 4 * h) =
              make_float4(v[nb][4 * q], v[nb][4 * q + 1], v[nb][4 * q + 2], v[nb][4 * q + 3]);
    } else {
      w_store_bf16((uint16_t*)p.C + o, n, h, live, v[nb]);
    }
  }
}

template <int MT, int ST>
__global__ __launch_bounds__(256, 1) void k_gemm_w(GemmWArgs p) {
  extern __shared__ __align__(16) uint8_t lds[];
  constexpr int BM = 32 * MT, RA = kWRA, RW = kWRW, AB = w_abytes(MT), HA = (MT + 1) / 2;
  static_assert(RW >= RA + 2 && (RA - 1) * (MT + 3) <= 63 && w_lds(MT) <= 160 * 1024, "rings, vmcnt range");
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, j = lane & 31, h = lane >> 5;
  const int b = xcd_remap(blockIdx.x, gridDim.x), nblk = gridDim.x;
  const int nbands = t64_bands(p.N), G = p.K / kGroup;
  const uint32_t gstride = (uint32_t)nbands * kT64Tile;
  uint8_t* const aring = lds;
  uint8_t* const wring = lds + RA * AB;
  const __amdgpu_buffer_rsrc_t ra =
      __builtin_amdgcn_make_buffer_rsrc((void*)p.A, 0, (int)((uint32_t)p.M * p.lda * 2u), 0x00020000);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)p.wt, 0, (int)p.w_bytes, 0x00020000);

  // the block's segments: its share of the cut tiles (one or two pieces), then its whole tiles
  int u0 = 0, u1 = 0, hp = 0;
  if (b < p.nsk) {
    u0 = share_start(b, p.rem, p.nsk, G), u1 = share_start(b + 1, p.rem, p.nsk, G);
    hp = (u1 - 1) / G > u0 / G ? 2 : 1;
  }
  const int nseg = hp + (b < p.full ? (p.full - 1 - b) / nblk + 1 : 0);
  if (nseg == 0) return;
  auto segment = [&](int s, int& t, int& g0, int& ng) __attribute__((always_inline)) {
    if (s < hp) {
      t = u0 / G + s;
      g0 = s ? 0 : u0 - t * G;
      ng = min(u1 - t * G, G) - g0;
      t += p.full;
    } else {
      t = b + (s - hp) * nblk;
      g0 = 0, ng = G;
    }
  };

  // ---- the two DMA streams (activations, weights): each walks the segments' groups and then stays on the last one.
  // Rows past M re-read row M - 1, bands past the last one the last (their sums are not stored).
  uint32_t va[MT], vw[2], vs, a_so, w_so;
  int a_seg = 0, a_left, w_seg = 0, w_left;
  auto open_a = [&]() __attribute__((always_inline)) {
    int t, tm, tn, g0;
    segment(a_seg, t, g0, a_left);
    w_tile(t, p.tiles_m, p.tiles_n, tm, tn);
    a_so = (uint32_t)g0 * 2u * kGroup;
#pragma unroll
    for (int q = 0; q < MT; q++) {
      const int r = 8 * (MT * wave + q) + lane / 8, c = (lane & 7) ^ ((r >> 1) & 7);
      va[q] = (uint32_t)min(tm * BM + r, p.M - 1) * (uint32_t)p.lda * 2u + 16u * c;
    }
  };
  auto open_w = [&]() __attribute__((always_inline)) {
    int t, tm, tn, g0;
    segment(w_seg, t, g0, w_left);
    w_tile(t, p.tiles_m, p.tiles_n, tm, tn);
    w_so = (uint32_t)g0 * gstride;
#pragma unroll
    for (int nb = 0; nb < 2; nb++) vw[nb] = (uint32_t)min(w_band(p, tn, wave, nb), nbands - 1) * kT64Tile + 16u * lane;
    vs = (uint32_t)min(w_band(p, tn, wave, h), nbands - 1) * kT64Tile + kT64Codes + 4u * j;
  };
  auto adv_a = [&]() __attribute__((always_inline)) {
    if (--a_left) a_so += 2u * kGroup;
    else if (a_seg + 1 < nseg) a_seg++, open_a();
    else a_left = 1;
  };
  auto adv_w = [&]() __attribute__((always_inline)) {
    if (--w_left) w_so += gstride;
    else if (w_seg + 1 < nseg) w_seg++, open_w();
    else w_left = 1;
  };
  auto issue_a = [&](uint8_t* st, int d) __attribute__((always_inline)) {
    w_dma(ra, st + (MT * wave + d) * 1024, va[d], a_so);
  };
  auto issue_w = [&](uint8_t* st, int d) __attribute__((always_inline)) {  // codes of the two bands, their (s, b) rows
    if (d < 2) w_dma(rw, st + (2 * wave + d) * kT64Codes, vw[d], w_so);
    else w_dma4(rw, st + 8 * kT64Codes + 2 * wave * 128, vs, w_so);
  };
  open_a();
  open_w();

  f32x16 acc[2][MT];
#pragma unroll
  for (int nb = 0; nb < 2; nb++)
#pragma unroll
    for (int a = 0; a < MT; a++) acc[nb][a] = zero16();
  // af: activation fragments by sub-step parity; bf: the unit's dequantized words; cw, csb: the next unit's codes and
  // (s, b); w3: this unit's last code words, dequantized in its own first sub-step with sa, sb, bi (still this unit's)
  u32x4 af[2][MT], bf[2][4], cw[2];
  uint32_t csb[2], w3[2], asw[4];
  float sa[2], sb[2], bi[2];
#pragma unroll
  for (int t = 0; t < 4; t++) asw[t] = j * 128 + 16 * ((4 * h + t) ^ ((j >> 1) & 7));
  auto scales = [&](int nb) __attribute__((always_inline)) {
    const float s = bf2f((uint16_t)(csb[nb] & 0xFFFFu));
    bi[nb] = bf2f((uint16_t)(csb[nb] >> 16)), sa[nb] = t64_sa(s), sb[nb] = t64_sb(s);
  };
  auto read_codes = [&](const uint8_t* st, int nb) __attribute__((always_inline)) {
    cw[nb] = *(const u32x4*)(st + (2 * wave + nb) * kT64Codes + 16 * lane);
    csb[nb] = *(const uint32_t*)(st + 8 * kT64Codes + (2 * wave + nb) * 128 + 4 * j);
  };

  // Unit i issues the second half of A(i + RA - 1)'s DMAs (sub-step 0), W(i + RW - 1) (sub-step 1) and, after its
  // barrier, the first half of A(i + RA) (sub-step 3) into the slab whose last fragments were read in sub-step 2. The
  // prologue leaves the streams as if units 1 - RA .. -1 had run, in their order, so that the units' wait counts what was
  // issued from unit 0 on: W(0 .. RW - RA - 1), then A(s) and W(RW - RA + s) for s = 0 .. RA - 2, half of A(RA - 1).
  auto prologue_w = [&](int s) __attribute__((always_inline)) {
#pragma unroll
    for (int d = 0; d < 3; d++) issue_w(wring + s * kWStage, d);
    adv_w();
  };
#pragma unroll
  for (int s = 0; s < RW - RA; s++) prologue_w(s);
#pragma unroll
  for (int s = 0; s < RA; s++) {
#pragma unroll
    for (int d = 0; d < (s + 1 < RA ? MT : HA); d++) issue_a(aring + s * AB, d);
    if (s + 1 < RA) {
      adv_a();
      prologue_w(RW - RA + s);
    }
  }
  // W(0), W(1) and A(0) have landed: the younger DMAs are W(RW - RA .. RW - 2), A(1 .. RA - 2) and the half
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((RA - 1) * 3 + (RA - 2) * MT + HA) : "memory");
#pragma unroll
  for (int nb = 0; nb < 2; nb++) {
    read_codes(wring, nb);
    scales(nb);
#pragma unroll
    for (int t = 0; t < 3; t++) bf[nb][t] = t64_dequant(cw[nb][t], sa[nb], sb[nb], bi[nb]);
    w3[nb] = cw[nb][3];
    read_codes(wring + kWStage, nb);
  }
#pragma unroll
  for (int a = 0; a < MT; a++) af[0][a] = *(const u32x4*)(aring + asw[0] + a * 4096);

  // One unit. Offsets of its slab (sl), the slab of the unit before (slp) and after (sln), of the weight stages of
  // units i + 2 (rd2) and i + RW - 1 (wr): scalars, so that the loop body is one unit and the sums stay where they are.
  int sl = 0, slp = (RA - 1) * AB, sln = AB, rd2 = 2 * kWStage, wr = (RW - 1) * kWStage;
  auto unit = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 4; t++) {
      if (t == 1)
#pragma unroll
        for (int nb = 0; nb < 2; nb++) scales(nb), w3[nb] = cw[nb][3];
      // A(i + 1) and, older, W(i + 2) have landed: younger are A(i + 2 .. i + RA - 1) and the W of the RA - 1 units that
      // issued them, this one included
      if (t == 3)
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((RA - 2) * (MT + 3) + 3) : "memory");
      const uint8_t* const src = aring + (asw[(t + 1) & 3] + (t == 3 ? sln : sl));
      const int tw = (t + 3) & 3;  // the word dequantized: the one of the sub-step before
#pragma unroll
      for (int g = 0; g < MT; g++) {
        if (t == 3 && g < HA) issue_a(aring + sl, g);
        if (t == 0 && HA + g < MT) issue_a(aring + slp, HA + g);
        if (t == 1 && g < 3) issue_w(wring + wr, g);
        af[(t + 1) & 1][g] = *(const u32x4*)(src + g * 4096);
#pragma unroll
        for (int e = g * 8 / MT; e < (g + 1) * 8 / MT; e++) {  // code pair e % 4 of band e / 4 (t64_dequant's steps)
          const int nb = e / 4, pr = e % 4;
          const uint32_t w = t == 0 ? w3[nb] : cw[nb][tw];
          const uint32_t x = (pr < 2 ? w : w >> 8) & (pr % 2 ? 0x00F000F0u : 0x000F000Fu);
          const float sc = pr % 2 ? sb[nb] : sa[nb];
          bf[nb][tw][pr] = pack_bf2(__builtin_fmaf(sc, h16_lo(x), bi[nb]), __builtin_fmaf(sc, h16_hi(x), bi[nb]));
        }
#pragma unroll
        for (int nb = 0; nb < 2; nb++)
          acc[nb][g] = ST == kWScalar ? mfma_bf16(af[t & 1][g], bf[nb][t], acc[nb][g])
                                      : mfma_bf16(bf[nb][t], af[t & 1][g], acc[nb][g]);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
        __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);  // VALU
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (t == 0) adv_a();
      if (t == 1) adv_w();
      if (t == 3)
#pragma unroll
        for (int nb = 0; nb < 2; nb++) read_codes(wring + rd2, nb);
    }
    slp = sl, sl = sln;
    sln = sln + AB == RA * AB ? 0 : sln + AB;
    rd2 = rd2 + kWStage == RW * kWStage ? 0 : rd2 + kWStage;
    wr = wr + kWStage == RW * kWStage ? 0 : wr + kWStage;
  };

#pragma clang loop unroll(disable)
  for (int s = 0; s < nseg; s++) {
    int t, g0, ng;
    segment(s, t, g0, ng);
#pragma clang loop unroll(disable)
    for (int i = 0; i < ng; i++) unit();
    // the segment's sums: lane (j, h) holds row 32 a + j, columns 8 q + 4 h + e of its two bands (kWScalar: the converse)
    if (s < hp) {
      float4* const slot =
          (float4*)p.part + (size_t)share_piece(b, t - p.full, p.rem, p.nsk) * 8 * MT * 4 * 64 + lane;
#pragma unroll
      for (int nb = 0; nb < 2; nb++)
#pragma unroll
        for (int a = 0; a < MT; a++)
#pragma unroll
          for (int q = 0; q < 4; q++)
            slot[((size_t)((2 * wave + nb) * MT + a) * 4 + q) * 64] = make_float4(
                acc[nb][a][4 * q], acc[nb][a][4 * q + 1], acc[nb][a][4 * q + 2], acc[nb][a][4 * q + 3]);
    } else {
      // read by asm, so that the compiler keeps every other tile's sums in AGPRs meanwhile; the wait covers the last
      // MFMA's 18 states before such a read
      asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
      int tm, tn;
      w_tile(t, p.tiles_m, p.tiles_n, tm, tn);
      // the residual rows of up to four row tiles are requested together: their latency is paid per group
      constexpr int GA = ST == kWAdd ? 4 : ST == kWScalar ? 2 : 1;
      WOld old[GA];
#pragma unroll
      for (int a = 0; a < MT; a++) {
        if (a % GA == 0 && (ST == kWAdd || (ST == kWScalar && p.mode == 1))) {
#pragma unroll
          for (int i = 0; i < GA; i++)
            if (a + i < MT) w_load_old<ST>(p, tm * BM + 32 * (a + i) + j, tn, wave, j, h, old[i]);
          __builtin_amdgcn_sched_barrier(0);
        }
        f32x16 x[2];
#pragma unroll
        for (int nb = 0; nb < 2; nb++)
#pragma unroll
          for (int e = 0; e < 16; e++) asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(x[nb][e]) : "a"(acc[nb][a][e]));
        w_emit<ST>(p, tm * BM + 32 * a + j, tn, wave, j, h, x[0], x[1], old[a % GA]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int nb = 0; nb < 2; nb++)
#pragma unroll
      for (int a = 0; a < MT; a++) acc[nb][a] = zero16();
  }
  // the streams' last DMAs land before the block's LDS is given back
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
}

// The cut tiles: block (tile, row tile a), wave w: its two bands' pieces summed in K order and stored.
template <int MT, int ST>
__global__ __launch_bounds__(256) void k_gemm_w_fixup(GemmWArgs p) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, j = lane & 31, h = lane >> 5, a = blockIdx.y;
  int tm, tn;
  w_tile(p.full + blockIdx.x, p.tiles_m, p.tiles_n, tm, tn);
  if (tm * 32 * MT + 32 * a >= p.M) return;
  const int tile = blockIdx.x, G = p.K / kGroup;
  const int b0 = share_of(tile * G, p.rem, p.nsk, G), b1 = share_of(tile * G + G - 1, p.rem, p.nsk, G);
  const float4* const slot =
      (const float4*)p.part + (size_t)share_piece(b0, tile, p.rem, p.nsk) * 8 * MT * 4 * 64 + lane;
  f32x16 x[2] = {zero16(), zero16()};
  WOld old;
  if (p.mode == 1) w_load_old<ST>(p, tm * 32 * MT + 32 * a + j, tn, wave, j, h, old);
#pragma unroll 2
  for (int z = 0; z <= b1 - b0; z++) {
    float4 v[2][4];
#pragma unroll
    for (int nb = 0; nb < 2; nb++)
#pragma unroll
      for (int q = 0; q < 4; q++) v[nb][q] = slot[((size_t)((z * 8 + 2 * wave + nb) * MT + a) * 4 + q) * 64];
#pragma unroll
    for (int nb = 0; nb < 2; nb++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        x[nb][4 * q] += v[nb][q].x, x[nb][4 * q + 1] += v[nb][q].y;
        x[nb][4 * q + 2] += v[nb][q].z, x[nb][4 * q + 3] += v[nb][q].w;
      }
  }
  w_emit<ST>(p, tm * 32 * MT + 32 * a + j, tn, wave, j, h, x[0], x[1], old);
}

// ---- host side
struct WPlan {
  int MT, tiles_m, tiles_n, full, rem, nsk;
  double ns;  // estimated time
};
// ns of a step by MT, at the clock that a long run of steps holds (taller tiles keep the matrix cores busier and the
// clock lower), of what a segment costs beside its steps (first loads, stores), and of a fixup launch; its bytes are
// written and read at about 5 TB/s each
static double w_step(int MT) { return MT == 8 ? 1560 : MT == 7 ? 1410 : MT == 6 ? 1250 : MT == 5 ? 1100 : 890; }
constexpr double kWSegment = 3000, kWFixup = 5000, kWBytesPerNs = 5000;

static WPlan w_plan_mt(int MT, int M, int N, int K, size_t part_bytes) {
  WPlan pl{};
  pl.MT = MT;
  pl.tiles_m = (M + 32 * MT - 1) / (32 * MT);
  pl.tiles_n = (t64_bands(N) + 7) / 8;
  const int G = K / kGroup, cu = cu_count();
  const long tiles = (long)pl.tiles_m * pl.tiles_n;
  const int rem = (int)(tiles % cu);
  const double step = w_step(MT), whole = (double)(tiles / cu) * (G * step + kWSegment);
  pl.full = (int)tiles;
  pl.ns = whole + (rem ? G * step + kWSegment : 0);
  // the last round's tiles shared by S blocks each, or (S = 0) by all CUs
  for (int S = 0; rem && S <= std::min(cu / rem, 16); S++) {
    const int nsk = S ? rem * S : cu;
    const size_t bytes = (size_t)share_pieces(rem, nsk) * w_slot_bytes(MT);
    const double share = (double)rem * G / nsk;
    if (S == 1 || share < 4 || bytes > part_bytes) continue;
    const double ns = whole + std::ceil(share) * step + kWSegment * (nsk % rem ? 1.5 : 1) + kWFixup +
                      2.0 * bytes / kWBytesPerNs;
    if (ns < pl.ns) pl.ns = ns, pl.full = (int)tiles - rem, pl.rem = rem, pl.nsk = nsk;
  }
  return pl;
}
// The row-tile height with the least estimated time: it fits M (a 777-row prompt is five tiles of 160 rows rather than
// four of 256) and the CUs' rounds.
static WPlan w_plan(int M, int N, int K, size_t part_bytes) {
  WPlan best = w_plan_mt(8, M, N, K, part_bytes);
  for (int MT = 7; MT >= 4; MT--) {
    const WPlan pl = w_plan_mt(MT, M, N, K, part_bytes);
    if (pl.ns < best.ns) best = pl;
  }
  return best;
}
constexpr size_t kWPartMax = (size_t)64 << 20;

bool gemm_w_applies(int M, int N, int K, int mode) {
  if (M <= 128 || K % kGroup || K / kGroup < 4 || t64_bytes(N, K) >= ((size_t)1 << 31)) return false;
  return mode != kModeSwiglu || N % 256 == 0;
}

size_t gemm_w_workspace(int M, int N, int K) {
  const WPlan pl = w_plan(M, N, K, kWPartMax);
  return (size_t)share_pieces(pl.rem, pl.nsk) * w_slot_bytes(pl.MT);
}

template <int MT, int ST>
static int launch_w_cfg(const GemmWArgs& a, hipStream_t st) {
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute((const void*)k_gemm_w<MT, ST>, hipFuncAttributeMaxDynamicSharedMemorySize, w_lds(MT));
    attr = true;
  }
  const int nblk = std::max(std::min(a.full, cu_count()), a.nsk);
  hipLaunchKernelGGL((k_gemm_w<MT, ST>), dim3(nblk), dim3(256), w_lds(MT), st, a);
  IFD_TRY(check_launch("gemm_w"));
  if (!a.rem) return IFD_OK;
  hipLaunchKernelGGL((k_gemm_w_fixup<MT, ST>), dim3(a.rem, MT), dim3(256), 0, st, a);
  return check_launch("gemm_w fixup");
}
template <int MT>
static int launch_w_st(const GemmWArgs& a, hipStream_t st) {
  const bool vec = aligned(a.C, 16) && a.ldc % (a.mode == 2 ? 4 : 8) == 0 && a.N % 16 == 0;
  if (!vec) return launch_w_cfg<MT, kWScalar>(a, st);
  switch (a.mode) {
    case 1: return launch_w_cfg<MT, kWAdd>(a, st);
    case 2: return launch_w_cfg<MT, kWF32>(a, st);
    case kModeSwiglu: return launch_w_cfg<MT, kWSwiglu>(a, st);
    default: return launch_w_cfg<MT, kWBf16>(a, st);
  }
}

int launch_gemm_w(const uint16_t* A, int lda, const void* wt, int N, int K, void* C, int ldc, int M, int mode,
                  void* ws, size_t ws_bytes, hipStream_t st) {
  if (M == 0) return IFD_OK;
  if ((size_t)M * lda * 2 >= ((size_t)1 << 31)) return fail(IFD_ERR_UNSUPPORTED, "gemm_w: operands past 2 GiB");
  const WPlan pl = w_plan(M, N, K, ws ? std::min(ws_bytes, kWPartMax) : 0);
  GemmWArgs a{A, lda, (const uint8_t*)wt, (uint32_t)t64_bytes(N, K), N, K, C, ldc, M, mode, (float*)ws, pl.tiles_m,
              pl.tiles_n, N % 256 == 0 ? N / 64 : 0, pl.full, pl.rem, pl.nsk};
  switch (pl.MT) {
    case 4: return launch_w_st<4>(a, st);
    case 5: return launch_w_st<5>(a, st);
    case 6: return launch_w_st<6>(a, st);
    case 7: return launch_w_st<7>(a, st);
    default: return launch_w_st<8>(a, st);
  }
}

}  // namespace ifd
