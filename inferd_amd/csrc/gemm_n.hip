// GEMM on T64 weights for decode batches (16 < M <= 128): C (mode) = A . W^T, and with the SwiGLU its gate/up pair.
// Serves the reference's affine_qmm_t_nax (third_party/mlx/.../quantized_nax.h:938-1076) with its split-K variant
// (engine/kernels/qmm_splitk.metal:14-107) and the gemm -> silu_mul pair of the MLP (engine/src/qwen35.h:1693-1700).
//
// A block sums a tile of all M rows (MT row tiles of 32) x 4 bands (128 columns) on NKQ K-groups of two waves: K-group
// kq takes 64-groups kq, kq + NKQ, .., and wave w of a K-group two bands over all MT row tiles. At the end of a tile
// the K-groups' sums meet in LDS.
// Why so:
// - A single wave issues one instruction per about 5 cycles, two on a SIMD one per 2.4 (3.5 for the conversions of
//   the dequant), four one per 1.7 (2.8), measured. With one wave per SIMD (the stream-K kernel that served these rows
//   before) a step of 32 MFMAs took about 1450 cycles at best, against 1100 for two waves that share the SIMD. Waves
//   that split K instead of columns or rows neither dequantize a weight twice nor read more activations from LDS.
// - Narrow tiles: with 8-band tiles a 34816-column linear has 136 tiles for 256 CUs, and cutting every tile wrote and
//   read 50 MB of fp32 pieces at M = 128, half of the call's time. With 4 bands 256 tiles are summed whole and only the
//   other 16 are shared out (k_gemm_n_fixup adds their pieces in K order).
// - The weights go straight to registers, two units ahead (no other wave needs them), so that LDS holds RA activation
//   slabs per K-group. Not so in FORM 2: the compiler takes the LDS read of the row scales for dependent on every DMA in
//   flight and waits for all loads before it, once per unit.
// FORM 0: weights dequantized to bf16(s q + b) (MLX qmm rounding, quantized.h:528-535), in place, one sub-step behind
// the MFMAs. FORM 1: the decode GEMV's arithmetic (core.metal:85-171): 128 + q as exact bf16, and per 64-group the fp32
// epilogue adds s P + (b - 128 s) X, X from an MFMA against ones. FORM 2: the reference's W4A8 with per-(row, 64-group)
// int8 activations (w4a8.metal:24-98): A holds the codes xq as exact bf16 integers, so P = sum (128 + q) xq and
// X = sum xq are exact (integers below 2^24), and the epilogue adds sx (s P + (b - 128 s) X) with the row's scale for
// that group; more than 64 rows are blocks of 64, neighbours in the tile order.
// What bounds it: at 128 rows rounds at 1.65 us per 4 units (1.3 PFLOP/s, the clock that the matrix cores hold under load)
// and about 12 us of first loads, sums and stores, so that the matrix cores are busy for half of the kernel's cycles; below,
// the weight stream (0.9 us per round at 32 rows for 0.8 at 6 TB/s) and the same 12 us. A tile change pays a memory latency:
// the compiler waits for all loads before the first LDS write of the sums, so open_w's loads do not run on over them.
// Measured, whole call on weights from memory, same box, before (stream-K or K-split tiles) -> after: 32768 x 5120 at M =
// 128 / 64 / 32 62.9 / 40.2 / 31.4 -> 51.9 / 31.2 / 24.6 us; gate and up with SwiGLU, 34816 x 5120 (16 shared tiles), 61.1 /
// 42.5 / 35.5 -> 56.4 / 39.7 / 31.2; 5120 x 17408 41.2 / 34.0 / 25.2 -> 37.5 / 29.1 / 20.7. FORM 2 (with its prep), before
// the K-split tiles: 34816 x 5120 at M = 24 / 64 / 128 / 255 55.8 / 89.5 / 127.4 / 215.5 -> 39.7 / 52.5 / 87.1 / 158.9 us;
// 5120 x 17408 at M = 24 28.1 -> 26.5.
// Deeper register sets (NS 5 to 7) measured slower at 32 and 64 rows.
// Activation slabs: [32 MT][64 bf16], 16-byte columns XOR-swizzled by row pair, filled by direct global -> LDS DMA, each
// issued by a whole wave under wave-uniform control flow (the LDS base goes to M0).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"
#include "dma.h"
#include "host.h"
#include "kernels.h"
#include "share.h"
#include "t64.h"
#include "t64_dev.h"

namespace ifd {

__host__ __device__ constexpr int n_ra(int MT) { return MT == 4 ? 2 : MT == 3 ? 3 : 4; }
__host__ __device__ constexpr int n_ring(int MT, int NKQ) { return NKQ * n_ra(MT) * MT * 4096; }
__host__ __device__ constexpr int n_lds(int MT, int NKQ, int FORM) {
  return n_ring(MT, NKQ) + (FORM == 2 ? NKQ * (n_ra(MT) + 1) * 256 : 0);
}
__host__ __device__ constexpr size_t n_slot_bytes(int MT) { return (size_t)4 * MT * 16 * 64 * sizeof(float); }

struct GemmNArgs {
  const uint16_t* A;
  int lda;
  const uint8_t* wt;
  uint32_t w_bytes;  // bytes of the T64 weights (buffer bound)
  int N, K;
  void* C;
  int ldc, M, mode;
  const float* sxT;   // FORM 2: the activation scales transposed, [G][Mp], Mp >= 64 tiles_m + 64
  int Mp;
  int tiles_m;        // row blocks of 32 MT (row block fastest in the tile order)
  float* part;        // piece slots [][2 waves][2 bands][MT * 4][64] float4
  int half;           // bands per half of the columns (N % 128 == 0), or 0: a tile is 4 neighbouring bands
  int full;           // tiles 0 .. full - 1 are summed whole, block b taking b, b + gridDim.x, ..
  int rem, nsk;       // the rem other tiles' rounds are shared evenly among blocks 0 .. nsk - 1 (rem < nsk)
};

// physical band of wave w's band nb of tile t (may lie past the last one when half == 0)
__device__ __forceinline__ int n_band(const GemmNArgs& p, int t, int w, int nb) {
  return p.half ? nb * p.half + 2 * t + w : 4 * t + 2 * w + nb;
}

// Rows r0 .. r0 + 3 of column j of wave w's two bands of tile t, stored by the mode.
template <int MODE>
__device__ __forceinline__ void n_emit(const GemmNArgs& p, int t, int w, int r0, int j, const float (&v0)[4],
                                       const float (&v1)[4]) {
  if constexpr (MODE == kModeSwiglu) {
    uint16_t* const o = (uint16_t*)p.C + (2 * t + w) * 32 + j;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const uint16_t y = f2bf(swiglu_f(bf2f(f2bf(v0[e])), bf2f(f2bf(v1[e]))));
      if (r0 + e < p.M) o[(size_t)(r0 + e) * p.ldc] = y;
    }
    return;
  }
#pragma unroll
  for (int nb = 0; nb < 2; nb++) {
    const int col = n_band(p, t, w, nb) * 32 + j;
    float v[4], old[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = nb ? v1[e] : v0[e];
    if constexpr (MODE == 1)
#pragma unroll
      for (int e = 0; e < 4; e++)
        old[e] = bf2f(((const uint16_t*)p.C)[(size_t)min(r0 + e, p.M - 1) * p.ldc + min(col, p.N - 1)]);
    if (col < p.N)
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (r0 + e < p.M) store_mode(p.C, (size_t)(r0 + e) * p.ldc + col, v[e] + old[e], MODE & 2);
  }
}

template <int K, int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (K < N) {
    f(std::integral_constant<int, K>{});
    static_for<K + 1, N>(f);
  }
}

template <int MT, int NKQ, int FORM, int NS, int MODE>
__global__ __launch_bounds__(128 * NKQ, 1) void k_gemm_n(GemmNArgs p) {
  extern __shared__ __align__(16) uint8_t lds[];
  constexpr int RA = n_ra(MT), AB = MT * 4096;
  constexpr int SX = FORM == 2 ? 1 : 0;
  static_assert((RA - 1) * 4 + (RA - 2) * (2 * MT + SX) <= 63 && n_lds(MT, NKQ, FORM) <= 160 * 1024, "vmcnt range, LDS");
  static_assert(FORM != 2 || MT <= 2, "one scale DMA covers 64 rows");
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kq = wv >> 1, w = wv & 1;
  const int lane = threadIdx.x & 63, j = lane & 31, h = lane >> 5;
  const int b = xcd_remap(blockIdx.x, gridDim.x), nblk = gridDim.x;
  const int nbands = t64_bands(p.N), R = p.K / kGroup / NKQ;  // rounds per tile
  const uint32_t gstride = (uint32_t)nbands * kT64Tile;
  uint8_t* const ring = lds + kq * RA * AB;
  // FORM 2: the units' row scales, RA + 1 slots of 64 floats: a slot is refilled a unit later than its slab, when both
  // waves are past the epilogue that read it
  uint8_t* const sxring = lds + n_ring(MT, NKQ) + kq * (RA + 1) * 256;
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      (void*)p.sxT, 0, FORM == 2 ? (int)((uint32_t)(p.K / kGroup) * p.Mp * 4u) : 0, 0x00020000);
  const __amdgpu_buffer_rsrc_t ra =
      __builtin_amdgcn_make_buffer_rsrc((void*)p.A, 0, (int)((uint32_t)p.M * p.lda * 2u), 0x00020000);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)p.wt, 0, (int)p.w_bytes, 0x00020000);

  int u0 = 0, u1 = 0, hp = 0;
  if (b < p.nsk) {
    u0 = share_start(b, p.rem, p.nsk, R), u1 = share_start(b + 1, p.rem, p.nsk, R);
    hp = u1 == u0 ? 0 : (u1 - 1) / R > u0 / R ? 2 : 1;
  }
  const int nseg = hp + (b < p.full ? (p.full - 1 - b) / nblk + 1 : 0);

  // activation DMA d (0 .. 2 MT - 1) of wave w covers rows 8 (2 MT w + d) .. + 7 of the slab: lane -> row + lane / 8,
  // physical 16-byte column lane % 8 holding logical column (lane % 8) ^ ((row / 2) % 8). Rows past M lie past the
  // buffer: those loads are dropped, and their sums not stored.
  uint32_t va[2];
#pragma unroll
  for (int o = 0; o < 2; o++) {
    const int r = 8 * (2 * MT * w + o) + lane / 8, c = (lane & 7) ^ ((r >> 1) & 7);
    va[o] = (uint32_t)r * (uint32_t)p.lda * 2u + 16u * c;
  }
  const uint32_t asw = j * 128 + 16 * ((4 * h) ^ ((j >> 1) & 7));  // fragment addresses: sub-step k's is asw ^ 16 k
  const u32x4 ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};

  auto segment = [&](int sg, int& t, int& r0, int& nr) __attribute__((always_inline)) {
    if (sg < hp) {
      t = u0 / R + sg;
      r0 = sg ? 0 : u0 - t * R;
      nr = min(u1 - t * R, R) - r0;
      t += p.full;
    } else {
      t = b + (sg - hp) * nblk, r0 = 0, nr = R;
    }
  };
  // NS units' weights, loaded NS - 1 units ahead. The stream walks the K-group's units r0 .. r0 + nr - 1 of a segment and
  // then stays on the last one; open_w starts it on a segment, before the one before has stored its sums (after which the
  // compiler waits for these loads: see above).
  u32x4 cw[NS][2];
  uint32_t csb[NS][2], vw[2], w_so;
  int w_left;
  auto load_w = [&](auto SC) __attribute__((always_inline)) {
    constexpr int s = decltype(SC)::value;
#pragma unroll
    for (int nb = 0; nb < 2; nb++) {
      cw[s][nb] = __builtin_amdgcn_raw_buffer_load_b128(rw, 16 * lane, w_so + vw[nb], 2);
      csb[s][nb] = __builtin_amdgcn_raw_buffer_load_b32(rw, 4 * j + kT64Codes, w_so + vw[nb], 2);
    }
    w_so += --w_left > 0 ? gstride * NKQ : 0u;
  };
  auto open_w = [&](int sg) __attribute__((always_inline)) {
    int t, r0;
    segment(sg, t, r0, w_left);
    w_so = (uint32_t)(r0 * NKQ + kq) * gstride;
#pragma unroll
    for (int nb = 0; nb < 2; nb++) vw[nb] = (uint32_t)min(n_band(p, t / p.tiles_m, w, nb), nbands - 1) * kT64Tile;
    static_for<0, FORM == 0 ? NS : NS - 1>([&](auto SC) __attribute__((always_inline)) { load_w(SC); });
    __builtin_amdgcn_sched_barrier(0);
  };
  if (nseg == 0) return;
  open_w(0);

#pragma clang loop unroll(disable)
  for (int sg = 0; sg < nseg; sg++) {
    int t, r0, nr;
    segment(sg, t, r0, nr);
    const int tm = t % p.tiles_m, tn = t / p.tiles_m;
    const uint32_t m_off = (uint32_t)tm * 32u * MT * p.lda * 2u;
    uint32_t a_so = (uint32_t)(r0 * NKQ + kq) * 2u * kGroup;
    int a_left = nr;
    uint32_t x_so = ((uint32_t)(r0 * NKQ + kq) * p.Mp + (uint32_t)tm * 32u * MT) * 4u;
    auto adv_a = [&]() __attribute__((always_inline)) {
      const bool on = --a_left > 0;
      a_so += on ? 2u * kGroup * NKQ : 0u;
      if constexpr (FORM == 2) x_so += on ? (uint32_t)p.Mp * 4u * NKQ : 0u;
    };
    auto issue_x = [&](int slot) __attribute__((always_inline)) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_void_t*)(sxring + slot), 4, 4 * lane, (int)x_so, 0, 0);
    };
    auto issue_a = [&](uint8_t* st, int d) __attribute__((always_inline)) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_void_t*)(st + (2 * MT * w + d) * 1024), 16,
                                               (int)(va[d & 1] + m_off + (uint32_t)(d & ~1) * 16u * p.lda), (int)a_so, 0, 0);
    };

    f32x16 acc[2][MT], P[2][MT], X[MT];
#pragma unroll
    for (int nb = 0; nb < 2; nb++)
#pragma unroll
      for (int a = 0; a < MT; a++) acc[nb][a] = zero16();
    u32x4 af[MT], bf[2][4];
    uint32_t w3[2];
    float sa[2], sb[2], bi[2];

    // prologue, after the weights': A(0 .. RA - 2) and half of A(RA - 1). All but the half land before the first unit:
    // the count of the units' wait (below) is that of a stream with weights between the slabs, which begins here, so
    // it covers the slabs that the units issue (from A(RA - 1)) and not these.
#pragma unroll
    for (int s = 0; s < RA; s++) {
#pragma unroll
      for (int d = 0; d < (s + 1 < RA ? 2 * MT : MT); d++) issue_a(ring + s * AB, d);
      if (s + 1 < RA) {
        if constexpr (FORM == 2) issue_x(s * 256);
        adv_a();
      }
    }
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(MT) : "memory");
#pragma unroll
    for (int a = 0; a < MT; a++) af[a] = *(const u32x4*)(ring + asw + a * 4096);
    auto scales = [&](uint32_t x, int nb) __attribute__((always_inline)) {
      const float s = bf2f((uint16_t)(x & 0xFFFFu));
      bi[nb] = bf2f((uint16_t)(x >> 16));
      if constexpr (FORM == 0) sa[nb] = t64_sa(s), sb[nb] = t64_sb(s);
      else sa[nb] = s, bi[nb] -= 128.f * s;
    };
    if constexpr (FORM == 0)
#pragma unroll
      for (int nb = 0; nb < 2; nb++) {
        scales(csb[0][nb], nb);
#pragma unroll
        for (int k = 0; k < 3; k++) bf[nb][k] = t64_dequant(cw[0][nb][k], sa[nb], sb[nb], bi[nb]);
        w3[nb] = cw[0][nb][3];
      }

    // One unit i (SC = i mod NS); offsets of its slab, the one before and after. Sub-step k issues, after barriers as in
    // the comment of each: the second half of A(i + RA - 1) (k = 0), W(i + NS) or, FORM 1, W(i + NS - 1) into the
    // registers of W(i) or W(i - 1) (k = 1), the first half of A(i + RA) (k = 3, into the slab whose last fragments were read at k = 2).
    int sl = 0, slp = (RA - 1) * AB, sln = AB, xr = 0, xw = (RA - 1) * 256;
    // TAIL: one of the segment's last units, past the whole turns of the register sets. Nothing reads what it would load
    // (the compiler may drop such a load, and the count with it), so it loads no weights and its wait counts none.
    auto unit = [&](auto SC, auto TAIL) __attribute__((always_inline)) {
      constexpr int YOUNGER = (RA - 2) * (2 * MT + SX) + (TAIL.value ? 0 : (RA - 1) * 4);
      constexpr int S = decltype(SC)::value, S1 = (S + 1) % NS, SL = (S + NS - 1) % NS;
      if constexpr (FORM != 0)
#pragma unroll
        for (int nb = 0; nb < 2; nb++) scales(csb[S][nb], nb);
#pragma unroll
      for (int k = 0; k < 4; k++) {
        if (FORM == 0 && k == 1)
#pragma unroll
          for (int nb = 0; nb < 2; nb++) scales(csb[S1][nb], nb), w3[nb] = cw[S1][nb][3];
        if (k == 1 && !TAIL.value) load_w(std::integral_constant<int, FORM == 0 ? S : SL>{});
        // A(i + 1) has landed: in the prologue (i + 1 < RA - 1), or else, its second half being unit i + 2 - RA's, younger
        // are A(i + 2 .. i + RA - 1) and the weights of units i + 2 - RA .. i
        if (k == 3)
          asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(YOUNGER) : "memory");
        const uint8_t* const src = ring + ((asw ^ (16u * ((k + 1) & 3))) + (k == 3 ? sln : sl));
        const int kw = (k + 3) & 3;
        if constexpr (FORM != 0)
#pragma unroll
          for (int nb = 0; nb < 2; nb++) bf[nb][k] = t64_off128(cw[S][nb][k]);
#pragma unroll
        for (int g = 0; g < MT; g++) {
          if (k == 3) issue_a(ring + sl, g);
          if (k == 0) issue_a(ring + slp, MT + g);
          if constexpr (FORM == 0) {
#pragma unroll
            for (int nb = 0; nb < 2; nb++) acc[nb][g] = mfma_bf16(af[g], bf[nb][k], acc[nb][g]);
          } else {
#pragma unroll
            for (int nb = 0; nb < 2; nb++) P[nb][g] = mfma_bf16(af[g], bf[nb][k], k ? P[nb][g] : zero16());
            X[g] = mfma_bf16(af[g], ones, k ? X[g] : zero16());
          }
          af[g] = *(const u32x4*)(src + g * 4096);
          if constexpr (FORM == 0) {
#pragma unroll
            for (int e = g * 8 / MT; e < (g + 1) * 8 / MT; e++) {  // code pair e % 4 of band e / 4 (t64_dequant's steps)
              const int nb = e / 4, pr = e % 4;
              const uint32_t x0 = k == 0 ? w3[nb] : cw[S1][nb][kw];
              const uint32_t x = (pr < 2 ? x0 : x0 >> 8) & (pr % 2 ? 0x00F000F0u : 0x000F000Fu);
              const float sc = pr % 2 ? sb[nb] : sa[nb];
              bf[nb][kw][pr] = pack_bf2(__builtin_fmaf(sc, h16_lo(x), bi[nb]), __builtin_fmaf(sc, h16_hi(x), bi[nb]));
            }
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
            __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);  // VALU
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
            __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        if (k == 0) {
          if constexpr (FORM == 2) {
            issue_x(xw);
            xw = xw == RA * 256 ? 0 : xw + 256;
          }
          adv_a();
        }
      }
      if constexpr (FORM == 1)
#pragma unroll
        for (int nb = 0; nb < 2; nb++)
#pragma unroll
          for (int a = 0; a < MT; a++)
#pragma unroll
            for (int e = 0; e < 16; e++)
              acc[nb][a][e] = __builtin_fmaf(sa[nb], P[nb][a][e], __builtin_fmaf(bi[nb], X[a][e], acc[nb][a][e]));
      if constexpr (FORM == 2) {
#pragma unroll
        for (int a = 0; a < MT; a++)
#pragma unroll
          for (int c = 0; c < 4; c++) {
            const float4 x = *(const float4*)(sxring + xr + (32 * a + 8 * c + 4 * h) * 4);
            const float sx[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
            for (int nb = 0; nb < 2; nb++)
#pragma unroll
              for (int e = 0; e < 4; e++)
                acc[nb][a][4 * c + e] = __builtin_fmaf(
                    sx[e], __builtin_fmaf(sa[nb], P[nb][a][4 * c + e], bi[nb] * X[a][4 * c + e]), acc[nb][a][4 * c + e]);
          }
        xr = xr == RA * 256 ? 0 : xr + 256;
      }
      slp = sl, sl = sln;
      sln = sln + AB == RA * AB ? 0 : sln + AB;
    };
    // whole turns of the register sets, then the rest (the compiler's waits for the weights count exactly in a loop
    // without exits in its middle)
    const int turns = nr / NS, rest = nr - turns * NS;
#pragma clang loop unroll(disable)
    for (int i = 0; i < turns; i++)
      static_for<0, NS>([&](auto SC) __attribute__((always_inline)) { unit(SC, std::false_type{}); });
    static_for<0, NS - 1>([&](auto SC) __attribute__((always_inline)) {
      if (SC.value < rest) unit(SC, std::true_type{});
    });

    // ---- the K-groups' sums meet in LDS, PQ quads of rows (quad c: rows 8 c + 4 h .. + 3) at a time:
    // [K-group][wave][band][quad][lane] float4. K-group kq adds them, in K-group order, for quads kq, kq + NKQ, ..
    constexpr int Q = 4 * MT, PQ = NKQ * Q * 4096 <= n_ring(MT, NKQ) ? Q : Q / 2;
    float4* const red = (float4*)lds;
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (sg + 1 < nseg) open_w(sg + 1);
#pragma unroll
    for (int c0 = 0; c0 < Q; c0 += PQ) {
      if (c0) __syncthreads();
#pragma unroll
      for (int nb = 0; nb < 2; nb++)
#pragma unroll
        for (int c = 0; c < PQ; c++) {
          const f32x16& x = acc[nb][(c0 + c) / 4];
          const int e = (c0 + c) % 4 * 4;
          red[(((kq * 2 + w) * 2 + nb) * PQ + c) * 64 + lane] = make_float4(x[e], x[e + 1], x[e + 2], x[e + 3]);
        }
      __syncthreads();
#pragma clang loop unroll(disable)
      for (int c = kq; c < PQ; c += NKQ) {
        float4 x[2][NKQ];
#pragma unroll
        for (int nb = 0; nb < 2; nb++)
#pragma unroll
          for (int z = 0; z < NKQ; z++) x[nb][z] = red[(((z * 2 + w) * 2 + nb) * PQ + c) * 64 + lane];
        float v[2][4] = {};
#pragma unroll
        for (int nb = 0; nb < 2; nb++)
#pragma unroll
          for (int z = 0; z < NKQ; z++)
            v[nb][0] += x[nb][z].x, v[nb][1] += x[nb][z].y, v[nb][2] += x[nb][z].z, v[nb][3] += x[nb][z].w;
        if (sg < hp) {
          float4* const slot = (float4*)p.part + (size_t)share_piece(b, t - p.full, p.rem, p.nsk) * 4 * Q * 64 + lane;
#pragma unroll
          for (int nb = 0; nb < 2; nb++)
            slot[((w * 2 + nb) * Q + c0 + c) * 64] = make_float4(v[nb][0], v[nb][1], v[nb][2], v[nb][3]);
        } else {
          n_emit<MODE>(p, tn, w, 32 * MT * tm + 8 * (c0 + c) + 4 * h, j, v[0], v[1]);
        }
      }
    }
    __syncthreads();
  }
}

// The shared tiles: block (tile, quad pair), wave (w, one of the pair): its two bands' pieces summed in K order.
template <int MT, int MODE>
__global__ __launch_bounds__(256) void k_gemm_n_fixup(GemmNArgs p, int R) {
  constexpr int Q = 4 * MT;
  const int wv = threadIdx.x >> 6, w = wv & 1, c = blockIdx.y * 2 + (wv >> 1);
  const int lane = threadIdx.x & 63, j = lane & 31, h = lane >> 5, tile = blockIdx.x;
  const int tm = (p.full + tile) % p.tiles_m, tn = (p.full + tile) / p.tiles_m;
  if (32 * MT * tm + 8 * c >= p.M) return;
  const int b0 = share_of(tile * R, p.rem, p.nsk, R), b1 = share_of(tile * R + R - 1, p.rem, p.nsk, R);
  const float4* const slot = (const float4*)p.part + (size_t)share_piece(b0, tile, p.rem, p.nsk) * 4 * Q * 64 + lane;
  float v[2][4] = {};
#pragma unroll 4
  for (int z = 0; z <= b1 - b0; z++) {
    float4 x[2];
#pragma unroll
    for (int nb = 0; nb < 2; nb++) x[nb] = slot[((size_t)(z * 2 + w) * 2 + nb) * Q * 64 + c * 64];
#pragma unroll
    for (int nb = 0; nb < 2; nb++) v[nb][0] += x[nb].x, v[nb][1] += x[nb].y, v[nb][2] += x[nb].z, v[nb][3] += x[nb].w;
  }
  n_emit<MODE>(p, tn, w, 32 * MT * tm + 8 * c + 4 * h, j, v[0], v[1]);
}

// ---- host side
struct NPlan {
  int MT, NKQ, form, tiles_m, full, rem, nsk;
  double ns;
};
constexpr double kNSegment = 4000, kNFixup = 5000, kNBytesPerNs = 5000;
// ns of a round: the MFMAs and dequant of NKQ units, or their weights at a CU's share of 6 TB/s
static double n_round(int MT) { return MT == 4 ? 1650 : MT == 3 ? 1400 : MT == 2 ? 1150 : 900; }

// form: 0 dequantized weights, 1 the decode GEMV's arithmetic (up to 64 rows), 2 the same on int8 rows with scales per
// 64-group (blocks of at most 64 rows); the pieces of shared tiles fit in part_bytes
static NPlan n_plan(int M, int N, int K, int form, size_t part_bytes = SIZE_MAX) {
  NPlan pl{};
  pl.form = form;
  pl.MT = form == 2 ? (M > 32 ? 2 : 1) : (M + 31) / 32;
  pl.tiles_m = (M + 32 * pl.MT - 1) / (32 * pl.MT);
  const int G = K / kGroup, cu = cu_count();
  pl.NKQ = 4;
  const int R = G / pl.NKQ, tiles = pl.tiles_m * ((t64_bands(N) + 3) / 4), rem = tiles % cu;
  const double rd = n_round(pl.MT), whole = (tiles / cu) * (R * rd + kNSegment);
  pl.full = tiles;
  pl.ns = whole + (rem ? R * rd + kNSegment : 0);
  for (int S = 0; rem && S <= std::min(cu / rem, 32); S++) {
    const int nsk = S ? rem * S : cu;
    const double share = (double)rem * R / nsk, bytes = (double)share_pieces(rem, nsk) * n_slot_bytes(pl.MT);
    if (S == 1 || share < 1 || bytes > part_bytes) continue;
    const double ns = whole + std::ceil(share) * rd + kNSegment * (nsk % rem ? 1.5 : 1) + kNFixup + 2 * bytes / kNBytesPerNs;
    if (ns < pl.ns) pl.ns = ns, pl.full = tiles - rem, pl.rem = rem, pl.nsk = nsk;
  }
  return pl;
}

bool gemm_n_applies(int M, int N, int K, int mode) {
  if (M <= 16 || M > 128 || K % 256 || t64_bytes(N, K) >= ((size_t)1 << 31)) return false;
  return mode != kModeSwiglu || N % 128 == 0;
}
bool gemm_n_a8_applies(int M, int N, int K) {
  return M > 16 && (size_t)M * K * 2 < ((size_t)1 << 31) && K % 256 == 0 && t64_bytes(N, K) < ((size_t)1 << 31);
}
size_t gemm_n_workspace(int M, int N, int K, int form) {
  const NPlan pl = n_plan(M, N, K, form);
  return (size_t)share_pieces(pl.rem, pl.nsk) * n_slot_bytes(pl.MT);
}

template <int MT, int NKQ, int FORM, int NS, int MODE>
static int launch_n_mode(const GemmNArgs& a, hipStream_t st) {
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute((const void*)k_gemm_n<MT, NKQ, FORM, NS, MODE>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, n_lds(MT, NKQ, FORM));
    attr = true;
  }
  const int nblk = std::max(std::min(a.full, cu_count()), a.nsk);
  hipLaunchKernelGGL((k_gemm_n<MT, NKQ, FORM, NS, MODE>), dim3(nblk), dim3(128 * NKQ), n_lds(MT, NKQ, FORM), st, a);
  IFD_TRY(check_launch("gemm_n"));
  if (!a.rem) return IFD_OK;
  hipLaunchKernelGGL((k_gemm_n_fixup<MT, MODE>), dim3(a.rem, 2 * MT), dim3(256), 0, st, a, a.K / kGroup / NKQ);
  return check_launch("gemm_n fixup");
}
template <int MT, int NKQ, int FORM, int NS>
static int launch_n_cfg(const GemmNArgs& a, hipStream_t st) {
  switch (a.mode) {
    case 1: return launch_n_mode<MT, NKQ, FORM, NS, 1>(a, st);
    case 2: return launch_n_mode<MT, NKQ, FORM, NS, 2>(a, st);
    case kModeSwiglu:
      if constexpr (FORM != 2) return launch_n_mode<MT, NKQ, FORM, NS, kModeSwiglu>(a, st);
      return fail(IFD_ERR_UNSUPPORTED, "gemm_n: no SwiGLU on int8 rows");
    default: return launch_n_mode<MT, NKQ, FORM, NS, 0>(a, st);
  }
}

int launch_gemm_n(const uint16_t* A, int lda, const float* sxT, int Mp, const void* wt, int N, int K, void* C, int ldc,
                  int M, int mode, int form, void* ws, size_t ws_bytes, hipStream_t st) {
  if (M == 0) return IFD_OK;
  if ((size_t)M * lda * 2 >= ((size_t)1 << 31) || (size_t)(K / kGroup) * Mp * 4 >= ((size_t)1 << 31))
    return fail(IFD_ERR_UNSUPPORTED, "gemm_n: operands past 2 GiB");
  const NPlan pl = n_plan(M, N, K, form, ws ? ws_bytes : 0);
  GemmNArgs a{A, lda, (const uint8_t*)wt, (uint32_t)t64_bytes(N, K), N, K, C, ldc, M, mode, sxT, Mp, pl.tiles_m, (float*)ws,
              N % 128 == 0 ? N / 64 : 0, pl.full, pl.rem, pl.nsk};
  if (form == 2) return pl.MT == 1 ? launch_n_cfg<1, 4, 2, 3>(a, st) : launch_n_cfg<2, 4, 2, 3>(a, st);
  if (pl.MT == 1) return form ? launch_n_cfg<1, 4, 1, 3>(a, st) : launch_n_cfg<1, 4, 0, 3>(a, st);
  if (pl.MT == 2) return form ? launch_n_cfg<2, 4, 1, 3>(a, st) : launch_n_cfg<2, 4, 0, 3>(a, st);
  return pl.MT == 3 ? launch_n_cfg<3, 4, 0, 3>(a, st) : launch_n_cfg<4, 4, 0, 3>(a, st);
}

}  // namespace ifd
