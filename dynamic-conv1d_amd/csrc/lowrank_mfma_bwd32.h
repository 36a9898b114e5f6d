// Lowrank backward on gfx950 matrix cores, one and two rank chunks (bf16 / fp16):
// every pass of a problem that takes several, and one-pass problems up to the size of
// the last-level cache (larger ones: bwd_streams in lowrank_mfma_bwd.hip).
//
// One pass over x and dy produces dx, dz, dU and dstatic_w (reference:
// lowrank.py:87-140 and 159-205, two kernels that both read dy).
//
// Tile: a wavefront owns 32 rows x 32 channels; lane l = 16q + n owns the eight
// rows 8q..8q+7 and the channels 2n, 2n+1 (one 4-byte load per row, 64
// contiguous bytes per row across a group's 16 lanes; the workgroup's 8
// wavefronts lie side by side on 256 channels of the same rows).  With
// G_k[t, d] = bf16(dy[t, d] * x[t-k, d]) (the reference also rounds this
// product to bf16 before its dot products, lowrank.py:128):
//   * dU[r, kD+d] += sum_t z_eff[t, r] G_k[t, d]: 16x16x32 MFMA with K = the 32
//     rows.  A lane's eight G values of a channel are the B operand as they lie
//     (rows 8q..8q+7 of column n); A is z_eff transposed.
//   * dz[t, r] += sum_d G_k[t, d] U_eff[r, kD+d]: K = the 32 channels.  The
//     packed G goes through the wavefront's LDS slot and comes back by row with
//     transposing reads (ds_read_b64_tr_b16).  Rows 4a..4a+3 of a half h of the
//     tile are rows 8a+4h..8a+4h+3, and each octet's channels come even ones first:
//     MFMA rows and the K index may be permuted alike in both operands.
//   * Tap weights Kw[t, k, :] = z_eff[t, :] U_eff[:, k]: per half one 16x16x16
//     MFMA (one rank chunk) or 16x16x32 (two, K = 32 ranks); the lane's result
//     is rows 8q+4h..+3 of its own channel.
//   * dx[t, d] = sum_k dy[t+k, d] Kw[t+k, k, d] (+ dy: tap 0's accumulator
//     starts at 1) in scatter form: dy[s] Kw[s, k] is added to row s-k; the
//     W-1 <= 7 rows of the group above pass up with one ds_bpermute each, and
//     group 3's open rows wait one tile for group 0's sums of the next.
//
// Why eight rows to a lane: what a lane does per tile beside its products
// (halo rows of x, sums for the group above, row closing, tap-weight operands)
// is per lane and not per row, so it halves against four rows to a lane; dU
// takes K = 32 rows per MFMA, twice the rate of K = 16; the dU accumulators of
// 32 channels take half the registers of 64; and the scatter form, whose sums
// reach one group up, serves W <= 8.
// Measured, B4 T4096 D2048 bf16, whole backward, inputs out of the cache, 16-row tiles
// -> these: W 8 R15 + static 82.7 -> 78.0 us, W 16 R16 174 -> 168, W 2 R31 + static 58.6
// -> 55.3, R63 + static 156 -> 140 (the two passes of ranks as one launch); W 4 R16 56.9
// -> 56.1 and R31 + static 67.6 -> 67.8 (equal; inputs left in the cache 53 -> 46 and 67
// -> 63); B2 T512 D256 R15 + static 16.9 -> 13.5 (a launch's serial start, below); R16 at
// W 1 and 2 44.8 -> 49.3 and 45.8 -> 51.1 (left in the cache equal and 43 -> 40).
// What bounds it: the chain of one tile (loads, conversions, products, the LDS
// transposes, sums), which two wavefronts per SIMD overlap in part.  W 4 R16 waits for
// 28% of its wavefronts' cycles and issues for 39%, W 4 with two rank chunks 37% and 33%,
// passes that add to dx 43% and 29%, passes of ranks without dx 50% and 29%; the matrix
// pipe is busy for 13-19%.  Transposing G with identity products instead of LDS took two
// rank chunks to 140 us, a second tile in flight changed nothing.
//
// The launch's start is kept short, since a small problem is little else: the
// group's pointers are scalar loads at a run-time offset, and the U operands are
// staged without branches, rolled where they go to LDS (6.3 -> 4.5 us to the
// first tile).
//
// A tile's rows are loaded into the registers of one whose rows have just been
// converted to fp32, so one tile is in flight while one is computed (a second one in
// flight at W <= 4: B4 T4096 D2048 R16 W 2 40 -> 42 us, B8 T8192 D4096 equal).
//
// dz partial sums over the 256 channels are added in LDS in wave order, once
// per DZB tiles, and written as one fp32 partial per 256-channel group; dU
// accumulates in registers over the run and goes out as one fp32 partial per
// run.  reduce_partials sums both in a fixed order.
//
// Passes (ACC, DXM), groups and layouts: see lowrank_mfma_bwd.hip.
#pragma once

#include "lowrank_mfma_bwd.h"

namespace dc {

// v_perm selectors: the low (high) halves of two words, packed.
constexpr uint32_t kEven = 0x05040100u, kOdd = 0x07060302u;

// Sum of two byte offsets, either of which may be kOobLane (out of range).
__device__ __forceinline__ int oob_add(int a, int b) { return (a | b) >= kOobLane ? kOobLane : a + b; }

template <typename T, int W, int RC, bool ACC, int DXM>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void lr_bwd_t32(LrBwdArgs a) {
  static_assert((RC == 1 && W <= 8) || (RC == 2 && W <= 4), "operands and accumulators of one pass");
  constexpr int NW = 8;                     // wavefronts: 256 channels
  constexpr int NR = W + 7;                 // x rows 8q-W+1 .. 8q+7 per lane
  // halo rows of x from the neighbour lanes where the registers hold the previous
  // tile's (B4 T4096 D2048 backward R16 59.2 -> 58.5 us, R63 + static 151.5 -> 148.9;
  // two rank chunks with dx spill with it: 123 -> 129 us), else loaded
  constexpr bool HX = W > 1 && ((RC == 1 && W <= 4) || DXM == 3);
  constexpr int NX = HX ? 8 : NR;           // x rows loaded per lane
  constexpr int NO = W > 1 ? W - 1 : 1;     // open rows of a group (none at W 1)
  constexpr int kFirstOpen = 9 - W;         // rows kFirstOpen .. 7 take the group below's sums
  constexpr bool NODX = DXM == 3;
  // U operands in registers where they fit (one rank chunk, W <= 4), else in LDS
  constexpr bool UREG = RC == 1 && W <= 4;
  constexpr int DZB = RC == 1 ? 2 : 1;      // tiles per dz batch
  constexpr int GPL = 272;                  // bytes per 4-row plane of the G tile (32 channels x 8 B + 16)
  typedef Pair LV;
  typedef DxVec<T, DXM == 1 || DXM == 2> DV;
  typedef DxVec<T, DXM == 1> DVS;
  typedef ZRaw<T, RC, true> ZR;
  // Passes that add to an earlier one's dx (ACC): when its rows are loaded (load_dxo).
  // Two rank chunks at W 4 and one at any W have no registers for them beside a
  // tile's fp32 rows, and take them before the last tap; the fp32 accumulator's at W <=
  // 2 come with the tile, which is too short to hide them, at W 3 at its start.  And the
  // passes that stream more than the last-level cache keeps (an fp32 accumulator, or
  // two rank chunks at W 4) read dy and store dx nontemporal.  B4 T4096 D2048, inputs
  // out of the cache, rows held from the tile's start with the open ones carried (8-12
  // registers spilled) -> now: R31 + static W 8 155 -> 149 us, W 12 227 -> 215, W 20 515
  // -> 453, R64 W 20 1113 -> 947, R127 + static W 8 934 -> 813, R160 W 1 380 -> 372, R255 +
  // static W 4 919 -> 794.  Rows with the tile at W 4 spill (W 20: 788).
  enum { kDxoTile, kDxoLastTap, kDxoAhead };
  constexpr int DXO = RC == 1 || DXM == 0 || W == 4 ? kDxoLastTap : W <= 2 ? kDxoAhead : kDxoTile;
  constexpr bool NTP = RC == 2 && (DXM == 1 || DXM == 2 || (ACC && W == 4));
  __shared__ u32x4 us[NW][UREG ? 1 : W * RC * 64];
  __shared__ __attribute__((aligned(16))) uint8_t gtile[NW][8 * GPL];
  __shared__ __attribute__((aligned(16))) float dzred[2][DZB][NW][RC * 512];

  const int lane = threadIdx.x & 63, wave = wave_id();
  const int q = lane >> 4, n = lane & 15;
  const int lb0 = xcd_remap(blockIdx.x, a.nblk);
  const int g = __builtin_amdgcn_readfirstlane(lb0 / a.nblk1);
  const int lb = lb0 - g * a.nblk1;
  // the group's pointers by scalar loads at a uniform offset of the argument block
  const auto* gp = kernel_args<LrBwdArgs>()->grp + g;
  const uint16_t* __restrict__ x = reinterpret_cast<const uint16_t*>(gp->x);
  const uint16_t* __restrict__ z = reinterpret_cast<const uint16_t*>(gp->z);
  const uint16_t* __restrict__ U = reinterpret_cast<const uint16_t*>(gp->U);
  const uint16_t* __restrict__ sw = reinterpret_cast<const uint16_t*>(gp->sw);
  const uint16_t* __restrict__ dy = reinterpret_cast<const uint16_t*>(gp->dy);
  char* __restrict__ dx = reinterpret_cast<char*>(gp->dx);
  float* __restrict__ part_dz = gp->part_dz;
  float* __restrict__ part_du = gp->part_du;
  // passes of ranks without dx (NODX) share one launch: neighbouring blocks take
  // the same rows and channels, so the second pass reads x and dy from the L2
  const int ps = NODX ? lb % a.nrp : 0, cl0 = NODX ? lb / a.nrp : lb;
  const int cg = cl0 % a.ncg, du_slot = cl0 / a.ncg, sp = a.sp0 + du_slot;
  const int D = a.D, Tn = a.Tn;
  const int d0 = (cg * NW + wave) * 32;
  const int col = d0 + 2 * n;
  const bool chv = col < D;  // the lane's 2 channels inside D (D % 8 == 0: both or none)
  const int ntile = (Tn + 31) >> 5;
  // the workgroup's run: tiles [tile0, tile1) of sequence b; its buffer resources start at row rb
  const int b = sp / a.nspb;
  const int tile0 = (sp - b * a.nspb) * a.seg;
  const int tile1 = min(tile0 + a.seg, ntile);
  const int rb = run_base_row(2 * tile0);
  const int64_t row0 = (int64_t)b * Tn, rrow = row0 + rb;
  const int rofs = NODX ? 32 * ps : 0;
  const int R = NODX ? max(min(a.R - rofs, 32), 0) : a.R, RK = NODX ? min(a.RK - rofs, 32) : a.RK;
  if constexpr (NODX) {
    z += rofs;
    U += (int64_t)rofs * a.uld;
    part_dz += rofs;
    part_du += (int64_t)rofs * a.uld;
  }
  const int kofs = ACC || NODX ? a.kofs : 0;  // a later pass of taps: x read, dx stored kofs rows earlier
  const float res = a.residual && a.kofs == 0 ? 1.f : 0.f;
  // head-major dy: the wavefront's channels lie in one head (yhd % 64 == 0), whose [T, yhd] block rdy covers
  const int yhd = a.yhd, head = d0 / yhd;
  const int rowb = yhd * 2, xrowb = a.xld * 2, dxrowb = a.dxld * DV::ES;
  const int dxsld = DXM == 2 ? a.dxsld : a.dxld, dxsrowb = dxsld * DVS::ES;
  const rsrc_t rx = run_rsrc(x + rrow * a.xld, Tn - rb, xrowb);
  const rsrc_t rdy = run_rsrc(dy + row0 * D + ((int64_t)head * Tn + rb) * yhd, Tn - rb, rowb);
  const rsrc_t rdx = run_rsrc(dx + rrow * a.dxld * DV::ES, Tn - rb, dxrowb);
  char* __restrict__ dxs = DXM == 2 ? reinterpret_cast<char*>(gp->dxs) : dx;
  const rsrc_t rdxs = DXM == 2 ? run_rsrc(dxs + rrow * dxsld * DVS::ES, Tn - rb, dxsrowb) : rdx;
  const int zld = a.zld, zr = a.zr, zrk = a.zrk;
  const rsrc_t rz = run_rsrc(z + rrow * zld, Tn - rb, zld * 2);
  const rsrc_t rpz = run_rsrc(part_dz + ((int64_t)cg * a.BT + rrow) * a.dzld, Tn - rb, a.dzld * 4);
  // byte offsets of the lane's row-8q channels in dy, x and dx
  const int lane_off = chv ? (8 * q * yhd + col - head * yhd) * 2 : kOobLane;
  const int xlane_off = chv ? (8 * q * a.xld + col) * 2 : kOobLane;
  const int dxlane_off = chv ? (8 * q * a.dxld + col) * DV::ES : kOobLane;
  const int dxslane_off = chv ? (8 * q * dxsld + col) * DVS::ES : kOobLane;
  // ACC: the earlier passes' dx of the rows that close_rows(tile) stores
  auto load_dxo = [&](int tile, typename DV::type(&dxo)[ACC ? 8 : 1]) {
    if constexpr (ACC) {
      const int cur = tile < tile1 ? dxlane_off + (tile * 32 - rb - kofs) * dxrowb : kOobTile;
      const int prev = tile > tile0 ? dxlane_off + ((tile - 1) * 32 - rb - kofs) * dxrowb : kOobTile;
#pragma unroll
      for (int i = 0; i < 8; ++i)
        dxo[i] = DV::load(rdx, (W > 1 && i >= kFirstOpen && q == 3 ? prev : cur) + i * dxrowb);
    }
  };
  const int zrow = 8 * (n >> 2) + (n & 3);  // tile row of the lane's z operand in half 0 (half 1: + 4)

  // Tile inputs (buffer loads: rows outside the sequence and channels past D
  // read 0; a tile past the run the out-of-range offset kOobTile).  dy and z of
  // the tile after the run are read too: its first rows close the run's last dx rows.
  struct TileIn {
    uint32_t xr[NX], dyr[8];
    ZR zraw[RC == 2 ? 1 : 2];
    u32x4 z32[RC == 2 ? 2 : 1];
    typename DV::type dxo[ACC && DXO == kDxoAhead ? 8 : 1];
  };
  TileIn in;
  auto load_tile = [&](int tile) {
    const int xtoff = tile < tile1 ? (tile * 32 - rb - kofs) * xrowb : kOobTile;
    const bool ylive = NODX ? tile < tile1 : tile <= tile1;
    const int toff = ylive ? (tile * 32 - rb) * rowb : kOobTile;
#pragma unroll
    for (int m = 0; m < NX; ++m) in.xr[m] = LV::load(rx, xlane_off + xtoff + (m + 8 - NX) * xrowb);
#pragma unroll
    for (int m = 0; m < 8; ++m) in.dyr[m] = bload32<NTP ? kNt : 0>(rdy, lane_off + toff + m * rowb);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int zoff = ylive ? (tile * 32 + zrow + 4 * h - rb) * zld * 2 : kOobTile;
      if constexpr (RC == 2)
        in.z32[h] = bload128(rz, ylive ? zoff + 16 * q : kOobTile);
      else
        in.zraw[h].load(rz, zoff, zr, q);
    }
    if constexpr (ACC && DXO == kDxoAhead) load_dxo(tile, in.dxo);
  };
  load_tile(tile0);
  // HX: x rows 8q-W+1 .. 8q-1 are own rows of the lane group above (lane - 16),
  // or for group 0 those of group 3 in the tile before (prev: loaded for the run's
  // first tile), passed with one ds_bpermute each.
  uint32_t prev[NO];
  if constexpr (HX) {
#pragma unroll
    for (int m = 0; m < W - 1; ++m)
      prev[m] = LV::load(rx, (chv ? col * 2 : kOobLane) + (tile0 * 32 - kofs + m - (W - 1) - rb) * xrowb);
  }
  __builtin_amdgcn_sched_barrier(0);  // the first tile's loads go out before the U staging waits

  // ---- U_eff operands of the wavefront's 32 channels (rows >= R of U and
  // channels past D read 0; the static row is OR-ed in).  Per tap k and chunk c:
  //   uz: rank 16c+n, channels 8q, 8q+2, 8q+4, 8q+6, then 8q+1 .. 8q+7: B operand
  //       of the dz MFMA (the K order of its A operand, read back from the G tile);
  //   uw: ranks 4q..4q+3 (8q..8q+7 with two chunks) of channel 2n+j: B operand of
  //       the tap-weight MFMA, in registers (UREG), else read back from uz's
  //       LDS copy with transposing reads.
  u32x2 uw[UREG && !NODX ? W * 2 : 1];
  u32x4 uzr[UREG ? W : 1];
  u32x4* __restrict__ my_us = us[wave];
  const int us_lane = 16 * q + (n ^ (4 * q));  // slot of channel octet q, rank n (swizzled for the transposing reads)
  {
    const rsrc_t ru = make_rsrc(U, lr_u_bytes(R, a.uld, a.kofs, D, 2));
    const rsrc_t rs = make_rsrc(sw, lr_sw_bytes(RK > R, W, D, 2));
    const int rowb = a.uld * 2, tapb = D * 2;
    // Offsets of tap 0 (a tap adds k * tapb to an out-of-range one too: below 2^31,
    // the host keeps (RK + 16) rows of U under kOobLane).  Lanes past D or off the
    // row are out of range, so every load is issued without a branch.
    const int c0 = d0 + 8 * q < D ? (d0 + 8 * q) * 2 : kOobLane;  // D % 8 == 0
    int zu[RC], zs[RC];
#pragma unroll
    for (int c = 0; c < RC; ++c) {
      const int r = 16 * c + n;
      zu[c] = r < R ? r * rowb : kOobLane;
      zs[c] = RK > R && r == R ? 0 : kOobLane;
    }
    auto load_uz = [&](int k, int c) {
      const u32x4 v = bload128(ru, oob_add(c0, zu[c]) + k * tapb) | bload128(rs, oob_add(c0, zs[c]) + k * tapb);
      return u32x4{__builtin_amdgcn_perm(v[1], v[0], kEven), __builtin_amdgcn_perm(v[3], v[2], kEven),
                   __builtin_amdgcn_perm(v[1], v[0], kOdd), __builtin_amdgcn_perm(v[3], v[2], kOdd)};
    };
    if constexpr (UREG) {
      uint32_t row[NODX ? 1 : W][4];
      if constexpr (!NODX) {
        const int cl = chv ? col * 2 : kOobLane;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
          const int r = 4 * q + kk;
          const int wu = r < R ? oob_add(cl, r * rowb) : kOobLane, ws = RK > R && r == R ? cl : kOobLane;
#pragma unroll
          for (int k = 0; k < W; ++k) row[k][kk] = bload32(ru, wu + k * tapb) | bload32(rs, ws + k * tapb);
        }
      }
#pragma unroll
      for (int k = 0; k < W; ++k) uzr[k] = load_uz(k, 0);
      if constexpr (!NODX) {
#pragma unroll
        for (int k = 0; k < W; ++k)
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const uint32_t hl = j ? kOdd : kEven;
            uw[k * 2 + j][0] = __builtin_amdgcn_perm(row[k][1], row[k][0], hl);
            uw[k * 2 + j][1] = __builtin_amdgcn_perm(row[k][3], row[k][2], hl);
          }
      }
    } else {
      // rolled: straight-line code runs at the rate it is fetched at, once per launch
#pragma unroll 1
      for (int k0 = 0; k0 < W; k0 += 2) {
        u32x4 v[2][RC];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int c = 0; c < RC; ++c) v[h][c] = load_uz(k0 + h < W ? k0 + h : k0, c);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int c = 0; c < RC; ++c) my_us[((k0 + h < W ? k0 + h : k0) * RC + c) * 64 + us_lane] = v[h][c];
      }
    }
  }
  // Transposing read of the tap-weight operand from my_us: lane a + 4i of group q
  // addresses rank base + i (base 4q, or 8q + 4s with two chunks) of the channels
  // 8a + 2e + j, e < 4: half j of octet a's slot.
  const int ul_rank = RC == 2 ? 8 * (q & 1) + (n >> 2) : 4 * q + (n >> 2), ul_oct = n & 3;
  const int ul_base = (RC == 2 ? (q >> 1) * 64 : 0) + 16 * ul_oct;
  const int ul_lane[2] = {(ul_base + (ul_rank ^ (4 * ul_oct))) * 16, (ul_base + ((ul_rank + 4) ^ (4 * ul_oct))) * 16};
  const uint8_t* const my_ul = reinterpret_cast<const uint8_t*>(my_us);

  // G tile: the 4-row group h of rows 8q.. at plane 2q+h, even channels, then odd ones
  uint8_t* const my_g = gtile[wave];
  const int gw_lane = 2 * q * GPL + 8 * n;
  const int gr_lane = 2 * (n & 3) * GPL + (4 * q + (n >> 2)) * 8;  // even channels; the odd ones 128 bytes on

  // Identity (one chunk) or rank-selection (two) matrices as the B operand that transposes z_eff.
  u32x2 ident;
  u32x4 sel[RC == 2 ? 2 : 1];
  {
    const uint32_t one = Mma16<T>::kOne;
    if constexpr (RC == 1) {
      uint32_t e[4];
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) e[kk] = 4 * q + kk == n ? one : 0u;
      ident[0] = e[0] | (e[1] << 16);
      ident[1] = e[2] | (e[3] << 16);
    } else {
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const uint32_t lo = 8 * q + 2 * h == 16 * c + n ? one : 0u;
          const uint32_t hi = 8 * q + 2 * h + 1 == 16 * c + n ? one : 0u;
          sel[c][h] = lo | (hi << 16);
        }
    }
  }

  f32x4 du[W][RC][2];
#pragma unroll
  for (int k = 0; k < W; ++k)
#pragma unroll
    for (int c = 0; c < RC; ++c)
#pragma unroll
      for (int j = 0; j < 2; ++j) du[k][c][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  struct ZA {
    u32x2 c[1];  // one rank chunk: ranks 4q..4q+3
    u32x4 v;     // two: ranks 8q..8q+7
  };
  // the tile's z operands of half h, from the loaded registers
  auto z_op = [&](int tile, int h) {
    ZA o;
    if constexpr (RC == 2)
      o.v = in.z32[h];
    else
      in.zraw[h].finish(o.c, tile * 32 + zrow + 4 * h, zr, zrk, Tn, q);
    return o;
  };
  // tap k's weights of half h for channel 2n+j, accumulator started at w0
  auto tap_w = [&](const ZA& za, const u32x4& uo, float w0) {
    const f32x4 wk = {w0, w0, w0, w0};
    if constexpr (RC == 2)
      return Mma32<T>::run(za.v, uo, wk);
    else
      return Mma16<T>::run(za.c[0], u32x2{uo[0], uo[1]}, wk);
  };
  auto tap_op = [&](int k, int j) {
    if constexpr (UREG) {
      return u32x4{uw[NODX ? 0 : k * 2 + j][0], uw[NODX ? 0 : k * 2 + j][1], 0u, 0u};
    } else {
      const u32x2 lo = lds_read_tr16(my_ul + ul_lane[0] + k * RC * 1024 + j * 8);
      if constexpr (RC == 1) return u32x4{lo[0], lo[1], 0u, 0u};
      const u32x2 hi = lds_read_tr16(my_ul + ul_lane[1] + k * RC * 1024 + j * 8);
      return u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
  };
  // row 4h+i of the lane's dy times tap k's weight: to dx row 4h+i-k, of the lane or of the group above
  auto scatter = [&](const f32x4& wk, const float(&dyf)[8][2], int k, int j, int h, float(&own)[8][2],
                     float(&S)[NO][2]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 4 * h + i, r = row - k;
      if (r >= 0)
        own[r][j] = fmaf(dyf[row][j], wk[i], own[r][j]);
      else
        S[-r - 1][j] = fmaf(dyf[row][j], wk[i], S[-r - 1][j]);
    }
  };

  // S[m]: the lane's sums for row 8q-1-m (the group above).  Groups 0-2 close
  // their rows with the group below's sums; group 3 stores its first rows now
  // and its open rows one tile later, with group 0's sums of the next tile.
  float carry[NO][2];
#pragma unroll
  for (int i = 0; i < NO; ++i) carry[i][0] = carry[i][1] = 0.f;
  auto close_rows = [&](const float(&own)[8][2], const float(&S)[NO][2], int tile,
                        const typename DV::type(&dxo)[ACC ? 8 : 1]) {
    const int src = ((lane + 16) & 63) << 2;  // ds_bpermute byte index of the group below
    float recv[NO][2];
#pragma unroll
    for (int m = 0; m < NO; ++m)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        recv[m][j] = W > 1 ? __int_as_float(__builtin_amdgcn_ds_bpermute(src, __float_as_int(S[m][j]))) : 0.f;
    const bool top = q == 3;
    const int cur_off = tile < tile1 ? dxslane_off + (tile * 32 - rb - kofs) * dxsrowb : kOobTile;
    const int prev_off = tile > tile0 ? dxslane_off + ((tile - 1) * 32 - rb - kofs) * dxsrowb : kOobTile;
    const int open_off = top ? prev_off : cur_off;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const bool open = W > 1 && i >= kFirstOpen;
      float v[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        v[j] = own[i][j];
        if (open) v[j] = (top ? carry[i - kFirstOpen][j] : v[j]) + recv[7 - i][j];
      }
      if constexpr (ACC) {  // a later pass adds to the stored rows
        typename DV::type o = dxo[i];
#pragma unroll
        for (int j = 0; j < 2; ++j) v[j] += DV::get(o, j);
      }
      DVS::template store<NTP>(DVS::make(v), rdxs, (open ? open_off : cur_off) + i * dxsrowb);
    }
    if constexpr (W > 1) {
#pragma unroll
      for (int i = 0; i < NO; ++i) {
#pragma unroll
        for (int j = 0; j < 2; ++j) carry[i][j] = own[kFirstOpen + i][j];
      }
    }
  };

  const int nit = tile1 - tile0;
  auto do_tile = [&](int it) {
    const int tile = tile0 + it;
    float xf[NR][2], dyf[8][2];
    const int above = ((lane + 48) & 63) << 2;  // ds_bpermute byte index of lane - 16
#pragma unroll
    for (int m = 0; m < NR; ++m) {
      uint32_t v;
      if (HX && m < W - 1) {
        const uint32_t own = in.xr[HX ? (m + 9 - W) % NX : 0];  // row 8q+9-W+m
        v = (uint32_t)__builtin_amdgcn_ds_bpermute(above, (int)(q == 3 ? prev[m % NO] : own));
        prev[m % NO] = own;
      } else {
        v = in.xr[m - (NR - NX)];
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) xf[m][j] = Mma16<T>::to_f(LV::elem(v, j));
    }
#pragma unroll
    for (int m = 0; m < 8; ++m)
#pragma unroll
      for (int j = 0; j < 2; ++j) dyf[m][j] = Mma16<T>::to_f(LV::elem(in.dyr[m], j));
    ZA zA[2] = {z_op(tile, 0), z_op(tile, 1)};
    __builtin_amdgcn_sched_barrier(0);
    typename DV::type dxo[ACC ? 8 : 1] = {};
    if constexpr (ACC && DXO == kDxoTile) load_dxo(tile, dxo);
    if constexpr (ACC && DXO == kDxoAhead) {
#pragma unroll
      for (int i = 0; i < 8; ++i) dxo[i] = in.dxo[DXO == kDxoAhead ? i : 0];
    }
    load_tile(tile + 1);
    __builtin_amdgcn_sched_barrier(0);  // the next tile's loads go out before this tile's products

    // z_eff transposed (rank n, rows 8q..8q+7): exact identity / selection products
    u32x4 zT[RC];
#pragma unroll
    for (int c = 0; c < RC; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        f32x4 tz;
        if constexpr (RC == 2)
          tz = Mma32<T>::run(zA[h].v, sel[c], f32x4{0.f, 0.f, 0.f, 0.f});
        else
          tz = Mma16<T>::run(zA[h].c[0], ident, f32x4{0.f, 0.f, 0.f, 0.f});
        zT[c][2 * h] = pack2<T>(tz[0], tz[1]);
        zT[c][2 * h + 1] = pack2<T>(tz[2], tz[3]);
      }
    float own[8][2], S[NO][2];
#pragma unroll
    for (int i = 0; i < 8; ++i) own[i][0] = own[i][1] = 0.f;
#pragma unroll
    for (int i = 0; i < NO; ++i) S[i][0] = S[i][1] = 0.f;
    f32x4 dz[2][RC];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int c = 0; c < RC; ++c) dz[h][c] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
    for (int k = 0; k < W; ++k) {
      if (ACC && DXO == kDxoLastTap && k == W - 1) {
        load_dxo(tile, dxo);
        __builtin_amdgcn_sched_barrier(0);
      }
      // G_k of the lane's rows and channels (fp32 products, rounded once); the
      // wave barriers keep the compiler from moving an LDS write above another
      // lane's read (the hardware keeps a wavefront's LDS order)
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        u32x4 gp;
#pragma unroll
        for (int h = 0; h < 4; ++h)
          gp[h] = pack2<T>(dyf[2 * h][j] * xf[2 * h - k + W - 1][j], dyf[2 * h + 1][j] * xf[2 * h + 1 - k + W - 1][j]);
        *reinterpret_cast<u32x2*>(my_g + gw_lane + 128 * j) = u32x2{gp[0], gp[1]};
        *reinterpret_cast<u32x2*>(my_g + gw_lane + 128 * j + GPL) = u32x2{gp[2], gp[3]};
#pragma unroll
        for (int c = 0; c < RC; ++c) du[k][c][j] = Mma32<T>::run(zT[c], gp, du[k][c][j]);
      }
      __builtin_amdgcn_wave_barrier();
      u32x4 ga[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const u32x2 lo = lds_read_tr16(my_g + gr_lane + h * GPL);
        const u32x2 hi = lds_read_tr16(my_g + gr_lane + h * GPL + 128);
        ga[h] = u32x4{lo[0], lo[1], hi[0], hi[1]};
      }
      if constexpr (!NODX) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const u32x4 uo = tap_op(k, j);
#pragma unroll
          for (int h = 0; h < 2; ++h) scatter(tap_w(zA[h], uo, k == 0 ? res : 0.f), dyf, k, j, h, own, S);
        }
      }
#pragma unroll
      for (int c = 0; c < RC; ++c) {
        const u32x4 uz = UREG ? uzr[UREG ? k : 0] : my_us[UREG ? 0 : (k * RC + c) * 64 + us_lane];
#pragma unroll
        for (int h = 0; h < 2; ++h) dz[h][c] = Mma32<T>::run(ga[h], uz, dz[h][c]);
      }
    }
    if constexpr (!NODX) close_rows(own, S, tile, dxo);

    // ---- dz: row 8q+4h+i, rank 16c+n of the tile at (16 row + n) ^ (q << 4) of chunk c's 512
    const int slot = it % DZB;
    const int buf = (it / DZB) & 1;
#pragma unroll
    for (int c = 0; c < RC; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          dzred[buf][slot][wave][c * 512 + (((8 * q + 4 * h + i) * 16 + n) ^ (q << 4))] = dz[h][c][i];
    if (slot == DZB - 1 || it == nit - 1) {
      __syncthreads();
      // the batch's sums go out at raised wave priority: every wavefront waits
      // at the next batch's barrier for the slowest one here
      __builtin_amdgcn_s_setprio(1);
      static_assert(DZB * RC * 512 == 2 * 512, "one pair of ranks per thread");
      const int e2 = 2 * (int)threadIdx.x;
      const int sl = e2 / (RC * 512), rem = e2 - sl * (RC * 512);
      const int c = rem >> 9, el = rem & 511, rr = el >> 4, r = 16 * c + (el & 15);
      const int pos = c * 512 + (el ^ (((el >> 7) & 3) << 4));
      f32x2 v = *reinterpret_cast<const f32x2*>(&dzred[buf][sl][0][pos]);
#pragma unroll
      for (int w2 = 1; w2 < NW; ++w2) {
        const f32x2 u = *reinterpret_cast<const f32x2*>(&dzred[buf][sl][w2][pos]);
        v[0] += u[0];
        v[1] += u[1];
      }
      // slots past a short last batch and ranks >= R store nothing (rows past T lie outside the resource)
      const int off = (((tile - slot + sl) * 32 + rr - rb) * a.dzld + r) * 4;
      const bool ok = sl <= slot;
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v[0]), rpz, ok && r < R ? off : kOobLane, 0, 0);
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v[1]), rpz, ok && r + 1 < R ? off + 4 : kOobLane, 0, 0);
      __builtin_amdgcn_s_setprio(0);
    }
  };
  for (int it = 0; it < nit; ++it) do_tile(it);
  if constexpr (!NODX && W > 1) {
    // The tile after the run (loaded) closes its last rows: rows 0 .. W-2 only.
    float dyf[8][2], own[8][2], S[NO][2];
#pragma unroll
    for (int m = 0; m < 8; ++m) {
#pragma unroll
      for (int j = 0; j < 2; ++j) dyf[m][j] = Mma16<T>::to_f(LV::elem(in.dyr[m], j));
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) own[i][0] = own[i][1] = 0.f;
#pragma unroll
    for (int i = 0; i < NO; ++i) S[i][0] = S[i][1] = 0.f;
#pragma unroll
    for (int h = 0; h < (W <= 5 ? 1 : 2); ++h) {
      const ZA za = z_op(tile1, h);
#pragma unroll
      for (int k = 1; k < W; ++k)
#pragma unroll
        for (int j = 0; j < 2; ++j) scatter(tap_w(za, tap_op(k, j), 0.f), dyf, k, j, h, own, S);
    }
    typename DV::type dxo[ACC ? 8 : 1] = {};
    load_dxo(tile1, dxo);
    close_rows(own, S, tile1, dxo);
  }

  // ---- dU partial of this run: rows r < RK of U_eff, the wavefront's 32 columns
  // per tap (rows >= RK fall outside the resource; see lowrank_mfma_bwd.hip)
  const int UL = a.uld;
  const rsrc_t rdu = make_rsrc(part_du + (int64_t)du_slot * a.dupr * UL, lr_dupart_bytes(RK, UL, a.kofs, D));
  const int du_lane = chv ? (4 * q * UL + col) * 4 : kOobLane;
#pragma unroll
  for (int k = 0; k < W; ++k)
#pragma unroll
    for (int c = 0; c < RC; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        __builtin_amdgcn_raw_buffer_store_b64(
            u32x2{__float_as_uint(du[k][c][0][i]), __float_as_uint(du[k][c][1][i])}, rdu,
            du_lane + ((16 * c + i) * UL + k * D) * 4, 0, 0);
}

template <typename T, int W, int RC>
hipError_t lr_bwd_t32_one(const LrBwdArgs& a, bool f32, hipStream_t stream) {
  if constexpr (RC == 2) {
    if (a.nodx) {  // dz and dU only (lr_dx_t32 forms dx)
      lr_bwd_t32<T, W, RC, false, 3><<<a.nblk, 512, 0, stream>>>(a);
      return hipGetLastError();
    }
    if (f32) {  // every pass on the fp32 dx accumulator; the last one stores dx itself
      if (a.accdx && a.dxsld > 0)
        lr_bwd_t32<T, W, RC, true, 2><<<a.nblk, 512, 0, stream>>>(a);
      else if (a.accdx)
        lr_bwd_t32<T, W, RC, true, 1><<<a.nblk, 512, 0, stream>>>(a);
      else
        lr_bwd_t32<T, W, RC, false, 1><<<a.nblk, 512, 0, stream>>>(a);
      return hipGetLastError();
    }
  }
  if (f32 || a.nodx) return hipErrorInvalidValue;  // one rank chunk takes at most four passes, with dx
  if (a.accdx)
    lr_bwd_t32<T, W, RC, true, 0><<<a.nblk, 512, 0, stream>>>(a);
  else
    lr_bwd_t32<T, W, RC, false, 0><<<a.nblk, 512, 0, stream>>>(a);
  return hipGetLastError();
}

template <typename T>
hipError_t lr_bwd_t32_launch(const LrBwdArgs& a, int W, int RC, bool f32, hipStream_t stream) {
  if (RC == 2) {
    switch (W) {
      case 1: return lr_bwd_t32_one<T, 1, 2>(a, f32, stream);
      case 2: return lr_bwd_t32_one<T, 2, 2>(a, f32, stream);
      case 3: return lr_bwd_t32_one<T, 3, 2>(a, f32, stream);
      case 4: return lr_bwd_t32_one<T, 4, 2>(a, f32, stream);
      default: return hipErrorInvalidValue;
    }
  }
  if (RC != 1) return hipErrorInvalidValue;
  switch (W) {
    case 1: return lr_bwd_t32_one<T, 1, 1>(a, f32, stream);
    case 2: return lr_bwd_t32_one<T, 2, 1>(a, f32, stream);
    case 3: return lr_bwd_t32_one<T, 3, 1>(a, f32, stream);
    case 4: return lr_bwd_t32_one<T, 4, 1>(a, f32, stream);
    case 5: return lr_bwd_t32_one<T, 5, 1>(a, f32, stream);
    case 6: return lr_bwd_t32_one<T, 6, 1>(a, f32, stream);
    case 7: return lr_bwd_t32_one<T, 7, 1>(a, f32, stream);
    case 8: return lr_bwd_t32_one<T, 8, 1>(a, f32, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace dc
