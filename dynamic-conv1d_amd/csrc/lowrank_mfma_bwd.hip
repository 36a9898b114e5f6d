// Lowrank backward on gfx950 matrix cores (bf16 / fp16): dx, dz, dU, dstatic_w.
#include "lowrank_mfma_bwd.h"

namespace dc {

// ---------------------------------------------------------------- backward
//
// Host side of the backward (launch plans, passes, workspace), and the kernel of
// the one-pass problems of three and four rank chunks (kernel ranks 33-48 at
// W <= 2, 49-64 at W 1) and of those of one and two chunks that stream past the
// last-level cache (bwd_streams).  Other problems of one and two chunks, and every
// problem that runs as passes, take lr_bwd_t32 (lowrank_mfma_bwd32.h).
//
// lr_bwd_mfma: one pass over x and dy produces dx, dz, dU and dstatic_w
// (reference: lowrank.py:87-140 and 159-205, two kernels that both read dy).
// A wavefront owns 16 rows x CPW channels (64, or 32 at two rank chunks); lane
// l = 16q + n owns rows 4q..4q+3 and the NJ = CPW/16 channels NJ*n .. (one 8- or
// 4-byte load per row).  With
// G_k[t, d] = bf16(dy[t, d] * x[t-k, d]) (the reference also rounds this
// product to bf16 before its dot products, lowrank.py:128):
//   * dU[r, kD+d] += sum_t z_eff[t, r] G_k[t, d]: MFMA with K = the 16 rows; the
//     lane's four G values of column NJ*n+j are the B operand.
//   * dz[t, r] += sum_d G_k[t, d] U_eff[r, kD+d]: K = 32 channels; the packed dU
//     operands go through the wavefront's LDS slot and come back by row with
//     transposing reads (ds_read_b64_tr_b16).
//   * Tap weights Kw[t, k, :] = z_eff[t, :] U_eff[:, k]: one 16x16x16 MFMA per
//     rank chunk, or one 16x16x32 over two.  The residual's dy rides on tap 0:
//     its accumulator starts at 1.
//   * dx[t, d] = sum_k dy[t+k, d] Kw[t+k, k, d] (+ dy) in scatter form: dy[s]
//     Kw[s, k] goes to row s-k; the sums for the group above pass up with a
//     ds_bpermute each, and group 3's open rows wait one tile.
// A workgroup covers 256 adjacent channels of one run of rows, or of two (one
// rank chunk: half the dU partials).  dz sums over the 256 channels are added in
// LDS in wave order, dU accumulates in registers over the run (the second run's
// is added to the first's at the end); both go out as fp32 partials that
// reduce_partials sums in a fixed order.
//
// Passes of taps (lr_bwd_t32): a launch holds the operands and accumulators of
// at most pass_taps(W, RC) taps, so wider problems run as consecutive launches
// over taps kofs .. kofs+W'-1: the W'-tap problem on x shifted down by kofs
// rows, whose dx rows land kofs rows earlier and are added to what the earlier
// passes stored (ACC), with U, static_w and the dU partial columns from tap
// kofs and dz partials in slots of their own.
//
// Groups: up to kMaxGroups independent problems of one shape share a launch
// (block index -> group); x and dx may have row strides xld, dxld > D, so the
// q / k / v convolutions read x out of a fused [B, T, 3D] projection and write
// dx into its gradient.

// NJ (4 or 2) 16-bit channels of one row held by a lane: one 8- or 4-byte unit.
template <int NJ> struct LaneVec;
template <> struct LaneVec<4> {
  typedef u32x2 type;
  template <int AUX>
  __device__ static __forceinline__ type load(rsrc_t r, int off) { return bload64<AUX>(r, off); }
  __device__ static __forceinline__ void store(type v, rsrc_t r, int off) { bstore64<true>(v, r, off); }
  __device__ static __forceinline__ uint32_t elem(const type& v, int j) { return elem16x2(v, j); }
  template <typename T>
  __device__ static __forceinline__ type pack(const float* f) {
    return type{pack2<T>(f[0], f[1]), pack2<T>(f[2], f[3])};
  }
};
template <> struct LaneVec<2> {
  typedef uint32_t type;
  template <int AUX>
  __device__ static __forceinline__ type load(rsrc_t r, int off) { return bload32<AUX>(r, off); }
  __device__ static __forceinline__ void store(type v, rsrc_t r, int off) {
    __builtin_amdgcn_raw_buffer_store_b32(v, r, off, 0, kNt);
  }
  __device__ static __forceinline__ uint32_t elem(const type& v, int j) { return j ? (v >> 16) : (v & 0xFFFFu); }
  template <typename T>
  __device__ static __forceinline__ type pack(const float* f) {
    return pack2<T>(f[0], f[1]);
  }
};

// U_eff operands of one wavefront's channels, staged once per run: the
// tap-weight operands in registers, the dz operands in LDS.  For tap k and rank
// chunk c, lane (q, n) holds
//   uw[j] (j < NJ): ranks 16c+4q..16c+4q+3 of channel NJ*n+j, packed (B operand
//                  of the 16x16x16 tap-weight MFMA); not with two chunks (stage_uw32);
//   uz[s] (s < NS): rank 16c+n, channels 32s+8q..32s+8q+7 as they lie in U (B
//                  operand of the 16x16x32 dz MFMA).
template <int W, int RC, int NJ, int NS, bool STAGE_UW>
__device__ __forceinline__ void stage_uops(u32x2 (&uw)[STAGE_UW ? W * RC * NJ : 1], u32x4* __restrict__ uz_lds,
                                           const uint16_t* __restrict__ U, const uint16_t* __restrict__ sw, int R,
                                           int RK, int D, int uld, int d0, int q, int n, int lane) {
  typedef LaneVec<NJ> LV;
  // Buffer loads, all issued before the first use: rows r >= R of U and lanes
  // outside D read 0; the static row (r == R < RK) is read from sw and OR-ed in.
  const rsrc_t ru = make_rsrc(U, lr_u_bytes(R, uld, 0, D, 2));
  const rsrc_t rs = make_rsrc(sw, lr_sw_bytes(RK > R, W, D, 2));
  const int cw = d0 + NJ * n < D ? (d0 + NJ * n) * 2 : kOobLane;  // the lane's tap-weight channels
  typename LV::type rows[W][RC][4];
  u32x4 zr[W][RC][NS];
#pragma unroll
  for (int k = 0; k < W; ++k)
#pragma unroll
    for (int c = 0; c < RC; ++c) {
      const bool has_static = RK > R && R >= 16 * c && R < 16 * c + 16;  // chunk c holds the static row
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        const int r = 16 * c + 4 * q + kk;
        if constexpr (STAGE_UW)
          rows[k][c][kk] = LV::template load<0>(ru, r < R ? cw + (r * uld + k * D) * 2 : kOobLane) |
                           LV::template load<0>(rs, has_static && r == R ? cw + k * D * 2 : kOobLane);
      }
      const int r = 16 * c + n;
#pragma unroll
      for (int s2 = 0; s2 < NS; ++s2) {
        const int dd = d0 + 32 * s2 + 8 * q;  // multiple of 8; D % 8 == 0, so dd < D means dd + 8 <= D
        const int cz = dd < D ? dd * 2 : kOobLane;
        zr[k][c][s2] = bload128(ru, r < R ? cz + (r * uld + k * D) * 2 : kOobLane) |
                       bload128(rs, has_static && r == R ? cz + k * D * 2 : kOobLane);
      }
    }
#pragma unroll
  for (int k = 0; k < W; ++k)
#pragma unroll
    for (int c = 0; c < RC; ++c) {
#pragma unroll
      for (int j = 0; j < (STAGE_UW ? NJ : 0); ++j) {
        const typename LV::type(&rw)[4] = rows[k][c];
        uw[(k * RC + c) * NJ + j][0] = LV::elem(rw[0], j) | (LV::elem(rw[1], j) << 16);
        uw[(k * RC + c) * NJ + j][1] = LV::elem(rw[2], j) | (LV::elem(rw[3], j) << 16);
      }
#pragma unroll
      for (int s2 = 0; s2 < NS; ++s2) uz_lds[((k * RC + c) * NS + s2) * 64 + lane] = zr[k][c][s2];
    }
}

// Tap-weight operands for K = 32 ranks (two rank chunks): lane (q, n) gives
// ranks 8q..8q+7 of channel NJ*n+j, packed (B operand of the 16x16x32 MFMA
// whose A is z_eff row n, ranks 8q..8q+7).  Row R (< RK) is static_w.
template <int W, int NJ>
__device__ __forceinline__ void stage_uw32(u32x4 (&uw)[W * NJ], const uint16_t* __restrict__ U,
                                           const uint16_t* __restrict__ sw, int R, int RK, int D, int uld, int d0,
                                           int q, int n) {
  typedef LaneVec<NJ> LV;
  const rsrc_t ru = make_rsrc(U, lr_u_bytes(R, uld, 0, D, 2));
  const rsrc_t rs = make_rsrc(sw, lr_sw_bytes(RK > R, W, D, 2));
  const int cw = d0 + NJ * n < D ? (d0 + NJ * n) * 2 : kOobLane;
  typename LV::type rows[W][8];
#pragma unroll
  for (int k = 0; k < W; ++k)
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) {
      const int r = 8 * q + kk;
      rows[k][kk] = LV::template load<0>(ru, r < R ? cw + (r * uld + k * D) * 2 : kOobLane) |
                    LV::template load<0>(rs, RK > R && r == R ? cw + k * D * 2 : kOobLane);
    }
#pragma unroll
  for (int k = 0; k < W; ++k)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      u32x4 v;
#pragma unroll
      for (int h = 0; h < 4; ++h) v[h] = LV::elem(rows[k][2 * h], j) | (LV::elem(rows[k][2 * h + 1], j) << 16);
      uw[k * NJ + j] = v;
    }
}

// A operands of the tap-weight MFMA: four ranks per rank chunk (16x16x16) or,
// with two rank chunks, eight ranks (16x16x32).
template <int RC> struct ZOp { u32x2 c[RC]; };
template <> struct ZOp<2> { u32x4 v; };

// CPW channels to a wavefront, NRW runs to a workgroup (bwd_shape).
template <typename T, int W, int RC, int NRW, int CPW>
__global__ __launch_bounds__(64 * (256 / CPW) * NRW)
__attribute__((amdgpu_waves_per_eu(RC <= 2 ? 2 : 1, 8))) void lr_bwd_mfma(LrBwdArgs a) {
  static_assert(W <= 4 && W * RC <= 8, "tap-weight operands in registers");
  static_assert(NRW == 1 || (RC == 1 && CPW == 64), "two runs per workgroup: one rank chunk");
  constexpr int NJ = CPW / 16;     // channels per lane
  constexpr int NS = CPW / 32;     // 32-channel K blocks of the dz MFMA
  constexpr int NCW = 256 / CPW;   // channel-chunk wavefronts per run: 256 channels per workgroup
  constexpr int NW = NCW * NRW;    // wavefronts per workgroup
  constexpr bool K32 = RC == 2;    // tap weights over 32 ranks in one 16x16x32 MFMA (z rows of exactly 32 ranks)
  constexpr int NR = W + 3;        // x rows 4q-W+1 .. 4q+3 per lane
  constexpr int NSC = W > 1 ? W - 1 : 1;  // open rows of a group (none at W 1)
  constexpr int kFirstOpen = 5 - W;       // rows kFirstOpen .. 3 take the group below's sums
  typedef LaneVec<NJ> LV;
  typedef ZOp<RC> ZO;
  typedef ZRaw<T, RC, true> ZR;  // 8-byte z loads: rows of zld % 4 == 0 elements
  constexpr int NUZ = W * RC * NS;  // dz operands per lane
  // G tile in LDS, transposed: channel c's rows 4p..4p+3 (8 bytes) at byte
  // p*GPL + 8c + 8(c/16).  The pad of 8 bytes per 16 channels keeps both access
  // patterns within two-way bank conflicts.
  constexpr int GPL = 8 * CPW + CPW / 2;  // bytes per 4-row plane
  __shared__ u32x4 uz_lds[NW][NUZ * 64];
  __shared__ __attribute__((aligned(16))) uint8_t gtile[NW][4 * GPL];
  // dz sums of the workgroup's chunks, gathered for DZB tiles (double-buffered:
  // one barrier per batch).  Row r, rank n of a tile sits at (16r + n) ^ ((r /
  // 4) << 4): the XOR puts the four row groups a lane quarter writes at once in
  // different banks.
  constexpr int DZB = RC == 1 ? 4 : RC == 2 && W >= 2 ? 2 : 1;
  __shared__ float dzred[2][NRW][NCW][DZB][RC * 256];

  const int lane = threadIdx.x & 63, wave = wave_id();
  const int cw = wave % NCW, rw = wave / NCW;  // chunk and run of this wavefront in the workgroup
  const int q = lane >> 4, n = lane & 15;
  const int lb0 = xcd_remap(blockIdx.x, a.nblk);
  const int g = __builtin_amdgcn_readfirstlane(lb0 / a.nblk1);
  const int lb = lb0 - g * a.nblk1;
  const auto* gp = kernel_args<LrBwdArgs>()->grp + g;
  const uint16_t* __restrict__ x = reinterpret_cast<const uint16_t*>(gp->x);
  const uint16_t* __restrict__ z = reinterpret_cast<const uint16_t*>(gp->z);
  const uint16_t* __restrict__ U = reinterpret_cast<const uint16_t*>(gp->U);
  const uint16_t* __restrict__ sw = reinterpret_cast<const uint16_t*>(gp->sw);
  const uint16_t* __restrict__ dy = reinterpret_cast<const uint16_t*>(gp->dy);
  uint16_t* __restrict__ dx = reinterpret_cast<uint16_t*>(gp->dx);
  float* __restrict__ part_dz = gp->part_dz;
  float* __restrict__ part_du = gp->part_du;
  const int cg = lb % a.ncg, du_slot = lb / a.ncg, sp = a.sp0 + du_slot * NRW;
  const int D = a.D, Tn = a.Tn;
  const int d0 = (cg * NCW + cw) * CPW;
  const int col = d0 + NJ * n;
  const bool chv = col < D;  // the lane's NJ channels inside D (D % 8 == 0: all or none)
  const int ntile = (Tn + 15) >> 4;
  // Run s: tiles [tile0, tile1) of sequence b, whose buffer resources start at
  // row rb.  A workgroup's last run can lie past nseg (odd nseg): it has no tiles.
  struct Run {
    int tile0, tile1, rb;
    int64_t row0;
  };
  auto run_of = [&](int s) {
    Run r{0, 0, 0, 0};
    if (s < a.nseg) {
      const int b = s / a.nspb;
      r.tile0 = (s - b * a.nspb) * a.seg;
      r.tile1 = min(r.tile0 + a.seg, ntile);
      r.rb = run_base_row(r.tile0);
      r.row0 = (int64_t)b * Tn;
    }
    return r;
  };
  Run runs[NRW];
  int nit = 0;  // iterations of every wavefront: the longest run of the workgroup
#pragma unroll
  for (int i = 0; i < NRW; ++i) {
    runs[i] = run_of(sp + i);
    nit = max(nit, runs[i].tile1 - runs[i].tile0);
  }
  const Run me = rw == 0 ? runs[0] : runs[NRW - 1];
  const int tile0 = me.tile0, tile1 = me.tile1, rb = me.rb;
  const int64_t row0 = me.row0, rrow = row0 + rb;
  const int R = a.R, RK = a.RK;
  u32x4* __restrict__ my_uz = uz_lds[wave];
  // G^T write position of the lane's channel NJ*n (plus 8j), and the transposed-read
  // position that returns row n, channels 8q..8q+3 (plus 32 for 8q+4..8q+7, plus
  // 8*32+16 per 32-channel block)
  uint8_t* const my_g = gtile[wave];
  const int gw_lane = q * GPL + NJ * 8 * n + (n / (16 / NJ)) * 8;
  const int gr_lane = (n & 3) * GPL + (8 * q + (n >> 2)) * 8 + (q >> 1) * 8;
  const float res = a.residual ? 1.f : 0.f;  // tap 0's weight + 1: the residual term dy
  // dy is [B, T, D] (yhd == D) or head-major [B, D/yhd, T, yhd] (yhd % 64 == 0: a
  // wavefront's channels lie in one head, whose [T, yhd] block rdy covers)
  const int yhd = a.yhd, head = d0 / yhd;
  const int rowb = yhd * 2, xrowb = a.xld * 2, dxrowb = a.dxld * 2;
  const rsrc_t rx = run_rsrc(x + rrow * a.xld, Tn - rb, xrowb);
  const rsrc_t rdy = run_rsrc(dy + row0 * D + ((int64_t)head * Tn + rb) * yhd, Tn - rb, rowb);
  const rsrc_t rdx = run_rsrc(dx + rrow * a.dxld, Tn - rb, dxrowb);
  const int zld = a.zld, zr = a.zr, zrk = a.zrk;
  const rsrc_t rz = run_rsrc(z + rrow * zld, Tn - rb, zld * 2);
  // byte offsets of the lane's row-4q channels in dy, x and dx
  const int lane_off = chv ? (4 * q * yhd + col - head * yhd) * 2 : kOobLane;
  const int xlane_off = chv ? (4 * q * a.xld + col) * 2 : kOobLane;
  const int dxlane_off = chv ? (4 * q * a.dxld + col) * 2 : kOobLane;

  u32x2 uw[K32 ? 1 : W * RC * NJ];  // staged below, after the first tile's loads are issued
  u32x4 uw32[K32 ? W * NJ : 1];
  // Identity (or, for 32 ranks, rank-selection) matrices as the B operand that transposes z_eff.
  u32x2 ident;
  u32x4 sel[K32 ? 2 : 1];
  {
    const uint32_t one = Mma16<T>::kOne;
    uint32_t e[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) e[kk] = (4 * q + kk == n) ? one : 0u;
    ident[0] = e[0] | (e[1] << 16);
    ident[1] = e[2] | (e[3] << 16);
    if constexpr (K32) {
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const uint32_t lo = (8 * q + 2 * h == 16 * c + n) ? one : 0u;
          const uint32_t hi = (8 * q + 2 * h + 1 == 16 * c + n) ? one : 0u;
          sel[c][h] = lo | (hi << 16);
        }
    }
  }
  f32x4 du[W][RC][NJ];
#pragma unroll
  for (int k = 0; k < W; ++k)
#pragma unroll
    for (int c = 0; c < RC; ++c)
#pragma unroll
      for (int j = 0; j < NJ; ++j) du[k][c][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Tile inputs (buffer loads: out-of-range rows / channels read as 0).  Two
  // buffers alternate: while one tile is computed the next one's loads are in
  // flight.  A tile past the run reads the out-of-range offset kOobTile; dy and z
  // of the tile after the run are read too (its first rows close the last dx rows).
  // dy rows are read once: nontemporal (B4 T4096 D2048 R16 60.0 -> 58.8 us), but
  // not in the short tiles of W 1 and the long ones of three and four chunks, which
  // wait for them (R63 + static W 1 71 -> 62 us without).
  struct TileIn {
    typename LV::type xr[NR], dyr[4];
    ZR zr;
    u32x4 z32;
  };
  auto load_tile = [&](int tile, TileIn& in) {
    const bool live = tile < tile1, ylive = W > 1 ? tile <= tile1 : live;
    const int xtoff = live ? (tile * 16 - rb) * xrowb : kOobTile;
    const int toff = ylive ? (tile * 16 - rb) * rowb : kOobTile;
#pragma unroll
    for (int m = 0; m < NR; ++m) in.xr[m] = LV::template load<0>(rx, xlane_off + xtoff + (m - (W - 1)) * xrowb);
#pragma unroll
    for (int m = 0; m < 4; ++m) in.dyr[m] = LV::template load<W == 1 || RC >= 3 ? 0 : kNt>(rdy, lane_off + toff + m * rowb);
    if constexpr (K32)
      in.z32 = bload128(rz, ylive ? ((tile * 16 + n - rb) * zld + 8 * q) * 2 : kOobTile);
    else
      in.zr.load(rz, ylive ? (tile * 16 + n - rb) * zld * 2 : kOobTile, zr, q);
  };
  auto z_op = [&](const TileIn& in, int tile) {
    ZO o;
    if constexpr (K32)
      o.v = in.z32;
    else
      in.zr.finish(o.c, tile * 16 + n, zr, zrk, Tn, q);
    return o;
  };
  // Tap k's weights of the lane's rows for channel NJ*n+j, accumulator started at w0.
  auto tap_w = [&](const ZO& za, int k, int j, float w0) {
    f32x4 wk = {w0, w0, w0, w0};
    if constexpr (K32) {
      wk = Mma32<T>::run(za.v, uw32[k * NJ + j], wk);
    } else {
#pragma unroll
      for (int c = 0; c < RC; ++c) wk = Mma16<T>::run(za.c[c], uw[(k * RC + c) * NJ + j], wk);
    }
    return wk;
  };
  auto scatter = [&](const f32x4& wk, const float(&dyf)[4][NJ], int k, int j, float(&own)[4][NJ],
                     float(&S)[NSC][NJ]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = i - k;  // dx row of this contribution, relative to 4q
      if (r >= 0)
        own[r][j] = fmaf(dyf[i][j], wk[i], own[r][j]);
      else
        S[-r - 1][j] = fmaf(dyf[i][j], wk[i], S[-r - 1][j]);  // row 4q-1-m of the group above
    }
  };
  float carry[NSC][NJ];  // group 3's open rows of the tile before
#pragma unroll
  for (int i = 0; i < NSC; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) carry[i][j] = 0.f;
  auto close_rows = [&](const float(&own)[4][NJ], const float(&S)[NSC][NJ], int tile) {
    const int src = ((lane + 16) & 63) << 2;  // ds_bpermute byte index of the group below
    const bool top = q == 3;
    float recv[NSC][NJ];
#pragma unroll
    for (int m = 0; m < NSC; ++m)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        recv[m][j] = W > 1 ? __int_as_float(__builtin_amdgcn_ds_bpermute(src, __float_as_int(S[m][j]))) : 0.f;
    const int cur_off = tile < tile1 ? dxlane_off + (tile * 16 - rb) * dxrowb : kOobTile;
    const int prev_off = tile > tile0 && tile <= tile1 ? dxlane_off + ((tile - 1) * 16 - rb) * dxrowb : kOobTile;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool open = W > 1 && i >= kFirstOpen;  // takes the group below's sums
      float v[NJ];
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        v[j] = own[i][j];
        if (open) v[j] = (top ? carry[i - kFirstOpen][j] : v[j]) + recv[3 - i][j];
      }
      LV::store(LV::template pack<T>(v), rdx, (top && open ? prev_off : cur_off) + i * dxrowb);
    }
    if constexpr (W > 1) {
#pragma unroll
      for (int i = 0; i < NSC; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) carry[i][j] = own[kFirstOpen + i][j];
    }
  };
  auto compute_tile = [&](int it, const TileIn& in) {
    const int tile = tile0 + it;
    const ZO zA = z_op(in, tile);
    u32x2 zT[RC];  // z_eff transposed (rank n, rows 4q..4q+3) through an exact identity / selection product
#pragma unroll
    for (int c = 0; c < RC; ++c) {
      f32x4 tz;
      if constexpr (K32)
        tz = Mma32<T>::run(zA.v, sel[c], f32x4{0.f, 0.f, 0.f, 0.f});
      else
        tz = Mma16<T>::run(zA.c[c], ident, f32x4{0.f, 0.f, 0.f, 0.f});
      zT[c] = u32x2{pack2<T>(tz[0], tz[1]), pack2<T>(tz[2], tz[3])};
    }
    float dyf[4][NJ], own[4][NJ], S[NSC][NJ];
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        dyf[m][j] = Mma16<T>::to_f(LV::elem(in.dyr[m], j));
        own[m][j] = 0.f;
      }
#pragma unroll
    for (int m = 0; m < NSC; ++m)
#pragma unroll
      for (int j = 0; j < NJ; ++j) S[m][j] = 0.f;
    f32x4 dz[RC];
#pragma unroll
    for (int c = 0; c < RC; ++c) dz[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < W; ++k) {
      // the wave barriers keep the compiler from moving an LDS write above
      // another lane's read (the hardware keeps a wavefront's LDS order)
      __builtin_amdgcn_wave_barrier();
      float gf[4][NJ];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) gf[i][j] = dyf[i][j] * Mma16<T>::to_f(LV::elem(in.xr[i - k + W - 1], j));
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        scatter(tap_w(zA, k, j, k == 0 ? res : 0.f), dyf, k, j, own, S);
        const u32x2 gk = {pack2<T>(gf[0][j], gf[1][j]), pack2<T>(gf[2][j], gf[3][j])};
        *reinterpret_cast<u32x2*>(my_g + gw_lane + 8 * j) = gk;
#pragma unroll
        for (int c = 0; c < RC; ++c) du[k][c][j] = Mma16<T>::run(zT[c], gk, du[k][c][j]);
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int s2 = 0; s2 < NS; ++s2) {
        const u32x2 lo = lds_read_tr16(my_g + gr_lane + s2 * (8 * 32 + 16));
        const u32x2 hi = lds_read_tr16(my_g + gr_lane + s2 * (8 * 32 + 16) + 32);
        const u32x4 ga = {lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
        for (int c = 0; c < RC; ++c) dz[c] = Mma32<T>::run(ga, my_uz[((k * RC + c) * NS + s2) * 64 + lane], dz[c]);
      }
    }
    close_rows(own, S, tile);
    const int slot = it % DZB;
    const int buf = (it / DZB) & 1;
#pragma unroll
    for (int c = 0; c < RC; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) dzred[buf][rw][cw][slot][c * 256 + (((4 * q + i) * 16 + n) ^ (q << 4))] = dz[c][i];
    if (slot == DZB - 1 || it == nit - 1) {
      __syncthreads();
      // the batch's sums go out at raised wave priority: every wavefront waits
      // at the next batch's barrier for the slowest one here
      __builtin_amdgcn_s_setprio(1);
      constexpr int PER_RUN = RC * 256;
      constexpr int NTH = 64 * NW;
      static_assert(DZB * PER_RUN % NTH == 0, "whole passes over a full batch");
#pragma unroll
      for (int ri = 0; ri < NRW; ++ri) {
        const Run& ru = ri == 0 ? runs[0] : runs[NRW - 1];
        // rows of run ri from its base row; t >= T falls outside the resource
        const rsrc_t rout = run_rsrc(part_dz + ((int64_t)cg * a.BT + ru.row0 + ru.rb) * a.dzld, Tn - ru.rb, a.dzld * 4);
        const int tb = ru.tile0 + it - slot;  // run ri's tile of slot 0
#pragma unroll
        for (int m = 0; m < DZB * PER_RUN / NTH; ++m) {
          const int e2 = (int)threadIdx.x + m * NTH;
          const int sl = e2 / PER_RUN, rem = e2 - sl * PER_RUN;
          const int c = rem >> 8, rr = (rem >> 4) & 15, nn = rem & 15;
          const int r = 16 * c + nn;
          const int ti = tb + sl;  // the slot's tile of run ri
          const int pos = rem ^ (((rem >> 6) & 3) << 4);  // as written
          float v = dzred[buf][ri][0][sl][pos];
#pragma unroll
          for (int w2 = 1; w2 < NCW; ++w2) v += dzred[buf][ri][w2][sl][pos];
          // slots past this batch, tiles past the run and ranks >= R store nothing
          const bool ok = sl <= slot && ti < ru.tile1 && r < R;
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rout,
                                                ok ? ((ti * 16 + rr - ru.rb) * a.dzld + r) * 4 : kOobLane, 0, 0);
        }
      }
      __builtin_amdgcn_s_setprio(0);
    }
  };

  // Every wavefront of the workgroup runs nit iterations (the barriers of the
  // dz batches are shared); tiles past its own run load and store nothing.
  TileIn ta, tb;
  load_tile(tile0, ta);
  __builtin_amdgcn_sched_barrier(0);  // the first tile's loads go out before the U staging waits
  stage_uops<W, RC, NJ, NS, !K32>(uw, my_uz, U, sw, R, RK, D, a.uld, d0, q, n, lane);
  if constexpr (K32) stage_uw32<W, NJ>(uw32, U, sw, R, RK, D, a.uld, d0, q, n);
  for (int it = 0; it < nit; it += 2) {
    load_tile(tile0 + it + 1, tb);
    __builtin_amdgcn_sched_barrier(0);  // issue the next tile's loads before this tile's waits
    compute_tile(it, ta);
    load_tile(tile0 + it + 2, ta);
    __builtin_amdgcn_sched_barrier(0);
    if (it + 1 < nit) compute_tile(it + 1, tb);
  }
  if constexpr (W > 1) {
    // The tile after the longest run (loaded into the buffer that is next in
    // turn) closes that run's last rows; in a shorter run it lies past tile1
    // and stores nothing.
    auto flush = [&](const TileIn& in) {
      const int tile = tile0 + nit;
      const ZO zA = z_op(in, tile);
      float dyf[4][NJ], own[4][NJ], S[NSC][NJ];
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          dyf[m][j] = Mma16<T>::to_f(LV::elem(in.dyr[m], j));
          own[m][j] = 0.f;
        }
#pragma unroll
      for (int m = 0; m < NSC; ++m)
#pragma unroll
        for (int j = 0; j < NJ; ++j) S[m][j] = 0.f;
#pragma unroll
      for (int k = 1; k < W; ++k)
#pragma unroll
        for (int j = 0; j < NJ; ++j) scatter(tap_w(zA, k, j, 0.f), dyf, k, j, own, S);
      close_rows(own, S, tile);
    };
    if (nit & 1)
      flush(tb);
    else
      flush(ta);
  }

  if constexpr (NRW == 2) {
    // The second run's wavefronts hand their dU sums to the first run's
    // wavefronts of the same chunk through LDS (the dz buffers, now free).
    float* xch = &dzred[0][0][0][0][0];
    constexpr int NDU = W * RC * NJ * 4;  // dU floats per lane
    static_assert(NCW * NDU * 64 <= 2 * NRW * NCW * DZB * RC * 256, "dU exchange fits the dz buffers");
    __syncthreads();
    if (rw == 1) {
#pragma unroll
      for (int k = 0; k < W; ++k)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) xch[((cw * W + k) * 16 + j * 4 + i) * 64 + lane] = du[k][0][j][i];
    }
    __syncthreads();
    if (rw == 1) return;
#pragma unroll
    for (int k = 0; k < W; ++k)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) du[k][0][j][i] += xch[((cw * W + k) * 16 + j * 4 + i) * 64 + lane];
  }

  // ---- dU partial of this workgroup row: rows r < RK of U_eff, the wavefront's
  // CPW columns per tap.  The resource spans the RK x W*D partial, so rows r >=
  // RK fall outside it (the host keeps (RK + 16) * W * D * 4 bytes below
  // kOobLane, so no offset wraps).
  const rsrc_t rdu = make_rsrc(part_du + (int64_t)du_slot * a.dupr * a.uld, lr_dupart_bytes(RK, a.uld, 0, D));
  const int du_lane = chv ? (4 * q * a.uld + col) * 4 : kOobLane;
#pragma unroll
  for (int k = 0; k < W; ++k)
#pragma unroll
    for (int c = 0; c < RC; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int off = du_lane + ((16 * c + i) * a.uld + k * D) * 4;
        if constexpr (NJ == 4)
          bstore128<false>(u32x4{__float_as_uint(du[k][c][0][i]), __float_as_uint(du[k][c][1][i]),
                                 __float_as_uint(du[k][c][2][i]), __float_as_uint(du[k][c][3][i])},
                           rdu, off);
        else
          __builtin_amdgcn_raw_buffer_store_b64(u32x2{__float_as_uint(du[k][c][0][i]), __float_as_uint(du[k][c][1][i])},
                                                rdu, off, 0, 0);
      }
}

// ------------------------------------------------------------------- host
namespace {

// Taps per backward pass: what one pass's tap-weight and dz operands (registers
// and LDS) and dU accumulators hold for RC rank chunks.  Wider problems run as
// consecutive passes of taps kofs .. kofs+taps-1, reading x and dy once per
// pass.  (Three and four chunks take their one pass at W 2 and W 1 only:
// lr_bwd_rank_split.)
constexpr int pass_taps(int W, int RC) {
  return RC == 1 ? (W <= 8 ? W : 8) : RC == 2 ? (W < 4 ? W : 4) : RC == 3 ? (W < 2 ? W : 2) : 1;
}
constexpr int npasses(int W, int RC) { return (W + pass_taps(W, RC) - 1) / pass_taps(W, RC); }

// Rank chunks of a problem's launch shape: its own (one to four), or passes of
// kBwdRankPass ranks on the two-chunk kernels where lr_bwd_rank_split holds.
constexpr int kBwdRankPass = 32;
inline bool bwd_rank_split(const LrProblem& p) { return lr_bwd_rank_split(p.R + (p.static_w ? 1 : 0), p.W); }
inline int bwd_rc(const LrProblem& p) {
  const int rk = (int)(p.R + (p.static_w ? 1 : 0));
  return bwd_rank_split(p) ? 2 : (rk + 15) / 16;
}
inline int bwd_rank_passes(const LrProblem& p) {
  const int rk = (int)(p.R + (p.static_w ? 1 : 0));
  return bwd_rank_split(p) ? (rk + kBwdRankPass - 1) / kBwdRankPass : 1;
}

// More than four passes (ranks x taps) add dx into an fp32 accumulator in the
// workspace, whose last pass stores dx itself, rounded once (DXM 2; a launch
// that rounded the whole accumulator after the passes took 55 us more at B4
// T4096 D2048 R127 + static W4: 456 -> 400 us) (above W 16 at two rank chunks,
// above W 8 at three, above W 4 at four; one rank chunk takes at most four
// passes of 8 taps up to W 32), and so do more than two where the passes split
// the ranks: each rank pass adds a partial tap weight whose terms can cancel
// (dx near zero from partials of several units), and three or four roundings
// of such partials left single entries past the elementwise bar in a random
// sweep (|dx - dx_oracle| 0.0217 at R104 + static W1, 4 passes, and 0.0219 at
// R73 + static W2, 3 passes, against 0.02 + 2%).
constexpr int kBwdMaxBf16DxPasses = 4;
constexpr int kBwdMaxBf16DxRankPasses = 2;
// Passes of ranks whose dx fits one launch
// (lr_dx_split_shape: W <= 8 up to kernel rank 64, W 5 / 4 up to 96 / 128) or
// two (W 9-16 up to 64, over the fp32 accumulator), with dy in either layout: the
// passes form dz and dU only (DXM 3) and lr_dx_t32 forms dx over all ranks and
// taps in one launch, rounded once (no fp32 accumulator).  Passes of taps alone
// (two rank chunks above W 4) keep dx: split off it measured 160 -> 166 us at B4
// T4096 D2048 R31 + static W 8.
inline bool bwd_dx_split(const LrProblem& p) {
  const int64_t hd = p.yhd();
  // head-major dy: where a 128-channel chunk lies in one head, or its heads fit one resource
  const bool dy_ok = hd == p.D || hd % 128 == 0 || (127 / hd + 2) * (p.T + 64) * hd * 2 < kMaxSeqBytes;
  return bwd_rank_split(p) && lr_dx_split_shape(p.R + (p.static_w ? 1 : 0), p.W) && dy_ok;
}
// The workspace keeps room for the accumulator whether or not dx is split off:
// the size queries do not see dy's layout, on which the split depends.
inline bool bwd_f32dx_room(const LrProblem& p) {
  const int np = bwd_rank_passes(p) * npasses((int)p.W, bwd_rc(p));
  return np > kBwdMaxBf16DxPasses || (bwd_rank_passes(p) > 1 && np > kBwdMaxBf16DxRankPasses);
}
inline bool bwd_f32dx(const LrProblem& p) { return !bwd_dx_split(p) && bwd_f32dx_room(p); }

// One-pass problems of one rank chunk (W <= 4), and of two at W 1 and 4, whose x,
// dy and dx together are more than the last-level cache (256 MB) keeps, with
// rows of whole 128-byte lines: lr_bwd_mfma's 16-row tiles (at one chunk its loads
// and stores are whole lines; for lr_bwd_t32 neither cache policies nor a second
// tile in flight nor other run lengths closed the gap).  bf16, t32 -> 16-row tiles, inputs
// partly left in the cache (and out of it): B4 T8192 D2048 R16 W 1 93 -> 74 us (95 -> 83),
// W 2 96 -> 75 (97 -> 82), W 4 101 -> 91 (102 -> 97), R31 + static W 1 98 -> 88 (99 -> 92),
// W 4 127 -> 121 (119 -> 117); B16 T4096 D2048 R16 W 2 184 -> 151; B2 T8192 D4096 R31 +
// static W 4 125 -> 121 (116 -> 115).  Below, B4 T4096 D2048 (201 MB): R16 W 2 40 -> 44
// (51 -> 46), W 4 46 -> 54 (57 -> 58), and B3 T5000 D2560 R16 W 2 46 -> 80 (64 -> 87); rows of 6000 bytes (D 3000) R16 W 4 282 -> 319; two chunks at W 2 78 -> 82
// (B6 T4096 D2048), W 3 equal.  The sizes are one group's, so that a grouped
// call's results are those of its groups' single calls.
inline bool bwd_streams(const LrProblem& p) {
  const int64_t rk = p.R + (p.static_w ? 1 : 0), bytes = 3 * p.B * p.T * p.D * 2;
  if (rk > 32 || p.W > 4 || p.D % 64 != 0) return false;
  if (rk <= 16 || p.W == 1) return bytes > 240000000;
  return p.W == 4 && bytes > 280000000;
}

// A launch's kernel and workgroups: lr_bwd_t32 (32 channels to a wavefront, rows
// 32 to a tile), or lr_bwd_mfma (16 rows): two runs to a workgroup and 64
// channels at one rank chunk, 32 channels at two, 64 at three and four.
struct BwdShape {
  bool t32;
  int rows, cpw, nrw;
};
inline BwdShape bwd_shape(const LrProblem& p) {
  const int rc = bwd_rc(p);
  if (rc <= 2 && !bwd_streams(p)) return {true, kT32Rows, kT32Chan, 1};
  return {false, 16, rc == 2 ? 32 : 64, rc == 1 ? 2 : 1};
}

}  // namespace

// The passes of a backward launch sequence: kernel ranks rofs .. rofs+RK-1 (R
// of them dynamic) and taps kofs .. kofs+W-1; slot: the pass's dz partial slot
// (its pass of taps: the passes of ranks write disjoint columns of the same
// slots).  Every pass takes the same launch shape (bwd_rc), so the dU partial
// rows of all passes line up.
int bwd_plan(const LrProblem& p, BwdPass* out) {
  const int RK = (int)(p.R + (p.static_w ? 1 : 0)), W = (int)p.W, rc = bwd_rc(p);
  const int nrp = bwd_rank_passes(p), step = nrp > 1 ? kBwdRankPass : RK;
  const int ntp = npasses(W, rc);
  if (nrp * ntp > kBwdMaxPlan) return -1;
  int n = 0;
  for (int i = 0; i < nrp; ++i) {
    const int rofs = i * step, rk = RK - rofs < step ? RK - rofs : step;
    const int rd = (int)p.R - rofs < 0 ? 0 : ((int)p.R - rofs < rk ? (int)p.R - rofs : rk);
    // taps split as evenly as the pass count allows, the longer passes first
    // (each at most wp): a pass costs about one sweep of x, dy and dx plus its
    // taps' products, so W 9 as 5 + 4 beats 8 + 1
    for (int t = 0, kofs = 0; t < ntp; ++t) {
      BwdPass& b = out[n++];
      b.rofs = rofs;
      b.R = rd;
      b.RK = rk;
      b.kofs = kofs;
      b.W = W / ntp + (t < W % ntp ? 1 : 0);
      b.slot = t;
      kofs += b.W;
    }
  }
  return n;
}

// Longest backward run (16-row tiles) whose resources fit (see run_rsrc): rows of
// x, dx, dy (one head's block of head-major dy), the z rows the kernel reads (z
// itself or the padded copy) and the fp32 dz partials.  An even number where the
// kernel's tiles are 32 rows.
int64_t lr_bwd_max_run_tiles(const LrProblem& p) {
  int64_t rowb = p.xld() * 2;
  // past four passes of taps the passes' dx rows are the fp32 accumulator (D floats each)
  const int64_t dxb = bwd_f32dx_room(p) ? p.D * 4 : p.dxld() * 2;
  // (the last pass over the accumulator also stores dx rows of dxld elements)
  const int64_t others[5] = {dxb, p.dxld() * 2, p.yhd() * 2, lr_bwd_zrow(p.R, p.static_w != nullptr, p.W) * 2,
                             p.R * 4};
  for (int64_t v : others) rowb = rowb > v ? rowb : v;
  const int64_t tiles = run_tiles_cap(rowb);
  return bwd_rc(p) <= 2 ? tiles / 2 * 2 : tiles;
}

namespace {

// Tiles per run: a CU holds one of its workgroups, so a launch
// takes ceil(workgroups / 256) rounds of a run's length each, and a few
// workgroups past a round cost as much as a full one (B1 T8192 D768 R15 + static
// W 8: runs of 3 tiles are 258 workgroups and took 48 us, runs of 4 31 us; B3
// T4788 D3712 R32: 270 workgroups 163 us, 225 116 us).  Of the run
// lengths that fill one to eight rounds, the one with the least time by a
// model: per round a launch's start and end (6 us) and the run's tiles, and
// every dU partial (one to nrw runs) written and read once.  The plan is one group's: a
// grouped launch has G times the workgroups, but its results are to be those of its
// groups' single calls, and so are its workspace shares.  dflt: no such length
// (more sequences than eight rounds hold).
int64_t bwd_run_tiles(const LrProblem& p, int rows, int nrw, int64_t ntile, int64_t cols, int64_t dflt) {
  constexpr int64_t kCus = 256;
  const double tile_us = 0.6 * (p.W < 2 ? 2 : p.W > 8 ? 8 : p.W) * (bwd_rc(p) == 2 ? 1.25 : 1.0) * rows / kT32Rows;
  const double part_us = (double)(p.R + (p.static_w ? 1 : 0)) * p.W * p.D * 8 / 5e6;
  int64_t best = dflt;
  double best_us = -1;
  for (int64_t rounds = 1; rounds <= 8; ++rounds) {
    const int64_t per_seq = rounds * kCus * nrw / (p.B * cols);  // runs a sequence may take
    if (per_seq < 1) continue;
    const int64_t seg = (ntile + per_seq - 1) / per_seq, runs = p.B * ((ntile + seg - 1) / seg);
    const double us = rounds * (6.0 + seg * tile_us) + (runs + nrw - 1) / nrw * part_us;
    if (best_us < 0 || us < best_us) {
      best = seg;
      best_us = us;
    }
  }
  return best;
}

// split: the passes of ranks form dz and dU in one launch (bwd_dx_split); each
// run is then nrp workgroup rows, so runs are nrp times as long for the same
// number of workgroups (and the dU partials nrp times fewer).
LrBwdArgs make_bwd_args(const LrProblem& p, int target_waves, bool split) {
  LrBwdArgs a;
  const BwdShape sh = bwd_shape(p);
  const int rows = sh.rows, ncw = 256 / sh.cpw;
  a.Tn = (int)p.T;
  a.D = (int)p.D;
  a.R = (int)p.R;
  a.RK = (int)p.R + (p.static_w ? 1 : 0);
  a.residual = p.residual;
  a.nch = (int)((p.D + sh.cpw - 1) / sh.cpw);
  a.ncg = (a.nch + ncw - 1) / ncw;
  const int64_t ntile = (p.T + rows - 1) / rows;
  a.nrp = split ? bwd_rank_passes(p) : 1;
  const int64_t cap = lr_bwd_max_run_tiles(p) * 16 / rows;  // >= 1 (lr_mfma_ok)
  int64_t seg = (p.B * ntile * a.ncg * ncw * a.nrp + target_waves - 1) / target_waves;
  if (bwd_rc(p) <= 2) seg = bwd_run_tiles(p, rows, sh.nrw, ntile, (int64_t)a.ncg * a.nrp, seg);
  if (seg < 1) seg = 1;
  if (seg > ntile) seg = ntile;
  if (seg > cap) seg = cap;
  a.seg = (int)seg;
  a.nspb = (int)((ntile + seg - 1) / seg);
  a.nseg = (int)(p.B * a.nspb);
  a.npair = (a.nseg + sh.nrw - 1) / sh.nrw;
  a.sp0 = 0;
  a.nblk = a.npair * a.ncg * a.nrp;
  a.BT = p.B * p.T;
  a.zld = a.zr = (int)p.R;
  a.zrk = a.RK;
  a.uld = (int)(p.W * p.D);
  a.kofs = 0;
  a.accdx = 0;
  a.dxsld = 0;
  a.nodx = 0;
  a.dzld = a.R;
  a.dupr = a.RK;
  return a;
}

// Ranks of the padded z_eff copy: RK rounded up to a multiple of 4, or 32 for
// two rank chunks (their 16x16x32 operands read ranks 8q..8q+7 of every row).
inline int64_t zpad_ranks(const LrProblem& p) { return lr_bwd_zrow(p.R, p.static_w != nullptr, p.W); }

// z_eff[t, r] = z[t, r] (r < R), 1 (r == R, static_w given), 0 up to RP: the
// backward's z operand when z cannot be read 8 bytes at a time.
struct ZpadArgs {
  const uint16_t* z[kMaxGroups];
  uint16_t* zp[kMaxGroups];
  int64_t n;  // BT * RP / 4: 4-rank pieces per group
  int R, RP, stat, one;
};
// One thread per 4 ranks of a padded row (RP % 4 == 0): four 2-byte reads of
// z (its rows need not be 4-byte aligned), one 8-byte store.  A grid-stride
// loop: the grid is capped (launch_zpad).
__global__ __launch_bounds__(256) void lr_zpad(ZpadArgs a) {
  const int g = blockIdx.y;
  const uint16_t* __restrict__ z = g == 0 ? a.z[0] : g == 1 ? a.z[1] : g == 2 ? a.z[2] : a.z[3];
  uint16_t* __restrict__ zp = g == 0 ? a.zp[0] : g == 1 ? a.zp[1] : g == 2 ? a.zp[2] : a.zp[3];
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < a.n; i += (int64_t)gridDim.x * 256) {
    const int64_t e = 4 * i;  // first element of the piece
    const int64_t t = e / a.RP;
    const int r0 = (int)(e - t * a.RP);
    uint32_t v[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const int r = r0 + kk;
      v[kk] = r < a.R ? z[t * a.R + r] : (r == a.R && a.stat ? (uint32_t)a.one : 0u);
    }
    *reinterpret_cast<u32x2*>(zp + e) = u32x2{v[0] | (v[1] << 16), v[2] | (v[3] << 16)};
  }
}

// lr_zpad over G problems: z_eff of group g into dst[g].
template <typename T>
hipError_t launch_zpad(const LrProblem* p, int G, void* const* dst) {
  if (auditing()) return hipSuccess;  // plain pointers
  ZpadArgs za;
  const int64_t RP = zpad_ranks(p[0]);
  za.n = p[0].B * p[0].T * RP / 4;
  za.R = (int)p[0].R;
  za.RP = (int)RP;
  za.stat = p[0].static_w != nullptr;
  za.one = Mma16<T>::kOne;
  for (int g = 0; g < kMaxGroups; ++g) {
    za.z[g] = (const uint16_t*)p[g < G ? g : 0].z;
    za.zp[g] = (uint16_t*)dst[g < G ? g : 0];
  }
  const int64_t blocks = (za.n + 255) / 256;
  lr_zpad<<<dim3((unsigned)(blocks < 65536 ? blocks : 65536), G), 256, 0, p[0].stream>>>(za);
  return hipGetLastError();
}

constexpr int kBwdTargetWaves = 2048;

// The byte counts lr_bwd_mfma gives its buffer resources for pass b of wq taps
// (the range audit; see the kernel): U, static_w and the dU partial per pass;
// x, dy, dx, z and the dz partials for the longest run (from row 0).
void audit_bwd_pass(const LrBwdArgs& b, int wq, bool f32) {
  const int64_t D = b.D;
  audit_range(lr_u_bytes(b.R, b.uld, b.kofs, D, 2), kOobLane);
  audit_range(lr_sw_bytes(b.RK > b.R, wq, D, 2), kOobLane);
  audit_range(lr_dupart_bytes(b.RK, b.uld, b.kofs, D), kOobLane);
  const int64_t rows[6] = {(int64_t)b.xld * 2, (int64_t)b.yhd * 2, (int64_t)b.dxld * (f32 ? 4 : 2),
                           (int64_t)b.zld * 2, (int64_t)b.dzld * 4, (int64_t)b.dxsld * 2};
  for (int64_t rowb : rows) audit_range(run_rsrc_bytes(b.Tn, rowb), kOobTile - 15 * rowb);
}

// dx rows T-kt .. T-1 of every sequence from the passes' fp32 accumulator
// (rows of D floats), rounded to the output type into dx rows dxld elements
// apart: the rows that the last pass over the accumulator, whose taps start at
// kt, does not store.
struct DxRoundGroup {
  const float* src;
  uint16_t* dst;
};
struct DxRoundArgs {
  int64_t n4;   // B * kt * D / 4 quads per group
  int dq;       // D / 4 quads per row
  int kt;       // rows per sequence
  int Tn;
  int64_t dld;  // row stride of dx (elements, a multiple of 4)
  DxRoundGroup grp[kMaxGroups];
};

template <typename T>
__global__ __launch_bounds__(256) void lr_dx_round_tail(DxRoundArgs a) {
  const int g = blockIdx.y;
  const float* __restrict__ src = pick(a.grp, g, &DxRoundGroup::src);
  uint16_t* __restrict__ dst = pick(a.grp, g, &DxRoundGroup::dst);
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < a.n4; e += (int64_t)gridDim.x * 256) {
    const int64_t rl = e / a.dq;  // the tail row of the sequences, in order
    const int c = (int)(e - rl * a.dq) * 4;
    const int64_t b = rl / a.kt;
    const int64_t row = b * a.Tn + a.Tn - a.kt + (rl - b * a.kt);
    const float4 v = *reinterpret_cast<const float4*>(src + row * a.dq * 4 + c);
    u32x2 o;
    o[0] = pack2<T>(v.x, v.y);
    o[1] = pack2<T>(v.z, v.w);
    *reinterpret_cast<u32x2*>(dst + row * a.dld + c) = o;
  }
}

template <typename T>
hipError_t launch_dx_round_tail(const LrProblem* p, int G, int64_t dxf_off, int kofs) {
  if (auditing()) return hipSuccess;  // plain pointers
  DxRoundArgs a;
  a.kt = (int)(kofs < p[0].T ? kofs : p[0].T);
  a.Tn = (int)p[0].T;
  a.dq = (int)(p[0].D / 4);
  a.n4 = p[0].B * a.kt * a.dq;
  a.dld = p[0].dxld();
  for (int g = 0; g < kMaxGroups; ++g) {
    const LrProblem& q = p[g < G ? g : 0];
    a.grp[g] = DxRoundGroup{(const float*)((const char*)q.ws + dxf_off), (uint16_t*)q.dx};
  }
  const int64_t blocks = (a.n4 + 255) / 256;
  lr_dx_round_tail<T><<<dim3((unsigned)(blocks < 8192 ? blocks : 8192), G), 256, 0, p[0].stream>>>(a);
  return hipGetLastError();
}

// Workspace: [dz partials: passes x ncg x BT x R fp32][dU partials: slots x RK
// x W*D fp32 (one per run of the contiguous problem: du_slots)][padded z_eff: BT
// x RP of z's type][past four passes, or two that split the ranks: the fp32 dx
// accumulator, BT x D], each 256-byte aligned.  The z_eff part is reserved
// whatever the pointers' alignment (the size query has none, and no row strides).
struct BwdWs {
  int64_t dz_off, du_off, zp_off, dxf_off, total;
  int slots;  // dU partials
};
BwdWs bwd_ws(const LrProblem& p, bool split) {
  const LrBwdArgs a = make_bwd_args(contiguous_problem(p), kBwdTargetWaves, split);
  BwdWs w;
  w.slots = du_slots(a.npair, a.seg);
  // one dz partial slot per pass of taps (the passes of ranks fill disjoint columns)
  const int64_t dz = (int64_t)npasses((int)p.W, bwd_rc(p)) * a.ncg * a.BT * a.R * 4;
  w.dz_off = 0;
  w.du_off = (dz + 255) / 256 * 256;
  w.zp_off = (w.du_off + (int64_t)w.slots * a.RK * p.W * p.D * 4 + 255) / 256 * 256;
  w.dxf_off = (w.zp_off + a.BT * zpad_ranks(p) * 2 + 255) / 256 * 256;
  w.total = w.dxf_off + (bwd_f32dx_room(p) ? a.BT * p.D * 4 : 0);
  return w;
}

// One pass's kernel for wq taps and rc rank chunks.
template <typename T>
hipError_t dispatch_bwd_kernel(const LrBwdArgs& a, const BwdShape& sh, int wq, int rc, bool f32, hipStream_t stream) {
  if (sh.t32) return lr_bwd_t32_launch<T>(a, wq, rc, f32, stream);
  if (f32 || a.accdx || a.nodx) return hipErrorInvalidValue;  // 16-row tiles take one pass
#define DC_BWD_CASE(WW, CC, NRW, CPW)                                                        \
  if (wq == WW && rc == CC) {                                                                \
    lr_bwd_mfma<T, WW, CC, NRW, CPW><<<a.nblk, 64 * (256 / CPW) * NRW, 0, stream>>>(a);      \
    return hipGetLastError();                                                                \
  }
  DC_BWD_CASE(1, 1, 2, 64) DC_BWD_CASE(2, 1, 2, 64) DC_BWD_CASE(3, 1, 2, 64) DC_BWD_CASE(4, 1, 2, 64)
  DC_BWD_CASE(1, 2, 1, 32) DC_BWD_CASE(4, 2, 1, 32)
  DC_BWD_CASE(1, 3, 1, 64) DC_BWD_CASE(2, 3, 1, 64) DC_BWD_CASE(1, 4, 1, 64)
#undef DC_BWD_CASE
  return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_bwd(const LrProblem* p, int G) {
  const int rc = bwd_rc(p[0]);
  BwdPass ps[kBwdMaxPlan];
  const int np = bwd_plan(p[0], ps);
  if (np < 1) return hipErrorInvalidValue;
  const bool f32 = bwd_f32dx(p[0]), dxs = bwd_dx_split(p[0]);
  LrBwdArgs a = make_bwd_args(p[0], kBwdTargetWaves, dxs);
  const BwdWs w = bwd_ws(p[0], dxs);
  const BwdShape sh = bwd_shape(p[0]);
  a.xld = (int)p[0].xld();
  a.dxld = (int)p[0].dxld();
  a.yhd = (int)p[0].yhd();
  // z itself when its rows are what the kernel reads: R % 4 == 0 and 8-byte
  // aligned, or (two rank chunks, and passes of 32 ranks) rows of a multiple
  // of 32 dynamic ranks without the static one, 16-byte aligned.
  const bool K32 = rc == 2;
  bool zvec = K32 ? (p[0].R % 32 == 0 && p[0].static_w == nullptr) : p[0].R % 4 == 0;
  for (int g = 0; g < G; ++g) {
    float* pdz = (float*)((char*)p[g].ws + w.dz_off);
    float* pdu = (float*)((char*)p[g].ws + w.du_off);
    a.grp[g] = LrBwdGroup{p[g].x, p[g].z, p[g].U, p[g].static_w, p[g].dy, p[g].dx, pdz, pdu};
    zvec = zvec && aligned_to(p[g].z, K32 ? 16 : 8);
  }
  hipError_t e;
  if (!zvec) {
    // padded z_eff rows: the forward's copy when the caller kept it, else
    // written into the workspace first
    bool saved = true;
    for (int g = 0; g < G; ++g) saved = saved && p[g].zeff != nullptr;
    void* zp[kMaxGroups];
    for (int g = 0; g < G; ++g) zp[g] = saved ? p[g].zeff : (char*)p[g].ws + w.zp_off;
    if (!saved && (e = launch_zpad<T>(p, G, zp)) != hipSuccess) return e;
    for (int g = 0; g < G; ++g) a.grp[g].z = zp[g];
    a.zld = a.zr = a.zrk = (int)zpad_ranks(p[0]);
  }
  const int64_t D = p[0].D, WD = p[0].W * D, RKWD = (int64_t)a.RK * WD, R = p[0].R;
  const int64_t dz_slot = (int64_t)a.ncg * a.BT * R;  // one pass of taps' dz partials
  // past four passes every pass works on the fp32 accumulator (rows of D floats)
  a.nodx = dxs ? 1 : 0;
  if (f32) {
    a.dxld = (int)D;
    for (int g = 0; g < G; ++g) a.grp[g].dx = (char*)p[g].ws + w.dxf_off;
  }
  a.dxsld = 0;
  // the passes over the runs that a.sp0 and a.npair name, dU partials from slot slot0 on
  auto passes = [&](int64_t slot0) {
    for (int i = 0; i < np; ++i) {
      // pass i: ranks rofs .. (z from column rofs, U and the dU partial rows from
      // row rofs, dz partial columns from rofs, static_w in the pass that holds
      // rank R), taps kofs .. (U, static_w and the dU partial columns from tap
      // kofs; dz partials in the slot of its pass of taps); the residual in the
      // first pass only
      const BwdPass& f = ps[i];
      LrBwdArgs b = a;
      b.R = f.R;
      b.RK = f.RK;
      b.kofs = f.kofs;
      b.accdx = i > 0;
      b.residual = a.residual && i == 0;
      if (f32 && i == np - 1) {  // the last pass adds to the accumulator and stores dx, rounded once
        b.dxsld = (int)p[0].dxld();
        for (int g = 0; g < G; ++g) b.grp[g].dxs = p[g].dx;
      }
      for (int g = 0; g < G; ++g) {
        b.grp[g].z = static_cast<const T*>(a.grp[g].z) + f.rofs;
        b.grp[g].U = (const T*)p[g].U + f.rofs * WD + f.kofs * D;
        b.grp[g].sw = p[g].static_w && f.RK > f.R ? (const void*)((const T*)p[g].static_w + f.kofs * D) : nullptr;
        b.grp[g].part_dz = a.grp[g].part_dz + f.slot * dz_slot + f.rofs;
        b.grp[g].part_du = a.grp[g].part_du + slot0 * RKWD + f.rofs * WD + f.kofs * D;
      }
      if (auditing()) {
        audit_bwd_pass(b, f.W, f32);
        continue;
      }
      if (dxs) {  // all passes of ranks of these taps in one launch, from the whole problem's ranks
        if (f.rofs > 0) continue;
        b.R = a.R;
        b.RK = a.RK;
        b.accdx = 0;
        b.residual = 0;
        for (int g = 0; g < G; ++g)
          b.grp[g].sw = p[g].static_w ? (const void*)((const T*)p[g].static_w + f.kofs * D) : nullptr;
      }
      if ((e = dispatch_bwd_kernel<T>(b, sh, f.W, rc, f32, p[0].stream)) != hipSuccess) return e;
    }
    return hipSuccess;
  };
  DuParts t(a.npair, w.slots);
  for (;; t.next()) {
    a.sp0 = t.run0 * sh.nrw;
    a.npair = t.n;
    a.nblk1 = a.npair * a.ncg * a.nrp;
    a.nblk = G * a.nblk1;
    if (auditing()) audit_range(w.du_off + t.used() * RKWD * 4, w.zp_off);
    if ((e = passes(t.slot0)) != hipSuccess) return e;
    if (!t.more()) break;
    PartialReduce folds[kMaxGroups];
    for (int g = 0; g < G; ++g) folds[g] = {a.grp[g].part_du, RKWD, t.used(), RKWD, a.grp[g].part_du};
    if ((e = reduce_partials_multi(folds, G, kFP32, p[0].stream)) != hipSuccess) return e;
  }
  if (auditing()) audit_range(w.total, p[0].ws_bytes);
  if (dxs) {
    const void* zs[kMaxGroups];
    for (int g = 0; g < G; ++g) zs[g] = a.grp[g].z;
    void* acc[kMaxGroups];
    for (int g = 0; g < G; ++g) acc[g] = (char*)p[g].ws + w.dxf_off;
    if ((e = lr_dx_mfma_launch<T>(p, G, zs, a.zld, acc)) != hipSuccess) return e;
    // the rows that the second launch's taps do not reach, from the accumulator
    if (lr_dx_two_passes(p[0].W) &&
        (e = launch_dx_round_tail<T>(p, G, w.dxf_off, (int)(p[0].W - p[0].W / 2))) != hipSuccess)
      return e;
  }
  // The last pass stores dx rows 0 .. T-1-kofs of its taps kofs ..; the rows
  // after those (no terms of its taps) are rounded from the accumulator here
  // (passes that split only the ranks have kofs 0: nothing left).
  if (f32 && ps[np - 1].kofs > 0 && (e = launch_dx_round_tail<T>(p, G, w.dxf_off, ps[np - 1].kofs)) != hipSuccess)
    return e;
  PartialReduce jobs[kMaxReduceJobs];
  int nj = 0;
  const int nslot = npasses((int)p[0].W, rc);
  for (int g = 0; g < G; ++g) {
    const float* pdz = a.grp[g].part_dz;
    const float* pdu = a.grp[g].part_du;
    jobs[nj++] = {pdu, RKWD, t.used(), R * WD, p[g].dU};
    jobs[nj++] = {pdu + R * WD, RKWD, t.used(), p[g].static_w ? WD : 0, p[g].dstatic_w};
    jobs[nj++] = {pdz, a.BT * R, nslot * a.ncg, a.BT * R, p[g].dz};
  }
  return reduce_partials_multi(jobs, nj, p[0].dtype, p[0].stream);
}

}  // namespace

int64_t lr_mfma_ws_bytes(const LrProblem& p) {
  // the plan depends on dy's layout (bwd_dx_split), which the size queries do not see: room for either
  const int64_t one = bwd_ws(p, false).total;
  const int64_t split = bwd_dx_split(contiguous_problem(p)) ? bwd_ws(p, true).total : 0;
  return one > split ? one : split;
}

hipError_t lr_zeff_fill(const LrProblem* p, int G) {
  void* dst[kMaxGroups];
  for (int g = 0; g < G; ++g) dst[g] = p[g].zeff;
  return p[0].dtype == kBF16 ? launch_zpad<bf16>(p, G, dst) : launch_zpad<fp16>(p, G, dst);
}

hipError_t lr_mfma_bwd(const LrProblem* p, int G) {
  return p[0].dtype == kBF16 ? launch_bwd<bf16>(p, G) : launch_bwd<fp16>(p, G);
}

}  // namespace dc
