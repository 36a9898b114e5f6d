// Lowrank backward on gfx950 matrix cores (bf16 / fp16): dx, dz, dU, dstatic_w.
#include "lowrank_mfma_bwd.h"

namespace dc {

// ---------------------------------------------------------------- backward
//
// Host side of the backward (launch plans, passes, workspace), and the kernel of
// the one-pass problems of three and four rank chunks (kernel ranks 33-48 at
// W <= 2, 49-64 at W 1).  One and two rank chunks, and every problem that runs
// as passes of ranks, take lr_bwd_t32 (lowrank_mfma_bwd32.h).
//
// lr_bwd_mfma: one pass over x and dy produces dx, dz, dU and dstatic_w
// (reference: lowrank.py:87-140 and 159-205, two kernels that both read dy).
// A wavefront owns 16 rows x 64 channels; lane l = 16q + n owns rows 4q..4q+3
// and the channels 4n..4n+3 (one 8-byte load per row).  With
// G_k[t, d] = bf16(dy[t, d] * x[t-k, d]) (the reference also rounds this
// product to bf16 before its dot products, lowrank.py:128):
//   * dU[r, kD+d] += sum_t z_eff[t, r] G_k[t, d]: MFMA with K = the 16 rows; the
//     lane's four G values of column 4n+j are the B operand.
//   * dz[t, r] += sum_d G_k[t, d] U_eff[r, kD+d]: K = 32 channels; the packed dU
//     operands go through the wavefront's LDS slot and come back by row with
//     transposing reads (ds_read_b64_tr_b16).
//   * Tap weights Kw[t, k, :] = z_eff[t, :] U_eff[:, k]: one 16x16x16 MFMA per
//     rank chunk.  The residual's dy rides on tap 0: its accumulator starts at 1.
//   * dx[t, d] = sum_k dy[t+k, d] Kw[t+k, k, d] (+ dy) in scatter form: dy[s]
//     Kw[s, k] goes to row s-k; the sums for the group above (W 2) pass up with
//     a ds_bpermute, and group 3's open row waits one tile.
// A workgroup is four wavefronts on 256 adjacent channels of one run of rows.
// dz sums over the 256 channels are added in LDS in wave order, dU accumulates
// in registers over the run; both go out as fp32 partials that reduce_partials
// sums in a fixed order.
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

// U_eff operands of one wavefront's 64-channel chunk, staged once per run: the
// tap-weight operands in registers, the dz operands in LDS.  For tap k and rank
// chunk c, lane (q, n) holds
//   uw[j] (j < 4): ranks 16c+4q..16c+4q+3 of channel 4n+j, packed (B operand of
//                  the 16x16x16 tap-weight MFMA);
//   uz[s] (s < 2): rank 16c+n, channels 32s+8q..32s+8q+7 as they lie in U (B
//                  operand of the 16x16x32 dz MFMA).
template <int W, int RC>
__device__ __forceinline__ void stage_uops(u32x2 (&uw)[W * RC * 4], u32x4* __restrict__ uz_lds,
                                           const uint16_t* __restrict__ U, const uint16_t* __restrict__ sw, int R,
                                           int RK, int D, int uld, int d0, int q, int n, int lane) {
  // Buffer loads, all issued before the first use: rows r >= R of U and lanes
  // outside D read 0; the static row (r == R < RK) is read from sw and OR-ed in.
  const rsrc_t ru = make_rsrc(U, lr_u_bytes(R, uld, 0, D, 2));
  const rsrc_t rs = make_rsrc(sw, lr_sw_bytes(RK > R, W, D, 2));
  const int cw = d0 + 4 * n < D ? (d0 + 4 * n) * 2 : kOobLane;  // the lane's tap-weight channels
  u32x2 rows[W][RC][4];
  u32x4 zr[W][RC][2];
#pragma unroll
  for (int k = 0; k < W; ++k)
#pragma unroll
    for (int c = 0; c < RC; ++c) {
      const bool has_static = RK > R && R >= 16 * c && R < 16 * c + 16;  // chunk c holds the static row
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        const int r = 16 * c + 4 * q + kk;
        rows[k][c][kk] = bload64(ru, r < R ? cw + (r * uld + k * D) * 2 : kOobLane) |
                         bload64(rs, has_static && r == R ? cw + k * D * 2 : kOobLane);
      }
      const int r = 16 * c + n;
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
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
      for (int j = 0; j < 4; ++j) {
        const u32x2(&rw)[4] = rows[k][c];
        uw[(k * RC + c) * 4 + j][0] = elem16x2(rw[0], j) | (elem16x2(rw[1], j) << 16);
        uw[(k * RC + c) * 4 + j][1] = elem16x2(rw[2], j) | (elem16x2(rw[3], j) << 16);
      }
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) uz_lds[((k * RC + c) * 2 + s2) * 64 + lane] = zr[k][c][s2];
    }
}

template <typename T, int W, int RC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 8))) void lr_bwd_mfma(LrBwdArgs a) {
  static_assert(W <= 2 && (RC == 3 || RC == 4), "the one-pass shapes of three and four rank chunks");
  typedef ZRaw<T, RC, true> ZR;   // 8-byte z loads: rows of zld % 4 == 0 elements
  constexpr int NR = W + 3;       // x rows 4q-W+1 .. 4q+3 per lane
  // G tile in LDS, transposed: channel c's rows 4p..4p+3 (8 bytes) at byte
  // p*GPL + 8c + 8(c/16).  The pad of 8 bytes per 16 channels keeps both access
  // patterns within two-way bank conflicts.
  constexpr int GPL = 8 * 64 + 32;  // bytes per 4-row plane
  __shared__ u32x4 uz_lds[4][W * RC * 2 * 64];
  __shared__ __attribute__((aligned(16))) uint8_t gtile[4][4 * GPL];
  // dz sums of the workgroup's chunks (double-buffered: one barrier per tile).
  // Row r, rank n of a tile sits at (16r + n) ^ ((r / 4) << 4): the XOR puts the
  // four row groups a lane quarter writes at once in different banks.
  __shared__ float dzred[2][4][RC * 256];

  const int lane = threadIdx.x & 63, wave = wave_id();
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
  const int cg = lb % a.ncg, du_slot = lb / a.ncg, sp = a.sp0 + du_slot;
  const int D = a.D, Tn = a.Tn;
  const int d0 = (cg * 4 + wave) * 64;
  const int col = d0 + 4 * n;
  const bool chv = col < D;  // the lane's 4 channels inside D (D % 8 == 0: all or none)
  const int ntile = (Tn + 15) >> 4;
  // the workgroup's run: tiles [tile0, tile1) of sequence b, whose buffer resources start at row rb
  const int b = sp / a.nspb;
  const int tile0 = (sp - b * a.nspb) * a.seg;
  const int tile1 = min(tile0 + a.seg, ntile);
  const int rb = run_base_row(tile0);
  const int64_t row0 = (int64_t)b * Tn, rrow = row0 + rb;
  const int R = a.R, RK = a.RK;
  u32x4* __restrict__ my_uz = uz_lds[wave];
  // G^T write position of the lane's channel 4n (plus 8j), and the transposed-read
  // position that returns row n, channels 8q..8q+3 (plus 32 for 8q+4..8q+7, plus
  // 8*32+16 per 32-channel block)
  uint8_t* const my_g = gtile[wave];
  const int gw_lane = q * GPL + 32 * n + (n / 4) * 8;
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
  const rsrc_t rpz = run_rsrc(part_dz + ((int64_t)cg * a.BT + rrow) * a.dzld, Tn - rb, a.dzld * 4);
  // byte offsets of the lane's row-4q channels in dy, x and dx
  const int lane_off = chv ? (4 * q * yhd + col - head * yhd) * 2 : kOobLane;
  const int xlane_off = chv ? (4 * q * a.xld + col) * 2 : kOobLane;
  const int dxlane_off = chv ? (4 * q * a.dxld + col) * 2 : kOobLane;

  // Identity as the B operand: lane (q, n) gives rows 4q..4q+3 of column n.
  u32x2 ident;
  {
    const uint32_t one = Mma16<T>::kOne;
    uint32_t e[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) e[kk] = (4 * q + kk == n) ? one : 0u;
    ident[0] = e[0] | (e[1] << 16);
    ident[1] = e[2] | (e[3] << 16);
  }
  u32x2 uw[W * RC * 4];
  f32x4 du[W][RC][4];
#pragma unroll
  for (int k = 0; k < W; ++k)
#pragma unroll
    for (int c = 0; c < RC; ++c)
#pragma unroll
      for (int j = 0; j < 4; ++j) du[k][c][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Tile inputs (buffer loads: out-of-range rows / channels read as 0).  Two
  // buffers alternate: while one tile is computed the next one's loads are in
  // flight.  A tile past the run reads the out-of-range offset kOobTile; dy and z
  // of the tile after the run are read too (its first row closes the last dx row).
  struct TileIn {
    u32x2 xr[NR], dyr[4];
    ZR zr;
  };
  auto load_tile = [&](int tile, TileIn& in) {
    const bool live = tile < tile1, ylive = tile <= tile1;
    const int xtoff = live ? (tile * 16 - rb) * xrowb : kOobTile;
    const int toff = ylive ? (tile * 16 - rb) * rowb : kOobTile;
#pragma unroll
    for (int m = 0; m < NR; ++m) in.xr[m] = bload64(rx, xlane_off + xtoff + (m - (W - 1)) * xrowb);
#pragma unroll
    for (int m = 0; m < 4; ++m) in.dyr[m] = bload64(rdy, lane_off + toff + m * rowb);  // nontemporal: 71 us for 62 (R63 + static)
    in.zr.load(rz, ylive ? (tile * 16 + n - rb) * zld * 2 : kOobTile, zr, q);
  };
  // Tap k's weights of the lane's rows for channel 4n+j, accumulator started at w0.
  auto tap_w = [&](const u32x2(&za)[RC], int k, int j, float w0) {
    f32x4 wk = {w0, w0, w0, w0};
#pragma unroll
    for (int c = 0; c < RC; ++c) wk = Mma16<T>::run(za[c], uw[(k * RC + c) * 4 + j], wk);
    return wk;
  };
  auto scatter = [&](const f32x4& wk, const float(&dyf)[4][4], int k, int j, float(&own)[4][4], float(&S)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (i >= k)
        own[i - k][j] = fmaf(dyf[i][j], wk[i], own[i - k][j]);
      else
        S[j] = fmaf(dyf[i][j], wk[i], S[j]);  // row 4q-1, of the group above
    }
  };
  float carry[4] = {0.f, 0.f, 0.f, 0.f};  // W 2: group 3's open row of the tile before
  auto close_rows = [&](const float(&own)[4][4], const float(&S)[4], int tile) {
    const int src = ((lane + 16) & 63) << 2;  // ds_bpermute byte index of the group below
    const bool top = q == 3;
    const int cur_off = tile < tile1 ? dxlane_off + (tile * 16 - rb) * dxrowb : kOobTile;
    const int prev_off = tile > tile0 ? dxlane_off + ((tile - 1) * 16 - rb) * dxrowb : kOobTile;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool open = W == 2 && i == 3;  // takes the group below's sums
      float v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[j] = own[i][j];
        if (open)
          v[j] = (top ? carry[j] : v[j]) + __int_as_float(__builtin_amdgcn_ds_bpermute(src, __float_as_int(S[j])));
      }
      bstore64<true>(u32x2{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])}, rdx,
                     (top && open ? prev_off : cur_off) + i * dxrowb);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) carry[j] = own[3][j];
  };
  auto compute_tile = [&](int it, const TileIn& in) {
    const int tile = tile0 + it;
    u32x2 zA[RC], zT[RC];
    in.zr.finish(zA, tile * 16 + n, zr, zrk, Tn, q);
    // z_eff transposed (rank n, rows 4q..4q+3) through an exact identity product
#pragma unroll
    for (int c = 0; c < RC; ++c) {
      const f32x4 tz = Mma16<T>::run(zA[c], ident, f32x4{0.f, 0.f, 0.f, 0.f});
      zT[c] = u32x2{pack2<T>(tz[0], tz[1]), pack2<T>(tz[2], tz[3])};
    }
    float dyf[4][4], own[4][4], S[4];
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        dyf[m][j] = Mma16<T>::to_f(elem16x2(in.dyr[m], j));
        own[m][j] = S[j] = 0.f;
      }
    f32x4 dz[RC];
#pragma unroll
    for (int c = 0; c < RC; ++c) dz[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < W; ++k) {
      // the wave barriers keep the compiler from moving an LDS write above
      // another lane's read (the hardware keeps a wavefront's LDS order)
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        scatter(tap_w(zA, k, j, k == 0 ? res : 0.f), dyf, k, j, own, S);
        float gf[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) gf[i] = dyf[i][j] * Mma16<T>::to_f(elem16x2(in.xr[i - k + W - 1], j));
        const u32x2 gk = {pack2<T>(gf[0], gf[1]), pack2<T>(gf[2], gf[3])};
        *reinterpret_cast<u32x2*>(my_g + gw_lane + 8 * j) = gk;
#pragma unroll
        for (int c = 0; c < RC; ++c) du[k][c][j] = Mma16<T>::run(zT[c], gk, du[k][c][j]);
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        const u32x2 lo = lds_read_tr16(my_g + gr_lane + s2 * (8 * 32 + 16));
        const u32x2 hi = lds_read_tr16(my_g + gr_lane + s2 * (8 * 32 + 16) + 32);
        const u32x4 ga = {lo[0], lo[1], hi[0], hi[1]};
#pragma unroll
        for (int c = 0; c < RC; ++c) dz[c] = Mma32<T>::run(ga, my_uz[((k * RC + c) * 2 + s2) * 64 + lane], dz[c]);
      }
    }
    close_rows(own, S, tile);
    const int buf = it & 1;
#pragma unroll
    for (int c = 0; c < RC; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) dzred[buf][wave][c * 256 + (((4 * q + i) * 16 + n) ^ (q << 4))] = dz[c][i];
    __syncthreads();
#pragma unroll
    for (int c = 0; c < RC; ++c) {
      const int e = (int)threadIdx.x, rr = e >> 4, r = 16 * c + (e & 15);
      const int pos = c * 256 + (e ^ (((e >> 6) & 3) << 4));
      float v = dzred[buf][0][pos];
#pragma unroll
      for (int w2 = 1; w2 < 4; ++w2) v += dzred[buf][w2][pos];
      // ranks >= R store nothing (rows past T lie outside the resource)
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rpz,
                                            r < R ? ((tile * 16 + rr - rb) * a.dzld + r) * 4 : kOobLane, 0, 0);
    }
  };

  TileIn ta, tb;
  load_tile(tile0, ta);
  __builtin_amdgcn_sched_barrier(0);  // the first tile's loads go out before the U staging waits
  stage_uops<W, RC>(uw, my_uz, U, sw, R, RK, D, a.uld, d0, q, n, lane);
  const int nit = tile1 - tile0;
  for (int it = 0; it < nit; it += 2) {
    load_tile(tile0 + it + 1, tb);
    __builtin_amdgcn_sched_barrier(0);  // issue the next tile's loads before this tile's waits
    compute_tile(it, ta);
    load_tile(tile0 + it + 2, ta);
    __builtin_amdgcn_sched_barrier(0);
    if (it + 1 < nit) compute_tile(it + 1, tb);
  }
  if constexpr (W == 2) {
    // the tile after the run closes its last row
    auto flush = [&](const TileIn& in) {
      u32x2 zA[RC];
      in.zr.finish(zA, tile1 * 16 + n, zr, zrk, Tn, q);
      float dyf[4][4], own[4][4], S[4];
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          dyf[m][j] = Mma16<T>::to_f(elem16x2(in.dyr[m], j));
          own[m][j] = S[j] = 0.f;
        }
#pragma unroll
      for (int j = 0; j < 4; ++j) scatter(tap_w(zA, 1, j, 0.f), dyf, 1, j, own, S);
      close_rows(own, S, tile1);
    };
    if (nit & 1)
      flush(tb);
    else
      flush(ta);
  }

  // ---- dU partial of this run: rows r < RK of U_eff, the wavefront's 64 columns
  // per tap.  The resource spans the run's RK x W*D partial, so rows r >= RK fall
  // outside it (the host keeps (RK + 16) * W * D * 4 bytes below kOobLane, so no
  // offset wraps).
  const rsrc_t rdu = make_rsrc(part_du + (int64_t)du_slot * a.dupr * a.uld, lr_dupart_bytes(RK, a.uld, 0, D));
  const int du_lane = chv ? (4 * q * a.uld + col) * 4 : kOobLane;
#pragma unroll
  for (int k = 0; k < W; ++k)
#pragma unroll
    for (int c = 0; c < RC; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        bstore128<false>(u32x4{__float_as_uint(du[k][c][0][i]), __float_as_uint(du[k][c][1][i]),
                               __float_as_uint(du[k][c][2][i]), __float_as_uint(du[k][c][3][i])},
                         rdu, du_lane + ((16 * c + i) * a.uld + k * D) * 4);
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
// Passes of ranks with dy in [B, T, D] whose dx fits one launch
// (lr_dx_split_shape: W <= 8 up to kernel rank 64, W 5 / 4 up to 96 / 128) or,
// with dy in either layout, two (W 9-16 up to 64, over the fp32 accumulator): the
// passes form dz and dU only (DXM 3) and lr_dx_t32 forms dx over all ranks and
// taps in one launch, rounded once (no fp32 accumulator).  Passes of taps alone
// (two rank chunks above W 4) keep dx: split off it measured 160 -> 166 us at B4
// T4096 D2048 R31 + static W 8.
inline bool bwd_dx_split(const LrProblem& p) {
  const int64_t hd = p.yhd();
  // head-major dy: two launches only, where a chunk's heads fit one resource
  const bool dy_ok = hd == p.D || (lr_dx_two_passes(p.W) && (127 / hd + 2) * (p.T + 64) * hd * 2 < kMaxSeqBytes);
  return bwd_rank_split(p) && lr_dx_split_shape(p.R + (p.static_w ? 1 : 0), p.W) && dy_ok;
}
// The workspace keeps room for the accumulator whether or not dx is split off:
// the size queries do not see dy's layout, on which the split depends.
inline bool bwd_f32dx_room(const LrProblem& p) {
  const int np = bwd_rank_passes(p) * npasses((int)p.W, bwd_rc(p));
  return np > kBwdMaxBf16DxPasses || (bwd_rank_passes(p) > 1 && np > kBwdMaxBf16DxRankPasses);
}
inline bool bwd_f32dx(const LrProblem& p) { return !bwd_dx_split(p) && bwd_f32dx_room(p); }

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

// Tiles per run of lr_bwd_t32: a CU holds one of its workgroups, so a launch
// takes ceil(workgroups / 256) rounds of a run's length each, and a few
// workgroups past a round cost as much as a full one (B1 T8192 D768 R15 + static
// W 8: runs of 3 tiles are 258 workgroups and took 48 us, runs of 4 31 us; B3
// T4788 D3712 R32: 270 workgroups 163 us, 225 116 us).  Of the run
// lengths that fill one to eight rounds, the one with the least time by a
// model: per round a launch's start and end (6 us) and the run's tiles, and
// every run's dU partial written and read once.  dflt: no such length (more
// sequences than eight rounds hold).
int64_t t32_run_tiles(const LrProblem& p, int64_t ntile, int64_t cols, int64_t dflt) {
  constexpr int64_t kCus = 256;
  const double tile_us = 0.6 * (p.W < 2 ? 2 : p.W > 8 ? 8 : p.W) * (bwd_rc(p) == 2 ? 1.25 : 1.0);
  const double part_us = (double)(p.R + (p.static_w ? 1 : 0)) * p.W * p.D * 8 / 5e6;
  int64_t best = dflt;
  double best_us = -1;
  for (int64_t rounds = 1; rounds <= 8; ++rounds) {
    const int64_t per_seq = rounds * kCus / (p.B * cols);  // runs a sequence may take
    if (per_seq < 1) continue;
    const int64_t seg = (ntile + per_seq - 1) / per_seq, runs = p.B * ((ntile + seg - 1) / seg);
    const double us = rounds * (6.0 + seg * tile_us) + runs * part_us;
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
  const int rc = bwd_rc(p);
  const bool t32 = rc <= 2;  // lr_bwd_t32, else lr_bwd_mfma
  const int cpw = t32 ? kT32Chan : 64, ncw = 256 / cpw, rows = t32 ? kT32Rows : 16;
  a.Tn = (int)p.T;
  a.D = (int)p.D;
  a.R = (int)p.R;
  a.RK = (int)p.R + (p.static_w ? 1 : 0);
  a.residual = p.residual;
  a.nch = (int)((p.D + cpw - 1) / cpw);
  a.ncg = (a.nch + ncw - 1) / ncw;
  const int64_t ntile = (p.T + rows - 1) / rows;
  a.nrp = split ? bwd_rank_passes(p) : 1;
  const int64_t cap = lr_bwd_max_run_tiles(p) * 16 / rows;  // >= 1 (lr_mfma_ok)
  int64_t seg = (p.B * ntile * a.ncg * ncw * a.nrp + target_waves - 1) / target_waves;
  if (t32) seg = t32_run_tiles(p, ntile, (int64_t)a.ncg * a.nrp, seg);
  if (seg < 1) seg = 1;
  if (seg > ntile) seg = ntile;
  if (seg > cap) seg = cap;
  a.seg = (int)seg;
  a.nspb = (int)((ntile + seg - 1) / seg);
  a.nseg = (int)(p.B * a.nspb);
  a.npair = a.nseg;
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
  w.slots = du_slots(a.nseg, a.seg);
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
hipError_t dispatch_bwd_kernel(const LrBwdArgs& a, int wq, int rc, bool f32, hipStream_t stream) {
  if (rc <= 2) return lr_bwd_t32_launch<T>(a, wq, rc, f32, stream);
  if (f32 || a.accdx || a.nodx) return hipErrorInvalidValue;  // three and four rank chunks take one pass
  if (rc == 3 && wq == 1)
    lr_bwd_mfma<T, 1, 3><<<a.nblk, 256, 0, stream>>>(a);
  else if (rc == 3 && wq == 2)
    lr_bwd_mfma<T, 2, 3><<<a.nblk, 256, 0, stream>>>(a);
  else if (rc == 4 && wq == 1)
    lr_bwd_mfma<T, 1, 4><<<a.nblk, 256, 0, stream>>>(a);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
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
      if ((e = dispatch_bwd_kernel<T>(b, f.W, rc, f32, p[0].stream)) != hipSuccess) return e;
    }
    return hipSuccess;
  };
  DuParts t(a.nseg, w.slots);
  for (;; t.next()) {
    a.sp0 = t.run0;
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
