// Lowrank forward and dx on gfx950 matrix cores with 32 ranks to a product
// (bf16 / fp16): kernel ranks 17-32 and 49-64 of the forward up to W 8, and the
// dx launch of the backwards that run as passes of ranks.
//
// A wavefront owns 32 rows x 128 channels; lane l = 16q + n owns rows 8q..8q+7
// and the channel octet 8n..8n+7 (16-byte loads, 256 contiguous bytes per row).
// The tap weights of tap k, channel 8n+j come from v_mfma_f32_16x16x32 over 32
// ranks, two per tap and channel (halves h: rows 8q+4h..+3), whose packed U
// operand (32 ranks of one channel of each lane) is read from LDS once for both.
//
// Against 16 rows and 16 ranks to a product (lr_fwd_mfma), per row and channel:
// half the LDS reads of U operands (at 64 ranks and W 4 these were 128 KB per 32
// rows and wavefront, 15 us of LDS time at B4 T4096 D2048) and half the matrix
// time (a 16x16x16 product takes as long as a 16x16x32 one).  Channels are
// computed a pair at a time: 16 accumulators and the pair's fp32 rows are live,
// the packed results replace the pair's raw rows.
// 60-133 VGPRs at 32 ranks, 74-248 at 64 (dx 88-256), none spilled.
// B4 T4096 D2048 bf16, inputs out of the cache, 16 ranks to a product -> this one,
// z_eff writer included: forward R31 + static 36.8 -> 30.6 us (4.5 TB/s of its
// bytes), W 8 47.0 -> 38.7, R63 + static 41.9 -> 37.3, W 8 73.8 -> 51.5, B2 T8192
// D4096 R31 + static 59.8 -> 56.0.  Without the writer (R32; inference) W 3-4 are 2-6%
// slower here (R32 30.1 -> 31.5) and 3-7% at B2 T10000 D1536, B3 T4788 D3712 and B6 T2048
// D4096, faster elsewhere (B12 T4096 D2048 107 -> 85, B2 T2048 D1024 21.6 -> 8.5).
// Backward with this dx launch: R63 + static 156 -> 140, W 8 390 -> 244, R127 + static
// 294 -> 244.
// What bounds the forward: at W 4 the wait for its rows (37% of the wavefronts' cycles;
// a plain copy of the same tensors reaches 5.1 TB/s); at W 8 issue (44%, 38% vector).
#pragma once

#include "lowrank_mfma_fwd_kernel.h"

namespace dc {

// Tiles per run of the dx launch: 2048 wavefronts where the problem has that many
// tiles, runs of about 4 tiles above, at most 4096 wavefronts (see fwd_target_waves).
inline int64_t t32_run_tiles(int64_t tiles) {
  int64_t w = tiles / 4;
  w = w < 2048 ? (tiles < 2048 ? tiles : 2048) : w > 4096 ? 4096 : w;
  return (tiles + w - 1) / w;
}

// Wavefronts per workgroup: as fwd_wg_waves (one workgroup per CU above 80 KiB of operands).
constexpr int t32_wg_waves(int W, int NC) { return W * NC > 10 ? 8 : 4; }

// Tiles per run of the forward: the length with the least time by a model of
// workgroups on 256 CUs, fitted at W x NC = 4, 8 and 16 to 84 sweeps of the run
// length (its choice is within 0.3% of the best length's time on average, 4% at
// most).  A CU works off k workgroups, each its start (staging of U; part) and its
// wavefronts' tiles (tile); or, with few of them, the serial chain of a round (lat
// per tile).  Runs of about 4 tiles whatever the rounds left 2.6 workgroups to a CU
// at B3 T4788 D3712: bf16 R32 W 4 55.2 -> 48 us, R63 + static W 4 77.4 -> 60.5; B4
// T6144 D2048 R63 + static W 8 89.9 -> 72.5, B2 T4096 D3072 R32 W 4 31.4 -> 25.5, B4
// T4096 D2048 equal (31.5).  A grouped call's workgroups count together; y does not
// depend on the runs.
inline int64_t t32_fwd_run_tiles(int64_t B, int64_t ntile, int64_t cols, int W, int NC) {
  struct Cost { double part, tile, lat, start; };
  constexpr Cost c4{0.46, 0.66, 4.4, 1.4}, c8{4.0, 0.91, 5.0, 9.0}, c16{7.2, 0.86, 8.8, 1.3};
  const int n = W * NC, nwv = t32_wg_waves(W, NC);
  const Cost &lo = n <= 8 ? c4 : c8, &hi = n <= 8 ? c8 : c16;
  const double f = n <= 4 ? 0 : n <= 8 ? (n - 4) / 4.0 : (n - 8) / 8.0;
  const auto mix = [f](double a, double b) { return a + f * (b - a); };
  const Cost c{mix(lo.part, hi.part), mix(lo.tile, hi.tile), mix(lo.lat, hi.lat), mix(lo.start, hi.start)};
  // bound by memory (n <= 4): more workgroups to a CU (B8 T4096 D4096 R31 + static W 4,
  // runs of 4, 8 and 16 tiles: 104.8, 106.3, 113.4 us)
  const int64_t longest = n <= 4 ? 4 : 64;
  const int64_t res = 256 * (n <= 5 ? 4 : 20 / n);  // workgroups resident at once (8 n KiB of 160 each)
  int64_t best = 1;
  double best_us = -1;
  for (int64_t seg = 1; seg <= ntile && seg <= longest; seg += seg < 16 ? 1 : seg / 4) {
    const int64_t runs = B * ((ntile + seg - 1) / seg), wg = (runs + nwv - 1) / nwv * cols;
    const double work = (double)((wg + 255) / 256) * (c.part + seg * nwv * c.tile);
    const double chain = (double)((wg + res - 1) / res) * (seg * c.lat + c.start);
    const double us = work > chain ? work : chain;
    if (best_us < 0 || us < best_us) {
      best = seg;
      best_us = us;
    }
  }
  return best;
}

// ub[((k*NC + c)*8 + j)*64 + lane] = U_eff[32c + 8q .. +7, k*D + dl + j], packed
// (row R is static_w, rows past RK zero; loads as in stage_u).
template <int W, int NC>
__device__ __forceinline__ void stage_u32(u32x4* __restrict__ lds, const uint16_t* __restrict__ U,
                                          const uint16_t* __restrict__ sw, int R, int RK, int D, int64_t WD, int dl,
                                          bool chv, int q, int lane, int wave) {
  const uint16_t* const safe = R > 0 ? U : sw;
  for (int kc = wave; kc < W * NC; kc += t32_wg_waves(W, NC)) {
    const int k = kc / NC, c = kc - k * NC;
    u32x4 rows[8];
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) {
      const int r = 32 * c + 8 * q + kk;
      const int64_t at = (int64_t)k * D + dl;
      const uint16_t* src = r < R ? U + r * WD + at : sw + at;
      src = chv && r < RK ? src : safe;
      rows[kk] = gload128(src);
    }
#pragma unroll
    for (int kk = 0; kk < 8; ++kk) {
      const bool ok = chv && 32 * c + 8 * q + kk < RK;
#pragma unroll
      for (int h = 0; h < 4; ++h) rows[kk][h] = ok ? rows[kk][h] : 0u;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t hl = j & 1 ? 0x07060302u : 0x05040100u;
      u32x4 v;
#pragma unroll
      for (int h = 0; h < 4; ++h) v[h] = __builtin_amdgcn_perm(rows[2 * h + 1][j >> 1], rows[2 * h][j >> 1], hl);
      lds[(kc * 8 + j) * 64 + lane] = v;
    }
  }
}

// z_eff operand of one row: ranks 32c+8q .. +7 for c < NC.  ZAL: rows of whole
// aligned 16-byte octets (R % 8 == 0 and 16-byte aligned rows, or a padded z_eff
// with R == RK == 32 NC).  Otherwise R % 8 == 7: octets load at the row's own
// 2-byte alignment, and the octet that R ends in loads the eight ranks that end at
// R, shifted down by one with the static rank (or 0) on top.
template <typename T, int NC, bool ZAL>
struct Z32 {
  u32x4 v[NC];
  __device__ __forceinline__ void load(rsrc_t rz, int base, int R, int q) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int r0 = 32 * c + 8 * q;
      const int s = ZAL || r0 + 8 <= R ? r0 : R - 8;
      v[c] = bload128(rz, r0 < R ? base + s * 2 : kOobTile);
    }
  }
  // t: the row; ranks past R: static (1) at R when the row is inside the sequence, else 0
  __device__ __forceinline__ void finish(u32x4 (&o)[NC], int t, int R, int RK, int Tn, int q) const {
    const uint32_t st = R < RK && t < Tn ? (uint32_t)Mma16<T>::kOne : 0u;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int r0 = 32 * c + 8 * q;
      o[c] = v[c];
      if constexpr (ZAL) {
        if (r0 == R) o[c][0] = st;  // a static rank that opens an octet (the load was out of range: 0)
      } else {
        const bool cut = r0 < R && r0 + 8 > R;
        u32x4 s;
#pragma unroll
        for (int h = 0; h < 3; ++h) s[h] = __builtin_amdgcn_alignbit(v[c][h + 1], v[c][h], 16);
        s[3] = (v[c][3] >> 16) | (st << 16);
#pragma unroll
        for (int h = 0; h < 4; ++h) o[c][h] = cut ? s[h] : v[c][h];
      }
    }
  }
};

// The wavefront's run and the buffer resources of its rows, common to both kernels.
struct T32Run {
  int tile0, tile1, rb;
  int64_t row0, rrow;
  __device__ __forceinline__ T32Run(const LrArgs& a, int sg) {
    const int b = sg / a.nspb;
    tile0 = (sg - b * a.nspb) * a.seg;
    tile1 = min(tile0 + a.seg, (a.Tn + 31) >> 5);
    rb = run_base_row(2 * tile0);
    row0 = (int64_t)b * a.Tn;
    rrow = row0 + rb;
  }
};

// Ends the work on one channel pair: its packed results exist here, and the LDS
// reads of the next pair's operands come after (a sched_barrier alone does not
// order pure arithmetic, and the pairs' weights, rows and sums then live together:
// 256 registers and up to 1.2 KB of spills, against 142 and none at W 4 and 64 ranks).
__device__ __forceinline__ void end_pair(u32x4 (&o)[8], int h4) {
  asm volatile("" : "+v"(o[0][h4]), "+v"(o[1][h4]), "+v"(o[2][h4]), "+v"(o[3][h4]), "+v"(o[4][h4]), "+v"(o[5][h4]),
               "+v"(o[6][h4]), "+v"(o[7][h4]) : : "memory");
}

// Tap weights of both halves for one tap and channel: rows 8q .. 8q+7.
template <typename T, int NC>
__device__ __forceinline__ void tap32(f32x4 (&wk)[2], const u32x4 (&z)[2][NC], const u32x4* __restrict__ u, float w0) {
#pragma unroll
  for (int h = 0; h < 2; ++h) wk[h] = f32x4{w0, w0, w0, w0};
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const u32x4 uo = u[c * 8 * 64];
#pragma unroll
    for (int h = 0; h < 2; ++h) wk[h] = Mma32<T>::run(z[h][c], uo, wk[h]);
  }
}

// ---------------------------------------------------------------- forward
// ZE: also write the padded z_eff rows (zrp ranks, a multiple of 8) for the
// backward; row r of a tile is written by the channel chunk r % nch.
template <typename T, int W, int NC, bool ZAL, bool ZE>
__global__ __launch_bounds__(64 * t32_wg_waves(W, NC)) void lr_fwd_t32(LrArgs a) {
  constexpr int NWV = t32_wg_waves(W, NC);
  constexpr bool HX = W >= 2 && W <= 4;  // halo rows from the lane group above (see lr_fwd_mfma)
  constexpr int NR = W + 7;              // x rows 8q-W+1 .. 8q+7
  constexpr int NH = W > 1 ? W - 1 : 1;
  __shared__ u32x4 ub[W * NC * 8 * 64];

  const int lane = threadIdx.x & 63, wave = wave_id();
  const int q = lane >> 4, n = lane & 15;
  const int lb0 = xcd_remap(blockIdx.x, a.nblk);
  const int g = __builtin_amdgcn_readfirstlane(lb0 / a.nblk1);
  const int lb = lb0 - g * a.nblk1;
  const auto* gp = kernel_args<LrArgs>()->grp + g;
  const uint16_t* __restrict__ x = reinterpret_cast<const uint16_t*>(gp->x);
  const uint16_t* __restrict__ z = reinterpret_cast<const uint16_t*>(gp->z);
  uint16_t* __restrict__ y = reinterpret_cast<uint16_t*>(gp->y);
  const int chunk = lb % a.nch, sgp = lb / a.nch;
  const int D = a.D, Tn = a.Tn, R = a.R, RK = a.RK;
  const int dl = chunk * 128 + 8 * n;
  const bool chv = dl < D;  // D % 8 == 0: octets are whole
  stage_u32<W, NC>(ub, reinterpret_cast<const uint16_t*>(gp->U), reinterpret_cast<const uint16_t*>(gp->sw), R, RK, D,
                   a.uld, dl, chv, q, lane, wave);
  __syncthreads();
  const int sg = sgp * NWV + wave;
  if (sg >= a.nseg) return;
  const T32Run run(a, sg);
  const int rb = run.rb;
  // y [B, T, D] (yhd == D) or head-major [B, D/yhd, T, yhd]: see lr_fwd_mfma
  const int yhd = a.yhd, yh = dl / yhd;
  const int yh0 = chunk * 128 / yhd, yhl = min(chunk * 128 + 127, D - 1) / yhd;
  const int rowb = yhd * 2, xrowb = a.xld * 2, zld = a.zld;
  const rsrc_t rx = run_rsrc(x + run.rrow * a.xld, Tn - rb, xrowb);
  const rsrc_t ry =
      run_rsrc(y + run.row0 * D + ((int64_t)yh0 * Tn + rb) * yhd, (int64_t)(yhl - yh0) * Tn + Tn - rb, rowb);
  const rsrc_t rz = run_rsrc(z + run.rrow * zld, Tn - rb, zld * 2);
  const int zrp = ZE ? a.zrp : 0;
  const rsrc_t rze =
      ZE ? run_rsrc(reinterpret_cast<const uint16_t*>(gp->zeff) + run.rrow * zrp, Tn - rb, zrp * 2) : make_rsrc(z, 0);
  const int lane_off = chv ? (((yh - yh0) * Tn + 8 * q) * yhd + dl - yh * yhd) * 2 : kOobLane;
  const int xlane_off = chv ? (8 * q * a.xld + dl) * 2 : kOobLane;
  const int above = ((lane + 48) & 63) << 2;  // ds_bpermute byte address of lane - 16
  const int zrow = 8 * (n >> 2) + (n & 3);    // tile row of the lane's z operand in half 0 (half 1: + 4)
  const float res = a.residual ? 1.f : 0.f;   // tap 0's weight + 1

  u32x4 prev[NH];  // HX: rows 32-W+1 .. 31 of the tile before (group 3 sends them)
  if constexpr (HX) {
#pragma unroll
    for (int m = 0; m < W - 1; ++m)
      prev[m] = bload128(rx, (chv ? dl * 2 : kOobLane) + (run.tile0 * 32 + m + 1 - W - rb) * xrowb);
  }
  for (int tile = run.tile0; tile < run.tile1; ++tile) {
    u32x4 xr[NR];
    const int xtoff = (tile * 32 - rb) * xrowb;
#pragma unroll
    for (int m = HX ? W - 1 : 0; m < NR; ++m)
      xr[m] = bload128<HX ? kNt : 0>(rx, xlane_off + xtoff + (m - (W - 1)) * xrowb);
    Z32<T, NC, ZAL> zr[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) zr[h].load(rz, (tile * 32 + zrow + 4 * h - rb) * zld * 2, R, q);
    u32x4 zc[2][NC];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int t = tile * 32 + zrow + 4 * h;
      zr[h].finish(zc[h], t, R, RK, Tn, q);
      if constexpr (ZE) {
        const bool mine = (zrow + 4 * h) % a.nch == chunk && t < Tn;
#pragma unroll
        for (int c = 0; c < NC; ++c)
          bstore128<false>(zc[h][c], rze, mine && 32 * c + 8 * q < zrp ? ((t - rb) * zrp + 32 * c + 8 * q) * 2 : kOobTile);
      }
    }
    if constexpr (HX) {
#pragma unroll
      for (int m = 0; m < W - 1; ++m) {
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const uint32_t s = q == 3 ? prev[m][h] : xr[m + 8][h];
          xr[m][h] = (uint32_t)__builtin_amdgcn_ds_bpermute(above, (int)s);
        }
        prev[m] = xr[m + 8];
      }
    }
    u32x4 out[8];
#pragma unroll
    for (int h4 = 0; h4 < 4; ++h4) {
      float acc[2][8];
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) {
        float xf[NR];
#pragma unroll
        for (int m = 0; m < NR; ++m) xf[m] = Mma16<T>::to_f(jj ? xr[m][h4] >> 16 : xr[m][h4] & 0xFFFFu);
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[jj][i] = 0.f;
#pragma unroll
        for (int k = 0; k < W; ++k) {
          f32x4 wk[2];
          tap32<T, NC>(wk, zc, ub + (k * NC * 8 + 2 * h4 + jj) * 64 + lane, k == 0 ? res : 0.f);
#pragma unroll
          for (int i = 0; i < 8; ++i) acc[jj][i] = fmaf(wk[i >> 2][i & 3], xf[i - k + W - 1], acc[jj][i]);
        }
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) out[i][h4] = pack2<T>(acc[0][i], acc[1][i]);
      end_pair(out, h4);
      __builtin_amdgcn_sched_barrier(0);
    }
    const int toff = (tile * 32 - rb) * rowb;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      bstore128<true>(out[i], ry, tile * 32 + 8 * q + i < Tn ? lane_off + toff + i * rowb : kOobTile);
  }
}

// --------------------------------------------------------------------- dx
// dx[t] = sum_k dy[t+k] * K[t+k, k] (+ dy[t]) over all kernel ranks, rounded once
// (lowrank.py:143-205), in scatter form: dy[s] K[s, k] goes to row s - k; the W-1
// rows of the group above (W <= 8) pass up with a ds_bpermute per channel, and
// group 3's open rows wait one tile in fp32 (carry).  The tile after a run closes
// its last rows.  z is read as z_eff rows of 32 NC ranks (grp.z, zld; static column
// included), grp.x is dy, grp.y dx (rows yhd apart).
//
// M: taps past one launch's operands take two (kernel rank 33-64 at W 9-16), over
// an fp32 accumulator (grp.zeff, rows of D): M 1 stores it, M 2 (taps kofs .., its
// rows kofs earlier) adds it and stores dx, rounded once; dx's last kofs rows, which
// get no terms of M 2's taps, are left to the caller.  Against passes of 32 ranks x 4
// taps that each added dx into the accumulator, whole backward at B4 T4096 D2048
// bf16: R40 W 12 530 -> 386 us, R64 W 16 772 -> 534 us.
template <typename T, int W, int NC, int M = 0, bool HM = M != 0>
__global__ __launch_bounds__(64 * t32_wg_waves(W, NC)) void lr_dx_t32(LrArgs a) {
  constexpr int NWV = t32_wg_waves(W, NC);
  constexpr int NO = W > 1 ? W - 1 : 1;  // open rows of a group (none at W 1)
  constexpr int kFirstOpen = 9 - W;
  __shared__ u32x4 ub[W * NC * 8 * 64];

  const int lane = threadIdx.x & 63, wave = wave_id();
  const int q = lane >> 4, n = lane & 15;
  const int lb0 = xcd_remap(blockIdx.x, a.nblk);
  const int g = __builtin_amdgcn_readfirstlane(lb0 / a.nblk1);
  const int lb = lb0 - g * a.nblk1;
  const auto* gp = kernel_args<LrArgs>()->grp + g;
  const uint16_t* __restrict__ dy = reinterpret_cast<const uint16_t*>(gp->x);
  const uint16_t* __restrict__ z = reinterpret_cast<const uint16_t*>(gp->z);
  uint16_t* __restrict__ dx = reinterpret_cast<uint16_t*>(gp->y);
  const int chunk = lb % a.nch, sgp = lb / a.nch;
  const int D = a.D, Tn = a.Tn, RK = a.RK;
  const int dl = chunk * 128 + 8 * n;
  const bool chv = dl < D;
  stage_u32<W, NC>(ub, reinterpret_cast<const uint16_t*>(gp->U), reinterpret_cast<const uint16_t*>(gp->sw), a.R, RK, D,
                   a.uld, dl, chv, q, lane, wave);
  __syncthreads();
  const int sg = sgp * NWV + wave;
  if (sg >= a.nseg) return;
  const T32Run run(a, sg);
  const int rb = run.rb, tile0 = run.tile0, tile1 = run.tile1, ntile = (Tn + 31) >> 5;
  // dy is [B, T, D] (hd == D) or, with HM, head-major [B, D/hd, T, hd]: the resource
  // then spans the chunk's heads (loads check the row against T)
  const int hd = HM ? a.zrp : a.xld, yh = HM ? dl / hd : 0, yh0 = HM ? chunk * 128 / hd : 0;
  const int yhl = HM ? min(chunk * 128 + 127, D - 1) / hd : 0;
  const int dyrowb = hd * 2, dxrowb = a.yhd * 2, zld = a.zld;
  const rsrc_t rdy = run_rsrc(dy + run.row0 * a.xld + ((int64_t)yh0 * Tn + rb) * hd,
                              (int64_t)(yhl - yh0) * Tn + Tn - rb, dyrowb);
  const rsrc_t rdx = run_rsrc(dx + run.rrow * a.yhd, Tn - rb, dxrowb);
  const rsrc_t rz = run_rsrc(z + run.rrow * zld, Tn - rb, zld * 2);
  const int dylane = chv ? (((yh - yh0) * Tn + 8 * q) * hd + dl - yh * hd) * 2 : kOobLane;
  const int dxlane = chv ? (8 * q * a.yhd + dl) * 2 : kOobLane;
  const int below = ((lane + 16) & 63) << 2;  // ds_bpermute byte index of the group below
  const int zrow = 8 * (n >> 2) + (n & 3);
  const float res = a.residual ? 1.f : 0.f;
  const bool top = q == 3;
  const int accrowb = D * 4, kofs = M == 2 ? a.kofs : 0;
  const rsrc_t racc = run_rsrc(reinterpret_cast<float*>(gp->zeff) + run.rrow * D, Tn - rb, M ? accrowb : 0);
  // M: the row of the resources that the lane's row i of a tile closes as (-1: none)
  auto acc_row = [&](int tile, int i) {
    const bool before = top && W > 1 && i >= kFirstOpen;  // group 3's open rows close a tile late
    const int t = (before ? tile - 1 : tile) * 32 + 8 * q + i;
    const bool ok = chv && (before ? tile > tile0 : tile < tile1) && t >= kofs && t < Tn;
    return ok ? t - kofs - rb : -1;
  };

  float carry[4][2][NO];  // group 3's open rows of the tile before (the run's first tile stores none)
#pragma unroll
  for (int h4 = 0; h4 < 4; ++h4)
#pragma unroll
    for (int jj = 0; jj < 2; ++jj)
#pragma unroll
      for (int m = 0; m < NO; ++m) carry[h4][jj][m] = 0.f;

  for (int tile = tile0; tile <= tile1; ++tile) {
    const bool live = tile < ntile;
    const int toff = live ? (tile * 32 - rb) * dyrowb : kOobTile;
    u32x4 dyr[8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
      dyr[i] = bload128(rdy, HM && tile * 32 + 8 * q + i >= Tn ? kOobTile : dylane + toff + i * dyrowb);
    u32x4 zc[2][NC];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int c = 0; c < NC; ++c)
        zc[h][c] = bload128(rz, live ? (tile * 32 + zrow + 4 * h - rb) * zld * 2 + (32 * c + 8 * q) * 2 : kOobTile);
    u32x4 acc[M ? 8 : 1][2];  // the accumulator's rows (M 1: to store)
    if constexpr (M == 2) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int r = acc_row(tile, i);
          acc[i][h] = bload128(racc, r >= 0 ? r * accrowb + dl * 4 + 16 * h : kOobTile);
        }
    }
    u32x4 out[8];
#pragma unroll
    for (int h4 = 0; h4 < 4; ++h4) {
      float v[2][8];
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) {
        float dyf[8], own[8], S[NO];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          dyf[i] = Mma16<T>::to_f(jj ? dyr[i][h4] >> 16 : dyr[i][h4] & 0xFFFFu);
          own[i] = 0.f;
        }
#pragma unroll
        for (int m = 0; m < NO; ++m) S[m] = 0.f;
#pragma unroll
        for (int k = 0; k < W; ++k) {
          f32x4 wk[2];
          tap32<T, NC>(wk, zc, ub + (k * NC * 8 + 2 * h4 + jj) * 64 + lane, k == 0 ? res : 0.f);
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const int r = i - k;
            if (r >= 0)
              own[r] = fmaf(wk[i >> 2][i & 3], dyf[i], own[r]);
            else
              S[-r - 1] = fmaf(wk[i >> 2][i & 3], dyf[i], S[-r - 1]);  // row 8q-1-m of the group above
          }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          v[jj][i] = own[i];
          if (W > 1 && i >= kFirstOpen) {
            const float recv = __int_as_float(__builtin_amdgcn_ds_bpermute(below, __float_as_int(S[(7 - i) % NO])));
            float& cy = carry[h4][jj][(i - kFirstOpen) % NO];
            v[jj][i] = (top ? cy : own[i]) + recv;
            cy = own[i];
          }
        }
      }
      if constexpr (M == 1) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int jj = 0; jj < 2; ++jj) {
            uint32_t o = __float_as_uint(v[jj][i]);
            asm volatile("" : "+v"(o) : : "memory");  // as end_pair
            acc[i][h4 >> 1][2 * (h4 & 1) + jj] = o;
          }
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          if constexpr (M == 2) {
#pragma unroll
            for (int jj = 0; jj < 2; ++jj) v[jj][i] += __uint_as_float(acc[i][h4 >> 1][2 * (h4 & 1) + jj]);
          }
          out[i][h4] = pack2<T>(v[0][i], v[1][i]);
        }
        end_pair(out, h4);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (M != 0) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int r = acc_row(tile, i);
        if constexpr (M == 2) {
          bstore128<true>(out[i], rdx, r >= 0 ? r * dxrowb + dl * 2 : kOobTile);
        } else {
#pragma unroll
          for (int h = 0; h < 2; ++h)
            bstore128<false>(acc[i][h], racc, r >= 0 ? r * accrowb + dl * 4 + 16 * h : kOobTile);
        }
      }
      continue;
    }
    const int cur_off = tile < tile1 ? dxlane + (tile * 32 - rb) * dxrowb : kOobTile;
    const int prev_off = tile > tile0 ? dxlane + ((tile - 1) * 32 - rb) * dxrowb : kOobTile;
    const int open_off = top ? prev_off : cur_off;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      bstore128<true>(out[i], rdx, (W > 1 && i >= kFirstOpen ? open_off : cur_off) + i * dxrowb);
  }
}

// Forward pass on lr_fwd_t32 (lowrank_mfma_fwd_t32_{bf16,fp16}.hip): a.zvec says ZAL, a.zrp > 0 ZE.
template <typename T>
hipError_t lr_fwd_t32_launch(const LrArgs& a, int W, int NC, hipStream_t stream);
// dx launch on lr_dx_t32.
template <typename T>
hipError_t lr_dx_t32_launch(const LrArgs& a, int W, int NC, int M, hipStream_t stream);

}  // namespace dc
