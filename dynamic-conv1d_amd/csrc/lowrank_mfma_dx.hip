// dx of the lowrank backward over all kernel ranks (lr_dx_t32, lowrank_mfma_t32.h),
// for the problems whose backward runs as passes of 32 ranks (lr_bwd_rank_split):
// those passes then form dz and dU only (lr_bwd_t32's DXM 3), and dx is rounded
// once.  Up to W 8 one launch takes all taps; at W 9-16 (kernel rank 33-64) two
// launches of half the taps each, over an fp32 accumulator that the first stores
// and the second adds, where the passes themselves would add to it once per
// 32 ranks and 4 taps.
#include "lowrank_mfma_t32.h"

namespace dc {

template <typename T>
hipError_t lr_dx_t32_launch(const LrArgs& a, int W, int NC, int M, hipStream_t s) {
#define DC_DX_CASE(WW, CC)                                                          \
  if (W == WW && NC == CC && M == 0) {                                              \
    if (a.zrp == a.xld)                                                             \
      lr_dx_t32<T, WW, CC><<<a.nblk, 64 * t32_wg_waves(WW, CC), 0, s>>>(a);         \
    else                                                                            \
      lr_dx_t32<T, WW, CC, 0, true><<<a.nblk, 64 * t32_wg_waves(WW, CC), 0, s>>>(a);\
    return hipGetLastError();                                                       \
  }
  // W x NC <= 16: up to 128 KiB of staged operands (lr_dx_split_shape)
  DC_DX_CASE(1, 2) DC_DX_CASE(2, 2) DC_DX_CASE(3, 2) DC_DX_CASE(4, 2)
  DC_DX_CASE(5, 2) DC_DX_CASE(6, 2) DC_DX_CASE(7, 2) DC_DX_CASE(8, 2)
  DC_DX_CASE(1, 3) DC_DX_CASE(2, 3) DC_DX_CASE(3, 3) DC_DX_CASE(4, 3) DC_DX_CASE(5, 3)
  DC_DX_CASE(1, 4) DC_DX_CASE(2, 4) DC_DX_CASE(3, 4) DC_DX_CASE(4, 4)
#undef DC_DX_CASE
  // the two launches of W 9-16 at 33-64 ranks: ceil(W / 2) taps, then the others
#define DC_DX_CASE2(WW, MM)                                                         \
  if (W == WW && NC == 2 && M == MM) {                                              \
    lr_dx_t32<T, WW, 2, MM><<<a.nblk, 64 * t32_wg_waves(WW, 2), 0, s>>>(a);         \
    return hipGetLastError();                                                       \
  }
  DC_DX_CASE2(5, 1) DC_DX_CASE2(6, 1) DC_DX_CASE2(7, 1) DC_DX_CASE2(8, 1)
  DC_DX_CASE2(4, 2) DC_DX_CASE2(5, 2) DC_DX_CASE2(6, 2) DC_DX_CASE2(7, 2) DC_DX_CASE2(8, 2)
#undef DC_DX_CASE2
  return hipErrorInvalidValue;
}

// Taps kofs .. kofs+W-1 of the problem (M, acc: see lr_dx_t32).
template <typename T>
static hipError_t dx_taps(const LrProblem* p, int G, const void* const* z, int zld, int kofs, int W, int M,
                          void* const* acc) {
  const LrProblem& p0 = p[0];
  const int RK = (int)p0.R + (p0.static_w ? 1 : 0), NC = (RK + 31) / 32;
  const int nwv = t32_wg_waves(W, NC);
  LrArgs a{};
  a.Tn = (int)p0.T;
  a.D = (int)p0.D;
  a.R = (int)p0.R;
  a.RK = RK;
  a.residual = p0.residual && kofs == 0;
  a.kofs = kofs;
  a.nch = (int)((p0.D + 127) / 128);
  a.zld = zld;
  a.xld = (int)p0.D;       // dy: [B, T, D],
  a.zrp = (int)p0.yhd();   // or head-major
  a.yhd = (int)p0.dxld();  // dx rows
  a.uld = p0.uld();
  // runs as the forward's, capped so that the rows of dy, dx and z a run
  // touches (its tiles, the halo, the tile after it) stay inside the resources
  const int64_t ntile = (p0.T + 31) / 32;
  int64_t seg = t32_run_tiles(p0.B * ntile * a.nch);
  int64_t rowb = p0.D > p0.dxld() ? p0.D : p0.dxld();
  rowb = 2 * (rowb > zld ? rowb : zld);
  if (M && p0.D * 4 > rowb) rowb = p0.D * 4;  // the accumulator's rows
  const int64_t cap = run_tiles_cap(rowb) / 2;  // >= 1 (lr_bwd_max_run_tiles)
  if (seg > cap) seg = cap;
  if (seg < 1) seg = 1;
  if (seg > ntile) seg = ntile;
  a.seg = (int)seg;
  a.nspb = (int)((ntile + seg - 1) / seg);
  a.nseg = (int)(p0.B * a.nspb);
  a.nblk1 = ((a.nseg + nwv - 1) / nwv) * a.nch;
  a.nblk = G * a.nblk1;
  for (int g = 0; g < G; ++g) {
    const T* sw = (const T*)p[g].static_w;
    a.grp[g] = LrFwdGroup{p[g].dy, z[g], (const T*)p[g].U + kofs * p0.D, sw ? sw + kofs * p0.D : nullptr, p[g].dx,
                          M ? acc[g] : nullptr};
  }
  if (auditing()) {
    const int64_t rows[4] = {(int64_t)a.xld * 2, (int64_t)a.yhd * 2, (int64_t)a.zld * 2, M ? p0.D * 4 : 4};
    for (int64_t rb : rows) audit_range(run_rsrc_bytes(a.Tn, rb), kOobTile - 15 * rb);
    const int64_t hd = p0.yhd();
    if (hd != p0.D) audit_range(run_rsrc_bytes((127 / hd + 2) * p0.T, hd * 2), kOobTile - 15 * hd * 2);
    return hipSuccess;
  }
  return lr_dx_t32_launch<T>(a, W, NC, M, p0.stream);
}

// z[g]: group g's z_eff rows as the passes read them, zld elements apart (a
// multiple of 32 ranks, static column included); acc[g]: the fp32 accumulator
// (two launches, lr_dx_two_passes; dx's last W / 2 rows are the caller's then).
template <typename T>
hipError_t lr_dx_mfma_launch(const LrProblem* p, int G, const void* const* z, int zld, void* const* acc) {
  const int W = (int)p[0].W;
  if (!lr_dx_two_passes(W)) return dx_taps<T>(p, G, z, zld, 0, W, 0, nullptr);
  const hipError_t e = dx_taps<T>(p, G, z, zld, 0, W - W / 2, 1, acc);
  return e == hipSuccess ? dx_taps<T>(p, G, z, zld, W - W / 2, W / 2, 2, acc) : e;
}

template hipError_t lr_dx_mfma_launch<bf16>(const LrProblem*, int, const void* const*, int, void* const*);
template hipError_t lr_dx_mfma_launch<fp16>(const LrProblem*, int, const void* const*, int, void* const*);

}  // namespace dc
