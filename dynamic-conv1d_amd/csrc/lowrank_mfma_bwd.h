// Shared pieces of the lowrank backward on gfx950 matrix cores (bf16 / fp16):
// the launch arguments and the row-piece types of its two kernels, lr_bwd_t32
// (lowrank_mfma_bwd32.h) and lr_bwd_mfma (lowrank_mfma_bwd.hip), and the host's
// launch of the first.
#pragma once

#include "lowrank_mfma.h"

namespace dc {

struct LrBwdGroup {
  const void* x;   // this group's first channel; rows xld elements apart
  const void* z;
  const void* U;
  const void* sw;
  const void* dy;
  void* dx;        // this group's first channel; rows dxld elements apart
  float* part_dz;
  float* part_du;
  void* dxs;       // the last pass over the fp32 accumulator (DXM 2): dx itself, rows dxsld apart
};

struct LrBwdArgs {
  int Tn, D, R, RK, residual;
  int nch;    // channel chunks of one wavefront (32 or 64 channels)
  int ncg;    // chunk groups of 256 channels: one workgroup column
  int seg;    // tiles per run
  int nspb;   // runs per sequence
  int nseg;   // B * nspb
  int npair;  // workgroup rows of a launch: a run, a dU partial each (lr_bwd_mfma: one or two; nseg, or a part: DuParts)
  int sp0;    // first run of the launch; its dU partial is part_du's first
  int nblk;   // ncg * npair * nrp * groups
  int nblk1;  // blocks per group
  int xld;    // row stride of x (elements)
  int dxld;   // row stride of dx (elements; the fp32 accumulator's D past four passes)
  int dxsld;  // row stride of dx for the last pass over the accumulator (DXM 2)
  int nodx;   // dz and dU only (DXM 3): launches of their own (lr_dx_t32) form dx over all ranks
  int nrp;    // with nodx: passes of 32 ranks in this launch (R and RK are then the problem's), else 1
  // z rows: zld elements apart, ranks < zr loaded, ranks zr .. zrk-1 of z_eff
  // added as the static rank (ZRaw).  z itself (zld = zr = R, zrk = RK) when
  // R % 4 == 0 and z is 8-byte aligned, else the padded z_eff copy in the
  // workspace (zld = zr = zrk = RP, the static column included).
  int zld, zr, zrk;
  int yhd;    // dy layout: D ([B, T, D]) or the head dim of [B, D/yhd, T, yhd]
  int uld;    // row stride of U and of the dU partials: the problem's W * D (all taps)
  int kofs;   // first tap of this pass (0 without a tap split)
  int accdx;  // add dx to what an earlier pass stored
  // A pass of ranks writes its dz and dU partial entries into the whole
  // problem's layout: dz partial rows dzld (its R) floats apart (part_dz starts
  // at the pass's first rank), dU partials of dupr (its kernel rank) rows each
  // (part_du starts at the pass's first rank row).  Without rank passes dzld = R
  // and dupr = RK.
  int dzld, dupr;
  int64_t BT;
  LrBwdGroup grp[kMaxGroups];
};


// A lane's two 16-bit channels of one row (lr_bwd_t32): one 4-byte unit.
struct Pair {
  __device__ static __forceinline__ uint32_t load(rsrc_t r, int off) { return bload32(r, off); }
  __device__ static __forceinline__ uint32_t elem(uint32_t v, int j) { return j ? (v >> 16) : (v & 0xFFFFu); }
};

// A lane's two channels of one dx row as the passes keep them: the output type
// (DxVec<T, false>), or past four passes (two that split the ranks) an fp32
// accumulator in the workspace (DxVec<T, true>), which the last pass rounds to
// dx once (more passes rounded in 16 bits each drift past the 2e-2 elementwise bar).
template <typename T, bool F32> struct DxVec {
  typedef uint32_t type;
  static constexpr int ES = 2;
  __device__ static __forceinline__ type load(rsrc_t r, int off) { return bload32(r, off); }
  // 16-bit rows leave in 64-byte pieces (half lines): the default policy lets the
  // L2 join two wavefronts' halves (B2 T8192 D4096 R31 + static backward 129 ->
  // 125 us against nontemporal stores, W 8 at R15 85 -> 83 us); NT: lr_bwd_t32's NTP
  template <bool NT>
  __device__ static __forceinline__ void store(type v, rsrc_t r, int off) {
    __builtin_amdgcn_raw_buffer_store_b32(v, r, off, 0, NT ? kNt : 0);
  }
  __device__ static __forceinline__ float get(type v, int j) { return Mma16<T>::to_f(Pair::elem(v, j)); }
  __device__ static __forceinline__ type make(const float* f) { return pack2<T>(f[0], f[1]); }
};
template <typename T> struct DxVec<T, true> {
  typedef u32x2 type;
  static constexpr int ES = 4;
  __device__ static __forceinline__ type load(rsrc_t r, int off) { return bload64(r, off); }
  template <bool NT>
  __device__ static __forceinline__ void store(type v, rsrc_t r, int off) { bstore64<true>(v, r, off); }
  __device__ static __forceinline__ float get(const type& v, int j) { return __uint_as_float(v[j]); }
  __device__ static __forceinline__ type make(const float* f) {
    return type{__float_as_uint(f[0]), __float_as_uint(f[1])};
  }
};

// Launch of lr_bwd_t32 for one pass of W taps and RC rank chunks (1 <= W <= 8
// at one chunk, 1 <= W <= 4 at two); accdx, nodx, dxsld and f32 pick the
// variant (ACC and DXM of the kernel).  Instantiated in lowrank_mfma_bwd32_{bf16,fp16}.hip.
template <typename T>
hipError_t lr_bwd_t32_launch(const LrBwdArgs& a, int W, int RC, bool f32, hipStream_t stream);

// Rows per tile and channels per workgroup of lr_bwd_t32.
constexpr int kT32Rows = 32, kT32Chan = 32;

}  // namespace dc
