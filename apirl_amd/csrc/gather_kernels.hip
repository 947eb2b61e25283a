// Deterministic backprojectors for gfx950: the voxel-driven gather, the 2D gather by patches and
// the 3D tile-walk form (each described at its kernels).
//
// The voxel-driven gather: one voxel per lane.  For each angle of the subset the lane finds the
// contiguous radial bins whose LOR can cross its voxel column, and for 3D, per segment, the
// contiguous range of sinograms whose ray can cross its slice.  For every candidate
// ray it reconstructs, without walking the ray, the state the reference's Siddon
// loop would be in when it emits this voxel (recon/src/Siddon.cpp:310-340, 615-639):
//   (a, b, c) = number of x, y, z crossings taken before the voxel,
//   the last crossing taken (alpha_c) and the next one (the segment end),
// using the exact values of the float accumulators (alpha_exact.h).  The voxel is
// on the ray's list iff every crossing taken precedes every crossing not taken in
// the loop's order (value, then x before y before z) and a + b + c is below the
// list length |di| + |dj| + |dk| (:220, :521), which reproduces the dropped exit
// voxel and the zero-length entry segments.  The weight (next - alpha_c) * L is then
// the reference's float, bit for bit.
//
// Terms are summed in a fixed order (angle, radial bin, segment, sinogram), so the
// result does not depend on scheduling: repeated runs are bit-identical.  No atomics.
#include <cfloat>
#include <algorithm>
#include <climits>
#include <cmath>
#include <vector>

#include "apirl_internal.h"
#include "alpha_exact.h"
#include "siddon_f64.h"

namespace apirl {

namespace {

constexpr int kGBlock = 256;
// axial margin of the sinogram search: covers the drift of the accumulated z
// crossings against the exact slab faces (well below 1e-3 mm here)
constexpr float kZMargin = 0.05f;

__device__ __forceinline__ float z_at(float za, float vz, float alpha) { return za + vz * alpha; }

// ZRay (apirl_internal.h): per-ray axial part of the Siddon setup for one subset
// (Siddon.cpp:150-182, 220, 244-255, 279-286) and the bin value, computed once per
// backprojection by zsetup_kernel.

// The axial part of one ray's setup in float (the reference's operations in its
// order): entry and exit slices, first z crossing and its increment, and the length.
__device__ __forceinline__ void zray_setup(const Geo& g, const RayXY& R, float za, float zb,
                                           ZRay& z) {
  const float vz = zb - za;
  const float z1 = za + vz * R.amin;
  const float z2 = za + vz * R.amax;
  const int kinc = vz > 0 ? 1 : (vz < 0 ? -1 : 0);
  z.kinc = (short)kinc;
  z.k0 = (int)floorf((z1 - g.offz) / g.dz);
  z.k1 = (short)(int)floorf((z2 - g.offz) / g.dz);
  z.azu = fabsf(g.dz / vz);
  if (vz > 0) z.az0 = (g.offz + (z.k0 + kinc) * g.dz - za) / vz;
  else if (vz < 0) z.az0 = (g.offz + z.k0 * g.dz - za) / vz;
  else z.az0 = FLT_MAX;
  const float ez = (za + vz) - za;
  z.L = sqrtf(R.lxy + ez * ez);
}

// nz_pair[ka * nr + r] != 0 iff some sinogram has a non-zero bin at (angle ka, r):
// the gather skips (angle, r) pairs whose bins are all zero (zero bins add nothing,
// SiddonProjector.cpp:496).
__device__ __forceinline__ void zsetup_one(const Geo& g, const RayXY* __restrict__ rays,
                                           const float2* __restrict__ zab,
                                           const float* __restrict__ sino, int kind,
                                           int nang_sub, int subset, int nsubsets,
                                           ZRay* __restrict__ out, int* __restrict__ nz_pair,
                                           float* __restrict__ ztab,
                                           const int* __restrict__ zsoff, int zblock,
                                           long idx, int f64s = 0) {
  const int rr = (int)(idx % g.nr);
  const long t = idx / g.nr;
  const int ka = (int)(t % nang_sub);
  const int s = (int)(t / nang_sub);
  const int a = subset + nsubsets * ka;
  const RayXY R = rays[(long)a * g.nr + rr];
  const float za = zab[s].x, zb = zab[s].y;
  const float vz = zb - za;
  ZRay z;
  const int kinc = vz > 0 ? 1 : (vz < 0 ? -1 : 0);
  z.kinc = (short)kinc;
  if (f64s) {
    // APIRL_PREC_F64_SETUP: the axial setup in double from the float LOR, rounded to
    // float, as the projector's F64_SETUP loop starts from it
    SetupXY64 xy;
    setup_xy_f64(g, R.p0x, R.p0y, R.vx, R.vy, xy);
    SetupZ64 zs;
    setup_z_f64(g, xy, za, R.vx, R.vy, (double)vz, zs);
    z.k0 = zs.k0;
    z.k1 = (short)zs.k1;
    z.az0 = (float)zs.az;
    z.azu = (float)zs.azu;
    z.L = (float)zs.L;
  } else {
    zray_setup(g, R, za, zb, z);
  }
  float b = 1.f;
  if (kind == BP_PLAIN) b = sino[idx];
  else if (kind == BP_MULT) b = sino[((long)s * g.nang + a) * g.nr + rr];
  z.b = b;
  // The ray's z crossings as the reference accumulates them (alpha_z += alpha_z_u,
  // Siddon.cpp:338): entry t is the value after t additions.  A ray with more
  // crossings than its slot (not expected: the slot bounds |Vz| (amax - amin) / dz)
  // is flagged and the gather reconstructs its crossings with alpha_after.
  // Entries are written for the slices k0 + kinc, k0 + 2 kinc, ... as far as the
  // slot reaches, at most |k1 - k0| + 2 of them (the loop's N steps can include a z
  // step more than the floor-based count when an x or y step fewer is taken);
  // zcount records how many, and the gather reconstructs any crossing beyond them
  // with alpha_after.
  const int nzc = abs((int)z.k1 - z.k0);
  int nw = 0;
  // a zero bin adds nothing (the gathers skip it once they have its record), so its
  // crossings are not written
  if (ztab && kinc != 0 && b != 0.f) {
    const int base = zsoff[s], slot = zsoff[s + 1] - base, kmin = zsoff[g.nsino + 1 + s];
    // entry e of the sinogram's slot lives at ((base + e) * nang_sub + ka) * nr + rr:
    // the rays of one (sinogram, angle) are adjacent, as the gather's lanes read them
    const long npair = (long)nang_sub * g.nr;
    float* dst = ztab + (long)ka * g.nr + rr;
    float az = z.az0;
    int kk = z.k0 + kinc;
    while (nw < nzc + 2 && kk - kmin >= 0 && kk - kmin < slot) {
      dst[(long)(base + kk - kmin) * npair] = az;  // entering slice kk: value after nw additions
      az = az + z.azu;
      kk += kinc;
      nw++;
    }
  }
  z.zcount = nw;
  z.pad = 0;
  out[idx] = z;  // (sinogram, angle, radial bin) order
  if (b != 0.f && (R.flags & RAY_VALID)) {
    int* f = &nz_pair[(long)ka * g.nr + rr];
    if (*f == 0) atomicOr(f, 1);
  }
}

__global__ __launch_bounds__(kGBlock) void zsetup_kernel(Geo g, const RayXY* __restrict__ rays,
                                                         const float2* __restrict__ zab,
                                                         const float* __restrict__ sino, int kind,
                                                         int nang_sub, int subset, int nsubsets,
                                                         long nrays, ZRay* __restrict__ out,
                                                         int* __restrict__ nz_pair,
                                                         float* __restrict__ ztab,
                                                         const int* __restrict__ zsoff,
                                                         int zblock, int f64s) {
  const long idx = (long)blockIdx.x * kGBlock + threadIdx.x;
  if (idx < nrays)
    zsetup_one(g, rays, zab, sino, kind, nang_sub, subset, nsubsets, out, nz_pair, ztab, zsoff,
               zblock, idx, f64s);
}

__global__ __launch_bounds__(kGBlock) void clear_int_kernel(int* __restrict__ p, long n) {
  const long i = (long)blockIdx.x * kGBlock + threadIdx.x;
  if (i < n) p[i] = 0;
}



// Voxel tile of one workgroup in the transaxial mapping: 16 x 16 voxels of one slice.
constexpr int kTile = 16;
constexpr int kWave = 64;

// Per-voxel accumulator of the gather for each precision mode.
template <int PREC>
struct Acc {
  using alpha_t = float;
  float s;
  __device__ void init(float v) { s = v; }
  __device__ void add(float t) { s = s + t; }
  // add(t) when c, else nothing (selected, so no branch)
  __device__ void add_if(bool c, float t) {
    const float n = s + t;
    s = c ? n : s;
  }
  __device__ void add_f64(double) {}
  __device__ float value() const { return s; }
};
template <>
struct Acc<APIRL_PREC_KAHAN> {
  using alpha_t = float;
  float s, c;
  __device__ void init(float v) { s = v; c = 0.f; }
  __device__ void add(float t) {
    const float y = t - c;
    const float u = s + y;
    c = (u - s) - y;
    s = u;
  }
  __device__ void add_if(bool cond, float t) {
    const float y = t - c;
    const float u = s + y;
    const float nc = (u - s) - y;
    s = cond ? u : s;
    c = cond ? nc : c;
  }
  __device__ void add_f64(double) {}
  __device__ float value() const { return s; }
};
// F64_SETUP: float crossings and weights from the double setup, summed as KAHAN.
template <>
struct Acc<APIRL_PREC_F64_SETUP> : Acc<APIRL_PREC_KAHAN> {};
template <>
struct Acc<APIRL_PREC_F64_ALPHA> {
  using alpha_t = double;
  double s;
  __device__ void init(float v) { s = v; }
  __device__ void add(float t) { s += t; }
  __device__ void add_f64(double t) { s += t; }
  __device__ float value() const { return (float)s; }
};

// First x / y crossings and increments of a ray.  REFERENCE and KAHAN use the
// reference's float values from the ray table (Siddon.cpp:253-286, with the 2D
// clamp of a negative first crossing to alpha_min, :590-606); F64_ALPHA in 2D
// recomputes them in double from the float entry voxel (3D F64_ALPHA does the whole
// setup in double, siddon_f64.h).
template <int PREC, int DIMS>
__device__ __forceinline__ void first_crossings(const Geo& g, const RayXY& t, int iinc, int jinc,
                                                typename Acc<PREC>::alpha_t& ax0,
                                                typename Acc<PREC>::alpha_t& axu,
                                                typename Acc<PREC>::alpha_t& ay0,
                                                typename Acc<PREC>::alpha_t& ayu) {
  if (PREC != APIRL_PREC_F64_ALPHA) {
    ax0 = t.ax;
    axu = t.axu;
    ay0 = t.ay;
    ayu = t.ayu;
  } else {
    const double R = g.R;
    const double vx = t.vx, vy = t.vy;
    ax0 = FLT_MAX;
    ay0 = FLT_MAX;
    axu = 0.0;
    ayu = 0.0;
    if (iinc != 0) {
      axu = fabs((double)g.dx / vx);
      ax0 = (-R + (double)(t.i0 + (iinc > 0 ? 1 : 0)) * g.dx - t.p0x) / vx;
      if (DIMS == 2 && ax0 < 0.0) ax0 = t.amin;
    }
    if (jinc != 0) {
      ayu = fabs((double)g.dy / vy);
      ay0 = (-R + (double)(t.j0 + (jinc > 0 ? 1 : 0)) * g.dy - t.p0y) / vy;
      if (DIMS == 2 && ay0 < 0.0) ay0 = t.amin;
    }
  }
}

// n-th crossing after the first: the exact float accumulator (alpha_exact.h) or,
// in double, a0 + n u.
// alpha_after out of line: the column kernel needs it only for the rare crossings the
// table does not hold, and inlined, parts of it are hoisted to every sinogram.
__device__ __noinline__ float alpha_after_call(float a, float u, int n) {
  return alpha_after(a, u, n);
}

template <int PREC>
__device__ __forceinline__ typename Acc<PREC>::alpha_t crossing(typename Acc<PREC>::alpha_t a0,
                                                               typename Acc<PREC>::alpha_t u,
                                                               int n) {
  if (PREC == APIRL_PREC_F64_ALPHA) return a0 + (double)n * u;
  else return alpha_after_call((float)a0, (float)u, n);
}

template <int PREC>
__device__ __forceinline__ void z_crossings(const Geo& g, const ZRay& z, float2 zz,
                                            typename Acc<PREC>::alpha_t& az0,
                                            typename Acc<PREC>::alpha_t& azu) {
  if (PREC != APIRL_PREC_F64_ALPHA) {
    az0 = z.az0;
    azu = z.azu;
  } else {
    const double za = zz.x, vz = (double)zz.y - zz.x;
    azu = fabs((double)g.dz / vz);
    if (vz > 0) az0 = ((double)g.offz + (double)(z.k0 + 1) * g.dz - za) / vz;
    else if (vz < 0) az0 = ((double)g.offz + (double)z.k0 * g.dz - za) / vz;
    else az0 = FLT_MAX;
  }
}

// Range [jlo, jhi] of bins whose LORs can pass within hw of a point at signed
// distance sc from the centre along their normal, from the radial lookup table
// (one grid step of slack on each side for rounding); empty when jlo > jhi.
__device__ __forceinline__ void lut_bins(const GatherArgs& A, float sc, float hw, int& jlo,
                                         int& jhi) {
  int kl = (int)floorf((sc - hw - A.rl0) * A.rl_inv_h) - 1;
  int kh = (int)ceilf((sc + hw - A.rl0) * A.rl_inv_h) + 1;
  kl = kl < 0 ? 0 : (kl > A.nrl - 1 ? A.nrl - 1 : kl);
  kh = kh < 0 ? 0 : (kh > A.nrl - 1 ? A.nrl - 1 : kh);
  jlo = A.rlut[kl].x;
  jhi = A.rlut[kh].y;
}

// Radial grid of a gather launch: known at compile time for single-job launches
// (uniform, or the lookup table), read from the arguments otherwise.
enum GatherGrid { kGridAny = 0, kGridUniform = 1, kGridLut = 2 };

template <int GRID>
__device__ __forceinline__ bool grid_lut(const GatherArgs& A) {
  return GRID == kGridLut || (GRID == kGridAny && A.rlut != nullptr);
}

// Candidate bins of angle a for a voxel column centred at (xc, yc): the bins whose
// LOR passes within the column's half-width (plus the float margin) of its centre.
// Even bins (lo0, hi0) and odd bins (lo1, hi1) get their own range; on the plan's
// uniform grid, where every bin of an angle shares it, the two ranges are equal.
template <int GRID>
__device__ __forceinline__ void candidate_bins(const GatherArgs& A, int a, float xc, float yc,
                                               float inv_dr, int& lo0, int& hi0, int& lo1,
                                               int& hi1) {
  const Geo& g = A.g;
  const float2 cs = A.angcs[a];
  const float sc = xc * cs.x + yc * cs.y;
  const float hw = 0.5f * g.dx * (fabsf(cs.x) + fabsf(cs.y)) + g.rmargin;
  if (!grid_lut<GRID>(A)) {
    int jlo = (int)ceilf((sc - hw - g.r0) * inv_dr);
    int jhi = (int)floorf((sc + hw - g.r0) * inv_dr);
    lo0 = lo1 = jlo < 0 ? 0 : jlo;
    hi0 = hi1 = jhi > g.nr - 1 ? g.nr - 1 : jhi;
    return;
  }
  lut_bins(A, sc, hw, lo0, hi0);
  const float2 co = A.angcs_odd[a];
  const float so = xc * co.x + yc * co.y;
  const float hwo = 0.5f * g.dx * (fabsf(co.x) + fabsf(co.y)) + g.rmargin;
  lut_bins(A, so, hwo, lo1, hi1);
}

// Bin rr is a candidate of its parity's range.
__device__ __forceinline__ bool in_parity_range(int rr, int lo0, int hi0, int lo1, int hi1) {
  return (rr & 1) ? (rr >= lo1 && rr <= hi1) : (rr >= lo0 && rr <= hi0);
}

// The sums start from zero instead of the image.  GatherArgs::fresh and upd_thr_at are the
// reference arithmetic's only: the column kernel holds its arguments in scalar registers, which
// it spills, and with these it took the other precisions 5.9 ms instead of 5.4 (12 angles of
// 344 x 837 bins into 256 x 256 x 81).
template <int PREC>
__device__ __forceinline__ bool sums_from_zero(const GatherArgs& A) {
  return PREC == APIRL_PREC_REFERENCE ? A.fresh != 0 : A.upd_sens != nullptr;
}

// A voxel's backprojection b: stored (forcePositive applied if asked for), or with the fused EM
// update (MlemSinogram3d.cpp:228-242, OsemSinogram3d.cpp:217-237, Mlem2d.cpp:171-185) applied
// to the image voxel it belongs to, as em_update_kernel computes it.
template <int PREC>
__device__ __forceinline__ void store_voxel(const GatherArgs& A, long v, float b) {
  constexpr bool kRef = PREC == APIRL_PREC_REFERENCE;
  if (!A.upd_sens) {
    A.img[v] = kRef && A.fresh == kFreshPositive && b < 0.f ? 0.f : b;  // Images.cpp:383-395
    return;
  }
  const float sv = A.upd_sens[v];
  const float thr = kRef && A.upd_thr_at ? *A.upd_thr_at : A.upd_thr;
  const bool ok = A.upd_strict ? (sv > thr) : (sv >= thr);
  A.img[v] = ok ? A.img[v] * b / sv : 0.f;
}

// alpha at which a ray leaves a column entered at lo, whose next x or y crossing is next: its list
// ends by amax, except that of an LOR that misses the image's square (lo > amax), which runs on.
__device__ __forceinline__ float column_exit(float amax, float lo, float next) {
  return amax < lo ? next : fminf(amax, next);
}

// Gather of one voxel (i, j, k): adds its terms to A.img[v] in the fixed order
// (angle, radial bin, segment, sinogram).  s_zab is the axial table in LDS (3D).
template <int DIMS, int PREC>
__device__ __forceinline__ void gather_voxel(const GatherArgs& A, const float2* s_zab, int i,
                                             int j, int k) {
  const Geo& g = A.g;
  const int* s_soff = (const int*)(s_zab + g.nsino);  // slot offsets follow the axial table
  const int* s_kmin = s_soff + g.nsino + 1;           // then the slots' first slices
  const long v = ((long)k * g.ny + j) * g.nx + i;
  // voxel centre for the candidate search
  const float xc = -g.R + g.dx * ((float)i + 0.5f);
  const float yc = -g.R + g.dy * ((float)j + 0.5f);
  const float zk0 = g.offz + k * g.dz, zk1 = zk0 + g.dz;
  const float inv_dr = 1.0f / g.dr;
  // Accumulator: float in the reference order (REFERENCE), float with a Kahan
  // compensation term (KAHAN), or double (F64_ALPHA).
  Acc<PREC> acc;
  acc.init(sums_from_zero<PREC>(A) ? 0.f : A.img[v]);
  for (int ka = 0; ka < A.nang_sub; ka++) {
    const int a = A.subset + A.nsubsets * ka;
    int lo0, hi0, lo1, hi1;
    candidate_bins<kGridAny>(A, a, xc, yc, inv_dr, lo0, hi0, lo1, hi1);
    const int jlo = lo0 < lo1 ? lo0 : lo1, jhi = hi0 > hi1 ? hi0 : hi1;
    for (int rr = jlo; rr <= jhi; rr++) {
      if (A.rlut && !in_parity_range(rr, lo0, hi0, lo1, hi1)) continue;
      if (DIMS == 3 && A.nz_pair[(long)ka * g.nr + rr] == 0) continue;
      const RayXY t = A.rays[(long)a * g.nr + rr];
      if (!(t.flags & RAY_VALID)) continue;
      const int iinc = ray_iinc(t.flags), jinc = ray_jinc(t.flags);
      // Entry voxel, transaxial list length and alpha range of the ray: the
      // reference's float setup from the ray table, or (F64_ALPHA, 3D) the same
      // setup carried out in double (siddon_f64.h).
      using R = typename Acc<PREC>::alpha_t;
      constexpr bool kF64Setup =
          (PREC == APIRL_PREC_F64_ALPHA || PREC == APIRL_PREC_F64_SETUP) && DIMS == 3;
      // crossings from the (double) setup by repeated addition rather than the plan's
      // float-setup tables
      constexpr bool kOwnCrossings = PREC == APIRL_PREC_F64_ALPHA || kF64Setup;
      int ti0 = t.i0, tj0 = t.j0, tnxy = t.nxy;
      R tamin = t.amin, tamax = t.amax;
      R ax0, axu, ay0, ayu;
      SetupXY64 xy;
      if (kF64Setup) {
        setup_xy_f64(g, t.p0x, t.p0y, t.vx, t.vy, xy);
        ti0 = xy.i0;
        tj0 = xy.j0;
        tnxy = abs(xy.i1 - xy.i0) + abs(xy.j1 - xy.j0);
        tamin = (R)xy.amin;
        tamax = (R)xy.amax;
        ax0 = (R)xy.ax;
        axu = (R)xy.axu;
        ay0 = (R)xy.ay;
        ayu = (R)xy.ayu;
      } else {
        first_crossings<PREC, DIMS>(g, t, iinc, jinc, ax0, axu, ay0, ayu);
      }
      int na, nb;
      if (iinc == 0) {
        if (i != ti0) continue;
        na = 0;
      } else {
        na = (i - ti0) * iinc;
        if (na < 0) continue;
      }
      if (jinc == 0) {
        if (j != tj0) continue;
        nb = 0;
      } else {
        nb = (j - tj0) * jinc;
        if (nb < 0) continue;
      }
      if (na + nb >= tnxy + (DIMS == 3 ? g.nz + 1 : 0)) continue;
      // x / y crossings around the column: the float accumulators of the reference
      // loop reconstructed exactly, or (F64_ALPHA) the crossings in double
      R Xp = -FLT_MAX, Xn, Yp = -FLT_MAX, Yn;
      Xn = ax0;
      Yn = ay0;
      if (kOwnCrossings) {
        if (na > 0) {
          Xp = crossing<PREC>(ax0, axu, na - 1);
          Xn = Xp + axu;
        }
        if (nb > 0) {
          Yp = crossing<PREC>(ay0, ayu, nb - 1);
          Yn = Yp + ayu;
        }
      } else {
        // the accumulated crossings by which the ray enters column i and row j
        // (plan-level table, written by repeated float addition)
        const float* xy = A.xytab + ((long)a * g.nr + rr) * (g.nx + g.ny);
        if (na > 0) {
          Xp = xy[i];
          Xn = Xp + axu;
        }
        if (nb > 0) {
          Yp = xy[g.nx + j];
          Yn = Yp + ayu;
        }
      }
      // taken x before untaken y (x wins ties), taken y before untaken x (strict)
      if (na > 0 && !(Xp <= Yn)) continue;
      if (nb > 0 && !(Yp < Xn)) continue;
      if (DIMS == 2) {
        const int m = na + nb;
        if (m >= tnxy) continue;
        R ac = tamin;
        if (m > 0) ac = Xp > Yp ? Xp : Yp;
        const R an = Xn < Yn ? Xn : Yn;
        float b = 1.f;
        if (A.kind == BP_PLAIN) b = A.sino[(long)ka * g.nr + rr];
        else if (A.kind == BP_MULT) b = A.sino[(long)a * g.nr + rr];
        if (PREC == APIRL_PREC_F64_ALPHA) {
          acc.add_f64((an - ac) * sqrt((double)t.vx * t.vx + (double)t.vy * t.vy) * b);
        } else {
          const float w = (float)(an - ac) * sqrtf(t.lxy);
          acc.add(w * b * 1.0f);  // SiddonProjector.cpp:72
        }
        continue;
      }
      // alpha interval of the column; the sinograms whose ray crosses the slab
      // [zk0, zk1] inside it form a contiguous run of each segment (the mean ring
      // coordinates grow with the index), found by a short scan from an estimate.
      const float lo = fmaxf((float)tamin, fmaxf((float)Xp, (float)Yp));
      const float hi = column_exit((float)tamax, lo, fminf((float)Xn, (float)Yn));
      const float amid = 0.5f * (lo + hi) - 0.5f;
      const float zlo_t = zk0 - kZMargin, zhi_t = zk1 + kZMargin;
      for (int sg = 0; sg < A.nseg; sg++) {
        const GatherSeg S = A.segs[sg];
        int sl = (int)floorf((0.5f * (zk0 + zk1) - amid * S.dlo - S.z0) * S.dhi + 0.5f);
        sl = sl < 0 ? 0 : (sl > S.count - 1 ? S.count - 1 : sl);
        // first sinogram whose ray reaches the slab's lower face
        while (sl > 0) {
          const float2 z = s_zab[S.first + sl - 1];
          const float vz = z.y - z.x;
          if (fmaxf(z.x + vz * lo, z.x + vz * hi) < zlo_t) break;
          sl--;
        }
        for (; sl < S.count; sl++) {
          const int s = S.first + sl;
          const float2 zz = s_zab[s];
          const float vzz = zz.y - zz.x;
          const float za_lo = z_at(zz.x, vzz, lo), za_hi = z_at(zz.x, vzz, hi);
          if (fmaxf(za_lo, za_hi) < zlo_t) continue;
          if (fminf(za_lo, za_hi) > zhi_t) break;
          const ZRay z = A.zr[((long)s * A.nang_sub + ka) * g.nr + rr];
          // the table entry for this slice, loaded alongside the record (its address
          // does not depend on it); used only when the ray enters the slice by a z
          // crossing of its own, which makes it the entry zsetup wrote
          float ztv = 0.f;
          if (!kOwnCrossings && A.ztab) {
            const int slot = s_soff[s + 1] - s_soff[s];
            int kk = k - s_kmin[s];
            kk = kk < 0 ? 0 : (kk >= slot ? slot - 1 : kk);
            ztv = A.ztab[((long)(s_soff[s] + kk) * A.nang_sub + ka) * g.nr + rr];
          }
          if (z.b == 0.f) continue;  // SiddonProjector.cpp:496
          int zk0 = z.k0, zk1 = z.k1, zkinc = z.kinc;
          R az0, azu;
          double Ld = 0.0;
          float Lf = z.L;
          if (kF64Setup) {
            SetupZ64 zs;
            setup_z_f64(g, xy, zz.x, t.vx, t.vy, (double)(zz.y - zz.x), zs);
            zk0 = zs.k0;
            zk1 = zs.k1;
            zkinc = zs.kinc;
            az0 = (R)zs.az;
            azu = (R)zs.azu;
            Ld = zs.L;
            Lf = (float)zs.L;
          } else {
            z_crossings<PREC>(g, z, zz, az0, azu);
          }
          int nc;
          if (zkinc == 0) {
            if (k != zk0) continue;
            nc = 0;
          } else {
            nc = (k - zk0) * zkinc;
            if (nc < 0) continue;
          }
          const int m = na + nb + nc;
          if (m >= tnxy + abs(zk1 - zk0)) continue;
          R Zp = -FLT_MAX, Zn = az0;
          if (nc > 0) {
            if (kOwnCrossings) {
              Zp = crossing<PREC>(az0, azu, nc - 1);
            } else {
              Zp = nc <= z.zcount ? ztv : crossing<PREC>(az0, azu, nc - 1);
            }
            Zn = Zp + azu;
          }
          // cross-axis order (x before y before z on ties)
          if (na > 0 && !(Xp <= Zn)) continue;
          if (nb > 0 && !(Yp <= Zn)) continue;
          if (nc > 0 && !(Zp < Xn && Zp < Yn)) continue;
          R ac = tamin;
          if (m > 0) {
            ac = Xp > Yp ? Xp : Yp;
            ac = ac > Zp ? ac : Zp;
          }
          R an = Xn < Yn ? Xn : Yn;
          an = an < Zn ? an : Zn;
          if (PREC == APIRL_PREC_F64_ALPHA) {
            acc.add_f64((an - ac) * Ld * z.b);
          } else {
            const float w = (float)(an - ac) * Lf;
            acc.add(w * 1.0f * z.b);  // SiddonProjector.cpp:546
          }
        }
      }
    }
  }
  store_voxel<PREC>(A, v, acc.value());
}

// One 32-byte record as two 16-byte loads.
__device__ __forceinline__ ZRay load_zray(const ZRay* p) {
  const int4* q = reinterpret_cast<const int4*>(p);
  const int4 a = q[0], b = q[1];
  ZRay z;
  z.k0 = a.x;
  z.k1 = (short)(a.y & 0xffff);
  z.kinc = (short)(a.y >> 16);
  z.azu = __int_as_float(a.z);
  z.az0 = __int_as_float(a.w);
  z.L = __int_as_float(b.x);
  z.b = __int_as_float(b.y);
  z.zcount = b.z;
  z.pad = b.w;
  return z;
}

// LDS of the column kernel: the axial table (float2 per sinogram), per sinogram where
// slice k's crossing-table entry lives (entry index clamp(k + x, y, z) with x = slot
// start - first slice, [y, z] = the slot's entries; int4, 16-byte aligned), and the
// segments' sinogram runs (read once per candidate ray and segment: from LDS rather
// than by scalar loads, 2.53 -> 2.48 ms per C2 subset).
__host__ __device__ inline size_t column_lds_off(int nsino) { return ((size_t)nsino * sizeof(float2) + 15) / 16 * 16; }
inline size_t column_lds_bytes(int nsino, int nseg = 0) {
  return column_lds_off(nsino) + (size_t)nsino * sizeof(int4) + (size_t)nseg * sizeof(GatherSeg);
}

// 3D gather of ZV voxels of one column, (i, j, kb) .. (i, j, kb + ZV - 1), by one lane
// (float precision modes).  Each voxel receives exactly the terms gather_voxel gives
// it, in the same order (angle, radial bin, segment, sinogram): the voxels share the
// transaxial part of every candidate ray (its column tests and x / y crossings) and
// one scan of each segment's sinograms over the union of their slabs.  Inside the
// scan, each sinogram is tested against each voxel's own slab exactly as
// gather_voxel tests it.  Record and table addresses are formed from a per-(angle,
// radial bin) base and 32-bit offsets s npair and e npair, formed with 24-bit
// multiplies: gather_fits admits a subset only when its records number below 2^31,
// the z-table offsets stay below 2^32 (the table is held under 1 GiB) and
// npair, the sinograms and the table slots stay below 2^24, which makes both exact.
template <int PREC, int ZV, int GRID = kGridAny>
__device__ __forceinline__ void gather_column(const GatherArgs& A, const float2* s_zab,
                                              const int4* s_slot, const GatherSeg* segs, int i,
                                              int j, int kb) {
  static_assert(PREC != APIRL_PREC_F64_ALPHA && PREC != APIRL_PREC_F64_SETUP,
                "double-precision setup uses gather_voxel");
  const Geo& g = A.g;
  const int nk = g.nz - kb < ZV ? g.nz - kb : ZV;  // voxels of this column segment (>= 1)
  const long nxy = (long)g.nx * g.ny;
  const long v0 = ((long)kb * g.ny + j) * g.nx + i;
  const float xc = -g.R + g.dx * ((float)i + 0.5f);
  const float yc = -g.R + g.dy * ((float)j + 0.5f);
  const float inv_dr = 1.0f / g.dr;
  const unsigned npair = (unsigned)A.nang_sub * (unsigned)g.nr;
  // each voxel's slab and search bounds, as gather_voxel computes them
  float zlo_t[ZV], zhi_t[ZV];
  Acc<PREC> acc[ZV];
#pragma unroll
  for (int q = 0; q < ZV; q++) {
    const int k = kb + q;
    const float zk0 = g.offz + k * g.dz, zk1 = zk0 + g.dz;
    zlo_t[q] = zk0 - kZMargin;
    zhi_t[q] = zk1 + kZMargin;
    acc[q].init(q < nk && !sums_from_zero<PREC>(A) ? A.img[v0 + q * nxy] : 0.f);
  }
  const float zlo_all = zlo_t[0];
  float zhi_all = zhi_t[0];
#pragma unroll
  for (int q = 1; q < ZV; q++)
    if (q < nk) zhi_all = zhi_t[q];
  const float zmid_all = 0.5f * (zlo_all + zhi_all);
  for (int ka = 0; ka < A.nang_sub; ka++) {
    const int a = A.subset + A.nsubsets * ka;
    int lo0, hi0, lo1, hi1;
    candidate_bins<GRID>(A, a, xc, yc, inv_dr, lo0, hi0, lo1, hi1);
    const int jlo = lo0 < lo1 ? lo0 : lo1, jhi = hi0 > hi1 ? hi0 : hi1;
    for (int rr = jlo; rr <= jhi; rr++) {
      if (grid_lut<GRID>(A) && !in_parity_range(rr, lo0, hi0, lo1, hi1)) continue;
      const unsigned pair = (unsigned)ka * (unsigned)g.nr + (unsigned)rr;
      if (A.nz_pair[pair] == 0) continue;
      const RayXY t = A.rays[(long)a * g.nr + rr];
      const float* xy = A.xytab + ((long)a * g.nr + rr) * (g.nx + g.ny);
      // entry crossings of column i and row j (table entries exist for every i, j, so
      // they are loaded before the tests that decide whether they are used)
      const float xyi = xy[i], xyj = xy[g.nx + j];
      const int iinc = ray_iinc(t.flags), jinc = ray_jinc(t.flags);
      const int tnxy = t.nxy;
      const float tamin = t.amin, tamax = t.amax;
      float ax0, axu, ay0, ayu;
      first_crossings<PREC, 3>(g, t, iinc, jinc, ax0, axu, ay0, ayu);
      // the transaxial tests of gather_voxel as one predicate
      // crossings already taken in x and y (increments are -1, 0 or 1: a 24-bit
      // multiply is exact and full rate)
      const int na = __mul24(i - t.i0, iinc), nb = __mul24(j - t.j0, jinc);
      // (iinc == 0 ? i == i0 : na >= 0) and the same for j, as lane-mask operations
      bool okt = (t.flags & RAY_VALID) != 0;
      okt &= (i == t.i0) | ((iinc != 0) & (na >= 0));
      okt &= (j == t.j0) | ((jinc != 0) & (nb >= 0));
      okt &= na + nb < tnxy + g.nz + 1;
      const float Xp = na > 0 ? xyi : -FLT_MAX, Xn = na > 0 ? xyi + axu : ax0;
      const float Yp = nb > 0 ? xyj : -FLT_MAX, Yn = nb > 0 ? xyj + ayu : ay0;
      okt &= ((na <= 0) | (Xp <= Yn)) & ((nb <= 0) | (Yp < Xn));
      if (!okt) continue;
      const float lo = fmaxf(tamin, fmaxf(Xp, Yp));
      const float hi = column_exit(tamax, lo, fminf(Xn, Yn));
      const float amid = 0.5f * (lo + hi) - 0.5f;
      const ZRay* zr_pair = A.zr + pair;            // record of sinogram s: [s * npair]
      const float* zt_pair = A.ztab ? A.ztab + pair : nullptr;  // entry e: [e * npair]
      for (int sg = 0; sg < A.nseg; sg++) {
        const GatherSeg S = segs[sg];
        int sl = (int)floorf((zmid_all - amid * S.dlo - S.z0) * S.dhi + 0.5f);
        sl = sl < 0 ? 0 : (sl > S.count - 1 ? S.count - 1 : sl);
        while (sl > 0) {
          const float2 z = s_zab[S.first + sl - 1];
          const float vz = z.y - z.x;
          if (fmaxf(z.x + vz * lo, z.x + vz * hi) < zlo_all) break;
          sl--;
        }
        for (; sl < S.count; sl++) {
          const int s = S.first + sl;
          const float2 zz = s_zab[s];
          const float vzz = zz.y - zz.x;
          const float za_lo = z_at(zz.x, vzz, lo), za_hi = z_at(zz.x, vzz, hi);
          const float zmax = fmaxf(za_lo, za_hi), zmin = fminf(za_lo, za_hi);
          if (zmax < zlo_all) continue;
          if (zmin > zhi_all) break;
          const ZRay z = load_zray(zr_pair + __umul24((unsigned)s, npair));
          // the table entry of each slice this sinogram can reach, loaded alongside the
          // record (its address does not depend on it) and used only when the ray
          // enters that slice by a z crossing of its own, which makes it an entry
          // zsetup wrote
          float ztv[ZV];
          bool hit[ZV];
#pragma unroll
          for (int q = 0; q < ZV; q++) {
            hit[q] = (q < nk) & !(zmax < zlo_t[q]) & !(zmin > zhi_t[q]);
            ztv[q] = 0.f;
          }
          if (zt_pair) {
            const int4 sl4 = s_slot[s];
#pragma unroll
            for (int q = 0; q < ZV; q++) {
              int e = kb + q + sl4.x;
              e = e < sl4.y ? sl4.y : (e > sl4.z ? sl4.z : e);
              if (hit[q]) ztv[q] = zt_pair[__umul24((unsigned)e, npair)];
            }
          }
          if (z.b == 0.f) continue;  // SiddonProjector.cpp:496
          const float az0 = z.az0, azu = z.azu;
          const int zk0r = z.k0, zkinc = z.kinc, zn = abs((int)z.k1 - z.k0);
#pragma unroll
          for (int q = 0; q < ZV; q++) {
            if (!hit[q]) continue;
            // the tests of gather_voxel, evaluated as one predicate (selects, not
            // branches); the term is added only when all hold
            const int k = kb + q;
            const int nc = __mul24(k - zk0r, zkinc);
            // (zkinc == 0 ? k == zk0r : nc >= 0), as lane-mask operations
            bool ok = (k == zk0r) | ((zkinc != 0) & (nc >= 0));
            const int m = na + nb + nc;
            ok &= m < tnxy + zn;
            if (!ok) continue;  // whole wavefronts often fail the count tests
            const bool hz = nc > 0;
            float Zt = ztv[q];
            if (ok & hz & !(zt_pair && nc <= z.zcount)) Zt = crossing<PREC>(az0, azu, nc - 1);
            const float Zp = hz ? Zt : -FLT_MAX;
            const float Zn = hz ? Zt + azu : az0;
            ok &= ((na <= 0) | (Xp <= Zn)) & ((nb <= 0) | (Yp <= Zn)) &
                  (!hz | ((Zp < Xn) & (Zp < Yn)));
            float ac = Xp > Yp ? Xp : Yp;
            ac = ac > Zp ? ac : Zp;
            ac = m > 0 ? ac : tamin;
            float an = Xn < Yn ? Xn : Yn;
            an = an < Zn ? an : Zn;
            const float w = (an - ac) * z.L;
            acc[q].add_if(ok, w * 1.0f * z.b);  // SiddonProjector.cpp:546
          }
        }
      }
    }
  }
#pragma unroll
  for (int q = 0; q < ZV; q++)
    if (q < nk) store_voxel<PREC>(A, v0 + q * nxy, acc[q].value());
}

// Eight waves per SIMD for up to three voxels per lane: the kernel waits mostly on
// its record and table loads, and the two extra waves hide more of that latency than
// the few registers spilled at 64 VGPRs cost (3.29 -> 3.03 ms per C2 subset).
template <int PREC, int ZV, int GRID>
__global__ __launch_bounds__(kGBlock, ZV <= 3 ? 8 : 6) void gather_column_kernel(GatherArgs A) {
  extern __shared__ float2 s_zab[];
  const Geo& g = A.g;
  int4* s_slot = (int4*)((char*)s_zab + column_lds_off(g.nsino));
  GatherSeg* s_seg = (GatherSeg*)(s_slot + g.nsino);
  for (int q = threadIdx.x; q < g.nsino; q += kGBlock) {
    s_zab[q] = A.zab[q];
    if (A.zsoff) {
      const int so = A.zsoff[q], so1 = A.zsoff[q + 1], km = A.zsoff[g.nsino + 1 + q];
      s_slot[q] = make_int4(so - km, so, so1 - 1 < so ? so : so1 - 1, 0);
    }
  }
  for (int q = threadIdx.x; q < A.nseg; q += kGBlock) s_seg[q] = A.segs[q];
  __syncthreads();
  // a workgroup is a 16 x 16 tile of columns, ZV slices deep: the grid's own tile, or
  // the one the tile map gives this slot
  int tx = blockIdx.x, ty = blockIdx.y, tz = blockIdx.z;
  if (A.tile_map) {
    const int t = A.tile_map[blockIdx.x];
    if (t < 0) return;
    const int ntx = (g.nx + kTile - 1) / kTile, nty = (g.ny + kTile - 1) / kTile;
    tx = t % ntx;
    ty = (t / ntx) % nty;
    tz = t / (ntx * nty);
  }
  const int i = tx * kTile + (threadIdx.x % kTile);
  const int j = ty * kTile + (threadIdx.x / kTile);
  const int kb = tz * ZV;
  if (i >= g.nx || j >= g.ny || kb >= g.nz) return;
  gather_column<PREC, ZV, GRID>(A, s_zab, s_slot, s_seg, i, j, kb);
}

template <int DIMS, int PREC>
__global__ __launch_bounds__(kGBlock) void gather_kernel(GatherArgs A) {
  extern __shared__ float2 s_zab[];  // (P1.Z, P2.Z) of every sinogram
  const Geo& g = A.g;
  if (DIMS == 3) {
    int* s_soff = (int*)(s_zab + g.nsino);
    for (int q = threadIdx.x; q < g.nsino; q += kGBlock) s_zab[q] = A.zab[q];
    if (A.zsoff)
      for (int q = threadIdx.x; q <= 2 * g.nsino; q += kGBlock) s_soff[q] = A.zsoff[q];
    __syncthreads();
  }
  // Voxel of this lane.
  //   zlanes <= 1: a workgroup is a 16 x 16 tile of one slice (grid nx/16, ny/16, nz).
  //   zlanes = Z > 1: a wavefront holds 64 / Z voxel columns (neighbours along x) times
  //     Z consecutive slices; every lane of a column shares the column's candidate
  //     rays, so the transaxial tests agree across those lanes and only the axial
  //     part differs.  1D grid; workgroups are remapped so that each XCD takes one
  //     contiguous run of columns (round-robin dispatch puts block b on XCD b % 8).
  int i, j, k;
  if (A.zlanes <= 1) {
    i = blockIdx.x * kTile + (threadIdx.x % kTile);
    j = blockIdx.y * kTile + (threadIdx.x / kTile);
    k = blockIdx.z;
    if (i >= g.nx || j >= g.ny) return;
  } else {
    const unsigned nb = gridDim.x, b = blockIdx.x;
    const unsigned xcd = b % 8, per = nb / 8, rem = nb % 8;
    const unsigned lb = xcd * per + (xcd < rem ? xcd : rem) + b / 8;
    const int Z = A.zlanes, C = kWave / Z;
    const int nch = (g.nz + Z - 1) / Z;
    const long wave = ((long)lb * kGBlock + threadIdx.x) / kWave;
    const int lane = threadIdx.x % kWave;
    const int c = lane / Z, kk = lane % Z;
    const long q = (wave / nch) * C + c;
    k = (int)(wave % nch) * Z + kk;
    if (c >= C || k >= g.nz || q >= (long)g.nx * g.ny) return;
    i = (int)(q % g.nx);
    j = (int)(q / g.nx);
  }
  gather_voxel<DIMS, PREC>(A, s_zab, i, j, k);
}

// ---- 2D gather, reference arithmetic ------------------------------------------------
//
// A workgroup takes a patch of P x P voxels.  Its first nw wavefronts walk the rays of a few
// angles each per round, one ray per lane, through the patch, and write each voxel's term to the
// LDS slot of the ray's rank among the voxel's candidate bins (a slot no ray writes holds 0);
// the next wavefront, a voxel per lane, adds the terms of the round before in the reference's
// order (angle, radial bin).  The sums are gather_kernel's, bit for bit.
//
// gather_kernel (one lane per voxel, its angles in turn) waits for its loads with too few
// wavefronts (256 for 128 x 128: 569 us from 192 x 192 bins).  One voxel per lane and an angle
// per wavefront, its rays staged in LDS, is VALU-bound: 570 instructions an angle and patch,
// most for bins that miss the voxel (48 us).  A ray's steps through an 8 x 8 patch are 15 at the
// most, 23 instructions each, for 3 angles at a time there.  Calls, 17 us of host work
// included, voxel per lane -> ray per lane: 128 x 128 from 192 x 192 50 -> 33 us, from 252 x 344
// 118 -> 61; 64 x 64 from 192 x 192 108 -> 29; 32 x 32 from 252 x 344 1575 -> 82; 512 x 512 from
// 252 x 344 381 -> 212.
constexpr int kG2Waves = 16;                  // wavefronts of the workgroup, one of them sums
constexpr int kG2LdsFloats = 16 * 1024 - 64;  // a grouped launch's two rounds of terms: 64 KiB
                                              // less the batch's block number

struct G2Plan {
  int slots;   // of a voxel and angle: its candidates and one more (a rank is rounded down)
  int rays;    // of an angle, that can cross a patch (64: or more)
  int angles;  // of a wavefront's round
  int nw;      // wavefronts that walk; 0: one angle's terms do not fit
};
// The half-width of a patch's bins: its own, a hundredth of a bin and 2 um more than its voxels'
// own ranges, whose rounding is far below that.
template <int P>
__host__ __device__ inline float gather2_half(const Geo& g, float c, float s) {
  return 0.5f * P * (g.dx * c + g.dy * s) + 0.5f * fabsf(g.dx - g.dy) + g.rmargin + 0.01f * g.dr +
         2e-3f;
}
template <int P>
__host__ __device__ inline G2Plan gather2_plan(const Geo& g, int maxc, int nang_sub,
                                               int lds_floats) {
  G2Plan q;
  q.slots = (maxc > 0 ? maxc : 1) + 1;
  const float r = 2.f * gather2_half<P>(g, 0.7072f, 0.7072f) / g.dr + 2.f;  // widest: 45 degrees
  q.rays = r < (float)kWave ? (int)r : kWave;
  q.angles = kWave / q.rays;
  const int fit = lds_floats / (2 * q.angles * q.slots * P * P);
  const int need = (nang_sub + q.angles - 1) / q.angles;
  q.nw = fit < kG2Waves - 1 ? fit : kG2Waves - 1;
  q.nw = q.nw < need ? q.nw : need;
  return q;
}
template <int P>
inline size_t gather2_lds(const G2Plan& q) {
  return (size_t)q.nw * 2 * q.angles * q.slots * P * P * sizeof(float);
}

// Orders a wavefront's LDS accesses before and after this point (lanes read what
// other lanes of the wavefront wrote).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The terms of angles ka0 .. ka0 + q.angles - 1 for the voxels of patch (px, py), to
// T[((angle * q.slots) + rank) * P * P + voxel].
template <int P>
__device__ __forceinline__ void gather2_terms(const GatherArgs& A, const G2Plan& q, int ka0, int px,
                                              int py, float inv_dr, int al, int rl, float* T) {
  const Geo& g = A.g;
  const int lane = threadIdx.x & (kWave - 1);
  for (int c = lane * 4; c < q.angles * q.slots * P * P; c += kWave * 4)
    *reinterpret_cast<float4*>(T + c) = make_float4(0.f, 0.f, 0.f, 0.f);
  wave_lds_sync();
  const int ka = ka0 + al;
  if (al >= q.angles || ka >= A.nang_sub) return;
  const int a = A.subset + A.nsubsets * ka, ci0 = px * P, cj0 = py * P;
  const float2 cs = A.angcs[a];
  // the patch's bins
  const float sp = (-g.R + g.dx * (float)(ci0 + P / 2)) * cs.x +
                   (-g.R + g.dy * (float)(cj0 + P / 2)) * cs.y;
  const float hp = gather2_half<P>(g, fabsf(cs.x), fabsf(cs.y));
  int p0 = (int)ceilf((sp - hp - g.r0) * inv_dr), p1 = (int)floorf((sp + hp - g.r0) * inv_dr);
  p0 = p0 < 0 ? 0 : p0;
  p1 = p1 > g.nr - 1 ? g.nr - 1 : p1;
  // a voxel's first candidate is the bin at or after t0 + i tx + j ty (candidate_bins; a
  // thousandth of a bin early for the rounding here).  In 2^-16 bins, from bin p0: whole
  // numbers, so a voxel's is the same whatever the path to it.
  const float hw = 0.5f * (g.dx * fabsf(cs.x) + g.dy * fabsf(cs.y)) + g.rmargin;
  const int tx = (int)rintf(g.dx * cs.x * inv_dr * 65536.f);
  const int ty = (int)rintf(g.dy * cs.y * inv_dr * 65536.f);
  const float t0 = ((-g.R + g.dx * ((float)ci0 + 0.5f)) * cs.x +
                    (-g.R + g.dy * ((float)cj0 + 0.5f)) * cs.y - hw - g.r0) * inv_dr - 1e-3f;
  const int u0 = (int)((float)p0 * 65536.f - t0 * 65536.f);
  const int ci1 = ci0 + P - 1 < g.nx ? ci0 + P - 1 : g.nx - 1;
  const int cj1 = cj0 + P - 1 < g.ny ? cj0 + P - 1 : g.ny - 1;
  // byte addresses in LDS: a rank's terms are kSlot bytes, so that a rank in 2^-16 ranks, shifted
  // and its fraction replaced by the voxel's offset, is the term's address
  constexpr int kSlot = P * P * 4, kShift = 16 - (P == 8 ? 8 : 6);
  constexpr int kRow = 2 * P;  // (row, column) as one number, a guard bit above each
  constexpr unsigned kGuards = ~(unsigned)((P - 1) | (P - 1) * kRow | 63 << 16);
  typedef __attribute__((address_space(3))) char* lds_bytes;
  typedef __attribute__((address_space(3))) float* lds_float;
  const int slot0 = (int)(unsigned)(uintptr_t)(lds_bytes)(char*)(T + al * q.slots * P * P) / kSlot;
  const int ulo = slot0 << 16, uhi = ulo + (q.slots << 16) - 1;
  for (int rr = p0 + rl; rr <= p1; rr += q.rays) {
    const float b = A.kind == BP_PLAIN ? A.sino[(long)ka * g.nr + rr]
                                       : (A.kind == BP_MULT ? A.sino[(long)a * g.nr + rr] : 1.f);
    if (b == 0.f) continue;  // its terms are 0, as its slots are
    const float4* ray = reinterpret_cast<const float4*>(A.rays + (long)a * g.nr + rr);
    const float4 q1 = ray[1], q2 = ray[2], q3 = ray[3];
    const float amin = q1.x, ax = q1.z, ay = q1.w, axu = q2.x, ayu = q2.y, len = q3.w;
    const int i0 = __float_as_int(q2.w), j0 = __float_as_int(q3.x);
    const int nxy = __float_as_int(q3.y), flags = __float_as_int(q3.z);
    const int iinc = ray_iinc(flags), jinc = ray_jinc(flags);
    // the columns and rows the ray has to come to first, and the steps to them
    const int ic = iinc > 0 ? (i0 > ci0 ? i0 : ci0) : (i0 < ci1 ? i0 : ci1);
    const int jc = jinc > 0 ? (j0 > cj0 ? j0 : cj0) : (j0 < cj1 ? j0 : cj1);
    const int na = (ic - i0) * iinc, nb = (jc - j0) * jinc;
    int il = ic - ci0, jl = jc - cj0;
    bool ok = (flags & RAY_VALID) != 0 && (unsigned)(il | jl) < (unsigned)P;
    ok &= (iinc != 0) | (ic == i0);
    ok &= (jinc != 0) | (jc == j0);
    if (!ok) continue;
    const float* xytab = A.xytab + ((long)a * g.nr + rr) * (g.nx + g.ny);
    const float Xi = na > 0 ? xytab[ic] : -FLT_MAX, Yi = nb > 0 ? xytab[g.nx + jc] : -FLT_MAX;
    float X = na > 0 ? Xi + axu : ax, Y = nb > 0 ? Yi + ayu : ay;
    // rows, columns and the steps left in the list (of 64) in one number, whose guard bits say
    // when one runs out; the term's rank; the voxel's offset
    int left = nxy - na - nb;
    left = left < 0 ? 0 : (left > 63 ? 63 : left);
    int at = il + jl * kRow + ((64 - left) << 16);
    int u = u0 + ((rr - p0) << 16) + ulo - il * tx - jl * ty;
    int off = (jl * P + il) * 4;
    const int atx = iinc + (1 << 16), aty = jinc * kRow + (1 << 16);
    const int ux = -iinc * tx, uy = -jinc * ty, ox = iinc * 4, oy = jinc * P * 4;
    // the later of the two crossings enters the patch; the other chain's crossings before it
    // (x first on ties) are taken first
    float ac = Xi > Yi ? Xi : Yi;
    if (na + nb == 0) {
      ac = amin;
    } else if (Xi > Yi) {
      while (Y < Xi && !(at & kGuards)) {
        Y = Y + ayu;
        at += aty;
        u += uy;
        off += oy;
      }
    } else {
      while (X <= Yi && !(at & kGuards)) {
        X = X + axu;
        at += atx;
        u += ux;
        off += ox;
      }
    }
    while (!(at & kGuards)) {
      const bool bx = X <= Y;
      const float an = bx ? X : Y;
      const float w = (an - ac) * len;
      ac = an;
      const int c = u < ulo ? ulo : (u > uhi ? uhi : u);
      *(lds_float)(lds_bytes)(uintptr_t)(unsigned)(((c >> kShift) & ~(kSlot - 1)) |
                                                   (off & (kSlot - 1))) =
          w * b * 1.0f;  // SiddonProjector.cpp:72
      const float nX = X + axu, nY = Y + ayu;
      X = bx ? nX : X;
      Y = bx ? Y : nY;
      at += bx ? atx : aty;
      u += bx ? ux : uy;
      off += bx ? ox : oy;
    }
  }
}

// Patch (px, py) by the whole workgroup (more than q.nw wavefronts, q.nw >= 1); lds:
// gather2_lds(q) bytes.
template <int P>
__device__ __forceinline__ void gather2_patch(const GatherArgs& A, const G2Plan& q, int px, int py,
                                              float* lds) {
  const Geo& g = A.g;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & (kWave - 1);
  const int mine = q.angles * q.slots * P * P, buf = q.nw * mine, round = q.nw * q.angles;
  const int rounds = (A.nang_sub + round - 1) / round;
  // the two kinds of wavefront meet at the same barriers, rounds + 1 of them
  if (wave < q.nw) {
    const float inv_dr = 1.0f / g.dr;
    const int al = lane / q.rays, rl = lane % q.rays;
    for (int it = 0; it <= rounds; it++) {
      const int ka0 = it * round + wave * q.angles;
      if (ka0 < A.nang_sub)
        gather2_terms<P>(A, q, ka0, px, py, inv_dr, al, rl, lds + (it & 1) * buf + wave * mine);
      __syncthreads();
    }
  } else {
    const int ir = px * P + lane % P, jr = py * P + lane / P;
    const bool in = wave == q.nw && lane < P * P && ir < g.nx && jr < g.ny;
    const long v = (long)jr * g.nx + ir;
    float acc = in && !A.fresh ? A.img[v] : 0.f;
    for (int it = 0; it <= rounds; it++) {
      if (it > 0 && in) {
        const float* s = lds + ((it - 1) & 1) * buf + lane;
        const int left = A.nang_sub - (it - 1) * round;
        const int n = (left < round ? left : round) * q.slots;
#pragma unroll 8
        for (int c = 0; c < n; c++) acc = acc + s[c * (P * P)];
      }
      __syncthreads();
    }
    if (in) store_voxel<APIRL_PREC_REFERENCE>(A, v, acc);
  }
}

template <int P>
__global__ __launch_bounds__(kG2Waves * kWave, 8) void gather2_kernel(GatherArgs A, G2Plan q) {
  extern __shared__ __align__(256) float g2lds[];  // a slot's alignment (gather2_terms)
  gather2_patch<P>(A, q, blockIdx.x, blockIdx.y, g2lds);
}

// ---- grouped (multi-job) launch -----------------------------------------------
#include "group_common.h"

// Each virtual block is one 8 x 8 patch of one 2D job, by the whole workgroup.
__global__ __launch_bounds__(kG2Waves * kWave, 8) void gather2_group_kernel(
    BatchHeader* __restrict__ hdr, const GJob* __restrict__ jobs) {
  extern __shared__ __align__(256) float g2lds[];  // a slot's alignment (gather2_terms)
  const int n = hdr->count[PH_GATHER2];
  const long total = hdr->total[PH_GATHER2];
  const int grab = grab_size(hdr);
  for (long v0 = first_vb(grab); v0 < total; v0 = next_vb(&hdr->next[PH_GATHER2], grab, total))
    for (long vb = v0; vb < v0 + grab && vb < total; vb++) {
      const GJob& J = jobs[find_job(jobs, n, vb)];
      const int lb = (int)(vb - J.first), px = lb % J.ntx, py = lb / J.ntx;
      const G2Plan q = gather2_plan<kPatch2>(J.A.g, J.A.maxc, J.A.nang_sub, kG2LdsFloats);
      if (q.nw > 0) {
        gather2_patch<kPatch2>(J.A, q, px, py, g2lds);
      } else if (threadIdx.x < kWave) {  // more candidates per angle than the LDS holds
        const int i = px * kPatch2 + threadIdx.x % kPatch2, j = py * kPatch2 + threadIdx.x / kPatch2;
        if (threadIdx.x < kPatch2 * kPatch2 && i < J.A.g.nx && j < J.A.g.ny)
          gather_voxel<2, APIRL_PREC_REFERENCE>(J.A, nullptr, i, j, 0);
      }
    }
}

inline unsigned ggrid(long n) { return (unsigned)((n + kGBlock - 1) / kGBlock); }

template <int PREC, int ZV>
void launch_gather_column(const GatherArgs& A, hipStream_t st) {
  const Geo& g = A.g;
  const dim3 grid = A.tile_map ? dim3((unsigned)A.tile_slots)
                               : dim3((g.nx + kTile - 1) / kTile, (g.ny + kTile - 1) / kTile,
                                      (g.nz + ZV - 1) / ZV);
  if (A.rlut)
    hipLaunchKernelGGL((gather_column_kernel<PREC, ZV, kGridLut>), grid, dim3(kGBlock),
                       column_lds_bytes(g.nsino, A.nseg), st, A);
  else
    hipLaunchKernelGGL((gather_column_kernel<PREC, ZV, kGridUniform>), grid, dim3(kGBlock),
                       column_lds_bytes(g.nsino, A.nseg), st, A);
}

template <int PREC>
void launch_gather3(const GatherArgs& A, int zlanes, int zvox, hipStream_t st) {
  const Geo& g = A.g;
  const size_t lds =
      (size_t)g.nsino * sizeof(float2) + (size_t)(2 * g.nsino + 1) * sizeof(int);
  // (the one-voxel kernel where the column kernel's tables, with their runs, exceed the LDS of a
  // workgroup: from 2700 sinograms of few runs, 1330 of runs of two)
  if (PREC != APIRL_PREC_F64_ALPHA && PREC != APIRL_PREC_F64_SETUP && zlanes <= 1 &&
      zvox >= 1 && column_lds_bytes(g.nsino, A.nseg) <= 65536) {
    constexpr int P =
        (PREC == APIRL_PREC_F64_ALPHA || PREC == APIRL_PREC_F64_SETUP) ? APIRL_PREC_REFERENCE
                                                                       : PREC;
    if (zvox == 1) launch_gather_column<P, 1>(A, st);
    else if (zvox == 2) launch_gather_column<P, 2>(A, st);
    else if (zvox == 3) launch_gather_column<P, 3>(A, st);
    else launch_gather_column<P, 4>(A, st);
    return;
  }
  if (zlanes <= 1) {
    const dim3 grid((g.nx + kTile - 1) / kTile, (g.ny + kTile - 1) / kTile, g.nz);
    hipLaunchKernelGGL((gather_kernel<3, PREC>), grid, dim3(kGBlock), lds, st, A);
    return;
  }
  const long ncol = (long)g.nx * g.ny;
  const int C = kWave / zlanes;
  const long nwaves = (ncol + C - 1) / C * ((g.nz + zlanes - 1) / zlanes);
  const long nblocks = (nwaves * kWave + kGBlock - 1) / kGBlock;
  hipLaunchKernelGGL((gather_kernel<3, PREC>), dim3((unsigned)nblocks), dim3(kGBlock), lds, st,
                     A);
}

// 4 x 4 patches for images of up to this many 8 x 8 ones, which would leave half of the CUs idle
// (8 x 8 / 4 x 4: 64 x 64 from 192 x 192 bins 68 / 31 us, 252 x 344 108 / 57; 88 x 88 48 / 38);
// from 96 x 96 on the 8 x 8 patches, whose rays' setup serves more voxels, are ahead (98 / 105 us
// there, 42 / 52 at 128 x 128).  A grouped launch, which has several images' patches, keeps 8 x 8
// (17 of 64 x 64: 2.36 / 2.59 ms).
constexpr int kG2SmallPatches = 128;

// The patches a CU gets share its LDS: more wavefronts at work on one patch while there are few
// of them (128 x 128, one a CU: 48, 64 and 96 KiB 42, 42 and 37 us), less waiting at the rounds'
// ends with several workgroups a CU (256 x 256 from 96 x 192: 32, 64 and 96 KiB 34, 39, 51 us).
constexpr int kG2MostLds = 24 * 1024;
inline int gather2_lds_floats(long patches) {
  constexpr int kCus = 256;
  const long per = (patches + kCus - 1) / kCus, share = 40 * 1024 / (per > 0 ? per : 1);
  return (int)(share > kG2MostLds ? kG2MostLds : (share < 8 * 1024 ? 8 * 1024 : share));
}

template <int P>
void launch_gather2_patches(const GatherArgs& A, hipStream_t st) {
  const Geo& g = A.g;
  const dim3 grid((g.nx + P - 1) / P, (g.ny + P - 1) / P);
  const int lds = gather2_lds_floats((long)grid.x * grid.y);
  G2Plan q = gather2_plan<P>(g, A.maxc, A.nang_sub, lds);
  if (q.nw == 0) q = gather2_plan<P>(g, A.maxc, A.nang_sub, kG2MostLds);  // gather2_fits: not 0
  hipLaunchKernelGGL(gather2_kernel<P>, grid, dim3((q.nw + 1) * kWave), gather2_lds<P>(q), st, A,
                     q);
}

// bins within a column's half-width (candidate_bins) of its centre, on a uniform grid
inline int gather2_candidates(const Geo& g) {
  return (int)std::min(1e6, std::floor((1.41421357 * std::max(g.dx, g.dy) + 2.0 * g.rmargin) /
                                           g.dr * 1.0001 + 1e-3) + 1);
}

inline bool gather2_small(const Geo& g) {
  return (long)((g.nx + 7) / 8) * ((g.ny + 7) / 8) <= kG2SmallPatches;
}
inline bool gather2_fits(const Geo& g, int maxc, int nang_sub) {
  return (gather2_small(g) ? gather2_plan<4>(g, maxc, nang_sub, kG2MostLds)
                           : gather2_plan<8>(g, maxc, nang_sub, kG2MostLds)).nw > 0;
}

template <int PREC>
void launch_gather2(const GatherArgs& A, hipStream_t st) {
  const Geo& g = A.g;
  if (PREC == APIRL_PREC_REFERENCE && gather2_fits(g, A.maxc, A.nang_sub)) {
    if (gather2_small(g)) launch_gather2_patches<4>(A, st);
    else launch_gather2_patches<8>(A, st);
    return;
  }
  const dim3 grid((g.nx + kTile - 1) / kTile, (g.ny + kTile - 1) / kTile, g.nz);
  hipLaunchKernelGGL((gather_kernel<2, PREC>), grid, dim3(kGBlock), 0, st, A);
}


// ---- Tile-walk backprojector (3D, APIRL_PREC_REFERENCE) -----------------------------
//
// A wavefront owns an item: kTW x kTW voxel columns (a tile) times a slab of slices,
// summed in its own LDS.  For every ray (angle, radial bin) of the subset that crosses
// the tile (its entry and path there are found once per subset: the rays of all sinograms
// share them) its lanes take the sinograms whose rays can reach the slab there, one ray
// per lane.  Each lane resumes the reference's Siddon loop (Siddon.cpp:310-340) at the
// tile's entry: the x / y crossings are the loop's accumulated float values from the plan's
// table, its z crossings come from the first one by the loop's own additions.  It walks to
// the tile's exit, adding (alpha - alpha_c) L b (SiddonProjector.cpp:546) to the voxels it
// visits inside the slab, while its step count stays below the list length
// |di| + |dj| + |dk| (:220, the dropped exit voxel), and only there: the voxels, weights and
// terms are the reference's floats, bit for bit.  Each voxel's terms are summed in double in
// the wavefront's order, which depends on the data only (one wavefront per item), so
// repeated runs are bit-identical, and rounded to float once.
//
// An image of few tiles is split further: each (tile, slab) into chunks of the tile's rays,
// whose sums go to memory in double and are added in chunk order.
//
// VALU issue bounds it (4.3e8 wave-instructions for 12 of 252 angles of 344 x 837 bins into
// 256 x 256 x 81, 14 a step, two thirds of the lanes at work), the LDS next (70 % of the time):
// the sinograms of several rays share a pass, so that a pass has 64 lanes, zero bins are left
// out before it, and slabs of about 12 slices keep both the passes full and the walks through
// other slabs few.  That update took 1.35 ms when each (tile, slab, ray) read a kept list of its
// sinograms, zero bins included, and 2.9 ms voxel-driven; the 192 x 192 x 233 sensitivity of
// 128 x 128 x 47, 12.6 ms voxel-driven.  Now 0.78 and 2.18 ms.

constexpr int kTW = 8;      // item tile width in columns (kTW * kTW = one lane per column)

struct TileEntry {
  int i, j;      // column and row of the ray's first voxel in the tile
  int mxy;       // x and y crossings the loop has taken there
  float ce;      // alpha_c there: the crossing just taken, or alpha_min (first voxel)
  float Xn, Yn;  // the next x and y crossings (the loop's accumulated values)
  float aout;    // alpha near the tile's exit (sinogram candidates only)
};

// A ray that enters a tile: the loop's state there and the transaxial part of its walk
// through the tile, the same for every sinogram: the columns it visits in order, for each
// the alpha at which the loop leaves it by an x or y crossing (the smaller accumulated
// crossing there; x before y on ties, Siddon.cpp:318-331) and the bytes from the column's
// sums to the next one's.  At most 2 kTW - 1 columns; the last one's step leaves the slab for
// good, and two entries follow that lead nowhere, so a walk may go on a step past its end.
constexpr int kTPath = 2 * kTW + 2;
constexpr int kTileAway = 1 << 29;
struct TileStep {
  float ae;
  int step;
};
struct alignas(16) TileRay {
  float ce, aout;  // alpha at the entry (alpha_c) and where the walk leaves the tile
  int pair;        // ka * nr + r
  int mxy;         // x and y crossings the loop has taken at the entry
  int nxy;         // the ray's transaxial list length |di| + |dj|
  int ncol;        // columns on its path through the tile
  int col0;        // byte offset of the first column's sums
  int pad;
  TileStep path[kTPath];
};
static_assert(sizeof(TileRay) == 32 + 8 * kTPath, "TileRay is whole 16-byte words");

// Axial record of one ray with its bin value, (angle, r, sinogram) order: with the
// sinogram's crossing increment (apirl_plan::d_zinc) what a lane needs beside the TileRay.
struct alignas(16) TileZ {
  float az0;  // first z crossing
  float L;    // ray length
  float b;    // bin value
  int k01;    // entry and exit slice, 16 bits each
};
static_assert(sizeof(TileZ) == 16, "TileZ is one 16-byte load");

// Crossings p after which index i0 + inc p enters [lo, hi] (pin) and first lies
// beyond it (pout); false when it never lies in it.
__device__ __forceinline__ bool axis_span(int i0, int inc, int lo, int hi, int& pin, int& pout) {
  if (inc == 0) {
    pin = 0;
    pout = INT_MAX;
    return i0 >= lo && i0 <= hi;
  }
  if (inc > 0) {
    pin = lo - i0 > 0 ? lo - i0 : 0;
    pout = hi - i0 + 1;
    return i0 <= hi;
  }
  pin = i0 - hi > 0 ? i0 - hi : 0;
  pout = i0 - lo + 1;
  return i0 >= lo;
}

// Crossing p >= 1 along one axis: the table's value for index c = i0 + inc p, or, for
// the one index past the image that an item at its edge asks for, the loop's next
// addition to the previous crossing.
__device__ __forceinline__ float axis_cross(const float* tab, int n, int i0, int inc, float a0,
                                            float au, int p) {
  const int c = i0 + inc * p;
  if (c >= 0 && c < n) return tab[c];
  return p == 1 ? a0 : tab[c - inc] + au;
}

// Number of crossings p >= 1 whose value is <= v (strict: < v), given that crossing
// plo (when plo >= 1) is and that the answer is taken as phi once it reaches phi:
// the linear estimate, corrected against the exact values.
__device__ __forceinline__ int axis_count(const float* tab, int n, int i0, int inc, float a0,
                                          float au, int plo, int phi, float v, bool strict) {
  const float e = (v - a0) / au + 1.f;
  int p = !(e > (float)plo) ? plo : (e < (float)phi ? (int)e : phi);
  while (p > plo) {
    const float x = axis_cross(tab, n, i0, inc, a0, au, p);
    if (strict ? x < v : x <= v) break;
    p--;
  }
  while (p < phi) {
    const float x = axis_cross(tab, n, i0, inc, a0, au, p + 1);
    if (!(strict ? x < v : x <= v)) break;
    p++;
  }
  return p;
}

// Where ray t enters the tile [ti0, ti1] x [tj0, tj1]: the loop's state after the
// later of the crossings that bring i and j into range (an x crossing at the same
// alpha as a y crossing is taken first, Siddon.cpp:318-331); false when the ray's
// path misses the tile.
__device__ __forceinline__ bool tile_entry(const Geo& g, const RayXY& t, const float* xy, int ti0,
                                           int ti1, int tj0, int tj1, TileEntry& E) {
  const int iinc = ray_iinc(t.flags), jinc = ray_jinc(t.flags);
  int pin, pout, qin, qout;
  if (!axis_span(t.i0, iinc, ti0, ti1, pin, pout) || !axis_span(t.j0, jinc, tj0, tj1, qin, qout))
    return false;
  const float* yt = xy + g.nx;
  int p = 0, q = 0;
  float ce = t.amin;
  if (pin > 0 || qin > 0) {
    const float Xin = pin > 0 ? axis_cross(xy, g.nx, t.i0, iinc, t.ax, t.axu, pin) : -FLT_MAX;
    const float Yin = qin > 0 ? axis_cross(yt, g.ny, t.j0, jinc, t.ay, t.ayu, qin) : -FLT_MAX;
    if (Xin <= Yin) {  // entered by y crossing qin; x crossings up to its alpha are taken
      q = qin;
      ce = Yin;
      if (iinc != 0) {
        p = axis_count(xy, g.nx, t.i0, iinc, t.ax, t.axu, pin, pout, Yin, false);
        if (p >= pout) return false;
      }
    } else {  // entered by x crossing pin; y crossings below its alpha are taken
      p = pin;
      ce = Xin;
      if (jinc != 0) {
        q = axis_count(yt, g.ny, t.j0, jinc, t.ay, t.ayu, qin, qout, Xin, true);
        if (q >= qout) return false;
      }
    }
  }
  E.i = t.i0 + iinc * p;
  E.j = t.j0 + jinc * q;
  E.mxy = p + q;
  E.ce = ce;
  E.Xn = (iinc == 0 || p == 0) ? t.ax : xy[E.i] + t.axu;
  E.Yn = (jinc == 0 || q == 0) ? t.ay : yt[E.j] + t.ayu;
  const float xo = iinc == 0 ? FLT_MAX : t.ax + (float)(pout - 1) * t.axu;
  const float yo = jinc == 0 ? FLT_MAX : t.ay + (float)(qout - 1) * t.ayu;
  E.aout = fminf(t.amax, fminf(xo, yo));
  return true;
}

// Radial bins of angle a whose LORs can cross a tile centred at (xc, yc) with
// half-widths (hx, hy): candidate_bins for a rectangle.
__device__ __forceinline__ void tile_bins(const GatherArgs& A, int a, float xc, float yc, float hx,
                                          float hy, float inv_dr, int& lo0, int& hi0, int& lo1,
                                          int& hi1) {
  const Geo& g = A.g;
  const float2 cs = A.angcs[a];
  const float sc = xc * cs.x + yc * cs.y;
  const float hw = hx * fabsf(cs.x) + hy * fabsf(cs.y) + g.rmargin;
  if (!grid_lut<kGridAny>(A)) {
    int jlo = (int)ceilf((sc - hw - g.r0) * inv_dr);
    int jhi = (int)floorf((sc + hw - g.r0) * inv_dr);
    lo0 = lo1 = jlo < 0 ? 0 : jlo;
    hi0 = hi1 = jhi > g.nr - 1 ? g.nr - 1 : jhi;
    return;
  }
  lut_bins(A, sc, hw, lo0, hi0);
  const float2 co = A.angcs_odd[a];
  const float so = xc * co.x + yc * co.y;
  const float hwo = hx * fabsf(co.x) + hy * fabsf(co.y) + g.rmargin;
  lut_bins(A, so, hwo, lo1, hi1);
}

// Byte distance of neighbouring slices' sums in an item: one word pair more than the tile's
// columns, so that lanes on one column and neighbouring slices take different LDS banks.
constexpr int kTPitch = (kTW * kTW + 1) * 8;

typedef __attribute__((address_space(3))) double LdsDouble;
typedef __attribute__((address_space(3))) const TileStep LdsTileStep;
typedef __attribute__((address_space(3))) const char LdsByte;

// One step of the reference's loop in an item: the term goes to the sum of the lane's voxel
// (at LDS address v; only where that lies in the slab, below lim), then the lane moves on
// along its path (at LDS address ep).  14 VALU instructions with the end test of every
// second step.
__device__ __forceinline__ void tile_step(unsigned& ep, float& Zn, float& ac, unsigned& v,
                                          float azu, float L, float b, int kstep, unsigned lim) {
  LdsTileStep* p = (LdsTileStep*)(uintptr_t)ep;
  const float ae = p->ae;
  const int step = p->step;
  const bool zst = Zn < ae;  // Siddon.cpp:318-339: x, then y, then z on ties
  const float an = zst ? Zn : ae;
  const float term = (an - ac) * L * b;  // the reference's float term (geomFactor 1)
  if (v < lim)
    __hip_atomic_fetch_add((LdsDouble*)(uintptr_t)v, (double)term, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WAVEFRONT);
  ac = an;
  Zn = Zn + (zst ? azu : 0.f);
  v += (unsigned)(zst ? kstep : step);
  ep += zst ? 0u : (unsigned)sizeof(TileStep);
}

// One lane: the ray (R, z, zinc) from the tile's entry to its exit, its terms added to the
// item's sums (slice kz0 + q of column c at LDS address q kTPitch + 8 c, below lim: the sums
// are the first thing in the workgroup's LDS).
__device__ __forceinline__ void tile_lane(const TileRay& R, const TileZ& z, float zinc, int kz0,
                                          unsigned lim) {
  const float azu = fabsf(zinc), ce = R.ce;
  const int kinc = zinc > 0.f ? 1 : -1;  // no z step where Vz is 0: az0 is FLT_MAX
  int k = (short)(z.k01 & 0xffff);
  int left = R.nxy + abs((z.k01 >> 16) - k) - R.mxy;
  float Zn = z.az0;
  // z crossings taken before the entry: those below its alpha (a z crossing at the
  // alpha of an x or y crossing is taken after it, Siddon.cpp:318-339), by the
  // loop's own additions, four at a time while all four are (one test in four: 1.08 -> 0.94 ms
  // for 12 of 252 angles of 344 x 837 bins into 256 x 256 x 81, whose rays cross up to 70 slices)
  if (R.mxy > 0) {
    int c = 0;
    float z1 = Zn + azu, z2 = z1 + azu, z3 = z2 + azu;
    while (z3 < ce && c < left) {
      Zn = z3 + azu;
      z1 = Zn + azu;
      z2 = z1 + azu;
      z3 = z2 + azu;
      c += 4;
    }
    c += (Zn < ce ? 1 : 0) + (z1 < ce ? 1 : 0) + (z2 < ce ? 1 : 0);
    Zn = z2 < ce ? z3 : (z1 < ce ? z2 : (Zn < ce ? z1 : Zn));
    k += c * kinc;
    left -= c;
  }
  unsigned v = (unsigned)((k - kz0) * kTPitch + R.col0);
  const int kstep = kinc * kTPitch;
  unsigned ep = (unsigned)(size_t)(LdsByte*)(const char*)R.path;
  const unsigned eend = ep + R.ncol * (unsigned)sizeof(TileStep);
  float ac = ce;
  // far from the list's end the walk cannot reach it in the next kTFar steps
  constexpr int kTFar = 2 * kTPath;
  if (left >= kTFar) {
    left -= kTFar;
    for (int m = 0; m < kTFar; m += 2) {
      tile_step(ep, Zn, ac, v, azu, z.L, z.b, kstep, lim);
      tile_step(ep, Zn, ac, v, azu, z.L, z.b, kstep, lim);
      if (ep >= eend) return;
    }
  }
  for (; left > 0 && ep < eend; left--)
    tile_step(ep, Zn, ac, v, azu, z.L, z.b, kstep, lim);
}

constexpr int kTSlots = 4;    // rays in flight per wavefront
constexpr int kTQueue = 128;  // pending (ray, sinogram) entries per wavefront

// LDS of one item: its sums (double: LDS adds of doubles run about 20 times faster than of
// floats here, and sum more exactly), the rays in flight, and the queue of pending (ray,
// sinogram) entries.
__host__ __device__ inline int tile_acc_bytes(int zs) { return (zs * kTPitch + 15) / 16 * 16; }
inline size_t tile_lds_bytes(int zs) {
  return (size_t)tile_acc_bytes(zs) + kTSlots * sizeof(TileRay) + kTQueue * 4;
}

// Columns a ray visits in the tile [ti0, ti1] x [tj0, tj1] from its entry E on, by the loop's
// x / y steps; step(q, ae, bx) for each: the alpha at which it leaves the q-th, by an x step or
// by a y step.
template <class Step>
__device__ __forceinline__ int tile_path(const RayXY& t, const TileEntry& E, int ti0, int ti1,
                                         int tj0, int tj1, Step&& step) {
  const int iinc = ray_iinc(t.flags), jinc = ray_jinc(t.flags);
  float Xn = E.Xn, Yn = E.Yn;
  int i = E.i, j = E.j, q = 0;
  while (q < kTPath - 2) {
    const bool bx = Xn <= Yn;
    step(q, Xn < Yn ? Xn : Yn, bx);
    q++;
    if (bx) {
      i += iinc;
      Xn = Xn + t.axu;
    } else {
      j += jinc;
      Yn = Yn + t.ayu;
    }
    if (i < ti0 || i > ti1 || j < tj0 || j > tj1) break;
  }
  return q;
}

// The rays of one tile per workgroup: candidate c of angle ka (the c-th bin of the angle's
// candidate range) is kept when its LOR is valid and its path enters the tile.  The kept rays
// go to the front of the tile's slots, the longest paths first and in (angle, bin) order among
// equal ones: the lanes of a pass then walk about equally far.  The workgroup also finds its
// tile's place in the order of tile_bp_kernel's items: by the distance from the image centre, and
// by number among equal ones.
__global__ __launch_bounds__(kGBlock) void tile_rays_kernel(GatherArgs A, int maxc, int nslot,
                                                            TileRay* __restrict__ rays,
                                                            int* __restrict__ pairs,
                                                            int* __restrict__ count,
                                                            int* __restrict__ order) {
  constexpr int kWaves = kGBlock / kWave;
  __shared__ int place[kTPath];            // next slot of each path length
  __shared__ int wcount[kWaves][kTPath];
  __shared__ int before;  // tiles before this one in the order
  const Geo& g = A.g;
  const int tile = blockIdx.x, wave = threadIdx.x / kWave;
  const int ntx = (g.nx + kTW - 1) / kTW;
  const int ti0 = (tile % ntx) * kTW, tj0 = (tile / ntx) * kTW;
  const int ti1 = (ti0 + kTW < g.nx ? ti0 + kTW : g.nx) - 1;
  const int tj1 = (tj0 + kTW < g.ny ? tj0 + kTW : g.ny) - 1;
  const float xt = -g.R + g.dx * 0.5f * (float)(ti0 + ti1 + 1);
  const float yt = -g.R + g.dy * 0.5f * (float)(tj0 + tj1 + 1);
  const float hx = 0.5f * g.dx * (float)(ti1 - ti0 + 1);
  const float hy = 0.5f * g.dy * (float)(tj1 - tj0 + 1);
  RayXY t;
  TileEntry E;
  int pair = 0;
  // the ray of candidate slot idx, the columns of its path (0: none)
  auto candidate = [&](int idx) -> int {
    if (idx >= nslot) return 0;
    const int c = idx % maxc, ka = idx / maxc, a = A.subset + A.nsubsets * ka;
    int lo0, hi0, lo1, hi1;
    tile_bins(A, a, xt, yt, hx, hy, 1.0f / g.dr, lo0, hi0, lo1, hi1);
    int rr = lo0 + c, last = hi0;
    if (grid_lut<kGridAny>(A)) {
      // even and odd bins in turn, each from its own range's first (the ranges of odd bins half
      // an angular step away can lie far apart)
      const int even = lo0 + (lo0 & 1), odds = lo1 + 1 - (lo1 & 1);
      const bool odd = ((c & 1) != 0) != (odds < even);
      rr = (odd ? odds : even) + 2 * (c >> 1);
      last = odd ? hi1 : hi0;
    }
    if (rr > last) return 0;
    pair = ka * g.nr + rr;
    t = A.rays[(long)a * g.nr + rr];
    if (!(t.flags & RAY_VALID) ||
        !tile_entry(g, t, A.xytab + ((long)a * g.nr + rr) * (g.nx + g.ny), ti0, ti1, tj0, tj1, E))
      return 0;
    return tile_path(t, E, ti0, ti1, tj0, tj1, [](int, float, bool) {});
  };
  if (threadIdx.x < kTPath) place[threadIdx.x] = 0;
  if (threadIdx.x == 0) before = 0;
  __syncthreads();
  {
    auto distance = [&](int t) -> long {  // squared, of twice the voxels
      const long x = (2 * (t % ntx) + 1) * (long)kTW - g.nx, y = (2 * (t / ntx) + 1) * (long)kTW - g.ny;
      return x * x + y * y;
    };
    const long mine = distance(tile);
    int n = 0;
    for (int t = threadIdx.x; t < (int)gridDim.x; t += kGBlock) {
      const long d = distance(t);
      n += d < mine || (d == mine && t < tile) ? 1 : 0;
    }
    if (n > 0) atomicAdd(&before, n);
  }
  for (int base = 0; base < nslot; base += kGBlock) {
    const int n = candidate(base + threadIdx.x);
    if (n > 0) atomicAdd(&place[n], 1);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    order[before] = tile;
    int run = 0;
    for (int n = kTPath - 1; n > 0; n--) {
      const int c = place[n];
      place[n] = run;
      run += c;
    }
    count[tile] = run;
  }
  __syncthreads();
  for (int base = 0; base < nslot; base += kGBlock) {
    const int ncol = candidate(base + threadIdx.x);
    int rank = 0;
    for (int n = 1; n < kTPath; n++) {
      const unsigned long long bal = __ballot(ncol == n);
      if (ncol == n)
        rank = __builtin_amdgcn_mbcnt_hi((unsigned)(bal >> 32),
                                         __builtin_amdgcn_mbcnt_lo((unsigned)bal, 0));
      if (threadIdx.x % kWave == 0) wcount[wave][n] = __popcll(bal);
    }
    __syncthreads();
    int d = place[ncol] + rank;
    for (int w = 0; w < wave; w++) d += ncol > 0 ? wcount[w][ncol] : 0;
    __syncthreads();
    if (threadIdx.x > 0 && threadIdx.x < kTPath)
      for (int w = 0; w < kWaves; w++) place[threadIdx.x] += wcount[w][threadIdx.x];
    __syncthreads();
    if (ncol == 0) continue;
    TileRay* R = rays + (long)tile * nslot + d;
    pairs[(long)tile * nslot + d] = pair;
    const int iinc = ray_iinc(t.flags), jinc = ray_jinc(t.flags);
    float last = E.ce;
    tile_path(t, E, ti0, ti1, tj0, tj1, [&](int q, float ae, bool bx) {
      TileStep e;
      e.ae = last = ae;
      e.step = q == ncol - 1 ? kTileAway : (bx ? iinc : jinc * kTW) * 8;
      R->path[q] = e;
    });
    for (int r = ncol; r < kTPath; r++)
      R->path[r] = TileStep{__int_as_float(0x7f800000), kTileAway};
    R->ce = E.ce;
    R->aout = fmaxf(E.aout, last);
    R->pair = pair;
    R->mxy = E.mxy;
    R->nxy = t.nxy;
    R->ncol = ncol;
    R->col0 = ((E.j - tj0) * kTW + E.i - ti0) * 8;
    R->pad = 0;
  }
}

// The call's axial records out[(ka nr + r) nsino + s] (zray_setup and the bin value): a
// workgroup takes kTZBins bins of one angle with all of their sinograms, 32 at a time through
// an LDS tile, so that the sinogram is read along r and the records are written along s;
// nzmask[(ka nr + r) nwords + s / 32]: the sinograms of a valid LOR whose bin is not zero, a
// bit each; nz_pair[ka nr + r]: whether there is one.
constexpr int kTZBins = 8;
__host__ __device__ inline int tile_words(int nsino) { return (nsino + 63) / 64 * 2 + 2; }
__global__ __launch_bounds__(kGBlock) void tile_zsetup_kernel(GatherArgs A,
                                                              TileZ* __restrict__ out,
                                                              unsigned* __restrict__ nzmask,
                                                              int* __restrict__ nz_pair) {
  __shared__ float tb[32][kTZBins + 1];
  __shared__ int snz[kTZBins];
  const Geo& g = A.g;
  const int r0 = blockIdx.x * kTZBins, ka = blockIdx.y;
  const int a = A.subset + A.nsubsets * ka;
  const int rx = threadIdx.x % kTZBins, sx = threadIdx.x / kTZBins;  // 8 bins x 32 sinograms
  const int ty = threadIdx.x / 32, tx = threadIdx.x % 32;            // the same, s fastest
  RayXY R = A.rays[(long)a * g.nr + (r0 + ty < g.nr ? r0 + ty : g.nr - 1)];
  const int nwords = tile_words(g.nsino);
  bool nz = false;
  if (threadIdx.x < kTZBins) snz[threadIdx.x] = 0;
  for (int s0 = 0; s0 < g.nsino; s0 += 32) {
    __syncthreads();
    {
      const int s = s0 + sx, rr = r0 + rx;
      float b = 1.f;
      if (s < g.nsino && rr < g.nr) {
        if (A.kind == BP_PLAIN) b = A.sino[((long)s * A.nang_sub + ka) * g.nr + rr];
        else if (A.kind == BP_MULT) b = A.sino[((long)s * g.nang + a) * g.nr + rr];
      }
      tb[sx][rx] = b;
    }
    __syncthreads();
    const int s = s0 + tx, rr = r0 + ty;
    bool nzb = false;
    if (s < g.nsino && rr < g.nr) {
      const float2 zz = A.zab[s];
      ZRay z;
      zray_setup(g, R, zz.x, zz.y, z);
      TileZ o;
      o.az0 = z.az0;
      o.L = z.L;
      o.b = tb[tx][ty];
      o.k01 = (int)(((unsigned)(int)z.k1 << 16) | ((unsigned)z.k0 & 0xffffu));
      out[((long)ka * g.nr + rr) * g.nsino + s] = o;
      nzb = o.b != 0.f && (R.flags & RAY_VALID);
    }
    const unsigned bits = (unsigned)(__ballot(nzb) >> (threadIdx.x & 32));
    if (tx == 0 && rr < g.nr) nzmask[((long)ka * g.nr + rr) * nwords + s0 / 32] = bits;
    nz |= bits != 0u;
  }
  // words that a window of 64 sinograms may reach past the last one
  for (int w = (g.nsino + 31) / 32 + tx; w < nwords; w += 32)
    if (r0 + ty < g.nr) nzmask[((long)ka * g.nr + r0 + ty) * nwords + w] = 0u;
  __syncthreads();
  if (nz) snz[ty] = 1;
  __syncthreads();
  if (threadIdx.x < kTZBins && r0 + (int)threadIdx.x < g.nr)
    nz_pair[(long)ka * g.nr + r0 + threadIdx.x] = snz[threadIdx.x];
}

// Items b = (tile position * nslab + slab) * nchunk + chunk, the tiles in the order of
// order[] (the ones nearest the image centre first, whose rays are the most), one wavefront
// each.  The rays entering tile t are rays[t * nslot + c], c < count[t]; a chunk takes every
// nchunk-th of them.  The (ray, sinogram) pairs to walk go through a queue in LDS: a pass takes 64 of
// them as soon as there are, so a pass carries the sinograms of several rays.  parts: null,
// or the chunks' sums, [nchunk][voxels].
__global__ __launch_bounds__(kWave) void tile_bp_kernel(GatherArgs A, int zs, int nslab, int nchunk,
                                                        const int* __restrict__ order,
                                                        const TileRay* __restrict__ rays,
                                                        const int* __restrict__ pairs,
                                                        const int* __restrict__ count, int nslot,
                                                        const TileZ* __restrict__ zrec,
                                                        const unsigned* __restrict__ nzmask,
                                                        const float* __restrict__ zinc,
                                                        double* __restrict__ parts) {
  extern __shared__ __align__(16) char tlds[];
  const Geo& g = A.g;
  const int lane = threadIdx.x;
  char* acc = tlds;
  TileRay* slots = (TileRay*)(tlds + tile_acc_bytes(zs));
  unsigned* queue = (unsigned*)(slots + kTSlots);
  const int ntx = (g.nx + kTW - 1) / kTW;
  const int chunk = blockIdx.x % nchunk, ts = blockIdx.x / nchunk;
  const int slab = ts % nslab, tile = order[ts / nslab];
  const int ti0 = (tile % ntx) * kTW, tj0 = (tile / ntx) * kTW;
  const int kz0 = slab * zs, kz1 = (kz0 + zs < g.nz ? kz0 + zs : g.nz) - 1, nk = kz1 - kz0 + 1;
  const bool incol = ti0 + lane % kTW < g.nx && tj0 + lane / kTW < g.ny;
  const long nxy = (long)g.nx * g.ny;
  const long v0 = kz0 * nxy + (long)(tj0 + lane / kTW) * g.nx + ti0 + lane % kTW;
  const unsigned lim = (unsigned)(nk * kTPitch);
  double* col = (double*)acc + lane;
  for (int q = 0; q < nk; q++)
    col[q * (kTPitch / 8)] = (incol && !A.fresh && !parts) ? (double)A.img[v0 + q * nxy] : 0.0;
  // the slab's z range widened by the search margin
  const float zlo = g.offz + kz0 * g.dz - kZMargin, zhi = g.offz + (kz1 + 1) * g.dz + kZMargin;
  const TileRay* tr = rays + (long)tile * nslot;
  const int* tp = pairs + (long)tile * nslot;
  const int nray = count[tile];
  const int nwords = tile_words(g.nsino);
  int pend = 0;  // pending entries (ray number << 16 | sinogram), queue[0 .. pend)
  // one pass: the first n entries, one per lane; the ones after them move to the front
  auto run_pass = [&](int n) {
    wave_lds_sync();
    const unsigned e = queue[lane];
    const unsigned after = n == kWave ? queue[kWave + lane] : 0u;
    if (lane < n) {
      const TileRay& R = slots[(e >> 16) & (kTSlots - 1)];
      const int s = (int)(e & 0xffffu);
      const TileZ z = zrec[(long)R.pair * g.nsino + s];
      tile_lane(R, z, zinc[s], kz0, lim);
    }
    pend -= n;
    wave_lds_sync();
    if (lane < pend) queue[lane] = after;
  };
  int nlive = 0;  // rays taken so far (their numbers in the queue)
  for (int cb = chunk; cb < nray; cb += kWave * nchunk) {
    // the chunk's next 64 rays: those with a non-zero bin
    const int cl = cb + lane * nchunk, pr = cl < nray ? tp[cl] : -1;
    unsigned long long live = __ballot(pr >= 0 && A.nz_pair[pr < 0 ? 0 : pr] != 0);
    for (; live; live &= live - 1) {
      const int c = cb + (int)__builtin_ctzll(live) * nchunk;
      // the slot of ray number nlive is free once no pending entry belongs to the ray
      // kTSlots before it
      while (pend > 0) {
        wave_lds_sync();
        if ((((unsigned)nlive - (queue[0] >> 16)) & 0xffffu) < kTSlots) break;
        run_pass(pend < kWave ? pend : kWave);
      }
      wave_lds_sync();
      constexpr int kWords = sizeof(TileRay) / 4;
      if (lane < kWords)
        ((unsigned*)&slots[nlive & (kTSlots - 1)])[lane] = ((const unsigned*)(tr + c))[lane];
      wave_lds_sync();
      const unsigned taglane = (((unsigned)nlive & 0xffffu) << 16) + (unsigned)lane;
      nlive++;
      // The sinograms whose ray can reach the slab inside the tile: runs [first, first + cnt),
      // one per lane, of which those with a non-zero bin are queued (zero bins add nothing,
      // SiddonProjector.cpp:496).  With one slab all of them, 64 to a run; otherwise, per
      // segment run, the indices whose mean z lies within the slab widened by the run's slopes
      // over the tile's alpha range (z = zmean + (zb - za)(alpha - 1/2)) and its deviation from
      // the line.  The few that do not reach it add nothing.
      const float ulo = tr[c].ce - 0.5f, uhi = tr[c].aout - 0.5f;
      const unsigned* words = nzmask + (long)tr[c].pair * nwords;
      const int nrun = nslab == 1 ? (g.nsino + kWave - 1) / kWave : A.nseg;
      for (int rb = 0; rb < nrun; rb += kWave) {
        int first = 0, cnt = 0;
        if (rb + lane < nrun) {
          if (nslab == 1) {
            first = (rb + lane) * kWave;
            cnt = g.nsino - first < kWave ? g.nsino - first : kWave;
          } else {
            const GatherSeg S = A.segs[rb + lane];
            const float p1 = S.dmin * ulo, p2 = S.dmin * uhi, p3 = S.dmax * ulo, p4 = S.dmax * uhi;
            const float dlo = fminf(fminf(p1, p2), fminf(p3, p4));
            const float dhi = fmaxf(fmaxf(p1, p2), fmaxf(p3, p4));
            // 0.01 mm and a hundredth of an index for the rounding
            const float lf = ceilf((zlo - dhi - S.devz - 0.01f - S.z0) * S.dhi - 0.01f);
            const float hf = floorf((zhi - dlo + S.devz + 0.01f - S.z0) * S.dhi + 0.01f);
            const int l0 = lf > 0.f ? (lf < (float)S.count ? (int)lf : S.count) : 0;
            const int l1 = hf < (float)(S.count - 1) ? (int)hf : S.count - 1;
            first = S.first + l0;
            cnt = l1 >= l0 ? l1 - l0 + 1 : 0;
          }
        }
        while (__any(cnt > 0)) {
          // the next (up to) 64 of every run: their bits
          unsigned lo = 0, hi = 0;
          if (cnt > 0) {
            const unsigned* w = words + (first >> 5);
            const int sh = first & 31;
            lo = __builtin_amdgcn_alignbit(w[1], w[0], sh);
            hi = __builtin_amdgcn_alignbit(w[2], w[1], sh);
            if (cnt < 32) lo &= (1u << cnt) - 1u;
            hi = cnt <= 32 ? 0u : (cnt < 64 ? hi & ((1u << (cnt - 32)) - 1u) : hi);
          }
          unsigned long long some = __ballot((lo | hi) != 0u);
          if (!__any(hi != 0u)) {  // runs of at most 32: the usual case, half the work
            for (; some; some &= some - 1) {
              const int l = __builtin_ctzll(some);
              const unsigned m = (unsigned)__builtin_amdgcn_readlane(lo, l);
              const int f = __builtin_amdgcn_readlane(first, l);
              if (__builtin_amdgcn_inverse_ballot_w64((unsigned long long)m))
                queue[__builtin_amdgcn_mbcnt_lo(m, pend)] = taglane + (unsigned)f;
              pend += __popc(m);
              if (pend >= kWave) run_pass(kWave);
            }
          } else {
            for (; some; some &= some - 1) {
              const int l = __builtin_ctzll(some);
              const unsigned mlo = (unsigned)__builtin_amdgcn_readlane(lo, l);
              const unsigned mhi = (unsigned)__builtin_amdgcn_readlane(hi, l);
              const int f = __builtin_amdgcn_readlane(first, l);
              if (__builtin_amdgcn_inverse_ballot_w64(mlo | (unsigned long long)mhi << 32))
                queue[__builtin_amdgcn_mbcnt_hi(mhi, __builtin_amdgcn_mbcnt_lo(mlo, pend))] =
                    taglane + (unsigned)f;
              pend += __popc(mlo) + __popc(mhi);
              if (pend >= kWave) run_pass(kWave);
            }
          }
          first += kWave;
          cnt -= kWave;
        }
      }
    }
  }
  while (pend > 0) run_pass(pend < kWave ? pend : kWave);
  wave_lds_sync();
  if (incol)
    for (int q = 0; q < nk; q++) {
      const double b = col[q * (kTPitch / 8)];
      if (parts) parts[(long)chunk * nxy * g.nz + v0 + q * nxy] = b;
      else store_voxel<APIRL_PREC_REFERENCE>(A, v0 + q * nxy, (float)b);
    }
}

// The voxels' sums over the chunks, in their order.  Few wavefronts wait for the loads of tens
// of chunks: eight are in flight at a time (64 x 64 x 17, 28 chunks: 10.6 -> 5.7 us).
__global__ __launch_bounds__(kGBlock) void tile_reduce_kernel(GatherArgs A, long nvox, int nchunk,
                                                              const double* __restrict__ parts) {
  const long v = (long)blockIdx.x * kGBlock + threadIdx.x;
  if (v >= nvox) return;
  double b = A.fresh ? 0.0 : (double)A.img[v];
  const double* p = parts + v;
  int c = 0;
  for (; c + 8 <= nchunk; c += 8, p += 8 * nvox) {
    double t[8];
#pragma unroll
    for (int u = 0; u < 8; u++) t[u] = p[u * nvox];
#pragma unroll
    for (int u = 0; u < 8; u++) b += t[u];
  }
  for (; c < nchunk; c++, p += nvox) b += *p;
  store_voxel<APIRL_PREC_REFERENCE>(A, v, (float)b);
}

}  // namespace

hipError_t launch_backproject_gather(const apirl_plan* p, const float* sino, float* img,
                                     int subset, int nsubsets, int kind, int precision,
                                     void* scratch, size_t scratch_bytes, hipStream_t st,
                                     const EmFuse* fuse) {
  if (kind != BP_PLAIN && kind != BP_ONES && kind != BP_MULT) return hipErrorNotSupported;
  if (precision < APIRL_PREC_REFERENCE || precision > APIRL_PREC_F64_SETUP)
    return hipErrorInvalidValue;
  const Geo& g = p->geo;
  const int nang_sub = subset_num_angles(g.nang, nsubsets, subset);
  const long nrays = (long)g.nsino * nang_sub * g.nr;
  const long nvox = (long)g.nx * g.ny * g.nz;
  if (nrays == 0 || nvox == 0) return hipSuccess;
  if (g.dims == 3 && scratch_bytes < gather_scratch_bytes(p, subset, nsubsets))
    return hipErrorInvalidValue;
  GatherArgs A;
  ZRay* zr = nullptr;
  int* nzp = nullptr;
  gather_args_for(p, subset, nsubsets, kind, sino, img, g.dims == 3 ? scratch : nullptr, A, zr,
                  nzp);
  A.zlanes = g.dims == 3 ? p->gather_zlanes : 1;
  if (fuse) {
    A.upd_sens = fuse->sens;
    A.fresh = fuse->sens ? kFresh : fuse->fresh;
    A.upd_thr = fuse->thr;
    A.upd_thr_at = fuse->thr_at;
    A.upd_strict = fuse->strict;
  }
  if (g.dims == 3) {
    // APIRL_PREC_F64_SETUP with its tables (the rays' double transaxial setup, their
    // entry crossings, and zsetup's double axial setup): the column kernel, whose
    // terms are then those of the one-voxel F64_SETUP gather, summed as KAHAN
    const LorForm& F = p->forms[p->scanner];
    const bool f64s = precision == APIRL_PREC_F64_SETUP && A.zlanes <= 1 && p->gather_zvox >= 1 &&
                      F.rays_f64s && F.xytab_f64s;
    if (f64s) {
      A.rays = F.rays_f64s;
      A.xytab = F.xytab_f64s;
    }
    const long npair = (long)nang_sub * g.nr;
    hipLaunchKernelGGL(clear_int_kernel, dim3(ggrid(npair)), dim3(kGBlock), 0, st, nzp, npair);
    hipLaunchKernelGGL(zsetup_kernel, dim3(ggrid(nrays)), dim3(kGBlock), 0, st, g, p->d_rays,
                       p->d_zab, sino, kind, nang_sub, subset, nsubsets, nrays, zr, nzp, A.ztab,
                       A.zsoff, A.zblock, f64s ? 1 : 0);
    const int zv = p->gather_zvox;
    if (precision == APIRL_PREC_REFERENCE)
      launch_gather3<APIRL_PREC_REFERENCE>(A, A.zlanes, zv, st);
    else if (precision == APIRL_PREC_KAHAN || f64s)
      launch_gather3<APIRL_PREC_KAHAN>(A, A.zlanes, zv, st);
    else if (precision == APIRL_PREC_F64_SETUP)
      launch_gather3<APIRL_PREC_F64_SETUP>(A, A.zlanes, zv, st);
    else launch_gather3<APIRL_PREC_F64_ALPHA>(A, A.zlanes, zv, st);
  } else {
    if (precision == APIRL_PREC_REFERENCE) launch_gather2<APIRL_PREC_REFERENCE>(A, st);
    else if (precision == APIRL_PREC_KAHAN || precision == APIRL_PREC_F64_SETUP)
      launch_gather2<APIRL_PREC_KAHAN>(A, st);
    else launch_gather2<APIRL_PREC_F64_ALPHA>(A, st);
  }
  return hipGetLastError();
}

// Slab depth of the tile backprojector's items: the plan's tuning, or the whole image up to
// kTSlices slices, about kTSlices - 1 otherwise (a ray is walked through every slab it
// reaches in a tile, and deep slabs leave room for fewer wavefronts).
constexpr int kTSlices = 13;
int tile_slab_depth(const apirl_plan* p) {
  const int nz = p->geo.nz;
  if (p->tile_zs > 0) return p->tile_zs < nz ? p->tile_zs : nz;
  if (nz <= kTSlices) return nz;
  const int nslab = (nz + kTSlices - 2) / (kTSlices - 1);
  return (nz + nslab - 1) / nslab;
}

// Half-width along r of the bins whose LORs can cross a tile at the widest angle (tile_bins).
double tile_half_width(const Geo& g) {
  return 0.5 * kTW * std::max(g.dx, g.dy) * 1.41421357 + g.rmargin + 1e-3;
}

int tile_lut_candidates(const Geo& g, const std::vector<int2>& lut, float inv_h) {
  // entries between the two that lut_bins looks up, which rounds outwards and takes one more on
  // each side; two more for its own rounding
  const int n = (int)lut.size();
  const double d = std::ceil(2.0 * tile_half_width(g) * inv_h) + 6;
  const int step = d < n ? (int)d : n;
  int most = 0;
  for (int k = 0; k < n; k++)
    most = std::max(most, lut[std::min(k + step, n - 1)].y - lut[k].x + 1);
  return most + 1;  // the parity with one bin more, in turn with the other
}

// Upper bound on the candidate bins of one (tile, angle) of the active LOR form: counted in its
// lookup table (LorForm::tile_maxc), whose radial grid need not be the plan's, or the bins within
// the tile's half-width on the plan's uniform grid.
int tile_max_candidates(const apirl_plan* p) {
  const Geo& g = p->geo;
  if (p->d_rlut) return p->forms[p->scanner].tile_maxc;
  double drmin = g.dr > 0 ? g.dr : 1.0;
  for (size_t j = 1; j < p->r.size(); j++) drmin = std::min(drmin, (double)p->r[j] - p->r[j - 1]);
  if (!(drmin > 0)) drmin = 1e-3;
  const int c = (int)std::ceil(2 * tile_half_width(g) / drmin) + 3;
  return c < g.nr ? c : g.nr;
}

const char* tile_misfit(const apirl_plan* p) {
  if (p->geo.dims != 3) return "the tile backprojector is 3D only";
  if (p->geo.nsino >= 65536) return "the tile backprojector takes fewer than 65536 sinograms";
  if ((long)p->geo.nang * tile_max_candidates(p) >= 65536)
    return "the tile backprojector takes fewer than 65536 candidate rays per tile";
  if (tile_lds_bytes(tile_slab_depth(p)) > 65536)
    return "the tile backprojector's items exceed 64 KiB of LDS";
  if (!p->d_zinc || !p->slices16) return "the tile backprojector keeps slices in 16 bits";
  return nullptr;
}

int tile_count(const apirl_plan* p) {
  return ((p->geo.nx + kTW - 1) / kTW) * ((p->geo.ny + kTW - 1) / kTW);
}

namespace {
size_t align256(size_t n) { return (n + 255) / 256 * 256; }

struct TileSizes {
  int nang_sub, maxc, ntiles, nslot, zs, nslab, nchunk;
  long nrays, npair, nvox;
};

// Wavefronts the items should come to, by the pairs of a slot and a sinogram there are to walk.
// Few of them and the GPU (some 4600 wavefronts with an item's LDS) is not filled, or the last
// ones to finish are a large part; many of them and each spends its time on its own start, its
// sums and their way through memory (nchunk images of doubles).  The best of sweeps over 44
// subsets of 2e5 .. 8e7 pairs lay at 0.5 .. 3 times 4600, about as their 0.36th power: 2.0e5 pairs
// 32 us at 2300 wavefronts, 52 at 9200; 6.2e6 92, 80 and 90 us at 4600, 6900 and 13800; 8.5e7
// 1180, 623 and 618 us at 4600, 9200 and 13800.
constexpr double kTWaves = 30.0, kTWavesPower = 0.36;
constexpr int kTChunkRays = 4;                   // slots per chunk at least
constexpr size_t kTPartBytes = size_t(1) << 28;  // the chunks' sums at most

TileSizes tile_sizes(const apirl_plan* p, int subset, int nsubsets) {
  const Geo& g = p->geo;
  TileSizes z;
  z.nang_sub = subset_num_angles(g.nang, nsubsets, subset);
  z.npair = (long)z.nang_sub * g.nr;
  z.nrays = (long)g.nsino * z.npair;
  z.nvox = (long)g.nx * g.ny * g.nz;
  z.maxc = tile_max_candidates(p);
  z.ntiles = tile_count(p);
  z.nslot = z.nang_sub * z.maxc;
  z.zs = tile_slab_depth(p);
  z.nslab = (g.nz + z.zs - 1) / z.zs;
  const double waves = kTWaves * std::pow((double)z.ntiles * z.nslot * g.nsino, kTWavesPower);
  long c = std::lround(waves / ((double)z.ntiles * z.nslab));
  // whole eights, where there are some: a tile's chunk k then runs on XCD k % 8 in every tile and
  // slab, whose L2 has the rays' records (33 chunks against 32: 2.22 against 2.20 ms for the 128 x 128 x
  // 47 sensitivity, 95 against 90 us for a 55 x 55 x 50 update)
  if (c >= 12) c = (c + 4) / 8 * 8;
  c = std::min(c, (long)z.nslot / kTChunkRays);
  c = std::min(c, (long)(kTPartBytes / (z.nvox * sizeof(double))));
  z.nchunk = c < 1 ? 1 : (int)c;
  return z;
}

// geometry: [ray count per tile][order of the tiles][ray (angle, bin) pairs][rays]
struct TileGeoPtrs {
  int* count;
  int* order;
  int* pairs;
  TileRay* rays;
  size_t bytes;
};

TileGeoPtrs tile_geo_ptrs(const TileSizes& z, void* geo) {
  const size_t nslots = (size_t)z.ntiles * z.nslot;
  TileGeoPtrs q;
  char* c = (char*)geo;
  size_t o = 0;
  q.count = (int*)(c + o);
  o += align256((size_t)z.ntiles * sizeof(int));
  q.order = (int*)(c + o);
  o += align256((size_t)z.ntiles * sizeof(int));
  q.pairs = (int*)(c + o);
  o += align256(nslots * sizeof(int));
  q.rays = (TileRay*)(c + o);
  o += align256(nslots * sizeof(TileRay));
  q.bytes = o;
  return q;
}
}  // namespace

size_t tile_geo_bytes(const apirl_plan* p, int subset, int nsubsets) {
  return tile_geo_ptrs(tile_sizes(p, subset, nsubsets), nullptr).bytes;
}

// scratch: [TileZ x nrays, (angle, radial bin, sinogram) order][non-zero sinograms per
// (angle, r)][non-zero flag per (angle, r)][the chunks' sums][the geometry, when it is not
// kept]
size_t tile_scratch_bytes(const apirl_plan* p, int subset, int nsubsets, bool with_geo) {
  const TileSizes z = tile_sizes(p, subset, nsubsets);
  return align256((size_t)z.nrays * sizeof(TileZ)) +
         align256((size_t)z.npair * tile_words(p->geo.nsino) * sizeof(unsigned)) +
         align256((size_t)z.npair * sizeof(int)) +
         (z.nchunk > 1 ? align256((size_t)z.nchunk * z.nvox * sizeof(double)) : 0) +
         (with_geo ? tile_geo_bytes(p, subset, nsubsets) : 0);
}

hipError_t launch_backproject_tile(const apirl_plan* p, const float* sino, float* img,
                                   int subset, int nsubsets, int kind, void* scratch,
                                   size_t scratch_bytes, hipStream_t st, const EmFuse* fuse,
                                   void* geo, bool geo_ready) {
  if (kind != BP_PLAIN && kind != BP_ONES && kind != BP_MULT) return hipErrorNotSupported;
  if (tile_misfit(p)) return hipErrorNotSupported;
  const Geo& g = p->geo;
  const TileSizes z = tile_sizes(p, subset, nsubsets);
  if (z.nrays == 0 || z.nvox == 0) return hipSuccess;
  if (scratch_bytes < tile_scratch_bytes(p, subset, nsubsets, geo == nullptr))
    return hipErrorInvalidValue;
  char* sp = (char*)scratch;
  TileZ* zr = (TileZ*)sp;
  sp += align256((size_t)z.nrays * sizeof(TileZ));
  unsigned* nzmask = (unsigned*)sp;
  sp += align256((size_t)z.npair * tile_words(g.nsino) * sizeof(unsigned));
  int* nzp = (int*)sp;
  sp += align256((size_t)z.npair * sizeof(int));
  double* parts = nullptr;
  if (z.nchunk > 1) {
    parts = (double*)sp;
    sp += align256((size_t)z.nchunk * z.nvox * sizeof(double));
  }
  if (!geo) {
    geo = sp;
    geo_ready = false;
  }
  const TileGeoPtrs q = tile_geo_ptrs(z, geo);
  GatherArgs A;
  ZRay* unused_zr = nullptr;
  int* unused_nz = nullptr;
  gather_args_for(p, subset, nsubsets, kind, sino, img, nullptr, A, unused_zr, unused_nz);
  A.nz_pair = nzp;
  if (fuse) {
    A.upd_sens = fuse->sens;
    A.fresh = fuse->sens ? kFresh : fuse->fresh;
    A.upd_thr = fuse->thr;
    A.upd_thr_at = fuse->thr_at;
    A.upd_strict = fuse->strict;
  }
  // the subset's geometry: the rays of every tile with their paths
  if (!geo_ready)
    hipLaunchKernelGGL(tile_rays_kernel, dim3(z.ntiles), dim3(kGBlock), 0, st, A, z.maxc, z.nslot,
                       q.rays, q.pairs, q.count, q.order);
  // the call's axial records with their bin values, and the (angle, r) with a non-zero bin
  hipLaunchKernelGGL(tile_zsetup_kernel, dim3((g.nr + kTZBins - 1) / kTZBins, z.nang_sub),
                     dim3(kGBlock), 0, st, A, zr, nzmask, nzp);
  hipLaunchKernelGGL(tile_bp_kernel, dim3((unsigned)(z.ntiles * z.nslab * z.nchunk)), dim3(kWave),
                     tile_lds_bytes(z.zs), st, A, z.zs, z.nslab, z.nchunk, (const int*)q.order,
                     (const TileRay*)q.rays, (const int*)q.pairs, (const int*)q.count, z.nslot,
                     (const TileZ*)zr, (const unsigned*)nzmask, p->d_zinc, parts);
  if (parts)
    hipLaunchKernelGGL(tile_reduce_kernel, dim3(ggrid(z.nvox)), dim3(kGBlock), 0, st, A, z.nvox,
                       z.nchunk, (const double*)parts);
  return hipGetLastError();
}

// Bytes of the z-crossing table for a subset of nang_sub angles; 0 (no table: the
// gather reconstructs z crossings with alpha_after) above 1 GiB, e.g. for MLEM over
// all angles of a large sinogram.
size_t ztable_bytes(const apirl_plan* p, int nang_sub) {
  const size_t bytes = (size_t)nang_sub * p->geo.nr * (size_t)p->zblock * sizeof(float);
  return (p->d_zsoff && bytes <= ((size_t)1 << 30)) ? bytes : 0;
}

void gather_args_for(const apirl_plan* p, int subset, int nsubsets, int kind, const float* sino,
                     float* img, void* scratch, GatherArgs& A, ZRay*& zr, int*& nz_pair) {
  const Geo& g = p->geo;
  const int nang_sub = subset_num_angles(g.nang, nsubsets, subset);
  const long nrays = (long)g.nsino * nang_sub * g.nr;
  A.g = g;
  A.rays = p->d_rays;
  A.zab = p->d_zab;
  const float2* own = p->forms[p->scanner].angcs;
  A.angcs = own ? own : p->d_angcs;
  A.segs = p->d_segs;
  A.nseg = p->nseg;
  A.sino = sino;
  A.img = img;
  A.kind = kind;
  A.nang_sub = nang_sub;
  A.subset = subset;
  A.nsubsets = nsubsets;
  A.zlanes = 1;
  zr = nullptr;
  nz_pair = nullptr;
  A.ztab = nullptr;
  A.zsoff = p->d_zsoff;
  A.zblock = p->zblock;
  A.xytab = p->d_xytab;
  A.angcs_odd = p->d_angcs_odd;
  A.rlut = p->d_rlut;
  A.rl0 = p->rl0;
  A.rl_inv_h = p->rl_inv_h;
  A.nrl = p->nrl;
  // the column kernel's sector order when selected and built for the current depth
  const int zv = p->gather_zvox;
  const bool wedge = p->gather_xcd == APIRL_GATHER_XCD_WEDGES && zv >= 1 && zv <= 4 &&
                     p->d_tilemap[zv];
  A.tile_map = wedge ? p->d_tilemap[zv] : nullptr;
  A.tile_slots = wedge ? p->tilemap_slots[zv] : 0;
  if (g.dims == 3 && scratch) {
    // scratch: [ZRay x nrays][non-zero flag per (angle, r)][z-crossing table]
    const size_t npair = (size_t)nang_sub * g.nr;
    zr = (ZRay*)scratch;
    nz_pair = (int*)((char*)scratch + (size_t)nrays * sizeof(ZRay));
    if (ztable_bytes(p, nang_sub) > 0)
      A.ztab = (float*)((char*)scratch + (size_t)nrays * sizeof(ZRay) +
                        (npair * sizeof(int) + 255) / 256 * 256);
  }
  A.zr = zr;
  A.nz_pair = nz_pair;
  A.maxc = gather2_candidates(g);
  A.upd_sens = nullptr;
  A.fresh = 0;
  A.upd_thr = 0.f;
  A.upd_thr_at = nullptr;
  A.upd_strict = 0;
}

hipError_t launch_group_gather(BatchHeader* hdr, const GJob* jobs, int grid, hipStream_t st) {
  hipLaunchKernelGGL(gather2_group_kernel, dim3(grid), dim3(kG2Waves * kWave),
                     kG2LdsFloats * sizeof(float), st, hdr, jobs);
  return hipGetLastError();
}

bool gather2_takes(const apirl_plan* p, int subset, int nsubsets) {
  const Geo& g = p->geo;
  if (g.dims != 2 || g.ns * g.nas != 1 || !p->gather_ok) return false;
  const int nang_sub = subset_num_angles(g.nang, nsubsets, subset);
  return nang_sub > 0 && gather2_fits(g, gather2_candidates(g), nang_sub);
}

const char* gather_misfit(const apirl_plan* p, int subset, int nsubsets) {
  const Geo& g = p->geo;
  if (g.dims != 3) return nullptr;
  const long nang_sub = subset_num_angles(g.nang, nsubsets, subset);
  const long npair = nang_sub * g.nr;
  const long lim24 = 1L << 24;
  if ((long)g.nsino * npair >= (1L << 31)) return "the subset has 2^31 bins or more";
  if (npair >= lim24) return "the subset has 2^24 (angle, radial bin) pairs or more";
  if (g.nsino >= lim24) return "the sinogram count reaches 2^24";
  if (p->zblock >= lim24) return "the z-crossing table slots reach 2^24 entries";
  // the table offset e * npair (e < zblock) is a 32-bit product; the table exists only
  // below 1 GiB, 2^28 floats, which keeps it there, and this says so explicitly
  if (ztable_bytes(p, (int)nang_sub) > 0 && (unsigned long)p->zblock * npair >= (1UL << 32))
    return "the z-crossing table offsets reach 2^32";
  return nullptr;
}

void build_wedge_tile_map(int ntx, int nty, int nzb, std::vector<int>& map) {
  constexpr int kX = 8;  // XCDs; the hardware deals workgroup b to XCD b % 8
  std::vector<int> wedge((size_t)ntx * nty);
  const double kPi = 3.14159265358979323846;
  for (int ty = 0; ty < nty; ty++)
    for (int tx = 0; tx < ntx; tx++) {
      const double cx = tx + 0.5 - ntx / 2.0, cy = ty + 0.5 - nty / 2.0;
      int w = (int)std::floor((std::atan2(cy, cx) + kPi) / (2 * kPi / kX));
      wedge[(size_t)ty * ntx + tx] = w < 0 ? 0 : (w >= kX ? kX - 1 : w);
    }
  std::vector<std::vector<int>> lists(kX);
  for (int tz = 0; tz < nzb; tz++)
    for (int ty = 0; ty < nty; ty++)
      for (int tx = 0; tx < ntx; tx++)
        lists[wedge[(size_t)ty * ntx + tx]].push_back(tx + ntx * (ty + nty * tz));
  size_t len = 0;
  for (auto& l : lists) len = l.size() > len ? l.size() : len;
  map.assign(len * kX, -1);
  for (int x = 0; x < kX; x++)
    for (size_t k = 0; k < lists[x].size(); k++) map[k * kX + x] = lists[x][k];
}

bool gather_fits(const apirl_plan* p, int subset, int nsubsets) {
  return gather_misfit(p, subset, nsubsets) == nullptr;
}

size_t gather_scratch_bytes(const apirl_plan* p, int subset, int nsubsets) {
  const Geo& g = p->geo;
  if (g.dims != 3) return 0;
  const int nang_sub = subset_num_angles(g.nang, nsubsets, subset);
  const long nrays = (long)g.nsino * nang_sub * g.nr;
  const size_t npair = (size_t)nang_sub * g.nr;
  return (size_t)nrays * sizeof(ZRay) + (npair * sizeof(int) + 255) / 256 * 256 +
         ztable_bytes(p, nang_sub);
}

}  // namespace apirl
