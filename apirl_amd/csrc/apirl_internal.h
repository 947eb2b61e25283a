// Internal types shared by the host side (capi.cpp, geometry.cpp) and the gfx950
// kernels (siddon_kernels.hip).  Not part of the C-ABI.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <string>
#include <vector>

#include "apirl_hip.h"

namespace apirl {

// Per-LOR (angle, r) part of the Siddon setup that depends only on the transaxial
// geometry: recon/src/Siddon.cpp:83-145 (square-FOV alpha clip and clamp),
// :148-152/:494-498 (entry/exit points), :177-181/:509-512 (entry indices),
// :253-286/:583-606 (alpha increments and first crossings) and the xy part of the
// ray length (:248-250/:579-580).  Computed on the host in float with the reference's
// operation order and uploaded once; 64 bytes so one lane reads one line.
struct alignas(16) RayXY {
  float p0x, p0y;  // LOR.P0 (P1 of the bin)
  float vx, vy;    // LOR.Vx, LOR.Vy = P2 - P1
  float amin, amax;
  float ax, ay;    // first x / y crossing (2D: negative values clamped to amin)
  float axu, ayu;  // |dx / Vx|, |dy / Vy|
  float lxy;       // ((P0.X+Vx)-P0.X)^2 + ((P0.Y+Vy)-P0.Y)^2
  int i0, j0;      // entry voxel indices (may be -1 or n)
  int nxy;         // |imax - imin| + |jmax - jmin|
  int flags;       // see RAY_* below
  float len;       // sqrtf(lxy): the ray length of a 2D LOR
};
static_assert(sizeof(RayXY) == 64, "RayXY must be one 64-byte line");

enum : int {
  RAY_VALID = 1,     // 2D: r <= rfov (Sinogram2DinCylindrical3Dpet.cpp:256-260)
  RAY_REJECTED = 2,  // 2D: both ends outside on one side (Siddon.cpp:515-519)
  RAY_XMAJOR = 64,   // |Vx| > |Vy|: neighbouring radial bins are offset along y
};
__host__ __device__ inline int ray_iinc(int flags) { return ((flags >> 2) & 3) - 1; }
__host__ __device__ inline int ray_jinc(int flags) { return ((flags >> 4) & 3) - 1; }
inline int ray_flags(int iinc, int jinc, int valid, int rejected) {
  return (valid ? RAY_VALID : 0) | (rejected ? RAY_REJECTED : 0) | ((iinc + 1) << 2) |
         ((jinc + 1) << 4);
}

// Geometry constants passed by value to every kernel.
struct Geo {
  int nx, ny, nz;
  float dx, dy, dz;
  float R;     // (dx * nx) / 2, Images.cpp:55
  float offz;  // dz / 2, Siddon.cpp:162
  int nr, nang, nsino;
  int dims;
  float r0, dr, rmargin;  // uniform radial grid r_j = r0 + j dr (gather candidate search)
  int walk24;  // voxel indices fit 24-bit multiplies (nx ny, nx, ny, nz below 2^23)
  int ns, nas;  // LORs per bin: transaxial x axial samples (oversampled 3D Siddon)
};

// A run of consecutive sinograms with increasing mean axial coordinate and ends that do not
// move back (one segment of the reference's enumeration): zmean(first + l) ~ z0 + l h.  The gather
// backprojector starts its sinogram scan at the index this line predicts for a ray
// of typical axial slope dlo (the middle sinogram's zb - za); dhi holds 1 / h.  The
// tile backprojector bounds the run's axial slopes zb - za by [dmin, dmax] and the
// deviation of zmean from the line by devz.
struct GatherSeg {
  int first, count;
  float z0, h, dlo, dhi, margin;
  int pad;
  float dmin, dmax, devz;
  int pad2;
};

// One geometry of a plan's LOR endpoints (APIRL_SCANNER_*) with the tables the
// projectors and the gather read for it.  A plan keeps every form it has built and
// points its active tables (apirl_plan::d_rays ...) at one of them.
struct LorForm {
  RayXY* rays = nullptr;        // [nang][nr][ns]
  float* xytab = nullptr;       // [nang][nr][nx + ny] gather entry crossings, or null
  float2* angcs = nullptr;      // [nang] the angles' (cos, sin); null: the plan's
  float2* angcs_odd = nullptr;  // [nang] odd bins' (cos, sin) (radial lookup search)
  int2* rlut = nullptr;         // radial position -> bin range; null on a uniform grid
  float rl0 = 0.f, rl_inv_h = 0.f;
  int nrl = 0;
  int tile_maxc = 0;            // with rlut: candidate bins of a tile and angle at most
  bool built = false;
  bool gather = false;          // the gather's tables exist for this form
  // APIRL_PREC_F64_SETUP tables of the gather's column kernel, built on its first
  // use: the rays with the double setup's entry voxel, list length, alpha range and
  // first crossings (rounded to float), and their entry-crossing table
  RayXY* rays_f64s = nullptr;
  float* xytab_f64s = nullptr;
};

}  // namespace apirl

struct apirl_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;
  // this device's copy of the file-scope partials array of apirl_project_ratio_noalloc
  // (hipGetSymbolAddress, taken once per device); null if that failed
  double* d_noalloc = nullptr;
  // scratch owned by the context (likelihood partials, reductions)
  double* d_red = nullptr;
  size_t red_cap = 0;
  bool red_captured = false;     // a graph reads d_red
  std::vector<void*> retired;    // ones that graphs read, kept until the context ends
  float* d_fred = nullptr;
  unsigned long long* d_ured = nullptr;
};

struct apirl_plan {
  apirl_ctx* ctx = nullptr;
  apirl_image_desc img{};
  apirl_sino_desc sino{};   // pointers inside are not kept
  apirl::Geo geo{};
  apirl::RayXY* d_rays = nullptr;  // [nang][nr][ns]
  float2* d_zab = nullptr;         // [nsino][nas] (P1.Z, P2.Z), 3D only
  // [16][nvox] per-XCD scatter targets, 8 in the image layout and 8 transposed
  // ([z][x][y]), allocated on the first scatter backprojection and zero between calls
  float* d_replicas = nullptr;
  bool replicas_failed = false;    // their allocation failed: direct atomics on the image
  // Oversampled plans (ns x nas LORs per bin): one plan of one LOR per bin for each
  // radial sub-LOR o and axial sample q (index o * nas + q), whose gathers add up to
  // the oversampled backprojection; built on the first gather, freed with the plan or
  // when the oversampling changes
  std::vector<apirl_plan*> os_parts;
  // copy of the projected image: in 3D with z fastest (path_image_floats), or transposed
  // ([nz][nx][ny]) for a ray per lane
  float* d_imgT = nullptr;
  int* d_zorder = nullptr;         // [nsino] sinograms sorted by mean axial coordinate
  float2* d_angcs = nullptr;       // [nang] (cos, sin) for the gather candidate search
  apirl::GatherSeg* d_segs = nullptr;
  int nseg = 0;
  bool gather_ok = false;          // uniform radial grid and increasing runs found
  int gather_zlanes = 1;           // 3D gather voxel mapping (1: 16x16 slice tiles; Z>1:
                                   // Z slices x 64/Z columns per wavefront)
  int gather_zvox = 3;             // 3D gather voxels per lane along z (1..4, tiles only)
  int gather_xcd = APIRL_GATHER_XCD_WEDGES;  // column kernel's tile order
  int tile_zs = 0;                 // tile backprojector's slab depth (0: tile_slab_depth's)
  float* d_zinc = nullptr;         // [nsino] z-crossing increment |dz / Vz|, negative for Vz < 0
  bool slices16 = false;           // every slice index of its rays fits 16 bits
  // its geometry per (LOR form, subset, subsets), kept from the first call on, within
  // tile_geo_budget bytes in all (apirl_tuning.tile_cache_mb); `ready` once the launch
  // that builds it is enqueued on `stream`, whose event `ev` follows it
  struct TileGeo {
    int form, subset, nsubsets;
    void* d;
    size_t bytes;
    bool ready;
    bool captured;  // a graph reads it
    hipStream_t stream;
    hipEvent_t ev;
  };
  std::vector<TileGeo> tile_geo;
  size_t tile_geo_used = 0;
  size_t tile_geo_budget = (size_t)16384 << 20;
  // its tile maps (APIRL_GATHER_XCD_WEDGES), one per voxels-per-lane depth 1..4, built
  // on first use and kept until the plan ends (captured launches may hold them)
  int* d_tilemap[5] = {};
  int tilemap_slots[5] = {};
  void* d_gscratch = nullptr;      // per-ray axial setup of the gather (grown on demand)
  float* d_divbins = nullptr;      // DivideAndBackproject's bin values for the gather
  size_t divbins_cap = 0;          //   (grown on demand)
  int* d_zsoff = nullptr;          // [2 nsino + 1] z-crossing table slots, first slices
  float* d_xytab = nullptr;        // [nang][nr][nx + ny] entry crossings (gather)
  int zblock = 0;                  // z-crossing table entries per (angle, radial bin)
  size_t gscratch_bytes = 0;
  bool gscratch_captured = false;  // a graph reads d_gscratch
  size_t gscratch_refused = SIZE_MAX;  // as much could not be allocated
  // scratch and tile geometry that graphs read, kept until the plan ends
  std::vector<void*> retired;
  std::vector<float> ang, r;       // host copies of the grids
  std::vector<float2> zab;         // [nsino] one axial sample per bin
  std::vector<float> z1m, z2m;     // [nsino] mean ring coordinates of each sinogram
  bool gather_tables = false;      // the gather's candidate-search tables common to every
                                   // LOR form (angle directions, segment runs, z slots)
  bool uniform_r = true;           // the plan's radial grid is uniform (closed-form search)
  float2* d_angcs_odd = nullptr;   // [nang] odd bins' (cos, sin) (mMR gather search)
  int2* d_rlut = nullptr;          // [nrl] radial position -> bin range (mMR gather search)
  float rl0 = 0.f, rl_inv_h = 0.f;
  int nrl = 0;
  int scanner = 0;                 // APIRL_SCANNER_*: geometry of the LOR endpoints
  apirl::LorForm forms[3];         // per APIRL_SCANNER_*, built on first use; the d_rays,
                                   // d_xytab, d_angcs_odd, d_rlut above alias forms[scanner]
};

namespace apirl {
// Points the plan's active LOR tables at form f (built); returns the previous form.
int use_lor_form(apirl_plan* p, int f);
// Builds form f of a 3D plan if needed (host tables, upload).  false: out of memory or
// not defined for the plan (message in the context).
bool build_lor_form(apirl_plan* p, int f);
// Holds form f active for a scope (host-side pointer swap: launches already enqueued
// keep the tables they were given).
struct ActiveForm {
  apirl_plan* p;
  int prev;
  ActiveForm(apirl_plan* plan, int f) : p(plan), prev(use_lor_form(plan, f)) {}
  ~ActiveForm() { use_lor_form(p, prev); }
};
}  // namespace apirl

namespace apirl {

// geometry.cpp
void build_ray_table(const apirl_image_desc& img, const apirl_sino_desc& sino,
                     const std::vector<float>& ang, const std::vector<float>& r,
                     std::vector<RayXY>& out);
void build_z_table(const apirl_sino_desc& sino, std::vector<float2>& zab);
// Ray records from explicit transaxial LOR endpoints (x1, y1, x2, y2) per bin; ok[n]
// false marks a LOR the geometry rejects.
void build_ray_table_pts(const apirl_image_desc& img, bool is2d, const std::vector<float4>& pts,
                         const std::vector<char>& ok, std::vector<RayXY>& out);
// Siemens Biograph mMR LOR endpoints of a nang x nr sinogram.
void mmr_lor_points(int nang, int nr, std::vector<float4>& pts);
// The LORs of the reference's mMR subset sinograms (APIRL_SCANNER_MMR_SUBSET):
// cylindrical, on the radius 328 mm, at the mMR's radial positions and angles.
void mmr_subset_lor_points(int nang, int nr, std::vector<float4>& pts);
// Oversampled bins (SiddonProjector.cpp:374-395, Sinogram2DinCylindrical3Dpet.cpp:
// 283-299): ns radial sub-LORs per bin and nas axial ones per sinogram.
void build_subsample_r(const std::vector<float>& r, int ns, std::vector<float>& r_sub);
void build_z_table_os(const std::vector<float>& z1m, const std::vector<float>& z2m,
                      float ring_width, int nas, std::vector<float2>& zab);
int subset_num_angles(int nang, int nsubsets, int subset);

// siddon_kernels.hip: launchers (enqueue on stream; return hipError_t)
struct FusedRatio {
  const float* meas = nullptr;      // full sinogram
  const float* additive = nullptr;  // full sinogram or null
  float* ratio = nullptr;           // subset sinogram
  double* lik_partials = nullptr;   // one per block, or null
  int lik_positive_only = 0;
  // angle of the additive sinogram added to bin (s, k, r) of subset `subset`:
  // 0 = the bin's own angle subset + nsubsets k; 1 = k, the subset-local index into
  // the full additive sinogram, as OsemSinogram3d.cpp:172-173 with
  // Sinogram3D::addBinToBin (Sinogram3D.cpp:857-873) reads it
  int additive_local = 0;
  int max_partials = 0;
};
// The fused form writes project_partials likelihood partials, one per workgroup.  With
// FusedRatio::max_partials (max_partials below) the path projector, which has one or more per
// (angle, bin), runs only where that holds them; a ray per lane has one per 256 bins.
// image_copy: where the projector's copy of the image goes (path_image_floats floats in 3D,
// the image's in 2D) instead of the plan's own buffer, for work on a stream of its own.
hipError_t launch_project(const apirl_plan* p, const float* img, float* sino, int subset,
                          int nsubsets, int precision, const FusedRatio* fused, int* nblocks_out,
                          hipStream_t st, float* image_copy = nullptr);
bool path_forward_ok(const apirl_plan* p, int precision, int subset, int nsubsets,
                     int max_partials = 0);
// Floats of the path forward projector's z-fastest image copy (apirl_plan::d_imgT).
size_t path_image_floats(const Geo& g);
int project_partials(const apirl_plan* p, int subset, int nsubsets, int precision,
                     int max_partials = 0);
hipError_t launch_backproject(const apirl_plan* p, const float* sino, const float* est,
                              float* img, int subset, int nsubsets, int kind, int mode,
                              hipStream_t st);
// zeroes the scatter's n-float image copies (device-scope stores, as the reduction
// clears them)
hipError_t launch_zero_floats(float* x, size_t n, hipStream_t st);
hipError_t launch_em_update(float* x, const float* b, const float* s, size_t n, float thr,
                            int strict, hipStream_t st);
hipError_t launch_force_positive(float* x, size_t n, hipStream_t st);
// DivideAndBackproject's per-bin value (3D and 2D rules) into out, for its gather form.
hipError_t launch_divide_rule(const float* meas, const float* est, float* out, size_t n,
                              int dims, hipStream_t st);
hipError_t launch_sum_partials(const double* partials, int n, double* out, hipStream_t st);
// Sums of rows of partials, stride apart: row r's first nmore where r % nsubsets < more, its
// first nless otherwise, to out[r], each in launch_sum_partials' order.
hipError_t launch_sum_partials_rows(const double* partials, int rows, long stride, int nsubsets,
                                    int more, int nmore, int nless, double* out, hipStream_t st);
// Partials of apirl_project_ratio_noalloc: a file-scope device array of
// siddon_kernels.hip of kNoallocPartials doubles (one per workgroup, of 256 bins at least where
// there are as many as APIRL_NOALLOC_MAX_BINS).
constexpr int kNoallocPartials = 1 << 19;
// The current device's address of that array (hipGetSymbolAddress).
hipError_t noalloc_scratch_address(double** out);
// The one-LOR-per-bin plans of an oversampled plan (apirl_plan::os_parts); false with
// the context's error set when they cannot be built.
bool ensure_os_parts(apirl_plan* p);
// The rays of an APIRL_PREC_F64_SETUP gather: each ray's transaxial setup carried out
// in double from its float LOR (setup_xy_f64), rounded to float as the projector's
// F64_SETUP loop starts from it.
void build_f64s_rays(const Geo& g, const std::vector<RayXY>& rays, std::vector<RayXY>& out);
void free_os_parts(apirl_plan* p);
// Likelihood sum y log(x) - x over x > 0 (positive_only) or x != 0, deterministic:
// block partials into `partials`, then a fixed-order sum into *out.
hipError_t launch_likelihood(const float* x, const float* y, long n, int positive_only,
                             double* partials, double* out, hipStream_t st);
// The MLEM update threshold from a sensitivity's smallest non-zero and largest value (Mlem.cpp:41).
__host__ __device__ inline float mlem_threshold(float least, float most) {
  return least + (most - least) * 0.0001f;
}
// d_out: [min_nz, max] and 2 kMinMaxBlocks floats of scratch.  d_thr: null, or where the MLEM
// threshold of a sensitivity x goes (mlem_threshold).
constexpr int kMinMaxBlocks = 512;
constexpr size_t kMinMaxFloats = 2 + 2 * (size_t)kMinMaxBlocks;
hipError_t launch_min_nz_max(const float* x, size_t n, float* d_out, float* d_thr, hipStream_t st);
hipError_t launch_count_intersections(const apirl_plan* p, int subset, int nsubsets,
                                      unsigned long long* d_out, hipStream_t st);

// The EM update a gather can apply to its voxels instead of storing their
// backprojection (GatherArgs::upd_sens): img is then the image being updated.  Or, with fresh
// (GatherArgs::fresh) and no sens, how a backprojection is stored whose image need not be cleared.
struct EmFuse {
  const float* sens;
  float thr;
  int strict;
  const float* thr_at = nullptr;  // device: the threshold, in place of thr
  int fresh = 0;
};
constexpr int kFresh = 1, kFreshPositive = 2;  // as it is; forcePositive applied
// The 2D gather by patches runs this subset's backprojection; the scatter form, whose atomics it
// outruns everywhere (34 / 19 us for 32 x 32 from 8 x 40 bins, 319 / 82 from 252 x 344; 164 / 20
// for 256 x 256 from 24 x 76, 531 / 99 from 252 x 320), then does too.
bool gather2_takes(const apirl_plan* p, int subset, int nsubsets);
hipError_t launch_backproject_gather(const apirl_plan* p, const float* sino, float* img,
                                     int subset, int nsubsets, int kind, int precision,
                                     void* scratch, size_t scratch_bytes, hipStream_t st,
                                     const EmFuse* fuse = nullptr);
// Tile-walk backprojector; tile_misfit says why a plan cannot take it (null when it can).
// Its geometry for one subset (the rays of every tile and their paths; tile_geo_bytes)
// depends on the plan's LOR form alone: with `geo` null it is built in the scratch on every
// call; otherwise it lives in `geo`, built there when `geo_ready` is false and reused as it
// stands when true.  The scratch (tile_scratch_bytes, with the geometry when `geo` is null)
// holds the call's axial records with their bin values and the sums of its chunks.
hipError_t launch_backproject_tile(const apirl_plan* p, const float* sino, float* img,
                                   int subset, int nsubsets, int kind, void* scratch,
                                   size_t scratch_bytes, hipStream_t st, const EmFuse* fuse,
                                   void* geo, bool geo_ready);
const char* tile_misfit(const apirl_plan* p);
// Candidate bins (even and odd ones counted alike) of one tile and angle at the most, on the
// radial grid of a lookup table.
int tile_lut_candidates(const Geo& g, const std::vector<int2>& lut, float inv_h);
// A batched 3D job's backprojections (one LOR per bin), as apirl_backproject runs them for
// APIRL_BP_GATHER, on any stream with a scratch of the job's own.  job_scratch_bytes: what a
// subset needs, after the memory of its kept geometry has been taken.  job_footprint: what the
// subsets of a job would need, scratch (their largest) and kept geometry that the plan does not
// hold yet, for a plan of one LOR per bin (parts: as many plans like it, sharing its budget).
size_t job_scratch_bytes(apirl_plan* p, int subset, int nsubsets);
void job_footprint(const apirl_plan* p, int nsubsets, int parts, size_t& scratch,
                   size_t& geometry);
hipError_t job_backproject(apirl_plan* p, const float* sino, float* img, int subset, int nsubsets,
                           int kind, const EmFuse* fuse, void* scratch, size_t scratch_bytes,
                           hipStream_t st);
size_t tile_geo_bytes(const apirl_plan* p, int subset, int nsubsets);
size_t tile_scratch_bytes(const apirl_plan* p, int subset, int nsubsets, bool with_geo);
size_t gather_scratch_bytes(const apirl_plan* p, int subset, int nsubsets);
// The 3D gather's 32-bit record and table offsets hold for this subset (fewer than
// 2^31 subset bins; angle x radial bins, sinograms and crossing-table slots below 2^24).
bool gather_fits(const apirl_plan* p, int subset, int nsubsets);
// Tile order of the column kernel that keeps each XCD on one angular sector of the
// image (APIRL_GATHER_XCD_WEDGES): 8 lists of tiles, one per 45-degree wedge about
// the image centre, z-block by z-block, interleaved so that slot b goes to list
// b % 8, the XCD that the hardware dispatches workgroup b to; -1 pads the lists.
void build_wedge_tile_map(int ntx, int nty, int nzb, std::vector<int>& map);
// Why a subset does not fit the gather's 32-bit offsets (nullptr when it fits).
const char* gather_misfit(const apirl_plan* p, int subset, int nsubsets);
size_t ztable_bytes(const apirl_plan* p, int nang_sub);
void build_xy_crossings(const apirl_image_desc& img, const std::vector<RayXY>& rays,
                        std::vector<float>& out);
// Radial positions of the mMR's bins (ascending) and the (cos, sin) of each angle's
// even and odd bins (half an angular step less), as the mMR LOR endpoints use them.
void mmr_radial_grid(int nang, int nr, std::vector<float>& r, std::vector<float2>& angcs,
                     std::vector<float2>& angcs_odd);
// Lookup table from a radial position to the range of bins around it, on a grid of
// spacing h from rl0 covering the ascending positions r with two points to spare:
// lut[k] = (first j with r[j] >= rl0 + k h, last j with r[j] <= rl0 + k h).
void build_radial_lut(const std::vector<float>& r, std::vector<int2>& lut, float& rl0,
                      float& inv_h);
void build_gather_tables(const apirl_plan& p, std::vector<float2>& angcs,
                         std::vector<GatherSeg>& segs, float& r0, float& dr, float& rmargin,
                         bool& ok);

// Backprojection kinds
enum { BP_PLAIN = 0, BP_ONES = 1, BP_DIVIDE = 2, BP_MULT = 3 };

// ---- batched jobs (batch.cpp, grouped kernels) --------------------------------
// A round runs one OSEM / MLEM sub-iteration of every active 2D job with one launch
// per phase; each launch walks a job table in device memory.  Every job owns a
// contiguous run of "virtual blocks" (first .. next job's first) of that phase;
// the launches are persistent (fixed grid) and their workgroups take virtual blocks
// from a per-phase counter (dynamic balance: tiles differ ~10x in cost), so the
// launch shapes never change and one captured graph serves every round.

// Per-ray axial part of the Siddon setup and the bin value of one subset bin, used
// by the gather backprojector (one 32-byte load per candidate ray).
struct alignas(32) ZRay {
  int k0;       // entry slice
  short k1;     // exit slice
  short kinc;   // sign of Vz
  float azu;    // |dz / Vz|
  float az0;    // first z crossing (FLT_MAX when Vz == 0)
  float L;      // ray length |P2 - P1| in the reference's operand order
  float b;      // bin value being backprojected
  int zcount;   // z crossings of the ray held by the crossing table (the rest: alpha_after)
  int pad;
};
static_assert(sizeof(ZRay) == 32, "ZRay is one 32-byte load");

struct GatherArgs {
  Geo g;
  const RayXY* rays;
  const float2* zab;
  const float2* angcs;  // (cos, sin) of every angle of the full sinogram
  const GatherSeg* segs;
  int nseg;
  const ZRay* zr;
  const int* nz_pair;
  const float* sino;  // subset sinogram (PLAIN), full sinogram (MULT) or null (ONES)
  float* img;
  int kind;           // BP_PLAIN, BP_ONES or BP_MULT
  int nang_sub, subset, nsubsets;
  int zlanes;         // voxel mapping (see gather_kernel)
  // z-crossing table: for every subset ray, the reference's accumulated z crossing
  // by which it enters slice k, at ztab[((zsoff[s] + k - kmin[s]) * nang_sub + ka) * nr + r]
  float* ztab;
  const int* zsoff;   // [nsino + 1] slot offsets, then [nsino] first slice kmin per sinogram
  int zblock;
  // x / y crossing table of the plan: xytab[(a * nr + r) * (nx + ny) + i] is the
  // accumulated x crossing by which ray (a, r) enters column i, [... + nx + j] the y
  // crossing by which it enters row j
  const float* xytab;
  // Candidate search on a non-uniform radial grid with odd bins at their own angle
  // (mMR; null for the plan's uniform grid): angcs_odd[a] is the (cos, sin) of the
  // odd bins of angle a; rlut[k] = (first bin with r >= rl0 + k h, last bin with
  // r <= rl0 + k h), k < nrl, rl_inv_h = 1 / h.
  const float2* angcs_odd;
  const int2* rlut;
  float rl0, rl_inv_h;
  int nrl;
  // Column kernel's workgroup order (null: the 3D grid itself): slot b of a 1D grid
  // takes tile tile_map[b] = tx + ntx (ty + nty tz), or nothing when it is -1.
  const int* tile_map;
  int tile_slots;
  // EM update fused into the gather (null: img accumulates the backprojection): img is
  // then the image x, and each voxel's backprojection b, summed from zero, updates it
  // to (s > thr or, not strict, s >= thr) ? (x b) / s : 0 with s = upd_sens[v]
  const float* upd_sens;
  // not 0: the sums start from zero, not from img (kFresh, as with upd_sens; kFreshPositive);
  // APIRL_PREC_REFERENCE only
  int fresh;
  float upd_thr;
  const float* upd_thr_at;  // null, or (device) the threshold in place of upd_thr
  int upd_strict;
  int maxc;  // 2D: upper bound on a voxel's candidate bins of one angle
};

struct BatchHeader {
  long total[2];                // virtual blocks of each phase (BatchPhase)
  int count[2];                 // jobs in each phase's table
  unsigned long long next[2];   // work counters (uploaded as 0 with every round's table)
  int grab;                     // virtual blocks a workgroup takes per counter draw (>= 1)
  int pad;
};
enum BatchPhase { PH_PROJ2 = 0, PH_GATHER2 };

struct ProjJob {  // fused projection + ratio of one subset (likelihood not taken)
  Geo g;
  const RayXY* rays;
  const float* img;
  FusedRatio fr;
  int nang_sub, subset, nsubsets, pad;
  long nrays;
  long first;
};
struct GJob {  // gather backprojection of one subset with the update fused in (8 x 8 patches)
  GatherArgs A;
  int ntx, nty;
  long first;
};
constexpr int kGroupRays = 64;       // rays of a virtual block of the grouped projection
constexpr int kGroupProject = 512;   // and its threads
inline long group_blocks(long n) { return (n + kGroupRays - 1) / kGroupRays; }
constexpr int kPatch2 = 8;  // the 2D gather's voxel patches are kPatch2 x kPatch2
inline long gather_patches(const Geo& g) {
  return (long)((g.nx + kPatch2 - 1) / kPatch2) * ((g.ny + kPatch2 - 1) / kPatch2);
}

hipError_t launch_group_project(BatchHeader* hdr, const ProjJob* jobs, int grid, hipStream_t st);
hipError_t launch_group_gather(BatchHeader* hdr, const GJob* jobs, int grid, hipStream_t st);
void gather_args_for(const apirl_plan* p, int subset, int nsubsets, int kind, const float* sino,
                     float* img, void* scratch, GatherArgs& A, ZRay*& zr, int*& nz_pair);

}  // namespace apirl
