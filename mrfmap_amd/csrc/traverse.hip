// Ray traversal for the BP inference path: pixel ray set-up, integer 3-D DDA
// over the brick grid, brick activation and emission of per-ray incidence
// lists.
//
// Replaces GVDB's hierarchical DDA `rayCast` + PREPARE_DDA_LEAF / NEXT_DDA /
// STEP_DDA as driven by render_cumulative_length_kernel and
// render_factors_to_node_kernel (src/cuda/gvdbkernels.cu:1164-1226,
// 1276-1302), and the endpoint activation of GVDBCamera::reprojectAndActivate
// -> GVDBMRFMap::activateSpace (src/GVDBCamera.cpp:70-112,
// src/GVDBMRFMap.cpp:117-135).
//
// Traversal rule (the contract the CPU oracle restates):
//  * ray of pixel (x, y): origin O = t/res + off, direction per metre of planar
//    depth D = R ((x-cx)/fx, (y-cy)/fy, 1) / res, both in voxel units and
//    rounded to fixed point Oi = rint(O 2^16), Di = rint(D 2^16);
//  * the ray is walked from max(0, box entry) through the voxel grid; every
//    voxel boundary crossing is the exact rational z = (k 2^16 - Oi_a) / Di_a,
//    compared by 64-bit cross multiplication, ties step all tied axes at once;
//  * a voxel is emitted when its brick is active, with chord length
//    l = (z_exit - z_entry) |D| evaluated in IEEE double from the rationals;
//    a run of skipped voxels after the first emission becomes one gap record;
//  * at the exit of every active brick the walk stops if
//    z + bias(z) >= d + 3 sigma(z) (src/cuda/gvdbkernels.cu:567-570, 1035-1037);
//    leaving the grid first marks the ray kRanOut (the "infinity" term,
//    src/cuda/gvdbkernels.cu:1196-1208).
// The file is compiled with -ffp-contract=off so each double operation is a
// single correctly rounded IEEE operation, as in the host oracle.

#include <algorithm>
#include <cmath>

#include "mrf_internal.h"
#include "mrf_kernels.h"

namespace mrf {

namespace {

__host__ __device__ __forceinline__ int tiled_pixels(const CamGeom& c) {
  return ((c.cols + 7) >> 3) * ((c.rows + 7) >> 3) * 64;
}

struct Rat {
  int64_t n, d;  // value n / d with d > 0
};

__device__ __forceinline__ bool rat_lt(const Rat& a, const Rat& b) { return a.n * b.d < b.n * a.d; }

__device__ __forceinline__ int64_t floor_div(int64_t x, int64_t y, bool* exact) {
  int64_t q = x / y, r = x % y;
  if (r != 0 && x < 0) q -= 1;
  *exact = (r == 0);
  return q;
}

struct RaySetup {
  int64_t Oi[3], Di[3];
  double norm;  // |D| in voxels per metre of planar depth
};

// Returns false for rays whose fixed-point set-up would leave the exact range
// of the 64-bit comparisons (|Oi| >= 2^29 or |Di| >= 2^26).
__device__ bool setup_ray(const CamGeom& c, const GridGeom& g, int x, int y, RaySetup& rs) {
  double ux = ((double)x - c.cx) / c.fx;
  double uy = ((double)y - c.cy) / c.fy;
  double n2 = 0.0;
  for (int a = 0; a < 3; ++a) {
    double dw = c.R[a * 3 + 0] * ux;
    dw = dw + c.R[a * 3 + 1] * uy;
    dw = dw + c.R[a * 3 + 2];
    double D = dw / g.res;
    double O = c.t[a] / g.res;
    O = O + g.off[a];
    double oi = rint(O * kFixScale), di = rint(D * kFixScale);
    if (!(fabs(oi) < 536870912.0) || !(fabs(di) < 67108864.0)) return false;
    rs.Oi[a] = (int64_t)oi;
    rs.Di[a] = (int64_t)di;
    double dd = (double)rs.Di[a] / kFixScale;
    n2 = n2 + dd * dd;
  }
  rs.norm = sqrt(n2);
  return rs.norm > 0.0;
}

// sigma(z) or bias(z) of a lookup cell in double; loaded before a walk, so
// that its loop neither loads them nor, waiting for such a load, waits for
// its own earlier stores.  Two coefficients: c2 = 0, which adds an exact 0.
struct PolyD {
  double c0, c1, c2;
  __device__ __forceinline__ PolyD(const float* c, int n)
      : c0((double)c[0]), c1((double)c[1]), c2(n == 3 ? (double)c[2] : 0.0) {}
  __device__ __forceinline__ double operator()(double s) const { return ((s * s) * c2 + s * c1) + c0; }
};

// Sensor model and truncation test of one ray: whether a walk that leaves an
// active brick at depth z stops there.
struct Truncation {
  PolyD sig, bia;
  double depth;
  __device__ __forceinline__ bool ends(double z) const { return z + bia(z) >= depth + 3.0 * sig(z); }
};

__device__ __forceinline__ bool pixel_valid(const CamGeom& c, int x, int y, float d) {
  if (!(d > 0.0f)) return false;  // NaN, 0 and negatives are invalid
  if (c.mask848 && c.cols == 848 && c.rows == 480 &&
      (x < 24 || x >= c.cols - 24 || y < 20 || y >= c.rows - 20))
    return false;
  return true;
}

__device__ __forceinline__ uint32_t lookup_offset(const CamGeom& c, int lookup_n, int x, int y) {
  int v = c.rows - 1 - y;  // the reference indexes its tables in the vertically flipped image
  return (uint32_t)((v / kLookupPx) * (c.lookup_u * lookup_n) + (x / kLookupPx) * lookup_n);
}

// kEmitAll: emission where every brick on the ray's way is active (full-ray
// activation, whose brick walk marked them)
enum WalkMode { kCount = 1, kEmit = 2, kEmitAll = 3 };

struct WalkOut {
  uint32_t n;
  float z0;
  bool ran_out;
  double last_exit;  // exact exit depth of the last voxel record (kEmit, kEmitAll)
};

// Entry of a pixel ray into the voxel grid: the exact entry depth zin (at
// least 0), the voxel there and the step sign of each axis; false when the
// ray misses the grid.
__device__ __forceinline__ bool ray_entry(const GridGeom& g, const RaySetup& rs, Rat& zin, int ix[3], int sg[3]) {
  const int N[3] = {g.nx, g.ny, g.nz};
  zin = {0, 1};
  Rat zout = {0, 1};
  bool has_out = false;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int64_t Oi = rs.Oi[a], Di = rs.Di[a], top = (int64_t)N[a] << kFix;
    if (Di == 0) {
      if (Oi < 0 || Oi >= top) return false;
      continue;
    }
    Rat lo, hi;
    if (Di > 0) {
      lo = {-Oi, Di};
      hi = {top - Oi, Di};
    } else {
      lo = {Oi - top, -Di};
      hi = {Oi, -Di};
    }
    if (rat_lt(zin, lo)) zin = lo;
    if (!has_out || rat_lt(hi, zout)) {
      zout = hi;
      has_out = true;
    }
  }
  if (!has_out || !rat_lt(zin, zout)) return false;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int64_t Oi = rs.Oi[a], Di = rs.Di[a];
    bool exact;
    int64_t X = Oi * zin.d + zin.n * Di;
    int64_t q = floor_div(X, zin.d << kFix, &exact);
    if (Di < 0 && exact) q -= 1;
    if (q < 0) q = 0;
    if (q > N[a] - 1) q = N[a] - 1;
    ix[a] = (int)q;
    sg[a] = Di > 0 ? 1 : (Di < 0 ? -1 : 0);
  }
  return true;
}

// Front/window split of one ray during its emission, with the ray kernel's
// own FP32 depth sums: the front ends at the first record whose exit depth s
// has d - (s + bias(s)) <= kFrontU * 3 sigma(s).  The Kahan state of the
// front's length sum is kept: the window continues it.
struct FrontSplit {
  Poly sig, bia;
  float z0, inv_norm, depth;
  Kahan kS;
  uint32_t nf;  // the first window record (valid once open is false)
  bool open;
  __device__ __forceinline__ void record(uint32_t k, float ln) {
    if (!open) return;
    const float s = z0 + kS.at(ln) * inv_norm;
    const float sg = sig(s);
    if (!(sg > 0.0f && depth - (s + bia(s)) > kFrontU * (3.0f * sg))) {
      nf = k;
      open = false;
      return;
    }
    kS.add(ln);
  }
};

// The next voxel-face crossing of each axis, t_a = n_a / d_a (n_a grows by
// 2^kFix per step; an axis that does not move has d_a = 0 and n_a = 1), and
// the cross differences X_ab = n_a d_b - n_b d_a (t_a < t_b iff X_ab < 0,
// equal iff 0; positive for an a that does not move against a b that does),
// kept and updated by additions: exact comparisons with no multiplications
// and no run-time indexing in the loop.  which(): the axes that step, every
// axis whose crossing equals the nearest one.  z(): the nearest crossing,
// n / d rounded once.
//
// The walks are bound by their arithmetic (a wavefront step of the emission
// took about 1700 issue cycles with 64-bit integers, whose additions, selects
// and comparisons cost two instructions or more, and with one FP64 division).
// Steps<true> keeps everything in FP64, whose fma runs at full rate, where all
// values are integers below 2^53 (dda_fits_f64): the same exact comparisons,
// selects as fma with a factor 0 or 1, and n / d from the reciprocal of d
// (rounded once, kept) with one residual correction.  That quotient is the
// correctly rounded one.  setup_ray keeps |Oi| below 2^29 and d below 2^26, and
// a grid has at most 2048 voxels an axis (2^27 in units of 2^-kFix), so n is
// below 2^30.  q + r e with e = n - d q exact has a relative error below 2^-100
// before its rounding; n / d and the middle between two doubles differ by at
// least 1 / (d 2^54) of their value, more than 2^-80, or are equal, which would
// take an n of 54 bits.  Rounding keeps the order, so the smallest of the three
// rounded crossings is the rounded nearest crossing.  Steps<false> is the
// general form.  Its quotients and those of the brick walk (mark_bricks) divide
// the same exact doubles, so all three give the same bits, also where the tied
// axes have other numerators: kEmitAll relies on it, since it takes every brick
// it meets for one that the brick walk marked.
template <bool F64>
struct Steps;

template <>
struct Steps<false> {
  int64_t n0, n1, n2, d0, d1, d2, s0, s1, s2, X01, X02, X12;
  __device__ __forceinline__ void init(const int64_t (&n)[3], const int64_t (&d)[3], int fix) {
    n0 = n[0], n1 = n[1], n2 = n[2];
    d0 = d[0], d1 = d[1], d2 = d[2];
    s0 = d0 << fix, s1 = d1 << fix, s2 = d2 << fix;
    X01 = n0 * d1 - n1 * d0, X02 = n0 * d2 - n2 * d0, X12 = n1 * d2 - n2 * d1;
  }
  __device__ __forceinline__ void which(bool& a, bool& b, bool& c) const {
    a = (X01 <= 0) & (X02 <= 0);
    b = (X01 >= 0) & (X12 <= 0);
    c = (X02 >= 0) & (X12 >= 0);
  }
  __device__ __forceinline__ double z() const {
    bool a, b, c;
    which(a, b, c);
    const int64_t ma = -(int64_t)a, mb = -(int64_t)(!a & b), mc = -(int64_t)(!a & !b);  // one of them all ones
    return (double)((n0 & ma) | (n1 & mb) | (n2 & mc)) / (double)((d0 & ma) | (d1 & mb) | (d2 & mc));
  }
  __device__ __forceinline__ void step(bool a, bool b, bool c, int fix) {
    const int64_t one = (int64_t)1 << fix;
    n0 += a ? one : 0;
    n1 += b ? one : 0;
    n2 += c ? one : 0;
    X01 += (a ? s1 : 0) - (b ? s0 : 0);
    X02 += (a ? s2 : 0) - (c ? s0 : 0);
    X12 += (b ? s2 : 0) - (c ? s1 : 0);
  }
};

template <>
struct Steps<true> {
  double n0, n1, n2, d0, d1, d2, r0, r1, r2, s0, s1, s2, X01, X02, X12;
  // an axis that does not move: a huge reciprocal, so that its crossing is last
  __device__ __forceinline__ static double rec(double d) { return d > 0.0 ? 1.0 / d : 1e300; }
  __device__ __forceinline__ void init(const int64_t (&n)[3], const int64_t (&d)[3], int fix) {
    n0 = (double)n[0], n1 = (double)n[1], n2 = (double)n[2];
    d0 = (double)d[0], d1 = (double)d[1], d2 = (double)d[2];
    r0 = rec(d0), r1 = rec(d1), r2 = rec(d2);
    const double one = (double)(1 << fix);
    s0 = d0 * one, s1 = d1 * one, s2 = d2 * one;
    X01 = n0 * d1 - n1 * d0, X02 = n0 * d2 - n2 * d0, X12 = n1 * d2 - n2 * d1;
  }
  __device__ __forceinline__ void which(bool& a, bool& b, bool& c) const {
    a = (X01 <= 0.0) & (X02 <= 0.0);
    b = (X01 >= 0.0) & (X12 <= 0.0);
    c = (X02 >= 0.0) & (X12 >= 0.0);
  }
  __device__ __forceinline__ static double quot(double n, double d, double r) {
    const double q = n * r;
    return fma(fma(-d, q, n), r, q);
  }
  __device__ __forceinline__ double z() const {
    return fmin(quot(n0, d0, r0), fmin(quot(n1, d1, r1), quot(n2, d2, r2)));
  }
  __device__ __forceinline__ void step(bool a, bool b, bool c, int fix) {
    const double fa = a ? 1.0 : 0.0, fb = b ? 1.0 : 0.0, fc = c ? 1.0 : 0.0, one = (double)(1 << fix);
    n0 = fma(fa, one, n0);
    n1 = fma(fb, one, n1);
    n2 = fma(fc, one, n2);
    X01 = fma(-fb, s0, fma(fa, s1, X01));
    X02 = fma(-fc, s0, fma(fa, s2, X02));
    X12 = fma(-fc, s1, fma(fb, s2, X12));
  }
};

// the crossings a ray in voxel ix meets next
template <bool F64>
__device__ __forceinline__ Steps<F64> first_crossings(const RaySetup& rs, const int (&ix)[3]) {
  int64_t n[3], d[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int64_t Oi = rs.Oi[a], Di = rs.Di[a];
    n[a] = Di > 0 ? (((int64_t)ix[a] + 1) << kFix) - Oi : (Di < 0 ? Oi - ((int64_t)ix[a] << kFix) : 1);
    d[a] = Di > 0 ? Di : -Di;
  }
  Steps<F64> st;
  st.init(n, d, kFix);
  return st;
}

// Records of one ray are written out[0], out[kSlice], out[2 kSlice], ... and
// their chord lengths to_len words further on (record k of the 64 rays of a
// pixel tile is contiguous: sliced ELL), the
// first cap of them (the count goes on past cap); vis, when given, splits
// them into front and window (vis->record(k, chord) per record in order,
// vis->z0 the planar depth at the entry of the first).  kEmit looks each
// brick's slot up and writes the voxels' pool ids; kEmitAll needs no look-up
// and writes (linear brick index) * 512 + voxel, so that its loop holds no
// load to wait for (a wait counts the earlier stores too): the copy into the
// final layout turns them into pool ids.
template <int MODE, bool F64>
__device__ __forceinline__ WalkOut walk(const GridGeom& g, const RaySetup& rs, const Truncation& trunc,
                                        const int32_t* __restrict__ slot, uint32_t* __restrict__ out, size_t to_len,
                                        uint32_t cap, FrontSplit* vis = nullptr) {
  constexpr bool kAll = MODE == kEmitAll, kWrites = MODE == kEmit || MODE == kEmitAll;
  WalkOut wo = {0u, 0.0f, true};
  Rat zin;
  int ix[3], sg[3];
  if (!ray_entry(g, rs, zin, ix, sg)) return wo;
  Steps<F64> st = first_crossings<F64>(rs, ix);
  double zc_d = (double)zin.n / (double)zin.d;
  double last_exit = 0.0;
  bool any = false, skipped = false;
  uint32_t cnt = 0;
  auto put = [&](uint32_t vox, float len) {
    out[(size_t)cnt * kSlice] = vox;
    out[(size_t)cnt * kSlice + to_len] = __float_as_uint(len);
  };
  // the brick's slot (kEmitAll: its linear index)
  auto brick_lookup = [&](void) -> int32_t {
    const int lin = ((ix[0] >> kBrickLog) * g.by + (ix[1] >> kBrickLog)) * g.bz + (ix[2] >> kBrickLog);
    return kAll ? lin : slot[lin];
  };
  int32_t bslot = brick_lookup();
  const int max_steps = g.nx + g.ny + g.nz + 3;
  for (int step = 0; step < max_steps; ++step) {
    // per-voxel depths only where records need them; the counting walk converts the exit depth at brick exits alone
    double zn_d = 0.0;
    if constexpr (kWrites) zn_d = st.z();
    const bool active = kAll || bslot >= 0;
    if (active) {
      if (!kAll && any && skipped) {
        if constexpr (kWrites) {
          float gl = (float)((zc_d - last_exit) * rs.norm);
          if (cnt < cap) put(kGapVox, gl);
          if (vis) vis->record(cnt, gl);
        }
        ++cnt;
        skipped = false;
      }
      if (!any) {
        wo.z0 = (float)zc_d;
        if constexpr (kWrites) {
          if (vis) vis->z0 = wo.z0;
        }
        any = true;
      }
      if constexpr (kWrites) {
        const uint32_t local = (uint32_t)((((ix[0] & 7) << 3) | (ix[1] & 7)) << 3 | (ix[2] & 7));
        const uint32_t vox = (uint32_t)bslot * kBrickVox + local;
        const float len = (float)((zn_d - zc_d) * rs.norm);
        if (cnt < cap) put(vox, len);
        if (vis) vis->record(cnt, len);
      }
      ++cnt;
      last_exit = zn_d;
    } else if (any) {
      skipped = true;
    }
    bool st0, st1, st2;
    st.which(st0, st1, st2);
    const int nx[3] = {ix[0] + (st0 ? sg[0] : 0), ix[1] + (st1 ? sg[1] : 0), ix[2] + (st2 ? sg[2] : 0)};
    // the grid is made of whole bricks, so leaving it changes the brick too
    const bool brick_change = (uint32_t)((nx[0] ^ ix[0]) | (nx[1] ^ ix[1]) | (nx[2] ^ ix[2])) >> kBrickLog != 0u;
    ix[0] = nx[0];
    ix[1] = nx[1];
    ix[2] = nx[2];
    if (brick_change) {
      if (active && trunc.ends(kWrites ? zn_d : st.z())) {
        wo.ran_out = false;
        break;
      }
      if ((uint32_t)nx[0] >= (uint32_t)g.nx || (uint32_t)nx[1] >= (uint32_t)g.ny || (uint32_t)nx[2] >= (uint32_t)g.nz)
        break;
      bslot = brick_lookup();
    }
    st.step(st0, st1, st2, kFix);
    zc_d = zn_d;
  }
  wo.n = cnt;
  wo.last_exit = last_exit;
  return wo;
}

struct PixelCtx {
  bool ok;
  int x, y;
  float d;
  RaySetup rs;
  uint32_t cell;
};

// Rays are enumerated in 8x8 pixel tiles (tiles row-major, pixels row-major
// inside a tile) so that rays sharing voxels sit next to each other in the
// lists and run together on the GPU.
__device__ __forceinline__ bool tile_pixel(const CamGeom& c, int t, int* x, int* y) {
  const int ntx = (c.cols + 7) >> 3;
  const int tile = t >> 6, l = t & 63;
  *x = (tile % ntx) * 8 + (l & 7);
  *y = (tile / ntx) * 8 + (l >> 3);
  return *x < c.cols && *y < c.rows;
}

__device__ __forceinline__ PixelCtx load_pixel(const CamGeom& c, const GridGeom& g, const float* depth,
                                               int t) {
  PixelCtx p;
  p.ok = false;
  if (!tile_pixel(c, t, &p.x, &p.y)) return p;
  p.d = depth[p.y * c.cols + p.x];
  if (!pixel_valid(c, p.x, p.y, p.d)) return p;
  if (!setup_ray(c, g, p.x, p.y, p.rs)) return p;
  p.cell = lookup_offset(c, g.lookup_n, p.x, p.y);
  p.ok = true;
  return p;
}

__device__ __forceinline__ Truncation truncation(const GridGeom& g, const PixelCtx& p, const float* sig,
                                                 const float* bia) {
  return {PolyD(sig + p.cell, g.lookup_n), PolyD(bia + p.cell, g.lookup_n), (double)p.d};
}

// Full-ray activation of one ray, walked over the brick grid: every brick
// the voxel walk would cross up to its truncation is marked.  Brick faces
// are voxel faces, so the bricks are met in the order of the voxel walk and
// each brick exit is the same exact rational (n 2^kFix - Oi) / Di, with the
// same tie rule (all tied axes step at once); the truncation test runs at
// each brick exit as in walk().  The return value bounds the voxel walk's
// record count: every voxel step advances at least one axis by one voxel,
// each axis runs monotonically from the entry voxel to a voxel of the last
// brick, so n <= 1 + sum over axes of |last - entry| with "last" the far
// voxel of that brick along the axis (ties and a stop short of that voxel
// only make n smaller).  0 for a ray that misses the grid.
__device__ uint32_t mark_bricks(const GridGeom& g, const RaySetup& rs, const Truncation& trunc,
                                uint8_t* __restrict__ bflags) {
  Rat zin;
  int ix[3], sg[3];
  if (!ray_entry(g, rs, zin, ix, sg)) return 0;
  const int NB[3] = {g.bx, g.by, g.bz};
  int b[3] = {ix[0] >> kBrickLog, ix[1] >> kBrickLog, ix[2] >> kBrickLog};
  // next brick-face crossing per moving axis: n_a / d_a, n_a growing by
  // 2^(kFix + kBrickLog) per brick; cross differences as in walk()
  int64_t n[3], d[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int64_t Oi = rs.Oi[a], Di = rs.Di[a];
    if (Di > 0) {
      n[a] = (((int64_t)b[a] + 1) << (kFix + kBrickLog)) - Oi;
      d[a] = Di;
    } else if (Di < 0) {
      n[a] = Oi - ((int64_t)b[a] << (kFix + kBrickLog));
      d[a] = -Di;
    } else {
      n[a] = 1;
      d[a] = 0;
    }
  }
  const bool m0 = sg[0] != 0, m1 = sg[1] != 0, m2 = sg[2] != 0;
  const int64_t s0 = d[0] << (kFix + kBrickLog), s1 = d[1] << (kFix + kBrickLog), s2 = d[2] << (kFix + kBrickLog);
  int64_t X01 = n[0] * d[1] - n[1] * d[0], X02 = n[0] * d[2] - n[2] * d[0], X12 = n[1] * d[2] - n[2] * d[1];
  const int max_steps = g.bx + g.by + g.bz + 3;
  for (int step = 0; step < max_steps; ++step) {
    bflags[(b[0] * g.by + b[1]) * g.bz + b[2]] = 1;
    int best = m0 ? 0 : (m1 ? 1 : 2);
    if (m1 && best == 0 && X01 > 0) best = 1;
    if (m2 && best != 2 && (best == 0 ? X02 > 0 : X12 > 0)) best = 2;
    const int64_t zn_n = best == 0 ? n[0] : (best == 1 ? n[1] : n[2]);
    const int64_t zn_dd = best == 0 ? d[0] : (best == 1 ? d[1] : d[2]);
    const double zb = (double)zn_n / (double)zn_dd;
    if (trunc.ends(zb)) break;
    const bool st0 = m0 && (best == 0 || (best == 1 ? X01 == 0 : X02 == 0));
    const bool st1 = m1 && (best == 1 || (best == 0 ? X01 == 0 : X12 == 0));
    const bool st2 = m2 && (best == 2 || (best == 0 ? X02 == 0 : X12 == 0));
    const int nb[3] = {b[0] + (st0 ? sg[0] : 0), b[1] + (st1 ? sg[1] : 0), b[2] + (st2 ? sg[2] : 0)};
    if (nb[0] < 0 || nb[0] >= NB[0] || nb[1] < 0 || nb[1] >= NB[1] || nb[2] < 0 || nb[2] >= NB[2]) break;
    if (st0) {
      n[0] += (int64_t)1 << (kFix + kBrickLog);
      X01 += s1;
      X02 += s2;
    }
    if (st1) {
      n[1] += (int64_t)1 << (kFix + kBrickLog);
      X01 -= s0;
      X12 += s2;
    }
    if (st2) {
      n[2] += (int64_t)1 << (kFix + kBrickLog);
      X02 -= s0;
      X12 -= s1;
    }
    b[0] = nb[0];
    b[1] = nb[1];
    b[2] = nb[2];
  }
  uint32_t bound = 1;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    if (sg[a] > 0) bound += (uint32_t)((b[a] << kBrickLog) + (1 << kBrickLog) - 1 - ix[a]);
    if (sg[a] < 0) bound += (uint32_t)(ix[a] - (b[a] << kBrickLog));
  }
  return bound;
}

// Full-ray activation: marks every brick a ray crosses up to its truncation.
// A ray's own walk activates every brick before and at its stopping brick,
// so its later list walk sees exactly these bricks, with no gaps; bound (per
// tiled pixel, when given) receives the bound of that walk's record count.
__global__ void k_mark_rays(CamGeom c, GridGeom g, const float* __restrict__ depth,
                            const float* __restrict__ sig, const float* __restrict__ bia,
                            uint8_t* __restrict__ bflags, uint32_t* __restrict__ bound) {
  const int pix = blockIdx.x * blockDim.x + threadIdx.x;
  if (pix >= tiled_pixels(c)) return;
  PixelCtx p = load_pixel(c, g, depth, pix);
  uint32_t n = 0;
  if (p.ok) n = mark_bricks(g, p.rs, truncation(g, p, sig, bia), bflags);
  if (bound) bound[pix] = n;
}

__global__ void k_mark_endpoints(CamGeom c, GridGeom g, const float* __restrict__ depth,
                                 uint8_t* __restrict__ bflags) {
  const int pix = blockIdx.x * blockDim.x + threadIdx.x;
  if (pix >= tiled_pixels(c)) return;
  PixelCtx p = load_pixel(c, g, depth, pix);
  if (!p.ok) return;
  const int M[3] = {g.mx, g.my, g.mz};
  const int N[3] = {g.nx, g.ny, g.nz};
  int lo[3], hi[3];
  for (int a = 0; a < 3; ++a) {
    double P = (double)p.d * (double)p.rs.Di[a];
    P = (double)p.rs.Oi[a] + P;
    P = P / kFixScale;
    if (!(P >= 0.0 && P < (double)M[a])) return;
    int l = (int)floor(P - 1.0), h = (int)floor(P + 1.0);
    if (l < 0) l = 0;
    if (h > N[a] - 1) h = N[a] - 1;
    lo[a] = l >> kBrickLog;
    hi[a] = h >> kBrickLog;
  }
  for (int i = lo[0]; i <= hi[0]; ++i)
    for (int j = lo[1]; j <= hi[1]; ++j)
      for (int k = lo[2]; k <= hi[2]; ++k) bflags[(i * g.by + j) * g.bz + k] = 1;
}

// Depth endpoints per voxel (a feature of the learned warm start): the voxel
// holding the endpoint of every valid pixel, with the endpoint formula and
// map-box gate of k_mark_endpoints; endpoints in inactive bricks are dropped.
__global__ void k_feat_hits(CamGeom c, GridGeom g, const float* __restrict__ depth,
                            const int32_t* __restrict__ slot, uint32_t* __restrict__ hits) {
  const int pix = blockIdx.x * blockDim.x + threadIdx.x;
  if (pix >= tiled_pixels(c)) return;
  PixelCtx p = load_pixel(c, g, depth, pix);
  if (!p.ok) return;
  const int M[3] = {g.mx, g.my, g.mz};
  int v[3];
  for (int a = 0; a < 3; ++a) {
    double P = (double)p.d * (double)p.rs.Di[a];
    P = (double)p.rs.Oi[a] + P;
    P = P / kFixScale;
    if (!(P >= 0.0 && P < (double)M[a])) return;
    v[a] = (int)floor(P);
  }
  const int sl = slot[((v[0] >> kBrickLog) * g.by + (v[1] >> kBrickLog)) * g.bz + (v[2] >> kBrickLog)];
  if (sl < 0) return;
  atomicAdd(&hits[(size_t)sl * kBrickVox + ((v[0] & 7) * 64 + (v[1] & 7) * 8 + (v[2] & 7))], 1u);
}

template <bool F64>
__global__ void k_count(CamGeom c, GridGeom g, const float* __restrict__ depth,
                        const float* __restrict__ sig, const float* __restrict__ bia,
                        const int32_t* __restrict__ slot, uint32_t* __restrict__ counts) {
  const int pix = blockIdx.x * blockDim.x + threadIdx.x;
  if (pix >= tiled_pixels(c)) return;
  PixelCtx p = load_pixel(c, g, depth, pix);
  uint32_t n = 0;
  if (p.ok) {
    const Truncation trunc = truncation(g, p, sig, bia);
    n = walk<kCount, F64>(g, p.rs, trunc, slot, nullptr, 0, 0u).n;
  }
  counts[pix] = n;
}

// Records per slice (max over the tile's 64 rays) and the slice's padded size.
__global__ void k_slice_len(const uint32_t* __restrict__ counts, uint32_t ntiles, uint32_t* __restrict__ slice_len,
                            uint32_t* __restrict__ slice_rec) {
  const uint32_t t = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (t >= ntiles) return;
  uint32_t m = counts[t * kSlice + (threadIdx.x & 63)];
  for (int o = 32; o > 0; o >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o));
  if ((threadIdx.x & 63) == 0) {
    slice_len[t] = m;
    slice_rec[t] = m * kSlice;
  }
}

// Emission of every ray's records into the staging lists, split into front
// and window as they go: front[pix].nf front records, then lanes[pix].nw
// window records; cnt_f / cnt_w per tiled pixel.
template <bool F64, bool ALL>
__global__ void k_emit(CamGeom c, GridGeom g, const float* __restrict__ depth, const float* __restrict__ sig,
                       const float* __restrict__ bia, const int32_t* __restrict__ slot,
                       const uint32_t* __restrict__ slice_off, const uint32_t* __restrict__ slice_len,
                       uint32_t* __restrict__ sell, size_t to_len, FrontRec* __restrict__ front,
                       RayRec* __restrict__ lanes,
                       uint32_t* __restrict__ cnt_f, uint32_t* __restrict__ cnt_w, uint32_t* __restrict__ overflow) {
  const int pix = blockIdx.x * blockDim.x + threadIdx.x;
  if (pix >= tiled_pixels(c)) return;
  const uint32_t tile = (uint32_t)pix >> 6, lane = (uint32_t)pix & 63u;
  uint32_t* out = sell + slice_off[tile] + lane;
  PixelCtx p = load_pixel(c, g, depth, pix);
  FrontRec f;
  f.off = slice_off[tile] + lane;  // front and window records follow each other until the reslice
  f.nf = 0;
  RayRec r;
  r.off_w = 0;
  r.nw = 0;
  r.ks = 0.0f;
  r.kc = 0.0f;
  r.z0 = 0.0f;
  r.inv_norm = 0.0f;
  r.depth = 0.0f;
  r.cell_flags = 0;
  if (p.ok) {
    FrontSplit sp;
    load_cell(sig, bia, g.lookup_n, p.cell, sp.sig, sp.bia);
    sp.inv_norm = (float)(1.0 / p.rs.norm);
    sp.depth = p.d;
    sp.z0 = 0.0f;
    sp.kS = {0.0f, 0.0f};
    sp.nf = 0;
    sp.open = true;
    const uint32_t cap = slice_len[tile];
    const Truncation trunc = truncation(g, p, sig, bia);
    WalkOut wo = walk<ALL ? kEmitAll : kEmit, F64>(g, p.rs, trunc, slot, out, to_len, cap, &sp);
    uint32_t n = wo.n;
    if (n > cap) {  // the slot's bound did not hold: an error, and the lists stay in bounds
      atomicOr(overflow, 1u);
      n = cap;
    }
    const uint32_t nf = sp.open ? n : min(sp.nf, n);
    f.nf = nf;
    r.nw = n - nf;
    r.ks = sp.kS.s;
    r.kc = sp.kS.c;
    r.z0 = wo.z0;
    r.inv_norm = sp.inv_norm;
    r.depth = p.d;
    // the infinity term's test d > s_n + bias(s_n) at the exact exit depth of
    // the last record, in FP64 as the traversal itself: an FP32 running sum
    // of chord lengths can land on either side when d is within an ulp
    const bool inf = wo.ran_out && (double)p.d > wo.last_exit + trunc.bia(wo.last_exit);
    r.cell_flags = p.cell | (wo.ran_out ? kRanOut : 0u) | (inf ? kInfTerm : 0u);
  }
  // records past the ray's own are never read: no padding
  front[pix] = f;
  lanes[pix] = r;
  cnt_f[pix] = f.nf;
  cnt_w[pix] = r.nw;
}

// ---------------------------------------------------------------- map evaluation
// One pixel ray walked through the current map to the end of the grid (no
// truncation), every voxel of an active brick read as its marginal
// occupancy p (0 where never updated, gvdbkernels.cu:469-476).  Per voxel:
// alpha = -ln(1 - p), Lambda += -alpha l, vis = e^Lambda, weight
// vis_prev - vis (Crispell's visibility model, gvdbkernels.cu:230-236).
//  * log-likelihood (rayLikelihoodBrick + render_likelihood_kernel,
//    gvdbkernels.cu:183-293, 1246-1274): sum of weight x p(z | voxel), with
//    p(z | voxel) = 0 below Z_MIN, (1 - LIKE_EPS) (psi(s) + psi(s_prev)) / 2
//    within 3 sigma of the measured depth, LIKE_EPS elsewhere; plus
//    vis_inf x (d >= Z_MAX ? 1 - LIKE_EPS : LIKE_EPS); the pixel's value is
//    its log; invalid depth gives 0.
//  * expected depth (rayExpectedDepthBrick + render_expected_depth_kernel,
//    gvdbkernels.cu:295-354, 1332-1363): sum of weight x the planar depth of
//    the voxel centre, over 1 - vis_inf + F_EPS; every pixel.
//  * accuracy (render_accuracy_kernel, gvdbkernels.cu:1066-1104): at the
//    voxel with the largest weight per unit length, 1 if its depth is within
//    1 sigma of the measurement else 0; -1 for an invalid pixel, a ray that
//    met nothing, or one that kept vis >= 0.9 and ended short of the
//    measurement (0 if it ended beyond it).
//  * simple accuracy (raySimpleAccuracyBrick + render_simple_accuracy_kernel,
//    gvdbkernels.cu:135-181, 1106-1134): the first voxel with
//    p >= acc_thresh gives 1 (within one voxel size of the measured depth) or
//    2; an active brick ending at or beyond the measured depth first gives 0;
//    otherwise -1.
// The prefix depth s is the planar depth at the voxel's exit; at an active
// brick's end the previous depth carried into the next brick is s + bias(s)
// (the reference passes it on in norm.x).
constexpr float kZMin = 0.1f;
constexpr float kLikeEps = 1e-3f;

// sigma(s) or bias(s) in FP32 (two coefficients: c2 = 0)
__device__ __forceinline__ float poly_f(const Poly& c, float s) { return (s * s) * c.c2 + s * c.c1 + c.c0; }

struct EvalRay {
  Poly sig, bia;
  float d, res, acc_thresh;
  bool valid;
  float prev_vis, lam, sum, prev_s, norm_x, peak, esum, sacc;
  int peak_ok;
  bool first, sdone;

  __device__ __forceinline__ float psi(float s) const {
    const float sg3 = 3.0f * poly_f(sig, s);
    const float u = (d - s - poly_f(bia, s)) / sg3;
    return 0.398942f * expf(-0.5f * u * u) / sg3;
  }
  // a voxel of an active brick with occupancy p, its chord, entry and exit depth and its centre's depth
  __device__ __forceinline__ void voxel(float p, float len, double z0, double z1, float zc) {
    const float s = (float)z1;
    if (first) {
      prev_s = (float)z0;
      first = false;
    }
    const float alpha = -logf(1.0f - p);
    lam += -alpha * len;
    const float vis = expf(lam);
    if (valid) {
      const float pdm = s + poly_f(bia, s) - d;
      const float sg = poly_f(sig, s);
      float prob;
      if (s < kZMin)
        prob = 0.0f;
      else if (fabsf(pdm) <= 3.0f * sg)
        prob = (1.0f - kLikeEps) * 0.5f * (psi(s) + psi(prev_s));
      else
        prob = kLikeEps;
      // the weight per unit length w, divided out only where it may exceed the peak
      if ((prev_vis - vis) * __builtin_amdgcn_rcpf(len) * 1.000001f >= peak) {
        const float w = (prev_vis - vis) / len;
        if (w > peak) {
          peak = w;
          peak_ok = fabsf(pdm) <= sg ? 1 : 0;
        }
      }
      sum += (prev_vis - vis) * prob;
      norm_x = pdm + d;
      if (!sdone && p >= acc_thresh) {
        sacc = fabsf(s - d) <= res ? 1.0f : 2.0f;
        sdone = true;
      }
    }
    esum += (prev_vis - vis) * zc;
    prev_vis = vis;
    prev_s = s;
  }
  __device__ __forceinline__ void brick_end(double z) {
    if (valid) {
      prev_s = norm_x;
      if (!sdone && (float)z >= d) {
        sacc = 0.0f;
        sdone = true;
      }
    }
  }
};

// The walk of k_eval, to the end of the grid.  cz: the depth of voxel ix's
// centre is cz[3] + sum cz[a] ix[a].  Bound by its arithmetic: taking the
// voxels four at a time, so that their slots and then their beliefs are
// loaded together, was slower (1.24 against 1.05 ms for a 640x480 frame in a
// 4x4x3 m map at 1 cm; 1.66 ms with the integer walk and the sensor model
// loaded per voxel).
template <bool F64>
__device__ __forceinline__ void eval_walk(const GridGeom& g, const RaySetup& rs, const int32_t* __restrict__ slot,
                                          const float* __restrict__ B, const uint8_t* __restrict__ upd,
                                          const double (&cz)[4], EvalRay& v) {
  Rat zin;
  int ix[3], sg[3];
  if (!ray_entry(g, rs, zin, ix, sg)) return;
  Steps<F64> st = first_crossings<F64>(rs, ix);
  double zc_d = (double)zin.n / (double)zin.d;
  auto brick_lookup = [&](void) -> int32_t {
    return slot[((ix[0] >> kBrickLog) * g.by + (ix[1] >> kBrickLog)) * g.bz + (ix[2] >> kBrickLog)];
  };
  int32_t bslot = brick_lookup();
  const int max_steps = g.nx + g.ny + g.nz + 3;
  for (int step = 0; step < max_steps; ++step) {
    const double zn_d = st.z();
    if (bslot >= 0) {
      const uint32_t local = (uint32_t)((((ix[0] & 7) << 3) | (ix[1] & 7)) << 3 | (ix[2] & 7));
      const size_t id = (size_t)bslot * kBrickVox + local;
      float neg = 1.0f / (1.0f + expf(B[id]));
      neg = fminf(fmaxf(neg, kFEps), 1.0f - kFEps);
      const double zc = fma(cz[0], (double)ix[0], fma(cz[1], (double)ix[1], fma(cz[2], (double)ix[2], cz[3])));
      v.voxel(upd[id] ? 1.0f - neg : 0.0f, (float)((zn_d - zc_d) * rs.norm), zc_d, zn_d, (float)zc);
    }
    bool st0, st1, st2;
    st.which(st0, st1, st2);
    const int nx[3] = {ix[0] + (st0 ? sg[0] : 0), ix[1] + (st1 ? sg[1] : 0), ix[2] + (st2 ? sg[2] : 0)};
    const bool brick_change = (uint32_t)((nx[0] ^ ix[0]) | (nx[1] ^ ix[1]) | (nx[2] ^ ix[2])) >> kBrickLog != 0u;
    ix[0] = nx[0];
    ix[1] = nx[1];
    ix[2] = nx[2];
    if (brick_change) {
      if (bslot >= 0) v.brick_end(zn_d);
      if ((uint32_t)nx[0] >= (uint32_t)g.nx || (uint32_t)nx[1] >= (uint32_t)g.ny || (uint32_t)nx[2] >= (uint32_t)g.nz)
        break;
      bslot = brick_lookup();
    }
    st.step(st0, st1, st2, kFix);
    zc_d = zn_d;
  }
}

template <bool F64>
__global__ __launch_bounds__(256) void k_eval(CamGeom c, GridGeom g, const float* __restrict__ depth,
                                              const float* __restrict__ sigt, const float* __restrict__ biat,
                                              const int32_t* __restrict__ slot, const float* __restrict__ B,
                                              const uint8_t* __restrict__ upd, float acc_thresh,
                                              float* __restrict__ out_ll, float* __restrict__ out_ed,
                                              float* __restrict__ out_acc, float* __restrict__ out_sacc,
                                              double* __restrict__ part, unsigned long long* __restrict__ counts) {
  __shared__ double sh[256];
  const int pix = blockIdx.x * blockDim.x + threadIdx.x;
  int x = 0, y = 0;
  const bool in = pix < tiled_pixels(c) && tile_pixel(c, pix, &x, &y);
  float ll = 0.0f, ed = 0.0f, acc = -1.0f, sacc = -1.0f;
  if (in) {
    const float d = depth ? depth[y * c.cols + x] : 0.0f;
    EvalRay v;
    load_cell(sigt, biat, g.lookup_n, lookup_offset(c, g.lookup_n, x, y), v.sig, v.bia);
    v.d = d;
    v.res = (float)g.res;
    v.acc_thresh = acc_thresh;
    v.valid = depth != nullptr && pixel_valid(c, x, y, d);
    // the camera's z axis over voxel centres: sum_a R_a2 ((ix_a + 1/2 - off_a) res - t_a)
    double cz[4] = {0.0, 0.0, 0.0, 0.0};
    for (int a = 0; a < 3; ++a) {
      cz[a] = c.R[a * 3 + 2] * g.res;
      cz[3] += c.R[a * 3 + 2] * ((0.5 - g.off[a]) * g.res - c.t[a]);
    }
    v.prev_vis = 1.0f;
    v.lam = v.sum = v.prev_s = v.norm_x = v.peak = v.esum = 0.0f;
    v.sacc = -1.0f;
    v.peak_ok = 0;
    v.first = true;
    v.sdone = false;
    RaySetup rs;
    if (setup_ray(c, g, x, y, rs)) eval_walk<F64>(g, rs, slot, B, upd, cz, v);
    ed = v.esum / (1.0f - v.prev_vis + kFEps);
    if (v.valid) {
      ll = logf(v.sum + v.prev_vis * (d >= kZMax ? 1.0f - kLikeEps : kLikeEps));
      if (v.peak > 0.0f && v.prev_vis >= 0.9f)
        acc = v.norm_x <= d ? -1.0f : 0.0f;
      else if (v.peak > 0.0f)
        acc = (float)v.peak_ok;
      sacc = v.sacc;
    }
    const int o = y * c.cols + x;
    if (out_ll) out_ll[o] = ll;
    if (out_ed) out_ed[o] = ed;
    if (out_acc) out_acc[o] = acc;
    if (out_sacc) out_sacc[o] = sacc;
  }
  // class counts: accuracy -1, 0, 1 then simple accuracy -1, 0, 1, 2 (pixels of the image only)
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int k = 0; k < 7; ++k) {
    const float want = k < 3 ? (float)(k - 1) : (float)(k - 4);
    const float val = k < 3 ? acc : sacc;
    const unsigned long long m = __ballot(in && val == want);
    if (lane == 0 && m) atomicAdd(counts + k, (unsigned long long)__popcll(m));
  }
  // fixed-order FP64 block sum of the log-likelihoods
  sh[threadIdx.x] = (double)ll;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

}  // namespace

int num_tiled_pixels(const CamGeom& c) { return tiled_pixels(c); }

namespace {

// Whether every ray of the camera keeps the walks' numbers below 2^52: the
// crossings' numerators are at most the distance from the origin to the far
// side of the grid (in 2^-kFix voxels) plus a step, the directions are linear
// in the pixel, so largest at a corner of the image.
bool dda_fits_f64(const CamGeom& c, const GridGeom& g) {
  const int N[3] = {g.nx, g.ny, g.nz};
  double n[3], d[3];
  for (int a = 0; a < 3; ++a) {
    const double O = (c.t[a] / g.res + g.off[a]) * kFixScale, top = (double)N[a] * kFixScale;
    n[a] = std::max(std::fabs(O), std::fabs(top - O)) + 2.0 * kFixScale;
    d[a] = 0.0;
    for (int k = 0; k < 4; ++k) {
      const double ux = ((k & 1 ? c.cols - 1 : 0) - c.cx) / c.fx, uy = ((k >> 1 ? c.rows - 1 : 0) - c.cy) / c.fy;
      d[a] = std::max(d[a], std::fabs(c.R[a * 3] * ux + c.R[a * 3 + 1] * uy + c.R[a * 3 + 2]) / g.res * kFixScale + 2.0);
    }
  }
  const double lim = 4503599627370496.0;  // 2^52
  return n[0] * d[1] + n[1] * d[0] < lim && n[0] * d[2] + n[2] * d[0] < lim && n[1] * d[2] + n[2] * d[1] < lim;
}

}  // namespace

unsigned eval_blocks(const CamGeom& c) { return (unsigned)((tiled_pixels(c) + 255) / 256); }

void launch_eval(const CamGeom& c, const GridGeom& g, const float* depth, const float* sig, const float* bia,
                 const int32_t* slot, const float* B, const uint8_t* upd, float acc_thresh, float* ll, float* ed,
                 float* acc, float* sacc, double* part, unsigned long long* counts, hipStream_t s) {
  auto* k = dda_fits_f64(c, g) ? k_eval<true> : k_eval<false>;
  hipLaunchKernelGGL(k, dim3(eval_blocks(c)), dim3(256), 0, s, c, g, depth, sig, bia, slot, B, upd, acc_thresh, ll, ed,
                     acc, sacc, part, counts);
}

void launch_mark_rays(const CamGeom& c, const GridGeom& g, const float* depth, const float* sig,
                      const float* bia, uint8_t* bflags, uint32_t* bound, hipStream_t s) {
  const int n = tiled_pixels(c);
  hipLaunchKernelGGL(k_mark_rays, dim3((n + 127) / 128), dim3(128), 0, s, c, g, depth, sig, bia, bflags, bound);
}

void launch_feat_hits(const CamGeom& c, const GridGeom& g, const float* depth, const int32_t* slot, uint32_t* hits,
                      hipStream_t s) {
  const int n = tiled_pixels(c);
  hipLaunchKernelGGL(k_feat_hits, dim3((n + 255) / 256), dim3(256), 0, s, c, g, depth, slot, hits);
}

void launch_mark_endpoints(const CamGeom& c, const GridGeom& g, const float* depth, uint8_t* bflags,
                           hipStream_t s) {
  const int n = tiled_pixels(c);
  hipLaunchKernelGGL(k_mark_endpoints, dim3((n + 255) / 256), dim3(256), 0, s, c, g, depth, bflags);
}

void launch_count(const CamGeom& c, const GridGeom& g, const float* depth, const float* sig,
                  const float* bia, const int32_t* slot, uint32_t* counts, hipStream_t s) {
  const int n = tiled_pixels(c);
  auto* k = dda_fits_f64(c, g) ? k_count<true> : k_count<false>;
  hipLaunchKernelGGL(k, dim3((n + 127) / 128), dim3(128), 0, s, c, g, depth, sig, bia, slot, counts);
}

void launch_slice_len(const uint32_t* counts, uint32_t ntiles, uint32_t* slice_len, uint32_t* slice_rec,
                      hipStream_t s) {
  if (ntiles == 0) return;
  hipLaunchKernelGGL(k_slice_len, dim3((ntiles + 3) / 4), dim3(256), 0, s, counts, ntiles, slice_len, slice_rec);
}

void launch_emit(const CamGeom& c, const GridGeom& g, const float* depth, const float* sig, const float* bia,
                 const int32_t* slot, const uint32_t* slice_off, const uint32_t* slice_len, uint32_t* sell,
                 size_t to_len, FrontRec* front, RayRec* lanes, uint32_t* cnt_f, uint32_t* cnt_w, uint32_t* overflow,
                 bool all_active, hipStream_t s) {
  const int n = tiled_pixels(c);
  const bool f64 = dda_fits_f64(c, g);
  auto* k = all_active ? (f64 ? k_emit<true, true> : k_emit<false, true>)
                       : (f64 ? k_emit<true, false> : k_emit<false, false>);
  hipLaunchKernelGGL(k, dim3((n + 127) / 128), dim3(128), 0, s, c, g, depth, sig, bia, slot, slice_off, slice_len, sell,
                     to_len, front, lanes, cnt_f, cnt_w, overflow);
}

}  // namespace mrf
