// Per-camera pair and window-segment layout of the incidence lists (built
// once per traversal, not per BP iteration).
//
// Pairs.  Every voxel the camera's live records touch is one (camera, voxel)
// pair.  Two byte flags over the brick pool -- touched by any record, by a
// window record -- number the pairs by their ranks (counts per brick, a scan
// over bricks, ranks inside the brick): the pairs with window records first,
// then the others, each group in voxel order, so that window segment m
// belongs to pair m.
//
// Per pair, the summed chord length C (what render_cumulative_length_kernel
// accumulates with float atomics in every camera pass,
// src/cuda/gvdbkernels.cu:519-571, 1276-1302) and the chord length of its
// front records (whose messages are the constant F_EPS * l) are summed in
// fixed point, each length as q 2^-24 + r 2^-48, both sums exact whatever
// their size (the carries of the 32-bit words are kept), so they do not
// depend on the order in which records arrive.  C is exact for every chord of
// at least 2^-25, and the epilogue gate C > 0.1f (gvdbkernels.cu:408) falls as
// it does on the exact sum, however close to 0.1f C lies.
//
// Window segments.  The window records are stably radix-sorted by pair, so
// each pair's records stay in record order; the BP iteration sums each
// segment in that order, gathered through win_idx (no atomics,
// bit-reproducible).  The pass that copies the records into their final
// regions puts each live record's pair in place of its voxel, sums the front
// part of C and writes the sort's input.
#include <hipcub/hipcub.hpp>

#include "mrf_kernels.h"

namespace mrf {

namespace {

constexpr double kFixLen = 16777216.0;  // 2^24: chord lengths (< 1.74) in fixed point, a 64-record sum < 2^31

// Pair numbering by brick (one wavefront per brick of the pool, 8 voxels
// per lane, the byte flags read 8 at a time): a voxel's rank among the
// touched voxels in voxel order is its brick's offset plus the touched
// voxels before it in the brick.

__device__ __forceinline__ uint32_t wave_sum_u32(uint32_t x) {
  for (int o = 32; o > 0; o >>= 1) x += (uint32_t)__shfl_xor((int)x, o, 64);
  return x;
}

__global__ __launch_bounds__(256) void k_brick_flag_counts(const uint8_t* __restrict__ any,
                                                           const uint8_t* __restrict__ wany, uint32_t nbricks,
                                                           uint64_t* __restrict__ counts) {
  const uint32_t b = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (b >= nbricks) return;  // uniform per wavefront
  const uint32_t l = threadIdx.x & 63u;
  const uint64_t a = reinterpret_cast<const uint64_t*>(any)[(size_t)b * 64 + l];
  const uint64_t w = reinterpret_cast<const uint64_t*>(wany)[(size_t)b * 64 + l];
  const uint32_t na = wave_sum_u32((uint32_t)__popcll(a)), nw = wave_sum_u32((uint32_t)__popcll(w));
  if (l == 0) counts[b] = (uint64_t)na | ((uint64_t)nw << 32);
}

// pid[v] and pair_vox[pid] of every touched voxel (window pairs first, the
// ranks of wany; then the others, nwp + the ranks of any minus those of
// wany); the flags are cleared behind (all zero again for the next camera)
__global__ __launch_bounds__(256) void k_pair_table(uint8_t* __restrict__ any, uint8_t* __restrict__ wany,
                                                    const uint64_t* __restrict__ boff, uint32_t nbricks,
                                                    uint32_t nwp, uint32_t* __restrict__ pid,
                                                    uint32_t* __restrict__ pair_vox) {
  const uint32_t b = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (b >= nbricks) return;  // uniform per wavefront
  const uint32_t l = threadIdx.x & 63u;
  uint64_t* A = reinterpret_cast<uint64_t*>(any) + (size_t)b * 64 + l;
  uint64_t* Wf = reinterpret_cast<uint64_t*>(wany) + (size_t)b * 64 + l;
  const uint64_t a = *A, w = *Wf;
  if (__ballot(a != 0) == 0) return;  // no touched voxel in the brick (uniform)
  // exclusive prefix of the lanes' counts
  const uint32_t na = (uint32_t)__popcll(a), nw = (uint32_t)__popcll(w);
  uint32_t ia = na, iw = nw;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t ua = (uint32_t)__shfl_up((int)ia, o, 64), uw = (uint32_t)__shfl_up((int)iw, o, 64);
    if (l >= (uint32_t)o) {
      ia += ua;
      iw += uw;
    }
  }
  const uint64_t o = boff[b];
  uint32_t ra = (uint32_t)o + ia - na, rw = (uint32_t)(o >> 32) + iw - nw;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const bool fa = ((a >> (8 * k)) & 1u) != 0, fw = ((w >> (8 * k)) & 1u) != 0;
    if (fa) {
      const uint32_t v = b * (uint32_t)kBrickVox + l * 8u + (uint32_t)k;
      const uint32_t p = fw ? rw : nwp + (ra - rw);
      pid[v] = p;
      pair_vox[p] = v;
    }
    ra += fa ? 1u : 0u;
    rw += fw ? 1u : 0u;
  }
  if (a) *A = 0;
  if (w) *Wf = 0;
}

template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_u(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, ROWS, 0xF, true);
}

// (x, f) <- (x_left, f_left) (+) (x, f): add the left value unless a run
// starts at or before this lane
template <int CTRL, int ROWS>
__device__ __forceinline__ void seg_step_u(uint32_t& x, uint32_t& x2, uint32_t& f) {
  const uint32_t y = dpp_u<CTRL, ROWS>(x);
  const uint32_t y2 = dpp_u<CTRL, ROWS>(x2);
  const uint32_t g = dpp_u<CTRL, ROWS>(f);
  x = f ? x : x + y;
  x2 = f ? x2 : x2 + y2;
  f |= g;
}

// Inclusive segmented sum over the 64 lanes (all active): row_shr 1/2/4/8
// inside each row of 16, then row_bcast 15 and 31.
__device__ __forceinline__ void wave_seg_sum_u(uint32_t& x, uint32_t& x2, uint32_t f) {
  seg_step_u<0x111, 0xF>(x, x2, f);
  seg_step_u<0x112, 0xF>(x, x2, f);
  seg_step_u<0x114, 0xF>(x, x2, f);
  seg_step_u<0x118, 0xF>(x, x2, f);
  seg_step_u<0x142, 0xA>(x, x2, f);
  seg_step_u<0x143, 0xC>(x, x2, f);
}

// Copy every ray's staged records into the front and window regions of the
// final record buffer (sliced: lane l of slice t at region offset + k * 64 +
// l), each live record with its pair instead of its voxel, padding each lane
// to its slice's length with gap records; the window records' sort input (key
// its pair, a sentinel that sorts last for a gap or padding record, value its
// position in the region); and the front sums of every pair: acc holds
// {sum of r (low word), sum of q (high word)} of its front records' lengths l =
// q 2^-24 + r 2^-48, hi the carries out of the two words.  The window part of
// C is summed after the window sort, where each pair's records are contiguous
// (k_window_layout).  SLOTS as in k_mark_voxels.
//
// The 64 records of a row share few voxels (the rays are neighbours, and with
// full-ray activation a voxel is the same step of every ray that meets it).
// A wave first sums runs of equal voxels along the pixel rows (near the camera
// all 64 rays lie in one voxel, and 64 LDS operations on one word follow each
// other: 1508 us without it), then across them in a table in LDS that holds a
// batch of 8 rows, and issues one 64-bit atomic per voxel and batch: a run
// whose slot holds another pair goes to memory by itself.  A ray meets a voxel
// once, so a sum in the table has at most 64 parts: r < 2^30 and q < 2^31
// never carry there.  In memory they may (a voxel met by more than 128 rays):
// the add whose low word wrapped takes the carry out of q again, and every
// carry and borrow is counted in hi, modulo 2^32 per word, so the two sums
// stay exact.  The window part of C summed here as well costs 490 us more
// (the far voxels are met by few rays of a tile) and saves 250 after the sort.
// 640x480 at 1 cm, 150 M records in 161 M places: 1051 us and 3.87 GB by the
// counters; the atomics take 356, the copy alone (2.6 GB) about 600.  A copy
// with voxels, then a pass that rewrote it in place, sorting each row's 64
// pairs across the lanes, took 795 + 1245 us (now 1051 + 362 for
// k_mark_voxels, and the emission 75 more for its second store).
constexpr uint32_t kTabLog = 9, kTab = 1u << kTabLog;
constexpr uint32_t kFree = 0xFFFFFFFFu;
template <bool SLOTS>
__global__ __launch_bounds__(256) void k_reslice(FrontRec* __restrict__ front, RayRec* __restrict__ lanes,
                                                 const uint32_t* __restrict__ ids, const uint32_t* __restrict__ lens,
                                                 const int32_t* __restrict__ slot, const uint32_t* __restrict__ pid,
                                                 const uint32_t* __restrict__ off_f, const uint32_t* __restrict__ len_f,
                                                 const uint32_t* __restrict__ off_w, const uint32_t* __restrict__ len_w,
                                                 uint32_t base_w, uint2* __restrict__ inc,
                                                 unsigned long long* __restrict__ acc,
                                                 unsigned long long* __restrict__ hi, uint32_t* __restrict__ wkeys,
                                                 uint32_t* __restrict__ wvals, uint32_t sentinel) {
  constexpr uint32_t kW = 4, kB = 8;
  __shared__ uint32_t tab_key[kW][kTab];
  __shared__ unsigned long long tab_sum[kW][kTab];
  const uint32_t t = blockIdx.x, wave = threadIdx.x >> 6, l = threadIdx.x & 63u, ray = t * kSlice + l;
  uint32_t* tk = tab_key[wave];
  unsigned long long* ts = tab_sum[wave];
  for (uint32_t i = l; i < kTab; i += 64u) {
    tk[i] = kFree;
    ts[i] = 0;
  }
  const FrontRec f = front[ray];
  const uint32_t rnw = lanes[ray].nw;
  const uint32_t fo = off_f[t] + l, wo = off_w[t] + l;
  const uint32_t lf = len_f[t], lw = len_w[t];
  // the pairs of a batch's records (kGapVox: none)
  auto pairs = [&](uint32_t(&e)[kB]) {
    if constexpr (SLOTS) {
      int32_t sl[kB];
#pragma unroll
      for (uint32_t u = 0; u < kB; ++u) sl[u] = slot[e[u] != kGapVox ? e[u] >> kBrickLog * 3 : 0u];
#pragma unroll
      for (uint32_t u = 0; u < kB; ++u)
        if (e[u] != kGapVox) e[u] = (uint32_t)sl[u] * kBrickVox + (e[u] & (kBrickVox - 1u));
    }
    uint32_t p[kB];
#pragma unroll
    for (uint32_t u = 0; u < kB; ++u) p[u] = pid[e[u] != kGapVox ? e[u] : 0u];
#pragma unroll
    for (uint32_t u = 0; u < kB; ++u)
      if (e[u] != kGapVox) e[u] = p[u];
  };
  for (uint32_t k0 = wave * kB; k0 < lf; k0 += kW * kB) {
    uint32_t e[kB], len[kB];
#pragma unroll
    for (uint32_t u = 0; u < kB; ++u) {
      const bool in = k0 + u < f.nf;
      e[u] = in ? ids[f.off + (size_t)(k0 + u) * kSlice] : kGapVox;
      len[u] = in ? lens[f.off + (size_t)(k0 + u) * kSlice] : 0u;
    }
    pairs(e);
#pragma unroll
    for (uint32_t u = 0; u < kB; ++u)
      if (k0 + u < lf) inc[fo + (size_t)(k0 + u) * kSlice] = make_uint2(e[u], len[u]);
    // the table: first the slots of all rows, then their sums
    unsigned long long x[kB];
    uint32_t at[kB], was[kB];
#pragma unroll
    for (uint32_t u = 0; u < kB; ++u) {
      // l 2^24 is exact in double; q its integer part (< 2^25), r the rest in
      // units of 2^-48 (< 2^24)
      const double d = (double)__uint_as_float(len[u]) * kFixLen;
      uint32_t q = (uint32_t)d, r = (uint32_t)((d - (double)q) * kFixLen);
      // first summed along the pixel row: the last ray of a run of equal
      // voxels keeps the run's sum
      const uint32_t right = (uint32_t)__shfl_down((int)e[u], 1, 64);
      uint32_t head = dpp_u<0x111, 0xF>(e[u]) != e[u] || (l & 7u) == 0u ? 1u : 0u;
      const bool ends = right != e[u] || (l & 7u) == 7u;
      seg_step_u<0x111, 0xF>(q, r, head);
      seg_step_u<0x112, 0xF>(q, r, head);
      seg_step_u<0x114, 0xF>(q, r, head);
      if (!ends) e[u] = kGapVox;
      x[u] = (unsigned long long)q << 32 | r;
      at[u] = (e[u] * 2654435761u) >> (32 - kTabLog);
      was[u] = e[u];
      if (e[u] != kGapVox) was[u] = atomicCAS(&tk[at[u]], kFree, e[u]);
    }
#pragma unroll
    for (uint32_t u = 0; u < kB; ++u)
      if (e[u] != kGapVox && (was[u] == kFree || was[u] == e[u])) atomicAdd(&ts[at[u]], x[u]);
    // the wave's own LDS operations complete in order
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (uint32_t u = 0; u < kB; ++u) {
      if (e[u] == kGapVox) continue;
      if (was[u] == kFree) {  // this lane took the slot: it passes the sum on and frees the slot
        x[u] = ts[at[u]];
        ts[at[u]] = 0;
        tk[at[u]] = kFree;
      } else if (was[u] == e[u]) {
        e[u] = kGapVox;  // in another lane's or row's sum
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // the adds, then their carries once the old values are back
    unsigned long long old[kB];
#pragma unroll
    for (uint32_t u = 0; u < kB; ++u) old[u] = e[u] != kGapVox ? atomicAdd(acc + e[u], x[u]) : 0ull;
#pragma unroll
    for (uint32_t u = 0; u < kB; ++u) {
      if (e[u] == kGapVox) continue;
      unsigned long long c = old[u] + x[u] < old[u] ? 1ull << 32 : 0ull;
      if ((uint32_t)old[u] + (uint32_t)x[u] < (uint32_t)old[u]) {
        c += 1ull;
        if (atomicAdd(acc + e[u], 0xFFFFFFFF00000000ull) >> 32 == 0) c -= 1ull << 32;
      }
      if (c) atomicAdd(hi + e[u], c);
    }
  }
  for (uint32_t k0 = wave * kB; k0 < lw; k0 += kW * kB) {
    uint32_t e[kB], len[kB];
#pragma unroll
    for (uint32_t u = 0; u < kB; ++u) {
      const bool in = k0 + u < rnw;
      e[u] = in ? ids[f.off + (size_t)(f.nf + k0 + u) * kSlice] : kGapVox;
      len[u] = in ? lens[f.off + (size_t)(f.nf + k0 + u) * kSlice] : 0u;
    }
    pairs(e);
#pragma unroll
    for (uint32_t u = 0; u < kB; ++u) {
      if (k0 + u < lw) {
        const size_t jw = wo + (size_t)(k0 + u) * kSlice;
        inc[base_w + jw] = make_uint2(e[u], len[u]);
        wkeys[jw] = e[u] == kGapVox ? sentinel : e[u];
        wvals[jw] = (uint32_t)jw;
      }
    }
  }
  __syncthreads();  // every wave has read the slice's descriptions
  if (wave != 0) return;
  front[ray].off = fo;
  lanes[ray].off_w = base_w + wo;
}

// a pair's sums of q (units of 2^-24) and r (2^-48) from their words
__device__ __forceinline__ uint64_t sum_q(uint64_t acc, uint64_t hi) { return acc >> 32 | (hi & 0xFFFFFFFF00000000ull); }
__device__ __forceinline__ uint64_t sum_r(uint64_t acc, uint64_t hi) { return (acc & 0xFFFFFFFFull) | hi << 32; }

// C in FP32 with the gate of the exact sum (C > 0.1f, gvdbkernels.cu:408) from
// the exact fixed-point sums of a pair: w, f in units of 2^-24 (window, front
// records), r the parts below in units of 2^-48.  Where rounding to float
// would move C onto kCumLenMin from above, C takes the next float up, so that
// the float gate falls as on the exact sum.  The integers are below 2^53: the
// doubles and their sum are exact.
__device__ __forceinline__ float pair_length(uint64_t w, uint64_t f, uint64_t r) {
  const double cd = ((double)w + (double)f) / kFixLen + (double)r / (kFixLen * kFixLen);
  float cf = (float)cd;
  if (cd > (double)kCumLenGate) {
    if (!(cf > kCumLenMin)) cf = __uint_as_float(__float_as_uint(kCumLenMin) + 1u);
  } else if (cf > kCumLenMin) {
    cf = kCumLenMin;
  }
  return cf;
}
// F_EPS x the chord length of the front records
__device__ __forceinline__ float front_message(uint64_t f) { return (float)((double)kFEps * ((double)f / kFixLen)); }

// Segment layout of the sorted window records (position m holds pair keys[m],
// record win_idx[m] of the window region) and C of the window pairs, a wave
// per tile of kTile positions.  Every window pair has live window records, so
// the sorted keys step through 0, 1, 2, ...: the key of a head is the number
// of heads before it, and the first position of a pair (wseg_off), the head
// bitmask and the heads before a tile (tile_h0) need no scan.  The lengths
// become the exact fixed-point parts of k_reslice; runs of equal pairs are
// summed by a segmented scan per row of 64, a row's last run is carried into
// the next row.  A pair whose records all lie in this tile is finished here;
// of the others, the part in this tile is added to acc_w (units of 2^-24) and
// acc_r (the parts below), both zeroed before, and k_pair_finish ends them.
// Bound by its loads, so all of them are in flight before the first is used
// (keys and indices, then the gathered records with the pairs' front sums)
// and every store comes after the last.  640x480 at 1 cm, 30 M positions: 313
// us and 62 us for k_pair_finish; heads, scan, offsets and bits as passes of
// their own with atomic length sums took 281 + 292 us and 79 us.
__global__ __launch_bounds__(256) void k_window_layout(const uint2* __restrict__ recw,
                                                       const uint32_t* __restrict__ keys,
                                                       const uint32_t* __restrict__ win_idx, uint32_t nwin,
                                                       uint32_t nwp, uint32_t* __restrict__ wseg_off,
                                                       uint64_t* __restrict__ bits, uint32_t* __restrict__ tile_h0,
                                                       const uint64_t* __restrict__ acc,
                                                       const uint64_t* __restrict__ hi,
                                                       unsigned long long* __restrict__ acc_w,
                                                       unsigned long long* __restrict__ acc_r,
                                                       float* __restrict__ pair_c, float* __restrict__ pair_sf) {
  constexpr int kRows = kTile / 64;
  const int lane = threadIdx.x & 63;
  const uint32_t tile = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (tile == 0 && lane == 0) wseg_off[nwp] = nwin;
  if ((uint64_t)tile * kTile >= nwin) return;  // uniform per wavefront
  const uint32_t m0 = tile * kTile;
  uint32_t key[kRows], len[kRows], next[kRows];
#pragma unroll
  for (int j = 0; j < kRows; ++j) {
    const uint32_t m = m0 + 64u * j + lane;
    key[j] = m < nwin ? keys[m] : 0xFFFFFFFFu;
    len[j] = m < nwin ? win_idx[m] : 0u;
  }
  // the keys on either side of the tile (no pair: none)
  const uint32_t left = m0 ? keys[m0 - 1] : 0xFFFFFFFFu;
  const uint32_t right = m0 + kTile < nwin ? keys[m0 + kTile] : 0xFFFFFFFFu;
#pragma unroll
  for (int j = 0; j < kRows; ++j) {
    const uint32_t after = j + 1 < kRows ? (uint32_t)__builtin_amdgcn_readfirstlane((int)key[j + 1 < kRows ? j + 1 : j])
                                         : right;
    const uint32_t down = (uint32_t)__shfl_down((int)key[j], 1, 64);
    next[j] = lane == 63 ? after : down;
  }
  // a run's last lane, of a pair that lies in the tile: its front sums
  uint64_t f[kRows], r[kRows];
#pragma unroll
  for (int j = 0; j < kRows; ++j) {
    len[j] = key[j] != 0xFFFFFFFFu ? recw[len[j]].y : 0u;
    const bool done = key[j] != 0xFFFFFFFFu && next[j] != key[j] && key[j] != left;
    f[j] = done ? acc[key[j]] : 0u;
    r[j] = done ? hi[key[j]] : 0u;
  }
  uint64_t w[kRows], hb[kRows];
  uint32_t before = left;             // the key before the row
  uint64_t carry_w = 0, carry_r = 0;  // the run that goes on from the row before
#pragma unroll
  for (int j = 0; j < kRows; ++j) {
    const uint32_t k = key[j];
    const uint32_t up = (uint32_t)__shfl_up((int)k, 1, 64), prev = lane == 0 ? before : up;
    hb[j] = __ballot(k != 0xFFFFFFFFu && prev != k);
    // l 2^24 is exact in double; ql its integer part (< 2^25), rl the rest in
    // units of 2^-48 (< 2^24)
    const double x = (double)__uint_as_float(len[j]) * kFixLen;
    uint32_t ql = (uint32_t)x;
    uint32_t rl = (uint32_t)((x - (double)ql) * kFixLen);
    wave_seg_sum_u(ql, rl, lane == 0 || prev != k ? 1u : 0u);
    const bool goes_on = (hb[j] & (~0ull >> (63 - lane))) == 0;  // still in the run from before the row
    w[j] = ql + (goes_on ? carry_w : 0u);
    const uint64_t rj = rl + (goes_on ? carry_r : 0u);
    const uint64_t fr = sum_r(f[j], r[j]) + rj;
    f[j] = sum_q(f[j], r[j]);
    r[j] = fr;
    before = (uint32_t)__builtin_amdgcn_readlane((int)k, 63);
    const bool carries = before == (uint32_t)__builtin_amdgcn_readlane((int)next[j], 63);
    const uint32_t w0 = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)w[j], 63),
                   w1 = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(w[j] >> 32), 63),
                   r0 = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)rj, 63),
                   r1 = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(rj >> 32), 63);
    carry_w = carries ? (uint64_t)w0 | (uint64_t)w1 << 32 : 0u;
    carry_r = carries ? (uint64_t)r0 | (uint64_t)r1 << 32 : 0u;
  }
  if (lane == 0) tile_h0[tile] = hb[0] & 1u ? key[0] : key[0] + 1u;
#pragma unroll
  for (int j = 0; j < kRows; ++j) {
    const uint32_t m = m0 + 64u * j + lane, k = key[j];
    if (lane == 0 && m < nwin) bits[m >> 6] = hb[j];
    if ((hb[j] >> lane) & 1u) wseg_off[k] = m;
    if (k == 0xFFFFFFFFu) continue;
    if (next[j] != k && k != left) {
      pair_c[k] = pair_length(w[j], f[j], r[j]);
      pair_sf[k] = front_message(f[j]);
    } else if (next[j] != k || (j + 1 == kRows && lane == 63)) {  // from or into another tile
      atomicAdd(acc_w + k, (unsigned long long)w[j]);
      if (r[j]) atomicAdd(acc_r + k, (unsigned long long)r[j]);
    }
  }
}

// C and the front messages of the pairs that k_window_layout left: the
// front-only pairs and the window pairs whose records cross a tile's end
__global__ void k_pair_finish(const uint64_t* __restrict__ acc, const uint64_t* __restrict__ hi,
                              const uint64_t* __restrict__ acc_w, const uint64_t* __restrict__ acc_r,
                              const uint32_t* __restrict__ wseg_off, uint32_t np, uint32_t nwp, float* __restrict__ pair_c, float* __restrict__ pair_sf) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  uint64_t w = 0, r = 0;
  if (p < nwp) {
    if (wseg_off[p] / kTile == (wseg_off[p + 1] - 1u) / kTile) return;
    w = acc_w[p];
    r = acc_r[p];
  }
  const uint64_t a = acc[p], h = hi[p], f = sum_q(a, h);
  pair_c[p] = pair_length(w, f, sum_r(a, h) + r);
  pair_sf[p] = front_message(f);
}

// record -> voxel (for export)
__global__ void k_export_vox(const uint2* __restrict__ rec, uint32_t n, const uint32_t* __restrict__ pair_vox,
                             uint2* __restrict__ out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint2 e = rec[i];
  if (e.x != kGapVox) e.x = pair_vox[e.x];
  out[i] = e;
}

inline unsigned blocks(size_t n, int t) { return (unsigned)((n + t - 1) / t); }
}  // namespace

size_t window_sort_temp_bytes(uint32_t n, int bits) {
  size_t bytes = 0;
  (void)hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, (const uint32_t*)nullptr, (uint32_t*)nullptr,
                                           (const uint32_t*)nullptr, (uint32_t*)nullptr, (int)n, 0, bits);
  return bytes;
}

void launch_brick_flag_counts(const uint8_t* any, const uint8_t* wany, uint32_t nbricks, uint64_t* counts,
                              hipStream_t s) {
  if (nbricks == 0) return;
  hipLaunchKernelGGL(k_brick_flag_counts, dim3(blocks(nbricks, 4)), dim3(256), 0, s, any, wany, nbricks, counts);
}

void launch_pair_table(uint8_t* any, uint8_t* wany, const uint64_t* boff, uint32_t nbricks, uint32_t nwp,
                       uint32_t* pid, uint32_t* pair_vox, hipStream_t s) {
  if (nbricks == 0) return;
  hipLaunchKernelGGL(k_pair_table, dim3(blocks(nbricks, 4)), dim3(256), 0, s, any, wany, boff, nbricks, nwp, pid,
                     pair_vox);
}

void launch_reslice(FrontRec* front, RayRec* lanes, uint32_t nslices, const uint32_t* ids, const uint32_t* lens,
                    const int32_t* slot, const uint32_t* pid, const uint32_t* off_f, const uint32_t* len_f,
                    const uint32_t* off_w, const uint32_t* len_w, uint32_t base_w, uint2* inc, uint64_t* acc,
                    uint64_t* hi, uint32_t np, uint32_t* wkeys, uint32_t* wvals, uint32_t sentinel, hipStream_t s) {
  if (nslices == 0) return;
  launch_zero_words(acc, (size_t)np * 8, s);
  launch_zero_words(hi, (size_t)np * 8, s);
  auto* k = slot ? k_reslice<true> : k_reslice<false>;
  hipLaunchKernelGGL(k, dim3(nslices), dim3(256), 0, s, front, lanes, ids, lens, slot, pid, off_f, len_f, off_w, len_w,
                     base_w, inc, reinterpret_cast<unsigned long long*>(acc), reinterpret_cast<unsigned long long*>(hi),
                     wkeys, wvals, sentinel);
}

void launch_window_layout(const uint2* recw, const uint32_t* keys, const uint32_t* win_idx, uint32_t nwin,
                          uint32_t nwp, uint32_t* wseg_off, uint64_t* bits, uint32_t* tile_h0, const uint64_t* acc,
                          const uint64_t* hi, uint64_t* acc_w, uint64_t* acc_r, float* pair_c, float* pair_sf,
                          hipStream_t s) {
  launch_zero_words(acc_w, (size_t)nwp * 8, s);
  launch_zero_words(acc_r, (size_t)nwp * 8, s);
  hipLaunchKernelGGL(k_window_layout, dim3(blocks(nwin ? nwin : 1, 4 * kTile)), dim3(256), 0, s, recw, keys, win_idx,
                     nwin, nwp, wseg_off, bits, tile_h0, acc, hi, reinterpret_cast<unsigned long long*>(acc_w),
                     reinterpret_cast<unsigned long long*>(acc_r), pair_c, pair_sf);
}

void launch_pair_finish(const uint64_t* acc, const uint64_t* hi, const uint64_t* acc_w, const uint64_t* acc_r,
                        const uint32_t* wseg_off, uint32_t np, uint32_t nwp, float* pair_c, float* pair_sf,
                        hipStream_t s) {
  if (np == 0) return;
  hipLaunchKernelGGL(k_pair_finish, dim3(blocks(np, 256)), dim3(256), 0, s, acc, hi, acc_w, acc_r, wseg_off, np, nwp,
                     pair_c, pair_sf);
}

hipError_t sort_window(uint32_t nwr, int bits, uint32_t* keys_in, uint32_t* keys_out, uint32_t* vals_in,
                       uint32_t* vals_out, void* temp, size_t temp_bytes, hipStream_t s) {
  if (nwr == 0) return hipSuccess;
  size_t tb = temp_bytes;
  return hipcub::DeviceRadixSort::SortPairs(temp, tb, keys_in, keys_out, vals_in, vals_out, (int)nwr, 0, bits, s);
}

void launch_export_vox(const uint2* rec, uint32_t n, const uint32_t* pair_vox, uint2* out, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_export_vox, dim3(blocks(n, 256)), dim3(256), 0, s, rec, n, pair_vox, out);
}

}  // namespace mrf
