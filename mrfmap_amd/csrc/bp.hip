// Loopy-BP message kernels of the MRFMap inference path.
//
//  * k_pair_msg: voxel->ray message log2 n of every (camera, voxel) pair
//    (gvdbkernels.cu:764-773) into a compact per-pair array.
//  * k_ray_messages: L lanes per ray over sliced-ELL pixel tiles; reads log2 n
//    of each record's pair, writes p*l into the record's slot of the
//    camera's voxel-sorted segment array.  Replaces
//    the pre pass (rayStartComputingMessagesFromBrickPre,
//    src/cuda/gvdbkernels.cu:689-819), the infinity term
//    (gvdbkernels.cu:1196-1208) and the post pass
//    (rayStartComputingMessagesFromBrickPost, gvdbkernels.cu:824-1038) with a
//    single launch.
//  * k_seg_sum / k_seg_update: per pair, the fixed-order sum S of
//    its slots, m = logit(clamp(S/C)), B += m - M_c, M_c = m
//    (compute_gvdb_message_to_factors, gvdbkernels.cu:396-496, live 457-479).
//  * residual / marginal / readback kernels (gvdbkernels.cu:469-476, 360-373).
#include <hip/hip_fp16.h>

#include "mrf_kernels.h"

namespace mrf {

namespace {

// ---------------------------------------------------------------- storage
template <int MT>
struct Msg;
// kOut: factor applied to ray->voxel messages p*l before storage (FP16 keeps
// them out of its subnormal range: p*l >= 1e-4 * l).
template <>
struct Msg<kMsgF32> {
  typedef float T;
  static constexpr float kOut = 1.0f;
  __device__ static float load(const T* p, uint32_t i) { return p[i]; }
  __device__ static void store(T* p, uint32_t i, float v) { p[i] = v; }
};
template <>
struct Msg<kMsgF16> {
  typedef __half T;
  static constexpr float kOut = 4096.0f;
  __device__ static float load(const T* p, uint32_t i) { return __half2float(p[i]); }
  __device__ static void store(T* p, uint32_t i, float v) { p[i] = __float2half_rn(v); }
};
template <>
struct Msg<kMsgBF16> {
  typedef uint16_t T;
  static constexpr float kOut = 1.0f;
  __device__ static float load(const T* p, uint32_t i) { return __uint_as_float((uint32_t)p[i] << 16); }
  __device__ static void store(T* p, uint32_t i, float v) {
    uint32_t u = __float_as_uint(v);
    u += 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even
    p[i] = (uint16_t)(u >> 16);
  }
};

// ---------------------------------------------------------------- wave ops
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, ROWS, 0xF, true));
}

// Inclusive prefix sum over the 64 lanes (all lanes must be active):
// row_shr 1/2/4/8 inside each row of 16, then row_bcast 15 and 31.
__device__ __forceinline__ float wave_scan(float x) {
  x += dpp<0x111, 0xF>(x);
  x += dpp<0x112, 0xF>(x);
  x += dpp<0x114, 0xF>(x);
  x += dpp<0x118, 0xF>(x);
  x += dpp<0x142, 0xA>(x);
  x += dpp<0x143, 0xC>(x);
  return x;
}

__device__ __forceinline__ float lane63(float x) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}

// ---------------------------------------------------------------- sensor model
// sigma(z), bias(z): p0 + p1 z (+ p2 z^2) per 20x20-pixel lookup cell
// (get_depth_sigma / get_depth_bias, gvdbkernels.cu:46-55).
// A linear cell has c2 = 0, for which fmaf(z, fmaf(z, 0, c1), c0) is
// fmaf(z, c1, c0) exactly.

// 0.398942 e^{-u^2/2}, the exponential as a power of 2 with the constants
// folded: e^{-u^2/2} = 2^{u^2 (-log2(e) / 2)}
constexpr float kNegHalfLog2e = -0.72134752044448170f;
__device__ __forceinline__ float gauss_a(float u) { return 0.398942f * __builtin_amdgcn_exp2f((u * u) * kNegHalfLog2e); }

// ---------------------------------------------------------------- segments
// A camera's incidences are stored pair-major: pair q owns positions
// [pair_off[q], pair_off[q+1]).  Segment heads are marked in a bitmask and
// each tile of kTile positions knows how many heads precede it, so the pair
// of every position follows from one 64-bit word and a popcount.  All
// segment kernels below work on position tiles (one wavefront per tile), so
// a pair with hundreds of thousands of incidences (the voxels at a camera's
// centre, which every ray of that camera crosses) is spread over many
// wavefronts instead of serialising one.

// Per-lane pair index of positions base + lane (word = head bits of the
// 64 positions starting at base, before = heads before base).
__device__ __forceinline__ uint32_t pair_of(uint64_t word, uint32_t before, int lane) {
  const uint64_t upto = lane == 63 ? ~0ull : ((2ull << lane) - 1ull);
  return before + (uint32_t)__popcll(word & upto) - 1u;
}

// Voxel -> ray message of every pair: n = clamp(1/(1+exp(B - M_c))), camera
// c's own previous message excluded from the belief (gvdbkernels.cu:764-773),
// stored as log2 n (the reference's ln n / ln 2): the ray kernels sum
// l log2 n and take exp2 of the sums (one multiply fewer per exponential than
// e^x = 2^(x log2 e)).
template <int MT>
__device__ __forceinline__ void pair_msg_qv(uint32_t q, uint32_t v, const float* __restrict__ B,
                                            const float* __restrict__ M, typename Msg<MT>::T* __restrict__ apair) {
  const float qv = B[v] - M[q];
  float nn = 1.0f / (1.0f + __expf(qv));
  nn = fminf(fmaxf(nn, kFEps), 1.0f - kFEps);
  Msg<MT>::store(apair, q, __builtin_amdgcn_logf(nn));
}

template <int MT>
__device__ __forceinline__ void pair_msg_one(uint32_t q, const uint32_t* __restrict__ pair_vox,
                                             const float* __restrict__ B, const float* __restrict__ M,
                                             typename Msg<MT>::T* __restrict__ apair) {
  pair_msg_qv<MT>(q, pair_vox[q], B, M, apair);
}

// The window pairs [0, nwp) change every iteration; of the front-only pairs,
// all while *msg_all (the first iterations of a call), afterwards only the
// list dyn (front-only pairs at voxels that some camera reaches with window
// records, each with its voxel, so that its message and belief are loaded
// together).  One launch: the window pairs one per thread, the others
// strided over the grid.
template <int MT>
__global__ __launch_bounds__(256) void k_pair_msg(const uint32_t* __restrict__ pair_vox, uint32_t nwp,
                                                  uint32_t npairs, const uint2* __restrict__ dyn, uint32_t ndyn,
                                                  const float* __restrict__ B, const float* __restrict__ M,
                                                  typename Msg<MT>::T* __restrict__ apair,
                                                  const uint32_t* __restrict__ msg_all) {
  const uint32_t tid = blockIdx.x * blockDim.x + threadIdx.x, stride = gridDim.x * blockDim.x;
  for (uint32_t q = tid; q < nwp; q += stride) pair_msg_one<MT>(q, pair_vox, B, M, apair);
  if (*msg_all) {
    for (uint32_t q = nwp + tid; q < npairs; q += stride) pair_msg_one<MT>(q, pair_vox, B, M, apair);
  } else {
    for (uint32_t k = tid; k < ndyn; k += stride) {
      const uint2 e = dyn[k];  // {pair, voxel}
      pair_msg_qv<MT>(e.x, e.y, B, M, apair);
    }
  }
}

// ---------------------------------------------------------------- list layout
// The voxels of every ray's staged records: per row (record k of the 64 rays
// of a slice) the voxel flags any[v] = 1 (every live record) and wany[v] = 1
// (live window records) are set, skipping a lane whose voxel equals that of
// the ray to its left or above in the pixel tile (the flags say only
// whether).  counts[slice] = {live records, live window records, records
// (gap records included), rays with records}, summed by k_slice_totals: four
// atomics per slice on the same words took 12 ns each (240 us for 640x480
// with few records).
// SLOTS: the staged records hold (linear brick index) * 512 + voxel, and the
// brick's slot is looked up here (neighbouring rays share their bricks).
//
// Brick entries of the window records (bstart; null when not wanted): record
// k of lane l enters a brick when it is a voxel record and the previous
// record of its ray is a gap record, lies in another brick, or does not
// exist.  The 64 lanes' flags of a window row form one 64-bit word.
// tail[lane]: when the first window record continues the brick of the last
// front record, the number of front records since that brick's entry (at most
// 22, the longest crossing of a brick), else 0.  Both look one record back.
//
// A block of four waves is one slice, batches of kB rows going to its waves
// in turn: a wave's batch is a chain of loads (record, slot) before its
// stores, and one wave per slice leaves four waves per SIMD at 640x480 and
// fewer than one below 160x120.  640x480 at 1 cm, 161 M voxels (0.65 GB): 362
// us, mostly the flags' byte stores; with few records (2 cm, endpoint
// activation) 28 us, and 160x120 at 4 cm 21 us.
template <bool SLOTS>
__global__ __launch_bounds__(256) void k_mark_voxels(const FrontRec* __restrict__ front,
                                                     const RayRec* __restrict__ lanes,
                                                     const uint32_t* __restrict__ ids, const int32_t* __restrict__ slot,
                                                     const uint32_t* __restrict__ len_f,
                                                     const uint32_t* __restrict__ off_w,
                                                     const uint32_t* __restrict__ len_w, uint8_t* __restrict__ any,
                                                     uint8_t* __restrict__ wany, uint64_t* __restrict__ bstart,
                                                     uint8_t* __restrict__ tail, uint4* __restrict__ counts) {
  constexpr uint32_t kW = 4, kB = 8;
  __shared__ uint32_t wave_counts[kW][2];
  const uint32_t t = blockIdx.x, wave = threadIdx.x >> 6, l = threadIdx.x & 63u, ray = t * kSlice + l;
  const FrontRec f = front[ray];
  const uint32_t rnw = lanes[ray].nw, nr = f.nf + rnw;
  const uint32_t* __restrict__ src = ids + f.off;
  // a voxel this lane need not flag: the left or the upper ray has it too
  auto dup = [&](uint32_t v) {
    const uint32_t left = (uint32_t)__shfl_up((int)v, 1, 64), up = (uint32_t)__shfl_up((int)v, 8, 64);
    return ((l & 7u) != 0u && left == v) || (l >= 8u && up == v);
  };
  // a batch's loads are in flight together (the bounds lf, lw are uniform per
  // wavefront, so every lane takes part in the shuffles)
  auto pool_ids = [&](uint32_t(&e)[kB]) {
    if constexpr (SLOTS) {
      int32_t sl[kB];
#pragma unroll
      for (uint32_t u = 0; u < kB; ++u) sl[u] = slot[e[u] != kGapVox ? e[u] >> kBrickLog * 3 : 0u];
#pragma unroll
      for (uint32_t u = 0; u < kB; ++u)
        if (e[u] != kGapVox) e[u] = (uint32_t)sl[u] * kBrickVox + (e[u] & (kBrickVox - 1u));
    }
  };
  uint32_t nl = 0, nw = 0;  // below 2^31: the records of a camera are
  const uint32_t lf = len_f[t], lw = len_w[t];
  for (uint32_t k0 = wave * kB; k0 < lf; k0 += kW * kB) {
    uint32_t e[kB];
#pragma unroll
    for (uint32_t u = 0; u < kB; ++u) e[u] = k0 + u < f.nf ? src[(size_t)(k0 + u) * kSlice] : kGapVox;
    pool_ids(e);
#pragma unroll
    for (uint32_t u = 0; u < kB; ++u) {
      const bool live = e[u] != kGapVox;
      nl += (uint32_t)__popcll(__ballot(live));
      const bool d = dup(e[u]);
      if (live && !d) any[e[u]] = 1;
    }
  }
  const uint32_t* __restrict__ srcw = src + (size_t)f.nf * kSlice;
  for (uint32_t k0 = wave * kB; k0 < lw; k0 += kW * kB) {
    uint32_t e[kB];
    uint32_t prev = kGapVox;  // the ray's record before the batch
    if (bstart && f.nf + k0 > 0 && k0 <= rnw) prev = src[(size_t)(f.nf + k0 - 1) * kSlice];
#pragma unroll
    for (uint32_t u = 0; u < kB; ++u) e[u] = k0 + u < rnw ? srcw[(size_t)(k0 + u) * kSlice] : kGapVox;
    if (bstart) {
      uint64_t mine = 0;  // lane u: the word of row k0 + u
#pragma unroll
      for (uint32_t u = 0; u < kB; ++u) {
        const uint32_t cur = e[u];
        const uint64_t m =
            __ballot(cur != kGapVox && (prev == kGapVox || (prev >> kBrickLog * 3) != (cur >> kBrickLog * 3)));
        if (l == u) mine = m;
        prev = cur;
      }
      if (l < kB && k0 + l < lw) bstart[off_w[t] / kSlice + k0 + l] = mine;
    }
    pool_ids(e);
#pragma unroll
    for (uint32_t u = 0; u < kB; ++u) {
      const bool live = e[u] != kGapVox;
      const uint32_t n = (uint32_t)__popcll(__ballot(live));
      nl += n;
      nw += n;
      const bool d = dup(e[u]);
      if (live && !d) {
        any[e[u]] = 1;
        wany[e[u]] = 1;
      }
    }
  }
  if (tail && wave == kW - 1) {  // the wave with the fewest batches
    uint32_t tl = 0;
    if (f.nf && rnw) {
      const uint32_t w0 = srcw[0], last = src[(size_t)(f.nf - 1) * kSlice];
      auto same = [&](uint32_t v) { return v != kGapVox && (v >> kBrickLog * 3) == (w0 >> kBrickLog * 3); };
      if (w0 != kGapVox && same(last)) {
        bool more = true;
        for (tl = 1; more;) {  // records back from the last front record, kB at a time
          uint32_t pv[kB];
#pragma unroll
          for (uint32_t u = 0; u < kB; ++u)
            pv[u] = tl + u < f.nf ? src[(size_t)(f.nf - 1 - tl - u) * kSlice] : kGapVox;
#pragma unroll
          for (uint32_t u = 0; u < kB; ++u) {
            more = more && same(pv[u]);
            if (more) ++tl;
          }
        }
      }
    }
    tail[ray] = (uint8_t)tl;
  }
  if (l == 0) {
    wave_counts[wave][0] = nl;
    wave_counts[wave][1] = nw;
  }
  __syncthreads();
  if (wave != 0) return;
  const uint32_t nray = (uint32_t)__popcll(__ballot(nr != 0u));
  uint32_t nrec = nr;
  for (int o = 32; o > 0; o >>= 1) nrec += (uint32_t)__shfl_xor((int)nrec, o, 64);
  if (l == 0) {
    for (uint32_t w = 1; w < kW; ++w) {
      nl += wave_counts[w][0];
      nw += wave_counts[w][1];
    }
    counts[t] = make_uint4(nl, nw, nrec, nray);
  }
}

// the sums of the slices' counts, in one block
__global__ __launch_bounds__(1024) void k_slice_totals(const uint4* __restrict__ counts, uint32_t nslices,
                                                       uint64_t* __restrict__ totals) {
  __shared__ uint64_t part[16][4];
  uint64_t s[4] = {0, 0, 0, 0};
  for (uint32_t t = threadIdx.x; t < nslices; t += 1024u) {
    const uint4 c = counts[t];
    s[0] += c.x, s[1] += c.y, s[2] += c.z, s[3] += c.w;
  }
  for (int o = 32; o > 0; o >>= 1)
    for (int k = 0; k < 4; ++k) s[k] += (uint64_t)__shfl_xor((unsigned long long)s[k], o, 64);
  if ((threadIdx.x & 63u) == 0u)
    for (int k = 0; k < 4; ++k) part[threadIdx.x >> 6][k] = s[k];
  __syncthreads();
  if (threadIdx.x < 4u) {
    uint64_t v = 0;
    for (int w = 0; w < 16; ++w) v += part[w][threadIdx.x];
    totals[threadIdx.x] = v;
  }
}

// Front chunks: a slice with window records needs ceil(len_f / kChunk) of
// them, a slice without none.
// (cnt[nslices] = 0, so that an exclusive scan of nslices + 1 counts ends
// with the total)
__global__ void k_chunk_counts(const uint32_t* __restrict__ len_f, const uint32_t* __restrict__ len_w,
                               uint32_t nslices, uint32_t* __restrict__ cnt) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t > nslices) return;
  cnt[t] = (t < nslices && len_w[t]) ? (len_f[t] + kChunk - 1) / kChunk : 0u;
}

// Chunk descriptors {chunk, slice, first row, end row} and, per lane of every
// slice, its front span {first record, records to sum: nf, 0 without window}.
__global__ void k_chunk_desc(const uint32_t* __restrict__ chunk_off, const uint32_t* __restrict__ len_f,
                             uint32_t nslices, uint4* __restrict__ desc) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= nslices) return;
  for (uint32_t w = chunk_off[t]; w < chunk_off[t + 1]; ++w) {
    const uint32_t k0 = (w - chunk_off[t]) * kChunk;
    desc[w] = make_uint4(w, t, k0, min(k0 + kChunk, len_f[t]));
  }
}
__global__ void k_front_span(const FrontRec* __restrict__ front, const RayRec* __restrict__ lanes, uint32_t n,
                             uint2* __restrict__ span) {
  const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r < n) span[r] = make_uint2(front[r].off, lanes[r].nw ? front[r].nf : 0u);
}
// Launch order of the slices in the window kernel: per XCD (block b of a grid
// runs on XCD b % 8) its slices, longest window first, by bins of 8 rows (the
// order inside a bin is free: the slices are independent).  Four waves of the
// window kernel fit a SIMD, so of the 4704 slices of a 640x480 image 608 wait
// for a free place, and a long one among them runs when the others are done;
// and with an eighth of the image per XCD, the XCD with the long windows ends
// last.  An XCD takes groups of kOrderGroup neighbouring slices in turn (they
// share lines in its L2; groups of 2 to 32 are within 1 %, of 128 10 %
// slower).  Window kernel in image order and longest first: 640x480 at 1 cm
// 191 and 181 us, 10x10x3 m at 1 cm (3437 slices) 210 and 188, 320x240 at 2
// cm 60.9 and 57.8, 160x120 at 4 cm 42.8 and 42.7.
constexpr uint32_t kOrderBins = 1024, kOrderGroup = 8, kNoSlice = 0xFFFFFFFFu;
__global__ __launch_bounds__(1024) void k_slice_order(const uint32_t* __restrict__ len_w, uint32_t nslices,
                                                      uint32_t per, uint32_t* __restrict__ order) {
  __shared__ uint32_t first[kOrderBins];
  const uint32_t i = threadIdx.x, xcd = blockIdx.x;
  auto slice = [&](uint32_t j) { return (j / kOrderGroup * 8u + xcd) * kOrderGroup + j % kOrderGroup; };
  auto bin = [&](uint32_t t) { return kOrderBins - 1u - min(len_w[t] / 8u, kOrderBins - 1u); };
  first[i] = 0;
  __syncthreads();
  for (uint32_t j = i; j < per; j += kOrderBins) {
    if (slice(j) < nslices) atomicAdd(&first[bin(slice(j))], 1u);
  }
  __syncthreads();
  const uint32_t n = first[i];
  for (uint32_t o = 1; o < kOrderBins; o <<= 1) {  // inclusive scan
    const uint32_t v = i >= o ? first[i - o] : 0u;
    __syncthreads();
    first[i] += v;
    __syncthreads();
  }
  const uint32_t e = first[i] - n, total = first[kOrderBins - 1];
  __syncthreads();
  first[i] = e;
  __syncthreads();
  for (uint32_t j = i; j < per; j += kOrderBins) {
    if (slice(j) < nslices) order[8u * atomicAdd(&first[bin(slice(j))], 1u) + xcd] = slice(j);
    if (j >= total) order[8u * j + xcd] = kNoSlice;
  }
}
__global__ void k_gather_desc(const uint4* __restrict__ desc, const uint32_t* __restrict__ idx, uint32_t n,
                              uint4* __restrict__ out) {
  const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < n) out[j] = desc[idx[j]];
}

// ---------------------------------------------------------------- ray kernels
// Front sums.  Front records have psi(s) = 0, so all they contribute to a ray
// is the visibility sum Lambda = sum l log2 n (in units of ln 2; the reference's visibility
// includes the voxel itself, gvdbkernels.cu:781-783); their messages are
// the constant F_EPS * l, summed per pair once per traversal, and their
// length sum is geometric (RayRec::ks/kc).  Chunk c of a slice is records
// [c * kChunk, (c + 1) * kChunk) of its 64 rays, one wavefront at a time,
// so the work splits into near-equal pieces whatever the ray lengths; each
// lane writes its Kahan-compensated partial sum.  Rays without window
// records are skipped.
//
// While the log2 n of all pairs are recomputed (the first two iterations of
// a call) every chunk is summed in record order, and the records whose log2 n
// stops changing (bit clear in the chunk-lane mask fdmask) are also summed
// on their own into fstatic.  Afterwards only the chunks with a changing
// record are visited (dyn_desc), and each lane adds its changing records,
// copied in order into a compact block of the chunk (dfront, rows of 64
// lanes, {first row, rows} in dcr), to its kept static sum: static records
// are not read again.  The two orders of summation differ only by FP32
// rounding.
template <int MI, int U>
__global__ __launch_bounds__(256) void k_front_sums(const uint2* __restrict__ fspan, const uint4* __restrict__ desc,
                                                    uint32_t nchunks, const uint4* __restrict__ dyn_desc,
                                                    uint32_t ndyn_chunks, const uint2* __restrict__ inc,
                                                    const typename Msg<MI>::T* __restrict__ Xi,
                                                    float* __restrict__ partial,
                                                    const uint32_t* __restrict__ msg_all,
                                                    const uint32_t* __restrict__ fdmask, float* __restrict__ fstatic,
                                                    const uint2* __restrict__ dfront, const uint2* __restrict__ dcr) {
  // a wave per entry of the descriptor list (one wave-uniform load per
  // chunk), the waves past the list's end exit at once.  The grid covers
  // every chunk; the loop strides for a smaller one.
  const bool all = *msg_all != 0u;
  const uint32_t n = all ? nchunks : ndyn_chunks;
  const uint32_t nwaves = gridDim.x * (blockDim.x >> 6);
  const uint32_t l = threadIdx.x & 63u;
  for (uint32_t i = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)); i < n;
       i += nwaves) {
    if (all) {
      const uint4 d = desc[i];  // {chunk, slice, first row, end row}
      const uint2 fs = fspan[d.y * kSlice + l];
      const uint32_t k1 = min(d.z + kChunk, fs.y);
      const uint2* __restrict__ rf = inc + fs.x;
      const uint32_t m = fdmask[(size_t)d.x * kSlice + l];
      Kahan acc = {0.f, 0.f}, accs = {0.f, 0.f};
      for (uint32_t kb = d.z; kb < d.w; kb += U) {
        uint2 e[U];
        float x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const uint32_t k = kb + u;
          e[u] = k < k1 ? rf[(size_t)k * kSlice] : make_uint2(kGapVox, 0u);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) x[u] = e[u].x != kGapVox ? Msg<MI>::load(Xi, e[u].x) : 0.0f;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const uint32_t k = kb + u;
          if (k < k1) {
            const float v = __uint_as_float(e[u].y) * x[u];
            acc.add(v);
            if (((m >> (k - d.z)) & 1u) == 0u) accs.add(v);
          }
        }
      }
      partial[(size_t)d.x * kSlice + l] = acc.at(0.0f);
      fstatic[(size_t)d.x * kSlice + l] = accs.at(0.0f);
    } else {
      const uint32_t w = dyn_desc[i].x;  // the chunk
      const uint2 cr = dcr[i];           // {first row, rows} of its compact block
      const uint32_t cnt = (uint32_t)__popc(fdmask[(size_t)w * kSlice + l]);
      const uint2* __restrict__ rf = dfront + (size_t)cr.x * kSlice + l;
      Kahan acc = {fstatic[(size_t)w * kSlice + l], 0.f};
      for (uint32_t rb = 0; rb < cr.y; rb += U) {
        uint2 e[U];
        float x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) e[u] = rb + u < cnt ? rf[(size_t)(rb + u) * kSlice] : make_uint2(kGapVox, 0u);
#pragma unroll
        for (int u = 0; u < U; ++u) x[u] = e[u].x != kGapVox ? Msg<MI>::load(Xi, e[u].x) : 0.0f;
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (rb + u < cnt) acc.add(__uint_as_float(e[u].y) * x[u]);
      }
      partial[(size_t)w * kSlice + l] = acc.at(0.0f);
    }
  }
}

// Per front chunk (the layout of k_front_sums): a record changes when it
// belongs to a window pair or to a front-only pair at a voxel that some
// camera reaches with window records (pflag[q - nwp] != 0); the others'
// log2 n stop changing after the first two iterations of a call.  Per lane,
// dmask has bit k - first row set for each changing record k; per chunk,
// rows = the most changing records of a lane (the rows of its compact
// block), 0 when no record changes (the chunk's partial sums can be kept).
// The live records that do not change, which the front sums stop reading
// after the first two iterations of a call, are counted into nstatic.
__global__ __launch_bounds__(1024) void k_chunk_static(const uint2* __restrict__ fspan,
                                                      const uint4* __restrict__ desc, uint32_t nchunks,
                                                      const uint2* __restrict__ inc,
                                                      uint32_t nwp, const uint32_t* __restrict__ pflag,
                                                      uint32_t* __restrict__ dyn_flag, uint32_t* __restrict__ dmask,
                                                      uint32_t* __restrict__ rows,
                                                      unsigned long long* __restrict__ nstatic) {
  __shared__ uint32_t block_kept[16];
  const uint32_t w = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const uint32_t l = threadIdx.x & 63u;
  if (w >= nchunks) {  // uniform per wavefront; still takes part in the block's sum
    if (l == 0) block_kept[threadIdx.x >> 6] = 0u;
    __syncthreads();
    return;
  }
  const uint4 d = desc[w];
  const uint2 fs = fspan[d.y * kSlice + l];
  const uint32_t k0 = d.z, k1 = min(k0 + kChunk, fs.y);
  const uint2* __restrict__ rf = inc + fs.x;
  // all loads of the chunk first, then the flags of its front-only pairs
  uint32_t q[kChunk], pf[kChunk];
#pragma unroll
  for (uint32_t b = 0; b < kChunk; ++b) q[b] = k0 + b < k1 ? rf[(size_t)(k0 + b) * kSlice].x : kGapVox;
#pragma unroll
  for (uint32_t b = 0; b < kChunk; ++b) pf[b] = q[b] != kGapVox && q[b] >= nwp ? pflag[q[b] - nwp] : 0u;
  uint32_t m = 0, live = 0;
#pragma unroll
  for (uint32_t b = 0; b < kChunk; ++b) {
    if (q[b] == kGapVox) continue;
    ++live;
    if (q[b] < nwp || pf[b] != 0u) m |= 1u << b;
  }
  dmask[(size_t)w * kSlice + l] = m;
  uint32_t nr = (uint32_t)__popc(m);
  uint32_t kept = live - nr;  // this lane's records whose sums are kept
  for (int o = 32; o > 0; o >>= 1) {
    nr = max(nr, (uint32_t)__shfl_xor((int)nr, o, 64));
    kept += (uint32_t)__shfl_xor((int)kept, o, 64);
  }
  if (l == 0) {
    dyn_flag[w] = nr ? 1u : 0u;
    rows[w] = nr;
    block_kept[threadIdx.x >> 6] = kept;
  }
  // one atomic per block, not per chunk: they all go to one address
  __syncthreads();
  if (threadIdx.x == 0) {
    uint64_t sum = 0;
    for (uint32_t i = 0; i < (blockDim.x >> 6); ++i) sum += block_kept[i];
    if (sum) atomicAdd(nstatic, (unsigned long long)sum);
  }
}

// rows of every changing chunk's compact block, in list order
__global__ void k_dyn_rows(const uint4* __restrict__ dyn_desc, uint32_t n, const uint32_t* __restrict__ rows,
                           uint32_t* __restrict__ out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = rows[dyn_desc[i].x];
}

// The compact blocks: per entry of the changing-chunk list (one wave), each
// lane copies its changing records of the chunk in order to rows
// first row + 0, 1, ... of the block; dcr[i] = {first row, rows}.
__global__ __launch_bounds__(256) void k_fill_dfront(const uint2* __restrict__ fspan,
                                                     const uint4* __restrict__ dyn_desc, uint32_t n,
                                                     const uint2* __restrict__ inc,
                                                     const uint32_t* __restrict__ dmask,
                                                     const uint32_t* __restrict__ rows,
                                                     const uint32_t* __restrict__ row_off, uint2* __restrict__ dfront,
                                                     uint2* __restrict__ dcr) {
  const uint32_t i = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (i >= n) return;  // uniform per wavefront
  const uint32_t l = threadIdx.x & 63u;
  const uint4 d = dyn_desc[i];
  const uint2 fs = fspan[d.y * kSlice + l];
  const uint2* __restrict__ rf = inc + fs.x;
  const uint32_t m = dmask[(size_t)d.x * kSlice + l];
  const uint32_t r0 = row_off[i];
  uint2 e[kChunk];
#pragma unroll
  for (uint32_t b = 0; b < kChunk; ++b) e[b] = (m >> b) & 1u ? rf[(size_t)(d.z + b) * kSlice] : make_uint2(0u, 0u);
  uint32_t r = 0;
#pragma unroll
  for (uint32_t b = 0; b < kChunk; ++b)
    if ((m >> b) & 1u) dfront[(size_t)(r0 + r++) * kSlice + l] = e[b];
  if (l == 0) dcr[i] = make_uint2(r0, rows[d.x]);
}

// ---------------------------------------------------------------- buffer access
// Raw buffer loads and stores through a wave-uniform resource (base address,
// size in bytes): the hardware's range check makes an access at or past the
// size read 0 or be dropped, and constant offsets fold into the instruction.
typedef __amdgpu_buffer_rsrc_t Rsrc;
constexpr int kRsrcWord3 = 0x00020000;  // gfx9 raw buffer: 32-bit data format, no swizzle
__device__ __forceinline__ Rsrc make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, kRsrcWord3);
}

template <int MT>
struct MsgB;
template <>
struct MsgB<kMsgF32> {
  static constexpr uint32_t kShift = 2;
  __device__ static float load(Rsrc r, uint32_t off) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
  }
  __device__ static void store(Rsrc r, uint32_t off, float v) {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, (int)off, 0, 0);
  }
};
template <>
struct MsgB<kMsgF16> {
  static constexpr uint32_t kShift = 1;
  __device__ static float load(Rsrc r, uint32_t off) {
    return __half2float(__ushort_as_half((unsigned short)__builtin_amdgcn_raw_buffer_load_b16(r, (int)off, 0, 0)));
  }
  __device__ static void store(Rsrc r, uint32_t off, float v) {
    __builtin_amdgcn_raw_buffer_store_b16(__half_as_ushort(__float2half_rn(v)), r, (int)off, 0, 0);
  }
};
template <>
struct MsgB<kMsgBF16> {
  static constexpr uint32_t kShift = 1;
  __device__ static float load(Rsrc r, uint32_t off) {
    return __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b16(r, (int)off, 0, 0) << 16);
  }
  __device__ static void store(Rsrc r, uint32_t off, float v) {
    uint32_t u = __float_as_uint(v);
    u += 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even
    __builtin_amdgcn_raw_buffer_store_b16((unsigned short)(u >> 16), r, (int)off, 0, 0);
  }
};

// Window of every ray: one thread per ray, the 64 rays of a slice in one
// wavefront; record k of all lanes of a slice is contiguous.  Lambda starts
// from the ray's front partial sums, the travelled length from the front's
// Kahan state.  Pass 1: vpsi_k = exp(Lambda_k) psi(s_k), tau_k = vpsi_k
// (1 - n_k), T = sum tau (+ V_n when the walk ran out and d lies beyond,
// gvdbkernels.cu:1196-1208).  Pass 2 restarts at the window with the saved
// sums and writes p = mu1 / (mu1 + mu0 + 1e-7), mu1 = P + vpsi,
// mu0 = P + R / n (gvdbkernels.cu:936-951) times l into the record's own
// slot of the window region (coalesced; the segment sums gather them in
// voxel order).  The file is built without FP contraction, so pass 2
// recomputes pass 1's terms bit for bit.
//
// Records are processed in batches of UW, software-pipelined: while a batch
// is computed, the message gathers of the next batch and the record loads of
// the one after are in flight (two batches of lengths and messages and one
// of records in registers, used in turn, so nothing is copied).  Every
// access goes through a buffer resource: the records and the message slots
// of the slice's window region, and the pair messages.  Loads past the
// region read {0, 0} (pair 0, length 0); a gap record's pair index is past
// the message array, so its message reads 0, and since every pair's
// log2 n <= log2(1 - F_EPS) < 0, a record is live exactly when its message is
// nonzero.  All lanes run to the slice's longest ray (uniform loop control);
// slots past a lane's last record are computed too: they have length 0, so
// the visibility and length sums add exact zeros, their taus are left out
// of T and P by a select, their stores land in the slice's padding or past
// the region (dropped), and no kernel reads those slots.
// UW records of a lane from row k0 on (record k at byte lane_off + k * 64 * 8)
template <int UW>
__device__ __forceinline__ void win_load(Rsrc rr, uint32_t lane_off, uint32_t k0, uint2 (&e)[UW]) {
#pragma unroll
  for (int u = 0; u < UW; ++u) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b64(rr, (int)(lane_off + (k0 + (uint32_t)u) * (kSlice * 8u)), 0, 0);
    e[u] = make_uint2((uint32_t)v[0], (uint32_t)v[1]);
  }
}
// gathers of the batch's messages; the lengths move to their own registers
template <int MI, int UW>
__device__ __forceinline__ void win_issue(Rsrc rx, const uint2 (&e)[UW], float (&ln)[UW], float (&x)[UW]) {
#pragma unroll
  for (int u = 0; u < UW; ++u) {
    x[u] = MsgB<MI>::load(rx, e[u].x << MsgB<MI>::kShift);
    ln[u] = __uint_as_float(e[u].y);
  }
}

struct WinRay {
  float z0, inv, d;
  Poly sig3, bia;  // 3 sigma(z) (the likelihood width) and bias(z)
  float rsig3;     // 1 / sig3.c0
};

// a = 0.398942 e^{-u^2/2} and psi(s; d) = N(d; s + bias(s), (3 sigma(s))^2) =
// a / (3 sigma(s)) (depth_potential, gvdbkernels.cu:57-72).  CS: every lookup
// cell's sigma and bias are constants (c1 = c2 = 0), so the polynomials and
// the reciprocal leave the loop with the same bits: fmaf(z, fmaf(z, 0, 0), c0)
// is c0.
template <bool CS>
__device__ __forceinline__ void win_psi(const WinRay& r, float s, float& ap, float& ps) {
  const float diff = fabsf(r.d - (s + (CS ? r.bia.c0 : r.bia(s))));
  const float inv = CS ? r.rsig3 : __builtin_amdgcn_rcpf(r.sig3(s));
  ap = gauss_a(diff * inv);
  ps = ap * inv;
}

// depth at the exit of a record: z0 + (travelled chord length) * inv
__device__ __forceinline__ float win_depth(const WinRay& r, const Kahan& kS, float ln) {
  return fmaf(kS.at(ln), r.inv, r.z0);
}

// terms of one record shared by both passes: a = l log2 n, vpsi, n
template <bool CS>
__device__ __forceinline__ void win_terms(const WinRay& r, const Kahan& kL, const Kahan& kS, float ln, float lnn,
                                          float& a, float& vpsi, float& nn) {
  a = ln * lnn;
  const float s = win_depth(r, kS, ln);
  float ap, ps;
  win_psi<CS>(r, s, ap, ps);
  // a gap or padding record (log2 n = 0) gets a vpsi but n = 1 exactly, so
  // its tau vpsi (1 - n) is exactly 0; its own message is never read
  vpsi = __builtin_amdgcn_exp2f(kL.at(a)) * ps;
  nn = __builtin_amdgcn_exp2f(lnn);
}

template <int UW, bool CS>
__device__ __forceinline__ void win_pass1(const WinRay& r, uint32_t k0, uint32_t nw, const float (&ln)[UW],
                                          const float (&x)[UW], Kahan& kL, Kahan& kS, float& T) {
#pragma unroll
  for (int u = 0; u < UW; ++u) {
    const bool valid = k0 + u < nw;
    float a, vpsi, nn;
    win_terms<CS>(r, kL, kS, ln[u], x[u], a, vpsi, nn);
    T += valid ? vpsi * (1.0f - nn) : 0.0f;
    kL.add(a);  // a = 0 and l = 0 past the lane's last record: no select needed
    kS.add(ln[u]);
  }
}

// Pass 1 of the reference's pre pass with its flush-to-zero arithmetic
// (MRF_VIS_BRICK_LOCAL): a tau is non-zero there only when a = 0.398942
// e^{-u^2/2}, psi = a / (3 sigma), b = V (1 - n) and b psi are all at least
// the smallest normal float (gvdbkernels.cu:57-72, 792-795).  Until the
// first such tau the visibility sum restarts at every brick entry (bit l of
// the row's word in bsw; the restore at gvdbkernels.cu:708-715 tests the
// accumulated tau), and only such taus enter T.  The terms are those of
// win_terms, so a ray whose restarts change nothing gets the T of pass 1.
// The per-lane conditions are kept as wavefront masks in scalar registers (nz:
// the lanes that have a counted tau; bsw: the rows' brick-entry words, a
// batch loaded together), so a record costs two selects for the restart and
// one for the tau and the batch has no branches: with a branch and a scalar
// load per record the compiler waited for each word in turn.  4 x 160x120 at
// 4 cm (one wave per SIMD, bound by latency): 48.3 -> 42.8 us per camera pass
// together with the constant sensor model; 13 x 640x480 at 1 cm (bound by
// memory traffic): 190 us either way.
constexpr float kFtzMin = 0x1p-126f;

template <int UW, bool CS>
__device__ __forceinline__ void win_pass1_bl(const WinRay& r, uint32_t k0, uint32_t nw, const float (&ln)[UW],
                                             const float (&x)[UW], const uint64_t* __restrict__ bsw, Kahan& kL,
                                             Kahan& kS, float& T, uint64_t& nz) {
  uint64_t w[UW];
#pragma unroll
  for (int u = 0; u < UW; ++u) w[u] = bsw[k0 + u];
#pragma unroll
  for (int u = 0; u < UW; ++u) {
    const uint64_t valid = __ballot(k0 + u < nw);
    const bool restart = __builtin_amdgcn_inverse_ballot_w64(w[u] & valid & ~nz);
    kL.s = restart ? 0.0f : kL.s;
    kL.c = restart ? 0.0f : kL.c;
    const float lnn = x[u];
    const float a = ln[u] * lnn;
    const float s = win_depth(r, kS, ln[u]);
    float ap, ps;
    win_psi<CS>(r, s, ap, ps);
    const float V = __builtin_amdgcn_exp2f(kL.at(a));
    const float nn = __builtin_amdgcn_exp2f(lnn);
    const float b = V * (1.0f - nn);
    // every factor at least 2^-126 (log2 n = 0, a gap or padding record, gives b = 0)
    const uint64_t counted = valid & __ballot(fminf(fminf(ap, ps), fminf(b, b * ps)) >= kFtzMin);
    T += __builtin_amdgcn_inverse_ballot_w64(counted) ? (V * ps) * (1.0f - nn) : 0.0f;
    nz |= counted;
    kL.add(a);  // a = 0 and l = 0 past the lane's last record: no select needed
    kS.add(ln[u]);
  }
}

template <int UW, bool BL, bool CS>
__device__ __forceinline__ void win_pass1_any(const WinRay& r, uint32_t k0, uint32_t nw, const float (&ln)[UW],
                                              const float (&x)[UW], const uint64_t* __restrict__ bsw, Kahan& kL,
                                              Kahan& kS, float& T, uint64_t& nz) {
  if constexpr (BL)
    win_pass1_bl<UW, CS>(r, k0, nw, ln, x, bsw, kL, kS, T, nz);
  else
    win_pass1<UW, CS>(r, k0, nw, ln, x, kL, kS, T);
}

template <int MO, int UW, bool CS>
__device__ __forceinline__ void win_pass2(const WinRay& r, uint32_t k0, uint32_t nw, const float (&ln)[UW],
                                          const float (&x)[UW], float T, Rsrc ro, uint32_t lane_off, Kahan& kL,
                                          Kahan& kS, float& P) {
  typedef typename Msg<MO>::T TO;
#pragma unroll
  for (int u = 0; u < UW; ++u) {
    const bool valid = k0 + u < nw;
    float a, vpsi, nn;
    win_terms<CS>(r, kL, kS, ln[u], x[u], a, vpsi, nn);
    const float tau = vpsi * (1.0f - nn);
    const float R = (T - P) - tau;
    const float mu1 = P + vpsi;
    const float mu0 = P + R * __builtin_amdgcn_rcpf(nn);
    float p = mu1 * __builtin_amdgcn_rcpf(mu1 + mu0 + kMsgNormEps);
    p = fminf(fmaxf(p, kFEps), 1.0f - kFEps);
    MsgB<MO>::store(ro, lane_off + (k0 + (uint32_t)u) * (kSlice * (uint32_t)sizeof(TO)), p * ln[u] * Msg<MO>::kOut);
    kL.add(a);  // a = 0 and l = 0 past the lane's last record: no select needed
    kS.add(ln[u]);
    P += valid ? tau : 0.0f;
  }
}

template <int MI, int MO, int UW, bool BL, bool CS>
__global__ __launch_bounds__(64) void k_ray_window(const RayRec* __restrict__ lanes, const uint32_t* __restrict__ len_w,
                                                    const uint32_t* __restrict__ order,
                                                    const uint32_t* __restrict__ chunk_off,
                                                    const float* __restrict__ partial, const uint2* __restrict__ inc,
                                                    uint32_t base_w,
                                                    const typename Msg<MI>::T* __restrict__ Xi, uint32_t npairs,
                                                    typename Msg<MO>::T* __restrict__ Xo,
                                                    const float* __restrict__ sigt, const float* __restrict__ biat,
                                                    int lookup_n, const FrontRec* __restrict__ front,
                                                    const uint64_t* __restrict__ bstart,
                                                    const uint8_t* __restrict__ tail) {
  typedef typename Msg<MI>::T TI;
  typedef typename Msg<MO>::T TO;
  // one wave (one slice) per block, so that a finished wave frees its slot at
  // once
  const uint32_t t = order[blockIdx.x], l = threadIdx.x, ray = t * kSlice + l;
  if (t == kNoSlice) return;
  const uint32_t lw = len_w[t];
  if (lw == 0) return;
  const RayRec rec = lanes[ray];
  const uint32_t nw = rec.nw;
  // a lane without window records leaves: the ballots below have 0 for it, and
  // nothing below reads a value of another lane (what is read from the first
  // lane left, by readfirstlane, is the same in all of them)
  if (nw == 0) return;

  // the front's visibility sum: the partial sums of the slice's front chunks, loaded 8 at a time
  Kahan kL = {0.f, 0.f};
  const uint32_t c1 = chunk_off[t + 1];
  for (uint32_t c0 = chunk_off[t]; c0 < c1; c0 += 8) {
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = c0 + i < c1 ? partial[(size_t)(c0 + i) * kSlice + l] : 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (c0 + i < c1) kL.add(v[i]);
  }
  Kahan kS = {rec.ks, rec.kc};
  WinRay r;
  load_cell(sigt, biat, lookup_n, rec.cell_flags & kCellMask, r.sig3, r.bia);
  r.sig3.c0 *= 3.0f;
  r.sig3.c1 *= 3.0f;
  r.sig3.c2 *= 3.0f;
  r.rsig3 = __builtin_amdgcn_rcpf(r.sig3.c0);
  r.z0 = rec.z0;
  r.inv = rec.inv_norm;
  r.d = rec.depth;
  const Kahan L0 = kL, S0 = kS;
  // the slice's window region (record k of lane l at sw + k * 64 + l), wave-uniform
  const uint32_t sw = __builtin_amdgcn_readfirstlane(rec.off_w - l);
  const uint32_t lws = __builtin_amdgcn_readfirstlane(lw);
  const Rsrc rr = make_rsrc(inc + sw, lws * kSlice * 8u);
  const Rsrc rx = make_rsrc(Xi, npairs * (uint32_t)sizeof(TI));
  const Rsrc ro = make_rsrc(Xo + (sw - base_w), lws * kSlice * (uint32_t)sizeof(TO));
  const uint32_t lr = l * 8u, lo = l * (uint32_t)sizeof(TO);

  float lA[UW], xA[UW], lB[UW], xB[UW];
  uint2 e[UW];
  // pass 1
  float T = 0.0f;  // sum of the taus: positive terms, a plain sum
  uint64_t nz = 0;
  const uint64_t* bsw = nullptr;
  if constexpr (BL) {
    // the pre pass enters the window with the visibility sum of the front
    // records in the first window record's brick (every front tau is 0);
    // bit l of word k of bsw: window record k of this lane enters a brick
    // (the slice's rows of the word array, padded past the last slice)
    // (at most 22 records, the longest crossing of a brick; 8 record loads,
    // then their 8 gathers, in flight at a time, summed in record order)
    const FrontRec fr = front[ray];
    const uint32_t tl = tail[ray];
    const uint2* __restrict__ tr = inc + fr.off + (size_t)(fr.nf - tl) * kSlice;
    Kahan kp = {0.f, 0.f};
    for (uint32_t b = 0; b < tl; b += 8) {
      uint2 et[8];
      float tx[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) et[i] = b + i < tl ? tr[(size_t)(b + i) * kSlice] : make_uint2(0u, 0u);
#pragma unroll
      for (int i = 0; i < 8; ++i) tx[i] = b + i < tl ? Msg<MI>::load(Xi, et[i].x) : 0.0f;
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (b + i < tl) kp.add(__uint_as_float(et[i].y) * tx[i]);
    }
    kL = kp;
    bsw = bstart + (sw - base_w) / kSlice;
  }
  win_load<UW>(rr, lr, 0, e);
  win_issue<MI, UW>(rx, e, lA, xA);
  win_load<UW>(rr, lr, UW, e);
  for (uint32_t k0 = 0;; k0 += 2 * UW) {  // bounded by the slice's longest ray: uniform control flow
    win_issue<MI, UW>(rx, e, lB, xB);
    win_load<UW>(rr, lr, k0 + 2 * UW, e);
    win_pass1_any<UW, BL, CS>(r, k0, nw, lA, xA, bsw, kL, kS, T, nz);
    if (k0 + UW >= lws) break;
    win_issue<MI, UW>(rx, e, lA, xA);
    win_load<UW>(rr, lr, k0 + 3 * UW, e);
    win_pass1_any<UW, BL, CS>(r, k0 + UW, nw, lB, xB, bsw, kL, kS, T, nz);
    if (k0 + 2 * UW >= lws) break;
  }
  if (rec.cell_flags & kInfTerm) T += __builtin_amdgcn_exp2f(kL.at(0.0f));  // decided at traversal

  // pass 2
  kL = L0;
  kS = S0;
  float P = 0.0f;  // prefix sum of the taus
  win_load<UW>(rr, lr, 0, e);
  win_issue<MI, UW>(rx, e, lA, xA);
  win_load<UW>(rr, lr, UW, e);
  for (uint32_t k0 = 0;; k0 += 2 * UW) {
    win_issue<MI, UW>(rx, e, lB, xB);
    win_load<UW>(rr, lr, k0 + 2 * UW, e);
    win_pass2<MO, UW, CS>(r, k0, nw, lA, xA, T, ro, lo, kL, kS, P);
    if (k0 + UW >= lws) break;
    win_issue<MI, UW>(rx, e, lA, xA);
    win_load<UW>(rr, lr, k0 + 3 * UW, e);
    win_pass2<MO, UW, CS>(r, k0 + UW, nw, lB, xB, T, ro, lo, kL, kS, P);
    if (k0 + 2 * UW >= lws) break;
  }
}

// Segment sums S_q = sum of p*l over pair q's positions, in a fixed order.
// One wavefront per tile of kTile = 512 positions.  The kernel waits on the
// gather of the messages (4 B each from a region written in ray order), so
// consecutive lanes take consecutive positions: a pair's records lie close
// together (neighbouring rays at the same step) and share the cache lines of
// one load.  The messages then change hands through LDS: lane l sums the 8
// consecutive positions j0 + 8l .. j0 + 8l + 7.  The indices are read once
// per iteration and are not kept in the caches, which hold the messages.
// Groups of kSegGroup consecutive blocks (a brick or two of pairs) run on one
// XCD, whose L2 then serves the lines that neighbouring voxels share.
// 13 x 640x480 at 1 cm, 30 M messages per camera: 113 us with 8 consecutive
// positions per lane, 109 coalesced, 106 with the indices uncached, 100 with
// the XCD groups (126-136 us without the bounds-test-free path or with groups
// of 512 blocks).
// Each lane sums its runs serially and writes the segments that start and
// end inside it; the runs that cross lanes are joined by one segmented
// inclusive scan over the 64 lanes (DPP).  Of the segments that cross tiles,
// the part that started in an earlier tile goes to pf, the part that
// continues into the next tile to pl, and a tile lying wholly inside one
// segment to mid; k_seg_update joins them.

template <int CTRL, int ROWS>
__device__ __forceinline__ int dppi(int x) {
  return __builtin_amdgcn_update_dpp(0, x, CTRL, ROWS, 0xF, true);
}

// (x, f) <- (x_left, f_left) (+) (x, f): add the left value unless a segment
// starts at or before this lane.
template <int CTRL, int ROWS>
__device__ __forceinline__ void seg_step(float& x, int& f) {
  const float y = dpp<CTRL, ROWS>(x);
  const int g = dppi<CTRL, ROWS>(f);
  x = f ? x : x + y;
  f |= g;
}

__device__ __forceinline__ void wave_seg_scan(float& x, int& f) {
  seg_step<0x111, 0xF>(x, f);
  seg_step<0x112, 0xF>(x, f);
  seg_step<0x114, 0xF>(x, f);
  seg_step<0x118, 0xF>(x, f);
  seg_step<0x142, 0xA>(x, f);
  seg_step<0x143, 0xC>(x, f);
}

__device__ __forceinline__ int wave_scan_i(int x) {
  x += dppi<0x111, 0xF>(x);
  x += dppi<0x112, 0xF>(x);
  x += dppi<0x114, 0xF>(x);
  x += dppi<0x118, 0xF>(x);
  x += dppi<0x142, 0xA>(x);
  x += dppi<0x143, 0xC>(x);
  return x;
}

// Messages X[idx[j]] of positions [j0, j1) of a tile, 8 consecutive ones per
// lane (zero past j1); sh: the wavefront's kTile floats of LDS
template <int MT>
__device__ __forceinline__ void load_tile(const typename Msg<MT>::T* __restrict__ X, const uint32_t* __restrict__ idx,
                                          uint32_t j0, uint32_t j1, uint32_t lane, float* sh, float (&x)[8]) {
  float g[8];
  if (j0 + kTile <= j1) {  // uniform: every tile but the last, no bounds tests
    uint32_t ix[8];
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) ix[i] = __builtin_nontemporal_load(idx + j0 + 64u * i + lane);
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) g[i] = Msg<MT>::load(X, ix[i]);
  } else {
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) {
      const uint32_t j = j0 + 64u * i + lane;
      g[i] = j < j1 ? Msg<MT>::load(X, idx[j]) : 0.0f;
    }
  }
#pragma unroll
  for (uint32_t i = 0; i < 8; ++i) sh[64u * i + lane] = g[i];
  // one wavefront writes and reads: LDS operations of a wavefront complete in order
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  const float4 a = *reinterpret_cast<const float4*>(sh + 8u * lane);
  const float4 b = *reinterpret_cast<const float4*>(sh + 8u * lane + 4u);
  x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
  x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
}

constexpr uint32_t kSegGroup = 4;

template <int MT>
__global__ __launch_bounds__(256) void k_seg_sum(const uint64_t* __restrict__ heads, const uint32_t* __restrict__ tile_h0,
                                                 uint32_t nlive, const typename Msg<MT>::T* __restrict__ X,
                                                 const uint32_t* __restrict__ idx,
                                                 float* __restrict__ S,
                                                 float* __restrict__ pf_v,
                                                 float* __restrict__ pl_v, float* __restrict__ mid) {
  __shared__ __align__(16) float sh[4][kTile];
  const int lane = threadIdx.x & 63;
  const uint32_t lb = (blockIdx.x / (8u * kSegGroup)) * (8u * kSegGroup) + (blockIdx.x & 7u) * kSegGroup +
                      ((blockIdx.x >> 3) % kSegGroup);
  const uint32_t w = lb * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const uint32_t j0 = w * kTile;
  if (j0 >= nlive) return;  // uniform per wavefront
  const uint32_t j1 = min(j0 + kTile, nlive);
  const uint32_t p0 = j0 + 8u * (uint32_t)lane;
  // head bits of this lane's 8 positions (zero past nlive)
  const uint32_t hb = p0 < j1 ? (uint32_t)(heads[p0 >> 6] >> (p0 & 63)) & 0xFFu : 0u;
  float x[8];
  load_tile<MT>(X, idx, j0, j1, (uint32_t)lane, sh[threadIdx.x >> 6], x);
  const int nh = __popc(hb);
  const int incl = wave_scan_i(nh);
  const uint32_t before = tile_h0[w] + (uint32_t)(incl - nh);  // heads before p0
  // serial runs; segments that start and end in the lane are complete
  float run = 0.0f, headpart = 0.0f;
  int cnt = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    if ((hb >> i) & 1u) {
      if (cnt)
        S[before + (uint32_t)cnt - 1u] = run;
      else
        headpart = run;
      ++cnt;
      run = 0.0f;
    }
    run += x[i];
  }
  // join the runs across lanes: U = open run at the end of this lane
  float U = run;
  int F = cnt > 0;
  wave_seg_scan(U, F);
  float in = __shfl_up(U, 1);
  int fin = __shfl_up(F, 1);
  if (lane == 0) {
    in = 0.0f;
    fin = 0;
  }
  const bool open_first = ((heads[j0 >> 6] >> (j0 & 63)) & 1ull) == 0ull;  // tile starts inside a segment
  // the segment that ends just before this lane's first head
  bool pf_here = false;
  float pfv = 0.0f;
  if (cnt) {
    const float v = in + headpart;
    if (fin)
      S[before - 1u] = v;
    else if (open_first) {
      pf_here = true;  // first head of the tile: the segment began in an earlier tile
      pfv = v;
    }
  }
  // the run open at the end of the tile
  const float Ut = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(U), 63));
  const int Ft = __builtin_amdgcn_readlane(F, 63);
  const int ntile = __builtin_amdgcn_readlane(incl, 63);
  const uint32_t qt = tile_h0[w] + (uint32_t)ntile - 1u;  // pair of the tile's last head
  const bool ends_here = j1 >= nlive || (heads[j1 >> 6] & 1ull) != 0ull;
  const unsigned long long pfmask = __ballot(pf_here);
  const float pfv0 =
      pfmask ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pfv), __builtin_ctzll(pfmask))) : 0.0f;
  if (lane == 0) {
    float pv = pfmask ? pfv0 : 0.0f, lv = 0.0f, mv = 0.0f;
    if (ends_here) {
      if (Ft)
        S[qt] = Ut;
      else
        pv = Ut;  // no head in the tile: the whole tile ends an earlier segment
    } else if (Ft) {
      lv = Ut;  // the tile's last segment continues into the next tile
    } else {
      mv = Ut;  // the tile lies inside one segment
    }
    pf_v[w] = pv;
    pl_v[w] = lv;
    mid[w] = mv;
  }
}


// Camera message of each (camera, voxel) pair from its message sum:
// a = clamp(S/C), m = ln a - ln(1-a), B += m - M_c, M_c = m, for C > 0.1f
// (compute_gvdb_message_to_factors, gvdbkernels.cu:408, 457-479).
// S = (sum of the pair's constant front messages) + (its window segment
// sum); window pairs are numbered first.  A window segment inside one tile
// of the segment kernel has its sum in S; one that crosses tiles is joined
// from its parts: the head tile's pl, the tiles inside it (mid), the tail
// tile's pf.

// The update of pair q from its loaded operands: C, the front sum sf, the
// window sum Sw (0 for a front-only pair), the voxel v, its belief Bv and
// the pair's previous message mo.  Every operand is loaded before this test
// (the belief right after the voxel), so that a pair costs two memory round
// trips, not four.
__device__ __forceinline__ void apply_pair(uint32_t q, float C, float sf, float Sw, uint32_t v, float Bv, float mo,
                                           float* __restrict__ B, float* __restrict__ M,
                                           uint8_t* __restrict__ upd, bool mark) {
  if (!(C > kCumLenMin)) return;
  float a = (sf + Sw) / C;
  a = fminf(fmaxf(a, kFEps), 1.0f - kFEps);
  const float m = __logf(a) - __logf(1.0f - a);
  M[q] = m;
  B[v] = (Bv + m) - mo;
  if (mark) upd[v] = 1;
}

// The window pairs [0, nwp), one per thread, and while *all_pairs (the
// first iteration of a call) the front-only pairs [nwp, npairs), strided
// over the grid: a front-only pair's m is the same every iteration, and once
// it is in M the update B = (B + m) - M would add nothing but FP32 rounding.
// The update flags (a voxel's belief has been set by a message) are written
// in that first iteration only: every later iteration updates the same
// voxels.  A camera has one pair per voxel, so no two threads share a B[v].
__global__ __launch_bounds__(256) void k_seg_update(const uint32_t* __restrict__ pair_vox,
                                                    const float* __restrict__ pair_c,
                                                    const float* __restrict__ pair_sf, uint32_t nwp, uint32_t npairs,
                                                    const uint32_t* __restrict__ wseg_off, const float* __restrict__ S,
                                                    const float* __restrict__ pl_v, const float* __restrict__ pf_v,
                                                    const float* __restrict__ mid, float out_scale,
                                                    float* __restrict__ B, float* __restrict__ M,
                                                    uint8_t* __restrict__ upd, const uint32_t* __restrict__ all_pairs) {
  const uint32_t tid = blockIdx.x * blockDim.x + threadIdx.x, stride = gridDim.x * blockDim.x;
  const bool first = *all_pairs != 0u;
  for (uint32_t q = tid; q < nwp; q += stride) {
    const uint32_t o0 = wseg_off[q], o1 = wseg_off[q + 1];
    const float Sq = S[q];  // stale for a segment that crosses tiles: not used then
    const float C = pair_c[q], sf = pair_sf[q], mo = M[q];
    const uint32_t v = pair_vox[q];
    const float Bv = B[v];
    const uint32_t w = o0 / kTile, wt = (o1 - 1u) / kTile;
    float Sw = Sq;
    if (w != wt) {
      float acc = 0.0f;
      for (uint32_t t = w + 1; t < wt; ++t) acc += mid[t];
      Sw = (pl_v[w] + acc) + pf_v[wt];
    }
    apply_pair(q, C, sf, Sw / out_scale, v, Bv, mo, B, M, upd, first);
  }
  if (first)
    for (uint32_t q = nwp + tid; q < npairs; q += stride) {
      const float C = pair_c[q], sf = pair_sf[q], mo = M[q];
      const uint32_t v = pair_vox[q];
      apply_pair(q, C, sf, 0.0f, v, B[v], mo, B, M, upd, true);
    }
}

// Beliefs of an external map (distinct voxels): B = the given log-odds,
// marked as updated so that the marginal reads back.
__global__ void k_set_voxels(const uint32_t* __restrict__ vox, const float* __restrict__ logodds, uint32_t n,
                             float* __restrict__ B, uint8_t* __restrict__ upd) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  B[vox[i]] = logodds[i];
  upd[vox[i]] = 1;
}

// Summed chord length per voxel over one camera's pairs (a camera's pairs
// are distinct voxels, so cameras launched one after another need no atomics).
__global__ void k_cum_add(const uint32_t* __restrict__ pair_vox, const float* __restrict__ pair_c, uint32_t npairs,
                          float* __restrict__ cum) {
  const uint32_t q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < npairs) cum[pair_vox[q]] += pair_c[q];
}

// Voxels that no remaining ray reaches go back to the prior and read 0
// (reset_empty_voxels, gvdbkernels.cu:498-517) ...
__global__ void k_reset_empty(const float* __restrict__ cum, size_t n, float prior_logodds, float* __restrict__ B,
                              uint8_t* __restrict__ upd) {
  const size_t v = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= n || !(cum[v] < 0.05f)) return;
  B[v] = prior_logodds;
  upd[v] = 0;
}

// ... and lose the moved camera's message.
__global__ void k_reset_pair_msgs(const uint32_t* __restrict__ pair_vox, uint32_t npairs, const float* __restrict__ cum,
                                  float* __restrict__ M) {
  const uint32_t q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < npairs && cum[pair_vox[q]] < 0.05f) M[q] = 0.0f;
}

// Camera messages across a re-traversal: old pairs -> voxels -> new pairs.
__global__ void k_scatter_pairs(const uint32_t* __restrict__ pair_vox, const float* __restrict__ M, uint32_t npairs,
                                float* __restrict__ dense) {
  const uint32_t q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < npairs) dense[pair_vox[q]] = M[q];
}

__global__ void k_gather_pairs(const uint32_t* __restrict__ pair_vox, const float* __restrict__ dense, uint32_t npairs,
                               float* __restrict__ M) {
  const uint32_t q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < npairs) M[q] = dense[pair_vox[q]];
}

// marginal occupancy 1 - clamp(1/(1+e^B)) (gvdbkernels.cu:469-476)
__device__ __forceinline__ float marginal(float b) {
  float neg = 1.0f / (1.0f + expf(b));
  neg = fminf(fmaxf(neg, kFEps), 1.0f - kFEps);
  return 1.0f - neg;
}

__global__ void k_marginals(const float* __restrict__ B, float* __restrict__ A, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) A[i] = marginal(B[i]);
}

// max over the block's threads of m (>= 0) into *d_max through the ordered
// bit pattern of non-negative doubles: one atomic per block, none when it
// would not raise the maximum read before it (the atomics of a launch all go
// to one word, and thousands of them take longer than the sweep of a small map)
__device__ __forceinline__ void block_max(double m, unsigned long long* __restrict__ d_max) {
  __shared__ double sh[4];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
  if ((threadIdx.x & 63u) == 0u) sh[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    m = fmax(fmax(sh[0], sh[1]), fmax(sh[2], sh[3]));
    const unsigned long long bits = (unsigned long long)__double_as_longlong(m);
    if (bits > __hip_atomic_load(d_max, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(d_max, bits);
  }
}

// max |marginal(B) - Aprev| as an IEEE double; Aprev is refreshed in the same
// sweep (stored only where it changes: most voxels are saturated and keep
// their bits, so a third of the traffic is left out).  n is a multiple of 4.
__global__ __launch_bounds__(256) void k_residual(const float4* __restrict__ B, float4* __restrict__ A, size_t n4,
                                                   unsigned long long* __restrict__ d_max) {
  double m = 0.0;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += (size_t)gridDim.x * blockDim.x) {
    const float4 b = B[i], p = A[i];
    const float4 a = make_float4(marginal(b.x), marginal(b.y), marginal(b.z), marginal(b.w));
    const double dx = fabs((double)a.x - (double)p.x), dy = fabs((double)a.y - (double)p.y);
    const double dz = fabs((double)a.z - (double)p.z), dw = fabs((double)a.w - (double)p.w);
    const double d = fmax(fmax(dx, dy), fmax(dz, dw));
    if (!(d == 0.0)) A[i] = a;
    m = fmax(m, d);
  }
  block_max(m, d_max);
}

// max |alpha(v) - ref(v)| with alpha the readback marginal (A, or 0 where
// never updated); A holds the marginals of the current beliefs.
__global__ __launch_bounds__(256) void k_ref_error(const float* __restrict__ A, const uint8_t* __restrict__ upd,
                                                   const float* __restrict__ ref, size_t n,
                                                   unsigned long long* __restrict__ d_max) {
  double m = 0.0;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const float a = upd[i] ? A[i] : 0.0f;
    const double dlt = fabs((double)a - (double)ref[i]);
    m = dlt > m ? dlt : m;
  }
  block_max(m, d_max);
}

__global__ void k_alphas(const float* __restrict__ B, const uint8_t* __restrict__ upd, float* __restrict__ out,
                         size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = upd[i] ? marginal(B[i]) : 0.0f;
}

__global__ void k_fill_f32(float* p, float v, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}
// The state that the iterations of a call keep on the GPU, so that they can be
// launched one after the other without the host: flags[0], [1] what
// CamPass::all_pairs and msg_all point at, flags[2] the iterations so far, and
// each iteration's residual in trace (kTraceLen entries, the last ones).
__global__ void k_iter_begin(uint32_t* __restrict__ flags, uint64_t* __restrict__ resid) {
  if (threadIdx.x != 0) return;
  flags[0] = 1u;  // every pair's update
  flags[1] = 2u;  // every pair's log2 n, two iterations
  flags[2] = 0u;
  *resid = 0;
}
__global__ void k_iter_end(uint32_t* __restrict__ flags, uint64_t* __restrict__ resid, uint64_t* __restrict__ trace) {
  if (threadIdx.x != 0) return;
  flags[0] = 0u;  // front-only messages are in M now
  if (flags[1]) flags[1] -= 1u;
  const uint32_t n = flags[2]++;
  trace[n % kTraceLen] = *resid;
  *resid = 0;
}

// window-touched voxels: W[v] = 1 for the voxel of every window pair
__global__ void k_mark_window_voxels(const uint32_t* __restrict__ pair_vox, uint32_t nwp, uint32_t* __restrict__ W) {
  const uint32_t q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < nwp) W[pair_vox[q]] = 1u;
}

__global__ void k_dyn_flags(const uint32_t* __restrict__ pair_vox, uint32_t n, const uint32_t* __restrict__ W,
                            uint32_t* __restrict__ flags) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) flags[k] = W[pair_vox[k]];
}

__global__ void k_dyn_compact(const uint32_t* __restrict__ flags, const uint32_t* __restrict__ pos, uint32_t n,
                              uint32_t q0, uint32_t* __restrict__ dyn) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n && flags[k]) dyn[pos[k]] = q0 + k;
}

__global__ void k_dyn_pairs(const uint32_t* __restrict__ flags, const uint32_t* __restrict__ pos, uint32_t n,
                            uint32_t q0, const uint32_t* __restrict__ pair_vox, uint2* __restrict__ dyn) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n && flags[k]) dyn[pos[k]] = make_uint2(q0 + k, pair_vox[q0 + k]);
}

__global__ void k_fill_u32(uint32_t* p, uint32_t v, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__global__ void k_fill_u8(uint8_t* p, uint8_t v, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}
__global__ void k_zero_u32(uint32_t* p, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

inline unsigned grid_for(size_t n, int threads) { return (unsigned)((n + threads - 1) / threads); }
// slices per XCD of the window kernel's order
inline uint32_t order_rows(uint32_t nslices) { return (nslices + 8 * kOrderGroup - 1) / (8 * kOrderGroup) * kOrderGroup; }
// grid of the per-pair kernels: a thread per window pair, at most 4096
// blocks strided over the front-only pairs
inline unsigned pair_grid(const CamPass& a) {
  return std::max(1u, std::max(grid_for(a.nwp, 256), std::min<unsigned>(grid_for(a.npairs - a.nwp, 256), 4096u)));
}

}  // namespace

template <int MT>
void launch_pair_msgs_t(const CamPass& a, hipStream_t s) {
  typedef typename Msg<MT>::T T;
  hipLaunchKernelGGL(k_pair_msg<MT>, dim3(pair_grid(a)), dim3(256), 0, s, a.pair_vox, a.nwp, a.npairs, a.dyn, a.ndyn,
                     a.B, a.M, (T*)a.apair, a.msg_all);
}

void launch_pair_msgs(const CamPass& a, hipStream_t s) {
  if (a.npairs == 0) return;
  switch (msg_in_type(a.msg_type)) {
    case kMsgF16:
      launch_pair_msgs_t<kMsgF16>(a, s);
      break;
    case kMsgBF16:
      launch_pair_msgs_t<kMsgBF16>(a, s);
      break;
    default:
      launch_pair_msgs_t<kMsgF32>(a, s);
  }
}

template <int MI, int MO, int UF, int UW>
void launch_ray_t(const CamPass& a, hipStream_t s, int part) {
  const typename Msg<MI>::T* Xi = (const typename Msg<MI>::T*)a.apair;
  if (a.nchunks && part != 2)
    hipLaunchKernelGGL((k_front_sums<MI, UF>), dim3(grid_for(a.nchunks, 4)), dim3(256), 0, s,
                       a.fspan, a.chunk_desc, a.nchunks, a.dyn_desc, a.ndyn_chunks, a.inc, Xi, a.partial, a.msg_all,
                       a.fdmask, a.fstatic, a.dfront, a.dcr);
  if (part == 1) return;
  auto* k = a.brick_local ? (a.const_model ? k_ray_window<MI, MO, UW, true, true> : k_ray_window<MI, MO, UW, true, false>)
                          : (a.const_model ? k_ray_window<MI, MO, UW, false, true> : k_ray_window<MI, MO, UW, false, false>);
  hipLaunchKernelGGL(k, dim3(8 * order_rows(a.nslices)), dim3(64), 0, s, a.lanes, a.len_w, a.order, a.chunk_off, a.partial, a.inc, a.base_w,
                     Xi, a.npairs, (typename Msg<MO>::T*)a.Xo, a.sig, a.bia, a.lookup_n, a.front, a.bstart, a.tail);
}

template <int MI, int MO>
void launch_ray_sched(const CamPass& a, hipStream_t s, int part) {
  switch (a.ray_sched) {
    case kSchedF8W8: launch_ray_t<MI, MO, 8, 8>(a, s, part); break;
    case kSchedF16W4: launch_ray_t<MI, MO, 16, 4>(a, s, part); break;
    case kSchedF16W8: launch_ray_t<MI, MO, 16, 8>(a, s, part); break;
    case kSchedF4W4: launch_ray_t<MI, MO, 4, 4>(a, s, part); break;
    case kSchedF16W16: launch_ray_t<MI, MO, 16, 16>(a, s, part); break;
    default: launch_ray_t<MI, MO, 8, 4>(a, s, part);
  }
}

void launch_ray_messages(const CamPass& a, hipStream_t s, int part) {
  if (a.nslices == 0 || a.nwin == 0) return;
  switch (a.msg_type) {
    case kMsgF16: launch_ray_sched<kMsgF16, kMsgF16>(a, s, part); break;
    case kMsgBF16: launch_ray_sched<kMsgBF16, kMsgBF16>(a, s, part); break;
    case kMsgMixedF16: launch_ray_sched<kMsgF32, kMsgF16>(a, s, part); break;
    case kMsgMixedBF16: launch_ray_sched<kMsgF32, kMsgBF16>(a, s, part); break;
    default: launch_ray_sched<kMsgF32, kMsgF32>(a, s, part);
  }
}


void launch_epilogue(const CamPass& a, hipStream_t s, int part) {
  if (a.npairs == 0) return;
  const int mo = msg_out_type(a.msg_type);
  const float out_scale = mo == kMsgF16 ? Msg<kMsgF16>::kOut : (mo == kMsgBF16 ? Msg<kMsgBF16>::kOut : 1.0f);
  if (a.nwin && part != 2) {
    const uint32_t ntiles = (a.nwin + kTile - 1) / kTile;
    // whole groups of blocks for the block remapping
    dim3 grid((grid_for(ntiles, 4) + 8 * kSegGroup - 1) / (8 * kSegGroup) * (8 * kSegGroup)), block(256);
    switch (mo) {
      case kMsgF16:
        hipLaunchKernelGGL(k_seg_sum<kMsgF16>, grid, block, 0, s, a.heads, a.tile_h0, a.nwin, (const __half*)a.Xo,
                           a.win_idx, a.S, a.pf_v, a.pl_v, a.mid);
        break;
      case kMsgBF16:
        hipLaunchKernelGGL(k_seg_sum<kMsgBF16>, grid, block, 0, s, a.heads, a.tile_h0, a.nwin, (const uint16_t*)a.Xo,
                           a.win_idx, a.S, a.pf_v, a.pl_v, a.mid);
        break;
      default:
        hipLaunchKernelGGL(k_seg_sum<kMsgF32>, grid, block, 0, s, a.heads, a.tile_h0, a.nwin, (const float*)a.Xo,
                           a.win_idx, a.S, a.pf_v, a.pl_v, a.mid);
    }
  }
  if (part == 1) return;
  // the segments that cross tiles are joined by k_seg_update
  hipLaunchKernelGGL(k_seg_update, dim3(pair_grid(a)), dim3(256), 0, s, a.pair_vox, a.pair_c, a.pair_sf, a.nwp,
                     a.npairs, a.wseg_off, a.S, a.pl_v, a.pf_v, a.mid, out_scale, a.B, a.M, a.upd, a.all_pairs);
}

void launch_mark_voxels(const FrontRec* front, const RayRec* lanes, uint32_t nslices, const uint32_t* ids,
                        const int32_t* slot, const uint32_t* len_f, const uint32_t* off_w, const uint32_t* len_w,
                        uint8_t* any, uint8_t* wany, uint64_t* bstart, uint8_t* tail, uint32_t* counts,
                        uint64_t* totals, hipStream_t s) {
  auto* c4 = reinterpret_cast<uint4*>(counts);
  if (nslices) {
    auto* k = slot ? k_mark_voxels<true> : k_mark_voxels<false>;
    hipLaunchKernelGGL(k, dim3(nslices), dim3(256), 0, s, front, lanes, ids, slot, len_f, off_w, len_w, any, wany,
                       bstart, tail, c4);
  }
  hipLaunchKernelGGL(k_slice_totals, dim3(1), dim3(1024), 0, s, c4, nslices, totals);
}

void launch_chunk_counts(const uint32_t* len_f, const uint32_t* len_w, uint32_t nslices, uint32_t* cnt, hipStream_t s) {
  hipLaunchKernelGGL(k_chunk_counts, dim3(grid_for(nslices + 1, 256)), dim3(256), 0, s, len_f, len_w, nslices, cnt);
}

void launch_chunk_desc(const uint32_t* chunk_off, const uint32_t* len_f, uint32_t nslices, uint4* desc, hipStream_t s) {
  if (nslices == 0) return;
  hipLaunchKernelGGL(k_chunk_desc, dim3(grid_for(nslices, 256)), dim3(256), 0, s, chunk_off, len_f, nslices, desc);
}
void launch_front_span(const FrontRec* front, const RayRec* lanes, uint32_t n, uint2* span, hipStream_t s) {
  if (n) hipLaunchKernelGGL(k_front_span, dim3(grid_for(n, 256)), dim3(256), 0, s, front, lanes, n, span);
}
uint32_t slice_order_words(uint32_t nslices) { return 8 * order_rows(nslices); }
void launch_slice_order(const uint32_t* len_w, uint32_t nslices, uint32_t* order, hipStream_t s) {
  if (nslices)
    hipLaunchKernelGGL(k_slice_order, dim3(8), dim3(kOrderBins), 0, s, len_w, nslices, order_rows(nslices), order);
}
void launch_gather_desc(const uint4* desc, const uint32_t* idx, uint32_t n, uint4* out, hipStream_t s) {
  if (n) hipLaunchKernelGGL(k_gather_desc, dim3(grid_for(n, 256)), dim3(256), 0, s, desc, idx, n, out);
}

void launch_chunk_static(const CamPass& a, const uint32_t* pflag, uint32_t* dyn_flag, uint32_t* dmask, uint32_t* rows,
                         unsigned long long* nstatic, hipStream_t s) {
  if (a.nchunks == 0) return;
  hipLaunchKernelGGL(k_chunk_static, dim3(grid_for(a.nchunks, 16)), dim3(1024), 0, s, a.fspan, a.chunk_desc, a.nchunks,
                     a.inc, a.nwp, pflag, dyn_flag, dmask, rows, nstatic);
}

void launch_dyn_rows(const uint4* dyn_desc, uint32_t n, const uint32_t* rows, uint32_t* out, hipStream_t s) {
  if (n) hipLaunchKernelGGL(k_dyn_rows, dim3(grid_for(n, 256)), dim3(256), 0, s, dyn_desc, n, rows, out);
}

void launch_fill_dfront(const CamPass& a, const uint32_t* rows, const uint32_t* row_off, uint2* dfront, uint2* dcr,
                        hipStream_t s) {
  if (a.ndyn_chunks == 0) return;
  hipLaunchKernelGGL(k_fill_dfront, dim3(grid_for(a.ndyn_chunks, 4)), dim3(256), 0, s, a.fspan, a.dyn_desc,
                     a.ndyn_chunks, a.inc, a.fdmask, rows, row_off, dfront, dcr);
}

void launch_marginals(const float* B, float* A, size_t n, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_marginals, dim3(grid_for(n, 256)), dim3(256), 0, s, B, A, n);
}

void launch_residual(const float* B, float* A, size_t n, unsigned long long* d_max, hipStream_t s) {
  if (n == 0) return;
  // at most 8 blocks per CU; 2 float4 per thread before a small map gets fewer blocks
  const unsigned g = std::min(grid_for(n / 4, 512), 2048u);
  hipLaunchKernelGGL(k_residual, dim3(g), dim3(256), 0, s, (const float4*)B, (float4*)A, n / 4, d_max);
}

void launch_ref_error(const float* A, const uint8_t* upd, const float* ref, size_t n, unsigned long long* d_max,
                      hipStream_t s) {
  launch_zero_words(d_max, 8, s);
  if (n == 0) return;
  size_t g = grid_for(n, 256);
  if (g > 2048) g = 2048;
  hipLaunchKernelGGL(k_ref_error, dim3(g), dim3(256), 0, s, A, upd, ref, n, d_max);
}

void launch_alphas(const float* B, const uint8_t* upd, float* out, size_t n, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_alphas, dim3(grid_for(n, 256)), dim3(256), 0, s, B, upd, out, n);
}

void launch_set_voxels(const uint32_t* vox, const float* logodds, uint32_t n, float* B, uint8_t* upd, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_set_voxels, dim3(grid_for(n, 256)), dim3(256), 0, s, vox, logodds, n, B, upd);
}

void launch_cum_add(const uint32_t* pair_vox, const float* pair_c, uint32_t npairs, float* cum, hipStream_t s) {
  if (npairs == 0) return;
  hipLaunchKernelGGL(k_cum_add, dim3(grid_for(npairs, 256)), dim3(256), 0, s, pair_vox, pair_c, npairs, cum);
}

void launch_reset_empty(const float* cum, size_t n, float prior_logodds, float* B, uint8_t* upd, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_reset_empty, dim3(grid_for(n, 256)), dim3(256), 0, s, cum, n, prior_logodds, B, upd);
}

void launch_reset_pair_msgs(const uint32_t* pair_vox, uint32_t npairs, const float* cum, float* M, hipStream_t s) {
  if (npairs == 0) return;
  hipLaunchKernelGGL(k_reset_pair_msgs, dim3(grid_for(npairs, 256)), dim3(256), 0, s, pair_vox, npairs, cum, M);
}

void launch_scatter_pairs(const uint32_t* pair_vox, const float* M, uint32_t npairs, float* dense, hipStream_t s) {
  if (npairs == 0) return;
  hipLaunchKernelGGL(k_scatter_pairs, dim3(grid_for(npairs, 256)), dim3(256), 0, s, pair_vox, M, npairs, dense);
}

void launch_gather_pairs(const uint32_t* pair_vox, const float* dense, uint32_t npairs, float* M, hipStream_t s) {
  if (npairs == 0) return;
  hipLaunchKernelGGL(k_gather_pairs, dim3(grid_for(npairs, 256)), dim3(256), 0, s, pair_vox, dense, npairs, M);
}

void launch_fill_f32(float* p, float v, size_t n, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_fill_f32, dim3(grid_for(n, 256)), dim3(256), 0, s, p, v, n);
}

void launch_iter_begin(uint32_t* flags, uint64_t* resid, hipStream_t s) {
  hipLaunchKernelGGL(k_iter_begin, dim3(1), dim3(64), 0, s, flags, resid);
}
void launch_iter_end(uint32_t* flags, uint64_t* resid, uint64_t* trace, hipStream_t s) {
  hipLaunchKernelGGL(k_iter_end, dim3(1), dim3(64), 0, s, flags, resid, trace);
}

void launch_mark_window_voxels(const uint32_t* pair_vox, uint32_t nwp, uint32_t* W, hipStream_t s) {
  if (nwp) hipLaunchKernelGGL(k_mark_window_voxels, dim3(grid_for(nwp, 256)), dim3(256), 0, s, pair_vox, nwp, W);
}

void launch_dyn_flags(const uint32_t* pair_vox, uint32_t n, const uint32_t* W, uint32_t* flags, hipStream_t s) {
  if (n) hipLaunchKernelGGL(k_dyn_flags, dim3(grid_for(n, 256)), dim3(256), 0, s, pair_vox, n, W, flags);
}

void launch_dyn_compact(const uint32_t* flags, const uint32_t* pos, uint32_t n, uint32_t q0, uint32_t* dyn,
                        hipStream_t s) {
  if (n) hipLaunchKernelGGL(k_dyn_compact, dim3(grid_for(n, 256)), dim3(256), 0, s, flags, pos, n, q0, dyn);
}

void launch_dyn_pairs(const uint32_t* flags, const uint32_t* pos, uint32_t n, uint32_t q0, const uint32_t* pair_vox,
                      uint2* dyn, hipStream_t s) {
  if (n) hipLaunchKernelGGL(k_dyn_pairs, dim3(grid_for(n, 256)), dim3(256), 0, s, flags, pos, n, q0, pair_vox, dyn);
}

void launch_fill_u32(uint32_t* p, uint32_t v, size_t n, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(n, 256)), dim3(256), 0, s, p, v, n);
}

void launch_fill_u8(uint8_t* p, uint8_t v, size_t n, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_fill_u8, dim3(grid_for(n, 256)), dim3(256), 0, s, p, v, n);
}

void launch_zero_words(void* p, size_t bytes, hipStream_t s) {
  const size_t n = bytes / 4;
  if (n == 0) return;
  hipLaunchKernelGGL(k_zero_u32, dim3(grid_for(n, 256)), dim3(256), 0, s, (uint32_t*)p, n);
}

}  // namespace mrf
