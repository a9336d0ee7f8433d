// fg_kernels.hip -- gfx950 kernels and C ABI of the raster-scan generalised
// geodesic distance transform (see include/fastgeodis_hip.h).
//
// Semantics (reference FastGeodis v1.0.5):
//   candidate  cur = fl(fl(d_q + fl(l_eucl*LD)) + fl(l_grad*l)),  l = sum_c |I_c(p) - I_c(q)|
//              (fastgeodis_cpu.cpp:88-110, 257-277)
//   update     d(p) = min(d(p), cur) keeping d(p) unless cur is strictly smaller
//   passes     2D: rows then columns (fastgeodis_cpu.cpp:177-198)
//              3D: D, H, W pass pairs with per-pass step tables (fastgeodis_cpu.cpp:220-231, 359-404)
//
// Layout in HBM.  Every sweep runs along a non-contiguous axis A with lanes on
// the contiguous axis E and wave rows on the remaining axis B:
//   D pass: A=D, B=H, E=W on the native (D,H,W) array
//   H pass: A=H, B=D, E=W on the native array
//   W pass: A=W, B=H, E=D on a transposed (W,H,D) copy (image transposed once
//           per call; the distance enters that layout through the H pass's
//           backward sweep, which writes it directly, and leaves it through
//           the W pass's backward sweep, which writes the native layout; a
//           transpose instead where those forms do not apply (3-4 channels, 2
//           channels on the automatic shapes, other shapes, the W pass at
//           K > 5) and after a signed or GSF transform's last W pass, where it
//           applies the epilogue)
//   2D: rows A=H, E=W on (H,W); columns A=W, E=H on (W,H), the backward row
//       and column sweeps writing the other layout (through transposes in
//       launches of many row tiles, kRowWaveTiles)
// B and E are the reference's in-plane axes in its neighbour order (B outer,
// E inner), so the exact-order path visits candidates in the reference order.
//
// Engines.
//   tiled (default): one persistent kernel per sweep (all workgroups resident).
//     A workgroup owns a tile of the slice plane and walks along A.  Its
//     front (the previous slice) lives in VGPRs: lane = E position, register
//     = B row; E neighbours arrive through DPP wave shifts folded into the
//     arithmetic, B neighbours are other registers or, across waves, LDS.
//     The window is the tile grown by K on every tiled side; every K slices a
//     tile publishes its own values as (value, tag) pairs with device-scope
//     relaxed 64-bit stores and reloads its K-wide halo from its neighbours'
//     publications, spinning on the tag (bounded; expiry sets a status word).
//     Between exchanges the halo is recomputed redundantly: values at window
//     positions more than j slices from the window edge are exact at step j,
//     so the tile's own positions are exact for all K steps.  3D planes run
//     sweep_tiled_kernel; one-row planes (2D) row_sweep_kernel, the same tiling
//     with the front in one wave and the loads, image terms and stores in
//     others; a call on small 2D images small_call_kernel, one workgroup and
//     one launch per transform.
//   per-slice: one small launch per slice (any channel count); kept as the
//     fallback and as an independent second path for tests.
//
// Arithmetic.  Compiled with -ffp-contract=off (no FMA) and without fast-math.
// With l_grad and every l_eucl*LD non-negative (sign bit clear), no candidate
// can be -0, so min over candidates with IEEE minNum (v_min3_f32, NaN
// candidates ignored) followed by "(m < d) ? m : d" equals the reference's
// sequential std::min fold bit for bit; otherwise the exact path folds the
// candidates one by one in the reference order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <thread>
#include <type_traits>
#include <vector>

#include "fastgeodis_hip.h"

namespace {

constexpr float kInf = __builtin_huge_valf();
// Deepest halo: 2D rows use up to 30 lanes on each side of a 64-lane window (a
// lone image leaves most CUs idle); 3D windows of 32 rows stop at 15 by
// themselves.
constexpr int kMaxK = 30;
// s_sleep units (64 clocks each) between publishing a halo and first polling
// the neighbours' publications, and between polls.  A poll that comes too
// early costs a second round trip behind everything the CU has in flight, and
// polls slow the publications down.  32-row windows, 512^2 planes (K = 5, the
// memory system busy): a sweep took 615, 584, 577 and 582 us with 20, 28, 36
// and 44 units, and 563 us with 36 and 8 between polls.  At K = 10 (256^2
// planes, most CUs idle) 90.7, 89.4, 89.8 and 92.1 us with 16, 20, 28 and 36.
constexpr int kHaloPollDelay = 36, kHaloRepollDelay = 8;
constexpr int kHaloPollDelayDeep = 24;
// 16-row windows (256^2 planes, K = 5): 87.0, 84.1, 88.8 and 94.3 us with 16,
// 20, 28 and 36 units, 88.9 us with 20 and 8 between polls.
constexpr int kHaloPollDelay16 = 20, kHaloRepollDelay16 = 1;
// The same for row tiles: 512 clocks (256 and 64 measured 7 and 11 % slower
// sweeps of 512^2: more polls in the way of the publications).
constexpr int kRowPollDelay = 8;
// Multi-wave tiles skip the slab loads of window rows whose values at that
// step are not exact (see load_rows).
constexpr bool kSkipEdgeLoads = true;
// Waves that perform the halo exchanges in kernels with exchange waves.
constexpr int kCommWaves = 4;
// A-contiguous output (the W pass writing the native layout): slices staged
// per run (16 x 4 B = one 64-byte segment per position; measured in the
// sweep's streaming pattern: runs of 16 cost ~10 % more than plain row
// stores, runs of 8 ~50 %) and the padding between run slots in LDS (words).
constexpr int kRunLen = 16;
constexpr int kRunPad = 4;
// A completed run is stored at the next halo exchange, so the LDS ring also
// holds the slices staged until then (K - 1 at most, the host using this
// form with K == 5).
constexpr int kRunSlots = kRunLen + 4;
// Buckets of the exchange-wait histogram: bucket b counts waits of
// [2^(b-1), 2^b) ticks of the constant-rate device clock (bucket 0: 0 ticks).
constexpr int kXHistBuckets = 32;

// ---------------------------------------------------------------------------
// Descriptors
// ---------------------------------------------------------------------------

struct SweepDesc {
  const float *img;  // image channel 0 in this sweep's layout
  float *d;          // distance in this sweep's layout
  long long cs;      // image channel stride (elements)
  long long sA, sB;  // slice stride and row stride; lanes are contiguous
  int nA, nB, nE;
  int dir;  // +1 forward, -1 backward
  int C;
  float lg;
  float e1[9];  // fl(l_eucl * LD[i*3+j]), i = row offset + 1, j = lane offset + 1
  int nTB, nTE;  // tile grid
  int TB, TE;    // own tile extent
  int tile0;     // first tile of this descriptor within its launch
  long long halo0;  // first halo entry of this descriptor
  float *dxo;       // other-layout output: element (a, b, e) at
  long long sXe, sXa;  //   dxo[e * sXe + a * sXa + b] (XST, b contiguous)
  long long sXb;       //   dxo[e * sXe + b * sXb + a] (XSA, a contiguous)
  // First sweep of a transform: the input distance is the initialisation,
  // computed from the mask as it is loaded (init_mode 1: fl(v*m), 2:
  // fl(v*fl(1-m))), and the sweep's untouched first slice is written too.
  const float *init_src;  // mask channel 0 in this sweep's layout (init_mode != 0)
  float init_v;
  int init_mode;
};

// Transposes, optionally combining several sources elementwise (the epilogues
// of signed and GSF transforms, applied while their distances leave the W
// pass layout).
enum XposeKind : int {
  XK_COPY = 0,       // dst = src
  XK_SIGNED = 1,     // dst = src - src2                      (D(M) - D(1-M))
  XK_GSF_MID = 2,    // ds = src - src2; dst..dst4 = the inits of the four second-stage transforms
  XK_GSF_FINAL = 3,  // dst = -(src2 - src3) + (src4 - src)
};

struct XposeDesc {  // out[c][w][h][d] = in[c][d][h][w]
  const float *src;
  float *dst;
  int C, D, H, W;
  int tiles_dw;  // tiles per (c, h) plane
  int tile0;
  int kind;                          // XposeKind (C == 1 unless XK_COPY)
  const float *src2, *src3, *src4;   // further sources, same layout as src
  float *dst2, *dst3, *dst4;         // further outputs (XK_GSF_MID), same layout as dst
  float v, theta;
};

// ---------------------------------------------------------------------------
// Device helpers
// ---------------------------------------------------------------------------

// Lane l receives lane l-1 (J == 0) or lane l+1 (J == 2).  The wave's edge
// lane receives 0 (wave shift) or the opposite edge lane's value (ALT: wave
// rotate); that lane is always a halo lane, whose value stays outside the
// part of the window that is exact, or a pad lane, forced to +inf each step,
// so both forms give the same results.  A shift that several candidates use
// is computed once by the compiler and cannot fold into its users; shifting
// one front row for two new rows with the two different forms keeps each
// shift single-use, so it folds into the VALU instruction that consumes it
// (v_add_f32_dpp / v_sub_f32_dpp).  TAG keeps other call sites distinct.
template <int J, int TAG, bool ALT = false>
__device__ __forceinline__ float shiftE(float x) {
  if constexpr (J == 1) return x;
  else {
    constexpr int ctrl = (J == 0 ? 0x138 : 0x130) | (ALT ? 0x4 : 0x0);  // wave_shr/ror:1, wave_shl/rol:1
    return __int_as_float(__builtin_amdgcn_update_dpp(TAG, __float_as_int(x), ctrl, 0xF, 0xF, true));
  }
}

// Workgroups are dispatched round-robin over the 8 XCDs; give each XCD a
// contiguous range of tiles so that most neighbours share an L2.
__device__ __forceinline__ int xcd_remap(int g, int G) {
  constexpr int nx = 8;
  const int x = g % nx, i = g / nx;
  const int q = G / nx, rem = G % nx;
  return x * q + min(x, rem) + i;
}

__device__ __forceinline__ unsigned long long pack(float v, unsigned tag) {
  return ((unsigned long long)tag << 32) | (unsigned long long)__float_as_uint(v);
}

// sum over channels C0..CT-1 of |I_c(p) - I_c(q)|, accumulated left to right
template <int I, int J, int C0, int CT>
__device__ __forceinline__ float absdiff_sum(float acc, const float (&Iq)[CT], const float (&In)[CT]) {
  if constexpr (C0 >= CT) {
    return acc;
  } else {
    const float q = shiftE<J, 1 + C0 + I * 16 + J * 4, (I & 1) != 0>(Iq[C0]);
    return absdiff_sum<I, J, C0 + 1, CT>(acc + fabsf(q - In[C0]), Iq, In);
  }
}

// Candidate for the element at this lane from front row I (B offset I-1) and
// lane offset J-1:  (d_q + e1) + l_grad * sum_c |I_c(p) - I_c(q)|.  The
// channel sum starts from |I_0(p) - I_0(q)|, which equals the reference's
// 0.0f + |..| bit for bit.
template <int I, int J, int CT, bool LAMB1>
__device__ __forceinline__ float candidate(float dq, const float (&Iq)[CT], const float (&In)[CT], float e1,
                                           float lg) {
  // |q - p| == |p - q| exactly; the shifted operand goes first so that the
  // shift folds into v_sub_f32_dpp without commuting
  const float l =
      absdiff_sum<I, J, 1, CT>(fabsf(shiftE<J, 1 + I * 16 + J * 4, (I & 1) != 0>(Iq[0]) - In[0]), Iq, In);
  if constexpr (LAMB1) {
    // l_grad == 1 and l_eucl*LD == +0: fl(1*l) == l and dropping "+ 0" is exact here
    return shiftE<J, 64 + I * 4 + J, (I & 1) != 0>(dq) + l;
  } else {
    // the step is added before the shift, so that the candidates of several
    // new elements share the sums of a front element: with the table's equal
    // entries (step_of) 12 additions per two rows instead of 18
    return shiftE<J, 64 + I * 4 + J, (I & 1) != 0>(dq + e1) + lg * l;
  }
}

// The table entry of a candidate: steps to opposite neighbours have the same
// length (and bits), so each is taken from the first of its kind.
template <int I, int J>
__device__ __forceinline__ float step_of(const float (&e1)[9]) {
  return e1[(I == 2 ? 0 : I) * 3 + (J == 2 ? 0 : J)];
}

// The three candidates from front row I (its distance dq and image Iq).
template <int I, int CT, bool LAMB1>
__device__ __forceinline__ void candidates_row(float (&c)[3], float dq, const float (&Iq)[CT],
                                               const float (&In)[CT], const float (&e1)[9], float lg) {
  c[0] = candidate<I, 0, CT, LAMB1>(dq, Iq, In, step_of<I, 0>(e1), lg);
  c[1] = candidate<I, 1, CT, LAMB1>(dq, Iq, In, step_of<I, 1>(e1), lg);
  c[2] = candidate<I, 2, CT, LAMB1>(dq, Iq, In, step_of<I, 2>(e1), lg);
}

// v_min3_f32 of quiet operands (results of arithmetic).  Where one comes from
// another basic block, the compiler would quiet it first and fall back to
// two-operand minima: six more instructions per two rows behind the barrier.
__device__ __forceinline__ float min3(float a, float b, float c) {
  float r;
  asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// The nine candidates of one row element, taken in triples of a front row as
// they become available.
// FAST: folded with IEEE minNum as they come (any order gives the same value,
// as no candidate is -0); otherwise kept for the reference's order, and folded
// in it as far as they are there (`early`).
template <bool FAST>
struct Fold {
  float c[9];   // !FAST: candidate of front row i, lane offset j at i * 3 + j
  float nd;     // !FAST: the old value and the first candidates folded
  float m;      // FAST: minimum so far
  float left;   // FAST: a candidate that waits for the next pair
  int n = 0;    // triples taken
  __device__ __forceinline__ void take(int i, const float (&t)[3]) {
    if constexpr (FAST) {
      if (n == 0) {
        m = fminf(fminf(t[0], t[1]), t[2]);
      } else if (n == 1) {
        m = fminf(fminf(m, t[0]), t[1]);
        left = t[2];
      } else {
        m = min3(min3(m, left, t[0]), t[1], t[2]);
      }
      ++n;
    } else {
      for (int j = 0; j < 3; ++j) c[i * 3 + j] = t[j];
    }
  }
  // !FAST: folds the first k candidates (all taken by then)
  __device__ __forceinline__ void early(float dinit, int k) {
    nd = dinit;
#pragma unroll
    for (int q = 0; q < 9; ++q)
      if (q < k) nd = (c[q] < nd) ? c[q] : nd;
  }
  // the new value; k: candidates that `early` folded (0: it was not called)
  __device__ __forceinline__ float with(float dinit, int k) const {
    if constexpr (FAST) return (m < dinit) ? m : dinit;
    float v = k ? nd : dinit;
#pragma unroll
    for (int q = 0; q < 9; ++q)
      if (q >= k) v = (c[q] < v) ? c[q] : v;
    return v;
  }
};

// ---------------------------------------------------------------------------
// Tiled persistent sweep kernel
// ---------------------------------------------------------------------------

// Global-address-space view of the halo publications (64-bit atomics use
// SGPR base + VGPR offset addressing instead of flat addressing).
typedef __attribute__((address_space(1))) unsigned long long gu64;

// Publications as buffer operations at device scope (sc1) on the descriptor's
// part of the exchange buffer, one aligned 64-bit (value, tag) entry per lane,
// written and read whole.  A lane that publishes or needs nothing gets kNoHalo
// as its byte offset: its store is dropped, its load returns 0 without a
// memory access.  So neither needs a branch, and the loads of all rows are in
// flight together (under branches the compiler waited for each row's load
// before it issued the next one).  The offsets fit 32 bits: the tiles of a
// launch are resident together, and each has two slots of less than 64 KB.
// They are plain stores and loads, not atomics: what the exchange rests on is
// that the aligned 8 bytes that one lane's instruction writes become visible
// whole, so a reader that sees the tag has the value.  Nothing else is ordered
// by an entry, so there is no release or acquire.
constexpr unsigned kNoHalo = 0xFFFFFFFFu;
constexpr int kHaloCache = 16;  // sc1
typedef unsigned uint2v __attribute__((ext_vector_type(2)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t halo_rsrc(unsigned long long *base) {
  return __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, 0xFFFFFFF0u, 0x00020000);
}
__device__ __forceinline__ void halo_publish(__amdgpu_buffer_rsrc_t h, unsigned ofs, float v, unsigned tag) {
  __builtin_amdgcn_raw_buffer_store_b64(uint2v{__float_as_uint(v), tag}, h, (int)ofs, 0, kHaloCache);
}
__device__ __forceinline__ uint2v halo_read(__amdgpu_buffer_rsrc_t h, unsigned ofs) {
  asm volatile("" ::: "memory");  // every poll reads again
  return __builtin_amdgcn_raw_buffer_load_b64(h, (int)ofs, 0, kHaloCache);
}

// Waits until the entries at ofs[0..N-1] carry `tag` (x holds a first read of
// them); false after spin_limit more reads.
template <int N, int REPOLL>
__device__ __forceinline__ bool halo_wait(__amdgpu_buffer_rsrc_t h, const unsigned (&ofs)[N], uint2v (&x)[N],
                                          unsigned tag, int spin_limit) {
  for (int spins = 0;; ++spins) {
    bool late[N], waiting = false;
#pragma unroll
    for (int k = 0; k < N; ++k) {
      late[k] = ofs[k] != kNoHalo && x[k].y != tag;
      waiting = waiting || late[k];
    }
    if (__ballot(waiting) == 0) return true;
    if (spins >= spin_limit) return false;
    __builtin_amdgcn_s_sleep(REPOLL);
    uint2v y[N];
#pragma unroll
    for (int k = 0; k < N; ++k) y[k] = halo_read(h, late[k] ? ofs[k] : kNoHalo);
#pragma unroll
    for (int k = 0; k < N; ++k) x[k] = late[k] ? y[k] : x[k];
  }
}

template <int R, int CT>
struct Slab {  // one prefetched slice: image rows -1..R, distance rows 0..R-1
  float I[CT][R + 2];
  float d[R];
};

// NW waves per workgroup, R window rows per wave (register rows), P slices
// prefetched ahead, CT image channels.
// A sweep is a chain of steps and exchanges, and both bound it.  A step: the
// vector issue of its candidates (4 waves a SIMD, 1.05 ns per add and 1.75 per
// minimum or lane shift of a wave), then the edge rows through LDS and one
// barrier; so the candidates of a wave's own front rows are evaluated between
// its LDS writes and the barrier, waves compute only the steps that still reach
// own rows, new elements share the sums of a front element and take minima of
// three.  An exchange (every K steps): two rows' publications and polls in
// flight together, nothing else of the wave's before them in the queue.
// Whole calls before / after these: 512^3 lamb 1 iter 4 15.68 / 13.98 ms,
// 128 x 256 x 256 lamb 0.5 4.52 / 3.51 ms (with 16-row windows), 20 x 120 x 140
// 1.63 / 1.33 ms.  512^2 planes, K = 5: 439 of the 634 us of a sweep remained
// without exchanges, 271 without exchanges, loads and stores.
// XS, the output form: 0 writes slice a in the sweep's own layout.
//   1 (XST): writes it to Dd.dxo with B contiguous (the H pass writes the
//     (W, H, D) layout of the W pass), staging each slice's window through
//     LDS so each store covers a run of consecutive B.
//   2 (XSA): writes it to Dd.dxo with A contiguous (the W pass writing the
//     native (D, H, W) layout): each wave stages kRunLen consecutive slices
//     in LDS so that each store covers runs of kRunLen consecutive A.
// INIT: the first sweep of a transform, whose input distance is computed from
// the mask as it is loaded (SweepDesc::init_mode).
// COMM: kCommWaves more waves (indices NW, NW + 1, ...) that hold no rows and
// perform every halo exchange of the tile, each for its share of the window
// rows: the compute waves leave their front in LDS and wait at a barrier while
// they publish and poll, so the compute waves' prefetch loads stay in flight
// (a wave's wait for a halo load is also a wait for every load it issued
// earlier).
template <int NW, int R, int P, int CT, bool LAMB1, bool FAST, int XS = 0, bool INIT = false,
          bool COMM = false>
__global__ __launch_bounds__((NW + (COMM ? kCommWaves : 0)) * 64) void sweep_tiled_kernel(
    const SweepDesc *__restrict__ descs, int ndesc, SweepDesc one, int K, unsigned tag_base,
    unsigned long long *__restrict__ halo_base, int *__restrict__ status, int spin_limit,
    unsigned *__restrict__ xhist) {
  constexpr bool XST = XS == 1, XSA = XS == 2;
  static_assert(NW > 1, "one-row planes run on row_sweep_kernel");
  // LDS slots of the edge rows (and of a B-contiguous window): a slot's reads
  // and its next rewrite must be at least two steps apart (one barrier per
  // step), so ring positions alternate between two slots and the last
  // position of an odd ring has a third.  XSA needs the LDS for its runs: two
  // slots, alternating by step parity.
  constexpr int ES = (XSA || P % 2 == 0) ? 2 : 3;
  auto edge_slot = [](int position) constexpr { return (P % 2 == 1 && position == P - 1) ? 2 : position % 2; };
  __shared__ float edge_first[ES][NW][64];
  __shared__ float edge_last[ES][NW][64];
  __shared__ float edgeI_first[ES][NW][CT][64];
  __shared__ float edgeI_last[ES][NW][CT][64];
  constexpr int NWR = NW * R;  // window rows
  static_assert(!XST || (NW > 1 && 64 % NWR == 0), "transposed output needs a multi-wave window of 16/32/64 rows");
  static_assert(!XSA || (NW > 1 && !COMM && !INIT && NWR > 2 * P), "A-contiguous output is a plain-sweep form");
  __shared__ float xtile[XST ? ES : 1][XST ? NWR : 1][65];
  // XSA: slot a % kRunSlots holds slice a, one 64-lane row per own row of
  // the tile (window rows K .. K + TB - 1; the host uses this form only on
  // planes of several tiles along B, where TB <= NWR - 2K); the slots are
  // kRunPad words apart beyond their rows, so the 16 lanes that read one
  // position's run hit different banks
  constexpr int XOR = NWR - 2 * P;  // own rows at the shallowest halo (+ 1 spare row)
  __shared__ float xrun[XSA ? kRunSlots : 1][XSA ? (XOR + 1) * 64 + kRunPad : 1];
  __shared__ unsigned xhist_wg[kXHistBuckets];  // this workgroup's exchange-wait counts (measurement)
  static_assert(!COMM || (NW > 1 && NWR % kCommWaves == 0), "exchange waves serve multi-wave sweeps");
  __shared__ float xfront[COMM ? NWR : 1][64];     // COMM: the front around an exchange

  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave index: uniform
  const int tile = xcd_remap(blockIdx.x, gridDim.x);
  if (xhist) {
    if (threadIdx.x < kXHistBuckets) xhist_wg[threadIdx.x] = 0u;
    __syncthreads();
  }

  // descriptor owning this tile: the launch's only one (passed by value when
  // descs is null) or a binary search on tile0 (uniform branches and loads,
  // so the copy's fields stay in scalar registers)
  SweepDesc Dd;
  if (descs) {
    int lo = 0, hi = ndesc - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (descs[mid].tile0 <= tile) lo = mid; else hi = mid - 1;
    }
    Dd = descs[lo];
  } else {
    Dd = one;
  }
  unsigned long long *const halo = halo_base + Dd.halo0;
  const long long cs = Dd.cs, sA = Dd.sA, sB = Dd.sB;
  const int nA = Dd.nA, nB = Dd.nB, nE = Dd.nE, dir = Dd.dir;
  const float lg = Dd.lg;
  float e1[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) e1[k] = Dd.e1[k];
  const int nTB = Dd.nTB, nTE = Dd.nTE, TB = Dd.TB, TE = Dd.TE;
  const int lt = tile - Dd.tile0;
  const int tb = lt / nTE, te = lt - tb * nTE;
  const int b_own0 = tb * TB, b_own1 = min(nB, b_own0 + TB);
  const int e_own0 = te * TE, e_own1 = min(nE, e_own0 + TE);
  const int bw0 = (nTB > 1) ? b_own0 - K : 0;
  const int ew0 = (nTE > 1) ? e_own0 - K : -1;
  const int e = ew0 + lane;
  const bool lane_valid = (e >= 0) && (e < nE);
  const unsigned ec = (unsigned)min(max(e, 0), nE - 1);  // clamped: loads never leave the row
  const unsigned ecb = ec * 4u;                             // its byte offset within a row
  const bool lane_own = (e >= e_own0) && (e < e_own1);
  // Byte offsets (within a parity's slots) of the entry that window row b
  // publishes, or kNoHalo: own positions within K of a tile edge that has a
  // neighbour; and of the entry that it reloads, or kNoHalo: non-own
  // positions within K of the own region (the only ones whose values reach
  // own positions in K steps), published by the tile that owns them, which
  // lies across that edge.
  const int tile_slots = TB * TE;
  const int ote = lane_valid ? (e / TE) : 0;
  const int ow = min(nE, ote * TE + TE) - ote * TE;
  const int lane_dist = max(max(e_own0 - e, e - (e_own1 - 1)), 0);
  const bool lane_band = (te > 0 && e - e_own0 < K) || (te < nTE - 1 && e_own1 - 1 - e < K);
  auto publish_ofs = [&](int b) -> unsigned {
    const bool row_band = (tb > 0 && b - b_own0 < K) || (tb < nTB - 1 && b_own1 - 1 - b < K);
    if (!(b >= b_own0 && b < b_own1 && lane_own && (row_band || lane_band))) return kNoHalo;
    return (unsigned)(lt * 2 * tile_slots + (b - b_own0) * (e_own1 - e_own0) + (e - e_own0)) * 8u;
  };
  auto reload_ofs = [&](int b) -> unsigned {
    const bool own = b >= b_own0 && b < b_own1 && lane_own;
    const int row_dist = max(max(b_own0 - b, b - (b_own1 - 1)), 0);
    if (b < 0 || b >= nB || !lane_valid || own || max(row_dist, lane_dist) > K) return kNoHalo;
    const int otb = b / TB;
    return (unsigned)((otb * nTE + ote) * 2 * tile_slots + (b - otb * TB) * ow + (e - ote * TE)) * 8u;
  };

  // The block loop below advances in groups of P steps and exchanges halos
  // every K steps; it stays within the sweep only when K is a positive
  // multiple of P.  A launch that breaks this is refused before any store,
  // and so is an A-contiguous output whose own rows or staged slices would
  // not fit its LDS ring.
  if (K <= 0 || K % P != 0 || (XSA && (Dd.nTB < 2 || Dd.TB > XOR || K > kRunSlots - kRunLen + 1))) {
    if (threadIdx.x == 0) __hip_atomic_store(status, FG_EINVAL, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    return;
  }
  const int nsteps = nA - 1;
  if (nsteps <= 0) return;
  const int a_first = (dir > 0) ? 1 : nA - 2;
  const int nblocks_all = (nsteps + K - 1) / K;

  // Last wave with rows in the plane; later ones leave now (their rows are
  // never read: wave w_last takes its lower neighbour row as outside), unless
  // they still move staged windows or exchange halos.
  const int w_last = min(NW - 1, (nB - 1 - bw0) / R);
  if constexpr (!XST && !COMM)
    if (w > w_last) return;

  // The exchange wave: the same barrier sequence as the compute waves (one
  // per step, two per exchange), publishing and polling between the two
  // barriers of each exchange for every row of the window.
  if constexpr (COMM) {
    if (w >= NW) {
      constexpr int CR = NWR / kCommWaves;  // window rows per exchange wave
      const int cr0 = (w - NW) * CR;
      unsigned pub[CR], src[CR];
#pragma unroll
      for (int k = 0; k < CR; ++k) {
        pub[k] = publish_ofs(bw0 + cr0 + k);
        src[k] = reload_ofs(bw0 + cr0 + k);
      }
      bool tripped = false;
      for (int blk = 0;; ++blk) {
        for (int st = 0; st < K; ++st) __syncthreads();
        if (blk + 1 >= nblocks_all) break;
        __syncthreads();  // the compute waves' front is in xfront
        const unsigned long long t_in = xhist ? wall_clock64() : 0ull;
        const unsigned tag = tag_base + (unsigned)(blk + 1);
        const __amdgpu_buffer_rsrc_t h = halo_rsrc(halo + ((blk + 1) & 1) * tile_slots);
#pragma unroll
        for (int k = 0; k < CR; ++k) halo_publish(h, pub[k], xfront[cr0 + k][lane], tag);
        __builtin_amdgcn_s_sleep(kHaloPollDelay);
        uint2v x[CR];
#pragma unroll
        for (int k = 0; k < CR; ++k) x[k] = halo_read(h, src[k]);
        if (!halo_wait<CR, kHaloRepollDelay>(h, src, x, tag, tripped ? 0 : spin_limit)) {
          __hip_atomic_store(status, FG_EWATCHDOG, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
          tripped = true;
        }
#pragma unroll
        for (int k = 0; k < CR; ++k)
          if (src[k] != kNoHalo) xfront[cr0 + k][lane] = __uint_as_float(x[k].x);
        if (xhist && lane == 0) {
          const unsigned long long dt = wall_clock64() - t_in;
          const int bucket = dt ? min(64 - __clzll(dt), kXHistBuckets - 1) : 0;
          atomicAdd(&xhist_wg[bucket], 1u);
        }
        __syncthreads();  // the halo is in xfront
      }
      if constexpr (XST) __syncthreads();  // the last staged slice
      if (xhist) __syncthreads();           // the workgroup's histogram flush
      return;
    }
  }

  // Row bookkeeping: rows -1..R relative to this wave.  rofs[r] is the byte
  // offset of this lane's element of row r (clamped into the plane) within
  // a slice; the host runs this kernel only on arrays of less than 4 GiB per
  // channel, so every offset in a slice fits 32 bits and all loads and
  // stores use a per-slice buffer resource plus this loop-invariant offset.
  int rb[R + 2];
  bool rvalid[R + 2];
  unsigned rofs[R + 2];
#pragma unroll
  for (int r = 0; r < R + 2; ++r) {
    rb[r] = bw0 + w * R + r - 1;
    rvalid[r] = rb[r] >= 0 && rb[r] < nB;
    rofs[r] = (unsigned)((long long)min(max(rb[r], 0), nB - 1) * sB * 4) + ecb;
  }
  // Buffer resources are raw and byte-addressed; offsets at or beyond the
  // range are out of bounds, and stores there are dropped.
  // Slice cursor of a step: its slice a and that slice's byte offset
  // a * sA * 4, advanced together by one slice per step (two scalar adds
  // instead of a 64-bit multiply per array).  A slice outside [0, nA) (the
  // prefetches and stores of steps past the end of the sweep) gets an empty
  // buffer range: its loads return 0 and its stores are dropped, without a
  // memory access.
  struct Cursor {
    int a;
    long long off;
  };
  const long long dAb = (long long)dir * sA * 4;
  auto cursor_of = [&](int step) {
    const int a = a_first + step * dir;
    return Cursor{a, (long long)a * sA * 4};
  };
  auto advance = [&](Cursor &c) {
    c.a += dir;
    c.off += dAb;
  };
  auto cursor_rsrc = [&](const float *base, const Cursor &c) {
    const bool in = (unsigned)c.a < (unsigned)nA;
    return __builtin_amdgcn_make_buffer_rsrc((void *)((const char *)base + c.off), 0, in ? 0xFFFFFFF0u : 0u,
                                             0x00020000);
  };
  // the out-of-range offset of a lane that stores nothing
  constexpr unsigned kNowhere = 0xFFFFFFFFu;

  // Transposed output: wave w moves window columns (w * R + k) * (64 / NWR)
  // + lane / NWR, rows lane % NWR, for k < R; the byte offset of each element
  // in its output slice (out-of-range for positions this tile does not own).
  unsigned xoff[XST ? R : 1];
  if constexpr (XST) {
#pragma unroll
    for (int k = 0; k < R; ++k) {
      const int col = (w * R + k) * (64 / NWR) + lane / NWR, row = lane % NWR;
      const int eg = ew0 + col, bg = bw0 + row;
      const bool own = eg >= e_own0 && eg < e_own1 && bg >= b_own0 && bg < b_own1;
      xoff[k] = own ? (unsigned)(((long long)eg * Dd.sXe + bg) * 4) : 0xFFFFFFFFu;
    }
  }
  // stores the staged window of step sp (LDS slot ps) to the output; step -1
  // is the sweep's first slice, which the sweep itself never changes but the
  // output array must also hold
  auto xflush = [&](int ps, int sp) {
    if constexpr (XST) {
      const bool live = sp >= -1 && sp < nsteps;
      const int ap = min(max(a_first + sp * dir, 0), nA - 1);
      const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
          (void *)(Dd.dxo + (long long)ap * Dd.sXa), 0, live ? 0xFFFFFFF0u : 0u, 0x00020000);
#pragma unroll
      for (int k = 0; k < R; ++k) {
        const int col = (w * R + k) * (64 / NWR) + lane / NWR, row = lane % NWR;
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(xtile[ps][row][col]), rx, (int)xoff[k], 0, 0);
      }
    }
  };

  // Prefetch loads are raw loads at clamped coordinates (always in bounds) and
  // carry no masking, so no instruction waits on them until the slab is
  // consumed.  Values at pad positions (outside the plane) are never used:
  // a pad's own result is forced to +inf after every step, and its image
  // value only enters candidates whose distance operand is that +inf.
  // With several waves, image rows -1 and R of a slab are the neighbour
  // waves' rows R-1 and 0: they arrive through LDS when the slab is consumed
  // (see step), so only rows 0..R-1 are loaded.  The initial front loads all
  // rows.
  // the initialisation from the loaded mask value: fl(v*m) (mode 1) or
  // fl(v*fl(1-m)) (mode 2), by a select rather than a branch
  const bool init_inv = Dd.init_mode == 2;
  const float init_v = Dd.init_v;
  auto init_of = [&](float m) -> float {
    if constexpr (INIT) {
      const float t = 1.0f - m;
      return init_v * (init_inv ? t : m);
    } else {
      return m;
    }
  };
  // Slab offsets per ring slot.  With K == P a block is one turn of the ring
  // and slot t always holds block step t + 1.  At block step j the window
  // rows less than j rows from a window edge that faces a neighbour tile
  // depend on positions outside the window: their values are not exact and
  // are never stored or published (the next exchange replaces them), so
  // their loads get an out-of-range offset (the load returns 0 without a
  // memory access).  The image rows of a block's last step (slot P - 1) are
  // all loaded: after the exchange they are the front image of the next
  // block's first step, whose rows are all exact again.  Computed once, so
  // the steps pay nothing for it; with K > P every row is loaded.
  constexpr int SK = kSkipEdgeLoads ? P : 1;
  unsigned slot_ofs[SK][R];
#pragma unroll
  for (int t = 0; t < SK; ++t)
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int wr = w * R + r;  // window row (uniform)
      const bool skip = SK > 1 && K == P && nTB > 1 && min(wr, NWR - 1 - wr) <= t;
      slot_ofs[t][r] = skip ? 0xFFFFFFFFu : rofs[r + 1];
    }
  // t: the ring slot the slab fills, or -1 (every row loaded)
  auto load_rows = [&](Slab<R, CT> &S, const Cursor &cur, int r0, int r1, int t) {
    const __amdgpu_buffer_rsrc_t rd = cursor_rsrc(INIT ? Dd.init_src : Dd.d, cur);
    __amdgpu_buffer_rsrc_t ri[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) ri[c] = cursor_rsrc(Dd.img + c * cs, cur);
#pragma unroll
    for (int r = 0; r < R + 2; ++r) {
      const bool slotted = SK > 1 && t >= 0 && r >= 1 && r <= R;
      const unsigned od = slotted ? slot_ofs[t][r - 1] : rofs[r];
      const unsigned oi = (slotted && t < P - 1) ? slot_ofs[t][r - 1] : rofs[r];
      if (r >= r0 && r < r1) {
#pragma unroll
        for (int c = 0; c < CT; ++c)
          S.I[c][r] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(ri[c], (int)oi, 0, 0));
      }
      if (r >= 1 && r <= R)
        S.d[r - 1] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rd, (int)od, 0, 0));
    }
  };
  auto load_slab = [&](Slab<R, CT> &S, const Cursor &cur, int t) {
    load_rows(S, cur, 1, R + 1, t);
  };

  // per-row validity of this lane (pad positions hold +inf in the front) and
  // ownership of each wave row (uniform)
  bool pvalid[R], row_own[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    pvalid[r] = rvalid[r + 1] && lane_valid;
    row_own[r] = rb[r + 1] >= b_own0 && rb[r + 1] < b_own1;
  }

  // XSA: stage the wave's own-row values of slice a in LDS slot a % kRunSlots.
  // Runs are the kRunLen slices a0 .. a0 + kRunLen - 1 with a0 a multiple of
  // kRunLen (clipped to the sweep).  A run whose slices have all been staged
  // is stored at the next halo exchange, after the tile's publications,
  // where the wave waits for its earlier memory operations anyway (stores
  // issued inside the steps made the compiler's waits for the prefetched
  // slabs conservative on every path); the K <= kRunSlots -
  // kRunLen slices staged before then fill free slots.  Lane l moves slot
  // a0 + l % 16 of window lane 4j + l / 16, for j < 16, so every 16 lanes
  // store one 64-byte segment of the output.  Only this wave reads what it
  // staged and a wave's LDS accesses complete in order, so no barrier is
  // needed; the wave-scope fences keep the compiler from moving the accesses
  // across each other.  Slices past the end of the array (a partial first or
  // last run) and positions the tile does not own get an out-of-range
  // offset.  The host uses this form only for outputs of less than 4 GiB,
  // so 32-bit offsets address every element (the wrapped products of a
  // negative window lane are replaced before use).
  int xa_a0 = -1;  // first slice of the run awaiting its stores, or -1
  auto xa_flush = [&]() {
    if constexpr (XSA) {
      constexpr int LPR = kRunLen, PPI = 64 / kRunLen;
      static_assert(64 % kRunLen == 0, "run layout");
      if (xa_a0 >= 0) {
        const int q = lane % LPR, pl = lane / LPR;
        const int sq = (xa_a0 + q) % kRunSlots;  // LDS slot of this lane's slice
        const unsigned sXe4 = (unsigned)Dd.sXe * 4u;
        const unsigned lane_base = (unsigned)(ew0 + pl) * sXe4 + (unsigned)(xa_a0 + q) * 4u;
        const bool a_ok = xa_a0 + q < nA;
        const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)Dd.dxo, 0, 0xFFFFFFF0u, 0x00020000);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int r = 0; r < R; ++r) {
          if (!row_own[r]) continue;
          const unsigned row_base = (unsigned)rb[r + 1] * (unsigned)Dd.sXb * 4u;
#pragma unroll
          for (int j = 0; j < kRunLen; ++j) {
            const int p = j * PPI + pl;  // window lane
            const int ep = ew0 + p;
            const bool own = a_ok && ep >= e_own0 && ep < e_own1;
            const float x = xrun[sq][(w * R + r - K) * 64 + p];
            const unsigned off = own ? lane_base + (unsigned)(j * PPI) * sXe4 + row_base : 0xFFFFFFFFu;
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x), rx, (int)off, 0, 0);
          }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        xa_a0 = -1;
      }
    }
  };
  // Branch-free staging (a branch in the step keeps the compiler from
  // moving work across it): rows the tile does not own write a spare row,
  // and the padded steps past either end (a >= -(K - 1), K <= kXsaMaxK)
  // write slots that hold no pending slice.
  int xrow[XSA ? R : 1];
#pragma unroll
  for (int r = 0; r < (XSA ? R : 0); ++r) xrow[r] = (row_own[r] ? w * R + r - K : XOR) * 64 + lane;
  auto xa_stage = [&](const float (&v)[R], int a) {
    if constexpr (XSA) {
      const int sa = (a + kRunSlots) % kRunSlots;
#pragma unroll
      for (int r = 0; r < R; ++r) xrun[sa][xrow[r]] = v[r];
      // one run completes per block at most (K < kRunLen); a forward
      // sweep's partial last run is stored after the loop
      const int g = a & (kRunLen - 1);
      const bool done = (unsigned)a < (unsigned)nA && (dir < 0 ? g == 0 : g == kRunLen - 1);
      xa_a0 = done ? a - g : xa_a0;
    }
  };

  // At block step j only rows within K - j of the tile's own rows can still
  // reach them by the next exchange, so a wave computes in its first
  // live_steps steps of a block: K with an own row, K less its distance to
  // them otherwise, 0 without a row in the plane.  (It still passes its edge
  // rows on: the neighbour wave's next step needs the last ones.)  At K = 10,
  // where a 32-row window holds 12 own rows, this is a quarter of the work.
  int live_steps = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int b = rb[r + 1];
    if (b >= 0 && b < nB) live_steps = max(live_steps, K - max(max(b_own0 - b, b - (b_own1 - 1)), 0));
  }

  // Slab ring: the slab of step s is S[s % P]; its image rows are also the
  // front image of step s + 1, so a slab is refilled (with the slice of step
  // s + P) only after step s + 1 has used it; the front of step 0 starts in
  // S[P - 1].  Slabs stay in fixed registers this way.
  float Fd[R];  // front distance rows 0..R-1
  Slab<R, CT> S[P];
  load_rows(S[P - 1], cursor_of(-1), 0, R + 2, -1);  // front slice: not modified by this sweep
#pragma unroll
  for (int r = 0; r < R; ++r) Fd[r] = pvalid[r] ? init_of(S[P - 1].d[r]) : kInf;
  if constexpr (INIT) {
    // the output's copy of the untouched first slice: its initialisation
    const Cursor c0 = cursor_of(-1);
    const __amdgpu_buffer_rsrc_t rs = cursor_rsrc(Dd.d, c0);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const unsigned off = (row_own[r] && lane_own) ? rofs[r + 1] : kNowhere;
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(Fd[r]), rs, (int)off, 0, 0);
    }
  }
  if constexpr (XST) {  // stage the first slice as step -1 (ring slot P - 1)
#pragma unroll
    for (int r = 0; r < R; ++r) xtile[edge_slot(P - 1)][w * R + r][lane] = Fd[r];
  }
  xa_stage(Fd, a_first - dir);  // XSA: the sweep's untouched first slice
#pragma unroll
  for (int p = 0; p < P - 1; ++p) load_slab(S[p], cursor_of(p), p);
  // the slices that the loop stores (step s) and prefetches (step s + P - 1)
  Cursor cur_st = cursor_of(0), cur_pf = cursor_of(P - 1);

  // Own-layout output of the slice at cursor c, whose values the front holds:
  // raw buffer stores; non-own lanes get an out-of-range offset and the
  // hardware drops their writes, and so do rows the tile does not own on the
  // short rings.  On the 5-slice ring those rows branch around the store
  // (512^3: 611 against 631 us a sweep; on the 3-slice ring the branch makes
  // the waits for the prefetched slabs conservative: 919 against 811 us).  A
  // padded step's slice is outside the array: all its stores are dropped.
  auto store_own = [&](const Cursor &c) {
    const __amdgpu_buffer_rsrc_t rs = cursor_rsrc(Dd.d, c);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const unsigned off = (row_own[r] && lane_own) ? rofs[r + 1] : kNowhere;
      if (P < 5 || row_own[r]) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(Fd[r]), rs, (int)off, 0, 0);
    }
  };
  // the stores that the block's last step left
  auto store_last = [&]() {
    if constexpr (XS == 0) store_own(Cursor{cur_st.a - dir, cur_st.off - dAb});
  };

  // Publishes the tile's own front values that neighbours read and reloads
  // the halo positions of the window from the neighbours' publications
  // (publish_ofs, reload_ofs).  Pending rows are polled together, so one
  // memory round trip serves all of them.  A wave's loads return in order, so
  // the block's last stores and the prefetch of the next slice follow the
  // wait: a poll behind them waited for them too (512^3: 702 against 585 us a
  // sweep with the prefetch before the wait).
  bool wd_tripped = false;
  unsigned pub[R], src[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    pub[r] = publish_ofs(rb[r + 1]);
    src[r] = reload_ofs(rb[r + 1]);
  }
  // COMM: hand the front to the exchange wave and take the halo back from it
  auto exchange_via_comm = [&](int blk, Slab<R, CT> &pf_slab) {
    (void)blk;
#pragma unroll
    for (int r = 0; r < R; ++r) xfront[w * R + r][lane] = Fd[r];
    store_last();
    load_slab(pf_slab, cur_pf, P - 2);
    advance(cur_pf);
    __syncthreads();  // front visible to the exchange wave
    __syncthreads();  // halo values written by it
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (src[r] != kNoHalo) Fd[r] = xfront[w * R + r][lane];
  };
  auto exchange = [&](int blk, Slab<R, CT> &pf_slab) {
    // measurement only (xhist non-null): how long this wave spends in the
    // exchange, from its publications to the last halo value it waits for,
    // as a histogram of the device's constant-rate clock (log2 buckets)
    const unsigned long long t_in = xhist ? wall_clock64() : 0ull;
    const unsigned tag = tag_base + (unsigned)blk;
    const __amdgpu_buffer_rsrc_t h = halo_rsrc(halo + (blk & 1) * tile_slots);
#pragma unroll
    for (int r = 0; r < R; ++r) halo_publish(h, pub[r], Fd[r], tag);
    // XSA: a run completed in this block is stored after the publications (which then leave first) and drains
    // while the wave waits to poll; the halo wait below also waits for it,
    // so every path leaves the exchange with the same loads in flight
    xa_flush();
    // Neighbours publish at about the same moment; polling right away mostly
    // finds their values not yet visible.
    if constexpr (NWR <= 16) __builtin_amdgcn_s_sleep(kHaloPollDelay16);
    else if (K == P) __builtin_amdgcn_s_sleep(kHaloPollDelay);
    else __builtin_amdgcn_s_sleep(kHaloPollDelayDeep);
    uint2v x[R];
#pragma unroll
    for (int r = 0; r < R; ++r) x[r] = halo_read(h, src[r]);
    // after an expiry this wave waits no more: the sweep then finishes
    // (with wrong values, reported through the status word) instead of
    // spending the full limit again at every later exchange
    if (!halo_wait<R, (NWR <= 16 ? kHaloRepollDelay16 : kHaloRepollDelay)>(h, src, x, tag, wd_tripped ? 0 : spin_limit)) {
      __hip_atomic_store(status, FG_EWATCHDOG, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      wd_tripped = true;
    }
    load_slab(pf_slab, cur_pf, P - 2);
    advance(cur_pf);
    store_last();
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (src[r] != kNoHalo) Fd[r] = __uint_as_float(x[r].x);
    if (xhist && lane == 0) {
      const unsigned long long dt = wall_clock64() - t_in;
      const int bucket = dt ? min(64 - __clzll(dt), kXHistBuckets - 1) : 0;
      atomicAdd(&xhist_wg[bucket], 1u);  // LDS; added to the device histogram at the end
    }
  };

  // One slice: Sl holds the new slice (ring slot `slot`), Fr the previous
  // one (front image).  Afterwards Fr is refilled with the slice of step
  // s + P - 1.
  // j: its number in the block (1..K); the block's last step (no prefetch)
  // leaves its own-layout stores to the exchange.
  auto step = [&](Slab<R, CT> &Sl, Slab<R, CT> &Fr, int s, int j, int slot, bool prefetch) {
    // steps past the end of the sweep (the last block is padded to K steps)
    // compute on slices of zeros and store nothing
    (void)s;
    // Wave-boundary front rows through LDS, and the new slice's image rows
    // -1 and R (the front image of the next step) from the neighbour waves
    // (branch-free: the edge waves read their own slot and select +inf for
    // the distance; their outer image rows then only meet +inf candidates).
    // The candidates whose front row the wave holds itself are computed
    // between the writes and the barrier, so that neither the writes' latency
    // nor the slowest wave's barrier is idle time, and the image differences
    // to the neighbours' rows while the reads are under way.
    const int es = XSA ? (s & 1) : edge_slot(slot);
    edge_first[es][w][lane] = Fd[0];
    edge_last[es][w][lane] = Fd[R - 1];
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      edgeI_first[es][w][c][lane] = Sl.I[c][1];
      edgeI_last[es][w][c][lane] = Sl.I[c][R];
    }
    float In[R][CT];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int c = 0; c < CT; ++c) In[r][c] = Sl.I[c][r + 1];
    auto front_image = [&](int row, float (&Iq)[CT]) {  // image row -1..R of the previous slice
#pragma unroll
      for (int c = 0; c < CT; ++c) Iq[c] = Fr.I[c][row + 1];
    };
    Fold<FAST> fold[R];
    // triples of row r from front row r + I - 1, whose distance is dq
    auto triple = [&](auto I_, int r, float dq) {
      constexpr int I = decltype(I_)::value;
      float Iq[CT], t[3];
      front_image(r + I - 1, Iq);
      candidates_row<I, CT, LAMB1>(t, dq, Iq, In[r], e1, lg);
      fold[r].take(I, t);
    };
    constexpr std::integral_constant<int, 0> above{};
    constexpr std::integral_constant<int, 1> same{};
    constexpr std::integral_constant<int, 2> below{};
    // Candidates of row r, first in the reference's order, that are folded
    // before the barrier: the row then holds one value over it instead.  Where
    // registers decide how many workgroups a unit holds: 8 x 4 with 4 channels
    // takes 124 of them instead of 132 (two workgroups, else one), 4 x 8 with 2
    // channels 140 instead of 184 (three, else two).  Elsewhere it is no gain
    // (lamb 1.5, 20 x 120 x 140 888 / 910 us, 256 x 400 x 400 4187 / 4231).
    constexpr bool kEarly = !FAST && P == 2 && (R == 8 || CT == 4);
    auto early_of = [](int r) { return !kEarly || r == 0 ? 0 : r < R - 1 ? 9 : 6; };
    const bool live = j <= live_steps;
    if (live) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        triple(same, r, Fd[r]);
        if (r > 0) triple(above, r, Fd[r - 1]);
        if (r < R - 1) triple(below, r, Fd[r + 1]);
        if (early_of(r) > 0) fold[r].early(init_of(Sl.d[r]), early_of(r));
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // (the compiler would move these past the barrier)
    __syncthreads();
    const float t = edge_last[es][max(w - 1, 0)][lane];
    const float u = edge_first[es][min(w + 1, NW - 1)][lane];
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      Sl.I[c][0] = edgeI_last[es][max(w - 1, 0)][c][lane];
      Sl.I[c][R + 1] = edgeI_first[es][min(w + 1, NW - 1)][c][lane];
    }
    // the previous step's staged window is complete (barrier above)
    xflush(edge_slot((slot + P - 1) % P), s - 1);
    if (live) {
      triple(above, 0, (w > 0) ? t : kInf);
      triple(below, R - 1, (w < w_last) ? u : kInf);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float v = fold[r].with(init_of(Sl.d[r]), early_of(r));
        Fd[r] = pvalid[r] ? v : kInf;
      }
    }
    if constexpr (XST) {
#pragma unroll
      for (int r = 0; r < R; ++r) xtile[edge_slot(slot)][w * R + r][lane] = Fd[r];
    } else if constexpr (XSA) {
      xa_stage(Fd, cur_st.a);
    } else if (prefetch) {
      store_own(cur_st);
    }
    advance(cur_st);
    // prefetch without a branch: past the end of the sweep the loads return 0
    // and the data is never consumed (only steps that store nothing use it)
    if (prefetch) {
      load_slab(Fr, cur_pf, (slot + P - 1) % P);
      advance(cur_pf);
    }
  };

  // Blocks of exactly K steps (K a multiple of P, so a block starts at a
  // step s with s % P == 0 and slab p always sits in S[p]); the last block is
  // padded with steps that store nothing.  Every path into the group loop
  // and the block loop holds the ring in the same registers, so the waits
  // on prefetched slabs stay precise (no block boundary drains the loads).
  // The last step of a block defers its prefetch into the exchange.
  const int groups = K / P;
  const int nblocks = (nsteps + K - 1) / K;
  for (int blk = 0;; ++blk) {
    const int s0 = blk * K;
    for (int g = 0; g < groups - 1; ++g) {
#pragma unroll
      for (int p = 0; p < P; ++p) step(S[p], S[(p + P - 1) % P], s0 + g * P + p, g * P + p + 1, p, true);
    }
    const int sl = s0 + K - P;
#pragma unroll
    for (int p = 0; p < P - 1; ++p) step(S[p], S[(p + P - 1) % P], sl + p, K - P + p + 1, p, true);
    step(S[P - 1], S[P - 2], sl + P - 1, K, P - 1, false);
    if (blk + 1 >= nblocks) {
      store_last();
      break;
    }
    // deferred prefetch of step s0 + K - 1: the slice of step s0 + K + P - 2
    if constexpr (COMM) exchange_via_comm(blk + 1, S[P - 2]);
    else exchange(blk + 1, S[P - 2]);
  }
  if constexpr (XST) {
    __syncthreads();
    xflush(edge_slot(P - 1), nblocks * K - 1);  // the last step sits in slot P - 1
  }
  if constexpr (XSA) {
    xa_flush();  // a run completed in the last block
    if (dir > 0 && ((nA - 1) & (kRunLen - 1)) != kRunLen - 1) {  // a forward sweep's partial last run
      xa_a0 = (nA - 1) & ~(kRunLen - 1);
      xa_flush();
    }
  }
  if (xhist) {
    __syncthreads();
    if (threadIdx.x < kXHistBuckets && xhist_wg[threadIdx.x]) atomicAdd(xhist + threadIdx.x, xhist_wg[threadIdx.x]);
  }
}

// ---------------------------------------------------------------------------
// One-row sweeps (2D rows and columns, planes of one row)
// ---------------------------------------------------------------------------

// Waves of a row workgroup that read global memory and prepare the steps.
constexpr int kRowProducers = 6;
constexpr int kRowThreads = (1 + kRowProducers) * 64;
// Halo depths with compiled kernels are the multiples of this.
constexpr int kRowHaloStep = 6;
// Steps that the front wave reads from LDS ahead of their use.
constexpr int kRowAhead = 6;
// Row workgroups per compute unit that a plan counts on at halo depth K.  LDS
// would hold two at K = 30, but they ran slower than one at K = 24 (a 1536^2
// image with 3 channels: 384 workgroups at K = 30 1108 us, 96 at K = 24
// 793 us; four times 1292 lanes, 324 workgroups at K = 24 1326 us, 188 at
// K = 18 1543 us).
constexpr int row_groups_per_cu(int K) { return K >= 30 ? 1 : K >= 24 ? 2 : K >= 18 ? 3 : 4; }

// Everything of a row tile that both kinds of wave use.
struct RowTile {
  int te, lane, e, ew0, e_own0, e_own1;
  bool lane_valid, lane_own;
  int nA, dir, a_first, nsteps, nblocks;
  unsigned stride4;     // bytes of a slice (a row of lanes)
  unsigned dstride4;    // from one step's slice to the next (modulo 2^32)
  unsigned range;       // bytes of the array
  unsigned lofs;        // this lane's byte offset in a slice, clamped into it
};

__device__ __forceinline__ RowTile row_tile(const SweepDesc &Dd, int te, int K) {
  const int nTE = Dd.nTE, TE = Dd.TE, nE = Dd.nE;
  RowTile T;
  T.te = te;
  T.lane = threadIdx.x & 63;
  T.e_own0 = te * TE;
  T.e_own1 = min(nE, T.e_own0 + TE);
  T.ew0 = (nTE > 1) ? T.e_own0 - K : -1;
  T.e = T.ew0 + T.lane;
  T.lane_valid = T.e >= 0 && T.e < nE;
  T.lane_own = T.e >= T.e_own0 && T.e < T.e_own1;
  T.nA = Dd.nA;
  T.dir = Dd.dir;
  T.nsteps = Dd.nA - 1;
  T.nblocks = (T.nsteps + K - 1) / K;
  T.a_first = Dd.dir > 0 ? 1 : Dd.nA - 2;
  T.stride4 = (unsigned)Dd.sA * 4u;
  T.dstride4 = (unsigned)Dd.dir * T.stride4;
  T.range = (unsigned)((long long)Dd.nA * Dd.sA * 4);
  T.lofs = (unsigned)min(max(T.e, 0), nE - 1) * 4u;
  return T;
}

// Byte offset of slice a of the sweep's arrays.  Slices before the first or
// past the last one give offsets at or beyond the array's range (the host
// runs these kernels only when (nA + 32) * stride4 <= 2^31), so their loads
// return 0.
__device__ __forceinline__ unsigned row_ofs(const RowTile &T, int a) { return (unsigned)a * T.stride4 + T.lofs; }

// LDS of a row workgroup: two blocks of prepared steps and of new values.
template <int K>
struct RowShared {
  float4 pay[2][K][64];
  float res[2][K][64];  // (what the front wave reads ahead past pay lies in here)
  float spare[(K < 2 * kRowAhead ? 2 * kRowAhead - K : 0) * 128 + 1];
  unsigned xhist[kXHistBuckets];
};
static_assert(sizeof(RowShared<24>) * row_groups_per_cu(24) <= 160 << 10 &&
                  sizeof(RowShared<18>) * row_groups_per_cu(18) <= 160 << 10 &&
                  sizeof(RowShared<12>) * row_groups_per_cu(12) <= 160 << 10,
              "row workgroups share a CU's LDS");

// The part of block b that producer pw prepares: steps pw * SP .. pw * SP + SP - 1.
template <int SP, int CT>
struct RowSteps {
  float I[SP + 1][CT];  // image: the slice before the first step, then each step's
  float d[SP];          // old distance (or the mask, initialising sweeps)
};

template <int K, int CT, bool LAMB1>
__device__ __forceinline__ void row_produce(const SweepDesc &Dd, const RowTile &T, int pw,
                                            float4 (*__restrict__ pay)[K][64], float (*__restrict__ res)[K][64]) {
  constexpr int SP = K / kRowProducers;
  const bool init = Dd.init_mode != 0, init_inv = Dd.init_mode == 2;
  RowSteps<SP, CT> S;
  auto load = [&](int b) {
    const __amdgpu_buffer_rsrc_t rd =
        __builtin_amdgcn_make_buffer_rsrc((void *)(init ? Dd.init_src : Dd.d), 0, T.range, 0x00020000);
    unsigned o = row_ofs(T, T.a_first + (b * K + pw * SP - 1) * T.dir);  // the slice before the first step's
#pragma unroll
    for (int i = 0; i <= SP; ++i, o += T.dstride4) {
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        const __amdgpu_buffer_rsrc_t ri =
            __builtin_amdgcn_make_buffer_rsrc((void *)(Dd.img + c * Dd.cs), 0, T.range, 0x00020000);
        S.I[i][c] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(ri, (int)o, 0, 0));
      }
      if (i > 0) S.d[i - 1] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rd, (int)o, 0, 0));
    }
  };
  // the weighted image differences of each step's three candidates and its
  // old distance.  Pad lanes get +inf, so their new value is +inf.  Where the
  // old distance is NaN the differences are too, so that the front wave's
  // plain minimum keeps it (see row_relax).
  auto make = [&](int b) {
#pragma unroll
    for (int i = 0; i < SP; ++i) {
      float l[3];
      l[0] = absdiff_sum<1, 0, 1, CT>(fabsf(shiftE<0, 17>(S.I[i][0]) - S.I[i + 1][0]), S.I[i], S.I[i + 1]);
      l[1] = absdiff_sum<1, 1, 1, CT>(fabsf(S.I[i][0] - S.I[i + 1][0]), S.I[i], S.I[i + 1]);
      l[2] = absdiff_sum<1, 2, 1, CT>(fabsf(shiftE<2, 19>(S.I[i][0]) - S.I[i + 1][0]), S.I[i], S.I[i + 1]);
      float d = S.d[i];
      if (init) {
        const float t = 1.0f - d;
        d = Dd.init_v * (init_inv ? t : d);
      }
      d = T.lane_valid ? d : kInf;
      const bool keep = !T.lane_valid || __builtin_isnan(d);
      float4 q;
      q.x = keep ? d : (LAMB1 ? l[0] : Dd.lg * l[0]);
      q.y = keep ? d : (LAMB1 ? l[1] : Dd.lg * l[1]);
      q.z = keep ? d : (LAMB1 ? l[2] : Dd.lg * l[2]);
      q.w = d;
      pay[b & 1][pw * SP + i][T.lane] = q;
    }
  };
  // block b's new values of the tile's own lanes
  auto store = [&](int b) {
    if (Dd.dxo) {  // the other 2D layout: runs of consecutive slices per lane
      const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)Dd.dxo, 0, T.range, 0x00020000);
      const int n = (T.e_own1 - T.e_own0) * K;
      for (int k = pw * 64 + T.lane; k < n; k += kRowProducers * 64) {
        const int el = k / K, sl = k - el * K;
        const int s = b * K + sl;
        const float v = res[b & 1][sl][T.e_own0 - T.ew0 + el];
        const unsigned o = (unsigned)(T.e_own0 + el) * (unsigned)Dd.sXe * 4u +
                           (unsigned)(T.a_first + s * T.dir) * (unsigned)Dd.sXa * 4u;
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rx, (int)(s < T.nsteps ? o : 0xFFFFFFFFu), 0, 0);
      }
    } else {
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)Dd.d, 0, T.range, 0x00020000);
      const int s0 = b * K + pw * SP;
      unsigned o = row_ofs(T, T.a_first + s0 * T.dir);
#pragma unroll
      for (int i = 0; i < SP; ++i, o += T.dstride4) {
        const float v = res[b & 1][pw * SP + i][T.lane];
        const bool own = T.lane_own && s0 + i < T.nsteps;
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rs, (int)(own ? o : 0xFFFFFFFFu), 0, 0);
      }
    }
  };
  // While the front wave runs block b: prepare b + 1, read b + 2, store
  // b - 1.  One copy of the code serves the first and last blocks too: a
  // launch starts with cold instruction caches, and straight-line code of
  // its own for them cost several microseconds a sweep.
  for (int b = -2; b <= T.nblocks; ++b) {
    if (b >= -1 && b + 1 < T.nblocks) make(b + 1);
    if (b + 2 < T.nblocks) load(b + 2);
    if (b > 0) store(b - 1);
    if (b >= -1 && b < T.nblocks) __syncthreads();
  }
}

// One step of the front wave: the new values from the front F and the prepared
// differences q.x, q.y, q.z (neighbours -1, 0, +1) and old distances q.w.
// Every instruction here is on the sweep's serial chain.  FAST: v_min3 drops
// NaN candidates, and v_min_f32 of (m, old) returns old when m is NaN; where
// old is NaN all candidates are (the producers see to it), so the result is
// the reference's fold without its compare and select, whose mask write and
// read cost the chain ~13 clocks more.  Written as one block because the
// compiler would quiet the loaded operand of a minimum with one more
// instruction.  A lane-shifted operand must not be read within two wait
// states of its write: the add before it (and s_nop, or a second add)
// stands between.
template <bool LAMB1, bool FAST>
__device__ __forceinline__ float row_relax(float F, const float4 &q, float e1s, float e1c) {
  if constexpr (FAST) {
    float c3, c4, c5;
    if constexpr (LAMB1) {
      asm("v_add_f32 %[c4], %[F], %[q4]\n\t"
          "s_nop 0\n\t"
          "v_add_f32_dpp %[c3], %[F], %[q3] wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
          "v_add_f32_dpp %[c5], %[F], %[q5] wave_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
          "v_min3_f32 %[c3], %[c3], %[c4], %[c5]\n\t"
          "v_min_f32 %[F], %[c3], %[d]"
          : [F] "+v"(F), [c3] "=&v"(c3), [c4] "=&v"(c4), [c5] "=&v"(c5)
          : [q3] "v"(q.x), [q4] "v"(q.y), [q5] "v"(q.z), [d] "v"(q.w));
    } else {
      float ts;
      asm("v_add_f32 %[ts], %[F], %[es]\n\t"
          "v_add_f32 %[c4], %[F], %[ec]\n\t"
          "v_add_f32 %[c4], %[c4], %[q4]\n\t"
          "v_add_f32_dpp %[c3], %[ts], %[q3] wave_shr:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
          "v_add_f32_dpp %[c5], %[ts], %[q5] wave_shl:1 row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
          "v_min3_f32 %[c3], %[c3], %[c4], %[c5]\n\t"
          "v_min_f32 %[F], %[c3], %[d]"
          : [F] "+v"(F), [ts] "=&v"(ts), [c3] "=&v"(c3), [c4] "=&v"(c4), [c5] "=&v"(c5)
          : [q3] "v"(q.x), [q4] "v"(q.y), [q5] "v"(q.z), [d] "v"(q.w), [es] "v"(e1s), [ec] "v"(e1c));
    }
    return F;
  } else {
    // candidates may be -0: folded one by one in the reference's order
    const float ts = F + e1s;
    const float c[3] = {shiftE<0, 81>(ts) + q.x, (F + e1c) + q.y, shiftE<2, 83>(ts) + q.z};
    float nd = q.w;
#pragma unroll
    for (int k = 0; k < 3; ++k) nd = (c[k] < nd) ? c[k] : nd;
    return nd;
  }
}

// A row sweep is a chain of nA - 1 dependent steps, so a tile's time is its
// longest wave's instructions per step plus an exchange every K steps.  The
// work that does not depend on the front (loads, image differences and
// weights of every channel, the initialisation, pad lanes, stores) is taken
// off the chain: wave 0, the front wave, only reads a prepared step from LDS
// (16 bytes a lane), adds, takes the minimum and leaves the new value in LDS,
// while the producer waves of the workgroup prepare block b + 1, read global
// memory for block b + 2 and store block b - 1.  One barrier per block of K steps.  Window, halo and publications
// are those of the tiled kernel with one row.
// Measured, 512^2, one channel, K = 30: 1690 clocks of steps (56 each), ~180 to
// publish and ~1100 until the neighbours' values are there, per block of 30
// steps; a sweep 35 us against 43 us for one wave doing everything with its
// steps in a 30-slice register ring (20 instructions a step); 1536^2 with 3
// channels 97 against 225 us.  Producers in six waves: with three a 3-channel
// block waited ~750 clocks for them.
template <int K, bool LAMB1, bool FAST>
__global__ __launch_bounds__(kRowThreads)
    __attribute__((amdgpu_waves_per_eu((row_groups_per_cu(K) * (kRowThreads / 64) + 3) / 4))) void row_sweep_kernel(
    const SweepDesc *__restrict__ descs, int ndesc, SweepDesc one, int Karg, unsigned tag_base,
    unsigned long long *__restrict__ halo_base, int *__restrict__ status, int spin_limit,
    unsigned *__restrict__ xhist) {
  static_assert(K % kRowProducers == 0, "producers prepare equal parts of a block");
  __shared__ RowShared<K> sh;
  float4 (*const pay)[K][64] = sh.pay;
  float (*const res)[K][64] = sh.res;
  unsigned *const xhist_wg = sh.xhist;
  // role 0 is the front wave: wave 3, whose SIMD holds no other wave of the
  // workgroup, and another one in each next round of 256 workgroups, so that
  // two front waves on one CU run on different SIMDs
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), front = 3 - ((blockIdx.x >> 8) & 3);
  const int w = wave >= front ? wave - front : wave - front + 1 + kRowProducers;
  const int tile = xcd_remap(blockIdx.x, gridDim.x);
  if (xhist) {
    if (threadIdx.x < kXHistBuckets) xhist_wg[threadIdx.x] = 0u;
    __syncthreads();
  }
  SweepDesc Dd;
  if (descs) {
    int lo = 0, hi = ndesc - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (descs[mid].tile0 <= tile) lo = mid; else hi = mid - 1;
    }
    Dd = descs[lo];
  } else {
    Dd = one;
  }
  if (Karg != K || Dd.nB != 1 || Dd.C < 1 || Dd.C > 4) {
    if (threadIdx.x == 0) __hip_atomic_store(status, FG_EINVAL, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    return;
  }
  const RowTile T = row_tile(Dd, tile - Dd.tile0, K);
  const int nTE = Dd.nTE, TE = Dd.TE, te = T.te;
  if (T.nsteps <= 0) return;

  if (w > 0) {
    switch (Dd.C) {
      case 1: row_produce<K, 1, LAMB1>(Dd, T, w - 1, pay, res); break;
      case 2: row_produce<K, 2, LAMB1>(Dd, T, w - 1, pay, res); break;
      case 3: row_produce<K, 3, LAMB1>(Dd, T, w - 1, pay, res); break;
      default: row_produce<K, 4, LAMB1>(Dd, T, w - 1, pay, res); break;
    }
  } else {
    __builtin_amdgcn_s_setprio(3);  // ahead of producers on its SIMD
    const int lane = T.lane;
    const float e1s = Dd.e1[3], e1c = Dd.e1[4];
    // the front: the sweep's untouched first slice, which an initialising
    // sweep and one that writes the other layout also store
    float F;
    {
      const bool init = Dd.init_mode != 0;
      const __amdgpu_buffer_rsrc_t rd =
          __builtin_amdgcn_make_buffer_rsrc((void *)(init ? Dd.init_src : Dd.d), 0, T.range, 0x00020000);
      const int a = T.a_first - T.dir;
      float x = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rd, (int)row_ofs(T, a), 0, 0));
      if (init) {
        const float t = 1.0f - x;
        x = Dd.init_v * (Dd.init_mode == 2 ? t : x);
      }
      F = T.lane_valid ? x : kInf;
      // (a buffer store: a flat store in flight would make every wait for an
      // LDS read below a wait for all of them)
      const __amdgpu_buffer_rsrc_t rs =
          __builtin_amdgcn_make_buffer_rsrc((void *)(Dd.dxo ? Dd.dxo : Dd.d), 0, T.range, 0x00020000);
      const unsigned o = Dd.dxo ? (unsigned)T.e * (unsigned)Dd.sXe * 4u + (unsigned)a * (unsigned)Dd.sXa * 4u
                                : row_ofs(T, a);
      if (T.lane_own && (Dd.dxo || init)) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(F), rs, (int)o, 0, 0);
    }
    // the halo: own lanes within K of a neighbour publish, the other lanes
    // of the plane reload from the tile that owns them
    gu64 *halo = (gu64 *)halo_base + Dd.halo0;
    const bool pub = T.lane_own && ((te > 0 && T.e - T.e_own0 < K) || (te < nTE - 1 && T.e_own1 - 1 - T.e < K));
    const bool need = T.lane_valid && !T.lane_own && max(T.e_own0 - T.e, T.e - (T.e_own1 - 1)) <= K;
    const int ote = T.lane_valid ? T.e / TE : te;
    gu64 *pub_at = halo + (long long)te * 2 * TE + (T.lane_own ? T.e - T.e_own0 : 0);
    const gu64 *src_at = halo + (long long)ote * 2 * TE + (T.lane_valid ? T.e - ote * TE : 0);
    bool tripped = false;
    __syncthreads();
    for (int b = 0;; ++b) {
      // prepared steps are read kAhead steps early; the scheduling fences keep
      // the reads there (left alone, the compiler moves each next to its use
      // and the chain waits for LDS at every step)
      constexpr int kAhead = kRowAhead;
      static_assert(K % kAhead == 0, "the steps run in groups of kAhead");
      const float4 *pq = &pay[b & 1][0][lane];
      float *pr = &res[b & 1][0][lane];
      float4 q[kAhead];
#pragma unroll
      for (int s = 0; s < kAhead; ++s) q[s] = pq[s * 64];
#pragma unroll
      for (int g = 0; g < K / kAhead; ++g) {
        // (the last group reads on past its block, inside RowShared; unused)
        pq += kAhead * 64;
#pragma unroll
        for (int s = 0; s < kAhead; ++s) {
          __builtin_amdgcn_sched_barrier(0);
          F = row_relax<LAMB1, FAST>(F, q[s], e1s, e1c);
          q[s] = pq[s * 64];
          pr[s * 64] = F;
        }
        __builtin_amdgcn_sched_barrier(0);
        pr += kAhead * 64;
      }
      if (b + 1 >= T.nblocks) break;
      const unsigned long long t_in = xhist ? wall_clock64() : 0ull;
      const unsigned tag = tag_base + (unsigned)(b + 1);
      const int hslot = ((b + 1) & 1) * TE;
      if (pub) __hip_atomic_store(pub_at + hslot, pack(F, tag), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();  // block b is in res, block b + 1 in pay
      if (need) {
        __builtin_amdgcn_s_sleep(kRowPollDelay);
        unsigned long long x = __hip_atomic_load(src_at + hslot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // after an expiry this wave waits no more: the sweep then finishes
        // (with wrong values, reported through the status word)
        int spins = tripped ? spin_limit : 0;
        while ((unsigned)(x >> 32) != tag) {
          if (++spins > spin_limit) {
            __hip_atomic_store(status, FG_EWATCHDOG, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            tripped = true;
            break;
          }
          x = __hip_atomic_load(src_at + hslot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        F = __uint_as_float((unsigned)x);
      }
      if (xhist && lane == 0) {
        const unsigned long long dt = wall_clock64() - t_in;
        const int bucket = dt ? min(64 - __clzll(dt), kXHistBuckets - 1) : 0;
        atomicAdd(&xhist_wg[bucket], 1u);
      }
    }
    __syncthreads();
  }
  if (xhist) {
    __syncthreads();
    if (threadIdx.x < kXHistBuckets && xhist_wg[threadIdx.x]) atomicAdd(xhist + threadIdx.x, xhist_wg[threadIdx.x]);
  }
}

// The one-wave form: a wave per tile does everything, with the steps in a ring
// of 6 slices in registers.  Its chain is longer (20 instructions a step with
// one channel), but a tile issues half the instructions that a front wave and
// its producers do, which counts where a pass has more tiles than compute
// units can serve at once (see kRowWaveTiles).
constexpr int kRowWaveMaxK = 30;
template <int CT, bool LAMB1, bool FAST, bool INIT>
__device__ __forceinline__ void row_wave_run(const SweepDesc &Dd, const RowTile &T, int K, unsigned tag_base,
                                             gu64 *__restrict__ halo, int *__restrict__ status, int spin_limit,
                                             unsigned *xhist_wg) {
  constexpr int P = kRowHaloStep;
  struct Step {
    float I[CT], d;
  } S[P];
  const __amdgpu_buffer_rsrc_t rd =
      __builtin_amdgcn_make_buffer_rsrc((void *)(INIT ? Dd.init_src : Dd.d), 0, T.range, 0x00020000);
  auto load = [&](Step &q, unsigned o) {
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      const __amdgpu_buffer_rsrc_t ri =
          __builtin_amdgcn_make_buffer_rsrc((void *)(Dd.img + c * Dd.cs), 0, T.range, 0x00020000);
      q.I[c] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(ri, (int)o, 0, 0));
    }
    q.d = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rd, (int)o, 0, 0));
  };
  const bool init_inv = Dd.init_mode == 2;
  auto init_of = [&](float m) {
    const float t = 1.0f - m;
    return INIT ? Dd.init_v * (init_inv ? t : m) : m;
  };
  // stores: the offsets of slices past either end and, based at 2^31, of lanes
  // of other tiles are out of range (see row_ofs)
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)Dd.d, 0, T.range, 0x00020000);
  const unsigned out0 = T.lane_own ? T.lofs : 0x80000000u;
  unsigned st = (unsigned)T.a_first * T.stride4;
  const float e1s = Dd.e1[3], e1c = Dd.e1[4], e1n = Dd.e1[5], lg = Dd.lg;

  const int a0 = T.a_first - T.dir;  // the sweep's untouched first slice
  load(S[P - 1], row_ofs(T, a0));
  float F = T.lane_valid ? init_of(S[P - 1].d) : kInf;
  if (INIT)
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(F), rs, (int)(out0 + (unsigned)a0 * T.stride4), 0, 0);
  unsigned pf = row_ofs(T, T.a_first);
#pragma unroll
  for (int p = 0; p < P - 1; ++p, pf += T.dstride4) load(S[p], pf);

  // The next step, with its slice in S[slot] and the front's image in the slot
  // before, which is then refilled with the slice P - 1 steps on.
  auto step = [&](int slot, bool prefetch) {
    Step &Fr = S[(slot + P - 1) % P], &Sl = S[slot];
    const float c3 = candidate<1, 0, CT, LAMB1>(F, Fr.I, Sl.I, e1s, lg);
    const float c4 = candidate<1, 1, CT, LAMB1>(F, Fr.I, Sl.I, e1c, lg);
    const float c5 = candidate<1, 2, CT, LAMB1>(F, Fr.I, Sl.I, e1n, lg);
    float nd = init_of(Sl.d);
    if constexpr (FAST) {
      const float m = fminf(fminf(c3, c4), c5);
      nd = (m < nd) ? m : nd;
    } else {
      nd = (c3 < nd) ? c3 : nd;
      nd = (c4 < nd) ? c4 : nd;
      nd = (c5 < nd) ? c5 : nd;
    }
    F = T.lane_valid ? nd : kInf;
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(F), rs, (int)(out0 + st), 0, 0);
    st += T.dstride4;
    if (prefetch) {
      load(Fr, pf);
      pf += T.dstride4;
    }
  };
  const int nTE = Dd.nTE, TE = Dd.TE, te = T.te;
  const bool pub = T.lane_own && ((te > 0 && T.e - T.e_own0 < K) || (te < nTE - 1 && T.e_own1 - 1 - T.e < K));
  const bool need = T.lane_valid && !T.lane_own && max(T.e_own0 - T.e, T.e - (T.e_own1 - 1)) <= K;
  const int ote = T.lane_valid ? T.e / TE : te;
  gu64 *pub_at = halo + (long long)te * 2 * TE + (T.lane_own ? T.e - T.e_own0 : 0);
  const gu64 *src_at = halo + (long long)ote * 2 * TE + (T.lane_valid ? T.e - ote * TE : 0);
  bool tripped = false;
  for (int b = 0;; ++b) {
    for (int g = 1; g < K / P; ++g) {
#pragma unroll
      for (int p = 0; p < P; ++p) step(p, true);
    }
#pragma unroll
    for (int p = 0; p < P; ++p) step(p, p < P - 1);  // (the last prefetch follows the poll below)
    if (b + 1 >= T.nblocks) break;
    const unsigned long long t_in = xhist_wg ? wall_clock64() : 0ull;
    const unsigned tag = tag_base + (unsigned)(b + 1);
    const int hslot = ((b + 1) & 1) * TE;
    if (pub) __hip_atomic_store(pub_at + hslot, pack(F, tag), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_s_sleep(kRowPollDelay);
    unsigned long long x = (unsigned long long)tag << 32;
    if (need) x = __hip_atomic_load(src_at + hslot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    load(S[P - 2], pf);
    pf += T.dstride4;
    // (bounded as in row_sweep_kernel)
    int spins = tripped ? spin_limit : 0;
    while ((unsigned)(x >> 32) != tag) {
      if (++spins > spin_limit) {
        __hip_atomic_store(status, FG_EWATCHDOG, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        tripped = true;
        break;
      }
      x = __hip_atomic_load(src_at + hslot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (need) F = __uint_as_float((unsigned)x);
    if (xhist_wg && T.lane == 0) {
      const unsigned long long dt = wall_clock64() - t_in;
      atomicAdd(&xhist_wg[dt ? min(64 - __clzll(dt), kXHistBuckets - 1) : 0], 1u);
    }
  }
}

// MC: the most channels of a transform of the launch.  A kernel holds the
// registers of its widest ring, and tiles wait for their neighbours, so a plane
// of more tiles than are resident cannot run on it.  One kernel for 1-4 channels
// took 118 registers (16 waves a CU); by MC 57-63, 63-70, 76-79, 77-79: 32, 28,
// 24 and 24 waves, up to 8192 tiles of one channel (a line of 426 000).
template <int MC, bool LAMB1, bool FAST>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(MC == 1 ? 8 : MC == 2 ? 7 : 6))) void row_wave_kernel(
    const SweepDesc *__restrict__ descs, int ndesc, SweepDesc one, int K, unsigned tag_base,
    unsigned long long *__restrict__ halo_base, int *__restrict__ status, int spin_limit,
    unsigned *__restrict__ xhist) {
  __shared__ unsigned xhist_wg[kXHistBuckets];
  const int tile = xcd_remap(blockIdx.x, gridDim.x);
  if (xhist) {
    if (threadIdx.x < kXHistBuckets) xhist_wg[threadIdx.x] = 0u;
    __syncthreads();
  }
  SweepDesc Dd;
  if (descs) {
    int lo = 0, hi = ndesc - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (descs[mid].tile0 <= tile) lo = mid; else hi = mid - 1;
    }
    Dd = descs[lo];
  } else {
    Dd = one;
  }
  // A sweep's padded last block prefetches slices -(K + P - 3) .. nA + K + P - 4
  // at most and stores to -(K - 1) .. nA + K - 2: with (nA + 32) slices in 2^31
  // bytes, 33 slices to either side and stores based at 2^31 up to 32 of them
  // stay between the array's range and 2^32.
  static_assert(kRowWaveMaxK + kRowHaloStep - 3 <= 33 && kRowWaveMaxK <= 32, "slices past the ends stay out of range");
  if (K <= 0 || K % kRowHaloStep != 0 || K > kRowWaveMaxK || Dd.nB != 1 || Dd.dxo || Dd.C < 1 || Dd.C > MC) {
    if (threadIdx.x == 0) __hip_atomic_store(status, FG_EINVAL, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    return;
  }
  const RowTile T = row_tile(Dd, tile - Dd.tile0, K);
  if (T.nsteps <= 0) return;
  gu64 *const halo = (gu64 *)halo_base + Dd.halo0;
  unsigned *const xh = xhist ? xhist_wg : nullptr;
  auto run = [&](auto ct) {
    constexpr int CT = decltype(ct)::value;
    if (Dd.init_mode) row_wave_run<CT, LAMB1, FAST, true>(Dd, T, K, tag_base, halo, status, spin_limit, xh);
    else row_wave_run<CT, LAMB1, FAST, false>(Dd, T, K, tag_base, halo, status, spin_limit, xh);
  };
  if (MC == 1 || Dd.C == 1) run(std::integral_constant<int, 1>{});
  if constexpr (MC > 1)
    if (Dd.C == 2) run(std::integral_constant<int, 2>{});
  if constexpr (MC > 2)
    if (Dd.C == 3) run(std::integral_constant<int, 3>{});
  if constexpr (MC > 3)
    if (Dd.C == 4) run(std::integral_constant<int, 4>{});
  if (xhist) {
    __syncthreads();
    if (threadIdx.x < kXHistBuckets && xhist_wg[threadIdx.x]) atomicAdd(xhist + threadIdx.x, xhist_wg[threadIdx.x]);
  }
}

// ---------------------------------------------------------------------------
// Small 2D images: a whole transform in one workgroup
// ---------------------------------------------------------------------------

// One transform, every sweep of every iteration, with image and distance in
// LDS.
struct SmallDesc {
  const float *img;  // (C, H, W)
  const float *src;  // mask (init_mode 1: v*m, 2: v*(1-m)) or initial distance (0)
  float *out;        // (H, W), or (W, H) with `flip`
  int C, H, W, iters;
  int init_mode, flip;
  float v, lg, e1s, e1c;  // e1s: step to a side neighbour of the previous line, e1c: to the middle one
};

// The transforms of one call (signed 2, GSF 4) travel in the kernel's
// arguments: a descriptor copy of its own would cost ~15 us on the stream.
constexpr int kSmallByValue = 4;
struct SmallDescs {
  SmallDesc d[kSmallByValue];
};

constexpr int kSmallWaves = 4, kSmallHalo = 16, kSmallOwn = 64 - 2 * kSmallHalo;
constexpr int kSmallSide = kSmallWaves * kSmallOwn;  // longest side
constexpr int kSmallAhead = 4;                       // lines read ahead
// Floats per element in LDS: the distance and up to 1 or 3 image channels.
constexpr int small_element(int C) { return C == 1 ? 2 : 4; }
// Floats before and after the image that reads ahead of the last line touch.
constexpr int small_guard(int C, int W) { return kSmallAhead * (W | 1) * small_element(C); }
// LDS of an H x W image: rows of odd pitch, so that both lines of consecutive
// elements and columns spread over the banks; the guards; one word per thread
// for the lanes that store nothing.
constexpr size_t small_lds(int C, int H, int W) {
  return ((size_t)H * (W | 1) * small_element(C) + 2 * small_guard(C, W) + kSmallWaves * 64) * sizeof(float);
}

template <int EL>
struct SmallElement;
template <>
struct SmallElement<2> { typedef float2 type; };
template <>
struct SmallElement<4> { typedef float4 type; };

// A call on a small image is launches: at 64^2 a sweep's 63 steps take ~2 us
// of the ~8 us that its launch, first loads and exchanges cost.  Here one
// launch does everything: the image and the distance sit in LDS, a line of up
// to 64 elements is one wave's, a longer one is split over up to four waves
// with 32 own lanes each and 16 lanes of halo to either side, which are read
// back from the lines in LDS every 16 steps behind a barrier.  64^2, one
// channel, iter 2: 73 -> 33 us a call; 128^2 98 -> 78 us.  A step takes 53-58 ns
// (3 channels 90), as its image term is on the chain; up to a side of 64 one
// wave of the four walks it.
// Between barriers a wave's halo lanes may read a line's old distances after
// the wave that owns them has replaced them.  That changes no result: a halo
// lane that still counts computes the same minimum from the replaced value (it
// is the minimum of the old one and the same candidates, and is kept by both
// folds), and the others reach no own lane before they are read back.
template <int CT, bool LAMB1, bool FAST>
__global__ __launch_bounds__(kSmallWaves * 64) void small_call_kernel(const SmallDesc *__restrict__ descs,
                                                                      SmallDescs few) {
  constexpr int EL = CT == 1 ? 2 : 4;
  typedef typename SmallElement<EL>::type Element;
  extern __shared__ __align__(16) float small_mem[];
  SmallDesc S;
  if (descs) {
    S = descs[blockIdx.x];
  } else {
    S = few.d[0];
#pragma unroll
    for (int k = 1; k < kSmallByValue; ++k)
      if ((int)blockIdx.x == k) S = few.d[k];
  }
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int H = S.H, W = S.W, pitch = W | 1;
  const long long N = (long long)H * W;
  const int guard = small_guard(CT, W);
  float *const mem = small_mem + guard;
  for (int h = wave; h < H; h += kSmallWaves)
    for (int x = lane; x < W; x += 64) {
      const int k = h * W + x;
      const float m = S.src[k], t = 1.0f - m;
      float *el = mem + (h * pitch + x) * EL;
      el[0] = S.init_mode == 0 ? m : S.v * (S.init_mode == 2 ? t : m);
#pragma unroll
      for (int c = 0; c < CT; ++c) el[1 + c] = S.img[c * N + k];
    }
  __syncthreads();

  const float e1[9] = {0.f, 0.f, 0.f, S.e1s, S.e1c, S.e1s, 0.f, 0.f, 0.f};
  const float lg = S.lg;
  for (int sweep = 0; sweep < 4 * S.iters; ++sweep) {
    const bool rows = (sweep & 2) == 0;
    const int dir = (sweep & 1) ? -1 : 1;
    const int nA = rows ? H : W, nE = rows ? W : H;
    const int sA = (rows ? pitch : 1) * EL, sE = (rows ? 1 : pitch) * EL;  // floats
    const int nsteps = nA - 1, a0 = dir > 0 ? 0 : nA - 1;
    const bool split = nE > 64;
    const int e = split ? wave * kSmallOwn - kSmallHalo + lane : lane;
    const bool own = e >= 0 && e < nE && (!split || (lane >= kSmallHalo && lane < 64 - kSmallHalo));
    const bool has_left = e > 0, has_right = e < nE - 1;
    const bool active = wave == 0 || (split && wave * kSmallOwn < nE);
    // read position kSmallAhead lines ahead of the step, write position; lanes
    // that store nothing write a word of their own
    const float *rp = mem + a0 * sA + min(max(e, 0), nE - 1) * sE;
    float *wp = own ? mem + (a0 + dir) * sA + e * sE : small_mem + H * pitch * EL + 2 * guard + threadIdx.x;
    const int rs = dir * sA, ws = own ? rs : 0;
    float F = 0.f, Iq[CT];
    Element q[kSmallAhead];
    auto read = [&]() {
      const Element x = *reinterpret_cast<const Element *>(rp);
      rp += rs;
      return x;
    };
    if (active) {
      const Element f = read();
      const float *pf = reinterpret_cast<const float *>(&f);
      F = pf[0];
#pragma unroll
      for (int c = 0; c < CT; ++c) Iq[c] = pf[1 + c];
#pragma unroll
      for (int k = 0; k < kSmallAhead; ++k) q[k] = read();
    }
    auto step = [&](Element &x) {
      const float *pq = reinterpret_cast<const float *>(&x);
      const float dinit = pq[0];
      float In[CT];
#pragma unroll
      for (int c = 0; c < CT; ++c) In[c] = pq[1 + c];
      x = read();
      float t[3];
      candidates_row<1, CT, LAMB1>(t, F, Iq, In, e1, lg);
      t[0] = has_left ? t[0] : kInf;
      t[2] = has_right ? t[2] : kInf;
      if constexpr (FAST) {
        const float m = fminf(fminf(t[0], t[1]), t[2]);
        F = (m < dinit) ? m : dinit;
      } else {
        F = dinit;
#pragma unroll
        for (int i = 0; i < 3; ++i) F = (t[i] < F) ? t[i] : F;
      }
#pragma unroll
      for (int c = 0; c < CT; ++c) Iq[c] = In[c];
      *wp = F;
      wp += ws;
    };
    for (int s0 = 0; s0 < nsteps; s0 += kSmallHalo) {
      if (split && s0 > 0) {
        __syncthreads();  // every wave's own part of the last line is in LDS
        if (active) {
          const float x = rp[-(1 + kSmallAhead) * rs];
          F = own ? F : x;
        }
      }
      if (active) {
        const int n = min(kSmallHalo, nsteps - s0);
        int j = 0;
        for (; j + kSmallAhead <= n; j += kSmallAhead) {
#pragma unroll
          for (int k = 0; k < kSmallAhead; ++k) step(q[k]);
        }
#pragma unroll
        for (int k = 0; k < kSmallAhead - 1; ++k)
          if (j + k < n) step(q[k]);
      }
    }
    __syncthreads();
  }

  if (!S.flip) {
    for (int h = wave; h < H; h += kSmallWaves)
      for (int x = lane; x < W; x += 64) S.out[h * W + x] = mem[(h * pitch + x) * EL];
  } else {
    for (int x = wave; x < W; x += kSmallWaves)
      for (int h = lane; h < H; h += 64) S.out[x * H + h] = mem[(h * pitch + x) * EL];
  }
}

// ---------------------------------------------------------------------------
// Per-slice engine: one launch updates one slice from the previous one.
// Visits candidates in the reference order with the reference's min rule.
// ---------------------------------------------------------------------------

struct SliceDesc {
  const float *img;
  float *d;
  long long cs, sA, sB;
  int nB, nE, C;
  float lg;
  float e1[9];
};

__global__ void slice_kernel(SliceDesc D, int a, int aq) {
  const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long nplane = (long long)D.nB * D.nE;
  if (idx >= nplane) return;
  const int b = (int)(idx / D.nE), e = (int)(idx - (long long)b * D.nE);
  const long long p = (long long)a * D.sA + (long long)b * D.sB + e;
  float nd = D.d[p];
  for (int i = 0; i < 3; ++i) {
    const int bq = b + i - 1;
    if (bq < 0 || bq >= D.nB) continue;
    for (int j = 0; j < 3; ++j) {
      const int eq = e + j - 1;
      if (eq < 0 || eq >= D.nE) continue;
      const long long q = (long long)aq * D.sA + (long long)bq * D.sB + eq;
      float l = 0.0f;
      if (D.C == 1) {
        l = fabsf(D.img[p] - D.img[q]);
      } else {
        for (int c = 0; c < D.C; ++c) l += fabsf(D.img[c * D.cs + p] - D.img[c * D.cs + q]);
      }
      const float cur = (D.d[q] + D.e1[i * 3 + j]) + D.lg * l;
      nd = (cur < nd) ? cur : nd;
    }
  }
  D.d[p] = nd;
}

// ---------------------------------------------------------------------------
// Transposes (batched): out[c][w][h][d] = in[c][d][h][w]
// ---------------------------------------------------------------------------

constexpr int kXT = 64;

// Value of the combined sources at element k of the source layout.
__device__ __forceinline__ float xsrc(const XposeDesc &X, long long k) {
  const float a = X.src[k];
  if (X.kind == XK_SIGNED || X.kind == XK_GSF_MID) return a - X.src2[k];
  if (X.kind == XK_GSF_FINAL) return -(X.src2[k] - X.src3[k]) + (X.src4[k] - a);
  return a;
}

// Writes the (combined) value x to element k of the destination layout(s).
__device__ __forceinline__ void xdst(const XposeDesc &X, long long k, float x) {
  if (X.kind == XK_GSF_MID) {
    // x = Ds = D(M) - D(1-M); Md = Ds > theta, Me = Ds > -theta
    const float md = (x > X.theta) ? 1.0f : 0.0f;
    const float me = (x > -X.theta) ? 1.0f : 0.0f;
    const float m1 = 1.0f - md;  // mask of signed(image, 1 - Md)
    X.dst2[k] = X.v * m1;        // D(1-Md) init
    X.dst3[k] = X.v * (1.0f - m1);  // D(1-(1-Md)) init
    X.dst4[k] = X.v * me;        // D(Me) init
    X.dst[k] = X.v * (1.0f - me);   // D(1-Me) init
  } else {
    X.dst[k] = x;
  }
}

__global__ __launch_bounds__(256) void xpose_kernel(const XposeDesc *__restrict__ descs, int ndesc, XposeDesc one) {
  __shared__ float tile[kXT][kXT + 1];
  const int t = blockIdx.x;
  XposeDesc X;
  if (descs) {
    int lo = 0, hi = ndesc - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (descs[mid].tile0 <= t) lo = mid; else hi = mid - 1;
    }
    X = descs[lo];
  } else {
    X = one;
  }
  const int lt = t - X.tile0;
  const int plane = lt / X.tiles_dw, tt = lt - plane * X.tiles_dw;
  const int c = plane / X.H, h = plane - c * X.H;
  const int ntw = (X.W + kXT - 1) / kXT;
  const int td = tt / ntw, tw = tt - td * ntw;
  const int d0 = td * kXT, w0 = tw * kXT;
  const long long HW = (long long)X.H * X.W, HD = (long long)X.H * X.D;
  const long long cn = (long long)X.D * HW;
  const long long sbase = c * cn + (long long)h * X.W;  // element offsets of this (c, h) plane
  const long long dbase = c * cn + (long long)h * X.D;
  if (X.kind == XK_COPY && (X.W & 3) == 0 && (X.D & 3) == 0 && d0 + kXT <= X.D && w0 + kXT <= X.W &&
      (((uintptr_t)X.src | (uintptr_t)X.dst) & 15) == 0) {
    // full tile, 16-byte rows: each thread moves float4s (16 threads per
    // 256-byte row segment) and the LDS tile keeps its padded scalar layout
    const float *src = X.src + sbase;
    float *dst = X.dst + dbase;
    const int q = threadIdx.x & 15, r0 = threadIdx.x >> 4;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int r = r0 + 16 * k;
      const float4 v = *reinterpret_cast<const float4 *>(src + (long long)(d0 + r) * HW + w0 + 4 * q);
      tile[r][4 * q + 0] = v.x;
      tile[r][4 * q + 1] = v.y;
      tile[r][4 * q + 2] = v.z;
      tile[r][4 * q + 3] = v.w;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int r = r0 + 16 * k;  // output row (w)
      float4 v;
      v.x = tile[4 * q + 0][r];
      v.y = tile[4 * q + 1][r];
      v.z = tile[4 * q + 2][r];
      v.w = tile[4 * q + 3][r];
      *reinterpret_cast<float4 *>(dst + (long long)(w0 + r) * HD + d0 + 4 * q) = v;
    }
    return;
  }
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int r = ty; r < kXT; r += 4) {
    const int d = d0 + r, w = w0 + tx;
    if (d < X.D && w < X.W) tile[r][tx] = xsrc(X, sbase + (long long)d * HW + w);
  }
  __syncthreads();
  for (int r = ty; r < kXT; r += 4) {
    const int w = w0 + r, d = d0 + tx;
    if (d < X.D && w < X.W) xdst(X, dbase + (long long)w * HD + d, tile[tx][r]);
  }
}

// ---------------------------------------------------------------------------
// Elementwise init / epilogue kernels (batched through small descriptors)
// ---------------------------------------------------------------------------

enum EwKind : int {
  EW_INIT_UNSIGNED = 0,  // out = v*m (all channels)
  EW_INIT_SIGNED = 1,    // out = v*m (all channels); a = v*(1-m) (channel 0)
  EW_FINAL_SIGNED = 2,   // out0 -= a;  out_c -= v*(1-m_c) for c >= 1
  EW_GSF_MID = 3,        // from (out0, a): thresholds -> inits of the 4 stage-2 transforms
  EW_GSF_FINAL = 4,      // out0 = -(a - b) + (c2 - out0); channels >= 1 in closed form
  EW_FILL_U64 = 5,       // zero a range of 64-bit words
  EW_CHANNELS = 6,       // mask channels >= 1 (elements [n0, n0*Cm)): the op's closed form of the mask
};

struct EwDesc {
  int kind;
  long long n0;   // voxels per channel
  int Cm;
  int op;         // EW_CHANNELS: FG_OP_*
  const float *mask;
  float *out;
  float *a, *b, *c2;
  float v, theta;
  unsigned long long *u64;
  long long nu64;
  long long blk0;   // first block of this descriptor in the launch
  long long nelem;
};

// Elements per ew_kernel block (256 threads x 4).
constexpr int kEwPerBlock = 1024;

__device__ __forceinline__ float signed_closed(float v, float m) {
  // untransformed channels of signed: v*m - v*(1-m)
  return v * m - v * (1.0f - m);
}

__device__ __forceinline__ void ew_one(const EwDesc &E, long long i);

// Each block handles kEwPerBlock consecutive elements of one descriptor (the
// block-uniform search runs on scalar loads once per block), each thread 4
// of them; the unsigned initialisation (every plain call) uses one 16-byte
// load and store when the 4 elements are aligned.
__global__ __launch_bounds__(256) void ew_kernel(const EwDesc *__restrict__ descs, int ndesc, EwDesc one) {
  const long long b = blockIdx.x;
  EwDesc E;
  if (descs) {
    int lo = 0, hi = ndesc - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (descs[mid].blk0 <= b) lo = mid; else hi = mid - 1;
    }
    E = descs[lo];
  } else {
    E = one;
  }
  const long long i0 = (b - E.blk0) * kEwPerBlock + (long long)threadIdx.x * 4;
  if (i0 >= E.nelem) return;
  if (E.kind == EW_INIT_UNSIGNED && i0 + 4 <= E.nelem &&
      (((uintptr_t)(E.out + i0) | (uintptr_t)(E.mask + i0)) & 15) == 0) {
    const float4 m = *reinterpret_cast<const float4 *>(E.mask + i0);
    float4 o;
    o.x = E.v * m.x;
    o.y = E.v * m.y;
    o.z = E.v * m.z;
    o.w = E.v * m.w;
    *reinterpret_cast<float4 *>(E.out + i0) = o;
    return;
  }
  for (int j = 0; j < 4 && i0 + j < E.nelem; ++j) ew_one(E, i0 + j);
}

__device__ __forceinline__ void ew_one(const EwDesc &E, long long i) {
  {
    const float v = E.v;
    switch (E.kind) {
      case EW_INIT_UNSIGNED:
        E.out[i] = v * E.mask[i];
        break;
      case EW_INIT_SIGNED: {
        const float m = E.mask[i];
        E.out[i] = v * m;
        if (i < E.n0) E.a[i] = v * (1.0f - m);
        break;
      }
      case EW_FINAL_SIGNED:
        if (i < E.n0) E.out[i] = E.out[i] - E.a[i];
        else E.out[i] = E.out[i] - v * (1.0f - E.mask[i]);
        break;
      case EW_GSF_MID: {
        // Ds = D(M) - D(1-M); Md = Ds > theta; Me = Ds > -theta
        const float ds = E.out[i] - E.a[i];
        const float md = (ds > E.theta) ? 1.0f : 0.0f;
        const float me = (ds > -E.theta) ? 1.0f : 0.0f;
        const float m1 = 1.0f - md;        // mask of signed(image, 1 - Md)
        E.a[i] = v * m1;                   // D(1-Md) init
        E.b[i] = v * (1.0f - m1);          // D(1-(1-Md)) init
        E.c2[i] = v * me;                  // D(Me) init
        E.out[i] = v * (1.0f - me);        // D(1-Me) init
        break;
      }
      case EW_GSF_FINAL:
        if (i < E.n0) {
          E.out[i] = -(E.a[i] - E.b[i]) + (E.c2[i] - E.out[i]);
        } else {
          const float m = E.mask[i];
          const float ds = signed_closed(v, m);
          const float md = (ds > E.theta) ? 1.0f : 0.0f;
          const float me = (ds > -E.theta) ? 1.0f : 0.0f;
          const float dd = -signed_closed(v, 1.0f - md);
          const float de = signed_closed(v, me);
          E.out[i] = dd + de;
        }
        break;
      case EW_FILL_U64:
        E.u64[i] = 0ull;
        break;
      case EW_CHANNELS: {
        // element n0 + i: an untransformed channel (reference: channels >= 1
        // keep their initialisation through every pass)
        const long long k = E.n0 + i;
        const float m = E.mask[k];
        if (E.op == FG_OP_UNSIGNED) {
          E.out[k] = v * m;
        } else if (E.op == FG_OP_SIGNED) {
          E.out[k] = signed_closed(v, m);
        } else {
          const float ds = signed_closed(v, m);
          const float md = (ds > E.theta) ? 1.0f : 0.0f;
          const float me = (ds > -E.theta) ? 1.0f : 0.0f;
          E.out[k] = -signed_closed(v, 1.0f - md) + signed_closed(v, me);
        }
        break;
      }
      default:
        break;
    }
  }
}

// Single-voxel writes (click edits of resident masks), passed by value in
// groups of up to kVoxelsPerLaunch.
constexpr int kVoxelsPerLaunch = 96;
struct VoxelBatch {
  fg_voxel_set it[kVoxelsPerLaunch];
};

__global__ __launch_bounds__(128) void set_voxels_kernel(VoxelBatch b, int n) {
  const int i = threadIdx.x;
  if (i < n) b.it[i].dst[b.it[i].index] = b.it[i].value;
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------

thread_local std::string g_err;
thread_local fg_tuning g_tune = {1, 0, 0, 0};

// Requested halo depth: 0 = automatic (per plane), otherwise 1..kMaxK.
int current_halo() { return std::max(0, std::min(g_tune.halo, kMaxK)); }

// Per-launch timing of tiled sweeps (fg_profile_enable / fg_profile_collect).
struct ProfRec {
  hipEvent_t start, stop;
  double bytes;
};
thread_local bool g_prof_on = false;     // events around tiled launches
thread_local bool g_prof_xhist = false;  // exchange-wait histogram
// Checks of a pending halo value before a wait expires (0 = default); set by
// fg_set_wait_limit.
thread_local int g_wait_limit = 0;
thread_local std::vector<ProfRec> g_prof;

int fail(int code, const std::string &msg) {
  g_err = msg;
  return code;
}

#define FG_HIP(x)                                                                \
  do {                                                                           \
    hipError_t e_ = (x);                                                         \
    if (e_ != hipSuccess)                                                        \
      return fail(FG_EHIP, std::string(#x " failed: ") + hipGetErrorString(e_)); \
  } while (0)

// Step table of one pass: sqrt((s0 + |i-1|*s1) + |j-1|*s2) in float, in this
// summation order (reference fastgeodis_cpu.cpp:220-231).
void table3d(float s0, float s1, float s2, float ld[9]) {
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) {
      float v = s0;
      v += (float)std::abs(i - 1) * s1;
      v += (float)std::abs(j - 1) * s2;
      ld[i * 3 + j] = std::sqrt(v);
    }
}

void table2d(float ld[9]) {  // {sqrt2, 1, sqrt2} (reference fastgeodis_cpu.cpp:67)
  const float r2 = std::sqrt(2.0f);
  const float row[3] = {r2, 1.0f, r2};
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) ld[i * 3 + j] = row[j];
}

int ceil_div(long long a, long long b) { return (int)((a + b - 1) / b); }

// One unsigned transform to run.
struct Xform {
  const float *img;   // native (C, D, H, W) or (C, H, W)
  const float *imgT;  // transposed (C, W, H, D) or (C, W, H)
  float *d;           // native layout
  float *dT;          // transposed scratch
  int C, D, H, W;
  bool is2d;
  float lg;
  float e1[3][9];  // per pass: D, H, W (2D: [1] rows pass, [2] columns pass)
  bool lamb1, fast;
  int iters;
  int it = 0;  // the iteration being recorded
  bool small = false;  // runs in one workgroup (small_call_kernel)
  bool xst;  // this iteration's H-backward sweep writes dT directly (no transpose before the W pass)
  bool xsa = false;  // this iteration's W-backward sweep writes d directly (no transpose after the W pass)
  // The first sweep initialises the distance from the mask (init_mode 1: v*m,
  // 2: v*(1-m)) instead of reading it; set only when that sweep is tiled.
  int init_mode = 0;
  const float *init_src = nullptr;
  float init_v = 0.f;
  // Transpose back after the last iteration: the first transform of a group
  // (signed pair, GSF stages) combines the group's distances (fin_kind) into
  // fin_dst; the other members (fin_member) contribute their dT only.
  int fin_kind = XK_COPY;
  bool fin_member = false;
  const float *fin_src[3] = {nullptr, nullptr, nullptr};
  float *fin_dst[4] = {nullptr, nullptr, nullptr, nullptr};
  float fin_v = 0.f, fin_theta = 0.f;
};

// The pass of a transform's first sweep: rows (1) in 2D, D (0) in 3D.
int first_pass(const Xform &x) { return x.is2d ? 1 : 0; }

// Tiled plan for one sweep plane.
struct Plan {
  int NW, R;
  bool comm;  // one more wave that performs the halo exchanges
  int P;  // slab ring size of the kernel that runs this plan
  int K;  // halo depth actually used: the requested depth rounded up to a multiple of P
  int nTB, nTE, TB, TE;
  bool ok;
};

struct Shape {
  int NW, R;
  int P12, P34;  // slab ring size for 1-2 / 3-4 image channels (prefetch distance P - 1)
  bool comm;     // plus kCommWaves waves that perform the halo exchanges
};
// Workgroup shapes with compiled kernels: index 0 serves 2D row sweeps
// (one row); the others tile 3D planes (selected by fg_tuning.shape).
constexpr Shape kShapes[] = {{1, 1, kRowHaloStep, kRowHaloStep, false},  {4, 8, 2, 2, false},  {8, 4, 3, 2, false},
                             {16, 2, 3, 3, false}, {8, 4, 5, 2, false},  {16, 2, 5, 3, false},
                             {8, 4, 5, 2, true},   {8, 2, 5, 3, false}};
constexpr int kNumShapes = 8;
constexpr int kAutoShape = 5;  // fastest on 512^2 planes: 16 x 2 with the deepest ring that keeps K = 5
// 16-row windows (8 x 2, K = 5): with the automatic shape and halo, a pass
// runs on them when its planes are 3D with 1-2 channels, have several tiles
// along B, and all their 16-row tiles are resident at one per compute unit
// (see Runner::pass_shape).  The 32-row windows leave compute units idle on
// such planes, and a step's time goes with a window's rows.  Planes of one
// tile along B take a deep halo on the 32-row windows instead, and so do
// those with lamb = 1 that reach K = 15 there.  Whole calls at iter 2, 16-row
// against 32-row windows at their best halo, us: 128 x 256 x 256 lamb 1 1651 /
// 1744, lamb 0.5 1964 / 2358, 2 channels 2373 / 3043; 256^3 lamb 1 2020 / 2134;
// 128^3 lamb 1 1044 / 1024 (K = 15), lamb 0.5 1226 / 1315; 20 x 120 x 140 lamb 1
// 780 / 704 (two passes of one tile along B or K = 15).  Passes whose 16-row
// tiles exceed the device ran slower on them (40 x 400 x 400 lamb 1 2234 / 2019).
constexpr int kSmallPlaneShape = 7;
thread_local int g_shape = kAutoShape;

// Sets this thread's shape for one pass and restores it on every way out.
struct ShapeScope {
  int saved;
  explicit ShapeScope(int shape) : saved(g_shape) { g_shape = shape; }
  ~ShapeScope() { g_shape = saved; }
};

Plan plan_fixed(int nB, int nE, int Kreq, int C, int shape = -1) {
  Plan p{};
  p.ok = false;
  const Shape s = nB == 1 ? kShapes[0] : kShapes[shape >= 0 ? shape : g_shape];
  p.NW = s.NW;
  p.R = s.R;
  p.comm = s.comm && C <= 2;  // exchange-wave kernels exist for 1-2 channels; 3-4 run the plain 8 x 4
  const int P = C <= 2 ? s.P12 : s.P34;
  p.P = P;
  const int K = ((Kreq + P - 1) / P) * P;
  p.K = K;
  const int WR = s.NW * s.R;
  if (nE <= 62) {
    p.nTE = 1;
    p.TE = nE;
  } else {
    const int cap = 64 - 2 * K;
    if (cap < 1) return p;
    p.nTE = ceil_div(nE, cap);
    p.TE = ceil_div(nE, p.nTE);
  }
  if (nB <= WR) {
    p.nTB = 1;
    p.TB = nB;
  } else {
    const int cap = WR - 2 * K;
    if (cap < 1) return p;
    p.nTB = ceil_div(nB, cap);
    p.TB = ceil_div(nB, p.nTB);
  }
  p.ok = true;
  return p;
}

// Tiles that a plan counts on: one 3D tile a compute unit, of rows as many
// workgroups as a unit serves at halo depth K, and never more than a workgroup
// cap (max_groups) allows in one launch.
struct TileBudget {
  int cus, max_groups;
  long long of(int nB, int K) const {
    const long long n = nB == 1 ? (long long)cus * row_groups_per_cu(K) : cus;
    return max_groups > 0 ? std::min<long long>(n, max_groups) : n;
  }
};

// Plan of one sweep plane.  Kreq > 0: that halo depth, rounded up to a
// multiple of the slab ring (a row whose tiles would not all be resident at
// that depth takes the deepest at which they are, in a 3D volume one whose
// entries fit the exchange buffer of the requested depth).  Kreq == 0 (automatic):
// the deepest halo (fewest exchanges) whose tiles still fit the budget, as
// every tile waits for its neighbours at each exchange; if even the shallowest
// halo, which has the fewest tiles, needs more, that one.
Plan plan_plane(int nB, int nE, int Kreq, int C, const TileBudget &budget, bool is2d) {
  if (Kreq > 0) {
    const Plan p = plan_fixed(nB, nE, Kreq, C);
    if (nB > 1 || p.nTE <= 2 * budget.cus) return p;
    for (int K = p.K - p.P; K > 0; K -= p.P) {
      const Plan q = plan_fixed(nB, nE, K, C);
      if ((q.nTE <= 2 * budget.cus || K == p.P) && (is2d || q.nTE * q.TE <= p.nTE * p.TE)) return q;
    }
    return p;
  }
  const Plan first = plan_fixed(nB, nE, 1, C);
  Plan best = first;
  for (int K = first.P; K <= kMaxK; K += first.P) {
    const Plan q = plan_fixed(nB, nE, K, C);
    if (!q.ok) break;
    if ((long long)q.nTB * q.nTE > budget.of(nB, K)) continue;
    best = q;
  }
  return best;
}

// (nB, nE) of each pass's sweep plane: 0 = D, 1 = H (2D: rows), 2 = W (2D: columns)
void pass_plane(const Xform &x, int pass, int &nA, int &nB, int &nE) {
  if (x.is2d) {
    nB = 1;
    if (pass == 1) { nA = x.H; nE = x.W; }
    else if (pass == 2) { nA = x.W; nE = x.H; }
    else { nA = 1; nE = x.W; }
    return;
  }
  if (pass == 0) { nA = x.D; nB = x.H; nE = x.W; }
  else if (pass == 1) { nA = x.H; nB = x.D; nE = x.W; }
  else { nA = x.W; nB = x.H; nE = x.D; }
}

template <int NW, int R, int P, int CT, bool L1, bool FA, int XS = 0, bool IN = false, bool CM = false>
const void *kernel_ptr() {
  return reinterpret_cast<const void *>(&sweep_tiled_kernel<NW, R, P, CT, L1, FA, XS, IN, CM>);
}

// lamb1 implies fast (l_grad == 1 and l_eucl*LD == +0 are non-negative).
// Only the channel counts a (shape, ring) pair serves are instantiated.
template <int NW, int R, int P, int CT, int XS = 0, bool IN = false, bool CM = false>
const void *pick_variant(bool lamb1, bool fast) {
  if (lamb1) return kernel_ptr<NW, R, P, CT, true, true, XS, IN, CM>();
  return fast ? kernel_ptr<NW, R, P, CT, false, true, XS, IN, CM>()
              : kernel_ptr<NW, R, P, CT, false, false, XS, IN, CM>();
}

template <int NW, int R, int P, int CT>
const void *pick_variant_init(bool lamb1, bool fast, bool init) {
  return init ? pick_variant<NW, R, P, CT, 0, true>(lamb1, fast) : pick_variant<NW, R, P, CT>(lamb1, fast);
}

// Kernels of the 8 x 4 shape with an exchange wave (ring 5, 1-2 channels).
const void *pick_comm_kernel(int C, bool lamb1, bool fast, int xs, bool init) {
  if (xs == 2) return nullptr;
  if (C == 1) {
    if (xs == 1) return pick_variant<8, 4, 5, 1, 1, false, true>(lamb1, fast);
    return init ? pick_variant<8, 4, 5, 1, 0, true, true>(lamb1, fast)
                : pick_variant<8, 4, 5, 1, 0, false, true>(lamb1, fast);
  }
  if (C == 2) {
    if (xs == 1) return pick_variant<8, 4, 5, 2, 1, false, true>(lamb1, fast);
    return init ? pick_variant<8, 4, 5, 2, 0, true, true>(lamb1, fast)
                : pick_variant<8, 4, 5, 2, 0, false, true>(lamb1, fast);
  }
  return nullptr;
}

template <int NW, int R, int P, int CLO, int CHI>
const void *pick_kernel_nr(int C, bool lamb1, bool fast, bool init) {
  if constexpr (CLO <= 1 && 1 <= CHI)
    if (C == 1) return pick_variant_init<NW, R, P, 1>(lamb1, fast, init);
  if constexpr (CLO <= 2 && 2 <= CHI)
    if (C == 2) return pick_variant_init<NW, R, P, 2>(lamb1, fast, init);
  if constexpr (CLO <= 3 && 3 <= CHI)
    if (C == 3) return pick_variant_init<NW, R, P, 3>(lamb1, fast, init);
  if constexpr (CLO <= 4 && 4 <= CHI)
    if (C == 4) return pick_variant_init<NW, R, P, 4>(lamb1, fast, init);
  return nullptr;
}

// The one-row kernel of halo depth K (1-4 channels, every output form and
// initialisation), or null.
template <int K>
const void *pick_row_variant(bool lamb1, bool fast) {
  if (lamb1) return reinterpret_cast<const void *>(&row_sweep_kernel<K, true, true>);
  return fast ? reinterpret_cast<const void *>(&row_sweep_kernel<K, false, true>)
              : reinterpret_cast<const void *>(&row_sweep_kernel<K, false, false>);
}

template <int MC>
const void *pick_row_wave(bool lamb1, bool fast) {
  if (lamb1) return reinterpret_cast<const void *>(&row_wave_kernel<MC, true, true>);
  return fast ? reinterpret_cast<const void *>(&row_wave_kernel<MC, false, true>)
              : reinterpret_cast<const void *>(&row_wave_kernel<MC, false, false>);
}

// wave: 0, or the most channels of a launch on the one-wave form
const void *pick_row_kernel(int K, bool lamb1, bool fast, int wave) {
  switch (wave) {
    case 1: return pick_row_wave<1>(lamb1, fast);
    case 2: return pick_row_wave<2>(lamb1, fast);
    case 3: return pick_row_wave<3>(lamb1, fast);
    case 4: return pick_row_wave<4>(lamb1, fast);
    default: break;
  }
  switch (K) {
    case 6: return pick_row_variant<6>(lamb1, fast);
    case 12: return pick_row_variant<12>(lamb1, fast);
    case 18: return pick_row_variant<18>(lamb1, fast);
    case 24: return pick_row_variant<24>(lamb1, fast);
    case 30: return pick_row_variant<30>(lamb1, fast);
    default: return nullptr;
  }
}

template <int CT>
const void *pick_small_variant(bool lamb1, bool fast) {
  if (lamb1) return reinterpret_cast<const void *>(&small_call_kernel<CT, true, true>);
  return fast ? reinterpret_cast<const void *>(&small_call_kernel<CT, false, true>)
              : reinterpret_cast<const void *>(&small_call_kernel<CT, false, false>);
}
const void *pick_small_kernel(int C, bool lamb1, bool fast) {
  switch (C) {
    case 1: return pick_small_variant<1>(lamb1, fast);
    case 2: return pick_small_variant<2>(lamb1, fast);
    case 3: return pick_small_variant<3>(lamb1, fast);
    default: return nullptr;
  }
}

// The kernel compiled for exactly this (NW, R, P) and channel count, or null.
// xs selects the output form (0 own layout, 1 B contiguous, 2 A contiguous).
// B-contiguous kernels exist for the 5-slice-ring 3D shapes with 1-2 channels
// (16 x 2: one; two would exceed the LDS), A-contiguous ones for the same
// shapes with 1 channel.
constexpr int kXstMaxC = 2;
constexpr int kXsaMaxC = 1;
constexpr int kXsaMaxK = kRunSlots - kRunLen + 1;
const void *pick_kernel(int NW, int R, int P, int C, bool lamb1, bool fast, int xs = 0, bool init = false,
                        bool comm = false) {
  if (xs && init) return nullptr;
  if (comm) return (NW == 8 && R == 4 && P == 5) ? pick_comm_kernel(C, lamb1, fast, xs, init) : nullptr;
  if (xs == 1) {
    if (NW == 8 && R == 4 && P == 5 && C == 1) return pick_variant<8, 4, 5, 1, 1>(lamb1, fast);
    if (NW == 8 && R == 4 && P == 5 && C == 2) return pick_variant<8, 4, 5, 2, 1>(lamb1, fast);
    if (NW == 16 && R == 2 && P == 5 && C == 1) return pick_variant<16, 2, 5, 1, 1>(lamb1, fast);
    if (NW == 8 && R == 2 && P == 5 && C == 1) return pick_variant<8, 2, 5, 1, 1>(lamb1, fast);
    if (NW == 8 && R == 2 && P == 5 && C == 2) return pick_variant<8, 2, 5, 2, 1>(lamb1, fast);
    return nullptr;
  }
  if (xs == 2) {
    if (NW == 8 && R == 4 && P == 5 && C == 1) return pick_variant<8, 4, 5, 1, 2>(lamb1, fast);
    if (NW == 16 && R == 2 && P == 5 && C == 1) return pick_variant<16, 2, 5, 1, 2>(lamb1, fast);
    if (NW == 8 && R == 2 && P == 5 && C == 1) return pick_variant<8, 2, 5, 1, 2>(lamb1, fast);
    return nullptr;
  }
#define FG_S(nw, r, p, clo, chi) \
  if (NW == nw && R == r && P == p && C >= clo && C <= chi) return pick_kernel_nr<nw, r, p, clo, chi>(C, lamb1, fast, init);
  FG_S(4, 8, 2, 1, 4)
  FG_S(8, 4, 3, 1, 2)
  FG_S(8, 4, 5, 1, 2)
  FG_S(16, 2, 5, 1, 2)
  FG_S(8, 4, 2, 3, 4)
  FG_S(16, 2, 3, 1, 4)
  FG_S(8, 2, 5, 1, 2)
  FG_S(8, 2, 3, 3, 4)
#undef FG_S
  return nullptr;
}

// Workspace layout helper: carves 256-byte aligned regions.
struct Carver {
  char *base;
  size_t cap, used = 0;
  bool dry;
  Carver(void *b, size_t c, bool dry_run) : base((char *)b), cap(c), dry(dry_run) {}
  void *take(size_t bytes) {
    used = (used + 255) & ~(size_t)255;
    void *p = dry ? nullptr : base + used;
    used += bytes;
    return p;
  }
  bool fits() const { return used <= cap; }
};

// Recorded launch.  Descriptor arrays live in one host blob that is copied to
// the workspace once per call, before any launch is issued.
struct Cmd {
  enum Type { TILED, SLICE, XPOSE, EW, SMALL } type;
  size_t lds = 0;  // dynamic LDS bytes
  SmallDescs small_few{};
  const void *kern = nullptr;
  int grid = 0, block = 0;
  size_t off = 0;  // descriptor offset in the blob
  int ndesc = 0;
  int K = 0;
  unsigned tag_base = 0;
  SliceDesc slice{};  // SLICE: descriptor by value
  int a = 0, aq = 0;
  double alg_bytes = 0;  // TILED: algorithmic HBM bytes of the launch
  // launches of one descriptor pass it by value (no blob entry)
  bool by_value = false;
  SweepDesc sweep1{};
  XposeDesc xpose1{};
  EwDesc ew1{};
};

struct Recorder {
  std::vector<unsigned char> blob;
  std::vector<std::pair<std::string, size_t>> seen;  // identical arrays share storage
  std::vector<Cmd> cmds;

  size_t put(const void *p, size_t bytes) {
    std::string key((const char *)p, bytes);
    for (auto &s : seen)
      if (s.first == key) return s.second;
    size_t off = (blob.size() + 255) & ~(size_t)255;
    blob.resize(off + bytes);
    std::memcpy(blob.data() + off, p, bytes);
    seen.emplace_back(std::move(key), off);
    return off;
  }
};

struct Device {
  int id = -1;
  int cus = 0;
};

int query_device(Device &dev) {
  int id = 0;
  FG_HIP(hipGetDevice(&id));
  int cus = 0;
  FG_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, id));
  dev.id = id;
  dev.cus = cus;
  return FG_OK;
}

// The tiled sweep needs all workgroups of a launch resident at once.  Its
// grid never exceeds the occupancy limit (coresident_groups), so on its own
// every workgroup starts; but two such launches running together (calls on
// different streams) could each hold part of the device and wait on
// workgroups that cannot start.  Calls that launch tiled sweeps are therefore
// ordered per device: the host lock covers a whole replay, and a call on a
// different stream than the previous one first waits for that call's end.
// (Plain launches: the cooperative launch API adds ~15 us per launch.)
//
// The same per-device state holds the status word: one int in pinned,
// host-mapped, coherent host memory that every launch of the device may set
// (system-scope store) when a bounded wait expires or a launch is refused.
// Nothing clears it on the device; the next call on the device (or
// fg_status) reads and clears it from the host without synchronising, so an
// expiry is reported at the latest by the call after the one it happened in.
//
// Descriptor blobs reach the device through pinned staging slots (a ring per
// device): the copy is asynchronous, and a slot is reused only after the
// event recorded behind its last copy has completed.
struct StageSlot {
  unsigned char *host = nullptr;
  size_t cap = 0;
  hipEvent_t copied{};
  bool has_event = false;
};
constexpr int kStageSlots = 8;

// Scratch of the no-allocation entry point (fg_geodesic3d_f32_noalloc): one
// static device array per device, held from the library's load on that device
// until the process ends.  Bytes [0, 256) hold that entry point's status word
// while the device has no pinned status word; the rest is its workspace.
// Host code uses the address from hipGetSymbolAddress, never the name.
constexpr size_t kNoAllocScratchBytes = size_t(256) << 20;
constexpr size_t kNoAllocStatusBytes = 256;

struct DeviceState {
  std::mutex m;  // held for a whole replay
  bool has = false;
  hipStream_t last{};
  hipEvent_t done{};
  int *status_host = nullptr;  // pinned word written by kernels
  int *status_dev = nullptr;   // its device address
  std::atomic<int> injected{0};  // set from the host (fg_inject_status)
  StageSlot stage[kStageSlots];
  int next_slot = 0;
  unsigned char *scratch = nullptr;  // device address of the no-allocation scratch (per device)
};

std::mutex g_reg_m;
std::map<int, std::unique_ptr<DeviceState>> g_reg;

DeviceState &device_state(int id) {
  std::lock_guard<std::mutex> g(g_reg_m);
  auto &slot = g_reg[id];
  if (!slot) slot.reset(new DeviceState());
  return *slot;
}

// Allocates the device's status word on first use (the device is current).
int ensure_status_word(DeviceState &s) {
  std::lock_guard<std::mutex> g(s.m);
  if (s.status_host) return FG_OK;
  void *h = nullptr;
  FG_HIP(hipHostMalloc(&h, 256, hipHostMallocMapped | hipHostMallocCoherent));
  std::memset(h, 0, 256);
  void *d = nullptr;
  hipError_t e = hipHostGetDevicePointer(&d, h, 0);
  if (e != hipSuccess) {
    (void)hipHostFree(h);
    return fail(FG_EHIP, std::string("hipHostGetDevicePointer: ") + hipGetErrorString(e));
  }
  s.status_host = (int *)h;
  s.status_dev = (int *)d;
  return FG_OK;
}

// Reads and clears the device's pending status (no synchronisation).
int take_status(DeviceState &s) {
  int v = s.injected.exchange(0);
  if (s.status_host) {
    const int w = __atomic_exchange_n(s.status_host, 0, __ATOMIC_SEQ_CST);
    if (v == 0) v = w;
  }
  return v;
}

int status_error(int st, const char *when) {
  if (st == FG_OK) return FG_OK;
  if (st == FG_EWATCHDOG)
    return fail(FG_EWATCHDOG, std::string(when) +
                                  ": a tile's bounded halo wait expired (another persistent kernel may have held "
                                  "compute units); the results of that call are invalid");
  if (st == FG_EINVAL)
    return fail(FG_EHIP, std::string(when) +
                             ": a sweep launch was refused (halo depth not a multiple of its ring, a one-row "
                             "kernel on a plane of several rows, or a native-layout output on a plane of one "
                             "tile row)");
  return fail(FG_EHIP, std::string(when) + ": device status " + std::to_string(st));
}

// Holds a device's order for one replay; on every way out (errors included)
// marks the end of what the replay enqueued on its stream.
struct OrderedReplay {
  DeviceState *ord = nullptr;
  hipStream_t stream{};
  std::unique_lock<std::mutex> lock;
  // order: the replay contains persistent sweeps and joins the device order;
  // create: the order's event may be created here (not for callers that
  // allocate nothing, which then join only an existing order)
  int begin(DeviceState &o, hipStream_t s, bool order, bool create = true) {
    lock = std::unique_lock<std::mutex>(o.m);
    if (!order || (!o.has && !create)) return FG_OK;
    if (!o.has) {
      FG_HIP(hipEventCreateWithFlags(&o.done, hipEventDisableTiming));
      o.has = true;
    } else if (o.last != s) {
      FG_HIP(hipStreamWaitEvent(s, o.done, 0));
    }
    o.last = s;
    ord = &o;
    stream = s;
    return FG_OK;
  }
  ~OrderedReplay() {
    if (ord) (void)hipEventRecord(ord->done, stream);
  }
};

// Copies `bytes` of `src` to `dst` on `stream` through a pinned staging slot
// of the device (the device's lock is held by the caller).
int stage_copy(DeviceState &s, void *dst, const void *src, size_t bytes, hipStream_t stream) {
  StageSlot &sl = s.stage[s.next_slot];
  s.next_slot = (s.next_slot + 1) % kStageSlots;
  if (sl.has_event) FG_HIP(hipEventSynchronize(sl.copied));
  if (sl.cap < bytes) {
    if (sl.host) FG_HIP(hipHostFree(sl.host));
    sl.host = nullptr;
    sl.cap = 0;
    const size_t cap = std::max<size_t>(bytes, 64 << 10);
    void *h = nullptr;
    FG_HIP(hipHostMalloc(&h, cap, hipHostMallocDefault));
    sl.host = (unsigned char *)h;
    sl.cap = cap;
  }
  if (!sl.has_event) {
    FG_HIP(hipEventCreateWithFlags(&sl.copied, hipEventDisableTiming));
    sl.has_event = true;
  }
  std::memcpy(sl.host, src, bytes);
  FG_HIP(hipMemcpyAsync(dst, sl.host, bytes, hipMemcpyHostToDevice, stream));
  FG_HIP(hipEventRecord(sl.copied, stream));
  return FG_OK;
}

// Occupancy-limited number of co-resident workgroups per kernel (cached per
// host thread and device).
int coresident_groups(const void *kern, int threads, const Device &dev, long long &cap) {
  struct Entry { const void *k; int dev; long long cap; };
  thread_local std::vector<Entry> cache;
  for (auto &e : cache)
    if (e.k == kern && e.dev == dev.id) { cap = e.cap; return FG_OK; }
  int per_cu = 0;
  FG_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, threads, 0));
  cap = (long long)per_cu * dev.cus;
  cache.push_back({kern, dev.id, cap});
  return FG_OK;
}

// Address of the exchange-wait histogram on device `dev` (the device is current).
int exchange_histogram_impl(int dev, unsigned **out);
inline int exchange_histogram(int dev, unsigned **out) { return exchange_histogram_impl(dev, out); }

// Executable graphs of repeated launch sequences.  A replay whose sequence of
// launches (kernel, grid and block of each, in order) repeats on a host
// thread and device runs as one hipGraphLaunch of a cached graph whose kernel
// nodes (a chain) get this call's arguments; the first occurrence of a
// sequence launches directly, the second builds the graph.  Graphs hold
// kernel nodes only (no memset or copy nodes).
thread_local bool g_graph_on = true;

struct GraphEntry {
  std::thread::id thread;
  uint64_t key = 0;
  int dev = -1;
  hipGraph_t graph{};
  hipGraphExec_t exec{};
  std::vector<hipGraphNode_t> nodes;
  uint64_t last_use = 0;
};
std::mutex g_graph_m;
std::vector<std::unique_ptr<GraphEntry>> g_graph_list;  // every thread's entries
thread_local std::vector<std::pair<uint64_t, int>> g_graph_seen;  // sequences seen once (key, device)
thread_local uint64_t g_graph_clock = 0;
constexpr int kGraphsPerThread = 8;

void destroy_graph(GraphEntry &e) {
  if (e.exec) (void)hipGraphExecDestroy(e.exec);
  if (e.graph) (void)hipGraphDestroy(e.graph);
  e.exec = nullptr;
  e.graph = nullptr;
}

struct SweepJob {
  Xform *x;
  int pass;
  int K;   // halo depth of this plane's plan (> 0)
  int xs;  // output form (SweepDesc::dxo)
};

// Row launches of more tiles than this a compute unit run the one-wave form.
// Front and producers / one wave, ms a call: 32 RGB 1024^2 GSF iter 4 (2560
// tiles) 31.4 / 20.0, 64 of 512^2 (832) 1.31 / 1.18; below the line a
// 1252 x 1292 GSF (324 tiles at K = 24) 1.3 / 2.1.  (One-wave tiles were the
// only form once and took 20.0 and 1.22 there: above the line nothing is
// gained, below it the front wave's shorter chain is.)  The one-wave form's
// tiles leave the layout change to transposes: storing the other layout
// themselves (runs of K elements a lane) they took 28.8 ms on the first.
constexpr int kRowWaveTiles = 3;

// What the sweeps of one launch share.  Row sweeps (row()) of any channel
// count, output form and initialisation share a kernel: C, xs and in are 0.
struct SweepGroup {
  int NW, R, P, K, C;
  bool l1, fa;
  int xs;
  bool in, cm;
  int wave;  // rows on the one-wave form: the most channels of a transform
  bool row() const { return NW == 1; }
  int threads() const { return row() ? (wave ? 64 : kRowThreads) : (NW + (cm ? kCommWaves : 0)) * 64; }
  const void *kernel() const {
    return row() ? pick_row_kernel(K, l1, fa, wave) : pick_kernel(NW, R, P, C, l1, fa, xs, in, cm);
  }
  bool operator==(const SweepGroup &o) const {
    return NW == o.NW && R == o.R && P == o.P && K == o.K && C == o.C && l1 == o.l1 && fa == o.fa && xs == o.xs &&
           in == o.in && cm == o.cm && wave == o.wave;
  }
};

struct Runner {
  Device dev;
  int K;
  int engine;
  int max_groups;
  size_t halo_cap;  // entries
  unsigned tag_base = 0;
  Recorder rec;

  bool no_graph = false;  // replay the launches directly (sequences that do not repeat)

  TileBudget budget() const { return {dev.cus, max_groups}; }

  void fill_desc(const Xform &x, int pass, int dir, SweepDesc &s, int xs = 0) {
    std::memset(&s, 0, sizeof s);
    if (x.init_mode && x.it == 0 && pass == first_pass(x) && dir > 0) {
      s.init_src = x.init_src;
      s.init_v = x.init_v;
      s.init_mode = x.init_mode;
    }
    const long long N = (long long)x.D * x.H * x.W;
    s.C = x.C;
    s.cs = N;
    s.dir = dir;
    s.lg = x.lg;
    pass_plane(x, pass, s.nA, s.nB, s.nE);
    if (x.is2d) {
      if (pass == 2) { s.img = x.imgT; s.d = x.dT; s.sA = x.H; }   // transposed (W, H)
      else { s.img = x.img; s.d = x.d; s.sA = x.W; }                 // native (H, W)
      s.sB = 0;
    } else if (pass == 0) {
      s.img = x.img; s.d = x.d; s.sA = (long long)x.H * x.W; s.sB = x.W;
    } else if (pass == 1) {
      s.img = x.img; s.d = x.d; s.sA = x.W; s.sB = (long long)x.H * x.W;
    } else {
      s.img = x.imgT; s.d = x.dT; s.sA = (long long)x.H * x.D; s.sB = x.D;
    }
    for (int k = 0; k < 9; ++k) s.e1[k] = x.e1[pass][k];
    if (xs == 1) {  // H pass (A = H, B = D, E = W) written as (W, H, D)
      s.dxo = x.dT;
      s.sXe = (long long)s.nA * s.nB;
      s.sXa = s.nB;
    } else if (xs == 2 && x.is2d) {  // rows (A = H, E = W) written as (W, H), columns as (H, W)
      s.dxo = pass == 1 ? x.dT : x.d;
      s.sXe = s.nA;
      s.sXa = 1;
      s.sXb = 0;
    } else if (xs == 2) {  // W pass (A = W, B = H, E = D) written as (D, H, W)
      s.dxo = x.d;
      s.sXe = (long long)x.H * x.W;
      s.sXb = x.W;
    }
  }

  // Whether the H-backward sweep of this transform can write the transposed
  // layout itself: 3D, tiled engine, a B-contiguous kernel for its channel count
  // on the thread's shape, and every output offset within 32 bits.  The pass may
  // still run on 16-row windows, and the choice is made again when it is
  // recorded; with the automatic shape two channels never get here (16 x 2 has
  // no such kernel for them), and their distance is transposed.
  bool xstore_candidate(const Xform &x) {
    if (x.is2d) return row_xsa_candidate(x, 1);
    if (engine == 0 || x.C > kXstMaxC) return false;
    int nA, nB, nE;
    pass_plane(x, 1, nA, nB, nE);
    if (nA <= 1 || nB <= 1) return false;
    const Plan p = plan_plane(nB, nE, K, x.C, budget(), x.is2d);
    if (!p.ok || !pick_kernel(p.NW, p.R, p.P, x.C, x.lamb1, x.fast, 1, false, p.comm)) return false;
    if ((long long)x.D * x.H * x.W * 4 >= 0xFFFFFFF0ll) return false;
    return slice_offsets_fit(x, 1);
  }

  // Whether the W-backward sweep of this transform may write the native
  // layout itself (the launch then also needs a plan of several tile rows
  // and an A-contiguous kernel for its shape, checked when it is recorded):
  // 3D, tiled engine, one channel, output offsets within 32 bits, and not
  // the last iteration of a transform whose result leaves through a
  // combining transpose (signed and GSF epilogues).
  bool xsa_candidate(const Xform &x) {
    if (x.it == x.iters - 1 && (x.fin_member || x.fin_kind != XK_COPY)) return false;
    if (x.is2d) return row_xsa_candidate(x, 2);
    if (engine == 0 || x.C > kXsaMaxC) return false;
    int nA, nB, nE;
    pass_plane(x, 2, nA, nB, nE);
    if (nA <= 1 || nB <= 1) return false;
    if ((long long)x.D * x.H * x.W * 4 >= 0xFFFFFFF0ll) return false;
    return slice_offsets_fit(x, 2);
  }

  // 2D: whether the backward sweep of rows (pass 1) may write the column
  // layout, or that of columns (pass 2) the native layout, itself; the launch
  // must also run the front-and-producers form (decided when it is recorded).
  // The output, like the input, is addressed with 32-bit offsets within 2^31
  // bytes.
  bool row_xsa_candidate(const Xform &x, int pass) {
    if (engine == 0 || x.C > 4) return false;
    int nA, nB, nE;
    pass_plane(x, pass, nA, nB, nE);
    if (nA <= 1) return false;
    return slice_offsets_fit(x, 1) && slice_offsets_fit(x, 2);
  }

  // The tiled kernel addresses elements of a slice with 32-bit byte offsets
  // from the slice start (buffer resources with a range of 0xFFFFFFF0 bytes);
  // the one-row kernel addresses the whole array with them, within 2^31
  // bytes including 32 slices of margin past its end.
  bool slice_offsets_fit(const Xform &x, int pass) {
    SweepDesc s;
    fill_desc(x, pass, 1, s);
    const long long span = ((long long)(s.nB - 1) * s.sB + s.nE) * 4;
    if (s.nB == 1 && (long long)(s.nA + 32) * s.sA * 4 > (1ll << 31)) return false;
    return span < 0xFFFFFFF0ll;
  }

  void record_per_slice(const Xform &x, int pass, int dir) {
    SweepDesc s;
    fill_desc(x, pass, dir, s);
    Cmd c;
    c.type = Cmd::SLICE;
    SliceDesc &sd = c.slice;
    sd.img = s.img; sd.d = s.d; sd.cs = s.cs; sd.sA = s.sA; sd.sB = s.sB;
    sd.nB = s.nB; sd.nE = s.nE; sd.C = s.C; sd.lg = s.lg;
    for (int k = 0; k < 9; ++k) sd.e1[k] = s.e1[k];
    c.grid = ceil_div((long long)s.nB * s.nE, 256);
    c.block = 256;
    if (dir > 0) {
      for (int a = 1; a < s.nA; ++a) { c.a = a; c.aq = a - 1; rec.cmds.push_back(c); }
    } else {
      for (int a = s.nA - 2; a >= 0; --a) { c.a = a; c.aq = a + 1; rec.cmds.push_back(c); }
    }
  }

  int record_tiled(std::vector<SweepJob> &jobs, int dir, const SweepGroup &g) {
    std::vector<SweepDesc> descs;
    long long halo_used = 0;
    int tiles = 0, max_blocks = 0;
    double alg = 0;
    for (auto &j : jobs) {
      SweepDesc s;
      fill_desc(*j.x, j.pass, dir, s, j.xs);
      alg += (double)(s.nA - 1) * s.nB * s.nE * (4.0 * s.C + 8.0);
      Plan p = plan_fixed(s.nB, s.nE, j.K, s.C);
      if (!p.ok || p.NW != g.NW || p.R != g.R || p.P != g.P || p.comm != g.cm || p.K % g.P != 0 || p.K != g.K)
        return fail(FG_EINVAL, "internal: sweep plan does not match the selected kernel");
      s.nTB = p.nTB; s.nTE = p.nTE; s.TB = p.TB; s.TE = p.TE;
      s.tile0 = tiles;
      s.halo0 = halo_used;
      const int nt = p.nTB * p.nTE;
      tiles += nt;
      halo_used += (long long)nt * 2 * p.TB * p.TE;
      max_blocks = std::max(max_blocks, (s.nA - 1) / p.K + 1);
      descs.push_back(s);
    }
    if (descs.empty()) return FG_OK;
    if ((size_t)halo_used > halo_cap) return fail(FG_EWORKSPACE, "workspace too small for the sweep plan");
    if ((unsigned long long)tag_base + max_blocks + 2 >= 0x7fffffffull) {
      record_zero_halo();
      tag_base = 0;
    }
    Cmd c;
    c.type = Cmd::TILED;
    c.kern = g.kernel();
    if (!c.kern) return fail(FG_EINVAL, "no tiled kernel for this shape");
    c.grid = tiles;
    c.block = g.threads();
    c.ndesc = (int)descs.size();
    if (c.ndesc == 1) {
      c.by_value = true;
      c.sweep1 = descs[0];
    } else {
      c.off = rec.put(descs.data(), descs.size() * sizeof(SweepDesc));
    }
    c.K = g.K;
    c.tag_base = tag_base;
    c.alg_bytes = alg;
    rec.cmds.push_back(c);
    tag_base += (unsigned)max_blocks + 1;
    return FG_OK;
  }

  void record_zero_halo() {
    if (halo_cap == 0) return;
    EwDesc e{};
    e.kind = EW_FILL_U64;
    e.u64 = nullptr;  // patched at replay: the halo base
    e.nelem = (long long)halo_cap;
    record_ew({e});
  }

  void record_ew(const std::vector<EwDesc> &in) {
    std::vector<EwDesc> ds = in;
    long long blocks = 0;
    for (auto &e : ds) {
      e.blk0 = blocks;
      blocks += ceil_div(e.nelem, (long long)kEwPerBlock);
    }
    if (blocks == 0) return;
    Cmd c;
    c.type = Cmd::EW;
    c.ndesc = (int)ds.size();
    if (c.ndesc == 1) {
      c.by_value = true;
      c.ew1 = ds[0];
    } else {
      c.off = rec.put(ds.data(), ds.size() * sizeof(EwDesc));
    }
    c.block = 256;
    c.grid = (int)blocks;  // < 2^31: 2^41 elements would not fit any device
    rec.cmds.push_back(c);
  }

  void record_xpose(const std::vector<XposeDesc> &in) {
    std::vector<XposeDesc> ds = in;
    int tiles = 0;
    for (auto &x : ds) {
      x.tiles_dw = ceil_div(x.D, kXT) * ceil_div(x.W, kXT);
      x.tile0 = tiles;
      tiles += x.C * x.H * x.tiles_dw;
    }
    if (tiles == 0) return;
    Cmd c;
    c.type = Cmd::XPOSE;
    c.ndesc = (int)ds.size();
    if (c.ndesc == 1) {
      c.by_value = true;
      c.xpose1 = ds[0];
    } else {
      c.off = rec.put(ds.data(), ds.size() * sizeof(XposeDesc));
    }
    c.grid = tiles;
    c.block = 256;
    rec.cmds.push_back(c);
  }

  static XposeDesc xd(const float *src, float *dst, int C, int D, int H, int W) {
    XposeDesc x{};
    x.src = src; x.dst = dst; x.C = C; x.D = D; x.H = H; x.W = W;
    return x;
  }
  static void native_dims(const Xform &x, int &D, int &H, int &W) {
    if (x.is2d) { D = x.H; H = 1; W = x.W; }  // (H, W) seen as (D'=H, H'=1, W'=W)
    else { D = x.D; H = x.H; W = x.W; }
  }

  // Whether a transform's sweeps of this pass run on the tiled engine.
  bool tiled_eligible(const Xform &x, int pass) {
    int nA, nB, nE;
    pass_plane(x, pass, nA, nB, nE);
    if (nA <= 1 || engine == 0 || x.C > 4) return false;
    return plan_plane(nB, nE, K, x.C, budget(), x.is2d).ok && slice_offsets_fit(x, pass);
  }

  // Halo depth of each transform's plane in this pass.  Requested depths
  // apply as they are, but for rows that are too many for them (plan_plane;
  // 2D rows at K = 30, 4 own lanes of 64, whose tiles together are not resident
  // take K = 24: 48 images of 400 x 500 iter 2 at a requested 30 3.56 ms in
  // launches of 512 tiles, 2.46 on the one-wave form, 0.98 at 24).
  // Automatic: a lone plane takes the deepest halo whose
  // tiles fit one per CU (idle CUs cost nothing, and fewer exchanges shorten
  // the sweep).  Planes that share the pass (batches, the halves of a signed
  // or GSF call) are planned together: the deepest halo at which all their
  // tiles still fit the device, and the shallowest one when none does, as a
  // deeper halo then only adds window arithmetic (a 32 x 64 window computes
  // 1.7 x its own tile at K = 5 and 3.9 x at K = 10; a 64-lane row 1.23 x at
  // K = 6 and 16 x at K = 30).  3D tiles fill a CU each; several row
  // workgroups share one (row_groups_per_cu).
  std::vector<int> pass_halos(const std::vector<Xform *> &active, int pass) {
    std::vector<int> ks(active.size(), 0);
    std::vector<int> rows, planes;  // automatic 2D rows and 3D planes
    long long deepest = 0;          // tiles of 2D rows at the deepest requested depth
    for (size_t i = 0; i < active.size(); ++i) {
      int nA, nB, nE;
      pass_plane(*active[i], pass, nA, nB, nE);
      if (!tiled_eligible(*active[i], pass)) continue;
      const Plan p = plan_plane(nB, nE, K, active[i]->C, budget(), active[i]->is2d);
      ks[i] = p.K;
      if (K > 0 && active[i]->is2d && p.K == kMaxK) deepest += p.nTE;
      if (K == 0) (nB > 1 ? planes : rows).push_back((int)i);
    }
    if (deepest > 2 * dev.cus)
      for (size_t i = 0; i < active.size(); ++i)
        if (active[i]->is2d && ks[i] == kMaxK) ks[i] -= kRowHaloStep;
    if (rows.size() > 1) share_halo(active, pass, rows, ks);
    if (planes.size() > 1) share_halo(active, pass, planes, ks);
    return ks;
  }

  // One halo depth per slab-ring length for the planes `idx` (channel
  // classes use different rings), all rows or all 3D planes: the deepest whose
  // tiles fit the device, else the shallowest.
  void share_halo(const std::vector<Xform *> &active, int pass, const std::vector<int> &idx, std::vector<int> &ks) {
    auto ring = [&](int i) {
      int nA, nB, nE;
      pass_plane(*active[i], pass, nA, nB, nE);
      return plan_fixed(nB, nE, 1, active[i]->C).P;
    };
    std::vector<int> rings;
    for (int i : idx)
      if (std::find(rings.begin(), rings.end(), ring(i)) == rings.end()) rings.push_back(ring(i));
    for (int P : rings) {
      int best = P;
      for (int k = P; k <= kMaxK; k += P) {
        long long tiles = 0, fits = 0;
        bool ok = true;
        for (int i : idx) {
          if (ring(i) != P) continue;
          int nA, nB, nE;
          pass_plane(*active[i], pass, nA, nB, nE);
          fits = budget().of(nB, k);
          const Plan q = plan_fixed(nB, nE, k, active[i]->C);
          if (!q.ok) { ok = false; break; }
          tiles += (long long)q.nTB * q.nTE;
        }
        if (!ok) break;
        if (tiles <= fits) best = k;
      }
      for (int i : idx)
        if (ring(i) == P) ks[i] = best;
    }
  }

  // The 3D workgroup shape of a pass: the tuned one, or with the automatic
  // shape the 16-row windows when the pass's planes qualify (kSmallPlaneShape).
  int pass_shape(const std::vector<Xform *> &active, int pass) {
    if (g_tune.shape != 0 || K != 0 || engine == 0) return g_shape;  // tuned shape or halo
    const std::vector<int> ks = pass_halos(active, pass);  // with the 32-row windows
    long long t16 = 0;
    for (size_t i = 0; i < active.size(); ++i) {
      const Xform *x = active[i];
      int nA, nB, nE;
      pass_plane(*x, pass, nA, nB, nE);
      if (nA <= 1) continue;
      if (x->is2d || nB <= 1 || x->C > 2 || ks[i] == 0 || (x->lamb1 && ks[i] >= 15)) return g_shape;
      const Plan a = plan_fixed(nB, nE, ks[i], x->C);
      const Plan b = plan_fixed(nB, nE, 5, x->C, kSmallPlaneShape);
      if (!a.ok || !b.ok || a.nTB == 1) return g_shape;
      t16 += (long long)b.nTB * b.nTE;
    }
    return (t16 > 0 && t16 <= budget().of(2, 5)) ? kSmallPlaneShape : g_shape;
  }

  // Whether a row launch runs the one-wave form: one of more tiles than
  // kRowWaveTiles a compute unit, or with a plane (its widest) of more tiles
  // than workgroups with a front and producers are resident at once (512 at
  // K >= 24; a requested depth can ask for it).
  int row_wave(long long tiles, long long widest, int K, bool lamb1, bool fast, bool &wave) const {
    if (max_groups > 0) tiles = std::min<long long>(tiles, max_groups);  // a launch has no more
    wave = tiles > (long long)kRowWaveTiles * dev.cus;
    if (wave || widest <= dev.cus) return FG_OK;  // (at least one a compute unit is resident)
    const void *kern = pick_row_kernel(K, lamb1, fast, 0);
    long long cap = 0;
    if (!kern) return fail(FG_EINVAL, "no row kernel for this depth");
    if (const int rc = coresident_groups(kern, kRowThreads, dev, cap)) return rc;
    wave = widest > cap;
    return FG_OK;
  }

  // Which of a pass's transforms run on it (the most channels of its launch, or
  // 0): the rows that share a launch (same depth, lamb class and fold) are
  // counted together, once for the pass (a
  // count per transform made the recording of a batch quadratic: 1024 images of
  // 150 x 170 12.3 ms a call instead of 6.9).
  int row_waves(const std::vector<Xform *> &active, int pass, const std::vector<int> &ks, std::vector<char> &wave) const {
    struct Launch { long long tiles = 0, widest = 0; int channels = 0; bool wave = false; };
    Launch launch[kMaxK + 1][2][2];
    wave.assign(active.size(), 0);
    for (size_t i = 0; i < active.size(); ++i) {
      const Xform *x = active[i];
      int nA, nB, nE;
      pass_plane(*x, pass, nA, nB, nE);
      if (nB > 1 || nA <= 1 || ks[i] == 0) continue;
      wave[i] = 1;  // a row
      Launch &l = launch[ks[i]][x->lamb1][x->fast];
      const int n = plan_fixed(nB, nE, ks[i], x->C).nTE;
      l.tiles += n;
      l.widest = std::max<long long>(l.widest, n);
      l.channels = std::max(l.channels, x->C);
    }
    for (int k = 1; k <= kMaxK; ++k)
      for (int lamb1 = 0; lamb1 < 2; ++lamb1)
        for (int fast = 0; fast < 2; ++fast) {
          Launch &l = launch[k][lamb1][fast];
          if (l.tiles == 0) continue;
          if (const int rc = row_wave(l.tiles, l.widest, k, lamb1, fast, l.wave)) return rc;
        }
    for (size_t i = 0; i < active.size(); ++i) {
      if (!wave[i]) continue;
      const Launch &l = launch[ks[i]][active[i]->lamb1][active[i]->fast];
      wave[i] = l.wave ? (char)l.channels : 0;
    }
    return FG_OK;
  }

  // Record one pass (forward then backward) for the active transforms.
  int sweep_pass(std::vector<Xform *> &active, int pass) {
    ShapeScope shape_scope(pass_shape(active, pass));
    const std::vector<int> ks = pass_halos(active, pass);
    std::vector<char> wave;
    if (const int rc = row_waves(active, pass, ks, wave)) return rc;
    for (int dir : {+1, -1}) {
      std::vector<std::pair<SweepGroup, std::vector<SweepJob>>> groups;
      for (size_t i = 0; i < active.size(); ++i) {
        Xform *x = active[i];
        int nA, nB, nE;
        pass_plane(*x, pass, nA, nB, nE);
        if (nA <= 1) continue;
        const bool in = x->init_mode && x->it == 0 && pass == first_pass(*x) && dir > 0;
        if (ks[i] == 0) {
          if (in) return fail(FG_EINVAL, "internal: an initialising sweep was planned on the per-slice engine");
          record_per_slice(*x, pass, dir);
          if (pass == 1) x->xst = false;  // its output stays in the native layout
          if (pass == 2) x->xsa = false;  // its output stays in the W pass layout
          continue;
        }
        const Plan p = plan_fixed(nB, nE, ks[i], x->C);
        // Backward sweeps that write the next layout themselves: 2D row tiles
        // store every block from LDS in either layout (the one-wave form only
        // its own); 3D tiles stage the own
        // rows of a tile of several along B, and the slices of one block
        // beyond a run.  Otherwise the distance moves between layouts through
        // a transpose.
        int xs = 0;
        if (pass == 1 && dir < 0 && x->xst) {
          // (the pass may run on a shape without a B-contiguous kernel)
          if (x->is2d && !wave[i]) xs = 2;
          else if (p.NW > 1 && pick_kernel(p.NW, p.R, p.P, x->C, x->lamb1, x->fast, 1, in, p.comm)) xs = 1;
          else x->xst = false;
        }
        if (pass == 2 && dir < 0 && x->xsa) {
          if ((x->is2d && !wave[i]) ||
              (p.nTB > 1 && p.K <= kXsaMaxK && pick_kernel(p.NW, p.R, p.P, x->C, x->lamb1, x->fast, 2, in, p.comm)))
            xs = 2;
          else
            x->xsa = false;
        }
        const bool row = p.NW == 1;
        const SweepGroup key{p.NW, p.R, p.P, p.K, row ? 0 : x->C, x->lamb1, x->fast, row ? 0 : xs, row ? false : in,
                             p.comm, wave[i]};
        auto g = std::find_if(groups.begin(), groups.end(), [&](const auto &q) { return q.first == key; });
        if (g == groups.end()) g = groups.insert(groups.end(), {key, {}});
        g->second.push_back({x, pass, p.K, xs});
      }
      for (auto &g : groups) {
        int rc = record_group(g.second, dir, g.first);
        if (rc) return rc;
      }
    }
    return FG_OK;
  }

  // A group is split into launches whose tiles can all be co-resident.  For the
  // automatic 3D shape that is one workgroup a compute unit, as its kernels take
  // more than 64 registers (65-97); two in turn finish sooner than two at once
  // (clicks in eight volumes 10.27 / 11.21 ms).
  int record_group(std::vector<SweepJob> &jobs, int dir, const SweepGroup &g) {
    const void *kern = g.kernel();
    if (!kern) return fail(FG_EINVAL, "no tiled kernel for this shape");
    long long cap = 0;
    int rc = coresident_groups(kern, g.threads(), dev, cap);
    if (rc) return rc;
    if (max_groups > 0) cap = std::min<long long>(cap, max_groups);
    // A launch lasts as long as its longest sweep: pack planes of similar
    // step counts together (longest first).
    std::stable_sort(jobs.begin(), jobs.end(), [](const SweepJob &u, const SweepJob &v) {
      int au, bu, eu, av, bv, ev;
      pass_plane(*u.x, u.pass, au, bu, eu);
      pass_plane(*v.x, v.pass, av, bv, ev);
      return au > av;
    });
    std::vector<SweepJob> chunk;
    long long tiles = 0;
    for (auto &j : jobs) {
      int nA, nB, nE;
      pass_plane(*j.x, j.pass, nA, nB, nE);
      Plan p = plan_fixed(nB, nE, j.K, j.x->C);
      const long long nt = (long long)p.nTB * p.nTE;
      if (nt > cap && g.wave > j.x->C) {  // its own channel count's kernel holds more tiles
        std::vector<SweepJob> alone{j};
        SweepGroup own = g;
        own.wave = j.x->C;
        if ((rc = record_group(alone, dir, own))) return rc;
        continue;
      }
      if (nt > cap) {  // one plane alone cannot be co-resident: per-slice engine
        if (j.x->init_mode && j.x->it == 0 && j.pass == first_pass(*j.x) && dir > 0)
          return fail(FG_EINVAL, "internal: an initialising sweep was planned on the per-slice engine");
        record_per_slice(*j.x, j.pass, dir);
        if (j.pass == 1) j.x->xst = false;  // its output stays in the native layout
        if (j.pass == 2) j.x->xsa = false;  // its output stays in the W pass layout
        continue;
      }
      if (tiles + nt > cap) {
        if ((rc = record_tiled(chunk, dir, g))) return rc;
        chunk.clear();
        tiles = 0;
      }
      chunk.push_back(j);
      tiles += nt;
    }
    if (!chunk.empty()) return record_tiled(chunk, dir, g);
    return FG_OK;
  }

  // The transposes around a W pass: into its layout (unless the H pass's
  // backward sweep wrote it) and, once the W pass is recorded, back (unless
  // its backward sweep wrote the native layout), the last iteration's
  // carrying the group's epilogue (members of a group contribute through its
  // first one).
  void w_pass_to(const std::vector<Xform *> &active, std::vector<XposeDesc> &to) {
    for (auto *x : active) {
      int D, H, W;
      native_dims(*x, D, H, W);
      if (!x->xst) to.push_back(xd(x->d, x->dT, 1, D, H, W));
    }
  }
  void w_pass_back(const std::vector<Xform *> &active, std::vector<XposeDesc> &back) {
    for (auto *x : active) {
      if (x->xsa) continue;
      int D, H, W;
      native_dims(*x, D, H, W);
      const bool last = x->it == x->iters - 1;
      if (last && x->fin_member) continue;  // part of its group's combined transpose
      XposeDesc b = xd(x->dT, x->d, 1, W, H, D);
      if (last && x->fin_kind != XK_COPY) {
        b.kind = x->fin_kind;
        b.src2 = x->fin_src[0];
        b.src3 = x->fin_src[1];
        b.src4 = x->fin_src[2];
        b.dst = x->fin_dst[0];
        b.dst2 = x->fin_dst[1];
        b.dst3 = x->fin_dst[2];
        b.dst4 = x->fin_dst[3];
        b.v = x->fin_v;
        b.theta = x->fin_theta;
      }
      back.push_back(b);
    }
  }

  // The small transforms of a run: one workgroup each, one launch per kernel
  // and LDS size class, then the epilogues of their groups.
  int record_small(std::vector<Xform> &xs) {
    struct Launch { const void *kern; size_t lds; std::vector<SmallDesc> descs; };
    std::vector<Launch> launches;
    std::vector<Xform *> mine;
    for (auto &x : xs) {
      if (!x.small) continue;
      const bool flip = x.fin_member || x.fin_kind != XK_COPY;  // an epilogue reads the W pass layout
      SmallDesc d{};
      d.img = x.img;
      d.src = x.init_mode ? x.init_src : x.d;
      d.out = flip ? x.dT : x.d;
      d.C = x.C; d.H = x.H; d.W = x.W; d.iters = x.iters;
      d.init_mode = x.init_mode;
      d.flip = flip;
      d.v = x.init_v;
      d.lg = x.lg;
      d.e1s = x.e1[1][3];
      d.e1c = x.e1[1][4];
      const void *kern = pick_small_kernel(x.C, x.lamb1, x.fast);
      if (!kern) return fail(FG_EINVAL, "internal: no kernel for a small image");
      const size_t lds = small_lds(x.C, x.H, x.W);
      // (workgroups of one launch reserve the same LDS: a class per 32 KB)
      auto l = std::find_if(launches.begin(), launches.end(),
                            [&](const Launch &q) { return q.kern == kern && (q.lds >> 15) == (lds >> 15); });
      if (l == launches.end()) l = launches.insert(launches.end(), {kern, lds, {}});
      l->lds = std::max(l->lds, lds);
      l->descs.push_back(d);
      x.it = x.iters - 1;
      x.xsa = !flip;
      mine.push_back(&x);
    }
    for (auto &l : launches) {
      Cmd c;
      c.type = Cmd::SMALL;
      c.kern = l.kern;
      c.lds = l.lds;
      c.grid = c.ndesc = (int)l.descs.size();
      c.block = kSmallWaves * 64;
      if (c.ndesc <= kSmallByValue) {
        c.by_value = true;
        std::copy(l.descs.begin(), l.descs.end(), c.small_few.d);
      } else {
        c.off = rec.put(l.descs.data(), l.descs.size() * sizeof(SmallDesc));
      }
      rec.cmds.push_back(c);
    }
    std::vector<XposeDesc> back;
    w_pass_back(mine, back);
    record_xpose(back);
    return FG_OK;
  }

  int record_run(std::vector<Xform> &xs) {
    if (const int rc = record_small(xs)) return rc;
    int max_it = 0;
    for (auto &x : xs)
      if (!x.small) max_it = std::max(max_it, x.iters);
    for (int it = 0; it < max_it; ++it) {
      std::vector<Xform *> active;
      for (auto &x : xs)
        if (!x.small && x.iters > it) {
          x.it = it;
          active.push_back(&x);
        }
      int rc;
      for (auto *x : active) {
        x->xst = xstore_candidate(*x);
        x->xsa = xsa_candidate(*x);
      }
      if ((rc = sweep_pass(active, 0))) return rc;
      if ((rc = sweep_pass(active, 1))) return rc;
      std::vector<XposeDesc> to, back;
      w_pass_to(active, to);
      record_xpose(to);
      if ((rc = sweep_pass(active, 2))) return rc;
      w_pass_back(active, back);
      record_xpose(back);
    }
    return FG_OK;
  }

  // Whether the first sweep of x runs on the tiled engine whatever halo depth
  // and shape its pass is planned with: the plane's tiles at the requested
  // depth's plan, or automatically at the shallowest halo, which has the
  // fewest, are co-resident (and within a workgroup cap).
  // Deeper halos and 16-row windows are planned only where their tiles fit
  // the budget, which is within both.
  int first_sweep_tiled(const Xform &x, bool &tiled) {
    tiled = false;
    const int pass = first_pass(x);
    if (x.iters <= 0 || !tiled_eligible(x, pass)) return FG_OK;
    int nA, nB, nE;
    pass_plane(x, pass, nA, nB, nE);
    const Plan p = K > 0 ? plan_plane(nB, nE, K, x.C, budget(), x.is2d) : plan_fixed(nB, nE, 1, x.C);
    if (!p.ok) return FG_OK;
    bool wave = false;
    int rc = FG_OK;
    if (nB == 1 && (rc = row_wave(p.nTE, p.nTE, p.K, x.lamb1, x.fast, wave))) return rc;
    const SweepGroup g{p.NW, p.R, p.P, p.K, x.C, x.lamb1, x.fast, 0, true, p.comm, wave ? x.C : 0};
    const void *kern = g.kernel();
    if (!kern) return FG_OK;
    long long cap = 0;
    rc = coresident_groups(kern, g.threads(), dev, cap);
    if (rc) return rc;
    if (max_groups > 0) cap = std::min<long long>(cap, max_groups);
    tiled = (long long)p.nTB * p.nTE <= cap;
    return FG_OK;
  }

  // status: the status word the launches write; no_alloc: create nothing on the
  // host side (no pinned staging, no events) and pass every descriptor by value
  int replay(hipStream_t stream, unsigned char *blob_dev, size_t blob_cap, unsigned long long *halo, int *status,
             bool no_alloc) {
    if (rec.blob.size() > blob_cap) return fail(FG_EWORKSPACE, "descriptor area too small");
    // the halo base is only known now: patch fill descriptors
    for (auto &c : rec.cmds)
      if (c.type == Cmd::EW) {
        EwDesc *ds = c.by_value ? &c.ew1 : reinterpret_cast<EwDesc *>(rec.blob.data() + c.off);
        for (int i = 0; i < c.ndesc; ++i)
          if (ds[i].kind == EW_FILL_U64) ds[i].u64 = halo;
      }
    bool tiled = false;
    for (auto &c : rec.cmds) tiled = tiled || c.type == Cmd::TILED;
    DeviceState &ds = device_state(dev.id);
    if (no_alloc && !rec.blob.empty())
      return fail(FG_EINVAL, "internal: a launch of this call needs a descriptor array");
    OrderedReplay order;
    int rc = order.begin(ds, stream, tiled, !no_alloc);
    if (rc) return rc;
    if (!rec.blob.empty() && (rc = stage_copy(ds, blob_dev, rec.blob.data(), rec.blob.size(), stream))) return rc;
    // the kernel expires a wait when a check finds a halo value pending after spin re-polls
    const int spin = g_wait_limit > 0 ? g_wait_limit - 1 : (1 << 21);

    // Argument values of every launch (the arrays point into `vals`, which
    // outlives the launches and graph updates below).
    struct Vals {
      const void *dp;
      int ndesc, k, sp, a, aq;
      unsigned tb;
    };
    const size_t n = rec.cmds.size();
    std::vector<Vals> vals(n);
    std::vector<std::array<void *, 9>> args(n);
    // exchange-wait histogram of this device while profiling
    unsigned *xhist = nullptr;
    if (g_prof_xhist && (rc = exchange_histogram(dev.id, &xhist))) return rc;
    std::vector<const void *> funcs(n);
    bool slice = false;
    for (size_t i = 0; i < n; ++i) {
      Cmd &c = rec.cmds[i];
      Vals &v = vals[i];
      v.ndesc = c.ndesc;
      auto &a = args[i];
      switch (c.type) {
        case Cmd::TILED:
          v.dp = c.by_value ? nullptr : blob_dev + c.off;
          v.k = c.K;
          v.sp = spin;
          v.tb = c.tag_base;
          a = {(void *)&v.dp, &v.ndesc, (void *)&c.sweep1, &v.k, &v.tb, (void *)&halo, (void *)&status, &v.sp,
               (void *)&xhist};
          funcs[i] = c.kern;
          break;
        case Cmd::SLICE:
          v.a = c.a;
          v.aq = c.aq;
          a = {(void *)&c.slice, &v.a, &v.aq, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
          funcs[i] = reinterpret_cast<const void *>(&slice_kernel);
          slice = true;
          break;
        case Cmd::XPOSE:
          v.dp = c.by_value ? nullptr : blob_dev + c.off;
          a = {(void *)&v.dp, &v.ndesc, (void *)&c.xpose1, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
          funcs[i] = reinterpret_cast<const void *>(&xpose_kernel);
          break;
        case Cmd::SMALL:
          v.dp = c.by_value ? nullptr : blob_dev + c.off;
          a = {(void *)&v.dp, (void *)&c.small_few, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
          funcs[i] = c.kern;
          break;
        case Cmd::EW:
          v.dp = c.by_value ? nullptr : blob_dev + c.off;
          a = {(void *)&v.dp, &v.ndesc, (void *)&c.ew1, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
          funcs[i] = reinterpret_cast<const void *>(&ew_kernel);
          break;
      }
    }
    auto node_params = [&](size_t i) {
      hipKernelNodeParams p{};
      p.func = const_cast<void *>(funcs[i]);
      p.gridDim = dim3(rec.cmds[i].grid);
      p.blockDim = dim3(rec.cmds[i].block);
      p.sharedMemBytes = (unsigned)rec.cmds[i].lds;
      p.kernelParams = args[i].data();
      p.extra = nullptr;
      return p;
    };

    // graph replay of a repeated sequence (not while profiling per launch, not
    // for the per-slice engine's hundreds of launches, never without allocating)
    if (g_graph_on && !no_graph && !g_prof_on && !g_prof_xhist && !slice && !no_alloc && n >= 2) {
      uint64_t key = 1469598103934665603ull;
      auto mix = [&](uint64_t x) { key = (key ^ x) * 1099511628211ull; };
      for (size_t i = 0; i < n; ++i) {
        mix((uint64_t)(uintptr_t)funcs[i]);
        mix((uint64_t)rec.cmds[i].grid);
        mix((uint64_t)rec.cmds[i].block);
        mix((uint64_t)rec.cmds[i].lds);
      }
      GraphEntry *e = nullptr;
      {
        std::lock_guard<std::mutex> g(g_graph_m);
        for (auto &p : g_graph_list)
          if (p->thread == std::this_thread::get_id() && p->key == key && p->dev == dev.id && p->nodes.size() == n)
            e = p.get();
      }
      bool fresh = false;
      if (!e) {
        auto seen = std::find(g_graph_seen.begin(), g_graph_seen.end(), std::make_pair(key, dev.id));
        if (seen == g_graph_seen.end()) {
          g_graph_seen.push_back({key, dev.id});
          if (g_graph_seen.size() > 32) g_graph_seen.erase(g_graph_seen.begin());
        } else {
          std::unique_ptr<GraphEntry> ne(new GraphEntry());
          ne->thread = std::this_thread::get_id();
          ne->key = key;
          ne->dev = dev.id;
          bool ok = hipGraphCreate(&ne->graph, 0) == hipSuccess;
          for (size_t i = 0; ok && i < n; ++i) {
            hipGraphNode_t node{};
            const hipKernelNodeParams p = node_params(i);
            ok = hipGraphAddKernelNode(&node, ne->graph, i ? &ne->nodes.back() : nullptr, i ? 1 : 0, &p) ==
                 hipSuccess;
            if (ok) ne->nodes.push_back(node);
          }
          ok = ok && hipGraphInstantiate(&ne->exec, ne->graph, nullptr, nullptr, 0) == hipSuccess;
          if (ok) {
            std::lock_guard<std::mutex> g(g_graph_m);
            // keep at most kGraphsPerThread entries per thread: drop the least recently used
            std::vector<GraphEntry *> mine;
            for (auto &p : g_graph_list)
              if (p->thread == ne->thread) mine.push_back(p.get());
            if ((int)mine.size() >= kGraphsPerThread) {
              GraphEntry *old = *std::min_element(mine.begin(), mine.end(), [](GraphEntry *x, GraphEntry *y) {
                return x->last_use < y->last_use;
              });
              destroy_graph(*old);
              g_graph_list.erase(std::find_if(g_graph_list.begin(), g_graph_list.end(),
                                              [&](const std::unique_ptr<GraphEntry> &p) { return p.get() == old; }));
            }
            e = ne.get();
            g_graph_list.push_back(std::move(ne));
            fresh = true;
          } else {
            destroy_graph(*ne);
            (void)hipGetLastError();
          }
        }
      }
      if (e) {
        e->last_use = ++g_graph_clock;
        bool ok = true;
        for (size_t i = 0; ok && !fresh && i < n; ++i) {
          const hipKernelNodeParams p = node_params(i);
          ok = hipGraphExecKernelNodeSetParams(e->exec, e->nodes[i], &p) == hipSuccess;
        }
        if (ok) {
          FG_HIP(hipGraphLaunch(e->exec, stream));
          return FG_OK;
        }
        (void)hipGetLastError();  // an update failed: launch directly this time
      }
    }

    for (size_t i = 0; i < n; ++i) {
      Cmd &c = rec.cmds[i];
      ProfRec pr{};
      const bool prof = g_prof_on && c.type == Cmd::TILED;
      if (prof) {
        FG_HIP(hipEventCreate(&pr.start));
        FG_HIP(hipEventCreate(&pr.stop));
        FG_HIP(hipEventRecord(pr.start, stream));
      }
      FG_HIP(hipLaunchKernel(funcs[i], dim3(c.grid), dim3(c.block), args[i].data(), c.lds, stream));
      if (prof) {
        FG_HIP(hipEventRecord(pr.stop, stream));
        pr.bytes = c.alg_bytes;
        g_prof.push_back(pr);
      }
    }
    return FG_OK;
  }
};

// ---------------------------------------------------------------------------
// Operation planning shared by the single-call and batched entry points
// ---------------------------------------------------------------------------

struct OpSpec {
  const float *image;
  const float *imageT;  // the image already in the W pass layout (C, W, H, D) / (C, W, H), or null
  const float *mask;
  float *out;
  int C, Cm, D, H, W;
  bool is2d;
  int op;
  int iters;
  float spacing[3];
  float v, lg, le, theta;
};

bool non_negative(float x) { return !std::signbit(x); }

void make_xform(const OpSpec &o, float lg, float le, Xform &x) {
  x.C = o.C; x.D = o.D; x.H = o.H; x.W = o.W; x.is2d = o.is2d; x.lg = lg; x.iters = o.iters;
  float ld[3][9];
  if (o.is2d) {
    table2d(ld[0]);
    table2d(ld[1]);
    table2d(ld[2]);
  } else {
    float sq[3];
    for (int k = 0; k < 3; ++k) sq[k] = o.spacing[k] * o.spacing[k];
    table3d(sq[0], sq[1], sq[2], ld[0]);  // D pass: in-plane (H, W)
    table3d(sq[1], sq[0], sq[2], ld[1]);  // H pass: in-plane (D, W)
    table3d(sq[2], sq[1], sq[0], ld[2]);  // W pass: in-plane (H, D)
  }
  bool fast = non_negative(lg);
  bool e1zero = true;
  for (int p = 0; p < 3; ++p)
    for (int k = 0; k < 9; ++k) {
      x.e1[p][k] = le * ld[p][k];
      fast = fast && non_negative(x.e1[p][k]);
      uint32_t bits;
      std::memcpy(&bits, &x.e1[p][k], 4);
      e1zero = e1zero && bits == 0u;
    }
  x.fast = fast;
  x.lamb1 = (lg == 1.0f) && e1zero;
}

long long vox(const OpSpec &o) { return (long long)o.D * o.H * o.W; }

// Whether an op's transforms can run in one workgroup each: 2D, one channel with
// sides up to kSmallSide or 2-3 channels with sides up to 64, the tiled engine
// and no requested halo depth or workgroup cap.  The one front wave of
// small_call_kernel takes longer per step than row_sweep_kernel's (~60 ns with
// one channel, ~110 with 3, against ~42) but nothing per launch.  us a call at
// iter 2, this kernel / one launch per sweep: 64^2 33 / 73, 128^2 78 / 98,
// 128 x 100 lamb 0.5 87 / 96; 3 channels lamb 0.5: 64^2 57 / 77, 90^2 92 / 82.
bool small_op(const OpSpec &o) {
  const int side = std::max(o.H, o.W);
  return o.is2d && o.iters > 0 && side <= (o.C == 1 ? kSmallSide : 64) && o.C <= 3 && g_tune.engine != 0 &&
         g_tune.halo == 0 && g_tune.max_groups == 0 && small_lds(o.C, o.H, o.W) <= (160u << 10);
}
// They do when all ops of the call can, however many there are: workgroups of
// more than 80 KB (a side of ~96) take a compute unit each, so large batches run
// in rounds of 256, and still take less than their sweeps would, host time
// included.  Calls of n images, this kernel / sweeps, us: 128^2, n = 64 327 /
// 443, 256 990 / 1403, 1024 3916 / 5091; GSF 256 1663 / 3765; 90^2, 1024 3916 /
// 5007; 3 channels of 64^2, 1024 3791 / 5110.  Beside larger images they share
// those launches at no cost of their own (a batch of 48 images and 8 volumes:
// 4735 us, 4896 with its small images in launches of their own).
bool small_ops(const std::vector<OpSpec> &ops) { return std::all_of(ops.begin(), ops.end(), small_op); }

int n_dist(int op) { return op == FG_OP_UNSIGNED ? 1 : (op == FG_OP_SIGNED ? 2 : 4); }

size_t halo_entries_for(const std::vector<OpSpec> &ops, int K) {
  size_t total = 0;
  for (auto &o : ops) {
    Xform x{};
    x.D = o.D; x.H = o.H; x.W = o.W; x.is2d = o.is2d;
    size_t worst = 0;
    for (int p = 0; p < 3; ++p) {
      int nA, nB, nE;
      pass_plane(x, p, nA, nB, nE);
      const bool any = K <= 0 || o.is2d;  // depths the plan may take
      for (int k = (any ? 1 : K); k <= (any ? kMaxK : K); ++k) {
        for (int sh : {g_shape, (g_tune.shape == 0 && K <= 0) ? kSmallPlaneShape : g_shape}) {
          Plan pl = plan_fixed(nB, nE, k, o.C, sh);
          if (!pl.ok) continue;
          worst = std::max(worst, (size_t)pl.nTB * pl.nTE * 2 * pl.TB * pl.TE);
        }
      }
    }
    total += worst * (size_t)n_dist(o.op);
  }
  return total;
}

// Upper bound of the descriptor blob: identical descriptor arrays are stored
// once, and the active set of transforms changes at most once per distinct
// iteration count.
size_t blob_bytes_for(const std::vector<OpSpec> &ops) {
  size_t ntrans = 0, n2d = 0;
  std::vector<int> its;
  for (auto &o : ops) {
    ntrans += n_dist(o.op);
    if (o.is2d) n2d += n_dist(o.op);
    if (std::find(its.begin(), its.end(), o.iters) == its.end()) its.push_back(o.iters);
  }
  const size_t sets = its.size() + 1;
  const size_t nsweep = 2 * 6 * sets;  // (pass, dir) x active sets, x2 for GSF stages
  size_t bytes = 0;
  bytes += nsweep * (ntrans * sizeof(SweepDesc) + 256) * 2;
  bytes += (4 * sets + 2) * (ntrans * sizeof(XposeDesc) + 256) + (ops.size() * sizeof(XposeDesc) + 256);
  bytes += 8 * (ops.size() * sizeof(EwDesc) + 256);
  bytes += 2 * (n2d * (sizeof(SmallDesc) + 256));
  return bytes + 4096;
}

struct Layout {
  unsigned char *blob;
  size_t blob_cap;
  unsigned long long *halo;
  size_t halo_cap;
};

void layout_common(const std::vector<OpSpec> &ops, int K, Layout &L, Carver &cv) {
  L.blob_cap = blob_bytes_for(ops);
  L.blob = (unsigned char *)cv.take(L.blob_cap);
  L.halo_cap = halo_entries_for(ops, K);
  L.halo = (unsigned long long *)cv.take(L.halo_cap * sizeof(unsigned long long) + 8);
}

size_t op_buffers_bytes(const OpSpec &o) {
  const long long N = vox(o);
  const int nd = n_dist(o.op);
  // image transpose (C*N, unless given) + extra distances (nd-1) + transposed distances (nd)
  const size_t floats = (o.imageT ? 0 : (size_t)o.C * N) + (size_t)(nd - 1) * N + (size_t)nd * N;
  return floats * sizeof(float) + 16 * 256;
}

size_t workspace_for(const std::vector<OpSpec> &ops, int K) {
  Layout L{};
  Carver cv(nullptr, 0, true);
  layout_common(ops, K, L, cv);
  for (auto &o : ops) cv.take(op_buffers_bytes(o));
  return ((cv.used + 255) & ~(size_t)255) + 256;
}

int validate(const OpSpec &o) {
  if (!o.image || !o.mask || !o.out) return fail(FG_EINVAL, "null pointer");
  if (o.C < 1 || o.Cm < 1 || o.D < 1 || o.H < 1 || o.W < 1)
    return fail(FG_EINVAL, "extents and channel counts must be >= 1");
  if (o.is2d && o.D != 1) return fail(FG_EINVAL, "2D instance must have D == 1");
  if (o.op < FG_OP_UNSIGNED || o.op > FG_OP_GSF) return fail(FG_EINVAL, "unknown op");
  if (vox(o) * std::max(o.C, o.Cm) >= (1ll << 40)) return fail(FG_EINVAL, "volume too large");
  if (o.H >= (1 << 30) || o.W >= (1 << 30) || o.D >= (1 << 30)) return fail(FG_EINVAL, "extent too large");
  return FG_OK;
}

struct RunOpts {
  bool no_alloc = false;           // create nothing (no pinned status word, staging or events)
  int *fallback_status = nullptr;  // status word to use while the device has no pinned one
};

int run_ops(std::vector<OpSpec> &ops, void *ws, size_t wsb, hipStream_t stream, const RunOpts &opt = RunOpts()) {
  for (auto &o : ops) {
    int rc = validate(o);
    if (rc) return rc;
  }
  const int K = current_halo();
  const size_t need = workspace_for(ops, K);
  if (!ws || wsb < need)
    return fail(FG_EWORKSPACE, "workspace too small: need " + std::to_string(need) + " bytes");
  Layout L{};
  Carver cv(ws, wsb, false);
  layout_common(ops, K, L, cv);

  Runner run{};
  int rc = query_device(run.dev);
  if (rc) return rc;
  // an expiry left by an earlier call on this device is reported here
  DeviceState &dstate = device_state(run.dev.id);
  if (!opt.no_alloc && (rc = ensure_status_word(dstate))) return rc;
  if ((rc = status_error(take_status(dstate), "an earlier call on this device"))) return rc;
  int *status = dstate.status_dev ? dstate.status_dev : opt.fallback_status;
  if (!status) return fail(FG_EINVAL, "internal: no status word");
  run.K = K;
  run.engine = g_tune.engine;
  run.max_groups = g_tune.max_groups;
  run.halo_cap = L.halo_cap;

  struct OpBufs { float *imgT; float *dist[4]; float *dT[4]; };
  std::vector<OpBufs> bufs(ops.size());
  for (size_t i = 0; i < ops.size(); ++i) {
    const OpSpec &o = ops[i];
    const long long N = vox(o);
    const int nd = n_dist(o.op);
    const size_t start = cv.used;
    bufs[i].imgT = o.imageT ? const_cast<float *>(o.imageT) : (float *)cv.take((size_t)o.C * N * sizeof(float));
    bufs[i].dist[0] = o.out;
    for (int k = 1; k < nd; ++k) bufs[i].dist[k] = (float *)cv.take((size_t)N * sizeof(float));
    for (int k = 0; k < nd; ++k) bufs[i].dT[k] = (float *)cv.take((size_t)N * sizeof(float));
    cv.used = start;
    cv.take(op_buffers_bytes(o));
  }
  if (!cv.fits()) return fail(FG_EWORKSPACE, "workspace too small");

  // the halo tags start from zero on every call
  const bool small = small_ops(ops);
  if (!small) run.record_zero_halo();

  // image transposes (once per op)
  {
    std::vector<XposeDesc> xs;
    for (size_t i = 0; i < ops.size(); ++i) {
      const OpSpec &o = ops[i];
      if (o.imageT || small) continue;  // the caller keeps the transposed image; small ones need none
      if (o.is2d) xs.push_back(Runner::xd(o.image, bufs[i].imgT, o.C, o.H, 1, o.W));
      else xs.push_back(Runner::xd(o.image, bufs[i].imgT, o.C, o.D, o.H, o.W));
    }
    run.record_xpose(xs);
  }

  // Stage 1: initialise and transform.  With iterations, a transform's first
  // sweep computes its initialisation from the mask (when that sweep is
  // tiled), mask channels >= 1 get their closed form in one elementwise pass,
  // and each op's epilogue is applied by its last transpose back (signed:
  // D(M) - D(1-M); GSF: the thresholds that initialise stage 2).  Without
  // iterations the elementwise kernels do all of it.
  std::vector<EwDesc> init, chans;
  std::vector<Xform> xs;
  std::vector<char> fused(ops.size(), 0);
  for (size_t i = 0; i < ops.size(); ++i) {
    const OpSpec &o = ops[i];
    const long long N = vox(o);
    fused[i] = o.iters > 0;
    EwDesc e{};
    e.n0 = N;
    e.Cm = o.Cm;
    e.op = o.op;
    e.mask = o.mask;
    e.out = o.out;
    e.v = o.v;
    e.theta = o.theta;
    float lg = o.lg, le = o.le;
    if (o.op == FG_OP_GSF) le = 1 - o.lg;  // reference fastgeodis.cpp:321: 1 - lambda in float
    const int nd = (o.op == FG_OP_UNSIGNED) ? 1 : 2;
    const size_t j0 = xs.size();
    for (int k = 0; k < nd; ++k) {
      Xform x{};
      make_xform(o, lg, le, x);
      x.img = o.image;
      x.imgT = bufs[i].imgT;
      x.d = bufs[i].dist[k];
      x.dT = bufs[i].dT[k];
      xs.push_back(x);
    }
    EwDesc ie = e;
    ie.kind = (o.op == FG_OP_UNSIGNED) ? EW_INIT_UNSIGNED : EW_INIT_SIGNED;
    ie.a = bufs[i].dist[1];
    if (!fused[i]) {
      ie.nelem = N * o.Cm;  // every channel
      init.push_back(ie);
      continue;
    }
    if (o.Cm > 1) {
      EwDesc c = e;
      c.kind = EW_CHANNELS;
      c.nelem = N * (o.Cm - 1);
      chans.push_back(c);
    }
    for (int k = 0; k < nd; ++k) xs[j0 + k].small = small;
    bool tiled = xs[j0].small;
    if (!tiled && (rc = run.first_sweep_tiled(xs[j0], tiled))) return rc;
    if (tiled) {
      for (int k = 0; k < nd; ++k) {
        xs[j0 + k].init_mode = (k == 0) ? 1 : 2;
        xs[j0 + k].init_src = o.mask;
        xs[j0 + k].init_v = o.v;
      }
    } else {
      ie.nelem = N;  // channel 0
      init.push_back(ie);
    }
    if (o.op != FG_OP_UNSIGNED) {
      Xform &x0 = xs[j0];
      x0.fin_kind = (o.op == FG_OP_SIGNED) ? XK_SIGNED : XK_GSF_MID;
      x0.fin_src[0] = xs[j0 + 1].dT;
      x0.fin_dst[0] = o.out;
      if (o.op == FG_OP_GSF)
        for (int k = 1; k < 4; ++k) x0.fin_dst[k] = bufs[i].dist[k];
      x0.fin_v = o.v;
      x0.fin_theta = o.theta;
      xs[j0 + 1].fin_member = true;
    }
  }
  run.record_ew(init);
  run.record_ew(chans);
  if ((rc = run.record_run(xs))) return rc;

  // Stage 2 (GSF): four more transforms from the thresholds.
  std::vector<EwDesc> mid, fin;
  std::vector<Xform> xs2;
  for (size_t i = 0; i < ops.size(); ++i) {
    const OpSpec &o = ops[i];
    const long long N = vox(o);
    EwDesc e{};
    e.n0 = N;
    e.Cm = o.Cm;
    e.op = o.op;
    e.mask = o.mask;
    e.out = o.out;
    e.v = o.v;
    e.theta = o.theta;
    if (o.op == FG_OP_SIGNED && !fused[i]) {
      e.kind = EW_FINAL_SIGNED;
      e.a = bufs[i].dist[1];
      e.nelem = N * o.Cm;
      fin.push_back(e);
    } else if (o.op == FG_OP_GSF) {
      if (!fused[i]) {
        EwDesc m = e;
        m.kind = EW_GSF_MID;
        m.a = bufs[i].dist[1];
        m.b = bufs[i].dist[2];
        m.c2 = bufs[i].dist[3];
        m.nelem = N;
        mid.push_back(m);
        EwDesc f = m;
        f.kind = EW_GSF_FINAL;
        f.nelem = N * o.Cm;
        fin.push_back(f);
      }
      const float le = 1 - o.lg;
      // dist[0] = out: D(1-Me); dist[1]: D(1-Md); dist[2]: D(Md); dist[3]: D(Me)
      const size_t j0 = xs2.size();
      for (int k = 0; k < 4; ++k) {
        Xform x{};
        make_xform(o, o.lg, le, x);
        x.img = o.image;
        x.imgT = bufs[i].imgT;
        x.d = bufs[i].dist[k];
        x.dT = bufs[i].dT[k];
        x.small = small;
        xs2.push_back(x);
      }
      if (fused[i]) {
        Xform &x0 = xs2[j0];
        x0.fin_kind = XK_GSF_FINAL;
        for (int k = 1; k < 4; ++k) {
          x0.fin_src[k - 1] = xs2[j0 + k].dT;
          xs2[j0 + k].fin_member = true;
        }
        x0.fin_dst[0] = o.out;
      }
    }
  }
  run.record_ew(mid);
  if (!xs2.empty() && (rc = run.record_run(xs2))) return rc;
  run.record_ew(fin);
  return run.replay(stream, L.blob, L.blob_cap, L.halo, status, opt.no_alloc);
}

OpSpec spec2d(const float *image, const float *mask, float *out, int C, int Cm, int H, int W, int op,
              int iters, float v, float lg, float le, float theta) {
  OpSpec o{};
  o.image = image; o.mask = mask; o.out = out; o.C = C; o.Cm = Cm; o.D = 1; o.H = H; o.W = W;
  o.is2d = true; o.op = op; o.iters = iters; o.v = v; o.lg = lg; o.le = le; o.theta = theta;
  o.spacing[0] = o.spacing[1] = o.spacing[2] = 1.0f;
  return o;
}

OpSpec spec3d(const float *image, const float *mask, float *out, int C, int Cm, int D, int H, int W,
              const float *spacing, int op, int iters, float v, float lg, float le, float theta) {
  OpSpec o{};
  o.image = image; o.mask = mask; o.out = out; o.C = C; o.Cm = Cm; o.D = D; o.H = H; o.W = W;
  o.is2d = false; o.op = op; o.iters = iters; o.v = v; o.lg = lg; o.le = le; o.theta = theta;
  for (int k = 0; k < 3; ++k) o.spacing[k] = spacing ? spacing[k] : 1.0f;
  return o;
}

int run_single(OpSpec o, void *ws, size_t wsb, void *stream) {
  std::vector<OpSpec> ops{o};
  return run_ops(ops, ws, wsb, (hipStream_t)stream);
}

// ---------------------------------------------------------------------------
// Stepper: transforms that advance one pass pair per step, so that new ones
// join between steps (continuous batching of a serving loop).  Each step
// records, for every active transform, its next pass pair (forward and
// backward sweep) in launches shared with every other transform at that
// pass, plus the transposes around W passes; a transform that has run its
// last W pass leaves with its epilogue applied.  Results equal the same
// transform run alone: a transform computes exactly the launches of its
// plain call, only in the company of others.
// ---------------------------------------------------------------------------

struct StepOp {
  OpSpec o;
  int ticket = 0;
  bool started = false;   // its first step (image transpose, mask channels >= 1) recorded
  int it = 0;             // iteration of its next pass pair
  int pass = 0;           // next pass: 0 D, 1 H, 2 W (2D: 1 rows, 2 columns)
  float *imgT = nullptr;  // the image in the W pass layout
  std::vector<Xform> xs;  // 1 (unsigned) or 2 (signed: D(M), D(1-M))
  size_t halo_entries = 0;
};

struct Stepper {
  int device = -1;
  unsigned long long *halo = nullptr;
  size_t halo_cap = 0;  // entries
  unsigned char *blob = nullptr;
  size_t blob_cap = 0;
  bool halo_clear = false;  // the first step clears the exchange buffer
  unsigned tag_base = 0;
  int next_ticket = 1;
  size_t halo_used = 0;  // entries reserved by the active transforms
  std::vector<StepOp> ops;
};

size_t stepper_blob_bytes(int max_transforms) {
  const size_t n = (size_t)std::max(max_transforms, 1);
  // per step: 3 passes x 2 directions of sweeps, 3 transpose launches, 2 elementwise
  return 6 * (n * sizeof(SweepDesc) + 256) * 2 + 3 * (n * sizeof(XposeDesc) + 256) +
         2 * (n * sizeof(EwDesc) + 256) + 4096;
}

int stepper_runner(const Stepper &st, Runner &run) {
  int rc = query_device(run.dev);
  if (rc) return rc;
  if (run.dev.id != st.device) return fail(FG_EINVAL, "the stepper belongs to another device");
  run.K = current_halo();
  run.engine = g_tune.engine;
  run.max_groups = g_tune.max_groups;
  run.halo_cap = st.halo_cap;
  run.tag_base = st.tag_base;
  run.no_graph = true;
  return FG_OK;
}

int stepper_add(Stepper &st, const OpSpec &o, void *ws, size_t wsb, int *ticket) {
  int rc = validate(o);
  if (rc) return rc;
  if (o.op != FG_OP_UNSIGNED && o.op != FG_OP_SIGNED) return fail(FG_EINVAL, "the stepper runs unsigned and signed transforms");
  if (o.iters < 1) return fail(FG_EINVAL, "the stepper needs iterations >= 1");
  if (!ws || wsb < op_buffers_bytes(o)) return fail(FG_EWORKSPACE, "transform workspace too small");
  Runner run{};
  if ((rc = stepper_runner(st, run))) return rc;
  const size_t hneed = halo_entries_for({o}, run.K);
  if (st.halo_used + hneed > st.halo_cap) return fail(FG_EWORKSPACE, "the stepper's exchange buffer is full");

  StepOp op;
  op.o = o;
  const long long N = vox(o);
  const int nd = n_dist(o.op);
  Carver cv(ws, wsb, false);
  op.imgT = o.imageT ? const_cast<float *>(o.imageT) : (float *)cv.take((size_t)o.C * N * sizeof(float));
  float *dist[2] = {o.out, nd > 1 ? (float *)cv.take((size_t)N * sizeof(float)) : nullptr};
  float *dT[2] = {nullptr, nullptr};
  for (int k = 0; k < nd; ++k) dT[k] = (float *)cv.take((size_t)N * sizeof(float));
  if (!cv.fits()) return fail(FG_EWORKSPACE, "transform workspace too small");
  for (int k = 0; k < nd; ++k) {
    Xform x{};
    make_xform(o, o.lg, o.le, x);
    x.img = o.image;
    x.imgT = op.imgT;
    x.d = dist[k];
    x.dT = dT[k];
    op.xs.push_back(x);
  }
  // the initialisation is computed by the first sweep, which therefore must
  // run on the tiled engine
  bool tiled = false;
  if ((rc = run.first_sweep_tiled(op.xs[0], tiled))) return rc;
  if (!tiled) return fail(FG_EINVAL, "the stepper needs a first sweep on the tiled engine (plane too large)");
  for (int k = 0; k < nd; ++k) {
    op.xs[k].init_mode = (k == 0) ? 1 : 2;
    op.xs[k].init_src = o.mask;
    op.xs[k].init_v = o.v;
  }
  if (o.op == FG_OP_SIGNED) {
    op.xs[0].fin_kind = XK_SIGNED;
    op.xs[0].fin_src[0] = op.xs[1].dT;
    op.xs[0].fin_dst[0] = o.out;
    op.xs[0].fin_v = o.v;
    op.xs[1].fin_member = true;
  }
  op.pass = first_pass(op.xs[0]);
  op.ticket = st.next_ticket++;
  if (st.next_ticket <= 0) st.next_ticket = 1;
  op.halo_entries = hneed;
  st.halo_used += hneed;
  *ticket = op.ticket;
  st.ops.push_back(std::move(op));
  return FG_OK;
}

int stepper_step(Stepper &st, hipStream_t stream, int *done, int cap, int *ndone) {
  *ndone = 0;
  if (st.ops.empty()) return FG_OK;
  Runner run{};
  int rc = stepper_runner(st, run);
  if (rc) return rc;
  DeviceState &dstate = device_state(run.dev.id);
  if ((rc = ensure_status_word(dstate))) return rc;
  if ((rc = status_error(take_status(dstate), "an earlier call on this device"))) return rc;
  if (!st.halo_clear) run.record_zero_halo();

  // first steps: image transposes and mask channels >= 1 (closed form)
  std::vector<XposeDesc> ximg;
  std::vector<EwDesc> chans;
  for (auto &op : st.ops) {
    if (op.started) continue;
    const OpSpec &o = op.o;
    if (!o.imageT) {
      if (o.is2d) ximg.push_back(Runner::xd(o.image, op.imgT, o.C, o.H, 1, o.W));
      else ximg.push_back(Runner::xd(o.image, op.imgT, o.C, o.D, o.H, o.W));
    }
    if (o.Cm > 1) {
      EwDesc c{};
      c.n0 = vox(o);
      c.Cm = o.Cm;
      c.op = o.op;
      c.mask = o.mask;
      c.out = o.out;
      c.v = o.v;
      c.theta = o.theta;
      c.kind = EW_CHANNELS;
      c.nelem = vox(o) * (o.Cm - 1);
      chans.push_back(c);
    }
  }
  run.record_xpose(ximg);
  run.record_ew(chans);

  std::vector<Xform *> act[3];
  for (auto &op : st.ops)
    for (auto &x : op.xs) {
      x.it = op.it;
      act[op.pass].push_back(&x);
    }
  for (auto *x : act[1]) x->xst = run.xstore_candidate(*x);
  for (auto *x : act[2]) x->xsa = run.xsa_candidate(*x);
  std::vector<XposeDesc> to, back;
  run.w_pass_to(act[2], to);
  run.record_xpose(to);
  for (int pass = 0; pass < 3; ++pass)
    if (!act[pass].empty() && (rc = run.sweep_pass(act[pass], pass))) return rc;
  run.w_pass_back(act[2], back);
  run.record_xpose(back);
  if ((rc = run.replay(stream, st.blob, st.blob_cap, st.halo, dstate.status_dev, false))) return rc;
  st.halo_clear = true;
  st.tag_base = run.tag_base;

  // advance; transforms past their last W pass leave
  std::vector<StepOp> keep;
  for (auto &op : st.ops) {
    op.started = true;
    if (op.pass == 2) {
      op.pass = first_pass(op.xs[0]);
      if (++op.it == op.o.iters) {
        if (*ndone < cap) done[(*ndone)++] = op.ticket;
        st.halo_used -= op.halo_entries;
        continue;
      }
    } else {
      ++op.pass;
    }
    keep.push_back(std::move(op));
  }
  st.ops.swap(keep);
  return FG_OK;
}


}  // namespace

static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

// Exchange-wait histogram filled by the sweep kernels while profiling.
static __device__ unsigned xhist_dev[kXHistBuckets];

namespace {

std::mutex g_xhist_m;
std::map<int, unsigned *> g_xhist_ptr;  // device -> address of xhist_dev

int exchange_histogram_impl(int dev, unsigned **out) {
  std::lock_guard<std::mutex> g(g_xhist_m);
  auto it = g_xhist_ptr.find(dev);
  if (it == g_xhist_ptr.end()) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(xhist_dev));
    if (e != hipSuccess || !p) return fail(FG_EHIP, std::string("hipGetSymbolAddress(xhist): ") + hipGetErrorString(e));
    it = g_xhist_ptr.emplace(dev, (unsigned *)p).first;
  }
  *out = it->second;
  return FG_OK;
}

// Device address of this device's scratch array (the device is current),
// looked up once per device.
int noalloc_scratch(DeviceState &ds, unsigned char **out) {
  std::lock_guard<std::mutex> g(ds.m);
  if (!ds.scratch) {
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(FG_EHIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    ds.scratch = (unsigned char *)p;
  }
  *out = ds.scratch;
  return FG_OK;
}

}  // namespace

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------

extern "C" {

int fg_abi_version(void) { return 4; }

const char *fg_last_error(void) { return g_err.c_str(); }

size_t fg_workspace_bytes(int op, int C, int D, int H, int W) {
  OpSpec o{};
  o.op = (op < FG_OP_UNSIGNED || op > FG_OP_GSF) ? FG_OP_GSF : op;
  o.C = std::max(C, 1); o.Cm = 1; o.D = std::max(D, 1); o.H = std::max(H, 1); o.W = std::max(W, 1);
  o.is2d = (D <= 0);
  o.iters = 1;
  std::vector<OpSpec> ops{o};
  return workspace_for(ops, current_halo());
}

int fg_geodesic2d_f32(const float *image, const float *mask, float *out, int C, int Cm, int H, int W,
                      float v, float l_grad, float l_eucl, int iterations, void *workspace,
                      size_t workspace_bytes, void *stream) {
  return run_single(spec2d(image, mask, out, C, Cm, H, W, FG_OP_UNSIGNED, iterations, v, l_grad, l_eucl, 0.f),
                    workspace, workspace_bytes, stream);
}

int fg_geodesic3d_f32(const float *image, const float *mask, float *out, int C, int Cm, int D, int H, int W,
                      const float spacing[3], float v, float l_grad, float l_eucl, int iterations,
                      void *workspace, size_t workspace_bytes, void *stream) {
  if (!spacing) return fail(FG_EINVAL, "spacing must have 3 entries");
  return run_single(
      spec3d(image, mask, out, C, Cm, D, H, W, spacing, FG_OP_UNSIGNED, iterations, v, l_grad, l_eucl, 0.f),
      workspace, workspace_bytes, stream);
}

int fg_signed_geodesic2d_f32(const float *image, const float *mask, float *out, int C, int Cm, int H, int W,
                             float v, float l_grad, float l_eucl, int iterations, void *workspace,
                             size_t workspace_bytes, void *stream) {
  return run_single(spec2d(image, mask, out, C, Cm, H, W, FG_OP_SIGNED, iterations, v, l_grad, l_eucl, 0.f),
                    workspace, workspace_bytes, stream);
}

int fg_signed_geodesic3d_f32(const float *image, const float *mask, float *out, int C, int Cm, int D, int H,
                             int W, const float spacing[3], float v, float l_grad, float l_eucl,
                             int iterations, void *workspace, size_t workspace_bytes, void *stream) {
  if (!spacing) return fail(FG_EINVAL, "spacing must have 3 entries");
  return run_single(
      spec3d(image, mask, out, C, Cm, D, H, W, spacing, FG_OP_SIGNED, iterations, v, l_grad, l_eucl, 0.f),
      workspace, workspace_bytes, stream);
}

int fg_gsf2d_f32(const float *image, const float *mask, float *out, int C, int Cm, int H, int W, float theta,
                 float v, float lambda, int iterations, void *workspace, size_t workspace_bytes,
                 void *stream) {
  return run_single(spec2d(image, mask, out, C, Cm, H, W, FG_OP_GSF, iterations, v, lambda, 0.f, theta),
                    workspace, workspace_bytes, stream);
}

int fg_gsf3d_f32(const float *image, const float *mask, float *out, int C, int Cm, int D, int H, int W,
                 float theta, const float spacing[3], float v, float lambda, int iterations, void *workspace,
                 size_t workspace_bytes, void *stream) {
  if (!spacing) return fail(FG_EINVAL, "spacing must have 3 entries");
  return run_single(
      spec3d(image, mask, out, C, Cm, D, H, W, spacing, FG_OP_GSF, iterations, v, lambda, 0.f, theta),
      workspace, workspace_bytes, stream);
}

int fg_geodesic3d_f32_noalloc(const float *image, const float *mask, float *out, int C, int Cm, int D, int H,
                              int W, const float spacing[3], float v, float l_grad, float l_eucl, int iterations,
                              void *stream) {
  if (!spacing) return fail(FG_EINVAL, "spacing must have 3 entries");
  std::vector<OpSpec> ops{
      spec3d(image, mask, out, C, Cm, D, H, W, spacing, FG_OP_UNSIGNED, iterations, v, l_grad, l_eucl, 0.f)};
  int rc = validate(ops[0]);
  if (rc) return rc;
  const size_t need = workspace_for(ops, current_halo());
  if (need > kNoAllocScratchBytes - kNoAllocStatusBytes)
    return fail(FG_EWORKSPACE, "fg_geodesic3d_f32_noalloc: this volume needs " + std::to_string(need) +
                                   " bytes of scratch; the no-allocation entry point holds " +
                                   std::to_string(kNoAllocScratchBytes - kNoAllocStatusBytes) +
                                   " (use fg_geodesic3d_f32 with a workspace)");
  int id = 0;
  hipError_t e = hipGetDevice(&id);
  if (e != hipSuccess) return fail(FG_EHIP, std::string("hipGetDevice: ") + hipGetErrorString(e));
  DeviceState &ds = device_state(id);
  unsigned char *sp = nullptr;
  if ((rc = noalloc_scratch(ds, &sp))) return rc;
  RunOpts opt;
  opt.no_alloc = true;
  opt.fallback_status = (int *)sp;
  return run_ops(ops, sp + kNoAllocStatusBytes, kNoAllocScratchBytes - kNoAllocStatusBytes, (hipStream_t)stream,
                 opt);
}

size_t fg_noalloc_scratch_bytes(void) { return kNoAllocScratchBytes - kNoAllocStatusBytes; }

static int to_specs(const fg_instance *inst, int n, std::vector<OpSpec> &ops) {
  if (n < 0 || (n > 0 && !inst)) return fail(FG_EINVAL, "bad instance array");
  for (int i = 0; i < n; ++i) {
    const fg_instance &f = inst[i];
    if (f.is2d && f.D != 1) return fail(FG_EINVAL, "2D instance must have D == 1");
    if (f.is2d)
      ops.push_back(spec2d(f.image, f.mask, f.out, f.C, f.Cm, f.H, f.W, f.op, f.iterations, f.v, f.l_grad,
                           f.l_eucl, f.theta));
    else
      ops.push_back(spec3d(f.image, f.mask, f.out, f.C, f.Cm, f.D, f.H, f.W, f.spacing, f.op, f.iterations,
                           f.v, f.l_grad, f.l_eucl, f.theta));
    ops.back().imageT = f.imageT;
  }
  return FG_OK;
}

size_t fg_batch_workspace_bytes(const fg_instance *inst, int n) {
  std::vector<OpSpec> ops;
  if (to_specs(inst, n, ops)) return 0;
  return workspace_for(ops, current_halo());
}

int fg_geodesic_batch_f32(const fg_instance *inst, int n, void *workspace, size_t workspace_bytes,
                          void *stream) {
  std::vector<OpSpec> ops;
  int rc = to_specs(inst, n, ops);
  if (rc) return rc;
  if (ops.empty()) return FG_OK;
  return run_ops(ops, workspace, workspace_bytes, (hipStream_t)stream);
}

struct fg_stepper {
  Stepper impl;
};

size_t fg_stepper_blob_bytes(int max_transforms) { return stepper_blob_bytes(max_transforms); }

size_t fg_stepper_op_bytes(const fg_instance *inst, size_t *halo_bytes) {
  std::vector<OpSpec> ops;
  if (!inst || to_specs(inst, 1, ops)) return 0;
  if (halo_bytes) *halo_bytes = halo_entries_for(ops, current_halo()) * sizeof(unsigned long long);
  return op_buffers_bytes(ops[0]);
}

int fg_stepper_create(fg_stepper **out, void *halo, size_t halo_bytes, void *blob, size_t blob_bytes) {
  if (!out || !halo || !blob) return fail(FG_EINVAL, "null argument");
  if (halo_bytes < 16 || blob_bytes < 4096) return fail(FG_EWORKSPACE, "stepper buffers too small");
  int dev = 0;
  FG_HIP(hipGetDevice(&dev));
  fg_stepper *p = new (std::nothrow) fg_stepper();
  if (!p) return fail(FG_EHIP, "out of host memory");
  p->impl.device = dev;
  p->impl.halo = (unsigned long long *)halo;
  p->impl.halo_cap = (halo_bytes - 8) / sizeof(unsigned long long);
  p->impl.blob = (unsigned char *)blob;
  p->impl.blob_cap = blob_bytes;
  *out = p;
  return FG_OK;
}

int fg_stepper_add(fg_stepper *s, const fg_instance *inst, void *workspace, size_t workspace_bytes,
                   int *ticket) {
  if (!s || !inst || !ticket) return fail(FG_EINVAL, "null argument");
  std::vector<OpSpec> ops;
  int rc = to_specs(inst, 1, ops);
  if (rc) return rc;
  return stepper_add(s->impl, ops[0], workspace, workspace_bytes, ticket);
}

int fg_stepper_step(fg_stepper *s, void *stream, int *done, int cap, int *ndone) {
  if (!s || !ndone || (cap > 0 && !done)) return fail(FG_EINVAL, "null argument");
  if (cap < (int)s->impl.ops.size()) return fail(FG_EINVAL, "done array smaller than the active transforms");
  return stepper_step(s->impl, (hipStream_t)stream, done, cap, ndone);
}

int fg_stepper_active(const fg_stepper *s) { return s ? (int)s->impl.ops.size() : 0; }

void fg_stepper_destroy(fg_stepper *s) { delete s; }

int fg_set_voxels_f32(const fg_voxel_set *items, int n, void *stream) {
  if (n < 0 || (n > 0 && !items)) return fail(FG_EINVAL, "bad voxel array");
  for (int i = 0; i < n; ++i)
    if (!items[i].dst || items[i].index < 0) return fail(FG_EINVAL, "voxel " + std::to_string(i) + ": bad target");
  for (int i0 = 0; i0 < n; i0 += kVoxelsPerLaunch) {
    VoxelBatch b;
    const int k = std::min(kVoxelsPerLaunch, n - i0);
    std::memcpy(b.it, items + i0, (size_t)k * sizeof(fg_voxel_set));
    hipLaunchKernelGGL(set_voxels_kernel, dim3(1), dim3(128), 0, (hipStream_t)stream, b, k);
    FG_HIP(hipGetLastError());
  }
  return FG_OK;
}

int fg_tuning_set(const fg_tuning *t) {
  if (!t) return fail(FG_EINVAL, "null tuning");
  if (t->engine < 0 || t->engine > 1) return fail(FG_EINVAL, "engine must be 0 or 1");
  if (t->halo < 0 || t->halo > kMaxK) return fail(FG_EINVAL, "halo must be 0 (automatic) or in [1, 30]");
  if (t->max_groups < 0) return fail(FG_EINVAL, "max_groups must be >= 0");
  if (t->shape < 0 || t->shape >= kNumShapes) return fail(FG_EINVAL, "shape must be in [0, 7]");
  g_tune = *t;
  g_shape = t->shape == 0 ? kAutoShape : t->shape;
  return FG_OK;
}

int fg_tuning_get(fg_tuning *t) {
  if (!t) return fail(FG_EINVAL, "null tuning");
  *t = g_tune;
  return FG_OK;
}

int fg_profile_enable(int on) {
  g_prof_on = (on & 1) != 0;
  g_prof_xhist = (on & 2) != 0;
  if (g_prof_xhist) {  // start a new exchange-wait histogram on the current device
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return fail(FG_EHIP, std::string("hipGetDevice: ") + hipGetErrorString(e));
    unsigned *h = nullptr;
    const int rc = exchange_histogram_impl(dev, &h);
    if (rc) return rc;
    e = hipMemset(h, 0, kXHistBuckets * sizeof(unsigned));
    if (e != hipSuccess) return fail(FG_EHIP, std::string("hipMemset: ") + hipGetErrorString(e));
  }
  return FG_OK;
}

int fg_profile_exchange_histogram(unsigned *counts, int n) {
  if (!counts || n < kXHistBuckets) return fail(FG_EINVAL, "need room for 32 buckets");
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(FG_EHIP, std::string("hipGetDevice: ") + hipGetErrorString(e));
  unsigned *h = nullptr;
  const int rc = exchange_histogram_impl(dev, &h);
  if (rc) return rc;
  e = hipDeviceSynchronize();
  if (e == hipSuccess) e = hipMemcpy(counts, h, kXHistBuckets * sizeof(unsigned), hipMemcpyDeviceToHost);
  if (e != hipSuccess) return fail(FG_EHIP, std::string("histogram copy: ") + hipGetErrorString(e));
  return FG_OK;
}

int fg_profile_collect(int *launches, double *total_ms, double *alg_bytes) {
  double ms = 0, bytes = 0;
  int n = 0, rc = FG_OK;
  for (auto &p : g_prof) {
    float t = 0;
    hipError_t e = hipEventSynchronize(p.stop);
    if (e == hipSuccess) e = hipEventElapsedTime(&t, p.start, p.stop);
    if (e != hipSuccess && rc == FG_OK) rc = fail(FG_EHIP, std::string("profile events: ") + hipGetErrorString(e));
    (void)hipEventDestroy(p.start);
    (void)hipEventDestroy(p.stop);
    ms += t;
    bytes += p.bytes;
    ++n;
  }
  g_prof.clear();
  if (launches) *launches = n;
  if (total_ms) *total_ms = ms;
  if (alg_bytes) *alg_bytes = bytes;
  return rc;
}

int fg_status(void *stream) {
  int id = 0;
  hipError_t e = hipGetDevice(&id);
  if (e != hipSuccess) return fail(FG_EHIP, std::string("hipGetDevice: ") + hipGetErrorString(e));
  e = hipStreamSynchronize((hipStream_t)stream);
  if (e != hipSuccess) return fail(FG_EHIP, std::string("hipStreamSynchronize: ") + hipGetErrorString(e));
  DeviceState &ds = device_state(id);
  int st = take_status(ds);
  if (ds.scratch) {  // the no-allocation entry point's word, used before a pinned one existed
    int w = 0;
    e = hipMemcpy(&w, ds.scratch, sizeof w, hipMemcpyDeviceToHost);
    if (e != hipSuccess) return fail(FG_EHIP, std::string("hipMemcpy: ") + hipGetErrorString(e));
    if (w != 0) {
      const int zero = 0;
      e = hipMemcpy(ds.scratch, &zero, sizeof zero, hipMemcpyHostToDevice);
      if (e != hipSuccess) return fail(FG_EHIP, std::string("hipMemcpy: ") + hipGetErrorString(e));
      if (st == FG_OK) st = w;
    }
  }
  return status_error(st, "status");
}

int fg_pending_status(int device) {
  if (device < 0) return fail(FG_EINVAL, "device must be >= 0");
  return take_status(device_state(device));
}

int fg_inject_status(int device, int code) {
  if (device < 0) return fail(FG_EINVAL, "device must be >= 0");
  device_state(device).injected.store(code);
  return FG_OK;
}

int fg_set_graphs(int on) {
  g_graph_on = on != 0;
  return FG_OK;
}

int fg_set_wait_limit(int spins) {
  if (spins < 0) return fail(FG_EINVAL, "wait limit must be >= 0");
  g_wait_limit = spins;
  return FG_OK;
}

void fg_release(void) {
  int rc = fg_profile_collect(nullptr, nullptr, nullptr);
  (void)rc;
  {
    std::lock_guard<std::mutex> g(g_graph_m);
    for (auto &p : g_graph_list) destroy_graph(*p);
    g_graph_list.clear();
  }
  std::lock_guard<std::mutex> g(g_reg_m);
  for (auto &kv : g_reg) {
    DeviceState &s = *kv.second;
    std::lock_guard<std::mutex> l(s.m);
    if (s.has) (void)hipEventSynchronize(s.done);
    for (auto &sl : s.stage) {
      if (sl.has_event) {
        (void)hipEventSynchronize(sl.copied);
        (void)hipEventDestroy(sl.copied);
        sl.has_event = false;
      }
      if (sl.host) (void)hipHostFree(sl.host);
      sl.host = nullptr;
      sl.cap = 0;
    }
    if (s.has) (void)hipEventDestroy(s.done);
    s.has = false;
    if (s.status_host) (void)hipHostFree(s.status_host);
    s.status_host = s.status_dev = nullptr;
  }
}

}  // extern "C"
