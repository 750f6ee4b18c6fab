// findLocalMax (objectdetect_aux.cpp:193-251) on device grids.
//
// A point (d, y, x) of a [D][H][W] grid is kept when no spatial 8-neighbour
// in its slice is strictly greater and the slices d-1 and d+1 (where they
// exist) are strictly lower at (y, x).  With at most max_n points the
// reference returns them in its scan order (d, then x, then y); with more it
// keeps the max_n largest values, sorted by value (ties by scan order here;
// the reference's std::sort leaves their order unspecified).
//
//   k_lmax_mark     the test, one bit per point and a histogram of the marked
//                   values' leading 11 bits per grid
//   k_lmax_refine   a second histogram (the next 11 bits) inside the bin that
//                   holds the max_n-th largest
//   k_lmax_collect  the keys at or above that 22-bit threshold (all of them
//                   when there are at most max_n)
//   k_lmax_select   one workgroup per grid sorts those few in LDS
// (k_lmax_small does all that for grids of no more points than LDS takes.)
// Where some grid has more of those keys than LDS takes (k_lmax_select tells
// the host), it goes on with a third histogram (the last 10 bits) and, where too
// many values equal that threshold, with three more of their scan indices, and
// collects again.
// Grids near LOG_ZERO do it (the bin spans 64 units of value there), grids of few
// distinct values, plateaus.  Selected by one workgroup from every mark, byte by
// byte, such a grid of 24 x 300 x 300 took 7.6 ms, now 0.62 (0.17 without the second
// part), a plateau of 1000 x 1000 6.2 and now 0.40 ms.
// key = (order key of value) << 32 | (2^32-1 - scan index): distinct, so the
// result does not depend on the order in which the keys were collected.
//
// The marks are read twice more from a mask of 1/32 of the grids' bytes and
// only marked values are touched again; the keys appended one by one with an
// atomic on a counter per grid, into 8 bytes for every point, took 3.6 ms for
// ten 24 x 300 x 300 grids with 2e5 maxima each, and reading them in one
// workgroup per grid 0.29 ms; now 69 + 27 + 32 + 18 us, the mark reading the
// grids at 1.3 TB/s (of 5.2 a large copy reaches).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/partapp_ps.h"
#include "ps_device.hpp"
#include "ps_plan.hpp"
#include "ps_pool.hpp"

namespace ps {

namespace {

struct LmGrid {
  long long off;       // grid start in the input array (elements)
  long long mask_off;  // start of its marks (64-bit words)
  int D, H, W;
  int wq;              // words per row
};
// the grids of one set of launches, passed by value
struct LmBatch {
  static constexpr int kMax = 96;
  LmGrid g[kMax];
};

constexpr int kSelThreads = 1024;
constexpr int kMaxLocalMax = 4096;
constexpr int kBins = 2048;     // 11 bits
constexpr int kCap = 8192;      // keys collected per grid (64 KB, sorted in LDS)
constexpr int kMarkRows = 16;   // rows of a wave's 64-column tile
constexpr int kTabGrids = 1024; // grids of one set of launches that reads a table

// per grid: the histograms of the first part, the marked points and the
// collected keys; from the second part's kernels the 22-bit threshold, the 32-bit
// one and the leading bits of the scan threshold, each with the max_n-th largest's
// place in its bin, and whether they were needed; its histograms
struct LmState {
  unsigned hist[2][kBins];
  unsigned marked;
  unsigned collected, third, thr22, need2, tie, thr32, need3, scan11, need4, scan22, need5;
  unsigned pad_[52];
  unsigned more[4][kBins];
};
constexpr int kStateWords = sizeof(LmState) / 4, kFirstWords = 2 * kBins + 64;  // the first part clears those
constexpr int kSecondFrom = 2 * kBins + 1;                                     // the second part from there on

__device__ __forceinline__ unsigned okey(float f) {
  unsigned u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float okey_inv(unsigned k) {
  unsigned u = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
  return __uint_as_float(u);
}

// words [from, to) of each of n states
__global__ __launch_bounds__(256) void k_lmax_clear(LmState *__restrict__ st, int n, int from, int to) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int per = to - from, g = (int)(i / per);
  if (g < n) reinterpret_cast<unsigned *>(st + g)[from + (int)(i - (long long)g * per)] = 0u;
}

// grid i of a launch: from the arguments, or (TAB) from the table.  Two
// variants of each kernel: chosen at run time, its sizes end up in vector
// registers and every address with them, and marking takes 1.5 times as long.
template <bool TAB>
__device__ __forceinline__ const LmGrid &lm_grid(const LmBatch &b, const LmGrid *__restrict__ tab, unsigned i) {
  if constexpr (TAB) return tab[i];
  else return b.g[i];
}

__device__ __forceinline__ unsigned long long lm_key(const LmGrid &G, float v, int d, int y, int x) {
  const unsigned scan = (unsigned)(((long long)d * G.W + x) * G.H + y);  // d, then x, then y
  return ((unsigned long long)okey(v) << 32) | (unsigned long long)(0xffffffffu - scan);
}

// One wave per 64 columns x 16 rows of a slice, a lane per column, the 3 x 3
// neighbourhood sliding down: five loads per point, four of them lines that
// the wave or its neighbours have just read.
template <bool TAB>
__global__ __launch_bounds__(256) void k_lmax_mark(const float *__restrict__ grids, LmBatch gd,
                                                   const LmGrid *__restrict__ tab, unsigned long long *__restrict__ mask, LmState *__restrict__ st) {
  __shared__ unsigned hist[kBins];
  unsigned bx, by;
  xcd_block(bx, by);
  const LmGrid &G = lm_grid<TAB>(gd, tab, by);
  const int D = G.D, H = G.H, W = G.W;
  const unsigned yt = (unsigned)(H + kMarkRows - 1) / kMarkRows, wq = (unsigned)G.wq;
  const unsigned tiles = (unsigned)D * yt * wq;  // at most D H W < 2^31
  if (bx * 4u >= tiles) return;
  for (int i = threadIdx.x; i < kBins; i += 256) hist[i] = 0u;
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const unsigned wave = (unsigned)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  unsigned n_marked = 0u;
  for (unsigned t = bx * 4u + wave; t < tiles; t += gridDim.x * 4u) {
    const unsigned dt = t / wq, q = t - dt * wq;
    const int d = (int)(dt / yt);
    const int y0 = (int)(dt - (unsigned)d * yt) * kMarkRows;
    const int x = (int)q * 64 + lane;
    const bool xin = x < W;
    const int xc = min(x, W - 1), xl = max(xc - 1, 0), xr = min(xc + 1, W - 1);
    const long long HW = (long long)H * W;
    const float *g = grids + G.off + (long long)d * HW;
    const float *gp = d > 0 ? g - HW : g, *gn = d < D - 1 ? g + HW : g;
    // a neighbour outside the grid is a copy of the point itself or of one
    // inside the neighbourhood: it never adds a greater value
    auto row3 = [&](int y, float &l, float &c, float &r) {
      const float *p = g + (long long)min(max(y, 0), H - 1) * W;
      l = p[xl];
      c = p[xc];
      r = p[xr];
    };
    // fmaxf leaves a NaN out, as the comparison with one does
    float l, c, r, al, ac, ar;
    row3(y0 - 1, al, ac, ar);
    float above = fmaxf(fmaxf(al, ar), ac);
    row3(y0, l, c, r);
    unsigned long long *m = mask + G.mask_off + ((long long)d * H + y0) * wq + q;
#pragma unroll
    for (int k = 0; k < kMarkRows; ++k) {
      const bool in = y0 + k < H;
      const long long yo = (long long)min(y0 + k, H - 1) * W + xc;
      float nl, nc, nr;
      row3(y0 + k + 1, nl, nc, nr);
      const float vp = gp[yo], vn = gn[yo];
      const float below = fmaxf(fmaxf(nl, nr), nc);
      const float side = fmaxf(l, r);
      const bool keep = in && xin && !(above > c) && !(below > c) && !(side > c) && (d == 0 || vp < c) &&
                        (d == D - 1 || vn < c);
      const unsigned long long w = __ballot(keep);
      if (lane == 0 && in) m[(long long)k * wq] = w;
      if (keep) atomicAdd(&hist[okey(c) >> 21], 1u);
      n_marked += (unsigned)__popcll(w);
      above = fmaxf(side, c);
      l = nl;
      c = nc;
      r = nr;
    }
  }
  __syncthreads();
  LmState &S = st[by];
  for (int i = threadIdx.x; i < kBins; i += 256)
    if (hist[i]) atomicAdd(&S.hist[0][i], hist[i]);
  if (lane == 0 && n_marked) atomicAdd(&S.marked, n_marked);
}

// The bin of a histogram that holds the need-th largest entry and, in `need`,
// its place inside the bin; every thread of a 256-thread block calls it.
__device__ __forceinline__ int lm_bin(const unsigned *__restrict__ h, unsigned &need, unsigned (&part)[4]) {
  constexpr int kPer = kBins / 256;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // thread t holds bins kBins - 1 - kPer t downwards
  unsigned c[kPer], sum = 0u;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    c[i] = h[kBins - 1 - (int)threadIdx.x * kPer - i];
    sum += c[i];
  }
  unsigned run = sum;  // inclusive sum over the wave
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned v = (unsigned)__shfl_up((int)run, o, 64);
    if (lane >= o) run += v;
  }
  __shared__ int bin_s;
  __shared__ unsigned need_s;
  if (lane == 63) part[wave] = run;
  __syncthreads();
  unsigned before = run - sum;
  for (int w = 0; w < wave; ++w) before += part[w];
  if (before < need && need <= before + sum) {
    int i = 0;
#pragma unroll
    for (int k = 0; k < kPer - 1; ++k)
      if (i == k && before + c[k] < need) {
        before += c[k];
        i = k + 1;
      }
    bin_s = kBins - 1 - (int)threadIdx.x * kPer - i;
    need_s = need - before;
  }
  __syncthreads();
  need = need_s;
  const int b = bin_s;
  __syncthreads();
  return b;
}

// f(value, d, y, x) of every marked point of the block's share of a grid; a
// lane whose point is not marked gets marked = false.  Eight words per wave
// are in flight.
template <class F>
__device__ __forceinline__ void lm_marked(const float *__restrict__ grids, const LmGrid &G,
                                          const unsigned long long *__restrict__ mask, unsigned first, unsigned step,
                                          F &&f) {
  constexpr unsigned kU = 8;
  const int lane = threadIdx.x & 63;
  const unsigned wq = (unsigned)G.wq, H = (unsigned)G.H, words = (unsigned)G.D * H * wq;
  const float *g = grids + G.off;
  const unsigned long long *m = mask + G.mask_off;
  for (unsigned w0 = first * kU; w0 < words; w0 += step * kU) {
    float v[kU];
    bool on[kU];
    unsigned row = w0 / wq, q = w0 - row * wq;
    const unsigned row0 = row, q0 = q;
#pragma unroll
    for (unsigned u = 0; u < kU; ++u) {
      on[u] = w0 + u < words && ((m[min(w0 + u, words - 1)] >> lane) & 1ull);
      v[u] = on[u] ? g[(long long)row * G.W + (q * 64 + lane)] : 0.0f;
      if (++q == wq) q = 0, ++row;
    }
    row = row0;
    q = q0;
    unsigned d = row / H, y = row - d * H;
#pragma unroll
    for (unsigned u = 0; u < kU; ++u) {
      f(on[u], v[u], (int)d, (int)y, (int)(q * 64 + lane));
      if (++q == wq) {
        q = 0;
        if (++y == H) y = 0, ++d;
      }
    }
  }
}

// One more histogram, of the values (DIGIT 1: bits 20 to 10, 2: 9 to 0) or, of
// values equal to the threshold, of 2^32-1 - scan (3: bits 31 to 21, 4: 20 to 10,
// 5: 9 to 0) whose leading bits are those that hold the max_n-th largest.
template <int DIGIT, bool TAB>
__global__ __launch_bounds__(256) void k_lmax_refine(const float *__restrict__ grids, LmBatch gd,
                                                     const LmGrid *__restrict__ tab,
                                                     const unsigned long long *__restrict__ mask,
                                                     LmState *__restrict__ st, int max_n) {
  __shared__ unsigned hist[kBins], part[4];
  LmState &S = st[blockIdx.y];
  const bool first = blockIdx.x == 0 && threadIdx.x == 0;
  unsigned top, v0 = 0u;  // leading bits of what is counted; of what value
  if (DIGIT <= 2) {
    if (S.marked <= (unsigned)max_n) return;
    unsigned need = (unsigned)max_n;
    top = (unsigned)lm_bin(S.hist[0], need, part);
    if (DIGIT == 2) {
      const unsigned b = (unsigned)lm_bin(S.hist[1], need, part);
      top = top << 11 | b;
      // the keys at or above the 22-bit threshold
      const bool third = (unsigned)max_n - need + S.hist[1][b] > (unsigned)kCap;
      if (first) S.third = third, S.thr22 = top, S.need2 = need;
      if (!third) return;
    }
  } else if (DIGIT == 3) {
    if (!S.third) return;
    unsigned need = S.need2;
    const unsigned b = (unsigned)lm_bin(S.more[0], need, part);
    const bool tie = (unsigned)max_n - need + S.more[0][b] > (unsigned)kCap;
    v0 = S.thr22 << 10 | b;
    if (first) S.tie = tie, S.thr32 = v0, S.need3 = need;
    if (!tie) return;
    top = 0u;
  } else {
    if (!S.tie) return;
    v0 = S.thr32;
    unsigned need = DIGIT == 4 ? S.need3 : S.need4;
    const unsigned b = (unsigned)lm_bin(S.more[DIGIT - 3], need, part);
    top = DIGIT == 4 ? b : S.scan11 << 11 | b;
    if (first && DIGIT == 4) S.scan11 = top, S.need4 = need;
    if (first && DIGIT == 5) S.scan22 = top, S.need5 = need;
  }
  constexpr int kShift = DIGIT == 1 || DIGIT == 4 ? 10 : DIGIT == 3 ? 21 : 0;
  constexpr int kBits = DIGIT == 2 || DIGIT == 5 ? 10 : 11;
  for (int i = threadIdx.x; i < kBins; i += 256) hist[i] = 0u;
  __syncthreads();
  const LmGrid &G = lm_grid<TAB>(gd, tab, blockIdx.y);
  const unsigned wave = (unsigned)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  lm_marked(grids, G, mask, blockIdx.x * 4 + wave, gridDim.x * 4, [&](bool on, float v, int d, int y, int x) {
    const unsigned k = DIGIT <= 2 ? okey(v) : (unsigned)lm_key(G, v, d, y, x);
    const bool in = on && (DIGIT <= 2 || okey(v) == v0) && (DIGIT == 3 || (k >> (kShift + kBits) % 32) == top);
    if (in) atomicAdd(&hist[(k >> kShift) & ((1u << kBits) - 1u)], 1u);
  });
  __syncthreads();
  unsigned *h = DIGIT == 1 ? S.hist[1] : S.more[DIGIT - (DIGIT == 1 ? 1 : 2)];
  for (int i = threadIdx.x; i < kBins; i += 256)
    if (hist[i]) atomicAdd(h + i, hist[i]);
}

template <bool SECOND, bool TAB>
__global__ __launch_bounds__(256) void k_lmax_collect(const float *__restrict__ grids, LmBatch gd,
                                                      const LmGrid *__restrict__ tab,
                                                      const unsigned long long *__restrict__ mask,
                                                      LmState *__restrict__ st, int max_n,
                                                      unsigned long long *__restrict__ keys) {
  __shared__ unsigned part[4];
  LmState &S = st[blockIdx.y];
  const LmGrid &G = lm_grid<TAB>(gd, tab, blockIdx.y);
  unsigned thr = 0u, thr_scan = 0u;  // least value key that is collected; of its ties the least 2^32-1 - scan
  const unsigned marked = S.marked;
  bool tie = false;
  if (SECOND && S.third) {
    tie = S.tie != 0u;
    thr = S.thr32;
    if (tie) {
      unsigned need = S.need5;
      thr_scan = S.scan22 << 10 | (unsigned)lm_bin(S.more[3], need, part);
    }
  } else if (marked > (unsigned)max_n) {
    unsigned need = (unsigned)max_n;
    const unsigned b1 = (unsigned)lm_bin(S.hist[0], need, part);
    const unsigned b2 = (unsigned)lm_bin(S.hist[1], need, part);
    thr = b1 << 21 | b2 << 10;
  }
  unsigned long long *out = keys + (long long)blockIdx.y * kCap;
  const int lane = threadIdx.x & 63;
  const unsigned wave = (unsigned)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  lm_marked(grids, G, mask, blockIdx.x * 4 + wave, gridDim.x * 4, [&](bool on, float v, int d, int y, int x) {
    bool take = on && okey(v) >= thr;
    if (SECOND && tie) take = take && (okey(v) > thr || (unsigned)lm_key(G, v, d, y, x) >= thr_scan);
    const unsigned long long w = __ballot(take);
    if (w == 0ull) return;
    unsigned at = 0u;
    if (lane == 0) at = atomicAdd(&S.collected, (unsigned)__popcll(w));
    at = (unsigned)__shfl((int)at, 0, 64) + (unsigned)__popcll(w & ((1ull << lane) - 1ull));
    // more than fit: counted only
    if (take && at < (unsigned)kCap) out[at] = lm_key(G, v, d, y, x);
  });
}

// bitonic sort of n (a power of two up to kCap) keys in LDS, descending
__device__ void bitonic_desc(unsigned long long *s, int n) {
  for (int k = 2; k <= n; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      __syncthreads();
      for (int i = threadIdx.x; i < (n >> 1); i += blockDim.x) {
        const int lo = 2 * i - (i & (j - 1)), hi = lo + j;  // the i-th pair j apart
        const unsigned long long a = s[lo], b = s[hi];
        if ((lo & k) == 0 ? a < b : a > b) {
          s[lo] = b;
          s[hi] = a;
        }
      }
    }
  __syncthreads();
}

__device__ __forceinline__ unsigned long long swap_halves(unsigned long long k) { return (k << 32) | (k >> 32); }

// the first `keep` keys of s as records; every thread of the block calls it
__device__ __forceinline__ void lm_write(const LmGrid &G, const unsigned long long *s, int keep,
                                         ps_local_max *__restrict__ o, int *__restrict__ o_n) {
  for (int i = threadIdx.x; i < keep; i += blockDim.x) {
    const unsigned long long k = s[i];
    const unsigned scan = 0xffffffffu - (unsigned)(k & 0xffffffffull);
    ps_local_max r;
    const unsigned hw = (unsigned)G.H * (unsigned)G.W;
    r.d = (int)(scan / hw);
    const unsigned rem = scan - (unsigned)r.d * hw;
    r.x = (int)(rem / (unsigned)G.H);
    r.y = (int)(rem - (unsigned)r.x * (unsigned)G.H);
    r.score = okey_inv((unsigned)(k >> 32));
    o[i] = r;
  }
  if (threadIdx.x == 0) *o_n = keep;
}

template <bool TAB>
__global__ __launch_bounds__(kSelThreads) void k_lmax_select(LmBatch gd, const LmGrid *__restrict__ tab,
                                                             const LmState *__restrict__ st,
                                                             const unsigned long long *__restrict__ keys, int max_n,
                                                             ps_local_max *__restrict__ out, int *__restrict__ out_n,
                                                             unsigned *more_host) {
  __shared__ unsigned long long s[kCap];
  const LmGrid &G = lm_grid<TAB>(gd, tab, blockIdx.x);
  const LmState &S = st[blockIdx.x];
  const unsigned long long *c = keys + (long long)blockIdx.x * kCap;
  const unsigned marked = S.marked, n = S.collected;
  const int keep = (int)min(marked, (unsigned)max_n);
  if (n > (unsigned)kCap) {  // the first part only
    if (threadIdx.x == 0) __hip_atomic_store(more_host, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    return;
  }
  // all of them in scan order (by 2^32-1 - scan descending), or the largest
  const bool all = marked <= (unsigned)max_n;
  int n2 = 1;
  while (n2 < (int)n) n2 <<= 1;
  for (int i = threadIdx.x; i < n2; i += blockDim.x) s[i] = i < (int)n ? (all ? swap_halves(c[i]) : c[i]) : 0ull;
  bitonic_desc(s, n2);
  if (all) {
    for (int i = threadIdx.x; i < keep; i += blockDim.x) s[i] = swap_halves(s[i]);
    __syncthreads();
  }
  lm_write(G, s, keep, out + (long long)blockIdx.x * max_n, out_n + blockIdx.x);
}

// All of it for a grid of at most kCap points, one workgroup each: five launches
// take such a call longer than their work (six grids of 24x25x2: 97 us a call with
// them, 80 with one).
template <bool TAB>
__global__ __launch_bounds__(kSelThreads) void k_lmax_small(const float *__restrict__ grids, LmBatch gd,
                                                            const LmGrid *__restrict__ tab, int max_n,
                                                            ps_local_max *__restrict__ out, int *__restrict__ out_n) {
  __shared__ unsigned long long s[kCap];
  __shared__ unsigned fill_s;
  const LmGrid &G = lm_grid<TAB>(gd, tab, blockIdx.x);
  const int D = G.D, H = G.H, W = G.W, HW = H * W, n = D * HW;
  const float *g = grids + G.off;
  if (threadIdx.x == 0) fill_s = 0u;
  __syncthreads();
  for (int e = threadIdx.x; e < n; e += kSelThreads) {
    const int d = e / HW, rem = e - d * HW, y = rem / W, x = rem - y * W;
    const float *p = g + d * HW;
    const int xl = max(x - 1, 0), xr = min(x + 1, W - 1);
    // (a neighbour outside the grid is one inside the neighbourhood again;
    // fmaxf leaves a NaN out, as the comparison with one does)
    auto row = [&](int yy) {
      const float *q = p + min(max(yy, 0), H - 1) * W;
      return fmaxf(fmaxf(q[xl], q[xr]), q[x]);
    };
    const float c = p[rem], above = row(y - 1), below = row(y + 1), side = fmaxf(p[y * W + xl], p[y * W + xr]);
    const float vp = d > 0 ? g[e - HW] : c, vn = d < D - 1 ? g[e + HW] : c;
    if (!(above > c) && !(below > c) && !(side > c) && (d == 0 || vp < c) && (d == D - 1 || vn < c))
      s[atomicAdd(&fill_s, 1u)] = lm_key(G, c, d, y, x);
  }
  __syncthreads();
  const int marked = (int)fill_s, keep = min(marked, max_n);
  const bool all = marked <= max_n;
  int n2 = 1;
  while (n2 < marked) n2 <<= 1;
  for (int i = threadIdx.x; i < n2; i += kSelThreads) s[i] = i < marked ? (all ? swap_halves(s[i]) : s[i]) : 0ull;
  bitonic_desc(s, n2);
  if (all) {
    for (int i = threadIdx.x; i < keep; i += kSelThreads) s[i] = swap_halves(s[i]);
    __syncthreads();
  }
  lm_write(G, s, keep, out + (long long)blockIdx.x * max_n, out_n + blockIdx.x);
}

}  // namespace

}  // namespace ps

using namespace ps;

extern "C" int ps_find_local_max(const float *grids_dev, const long long *offsets, const int *dims, int n_grids,
                                 int max_n, ps_local_max *out_dev, int *count_dev, void *stream) {
  if (!grids_dev || !offsets || !dims || n_grids < 1 || !out_dev || !count_dev)
    return set_error(PS_ERR_INVALID_ARG, "null argument or n_grids < 1");
  if (max_n < 1 || max_n > kMaxLocalMax) return set_error(PS_ERR_UNSUPPORTED, "max_n must be in [1, 4096]");
  // grids of one set of launches: in the kernels' arguments, or in a table
  // where a call has very many
  const int step = n_grids <= LmBatch::kMax ? LmBatch::kMax : kTabGrids;
  std::vector<LmGrid> gd(n_grids);
  long long words = 0, most_words = 0;  // of one set
  for (int g = 0; g < n_grids; ++g) {
    const int D = dims[3 * g], H = dims[3 * g + 1], W = dims[3 * g + 2];
    if (D < 1 || H < 1 || W < 1 || offsets[g] < 0) return set_error(PS_ERR_INVALID_ARG, "bad grid dims or offset");
    if ((long long)D * H * W >= (1ll << 31)) return set_error(PS_ERR_UNSUPPORTED, "grid too large");
    if (g % step == 0) words = 0;
    gd[g].off = offsets[g];
    gd[g].mask_off = words;
    gd[g].D = D;
    gd[g].H = H;
    gd[g].W = W;
    gd[g].wq = (W + 63) / 64;
    words += (long long)D * H * gd[g].wq;
    most_words = std::max(most_words, words);
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  // workspace, used by one set after another: histograms and counters,
  // collected keys, marks; the table
  const size_t n_set = (size_t)std::min(n_grids, step);
  const size_t o_keys = sizeof(LmState) * n_set;
  const size_t o_mask = o_keys + sizeof(unsigned long long) * kCap * n_set;
  const size_t o_tab = o_mask + sizeof(unsigned long long) * (size_t)most_words;
  const bool table = n_grids > LmBatch::kMax;
  void *ws = nullptr;
  if (pool_get(&ws, o_tab + (table ? sizeof(LmGrid) * (size_t)n_grids : 0)) != hipSuccess)
    return set_error(PS_ERR_OUT_OF_MEMORY, "local max workspace");
  char *base = static_cast<char *>(ws);
  LmState *st = reinterpret_cast<LmState *>(base);
  unsigned long long *keys = reinterpret_cast<unsigned long long *>(base + o_keys);
  unsigned long long *mask = reinterpret_cast<unsigned long long *>(base + o_mask);
  LmGrid *tab = table ? reinterpret_cast<LmGrid *>(base + o_tab) : nullptr;
  unsigned *more = nullptr;  // in host memory
  hipError_t e = pool_get_host(&more);
  if (e == hipSuccess) *more = 0u;
  if (table && e == hipSuccess)
    e = hipMemcpyAsync(tab, gd.data(), sizeof(LmGrid) * (size_t)n_grids, hipMemcpyHostToDevice, s);
  for (const bool second : {false, true}) {
    for (int g0 = 0; g0 < n_grids && e == hipSuccess; g0 += step) {
      const int n = std::min(n_grids - g0, step);
      const LmGrid *one = gd.data() + g0, *t = table ? tab + g0 : nullptr;
      LmBatch b;
      if (!table) std::copy(one, one + n, b.g);
      long long tiles = 0, most = 0, points = 0;
      for (int i = 0; i < n; ++i) {
        points = std::max(points, (long long)one[i].D * one[i].H * one[i].W);
        tiles = std::max(tiles, (long long)one[i].D * ((one[i].H + kMarkRows - 1) / kMarkRows) * one[i].wq);
        most = std::max(most, (long long)one[i].D * one[i].H * one[i].wq);
      }
      if (points <= kCap) {
        auto small = [&](auto tabc) {
          hipLaunchKernelGGL((k_lmax_small<decltype(tabc)::value>), dim3((unsigned)n), dim3(kSelThreads), 0, s, grids_dev,
                             b, t, max_n, out_dev + (long long)g0 * max_n, count_dev + g0);
        };
        if (table) small(std::true_type());
        else small(std::false_type());
        e = hipGetLastError();
        continue;
      }
      // cleared by a small kernel (this entry point synchronizes and is not
      // capturable)
      auto clear = [&](int from, int to) {
        const long long words = (long long)n * (to - from);
        hipLaunchKernelGGL(k_lmax_clear, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, s, st, n, from, to);
      };
      const dim3 blk(256);
      // the marked points again: 8 words per wave and turn, at most 128 blocks a grid
      const dim3 again((unsigned)std::min<long long>(128, (most + 31) / 32), (unsigned)n);
      const dim3 mark((unsigned)std::min<long long>(1 << 20, (tiles + 3) / 4), (unsigned)n);
      auto launch = [&](auto tabc) {
        constexpr bool T = decltype(tabc)::value;
        // the second part goes on from the first where its marks are still there
        if (!second || n < n_grids) {
          clear(0, kFirstWords);
          hipLaunchKernelGGL((k_lmax_mark<T>), mark, blk, 0, s, grids_dev, b, t, mask, st);
          hipLaunchKernelGGL((k_lmax_refine<1, T>), again, blk, 0, s, grids_dev, b, t, mask, st, max_n);
        }
        if (second) {
          clear(kSecondFrom, kStateWords);
          hipLaunchKernelGGL((k_lmax_refine<2, T>), again, blk, 0, s, grids_dev, b, t, mask, st, max_n);
          hipLaunchKernelGGL((k_lmax_refine<3, T>), again, blk, 0, s, grids_dev, b, t, mask, st, max_n);
          hipLaunchKernelGGL((k_lmax_refine<4, T>), again, blk, 0, s, grids_dev, b, t, mask, st, max_n);
          hipLaunchKernelGGL((k_lmax_refine<5, T>), again, blk, 0, s, grids_dev, b, t, mask, st, max_n);
        }
        if (second)
          hipLaunchKernelGGL((k_lmax_collect<true, T>), again, blk, 0, s, grids_dev, b, t, mask, st, max_n, keys);
        else
          hipLaunchKernelGGL((k_lmax_collect<false, T>), again, blk, 0, s, grids_dev, b, t, mask, st, max_n, keys);
        hipLaunchKernelGGL((k_lmax_select<T>), dim3((unsigned)n), dim3(kSelThreads), 0, s, b, t, st, keys, max_n,
                           out_dev + (long long)g0 * max_n, count_dev + g0, more);
      };
      if (table) launch(std::true_type());
      else launch(std::false_type());
      e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess || *more == 0u) break;
  }
  pool_put_host(more, e == hipSuccess);
  pool_put(ws, e == hipSuccess);
  if (e != hipSuccess) return set_error(PS_ERR_HIP, std::string("local max: ") + hipGetErrorString(e));
  return PS_OK;
}
