// gfx950 kernels of the pictorial-structure sweep.
//
// One message of the sum-product sweep (computeRotJointMarginal,
// objectdetect_findrot.cpp:292-456) is two launches over a whole level of
// messages (every instance, scale and chain of the level at once):
//
//   k_rowpass  one block per (message, row y): gathers the forward-warped
//              child belief of all R rotation slices (integer shift per
//              slice), exp(b - M), circular rotation filter, then the
//              truncated x filter from an LDS row with zero halo on the
//              matrix cores.  Writes the row-filtered grid T.
//   k_colpass  one block per (message, rotation, 64-column strip): truncated y
//              filter of T on the matrix cores from an LDS ring of rows, log,
//              +M, the inverse warp folded into the tile origin, and the
//              caller's accumulation (parent belief, root message slot, or
//              marginal + next downward source) fused as the epilogue,
//              together with the max / argmax reductions the next step needs.
//
// Arithmetic follows the reference order: every dot product accumulates its
// taps in ascending order with a fused multiply-add starting from 0, exactly
// like a sequential sdot; sums of grids are added in the reference's order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <map>
#include <mutex>
#include <type_traits>
#include <utility>

#include "ps_device.hpp"
#include "ps_rowgather.hpp"
#include "ps_internal.hpp"
#include "../../include/partapp_ps.h"

namespace ps {

// --------------------------------------------------------------- k_reset

// Clears the max keys, the argmax keys and their top-2 keys of the instances
// that run (keys_per_inst / map_per_inst consecutive entries per instance);
// with clear_active it also clears the per-instance flags (n_flags) that a
// later certification pass sets.
__global__ void k_reset(Bases b, int n_keys, int n_map, int keys_per_inst, int map_per_inst, unsigned *flags,
                        int n_flags) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n_keys && !skip_inst(b, i / keys_per_inst)) *max_key(b, i) = 0u;
  if (i < n_map && !skip_inst(b, i / map_per_inst)) {
    *map_key(b, i) = 0ull;
    if (b.top2_keys) *top2_key(b, i) = 0ull;
  }
  if (flags && i < n_flags) flags[i] = 0u;
}

// ---------------------------------------------------------------- k_upload
// A small table carried to device memory in a kernel's arguments: a copy from
// pageable memory costs the call some 20 us, a launch some 4.

struct UploadChunk {
  static constexpr int kUnits = 240;  // 16 bytes each, below the 4 KB of kernel arguments
  uint4 d[kUnits];
};
__global__ __launch_bounds__(256) void k_upload(UploadChunk c, uint4 *dst, int n) {
  const int i = threadIdx.x;
  if (i < n) dst[i] = c.d[i];
}

// `bytes` (a multiple of 16) of host memory to dst in stream order
hipError_t launch_upload(void *dst, const void *src, size_t bytes, hipStream_t s) {
  for (size_t o = 0; o < bytes; o += sizeof(UploadChunk)) {
    UploadChunk c;
    const size_t n = std::min(bytes - o, sizeof(UploadChunk));
    std::memcpy(c.d, static_cast<const char *>(src) + o, n);
    hipLaunchKernelGGL(k_upload, dim3(1), dim3(256), 0, s, c, reinterpret_cast<uint4 *>(static_cast<char *>(dst) + o),
                       (int)(n / 16));
  }
  return hipGetLastError();
}

// ------------------------------------------------- FP32 filters on the MFMA
// v_mfma_f32_4x4x1 holds 16 independent 4 x 4 products of depth 1: lane l =
// 4 b + n of block b has D[i] += A(lane 4 b + i) B(lane l), i = 0..3, each one
// fused multiply-add, bit for bit fmaf (checked on the device over 50-step
// chains with operands down to subnormals).  Four outputs next to each other
// along a filter of L taps, out[n] = sum_k x[k] f[k - n], therefore take L + 3
// steps in ascending order, the same sums as the sequential dot product with
// zero products before and after (0 x + a = a for finite x), at twice the
// rate of unpacked v_fma_f32 (131 against 65 TFLOP/s measured; the two do not
// overlap: a loop of both takes the sum of their times).  A zero product with
// a non-finite value would be a NaN outside the band, so data holding one goes
// an output at a time over its own taps.

typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4_t mfma4(float a, float b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 0, 0, 0);
}

// The taps of such a filter as that operand, in steps of four: copy n (n =
// lane % 4) holds f[k - n], k = 0 .. 4 chunks - 1 (zero off the filter); the
// copies' 16-byte units start in different LDS banks (an odd pitch).
__host__ __device__ __forceinline__ int tap4_chunks(int k) { return (2 * k + 1 + 3 + 3) >> 2; }
__host__ __device__ __forceinline__ int tap4_pitch(int k) { return 4 * (tap4_chunks(k) | 1); }
// A thread takes a tap to its place in the four copies; its first one is loaded
// ahead, to wait beside the pass's other loads (a launch of 112x128x24: 13.6 ->
// 12.9 us, of 32 300x300x24: 757 -> 743).
__device__ __forceinline__ float tap4_load(const float *__restrict__ f, int k) {
  return f[min(max((int)threadIdx.x - 3, 0), 2 * k)];
}
__device__ __forceinline__ void tap4_store(float *t4, float first, const float *__restrict__ f, int k, int nt) {
  const int L = 2 * k + 1, n4 = 4 * tap4_chunks(k), pitch = tap4_pitch(k);
  for (int i = threadIdx.x; i < n4 + 3; i += nt) {
    const int t = i - 3;
    float v = i == (int)threadIdx.x ? first : f[min(max(t, 0), 2 * k)];
    v = t >= 0 && t < L ? v : 0.0f;
#pragma unroll
    for (int n = 0; n < 4; ++n)
      if (t + n >= 0 && t + n < n4) t4[n * pitch + t + n] = v;
  }
}

// bit patterns from here on (infinities, NaNs, and anything negative, which
// no filter operand is) are not for the MFMA
constexpr unsigned kNonFinite = 0x7f800000u;
// The row pass looks at the values before the rotation filter, whose finite
// sums can overflow: below 2^122 they cannot, with at most 48 taps of at most
// 1 (a fill value exp(LOG_ZERO - M) lies above it where M < LOG_ZERO - 84.5).
constexpr unsigned kRowNonFinite = 0x7c800000u;
__device__ __forceinline__ unsigned max_bits(unsigned m, float v) { return max(m, __float_as_uint(v)); }

// ------------------------------------------------------------------ k_max
// Max of a leaf's source grid (getMinMax, multi_array_op.hpp:60-77).  Grids
// without masks are scanned flat with 16-byte loads, whatever their alignment;
// masked ones by rows, a wave each, over the states the masks leave.

__global__ __launch_bounds__(256) void k_max(Bases b, const MaxJob *__restrict__ jobs, int R, int chunk) {
  __shared__ uint4 red[4];
  const MaxJob &J = jobs[blockIdx.y];
  if (skip_inst(b, J.inst)) return;
  const int H = J.H, W = J.W;
  // 64 bits: a message's grid (any rotation count, full covariance) may hold
  // 2^31 states and more; in the chunk [e0, e0 + n) 32 do
  const long long total = (long long)R * H * W, e0 = (long long)blockIdx.x * chunk;
  if (e0 >= total) return;
  const int n = (int)min(total - e0, (long long)chunk);
  unsigned km = 0u;
  if (J.src_kind == kSrcZero) {
    km = f2key(0.0f);
  } else {
    const float *src = cptr(b, J.src);
    if (J.mask.rot_bits == 0ull && J.mask.strip == 0) {
      // [a0, a1): whole 16-byte units; the elements before and behind them
      src += e0;
      const int head = (int)((0u - (unsigned)(reinterpret_cast<uintptr_t>(src) >> 2)) & 3u);
      const int a0 = min(head, n), a1 = a0 + ((n - a0) & ~3);
      const int t = (int)threadIdx.x;
      if (t < a0) km = f2key(src[t]);
      else if (t >= 4 && t - 4 < n - a1) km = f2key(src[a1 + t - 4]);
      // four independent loads per thread in flight (a lane past the end
      // reads its first element again, which leaves the max unchanged)
      constexpr int kU = 4;
      const float4 *s4 = reinterpret_cast<const float4 *>(src + a0);
      const int n4 = (a1 - a0) >> 2;
      for (int i = t; i < n4; i += kU * blockDim.x) {
        float4 v[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
          const int j = i + u * (int)blockDim.x;
          v[u] = s4[j < n4 ? j : i];
        }
#pragma unroll
        for (int u = 0; u < kU; ++u)
          km = max(km, max(max(f2key(v[u].x), f2key(v[u].y)), max(f2key(v[u].z), f2key(v[u].w))));
      }
    } else {
      // the chunk's rows: those that begin in it
      const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
      const int row0 = (int)((e0 + W - 1) / W), row1 = (int)((e0 + n + W - 1) / W);
      const int x0 = J.mask.strip, x1 = W - J.mask.strip;
      bool any = J.mask.strip > 0;  // a masked state
      if (x1 - x0 <= 64) {
        // one or several rows a wave and turn, four turns in flight (row after row:
        // 55 instead of 15 us for the leaves of 6 images of 92x5x24 at three scales)
        int bits = 6;  // lanes a row, a power of two
        while (bits > 0 && (1 << (bits - 1)) >= x1 - x0) --bits;
        const int step = 4 << (6 - bits), x = x0 + (lane & ((1 << bits) - 1));
        constexpr int kU = 4;
        for (int row = row0 + (wave << (6 - bits)) + (lane >> bits); row < row1; row += kU * step) {
          float v[kU];
          bool use[kU];
#pragma unroll
          for (int u = 0; u < kU; ++u) {
            const int rr = row + u * step;
            const bool out = rr < row1 && masked(J.mask, rr / H, x0, W);
            any |= out;
            use[u] = rr < row1 && !out && x < x1;
            v[u] = use[u] ? src[(long long)rr * W + x] : 0.0f;
          }
#pragma unroll
          for (int u = 0; u < kU; ++u) km = max(km, use[u] ? f2key(v[u]) : 0u);
        }
      } else {
        for (int row = row0 + wave; row < row1; row += 4) {
          if (masked(J.mask, row / H, x0, W)) {
            any = true;
            continue;
          }
          constexpr int kU = 4;
          const float *p = src + (long long)row * W;
          for (int x = x0 + lane; x < x1; x += kU * 64) {
            float v[kU];
#pragma unroll
            for (int u = 0; u < kU; ++u) v[u] = p[x + 64 * u < x1 ? x + 64 * u : x];
#pragma unroll
            for (int u = 0; u < kU; ++u) km = max(km, f2key(v[u]));
          }
        }
      }
      if (any) km = max(km, f2key(kLogZero));
    }
  }
  KeyPart p;
  p.key = wave_max_u32(km);
  block_raise(red, p, max_key(b, J.key), nullptr, nullptr);
}

// -------------------------------------------------------------- k_rowpass
// One block per (message, row y), all R slices of the row.  LDS holds
// P[R][Pw]: the rotation-filtered rows with kx zeros on the left and a zero
// tail, Pw a multiple of 4, read by the x filter.

// slice groups the fixed-R row pass stages in LDS one after another: 48
// slices in two halves (36 KB instead of 72 KB of LDS per 300-wide row, 160
// VGPRs: 20.9 instead of 27.6 ms per 32 x 300x300x48 sweep), 24 in one (as
// two halves 9.7 instead of 8.8 ms per 32 x 300x300x24 sweep)
__host__ __device__ constexpr int row_groups(int R) { return R >= 48 ? 2 : 1; }

// LDS of the row pass with the x filter on the MFMA: P[position][pitch], the RG
// slices of a column next to each other (written and read at immediate
// offsets), kx zeros before the row and the last column's window behind it; the
// tap operand and the flag follow.  24 slices go through at once (12 at a time
// halve the LDS and cost a second pass over the rotation filter's inputs: 855
// against 765 us per launch of 32 images of 300x300x24) and are read in pairs
// (half the LDS instructions: 759 -> 733 us there, 153 -> 140 on uneven grids);
// 48 go in four groups of 12 (24 beside the 48 values held from group to group
// spill; three groups of 16, read four at a time, 77.6 against 74.5 us per launch
// of one 300x300 image).  The pitches spread the 16 positions x 4 slices of a
// read over all banks.
__host__ __device__ constexpr int row4_slices(int R) { return R == 24 ? 24 : 12; }
__host__ __device__ constexpr bool row4_pairs(int rg) { return rg % 8 == 0; }
__host__ __device__ constexpr int row4_pitch(int rg) { return row4_pairs(rg) ? rg + 2 : rg + 1; }
__host__ __device__ __forceinline__ int row4_len(int W, int k) { return ((W + 3) & ~3) + 4 * tap4_chunks(k); }
__host__ __device__ __forceinline__ size_t row4_floats(int rg, int W, int k) {
  return ((size_t)row4_len(W, k) * row4_pitch(rg) + 3) & ~(size_t)3;
}
__host__ __device__ __forceinline__ size_t row4_lds_bytes(int rg, int W, int k) {
  return sizeof(float) * (row4_floats(rg, W, k) + 4 * tap4_pitch(k) + 4);
}

// x filter of the RG rows of P (RG a multiple of 4), row y of T: wave w takes
// the 64-column tiles w, w + waves, ...; lane 4 b + m reads slices 4 s + m (in
// pairs: S m + s), s < S = RG / 4, from position 4 b of the tile on (past the row,
// its last positions again), and holds after the last step, in acc[s][i], slice
// 4 s + i (S i + s) at column `lane`: stores of whole lines.  One LDS read of
// four steps' taps serves the S groups of slices.
template <int RG>
__device__ __forceinline__ void xfilter4(const float *P, const float *t4, int kx, float *T, int tp, long long plane,
                                         int y, int W, int nt) {
  static_assert(RG % 4 == 0, "rows in groups of four");
  constexpr int S = RG / 4, Q = row4_pitch(RG);
  constexpr bool kPairs = row4_pairs(RG);
  const int lane = threadIdx.x & 63, m = lane & 3;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int NT = tap4_chunks(kx), tiles = (W + 63) >> 6;
  char *trow = reinterpret_cast<char *>(T + (long long)y * tp);
  const long long plane_b = plane * 4;
  for (int j = wave; j < tiles; j += nt >> 6) {
    const float4 *tv = reinterpret_cast<const float4 *>(t4 + m * tap4_pitch(kx));
    const float *d = P + min(64 * j + (lane & ~3), ((W + 3) & ~3) - 4) * Q + (kPairs ? m * S : m);
    f32x4_t acc[S];
#pragma unroll
    for (int s = 0; s < S; ++s) acc[s] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    for (int c = 0; c < NT; ++c) {
      const float4 t = *tv++;
      float x[4][S];
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int s = 0; s < S; ++s) {
          if (!kPairs) {
            x[k][s] = d[k * Q + 4 * s];
          } else if (s % 2 == 0) {
            const float2 v = *reinterpret_cast<const float2 *>(d + k * Q + s);
            x[k][s] = v.x;
            x[k][s + 1] = v.y;
          }
        }
      d += 4 * Q;
#pragma unroll
      for (int s = 0; s < S; ++s) acc[s] = mfma4(x[0][s], t.x, acc[s]);
#pragma unroll
      for (int s = 0; s < S; ++s) acc[s] = mfma4(x[1][s], t.y, acc[s]);
#pragma unroll
      for (int s = 0; s < S; ++s) acc[s] = mfma4(x[2][s], t.z, acc[s]);
#pragma unroll
      for (int s = 0; s < S; ++s) acc[s] = mfma4(x[3][s], t.w, acc[s]);
    }
    const unsigned xo = 64u * (unsigned)j + (unsigned)lane;
    if ((int)xo < tp) {
      char *o = trow;
#pragma unroll
      for (int n = 0; n < RG; ++n) {
        *reinterpret_cast<float *>(o + xo * 4u) = kPairs ? acc[n % S][n / S] : acc[n / 4][n % 4];
        o += plane_b;
      }
    }
  }
}

// Four taps of a filter on the vector unit: acc[i] += win[i + u] f[u], u
// ascending, the N values of the window and the four behind them, which become
// its last.
template <int N>
__device__ __forceinline__ void plain_taps(float (&acc)[N], float (&win)[N], const float (&behind)[4], const float *f) {
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const float t = f[u];
#pragma unroll
    for (int i = 0; i < N; ++i) acc[i] = fmaf(i + u < N ? win[(i + u) % N] : behind[(i + u) % 4], t, acc[i]);
  }
#pragma unroll
  for (int i = 0; i < N; ++i) win[i] = i + 4 < N ? win[(i + 4) % N] : behind[(i + 4) % 4];
}

// The same filter of rows holding a non-finite value, each output over its own
// taps (padded to a multiple of four with zeros, as the pool holds them): N
// outputs of a slice per thread (eight of 24 slices; of 48, whose 48 values a
// thread holds meanwhile, four: with eight the kernel takes 100 registers
// instead of 77 and two waves of six per SIMD).
template <int RG>
__device__ __forceinline__ void xfilter_plain(const float *P, const float *__restrict__ f, int kx, float *T, int tp,
                                              long long plane, int y, int W, int nt) {
  constexpr int Q = row4_pitch(RG), N = RG == 24 ? 8 : 4;
  const int Lp = (2 * kx + 1 + 3) & ~3, last = row4_len(W, kx) - 1;
  for (int i = threadIdx.x; i < RG * ((W + N - 1) / N); i += nt) {
    const int q = i / RG, r = i - q * RG;
    int pos = N * q;
    // (past the layout: its last position, for outputs past the row)
    auto next = [&] { return P[min(pos++, last) * Q + r]; };
    float a[N], win[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      a[j] = 0.0f;
      win[j] = next();
    }
    for (int t = 0; t < Lp; t += 4) {
      float behind[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) behind[j] = next();
      plain_taps<N>(a, win, behind, f + t);
    }
    float *o = T + r * plane + (long long)y * tp + N * q;
#pragma unroll
    for (int j = 0; j < N; ++j)
      if (N * q + j < W) o[j] = a[j];
  }
}

struct RowGeom {
  int Wo;    // groups of 8 outputs per row
  int nch;   // chunks of 8 taps (the last one a half chunk when tail4)
  int Pw;    // padded row pitch of P, a multiple of 8
  bool tail4;  // the taps, padded to a multiple of 4, end in a chunk of 4
};
__host__ __device__ __forceinline__ RowGeom row_geom(int W, int kx) {
  RowGeom g;
  g.Wo = (W + 7) >> 3;
  g.nch = (2 * kx + 1 + 7) >> 3;
  g.Pw = 8 * (g.Wo + g.nch + 1);
  g.tail4 = ((2 * kx + 1 + 3) & 7) == 4;
  return g;
}

// zero the halo columns [0, kx) and [kx + W, pitch) of every row of P
__device__ __forceinline__ void zero_halo(float *P, int R, int W, int kx, int pitch) {
  const int per_row = pitch - W;
  for (int i = threadIdx.x; i < R * per_row; i += blockDim.x) {
    const int r = i / per_row;
    const int c = i - r * per_row;
    P[r * pitch + (c < kx ? c : c + W)] = 0.0f;
  }
}

// truncated x filter (multi_array_filter.hpp:277-288) of every row of P:
// eight outputs per lane, taps in chunks of eight (zero padded), a 16-float
// window sliding along the row in two 16-byte LDS reads per chunk; writes
// row y of T (row pitch tp, a multiple of 32: the outputs past W land in the
// padding)
// NCH chunks known at compile time: the chunk loop unrolls, so the sliding
// window is renamed instead of copied.  With g.tail4 the last chunk runs its
// first 4 taps only (the others are the zero padding: an fmaf with a zero tap
// leaves the sum as it is)
template <int NCH>
__device__ __forceinline__ void xfilter_rows_n(const float *P, const float *taps_x, float *T, int R, int tp,
                                               long long plane, int y, const RowGeom &g) {
  const bool tail4 = g.tail4;
  const int n_items = R * g.Wo;
  const float inv_wo = 1.0f / (float)g.Wo;
  for (int item = threadIdx.x; item < n_items; item += blockDim.x) {
    int ro = (int)((float)item * inv_wo);
    if (ro * g.Wo > item) --ro;
    if ((ro + 1) * g.Wo <= item) ++ro;
    const int q = item - ro * g.Wo;
    // rows of P start on 32-byte boundaries (Pw is a multiple of 8)
    const float4 *P4 = reinterpret_cast<const float4 *>(
        __builtin_assume_aligned(P + ro * g.Pw + 8 * q, 16));
    float a[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) a[i] = 0.0f;
    float4 w0 = P4[0], w1 = P4[1];
    // the taps are re-read per item through the scalar cache rather than held
    // in vector registers for the whole loop
    const float *tx = taps_x;
    asm volatile("" : "+s"(tx));
#pragma unroll
    for (int c = 0; c < NCH - 1; ++c) {
      const float4 w2 = P4[2 * c + 2], w3 = P4[2 * c + 3];
      const float win[16] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w,
                             w2.x, w2.y, w2.z, w2.w, w3.x, w3.y, w3.z, w3.w};
      float f[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) f[u] = tx[8 * c + u];
#pragma unroll
      for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int i = 0; i < 8; ++i) a[i] = fmaf(win[i + u], f[u], a[i]);
      w0 = w2;
      w1 = w3;
    }
    {  // the last chunk: 4 or 8 taps
      constexpr int c = NCH - 1;
      const float4 w2 = P4[2 * c + 2];
      float f[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) f[u] = tx[8 * c + u];
      if (tail4) {
        const float win[12] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w, w2.x, w2.y, w2.z, w2.w};
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int i = 0; i < 8; ++i) a[i] = fmaf(win[i + u], f[u], a[i]);
      } else {
        const float4 w3 = P4[2 * c + 3];
        const float win[16] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w,
                               w2.x, w2.y, w2.z, w2.w, w3.x, w3.y, w3.z, w3.w};
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
          for (int i = 0; i < 8; ++i) a[i] = fmaf(win[i + u], f[u], a[i]);
      }
    }
    float *trow = T + ro * plane + (long long)y * tp;
    const int x0 = 8 * q;
    *reinterpret_cast<float4 *>(trow + x0) = make_float4(a[0], a[1], a[2], a[3]);
    *reinterpret_cast<float4 *>(trow + x0 + 4) = make_float4(a[4], a[5], a[6], a[7]);
  }
}

__device__ __forceinline__ void xfilter_rows(const float *P, const float *taps_x, float *T, int R, int tp,
                                             long long plane, int y, const RowGeom &g) {
  switch (g.nch) {  // half widths up to 43 (the filters of sigma <= 14.3 px)
    case 1: xfilter_rows_n<1>(P, taps_x, T, R, tp, plane, y, g); return;
    case 2: xfilter_rows_n<2>(P, taps_x, T, R, tp, plane, y, g); return;
    case 3: xfilter_rows_n<3>(P, taps_x, T, R, tp, plane, y, g); return;
    case 4: xfilter_rows_n<4>(P, taps_x, T, R, tp, plane, y, g); return;
    case 5: xfilter_rows_n<5>(P, taps_x, T, R, tp, plane, y, g); return;
    case 6: xfilter_rows_n<6>(P, taps_x, T, R, tp, plane, y, g); return;
    case 7: xfilter_rows_n<7>(P, taps_x, T, R, tp, plane, y, g); return;
    case 8: xfilter_rows_n<8>(P, taps_x, T, R, tp, plane, y, g); return;
    case 9: xfilter_rows_n<9>(P, taps_x, T, R, tp, plane, y, g); return;
    case 10: xfilter_rows_n<10>(P, taps_x, T, R, tp, plane, y, g); return;
    case 11: xfilter_rows_n<11>(P, taps_x, T, R, tp, plane, y, g); return;
    default: break;
  }
  const int n_items = R * g.Wo;
  const float inv_wo = 1.0f / (float)g.Wo;
  for (int item = threadIdx.x; item < n_items; item += blockDim.x) {
    int ro = (int)((float)item * inv_wo);
    if (ro * g.Wo > item) --ro;
    if ((ro + 1) * g.Wo <= item) ++ro;
    const int q = item - ro * g.Wo;
    const float4 *P4 = reinterpret_cast<const float4 *>(P + ro * g.Pw) + 2 * q;
    float a[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) a[i] = 0.0f;
    float4 w0 = P4[0], w1 = P4[1];
    for (int c = 0; c < g.nch; ++c) {
      const float4 w2 = P4[2 * c + 2], w3 = P4[2 * c + 3];
      const float win[16] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w,
                             w2.x, w2.y, w2.z, w2.w, w3.x, w3.y, w3.z, w3.w};
      float f[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) f[u] = taps_x[8 * c + u];
#pragma unroll
      for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int i = 0; i < 8; ++i) a[i] = fmaf(win[i + u], f[u], a[i]);
      w0 = w2;
      w1 = w3;
    }
    float *trow = T + ro * plane + (long long)y * tp;
    const int x0 = 8 * q;
    *reinterpret_cast<float4 *>(trow + x0) = make_float4(a[0], a[1], a[2], a[3]);
    *reinterpret_cast<float4 *>(trow + x0 + 4) = make_float4(a[4], a[5], a[6], a[7]);
  }
}

// Forward offsets of output slice ro (so = J.shifts + 4 R: the x offsets at
// so, the y offsets at so + 2 R) at row ys / column x.  SPLIT: the warp's
// offset changes once along an axis, by the step at so + 5 R (x) / so + 7 R
// (y) from the break at so + 4 R / so + 6 R on.
template <int R, bool SPLIT>
__device__ __forceinline__ int fwd_oy(const int *__restrict__ shifts, int so, int ro, int ys) {
  int oy = shifts[so + 2 * R + ro];  // masked rotations have no source row
  if (SPLIT && ys >= shifts[so + 6 * R + ro]) oy += shifts[so + 7 * R + ro];
  return oy;
}
template <int R, bool SPLIT>
__device__ __forceinline__ int fwd_ox(const int *__restrict__ shifts, int so, int ro, int x) {
  int ox = shifts[so + ro];
  if (SPLIT && x >= shifts[so + 4 * R + ro]) ox += shifts[so + 5 * R + ro];
  return ox;
}

// The R raw source values of column x, row y.  Per OUTPUT slice: the source
// slice is ro - delta (clamped into [0, R) at so + 3 R), read at (y + oyo, x +
// oxo) with oxo at so, oyo at so + 2 R (so = J.shifts + 4 R); slices without a
// source, or with a masked one, carry a row offset that fails the bounds test.
// Forward warp (objectdetect_findrot.cpp:342-359): every load unconditional (a
// slice without a source reads its clamped slice, a column outside the grid
// its nearest column), all R of them issued before any is used; the row
// address on the scalar unit, the column a byte offset from it.  The offsets
// are read through the scalar cache here and again by rowpass_exp (an empty
// asm keeps the reads apart) rather than held in scalar registers.
template <int R, bool SPLIT>
__device__ __forceinline__ void rowpass_gather(const MsgJob &J, const int *__restrict__ shifts, const float *src, int y,
                                               const int x, float (&v)[R]) {
  const int H = J.H, W = J.W;
  const int Ps = J.src.pitch;
  int HW = __builtin_amdgcn_readfirstlane(H * Ps);  // R * H * pitch < 2^31 is checked when the plan is built
  int so = __builtin_amdgcn_readfirstlane(J.shifts + 4 * R);
  const int ys = __builtin_amdgcn_readfirstlane(y);  // uniform: the row offsets on the scalar unit
  asm volatile("" : "+s"(so), "+s"(HW));
  const int x4 = x * 4, xmax4 = (W - 1) * 4;
#pragma unroll
  for (int ro = 0; ro < R; ++ro) {
    const int yy = min(max(ys + fwd_oy<R, SPLIT>(shifts, so, ro, ys), 0), H - 1);
    const char *srow = reinterpret_cast<const char *>(src + (unsigned)(shifts[so + 3 * R + ro] * HW + yy * Ps));
    const int xx4 = min(max(x4 + fwd_ox<R, SPLIT>(shifts, so, ro, x) * 4, 0), xmax4);
    v[ro] = *reinterpret_cast<const float *>(srow + (unsigned)xx4);
  }
}

// Masks, then exp(b - M) (:362-365) as 2^((b - M) log2 e) on the hardware exp2
// (values below 2^-126 flush to zero, where the reference's expf returns
// subnormals).  A source pixel outside the grid (the warp's LOG_ZERO fill) and
// a masked unary state (a masked rotation, or a column in the masked strips)
// both take e_fill = exp(LOG_ZERO - M): a masked rotation's row offset fails the
// test, the strips narrow the columns' range.
template <int R, bool SPLIT>
__device__ __forceinline__ void rowpass_exp(const MsgJob &J, const int *__restrict__ shifts, float negM, float e_fill,
                                            int y, const int x, const float (&v)[R], float (&e)[R]) {
  const int H = J.H, W = J.W;
  const bool zero_src = J.src_kind == kSrcZero;
  int so = __builtin_amdgcn_readfirstlane(J.shifts + 4 * R);
  const int ys = __builtin_amdgcn_readfirstlane(y);
  asm volatile("" : "+s"(so));
  const int lo = J.src_kind == kSrcUnary ? J.src_mask.strip : 0;
  const unsigned span = (unsigned)max(W - 2 * lo, 0);  // columns lo .. W - lo - 1 are read
#pragma unroll
  for (int ro = 0; ro < R; ++ro) {
    const bool row_ok = (unsigned)(ys + fwd_oy<R, SPLIT>(shifts, so, ro, ys)) < (unsigned)H;
    // a leaf without a detector has the zero log posterior (b = 0); the
    // exponential is computed for every lane (an empty asm keeps it out of a
    // branch), then selected
    float ev = __builtin_amdgcn_exp2f(((zero_src ? 0.0f : v[ro]) + negM) * kLog2eF);
    asm volatile("" : "+v"(ev));
    const bool ok = row_ok && (unsigned)(x + fwd_ox<R, SPLIT>(shifts, so, ro, x) - lo) < span;
    e[ro] = ok ? ev : e_fill;
  }
}

// Rotation filter of a column's values: the output slices G * RG .. (G + 1) *
// RG - 1 are written to out (pitch apart).
template <int R, int RG, int G, class Pitch>
__device__ __forceinline__ void rowpass_rotate(const MsgJob &J, const float *__restrict__ taps, const float (&e)[R],
                                               float *out, Pitch pitch) {
  if (J.rot_mode == kRotFilter) {
    RotDispatch<R, (R % 2 == 1) ? R - 2 : R - 1, G * RG, (G + 1) * RG>::run(J.rot_len, e, taps + J.taps_r, out, pitch);
  } else if (J.rot_mode == kRotCopy) {
#pragma unroll
    for (int k = 0; k < RG; ++k) out[k * pitch] = e[G * RG + k];
  } else {
#pragma unroll
    for (int k = 0; k < RG; ++k) out[k * pitch] = 0.0f;
  }
}

// Row pass for a rotation count fixed at compile time (24, and the
// reference's default 48), row y: lane t owns the columns x = t (mod
// blockDim.x); the slice groups go through P and the x filter one after
// another.  MFMA: the x filter on the matrix cores; with one column per lane
// its values stay in registers from group to group.  Else (row_on_mfma) on the
// vector unit.  Bound by latency: the filter, the exponentials and
// rotation filter, and the gather with the stores overlap between the 4 blocks
// that fit a CU only in part: 899 us per launch of 32 images of 300x300x24 with the filter on the
// vector unit, some 730 now (467 without the filter, which is what its 2.49 GB
// take at the rate of a copy).  48 slices: 118 -> 75 us per launch of an
// image of 300x300.
// KIND: the filter on the vector unit, on the matrix cores, or there with rows
// of more columns than threads, where waves past the row do nothing (a test that
// the narrower rows do without: with it 382 becomes 402 us per sweep of 8 images
// of 200x300x24; without it 834 instead of 736 at 200x520).
enum RowKind : int { kRowVector = 0, kRowMfma = 1, kRowMfmaWide = 2 };

template <int R, bool SPLIT, int KIND>
__device__ __forceinline__ void rowpass_body(const Bases &b, const MsgJob &J, const float *__restrict__ taps,
                                             const int *__restrict__ shifts, float *P, int y, int nt) {
  const int H = J.H, W = J.W;
  const int kx = J.kx;
  const RowGeom g = row_geom(W, kx);
  constexpr bool MFMA = KIND != kRowVector;
  constexpr int RG = MFMA ? row4_slices(R) : R / row_groups(R), NG = R / RG, Q = row4_pitch(RG);
  float *t4 = P + row4_floats(RG, W, kx);
  unsigned *bad = reinterpret_cast<unsigned *>(t4 + 4 * tap4_pitch(kx));  // P may hold a non-finite value
  if (MFMA) {
    // zeros before the row and as far behind it as a window reaches whose
    // first output is inside
    const int tail = (kx + W) * Q, end = (W + 4 * tap4_chunks(kx)) * Q;
    for (int i = threadIdx.x; i < kx * Q; i += nt) P[i] = 0.0f;
    for (int i = tail + (int)threadIdx.x; i < end; i += nt) P[i] = 0.0f;
    if (threadIdx.x == 0) *bad = 0u;
  } else {
    zero_halo(P, RG, W, kx, g.Pw);
  }

  const float M = key2f(*max_key(b, J.src_key));
  const float negM = -M;
  // exp(LOG_ZERO - M): the warp's fill value, on the path of every other value
  const float e_fill = __builtin_amdgcn_exp2f((kLogZero + negM) * kLog2eF);
  const float *src = cptr(b, J.src);
  float *T = mptr(b, J.tmp);
  const long long plane = (long long)H * J.tpitch;
  const bool one = MFMA && W <= nt;
  const float tap0 = MFMA ? tap4_load(taps + J.taps_x, kx) : 0.0f;
  float e[R];
  unsigned bits = 0u;
  auto values = [&](int x) {
    float v[R];
    rowpass_gather<R, SPLIT>(J, shifts, src, y, x, v);
    rowpass_exp<R, SPLIT>(J, shifts, negM, e_fill, y, x, v, e);
    if (MFMA) {
#pragma unroll
      for (int r = 0; r < R; ++r) bits = max_bits(bits, e[r]);
    }
  };
  auto group = [&](auto gc) {
    constexpr int G = decltype(gc)::value;
    if (G > 0) __syncthreads();  // every item of the group before is filtered
    for (int x0 = 0; x0 < W; x0 += nt) {
      const int x = x0 + (int)threadIdx.x;
      if (KIND != kRowMfma && __builtin_amdgcn_readfirstlane(x) >= W) break;
      if (!one || G == 0) values(min(x, W - 1));  // past the row: its last column again
      if (x < W) {
        if (MFMA) rowpass_rotate<R, RG, G>(J, taps, e, P + (kx + x) * Q, std::integral_constant<int, 1>{});
        else rowpass_rotate<R, RG, G>(J, taps, e, P + kx + x, g.Pw);
      }
    }
    if (MFMA && G == 0) {
      tap4_store(t4, tap0, taps + J.taps_x, kx, nt);
      __syncthreads();  // the flag is clear
    }
    if (MFMA && bits >= kRowNonFinite) *bad = 1u;
    __syncthreads();
    float *Tg = T + G * RG * plane;
    if (!MFMA) xfilter_rows(P, taps + J.taps_x, Tg, RG, J.tpitch, plane, y, g);
    else if (__builtin_amdgcn_readfirstlane(*bad) == 0u) xfilter4<RG>(P, t4, kx, Tg, J.tpitch, plane, y, W, nt);
    else xfilter_plain<RG>(P, taps + J.taps_x, kx, Tg, J.tpitch, plane, y, W, nt);
  };
  group(std::integral_constant<int, 0>{});
  if constexpr (NG > 1) group(std::integral_constant<int, 1>{});
  if constexpr (NG > 2) {
    group(std::integral_constant<int, 2>{});
    group(std::integral_constant<int, 3>{});
  }
}

// 24 slices on the matrix cores: at most 96 scalar registers, which the register
// count that seven waves a SIMD allow comes to.  More are allotted as 112, for
// seven waves instead of eight, and the first SIMD of a CU then takes no fourth
// block of five waves, two of which each block puts there: 2703 instead of 2835
// us of all row passes of 32 images of 300x300.
template <int R, bool SPLIT, int KIND>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(R == 24 && KIND != kRowVector ? 7 : 2))) void k_rowpass_r(Bases b, const MsgJob *__restrict__ jobs,
                                                   const float *__restrict__ taps, const int *__restrict__ shifts) {
  extern __shared__ float4 lds4[];
  float *P = reinterpret_cast<float *>(lds4);
  const int nt = (int)blockDim.x;
  unsigned bx, by;
  xcd_block(bx, by);
  const MsgJob &J = jobs[by];
  if (skip_inst(b, J.inst)) return;
  const int y = (int)bx;
  if (y >= J.H) return;
  // a warp whose offset changes along an axis takes the SPLIT variants
  if (SPLIT && J.split != 0) rowpass_body<R, SPLIT, KIND>(b, J, taps, shifts, P, y, nt);
  else rowpass_body<R, false, KIND>(b, J, taps, shifts, P, y, nt);
}

// Row pass for any rotation count: the exponentiated column goes through an
// LDS buffer E[R][Wa] before the rotation filter.
__global__ __launch_bounds__(512) void k_rowpass_any(Bases b, const MsgJob *__restrict__ jobs,
                                                     const float *__restrict__ taps, const int *__restrict__ shifts,
                                                     int R) {
  extern __shared__ float4 lds4[];
  unsigned bx, by;
  xcd_block(bx, by);
  const MsgJob &J = jobs[by];
  if (skip_inst(b, J.inst)) return;
  const int y = (int)bx;
  const int H = J.H, W = J.W;
  if (y >= H) return;
  const int kx = J.kx;
  const RowGeom g = row_geom(W, kx);
  const int Wa = (W + 3) & ~3;
  float *E = reinterpret_cast<float *>(lds4);
  float *P = E + R * Wa;
  zero_halo(P, R, W, kx, g.Pw);

  const float M = key2f(*max_key(b, J.src_key));
  const float negM = -M;
  const float e_fill = expf(kLogZero + negM);
  const float *src = cptr(b, J.src);
  const int Ps = J.src.pitch;
  const long long HW = (long long)H * Ps;
  const int *fox = shifts + J.shifts;
  const int *foy = fox + R;
  const int n_rot = J.rot_len >> 1;
  const float *fr = taps + J.taps_r;
  for (int x = threadIdx.x; x < W; x += blockDim.x) {
    for (int ro = 0; ro < R; ++ro) {
      const int rs = ro - J.delta;
      float e = e_fill;
      if (rs >= 0 && rs < R) {
        int oy = foy[rs], ox = fox[rs];
        if (J.split) {  // the breaks and steps by output slice
          const int *sp = shifts + J.shifts + 8 * R;
          if (x >= sp[ro]) ox += sp[R + ro];
          if (y >= sp[2 * R + ro]) oy += sp[3 * R + ro];
        }
        const int yy = y + oy;
        const int xx = x + ox;
        if (yy >= 0 && yy < H && xx >= 0 && xx < W) {
          float v;
          if (J.src_kind == kSrcZero) v = 0.0f;
          else if (J.src_kind == kSrcUnary && masked(J.src_mask, rs, xx, W)) v = kLogZero;
          else v = src[rs * HW + (long long)yy * Ps + xx];
          e = __builtin_amdgcn_exp2f((v + negM) * kLog2eF);
        }
      }
      E[ro * Wa + x] = e;
    }
    // the column was written by this thread: no barrier needed
    for (int ro = 0; ro < R; ++ro) {
      float acc;
      if (J.rot_mode == kRotFilter) {
        acc = 0.0f;
        for (int j = 0; j < J.rot_len; ++j) {
          int rr = ro - n_rot + j;
          rr = rr < 0 ? rr + R : (rr >= R ? rr - R : rr);
          acc = fmaf(E[rr * Wa + x], fr[j], acc);
        }
      } else if (J.rot_mode == kRotCopy) {
        acc = E[ro * Wa + x];
      } else {
        acc = 0.0f;
      }
      P[ro * g.Pw + kx + x] = acc;
    }
  }
  __syncthreads();
  xfilter_rows(P, taps + J.taps_x, mptr(b, J.tmp), R, J.tpitch, (long long)H * J.tpitch, y, g);
}

// -------------------------------------------------------------- k_colpass
// One block per (message, slice r, strip of 64 columns); it walks down the
// strip in tiles of 4 ROWS output rows.  Each tile stages the source rows it
// needs (4 ROWS + padded taps, zero outside the grid, inverse shift folded
// into the origin) in LDS; each of the four waves then computes ROWS rows,
// one column per lane, with a ROWS-row register ring fed from LDS.  Taps run
// in chunks of 8 (the tap pool is zero padded), so the ring indices are
// static.  ROWS = 8 (the default) or 16; the outputs are the same bit for bit.
//
// MFMA: the filter on the matrix cores, the staged rows a ring in LDS (nothing
// moves from tile to tile; with the move 1-4% slower).  Bound by memory at some
// 4 TB/s of scattered grids, and by the barriers between filter and epilogue;
// us per launch of 32 images of 300x300x24, by destination
// kind, vector unit / MFMA 8 rows / 16 rows: downward middle 1340 / 1286 /
// 1278, downward leaf 1055 / 948 / 1057, up root 978 / 870 / 935, up node 825
// / 780 / 838.  The vector unit's filter is left for taps so many that the
// operand does not fit LDS beside the rows.

constexpr int kColTileX = 64;
constexpr int kColWaves = 4;
constexpr int kColRowsDefault = 8;

__host__ __device__ __forceinline__ int col_padded_taps(int ky) { return (2 * ky + 1 + 3) & ~3; }
__host__ __device__ __forceinline__ int col_tile_rows(int ky, int rows) { return kColWaves * rows + col_padded_taps(ky); }
// rows moved per thread and pass when a tile hands its halo to the next one
constexpr int kColMove = 24;

// N (8 or 4) taps of the y filter starting at tap t; PH is the ring phase (t % ROWS)
template <int PH, int N, int ROWS>
__device__ __forceinline__ void col_chunk(float (&acc)[ROWS], float (&buf)[ROWS], const float *fy, const float *tw,
                                          int t) {
  float f[N];
#pragma unroll
  for (int u = 0; u < N; ++u) f[u] = fy[t + u];
#pragma unroll
  for (int u = 0; u < N; ++u) {
#pragma unroll
    for (int i = 0; i < ROWS; ++i) acc[i] = fmaf(buf[(i + u + PH) & (ROWS - 1)], f[u], acc[i]);
    buf[(u + PH) & (ROWS - 1)] = tw[(t + u + ROWS) * kColTileX];
  }
}

// The y filter of a wave's ROWS rows x 64 columns on the MFMA: lane = column,
// acc[g] = rows 4 g .. 4 g + 3, which take the taps f[k - i] against row k on
// from the wave's first; a ring of ROWS / 4 row quads in registers, each read
// once for all groups from the tile's ring of n rows (a multiple of 4; col:
// this lane's column, row: the wave's first row).  The quads read behind the
// tile's are the ring's oldest and multiplied by nothing.
template <int ROWS>
__device__ __forceinline__ void yfilter4(const float *col, int row, int n, const float *t4, int ky, float (&a)[ROWS]) {
  constexpr int G = ROWS / 4;
  const int NT = tap4_chunks(ky);
  const float4 *tv = reinterpret_cast<const float4 *>(t4 + (threadIdx.x & 3) * tap4_pitch(ky));
  f32x4_t acc[G];
  float x[G][4];
  auto quad = [&](float (&q)[4]) {
    const float *p = col + row * kColTileX;
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = p[i * kColTileX];
    row += 4;
    if (row >= n) row -= n;
  };
#pragma unroll
  for (int g = 0; g < G; ++g) {
    acc[g] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    quad(x[g]);
  }
  auto step = [&](auto uc) {
    constexpr int u = decltype(uc)::value;
    const float4 t = *tv++;
#pragma unroll
    for (int g = 0; g < G; ++g) acc[g] = mfma4(t.x, x[(u + g) % G][0], acc[g]);
#pragma unroll
    for (int g = 0; g < G; ++g) acc[g] = mfma4(t.y, x[(u + g) % G][1], acc[g]);
#pragma unroll
    for (int g = 0; g < G; ++g) acc[g] = mfma4(t.z, x[(u + g) % G][2], acc[g]);
#pragma unroll
    for (int g = 0; g < G; ++g) acc[g] = mfma4(t.w, x[(u + g) % G][3], acc[g]);
    quad(x[u]);
  };
  using std::integral_constant;
  int c = 0;
  for (; c + G <= NT; c += G) {
    step(integral_constant<int, 0>{});
    step(integral_constant<int, 1>{});
    if constexpr (G == 4) {
      step(integral_constant<int, 2>{});
      step(integral_constant<int, 3>{});
    }
  }
  if (c < NT) step(integral_constant<int, 0>{});
  if constexpr (G == 4) {
    if (c + 1 < NT) step(integral_constant<int, 1>{});
    if (c + 2 < NT) step(integral_constant<int, 2>{});
  }
#pragma unroll
  for (int i = 0; i < ROWS; ++i) a[i] = acc[i >> 2][i & 3];
}

// The same of a tile holding a non-finite value, each row over its own taps
// (padded to a multiple of four, Lp, with zeros).
template <int ROWS>
__device__ __forceinline__ void yfilter_plain(const float *col, int row, int n, const float *__restrict__ fy, int Lp,
                                              float (&a)[ROWS]) {
  auto next = [&] {
    const float v = col[row * kColTileX];
    if (++row == n) row = 0;
    return v;
  };
  float win[ROWS];
#pragma unroll
  for (int i = 0; i < ROWS; ++i) win[i] = next();
#pragma unroll 2
  for (int t = 0; t < Lp; t += 4) {
    float behind[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) behind[j] = next();
    plain_taps<ROWS>(a, win, behind, fy + t);
  }
}

// The caller's accumulation is a template (EPI, one variant per destination
// kind), so every load of a tile is unconditional straight-line code: the
// epilogue operands first, then the next tile's rows (always loaded, clamped
// into the grid, zeroed when they reach LDS), and the epilogue waits for its
// operands only.
// SPLIT: the launch may hold a split warp (J.split), whose inverse offsets
// change once along x (per lane) or y (a second segment of rows)
template <int EPI, int ROWS, bool SPLIT, bool MFMA>
__device__ __forceinline__ void colpass_strip(const Bases &b, const MsgJob &J, const float *__restrict__ taps,
                                              const int *__restrict__ shifts, int R, int r, int xt, int ya, int yb,
                                              float *tile) {
  constexpr int kColRows = ROWS;
  constexpr int kColTileY = kColRows * kColWaves;
  constexpr bool kNeedU = Epi<EPI>::kNeedU;
  constexpr bool kNeedB = Epi<EPI>::kNeedB;
  const int H = J.H, W = J.W;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int x = xt * kColTileX + lane;
  const bool xin = x < W;
  const int xo = xin ? x : W - 1;

  // inverse offsets of slice r (a split warp: the lane's column past the x
  // break takes the x step, the rows from the y break on the y step)
  int ox = shifts[J.shifts + 2 * R + r];
  const int oy0 = shifts[J.shifts + 3 * R + r];
  const bool split = SPLIT && J.split != 0;
  if (split && x >= shifts[J.shifts + 12 * R + r]) ox += shifts[J.shifts + 13 * R + r];
  const int ybrk = split ? shifts[J.shifts + 14 * R + r] : H;
  const int ystep = split ? shifts[J.shifts + 15 * R + r] : 0;
  const bool col_ok = xin && x + ox >= 0 && x + ox < W;
  int tp = J.tpitch;
  const float *Tr = cptr(b, J.tmp) + (long long)r * H * tp;
  const int ky = J.ky;
  const int Lp = col_padded_taps(ky);
  const int nrows = col_tile_rows(ky, ROWS);
  const float *fy = taps + J.taps_y;
  // MFMA: the tap operand and a flag (a non-finite value was staged: the
  // strip goes on on the vector unit) behind the tile
  float *t4 = tile + nrows * kColTileX;
  unsigned *bad = reinterpret_cast<unsigned *>(t4 + 4 * tap4_pitch(ky));
  unsigned bits = 0u;
  if (MFMA) {
    tap4_store(t4, tap4_load(fy, ky), fy, ky, kColWaves * 64);
    if (threadIdx.x == 0) *bad = 0u;
    __syncthreads();
  }
  const float M = key2f(*max_key(b, J.src_key));
  // row pitches: pa of dst (and of the unary a marginal adds), pb of the
  // grids at the other pitch (EpiPitch)
  const int pa = J.dst.pitch, pb = epi_pitch_b<EPI>(J);
  float *dst = mptr(b, J.dst) + r * H * pa;
  const float *dun = kNeedU ? cptr(b, J.dst_unary) + r * H * J.dst_unary.pitch : dst;
  float *dst2 = kNeedB ? mptr(b, J.dst2) + r * H * pb : dst;
  const float *bel = kNeedB ? cptr(b, J.dst_bel) + r * H * pb : dst;
  const bool leaf_u = J.dst_base == 1;  // a leaf's marginal: detected part (else its base is 0)
  const bool xmask = ((J.dst_mask.rot_bits >> r) & 1ull) || x < J.dst_mask.strip || x >= W - J.dst_mask.strip;
  // column loaded by this thread's lane slot (loads outside the grid go to its
  // nearest row and column; those values are zeroed when they reach LDS)
  const int lcol = xt * kColTileX + lane + ox;
  const bool lcol_ok = x < W && lcol >= 0 && lcol < W;
  const float *Tc = Tr + min(max(lcol, 0), W - 1);
  auto src_raw = [&](int row) -> float { return Tc[(long long)min(max(row, 0), H - 1) * tp]; };
  auto src_ok = [&](int row) -> bool { return lcol_ok && row >= 0 && row < H; };

  // The output rows [ya, yb) run in segments of one inverse row offset oy: up
  // to ybrk and, for a split warp, from it on.  Within a segment, tile t holds source
  // rows s_t + [0, nrows), s_t = ylo + kColTileY t + oy - ky.  Tile t+1 shares rows
  // [kColTileY, nrows) of tile t, which stay where they are in the ring (MFMA) or
  // move to [0, Lp) in LDS, and needs kColTileY new rows, fetched into registers
  // while tile t is filtered; in the ring they take the place of the oldest.
  constexpr int kNew = kColTileY / kColWaves;  // new rows per thread
  Epi<EPI> acc;
  // (the padding columns of the plan's grids are left unwritten here: the
  // extra stores cost what the whole lines save, 7.48 ms per sweep of 32
  // 300x300x24 images either way, and one image 352 -> 359 us)
  unsigned Wb = (unsigned)pa * 4u, Wb2 = (unsigned)pb * 4u;
  for (int seg = 0; seg < (SPLIT ? 2 : 1); ++seg) {
    const int ylo = seg == 0 ? ya : max(ya, ybrk), yhi = seg == 0 ? min(yb, ybrk) : yb;
    if (ylo >= yhi) continue;
    const int oy = seg == 0 ? oy0 : oy0 + ystep;
    if (seg) __syncthreads();  // every wave is done with the first segment's tile
    int base = 0;  // MFMA: ring row of the tile's first row
    for (int rr = wave; rr < nrows; rr += kColWaves) {
      const int row = ylo + oy - ky + rr;
      const float raw = src_raw(row), v = src_ok(row) ? raw : 0.0f;
      bits = max_bits(bits, v);
      tile[rr * kColTileX + lane] = v;
    }
    if (MFMA && bits >= kNonFinite) *bad = 1u;
    __syncthreads();

    for (int ty0 = ylo; ty0 < yhi; ty0 += kColTileY) {
      asm volatile("" : "+s"(Wb), "+s"(Wb2), "+s"(tp));  // per-row offsets recomputed per tile, not hoisted
      const bool more = ty0 + kColTileY < yhi;
      const int y0 = ty0 + wave * kColRows;
      const unsigned eb0 = (unsigned)(y0 * pa + xo) * 4u;
      const unsigned ebs0 = Epi<EPI>::kSide ? (unsigned)(y0 * pb + xo) * 4u : eb0;
      // the unary of the part written, loaded now so that its latency hides
      // behind the filter; the stored belief of the five-grid downward epilogue
      // is loaded after the filter (held through it, its 16 registers make the
      // kernel spill at 128 VGPRs)
      float pu[kColRows], pbel[kColRows];
      if (kNeedU || kNeedB) {
        // the unary: at the side pitch for a chain-node belief, else at dst's
        constexpr bool kUs = EPI == kEpiUpNodeU;
        if (ty0 + kColTileY <= H) {
#pragma unroll
          for (int i = 0; i < kColRows; ++i) {
            const unsigned eb = kUs ? ebs0 + (unsigned)i * Wb2 : eb0 + (unsigned)i * Wb;
            if (kNeedU) pu[i] = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(dun) + eb);
          }
        } else {
#pragma unroll
          for (int i = 0; i < kColRows; ++i) {
            const unsigned eb = (unsigned)(min(y0 + i, H - 1) * (kUs ? pb : pa) + xo) * 4u;
            if (kNeedU) pu[i] = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(dun) + eb);
          }
        }
      }
      // the next tile's new rows (in the last tile: clamped rows, unused)
      const int s1 = ty0 + kColTileY + oy - ky + Lp;
      float pre[kNew];
#pragma unroll
      for (int k = 0; k < kNew; ++k) pre[k] = src_raw(s1 + wave + kColWaves * k);

      const float *tw = tile + wave * kColRows * kColTileX + lane;
      float a[kColRows] = {};
      int row0 = base + wave * kColRows;  // of the ring (MFMA)
      if (row0 >= nrows) row0 -= nrows;
      if (MFMA && __builtin_amdgcn_readfirstlane(*bad) == 0u) {
        yfilter4<ROWS>(tile + lane, row0, nrows, t4, ky, a);
      } else if (MFMA) {
        yfilter_plain<ROWS>(tile + lane, row0, nrows, fy, Lp, a);
      } else {
        float buf[kColRows];
#pragma unroll
        for (int i = 0; i < kColRows; ++i) {
          a[i] = 0.0f;
          buf[i] = tw[i * kColTileX];
        }
        // taps in runs of the ring's period, then a tail (the tap count is
        // padded to a multiple of 4 with zero taps)
        int t0 = 0;
        for (; t0 + 8 <= Lp; t0 += 8) col_chunk<0, 8, ROWS>(a, buf, fy, tw, t0);
        if (Lp - t0 == 4) col_chunk<0, 4, ROWS>(a, buf, fy, tw, t0);
      }

      if (kNeedB) {
#pragma unroll
        for (int i = 0; i < kColRows; ++i) {
          const unsigned eb = (unsigned)(min(y0 + i, H - 1) * pb + xo) * 4u;
          pbel[i] = *reinterpret_cast<const float *>(reinterpret_cast<const char *>(bel) + eb);
        }
      }
#pragma unroll
      for (int i = 0; i < kColRows; ++i) {
        const int y = y0 + i;
        // log, +M (:432-435); inverse warp (:437-448): outside -> LOG_ZERO
        const float msg = (col_ok && (unsigned)(y + oy) < (unsigned)H) ? log0(a[i]) + M : kLogZero;
        if (xin && y < yhi)
          acc.store(dst, dst2, eb0 + (unsigned)i * Wb, ebs0 + (unsigned)i * Wb2, msg, kNeedU ? pu[i] : 0.0f,
                    kNeedB ? pbel[i] : 0.0f, xmask, leaf_u);
      }
      if (more) {
        if (MFMA) {
          __syncthreads();  // every wave is done with the ring's oldest rows
        } else {
          // move rows [kColTileY, nrows) to [0, Lp), then store the prefetched rows
          for (int c0 = 0; c0 < Lp; c0 += kColMove * kColWaves) {
            float mv[kColMove];
            __syncthreads();  // every wave is done with this tile
#pragma unroll
            for (int k = 0; k < kColMove; ++k) {
              const int rr = c0 + wave + kColWaves * k;
              if (rr < Lp) mv[k] = tile[(kColTileY + rr) * kColTileX + lane];
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < kColMove; ++k) {
              const int rr = c0 + wave + kColWaves * k;
              if (rr < Lp) tile[rr * kColTileX + lane] = mv[k];
            }
          }
        }
#pragma unroll
        for (int k = 0; k < kNew; ++k) {
          const int row = s1 + wave + kColWaves * k;
          const float v = src_ok(row) ? pre[k] : 0.0f;
          bits = max_bits(bits, v);
          int rr = (MFMA ? base : Lp) + wave + kColWaves * k;
          if (MFMA && rr >= nrows) rr -= nrows;
          tile[rr * kColTileX + lane] = v;
        }
        if (MFMA && bits >= kNonFinite) *bad = 1u;
        base += kColTileY;
        if (base >= nrows) base -= nrows;
        __syncthreads();
      }
    }
  }
  acc.flush(b, J, (long long)r * H * pa, tile);
}

// HI: the highest destination kind among the launch's jobs (the kernel holds
// only the epilogues up to it: 102-127 VGPRs below the five-grid downward
// one).  At most 128 VGPRs (4 waves per SIMD instead of 3): the five-grid
// epilogue fits without spilling vector registers once its stored belief is
// loaded after the filter (2.16 -> 1.33 ms per launch on 32 300x300x24
// grids; unbounded, at 156 VGPRs and 3 waves per SIMD, it takes 1.65 ms).
template <int HI, int ROWS, bool SPLIT, bool MFMA>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_colpass(
    Bases b, const MsgJob *__restrict__ jobs, const float *__restrict__ taps, const int *__restrict__ shifts, int R,
    int xtiles) {
  extern __shared__ float4 lds4[];
  float *tile = reinterpret_cast<float *>(lds4);
  unsigned bx, by;
  xcd_block(bx, by);
  const MsgJob &J = jobs[by];
  if (skip_inst(b, J.inst)) return;
  const int r = (int)bx / xtiles;
  const int xt = (int)bx - r * xtiles;
  if (xt * kColTileX >= J.W) return;
  int ya, yb;
  col_part(J.H, kColWaves * ROWS, ya, yb);
  if (ya >= yb) return;
  const int kind = epi_kind(J);
  if (HI == kEpiUpRoot || kind == kEpiUpRoot)
    colpass_strip<kEpiUpRoot, ROWS, SPLIT, MFMA>(b, J, taps, shifts, R, r, xt, ya, yb, tile);
  else if (HI == kEpiUpNode || kind == kEpiUpNode)
    colpass_strip<kEpiUpNode, ROWS, SPLIT, MFMA>(b, J, taps, shifts, R, r, xt, ya, yb, tile);
  else if (HI == kEpiUpNodeU || kind == kEpiUpNodeU)
    colpass_strip<kEpiUpNodeU, ROWS, SPLIT, MFMA>(b, J, taps, shifts, R, r, xt, ya, yb, tile);
  else if (HI == kEpiDownLeaf || kind == kEpiDownLeaf)
    colpass_strip<kEpiDownLeaf, ROWS, SPLIT, MFMA>(b, J, taps, shifts, R, r, xt, ya, yb, tile);
  else
    colpass_strip<kEpiDownMid, ROWS, SPLIT, MFMA>(b, J, taps, shifts, R, r, xt, ya, yb, tile);
}

// ----------------------------------------------------------------- k_root

// The root belief, its marginal and the children's log_from_root of a block of
// 128 pixels, 8 waves: two tiles of 64, a quarter of the rotations each, so
// that an image of 112x128 has 112 blocks of 6 steps in a row rather than 56 of
// 24.  Bound by memory (12 grids, 3.32 GB in 716 us for 32 images of
// 300x300x24), on one image by latency.  us before (a wave walks all rotations
// and raises its own keys) / now: 26 / 11.7 (112x128x24), 99 / 48.6 (300x300x48),
// 497 / 431 (6 uneven x48), 740 / 716 (32 300x300x24).  A block of 256 pixels:
// 13.7, 56, 425, 708; half the rotations per wave 18, 55, 443, 719.  Stores
// through the caches: odd grids' rows leave partial lines, which L2 merges;
// nontemporal ones took 394 instead of 302 us on an uneven batch, and 724 instead
// of 708 on the even one (blocks of 256 pixels).
//
// KC: the number of root children when it is at most 8 (fully unrolled),
// else kMaxRootChildren with the count read at run time.
// LSE64: the root posterior's log-sum-exp over rotations accumulated in FP64
// with a running maximum shift (the BF16 methods); otherwise in FP32 with
// no shift, as the reference sums expf (:713-726: a belief above ~88.7
// overflows to +inf there and here)
constexpr int kRootWaves = 4;  // per 64 pixels, a quarter of the rotations each
constexpr int kRootTiles = 2;  // 64-pixel tiles per block

template <int KC, bool LSE64>
__device__ __forceinline__ void root_pixels(const Bases &b, const RootJob &J, int R, int pix0, uint4 *red, float *bels) {
  const int H = J.H, W = J.W;
  const int HW = H * W;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = wv / kRootTiles, tile = wv % kRootTiles;
  const int r0 = wave * R / kRootWaves, r1 = (wave + 1) * R / kRootWaves;  // this wave's rotations
  const int pix = pix0 + tile * 64 + lane;
  const bool ok = pix < HW;
  const int pc = ok ? pix : HW - 1;  // loads of lanes past the end read the last pixel
  const int yc = pc / W;
  const int x = pc - yc * W;
  // the lanes walk the dense grids (unary, marginal, log_from_root, root
  // posterior: index r HW + pix), so each wave writes its rows' lines whole;
  // the upward messages are read from the plan's slots (row pitch pm)
  const int pm = J.msg[0].pitch;
  const int HPm = H * pm;
  const int pcm = yc * pm + x;
  const int K = KC <= 8 ? KC : J.K;
  const float *un = cptr(b, J.unary);
  float *marg = mptr(b, J.marginal);
  const bool posts = J.root_post.buf >= 0 && b.root;

  unsigned kmax[KC];
#pragma unroll
  for (int k = 0; k < KC; ++k) kmax[k] = 0u;
  unsigned long long amax = 0ull;
  unsigned second = 0u;  // second largest root belief (key), for the MAP certificate

  // the loads of slice r + 1 are issued before slice r is processed (its
  // stores could alias them as far as the compiler knows)
  float m[KC], u = 0.0f;
  auto load = [&](int r, float (&mm)[KC], float &uu) {
    const int e = r * HW + pc, em = r * HPm + pcm;
#pragma unroll
    for (int k = 0; k < KC; ++k) mm[k] = k < K ? cptr(b, J.msg[k])[em] : 0.0f;
    uu = un[e];
  };
  if (r0 < r1) load(r0, m, u);
  for (int r = r0; r < r1; ++r) {
    float mn[KC], un_next;
    load(r + 1 < r1 ? r + 1 : r, mn, un_next);
    const int e = r * HW + pix;
    const float uu = masked(J.mask, r, x, W) ? kLogZero : u;
    // root belief: messages in joint order (:637), then the unary (:652-654)
    float bel = 0.0f;
#pragma unroll
    for (int k = 0; k < KC; ++k)
      if (k < K) bel = bel + m[k];
    if (J.add_unary) bel = bel + uu;
    if (ok) {
      marg[e] = bel;
      const unsigned long long ak = amax_key(bel, (unsigned)e);
      const unsigned kv = (unsigned)(ak >> 32), kb = (unsigned)(amax >> 32);
      second = kv > kb ? kb : max(second, kv);
      amax = ak > amax ? ak : amax;
    }
    // log_from_root of child i: the other messages in order (:641-649), then
    // the root unary (:169)
#pragma unroll
    for (int i = 0; i < KC; ++i) {
      if (i < K) {
        float fr = 0.0f;
#pragma unroll
        for (int k = 0; k < KC; ++k)
          if (k < K && k != i) fr = fr + m[k];
        fr = fr + uu;
        if (ok) {
          mptr(b, J.fr[i])[e] = fr;
          kmax[i] = max(kmax[i], f2key(fr));
        }
      }
    }
    if (posts) bels[r * (64 * kRootTiles) + tile * 64 + lane] = LSE64 ? bel : expf(bel);
#pragma unroll
    for (int k = 0; k < KC; ++k) m[k] = mn[k];
    u = un_next;
  }

  // the keys, as block_raise does it, the children's by as many lanes at once
  unsigned *rk = reinterpret_cast<unsigned *>(red + kRootWaves * kRootTiles);  // [waves][KC]
  KeyPart part;
  if (b.top2_keys) part.second = wave_second((unsigned)(amax >> 32), second);
  part.amax = wave_max_u64(amax);
#pragma unroll
  for (int k = 0; k < KC; ++k) {
    if (k < K) {
      const unsigned v = wave_max_u32(kmax[k]);
      if (lane == 0) rk[wv * KC + k] = v;
    }
  }
  block_raise(red, part, nullptr, map_key(b, J.map_slot), top2_key(b, J.map_slot));
  if (wv == 1 && lane < K) {
    unsigned v = 0u;
    for (int w = 0; w < kRootWaves * kRootTiles; ++w) v = max(v, rk[w * KC + lane]);
    if (v) atomicMax(max_key(b, J.fr_key[lane]), v);
  }

  // root posterior over the valid rotations in ascending order (:713-726)
  if (!posts || wave != 0 || !ok) return;
  float out;
  if (LSE64) {
    double sum = 0.0;  // of exp(belief - mref)
    float mref = -INFINITY;  // the largest belief so far
    for (int r = 0; r < R; ++r) {
      if (!((J.valid_rot >> r) & 1ull)) continue;
      const float bel = bels[r * (64 * kRootTiles) + tile * 64 + lane];
      if (bel > mref) {
        sum *= (double)__builtin_amdgcn_exp2f((mref - bel) * kLog2eF);
        mref = bel;
      }
      sum += (double)__builtin_amdgcn_exp2f((bel - mref) * kLog2eF);
    }
    out = sum > 0.0 ? log0((float)sum) + mref : kLogZero;
  } else {
    float sum = 0.0f;
    for (int r = 0; r < R; ++r)
      if ((J.valid_rot >> r) & 1ull) sum += bels[r * (64 * kRootTiles) + tile * 64 + lane];
    out = log0(sum);
  }
  mptr(b, J.root_post)[pix] = out;
}

// one instantiation per child count, chosen on the host: the variant for a
// small tree then holds only its own K message registers (40 VGPRs for K = 5,
// 8 waves per SIMD), not those of the widest tree
template <int KC, bool LSE64>
__global__ __launch_bounds__(64 * kRootWaves * kRootTiles) void k_root(Bases b, const RootJob *__restrict__ jobs, int R) {
  // [R][64 kRootTiles] beliefs (FP32 sum: their exponentials), then the waves' keys
  extern __shared__ float4 lds4[];
  unsigned bx, by;
  xcd_block(bx, by);
  const RootJob &J = jobs[by];
  if (skip_inst(b, J.inst)) return;
  const int pix0 = (int)bx * 64 * kRootTiles;
  if (pix0 >= J.H * J.W) return;
  uint4 *red = reinterpret_cast<uint4 *>(lds4 + 16 * kRootTiles * R);
  root_pixels<KC, LSE64>(b, J, R, pix0, red, reinterpret_cast<float *>(lds4));
}

// ------------------------------------------------------------ k_map_decode

__global__ void k_map_decode(Bases b, const MapJob *__restrict__ jobs, int n, ps_map *out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const MapJob J = jobs[i];
  if (skip_inst(b, J.inst)) return;
  const unsigned long long k = *map_key(b, J.slot);
  ps_map m;
  if (k == 0ull) {
    m.rotidx = -1;
    m.y = -1;
    m.x = -1;
    m.score = -INFINITY;
  } else {
    const unsigned idx = 0xffffffffu - (unsigned)(k & 0xffffffffull);
    const unsigned hw = (unsigned)J.H * (unsigned)J.W;
    m.rotidx = (int)(idx / hw);
    const unsigned rem = idx - (unsigned)m.rotidx * hw;
    m.y = (int)(rem / (unsigned)J.W);
    m.x = (int)(rem - (unsigned)m.y * (unsigned)J.W);
    m.score = key2f((unsigned)(k >> 32));
  }
  out[J.out] = m;
}

// ------------------------------------------------------------- k_certify
// MAP certificate of one (instance, scale, part): with every log-marginal
// value off by at most eps, the computed argmax is the exact one whenever
// the computed best beats the second best by more than tau = 2 eps.  An
// instance with any slot at or below tau is flagged for re-evaluation.

__global__ void k_certify(const unsigned long long *__restrict__ top2, int n_map, int map_per_inst, float tau,
                          unsigned *flags) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_map) return;
  const unsigned long long t = top2[(size_t)i * kMapKeyStride];
  const unsigned k1 = (unsigned)(t >> 32), k2 = (unsigned)t;
  const float v1 = k1 ? key2f(k1) : -INFINITY;
  const float v2 = k2 ? key2f(k2) : -INFINITY;
  if (!(v1 - v2 > tau)) flags[i / map_per_inst] = 1u;
}

__global__ void k_invert_flags(const unsigned *__restrict__ in, unsigned *__restrict__ out, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = in[i] ? 0u : 1u;
}

// ------------------------------------------------------------ host launchers

hipError_t launch_invert_flags(const unsigned *in, unsigned *out, int n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_invert_flags, dim3((n + 255) / 256), dim3(256), 0, s, in, out, n);
  return hipGetLastError();
}

hipError_t launch_certify(const unsigned long long *top2, int n_map, int n_inst, float tau, unsigned *flags,
                          hipStream_t s) {
  if (n_map <= 0) return hipSuccess;
  const int mpi = std::max(1, n_map / std::max(1, n_inst));
  hipLaunchKernelGGL(k_certify, dim3((n_map + 255) / 256), dim3(256), 0, s, top2, n_map, mpi, tau, flags);
  return hipGetLastError();
}

hipError_t launch_reset(const Bases &b, int n_keys, int n_map, int n_inst, unsigned *flags, int n_flags,
                        hipStream_t s) {
  int n = std::max(std::max(n_keys, n_map), flags ? n_flags : 0);
  if (n <= 0) return hipSuccess;
  const int kpi = std::max(1, n_keys / std::max(1, n_inst)), mpi = std::max(1, n_map / std::max(1, n_inst));
  hipLaunchKernelGGL(k_reset, dim3((n + 255) / 256), dim3(256), 0, s, b, n_keys, n_map, kpi, mpi, flags, n_flags);
  return hipGetLastError();
}

hipError_t launch_max(const Bases &b, const MaxJob *jobs, int n_jobs, int R, int max_hw, hipStream_t s) {
  if (n_jobs <= 0) return hipSuccess;
  const int chunk = 16384;  // elements per block, a multiple of 4
  const long long n = (long long)R * max_hw;
  dim3 grid((unsigned)((n + chunk - 1) / chunk), n_jobs);
  hipLaunchKernelGGL(k_max, grid, dim3(256), 0, s, b, jobs, R, chunk);
  return hipGetLastError();
}

static bool rowpass_fixed(int R) { return R == 24 || R == 48; }

size_t rowpass_lds_bytes(int R, int W, int kx) {
  RowGeom g = row_geom(W, kx);
  // the fixed-R kernels stage one slice group at a time; the generic one all
  // slices and its E buffer
  size_t p = rowpass_fixed(R) ? (size_t)(R / row_groups(R)) * g.Pw : (size_t)R * g.Pw + (size_t)R * ((W + 3) & ~3);
  return sizeof(float) * p;
}
// with the x filter on the matrix cores; 0 where there is no such kernel
size_t rowpass4_lds_bytes(int R, int W, int kx) {
  return rowpass_fixed(R) ? row4_lds_bytes(row4_slices(R), W, kx) : 0;
}

// The dynamic-LDS attribute of a kernel is one process-wide value per device
// and function, while plans with different needs coexist: it is only ever
// raised (to the largest size asked for so far), under a lock, so a later
// plan never lowers what an earlier plan's launches rely on.
hipError_t raise_lds_limit(const void *f, size_t bytes) {
  if (bytes <= 64 * 1024) return hipSuccess;
  static std::mutex mu;
  static std::map<std::pair<int, const void *>, size_t> high;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lock(mu);
  size_t &h = high[std::make_pair(dev, f)];
  if (bytes <= h) return hipSuccess;
  e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (e == hipSuccess) h = bytes;
  return e;
}

template <int KIND>
static hipError_t rowpass_kind_set_lds_limit(size_t bytes) {
  hipError_t e = raise_lds_limit(reinterpret_cast<const void *>(&k_rowpass_r<24, false, KIND>), bytes);
  if (e == hipSuccess) e = raise_lds_limit(reinterpret_cast<const void *>(&k_rowpass_r<48, false, KIND>), bytes);
  if (e == hipSuccess) e = raise_lds_limit(reinterpret_cast<const void *>(&k_rowpass_r<24, true, KIND>), bytes);
  if (e == hipSuccess) e = raise_lds_limit(reinterpret_cast<const void *>(&k_rowpass_r<48, true, KIND>), bytes);
  return e;
}

// bytes, bytes4: the vector and the MFMA row pass's largest LDS
hipError_t rowpass_set_lds_limit(size_t bytes, size_t bytes4) {
  hipError_t e = rowpass_kind_set_lds_limit<kRowVector>(bytes);
  if (e == hipSuccess) e = rowpass_kind_set_lds_limit<kRowMfma>(bytes4);
  if (e == hipSuccess) e = rowpass_kind_set_lds_limit<kRowMfmaWide>(bytes4);
  if (e != hipSuccess) return e;
  return raise_lds_limit(reinterpret_cast<const void *>(&k_rowpass_any), bytes);
}

template <int ROWS, bool SPLIT, bool MFMA>
static hipError_t colpass_rows_set_lds_limit(size_t bytes) {
  hipError_t e = raise_lds_limit(reinterpret_cast<const void *>(&k_colpass<kEpiUpRoot, ROWS, SPLIT, MFMA>), bytes);
  if (e == hipSuccess) e = raise_lds_limit(reinterpret_cast<const void *>(&k_colpass<kEpiUpNode, ROWS, SPLIT, MFMA>), bytes);
  if (e == hipSuccess) e = raise_lds_limit(reinterpret_cast<const void *>(&k_colpass<kEpiUpNodeU, ROWS, SPLIT, MFMA>), bytes);
  if (e == hipSuccess) e = raise_lds_limit(reinterpret_cast<const void *>(&k_colpass<kEpiDownLeaf, ROWS, SPLIT, MFMA>), bytes);
  if (e == hipSuccess) e = raise_lds_limit(reinterpret_cast<const void *>(&k_colpass<kEpiDownMid, ROWS, SPLIT, MFMA>), bytes);
  return e;
}

// bytes: the LDS of the vector column pass; bytes4: of the MFMA one's 16-row
// tile (the larger one)
hipError_t colpass_set_lds_limit(size_t bytes, size_t bytes4) {
  hipError_t e = colpass_rows_set_lds_limit<8, false, false>(bytes);
  if (e == hipSuccess) e = colpass_rows_set_lds_limit<8, true, false>(bytes);
  if (e == hipSuccess) e = colpass_rows_set_lds_limit<8, false, true>(bytes4);
  if (e == hipSuccess) e = colpass_rows_set_lds_limit<16, false, true>(bytes4);
  if (e == hipSuccess) e = colpass_rows_set_lds_limit<8, true, true>(bytes4);
  return e;
}

template <int KIND>
static void launch_rowpass_r(int R, bool split, dim3 grid, dim3 blk, size_t lds_bytes, hipStream_t s, const Bases &b,
                             const MsgJob *jobs, const float *taps, const int *shifts) {
  if (R == 24 && !split)
    hipLaunchKernelGGL((k_rowpass_r<24, false, KIND>), grid, blk, lds_bytes, s, b, jobs, taps, shifts);
  else if (R == 24)
    hipLaunchKernelGGL((k_rowpass_r<24, true, KIND>), grid, blk, lds_bytes, s, b, jobs, taps, shifts);
  else if (!split)  // 48: the reference's default grid
    hipLaunchKernelGGL((k_rowpass_r<48, false, KIND>), grid, blk, lds_bytes, s, b, jobs, taps, shifts);
  else
    hipLaunchKernelGGL((k_rowpass_r<48, true, KIND>), grid, blk, lds_bytes, s, b, jobs, taps, shifts);
}

// Whether a launch of `blocks` rows of up to W columns takes its x filter to the
// matrix cores.  It does where the rows fit, but where that costs blocks per CU
// (its layout takes 26 floats a column of 24 slices, 24 on the vector unit) or,
// with more columns than threads, work: 48 slices go through in four groups
// rather than two, and a column's values are then gathered and exponentiated
// again for each.  us of all row passes of a sweep of 200-row images (half width
// 36), vector unit / matrix cores:
//   24 slices, 8 images: 877 / 757 (W 460, 3 / 2 blocks per CU), 1325 / 1593
//     (W 760, 2 / 1), 2103 / 1812 (W 800, 1 / 1)
//   48 slices, 4 images: 1343 / 838 (W 500, a column a thread), 1502 / 1821
//     (W 600, 2 / 3 blocks per CU), 2873 / 2197 (W 800, 1 / 2), 4268 / 5302
//     (W 1480, 1 / 1); three columns a thread 4049 / 4154 (W 1400, 1 / 2)
// Of rows of up to 16 columns a wave's tile of 64 is mostly empty (24 slices, 16
// images 300 rows high: 291 / 321 us at W 16, 293 / 285 at W 20).
static bool row_on_mfma(int R, int W, size_t lds, size_t lds4, long long blocks) {
  if (lds4 == 0 || (R == 24 && W <= 16)) return false;
  const int waves = std::min(512, (W + 63) / 64 * 64) / 64;
  // blocks per CU by LDS and by registers (waves of the kernel per CU), and no
  // more than there are
  auto per_cu = [&](size_t bytes, int max_waves) {
    return std::min({(long long)(160 * 1024 / bytes), (long long)(max_waves / waves), (blocks + 255) / 256});
  };
  const long long v = per_cu(lds, R == 24 ? 32 : 16), m = per_cu(lds4, R == 24 ? 32 : 24);
  return R == 24 || W <= 512 ? 2 * m > v : W <= 1024 && m >= 2 * v;
}

// threads: block size (a multiple of 64; 0 = one thread per column, at most
// 512); every loop of the row pass strides by the block size
// split: some job's warp changes its offset along an axis (MsgJob::split)
// lds4_bytes: LDS of the row pass with its x filter on the matrix cores, or 0
// where the rows do not fit it
hipError_t launch_rowpass(const Bases &b, const MsgJob *jobs, int n_jobs, const float *taps, const int *shifts,
                          int R, int max_h, int max_w, size_t lds_bytes, size_t lds4_bytes, hipStream_t s, int threads,
                          bool split) {
  if (n_jobs <= 0) return hipSuccess;
  dim3 grid(max_h, n_jobs);
  const int nt = threads > 0 ? std::min(threads, std::max(64, (max_w + 63) / 64 * 64))
                             : std::min(512, (max_w + 63) / 64 * 64);
  if (!rowpass_fixed(R))
    hipLaunchKernelGGL(k_rowpass_any, grid, dim3(nt), lds_bytes, s, b, jobs, taps, shifts, R);
  else if (!row_on_mfma(R, max_w, lds_bytes, lds4_bytes, (long long)max_h * n_jobs))
    launch_rowpass_r<kRowVector>(R, split, grid, dim3(nt), lds_bytes, s, b, jobs, taps, shifts);
  else if (max_w > 512)
    launch_rowpass_r<kRowMfmaWide>(R, split, grid, dim3(nt), lds4_bytes, s, b, jobs, taps, shifts);
  else
    launch_rowpass_r<kRowMfma>(R, split, grid, dim3(nt), lds4_bytes, s, b, jobs, taps, shifts);
  return hipGetLastError();
}

// LDS of the vector column pass's 16-row tile (the bound a filter is accepted
// by; its 8-row tile, the one that runs, takes 32 rows of 256 bytes less)
size_t colpass_lds_bytes(int ky, int rows) {
  return sizeof(float) * (size_t)col_tile_rows(ky, rows > 0 ? rows : 16) * kColTileX;
}
// LDS of the MFMA column pass's 16-row tile
size_t colpass4_lds_bytes(int ky) {
  return sizeof(float) * ((size_t)col_tile_rows(ky, 16) * kColTileX + 4 * tap4_pitch(ky) + 4);
}

template <int ROWS, bool SPLIT, bool MFMA>
static void launch_colpass_rows(int epi_hi, dim3 grid, size_t lds_bytes, hipStream_t s, const Bases &b,
                                const MsgJob *jobs, const float *taps, const int *shifts, int R, int xtiles) {
  const dim3 blk(kColWaves * 64);
  switch (epi_hi) {
    case kEpiUpRoot: hipLaunchKernelGGL((k_colpass<kEpiUpRoot, ROWS, SPLIT, MFMA>), grid, blk, lds_bytes, s, b, jobs, taps, shifts, R, xtiles); break;
    case kEpiUpNode: hipLaunchKernelGGL((k_colpass<kEpiUpNode, ROWS, SPLIT, MFMA>), grid, blk, lds_bytes, s, b, jobs, taps, shifts, R, xtiles); break;
    case kEpiUpNodeU: hipLaunchKernelGGL((k_colpass<kEpiUpNodeU, ROWS, SPLIT, MFMA>), grid, blk, lds_bytes, s, b, jobs, taps, shifts, R, xtiles); break;
    case kEpiDownLeaf: hipLaunchKernelGGL((k_colpass<kEpiDownLeaf, ROWS, SPLIT, MFMA>), grid, blk, lds_bytes, s, b, jobs, taps, shifts, R, xtiles); break;
    default: hipLaunchKernelGGL((k_colpass<kEpiDownMid, ROWS, SPLIT, MFMA>), grid, blk, lds_bytes, s, b, jobs, taps, shifts, R, xtiles); break;
  }
}

// A strip walks its tiles one after another, a few us each, most of it waiting.
// A launch of few strips cuts them into parts, each its own block, as long as
// all blocks fit the chip at once, 4 per CU; a part fills its own ring, whose
// extra rows cost more than the waits once the chip is full (300x300x48, 960
// strips: 94 instead of 86 us in two parts).  us per launch, one part / by this
// rule: 22.0 / 17.3, 21.4 / 17.8, 19.7 / 16.0 and 18.1 / 14.9 (FP32, 112x128x24,
// 192 or 240 strips), 21.1 / 17.4, 19.5 / 16.2, 18.2 / 16.0 and 15.7 / 13.1
// (fp16, 160x160x24, 288 or 360 strips), 10.8 / 8.6 (one message of 41x57x24).
int col_parts(int blocks, int tiles) { return std::max(1, std::min(tiles, 1024 / blocks)); }

// epi_hi: the highest destination kind (EpiKind) among the jobs; rows:
// output rows per lane (8 or 16; 0 = the default); lds_bytes_16, lds4_bytes_16:
// the LDS of the 16-row tile for the jobs' widest y filter, without and with
// the MFMA's tap operand (0: it does not fit, the filter runs on the vector
// unit, 8 rows per lane); an 8-row tile takes 32 rows of 256 bytes less
// (split: some job's warp changes its offset along an axis; those launches
// take 8 rows per lane)
hipError_t launch_colpass(const Bases &b, const MsgJob *jobs, int n_jobs, const float *taps, const int *shifts,
                          int R, int epi_hi, int max_h, int max_w, size_t lds_bytes_16, size_t lds4_bytes_16,
                          hipStream_t s, int rows, bool split) {
  if (n_jobs <= 0) return hipSuccess;
  if (rows == 0 || split) rows = kColRowsDefault;
  if (epi_hi < kEpiUpRoot || epi_hi > kEpiDownMid || (rows != 8 && rows != 16)) return hipErrorInvalidValue;
  const int xtiles = (max_w + kColTileX - 1) / kColTileX;
  // few rows of a tile to filter do not pay for the tap operand (us of all column
  // passes of 16 images of 300 columns x 24, half width 9, vector unit / matrix
  // cores: 107 / 115 at 4 rows, 121 / 122 at 12)
  if (max_h <= 12) lds4_bytes_16 = 0;
  const int tile_y = kColWaves * (lds4_bytes_16 == 0 ? kColRowsDefault : rows);
  dim3 grid(R * xtiles, n_jobs, col_parts(R * xtiles * n_jobs, (max_h + tile_y - 1) / tile_y));
  const size_t less = sizeof(float) * kColWaves * 8 * kColTileX;
  if (lds4_bytes_16 == 0 && split)
    launch_colpass_rows<8, true, false>(epi_hi, grid, lds_bytes_16 - less, s, b, jobs, taps, shifts, R, xtiles);
  else if (lds4_bytes_16 == 0)
    launch_colpass_rows<8, false, false>(epi_hi, grid, lds_bytes_16 - less, s, b, jobs, taps, shifts, R, xtiles);
  else if (split)
    launch_colpass_rows<8, true, true>(epi_hi, grid, lds4_bytes_16 - less, s, b, jobs, taps, shifts, R, xtiles);
  else if (rows == 16)
    launch_colpass_rows<16, false, true>(epi_hi, grid, lds4_bytes_16, s, b, jobs, taps, shifts, R, xtiles);
  else
    launch_colpass_rows<8, false, true>(epi_hi, grid, lds4_bytes_16 - less, s, b, jobs, taps, shifts, R, xtiles);
  return hipGetLastError();
}

// k: the root's child count, the same for every job (one tree per plan); a
// root without children and counts above 8 take the variant that reads J.K
template <bool LSE64>
static void launch_root_k(const Bases &b, const RootJob *jobs, int k, int R, dim3 grid, dim3 blk, hipStream_t s) {
  const int waves = kRootWaves * kRootTiles;
  const size_t lds = sizeof(float) * 64 * kRootTiles * R + waves * (sizeof(uint4) + sizeof(unsigned) * kMaxRootChildren);
  switch (k) {
    case 1: hipLaunchKernelGGL((k_root<1, LSE64>), grid, blk, lds, s, b, jobs, R); break;
    case 2: hipLaunchKernelGGL((k_root<2, LSE64>), grid, blk, lds, s, b, jobs, R); break;
    case 3: hipLaunchKernelGGL((k_root<3, LSE64>), grid, blk, lds, s, b, jobs, R); break;
    case 4: hipLaunchKernelGGL((k_root<4, LSE64>), grid, blk, lds, s, b, jobs, R); break;
    case 5: hipLaunchKernelGGL((k_root<5, LSE64>), grid, blk, lds, s, b, jobs, R); break;
    case 6: hipLaunchKernelGGL((k_root<6, LSE64>), grid, blk, lds, s, b, jobs, R); break;
    case 7: hipLaunchKernelGGL((k_root<7, LSE64>), grid, blk, lds, s, b, jobs, R); break;
    case 8: hipLaunchKernelGGL((k_root<8, LSE64>), grid, blk, lds, s, b, jobs, R); break;
    default: hipLaunchKernelGGL((k_root<kMaxRootChildren, LSE64>), grid, blk, lds, s, b, jobs, R); break;
  }
}

hipError_t launch_root(const Bases &b, const RootJob *jobs, int n_jobs, int k, int R, int max_hw, bool lse64,
                       hipStream_t s) {
  if (n_jobs <= 0) return hipSuccess;
  if (k < 0 || k > kMaxRootChildren) return hipErrorInvalidValue;
  dim3 grid((max_hw + 64 * kRootTiles - 1) / (64 * kRootTiles), n_jobs);
  const dim3 blk(64 * kRootWaves * kRootTiles);
  if (lse64)
    launch_root_k<true>(b, jobs, k, R, grid, blk, s);
  else
    launch_root_k<false>(b, jobs, k, R, grid, blk, s);
  return hipGetLastError();
}

hipError_t launch_map_decode(const Bases &b, const MapJob *jobs, int n, ps_map *out, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_map_decode, dim3((n + 255) / 256), dim3(256), 0, s, b, jobs, n, out);
  return hipGetLastError();
}

}  // namespace ps
