// Eigenbasis path of a message whose covariance has off-diagonal terms
// (gaussFilter2dOffset with offset 0, multi_array_filter.hpp:334-369, called
// per rotation slice by computeRotJointMarginal, objectdetect_findrot.cpp:
// 422-429).  The row pass has already written the rotation-filtered grid
// T[R][H][W] (exp(b - M) after the forward shift and the circular filter).
// Per slice:
//   k_od_x     the eigenbasis grid's cells, taken from T where they are
//       needed, and the x filter (multi_array_filter.hpp:211-321) with the
//       eigenvalue's taps.  A cell is the last source cell of the x-outer,
//       y-inner scan that the reference's nearest scatter (TM_DIRECT, sparse
//       models) leaves on it, zero cells not being written, or a bilinear
//       sample (TM_BILINEAR) (multi_array_transform.hpp:122-239)
//   k_od_y     the y filter
//   k_od_back  bilinear sample back to H x W, log, +M, the inverse shift and
//       the caller's accumulation (the column pass's epilogue)
// Coordinates are mapped in double with the reference's operation order; the
// bilinear weights are float; the filters add their taps in ascending order.
// Every launch covers the off-diagonal messages of one level.
//
// Of the six kernels that this was (keys cleared, scattered, or gathered, a
// tap at a time from global memory in both filters, one atomic per wave of 64
// pixels onto a part's argmax key), a sweep of 4 images of 200 x 200 x 24
// took 12.7 ms: back 5.4 (the atomics), y filter 4.0, x filter 2.0, scatter
// 0.95, gather 0.27, clear 0.12.  Now 1.9 ms: back 0.68, y 0.54, x 0.51.  The
// filters' multiply-adds alone take some 0.35 ms (100 taps on 1.9 times the
// states, 39 T a second), the grids' bytes 0.6 ms at a large copy's rate.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>

#include "ps_device.hpp"
#include "ps_internal.hpp"

namespace ps {

hipError_t raise_lds_limit(const void *f, size_t bytes);

namespace {

constexpr int kOdThreads = 256;

__device__ __forceinline__ float *od_a(const Bases &b, const MsgJob &J) { return mptr(b, J.od_buf); }
__device__ __forceinline__ float *od_x(const Bases &b, const MsgJob &J, int R) {
  return mptr(b, J.od_buf) + (long long)R * J.th * od_pitch(J.tw);
}

// The x filter's tile: kOdRows rows of at most kOdWide outputs, the row's
// tiles of equal width.
constexpr int kOdRows = 16, kOdWide = 384;
__host__ __device__ __forceinline__ int od_xtiles(int tw) { return (tw + kOdWide - 1) / kOdWide; }
__host__ __device__ __forceinline__ int od_xwidth(int tw) {
  const int n = od_xtiles(tw);
  return ((tw + n - 1) / n + 7) & ~7;
}
// LDS row of that tile: the outputs, the filter's reach and what the last
// output's 16-byte window reads beyond
__host__ __device__ __forceinline__ int od_xpitch(int tw, int k) { return (od_xwidth(tw) + 2 * k + 1 + 31) & ~7; }

// The y filter's tile: 64 columns x 64 rows, 16 rows per lane, the source rows
// staged for up to kOdTaps taps at a time (40 KB of LDS).
constexpr int kOdTaps = 96, kOdLane = 16, kOdTileY = 4 * kOdLane;

// TM_BILINEAR sample of a [h][w] grid (row pitch `pitch`) at (x1, y1)
// (multi_array_transform.hpp:218-236): within 10 float epsilons of a grid
// point the point itself, the last row and column (no right / lower
// neighbour) and outside: 0
__device__ __forceinline__ float bilinear_at(const float *g, int h, int w, int pitch, double x1, double y1) {
  const int ix = (int)floor(x1);
  const int iy = (int)floor(y1);
  float r = 0.0f;
  if (ix >= 0 && ix < w && iy >= 0 && iy < h) {
    const float eps10 = 10.0f * FLT_EPSILON;
    const float a = (float)(x1 - (double)ix);
    const float bb = (float)(y1 - (double)iy);
    const float *p = g + (long long)iy * pitch + ix;
    if (a < eps10 && bb < eps10) {
      r = p[0];
    } else if (ix < w - 1 && iy < h - 1) {
      const float t0 = (1.0f - bb) * (1.0f - a) * p[0];
      const float t1 = (1.0f - bb) * a * p[1];
      const float t2 = bb * (1.0f - a) * p[pitch];
      const float t3 = bb * a * p[pitch + 1];
      r = t0 + t1 + t2 + t3;
    }
  }
  return r;
}

}  // namespace

// N taps of a filter whose window of 16 values is lo, hi; N at most 8.  Only
// the filter's own taps are multiplied (a zero tap would spread a NaN).
template <int N>
__device__ __forceinline__ void od_taps(float (&acc)[8], const float (&lo)[8], const float (&hi)[8], const float *f,
                                        int n) {
#pragma unroll
  for (int u = 0; u < N; ++u) {
    if (N < 8 && u >= n) break;
    const float t = f[u];
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = fmaf(i + u < 8 ? lo[(i + u) & 7] : hi[(i + u) & 7], t, acc[i]);
  }
}
__device__ __forceinline__ void od_load8(float (&v)[8], const float *p) {
  const float4 a = *reinterpret_cast<const float4 *>(p), b = *reinterpret_cast<const float4 *>(p + 4);
  v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
}

// One block per (message, slice, 16 rows x up to 384 columns of the
// eigenbasis grid): its cells and the filter's reach beside them go to LDS,
// each found or sampled once, then eight outputs per lane from a sliding
// register window.  Direct: the grid is T turned and shifted, so at most 2 x 2
// source cells can land on a cell (CellWarp).
__global__ __launch_bounds__(kOdThreads) void k_od_x(Bases b, const MsgJob *__restrict__ jobs,
                                                     const float *__restrict__ taps, int R) {
  extern __shared__ float4 lds4[];
  float *P = reinterpret_cast<float *>(lds4);
  unsigned bx, by;
  xcd_block(bx, by);
  const MsgJob &J = jobs[by];
  if (skip_inst(b, J.inst)) return;
  const int th = J.th, tw = J.tw, H = J.H, W = J.W, tp = J.tpitch;
  const int nx = od_xtiles(tw), ny = (th + kOdRows - 1) / kOdRows;
  const int r = (int)bx / (nx * ny);
  if (r >= R) return;
  const int rem = (int)bx - r * (nx * ny);
  const int yt = rem / nx;
  const int xw = od_xwidth(tw), x0 = (rem - yt * nx) * xw, y0 = yt * kOdRows;
  const int k = J.kxe, L = 2 * k + 1;
  const int Pw = od_xpitch(tw, k), cw = xw + 2 * k;
  const float *T = cptr(b, J.tmp) + (long long)r * H * tp;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (J.od_direct) {
    const CellWarp cell(J.t_fwd);
    for (int row = wave; row < kOdRows; row += 4) {
      const int y3 = y0 + row;
      for (int c = lane; c < cw; c += 64) {
        const int x3 = x0 - k + c;
        float v = 0.0f;
        if (x3 >= 0 && x3 < tw && y3 < th) {
          float w[4];
          cell.load4(x3, y3, W, H, T, tp, w);
          v = last_cell(w);
        }
        P[row * Pw + c] = v;
      }
    }
  } else {
    const double m00 = J.t_fwd[0], m01 = J.t_fwd[1], m02 = J.t_fwd[2];
    const double m10 = J.t_fwd[3], m11 = J.t_fwd[4], m12 = J.t_fwd[5];
    for (int row = wave; row < kOdRows; row += 4) {
      const int y3 = y0 + row;
      for (int c = lane; c < cw; c += 64) {
        const int x3 = x0 - k + c;
        float v = 0.0f;
        if (x3 >= 0 && x3 < tw && y3 < th) {
          const double x1 = m00 * (double)x3 + m01 * (double)y3 + m02;
          const double y1 = m10 * (double)x3 + m11 * (double)y3 + m12;
          v = bilinear_at(T, H, W, tp, x1, y1);
        }
        P[row * Pw + c] = v;
      }
    }
  }
  __syncthreads();
  const float *fx = taps + J.taps_xe;
  const int pitch = od_pitch(tw), nq = xw >> 3;
  float *X = od_x(b, J, R) + ((long long)r * th + y0) * pitch;
  for (int item = threadIdx.x; item < kOdRows * nq; item += kOdThreads) {
    const int row = item / nq, q = item - row * nq;
    const int xo = x0 + 8 * q;
    if (y0 + row >= th || xo >= tw) continue;
    const float *p = P + row * Pw + 8 * q;
    float a[8], w0[8], w1[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) a[i] = 0.0f;
    od_load8(w0, p);
    od_load8(w1, p + 8);
    int t = 0;
    for (; t + 16 <= L; t += 16) {
      od_taps<8>(a, w0, w1, fx + t, 8);
      od_load8(w0, p + t + 16);
      od_taps<8>(a, w1, w0, fx + t + 8, 8);
      od_load8(w1, p + t + 24);
    }
    if (t + 8 <= L) {
      od_taps<8>(a, w0, w1, fx + t, 8);
      od_load8(w0, p + t + 16);
      od_taps<7>(a, w1, w0, fx + t + 8, L - t - 8);
    } else {
      od_taps<7>(a, w0, w1, fx + t, L - t);
    }
    float *o = X + (long long)row * pitch + xo;
    if ((pitch & 3) == 0) {
      *reinterpret_cast<float4 *>(o) = make_float4(a[0], a[1], a[2], a[3]);
      if (xo + 4 < pitch) *reinterpret_cast<float4 *>(o + 4) = make_float4(a[4], a[5], a[6], a[7]);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (xo + i < tw) o[i] = a[i];
    }
  }
}

// N taps (at most 8) of the y filter from tap t of the staged rows on; PH is
// the ring phase of the 16-row register window
template <int PH, int N>
__device__ __forceinline__ void od_ytaps(float (&acc)[kOdLane], float (&buf)[kOdLane], const float *f,
                                         const float *rows, int n) {
#pragma unroll
  for (int u = 0; u < N; ++u) {
    if (N < 8 && u >= n) break;
    const float t = f[u];
#pragma unroll
    for (int i = 0; i < kOdLane; ++i) acc[i] = fmaf(buf[(i + u + PH) & (kOdLane - 1)], t, acc[i]);
    buf[(u + PH) & (kOdLane - 1)] = rows[(u + kOdLane) * 64];
  }
}

// y filter of the eigenbasis grid, A = X * fy: one block per (message, slice,
// 64 columns x 64 rows), a column and 16 rows per lane from a register ring
// fed by LDS.  A filter of up to 96 taps (sigma up to 15.8 px) is staged at
// once, a longer one in turns.
__global__ __launch_bounds__(kOdThreads) void k_od_y(Bases b, const MsgJob *__restrict__ jobs,
                                                     const float *__restrict__ taps, int R) {
  __shared__ float tile[(kOdTileY + kOdTaps) * 64];
  unsigned bx, by;
  xcd_block(bx, by);
  const MsgJob &J = jobs[by];
  if (skip_inst(b, J.inst)) return;
  const int th = J.th, tw = J.tw;
  const int nx = (tw + 63) / 64, ny = (th + kOdTileY - 1) / kOdTileY;
  const int r = (int)bx / (nx * ny);
  if (r >= R) return;
  const int rem = (int)bx - r * (nx * ny);
  const int xt = rem / ny, y0 = (rem - xt * ny) * kOdTileY;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int x = xt * 64 + lane;
  const int pitch = od_pitch(tw);
  const float *col = od_x(b, J, R) + (long long)r * th * pitch + min(x, tw - 1);
  const int k = J.kye, L = 2 * k + 1;
  const float *fy = taps + J.taps_ye;
  float a[kOdLane];
#pragma unroll
  for (int i = 0; i < kOdLane; ++i) a[i] = 0.0f;
  for (int c = 0; c < L; c += kOdTaps) {
    const int n = min(L - c, kOdTaps);
    if (c) __syncthreads();  // every wave is done with the rows before
    const int s0 = y0 - k + c, rows = kOdTileY + n;
    for (int i0 = wave; i0 < rows; i0 += 32) {
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = col[(long long)min(max(s0 + i0 + 4 * j, 0), th - 1) * pitch];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int y = s0 + i0 + 4 * j;
        if (i0 + 4 * j < rows) tile[(i0 + 4 * j) * 64 + lane] = y >= 0 && y < th ? v[j] : 0.0f;
      }
    }
    __syncthreads();
    const float *p = tile + wave * kOdLane * 64 + lane;
    const float *f = fy + c;
    float buf[kOdLane];
#pragma unroll
    for (int i = 0; i < kOdLane; ++i) buf[i] = p[i * 64];
    int t = 0;
    for (; t + 16 <= n; t += 16) {
      od_ytaps<0, 8>(a, buf, f + t, p + t * 64, 8);
      od_ytaps<8, 8>(a, buf, f + t + 8, p + (t + 8) * 64, 8);
    }
    if (t + 8 <= n) {
      od_ytaps<0, 8>(a, buf, f + t, p + t * 64, 8);
      od_ytaps<8, 7>(a, buf, f + t + 8, p + (t + 8) * 64, n - t - 8);
    } else {
      od_ytaps<0, 7>(a, buf, f + t, p + t * 64, n - t);
    }
  }
  if (x >= tw) return;
  float *out = od_a(b, J) + (long long)r * th * pitch + x;
#pragma unroll
  for (int i = 0; i < kOdLane; ++i) {
    const int y = y0 + wave * kOdLane + i;
    if (y < th) out[(long long)y * pitch] = a[i];
  }
}

// Back to the grid: pixel (x, y) of slice r reads the smoothed slice at
// (x + inv_ox[r], y + inv_oy[r]) (the inverse nearest warp, LOG_ZERO outside,
// with a split warp's step past its break,
// objectdetect_findrot.cpp:437-448), which is the bilinear sample of the
// eigenbasis grid at T_back of that pixel, log, +M (:432-435); then the
// caller's accumulation.  One block per (message, slice, 64 x 32 pixels),
// eight rows per lane: a rotated block's samples stay in its CU's cache, and a
// wave's reductions cover 512 pixels before they reach the part's keys.
constexpr int kBackRows = 8;

__global__ __launch_bounds__(kOdThreads) void k_od_back(Bases b, const MsgJob *__restrict__ jobs,
                                                        const int *__restrict__ shifts, int R) {
  unsigned bx, by;
  xcd_block(bx, by);
  const MsgJob &J = jobs[by];
  if (skip_inst(b, J.inst)) return;
  const int H = J.H, W = J.W, th = J.th, tw = J.tw;
  const int nx = (W + 63) / 64, ny = (H + 4 * kBackRows - 1) / (4 * kBackRows);
  const int r = (int)bx / (nx * ny);
  if (r >= R) return;
  const int rem = (int)bx - r * (nx * ny);
  const int yt = rem / nx;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int x = (rem - yt * nx) * 64 + lane;
  const int y0 = (yt * 4 + wave) * kBackRows;
  const int *sh = shifts + J.shifts;
  // the inverse offsets, which change once along x / y where the warp is
  // split: breaks and steps from 12 R on
  int ox = sh[2 * R + r];
  const int oy0 = sh[3 * R + r];
  if (J.split && x >= sh[12 * R + r]) ox += sh[13 * R + r];
  const int ybrk = J.split ? sh[14 * R + r] : H, ystep = J.split ? sh[15 * R + r] : 0;
  const int xs = x + ox;
  const float M = key2f(*max_key(b, J.src_key));
  float *dst = mptr(b, J.dst);
  const float *dun = J.dst_unary.buf >= 0 ? cptr(b, J.dst_unary) : nullptr;
  float *dst2 = J.dst2.buf >= 0 ? mptr(b, J.dst2) : nullptr;
  const float *bel = J.dst_bel.buf >= 0 ? cptr(b, J.dst_bel) : nullptr;
  const bool need_u = (J.dst_kind == kDstUpNode && J.dst_add_unary) || J.dst_kind == kDstDown;
  const bool need_b = J.dst_kind == kDstDown && J.dst_base == 0;
  const bool xmask = ((J.dst_mask.rot_bits >> r) & 1ull) || x < J.dst_mask.strip || x >= W - J.dst_mask.strip;
  const double b0 = J.t_back[0], b1 = J.t_back[1], b2 = J.t_back[2];
  const double b3 = J.t_back[3], b4 = J.t_back[4], b5 = J.t_back[5];
  const int pitch = od_pitch(tw);
  const float *A = od_a(b, J) + (long long)r * th * pitch;
  // element (r, y, x) of a grid at its row pitch
  auto at = [&](const GridRef &g, int y) { return ((long long)r * H + y) * g.pitch + x; };
  DstAcc da;
  if (x < W) {
    // every load of the eight pixels before any store
    float v[kBackRows], pu[kBackRows], pb[kBackRows];
#pragma unroll
    for (int i = 0; i < kBackRows; ++i) {
      const int y = min(y0 + i, H - 1);
      const int ys = y + (y >= ybrk ? oy0 + ystep : oy0);
      v[i] = -1.0f;  // outside: LOG_ZERO, without the +M of a zero response
      if (xs >= 0 && xs < W && ys >= 0 && ys < H) {
        const double xe = b0 * (double)xs + b1 * (double)ys + b2;
        const double ye = b3 * (double)xs + b4 * (double)ys + b5;
        v[i] = bilinear_at(A, th, tw, pitch, xe, ye);
      }
      pu[i] = need_u ? dun[at(J.dst_unary, y)] : 0.0f;
      pb[i] = need_b ? bel[at(J.dst_bel, y)] : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < kBackRows; ++i) {
      const int y = y0 + i;
      if (y >= H) break;
      const int ys = y + (y >= ybrk ? oy0 + ystep : oy0);
      const bool in = xs >= 0 && xs < W && ys >= 0 && ys < H;
      const float msg = in ? log0(v[i]) + M : kLogZero;
      dst_store(J, dst, dst2, at(J.dst, y), dst2 ? at(J.dst2, y) : 0, (unsigned)(((long long)r * H + y) * W + x), xmask,
                msg, pu[i], pb[i], da);
    }
  }
  __shared__ uint4 red[4];
  dst_flush(b, J, dst2 != nullptr, da, red);
}

// ------------------------------------------------------------ host launcher

// The largest grids and LDS of the stages over off-diagonal jobs.
void od_extent(OdExtent &e, int R, const MsgJob &j) {
  e.x_blocks = std::max(e.x_blocks, (long long)R * od_xtiles(j.tw) * ((j.th + kOdRows - 1) / kOdRows));
  e.y_blocks = std::max(e.y_blocks, (long long)R * ((j.tw + 63) / 64) * ((j.th + kOdTileY - 1) / kOdTileY));
  e.b_blocks = std::max(e.b_blocks, (long long)R * ((j.W + 63) / 64) * ((j.H + 4 * kBackRows - 1) / (4 * kBackRows)));
  e.x_lds = std::max(e.x_lds, sizeof(float) * kOdRows * (size_t)od_xpitch(j.tw, j.kxe));
}

hipError_t od_set_lds_limit(const OdExtent &ext) {
  return raise_lds_limit(reinterpret_cast<const void *>(&k_od_x), ext.x_lds);
}

// The eigenbasis stages of n_jobs off-diagonal messages.
hipError_t launch_offdiag(const Bases &b, const MsgJob *jobs, int n_jobs, const float *taps, const int *shifts, int R,
                          const OdExtent &ext, hipStream_t s) {
  if (n_jobs <= 0) return hipSuccess;
  const dim3 blk(kOdThreads);
  hipLaunchKernelGGL(k_od_x, dim3((unsigned)ext.x_blocks, n_jobs), blk, ext.x_lds, s, b, jobs, taps, R);
  hipLaunchKernelGGL(k_od_y, dim3((unsigned)ext.y_blocks, n_jobs), blk, 0, s, b, jobs, taps, R);
  hipLaunchKernelGGL(k_od_back, dim3((unsigned)ext.b_blocks, n_jobs), blk, 0, s, b, jobs, shifts, R);
  return hipGetLastError();
}

}  // namespace ps
