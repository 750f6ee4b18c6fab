// Unary ingestion on the device: a part detector's score grids mapped to
// image coordinates, clipped and logged — the step right before the sweep.
//
//   PartApp::loadScoreGrid (partapp.cpp:866-899): each slice (scale,
//   rotation) of the score grid goes through transform_grid_fixed_size with
//   Tig = Ti2 T2g and NO_CLASS_VALUE = 0: a nearest scatter (TM_DIRECT, the
//   last source cell of the x-outer, y-inner scan wins, zero cells are not
//   written) or a bilinear gather (multi_array_transform.hpp:122-239);
//   then clip_scores_fill (objectdetect_aux.hpp:41-59: negative -> 1e-4) and
//   computeLogGrid (multi_array_op.hpp:154-166: 0 -> LOG_ZERO), as
//   findObjectImageRotJoints does (objectdetect_findrot.cpp:834-845).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <functional>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/partapp_ps.h"
#include "ps_device.hpp"
#include "ps_plan.hpp"
#include "ps_pool.hpp"

namespace ps {
extern thread_local std::string g_last_error;

namespace {

constexpr int kIngThreads = 256;

// clip_scores_fill then computeLogGrid of one value
__device__ __forceinline__ float clip_log(float v) {
  if (v < 0.0f) v = 0.0001f;
  return v == 0.0f ? kLogZero : logf(v);
}

}  // namespace

__global__ __launch_bounds__(kIngThreads) void k_ingest_clear(unsigned long long *keys, long long n) {
  for (long long i = (long long)blockIdx.x * kIngThreads + threadIdx.x; i < n; i += (long long)gridDim.x * kIngThreads)
    keys[i] = 0ull;
}

// TM_DIRECT: source cell (x1, y1) of slice s lands on the nearest output cell
// of Tig (x1, y1); the key (scan position + 1, value bits) keeps the last.
__global__ __launch_bounds__(kIngThreads) void k_ingest_scatter(const float *__restrict__ grid,
                                                                const double *__restrict__ mats, int n, int gh,
                                                                int gw, int H, int W,
                                                                unsigned long long *__restrict__ keys) {
  const long long cells = (long long)gh * gw;
  const long long total = n * cells;
  for (long long i = (long long)blockIdx.x * kIngThreads + threadIdx.x; i < total;
       i += (long long)gridDim.x * kIngThreads) {
    const float v = grid[i];
    if (v == 0.0f) continue;  // NO_CLASS_VALUE is not written
    const int s = (int)(i / cells);
    const int rem = (int)(i - s * cells);
    const int y1 = rem / gw;
    const int x1 = rem - y1 * gw;
    const double *m = mats + 6 * s;
    const double x3 = m[0] * (double)x1 + m[1] * (double)y1 + m[2];
    const double y3 = m[3] * (double)x1 + m[4] * (double)y1 + m[5];
    const int ix = (int)floor(x3 + 0.5);
    const int iy = (int)floor(y3 + 0.5);
    if (ix >= 0 && ix < W && iy >= 0 && iy < H) {
      const unsigned scan = (unsigned)x1 * (unsigned)gh + (unsigned)y1 + 1u;
      const unsigned long long key = ((unsigned long long)scan << 32) | (unsigned long long)__float_as_uint(v);
      atomicMax(keys + ((long long)s * H + iy) * W + ix, key);
    }
  }
}

__global__ __launch_bounds__(kIngThreads) void k_ingest_finish(const unsigned long long *__restrict__ keys,
                                                               long long n, float *__restrict__ out) {
  for (long long i = (long long)blockIdx.x * kIngThreads + threadIdx.x; i < n; i += (long long)gridDim.x * kIngThreads) {
    const unsigned long long k = keys[i];
    out[i] = clip_log(k ? __uint_as_float((unsigned)(k & 0xffffffffull)) : 0.0f);
  }
}

// A slice's warp, rows 0-1: grid -> image for TM_DIRECT, image -> grid for
// TM_BILINEAR.
struct IngestWarp {
  double m[6];
};
// The warps of one launch, passed by value: no table in device memory to
// allocate, fill and free around a call of some 100 us.
struct IngestSlices {
  static constexpr int kMax = 80;  // 48 bytes each, below the 4 KB of kernel arguments
  IngestWarp one[kMax];
};
struct IngestTable {
  const IngestWarp *__restrict__ one;
};
template <bool TAB>
using IngestWarps = std::conditional_t<TAB, IngestTable, IngestSlices>;

constexpr int kTile = 32;                    // output pixels per side of a block
constexpr int kPix = kTile * kTile / kIngThreads;  // pixels of a thread, kTile / kPix rows apart

enum IngestMode : int { kIngBilinear = 0, kIngDirect = 1, kIngDirect4 = 2 };

// One block per 32 x 32 output pixels of a slice, four rows of pixels per
// thread, so that the cells a rotated block reads (46 x 46 at 45 degrees) stay
// in its CU's cache; the blocks of a slice run behind one L2 (xcd_block).
//
// Direct (TM_DIRECT): the reference scatters source cell (x1, y1) to the
// nearest pixel of Tig (x1, y1), the last cell of the x-outer, y-inner scan
// staying.  Here pixel (ix, iy) looks for that cell itself: the cells that can
// land on it lie in the box of half widths ex, ey about its preimage
// (ingest_gather bounds both roundings), walked from the scan's end, and each
// is tested with the scatter's own double arithmetic, so the same cell is
// found.  Direct4: no box of the launch holds more than 2 x 2 cells (every
// warp that does not shrink): the cells of all four pixels are tested and
// their loads issued before any is used.  Bilinear (TM_BILINEAR): the sample
// at inverse(Tig) (ix, iy) (within 10 float epsilons of a grid point: that
// point; last row / column and outside: NO_CLASS_VALUE).
//
// Every cell is read once from HBM and every pixel written once: 240 slices of
// 425 x 425 cells onto 300 x 300 pixels in 92 us (2.8 TB/s; a large copy
// reaches 5.2), the rest being vector work on the warp (147 us with every test
// in double).  The scatter into 64-bit keys took 575 us, with clearing and
// reading the keys 646 us, and several ms of allocating 172 MB for them.
//
// TAB: the warps come from a table (a choice at run time leaves them in vector
// registers, and 4 KB of arguments cost a launch a microsecond).  FLAT: 1024 pixels in a row instead of 32 x 32, for slices that
// fill few such tiles.
template <int MODE, bool TAB, bool FLAT>
__global__ __launch_bounds__(kIngThreads) void k_ingest_tile(const float *__restrict__ grid, IngestWarps<TAB> warps,
                                                             int first, int gh, int gw, int H, int W, int tile0,
                                                             int xtiles, float *__restrict__ out) {
  unsigned bx, by;
  xcd_block(bx, by);
  double m[6];
#pragma unroll
  for (int i = 0; i < 6; ++i) m[i] = warps.one[by].m[i];
  const int s = first + (int)by;
  const int ty = (tile0 + (int)bx) / xtiles;
  const unsigned x0 = (unsigned)(tile0 + (int)bx - ty * xtiles) * kTile + (threadIdx.x & 31);
  const unsigned y0 = (unsigned)ty * kTile + (threadIdx.x >> 5);
  const unsigned p0 = (unsigned)(tile0 + (int)bx) * (kTile * kTile) + threadIdx.x;
  if (!FLAT && x0 >= (unsigned)W) return;
  // pixel k of the thread
  auto row = [&](int k) { return FLAT ? (p0 + k * kIngThreads) / (unsigned)W : y0 + k * (kTile / kPix); };
  auto col = [&](int k, unsigned y) { return FLAT ? p0 + k * kIngThreads - y * (unsigned)W : x0; };
  const float *src = grid + (long long)s * gh * gw;
  float *dst = out + (long long)s * H * W;
  if (MODE == kIngDirect4) {
    const CellWarp cell(m);
    float c[kPix][4];
#pragma unroll
    for (int k = 0; k < kPix; ++k) {
      const unsigned y = row(k);
      cell.load4((int)col(k, y), (int)y, gw, gh, src, gw, c[k]);
    }
#pragma unroll
    for (int k = 0; k < kPix; ++k) {
      const unsigned y = row(k);
      if (y < (unsigned)H) dst[(long long)y * W + col(k, y)] = clip_log(last_cell(c[k]));
    }
  } else if (MODE == kIngDirect) {
    const CellWarp cell(m);
    for (int k = 0; k < kPix; ++k) {
      const unsigned y = row(k), x = col(k, y);
      if (y >= (unsigned)H) break;
      const double xd = (double)x, yd = (double)y;
      const double cx = cell.a[0] * xd + cell.a[1] * yd + cell.a[2], cy = cell.a[3] * xd + cell.a[4] * yd + cell.a[5];
      const int x_hi = (int)fmin(floor(cx + cell.ex), (double)(gw - 1)), x_lo = (int)fmax(ceil(cx - cell.ex), 0.0);
      const int y_hi = (int)fmin(floor(cy + cell.ey), (double)(gh - 1)), y_lo = (int)fmax(ceil(cy - cell.ey), 0.0);
      float v = 0.0f;
      for (int x1 = x_hi; x1 >= x_lo && v == 0.0f; --x1) {
        const double p = m[0] * (double)x1, q = m[3] * (double)x1;
        for (int y1 = y_hi; y1 >= y_lo; --y1)
          if (cell.lands(p, q, (double)y1, xd, yd)) {
            v = src[(long long)y1 * gw + x1];
            if (v != 0.0f) break;  // NO_CLASS_VALUE is not written
          }
      }
      dst[(long long)y * W + x] = clip_log(v);
    }
  } else {
    const float eps10 = 10.0f * FLT_EPSILON;
#pragma unroll
    for (int k = 0; k < kPix; ++k) {
      const unsigned y = row(k), x = col(k, y);
      if (y >= (unsigned)H) break;
      const double x1 = m[0] * (double)x + m[1] * (double)y + m[2];
      const double y1 = m[3] * (double)x + m[4] * (double)y + m[5];
      const int ix = (int)floor(x1);
      const int iy = (int)floor(y1);
      float r = 0.0f;
      if (ix >= 0 && ix < gw && iy >= 0 && iy < gh) {
        const float a = (float)(x1 - (double)ix);
        const float b = (float)(y1 - (double)iy);
        const float *p = src + (long long)iy * gw + ix;
        if (a < eps10 && b < eps10) {
          r = p[0];
        } else if (ix < gw - 1 && iy < gh - 1) {
          const float t0 = (1.0f - b) * (1.0f - a) * p[0];
          const float t1 = (1.0f - b) * a * p[1];
          const float t2 = b * (1.0f - a) * p[gw];
          const float t3 = b * a * p[gw + 1];
          r = t0 + t1 + t2 + t3;
        }
      }
      dst[(long long)y * W + x] = clip_log(r);
    }
  }
}

// Whether the scatter of a slice with warp m (grid -> image) can be taken as
// a gather; four: its boxes hold at most 2 x 2 cells.  The cells of a pixel lie within
// half the absolute row sums of the inverse about its preimage, plus what
// rounding adds: of the inverse (cancellation in its determinant) and of the
// forward map, both bounded here and required to stay far below the slack
// that the kernel adds.  A test costs some 0.3 ps of the chip and an atomic of
// the scatter 14-30 ps, and a pixel has |det a| atomics: the gather takes
// boxes of up to 64 cells per atomic (beyond, an extreme shear), and of at
// most 4096 (a thread's serial walk).  Measured on 48 slices onto 300 x 300
// pixels, scatter against gather: 120 and 21 us without shrinking, 2.4 ms and 89 us at
// 1 / 4, 9.8 ms and 109 us at 1 / 8 (boxes of some 130 cells).
bool ingest_gather(const double (&m)[6], int gh, int gw, int H, int W, bool &four) {
  double a[6];
  affine_inverse(m, a);
  const double D = std::fabs(m[0] * m[4] - m[3] * m[1]);
  const double cancel = std::fabs(m[0] * m[4]) + std::fabs(m[3] * m[1]);
  const double ax = std::fabs(a[0]) + std::fabs(a[1]), ay = std::fabs(a[3]) + std::fabs(a[4]);
  const double reach = (double)W + (double)H + std::fabs(m[2]) + std::fabs(m[5]) + 2.0;
  const double fwd = (std::fabs(m[0]) + std::fabs(m[3]) + 1.0) * gw + (std::fabs(m[1]) + std::fabs(m[4]) + 1.0) * gh;
  const double err = 32.0 * 2.220446049250313e-16 * (ax + ay) * (reach * (1.0 + cancel / D) + fwd);
  const double box = (ax + 2.0) * (ay + 2.0);
  four = std::max(ax, ay) + 2.0 * kCellSlack < 2.0;
  return std::isfinite(err) && err < 0.01 * kCellSlack && box <= 64.0 * (1.0 + 1.0 / D) && box <= 4096.0;
}

}  // namespace ps

using namespace ps;

extern "C" int ps_ingest_scores(const float *score_grid_dev, int n, int grid_height, int grid_width,
                                const double *Tig, int interpolate, int height, int width, float *log_unary_dev,
                                void *stream) {
  if (!score_grid_dev || !Tig || !log_unary_dev) return set_error(PS_ERR_INVALID_ARG, "null argument");
  if (n < 1 || grid_height < 1 || grid_width < 1 || height < 1 || width < 1)
    return set_error(PS_ERR_INVALID_ARG, "counts and sizes must be >= 1");
  if ((long long)grid_height * grid_width >= (1ll << 31) || (long long)height * width >= (1ll << 31) ||
      (long long)grid_width * grid_height + 1 >= (1ll << 32))
    return set_error(PS_ERR_UNSUPPORTED, "grids must have fewer than 2^31 cells per slice");
  for (int s = 0; s < n; ++s) {
    const double *T = Tig + 9 * s;
    if (interpolate && !(T[0] * T[4] - T[3] * T[1] != 0.0))
      return set_error(PS_ERR_INVALID_ARG, "Tig of slice " + std::to_string(s) + " is singular");
  }
  int devcount = 0;
  if (hipGetDeviceCount(&devcount) != hipSuccess || devcount == 0)
    return set_error(PS_ERR_NO_DEVICE, "no HIP device");
  std::vector<IngestWarp> warps(n);
  for (int s = 0; s < n; ++s) warp_matrix(Tig + 9 * s, interpolate != 0, warps[s].m);
  hipStream_t st = static_cast<hipStream_t>(stream);
  // a nearest warp onto its own input (log_unary_dev overlapping the grid) is
  // the scatter's, whose keys hold every value before the first is written
  const float *grid_end = score_grid_dev + (long long)n * grid_height * grid_width;
  const float *out_end = log_unary_dev + (long long)n * height * width;
  const bool overlap = std::less<const float *>()(score_grid_dev, out_end) &&
                       std::less<const float *>()(log_unary_dev, grid_end);
  bool gather = interpolate || !overlap, four = true;
  for (int s = 0; s < n && !interpolate && gather; ++s) {
    bool f = false;
    gather = ingest_gather(warps[s].m, grid_height, grid_width, height, width, f);
    four = four && f;
  }
  if (gather) {
    // the warps of one launch ride in its arguments, those of more slices come
    // from a table (in the arguments of several launches, 4 to 6 us each, 1440
    // slices of 128 x 128 pixels took 152 us sampled and 212 us direct)
    IngestWarp *tab = nullptr;
    hipError_t eg = hipSuccess;
    if (n > IngestSlices::kMax) {
      if (pool_get(&tab, sizeof(IngestWarp) * n) != hipSuccess)
        return set_error(PS_ERR_OUT_OF_MEMORY, "ingest workspace");
      eg = hipMemcpyAsync(tab, warps.data(), sizeof(IngestWarp) * n, hipMemcpyHostToDevice, st);
    }
    const int xtiles = (width + kTile - 1) / kTile, step = tab ? 32768 : IngestSlices::kMax;
    const long long square = (long long)xtiles * ((height + kTile - 1) / kTile);
    const long long row = ((long long)height * width + kTile * kTile - 1) / (kTile * kTile);
    // tiles keep a rotated block's cells in its CU's cache, unless a third of
    // their pixels or more lie outside the slice (2000 slices of 40 x 40 pixels:
    // 4 of them each, 2 rows)
    const bool flat = 3 * row <= 2 * square;
    const long long tiles = flat ? row : square;
    constexpr long long kTiles = 1ll << 22;  // tiles of one launch
    for (int s0 = 0; s0 < n; s0 += step) {
      const int ns = std::min(n - s0, step);
      for (long long t0 = 0; t0 < tiles && eg == hipSuccess; t0 += kTiles) {
        const dim3 grid((unsigned)std::min(kTiles, tiles - t0), (unsigned)ns), blk(kIngThreads);
        auto launch = [&](auto tabc, auto flatc) {
          constexpr bool T = decltype(tabc)::value, F = decltype(flatc)::value;
          IngestWarps<T> w;
          if constexpr (T) w.one = tab + s0;
          else std::copy(warps.begin() + s0, warps.begin() + s0 + ns, w.one);
          auto mode = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, grid, blk, 0, st, score_grid_dev, w, s0, grid_height, grid_width, height, width,
                               (int)t0, xtiles, log_unary_dev);
          };
          if (interpolate) mode(k_ingest_tile<kIngBilinear, T, F>);
          else if (four) mode(k_ingest_tile<kIngDirect4, T, F>);
          else mode(k_ingest_tile<kIngDirect, T, F>);
        };
        const std::true_type yes;
        const std::false_type no;
        if (tab && flat) launch(yes, yes);
        else if (tab) launch(yes, no);
        else if (flat) launch(no, yes);
        else launch(no, no);
        eg = hipGetLastError();
      }
    }
    if (eg == hipSuccess) eg = hipStreamSynchronize(st);
    pool_put(tab, eg == hipSuccess);
    if (eg != hipSuccess) return set_error(PS_ERR_HIP, std::string("ingest: ") + hipGetErrorString(eg));
    return PS_OK;
  }
  // the buffers overlap, or some slice's warp is singular, too ill-conditioned
  // or shrinks too much for the gather: scatter with last-writer keys
  const long long out_n = (long long)n * height * width;
  const size_t mat_bytes = (sizeof(IngestWarp) * (size_t)n + 255) & ~(size_t)255;
  void *ws = nullptr;
  hipError_t e = pool_get(&ws, mat_bytes + (size_t)out_n * sizeof(unsigned long long));
  if (e != hipSuccess) return set_error(PS_ERR_OUT_OF_MEMORY, "ingest workspace");
  double *mats_dev = static_cast<double *>(ws);
  unsigned long long *keys = reinterpret_cast<unsigned long long *>(static_cast<char *>(ws) + mat_bytes);
  e = hipMemcpyAsync(mats_dev, warps.data(), sizeof(IngestWarp) * (size_t)n, hipMemcpyHostToDevice, st);
  auto blocks = [](long long m) {
    long long g = (m + kIngThreads - 1) / kIngThreads;
    return (unsigned)(g < 8192 ? (g < 1 ? 1 : g) : 8192);
  };
  if (e == hipSuccess) {
    const long long in_n = (long long)n * grid_height * grid_width;
    hipLaunchKernelGGL(k_ingest_clear, dim3(blocks(out_n)), dim3(kIngThreads), 0, st, keys, out_n);
    hipLaunchKernelGGL(k_ingest_scatter, dim3(blocks(in_n)), dim3(kIngThreads), 0, st, score_grid_dev, mats_dev, n,
                       grid_height, grid_width, height, width, keys);
    hipLaunchKernelGGL(k_ingest_finish, dim3(blocks(out_n)), dim3(kIngThreads), 0, st, keys, out_n, log_unary_dev);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  pool_put(ws, e == hipSuccess);
  if (e != hipSuccess) return set_error(PS_ERR_HIP, std::string("ingest: ") + hipGetErrorString(e));
  return PS_OK;
}

// ------------------------------------------------------------- extra unaries
// The additions findObjectImageRotJoints makes to the log unaries before the
// sweep (objectdetect_findrot.cpp:896-948), in place on device grids, with
// the reference's float / double mix (objectdetect_icps.cpp is compiled with
// `using namespace std`: log(float) is the float log, exp and pow(float, int)
// work in double, and `float += double` adds in double and rounds once).

namespace ps {
namespace {

// Slices per thread of the two adds below: a thread forms its pixel's term
// once for kAddSlices slices, whose loads are all in flight together (one
// thread per pixel with every slice in turn waits for each load: 8.5 and 11.9
// us per 24 x 300 x 300 grid, now 7.0 and 6.7).
constexpr int kAddSlices = 6;

// setTorsoPosPrior (objectdetect_icps.cpp:137-191): the clipped log prior of a
// pixel, added to its slices.
__global__ __launch_bounds__(kIngThreads) void k_torso_prior(float *g, int n_slices, int H, int W, float mu_x,
                                                             float mu_y, float var_x, float var_y, float weight) {
  const long long hw = (long long)H * W;
  const long long i = (long long)blockIdx.x * kIngThreads + threadIdx.x;
  if (i >= hw) return;
  for (int k0 = (int)blockIdx.y * kAddSlices; k0 < n_slices; k0 += (int)gridDim.y * kAddSlices) {
    float v[kAddSlices];
#pragma unroll
    for (int j = 0; j < kAddSlices; ++j) v[j] = g[(long long)min(k0 + j, n_slices - 1) * hw + i];
    const int iy = (int)(i / W), ix = (int)(i - (long long)iy * W);
    const float img_c_x = (float)(0.5 * W), img_c_y = (float)(0.5 * H);
    const float ix_rel = img_c_x - (float)ix;
    const float iy_rel = img_c_y - (float)iy;
    // pow(d, 2) of a float d is exact in double
    const double dx = (double)(ix_rel - mu_x), dy = (double)(iy_rel - mu_y);
    const float score_x = (float)exp(-0.5 * (dx * dx) / (double)var_x);
    const float score_y = (float)exp(-0.5 * (dy * dy) / (double)var_y);
    float score = weight * score_x * score_y;
    if ((double)score < 1e-4) score = 1e-4f;
    const double pred = (double)logf(score);
#pragma unroll
    for (int j = 0; j < kAddSlices; ++j)
      if (k0 + j < n_slices) g[(long long)(k0 + j) * hw + i] = (float)((double)v[j] + pred);
  }
}

// addLoadDPMScore's accumulation (:469-484, raw scores), addDPMScore
// (:490-524, log grids) and the torso path's computeLogGrid + addDPMScore
// (objectdetect_findrot.cpp:896-903)
__global__ __launch_bounds__(kIngThreads) void k_dpm_add(float *g, int S, int R, int H, int W, const float *dpm,
                                                         int n_dpm, float weight, int mode, double log_clip) {
  const long long hw = (long long)H * W;
  const long long i = (long long)blockIdx.x * kIngThreads + threadIdx.x;
  if (i >= hw) return;
  const bool per_r = mode == PS_DPM_RAW ? n_dpm == R : n_dpm > 1;
  const int n = S * R;
  for (int k0 = (int)blockIdx.y * kAddSlices; k0 < n; k0 += (int)gridDim.y * kAddSlices) {
    float v[kAddSlices], d[kAddSlices];
#pragma unroll
    for (int j = 0; j < kAddSlices; ++j) {
      const int k = min(k0 + j, n - 1);
      v[j] = g[(long long)k * hw + i];
      d[j] = dpm[(long long)(per_r ? k % R : 0) * hw + i];
    }
#pragma unroll
    for (int j = 0; j < kAddSlices; ++j) {
      if (k0 + j >= n) break;
      float *p = g + (long long)(k0 + j) * hw + i;
      if (mode == PS_DPM_RAW) {
        const double add = (double)d[j] > 1e-4 ? (double)(weight * logf(d[j])) : log_clip;
        *p = (float)((double)v[j] + add);
      } else {
        const float lv = mode == PS_DPM_LOG_OF_RAW ? (d[j] == 0.0f ? kLogZero : logf(d[j])) : d[j];
        *p = v[j] + weight * lv;
      }
    }
  }
}

// addExtraUnary (:526-548)
__global__ __launch_bounds__(kIngThreads) void k_add_scaled(float *g, const float *e, long long n, float weight) {
  for (long long i = (long long)blockIdx.x * kIngThreads + threadIdx.x; i < n; i += (long long)gridDim.x * kIngThreads)
    g[i] = g[i] + weight * e[i];
}

dim3 pixel_blocks(long long hw, long long n_slices) {
  return dim3((unsigned)((hw + kIngThreads - 1) / kIngThreads),
              (unsigned)std::min<long long>((n_slices + kAddSlices - 1) / kAddSlices, 65535));
}

}  // namespace
}  // namespace ps

extern "C" int ps_add_torso_pos_prior(float *root_unary_dev, int n_slices, int height, int width,
                                      const double params[4], float weight, void *stream) {
  if (!root_unary_dev || !params) return set_error(PS_ERR_INVALID_ARG, "null argument");
  if (n_slices < 1 || height < 1 || width < 1) return set_error(PS_ERR_INVALID_ARG, "counts and sizes must be >= 1");
  if ((long long)height * width >= (1ll << 40)) return set_error(PS_ERR_UNSUPPORTED, "grid too large");
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(k_torso_prior, pixel_blocks((long long)height * width, n_slices), dim3(kIngThreads), 0, st,
                     root_unary_dev, n_slices, height, width, (float)params[0], (float)params[1], (float)params[2],
                     (float)params[3], weight);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(PS_ERR_HIP, std::string("torso prior: ") + hipGetErrorString(e));
  return PS_OK;
}

extern "C" int ps_add_dpm_score(float *part_unary_dev, int S, int R, int height, int width, const float *dpm_dev,
                                int n_dpm, float weight, int mode, void *stream) {
  if (!part_unary_dev || !dpm_dev) return set_error(PS_ERR_INVALID_ARG, "null argument");
  if (S < 1 || R < 1 || height < 1 || width < 1 || n_dpm < 1)
    return set_error(PS_ERR_INVALID_ARG, "counts and sizes must be >= 1");
  if (mode != PS_DPM_RAW && mode != PS_DPM_LOG && mode != PS_DPM_LOG_OF_RAW)
    return set_error(PS_ERR_INVALID_ARG, "unknown DPM mode " + std::to_string(mode));
  if (mode != PS_DPM_RAW) {
    if (!(weight > 0)) return set_error(PS_ERR_INVALID_ARG, "dpm_weight must be > 0 (objectdetect_icps.cpp:501)");
    if (n_dpm > 1 && n_dpm < R) return set_error(PS_ERR_INVALID_ARG, "a rotation-dependent DPM prior needs R grids");
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  const long long hw = (long long)height * width, n = (long long)S * R;
  const bool per_r = mode == PS_DPM_RAW ? n_dpm == R : n_dpm > 1;
  auto add = [&](float *g, int s, int r, const float *dpm, int nd) {
    hipLaunchKernelGGL(k_dpm_add, pixel_blocks(hw, (long long)s * r), dim3(kIngThreads), 0, st, g, s, r, height, width,
                       dpm, nd, weight, mode, std::log(1e-4));
  };
  // scores that are slices of the part itself: a slice already added to is read
  // as it then is, so the slices go one after another
  const std::less<const float *> before;
  if (before(dpm_dev, part_unary_dev + n * hw) && before(part_unary_dev, dpm_dev + (per_r ? R : 1) * hw)) {
    for (long long k = 0; k < n; ++k) add(part_unary_dev + k * hw, 1, 1, dpm_dev + (per_r ? k % R : 0) * hw, 1);
  } else {
    add(part_unary_dev, S, R, dpm_dev, n_dpm);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(PS_ERR_HIP, std::string("dpm score: ") + hipGetErrorString(e));
  return PS_OK;
}

extern "C" int ps_add_extra_unary(float *log_unary_dev, const float *extra_dev, long long n, float weight,
                                  void *stream) {
  if (!log_unary_dev || !extra_dev) return set_error(PS_ERR_INVALID_ARG, "null argument");
  if (n < 0) return set_error(PS_ERR_INVALID_ARG, "n must be >= 0");
  if (n == 0) return PS_OK;
  long long g = (n + kIngThreads - 1) / kIngThreads;
  hipStream_t st = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(k_add_scaled, dim3((unsigned)(g < 65536 ? g : 65536)), dim3(kIngThreads), 0, st, log_unary_dev,
                     extra_dev, n, weight);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(PS_ERR_HIP, std::string("extra unary: ") + hipGetErrorString(e));
  return PS_OK;
}
