// Device helpers shared by the sweep kernels (ps_kernels.hip) and the
// eigenbasis path of off-diagonal covariances (ps_offdiag.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "ps_internal.hpp"

namespace ps {

// order-preserving 32-bit key of a float (larger float, larger key)
__device__ __forceinline__ unsigned f2key(float f) {
  unsigned u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float key2f(unsigned k) {
  unsigned u = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
  return __uint_as_float(u);
}
// argmax key: larger score wins, then the smaller flat index (the first
// maximum of a C-order scan, objectdetect_findrot.cpp:261-266)
__device__ __forceinline__ unsigned long long amax_key(float v, unsigned idx) {
  return ((unsigned long long)f2key(v) << 32) | (unsigned long long)(0xffffffffu - idx);
}

// The block of a 2-D grid (x fastest) renumbered so that each of the 8 XCDs,
// to which the dispatcher hands workgroups round-robin in launch order, gets
// one contiguous range of logical blocks.  Neighbouring tiles (which share the
// cache lines at their edges when grid rows are not 128-byte aligned) then run
// at the same time behind the same L2.
__device__ __forceinline__ void xcd_block(unsigned &bx, unsigned &by) {
  const unsigned n = gridDim.x * gridDim.y;
  const unsigned b = blockIdx.y * gridDim.x + blockIdx.x;
  const unsigned xcd = b & 7u, k = b >> 3;
  const unsigned q = n >> 3, rem = n & 7u;
  const unsigned l = xcd < rem ? xcd * (q + 1) + k : rem * (q + 1) + (xcd - rem) * q + k;
  by = l / gridDim.x;
  bx = l - by * gridDim.x;
}

// A column pass's rows [ya, yb), a part (gridDim.z of them) of a strip that
// walks tiles of th rows.
__device__ __forceinline__ void col_part(int H, int th, int &ya, int &yb) {
  const int rows = ((H + th - 1) / th + (int)gridDim.z - 1) / (int)gridDim.z * th;
  ya = (int)blockIdx.z * rows;
  yb = min(H, ya + rows);
}

__device__ __forceinline__ unsigned wave_max_u32(unsigned v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = max(v, (unsigned)__shfl_xor((int)v, o, 64));
  return v;
}
__device__ __forceinline__ unsigned long long wave_max_u64(unsigned long long v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    unsigned long long w = __shfl_xor(v, o, 64);
    v = w > v ? w : v;
  }
  return v;
}

// An instance left out of this execution (Bases::active names the instances
// that run): every block of its jobs exits at once.
__device__ __forceinline__ bool skip_inst(const Bases &b, int inst) { return b.active && b.active[inst] == 0u; }

__device__ __forceinline__ unsigned *max_key(const Bases &b, int k) { return b.max_keys + (size_t)k * kMaxKeyStride; }
__device__ __forceinline__ unsigned long long *map_key(const Bases &b, int k) {
  return b.map_keys + (size_t)k * kMapKeyStride;
}
// the MAP certificate's, or null where there is none
__device__ __forceinline__ unsigned long long *top2_key(const Bases &b, int k) {
  return b.top2_keys ? b.top2_keys + (size_t)k * kMapKeyStride : nullptr;
}

// A block's result for the keys it feeds: the waves' parts, each merged over
// its lanes, meet in LDS and one thread raises the keys.  Atomics on one cache
// line queue up at 4 to 13 ns each: by a wave each, all keys of an instance in
// one line, the leaf maxima of an image of 300x300x48 took 70 us for 17 us of
// reading (27 so, and 17 with a line per key).  (Reading a key first and raising
// it only where it is lower queues up just as much once thousands of waves are
// in flight, and each then waits for its answer: 957 instead of 299 us for the
// leaf maxima of 32 images.)
struct KeyPart {
  unsigned key = 0u;                // of a source's maximum
  unsigned long long amax = 0ull;   // (value key << 32) | flipped index of the best state
  unsigned second = 0u;             // value key of the second best state, for the MAP certificate
  __device__ __forceinline__ void merge(const KeyPart &o) {
    key = max(key, o.key);
    second = max(max(second, o.second), min((unsigned)(amax >> 32), (unsigned)(o.amax >> 32)));
    amax = o.amax > amax ? o.amax : amax;
  }
};
// the top-2 of a wave's lanes (k1 >= k2, every state seen by one lane only):
// the second key, in every lane
__device__ __forceinline__ unsigned wave_second(unsigned k1, unsigned k2) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned o1 = (unsigned)__shfl_xor((int)k1, o, 64), o2 = (unsigned)__shfl_xor((int)k2, o, 64);
    k2 = max(max(k2, o2), min(k1, o1));
    k1 = max(k1, o1);
  }
  return k2;
}
// A (best << 32) | second word raised by a compare-and-swap loop; the word
// only grows, so the loop ends.
__device__ __forceinline__ void top2_raise(unsigned long long *slot, unsigned k1, unsigned k2) {
  unsigned long long old = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (;;) {
    const unsigned a1 = (unsigned)(old >> 32), a2 = (unsigned)old;
    const unsigned long long nw = ((unsigned long long)max(a1, k1) << 32) | max(max(a2, k2), min(a1, k1));
    if (nw == old) break;
    const unsigned long long prev = atomicCAS(slot, old, nw);
    if (prev == old) break;
    old = prev;
  }
}
// Every thread of the block calls it, with its wave's part; red holds one
// entry per wave (LDS that no thread reads or writes any more).  Null keys are
// not fed.
__device__ __forceinline__ void block_raise(uint4 *red, KeyPart p, unsigned *max_key, unsigned long long *map_key,
                                            unsigned long long *top2_key) {
  const int waves = (int)(blockDim.x >> 6);
  if ((threadIdx.x & 63) == 0)
    red[threadIdx.x >> 6] = make_uint4(p.key, (unsigned)p.amax, (unsigned)(p.amax >> 32), p.second);
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int w = 1; w < waves; ++w) {
    const uint4 v = red[w];
    KeyPart o;
    o.key = v.x;
    o.amax = (unsigned long long)v.z << 32 | v.y;
    o.second = v.w;
    p.merge(o);
  }
  if (max_key && p.key) atomicMax(max_key, p.key);
  if (map_key && p.amax) atomicMax(map_key, p.amax);
  if (top2_key && p.amax) top2_raise(top2_key, (unsigned)(p.amax >> 32), p.second);
}
// one more value key into a lane's top-2
__device__ __forceinline__ void top2_add(unsigned &k1, unsigned &k2, unsigned k) {
  if (k > k1) {
    k2 = k1;
    k1 = k;
  } else if (k > k2) {
    k2 = k;
  }
}

// Base pointer of a GridRef.  Written as selects on the (uniform) buffer id
// so the kernel argument block is never copied to scratch for indexing.
__device__ __forceinline__ float *base_of(const Bases &b, int buf) {
  float *p = buf == kBufMarginal ? b.marginal : b.scratch;
  p = buf == kBufUnary ? const_cast<float *>(b.unary) : p;
  p = buf == kBufRoot ? b.root : p;
  return p;
}
__device__ __forceinline__ const float *cptr(const Bases &b, const GridRef &g) { return base_of(b, g.buf) + g.off; }
__device__ __forceinline__ float *mptr(const Bases &b, const GridRef &g) { return base_of(b, g.buf) + g.off; }

__device__ __forceinline__ bool masked(const UnaryMask &m, int r, int x, int W) {
  return ((m.rot_bits >> r) & 1ull) || x < m.strip || x >= W - m.strip;
}

// The nearest scatter (TM_DIRECT, multi_array_transform.hpp:122-239) seen from
// an output cell: which source cells (x1, y1) have
// floor(m (x1, y1) + 0.5) = (x, y).  They lie within half the absolute row
// sums of the inverse about the cell's preimage; kCellSlack covers what
// rounding adds (the callers make sure that it does).
constexpr double kCellSlack = 1e-3;

// the inverse of an affine map, rows 0-1
__host__ __device__ __forceinline__ void affine_inverse(const double *m, double (&a)[6]) {
  const double D = m[0] * m[4] - m[3] * m[1];
  a[0] = m[4] / D;
  a[1] = -m[1] / D;
  a[3] = -m[3] / D;
  a[4] = m[0] / D;
  a[2] = -(a[0] * m[2] + a[1] * m[5]);
  a[5] = -(a[3] * m[2] + a[4] * m[5]);
}

struct CellWarp {
  double m[6], a[6], ex, ey;
  __device__ __forceinline__ explicit CellWarp(const double *map) {
#pragma unroll
    for (int i = 0; i < 6; ++i) m[i] = map[i];
    affine_inverse(m, a);
    ex = 0.5 * (fabs(a[0]) + fabs(a[1])) + kCellSlack;
    ey = 0.5 * (fabs(a[3]) + fabs(a[4])) + kCellSlack;
  }
  // the scatter's own test of cell (x1, y1): p = m0 x1, q = m3 x1
  __device__ __forceinline__ bool lands(double p, double q, double y1, double xd, double yd) const {
    const double tx = (p + m[1] * y1 + m[2]) + 0.5, ty = (q + m[4] * y1 + m[5]) + 0.5;
    return tx >= xd && tx < xd + 1.0 && ty >= yd && ty < yd + 1.0;
  }
  // Where the box holds at most 2 x 2 cells: their values (0 for a cell that
  // does not land on (x, y) or lies outside), the scan's last first.  A
  // cell's landing point relative to the output cell's centre is formed in
  // float from the fractions of the double preimage, off by less than tol, so
  // only a cell that close to the edge takes the double test.
  __device__ __forceinline__ void load4(int x, int y, int gw, int gh, const float *src, int pitch,
                                        float (&c)[4]) const {
    const float n0 = (float)m[0], n1 = (float)m[1], n3 = (float)m[3], n4 = (float)m[4];
    const float tolx = 1e-6f * (1.0f + fabsf(n0) + fabsf(n1)), toly = 1e-6f * (1.0f + fabsf(n3) + fabsf(n4));
    const double xd = (double)x, yd = (double)y;
    const double cx = a[0] * xd + a[1] * yd + a[2], cy = a[3] * xd + a[4] * yd + a[5];
    const double xh = floor(cx + ex), yh = floor(cy + ey);  // the box's last column and row
    const float fx = (float)(xh - cx), fy = (float)(yh - cy);
    const int xi = (int)xh, yi = (int)yh;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int x1 = xi - (j >> 1), y1 = yi - (j & 1);
      const float u = fx - (float)(j >> 1), w = fy - (float)(j & 1);
      const float dx = fabsf(n0 * u + n1 * w) - 0.5f, dy = fabsf(n3 * u + n4 * w) - 0.5f;
      c[j] = 0.0f;
      if ((unsigned)x1 < (unsigned)gw && (unsigned)y1 < (unsigned)gh && dx < tolx && dy < toly) {
        bool hit = true;
        if (dx > -tolx || dy > -toly) hit = lands(m[0] * (double)x1, m[3] * (double)x1, (double)y1, xd, yd);
        if (hit) c[j] = src[(long long)y1 * pitch + x1];
      }
    }
  }
};
// the value that stays: the last of the scan that is not 0 (which is not written)
__device__ __forceinline__ float last_cell(const float (&c)[4]) {
  return c[0] != 0.0f ? c[0] : c[1] != 0.0f ? c[1] : c[2] != 0.0f ? c[2] : c[3];
}

// log of a filter response, 0 -> LOG_ZERO (multi_array_op.hpp:154-166), on
// the hardware log2 (v_log_f32, about 1 ulp): a response the hardware takes
// for 0 (below 2^-126 where it flushes) is LOG_ZERO too
__device__ __forceinline__ float log0(float v) {
  const float l = __builtin_amdgcn_logf(v);
  return l > -INFINITY ? l * 0.693147180559945309f : kLogZero;
}

// The caller's accumulation of a column pass specialised per destination
// kind (EpiKind), so that a kernel's loads for it are unconditional
// straight-line code.
template <int EPI>
struct Epi {
  static constexpr bool kNeedU = EPI >= kEpiUpNodeU;  // reads the unary of the part written
  static constexpr bool kNeedB = EPI == kEpiDownMid;  // reads the stored upward belief
  static constexpr bool kDown = EPI >= kEpiDownLeaf;
  // grids at a second row pitch (byte offset ebs): the unary a chain-node
  // belief adds (the belief is the plan's grid, the unary the caller's), or
  // the stored belief and the next source of a five-grid downward epilogue
  // (the marginal and the unary it adds are at dst's pitch)
  static constexpr bool kSide = EPI == kEpiUpNodeU || EPI == kEpiDownMid;
  float vmax = -INFINITY;  // max of the written next source / belief
  unsigned best_key = 0u, best_eb = 0u;  // argmax of the marginal (key, byte offset in the slice)
  unsigned second_key = 0u;              // second largest marginal value (key) of the lane

  // one output at byte offset eb of slice r of dst, ebs of dst2 (both point
  // at the slice); pu / pb are only read when the kind needs them
  __device__ __forceinline__ void store(float *dst, float *dst2, unsigned eb, unsigned ebs, float msg, float pu,
                                        float pb, bool xmask, bool leaf_u) {
    auto at = [](float *p, unsigned o) -> float & { return *reinterpret_cast<float *>(reinterpret_cast<char *>(p) + o); };
    if (EPI == kEpiUpRoot || EPI == kEpiUpNode) {
      at(dst, eb) = msg;
      if (EPI == kEpiUpNode) vmax = fmaxf(vmax, msg);
    } else if (EPI == kEpiUpNodeU) {
      const float v = msg + (xmask ? kLogZero : pu);
      at(dst, eb) = v;
      vmax = fmaxf(vmax, v);
    } else {
      const float u = xmask ? kLogZero : pu;
      const float mg = (kNeedB ? pb : (leaf_u ? u : 0.0f)) + msg;
      at(dst, eb) = mg;
      const unsigned k = f2key(mg);
      if (k > best_key) {  // a lane's outputs come in ascending flat order: the first maximum stays
        second_key = best_key;
        best_key = k;
        best_eb = eb;
      } else if (k > second_key) {
        second_key = k;
      }
      if (kNeedB) {
        const float v2 = u + msg;
        at(dst2, ebs) = v2;
        vmax = fmaxf(vmax, v2);
      }
    }
  }
  // a padding column of the plan's grids (past W, inside the row pitch):
  // LOG_ZERO, so that every line of such a row is written whole by one wave
  // (no reduction sees it)
  __device__ __forceinline__ void pad(float *dst, float *dst2, unsigned eb, unsigned ebs, bool pad_a, bool pad_b) {
    auto at = [](float *p, unsigned o) -> float & { return *reinterpret_cast<float *>(reinterpret_cast<char *>(p) + o); };
    if (pad_a) at(dst, eb) = kLogZero;
    if (kNeedB && pad_b) at(dst2, ebs) = kLogZero;
  }
  // the keys the outputs feed; every thread of the block calls it, and lds (16
  // bytes per wave) is free once all have
  __device__ __forceinline__ void flush(const Bases &b, const MsgJob &J, long long slice0, void *lds) {
    constexpr bool kKey = EPI == kEpiUpNode || EPI == kEpiUpNodeU || EPI == kEpiDownMid;
    if (!kKey && !kDown) return;
    KeyPart p;
    if (kKey) p.key = wave_max_u32(vmax > -INFINITY ? f2key(vmax) : 0u);
    if (kDown) {
      const unsigned flat = (unsigned)(slice0 + (best_eb >> 2));
      p.amax = wave_max_u64(best_key ? ((unsigned long long)best_key << 32) | (0xffffffffull - flat) : 0ull);
      if (b.top2_keys) p.second = wave_second(best_key, second_key);
    }
    __syncthreads();
    block_raise(static_cast<uint4 *>(lds), p, kKey ? max_key(b, kDown ? J.dst2_key : J.dst_key) : nullptr,
                kDown ? map_key(b, J.map_slot) : nullptr, kDown ? top2_key(b, J.map_slot) : nullptr);
  }
};

// Row pitch of an epilogue's side grids (Epi::kSide): the unary's for a
// chain-node belief, the next source's (and stored belief's) for the
// five-grid downward epilogue; dst's otherwise
template <int EPI>
__device__ __forceinline__ int epi_pitch_b(const MsgJob &J) {
  return EPI == kEpiUpNodeU ? J.dst_unary.pitch : (EPI == kEpiDownMid ? J.dst2.pitch : J.dst.pitch);
}

// Reductions a message's epilogue feeds: the max of the next upward source,
// the argmax of a marginal and the max of the next downward source.
struct DstAcc {
  unsigned kmax1 = 0u, kmax2 = 0u;
  unsigned long long amax = 0ull;
  unsigned second = 0u;  // second largest marginal value (key)
};

// The caller's accumulation of one message value msg at element
// flat = r*H*W + y*W + x of slice r, stored at dst[e] / dst2[e2] (each grid's
// own element of (r, y, x) at its row pitch).  pu is the unary of the part
// written (read when need_u), pb the stored upward belief (read when need_b),
// xmask the part's mask at (r, x).
//   up, parent = root:  the message slot (objectdetect_findrot.cpp:637-649)
//   up, chain node:     belief = 0 + message (+ unary) (:637, :652-654)
//   down:               marginal = belief + message (:201), next downward
//                       source = unary + message (:220-222)
__device__ __forceinline__ void dst_store(const MsgJob &J, float *dst, float *dst2, long long e, long long e2,
                                          unsigned flat, bool xmask, float msg, float pu, float pb, DstAcc &a) {
  if (J.dst_kind == kDstUpRoot) {
    dst[e] = msg;
  } else if (J.dst_kind == kDstUpNode) {
    float v = msg;
    if (J.dst_add_unary) v = v + (xmask ? kLogZero : pu);
    dst[e] = v;
    a.kmax1 = max(a.kmax1, f2key(v));
  } else {
    const float u = xmask ? kLogZero : pu;
    const float base = J.dst_base == 0 ? pb : (J.dst_base == 1 ? u : 0.0f);
    const float mg = base + msg;
    dst[e] = mg;
    const unsigned long long k = amax_key(mg, flat);
    const unsigned kv = (unsigned)(k >> 32), kb = (unsigned)(a.amax >> 32);
    a.second = kv > kb ? kb : max(a.second, kv);
    a.amax = k > a.amax ? k : a.amax;
    if (dst2) {
      const float v2 = u + msg;
      dst2[e2] = v2;
      a.kmax2 = max(a.kmax2, f2key(v2));
    }
  }
}

// The keys DstAcc feeds; every thread of the block calls it (red: LDS, an
// entry per wave).
__device__ __forceinline__ void dst_flush(const Bases &b, const MsgJob &J, bool has_dst2, const DstAcc &a, uint4 *red) {
  KeyPart p;
  if (J.dst_kind == kDstUpNode) {
    p.key = wave_max_u32(a.kmax1);
    block_raise(red, p, max_key(b, J.dst_key), nullptr, nullptr);
  } else if (J.dst_kind == kDstDown) {
    p.amax = wave_max_u64(a.amax);
    if (b.top2_keys) p.second = wave_second((unsigned)(a.amax >> 32), a.second);
    if (has_dst2) p.key = wave_max_u32(a.kmax2);
    block_raise(red, p, has_dst2 ? max_key(b, J.dst2_key) : nullptr, map_key(b, J.map_slot),
                top2_key(b, J.map_slot));
  }
}

}  // namespace ps
