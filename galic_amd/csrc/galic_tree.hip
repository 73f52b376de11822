// galic_tree.hip -- Barnes-Hut fill of the force and potential tables on gfx950.
//
// The reference builds an oct-tree by inserting particles one at a time
// (forcetree.c:369-495), sums monopole moments recursively
// (forcetree.c:591-722), and walks it once per target with a geometric opening
// criterion and Gadget-2 spline softening (forcetree_walk.c:12-222).  The tree
// that insertion produces is unique: a node exists for every cube of the
// subdivision that holds at least two particles, down to the depth where they
// separate.  Here the same tree is built in parallel:
//   1. integer positions exactly as forcetree.c:199-201 (52 mantissa bits of
//      (x - corner)/len + 1), Morton keys from their top 21 bits per axis with
//      the child numbering x + 2y + 4z of forcetree.c:216-217;
//   2. radix sort of the keys;
//   3. level by level, every node splits its sorted particle range into the 8
//      child ranges by binary search; ranges of >= 2 particles become nodes;
//   4. moments bottom-up in FP64, in child order 0..7 as the reference;
//   5. nextnode/sibling threading top-down, giving the reference's depth-first
//      walk order;
//   6. the tree is walked without a stack, one target per lane, the 64 targets of a wave on one path;
//      or by groups of targets with a list of interactions each (k_walk32g).
// Particles that share all 21 key levels (closer than len/2^21) stay together
// in a leaf bucket; opening it interacts with them one by one.  The reference
// would keep splitting; this changes results only for targets within that
// distance of such a pair.
#include <hip/hip_runtime.h>
#include <rocprim/device/device_radix_sort.hpp>
#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "../../include/galic_hip.h"
#include "galic_ctx.h"
#include "galic_kernels.h"
#include "galic_pool.h"

namespace galic {
galic_ctx *bound_ctx();
Ctx &ctx_state(galic_ctx *ctx);
namespace tree {

constexpr int kMaxDepth = 21;

struct Tree {
  int nsrc = 0;
  int cap = 0;
  double corner[3] = {0, 0, 0}, dlen = 1;  // the domain cube
  // sorted sources: position and mass
  double4 *src = nullptr;
  unsigned long long *key = nullptr;
  int *nextp = nullptr;  // next walk entry after each particle
  // nodes
  int *first = nullptr, *count = nullptr;
  int *child = nullptr;  // [node][8]: -1, particle (< nsrc) or nsrc + node
  double4 *com = nullptr;  // centre of mass and mass
  int4 *meta = nullptr;    // side length (float bits), sibling, nextnode, 1 for a leaf bucket
  double *quad = nullptr;  // [6][node] traceless quadrupole xx, yy, zz, xy, xz, yz (with quadrupole moments)
  float4 *quadf = nullptr; // [node][2] the same in FP32 for the FP32 walk: (xx, yy, zz, xy), (xz, yz, 0, 0)
  int *counter = nullptr;
  std::vector<int> level_lo;  // nodes of depth d are [level_lo[d], level_lo[d+1])
};

// Points of the host's interleaved arrays (stride 3) or of one array per coordinate (stride 1).
struct Points {
  const double *x, *y, *z;
  int stride;
};

__device__ __forceinline__ unsigned long long spread3(unsigned long long v) {
  v &= 0x1fffffULL;
  v = (v | (v << 32)) & 0x1f00000000ffffULL;
  v = (v | (v << 16)) & 0x1f0000ff0000ffULL;
  v = (v | (v << 8)) & 0x100f00f00f00f00fULL;
  v = (v | (v << 4)) & 0x10c30c30c30c30c3ULL;
  v = (v | (v << 2)) & 0x1249249249249249ULL;
  return v;
}

__device__ __forceinline__ unsigned long long mantissa(double d) {
  return (unsigned long long)__double_as_longlong(d) & 0xFFFFFFFFFFFFFull;
}

// forcetree.c:197-210 integer positions; Morton key from bits 51..31 of each
__global__ void k_keys(int n, Points P, double cx, double cy, double cz, double inv_len, unsigned long long *key,
                       int *idx) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i >= n) return;
  const size_t k = (size_t)i * P.stride;
  unsigned long long xb = mantissa(((P.x[k] - cx) * inv_len) + 1.0) >> 31;
  unsigned long long yb = mantissa(((P.y[k] - cy) * inv_len) + 1.0) >> 31;
  unsigned long long zb = mantissa(((P.z[k] - cz) * inv_len) + 1.0) >> 31;
  key[i] = spread3(xb) | (spread3(yb) << 1) | (spread3(zb) << 2);
  idx[i] = i;
}

__global__ void k_gather(int n, const int *idx, Points P, const double *pm, double4 *src) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i >= n) return;
  const int j = idx[i];
  const size_t k = (size_t)j * P.stride;
  src[i] = make_double4(P.x[k], P.y[k], P.z[k], pm[j]);
}

// Extent of the points: the smallest x, y, z then the largest, per workgroup.
__global__ void __launch_bounds__(256) k_extent(int n, Points P, double *out) {
  __shared__ double s[256];
  double v[6] = {1e30, 1e30, 1e30, -1e30, -1e30, -1e30};
  for(int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const size_t k = (size_t)i * P.stride;
    const double x[3] = {P.x[k], P.y[k], P.z[k]};
    for(int j = 0; j < 3; j++) {
      if(v[j] > x[j]) v[j] = x[j];
      if(v[3 + j] < x[j]) v[3 + j] = x[j];
    }
  }
  for(int j = 0; j < 6; j++) {
    s[threadIdx.x] = v[j];
    __syncthreads();
    for(int d = 128; d > 0; d >>= 1) {
      if((int)threadIdx.x < d) {
        const double a = s[threadIdx.x], b = s[threadIdx.x + d];
        s[threadIdx.x] = j < 3 ? (a > b ? b : a) : (a < b ? b : a);
      }
      __syncthreads();
    }
    if(threadIdx.x == 0) out[blockIdx.x * 6 + j] = s[0];
    __syncthreads();
  }
}

__device__ __forceinline__ int digit_at(unsigned long long key, int d) {  // child digit below depth d
  return (int)((key >> (3 * (kMaxDepth - 1 - d))) & 7ull);
}

// Split every node of depth d into its 8 child ranges (binary search on the sorted keys); ranges
// of >= 2 particles become nodes of depth d+1.  Eight threads per node, each with its own search.
// lev[k] counts the nodes of depth k: the nodes of a depth follow those of the depth above, so the
// levels are launched one after the other without the host reading their sizes.  A workgroup takes
// the ids of the nodes that its kSplitNodes nodes open with one atomic: atomics on one word bounded
// the split (1e7 sources, all levels: 7.3 ms with a thread and up to 8 atomics a node, 6.3 ms with
// an atomic a wave, 0.72 ms with an atomic a workgroup).  Ids in the order of the workgroups also
// keep the nodes that a walk opens together near each other (k_walk32g below: 32.2 -> 29.5 ms).
constexpr int kSplitNodes = 128;
__global__ void __launch_bounds__(8 * kSplitNodes) k_split(int d, int nsrc, int cap, const unsigned long long *key,
                                                           int *first, int *count, int *child, int4 *meta, int *lev) {
  __shared__ int wsum[8 * kSplitNodes / 64], base;
  int lo = 0;
  for(int k = 0; k < d; k++) lo += lev[k];
  const int n = min(lev[d], cap - lo), next = lo + lev[d], sub = threadIdx.x & 7, wave = threadIdx.x >> 6;
  for(int g0 = blockIdx.x * kSplitNodes; g0 < n; g0 += gridDim.x * kSplitNodes) {
    const int g = g0 + (threadIdx.x >> 3), nd = lo + min(g, n - 1);
    const int f = first[nd], c = g < n ? count[nd] : 0;
    const bool bucket = c >= 2 && d >= kMaxDepth;  // particles closer than the key resolution: a leaf bucket
    int l = f, r = bucket || sub == 0 ? f : f + c;  // first index in [l, r) with digit >= sub
    while(l < r) {
      const int mid = (l + r) >> 1;
      if(digit_at(key[mid], d) < sub)
        l = mid + 1;
      else
        r = mid;
    }
    int e = __shfl_down(l, 1, 8);
    if(sub == 7) e = f + c;
    const int cnt = bucket ? 0 : e - l;
    const unsigned long long opens = __ballot(cnt >= 2);
    if((threadIdx.x & 63) == 0) wsum[wave] = __popcll(opens);
    __syncthreads();
    if(threadIdx.x == 0) {
      int sum = 0;
      for(int w = 0; w < 8 * kSplitNodes / 64; w++) {
        const int v = wsum[w];
        wsum[w] = sum;
        sum += v;
      }
      base = sum > 0 ? next + atomicAdd(&lev[d + 1], sum) : 0;
    }
    __syncthreads();
    int ch = cnt == 1 ? l : -1;
    if(cnt >= 2) {
      const int id = base + wsum[wave] +
                     __builtin_amdgcn_mbcnt_hi((unsigned)(opens >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)opens, 0));
      if(id < cap) {  // (beyond: an overflow the host sees in lev)
        first[id] = l;
        count[id] = cnt;
        ch = nsrc + id;
      }
    }
    if(g < n) {
      if(sub == 0) meta[nd].w = bucket ? 1 : 0;
      child[(size_t)nd * 8 + sub] = ch;
    }
    __syncthreads();  // (wsum and base, before the next nodes)
  }
}

// Traceless quadrupole m (3 d_i d_j - d^2 delta_ij) of a point mass at offset d,
// added to q (xx, yy, zz, xy, xz, yz).
__device__ __forceinline__ void add_quad(double q[6], double m, double dx, double dy, double dz) {
  const double d2 = dx * dx + dy * dy + dz * dz;
  q[0] += m * (3 * dx * dx - d2);
  q[1] += m * (3 * dy * dy - d2);
  q[2] += m * (3 * dz * dz - d2);
  q[3] += m * 3 * dx * dy;
  q[4] += m * 3 * dx * dz;
  q[5] += m * 3 * dy * dz;
}

// Monopole moments of the nodes of one depth (forcetree.c:619-697), children in order 0..7.
// With quad (nnodes per component), also the traceless quadrupole about the
// centre of mass, from the children's own quadrupoles shifted to it.
// The node's side length (NODE.len, allvars.h:1095, held in float) goes beside them.
__global__ void k_moments(int lo, int hi, int nsrc, int nnodes, float len, const int *child, const int *first,
                          const int *count, const double4 *src, double4 *com, int4 *meta, double *quad) {
  int nd = lo + blockIdx.x * blockDim.x + threadIdx.x;
  if(nd >= hi) return;
  double ms = 0, s0 = 0, s1 = 0, s2 = 0;
  meta[nd].x = __float_as_int(len);
  const bool bucket = meta[nd].w;
  if(bucket) {
    for(int p = first[nd]; p < first[nd] + count[nd]; p++) {
      const double4 v = src[p];
      ms += v.w;
      s0 += v.w * v.x;
      s1 += v.w * v.y;
      s2 += v.w * v.z;
    }
  } else {
    const int *ch = child + (size_t)nd * 8;
    for(int k = 0; k < 8; k++) {
      int c = ch[k];
      if(c < 0) continue;
      const double4 v = c < nsrc ? src[c] : com[c - nsrc];
      ms += v.w;
      s0 += v.w * v.x;
      s1 += v.w * v.y;
      s2 += v.w * v.z;
    }
  }
  if(ms) {
    s0 /= ms;
    s1 /= ms;
    s2 /= ms;
  }
  com[nd] = make_double4(s0, s1, s2, ms);
  if(!quad) return;
  double q[6] = {0, 0, 0, 0, 0, 0};
  if(bucket) {
    for(int p = first[nd]; p < first[nd] + count[nd]; p++) {
      const double4 v = src[p];
      add_quad(q, v.w, v.x - s0, v.y - s1, v.z - s2);
    }
  } else {
    const int *ch = child + (size_t)nd * 8;
    for(int k = 0; k < 8; k++) {
      int c = ch[k];
      if(c < 0) continue;
      const double4 v = c < nsrc ? src[c] : com[c - nsrc];
      if(c >= nsrc)
        for(int j = 0; j < 6; j++) q[j] += quad[(size_t)j * nnodes + (c - nsrc)];
      add_quad(q, v.w, v.x - s0, v.y - s1, v.z - s2);
    }
  }
  for(int j = 0; j < 6; j++) quad[(size_t)j * nnodes + nd] = q[j];
}

// nextnode = first child; the sibling of a child is the next child, the last
// child inherits its parent's sibling (forcetree.c:624-638).
__global__ void k_thread(int lo, int hi, int nsrc, const int *child, int4 *meta, int *nextp) {
  int nd = lo + blockIdx.x * blockDim.x + threadIdx.x;
  if(nd >= hi) return;
  const int sib = nd == 0 ? -1 : meta[nd].y;
  if(nd == 0) meta[nd].y = -1;
  if(meta[nd].w) {
    meta[nd].z = sib;  // opened buckets are walked inline
    return;
  }
  const int *ch = child + (size_t)nd * 8;
  int list[8], n = 0;
  for(int k = 0; k < 8; k++)
    if(ch[k] >= 0) list[n++] = ch[k];
  meta[nd].z = n ? list[0] : sib;
  for(int k = 0; k < n; k++) {
    int nx = (k + 1 < n) ? list[k + 1] : sib;
    int c = list[k];
    if(c < nsrc)
      nextp[c] = nx;
    else
      meta[c - nsrc].y = nx;
  }
}

// FP32 copy of the quadrupoles, two 16-byte loads per node in the FP32 walk
__global__ void k_quadf(int nnodes, const double *quad, float4 *quadf) {
  int nd = blockIdx.x * blockDim.x + threadIdx.x;
  if(nd >= nnodes) return;
  const size_t nn = nnodes;
  quadf[2 * nd] = make_float4((float)quad[nd], (float)quad[nn + nd], (float)quad[2 * nn + nd], (float)quad[3 * nn + nd]);
  quadf[2 * nd + 1] = make_float4((float)quad[4 * nn + nd], (float)quad[5 * nn + nd], 0.f, 0.f);
}

struct WalkArgs {
  int nsrc, ntarget;
  Points X;             // the targets
  const int *order;     // per-target walks: the targets in walk order, or null
  const double4 *src;
  const int *nextp, *first, *count;
  const double4 *com;
  const int4 *meta;     // side length, sibling, nextnode, bucket (Tree)
  const double *quad;   // [6][nnodes] or null: monopole only
  const float4 *quadf;  // [nnodes][2] FP32 copy (FP32 walk)
  int nnodes;
  const int *child;     // [node][8] (the group walk)
  int blk_nb;           // targets are the (section, z, R) table nodes of nb x nb grids, a wave's an
                        // 8 x 8 block of one section; 0: 64 consecutive targets
  int tpw;              // per-target walks: targets of a wave, a power of two up to 64
  double theta, h, G;
  int plummer;          // Plummer softening of length eps instead of the spline of length h
  double eps;
  double *ax, *ay, *az, *pot;
  unsigned long long *nint;
};

// Gadget-2 cubic spline monopole (forcetree_walk.c:158-191)
__device__ __forceinline__ void interact64(double mass, double r2, double h, double &fac, double &wp) {
  double r = sqrt(r2);
  if(r >= h) {
    fac = mass / (r2 * r);
    wp = -mass / r;
  } else {
    double h_inv = 1.0 / h;
    double h3_inv = h_inv * h_inv * h_inv;
    double u = r * h_inv;
    if(u < 0.5) {
      fac = mass * h3_inv * (10.666666666667 + u * u * (32.0 * u - 38.4));
      wp = mass * h_inv * (-2.8 + u * u * (5.333333333333 + u * u * (6.4 * u - 9.6)));
    } else {
      fac = mass * h3_inv *
            (21.333333333333 - 48.0 * u + 38.4 * u * u - 10.666666666667 * u * u * u - 0.066666666667 / (u * u * u));
      wp = mass * h_inv *
           (-3.2 + 0.066666666667 / u + u * u * (10.666666666667 + u * (-16.0 + u * (9.6 - 2.133333333333 * u))));
    }
  }
}

__device__ __forceinline__ void interact32(float mass, float r2, float h, float &fac, float &wp) {
  float rinv = (r2 > 0.f) ? __builtin_amdgcn_rsqf(r2) : 0.f;
  float r = r2 * rinv;  // 0 for coincident points, which then take the u = 0 branch
  if(r >= h) {
    fac = mass * rinv * rinv * rinv;
    wp = -mass * rinv;
  } else {
    float h_inv = 1.0f / h;
    float h3_inv = h_inv * h_inv * h_inv;
    float u = r * h_inv;
    if(u < 0.5f) {
      fac = mass * h3_inv * (10.666666666667f + u * u * (32.0f * u - 38.4f));
      wp = mass * h_inv * (-2.8f + u * u * (5.333333333333f + u * u * (6.4f * u - 9.6f)));
    } else {
      float ui = 1.0f / u;
      fac = mass * h3_inv *
            (21.333333333333f - 48.0f * u + 38.4f * u * u - 10.666666666667f * u * u * u - 0.066666666667f * ui * ui * ui);
      wp = mass * h_inv *
           (-3.2f + 0.066666666667f * ui + u * u * (10.666666666667f + u * (-16.0f + u * (9.6f - 2.133333333333f * u))));
    }
  }
}

// Plummer-softened monopole: potential -m / sqrt(r^2 + eps^2)
__device__ __forceinline__ void plummer64(double mass, double r2, double eps, double &fac, double &wp) {
  const double s2 = r2 + eps * eps;
  const double sinv = 1.0 / sqrt(s2);
  fac = mass * sinv * sinv * sinv;
  wp = -mass * sinv;
}

__device__ __forceinline__ void plummer32(float mass, float r2, float eps, float &fac, float &wp) {
  const float sinv = __builtin_amdgcn_rsqf(r2 + eps * eps);
  fac = mass * sinv * sinv * sinv;
  wp = -mass * sinv;
}

// Quadrupole term of a node at offset d = (centre of mass - target), distance^2
// s2 (softened for Plummer): potential -(1/2) d.Q.d / s^5, acceleration
// -Q.d / s^5 + (5/2) (d.Q.d) d / s^7.
template <typename T>
__device__ __forceinline__ void quad_term(const T q[6], T dx, T dy, T dz, T s2, T sinv, T &ax, T &ay, T &az, T &pot) {
  const T qx = q[0] * dx + q[3] * dy + q[4] * dz;
  const T qy = q[3] * dx + q[1] * dy + q[5] * dz;
  const T qz = q[4] * dx + q[5] * dy + q[2] * dz;
  const T dqd = dx * qx + dy * qy + dz * qz;
  const T s5 = sinv * sinv * sinv * sinv * sinv;
  const T c = (T)2.5 * dqd * s5 / s2;
  ax += -qx * s5 + c * dx;
  ay += -qy * s5 + c * dy;
  az += -qz * s5 + c * dz;
  pot += (T)-0.5 * dqd * s5;
}

// The target of a lane: an 8 x 8 block of a section's table nodes per wave, or 64 targets in turn.
__device__ __forceinline__ long long wave_target(const WalkArgs &A, int g, int lane) {
  if(A.blk_nb > 0) {
    const int nbb = A.blk_nb / 8, s = g / (nbb * nbb), b = g % (nbb * nbb);
    return ((long long)s * A.blk_nb + (b / nbb) * 8 + lane / 8) * A.blk_nb + (b % nbb) * 8 + lane % 8;
  }
  return (long long)g * 64 + lane;
}

// Adds the interaction with a point of mass `mass` at offset (dx, dy, dz).
__device__ __forceinline__ void interact(const WalkArgs &A, double mass, double dx, double dy, double dz, double r2,
                                         double &ax, double &ay, double &az, double &pot) {
  double fac, wp;
  if(A.plummer)
    plummer64(mass, r2, A.eps, fac, wp);
  else
    interact64(mass, r2, A.h, fac, wp);
  ax += dx * fac;
  ay += dy * fac;
  az += dz * fac;
  pot += wp;
}
__device__ __forceinline__ void interact(const WalkArgs &A, float mass, float dx, float dy, float dz, float r2,
                                         float &ax, float &ay, float &az, float &pot) {
  float fac, wp;
  if(A.plummer)
    plummer32(mass, r2, (float)A.eps, fac, wp);
  else
    interact32(mass, r2, (float)A.h, fac, wp);
  ax += dx * fac;
  ay += dy * fac;
  az += dz * fac;
  pot += wp;
}

// forcetree_walk.c:58-192 (mode 0, one task), one target per lane, the 64 targets of a wave on one
// path.  The wave walks the nodes any of its targets opens; a lane whose target accepts a node
// waits until the walk reaches that node's sibling.  Every target interacts with the nodes and
// particles of its own walk in its own order, but the entry being walked is the same for the whole
// wave, so its moments and links are scalar loads: with each lane on its own path they were
// gathers of 64 lines, one after the other.  Neighbouring targets share most of their paths (the
// targets come in 8 x 8 blocks of a table section or in Morton order).  2e5 sources, 8 x 128^2
// targets, FP64: 11.7 -> 5.3 ms.
// A wave's time is the length of its path, and targets far from each other share little of it: where
// the launch leaves the chip idle, waves take fewer targets (kWalkWaves below), down to one.
// T = float: separations formed in FP64 (node centres of mass and particles stay FP64) and rounded
// once, the kernel and the sums in FP32 per target.
template <typename T>
__device__ __forceinline__ void walk_body(const WalkArgs &A) {
  const int lane = threadIdx.x & 63;
  const long long i = (long long)blockIdx.x * A.tpw + lane;
  long long t = wave_target(A, (int)(i >> 6), (int)(i & 63));
  const bool live = lane < A.tpw && t < A.ntarget;
  if(live && A.order) t = A.order[t];
  const size_t tk = live ? (size_t)t * A.X.stride : 0;
  const double px = live ? A.X.x[tk] : 0, py = live ? A.X.y[tk] : 0, pz = live ? A.X.z[tk] : 0;
  T ax = 0, ay = 0, az = 0, pot = 0;
  const T h = (T)A.h, eps = (T)A.eps, th2 = (T)(A.theta * A.theta);
  unsigned int nint = 0;
  constexpr int kGo = -2, kDead = -3;
  int resume = live ? kGo : kDead;  // kGo: the lane walks; an entry: it waits for it
  int no = A.nsrc;                  // root
  while(no >= 0) {
    no = __builtin_amdgcn_readfirstlane(no);
    if(resume == no) resume = kGo;
    const bool act = resume == kGo;
    if(no < A.nsrc) {
      const double4 s = A.src[no];
      const T dx = (T)(s.x - px), dy = (T)(s.y - py), dz = (T)(s.z - pz), mass = (T)s.w;
      if(act && mass != 0) {
        interact(A, mass, dx, dy, dz, dx * dx + dy * dy + dz * dz, ax, ay, az, pot);
        nint++;
      }
      no = A.nextp[no];
      continue;
    }
    const int q = no - A.nsrc;
    const double4 s = A.com[q];
    const int4 m = A.meta[q];
    const T dx = (T)(s.x - px), dy = (T)(s.y - py), dz = (T)(s.z - pz), mass = (T)s.w;
    const T r2 = dx * dx + dy * dy + dz * dz;
    const float l = __int_as_float(m.x), l2 = l * l;
    const bool wide = sizeof(T) == 8 ? l2 > r2 * A.theta * A.theta : l2 > r2 * th2;
    const bool open = act && wide;
    if(act && !wide) {
      if(A.quad && mass != 0) {
        T qq[6];
        if(sizeof(T) == 8) {
          const size_t nn = A.nnodes;
          for(int k = 0; k < 6; k++) qq[k] = A.quad[k * nn + q];
        } else {
          const float4 qa = A.quadf[2 * q], qb = A.quadf[2 * q + 1];
          qq[0] = qa.x;
          qq[1] = qa.y;
          qq[2] = qa.z;
          qq[3] = qa.w;
          qq[4] = qb.x;
          qq[5] = qb.y;
        }
        const T s2 = A.plummer ? r2 + eps * eps : r2;
        if(A.plummer || s2 >= h * h) {
          const T sinv = sizeof(T) == 8 ? (T)(1.0 / sqrt((double)s2)) : (T)__builtin_amdgcn_rsqf((float)s2);
          quad_term(qq, dx, dy, dz, s2, sinv, ax, ay, az, pot);
        }
      }
      if(mass != 0) {
        interact(A, mass, dx, dy, dz, r2, ax, ay, az, pot);
        nint++;
      }
    }
    if(__ballot(open) == 0) {
      no = m.y;
    } else if(m.w) {
      // a leaf bucket, its particles one by one
      const int p0 = A.first[q], p1 = p0 + A.count[q];
      for(int p = p0; p < p1; p++) {
        const double4 v = A.src[p];
        const T ex = (T)(v.x - px), ey = (T)(v.y - py), ez = (T)(v.z - pz);
        if(open && v.w != 0) {
          interact(A, (T)v.w, ex, ey, ez, ex * ex + ey * ey + ez * ez, ax, ay, az, pot);
          nint++;
        }
      }
      no = m.y;
    } else {
      if(act && !wide) resume = m.y;
      no = m.z;
    }
  }
  if(live) {
    A.ax[t] = (double)ax * A.G;
    A.ay[t] = (double)ay * A.G;
    A.az[t] = (double)az * A.G;
    A.pot[t] = (double)pot * A.G;
  }
  unsigned long long n = nint;
  for(int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o, 64);
  if(lane == 0) atomicAdd(A.nint, n);
}
__global__ void __launch_bounds__(64) k_walk64(WalkArgs A) { walk_body<double>(A); }
__global__ void __launch_bounds__(64) k_walk32(WalkArgs A) { walk_body<float>(A); }

// Table projection of grid.c:719-750: radial and vertical components summed
// over the FG_SECTIONS azimuthal sections in order, then averaged.
__global__ void k_project(int nb, const double *ax, const double *ay, const double *az, const double *pt,
                          const double *cs, const double *sn, double *dpotdr, double *dpotdz, double *pot) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i >= nb * nb) return;
  double r = 0, zz = 0, p = 0;
  for(int s = 0; s < GALIC_FG_SECTIONS; s++) {
    size_t n = (size_t)s * nb * nb + i;
    r += ax[n] * cs[s] + ay[n] * sn[s];
    zz += az[n];
    p += pt[n];
  }
  dpotdr[i] = r / GALIC_FG_SECTIONS;
  dpotdz[i] = zz / GALIC_FG_SECTIONS;
  pot[i] = p / GALIC_FG_SECTIONS;
}

// Table-fill targets (grid.c:680-704): node (s, k, j) at (R_j cos phi_s, R_j sin phi_s, z_k)
// with R_j = z_j = rj[j], the same products as the host-built targets.
__global__ void k_fill_targets(int nb, const double *rj, const double *cs, const double *sn, double *tx, double *ty,
                               double *tz) {
  const size_t n = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if(n >= (size_t)GALIC_FG_SECTIONS * nb * nb) return;
  const int s = (int)(n / ((size_t)nb * nb)), k = (int)((n / nb) % nb), j = (int)(n % nb);
  tx[n] = rj[j] * cs[s];
  ty[n] = rj[j] * sn[s];
  tz[n] = rj[k];
}

// The FP32 orbit kernels' force table (DPotDR, DPotDz) from the FP64 tables.
__global__ void k_acc_f(int n, const double *dr, const double *dz, float2 *out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if(i < n) out[i] = make_float2((float)dr[i], (float)dz[i]);
}

// Direct summation in FP64 with the walk's interaction (the check of the
// tree's force error): one target per lane, sources staged through LDS.
__global__ void __launch_bounds__(256) k_direct64(int nsrc, const double *sx, const double *sy, const double *sz,
                                                   const double *sm, int ntarget, const double *tx, const double *ty,
                                                   const double *tz, double h, int plummer, double eps, double G,
                                                   double *ax, double *ay, double *az, double *pot) {
  __shared__ double4 tile[256];
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = t < ntarget;
  const double px = live ? tx[t] : 0, py = live ? ty[t] : 0, pz = live ? tz[t] : 0;
  double acc_x = 0, acc_y = 0, acc_z = 0, potv = 0, fac, wp;
  for(int base = 0; base < nsrc; base += 256) {
    const int q = base + threadIdx.x;
    tile[threadIdx.x] = (q < nsrc) ? make_double4(sx[q], sy[q], sz[q], sm[q]) : make_double4(0, 0, 0, 0);
    __syncthreads();
    const int nt = min(256, nsrc - base);
    for(int k = 0; k < nt; k++) {
      const double4 s = tile[k];
      if(s.w != 0) {
        const double dx = s.x - px, dy = s.y - py, dz = s.z - pz;
        if(plummer)
          plummer64(s.w, dx * dx + dy * dy + dz * dz, eps, fac, wp);
        else
          interact64(s.w, dx * dx + dy * dy + dz * dz, h, fac, wp);
        acc_x += dx * fac;
        acc_y += dy * fac;
        acc_z += dz * fac;
        potv += wp;
      }
    }
    __syncthreads();
  }
  if(live) {
    ax[t] = acc_x * G;
    ay[t] = acc_y * G;
    az[t] = acc_z * G;
    pot[t] = potv * G;
  }
}

}  // namespace tree
}  // namespace galic

namespace {

using namespace galic::tree;

int terr(int code, const char *fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  return galic::set_error(code, buf);
}

// (An error that is reported is also dropped from the runtime's record, as in galic_api.hip.)
#define TCHK(expr)                                                                                 \
  do {                                                                                             \
    hipError_t e_ = (expr);                                                                        \
    if(e_ != hipSuccess) {                                                                         \
      (void)hipGetLastError();                                                                     \
      rc = terr(e_ == hipErrorOutOfMemory ? GALIC_ERR_NOMEM : GALIC_ERR_HIP, "%s: %s", #expr,      \
                hipGetErrorString(e_));                                                            \
      goto done;                                                                                   \
    }                                                                                              \
  } while(0)

inline int nb256(size_t n) { return (int)((n + 255) / 256); }

// Device times of the last tree call of this process (ms): build (sort, split,
// moments, threading), walk, and the interaction count.
double g_last_build_ms = 0, g_last_walk_ms = 0, g_last_interactions = 0;

// Device buffers of one call.
struct HipMem {
  typedef hipError_t Error;
  static Error get(void **p, size_t n) { return hipMalloc(p, n); }
  static void put(void *p) { (void)hipFree(p); }
  static Error good() { return hipSuccess; }
  static bool is_short(Error e) { return e == hipErrorOutOfMemory; }
  static void forget() { (void)hipGetLastError(); }
};
typedef galic::DevPool<HipMem> DevBufs;

// Moments bottom-up (monopole, and the quadrupole where T.quad is allocated), node side
// lengths DomainLen / 2^depth (NODE.len, allvars.h:1095, held in float), then the
// nextnode/sibling threading top-down (forcetree.c:591-722).
int tree_moments_dev(hipStream_t st, Tree &T, double dlen) {
  const int nnodes = T.level_lo.back(), nsrc = T.nsrc;
  const int ndepth = (int)T.level_lo.size() - 1;
  for(int d = ndepth - 1; d >= 0; d--) {
    int lo = T.level_lo[d], hi = T.level_lo[d + 1];
    if(hi <= lo) continue;
    hipLaunchKernelGGL(k_moments, dim3(nb256(hi - lo)), dim3(256), 0, st, lo, hi, nsrc, nnodes, (float)ldexp(dlen, -d),
                       (const int *)T.child, (const int *)T.first, (const int *)T.count, (const double4 *)T.src, T.com,
                       T.meta, T.quad);
    if(hipGetLastError() != hipSuccess) return terr(GALIC_ERR_HIP, "tree moments launch failed");
  }
  for(int d = 0; d < ndepth; d++) {
    int lo = T.level_lo[d], hi = T.level_lo[d + 1];
    if(hi <= lo) continue;
    hipLaunchKernelGGL(k_thread, dim3(nb256(hi - lo)), dim3(256), 0, st, lo, hi, nsrc, (const int *)T.child, T.meta,
                       T.nextp);
    if(hipGetLastError() != hipSuccess) return terr(GALIC_ERR_HIP, "tree threading launch failed");
  }
  if(T.quad && T.quadf) {
    hipLaunchKernelGGL(k_quadf, dim3(nb256(nnodes)), dim3(256), 0, st, nnodes, (const double *)T.quad, T.quadf);
    if(hipGetLastError() != hipSuccess) return terr(GALIC_ERR_HIP, "tree quadrupole copy failed");
  }
  return GALIC_OK;
}

// Builds the tree of nsrc sources (device SoA inputs, domain cube at corner with side dlen)
// into T, its buffers owned by B.  sorted (optional) receives the device array giving, for each
// sorted source, its index among the inputs.
int tree_build_dev(const galic_params *p, hipStream_t st, int nsrc, Points S, const double *dpm,
                   const double corner[3], double dlen, int precision,
                   DevBufs &B, Tree &T, int **sorted, float *build_ms) {
  int rc = GALIC_OK;
  unsigned long long *keys_in = nullptr;
  int *idx_in = nullptr, *idx = nullptr;
  void *tmp = nullptr;
  size_t tmp_bytes = 0;
  hipEvent_t eb = nullptr, ee = nullptr;
  (void)p;
  T.nsrc = nsrc;
  for(int j = 0; j < 3; j++) T.corner[j] = corner[j];
  T.dlen = dlen;
  TCHK(hipEventCreate(&eb));
  TCHK(hipEventCreate(&ee));
  TCHK(hipEventRecord(eb, st));
  TCHK(B.alloc(&keys_in, nsrc));
  TCHK(B.alloc(&T.key, nsrc));
  TCHK(B.alloc(&idx_in, nsrc));
  TCHK(B.alloc(&idx, nsrc));
  TCHK(B.alloc(&T.src, nsrc));
  TCHK(B.alloc(&T.nextp, nsrc));
  if(nsrc > 0) {
    hipLaunchKernelGGL(k_keys, dim3(nb256(nsrc)), dim3(256), 0, st, nsrc, S, corner[0], corner[1], corner[2],
                       1.0 / dlen, keys_in, idx_in);
    TCHK(hipGetLastError());
    TCHK(rocprim::radix_sort_pairs(nullptr, tmp_bytes, keys_in, T.key, idx_in, idx, (unsigned int)nsrc, 0, 63, st));
    TCHK(B.alloc((char **)&tmp, tmp_bytes));
    TCHK(rocprim::radix_sort_pairs(tmp, tmp_bytes, keys_in, T.key, idx_in, idx, (unsigned int)nsrc, 0, 63, st));
    hipLaunchKernelGGL(k_gather, dim3(nb256(nsrc)), dim3(256), 0, st, nsrc, (const int *)idx, S, dpm, T.src);
    TCHK(hipGetLastError());
  }
  if(sorted) *sorted = idx;
  {
    // nodes: the unique insertion tree has fewer than 2 nsrc nodes unless
    // particles pair up at great depth; grow and rebuild if needed
    // (the reference raises TreeAllocFactor and retries, forcetree.c:48-70)
    T.cap = 2 * nsrc + 64;
    for(int attempt = 0; attempt < 6; attempt++) {
      TCHK(B.alloc(&T.first, T.cap));
      TCHK(B.alloc(&T.count, T.cap));
      TCHK(B.alloc(&T.child, (size_t)T.cap * 8));
      TCHK(B.alloc(&T.meta, T.cap));
      TCHK(B.alloc(&T.counter, kMaxDepth + 2));
      const int root[2] = {0, nsrc};
      int lev[kMaxDepth + 2] = {1};
      TCHK(hipMemcpyAsync(T.first, &root[0], sizeof(int), hipMemcpyHostToDevice, st));
      TCHK(hipMemcpyAsync(T.count, &root[1], sizeof(int), hipMemcpyHostToDevice, st));
      TCHK(hipMemcpyAsync(T.counter, lev, sizeof(lev), hipMemcpyHostToDevice, st));
      for(int d = 0; d <= kMaxDepth; d++) {
        // at most 8^d nodes, of two particles at least (the root: of any number)
        const long long most = d < 8 ? std::min(1ll << (3 * d), (long long)nsrc / 2 + 1) : (long long)nsrc / 2 + 1;
        hipLaunchKernelGGL(k_split, dim3((unsigned int)std::min((most + kSplitNodes - 1) / kSplitNodes, 2048ll)),
                           dim3(8 * kSplitNodes), 0, st, d, nsrc, T.cap, (const unsigned long long *)T.key, T.first,
                           T.count, T.child, T.meta, T.counter);
        TCHK(hipGetLastError());
      }
      TCHK(hipMemcpyAsync(lev, T.counter, sizeof(lev), hipMemcpyDeviceToHost, st));
      TCHK(hipStreamSynchronize(st));
      T.level_lo.assign(1, 0);
      for(int d = 0; d <= kMaxDepth && lev[d] > 0; d++) T.level_lo.push_back(T.level_lo.back() + lev[d]);
      const bool overflow = T.level_lo.back() > T.cap;
      if(!overflow) break;
      T.cap *= 2;
      if(attempt == 5) {
        rc = terr(GALIC_ERR_NOMEM, "tree node pool overflow");
        goto done;
      }
    }
  }
  {
    const int nnodes = T.level_lo.back();
    TCHK(B.alloc(&T.com, nnodes));
    if(precision & GALIC_TREE_QUADRUPOLE) {
      TCHK(B.alloc(&T.quad, (size_t)6 * nnodes));
      if(precision & GALIC_TREE_FP32) TCHK(B.alloc(&T.quadf, (size_t)2 * nnodes));
    }
    if((rc = tree_moments_dev(st, T, dlen)) != GALIC_OK) goto done;
  }
  TCHK(hipEventRecord(ee, st));
  TCHK(hipEventSynchronize(ee));
  if(build_ms) TCHK(hipEventElapsedTime(build_ms, eb, ee));
done:
  if(eb) (void)hipEventDestroy(eb);
  if(ee) (void)hipEventDestroy(ee);
  return rc;
}

// The group walk (GALIC_TREE_GROUP, FP32 interactions): the 64 targets of a wave walk the tree
// together.  A node is accepted for the group only if the opening criterion holds at the point
// of the targets' bounding box nearest to its centre of mass, so every target interacts with
// nodes that its own criterion would accept, or with their descendants: more interactions than
// the per-target walk (forcetree_walk.c:12-222), none less accurate.  The wave takes up to 64
// pending entries of an LDS stack at a time (one per lane): accepted nodes, particles and
// opened leaf buckets go to an LDS interaction list, opened nodes push their children.  A full
// list is flushed: every lane adds the list's entries (read at wave-uniform addresses) to its
// own target.  With less stack room than 64 entries could need, one entry is taken at a time
// (a depth-first descent needs at most 7 entries per level).
constexpr int kGStack = 1024, kGList = 1024, kGDeep = 7 * (kMaxDepth + 3);

// One list entry's data: a node (q >= 0) with its moments, or a particle.
struct GroupEntry {
  int q;
  double4 s;
  float4 qa, qb;
};

// e uniform over the wave, not a bucket: scalar loads.
__device__ __forceinline__ GroupEntry group_load(const WalkArgs &A, int e) {
  GroupEntry g;
  g.q = e - A.nsrc;
  const double4 *s = g.q >= 0 ? A.com + g.q : A.src + e;
  g.s = *s;
  if(A.quadf) {
    const float4 *m = A.quadf + 2 * (size_t)max(g.q, 0);
    g.qa = m[0];
    g.qb = m[1];
  }
  return g;
}

__device__ __forceinline__ void group_add(const WalkArgs &A, const GroupEntry &g, double px, double py, double pz,
                                          float h, float eps, float &ax, float &ay, float &az, float &pot,
                                          unsigned int &nint) {
  float fac, wp;
  const float mass = (float)g.s.w;
  if(mass == 0) return;
  const float dx = (float)(g.s.x - px), dy = (float)(g.s.y - py), dz = (float)(g.s.z - pz);
  const float r2 = dx * dx + dy * dy + dz * dz;
  if(g.q >= 0 && A.quadf) {
    const float qq[6] = {g.qa.x, g.qa.y, g.qa.z, g.qa.w, g.qb.x, g.qb.y};
    const float s2 = A.plummer ? r2 + eps * eps : r2;
    if(A.plummer || s2 >= h * h) quad_term(qq, dx, dy, dz, s2, __builtin_amdgcn_rsqf(s2), ax, ay, az, pot);
  }
  if(A.plummer)
    plummer32(mass, r2, eps, fac, wp);
  else
    interact32(mass, r2, h, fac, wp);
  ax += dx * fac;
  ay += dy * fac;
  az += dz * fac;
  pot += wp;
  nint++;
}

// An opened leaf bucket: its particles one by one.
__device__ __forceinline__ void group_bucket(const WalkArgs &A, int q, double px, double py, double pz, float h,
                                             float eps, float &ax, float &ay, float &az, float &pot,
                                             unsigned int &nint) {
  const int p0 = A.first[q], p1 = p0 + A.count[q];
  for(int p = p0; p < p1; p++) {
    const GroupEntry g{-1, A.src[p], {}, {}};
    if(g.s.w != 0) group_add(A, g, px, py, pz, h, eps, ax, ay, az, pot, nint);
  }
}

// Adds the list's entries in their order to the lane's target, kGBatch at a time: the batch's
// loads go out together, so their latency (an LDS read, then a scalar load that depends on it) is
// paid once a batch instead of once an entry: that latency bounded the walk (512^2 x 8 targets and
// 1e7 sources, 9.1e9 interactions: 40.7 ms one entry at a time, 32.2 ms four at a time).  A batch
// with a bucket in it, and the list's end, go one by one.
constexpr int kGBatch = 4;
__device__ __forceinline__ void group_flush(const WalkArgs &A, const int *lst, int nl, double px, double py, double pz,
                                            float h, float eps, float &ax, float &ay, float &az, float &pot,
                                            unsigned int &nint) {
  for(int i = 0; i < nl; i += kGBatch) {
    const int4 e4 = *(const int4 *)(lst + i);  // (entries beyond nl are not used)
    const int e[kGBatch] = {__builtin_amdgcn_readfirstlane(e4.x), __builtin_amdgcn_readfirstlane(e4.y),
                            __builtin_amdgcn_readfirstlane(e4.z), __builtin_amdgcn_readfirstlane(e4.w)};
    if(i + kGBatch <= nl && (e[0] | e[1] | e[2] | e[3]) >= 0) {
      GroupEntry g[kGBatch];
#pragma unroll
      for(int k = 0; k < kGBatch; k++) g[k] = group_load(A, e[k]);
#pragma unroll
      for(int k = 0; k < kGBatch; k++) group_add(A, g[k], px, py, pz, h, eps, ax, ay, az, pot, nint);
    } else {
      for(int k = 0; k < kGBatch && i + k < nl; k++) {
        const int ek = __builtin_amdgcn_readfirstlane(lst[i + k]);
        if(ek >= 0)
          group_add(A, group_load(A, ek), px, py, pz, h, eps, ax, ay, az, pot, nint);
        else
          group_bucket(A, ~ek, px, py, pz, h, eps, ax, ay, az, pot, nint);
      }
    }
  }
}

__device__ __forceinline__ double wave_min(double v) {
  for(int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o, 64));
  return v;
}
__device__ __forceinline__ double wave_max(double v) {
  for(int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  return v;
}

__global__ void __launch_bounds__(64) k_walk32g(WalkArgs A) {
  __shared__ int stk[kGStack];
  __shared__ __align__(16) int lst[kGList];
  const int lane = threadIdx.x, g = blockIdx.x;
  const long long t = wave_target(A, g, lane);
  const bool live = t < A.ntarget;
  const long long tl = live ? t : (long long)g * 64;  // (dead lanes: the group's first target)
  const size_t tk = (size_t)tl * A.X.stride;
  const double px = A.X.x[tk], py = A.X.y[tk], pz = A.X.z[tk];
  const double bx0 = wave_min(px), by0 = wave_min(py), bz0 = wave_min(pz);
  const double bx1 = wave_max(px), by1 = wave_max(py), bz1 = wave_max(pz);
  const float h = (float)A.h, th2 = (float)(A.theta * A.theta), eps = (float)A.eps;
  float ax = 0, ay = 0, az = 0, pot = 0;
  unsigned int nint = 0;
  if(lane == 0) stk[0] = A.nsrc;  // the root node
  int top = A.nnodes > 0 ? 1 : 0, nl = 0;
  __syncthreads();
  while(top > 0) {
    const int k = (kGStack - top >= 7 * 64 + kGDeep) ? min(64, top) : 1;
    if(nl + k > kGList) {
      group_flush(A, lst, nl, px, py, pz, h, eps, ax, ay, az, pot, nint);
      nl = 0;
    }
    const int e = lane < k ? stk[top - 1 - lane] : -1;
    top -= k;
    __syncthreads();
    int item = 0, open = -1;  // item: the list entry (0: none)
    bool listed = false;
    if(lane < k) {
      if(e < A.nsrc) {
        listed = true;
        item = e;
      } else {
        const int q = e - A.nsrc;
        const double4 cm = A.com[q];
        const int4 mt = A.meta[q];
        const double cx = cm.x, cy = cm.y, cz = cm.z;
        const float dx = (float)fmax(fmax(bx0 - cx, cx - bx1), 0.0);
        const float dy = (float)fmax(fmax(by0 - cy, cy - by1), 0.0);
        const float dz = (float)fmax(fmax(bz0 - cz, cz - bz1), 0.0);
        const float l = __int_as_float(mt.x);
        if(l * l > (dx * dx + dy * dy + dz * dz) * th2) {
          if(mt.w) {
            listed = true;
            item = ~q;
          } else {
            open = q;
          }
        } else {
          listed = true;
          item = e;
        }
      }
    }
    const unsigned long long lm = __ballot(listed);
    if(listed) lst[nl + __builtin_amdgcn_mbcnt_hi((unsigned)(lm >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)lm, 0))] = item;
    nl += __popcll(lm);
    for(int c = 0; c < 8; c++) {
      const int ch = open >= 0 ? A.child[(size_t)open * 8 + c] : -1;
      const unsigned long long cm = __ballot(ch >= 0);
      if(ch >= 0) stk[top + __builtin_amdgcn_mbcnt_hi((unsigned)(cm >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)cm, 0))] = ch;
      top += __popcll(cm);
    }
    __syncthreads();
  }
  group_flush(A, lst, nl, px, py, pz, h, eps, ax, ay, az, pot, nint);
  if(live) {
    A.ax[t] = (double)ax * A.G;
    A.ay[t] = (double)ay * A.G;
    A.az[t] = (double)az * A.G;
    A.pot[t] = (double)pot * A.G;
    atomicAdd(A.nint, (unsigned long long)nint);
  }
}

// Waves of a per-target walk below which a wave takes fewer than 64 targets: one a SIMD.  Scattered
// targets, 2e5 sources, FP64, the walk: 64 targets in one wave 23.8 ms, one a wave 2.7 (a lane each on
// its own path: 6.3); 16000 in 250 waves 5.9, 1000 waves 4.0, 2000 4.8, 4000 6.7; 65000 in 1016
// waves 5.1, 2032 4.8, 4064 5.6.
constexpr int kWalkWaves = 1024;

// Walk of ntarget targets (device SoA) through T; the results are scaled by G (gravity_tree
// multiplies the walk's sums by G afterwards, gravtree.c:455-463).
// blk_nb > 0: the targets are table nodes (section, z, R) of blk_nb x blk_nb grids, which a wave
// takes in 8 x 8 blocks.
int tree_walk_dev(const galic_params *p, hipStream_t st, DevBufs &B, const Tree &T, int ntarget, Points X, double *dax,
                  double *day, double *daz, double *dpot, int precision, double G, long long *ninteractions,
                  float *walk_ms, int blk_nb = 0) {
  int rc = GALIC_OK;
  unsigned long long *nint = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  WalkArgs W;
  TCHK(B.alloc(&nint, 1));
  TCHK(hipMemsetAsync(nint, 0, sizeof(unsigned long long), st));
  W.nsrc = T.nsrc;
  W.ntarget = ntarget;
  W.X = X;
  W.order = nullptr;
  W.src = T.src;
  W.nextp = T.nextp;
  W.first = T.first;
  W.count = T.count;
  W.com = T.com;
  W.meta = T.meta;
  W.child = T.child;
  W.blk_nb = 0;
  W.quad = (precision & GALIC_TREE_QUADRUPOLE) ? T.quad : nullptr;
  W.quadf = (W.quad && (precision & GALIC_TREE_FP32)) ? T.quadf : nullptr;
  if(W.quad && (precision & GALIC_TREE_FP32) && !W.quadf) {
    rc = terr(GALIC_ERR_STATE, "the tree was built without the FP32 quadrupole copy");
    goto done;
  }
  if((precision & GALIC_TREE_QUADRUPOLE) && !T.quad) {
    rc = terr(GALIC_ERR_STATE, "the tree was built without quadrupole moments");
    goto done;
  }
  W.nnodes = T.level_lo.back();
  W.theta = p->ErrTolTheta;
  W.h = p->ForceSoftening;
  // ForceSoftening is 2.8 times the Softening parameter (init.c:78-84), the Plummer length
  W.plummer = (precision & GALIC_TREE_PLUMMER) ? 1 : 0;
  W.eps = p->ForceSoftening / 2.8;
  W.G = G;
  W.ax = dax;
  W.ay = day;
  W.az = daz;
  W.pot = dpot;
  W.nint = nint;
  TCHK(hipEventCreate(&e0));
  TCHK(hipEventCreate(&e1));
  TCHK(hipEventRecord(e0, st));
  if(ntarget > 0) {
    // table nodes in 8 x 8 blocks; other targets as they come in the group walk, whose groups are
    // the caller's, and in Morton order where each target walks for itself
    const bool blk = blk_nb > 0 && blk_nb % 8 == 0 && (long long)ntarget % ((long long)blk_nb * blk_nb) == 0;
    W.blk_nb = blk ? blk_nb : 0;
    W.tpw = 64;
    if(!(precision & GALIC_TREE_GROUP))
      while(W.tpw > 1 && ntarget / W.tpw < kWalkWaves) W.tpw /= 2;
    const dim3 grid((unsigned int)(((long long)ntarget + W.tpw - 1) / W.tpw)), block(64);
    if(precision & GALIC_TREE_GROUP) {
      hipLaunchKernelGGL(k_walk32g, grid, block, 0, st, W);
    } else {
      if(!blk && W.tpw > 1) {
        unsigned long long *k0 = nullptr, *k1 = nullptr;
        int *i0 = nullptr, *i1 = nullptr;
        char *tmp = nullptr;
        size_t tmp_bytes = 0;
        TCHK(B.alloc(&k0, ntarget));
        TCHK(B.alloc(&k1, ntarget));
        TCHK(B.alloc(&i0, ntarget));
        TCHK(B.alloc(&i1, ntarget));
        hipLaunchKernelGGL(k_keys, dim3(nb256(ntarget)), dim3(256), 0, st, ntarget, X, T.corner[0], T.corner[1],
                           T.corner[2], 1.0 / T.dlen, k0, i0);
        TCHK(hipGetLastError());
        TCHK(rocprim::radix_sort_pairs(nullptr, tmp_bytes, k0, k1, i0, i1, (unsigned int)ntarget, 0, 63, st));
        TCHK(B.alloc(&tmp, tmp_bytes));
        TCHK(rocprim::radix_sort_pairs(tmp, tmp_bytes, k0, k1, i0, i1, (unsigned int)ntarget, 0, 63, st));
        W.order = i1;
      }
      if(!(precision & GALIC_TREE_FP32))
        hipLaunchKernelGGL(k_walk64, grid, block, 0, st, W);
      else
        hipLaunchKernelGGL(k_walk32, grid, block, 0, st, W);
    }
    TCHK(hipGetLastError());
  }
  TCHK(hipEventRecord(e1, st));
  TCHK(hipEventSynchronize(e1));
  if(walk_ms) TCHK(hipEventElapsedTime(walk_ms, e0, e1));
  {
    unsigned long long ni = 0;
    TCHK(hipMemcpy(&ni, nint, sizeof(ni), hipMemcpyDeviceToHost));
    if(ninteractions) *ninteractions = (long long)ni;
  }
done:
  if(e0) (void)hipEventDestroy(e0);
  if(e1) (void)hipEventDestroy(e1);
  return rc;
}

// Build the tree of nsrc sources (device inputs) and walk ntarget targets.
int tree_forces_dev(const galic_params *p, hipStream_t st, DevBufs &B, int nsrc, Points S, const double *dpm,
                    int ntarget, Points X, double corner[3], double dlen, double *dax, double *day, double *daz,
                    double *dpot, int precision, long long *ninteractions, float *walk_ms, int blk_nb = 0) {
  Tree T;
  float build_ms = 0, wms = 0;
  long long ni = 0;
  int rc = tree_build_dev(p, st, nsrc, S, dpm, corner, dlen, precision, B, T, nullptr, &build_ms);
  if(rc != GALIC_OK) return rc;
  rc = tree_walk_dev(p, st, B, T, ntarget, X, dax, day, daz, dpot, precision, p->G, &ni, &wms, blk_nb);
  if(rc != GALIC_OK) return rc;
  if(ninteractions) *ninteractions = ni;
  if(walk_ms) *walk_ms = wms;
  g_last_build_ms = build_ms;
  g_last_walk_ms = wms;
  g_last_interactions = (double)ni;
  return GALIC_OK;
}

// The extent of points on the device, widened into lo and hi (domain_box.c:20-65).
int extend_domain(hipStream_t st, DevBufs &B, int n, Points P, double lo[3], double hi[3]) {
  if(n <= 0) return GALIC_OK;
  int rc = GALIC_OK;
  const int nblk = std::min(nb256(n), 512);
  double *d = nullptr;
  std::vector<double> h((size_t)nblk * 6);
  TCHK(B.alloc(&d, h.size()));
  hipLaunchKernelGGL(k_extent, dim3(nblk), dim3(256), 0, st, n, P, d);
  TCHK(hipGetLastError());
  TCHK(hipMemcpyAsync(h.data(), d, sizeof(double) * h.size(), hipMemcpyDeviceToHost, st));
  TCHK(hipStreamSynchronize(st));
  for(int b = 0; b < nblk; b++)
    for(int j = 0; j < 3; j++) {
      if(lo[j] > h[6 * b + j]) lo[j] = h[6 * b + j];
      if(hi[j] < h[6 * b + 3 + j]) hi[j] = h[6 * b + 3 + j];
    }
done:
  return rc;
}

// The cube over an extent (domain_box.c:20-65).
void domain_cube(const double lo[3], const double hi[3], double corner[3], double *len) {
  double l = 0;
  for(int j = 0; j < 3; j++)
    if(hi[j] - lo[j] > l) l = hi[j] - lo[j];
  l *= 1.00001;
  for(int j = 0; j < 3; j++) corner[j] = 0.5 * (lo[j] + hi[j]) - 0.5 * l;
  *len = l;
}

// The host's interleaved points onto the device.
int upload_points(hipStream_t st, DevBufs &B, int n, const double *aos, Points *P) {
  int rc = GALIC_OK;
  double *d = nullptr;
  TCHK(B.alloc(&d, 3 * (size_t)std::max(n, 1)));
  if(n > 0) TCHK(hipMemcpyAsync(d, aos, 3 * sizeof(double) * (size_t)n, hipMemcpyHostToDevice, st));
  *P = Points{d, d + 1, d + 2, 3};
done:
  return rc;
}

int upload_soa(hipStream_t st, int n, const double *aos, double *dx, double *dy, double *dz) {
  std::vector<double> t(std::max(n, 1));
  double *d[3] = {dx, dy, dz};
  for(int k = 0; k < 3; k++) {
    for(int i = 0; i < n; i++) t[i] = aos[3 * (size_t)i + k];
    if(n > 0 && hipMemcpyAsync(d[k], t.data(), sizeof(double) * n, hipMemcpyHostToDevice, st) != hipSuccess)
      return GALIC_ERR_HIP;
    if(hipStreamSynchronize(st) != hipSuccess) return GALIC_ERR_HIP;
  }
  return GALIC_OK;
}

// Node radii R_j = Rmin (Fac^j - 1) of the force grid (grid.c:680-704) and the section
// angles' cosines and sines, as galic_tree_fill computes them.
void fill_nodes(const galic_params *p, std::vector<double> &rj, std::vector<double> &cs, std::vector<double> &sn) {
  const int nb = p->FG_Nbin;
  rj.resize(nb);
  cs.resize(GALIC_FG_SECTIONS);
  sn.resize(GALIC_FG_SECTIONS);
  for(int j = 0; j < nb; j++) rj[j] = p->FG_Rmin * (pow(p->FG_Fac, j) - 1.0);
  for(int s = 0; s < GALIC_FG_SECTIONS; s++) {
    double phi = 2 * M_PI / GALIC_FG_SECTIONS * s;
    cs[s] = cos(phi);
    sn[s] = sin(phi);
  }
}

// The extent of the table fill's targets (R_j cos phi_s, R_j sin phi_s, z_k), widened into lo, hi.
void fill_extent(const std::vector<double> &rj, const std::vector<double> &cs, const std::vector<double> &sn,
                 double lo[3], double hi[3]) {
  for(size_t s = 0; s < cs.size(); s++)
    for(double r : rj) {
      lo[0] = std::min(lo[0], r * cs[s]);
      hi[0] = std::max(hi[0], r * cs[s]);
      lo[1] = std::min(lo[1], r * sn[s]);
      hi[1] = std::max(hi[1], r * sn[s]);
    }
  for(double r : rj) {
    lo[2] = std::min(lo[2], r);
    hi[2] = std::max(hi[2], r);
  }
}

// ------------------------------------------------ forcetree drop-ins' state --

// P[] of the forcetree drop-ins (allvars.h:844-868), caller-owned as the reference's P[]:
// positions, masses, types, and the GravAccel and Potential the walks write.
struct BoundParticles {
  int n = 0;
  double *pos = nullptr, *mass = nullptr, *acc = nullptr, *pot = nullptr;
  int *type = nullptr;
} g_P;

// The tree of the last force_treebuild, kept on the device for force_treeevaluate and
// force_update_node_recursive.
struct BoundTree {
  bool built = false;
  int device = 0;
  int npart = 0;                 // the build's npart: the root node's index (the reference's Tree_MaxPart)
  hipStream_t st = nullptr;
  DevBufs *B = nullptr;
  Tree T;
  int *sorted = nullptr;         // device: sorted source -> source index
  std::vector<int> src_of;       // source index -> index in P[]
  std::vector<int> targets;      // TargetList: the Type-5 particles (gravtree.c:115-119)
  double corner[3] = {0, 0, 0}, len = 0;
  galic_params p;
} g_T;

void tree_release() {
  if(g_T.B) {
    (void)hipSetDevice(g_T.device);
    delete g_T.B;
  }
  if(g_T.st) (void)hipStreamDestroy(g_T.st);
  g_T = BoundTree();
}

void tree_dropin_fail(const char *what) {
  // the reference terminates on errors in the tree code (allvars.h:129)
  fprintf(stderr, "galic forcetree drop-in %s failed: %s\n", what, galic_last_error());
  exit(1);
}

// Builds the bound tree over P[0..npart) without the Type-5 particles (forcetree.c:331);
// the domain cube covers every one of them (domain_box.c:20-65).  Returns the node count.
int tree_build_bound(int npart, int precision, bool exact = false) {
  galic_ctx *ctx = galic::bound_ctx();
  if(!ctx) return terr(GALIC_ERR_STATE, "no context bound (galic_bind): the tree takes its parameters from it");
  if(!g_P.pos || npart < 0 || npart > g_P.n)
    return terr(GALIC_ERR_ARG, "force_treebuild: npart %d beyond the %d bound particles (galic_bind_tree_particles)",
                npart, g_P.n);
  tree_release();
  const galic::Ctx &c = galic::ctx_state(ctx);
  g_T.p = c.p;
  g_T.device = c.device;
  g_T.npart = npart;
  int rc = GALIC_OK;
  std::vector<double> sx, sy, sz, sm, tp;
  std::vector<double> spos;
  for(int i = 0; i < npart; i++) {
    if(g_P.type[i] == 5) {
      g_T.targets.push_back(i);
      tp.insert(tp.end(), g_P.pos + 3 * (size_t)i, g_P.pos + 3 * (size_t)i + 3);
    } else {
      g_T.src_of.push_back(i);
      spos.insert(spos.end(), g_P.pos + 3 * (size_t)i, g_P.pos + 3 * (size_t)i + 3);
      sm.push_back(g_P.mass[i]);
    }
  }
  const int nsrc = (int)g_T.src_of.size();
  double *pm;
  Points S, X;
  double lo[3] = {1e30, 1e30, 1e30}, hi[3] = {-1e30, -1e30, -1e30};
  g_T.B = new DevBufs(exact);
  TCHK(hipSetDevice(g_T.device));
  TCHK(hipStreamCreate(&g_T.st));
  TCHK(g_T.B->alloc(&pm, nsrc));
  if((rc = upload_points(g_T.st, *g_T.B, nsrc, spos.data(), &S)) != GALIC_OK) goto done;
  if((rc = upload_points(g_T.st, *g_T.B, (int)g_T.targets.size(), tp.data(), &X)) != GALIC_OK) goto done;
  if((rc = extend_domain(g_T.st, *g_T.B, nsrc, S, lo, hi)) != GALIC_OK) goto done;
  if((rc = extend_domain(g_T.st, *g_T.B, (int)g_T.targets.size(), X, lo, hi)) != GALIC_OK) goto done;
  domain_cube(lo, hi, g_T.corner, &g_T.len);
  if(nsrc > 0) TCHK(hipMemcpy(pm, sm.data(), sizeof(double) * nsrc, hipMemcpyHostToDevice));
  rc = tree_build_dev(&g_T.p, g_T.st, nsrc, S, pm, g_T.corner, g_T.len, precision, *g_T.B, g_T.T,
                      &g_T.sorted, nullptr);
  if(rc == GALIC_OK) g_T.built = true;
done:
  if(rc != GALIC_OK) tree_release();
  if(rc == GALIC_ERR_NOMEM && !exact) return tree_build_bound(npart, precision, true);
  return rc == GALIC_OK ? g_T.T.level_lo.back() : rc;
}

// Walks n targets (positions pos, 3 each) of the bound tree; G scales the results.
int tree_walk_bound_with(DevBufs &B, int n, const double *pos, double *acc, double *pot, double G, long long *nint) {
  int rc = GALIC_OK;
  double *ax, *ay, *az, *pt;
  Points X;
  std::vector<double> h;
  TCHK(hipSetDevice(g_T.device));
  TCHK(B.alloc(&ax, n)); TCHK(B.alloc(&ay, n)); TCHK(B.alloc(&az, n)); TCHK(B.alloc(&pt, n));
  if((rc = upload_points(g_T.st, B, n, pos, &X)) != GALIC_OK) goto done;
  if((rc = tree_walk_dev(&g_T.p, g_T.st, B, g_T.T, n, X, ax, ay, az, pt, 0, G, nint, nullptr)) != GALIC_OK)
    goto done;
  h.resize(std::max(n, 1));
  {
    double *src[3] = {ax, ay, az};
    for(int k = 0; k < 3; k++) {
      if(n > 0) TCHK(hipMemcpy(h.data(), src[k], sizeof(double) * n, hipMemcpyDeviceToHost));
      for(int i = 0; i < n; i++) acc[3 * (size_t)i + k] = h[i];
    }
    if(n > 0) TCHK(hipMemcpy(pot, pt, sizeof(double) * n, hipMemcpyDeviceToHost));
  }
done:
  return rc;
}
int tree_walk_bound(int n, const double *pos, double *acc, double *pot, double G, long long *nint) {
  return galic::with_pool<DevBufs>(GALIC_ERR_NOMEM,
                                   [&](DevBufs &B) { return tree_walk_bound_with(B, n, pos, acc, pot, G, nint); });
}

// ---------------------------------------------------------- the tree calls --

int retabulate_with(DevBufs &B, galic_ctx *ctx, int precision, long long *ninteractions) {
  if(!ctx) return terr(GALIC_ERR_ARG, "null context");
  if((precision & ~15) || ((precision & GALIC_TREE_GROUP) && !(precision & GALIC_TREE_FP32)))
    return terr(GALIC_ERR_ARG, "mode: GALIC_TREE_FP32 | GALIC_TREE_QUADRUPOLE | GALIC_TREE_PLUMMER | "
                               "GALIC_TREE_GROUP (with GALIC_TREE_FP32)");
  galic::Ctx &c = galic::ctx_state(ctx);
  if(!c.tsrc || c.tsrc_n < 1) return terr(GALIC_ERR_STATE, "no tree sources (galic_set_tree_sources)");
  const galic_params *p = &c.p;
  const int nb = p->FG_Nbin, nsrc = c.tsrc_n;
  const size_t nn = (size_t)nb * nb, ns = GALIC_FG_SECTIONS * nn;
  std::vector<double> rj, cs, sn;
  fill_nodes(p, rj, cs, sn);
  // the domain over sources and targets, as galic_tree_fill forms it
  double lo[3], hi[3], corner[3], len = 0;
  for(int j = 0; j < 3; j++) {
    lo[j] = c.tsrc_lo[j];
    hi[j] = c.tsrc_hi[j];
  }
  fill_extent(rj, cs, sn, lo, hi);
  domain_cube(lo, hi, corner, &len);
  int rc = GALIC_OK;
  Tree T;
  double *drj, *dcs, *dsn, *tx, *ty, *tz, *ax, *ay, *az, *pt;
  long long ni = 0;
  float bms = 0, wms = 0;
  TCHK(hipSetDevice(c.device));
  TCHK(B.alloc(&drj, nb)); TCHK(B.alloc(&dcs, GALIC_FG_SECTIONS)); TCHK(B.alloc(&dsn, GALIC_FG_SECTIONS));
  TCHK(B.alloc(&tx, ns)); TCHK(B.alloc(&ty, ns)); TCHK(B.alloc(&tz, ns));
  TCHK(B.alloc(&ax, ns)); TCHK(B.alloc(&ay, ns)); TCHK(B.alloc(&az, ns)); TCHK(B.alloc(&pt, ns));
  TCHK(hipMemcpyAsync(drj, rj.data(), sizeof(double) * nb, hipMemcpyHostToDevice, c.stream));
  TCHK(hipMemcpyAsync(dcs, cs.data(), sizeof(double) * GALIC_FG_SECTIONS, hipMemcpyHostToDevice, c.stream));
  TCHK(hipMemcpyAsync(dsn, sn.data(), sizeof(double) * GALIC_FG_SECTIONS, hipMemcpyHostToDevice, c.stream));
  hipLaunchKernelGGL(k_fill_targets, dim3(nb256(ns)), dim3(256), 0, c.stream, nb, (const double *)drj,
                     (const double *)dcs, (const double *)dsn, tx, ty, tz);
  TCHK(hipGetLastError());
  if((rc = tree_build_dev(p, c.stream, nsrc, Points{c.tsrc, c.tsrc + nsrc, c.tsrc + 2 * (size_t)nsrc, 1},
                          c.tsrc + 3 * (size_t)nsrc, corner, len, precision, B, T, nullptr, &bms)) != GALIC_OK)
    goto done;
  if((rc = tree_walk_dev(p, c.stream, B, T, (int)ns, Points{tx, ty, tz, 1}, ax, ay, az, pt, precision, p->G, &ni, &wms,
                         nb)) != GALIC_OK)
    goto done;
  // installed as the context's tables: FG_DPotDR, FG_DPotDz, FG_Pot and the FP32 copy
  hipLaunchKernelGGL(k_project, dim3(nb256(nn)), dim3(256), 0, c.stream, nb, (const double *)ax, (const double *)ay,
                     (const double *)az, (const double *)pt, (const double *)dcs, (const double *)dsn, c.FG_DPotDR,
                     c.FG_DPotDz, c.FG_Pot);
  hipLaunchKernelGGL(k_acc_f, dim3(nb256(nn)), dim3(256), 0, c.stream, (int)nn, (const double *)c.FG_DPotDR,
                     (const double *)c.FG_DPotDz, c.FG_Acc_f);
  TCHK(hipGetLastError());
  TCHK(hipStreamSynchronize(c.stream));
  if(ninteractions) *ninteractions = ni;
  g_last_build_ms = bms;
  g_last_walk_ms = wms;
  g_last_interactions = (double)ni;
done:
  return rc;
}

int tree_forces_with(DevBufs &B, const galic_params *p, int device, int nsrc, const double *spos, const double *smass,
                      int ntarget, const double *tpos, double *acc, double *pot, int precision,
                      long long *ninteractions) {
  if(!p || nsrc < 0 || ntarget < 0 || (nsrc > 0 && (!spos || !smass)) || (ntarget > 0 && (!tpos || !acc || !pot)))
    return terr(GALIC_ERR_ARG, "bad tree arguments");
  if((precision & ~15) || ((precision & GALIC_TREE_GROUP) && !(precision & GALIC_TREE_FP32)))
    return terr(GALIC_ERR_ARG, "mode: GALIC_TREE_FP32 | GALIC_TREE_QUADRUPOLE | GALIC_TREE_PLUMMER | "
                               "GALIC_TREE_GROUP (with GALIC_TREE_FP32)");
  int rc = GALIC_OK;
  const hipStream_t st = hipStreamPerThread;
  double *pm, *ax, *ay, *az, *pt;
  Points S, X;
  double lo[3] = {1e30, 1e30, 1e30}, hi[3] = {-1e30, -1e30, -1e30}, corner[3], len;
  float ms = 0;
  std::vector<double> h;
  TCHK(hipSetDevice(device));
  TCHK(B.alloc(&pm, nsrc));
  TCHK(B.alloc(&ax, ntarget)); TCHK(B.alloc(&ay, ntarget)); TCHK(B.alloc(&az, ntarget)); TCHK(B.alloc(&pt, ntarget));
  if((rc = upload_points(st, B, nsrc, spos, &S)) != GALIC_OK) goto done;
  if((rc = upload_points(st, B, ntarget, tpos, &X)) != GALIC_OK) goto done;
  if(nsrc > 0) TCHK(hipMemcpyAsync(pm, smass, sizeof(double) * nsrc, hipMemcpyHostToDevice, st));
  if((rc = extend_domain(st, B, nsrc, S, lo, hi)) != GALIC_OK) goto done;
  if((rc = extend_domain(st, B, ntarget, X, lo, hi)) != GALIC_OK) goto done;
  domain_cube(lo, hi, corner, &len);
  rc = tree_forces_dev(p, st, B, nsrc, S, pm, ntarget, X, corner, len, ax, ay, az, pt, precision, ninteractions, &ms);
  if(rc != GALIC_OK) goto done;
  h.resize(std::max(ntarget, 1));
  {
    double *src[3] = {ax, ay, az};
    for(int k = 0; k < 3; k++) {
      if(ntarget > 0) TCHK(hipMemcpy(h.data(), src[k], sizeof(double) * ntarget, hipMemcpyDeviceToHost));
      for(int i = 0; i < ntarget; i++) acc[3 * (size_t)i + k] = h[i];
    }
    if(ntarget > 0) TCHK(hipMemcpy(pot, pt, sizeof(double) * ntarget, hipMemcpyDeviceToHost));
  }
done:
  (void)hipStreamSynchronize(st);  // (the buffers go next)
  return rc;
}

int tree_fill_with(DevBufs &B, const galic_params *p, int device, int nsrc, const double *spos, const double *smass,
                    double *pot, double *dpotdr, double *dpotdz, int precision, long long *ninteractions) {
  if(!p || nsrc < 0 || (nsrc > 0 && (!spos || !smass)) || !pot || !dpotdr || !dpotdz || p->FG_Nbin < 2)
    return terr(GALIC_ERR_ARG, "bad table-fill arguments");
  if((precision & ~15) || ((precision & GALIC_TREE_GROUP) && !(precision & GALIC_TREE_FP32)))
    return terr(GALIC_ERR_ARG, "mode: GALIC_TREE_FP32 | GALIC_TREE_QUADRUPOLE | GALIC_TREE_PLUMMER | "
                               "GALIC_TREE_GROUP (with GALIC_TREE_FP32)");
  const int nb = p->FG_Nbin;
  const size_t ns = (size_t)GALIC_FG_SECTIONS * nb * nb;
  if(ns > 0x7fffffff) return terr(GALIC_ERR_ARG, "FG_Nbin too large");
  // targets of grid.c:680-704: (R_j cos phi_s, R_j sin phi_s, z_k), formed on the device
  std::vector<double> rj, cs, sn;
  fill_nodes(p, rj, cs, sn);
  int rc = GALIC_OK;
  const hipStream_t st = hipStreamPerThread;
  double *pm, *tx, *ty, *tz, *ax, *ay, *az, *pt, *drj, *dcs, *dsn, *r0, *r1, *r2;
  Points S;
  double lo[3] = {1e30, 1e30, 1e30}, hi[3] = {-1e30, -1e30, -1e30}, corner[3], len;
  float ms = 0;
  TCHK(hipSetDevice(device));
  TCHK(B.alloc(&pm, nsrc));
  TCHK(B.alloc(&tx, ns)); TCHK(B.alloc(&ty, ns)); TCHK(B.alloc(&tz, ns));
  TCHK(B.alloc(&ax, ns)); TCHK(B.alloc(&ay, ns)); TCHK(B.alloc(&az, ns)); TCHK(B.alloc(&pt, ns));
  TCHK(B.alloc(&drj, nb)); TCHK(B.alloc(&dcs, GALIC_FG_SECTIONS)); TCHK(B.alloc(&dsn, GALIC_FG_SECTIONS));
  TCHK(B.alloc(&r0, (size_t)nb * nb)); TCHK(B.alloc(&r1, (size_t)nb * nb)); TCHK(B.alloc(&r2, (size_t)nb * nb));
  if((rc = upload_points(st, B, nsrc, spos, &S)) != GALIC_OK) goto done;
  if(nsrc > 0) TCHK(hipMemcpyAsync(pm, smass, sizeof(double) * nsrc, hipMemcpyHostToDevice, st));
  TCHK(hipMemcpyAsync(drj, rj.data(), sizeof(double) * nb, hipMemcpyHostToDevice, st));
  TCHK(hipMemcpyAsync(dcs, cs.data(), sizeof(double) * GALIC_FG_SECTIONS, hipMemcpyHostToDevice, st));
  TCHK(hipMemcpyAsync(dsn, sn.data(), sizeof(double) * GALIC_FG_SECTIONS, hipMemcpyHostToDevice, st));
  hipLaunchKernelGGL(k_fill_targets, dim3(nb256(ns)), dim3(256), 0, st, nb, (const double *)drj, (const double *)dcs,
                     (const double *)dsn, tx, ty, tz);
  TCHK(hipGetLastError());
  if((rc = extend_domain(st, B, nsrc, S, lo, hi)) != GALIC_OK) goto done;
  fill_extent(rj, cs, sn, lo, hi);
  domain_cube(lo, hi, corner, &len);
  rc = tree_forces_dev(p, st, B, nsrc, S, pm, (int)ns, Points{tx, ty, tz, 1}, corner, len, ax, ay, az, pt, precision,
                       ninteractions, &ms, nb);
  if(rc != GALIC_OK) goto done;
  hipLaunchKernelGGL(k_project, dim3(nb256((size_t)nb * nb)), dim3(256), 0, st, nb, (const double *)ax,
                     (const double *)ay, (const double *)az, (const double *)pt, (const double *)dcs,
                     (const double *)dsn, r1, r2, r0);
  TCHK(hipGetLastError());
  TCHK(hipMemcpyAsync(dpotdr, r1, sizeof(double) * nb * nb, hipMemcpyDeviceToHost, st));
  TCHK(hipMemcpyAsync(dpotdz, r2, sizeof(double) * nb * nb, hipMemcpyDeviceToHost, st));
  TCHK(hipMemcpyAsync(pot, r0, sizeof(double) * nb * nb, hipMemcpyDeviceToHost, st));
  TCHK(hipStreamSynchronize(st));
done:
  (void)hipStreamSynchronize(st);  // (the buffers and the host arrays of the copies go next)
  return rc;
}

int direct_forces_with(DevBufs &B, const galic_params *p, int device, int nsrc, const double *spos, const double *smass,
                             int ntarget, const double *tpos, double *acc, double *pot, int mode) {
  if(!p || nsrc < 0 || ntarget < 0 || (nsrc > 0 && (!spos || !smass)) || (ntarget > 0 && (!tpos || !acc || !pot)))
    return terr(GALIC_ERR_ARG, "bad direct-summation arguments");
  if(mode != 0 && mode != GALIC_TREE_PLUMMER) return terr(GALIC_ERR_ARG, "mode: 0 or GALIC_TREE_PLUMMER");
  int rc = GALIC_OK;
  hipStream_t st = nullptr;
  double *px, *py, *pz, *pm, *tx, *ty, *tz, *ax, *ay, *az, *pt;
  std::vector<double> h;
  TCHK(hipSetDevice(device));
  TCHK(hipStreamCreate(&st));
  TCHK(B.alloc(&px, nsrc)); TCHK(B.alloc(&py, nsrc)); TCHK(B.alloc(&pz, nsrc)); TCHK(B.alloc(&pm, nsrc));
  TCHK(B.alloc(&tx, ntarget)); TCHK(B.alloc(&ty, ntarget)); TCHK(B.alloc(&tz, ntarget));
  TCHK(B.alloc(&ax, ntarget)); TCHK(B.alloc(&ay, ntarget)); TCHK(B.alloc(&az, ntarget)); TCHK(B.alloc(&pt, ntarget));
  if((rc = upload_soa(st, nsrc, spos, px, py, pz)) != GALIC_OK) goto done;
  if((rc = upload_soa(st, ntarget, tpos, tx, ty, tz)) != GALIC_OK) goto done;
  if(nsrc > 0) TCHK(hipMemcpy(pm, smass, sizeof(double) * nsrc, hipMemcpyHostToDevice));
  if(ntarget > 0) {
    hipLaunchKernelGGL(galic::tree::k_direct64, dim3(nb256(ntarget)), dim3(256), 0, st, nsrc, (const double *)px,
                       (const double *)py, (const double *)pz, (const double *)pm, ntarget, (const double *)tx,
                       (const double *)ty, (const double *)tz, p->ForceSoftening, mode == GALIC_TREE_PLUMMER ? 1 : 0,
                       p->ForceSoftening / 2.8, p->G, ax, ay, az, pt);
    TCHK(hipGetLastError());
    TCHK(hipStreamSynchronize(st));
    h.resize(ntarget);
    double *src[3] = {ax, ay, az};
    for(int k = 0; k < 3; k++) {
      TCHK(hipMemcpy(h.data(), src[k], sizeof(double) * ntarget, hipMemcpyDeviceToHost));
      for(int i = 0; i < ntarget; i++) acc[3 * (size_t)i + k] = h[i];
    }
    TCHK(hipMemcpy(pot, pt, sizeof(double) * ntarget, hipMemcpyDeviceToHost));
  }
done:
  if(st) (void)hipStreamDestroy(st);
  return rc;
}

}  // namespace

extern "C" {

int galic_bind_tree_particles(int n, double *pos, double *mass, int *type, double *grav_accel, double *potential) {
  if(n < 0 || (n > 0 && (!pos || !mass || !type || !grav_accel || !potential)))
    return terr(GALIC_ERR_ARG, "galic_bind_tree_particles: bad arguments");
  tree_release();
  g_P.n = n;
  g_P.pos = pos;
  g_P.mass = mass;
  g_P.type = type;
  g_P.acc = grav_accel;
  g_P.pot = potential;
  return GALIC_OK;
}

int force_treebuild(int npart, int optimized_domain_mapping) {
  (void)optimized_domain_mapping;  // one GPU: no domain mapping to optimise
  const int r = tree_build_bound(npart, 0);
  if(r < 0) tree_dropin_fail("force_treebuild");
  return r;
}

void force_update_node_recursive(int no, int sib, int father, int *last) {
  if(!g_T.built) tree_dropin_fail("force_update_node_recursive (no tree built)");
  if(no != g_T.npart || sib != -1 || father != -1) {
    terr(GALIC_ERR_ARG, "node %d: the device tree numbers its own nodes; only the root (%d, sibling -1, father -1, "
         "as forcetree.c:86 calls it) is addressed", no, g_T.npart);
    tree_dropin_fail("force_update_node_recursive");
  }
  (void)hipSetDevice(g_T.device);
  if(tree_moments_dev(g_T.st, g_T.T, g_T.len) != GALIC_OK || hipStreamSynchronize(g_T.st) != hipSuccess)
    tree_dropin_fail("force_update_node_recursive");
  if(last) {
    // the walk order ends at the last source in key order (children are threaded in order)
    int s = -1;
    const int nsrc = g_T.T.nsrc;
    if(nsrc > 0 && hipMemcpy(&s, g_T.sorted + (nsrc - 1), sizeof(int), hipMemcpyDeviceToHost) != hipSuccess)
      tree_dropin_fail("force_update_node_recursive");
    *last = (s >= 0) ? g_T.src_of[s] : -1;
  }
}

int force_treeevaluate(int target, int mode, int thread_id) {
  (void)thread_id;
  if(!g_T.built) tree_dropin_fail("force_treeevaluate (no tree built)");
  if(mode != 0) {
    terr(GALIC_ERR_ARG, "mode %d: imported targets of other tasks have no counterpart on one GPU", mode);
    tree_dropin_fail("force_treeevaluate");
  }
  if(target < 0 || target >= (int)g_T.targets.size()) {
    terr(GALIC_ERR_ARG, "target %d beyond the %zu Type-5 particles", target, g_T.targets.size());
    tree_dropin_fail("force_treeevaluate");
  }
  // TargetList[target] (forcetree_walk.c:28-41); the sums are left without G, as the walk
  // leaves them (gravity_tree multiplies afterwards)
  const int i = g_T.targets[target];
  long long nint = 0;
  if(tree_walk_bound(1, g_P.pos + 3 * (size_t)i, g_P.acc + 3 * (size_t)i, g_P.pot + i, 1.0, &nint) != GALIC_OK)
    tree_dropin_fail("force_treeevaluate");
  return (int)nint;
}

void gravity(void) {
  // gravtree.c:35-50 and 88-467: build, walk every Type-5 particle, multiply by G, free
  if(tree_build_bound(g_P.n, 0) < 0) tree_dropin_fail("gravity");
  const int nt = (int)g_T.targets.size();
  std::vector<double> tp(3 * (size_t)nt), acc(3 * (size_t)nt), pot(nt);
  for(int k = 0; k < nt; k++)
    for(int j = 0; j < 3; j++) tp[3 * (size_t)k + j] = g_P.pos[3 * (size_t)g_T.targets[k] + j];
  if(tree_walk_bound(nt, tp.data(), acc.data(), pot.data(), g_T.p.G, nullptr) != GALIC_OK) tree_dropin_fail("gravity");
  for(int k = 0; k < nt; k++) {
    const int i = g_T.targets[k];
    for(int j = 0; j < 3; j++) g_P.acc[3 * (size_t)i + j] = acc[3 * (size_t)k + j];
    g_P.pot[i] = pot[k];
  }
  tree_release();
}

int galic_set_tree_sources(galic_ctx *ctx, int nsrc, const double *spos, const double *smass) {
  if(!ctx || nsrc < 1 || !spos || !smass) return terr(GALIC_ERR_ARG, "galic_set_tree_sources: bad arguments");
  galic::Ctx &c = galic::ctx_state(ctx);
  int rc = GALIC_OK;
  TCHK(hipSetDevice(c.device));
  if(c.tsrc) (void)hipFree(c.tsrc);
  c.tsrc = nullptr;
  c.tsrc_n = 0;
  TCHK(hipMalloc(&c.tsrc, sizeof(double) * 4 * (size_t)nsrc));
  c.tsrc_n = nsrc;
  for(int j = 0; j < 3; j++) {
    c.tsrc_lo[j] = 1e30;
    c.tsrc_hi[j] = -1e30;
  }
  for(int i = 0; i < nsrc; i++)
    for(int j = 0; j < 3; j++) {
      const double x = spos[3 * (size_t)i + j];
      if(c.tsrc_lo[j] > x) c.tsrc_lo[j] = x;
      if(c.tsrc_hi[j] < x) c.tsrc_hi[j] = x;
    }
  if((rc = upload_soa(c.stream, nsrc, spos, c.tsrc, c.tsrc + nsrc, c.tsrc + 2 * (size_t)nsrc)) != GALIC_OK) goto done;
  TCHK(hipMemcpy(c.tsrc + 3 * (size_t)nsrc, smass, sizeof(double) * nsrc, hipMemcpyHostToDevice));
done:
  return rc;
}

int galic_retabulate(galic_ctx *ctx, int precision, long long *ninteractions) {
  return galic::with_pool<DevBufs>(GALIC_ERR_NOMEM, [&](DevBufs &B) {
    return retabulate_with(B, ctx, precision, ninteractions);
  });
}

int galic_tree_forces(const galic_params *p, int device, int nsrc, const double *spos, const double *smass,
                      int ntarget, const double *tpos, double *acc, double *pot, int precision,
                      long long *ninteractions) {
  return galic::with_pool<DevBufs>(GALIC_ERR_NOMEM, [&](DevBufs &B) {
    return tree_forces_with(B, p, device, nsrc, spos, smass, ntarget, tpos, acc, pot, precision, ninteractions);
  });
}

int galic_tree_fill(const galic_params *p, int device, int nsrc, const double *spos, const double *smass,
                    double *pot, double *dpotdr, double *dpotdz, int precision, long long *ninteractions) {
  return galic::with_pool<DevBufs>(GALIC_ERR_NOMEM, [&](DevBufs &B) {
    return tree_fill_with(B, p, device, nsrc, spos, smass, pot, dpotdr, dpotdz, precision, ninteractions);
  });
}

int galic_direct_forces(const galic_params *p, int device, int nsrc, const double *spos, const double *smass,
                        int ntarget, const double *tpos, double *acc, double *pot) {
  return galic_direct_forces_mode(p, device, nsrc, spos, smass, ntarget, tpos, acc, pot, 0);
}

int galic_direct_forces_mode(const galic_params *p, int device, int nsrc, const double *spos, const double *smass,
                             int ntarget, const double *tpos, double *acc, double *pot, int mode) {
  return galic::with_pool<DevBufs>(GALIC_ERR_NOMEM, [&](DevBufs &B) {
    return direct_forces_with(B, p, device, nsrc, spos, smass, ntarget, tpos, acc, pot, mode);
  });
}

int galic_tree_last_timings(double *out3) {
  if(!out3) return terr(GALIC_ERR_ARG, "null argument");
  out3[0] = g_last_build_ms;
  out3[1] = g_last_walk_ms;
  out3[2] = g_last_interactions;
  return GALIC_OK;
}

}  // extern "C"
