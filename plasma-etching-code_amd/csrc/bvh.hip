// Morton-code LBVH over the surface triangles, rebuilt every step (replaces
// wp.Mesh(points, indices), threed.py:1674-1675):
//   prep     triangle centroids + per-block bounds        -> scene bounds (one workgroup)
//   morton   30-bit codes of the centroids                -> stable LDS radix sort (sort.hip)
//   leaves   triangle vertices gathered into Morton order (48 B per leaf)
//   karras   internal nodes from the sorted codes (Karras, HPG 2012), ties broken by index
//   refit    boxes of the nodes inside each 256-leaf tile in LDS, then those of the few nodes that
//            span tiles from the tiles' prefix, suffix and whole boxes
//   wide     4-wide nodes at binary-node indices: on large meshes a top-down collapse that
//            opens the larger-area inner child first (the top levels in one workgroup, then a
//            wavefront per subtree); on small ones every binary node at even depth (parity from
//            its parent chain) gathers its grandchildren (one parallel pass)
// plus the two query entry points used by the tests (the trace kernels inline the traversal).
#include "common.h"
#include <vector>

#include <stdlib.h>
#include "bvh.h"
#include "gridwalk.h"
#include "scan.h"

bool petch_grid_view(const petch_bvh* b, petch::GridView* v);
int petch_radix_sort_pairs(petch_ctx* ctx, uint32_t* keys, uint32_t* vals, uint32_t* ktmp,
                           uint32_t* vtmp, int n, int bits);

using petch::BvhNode;
using petch::BvhView;
using petch::BvhWide;

namespace {

constexpr int kBS = 256;

enum Hdr { H_COUNT, H_SIDE, H_LEVEL, H_OVER, H_OVER_LEVEL, H_DONE };

struct Work {  // device scratch owned by the BVH, carved from bvh->work
  float4* cen;
  uint32_t *keys, *vals, *ktmp, *vtmp;
  int *pint, *pleaf, *err;
  int* hdr;      // device state of the area-driven collapse and of the clustering (Hdr)
  float* part;   // per-block bounds (6 per block)
  float* scene;  // 6 floats
  float* root;   // 6 floats
};

size_t work_bytes(int cap_f) {
  size_t nb = (cap_f + kBS - 1) / kBS;
  return (size_t)cap_f * 16 + (size_t)cap_f * 4 * 4 + (size_t)cap_f * 4 * 2 + 64 +
         nb * 6 * 4 + 64 + 64 + 1024;
}

Work carve(void* base, int cap_f) {
  char* p = (char*)base;
  Work w;
  size_t nb = (cap_f + kBS - 1) / kBS;
  w.cen = (float4*)p; p += (size_t)cap_f * 16;
  w.keys = (uint32_t*)p; p += (size_t)cap_f * 4;
  w.vals = (uint32_t*)p; p += (size_t)cap_f * 4;
  w.ktmp = (uint32_t*)p; p += (size_t)cap_f * 4;
  w.vtmp = (uint32_t*)p; p += (size_t)cap_f * 4;
  w.pint = (int*)p; p += (size_t)cap_f * 4;
  w.pleaf = (int*)p; p += (size_t)cap_f * 4;
  w.err = (int*)p;
  w.hdr = w.err + 4; p += 64;
  w.part = (float*)p; p += nb * 6 * 4;
  w.scene = (float*)p; p += 64;
  w.root = (float*)p; p += 64;
  return w;
}

__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v = fminf(v, __shfl_xor(v, d, 64));
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v = fmaxf(v, __shfl_xor(v, d, 64));
  return v;
}

// Centroids of block lb's faces and the block's centroid bounds (6 floats at part[6 lb]).
__device__ __forceinline__ void bvh_prep_block(const float* __restrict__ verts,
                                               const int* __restrict__ faces, int nf,
                                               float4* __restrict__ cen, float* __restrict__ part,
                                               int lb) {
  int f = lb * kBS + threadIdx.x;
  float c[3] = {3.0e38f, 3.0e38f, 3.0e38f}, cmax[3] = {-3.0e38f, -3.0e38f, -3.0e38f};
  if (f < nf) {
    int a = faces[3 * f], b = faces[3 * f + 1], d = faces[3 * f + 2];
    float x = (verts[3 * a] + verts[3 * b] + verts[3 * d]) / 3.f;
    float y = (verts[3 * a + 1] + verts[3 * b + 1] + verts[3 * d + 1]) / 3.f;
    float z = (verts[3 * a + 2] + verts[3 * b + 2] + verts[3 * d + 2]) / 3.f;
    cen[f] = make_float4(x, y, z, 0.f);
    c[0] = cmax[0] = x;
    c[1] = cmax[1] = y;
    c[2] = cmax[2] = z;
  }
  __shared__ float s[kBS / 64][6];
  int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (int k = 0; k < 3; ++k) {
    float mn = wave_min(c[k]), mx = wave_max(cmax[k]);
    if (lane == 0) {
      s[w][k] = mn;
      s[w][3 + k] = mx;
    }
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    int k = threadIdx.x;
    float v = s[0][k];
    for (int q = 1; q < kBS / 64; ++q) v = (k < 3) ? fminf(v, s[q][k]) : fmaxf(v, s[q][k]);
    part[lb * 6 + k] = v;
  }
}

__global__ void __launch_bounds__(kBS) k_bvh_prep(const float* __restrict__ verts,
                                                  const int* __restrict__ faces, int nf,
                                                  float4* __restrict__ cen,
                                                  float* __restrict__ part) {
  bvh_prep_block(verts, faces, nf, cen, part, blockIdx.x);
}

// The scene bounds from nb block partials (one workgroup).
__device__ __forceinline__ void bvh_bounds_wg(const float* __restrict__ part, int nb,
                                              float* __restrict__ scene) {
  __shared__ float s[6][kBS];
  for (int k = 0; k < 6; ++k) {
    float v = (k < 3) ? 3.0e38f : -3.0e38f;
    for (int b = threadIdx.x; b < nb; b += kBS)
      v = (k < 3) ? fminf(v, part[b * 6 + k]) : fmaxf(v, part[b * 6 + k]);
    s[k][threadIdx.x] = v;
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    int k = threadIdx.x;
    float v = s[k][0];
    for (int q = 1; q < kBS; ++q) v = (k < 3) ? fminf(v, s[k][q]) : fmaxf(v, s[k][q]);
    scene[k] = v;
  }
}

__global__ void __launch_bounds__(kBS) k_bvh_bounds(const float* __restrict__ part, int nb,
                                                    float* __restrict__ scene) {
  bvh_bounds_wg(part, nb, scene);
}

__device__ __forceinline__ uint32_t spread10(uint32_t v) {
  v = (v * 0x00010001u) & 0xFF0000FFu;
  v = (v * 0x00000101u) & 0x0F00F00Fu;
  v = (v * 0x00000011u) & 0xC30C30C3u;
  v = (v * 0x00000005u) & 0x49249249u;
  return v;
}

__device__ __forceinline__ void bvh_morton_face(const float4* __restrict__ cen,
                                                const float* __restrict__ scene,
                                                uint32_t* __restrict__ keys,
                                                uint32_t* __restrict__ vals, int f) {
  float4 c = cen[f];
  float q[3] = {c.x, c.y, c.z};
  uint32_t u[3];
  for (int k = 0; k < 3; ++k) {
    float ext = scene[3 + k] - scene[k];
    float t = ext > 0.f ? (q[k] - scene[k]) / ext : 0.f;
    float s = fminf(fmaxf(t * 1024.f, 0.f), 1023.f);
    u[k] = (uint32_t)s;
  }
  keys[f] = (spread10(u[0]) << 2) | (spread10(u[1]) << 1) | spread10(u[2]);
  vals[f] = (uint32_t)f;
}

__global__ void k_bvh_morton(const float4* __restrict__ cen, int nf,
                             const float* __restrict__ scene, uint32_t* __restrict__ keys,
                             uint32_t* __restrict__ vals) {
  int f = blockIdx.x * kBS + threadIdx.x;
  if (f < nf) bvh_morton_face(cen, scene, keys, vals, f);
}

__device__ __forceinline__ void bvh_leaf(const float* __restrict__ verts,
                                         const int* __restrict__ faces,
                                         const uint32_t* __restrict__ vals,
                                         float4* __restrict__ tris, int s) {
  int f = (int)vals[s];
  int a = faces[3 * f], b = faces[3 * f + 1], c = faces[3 * f + 2];
  tris[3 * s] = make_float4(verts[3 * a], verts[3 * a + 1], verts[3 * a + 2], __int_as_float(f));
  tris[3 * s + 1] = make_float4(verts[3 * b], verts[3 * b + 1], verts[3 * b + 2], 0.f);
  tris[3 * s + 2] = make_float4(verts[3 * c], verts[3 * c + 1], verts[3 * c + 2], 0.f);
}

__global__ void k_bvh_leaves(const float* __restrict__ verts, const int* __restrict__ faces,
                             const uint32_t* __restrict__ vals, int nf,
                             float4* __restrict__ tris) {
  int s = blockIdx.x * kBS + threadIdx.x;
  if (s < nf) bvh_leaf(verts, faces, vals, tris, s);
}

__device__ __forceinline__ int delta(const uint32_t* __restrict__ k, int n, int i, int j) {
  if (j < 0 || j >= n) return -1;
  uint32_t a = k[i], b = k[j];
  if (a == b) return 32 + __clz((uint32_t)(i ^ j));
  return __clz(a ^ b);
}

__device__ __forceinline__ void bvh_karras_node(const uint32_t* __restrict__ keys, int n,
                                                BvhNode* __restrict__ nodes, int* __restrict__ pint,
                                                int* __restrict__ pleaf, int i) {
  int d = (delta(keys, n, i, i + 1) - delta(keys, n, i, i - 1)) >= 0 ? 1 : -1;
  int dmin = delta(keys, n, i, i - d);
  int lmax = 2;
  while (delta(keys, n, i, i + lmax * d) > dmin) lmax <<= 1;
  int l = 0;
  for (int t = lmax >> 1; t >= 1; t >>= 1)
    if (delta(keys, n, i, i + (l + t) * d) > dmin) l += t;
  int j = i + l * d;
  int dnode = delta(keys, n, i, j);
  int s = 0, t = l;
  while (true) {
    t = (t + 1) >> 1;
    if (delta(keys, n, i, i + (s + t) * d) > dnode) s += t;
    if (t <= 1) break;
  }
  int gamma = i + s * d + (d < 0 ? -1 : 0);
  int lo = i < j ? i : j, hi = i < j ? j : i;
  int left = (lo == gamma) ? ~gamma : gamma;
  int right = (hi == gamma + 1) ? ~(gamma + 1) : gamma + 1;
  nodes[i].d = make_int4(left, right, lo, hi);  // children, first and last leaf
  if (left < 0) pleaf[~left] = i; else pint[left] = i;
  if (right < 0) pleaf[~right] = i; else pint[right] = i;
  if (i == 0) pint[0] = -1;
}

// `done`, here and in the refit: where the clustered tree is complete there is nothing to do.
__global__ void k_bvh_karras(const uint32_t* __restrict__ keys, int n, BvhNode* __restrict__ nodes,
                             int* __restrict__ pint, int* __restrict__ pleaf,
                             const int* __restrict__ done) {
  if (done && *done) return;
  int i = blockIdx.x * kBS + threadIdx.x;
  if (i < n - 1) bvh_karras_node(keys, n, nodes, pint, pleaf, i);
}

__device__ __forceinline__ void put_child_box(BvhNode* nd, bool left, const float lo[3],
                                              const float hi[3]) {
  float* p = (float*)nd;
  if (left) {
    p[0] = lo[0]; p[1] = lo[1]; p[2] = lo[2]; p[3] = hi[0]; p[4] = hi[1]; p[5] = hi[2];
  } else {
    p[6] = lo[0]; p[7] = lo[1]; p[8] = lo[2]; p[9] = hi[0]; p[10] = hi[1]; p[11] = hi[2];
  }
}

// The refit: every node's two child boxes, from the leaves' triangles. One climb from the leaves
// with a flag in memory at each node is a chain of dependent global accesses as deep as the tree,
// each with an agent-scope release (51 us at 8k faces, 237 us at 47k), or with one workgroup a
// tree, so that workgroup scope is enough, a pass over all leaves by that workgroup (2.55 ms for
// 32 trees of 8 to 30k faces side by side). Here a workgroup takes a tile of kTile leaves in
// Morton order and climbs in LDS through the nodes whose leaves lie inside the tile; a node spanning tiles, a few
// for each tile, is the union of its first tile's suffix box, its last tile's prefix box and the
// whole tiles between, so no chain runs through memory: 16 us at 8k faces, 17 at 47k, 113 us for the
// 32 trees. The boxes are the same, minima and maxima of the same numbers.
constexpr int kTile = kBS;

struct RefitItem {
  const float4* tris;
  BvhNode* nodes;
  const int *pint, *pleaf;
  float* scr;        // prefix boxes, then suffix boxes, 6 floats a leaf (the wide nodes' memory)
  float* root;
  const int* done;   // nothing to refit where this is set
  int n;
  long long blk0;    // first tile of this tree in the launch
};

__device__ __forceinline__ const RefitItem& refit_item(const RefitItem* __restrict__ it, int n) {
  int lo = 0, hi = n - 1;
  const long long b = blockIdx.x;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (it[mid].blk0 <= b) lo = mid; else hi = mid - 1;
  }
  return it[lo];
}

__device__ __forceinline__ bool in_one_tile(int4 d) { return d.z / kTile == d.w / kTile; }

__device__ __forceinline__ void put_root(float* root, const float lo[3], const float hi[3]) {
  for (int k = 0; k < 3; ++k) {
    root[k] = lo[k];
    root[3 + k] = hi[k];
  }
}

__device__ __forceinline__ void refit_tile(const RefitItem& it, int tile) {
  __shared__ int4 s_d[kTile];
  __shared__ int s_par[kTile], s_flag[kTile];
  __shared__ float s_box[12][kTile];
  __shared__ float s_pre[kBS / 64][6], s_suf[kBS / 64][6];
  const int n = it.n, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int base = tile * kTile, i = base + tid;
  const bool node = i < n - 1, leaf = i < n;
  if (node) {
    s_d[tid] = it.nodes[i].d;
    s_par[tid] = it.pint[i];
    s_flag[tid] = 0;
  }
  float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
  if (leaf) {
    const float4 a = it.tris[3 * i], b = it.tris[3 * i + 1], c = it.tris[3 * i + 2];
    lo[0] = fminf(a.x, fminf(b.x, c.x)); hi[0] = fmaxf(a.x, fmaxf(b.x, c.x));
    lo[1] = fminf(a.y, fminf(b.y, c.y)); hi[1] = fmaxf(a.y, fmaxf(b.y, c.y));
    lo[2] = fminf(a.z, fminf(b.z, c.z)); hi[2] = fmaxf(a.z, fmaxf(b.z, c.z));
  }
  if (n > kTile) {
    float pre[6], suf[6];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      pre[k] = suf[k] = lo[k];
      pre[3 + k] = suf[3 + k] = hi[k];
    }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        const float u = __shfl_up(pre[k], d, 64), v = __shfl_down(suf[k], d, 64);
        if (lane >= d) pre[k] = k < 3 ? fminf(pre[k], u) : fmaxf(pre[k], u);
        if (lane + d < 64) suf[k] = k < 3 ? fminf(suf[k], v) : fmaxf(suf[k], v);
      }
    }
    if (lane == 63)
      for (int k = 0; k < 6; ++k) s_pre[w][k] = pre[k];
    if (lane == 0)
      for (int k = 0; k < 6; ++k) s_suf[w][k] = suf[k];
    __syncthreads();
    for (int q = 0; q < kBS / 64; ++q) {
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        if (q < w) pre[k] = k < 3 ? fminf(pre[k], s_pre[q][k]) : fmaxf(pre[k], s_pre[q][k]);
        if (q > w) suf[k] = k < 3 ? fminf(suf[k], s_suf[q][k]) : fmaxf(suf[k], s_suf[q][k]);
      }
    }
    if (leaf) {
      float* o = it.scr + 6LL * i;
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        o[k] = pre[k];
        o[6LL * n + k] = suf[k];
      }
    }
  }
  __syncthreads();
  if (leaf) {
    int child = ~i, p = it.pleaf[i];
    while (true) {
      const int l = p - base;
      if (l < 0 || l >= kTile || !in_one_tile(s_d[l])) {
        put_child_box(it.nodes + p, it.nodes[p].d.x == child, lo, hi);
        break;
      }
      const int side = s_d[l].x == child ? 0 : 6;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        s_box[side + k][l] = lo[k];
        s_box[side + 3 + k][l] = hi[k];
      }
      const int seen =
          __hip_atomic_fetch_add(s_flag + l, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
      if (seen == 0) break;   // the second child to arrive goes on
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        lo[k] = fminf(s_box[k][l], s_box[6 + k][l]);
        hi[k] = fmaxf(s_box[3 + k][l], s_box[9 + k][l]);
      }
      child = p;
      p = s_par[l];
      if (p < 0) {
        put_root(it.root, lo, hi);
        break;
      }
    }
  }
  __syncthreads();
  if (node && in_one_tile(s_d[tid])) {
    BvhNode* nd = it.nodes + i;
    nd->a = make_float4(s_box[0][tid], s_box[1][tid], s_box[2][tid], s_box[3][tid]);
    nd->b = make_float4(s_box[4][tid], s_box[5][tid], s_box[6][tid], s_box[7][tid]);
    nd->c = make_float4(s_box[8][tid], s_box[9][tid], s_box[10][tid], s_box[11][tid]);
  }
}

// The box of each node of the tile that spans tiles, into its parent's child slot. A long run of
// whole tiles is read by the wavefront together, a short one by its own lane.
constexpr int kSpanSerial = 8;
__device__ __forceinline__ void refit_span(const RefitItem& it, int tile) {
  const int n = it.n, i = tile * kTile + threadIdx.x, lane = threadIdx.x & 63;
  const float* suf = it.scr + 6LL * n;
  int4 d = make_int4(0, 0, 0, 0);
  if (i < n - 1) d = it.nodes[i].d;
  const bool span = !in_one_tile(d);
  const int t0 = d.z / kTile + 1, t1 = d.w / kTile;   // whole tiles t0 .. t1 - 1
  float box[6];
  for (int k = 0; k < 6; ++k) box[k] = k < 3 ? INFINITY : -INFINITY;
  if (span) {
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      const float a = suf[6LL * d.z + k], b = it.scr[6LL * d.w + k];
      box[k] = k < 3 ? fminf(a, b) : fmaxf(a, b);
    }
    if (t1 - t0 <= kSpanSerial) {
      for (int t = t0; t < t1; ++t) {
#pragma unroll
        for (int k = 0; k < 6; ++k) {
          const float v = suf[6LL * t * kTile + k];
          box[k] = k < 3 ? fminf(box[k], v) : fmaxf(box[k], v);
        }
      }
    }
  }
  unsigned long long todo = __ballot(span && t1 - t0 > kSpanSerial);
  while (todo) {
    const int who = __ffsll(todo) - 1;
    todo &= todo - 1;
    const int a = __shfl(t0, who, 64), e = __shfl(t1, who, 64);
    float part[6];
    for (int k = 0; k < 6; ++k) part[k] = k < 3 ? INFINITY : -INFINITY;
    for (int t = a + lane; t < e; t += 64) {
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        const float v = suf[6LL * t * kTile + k];
        part[k] = k < 3 ? fminf(part[k], v) : fmaxf(part[k], v);
      }
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) {
      const float v = k < 3 ? wave_min(part[k]) : wave_max(part[k]);
      if (lane == who) box[k] = k < 3 ? fminf(box[k], v) : fmaxf(box[k], v);
    }
  }
  if (span) {
    const int p = it.pint[i];
    if (p < 0) put_root(it.root, box, box + 3);
    else put_child_box(it.nodes + p, it.nodes[p].d.x == i, box, box + 3);
  }
}

__global__ void __launch_bounds__(kBS) k_bvh_refit_tile(RefitItem it) {
  if (it.done && *it.done) return;
  refit_tile(it, blockIdx.x);
}

__global__ void __launch_bounds__(kBS) k_bvh_refit_span(RefitItem it) {
  if (it.done && *it.done) return;
  refit_span(it, blockIdx.x);
}

// the trees of a batched build, one launch a stage
__global__ void __launch_bounds__(kBS) k_bvh_refit_tile_many(const RefitItem* __restrict__ items,
                                                             int n) {
  const RefitItem& it = refit_item(items, n);
  refit_tile(it, (int)(blockIdx.x - it.blk0));
}

__global__ void __launch_bounds__(kBS) k_bvh_refit_span_many(const RefitItem* __restrict__ items,
                                                             int n) {
  const RefitItem& it = refit_item(items, n);
  refit_span(it, (int)(blockIdx.x - it.blk0));
}

__device__ __forceinline__ void bvh_wide_node(const BvhNode* __restrict__ nodes,
                                              const int* __restrict__ pint, int n,
                                              BvhWide* __restrict__ wide, int i) {
  int depth = 0;
  int p = pint[i];
  for (int guard = 0; p >= 0 && p < n - 1 && guard < n; ++guard) {
    ++depth;
    p = pint[p];
  }
  if (depth & 1) return;
  float lo[4][3], hi[4][3];
  int ref[4];
  int m = 0;
  const BvhNode& N = nodes[i];
  const int kids[2] = {N.d.x, N.d.y};
  for (int side = 0; side < 2; ++side) {
    const int c = kids[side];
    if (c < 0 || c >= n - 1) {  // a leaf (an out-of-range reference is kept for the guard)
      const float* q = (const float*)&N + 6 * side;
      for (int k = 0; k < 3; ++k) {
        lo[m][k] = q[k];
        hi[m][k] = q[3 + k];
      }
      ref[m++] = c;
    } else {
      const BvhNode& C = nodes[c];
      const float* q = (const float*)&C;
      for (int g = 0; g < 2; ++g) {
        for (int k = 0; k < 3; ++k) {
          lo[m][k] = q[6 * g + k];
          hi[m][k] = q[6 * g + 3 + k];
        }
        ref[m++] = g == 0 ? C.d.x : C.d.y;
      }
    }
  }
  for (; m < 4; ++m) {
    for (int k = 0; k < 3; ++k) {
      lo[m][k] = INFINITY;
      hi[m][k] = INFINITY;
    }
    ref[m] = petch::kWideEmpty;
  }
  BvhWide w;
  w.lox = make_float4(lo[0][0], lo[1][0], lo[2][0], lo[3][0]);
  w.hix = make_float4(hi[0][0], hi[1][0], hi[2][0], hi[3][0]);
  w.loy = make_float4(lo[0][1], lo[1][1], lo[2][1], lo[3][1]);
  w.hiy = make_float4(hi[0][1], hi[1][1], hi[2][1], hi[3][1]);
  w.loz = make_float4(lo[0][2], lo[1][2], lo[2][2], lo[3][2]);
  w.hiz = make_float4(hi[0][2], hi[1][2], hi[2][2], hi[3][2]);
  w.ref = make_int4(ref[0], ref[1], ref[2], ref[3]);
  w.pad = make_int4(0, 0, 0, 0);
  wide[i] = w;
}

__global__ void k_bvh_wide(const BvhNode* __restrict__ nodes, const int* __restrict__ pint, int n,
                           BvhWide* __restrict__ wide) {
  int i = blockIdx.x * kBS + threadIdx.x;
  if (i < n - 1) bvh_wide_node(nodes, pint, n, wide, i);
}

// The Morton-tree builds of many meshes (the features of a batched step) side by side: one
// launch per stage for all of them. Item t owns the workgroups [fblk0[t], fblk0[t+1]) of the
// launches over faces and [nblk0[t], nblk0[t+1]) of those over internal nodes; every stage runs
// the same device code as the single build, so the trees are the same.
struct BuildItem {
  const float* verts;
  const int* faces;
  int nf, nfb;               // faces, and workgroups over them
  Work w;
  BvhNode* nodes;
  BvhWide* wide;
  float4* tris;
  long long fblk0, nblk0;
};

__device__ __forceinline__ int build_item_of(const BuildItem* __restrict__ it, int n, bool nodes) {
  int lo = 0, hi = n - 1;
  const long long b = blockIdx.x;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if ((nodes ? it[mid].nblk0 : it[mid].fblk0) <= b) lo = mid; else hi = mid - 1;
  }
  return lo;
}

__global__ void __launch_bounds__(kBS) k_bvh_prep_many(const BuildItem* __restrict__ items, int n) {
  const BuildItem& it = items[build_item_of(items, n, false)];
  bvh_prep_block(it.verts, it.faces, it.nf, it.w.cen, it.w.part, (int)(blockIdx.x - it.fblk0));
}

// one workgroup per item: the scene bounds, and the traversal error flag cleared
__global__ void __launch_bounds__(kBS) k_bvh_bounds_many(const BuildItem* __restrict__ items) {
  const BuildItem& it = items[blockIdx.x];
  bvh_bounds_wg(it.w.part, it.nfb, it.w.scene);
  if (threadIdx.x == 0) *it.w.err = 0;
}

__global__ void k_bvh_morton_many(const BuildItem* __restrict__ items, int n) {
  const BuildItem& it = items[build_item_of(items, n, false)];
  const int f = (int)(blockIdx.x - it.fblk0) * kBS + threadIdx.x;
  if (f < it.nf) bvh_morton_face(it.w.cen, it.w.scene, it.w.keys, it.w.vals, f);
}

// the leaves in Morton order
__global__ void k_bvh_leaves_many(const BuildItem* __restrict__ items, int n) {
  const BuildItem& it = items[build_item_of(items, n, false)];
  const int f = (int)(blockIdx.x - it.fblk0) * kBS + threadIdx.x;
  if (f < it.nf) bvh_leaf(it.verts, it.faces, it.w.vals, it.tris, f);
}

__global__ void k_bvh_karras_many(const BuildItem* __restrict__ items, int n) {
  const BuildItem& it = items[build_item_of(items, n, true)];
  const int i = (int)(blockIdx.x - it.nblk0) * kBS + threadIdx.x;
  if (i < it.nf - 1) bvh_karras_node(it.w.keys, it.nf, it.nodes, it.w.pint, it.w.pleaf, i);
}

__global__ void k_bvh_wide_many(const BuildItem* __restrict__ items, int n) {
  const BuildItem& it = items[build_item_of(items, n, true)];
  const int i = (int)(blockIdx.x - it.nblk0) * kBS + threadIdx.x;
  if (i < it.nf - 1) bvh_wide_node(it.nodes, it.w.pint, it.nf, it.wide, i);
}

// Surface area of the box lo..hi (0 for an inverted box).
__device__ __forceinline__ float box_area(const float* lo, const float* hi) {
  const float x = fmaxf(hi[0] - lo[0], 0.f), y = fmaxf(hi[1] - lo[1], 0.f),
              z = fmaxf(hi[2] - lo[2], 0.f);
  return x * y + y * z + z * x;
}

constexpr int kWideBS = 1024;
constexpr int kWideMaxLevels = 96;
// The clustering and the area-driven collapse add ~0.28 ms to a build of 47k faces and save ~7 %
// of the time of traces on the tree (on surfaces with a grid the traces walk that instead). Unless
// the caller chose a quality (petch_bvh_set_quality), meshes below this size get the Morton tree
// and the per-level grandchildren rule (one parallel pass).
constexpr int kWideSahMinFaces = 32768;

// The wide node of binary node b: its two children and, twice, the inner child of largest surface
// area replaced by that child's two children (a leaf stays a leaf), so big boxes are split first.
// The wide node is stored at its binary node's index; ref: its children; returns their number.
__device__ __forceinline__ int wide_sah_node(const BvhNode* __restrict__ nodes, int n,
                                             BvhWide* __restrict__ wide, int b, int ref[4]) {
  float lo[4][3], hi[4][3];
  const float* q = (const float*)(nodes + b);
  for (int side = 0; side < 2; ++side) {
    for (int k = 0; k < 3; ++k) {
      lo[side][k] = q[6 * side + k];
      hi[side][k] = q[6 * side + 3 + k];
    }
    ref[side] = side == 0 ? nodes[b].d.x : nodes[b].d.y;
  }
  int cnt = 2;
#pragma unroll
  for (int grow = 0; grow < 2; ++grow) {
    int best = -1;
    float best_a = -1.f;
#pragma unroll
    for (int c = 0; c < 2 + grow; ++c) {
      if (ref[c] < 0 || ref[c] >= n - 1) continue;   // leaves (and bad refs) stay
      const float a = box_area(lo[c], hi[c]);
      if (a > best_a) {
        best_a = a;
        best = c;
      }
    }
    const int r = best == 0 ? ref[0] : best == 1 ? ref[1] : best == 2 ? ref[2] : -1;
    const int at = 2 + grow;
    for (int k = 0; k < 3; ++k) {
      lo[at][k] = INFINITY;
      hi[at][k] = INFINITY;
    }
    ref[at] = petch::kWideEmpty;
    if (r >= 0) {
      const BvhNode g = nodes[r];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        if (c == best) {
          lo[c][0] = g.a.x; lo[c][1] = g.a.y; lo[c][2] = g.a.z;
          hi[c][0] = g.a.w; hi[c][1] = g.b.x; hi[c][2] = g.b.y;
          ref[c] = g.d.x;
        }
      }
      lo[at][0] = g.b.z; lo[at][1] = g.b.w; lo[at][2] = g.c.x;
      hi[at][0] = g.c.y; hi[at][1] = g.c.z; hi[at][2] = g.c.w;
      ref[at] = g.d.y;
      ++cnt;
    }
  }
  BvhWide w;
  w.lox = make_float4(lo[0][0], lo[1][0], lo[2][0], lo[3][0]);
  w.hix = make_float4(hi[0][0], hi[1][0], hi[2][0], hi[3][0]);
  w.loy = make_float4(lo[0][1], lo[1][1], lo[2][1], lo[3][1]);
  w.hiy = make_float4(hi[0][1], hi[1][1], hi[2][1], hi[3][1]);
  w.loz = make_float4(lo[0][2], lo[1][2], lo[2][2], lo[3][2]);
  w.hiz = make_float4(hi[0][2], hi[1][2], hi[2][2], hi[3][2]);
  w.ref = make_int4(ref[0], ref[1], ref[2], ref[3]);
  w.pad = make_int4(0, 0, 0, 0);
  wide[b] = w;
  return cnt;
}

// Top-down collapse into 4-wide nodes, level by level: the inner children of a level's wide nodes
// form the next level. Each level is a chain of three dependent fetches a node, so one workgroup
// (330 us for 47k faces) is bound by how many nodes it has in flight. Here it does the levels
// below kWideSplit nodes (k_wide_levels with first = true); each workgroup of k_wide_subtrees, one
// wavefront, then takes its share of the next level down to the leaves, with its lists in LDS.
// What finds no place there goes to a list in memory that a last launch of k_wide_levels works
// through (empty unless a subtree is very unbalanced). 28 + 13 + 2 us for the 47k faces.
// A tree deeper than kWideMaxLevels wide levels leaves error flag 3 (never for Morton trees,
// whose depth is bounded by the code length plus the index tie-break).
constexpr int kWideSplit = 1024;
constexpr int kWideList = 1024;   // nodes of one subtree level held in LDS

__global__ void __launch_bounds__(kWideBS) k_wide_levels(const BvhNode* __restrict__ nodes,
                                                         int n, BvhWide* __restrict__ wide,
                                                         int* __restrict__ list_a,
                                                         int* __restrict__ list_b,
                                                         int* __restrict__ hdr,
                                                         int* __restrict__ err, bool first) {
  __shared__ int cnt_cur, cnt_next;
  const int side = first ? 0 : hdr[H_SIDE] ^ 1;   // the second launch's list: the overflow
  if (threadIdx.x == 0) {
    if (first) list_a[0] = 0;
    cnt_cur = first ? 1 : hdr[H_OVER];
    cnt_next = 0;
  }
  __syncthreads();
  int* cur = side ? list_b : list_a;
  int* nxt = side ? list_a : list_b;
  int flip = side, level = first ? 0 : hdr[H_OVER_LEVEL];
  for (; level < kWideMaxLevels; ++level) {
    const int m = cnt_cur;
    if (m == 0 || (first && m >= kWideSplit)) break;
    for (int t = threadIdx.x; t < m; t += kWideBS) {
      int ref[4];
      const int cnt = wide_sah_node(nodes, n, wide, cur[t], ref);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if (c < cnt && ref[c] >= 0 && ref[c] < n - 1) {
          const int slot = atomicAdd(&cnt_next, 1);
          if (slot < n - 1) nxt[slot] = ref[c];
        }
      }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      cnt_cur = cnt_next < n - 1 ? cnt_next : n - 1;
      cnt_next = 0;
    }
    __syncthreads();
    int* tmp = cur;
    cur = nxt;
    nxt = tmp;
    flip ^= 1;
  }
  if (threadIdx.x == 0) {
    if (first) {
      hdr[H_COUNT] = cnt_cur;
      hdr[H_SIDE] = flip;
      hdr[H_LEVEL] = level;
      hdr[H_OVER] = 0;
      hdr[H_OVER_LEVEL] = 0;
    }
    if (cnt_cur > 0 && level >= kWideMaxLevels && err) *err = 3;
  }
}

__global__ void __launch_bounds__(64) k_wide_subtrees(const BvhNode* __restrict__ nodes, int n,
                                                      BvhWide* __restrict__ wide,
                                                      int* __restrict__ list_a,
                                                      int* __restrict__ list_b,
                                                      int* __restrict__ hdr,
                                                      int* __restrict__ err) {
  __shared__ int lists[2][kWideList];
  __shared__ int cnt_next;
  const int total = hdr[H_COUNT], first_level = hdr[H_LEVEL];
  const int* from = hdr[H_SIDE] ? list_b : list_a;
  int* over = hdr[H_SIDE] ? list_a : list_b;
  if (first_level >= kWideMaxLevels) return;
  // (a level below kWideSplit nodes has fewer than 4 kWideSplit children, a few each workgroup)
  int m = 0;
  for (int t = blockIdx.x; t < total && m < kWideList; t += gridDim.x) ++m;
  for (int t = threadIdx.x; t < m; t += 64) lists[0][t] = from[blockIdx.x + t * gridDim.x];
  if (threadIdx.x == 0) cnt_next = 0;
  __syncthreads();
  int level = first_level;
  for (; m > 0 && level < kWideMaxLevels; ++level) {
    const int* cur = lists[(level - first_level) & 1];
    int* nxt = lists[((level - first_level) & 1) ^ 1];
    for (int t = threadIdx.x; t < m; t += 64) {
      int ref[4];
      const int cnt = wide_sah_node(nodes, n, wide, cur[t], ref);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if (c < cnt && ref[c] >= 0 && ref[c] < n - 1) {
          const int slot = atomicAdd(&cnt_next, 1);
          if (slot < kWideList) {
            nxt[slot] = ref[c];
          } else {
            const int o = atomicAdd(hdr + H_OVER, 1);
            if (o < n - 1) over[o] = ref[c];
            atomicMax(hdr + H_OVER_LEVEL, level + 1);
          }
        }
      }
    }
    __syncthreads();
    m = cnt_next < kWideList ? cnt_next : kWideList;
    __syncthreads();
    if (threadIdx.x == 0) cnt_next = 0;
    __syncthreads();
  }
  if (threadIdx.x == 0 && m > 0 && err) *err = 3;
}

// ---------------------------------------------------------------------------- PLOC
// Parallel locally-ordered clustering (Meister & Bittner, IEEE TVCG 2018) over the Morton-sorted
// leaves: every cluster finds, within kPlocRadius places of it in Morton order, the cluster whose
// union box has the smallest surface area; mutual nearest pairs merge into a new internal node;
// the survivors are compacted in order, and the rounds repeat until one cluster is left. Node
// indices count down from n-2, so the last merge is the root, node 0, as in the Morton tree.
// Builds a tree closer to a surface-area-optimal one than the Morton split. The first rounds
// are one grid-wide launch each; the remaining few thousand clusters are finished by one
// workgroup with the clusters in LDS. If the rounds do not get down to one cluster the Morton
// tree is built after all.
constexpr int kPlocRadius = 16;
constexpr int kPlocTile = kBS;          // clusters of one workgroup of a grid-wide round
constexpr int kPlocMaxRounds = 40;      // grid-wide rounds at most
constexpr int kPlocFinishRounds = 512;  // then one workgroup finishes the (small) rest
constexpr int kFinBS = 1024;
constexpr int kFinCap = 2048;           // clusters that the finishing workgroup holds in LDS

// The clusters between two rounds: tile t's survivors, in order, at [t kPlocTile, + cnt[t]), so
// that no round needs a compaction of its own; sup[u] sums the counts of 256 tiles.
struct PlocSet {
  float4 *lo, *hi;  // cluster boxes
  int* ref;         // >= 0 node, < 0 leaf ~slot
  int *cnt, *sup;
};

struct PlocWork {
  PlocSet set[2];
  int* sup;         // the sums of every round, ns each
  int* nn;
  int* alloc;       // merges so far
  int tiles, ns;
};

size_t ploc_tiles(int nf) { return ((size_t)nf + kPlocTile - 1) / kPlocTile; }

size_t ploc_bytes(int nf) {
  const size_t t = ploc_tiles(nf), ns = (t + 255) / 256;
  return t * kPlocTile * (2 * 36 + 4) + 2 * t * 4 + (kPlocMaxRounds + 1) * ns * 4 + 64;
}

PlocWork ploc_carve(void* base, int nf) {
  PlocWork w;
  const size_t t = ploc_tiles(nf), cap = t * kPlocTile, ns = (t + 255) / 256;
  char* p = (char*)base;
  for (PlocSet& q : w.set) {
    q.lo = (float4*)p; p += cap * 16;
    q.hi = (float4*)p; p += cap * 16;
  }
  for (PlocSet& q : w.set) {
    q.ref = (int*)p; p += cap * 4;
    q.cnt = (int*)p; p += t * 4;
    q.sup = nullptr;
  }
  w.nn = (int*)p; p += cap * 4;
  w.sup = (int*)p; p += (kPlocMaxRounds + 1) * ns * 4;
  w.alloc = (int*)p;
  w.tiles = (int)t;
  w.ns = (int)ns;
  return w;
}

__device__ __forceinline__ float union_area(float4 alo, float4 ahi, float4 blo, float4 bhi) {
  const float x = fmaxf(ahi.x, bhi.x) - fminf(alo.x, blo.x);
  const float y = fmaxf(ahi.y, bhi.y) - fminf(alo.y, blo.y);
  const float z = fmaxf(ahi.z, bhi.z) - fminf(alo.z, blo.z);
  return x * y + y * z + z * x;
}

// The leaves as clusters; sup: the first round's sums, then `rounds` rounds' to be added to.
__global__ void __launch_bounds__(kBS) k_ploc_init(const float4* __restrict__ tris, int n,
                                                   PlocSet out, int tiles, int ns, int rounds,
                                                   int* __restrict__ sup, int* __restrict__ alloc) {
  const int i = blockIdx.x * kBS + threadIdx.x;
  if (i == 0) *alloc = 0;
  for (long long k = i; k < (long long)(rounds + 1) * ns; k += (long long)gridDim.x * kBS) {
    const long long left = n - k * 256 * kPlocTile;
    sup[k] = k >= ns ? 0 : (int)(left < 256 * kPlocTile ? left : 256 * kPlocTile);
  }
  if (i < tiles) out.cnt[i] = n - i * kPlocTile < kPlocTile ? n - i * kPlocTile : kPlocTile;
  if (i >= n) return;
  const float4 a = tris[3 * i], b = tris[3 * i + 1], c = tris[3 * i + 2];
  out.ref[i] = ~i;
  out.lo[i] = make_float4(fminf(a.x, fminf(b.x, c.x)), fminf(a.y, fminf(b.y, c.y)),
                          fminf(a.z, fminf(b.z, c.z)), 0.f);
  out.hi[i] = make_float4(fmaxf(a.x, fmaxf(b.x, c.x)), fmaxf(a.y, fmaxf(b.y, c.y)),
                          fmaxf(a.z, fmaxf(b.z, c.z)), 0.f);
}

// The nearest cluster of cluster q among [0, count) (lo, hi: cluster `first` onwards), by lane l
// of the `sub` lanes that share the search; ties keep the smaller index.
__device__ __forceinline__ int ploc_nearest(const float4* lo, const float4* hi, int first, int q,
                                            int count, int l, int sub) {
  const float4 qlo = lo[q - first], qhi = hi[q - first];
  int best = -1;
  float best_a = INFINITY;
  const int j0 = q - kPlocRadius < 0 ? 0 : q - kPlocRadius;
  const int j1 = q + kPlocRadius > count - 1 ? count - 1 : q + kPlocRadius;
#pragma unroll 4
  for (int j = j0 + l; j <= j1; j += sub) {
    const float a = union_area(qlo, qhi, lo[j - first], hi[j - first]);
    if (j != q && a < best_a) {
      best_a = a;
      best = j;
    }
  }
  for (int d = sub >> 1; d >= 1; d >>= 1) {
    const float oa = __shfl_xor(best_a, d, 64);
    const int oj = __shfl_xor(best, d, 64);
    if (oj >= 0 && (best < 0 || oa < best_a || (oa == best_a && oj < best))) {
      best_a = oa;
      best = oj;
    }
  }
  return best;
}

__device__ __forceinline__ void ploc_node(BvhNode* nd, float4 l0, float4 l1, float4 r0, float4 r1,
                                          int left, int right) {
  nd->a = make_float4(l0.x, l0.y, l0.z, l1.x);
  nd->b = make_float4(l1.y, l1.z, r0.x, r0.y);
  nd->c = make_float4(r0.z, r1.x, r1.y, r1.z);
  nd->d = make_int4(left, right, 0, 0);
}

__device__ __forceinline__ float4 min4(float4 a, float4 b) {
  return make_float4(fminf(a.x, b.x), fminf(a.y, b.y), fminf(a.z, b.z), 0.f);
}
__device__ __forceinline__ float4 max4(float4 a, float4 b) {
  return make_float4(fmaxf(a.x, b.x), fmaxf(a.y, b.y), fmaxf(a.z, b.z), 0.f);
}

// One round, one launch: workgroup b takes the clusters [b kPlocTile, (b + 1) kPlocTile) of all
// that are left. It finds where they lie from the tiles' counts, stages them with 2 kPlocRadius
// neighbours each side in LDS, finds the nearest of its own and of kPlocRadius each side (which
// tells whether its own pairs are mutual), merges, and leaves its survivors packed in its tile.
// 10 us a round at 47k faces, half of it the chain of fetches that finds the clusters (25 us as
// nearest, merge, scan and scatter launches through memory).
// A full tile keeps at least 120 of its 256 (at most 16 go to the tile before it, the others in
// pairs), so the 320 staged clusters lie in at most 5 tiles.
constexpr int kPlocWin = kPlocTile + 4 * kPlocRadius;   // and threads: one a staged cluster
constexpr int kPlocSpan = 8;
__global__ void __launch_bounds__(kPlocWin) k_ploc_round(PlocSet in, PlocSet out, int tiles, int ns,
                                                    BvhNode* __restrict__ nodes,
                                                    int* __restrict__ alloc, int n) {
  __shared__ float4 s_lo[kPlocWin], s_hi[kPlocWin];
  __shared__ int s_ref[kPlocWin], s_nn[kPlocTile + 2 * kPlocRadius];
  __shared__ int s_at[3], s_pre[kPlocSpan + 1];
  const int tid = threadIdx.x, b0 = blockIdx.x * kPlocTile;
  const int start = b0 < 2 * kPlocRadius ? 0 : b0 - 2 * kPlocRadius;
  int total = 0;
  for (int c = 0; c < ns; c += kPlocWin) {
    const int v = c + tid < ns ? in.sup[c + tid] : 0;
    int sum;
    const int ex = total + petch::block_excl_scan<kPlocWin>(v, sum);
    if (start >= ex && start < ex + v) {
      s_at[0] = c + tid;
      s_at[1] = ex;
    }
    total += sum;
  }
  if (b0 >= total) {
    if (tid == 0) out.cnt[blockIdx.x] = 0;
    return;
  }
  __syncthreads();
  {
    const int t = s_at[0] * 256 + tid;
    const int v = tid < 256 && t < tiles ? in.cnt[t] : 0;
    int sum;
    const int ex = s_at[1] + petch::block_excl_scan<kPlocWin>(v, sum);
    if (start >= ex && start < ex + v) {
      s_at[2] = t;
      s_pre[0] = ex;
    }
  }
  __syncthreads();
  const int t0 = s_at[2];
  if (tid == 0) {
#pragma unroll
    for (int k = 0; k < kPlocSpan; ++k)
      s_pre[k + 1] = s_pre[k] + (t0 + k < tiles ? in.cnt[t0 + k] : 0);
  }
  __syncthreads();
  const int past = b0 + kPlocTile + 2 * kPlocRadius, end = total < past ? total : past;
  if (const int q = start + tid; q < end) {
    int k = 0;
    while (k < kPlocSpan - 1 && q >= s_pre[k + 1]) ++k;
    const int src = (t0 + k) * kPlocTile + (q - s_pre[k]);
    if (src < tiles * kPlocTile) {
      s_lo[q - start] = in.lo[src];
      s_hi[q - start] = in.hi[src];
      s_ref[q - start] = in.ref[src];
    }
  }
  __syncthreads();
  const int n0 = b0 < kPlocRadius ? 0 : b0 - kPlocRadius;
  const int n1 = total < b0 + kPlocTile + kPlocRadius ? total : b0 + kPlocTile + kPlocRadius;
  if (const int q = n0 + tid; q < n1)
    s_nn[q - n0] = ploc_nearest(s_lo, s_hi, start, q, total, 0, 1);
  __syncthreads();
  const int i = b0 + tid;
  const bool own = tid < kPlocTile && i < total;
  const int j = own ? s_nn[i - n0] : -1;
  const bool mutual = j >= 0 && s_nn[j - n0] == i;
  const bool merge = mutual && i < j;                 // the smaller index builds the node
  const bool keep = own && !(mutual && i > j);  // and keeps its place
  int sum;
  const int ex = petch::block_excl_scan<kPlocWin>((keep ? 1 : 0) | (merge ? 0x10000 : 0), sum);
  if (tid == 0) {
    out.cnt[blockIdx.x] = sum & 0xffff;
    atomicAdd(out.sup + (blockIdx.x >> 8), sum & 0xffff);
    s_at[0] = atomicAdd(alloc, sum >> 16);
  }
  __syncthreads();
  if (!keep) return;
  float4 lo = s_lo[i - start], hi = s_hi[i - start];
  int ref = s_ref[i - start];
  if (merge) {
    const int node = (n - 2) - (s_at[0] + (ex >> 16));
    const float4 rlo = s_lo[j - start], rhi = s_hi[j - start];
    if (node >= 0) ploc_node(nodes + node, lo, hi, rlo, rhi, ref, s_ref[j - start]);
    lo = min4(lo, rlo);
    hi = max4(hi, rhi);
    ref = node;
  }
  const int o = b0 + (ex & 0xffff);   // at most 256 kept: within the tile
  out.lo[o] = lo;
  out.hi[o] = hi;
  out.ref[o] = ref;
}

// Rounds of one workgroup over clusters [0, count) at lo, hi, ref, compacted in place, until at
// most `stop` are left or `rounds` is spent. With few clusters several lanes share a search.
__device__ __forceinline__ void ploc_rounds(float4* lo, float4* hi, int* ref, int* nn, int& count,
                                            int stop, int& rounds, int& merged, BvhNode* nodes,
                                            int n) {
  const int tid = threadIdx.x;
  for (; rounds > 0 && count > stop; --rounds) {
    int sub = 16;
    while (sub > 1 && count * sub > kFinBS) sub >>= 1;
    for (int i = tid / sub; i < count; i += kFinBS / sub) {
      const int j = ploc_nearest(lo, hi, 0, i, count, tid % sub, sub);
      if (tid % sub == 0) nn[i] = j;
    }
    __syncthreads();
    int carry = 0;
    for (int base = 0; base < count; base += kFinBS) {
      const int i = base + tid;
      const int j = i < count ? nn[i] : -1;
      const bool mutual = j >= 0 && nn[j] == i;
      const bool merge = mutual && i < j;
      const bool keep = i < count && !(mutual && i > j);
      float4 l0, l1, r0, r1;
      int ri = 0, rj = 0;
      if (keep) {
        l0 = lo[i];
        l1 = hi[i];
        ri = ref[i];
      }
      if (merge) {
        r0 = lo[j];
        r1 = hi[j];
        rj = ref[j];
      }
      // (the scan's barriers part these reads from the writes below, which stay below base +
      // kFinBS: nothing that a later pass reads)
      int sum;
      const int ex = petch::block_excl_scan<kFinBS>((keep ? 1 : 0) | (merge ? 0x10000 : 0), sum);
      if (merge) {
        const int node = (n - 2) - (merged + (ex >> 16));
        if (node >= 0) ploc_node(nodes + node, l0, l1, r0, r1, ri, rj);
        l0 = min4(l0, r0);
        l1 = max4(l1, r1);
        ri = node;
      }
      if (keep) {
        const int k = carry + (ex & 0xffff);
        lo[k] = l0;
        hi[k] = l1;
        ref[k] = ri;
      }
      carry += sum & 0xffff;
      merged += sum >> 16;
    }
    __syncthreads();
    count = carry;
  }
}

// The remaining rounds in one workgroup, the clusters packed into LDS (through memory, at buf,
// while there are more than fit). Its 27 rounds are bound by LDS latency and barriers: 93 us for
// 47k faces (685 through memory, from 9k clusters on). *done: the tree is complete, and root its
// box.
__global__ void __launch_bounds__(kFinBS) k_ploc_finish(PlocSet in, PlocSet buf, int tiles, int ns,
                                                        int* __restrict__ nn,
                                                        BvhNode* __restrict__ nodes,
                                                        const int* __restrict__ alloc, int n,
                                                        int* __restrict__ done,
                                                        float* __restrict__ root) {
  __shared__ float4 s_lo[kFinCap], s_hi[kFinCap];
  __shared__ int s_ref[kFinCap], s_nn[kFinCap];
  __shared__ int s_pre[kFinBS], s_cnt[kFinBS];
  const int tid = threadIdx.x;
  int count = 0;
  for (int k = tid; k < ns; k += kFinBS) count += in.sup[k];
  count = petch::block_sum<kFinBS>(count);
  const bool fits = count <= kFinCap;
  int carry = 0;
  for (int c = 0; c < tiles && carry < count; c += kFinBS) {
    const int v = c + tid < tiles ? in.cnt[c + tid] : 0;
    int sum;
    s_pre[tid] = carry + petch::block_excl_scan<kFinBS>(v, sum);
    s_cnt[tid] = v;
    carry += sum;
    __syncthreads();
    for (int t = tid / kPlocTile; t < kFinBS && s_pre[t] < carry; t += kFinBS / kPlocTile) {
      const int k = tid % kPlocTile;
      if (k < s_cnt[t]) {
        const int src = (c + t) * kPlocTile + k, o = s_pre[t] + k;
        if (fits) {
          s_lo[o] = in.lo[src];
          s_hi[o] = in.hi[src];
          s_ref[o] = in.ref[src];
        } else {
          buf.lo[o] = in.lo[src];
          buf.hi[o] = in.hi[src];
          buf.ref[o] = in.ref[src];
        }
      }
    }
    __syncthreads();
  }
  int rounds = kPlocFinishRounds, merged = *alloc;
  if (!fits) {
    ploc_rounds(buf.lo, buf.hi, buf.ref, nn, count, kFinCap, rounds, merged, nodes, n);
    if (count <= kFinCap) {
      for (int k = tid; k < count; k += kFinBS) {
        s_lo[k] = buf.lo[k];
        s_hi[k] = buf.hi[k];
        s_ref[k] = buf.ref[k];
      }
    }
    __syncthreads();
  }
  if (count <= kFinCap) ploc_rounds(s_lo, s_hi, s_ref, s_nn, count, 1, rounds, merged, nodes, n);
  if (tid == 0) {
    const bool whole = count == 1 && merged == n - 1;
    *done = whole;
    if (whole) {
      root[0] = s_lo[0].x; root[1] = s_lo[0].y; root[2] = s_lo[0].z;
      root[3] = s_hi[0].x; root[4] = s_hi[0].y; root[5] = s_hi[0].z;
    }
  }
}

__global__ void k_query_ray(BvhView b, const float* __restrict__ o, const float* __restrict__ d,
                            int n, float tmax, int* __restrict__ face, float* __restrict__ tout) {
  int i = blockIdx.x * kBS + threadIdx.x;
  if (i >= n) return;
  petch::Hit h = petch::bvh_closest_hit(b, petch::v3(o[3 * i], o[3 * i + 1], o[3 * i + 2]),
                                        petch::v3(d[3 * i], d[3 * i + 1], d[3 * i + 2]), tmax);
  face[i] = h.face;
  if (tout) tout[i] = h.face >= 0 ? h.t : -1.f;
}

__global__ void k_query_ray_walk(petch::GridView g, BvhView tree, const float* __restrict__ o,
                                 const float* __restrict__ d, int n, float tmax,
                                 int* __restrict__ face, float* __restrict__ tout) {
  int i = blockIdx.x * kBS + threadIdx.x;
  if (i >= n) return;
  petch::Hit h = petch::walk_closest_hit(g, tree, petch::v3(o[3 * i], o[3 * i + 1], o[3 * i + 2]),
                                         petch::v3(d[3 * i], d[3 * i + 1], d[3 * i + 2]), tmax);
  face[i] = h.face;
  if (tout) tout[i] = h.face >= 0 ? h.t : -1.f;
}

__global__ void k_query_point(BvhView b, const float* __restrict__ p, int n, float maxd,
                              int* __restrict__ face, float* __restrict__ dist) {
  int i = blockIdx.x * kBS + threadIdx.x;
  if (i >= n) return;
  petch::ScratchStack stk;
  petch::PointHit h =
      petch::bvh_closest_point(b, petch::v3(p[3 * i], p[3 * i + 1], p[3 * i + 2]), maxd, stk);
  face[i] = h.face;
  if (dist) dist[i] = h.face >= 0 ? sqrtf(h.d2) : -1.f;
}

}  // namespace

BvhView petch_bvh_view(const petch_bvh* b) {
  BvhView v;
  v.nodes = (const BvhNode*)b->nodes;
  v.wide = (const BvhWide*)b->wide;
  v.tris = (const float4*)b->tris;
  v.nf = b->nf;
  v.err = b->work ? carve(b->work, b->cap_f).err : nullptr;
  v.root = (b->work && b->nf > 1) ? carve(b->work, b->cap_f).root : nullptr;
  return v;
}

int* petch_bvh_err(const petch_bvh* b) { return b->work ? carve(b->work, b->cap_f).err : nullptr; }

extern "C" int petch_bvh_create(petch_ctx* ctx, petch_bvh** out) {
  PETCH_ARG(ctx, ctx && out, "bvh_create: null pointer");
  petch_bvh* b = (petch_bvh*)calloc(1, sizeof(petch_bvh));
  if (!b) return petch_set_error(ctx, PETCH_E_HIP, "bvh_create: out of host memory");
  b->device = ctx->device;
  b->quality = -1;
  *out = b;
  return PETCH_OK;
}

extern "C" int petch_bvh_set_quality(petch_ctx* ctx, petch_bvh* b, int quality) {
  PETCH_ARG(ctx, ctx && b, "bvh_set_quality: null pointer");
  PETCH_ARG(ctx, quality >= -1 && quality <= 2, "bvh_set_quality: quality %d not in -1..2",
            quality);
  b->quality = quality;
  return PETCH_OK;
}

extern "C" int petch_bvh_destroy(petch_ctx* ctx, petch_bvh* b) {
  if (!b) return PETCH_OK;
  if (ctx) (void)hipStreamSynchronize(ctx->stream);
  if (b->nodes) (void)hipFree(b->nodes);
  if (b->wide) (void)hipFree(b->wide);
  if (b->tris) (void)hipFree(b->tris);
  if (b->work) (void)hipFree(b->work);
  if (b->aux) (void)hipFree(b->aux);
  if (b->cells) (void)hipFree(b->cells);
  if (b->gtris) (void)hipFree(b->gtris);
  free(b);
  return PETCH_OK;
}

namespace {

// PLOC rounds over the leaves of b (tris already in Morton order) into b->nodes; *done, on the
// device, tells whether they hold a complete tree.
int ploc_build(petch_ctx* ctx, petch_bvh* b, int nf, int* done, float* root) {
  const size_t need = ploc_bytes(nf);
  if (b->aux_cap < need) {
    PETCH_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (b->aux) (void)hipFree(b->aux);
    b->aux = nullptr;
    b->aux_cap = 0;
    const size_t want = need + need / 2;
    PETCH_HIP(ctx, hipMalloc(&b->aux, want));
    b->aux_cap = want;
  }
  PlocWork p = ploc_carve(b->aux, nf);
  // the first round keeps about 0.57 of its clusters (most leaves pair up), each later one 0.81:
  // as many as bring them into the finishing workgroup's LDS
  int rounds = nf > kFinCap ? 1 : 0;
  for (long long c = nf * 9LL / 16; c > kFinCap && rounds < kPlocMaxRounds; c -= c * 3 / 16)
    ++rounds;
  const unsigned g = (unsigned)p.tiles;
  p.set[0].sup = p.sup;
  hipLaunchKernelGGL(k_ploc_init, dim3(g), dim3(kBS), 0, ctx->stream, (const float4*)b->tris, nf,
                     p.set[0], p.tiles, p.ns, rounds, p.sup, p.alloc);
  PETCH_LAUNCH_CHECK(ctx);
  for (int r = 0; r < rounds; ++r) {
    p.set[(r + 1) & 1].sup = p.sup + (size_t)(r + 1) * p.ns;
    hipLaunchKernelGGL(k_ploc_round, dim3(g), dim3(kPlocWin), 0, ctx->stream, p.set[r & 1],
                       p.set[(r + 1) & 1], p.tiles, p.ns, (BvhNode*)b->nodes, p.alloc, nf);
    PETCH_LAUNCH_CHECK(ctx);
  }
  hipLaunchKernelGGL(k_ploc_finish, dim3(1), dim3(kFinBS), 0, ctx->stream, p.set[rounds & 1],
                     p.set[(rounds + 1) & 1], p.tiles, p.ns, p.nn, (BvhNode*)b->nodes, p.alloc, nf,
                     done, root);
  PETCH_LAUNCH_CHECK(ctx);
  return PETCH_OK;
}

}  // namespace

namespace {

// Grows the BVH's device buffers to hold nf faces (they are never shrunk); a BVH that was never
// built gets a minimal set, so its error flag is valid. A regrowth waits for the stream and
// frees and allocates four buffers (hundreds of microseconds with the device idle), and an
// etching surface keeps growing, so the new capacity is twice the request.
int ensure_capacity(petch_ctx* ctx, petch_bvh* b, int nf) {
  if (nf > b->cap_f) {
    PETCH_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (b->nodes) (void)hipFree(b->nodes);
    if (b->wide) (void)hipFree(b->wide);
    if (b->tris) (void)hipFree(b->tris);
    if (b->work) (void)hipFree(b->work);
    b->nodes = b->wide = b->tris = b->work = nullptr;
    int cap = nf > (0x7fffffff - 1024) / 2 ? nf : 2 * nf + 1024;
    PETCH_HIP(ctx, hipMalloc(&b->nodes, (size_t)cap * sizeof(BvhNode)));
    PETCH_HIP(ctx, hipMalloc(&b->wide, (size_t)cap * sizeof(BvhWide)));
    PETCH_HIP(ctx, hipMalloc(&b->tris, (size_t)cap * 48));
    PETCH_HIP(ctx, hipMalloc(&b->work, work_bytes(cap)));
    b->cap_f = cap;
  }
  if (b->cap_f == 0) {  // never built: keep a valid error flag
    int cap = 256;
    PETCH_HIP(ctx, hipMalloc(&b->nodes, (size_t)cap * sizeof(BvhNode)));
    PETCH_HIP(ctx, hipMalloc(&b->wide, (size_t)cap * sizeof(BvhWide)));
    PETCH_HIP(ctx, hipMalloc(&b->tris, (size_t)cap * 48));
    PETCH_HIP(ctx, hipMalloc(&b->work, work_bytes(cap)));
    b->cap_f = cap;
  }
  return PETCH_OK;
}

// The quality a build of nf faces gets.
int build_quality(const petch_bvh* b, int nf) {
  return b->quality >= 0 ? b->quality : (nf >= kWideSahMinFaces ? 2 : 0);
}

// Everything of a build up to the refit: buffers, centroids, Morton sort, leaves, then the
// clustered tree where the quality asks for it and the Morton tree's nodes where that one isn't
// complete. Returns the refit's item (n = nf; nothing to refit when nf < 2).
int build_prepare(petch_ctx* ctx, petch_bvh* b, const float* verts, const int* faces, int nv,
                  int nf, RefitItem* refit) {
  PETCH_ARG(ctx, ctx && b, "bvh_build: null pointer");
  PETCH_ARG(ctx, nf >= 0 && nv >= 0, "bvh_build: negative size");
  PETCH_ARG(ctx, nf == 0 || (verts && faces), "bvh_build: null mesh");
  b->nv = nv;
  b->nf = 0;
  b->grid_n[0] = 0;
  refit->n = 0;
  const int rc0 = ensure_capacity(ctx, b, nf);
  if (rc0 != PETCH_OK) return rc0;
  Work w = carve(b->work, b->cap_f);
  PETCH_HIP(ctx, hipMemsetAsync(w.err, 0, sizeof(int), ctx->stream));
  if (nf == 0) return PETCH_OK;
  unsigned g = petch_blocks(nf, kBS);
  hipLaunchKernelGGL(k_bvh_prep, dim3(g), dim3(kBS), 0, ctx->stream, verts, faces, nf, w.cen,
                     w.part);
  PETCH_LAUNCH_CHECK(ctx);
  hipLaunchKernelGGL(k_bvh_bounds, dim3(1), dim3(kBS), 0, ctx->stream, w.part, (int)g, w.scene);
  PETCH_LAUNCH_CHECK(ctx);
  hipLaunchKernelGGL(k_bvh_morton, dim3(g), dim3(kBS), 0, ctx->stream, w.cen, nf, w.scene, w.keys,
                     w.vals);
  PETCH_LAUNCH_CHECK(ctx);
  int rc = petch_radix_sort_pairs(ctx, w.keys, w.vals, w.ktmp, w.vtmp, nf, 30);
  if (rc != PETCH_OK) return rc;
  hipLaunchKernelGGL(k_bvh_leaves, dim3(g), dim3(kBS), 0, ctx->stream, verts, faces, w.vals, nf,
                     (float4*)b->tris);
  PETCH_LAUNCH_CHECK(ctx);
  if (nf > 1) {
    const int* done = nullptr;
    if (build_quality(b, nf) >= 2) {
      rc = ploc_build(ctx, b, nf, w.hdr + H_DONE, w.root);
      if (rc != PETCH_OK) return rc;
      done = w.hdr + H_DONE;
    }
    hipLaunchKernelGGL(k_bvh_karras, dim3(petch_blocks(nf - 1, kBS)), dim3(kBS), 0, ctx->stream,
                       w.keys, nf, (BvhNode*)b->nodes, w.pint, w.pleaf, done);
    PETCH_LAUNCH_CHECK(ctx);
    *refit = RefitItem{(const float4*)b->tris, (BvhNode*)b->nodes, w.pint, w.pleaf,
                       (float*)b->wide, w.root, done, nf, 0};
  }
  return PETCH_OK;
}

int build_refit(petch_ctx* ctx, const RefitItem& r) {
  if (r.n < 2) return PETCH_OK;
  const unsigned g = petch_blocks(r.n, kTile);
  hipLaunchKernelGGL(k_bvh_refit_tile, dim3(g), dim3(kBS), 0, ctx->stream, r);
  PETCH_LAUNCH_CHECK(ctx);
  if (g > 1) {
    hipLaunchKernelGGL(k_bvh_refit_span, dim3(g), dim3(kBS), 0, ctx->stream, r);
    PETCH_LAUNCH_CHECK(ctx);
  }
  return PETCH_OK;
}

// The rest of a build after the refit: the 4-wide nodes that the queries walk.
int build_finish(petch_ctx* ctx, petch_bvh* b, int nf) {
  if (nf > 1) {
    Work w = carve(b->work, b->cap_f);
    if (build_quality(b, nf) >= 1) {
      int *la = (int*)w.ktmp, *lb = (int*)w.vtmp;
      const BvhNode* nodes = (const BvhNode*)b->nodes;
      BvhWide* wide = (BvhWide*)b->wide;
      hipLaunchKernelGGL(k_wide_levels, dim3(1), dim3(kWideBS), 0, ctx->stream, nodes, nf, wide,
                         la, lb, w.hdr, w.err, true);
      PETCH_LAUNCH_CHECK(ctx);
      hipLaunchKernelGGL(k_wide_subtrees, dim3(kWideSplit), dim3(64), 0, ctx->stream, nodes, nf,
                         wide, la, lb, w.hdr, w.err);
      PETCH_LAUNCH_CHECK(ctx);
      hipLaunchKernelGGL(k_wide_levels, dim3(1), dim3(kWideBS), 0, ctx->stream, nodes, nf, wide,
                         la, lb, w.hdr, w.err, false);
    } else {
      hipLaunchKernelGGL(k_bvh_wide, dim3(petch_blocks(nf - 1, kBS)), dim3(kBS), 0, ctx->stream,
                         (const BvhNode*)b->nodes, w.pint, nf, (BvhWide*)b->wide);
    }
    PETCH_LAUNCH_CHECK(ctx);
  }
  b->nf = nf;
  return PETCH_OK;
}

}  // namespace

extern "C" int petch_bvh_build(petch_ctx* ctx, petch_bvh* b, const float* verts, const int* faces,
                               int nv, int nf) {
  RefitItem r;
  int rc = build_prepare(ctx, b, verts, faces, nv, nf, &r);
  if (rc != PETCH_OK) return rc;
  rc = build_refit(ctx, r);
  if (rc != PETCH_OK) return rc;
  return build_finish(ctx, b, nf);
}

extern "C" int petch_bvh_build_batch(petch_ctx* ctx, int n, petch_bvh* const* bvhs,
                                     const float* const* verts, const int* const* faces,
                                     const int* nv, const int* nf) {
  PETCH_ARG(ctx, ctx && (n == 0 || (bvhs && verts && faces && nv && nf)),
            "bvh_build_batch: null pointer");
  PETCH_ARG(ctx, n >= 0, "bvh_build_batch: n < 0");
  if (n == 0) return PETCH_OK;
  for (int t = 0; t < n; ++t) {
    PETCH_ARG(ctx, bvhs[t], "bvh_build_batch: item %d has a null BVH", t);
    PETCH_ARG(ctx, nf[t] >= 0 && nv[t] >= 0, "bvh_build_batch: item %d has a negative size", t);
    PETCH_ARG(ctx, nf[t] == 0 || (verts[t] && faces[t]), "bvh_build_batch: item %d has a null "
              "mesh", t);
  }
  // Morton trees of two or more faces take the batched stages; the others (clustered or
  // area-collapsed trees, meshes under two faces) are prepared one by one
  std::vector<RefitItem> refit;
  std::vector<BuildItem> fast;
  std::vector<petch_sort_item> sorts;
  std::vector<int> fast_t;
  long long fb = 0, nb = 0, tiles = 0, tab = 0;
  for (int t = 0; t < n; ++t) {
    petch_bvh* b = bvhs[t];
    if (build_quality(b, nf[t]) != 0 || nf[t] < 2) {
      RefitItem r;
      int rc = build_prepare(ctx, b, verts[t], faces[t], nv[t], nf[t], &r);
      if (rc == PETCH_OK) rc = build_refit(ctx, r);
      if (rc != PETCH_OK) return rc;
      continue;
    }
    b->nv = nv[t];
    b->nf = 0;
    b->grid_n[0] = 0;
    const int rc = ensure_capacity(ctx, b, nf[t]);
    if (rc != PETCH_OK) return rc;
    BuildItem it;
    it.verts = verts[t];
    it.faces = faces[t];
    it.nf = nf[t];
    it.nfb = (int)petch_blocks(nf[t], kBS);
    it.w = carve(b->work, b->cap_f);
    it.nodes = (BvhNode*)b->nodes;
    it.wide = (BvhWide*)b->wide;
    it.tris = (float4*)b->tris;
    it.fblk0 = fb;
    it.nblk0 = nb;
    fb += it.nfb;
    nb += petch_blocks(nf[t] - 1, kBS);
    petch_sort_item si;
    si.keys = it.w.keys;
    si.vals = it.w.vals;
    si.ktmp = it.w.ktmp;
    si.vtmp = it.w.vtmp;
    si.n = nf[t];
    si.nblocks = petch_sort_tiles(nf[t]);
    si.tblk0 = tiles;
    si.hist = si.offs = nullptr;
    tiles += si.nblocks;
    tab += 2LL * 256 * si.nblocks;
    fast.push_back(it);
    sorts.push_back(si);
    fast_t.push_back(t);
    refit.push_back(RefitItem{it.tris, it.nodes, it.w.pint, it.w.pleaf, (float*)it.wide, it.w.root,
                              nullptr, it.nf, it.fblk0});
  }
  PETCH_ARG(ctx, fb <= 0x7fffffffLL && tiles <= 0x7fffffffLL,
            "bvh_build_batch: too many faces for one launch");
  const int m = (int)fast.size();
  if (m > 0) {
    int* tabs = (int*)petch_scratch(ctx, SCR_SORT_MANY, (size_t)tab * sizeof(int));
    if (!tabs) return PETCH_E_HIP;
    long long off = 0;
    for (auto& si : sorts) {
      si.hist = tabs + off;
      si.offs = tabs + off + 256LL * si.nblocks;
      off += 2LL * 256 * si.nblocks;
    }
  }
  // one table upload for every stage: build items, sort items, refit items
  const size_t sz_b = fast.size() * sizeof(BuildItem), sz_s = sorts.size() * sizeof(petch_sort_item);
  const size_t off_s = (sz_b + 255) & ~(size_t)255, off_r = off_s + ((sz_s + 255) & ~(size_t)255);
  const size_t total = off_r + refit.size() * sizeof(RefitItem);
  if (refit.empty()) {
    for (int t = 0; t < n; ++t) {
      const int rc = build_finish(ctx, bvhs[t], nf[t]);
      if (rc != PETCH_OK) return rc;
    }
    return PETCH_OK;
  }
  std::vector<char> blob(total);
  if (sz_b) memcpy(blob.data(), fast.data(), sz_b);
  if (sz_s) memcpy(blob.data() + off_s, sorts.data(), sz_s);
  memcpy(blob.data() + off_r, refit.data(), refit.size() * sizeof(RefitItem));
  char* d = (char*)petch_upload_table(ctx, blob.data(), total);
  if (!d) return PETCH_E_HIP;
  const BuildItem* db = (const BuildItem*)d;
  const petch_sort_item* ds = (const petch_sort_item*)(d + off_s);
  const RefitItem* dr = (const RefitItem*)(d + off_r);
  if (m > 0) {
    hipLaunchKernelGGL(k_bvh_prep_many, dim3((unsigned)fb), dim3(kBS), 0, ctx->stream, db, m);
    PETCH_LAUNCH_CHECK(ctx);
    hipLaunchKernelGGL(k_bvh_bounds_many, dim3((unsigned)m), dim3(kBS), 0, ctx->stream, db);
    PETCH_LAUNCH_CHECK(ctx);
    hipLaunchKernelGGL(k_bvh_morton_many, dim3((unsigned)fb), dim3(kBS), 0, ctx->stream, db, m);
    PETCH_LAUNCH_CHECK(ctx);
    const int rc = petch_radix_sort_pairs_many(ctx, ds, m, tiles);
    if (rc != PETCH_OK) return rc;
    hipLaunchKernelGGL(k_bvh_leaves_many, dim3((unsigned)fb), dim3(kBS), 0, ctx->stream, db, m);
    PETCH_LAUNCH_CHECK(ctx);
    hipLaunchKernelGGL(k_bvh_karras_many, dim3((unsigned)nb), dim3(kBS), 0, ctx->stream, db, m);
    PETCH_LAUNCH_CHECK(ctx);
  }
  if (m > 0) {
    hipLaunchKernelGGL(k_bvh_refit_tile_many, dim3((unsigned)fb), dim3(kBS), 0, ctx->stream, dr, m);
    PETCH_LAUNCH_CHECK(ctx);
    hipLaunchKernelGGL(k_bvh_refit_span_many, dim3((unsigned)fb), dim3(kBS), 0, ctx->stream, dr, m);
    PETCH_LAUNCH_CHECK(ctx);
    hipLaunchKernelGGL(k_bvh_wide_many, dim3((unsigned)nb), dim3(kBS), 0, ctx->stream, db, m);
    PETCH_LAUNCH_CHECK(ctx);
    for (int k = 0; k < m; ++k) bvhs[fast_t[k]]->nf = nf[fast_t[k]];
  }
  // the others: their clustered tree / area-driven collapse, one by one
  std::vector<char> done((size_t)n, 0);
  for (int k = 0; k < m; ++k) done[(size_t)fast_t[k]] = 1;
  for (int t = 0; t < n; ++t) {
    if (done[(size_t)t]) continue;
    const int rc = build_finish(ctx, bvhs[t], nf[t]);
    if (rc != PETCH_OK) return rc;
  }
  return PETCH_OK;
}

extern "C" int petch_bvh_query_ray(petch_ctx* ctx, const petch_bvh* b, const float* orig,
                                   const float* dir, int n, float tmax, int* face, float* t) {
  PETCH_ARG(ctx, ctx && b && orig && dir && face, "bvh_query_ray: null pointer");
  PETCH_ARG(ctx, n >= 0, "bvh_query_ray: n < 0");
  if (n == 0) return PETCH_OK;
  petch::GridView g;
  if (petch_grid_view(b, &g)) {
    hipLaunchKernelGGL(k_query_ray_walk, dim3(petch_blocks(n, kBS)), dim3(kBS), 0, ctx->stream, g,
                       petch_bvh_view(b), orig, dir, n, tmax, face, t);
    PETCH_LAUNCH_CHECK(ctx);
    return PETCH_OK;
  }
  hipLaunchKernelGGL(k_query_ray, dim3(petch_blocks(n, kBS)), dim3(kBS), 0, ctx->stream,
                     petch_bvh_view(b), orig, dir, n, tmax, face, t);
  PETCH_LAUNCH_CHECK(ctx);
  return PETCH_OK;
}

extern "C" int petch_bvh_query_point(petch_ctx* ctx, const petch_bvh* b, const float* pts, int n,
                                     float max_dist, int* face, float* dist) {
  PETCH_ARG(ctx, ctx && b && pts && face, "bvh_query_point: null pointer");
  PETCH_ARG(ctx, n >= 0, "bvh_query_point: n < 0");
  if (n == 0) return PETCH_OK;
  hipLaunchKernelGGL(k_query_point, dim3(petch_blocks(n, kBS)), dim3(kBS), 0, ctx->stream,
                     petch_bvh_view(b), pts, n, max_dist, face, dist);
  PETCH_LAUNCH_CHECK(ctx);
  return PETCH_OK;
}

extern "C" int petch_bvh_status(petch_ctx* ctx, const petch_bvh* b, int* err_host) {
  PETCH_ARG(ctx, ctx && b && err_host, "bvh_status: null pointer");
  *err_host = 0;
  if (!b->work) return PETCH_OK;
  int* h = (int*)petch_pinned(ctx, sizeof(int));
  if (!h) return PETCH_E_HIP;
  PETCH_HIP(ctx, hipMemcpyAsync(h, carve(b->work, b->cap_f).err, sizeof(int),
                                hipMemcpyDeviceToHost, ctx->stream));
  PETCH_HIP(ctx, hipStreamSynchronize(ctx->stream));
  *err_host = *h;
  return PETCH_OK;
}

extern "C" int petch_bvh_status_async(petch_ctx* ctx, const petch_bvh* b, int* err_dev) {
  PETCH_ARG(ctx, ctx && b && err_dev, "bvh_status_async: null pointer");
  if (!b->work) {
    PETCH_HIP(ctx, hipMemsetAsync(err_dev, 0, sizeof(int), ctx->stream));
    return PETCH_OK;
  }
  PETCH_HIP(ctx, hipMemcpyAsync(err_dev, carve(b->work, b->cap_f).err, sizeof(int),
                                hipMemcpyDeviceToDevice, ctx->stream));
  return PETCH_OK;
}

extern "C" int petch_bvh_root_bounds(petch_ctx* ctx, const petch_bvh* b, float* lohi_host) {
  PETCH_ARG(ctx, ctx && b && lohi_host, "bvh_root_bounds: null pointer");
  PETCH_ARG(ctx, b->work && b->nf > 1, "bvh_root_bounds: BVH has no internal nodes");
  PETCH_HIP(ctx, hipMemcpyAsync(lohi_host, carve(b->work, b->cap_f).root, 6 * sizeof(float),
                                hipMemcpyDeviceToHost, ctx->stream));
  PETCH_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return PETCH_OK;
}
