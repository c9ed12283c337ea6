// The cells of a marching-cubes surface's grid, as the ray walks read them (gridwalk.h): the
// occupied cells' words from marching cubes, the empty cells' Chebyshev distance to the nearest
// occupied one, and the triangles in face order.
//
// The distance is separable: along z to the nearest occupied cell, then over y the least of
// max(|dy|, that), then over x. The first pass takes the nearest set bits of the wavefront's
// occupancy mask. The other two look outward from four cells of a column at a time (one word of
// the byte planes, whose columns are padded to whole words) and stop once the offset reaches the
// largest of the four values, so cells near the surface take a few reads and no four more than
// 2 kGridFar + 1; the byte planes stay in the L2. Three launches, whatever the number of surfaces.
// (Cell by cell, with byte reads: 2.80 ms for the 32 surfaces of a batched step, 80 us for a
// 47k-face trench; now 1.00 ms and 44 us, bound by the chain of reads of the cells far from the surface.)
#include "common.h"
#include "fastdiv.h"
#include "gridwalk.h"

#include <algorithm>
#include <vector>

int* petch_bvh_err(const petch_bvh* b);
petch::BvhView petch_bvh_view(const petch_bvh* b);

namespace {

constexpr int kBS = 256;

struct GridBuild {
  const float* verts;
  const int* faces;
  const uint32_t* raw;
  uint32_t* cells;
  float4* tris;
  uint8_t *dz, *dyz;  // distances after the z pass, after the y pass
  int* err;
  int nx, ny, nz, nf, N;
  int nw, N4;             // words of a column of the byte planes, and of a plane
  float inv_dx, tol;
  petch::FastDiv fy, fz, fw;
  long long blk0, nblk0;  // first workgroup of the first pass (nodes, then faces), of the others
};

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// The four values of a word of a byte plane, as two pairs (bytes 0 and 2, 1 and 3).
struct Four {
  u16x2 e, o;
};
__device__ __forceinline__ Four four(uint32_t w) {
  return Four{__builtin_bit_cast(u16x2, w & 0x00ff00ffu),
              __builtin_bit_cast(u16x2, (w >> 8) & 0x00ff00ffu)};
}
__device__ __forceinline__ uint32_t word(Four f) {
  return __builtin_bit_cast(uint32_t, f.e) | (__builtin_bit_cast(uint32_t, f.o) << 8);
}

// Least max(r, plane[n +- r st]) over r for four cells at once, the offsets staying within
// [0, len) of position p.
__device__ __forceinline__ Four spread(const uint32_t* __restrict__ plane, int n, int st, int p,
                                       int len) {
  Four best = four(plane[n]);
  for (int r = 1;; ++r) {
    const u16x2 m = __builtin_elementwise_max(best.e, best.o);
    if (r >= max((int)m.x, (int)m.y)) return best;
    const u16x2 rr = (unsigned short)r;
    if (p >= r) {
      const Four q = four(plane[n - r * st]);
      best.e = __builtin_elementwise_min(best.e, __builtin_elementwise_max(q.e, rr));
      best.o = __builtin_elementwise_min(best.o, __builtin_elementwise_max(q.o, rr));
    }
    if (p + r < len) {
      const Four q = four(plane[n + r * st]);
      best.e = __builtin_elementwise_min(best.e, __builtin_elementwise_max(q.e, rr));
      best.o = __builtin_elementwise_min(best.o, __builtin_elementwise_max(q.o, rr));
    }
  }
}

// The occupancy of the wavefront's 64 consecutive nodes and of the 16 on each side as bit masks
// (all lanes take part; n >= N reads none); the nearest set bit that lies in the node's own column.
__device__ __forceinline__ void grid_pass_z(const GridBuild& b, int n) {
  const int lane = threadIdx.x & 63, h = lane < 16 ? n - 16 : n + 16;
  const unsigned long long m = __ballot(n < b.N && (b.raw[n] & 15u));
  const unsigned long long side =
      __ballot((lane < 16 || lane >= 48) && h >= 0 && h < b.N && (b.raw[h] & 15u));
  if (n >= b.N) return;
  const uint32_t c = petch::fastdiv((uint32_t)n, b.fz);
  const int k = (int)((uint32_t)n - c * b.fz.d);
  // bit d: the node d above, below
  unsigned long long up = m >> lane, dn = m << (63 - lane);
  if (lane >= 48) up |= (side >> 48) << (64 - lane);
  if (lane < 16) dn |= (side << 48) >> (lane + 1);
  const int du = up ? __ffsll(up) - 1 : 64, dd = dn ? __clzll((long long)dn) : 64;
  int best = petch::kGridFar;
  if (k + du < b.nz) best = min(best, du);
  if (dd <= k) best = min(best, dd);
  uint8_t* col = b.dz + 4 * (size_t)b.nw * c;
  col[k] = (uint8_t)best;
  if (k == b.nz - 1)
    for (int q = b.nz; q < 4 * b.nw; ++q) col[q] = petch::kGridFar;
}

__device__ __forceinline__ void grid_tri(const GridBuild& b, int f) {
  const int* q = b.faces + 3LL * f;
#pragma unroll
  for (int v = 0; v < 3; ++v) {
    const float* p = b.verts + 3LL * q[v];
    b.tris[3LL * f + v] = make_float4(p[0], p[1], p[2], v == 0 ? __int_as_float(f) : 0.f);
  }
}

__device__ __forceinline__ void grid_first(const GridBuild& b, long long blk) {
  const int nodes = (b.N + kBS - 1) / kBS;
  if (blk < nodes) {
    const int n = (int)blk * kBS + threadIdx.x;
    grid_pass_z(b, n);
  } else {
    const int f = (int)(blk - nodes) * kBS + threadIdx.x;
    if (f < b.nf) grid_tri(b, f);
  }
}

__device__ __forceinline__ void grid_pass_y(const GridBuild& b, int n) {
  const uint32_t c = petch::fastdiv((uint32_t)n, b.fw);
  const int j = (int)(c - petch::fastdiv(c, b.fy) * b.fy.d);
  ((uint32_t*)b.dyz)[n] = word(spread((const uint32_t*)b.dz, n, b.nw, j, b.ny));
}

// The last pass writes the words; an occupied cell's triangles must lie in it to within tol (a
// thousandth of a cell plus the rounding of their vertices), or the walk could miss them.
__device__ __forceinline__ void grid_pass_x(const GridBuild& b, int n) {
  const uint32_t c = petch::fastdiv((uint32_t)n, b.fw);
  const int k0 = 4 * (int)((uint32_t)n - c * b.fw.d);
  const int i = (int)petch::fastdiv(c, b.fy);
  const int j = (int)(c - (uint32_t)i * b.fy.d);
  const uint32_t far4 = word(spread((const uint32_t*)b.dyz, n, b.ny * b.nw, i, b.nx));
  for (int q = 0; q < 4 && k0 + q < b.nz; ++q) {
    const int k = k0 + q, at = (int)c * b.nz + k;
    const uint32_t far = (far4 >> (8 * q)) & 255u;
    uint32_t out = far << 4;
    if (far == 0) {   // the cell is occupied itself
      out = b.raw[at];
      const int f0 = (int)(out >> 4), f1 = f0 + (int)(out & 15u);
      bool ok = f1 <= b.nf;
      for (int f = f0; ok && f < f1; ++f) {
        for (int v = 0; v < 3; ++v) {
          const float* p = b.verts + 3LL * b.faces[3LL * f + v];
          const float x = p[0] * b.inv_dx - (float)i, y = p[1] * b.inv_dx - (float)j,
                      z = p[2] * b.inv_dx - (float)k;
          ok = ok && !(fminf(fminf(x, y), z) < -b.tol || fmaxf(fmaxf(x, y), z) > 1.f + b.tol);
        }
      }
      if (!ok) {      // a bad word never reaches a walk
        out = 1u << 4;
        *b.err = 4;
      }
    }
    b.cells[at] = out;
  }
}

__global__ void k_grid_first(GridBuild b) { grid_first(b, blockIdx.x); }
__global__ void k_grid_y(GridBuild b) {
  const int n = blockIdx.x * kBS + threadIdx.x;
  if (n < b.N4) grid_pass_y(b, n);
}
__global__ void k_grid_x(GridBuild b) {
  const int n = blockIdx.x * kBS + threadIdx.x;
  if (n < b.N4) grid_pass_x(b, n);
}

// The passes of many surfaces (the features of a batched step), one launch each.
__device__ __forceinline__ int grid_item_of(const GridBuild* __restrict__ t, int n, bool first) {
  int lo = 0, hi = n - 1;
  const long long b = blockIdx.x;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if ((first ? t[mid].blk0 : t[mid].nblk0) <= b) lo = mid; else hi = mid - 1;
  }
  return lo;
}

__global__ void k_grid_first_many(const GridBuild* __restrict__ t, int n) {
  const GridBuild& b = t[grid_item_of(t, n, true)];
  grid_first(b, blockIdx.x - b.blk0);
}
__global__ void k_grid_y_many(const GridBuild* __restrict__ t, int n) {
  const GridBuild& b = t[grid_item_of(t, n, false)];
  const int i = (int)(blockIdx.x - b.nblk0) * kBS + threadIdx.x;
  if (i < b.N4) grid_pass_y(b, i);
}
__global__ void k_grid_x_many(const GridBuild* __restrict__ t, int n) {
  const GridBuild& b = t[grid_item_of(t, n, false)];
  const int i = (int)(blockIdx.x - b.nblk0) * kBS + threadIdx.x;
  if (i < b.N4) grid_pass_x(b, i);
}

int max_axis(int x, int y, int z) { return x > y ? (x > z ? x : z) : (y > z ? y : z); }

// Checks an item and grows its BVH's buffers (a regrowth waits for the stream). The BVH has no grid
// until grid_done, so that a call that fails on the way leaves it to its tree.
int grid_prepare(petch_ctx* ctx, const petch_grid_item& a, GridBuild& b) {
  PETCH_ARG(ctx, a.bvh && a.bvh->nf > 0 && a.verts && a.faces && a.cells,
            "bvh_set_grid: null pointer or no faces");
  PETCH_ARG(ctx, a.nx > 1 && a.ny > 1 && a.nz > 1 && a.dx > 0.0, "bvh_set_grid: bad grid");
  const long long N = (long long)a.nx * a.ny * a.nz;
  PETCH_ARG(ctx, N < (1LL << 30) && (long long)a.nx * a.ny < (1LL << 24) && a.bvh->nf < (1 << 28),
            "bvh_set_grid: more than 2^30-1 nodes, 2^24-1 columns or 2^28-1 faces");
  petch_bvh* v = a.bvh;
  v->grid_n[0] = 0;
  if (v->cells_cap < (size_t)N) {
    PETCH_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (v->cells) (void)hipFree(v->cells);
    v->cells = nullptr;
    v->cells_cap = 0;
    PETCH_HIP(ctx, hipMalloc(&v->cells, (size_t)N * sizeof(uint32_t)));
    v->cells_cap = (size_t)N;
  }
  if (v->gtris_cap < v->nf) {
    PETCH_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (v->gtris) (void)hipFree(v->gtris);
    v->gtris = nullptr;
    v->gtris_cap = 0;
    PETCH_HIP(ctx, hipMalloc(&v->gtris, (size_t)v->cap_f * 48));
    v->gtris_cap = v->cap_f;
  }
  b.verts = a.verts;
  b.faces = a.faces;
  b.raw = a.cells;
  b.cells = v->cells;
  b.tris = (float4*)v->gtris;
  b.err = petch_bvh_err(v);
  b.nx = a.nx;
  b.ny = a.ny;
  b.nz = a.nz;
  b.nf = v->nf;
  b.N = (int)N;
  b.inv_dx = (float)(1.0 / a.dx);
  b.tol = 1.0e-3f + 1.0e-6f * (float)max_axis(a.nx, a.ny, a.nz);
  b.fy = petch::make_fastdiv((uint32_t)a.ny);
  b.fz = petch::make_fastdiv((uint32_t)a.nz);
  b.nw = (a.nz + 3) / 4;
  b.N4 = a.nx * a.ny * b.nw;
  b.fw = petch::make_fastdiv((uint32_t)b.nw);
  b.blk0 = b.nblk0 = 0;
  return PETCH_OK;
}

void grid_done(const petch_grid_item& a) {
  a.bvh->grid_n[0] = a.nx;
  a.bvh->grid_n[1] = a.ny;
  a.bvh->grid_n[2] = a.nz;
  a.bvh->grid_dx = a.dx;
}

}  // namespace

bool petch_grid_view(const petch_bvh* b, petch::GridView* v) {
  *v = petch::GridView{};
  if (b->grid_n[0] < 2 || b->nf < 1) return false;
  v->cells = b->cells;
  v->tris = (const float4*)b->gtris;
  v->mx = b->grid_n[0] - 1;
  v->my = b->grid_n[1] - 1;
  v->mz = b->grid_n[2] - 1;
  v->dx = (float)b->grid_dx;
  v->inv_dx = (float)(1.0 / b->grid_dx);
  v->eps = 1.0e-4f + 1.0e-6f * (float)max_axis(v->mx, v->my, v->mz);
  v->slack = 0.25f * v->eps * v->dx;
  // (an ulp there is half of slack; it lies past the grid's length and past 100 cells)
  v->reach = 4194304.f * v->slack;
  v->root = petch_bvh_view(b).root;
  return true;
}

extern "C" int petch_bvh_set_grid(petch_ctx* ctx, const petch_grid_item* item) {
  PETCH_ARG(ctx, ctx && item, "bvh_set_grid: null pointer");
  GridBuild b;
  const int rc = grid_prepare(ctx, *item, b);
  if (rc != PETCH_OK) return rc;
  b.dz = (uint8_t*)petch_scratch(ctx, SCR_GRID, 8 * (size_t)b.N4);
  if (!b.dz) return PETCH_E_HIP;
  b.dyz = b.dz + 4 * (size_t)b.N4;
  const unsigned gn = petch_blocks(b.N, kBS), gf = petch_blocks(b.nf, kBS),
                 gw = petch_blocks(b.N4, kBS);
  hipLaunchKernelGGL(k_grid_first, dim3(gn + gf), dim3(kBS), 0, ctx->stream, b);
  PETCH_LAUNCH_CHECK(ctx);
  hipLaunchKernelGGL(k_grid_y, dim3(gw), dim3(kBS), 0, ctx->stream, b);
  PETCH_LAUNCH_CHECK(ctx);
  hipLaunchKernelGGL(k_grid_x, dim3(gw), dim3(kBS), 0, ctx->stream, b);
  PETCH_LAUNCH_CHECK(ctx);
  grid_done(*item);
  return PETCH_OK;
}

extern "C" int petch_bvh_set_grid_batch(petch_ctx* ctx, int n, const petch_grid_item* items) {
  PETCH_ARG(ctx, ctx && n >= 0 && (n == 0 || items), "bvh_set_grid_batch: null pointer or n < 0");
  if (n == 0) return PETCH_OK;
  // (a BVH twice: growing its buffers for the second would free the first's)
  std::vector<const petch_bvh*> seen((size_t)n);
  for (int k = 0; k < n; ++k) seen[k] = items[k].bvh;
  std::sort(seen.begin(), seen.end());
  PETCH_ARG(ctx, std::adjacent_find(seen.begin(), seen.end()) == seen.end(),
            "bvh_set_grid_batch: a BVH is listed twice");
  std::vector<GridBuild> t((size_t)n);
  long long first = 0, rest = 0;
  size_t bytes = 0;
  for (int k = 0; k < n; ++k) {
    const int rc = grid_prepare(ctx, items[k], t[k]);
    if (rc != PETCH_OK) return rc;
    t[k].blk0 = first;
    t[k].nblk0 = rest;
    first += petch_blocks(t[k].N, kBS) + petch_blocks(t[k].nf, kBS);
    rest += petch_blocks(t[k].N4, kBS);
    bytes += 8 * (size_t)t[k].N4;
  }
  PETCH_ARG(ctx, first <= 0x7fffffffLL, "bvh_set_grid_batch: too many nodes for one launch");
  uint8_t* plane = (uint8_t*)petch_scratch(ctx, SCR_GRID, bytes);
  if (!plane) return PETCH_E_HIP;
  for (GridBuild& b : t) {
    b.dz = plane;
    b.dyz = plane + 4 * (size_t)b.N4;
    plane += 8 * (size_t)b.N4;
  }
  const GridBuild* d = (const GridBuild*)petch_upload_table(ctx, t.data(), t.size() * sizeof(GridBuild));
  if (!d) return PETCH_E_HIP;
  hipLaunchKernelGGL(k_grid_first_many, dim3((unsigned)first), dim3(kBS), 0, ctx->stream, d, n);
  PETCH_LAUNCH_CHECK(ctx);
  hipLaunchKernelGGL(k_grid_y_many, dim3((unsigned)rest), dim3(kBS), 0, ctx->stream, d, n);
  PETCH_LAUNCH_CHECK(ctx);
  hipLaunchKernelGGL(k_grid_x_many, dim3((unsigned)rest), dim3(kBS), 0, ctx->stream, d, n);
  PETCH_LAUNCH_CHECK(ctx);
  for (int k = 0; k < n; ++k) grid_done(items[k]);
  return PETCH_OK;
}
