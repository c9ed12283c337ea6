// Ray queries on a marching-cubes surface by walking the level set's own cells.
//
// Every triangle of such a surface lies in one cell of the grid it was cut from, and faces come
// out in cell order, so a cell's triangles are consecutive faces. One 32-bit word per node holds
// what a ray needs to know of the cell that starts there:
//   occupied: first face << 4 | number of faces (1..15)
//   empty:    Chebyshev distance in cells to the nearest occupied cell << 4, at most kGridFar
// (the words lie node by node, (nx, ny, nz) in C order; the last layer of each axis starts no
// cell). A ray in an empty cell of distance D leaps to the edge of the cube of 2D - 1 empty cells
// around it; in an occupied cell it tests the cell's triangles (ray_tri, the test of the BVH
// leaves) and is done once its best hit lies before the cell's exit. Against the 4-wide tree this
// takes about as many steps per query (6.6 and 3.1 triangle tests against 8.1 and 1.5, AR-10
// trench), but a step is one dependent 4-byte load instead of a 112-byte node and a third of its
// instructions, and the triangle tests of many lanes are batched. Whole fluxes: 6.78 -> 5.60 ms
// (hole, 200k rays a species), 6.98 -> 5.22 ms (60x10x240 trench, 1M), one step of the AR-10 trench
// with 88M rays 73.3 -> 63.0 ms; what bounds the small ones is the longest ray's chain of steps.
//
// Hits are the tree's, by the same triangle test, but where a ray meets two faces at one distance
// (an edge or a vertex, met exactly): there the tree takes the face that its traversal tests
// first. A walk notes such a tie, and the caller leaves the ray to the tree; one query in ten
// million ends so where faces don't coincide.
//
// Rounding. A plane crossing or a position is exact to a few ulps of the coordinates, 3e-5 of a
// cell at 260 cells, and a triangle's vertices lie within as much of its cell; eps, 1e-4 of a cell
// plus 1e-6 of the grid's length in cells, bounds what adds up. Within eps of a plane either side
// may hold the hit, and a ray nearly along a plane stays beside it for many cells: the cells beside
// the ray are tested too wherever it starts, wherever it enters a cell within eps (and the
// crossing's own error along the ray) of a second plane, ahead or just left behind, and where it
// ends just before a plane. (The check of each entry costs 1 to 3 % of a flux.) Each step leaves
// its cell through a plane ahead, and a leap sets the other axes back by less than it gains, so a
// walk ends after at most nx + ny + nz steps. All this is about origins in the grid or some grid
// lengths off; the rounding of a farther one grows with it, and its ray is left to the tree
// (GridView::reach).
#pragma once
#include "bvh.h"

namespace petch {

constexpr int kGridFar = 15;

struct GridView {
  const uint32_t* cells;
  const float4* tris;  // v0 (w = face id bits), v1, v2 of every face, in face order
  int mx, my, mz;      // cells per axis
  float dx, inv_dx, eps;  // eps in cells
  float slack;            // a quarter of eps in length units
  float reach;            // largest coordinate of an origin that the walk takes
  const float* root;   // bounds of all triangles (lo xyz, hi xyz); null below two faces
};

// The watertight test of ray_tri with the axes rotated by the ray's kz alone (kx and ky follow
// from it): the same operations in the same order.
__device__ __forceinline__ Vec3 rot_axes(Vec3 v, bool k0, bool k2) {
  return v3(k2 ? v.x : (k0 ? v.y : v.z), k2 ? v.y : (k0 ? v.z : v.x), k2 ? v.z : (k0 ? v.x : v.y));
}

// A ray's constants for the walk: reciprocals for the cell planes, axis and shear for the
// triangle test.
struct WalkRay {
  Vec3 inv;
  int kz;
  float Sx, Sy, Sz;
};

__device__ __forceinline__ WalkRay walk_ray(Vec3 d) {
  const RayPre r = ray_pre(v3(0.f, 0.f, 0.f), d);
  return WalkRay{r.inv, r.kz, r.Sx, r.Sy, r.Sz};
}

// `tie` is set by a hit as far as tbest to within rounding, either way.
__device__ __forceinline__ bool walk_tri(Vec3 o, const WalkRay& r, Vec3 p0, Vec3 p1, Vec3 p2,
                                         float tbest, float& t, bool& tie) {
#pragma clang fp contract(off)
  const bool k0 = r.kz == 0, k2 = r.kz == 2;
  const Vec3 A = rot_axes(p0 - o, k0, k2), B = rot_axes(p1 - o, k0, k2),
             C = rot_axes(p2 - o, k0, k2);
  const float Ax = A.x - r.Sx * A.z, Ay = A.y - r.Sy * A.z;
  const float Bx = B.x - r.Sx * B.z, By = B.y - r.Sy * B.z;
  const float Cx = C.x - r.Sx * C.z, Cy = C.y - r.Sy * C.z;
  float U = Cx * By - Cy * Bx;
  float V = Ax * Cy - Ay * Cx;
  float W = Bx * Ay - By * Ax;
  if (U == 0.f || V == 0.f || W == 0.f) {
    U = (float)((double)Cx * By - (double)Cy * Bx);
    V = (float)((double)Ax * Cy - (double)Ay * Cx);
    W = (float)((double)Bx * Ay - (double)By * Ax);
  }
  if ((U < 0.f || V < 0.f || W < 0.f) && (U > 0.f || V > 0.f || W > 0.f)) return false;
  float det = U + V + W;
  if (det == 0.f) return false;
  float T = U * (r.Sz * A.z) + V * (r.Sz * B.z) + W * (r.Sz * C.z);
  if (det < 0.f) {
    T = -T;
    det = -det;
  }
  if (!(T > 0.f) || !(T < tbest * det * 1.000001f)) return false;
  t = T / det;
  tie = fabsf(t - tbest) <= 1.0e-6f * tbest;
  return t > 0.f && T < tbest * det && t < tbest;
}

// State of one query. cell (cx, cy, cz) with its leap D; faces [cur, end) of the cell still to be
// tested; amb: the neighbours still owed a test (two bits per axis: 1 the lower, 2 the upper
// neighbour; bits 6..8 the subset of axes tested last).
struct Walk {
  float t;   // best hit so far, or the bound on t
  int face;  // its face, -1 none
  int cx, cy, cz, D;
  int cur, end, amb;
  bool tie;
};

enum WalkState { kWalkOn = 1, kWalkTri = 2, kWalkMiss = 4, kWalkHit = 5 };

// (columns and words of one grid fit 24 and 30 bits, petch_bvh_set_grid)
__device__ __forceinline__ uint32_t grid_word(const GridView& g, int x, int y, int z) {
  const uint32_t c = __umul24((uint32_t)x, (uint32_t)(g.my + 1)) + (uint32_t)y;
  const uint32_t i = __umul24(c, (uint32_t)(g.mz + 1)) + (uint32_t)z;
  return *(const uint32_t*)((const char*)g.cells + 4u * i);
}

// The side of a neighbouring cell within eps of the coordinate q (in cells): 0 none, 1 the
// lower, 2 the upper.
__device__ __forceinline__ int grid_side(float q, float eps) {
  const float f = q - floorf(q);
  return f < eps ? 1 : (f > 1.f - eps ? 2 : 0);
}

// The coordinate q in cells, within the m cells of its axis and no nearer than half a cell to its
// ends (a ray may run along the outer planes; no neighbour lies across them).
__device__ __forceinline__ float grid_clamp(float q, int m) {
  return fminf(fmaxf(q, 0.5f), (float)m - 0.5f);
}
__device__ __forceinline__ float grid_coord(const GridView& g, float p, int m) {
  return grid_clamp(p * g.inv_dx, m);
}

// Takes up the cell just entered, whose word is w.
__device__ __forceinline__ WalkState walk_enter(Walk& T, uint32_t w, int amb) {
  const int n = (int)(w & 15u), v = (int)(w >> 4);
  T.cur = T.end = 0;
  T.amb = 0;
  T.D = n ? 1 : v;
  if (n) {
    T.cur = v;
    T.end = v + n;
  }
  if (T.D != 1) return kWalkOn;
  T.amb = amb;
  return (n || amb) ? kWalkTri : kWalkOn;
}

// Starts the query of the ray (o, d) for hits with 0 < t < tmax. The walk covers the stretch of the
// ray within the bounds of the triangles, eps wider: a ray that starts above the surface enters at
// its top, one that leaves upwards ends there. (The face that a ray starts on has its test as any
// other: where the coordinates' rounding exceeds the origin's offset the ray meets it again.)
__device__ __forceinline__ WalkState walk_begin(const GridView& g, Walk& T, Vec3 o, Vec3 d,
                                                const WalkRay& r, float tmax) {
  T.face = -1;
  const float far = fmaxf(fmaxf(fabsf(o.x), fabsf(o.y)), fabsf(o.z));
  const float e = __builtin_fmaf(far, 9.53674316e-7f, g.eps * g.dx);  // and 8 ulps of the origin
  Vec3 lo = v3(0.f, 0.f, 0.f),
       hi = v3((float)g.mx * g.dx, (float)g.my * g.dx, (float)g.mz * g.dx);
  if (g.root) {
    lo = v3(g.root[0], g.root[1], g.root[2]);
    hi = v3(g.root[3], g.root[4], g.root[5]);
  }
  const bool px = r.inv.x >= 0.f, py = r.inv.y >= 0.f, pz = r.inv.z >= 0.f;
  const float tn = fmaxf(fmaxf(((px ? lo.x - e : hi.x + e) - o.x) * r.inv.x,
                               ((py ? lo.y - e : hi.y + e) - o.y) * r.inv.y),
                         fmaxf(((pz ? lo.z - e : hi.z + e) - o.z) * r.inv.z, 0.f));
  const float tf = fminf(fminf(((px ? hi.x + e : lo.x - e) - o.x) * r.inv.x,
                               ((py ? hi.y + e : lo.y - e) - o.y) * r.inv.y),
                         ((pz ? hi.z + e : lo.z - e) - o.z) * r.inv.z);
  T.tie = false;
  if (!(tn <= tf)) return kWalkMiss;
  // an origin so far off that its rounding nears eps: to the tree, as a tie
  if (far > g.reach) {
    T.tie = true;
    return kWalkHit;
  }
  T.t = fminf(tmax, tf);
  const float qx = grid_coord(g, o.x + tn * d.x, g.mx),
              qy = grid_coord(g, o.y + tn * d.y, g.my),
              qz = grid_coord(g, o.z + tn * d.z, g.mz);
  T.cx = (int)qx;
  T.cy = (int)qy;
  T.cz = (int)qz;
  const uint32_t w = grid_word(g, T.cx, T.cy, T.cz);
  return walk_enter(T, w, grid_side(qx, g.eps) | (grid_side(qy, g.eps) << 2) |
                              (grid_side(qz, g.eps) << 4));
}

// Where the ray crosses the plane between cells c - 1 and c of one axis; never for a direction
// without a component along it (its reciprocal is +-1e20), also when it runs in the plane.
__device__ __forceinline__ float plane_t(const GridView& g, int c, float o, float inv) {
  const float t = ((float)c * g.dx - o) * inv;
  return fabsf(inv) < 1.0e20f ? t : 1.0e30f;
}

// The side (as grid_side) on which the coordinate q, in cells, lies within tol of the border of
// cell c or beyond it.
__device__ __forceinline__ int cell_side(float q, int c, float tol) {
  const float r = q - ((float)c + 0.5f);
  return fabsf(r) > 0.5f - tol ? (r > 0.f ? 2 : 1) : 0;
}

// Ends a query whose end (its best hit, or the bound on t) lies beside a plane ahead: the cell of
// that point and its neighbours within eps have their test first. D = 0 says that nothing else is
// owed then.
__device__ __forceinline__ WalkState walk_end(const GridView& g, Walk& T, Vec3 o, Vec3 d) {
  const float qx = grid_coord(g, __builtin_fmaf(T.t, d.x, o.x), g.mx),
              qy = grid_coord(g, __builtin_fmaf(T.t, d.y, o.y), g.my),
              qz = grid_coord(g, __builtin_fmaf(T.t, d.z, o.z), g.mz);
  T.cx = (int)qx;
  T.cy = (int)qy;
  T.cz = (int)qz;
  walk_enter(T, grid_word(g, T.cx, T.cy, T.cz), 0);
  T.amb = grid_side(qx, g.eps) | (grid_side(qy, g.eps) << 2) | (grid_side(qz, g.eps) << 4);
  T.D = 0;
  return kWalkTri;
}

// Leaves the current cell (or the empty cube around it) for the next.
__device__ __forceinline__ WalkState walk_step(const GridView& g, Walk& T, Vec3 o, Vec3 d,
                                               const WalkRay& r) {
  const int D = T.D, E = 1 - D;
  if (D == 0) return T.face >= 0 ? kWalkHit : kWalkMiss;
  const bool px = r.inv.x >= 0.f, py = r.inv.y >= 0.f, pz = r.inv.z >= 0.f;
  // the planes the ray leaves through
  const int wx = T.cx + (px ? D : E), wy = T.cy + (py ? D : E), wz = T.cz + (pz ? D : E);
  const float tx = plane_t(g, wx, o.x, r.inv.x);
  const float ty = plane_t(g, wy, o.y, r.inv.y);
  const float tz = plane_t(g, wz, o.z, r.inv.z);
  const float te = fminf(fminf(tx, ty), tz);
  const bool ax = tx <= te, ay = !ax && ty <= te, az = !ax && !ay;
  // how far the crossing may be off along the ray
  const float be = g.slack * fabsf(ax ? r.inv.x : (ay ? r.inv.y : r.inv.z));
  if (T.t <= te - 2.f * be) {
    const float s2 = 2.f * g.slack;
    if (T.t > fminf(fminf(tx - s2 * fabsf(r.inv.x), ty - s2 * fabsf(r.inv.y)),
                    tz - s2 * fabsf(r.inv.z)))
      return walk_end(g, T, o, d);
    return T.face >= 0 ? kWalkHit : kWalkMiss;
  }
  // the cell entered: across the plane left, on the other axes the cell held (one step) or the
  // one that the position says (a leap)
  const float qx = __builtin_fmaf(te, d.x, o.x) * g.inv_dx,
              qy = __builtin_fmaf(te, d.y, o.y) * g.inv_dx,
              qz = __builtin_fmaf(te, d.z, o.z) * g.inv_dx;
  T.cx = ax ? (px ? wx : wx - 1) : (D == 1 ? T.cx : (int)grid_clamp(qx, g.mx));
  T.cy = ay ? (py ? wy : wy - 1) : (D == 1 ? T.cy : (int)grid_clamp(qy, g.my));
  T.cz = az ? (pz ? wz : wz - 1) : (D == 1 ? T.cz : (int)grid_clamp(qz, g.mz));
  // Where the ray comes within tol of a second plane, ahead or just left behind, the cells beside
  // the one entered have their test too: across that plane, with those back over the plane it came
  // through. (The distances to the nearest plane of each axis; that of the plane left is about 0.)
  const float tol = g.eps + 2.f * be * g.inv_dx * fmaxf(fmaxf(fabsf(d.x), fabsf(d.y)), fabsf(d.z));
  int amb = 0;
  if (__builtin_amdgcn_fmed3f(fabsf(qx - rintf(qx)), fabsf(qy - rintf(qy)),
                              fabsf(qz - rintf(qz))) < tol) {
    const int sx = ax ? 0 : cell_side(grid_clamp(qx, g.mx), T.cx, tol),
              sy = ay ? 0 : cell_side(grid_clamp(qy, g.my), T.cy, tol),
              sz = az ? 0 : cell_side(grid_clamp(qz, g.mz), T.cz, tol);
    if (sx | sy | sz)
      amb = (ax ? (px ? 1 : 2) : sx) | (ay ? (py ? 1 : 2) : sy) << 2 | (az ? (pz ? 1 : 2) : sz) << 4;
  }
  if ((unsigned)T.cx >= (unsigned)g.mx || (unsigned)T.cy >= (unsigned)g.my ||
      (unsigned)T.cz >= (unsigned)g.mz) {
    // out of the grid, once the neighbours owed a test have had it
    if (!amb) return T.face >= 0 ? kWalkHit : kWalkMiss;
    return walk_enter(T, 1u << 4, amb);
  }
  const uint32_t w = grid_word(g, T.cx, T.cy, T.cz);
  return walk_enter(T, w, amb);
}

// Tests the next face of the current cell's list; when the list is done goes on to the next
// neighbour owed a test, or back to walking.
__device__ __forceinline__ WalkState walk_test(const GridView& g, Walk& T, Vec3 o,
                                               const WalkRay& r) {
  if (T.cur < T.end) {
    const float4* q = g.tris + 3 * (long long)T.cur;
    const float4 q0 = q[0], q1 = q[1], q2 = q[2];
    float t;
    bool tie = false;
    const bool better = walk_tri(o, r, v3(q0.x, q0.y, q0.z), v3(q1.x, q1.y, q1.z),
                                 v3(q2.x, q2.y, q2.z), T.t, t, tie);
    // (a neighbour's face may come up twice, and T.t starts as a bound)
    T.tie = T.tie || (tie && T.face >= 0 && T.face != T.cur);
    if (better) {
      T.t = t;
      T.face = T.cur;
    }
    ++T.cur;
  }
  if (T.cur < T.end) return kWalkTri;
  if (!T.amb) return kWalkOn;
  int m = T.amb >> 6;
  const int a0 = T.amb & 3, a1 = (T.amb >> 2) & 3, a2 = (T.amb >> 4) & 3;
  const int axes = (a0 ? 1 : 0) | (a1 ? 2 : 0) | (a2 ? 4 : 0);
  do {
    ++m;
  } while (m < 8 && (m & ~axes));
  if (m >= 8) {
    T.amb = 0;
    return kWalkOn;
  }
  T.amb = (T.amb & 63) | (m << 6);
  const int x = T.cx + ((m & 1) ? (a0 == 1 ? -1 : 1) : 0);
  const int y = T.cy + ((m & 2) ? (a1 == 1 ? -1 : 1) : 0);
  const int z = T.cz + ((m & 4) ? (a2 == 1 ? -1 : 1) : 0);
  if ((unsigned)x < (unsigned)g.mx && (unsigned)y < (unsigned)g.my && (unsigned)z < (unsigned)g.mz) {
    const uint32_t w = grid_word(g, x, y, z);
    if (w & 15u) {
      T.cur = (int)(w >> 4);
      T.end = T.cur + (int)(w & 15u);
    }
  }
  return kWalkTri;
}

// Closest hit with 0 < t < tmax of one ray, the whole query at once.
__device__ __forceinline__ Hit walk_closest_hit(const GridView& g, const BvhView& tree, Vec3 o,
                                                Vec3 d, float tmax) {
  const WalkRay r = walk_ray(d);
  Walk T;
  WalkState s = walk_begin(g, T, o, d, r, tmax);
  while (s == kWalkOn || s == kWalkTri) {
    if (s == kWalkTri) s = walk_test(g, T, o, r);
    else s = walk_step(g, T, o, d, r);
  }
  if (T.tie) return bvh_closest_hit(tree, o, d, tmax);
  return Hit{T.face, T.face, T.t};
}

}  // namespace petch
