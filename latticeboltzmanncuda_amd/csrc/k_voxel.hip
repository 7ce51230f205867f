// Mesh geometry on the GPU.
//
// lbm_voxelize_mesh: which lattice nodes lie inside a closed triangle mesh.  It replaces the host loop of
// Lattice::insertModel (reference Lattice.cpp:228-260) over
// Model::isPointInsideModel (reference Model.cpp:51-63) and decides every
// node as the host Model does: a node on a face (coplanar up to 1e-12
// relative, inside its three edges) is inside; otherwise the generalized
// winding number W = sum of signed solid angles / 4 pi decides, inside
// when |W| > 1/2.  Nodes outside the mesh's bounding box (with a 1e-9
// relative margin) are outside without a test: W is 0 there up to
// rounding and no face can touch them.
//
// A mesh whose faces close (every edge is run through as often one way as
// the other) has a whole W at every node off its faces: the signed count of
// the faces that a ray from the node crosses.  k_voxelize_lines counts them
// along z, one wavefront per lattice line, the side of each edge exact, so that
// the count is the W that the solid angles round to.  Other meshes take the
// sum of solid angles (k_voxelize; same formulas as the host, double
// precision, no contraction; only atan2 comes from the GPU's math library,
// and it cannot change a decision: W is within 1e-15 of 0.5 only for points
// closer to a face than the on-face tolerance).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "lbm_internal.h"
#include "lbm_lattice.h"
#include "lbm_scan.h"

#pragma clang fp contract(off)

namespace lbm {
namespace {

struct D3 {
  double x, y, z;
};
__device__ __forceinline__ D3 sub(D3 a, D3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ double dot(D3 a, D3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ D3 cross(D3 a, D3 b) {
  return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
__device__ __forceinline__ double norm(D3 a) { return sqrt(dot(a, a)); }

__device__ bool on_triangle(D3 p, D3 a, D3 b, D3 c) {
  const D3 n = cross(sub(b, a), sub(c, a));
  const double nn = norm(n);
  if (nn == 0.0) return false;
  const double off = dot(n, sub(p, a));
  const double scale = nn * (norm(sub(p, a)) + norm(sub(b, a)));
  if (fabs(off) > 1e-12 * scale) return false;
  const double tol = -1e-12 * nn * nn;
  return dot(cross(sub(b, a), sub(p, a)), n) >= tol && dot(cross(sub(c, b), sub(p, b)), n) >= tol &&
         dot(cross(sub(a, c), sub(p, c)), n) >= tol;
}

__device__ double solid_angle(D3 p, D3 a, D3 b, D3 c) {
  const D3 ra = sub(a, p), rb = sub(b, p), rc = sub(c, p);
  const double la = norm(ra), lb = norm(rb), lc = norm(rc);
  const double num = dot(ra, cross(rb, rc));
  const double den = la * lb * lc + dot(ra, rb) * lc + dot(rb, rc) * la + dot(rc, ra) * lb;
  return 2.0 * atan2(num, den);
}

constexpr int kBlock = 256;
constexpr int kFaceTile = 256;  // faces staged in LDS per pass

__device__ __forceinline__ D3 vert(const float* v, int i) {
  return {(double)v[3 * i], (double)v[3 * i + 1], (double)v[3 * i + 2]};
}

// One thread per node.  Faces are walked in the host's order (on-face pass
// first, then the winding sum in face order), staged through LDS.
__global__ void __launch_bounds__(kBlock)
    k_voxelize(Grid g, float spacing, const float* __restrict__ verts,
               const int32_t* __restrict__ faces, int32_t nf, float3 lo, float3 hi,
               uint8_t* __restrict__ inside) {
  __shared__ D3 tri[kFaceTile][3];
  const uint32_t n = blockIdx.x * kBlock + threadIdx.x;
  bool active = n < g.n;
  D3 p{0.0, 0.0, 0.0};
  if (active) {
    const uint32_t t = g.dz.div(n);
    const uint32_t z = n - t * g.nz, x = g.dy.div(t), y = t - x * g.ny;
    // the host forms the position in float, then widens it
    const float px = (float)x * spacing, py = (float)y * spacing, pz = (float)z * spacing;
    p = {(double)px, (double)py, (double)pz};
    if (px < lo.x || py < lo.y || pz < lo.z || px > hi.x || py > hi.y || pz > hi.z) {
      inside[n] = 0;
      active = false;
    }
  }
  const bool any = __syncthreads_or(active);
  if (!any) return;
  bool on = false;
  double omega = 0.0;
  // pass 0: on a face?  pass 1: winding number (only if on no face)
  for (int pass = 0; pass < 2; ++pass) {
    if (pass == 1 && !__syncthreads_or(active && !on)) break;
    for (int32_t f0 = 0; f0 < nf; f0 += kFaceTile) {
      const int cnt = min(kFaceTile, nf - f0);
      __syncthreads();
      for (int k = threadIdx.x; k < cnt; k += kBlock) {
        tri[k][0] = vert(verts, faces[3 * (f0 + k)]);
        tri[k][1] = vert(verts, faces[3 * (f0 + k) + 1]);
        tri[k][2] = vert(verts, faces[3 * (f0 + k) + 2]);
      }
      __syncthreads();
      if (!active) continue;
      if (pass == 0) {
        for (int k = 0; k < cnt && !on; ++k) on = on_triangle(p, tri[k][0], tri[k][1], tri[k][2]);
      } else if (!on) {
        for (int k = 0; k < cnt; ++k) omega += solid_angle(p, tri[k][0], tri[k][1], tri[k][2]);
      }
    }
  }
  if (active) {
    const double winding = omega / (4.0 * M_PI);
    inside[n] = (on || fabs(winding) > 0.5) ? 1 : 0;
  }
}

// Bounding box of a face, widened by more than the tolerances of the tests
// that it stands before (1e-12 of the face's size, 1e-9 of a link) and the
// rounding of positions: lo in [0], hi in [1].
struct Box {
  float3 lo, hi;
};
__global__ void __launch_bounds__(kBlock)
    k_face_boxes(const float* __restrict__ verts, const int32_t* __restrict__ faces, int32_t nf,
                 float spacing, Box* __restrict__ boxes) {
  const int32_t f = blockIdx.x * kBlock + threadIdx.x;
  if (f >= nf) return;
  float lo[3], hi[3], m = fabsf(spacing);
  for (int a = 0; a < 3; ++a) {
    const float u = verts[3 * faces[3 * f] + a], v = verts[3 * faces[3 * f + 1] + a],
                w = verts[3 * faces[3 * f + 2] + a];
    lo[a] = fminf(u, fminf(v, w));
    hi[a] = fmaxf(u, fmaxf(v, w));
    m = fmaxf(m, fmaxf(fabsf(lo[a]), fabsf(hi[a])));
  }
  m *= 1e-5f;
  boxes[f] = {{lo[0] - m, lo[1] - m, lo[2] - m}, {hi[0] + m, hi[1] + m, hi[2] + m}};
}

// Sign of a x b (two components), exact for the doubles given (without
// overflow and underflow, which float coordinates do not reach): rounding
// keeps the order, so products that round apart lie so, and where they round
// alike their rounding errors, which fma gives exactly, decide.
__device__ __forceinline__ int cross_sign(double ax, double ay, double bx, double by) {
  const double p = ax * by, q = ay * bx;
  if (p != q) return p > q ? 1 : -1;
  const double e = fma(ax, by, -p), f = fma(ay, bx, -q);
  return e > f ? 1 : (e < f ? -1 : 0);
}

// Side of the edge a -> b on which the origin's projection lies, a and b
// relative to the node.  On the edge, the side after a shift of the node by
// (eps, eps^2): one shift for all faces, so a line that meets an edge or a
// vertex crosses just the faces that the shifted line crosses.  0 for an
// edge that projects to a point.
__device__ __forceinline__ int edge_side(const D3& a, const D3& b) {
  const int c = cross_sign(a.x, a.y, b.x, b.y);
  if (c) return c;
  if (a.y != b.y) return a.y > b.y ? 1 : -1;
  return b.x > a.x ? 1 : (b.x < a.x ? -1 : 0);
}

// One wavefront per lattice line (x, y), lane by lane along z: per 64 faces
// the lanes look which boxes meet the line, then all lanes take those faces
// one after another -- on the face?  crossed above the node? -- so a face's
// work is done for 64 nodes at once and only near the line.  96^3, 1,520
// faces: 0.06 ms against 5.2 ms for all solid angles of all nodes.
__global__ void __launch_bounds__(kBlock)
    k_voxelize_lines(Grid g, float spacing, const float* __restrict__ verts,
                     const int32_t* __restrict__ faces, int32_t nf,
                     const Box* __restrict__ boxes, float3 lo, float3 hi,
                     uint8_t* __restrict__ inside, unsigned long long* __restrict__ count) {
  const uint32_t line = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  if (line >= g.nx * g.ny) return;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t x = g.dy.div(line), y = line - x * g.ny;
  const float px = (float)x * spacing, py = (float)y * spacing;
  const bool line_in = !(px < lo.x || py < lo.y || px > hi.x || py > hi.y);
  uint32_t total = 0;
  for (uint32_t z0 = 0; z0 < g.nz; z0 += 64) {
    const uint32_t z = z0 + lane;
    // the host forms the position in float, then widens it
    const float pz = (float)z * spacing;
    const bool active = line_in && z < g.nz && !(pz < lo.z || pz > hi.z);
    bool on = false;
    int winding = 0;
    if (__any(active)) {
      const D3 p{(double)px, (double)py, (double)pz};
      for (int32_t f0 = 0; f0 < nf; f0 += 64) {
        bool near = false;
        if (f0 + (int32_t)lane < nf) {
          const Box b = boxes[f0 + lane];
          near = px >= b.lo.x && px <= b.hi.x && py >= b.lo.y && py <= b.hi.y;
        }
        for (uint64_t m = __ballot(near); m; m &= m - 1) {
          const int32_t f = f0 + __builtin_ctzll(m);
          const Box b = boxes[f];
          const D3 A = vert(verts, faces[3 * f]), B = vert(verts, faces[3 * f + 1]),
                   C = vert(verts, faces[3 * f + 2]);
          if (active && pz >= b.lo.z && pz <= b.hi.z) on = on || on_triangle(p, A, B, C);
          const D3 ra = sub(A, p), rb = sub(B, p), rc = sub(C, p);
          const int side = edge_side(ra, rb);
          if (side && side == edge_side(rb, rc) && side == edge_side(rc, ra)) {
            // the plane's point on the line lies above the node
            const double off = dot(cross(sub(B, A), sub(C, A)), sub(p, A));
            if ((side > 0 ? off : -off) < 0.0) winding += side;
          }
        }
      }
    }
    const bool in = active && (on || winding != 0);
    if (z < g.nz) inside[(uint64_t)line * g.nz + z] = in ? 1 : 0;
    total += (uint32_t)__popcll(__ballot(in));
  }
  if (lane == 0 && total) atomicAdd(count, (unsigned long long)total);
}

// Whether every edge is run through as often from a to b as from b to a (by
// vertex index), and every vertex used is finite.
bool mesh_closes(const float* vertices, const int32_t* faces, int32_t nf) {
  size_t cap = 16;
  while (cap < 8 * (size_t)nf) cap *= 2;
  std::vector<uint64_t> key(cap, ~0ull);
  std::vector<int32_t> sum(cap, 0);
  int64_t open = 0;  // edges whose sum is not 0
  for (int32_t f = 0; f < nf; ++f)
    for (int e = 0; e < 3; ++e) {
      const uint32_t a = (uint32_t)faces[3 * (size_t)f + e],
                     b = (uint32_t)faces[3 * (size_t)f + (e + 1) % 3];
      for (int k = 0; k < 3; ++k)
        if (!std::isfinite(vertices[3 * (size_t)a + k])) return false;
      if (a == b) continue;
      const uint64_t id = (uint64_t)std::min(a, b) << 32 | std::max(a, b);
      size_t h = (size_t)((id * 0x9E3779B97F4A7C15ull) >> 20) & (cap - 1);
      while (key[h] != ~0ull && key[h] != id) h = (h + 1) & (cap - 1);
      key[h] = id;
      open -= sum[h] != 0;
      sum[h] += a < b ? 1 : -1;
      open += sum[h] != 0;
    }
  return open == 0;
}

// Whether no node of the lattice lies in the box [lo, hi].
bool box_is_empty(const Grid& g, float spacing, const float3& lo, const float3& hi) {
  if (!(spacing > 0.0f) || !std::isfinite(spacing)) return false;
  auto along = [&](float a, float b, uint32_t n) {  // (with room for rounding)
    return std::max(0.0, std::ceil((double)a / spacing - 1e-3)) <=
           std::min((double)n - 1.0, std::floor((double)b / spacing + 1e-3));
  };
  return !(along(lo.x, hi.x, g.nx) && along(lo.y, hi.y, g.ny) && along(lo.z, hi.z, g.nz));
}

// ---------------------------------------------------------------------
// lbm_build_reflections: the reflection tables of preProcessModel
// (reference Lattice.cpp:323-426, 450-477) on the GPU, one wavefront per
// internal node that has a link, with the host code's float / double operations in the
// same order (no contraction; sqrt and division correctly rounded); the
// sine and cosine of the half turn are computed on the host.
//
// For each link k of an internal node x whose source x + e_k is in the box
// and not internal: v = reflectionVector(h (x + e_k), h x), i.e. the unit
// vector from x to x + e_k rotated by pi about the normal of the first
// face hit by the ray (x + e_k) -> x (ties within 1e-9 of the nearest hit:
// lowest face index); rank the 27 directions by 2 - |v - e_j/|e_j|| (equal
// scores: higher index first); keep the first three whose target x + e_d is
// in the box and not internal, in slots INVERSE[k]*3 + rank; normalise the
// kept weights by their float sum (a kept rest direction, d = 0, keeps its
// weight as the host code does).

struct HalfTurn {
  float c, s, ci, si;  // cos, sin of +pi/2 and -pi/2 in float
};

__device__ double ray_hit(D3 o, D3 d, D3 a, D3 b, D3 c) {
  const D3 n = cross(sub(b, a), sub(c, a));
  const double denom = dot(n, d);
  const double scale = norm(n) * norm(d);
  if (scale == 0.0 || fabs(denom) <= 1e-14 * scale) return -1.0;
  const double t = dot(n, sub(a, o)) / denom;
  if (t < 0.0) return -1.0;
  const D3 q{o.x + t * d.x, o.y + t * d.y, o.z + t * d.z};
  const double tol = -1e-12 * dot(n, n);
  if (dot(cross(sub(b, a), sub(q, a)), n) < tol || dot(cross(sub(c, b), sub(q, b)), n) < tol ||
      dot(cross(sub(a, c), sub(q, c)), n) < tol)
    return -1.0;
  return t;
}

struct F3 {
  float x, y, z;
};

// The nearest face hit by the ray from p1 through p2 (-1: none): first face
// in index order within 1e-9 of the nearest hit.  face(i) gives the i-th of
// nf faces, in ascending order.
template <class Face>
__device__ __forceinline__ int32_t first_hit(D3 o, D3 d, const float* __restrict__ verts,
                                             const int32_t* __restrict__ faces, int32_t nf,
                                             Face&& face, double& best_t) {
  best_t = INFINITY;
  int32_t best = -1;
  auto hit = [&](int32_t t) {
    return ray_hit(o, d, vert(verts, faces[3 * t]), vert(verts, faces[3 * t + 1]),
                   vert(verts, faces[3 * t + 2]));
  };
  for (int32_t i = 0; i < nf; ++i) {
    const int32_t t = face(i);
    const double h = hit(t);
    if (h >= 0.0 && h < best_t) {
      best_t = h;
      best = t;
    }
  }
  if (best < 0) return -1;
  for (int32_t i = 0; i < nf; ++i) {
    const int32_t t = face(i);
    if (t >= best) break;
    const double h = hit(t);
    if (h >= 0.0 && h <= best_t + 1e-9) return t;
  }
  return best;
}

// Model::reflectionVector(p1, p2), given the face hit (-1: none)
__device__ F3 reflection_vector(F3 p1, F3 p2, int32_t best, const float* __restrict__ verts,
                                const int32_t* __restrict__ faces, const HalfTurn& ht) {
  F3 v{p1.x - p2.x, p1.y - p2.y, p1.z - p2.z};
  {
    const float nrm = sqrtf((v.x * v.x) + (v.y * v.y) + (v.z * v.z));
    v.x /= nrm;
    v.y /= nrm;
    v.z /= nrm;
  }
  if (best < 0) return F3{0.0f, 0.0f, 0.0f};
  const float* A = verts + 3 * faces[3 * best];
  const float* B = verts + 3 * faces[3 * best + 1];
  const float* C = verts + 3 * faces[3 * best + 2];
  const float e1[3] = {B[0] - A[0], B[1] - A[1], B[2] - A[2]};
  const float e2[3] = {C[0] - A[0], C[1] - A[1], C[2] - A[2]};
  F3 ax{(e1[1] * e2[2]) - (e1[2] * e2[1]), (e1[2] * e2[0]) - (e1[0] * e2[2]),
        (e1[0] * e2[1]) - (e1[1] * e2[0])};
  // rotateVectorAroundAxis(axis, v, pi) (Geometry.cpp:22-42)
  const float len = sqrtf((ax.x * ax.x) + (ax.y * ax.y) + (ax.z * ax.z));
  ax.x /= len;
  ax.y /= len;
  ax.z /= len;
  const float q[4] = {ht.c, ht.s * ax.x, ht.s * ax.y, ht.s * ax.z};
  const float qi[4] = {ht.ci, ht.si * ax.x, ht.si * ax.y, ht.si * ax.z};
  const float vv[4] = {0.0f, v.x, v.y, v.z};
  auto ham = [](const float* a, const float* b, float* r) {
    r[0] = (a[0] * b[0]) - (a[1] * b[1]) - (a[2] * b[2]) - (a[3] * b[3]);
    r[1] = (a[0] * b[1]) + (a[1] * b[0]) + (a[2] * b[3]) - (a[3] * b[2]);
    r[2] = (a[0] * b[2]) - (a[1] * b[3]) + (a[2] * b[0]) + (a[3] * b[1]);
    r[3] = (a[0] * b[3]) + (a[1] * b[2]) - (a[2] * b[1]) + (a[3] * b[0]);
  };
  float t1[4], r[4];
  ham(q, vv, t1);
  ham(t1, qi, r);
  return F3{r[1], r[2], r[3]};
}

// Whether the node at (x, y, z) lies in the box and outside the obstacle.
__device__ __forceinline__ bool is_free(const Grid& g, const uint8_t* __restrict__ flags, int x,
                                        int y, int z) {
  return x >= 0 && y >= 0 && z >= 0 && x < (int)g.nx && y < (int)g.ny && z < (int)g.nz &&
         !(flags[(uint32_t)z + g.nz * ((uint32_t)y + g.ny * (uint32_t)x)] & LBM_FLAG_INTERNAL);
}

// Internal nodes with a link to a free node (each of them gets a record:
// the link's own far end is a free target).
struct LinkedIn {
  Grid g;
  const uint8_t* flags;
  __device__ uint32_t operator()(uint32_t n) const {
    if (!(flags[n] & LBM_FLAG_INTERNAL)) return 0u;
    const uint32_t t = g.dz.div(n);
    const int z = (int)(n - t * g.nz), x = (int)g.dy.div(t), y = (int)(t - (uint32_t)x * g.ny);
    for (int k = 1; k < 27; ++k)
      if (is_free(g, flags, x + Lat<27>::E[k][0], y + Lat<27>::E[k][1], z + Lat<27>::E[k][2]))
        return 1u;
    return 0u;
  }
};
struct NodeOut {
  int32_t* node;
  __device__ void operator()(uint32_t n, uint32_t v, uint32_t at) const {
    if (v) node[at] = (int32_t)n;
  }
};

// One wavefront per record, lane k its link k.  All links lie within one
// cell of the node, so only the faces whose boxes meet that cell (found by
// the lanes together, a handful of them) can be hit on a link itself; a ray
// that hits none of those on its link (t <= 1) is followed through all
// faces.  96^3, 1,520 faces, 14,683 records: 61 ms with one thread per
// internal node and every face per ray, 0.16 ms here.
constexpr int kMaxNear = 256;
__global__ void __launch_bounds__(kBlock)
    k_build_reflections(Grid g, float h, const uint8_t* __restrict__ flags,
                        const int32_t* __restrict__ nodes, int32_t nrec,
                        const float* __restrict__ verts, const int32_t* __restrict__ faces,
                        int32_t nf, const Box* __restrict__ boxes, HalfTurn ht,
                        uint32_t* __restrict__ dirs, float* __restrict__ weights) {
  using L = Lat<27>;
  constexpr int kWaves = kBlock / 64;
  __shared__ int32_t near_s[kWaves][kMaxNear];
  __shared__ float w_s[kWaves][84];
  __shared__ uint8_t d_s[kWaves][84];
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int32_t r = blockIdx.x * kWaves + wv;
  const bool live = r < nrec;
  const uint32_t n = live ? (uint32_t)nodes[r] : 0u;
  const uint32_t tq = g.dz.div(n);
  const int z = (int)(n - tq * g.nz), x = (int)g.dy.div(tq), y = (int)(tq - (uint32_t)x * g.ny);
  const int k = lane < 27 ? lane : 0;
  const int sx = x + L::E[k][0], sy = y + L::E[k][1], sz = z + L::E[k][2];
  const bool link = live && lane < 27 && is_free(g, flags, sx, sy, sz);
  // the free directions: links to follow and targets to reflect to
  const uint32_t open = (uint32_t)__ballot(link);
  for (int i = lane; i < 84; i += 64) {
    w_s[wv][i] = 0.0f;
    d_s[wv][i] = 0;
  }
  // faces near the node, in ascending order
  int32_t nnear = 0;
  if (live) {
    const float x0 = h * (float)(x - 1), x1 = h * (float)(x + 1), y0 = h * (float)(y - 1),
                y1 = h * (float)(y + 1), z0 = h * (float)(z - 1), z1 = h * (float)(z + 1);
    const float3 cl{fminf(x0, x1), fminf(y0, y1), fminf(z0, z1)};
    const float3 ch{fmaxf(x0, x1), fmaxf(y0, y1), fmaxf(z0, z1)};
    for (int32_t f0 = 0; f0 < nf; f0 += 64) {
      bool near = false;
      if (f0 + lane < nf) {
        const Box b = boxes[f0 + lane];
        // (written so that a box of NaNs is near everything)
        near = !(b.hi.x < cl.x || b.lo.x > ch.x || b.hi.y < cl.y || b.lo.y > ch.y ||
                 b.hi.z < cl.z || b.lo.z > ch.z);
      }
      const uint64_t m = __ballot(near);
      const int32_t at = nnear + __popcll(m & ((1ull << lane) - 1ull));
      if (near && at < kMaxNear) near_s[wv][at] = f0 + lane;
      nnear += __popcll(m);
    }
  }
  __syncthreads();
  if (link) {
    const F3 p1{h * (float)sx, h * (float)sy, h * (float)sz};
    const F3 p2{h * (float)x, h * (float)y, h * (float)z};
    const D3 o{(double)p1.x, (double)p1.y, (double)p1.z};
    const D3 d{(double)p2.x - p1.x, (double)p2.y - p1.y, (double)p2.z - p1.z};
    double t = INFINITY;
    int32_t best = -1;
    if (nnear <= kMaxNear)
      best = first_hit(o, d, verts, faces, nnear, [&](int32_t i) { return near_s[wv][i]; }, t);
    if (!(t <= 1.0)) best = first_hit(o, d, verts, faces, nf, [](int32_t i) { return i; }, t);
    const F3 v = reflection_vector(p1, p2, best, verts, faces, ht);
    // distribute_vector: scores of the 27 directions
    float score[27];
#pragma unroll
    for (int j = 0; j < 27; ++j) {
      const int len2 = L::E[j][0] * L::E[j][0] + L::E[j][1] * L::E[j][1] + L::E[j][2] * L::E[j][2];
      const double inv = len2 == 0 ? 0.0
                                   : (len2 == 1 ? 1.0
                                                : (len2 == 2 ? 1.0 / 1.4142135623730951
                                                             : 1.0 / 1.7320508075688772));
      float unit[3];
      for (int a = 0; a < 3; ++a) unit[a] = L::E[j][a] == 0 ? 0.0f : (float)(L::E[j][a] * inv);
      const float dx = v.x - unit[0], dy = v.y - unit[1], dz = v.z - unit[2];
      score[j] = (float)(2.0 - (double)sqrtf((dx * dx) + (dy * dy) + (dz * dz)));
    }
    const int base = L::INV[k] * 3;
    int counter = 0;
    float total = 0.0f;
    uint32_t taken = 0u;
    // the ranked list in order: highest score first, equal scores by
    // higher index first
    for (int rank = 0; rank < 27 && counter < 3; ++rank) {
      int best_j = -1;
      float best_s = 0.0f;
#pragma unroll
      for (int j = 26; j >= 0; --j) {
        if ((taken >> j) & 1u) continue;
        if (best_j < 0 || score[j] > best_s) {
          best_j = j;
          best_s = score[j];
        }
      }
      taken |= 1u << best_j;
      if (!((open >> best_j) & 1u)) continue;
      d_s[wv][base + counter] = (uint8_t)best_j;
      w_s[wv][base + counter] = best_s;
      total += best_s;
      ++counter;
    }
    if (total != 0.0f)
      for (int i = 0; i < 3; ++i)
        if (d_s[wv][base + i] != 0) w_s[wv][base + i] /= total;
  }
  __syncthreads();
  if (!live) return;
  for (int i = lane; i < 81; i += 64) weights[81 * (size_t)r + i] = w_s[wv][i];
  if (lane < 14) {
    uint32_t word = 0;
    for (int i = 0; i < 6; ++i) word |= (uint32_t)d_s[wv][6 * lane + i] << (5 * i);
    dirs[14 * (size_t)r + lane] = word;
  }
}

}  // namespace
}  // namespace lbm

// Entry points of include/lbm.h (exported by lbm_exports.hip).
namespace lbm {
namespace api {

int lbm_build_reflections(lbm_ctx* c, const float* vertices, int32_t nv,
                          const int32_t* faces, int32_t nf, float spacing,
                          int32_t max_records, int32_t* node, uint32_t* dirs,
                          float* weights, int32_t* count) {
  if (!c) return fail(LBM_ERR_INVALID, "null context");
  TraceRange tr("lbm_build_reflections");
  if (c->cfg.mode != LBM_MODE_REFERENCE)
    return fail(LBM_ERR_STATE, "lbm_build_reflections needs a reference-mode lattice");
  if (!count || nv < 0 || nf < 0 || max_records < 0 || (nf > 0 && (!vertices || !faces)) ||
      (max_records > 0 && (!node || !dirs || !weights)))
    return fail(LBM_ERR_INVALID, "bad arguments");
  for (int64_t k = 0; k < 3 * (int64_t)nf; ++k)
    if (faces[k] < 0 || faces[k] >= nv) return fail(LBM_ERR_INVALID, "face index out of range");
  *count = 0;
  // the host's half turn: angle pi in float, halved in double, cos / sin
  // of the float overloads
  const float angle = (float)M_PI;
  const float half = (float)((double)angle / 2.0);
  const HalfTurn ht{std::cos(half), std::sin(half), std::cos(-half), std::sin(-half)};
  const uint32_t N = c->grid.n;
  DevArena in;
  const size_t o_v = in.add(12 * (size_t)nv), o_f = in.add(12 * (size_t)nf),
               o_b = in.add(sizeof(Box) * (size_t)nf), o_s = in.add(4ull * scan_tiles(N)),
               o_n = in.add(4);
  int rc;
  if ((rc = in.alloc("hipMalloc(reflection build)"))) return rc;
  const LinkedIn linked{c->grid, c->flags};
  uint32_t* sums = in.at<uint32_t>(o_s);
  int32_t nrec = 0;
  if ((rc = launch_scan_sums(linked, N, sums, in.at<uint32_t>(o_n), c->stream))) return rc;
  LBM_HIP(hipMemcpyAsync(&nrec, in.at<int32_t>(o_n), 4, hipMemcpyDeviceToHost, c->stream));
  if (nv > 0)
    LBM_HIP(hipMemcpyAsync(in.at<float>(o_v), vertices, 12 * (size_t)nv, hipMemcpyHostToDevice, c->stream));
  if (nf > 0)
    LBM_HIP(hipMemcpyAsync(in.at<int32_t>(o_f), faces, 12 * (size_t)nf, hipMemcpyHostToDevice, c->stream));
  LBM_HIP(hipStreamSynchronize(c->stream));
  *count = nrec;
  if (nrec > max_records)
    return fail(LBM_ERR_INVALID, "max_records is smaller than the number of records");
  if (nrec == 0) return LBM_OK;
  DevArena out;
  const size_t o_node = out.add(4 * (size_t)nrec), o_dirs = out.add(56 * (size_t)nrec),
               o_w = out.add(324 * (size_t)nrec);
  if ((rc = out.alloc("hipMalloc(reflection records)"))) return rc;
  int32_t* dnode = out.at<int32_t>(o_node);
  if ((rc = launch_scan_write(linked, N, sums, NodeOut{dnode}, c->stream))) return rc;
  const float* dv = in.at<float>(o_v);
  const int32_t* df = in.at<int32_t>(o_f);
  Box* db = in.at<Box>(o_b);
  if (nf > 0)
    hipLaunchKernelGGL(k_face_boxes, dim3((nf + kBlock - 1) / kBlock), dim3(kBlock), 0, c->stream,
                       dv, df, nf, spacing, db);
  hipLaunchKernelGGL(k_build_reflections, dim3((nrec + kBlock / 64 - 1) / (kBlock / 64)),
                     dim3(kBlock), 0, c->stream, c->grid, spacing, c->flags, dnode, nrec, dv, df,
                     nf, db, ht, out.at<uint32_t>(o_dirs), out.at<float>(o_w));
  LBM_HIP(hipGetLastError());
  LBM_HIP(hipMemcpyAsync(node, dnode, 4 * (size_t)nrec, hipMemcpyDeviceToHost, c->stream));
  const HostPiece d{dirs, 56 * (size_t)nrec}, w{weights, 324 * (size_t)nrec};
  if ((rc = copy_to_host(out.at<uint32_t>(o_dirs), &d, 1, c->stream))) return rc;
  return copy_to_host(out.at<float>(o_w), &w, 1, c->stream);
}

int lbm_voxelize_mesh(lbm_ctx* c, const float* vertices, int32_t nv,
                      const int32_t* faces, int32_t nf, float spacing,
                      uint8_t* inside, int64_t* count) {
  if (!c) return fail(LBM_ERR_INVALID, "null context");
  TraceRange tr("lbm_voxelize_mesh");
  if (!inside || nv < 0 || nf < 0 || (nf > 0 && (!vertices || !faces)))
    return fail(LBM_ERR_INVALID, "bad mesh arguments");
  for (int64_t k = 0; k < 3 * (int64_t)nf; ++k)
    if (faces[k] < 0 || faces[k] >= nv) return fail(LBM_ERR_INVALID, "face index out of range");
  const Grid& g = c->grid;
  float3 lo{0.f, 0.f, 0.f}, hi{-1.f, -1.f, -1.f};  // empty box: nothing inside
  if (nv > 0) {
    lo = {vertices[0], vertices[1], vertices[2]};
    hi = lo;
    for (int32_t v = 1; v < nv; ++v) {
      lo.x = std::fmin(lo.x, vertices[3 * v]);
      hi.x = std::fmax(hi.x, vertices[3 * v]);
      lo.y = std::fmin(lo.y, vertices[3 * v + 1]);
      hi.y = std::fmax(hi.y, vertices[3 * v + 1]);
      lo.z = std::fmin(lo.z, vertices[3 * v + 2]);
      hi.z = std::fmax(hi.z, vertices[3 * v + 2]);
    }
    const float m = 1e-9f * std::fmax(std::fmax(hi.x - lo.x, hi.y - lo.y),
                                      std::fmax(hi.z - lo.z, 1e-30f));
    lo = {lo.x - m, lo.y - m, lo.z - m};
    hi = {hi.x + m, hi.y + m, hi.z + m};
  }
  if (nf == 0) {
    for (uint32_t n = 0; n < g.n; ++n) inside[n] = 0;
    if (count) *count = 0;
    return LBM_OK;
  }
  DevArena mem;
  const size_t o_v = mem.add(12 * (size_t)nv), o_f = mem.add(12 * (size_t)nf),
               o_b = mem.add(sizeof(Box) * (size_t)nf), o_in = mem.add(g.n), o_n = mem.add(8);
  int rc;
  if ((rc = mem.alloc("hipMalloc(voxelisation)"))) return rc;
  float* dv = mem.at<float>(o_v);
  int32_t* df = mem.at<int32_t>(o_f);
  uint8_t* dout = mem.at<uint8_t>(o_in);
  LBM_HIP(hipMemcpyAsync(dv, vertices, 12 * (size_t)nv, hipMemcpyHostToDevice, c->stream));
  LBM_HIP(hipMemcpyAsync(df, faces, 12 * (size_t)nf, hipMemcpyHostToDevice, c->stream));
  // where no node lies in the mesh's box no face is tested, and whether the
  // mesh closes need not be known (14,160 faces: 85 us, with the look at their
  // edges 199)
  const bool closes = !box_is_empty(g, spacing, lo, hi) && mesh_closes(vertices, faces, nf);
  if (closes) {
    unsigned long long* dn = mem.at<unsigned long long>(o_n);
    Box* db = mem.at<Box>(o_b);
    LBM_HIP(hipMemsetAsync(dn, 0, 8, c->stream));
    hipLaunchKernelGGL(k_face_boxes, dim3((nf + kBlock - 1) / kBlock), dim3(kBlock), 0, c->stream,
                       dv, df, nf, spacing, db);
    hipLaunchKernelGGL(k_voxelize_lines,
                       dim3((unsigned)((g.nx * g.ny + kBlock / 64 - 1) / (kBlock / 64))),
                       dim3(kBlock), 0, c->stream, g, spacing, dv, df, nf, db, lo, hi, dout, dn);
  } else {
    hipLaunchKernelGGL(k_voxelize, dim3((g.n + kBlock - 1) / kBlock), dim3(kBlock), 0, c->stream, g,
                       spacing, dv, df, nf, lo, hi, dout);
  }
  LBM_HIP(hipGetLastError());
  const HostPiece map{inside, g.n};
  if ((rc = copy_to_host(dout, &map, 1, c->stream))) return rc;
  unsigned long long total = 0;
  if (closes)
    LBM_HIP(hipMemcpyAsync(&total, mem.at<char>(o_n), 8, hipMemcpyDeviceToHost, c->stream));
  LBM_HIP(hipStreamSynchronize(c->stream));
  if (count && !closes)
    for (uint32_t n = 0; n < g.n; ++n) total += inside[n];
  if (count) *count = (int64_t)total;
  return LBM_OK;
}

}  // namespace api
}  // namespace lbm
