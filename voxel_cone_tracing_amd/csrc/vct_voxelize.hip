// vct_voxelize.hip - voxelisation (kernel a).
//
// Replaces the voxelize program: voxelize.vert:24-30 (world position divided
// by cube_size, normal by the inverse-transpose model matrix),
// voxelize.geom:25-55 (projection onto the plane of the dominant axis of
// |cross(e1, e2)|, ties to XZ), GL rasterisation at pixel centres of a
// 2res x 2res viewport (renderer.cpp:339-343), and voxelize.frag:122-161
// (per-fragment direct lighting and the collision average into the voxel at
// ivec3(res * (0.5 p + 0.5))).
//
// MI355X design
//  1. setup (one lane per triangle): dominant axis, vertices snapped to
//     1/256 pixel, pixel bounding box in 2x2 quads, a 128-byte record; each
//     triangle is counted into the 8^3-voxel bricks its voxel box overlaps.
//  2. exclusive scan of the brick counts, then per-brick triangle lists.
//  3. one workgroup per brick: the pixel rows of its triangles' boxes inside
//     the brick's footprint are spread over the lanes, which queue the pixels
//     of each row's span; those are tested with exact 64-bit edge functions
//     (top-left rule) from records in LDS, and only fragments whose voxel lies
//     in the brick are shaded, so every fragment is found exactly once.
//  4a. exact mean (any storage): 16.16 fixed-point sums in LDS (exact, so
//     order-independent); the workgroup writes its brick's texels once.
//  4b. reference running average (RGBA8): the workgroup takes its brick's
//     triangles in their original order, a round's fragments at a time in
//     LDS, and replays the packed RGBA8 + count-nibble recurrence of
//     imageAtomicRGBA8Avg (voxelize.frag:95-120) on each voxel's in canonical
//     order - the result does not depend on scheduling.
// Bit-exact parts (coverage, voxel coordinates, fragment colours) use no
// fused multiply-add and correctly rounded division / square root.
#include <cmath>
#include <cstring>

#include <algorithm>

#include "vct_internal.h"

namespace vct {

struct Draw {
  const float* pos;
  const float* nrm;
  const uint32_t* mat;
  const uint32_t* perm;  // stored -> original triangle index
  uint32_t tri_base;    // first triangle of this draw in the batch
  uint32_t canon_base;  // original index of the draw's first triangle in the frame
  uint32_t ntri;
  float M[16];  // model matrix, column-major
  float N[9];   // mat3(transpose(inverse(model))), column-major
};

// The queued draws of a frame, in queue order, in device memory (no limit on
// their number).
struct DrawTable {
  const Draw* d;
  int ndraw;
  uint32_t ntri;
};

struct VoxParams {
  uint32_t res;
  float inv_unused;
  float cube_size;
  int average;   // VCT_AVG_*
  uint32_t unused;
  LightSet lights;
  // normalize(position) of each directional light, computed on the host with
  // the same IEEE float operations (sqrt, then three divisions), so the bits
  // equal what every fragment would compute
  float ldir[VCT_MAX_LIGHTS][3];
};

struct Setup {
  float w[3][3];   // world / cube_size
  int64_t X[3], Y[3];
  int axis;
  int qx0, qy0, qw, qh;
  int64_t area;
  bool swap;
  bool ok;
};

// Per-triangle record written once by the setup pass and read by the brick
// workgroups (coverage fields through LDS, the rest for covered pixels).
struct alignas(16) TriRec {
  int64_t area;     // doubled signed area in 1/256 pixel units, made positive
  int32_t X[3], Y[3];
  int32_t qx0, qy0, qw;
  uint32_t mat;
  uint32_t flags;   // bit 0: vertices 1, 2 swapped (CW); bits 1-2: dominant axis; bits 8-31: qh
  float w[3][3];    // world position / cube_size per vertex
  float n[3][3];    // normalised transformed normal per vertex
  uint32_t otri;   // original triangle index in the frame (canonical order)
};
static_assert(sizeof(TriRec) == 128, "TriRec must be 128 bytes");

// The material terms a fragment of the triangle needs (voxelize.frag:139-155),
// gathered per triangle by the set-up kernel in frame order, so a fragment
// reads them by triangle index rather than through its record's material id
// (a dependent gather into the material table; on a soup of 1M triangles
// with a material each the brick pass went from 360 to 336 us).  They depend
// on the materials and the queued models only, so frames that change
// neither keep them.
struct alignas(16) VoxShade {
  float diffuse[3], alpha;   // alpha: the dissolve of a transmissive material, else 1
  float emission[3], pad0;
  float tr[3], pad1;         // the transmittance of a transmissive material, else 1 (1 * c == c)
};
static_assert(sizeof(VoxShade) == 48, "VoxShade must be 48 bytes");

__device__ __forceinline__ VoxShade make_shade(const DevMaterial& m) {
  VoxShade h;
  const bool t = illum_transmissive(m.illum);
  for (int k = 0; k < 3; ++k) {
    h.diffuse[k] = m.diffuse[k];
    h.emission[k] = m.emission[k];
    h.tr[k] = t ? m.transmittance[k] : 1.0f;
  }
  h.alpha = t ? m.dissolve : 1.0f;
  h.pad0 = h.pad1 = 0.0f;
  return h;
}

// The draw holding stored triangle t: the last one with tri_base <= t.
__device__ __forceinline__ int find_draw(const DrawTable& b, uint32_t t) {
  int lo = 0, hi = b.ndraw - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (b.d[mid].tri_base <= t) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// voxelize.vert:26 + voxelize.geom:27-51 + viewport + snap.
__device__ __forceinline__ void tri_setup(const Draw& dr, uint32_t lt, uint32_t res, float cube_size, Setup& s) {
#pragma clang fp contract(off)
  const float* p = dr.pos + (size_t)lt * 9;
  for (int v = 0; v < 3; ++v) {
    const float px = p[v * 3 + 0], py = p[v * 3 + 1], pz = p[v * 3 + 2];
    for (int k = 0; k < 3; ++k) {
      float t = dr.M[0 + k] * px;
      t = t + dr.M[4 + k] * py;
      t = t + dr.M[8 + k] * pz;
      t = t + dr.M[12 + k];
      s.w[v][k] = t / cube_size;
    }
  }
  float e1[3], e2[3];
  for (int k = 0; k < 3; ++k) {
    e1[k] = s.w[1][k] - s.w[0][k];
    e2[k] = s.w[2][k] - s.w[0][k];
  }
  float cx = fabsf(e1[1] * e2[2] - e1[2] * e2[1]);
  float cy = fabsf(e1[2] * e2[0] - e1[0] * e2[2]);
  float cz = fabsf(e1[0] * e2[1] - e1[1] * e2[0]);
  int axis, ia, ib;
  if (cz > cx && cz > cy) {
    axis = 2; ia = 0; ib = 1;   // XY plane
  } else if (cx > cy && cx > cz) {
    axis = 0; ia = 1; ib = 2;   // YZ plane
  } else {
    axis = 1; ia = 0; ib = 2;   // XZ plane
  }
  s.axis = axis;
  const float fres = (float)res;
  bool ok = true;
  for (int v = 0; v < 3; ++v) {
    float a = s.w[v][ia], b = s.w[v][ib];
    if (!(fabsf(a) < 64.0f && fabsf(b) < 64.0f)) ok = false;
    float xw = a * fres + fres;  // viewport transform, scale = translate = res
    float yw = b * fres + fres;
    s.X[v] = (int64_t)__builtin_rintf((xw - 0.5f) * 256.0f);
    s.Y[v] = (int64_t)__builtin_rintf((yw - 0.5f) * 256.0f);
  }
  int64_t area = (s.X[1] - s.X[0]) * (s.Y[2] - s.Y[0]) - (s.Y[1] - s.Y[0]) * (s.X[2] - s.X[0]);
  s.swap = area < 0;
  s.area = area < 0 ? -area : area;
  if (area == 0) ok = false;
  int64_t xmin = min(s.X[0], min(s.X[1], s.X[2])), xmax = max(s.X[0], max(s.X[1], s.X[2]));
  int64_t ymin = min(s.Y[0], min(s.Y[1], s.Y[2])), ymax = max(s.Y[0], max(s.Y[1], s.Y[2]));
  const int64_t lim = 2 * (int64_t)res - 1;
  int64_t imin = (xmin + 255) >> 8, imax = xmax >> 8, jmin = (ymin + 255) >> 8, jmax = ymax >> 8;
  imin = imin < 0 ? 0 : imin;
  jmin = jmin < 0 ? 0 : jmin;
  imax = imax > lim ? lim : imax;
  jmax = jmax > lim ? lim : jmax;
  if (imin > imax || jmin > jmax) ok = false;
  s.ok = ok;
  if (ok) {
    s.qx0 = (int)(imin & ~1ll);
    s.qy0 = (int)(jmin & ~1ll);
    s.qw = (int)((imax - s.qx0) >> 1) + 1;
    s.qh = (int)((jmax - s.qy0) >> 1) + 1;
  } else {
    s.qx0 = s.qy0 = s.qw = s.qh = 0;
  }
}

// Record of a triangle that passed setup (s.ok).
__device__ __forceinline__ TriRec make_rec(const Draw& dr, uint32_t lt, const Setup& s) {
#pragma clang fp contract(off)
  TriRec r;
  r.area = s.area;
  for (int v = 0; v < 3; ++v) {
    r.X[v] = (int32_t)s.X[v];
    r.Y[v] = (int32_t)s.Y[v];
    for (int k = 0; k < 3; ++k) r.w[v][k] = s.w[v][k];
  }
  r.qx0 = s.qx0;
  r.qy0 = s.qy0;
  r.qw = s.qw;
  r.mat = dr.mat[lt];
  r.flags = (s.swap ? 1u : 0u) | ((uint32_t)s.axis << 1) | ((uint32_t)s.qh << 8);
  r.otri = dr.canon_base + dr.perm[lt];
  // normal: voxelize.vert:28 per vertex (normalize(N * n))
  const float* nr = dr.nrm + (size_t)lt * 9;
  for (int v = 0; v < 3; ++v) {
    float tt[3];
    for (int k = 0; k < 3; ++k) {
      float a = dr.N[0 + k] * nr[v * 3 + 0];
      a = a + dr.N[3 + k] * nr[v * 3 + 1];
      a = a + dr.N[6 + k] * nr[v * 3 + 2];
      tt[k] = a;
    }
    const float l = sqrtf(tt[0] * tt[0] + tt[1] * tt[1] + tt[2] * tt[2]);
    for (int k = 0; k < 3; ++k) r.n[v][k] = tt[k] / l;
  }
  return r;
}

__device__ __forceinline__ bool top_left(int64_t dx, int64_t dy) { return dy < 0 || (dy == 0 && dx < 0); }

// Edge functions of a record in CCW order (a, b, c) = (0, 1, 2) or (0, 2, 1)
// at pixel (i, j), and their exact per-column / per-row increments.
struct VEdges {
  int64_t w[3];
  int64_t ex[3], ey[3];
};

// Differences of snapped coordinates fit 32 bits (vertices lie within 65
// grid widths of the origin: |X|, |Y| < 2^25 in 1/256 pixel, and 256 i,
// 256 j < 2^20), so every product is a 32 x 32 -> 64-bit multiply.
template <typename Rec>
__device__ __forceinline__ void vox_edges(const Rec& s, int i, int j, VEdges& e) {
  const int32_t px = i * 256, py = j * 256;
  const bool sw = (s.flags & 1u) != 0u;
  const int32_t ax = s.X[0], ay = s.Y[0];
  const int32_t bx = sw ? s.X[2] : s.X[1], by = sw ? s.Y[2] : s.Y[1];
  const int32_t cx = sw ? s.X[1] : s.X[2], cy = sw ? s.Y[1] : s.Y[2];
  e.w[0] = (int64_t)(cx - bx) * (int64_t)(py - by) - (int64_t)(cy - by) * (int64_t)(px - bx);
  e.w[1] = (int64_t)(ax - cx) * (int64_t)(py - cy) - (int64_t)(ay - cy) * (int64_t)(px - cx);
  e.w[2] = (int64_t)(bx - ax) * (int64_t)(py - ay) - (int64_t)(by - ay) * (int64_t)(px - ax);
  e.ex[0] = cx - bx;
  e.ey[0] = cy - by;
  e.ex[1] = ax - cx;
  e.ey[1] = ay - cy;
  e.ex[2] = bx - ax;
  e.ey[2] = by - ay;
}

// Fragment at pixel (i, j) of the triangle's 2res x 2res raster given its
// edge values (wa, wb, wc): coverage, voxel (Morton index) and colour.
// Returns false if the pixel is not covered or the voxel falls outside the
// grid (with kBrick: also when the voxel's Morton index >> bshift is not
// bwant, before any shading).
// `c` holds the coverage fields (X, Y, area, flags), `sp` the whole record
// and `sh` the triangle's material terms (both read only for covered pixels).
template <bool kBrick = false, typename Rec>
__device__ __forceinline__ bool shade_w(const Rec& c, const TriRec* sp, const VoxShade* sh, const VEdges& e, int i,
                                        int j, int64_t wa, int64_t wb, int64_t wc, const VoxParams& vp,
                                        uint32_t& key, float4& color, uint32_t bshift = 0, uint32_t bwant = 0) {
#pragma clang fp contract(off)
  const int lim = 2 * (int)vp.res;
  if (i >= lim || j >= lim) return false;
  const bool sw = (c.flags & 1u) != 0u;
  if (wa < 0 || wb < 0 || wc < 0) return false;
  if (wa == 0 && !top_left(e.ex[0], e.ey[0])) return false;
  if (wb == 0 && !top_left(e.ex[1], e.ey[1])) return false;
  if (wc == 0 && !top_left(e.ex[2], e.ey[2])) return false;
  // weights of the original vertices 0, 1, 2
  const int64_t w0 = wa, w1 = sw ? wc : wb, w2 = sw ? wb : wc;
  const float fa = (float)c.area;
  const float b0 = (float)w0 / fa, b1 = (float)w1 / fa, b2 = (float)w2 / fa;
  const TriRec& s = *sp;
  float pos[3];
  for (int k = 0; k < 3; ++k) pos[k] = b0 * s.w[0][k] + b1 * s.w[1][k] + b2 * s.w[2][k];
  // voxel address, voxelize.frag:156-157 (truncation toward zero)
  int v[3];
  const float fres = (float)vp.res;
  for (int k = 0; k < 3; ++k) {
    float f = fres * (0.5f * pos[k] + 0.5f);
    if (!(f > -1.0f && f < fres)) return false;
    v[k] = (int)f;
  }
  key = brick_index((uint32_t)v[0], (uint32_t)v[1], (uint32_t)v[2]);
  if (kBrick && (key >> bshift) != bwant) return false;
  // normal: per-vertex normals (record), interpolated, normalised in the
  // fragment shader (voxelize.frag:134)
  float n[3];
  for (int k = 0; k < 3; ++k) n[k] = b0 * s.n[0][k] + b1 * s.n[1][k] + b2 * s.n[2][k];
  {
    float l = sqrtf(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
    for (int k = 0; k < 3; ++k) n[k] = n[k] / l;
  }
  // lighting, voxelize.frag:127-143
  float col[3] = {0.0f, 0.0f, 0.0f};
  const int nl = vp.lights.count < VCT_MAX_LIGHTS ? vp.lights.count : VCT_MAX_LIGHTS;
  for (int li = 0; li < nl; ++li) {
    const DevLight& L = vp.lights.l[li];
    float dir[3];
    float att;
    if (L.kind == VCT_LIGHT_DIRECTIONAL) {
      for (int k = 0; k < 3; ++k) dir[k] = vp.ldir[li][k];
      att = 1.0f;
    } else {
      float dv[3];
      for (int k = 0; k < 3; ++k) dv[k] = L.pos[k] / vp.cube_size - pos[k];
      float d = sqrtf(dv[0] * dv[0] + dv[1] * dv[1] + dv[2] * dv[2]);
      for (int k = 0; k < 3; ++k) dir[k] = dv[k] / d;
      att = 1.0f / (1.0f + d * d);
    }
    float c = n[0] * dir[0] + n[1] * dir[1] + n[2] * dir[2];
    c = c > 0.0f ? c : 0.0f;
    float ca = c * att;
    for (int k = 0; k < 3; ++k) col[k] = col[k] + ca * L.color[k] * L.intensity;
  }
  const VoxShade m = *sh;
  float out[4];
  for (int k = 0; k < 3; ++k) {
    float c = m.diffuse[k] * col[k] + m.emission[k];
    out[k] = m.tr[k] * c;
  }
  out[3] = m.alpha;
  for (int k = 0; k < 4; ++k) out[k] = fminf(fmaxf(out[k], 0.0f), 1.0f);
  color = make_float4(out[0], out[1], out[2], out[3]);
  return true;
}

// ---- exact mean: bricks of the grid accumulated in LDS ----------------------
// The grid is cut into cubes of kBrick^3 voxels (4^3 on small grids, brick_edge);
// a brick is one contiguous run of the Morton-ordered level 0, and the low
// 3 * log2(edge) bits of a voxel's Morton index are its index inside the
// brick.  Triangles are binned to the bricks their voxel bounding box
// overlaps; one workgroup per brick rasterises its triangles' pixels inside
// the brick's footprint on the projection plane, keeps the fragments whose
// voxel lies in the brick, and sums them in LDS as 16.16 fixed point (exact,
// so the order of the additions does not matter).  It then writes the
// brick's level-0 texels (mean = sum / count, 0 where empty) once.  8^3
// bricks with 256-lane workgroups (10 KiB of sums, several workgroups per CU)
// measured 15 % faster than 16^3 bricks with 1024 lanes (80 KiB, one per CU),
// which pay more for workgroup barriers and the load imbalance of the bricks
// than they save on triangles shared by neighbouring bricks.
constexpr int kBrick = 8;
constexpr int kBrickThreads = 256;
// (triangle, brick) items staged per round: a brick holds ~58 items on
// average (1.9 M over 32,768 bricks of a 1M-triangle soup at 256^3), so
// rounds of 128 rarely repeat, and the smaller stage leaves LDS for a 7th
// workgroup per CU (the registers' limit) where 256 allowed 6
constexpr int kBrickItems = 128;

// Grids up to 32^3 would be 64 bricks or fewer of 8^3, a quarter of the CUs
// with a workgroup each, and take bricks of 4^3: 103,000 triangles at 32^3
// voxelize in 0.07 ms instead of 0.18 (8^3 bricks), 1,700 in 0.047 instead of
// 0.10.  At 64^3 (512 bricks of 8^3) soups gain a fifth, but 34 triangles the
// size of the grid lose 5 %: the larger edge stays.
__host__ __device__ inline uint32_t brick_edge(uint32_t res) { return res <= 32u ? 4u : (uint32_t)kBrick; }

struct BrickGeom {
  uint32_t bits;    // log2(brick edge)
  uint32_t per;     // bricks per grid edge
};

__device__ __forceinline__ BrickGeom brick_geom(uint32_t res) {
  BrickGeom g;
  g.bits = 31u - __clz(brick_edge(res));
  g.per = res >> g.bits;
  return g;
}

struct BrickBox {
  int b0[3], nb[3];
  int n;
};

// Bricks overlapped by the voxel bounding box of a set-up triangle.  Fragment
// positions are convex combinations of the vertices up to rounding; 0.01
// voxel of margin covers it.
__device__ __forceinline__ BrickBox brick_box(const float (&pw)[3][3], bool ok, uint32_t res, BrickGeom g) {
#pragma clang fp contract(off)
  BrickBox bb;
  bb.n = 0;
  if (!ok) return bb;
  const float fres = (float)res;
  bb.n = 1;
  for (int k = 0; k < 3; ++k) {
    float lo = 3.0e38f, hi = -3.0e38f;
    for (int v = 0; v < 3; ++v) {
      const float f = fres * (0.5f * pw[v][k] + 0.5f);
      lo = fminf(lo, f);
      hi = fmaxf(hi, f);
    }
    lo -= 0.01f;
    hi += 0.01f;
    if (!(hi > -1.0f && lo < fres)) {  // every fragment would be dropped
      bb.n = 0;
      return bb;
    }
    const int vlo = lo <= 0.0f ? 0 : (int)lo;
    const int vhi = hi >= fres - 1.0f ? (int)res - 1 : (int)hi;
    bb.b0[k] = vlo >> g.bits;
    bb.nb[k] = (vhi >> g.bits) - bb.b0[k] + 1;
    bb.n *= bb.nb[k];
  }
  return bb;
}

__device__ __forceinline__ BrickBox brick_box(const Setup& s, uint32_t res, BrickGeom g) {
  return brick_box(s.w, s.ok, res, g);
}

__device__ __forceinline__ uint32_t brick_of(const BrickBox& bb, int k) {
  const int x = bb.b0[0] + k % bb.nb[0];
  const int y = bb.b0[1] + (k / bb.nb[0]) % bb.nb[1];
  const int z = bb.b0[2] + k / (bb.nb[0] * bb.nb[1]);
  return morton3((uint32_t)x, (uint32_t)y, (uint32_t)z);
}

// The brick box of a triangle packed into 8 bytes for the list write: first
// brick per axis, then bricks per axis (0: no brick), 8 bits each (at most
// 128 bricks per axis).
__device__ __forceinline__ uint2 pack_box(const BrickBox& bb) {
  if (bb.n == 0) return make_uint2(0u, 0u);
  return make_uint2((uint32_t)bb.b0[0] | ((uint32_t)bb.b0[1] << 8) | ((uint32_t)bb.b0[2] << 16),
                    (uint32_t)bb.nb[0] | ((uint32_t)bb.nb[1] << 8) | ((uint32_t)bb.nb[2] << 16));
}
__device__ __forceinline__ BrickBox unpack_box(uint2 p) {
  BrickBox bb;
  for (int k = 0; k < 3; ++k) {
    bb.b0[k] = (int)((p.x >> (8 * k)) & 255u);
    bb.nb[k] = (int)((p.y >> (8 * k)) & 255u);
  }
  bb.n = bb.nb[0] * bb.nb[1] * bb.nb[2];
  return bb;
}

// The bricks of a box as a triangle needs them.  A box of few bricks is
// counted whole, lane by lane with one atomic per distinct brick of the wave
// (neighbouring triangles share bricks).  Larger ones would hold their wave
// for a round trip per brick and put the triangle into many bricks it never
// touches, so the wave takes them one after another, its lanes over the
// triangle's bricks, and drops those the triangle cannot reach.
// Measured: the 34 triangles of the Cornell box at 64^3, count 67 and list
// write 89 us before; 4,000 triangles of 0.17 edge at 128^3, 99 and 154 us.
constexpr int kSmallBox = 8;

// False only where no fragment of the triangle can fall in brick `b` of its
// box: the brick's footprint on the projection plane lies outside an edge
// (exact integers, over the pixels the brick pass would test), or the
// triangle's plane passes the brick by.  The plane test is in float with
// margins far above its rounding (a quarter voxel, 2^-12 of the distance to
// vertex 0); a sliver whose normal is all rounding is kept.  No contraction:
// the count and the list write must decide alike.
__device__ __forceinline__ bool brick_reached(const TriRec& r, const int (&b)[3], uint32_t res, BrickGeom g) {
#pragma clang fp contract(off)
  const int axis = (int)((r.flags >> 1) & 3u);
  const int ia = axis == 0 ? 1 : 0, ib = axis == 2 ? 1 : 2;
  const int span = 2 << g.bits, lim = 2 * (int)res - 1;
  const int fx = (ia == 0 ? b[0] : b[1]) * span, fy = (ib == 1 ? b[1] : b[2]) * span;
  const int i0 = max(r.qx0, fx), i1 = min(min(r.qx0 + 2 * r.qw - 1, fx + span - 1), lim);
  const int j0 = max(r.qy0, fy), j1 = min(min(r.qy0 + 2 * (int)(r.flags >> 8) - 1, fy + span - 1), lim);
  if (i1 < i0 || j1 < j0) return false;
  VEdges e;
  vox_edges(r, i0, j0, e);
  const int64_t dw = 256 * (int64_t)(i1 - i0), dh = 256 * (int64_t)(j1 - j0);
  for (int k = 0; k < 3; ++k)  // w(i, j) = w + ex * 256 (j - j0) - ey * 256 (i - i0)
    if (e.w[k] + max((int64_t)0, e.ex[k] * dh) + max((int64_t)0, -e.ey[k] * dw) < 0) return false;
  // the plane against the brick, in voxels
  const float s = 0.5f * (float)res, h = 0.5f * (float)(1 << g.bits);
  float e1[3], e2[3], c[3], hx[3];
  for (int k = 0; k < 3; ++k) {
    e1[k] = (r.w[1][k] - r.w[0][k]) * s;
    e2[k] = (r.w[2][k] - r.w[0][k]) * s;
    c[k] = ((float)(b[k] << g.bits) + h) - (r.w[0][k] * s + s);
    hx[k] = h + 0.25f;
    if (b[k] == 0) hx[k] = h + 1.25f;  // fragments up to a voxel below the grid fall in its first voxel
  }
  const float n[3] = {e1[1] * e2[2] - e1[2] * e2[1], e1[2] * e2[0] - e1[0] * e2[2], e1[0] * e2[1] - e1[1] * e2[0]};
  const float nn = fabsf(n[0]) + fabsf(n[1]) + fabsf(n[2]);
  const float l1 = fabsf(e1[0]) + fabsf(e1[1]) + fabsf(e1[2]), l2 = fabsf(e2[0]) + fabsf(e2[1]) + fabsf(e2[2]);
  if (!(nn > 1e-2f * l1 * l2)) return true;
  const float d = fabsf(n[0] * c[0] + n[1] * c[1] + n[2] * c[2]);
  const float far = fabsf(c[0]) + fabsf(c[1]) + fabsf(c[2]);
  const float reach = fabsf(n[0]) * hx[0] + fabsf(n[1]) * hx[1] + fabsf(n[2]) * hx[2];
  return !(d > reach + nn * far * 2.44140625e-4f);
}

__device__ __forceinline__ void brick_at(const BrickBox& bb, int k, int (&b)[3]) {
  b[0] = bb.b0[0] + k % bb.nb[0];
  b[1] = bb.b0[1] + (k / bb.nb[0]) % bb.nb[1];
  b[2] = bb.b0[2] + k / (bb.nb[0] * bb.nb[1]);
}

// 1. setup (1 << lsh lanes per stored triangle, the first of them sets it up):
//    record + count into overlapped bricks.
__global__ __launch_bounds__(256) void vox_brick_count_kernel(DrawTable b, VoxParams vp, TriRec* __restrict__ recs,
                                                              const DevMaterial* __restrict__ mats,
                                                              VoxShade* __restrict__ shade, bool build_shade,
                                                              uint2* __restrict__ boxes, uint32_t* brick_count,
                                                              int lsh) {
  // each wave's records (128 B each, consecutive in memory) go out through
  // LDS as lane-contiguous 16-byte stores instead of one record per lane
  // (stride 9: a padded record, so the lanes' 16-byte pieces spread over banks)
  __shared__ uint4 s_out[4][64 * 9];
  const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t t = gid >> lsh;
  const bool own = (gid & ((1u << lsh) - 1u)) == 0u && t < b.ntri;
  const int slot = lane >> lsh, nrec = 64 >> lsh;      // the triangle's place in its wave, triangles per wave
  const uint32_t t0 = (gid - (uint32_t)lane) >> lsh;   // the wave's first triangle
  const BrickGeom g = brick_geom(vp.res);
  Setup s;
  s.ok = false;
  TriRec rec;
  memset(&rec, 0, sizeof(rec));  // a skipped triangle keeps area 0 (set-up triangles have area > 0)
  VoxShade h;
  memset(&h, 0, sizeof(h));
  if (own) {
    const int d = find_draw(b, t);
    const Draw& dr = b.d[d];
    const uint32_t lt = t - dr.tri_base;
    // every stored triangle's material id indexes the table (a default
    // material always exists), so the gather goes out before the set-up's
    // arithmetic instead of after its result
    DevMaterial m;
    if (build_shade) m = mats[dr.mat[lt]];
    tri_setup(dr, lt, vp.res, vp.cube_size, s);
    if (s.ok) rec = make_rec(dr, lt, s);
    if (build_shade) h = make_shade(m);  // also of a triangle that draws nothing in this frame
  }
  const BrickBox bb = brick_box(s, vp.res, g);
  uint4* w = s_out[wave];
  {
    const uint4* rp = reinterpret_cast<const uint4*>(&rec);
    if ((lane & ((1 << lsh) - 1)) == 0) {
#pragma unroll
      for (int q = 0; q < 8; ++q) w[slot * 9 + q] = rp[q];
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    uint4* out = reinterpret_cast<uint4*>(recs + t0);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int c = k * 64 + lane;  // 16-byte piece c of the wave's records: record c / 8, piece c % 8
      if ((c >> 3) < nrec && t0 + (uint32_t)(c >> 3) < b.ntri) out[c] = w[(c >> 3) * 9 + (c & 7)];
    }
  }
  if (own) boxes[t] = pack_box(bb);
  const int nsmall = bb.n <= kSmallBox ? bb.n : 0;
  for (int k = 0; __ballot(k < nsmall) != 0ull; ++k) {
    const bool act = k < nsmall;
    wave_add_one(brick_count, act ? brick_of(bb, k) : 0u, act);
  }
  for (unsigned long long big = __ballot(bb.n > kSmallBox); big; big &= big - 1ull) {
    const int lead = __ffsll((long long)big) - 1;
    BrickBox bx;
    for (int k = 0; k < 3; ++k) {
      bx.b0[k] = __builtin_amdgcn_readlane(bb.b0[k], lead);
      bx.nb[k] = __builtin_amdgcn_readlane(bb.nb[k], lead);
    }
    bx.n = bx.nb[0] * bx.nb[1] * bx.nb[2];
    const TriRec& r = *reinterpret_cast<const TriRec*>(&w[(lead >> lsh) * 9]);
    for (int k = lane; k < bx.n; k += 64) {
      int bk[3];
      brick_at(bx, k, bk);
      if (brick_reached(r, bk, vp.res, g))
        atomicAdd(brick_count + morton3((uint32_t)bk[0], (uint32_t)bk[1], (uint32_t)bk[2]), 1u);
    }
  }
  if (build_shade) {
    // the material terms the same way as the records (48 B per triangle: a
    // stride of three 16-byte pieces spreads over the banks unpadded)
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    const uint4* hp = reinterpret_cast<const uint4*>(&h);
    if ((lane & ((1 << lsh) - 1)) == 0) {
#pragma unroll
      for (int q = 0; q < 3; ++q) w[slot * 3 + q] = hp[q];
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    uint4* hout = reinterpret_cast<uint4*>(shade + t0);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int c = k * 64 + lane;  // piece c of the wave's material terms: triangle c / 3
      if (c / 3 < nrec && t0 + (uint32_t)c / 3u < b.ntri) hout[c] = w[c];
    }
  }
}

// 3. list write (1 << lsh lanes per triangle): the same brick boxes, as the
//    setup packed them.  Entries at or past `cap` are not written (their
//    bricks walk the boxes instead).
__global__ __launch_bounds__(256) void vox_brick_write_kernel(uint32_t ntri, uint32_t res,
                                                              const TriRec* __restrict__ recs,
                                                              const uint2* __restrict__ boxes,
                                                              const uint32_t* __restrict__ brick_off,
                                                              uint32_t* cursor, uint32_t* __restrict__ list,
                                                              uint32_t cap, int lsh) {
  const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = threadIdx.x & 63;
  const uint32_t t = gid >> lsh;
  const bool own = (gid & ((1u << lsh) - 1u)) == 0u && t < ntri;
  const BrickGeom g = brick_geom(res);
  const BrickBox bb = unpack_box(own ? boxes[t] : make_uint2(0u, 0u));
  const int nsmall = bb.n <= kSmallBox ? bb.n : 0;
  for (int k = 0; __ballot(k < nsmall) != 0ull; ++k) {
    const bool act = k < nsmall;
    const uint32_t key = act ? brick_of(bb, k) : 0u;
    const uint32_t slot = wave_add_one(cursor, key, act);
    if (act && (uint64_t)brick_off[key] + slot < (uint64_t)cap) list[brick_off[key] + slot] = t;
  }
  for (unsigned long long big = __ballot(bb.n > kSmallBox); big; big &= big - 1ull) {
    const int lead = __ffsll((long long)big) - 1;
    BrickBox bx;
    for (int k = 0; k < 3; ++k) {
      bx.b0[k] = __builtin_amdgcn_readlane(bb.b0[k], lead);
      bx.nb[k] = __builtin_amdgcn_readlane(bb.nb[k], lead);
    }
    bx.n = bx.nb[0] * bx.nb[1] * bx.nb[2];
    const uint32_t tl = (uint32_t)__builtin_amdgcn_readlane((int)t, lead);
    const TriRec& r = recs[tl];
    for (int k = lane; k < bx.n; k += 64) {
      int bk[3];
      brick_at(bx, k, bk);
      if (!brick_reached(r, bk, res, g)) continue;
      const uint32_t key = morton3((uint32_t)bk[0], (uint32_t)bk[1], (uint32_t)bk[2]);
      const uint32_t slot = atomicAdd(cursor + key, 1u);
      if ((uint64_t)brick_off[key] + slot < (uint64_t)cap) list[brick_off[key] + slot] = tl;
    }
  }
}

__device__ __forceinline__ uint32_t fixq(float c) { return (uint32_t)(c * 65536.0f + 0.5f); }

// mean of 16.16 fixed-point sums -> stored texel
template <int DT>
__device__ __forceinline__ void store_mean(void* level0, uint32_t v, uint32_t cnt, uint32_t r, uint32_t g, uint32_t b,
                                           uint32_t a) {
#pragma clang fp contract(off)
  float4 m = make_float4(0.f, 0.f, 0.f, 0.f);
  if (cnt) {
    const float fc = (float)cnt;
    const float s = 1.0f / 65536.0f;
    m.x = ((float)r / fc) * s;
    m.y = ((float)g / fc) * s;
    m.z = ((float)b / fc) * s;
    m.w = ((float)a / fc) * s;
  }
  if (DT == VCT_RGBA8) {
    reinterpret_cast<uint32_t*>(level0)[v] =
        to_unorm8(m.x) | (to_unorm8(m.y) << 8) | (to_unorm8(m.z) << 16) | (to_unorm8(m.w) << 24);
  } else if (DT == VCT_FP16) {
    reinterpret_cast<uint2*>(level0)[v] =
        make_uint2((uint32_t)f32_to_f16(m.x) | ((uint32_t)f32_to_f16(m.y) << 16),
                   (uint32_t)f32_to_f16(m.z) | ((uint32_t)f32_to_f16(m.w) << 16));
  } else if (DT == VCT_BF16) {
    reinterpret_cast<uint2*>(level0)[v] =
        make_uint2((uint32_t)f32_to_bf16(m.x) | ((uint32_t)f32_to_bf16(m.y) << 16),
                   (uint32_t)f32_to_bf16(m.z) | ((uint32_t)f32_to_bf16(m.w) << 16));
  } else {
    reinterpret_cast<float4*>(level0)[v] = m;
  }
}

// 4. one workgroup per brick (each workgroup maps its index to one brick's
//    Morton index, one to one).  The brick's triangles are taken kBrickItems
//    at a time; the pixel rows of their boxes inside the brick's footprint on
//    the projection plane are spread over the lanes (a lane finds its triangle
//    from the prefix of the row counts), the pixels of the rows' spans are
//    tested from a compact copy of the records in LDS, and only covered pixels
//    read the rest of the record.
struct CovRec {  // the coverage fields of a TriRec
  int64_t area;
  int32_t X[3], Y[3];
  uint32_t flags;
  uint32_t tri;
};

__device__ __forceinline__ void brick_add(uint32_t (*s_sum)[kBrick * kBrick * kBrick], uint32_t* s_cnt, uint32_t v,
                                          float4 color) {
  atomicAdd(&s_sum[0][v], fixq(color.x));
  atomicAdd(&s_sum[1][v], fixq(color.y));
  atomicAdd(&s_sum[2][v], fixq(color.z));
  atomicAdd(&s_sum[3][v], fixq(color.w));
  atomicAdd(&s_cnt[v], 1u);
}

// ---- reference running average -------------------------------------------
__device__ __forceinline__ uint32_t conv_vec4_to_rgba8(float x, float y, float z, float w) {
  // voxelize.frag:66-71: uint() truncation, & 0xFF
  return (((uint32_t)w & 0xffu) << 24) | (((uint32_t)z & 0xffu) << 16) | (((uint32_t)y & 0xffu) << 8) |
         ((uint32_t)x & 0xffu);
}
__device__ __forceinline__ uint32_t enc_nibble(uint32_t m, uint32_t n) {
  return (m & 0xFEFEFEFEu) | (n & 1u) | ((n & 2u) << 7) | ((n & 4u) << 14) | ((n & 8u) << 21);
}
__device__ __forceinline__ uint32_t dec_nibble(uint32_t m) {
  return (m & 1u) | ((m & 0x100u) >> 7) | ((m & 0x10000u) >> 14) | ((m & 0x1000000u) >> 21);
}

// One fragment (vx .. vw: its colour times 255) into a voxel's packed RGBA8 +
// count nibble, as imageAtomicRGBA8Avg does (voxelize.frag:95-120).
__device__ __forceinline__ uint32_t replay_step(uint32_t stored, float vx, float vy, float vz, float vw) {
#pragma clang fp contract(off)
  if (stored == 0u)  // imageAtomicCompSwap(0 -> new) succeeds
    return enc_nibble(conv_vec4_to_rgba8(vx, vy, vz, vw), 1u);
  const uint32_t cur = stored & 0xFEFEFEFEu;
  float rx = (float)(cur & 0xffu), ry = (float)((cur >> 8) & 0xffu), rz = (float)((cur >> 16) & 0xffu),
        rw = (float)(cur >> 24);
  uint32_t n = dec_nibble(stored);
  const float fn = (float)n;
  rx = rx * fn + vx;
  ry = ry * fn + vy;
  rz = rz * fn + vz;
  rw = rw * fn + vw;
  ++n;
  // x / n correctly rounded for n = 1 .. 16: the rounded reciprocal (one
  // Newton step from the approximation), the product and one correction by its
  // exact remainder (compared for every n and mantissa); 4 divisions cost four
  // times as many cycles
  const float fn1 = (float)n;
  float inv = __builtin_amdgcn_rcpf(fn1);
  inv = __builtin_fmaf(__builtin_fmaf(-fn1, inv, 1.0f), inv, inv);
  auto div = [&](float x) {
    const float q = x * inv;
    return __builtin_fmaf(__builtin_fmaf(-fn1, q, x), inv, q);
  };
  rx = div(rx);
  ry = div(ry);
  rz = div(rz);
  rw = div(rw);
  rx = __builtin_rintf(rx / 2.0f) * 2.0f;
  ry = __builtin_rintf(ry / 2.0f) * 2.0f;
  rz = __builtin_rintf(rz / 2.0f) * 2.0f;
  rw = __builtin_rintf(rw / 2.0f) * 2.0f;
  return enc_nibble(conv_vec4_to_rgba8(rx, ry, rz, rw), n);
}

// The brick lists' capacity: a brick whose range [off, off + count) runs past
// `cap` entries walks the packed brick boxes of all `ntri` triangles and keeps
// those that contain it: the triangles of its list, and ones that its list
// leaves out because they do not reach it, which give no fragment in it.
struct ListCap {
  const uint2* boxes;
  uint32_t ntri;
  uint32_t cap;
};

// A round of up to kBrickItems triangles of a brick, in LDS.
struct BrickRound {
  CovRec cov[kBrickItems];
  uint32_t end[kBrickItems];  // inclusive prefix of the row counts
  uint32_t org[kBrickItems];  // clipped box: i | j << 11 | width << 22 (width at most 16)
  uint32_t wsum[kBrickItems / 64];
  uint32_t q[kBrickThreads / 64][128];  // per-wave queue of pixels inside the spans
};

// Stages triangle t as entry `slot` of the round for the brick at bc (bricks);
// returns its rows: those of its box clipped to the brick's footprint.  A
// covered pixel (i, j) lands in voxel (i >> 1, j >> 1) on the projection
// plane: its centre sits a quarter voxel inside that voxel, and the
// interpolated position is a convex combination of the vertices that differs
// from the centre by the 1/512-pixel vertex snap plus rounding, far below a
// quarter voxel.  So pixels outside the footprint never land in the brick.
__device__ __forceinline__ uint32_t brick_stage(BrickRound& B, int slot, uint32_t t, const TriRec* __restrict__ recs,
                                                const uint32_t (&bc)[3], int span, int lim) {
  const TriRec* rp = recs + t;
  const uint32_t fl = rp->flags;
  const int axis = (int)((fl >> 1) & 3u);
  const int ia = axis == 0 ? 1 : 0, ib = axis == 2 ? 1 : 2;
  const int qh = (int)(fl >> 8);
  const int qx0 = rp->qx0, qy0 = rp->qy0, qw = rp->qw;
  const int fx = (int)bc[ia] * span, fy = (int)bc[ib] * span;
  const int i0 = max(qx0, fx), i1 = min(min(qx0 + 2 * qw - 1, fx + span - 1), lim);
  const int j0 = max(qy0, fy), j1 = min(min(qy0 + 2 * qh - 1, fy + span - 1), lim);
  if (i1 < i0 || j1 < j0) return 0u;
  B.org[slot] = (uint32_t)i0 | ((uint32_t)j0 << 11) | ((uint32_t)(i1 - i0 + 1) << 22);
  CovRec cr;
  cr.area = rp->area;
  for (int v = 0; v < 3; ++v) {
    cr.X[v] = rp->X[v];
    cr.Y[v] = rp->Y[v];
  }
  cr.flags = fl;
  cr.tri = t;
  B.cov[slot] = cr;
  return (uint32_t)(j1 - j0 + 1);
}

// Prefix of the entries' row counts (cnt of thread tid < kBrickItems);
// every thread of the workgroup calls it; returns the total.
__device__ __forceinline__ uint32_t brick_prefix(BrickRound& B, uint32_t cnt) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint32_t x = cnt;
  if (tid < kBrickItems) {
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    if (lane == 63) B.wsum[wave] = x;
  }
  __syncthreads();
  if (tid < kBrickItems) {
    for (int w = 0; w < wave; ++w) x += B.wsum[w];
    B.end[tid] = x;
  }
  __syncthreads();
  return B.end[kBrickItems - 1];
}

// Narrows [lo, hi] to the columns k where w - 256 ey k >= 0 may hold.  The
// crossing t = w / (256 ey) is bounded in float with a margin of 1e-3 pixel
// plus 2^-19 |t| (far above the rounding of the conversions, the reciprocal
// and the product), so it never drops a pixel the exact test would keep.
__device__ __forceinline__ void vox_span(int64_t w, int32_t ey, int& lo, int& hi) {
  if (ey == 0) {
    if (w < 0) hi = lo - 1;  // the whole row is outside this edge
    return;
  }
  float t = (float)w * __builtin_amdgcn_rcpf(256.0f * (float)ey);
  t = fminf(fmaxf(t, -4096.0f), 4096.0f);
  const float m = 1e-3f + fabsf(t) * 1.9073486e-6f;
  if (ey < 0) lo = max(lo, (int)ceilf(t - m));
  else hi = min(hi, (int)floorf(t + m));
}

// The round's pixels in two phases.  1: the rows of the triangles' boxes are
// dealt over the lanes; each lane bounds the span of its row inside the three
// edges, and the pixels of the spans are appended to the wave's queue in LDS.  2: whenever the queue
// holds 64, every lane takes one (entry | i << 8 | j << 19) and runs the exact
// fragment path (coverage, voxel address, brick test, shading, accumulation),
// so the expensive part runs with all lanes busy.  The set of fragments, and
// every value computed for one, is the same as testing each pixel of the boxes
// in full.  `fragment` is called by whole waves: fragment(d, on).
//
// Testing every pixel of the boxes, one per lane with its own three 64-bit
// edge functions, cost a pixel inside or outside the triangle the same; a row
// pays for its edges once and its pixels one queue entry each.  The voxelize
// pass of the 5M-triangle soup at 512^3 4.85 -> 4.08 ms, of the 1M-triangle
// one at 256^3 0.40 -> 0.37; a walk that also tests each pixel of the span
// exactly needs spills: 4.34 and 0.40.
template <class Frag>
__device__ __forceinline__ void brick_scan(BrickRound& B, uint32_t total, Frag&& fragment) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t* s_end = B.end;
  uint32_t* q = B.q[wave];
  uint32_t qn = 0;    // entries in the queue (the same in every lane)
  uint32_t own0 = 0;  // the entry of the wave's first row (the same in every lane; never decreases)
  for (uint32_t cb = (uint32_t)wave * 64u; cb < total; cb += kBrickThreads) {
    const uint32_t c = cb + (uint32_t)lane;
    // The entry (triangle) of each lane's row, for the window [cb, cb + 64) of
    // consecutive rows.  own0 moves to the first entry ending after cb: lane k
    // tests entry own0 + k and the ballot counts those ending at or before cb
    // (a prefix, the ends being sorted).  Lane k then holds the end of entry
    // own0 + k, and each lane finds how many of these end at or before its row
    // by a binary search over the lanes (register shuffles): that count from
    // own0 is its entry.  A window that spans more than 64 entries (entries
    // with one row or none) finishes with a per-lane walk.
    for (;;) {
      const uint32_t ek = own0 + (uint32_t)lane < kBrickItems ? s_end[own0 + lane] : 0xffffffffu;
      const uint32_t k = (uint32_t)__popcll(__ballot(ek <= cb));
      own0 += k;
      if (k < 64u) break;
    }
    const uint32_t ek = own0 + (uint32_t)lane < kBrickItems ? s_end[own0 + lane] : 0xffffffffu;
    // Only entries ending inside the window can end at or before a row: nend
    // of them, the first nend lanes (the ends are sorted).  A scan of few ends
    // read into scalar registers has no LDS round trip in its chain, where the
    // binary search takes seven dependent shuffles; the count is the same.
    const uint32_t nend = (uint32_t)__popcll(__ballot(ek < cb + 64u));
    uint32_t past = 0;
    if (nend <= 8u) {
      for (uint32_t k = 0; k < nend; ++k) past += (uint32_t)__builtin_amdgcn_readlane((int)ek, (int)k) <= c ? 1u : 0u;
    } else {
      for (uint32_t st = 32; st; st >>= 1)
        if ((uint32_t)__shfl(ek, (int)(past + st - 1u), 64) <= c) past += st;
      if ((uint32_t)__shfl(ek, (int)past, 64) <= c) ++past;
    }
    int len = 0;
    uint32_t desc = 0;
    if (c < total) {
      uint32_t lo = own0 + past;
      if (past == 64u)
        while (s_end[lo] <= c) ++lo;
      const uint32_t row = c - (lo ? s_end[lo - 1] : 0u);
      const uint32_t org = B.org[lo];
      const int i = (int)(org & 0x7ffu), j = (int)((org >> 11) & 0x7ffu) + (int)row;
      const CovRec cr = B.cov[lo];
      VEdges e;
      vox_edges(cr, i, j, e);
      int k0 = 0, k1 = (int)(org >> 22) - 1;
      vox_span(e.w[0], (int32_t)e.ey[0], k0, k1);
      vox_span(e.w[1], (int32_t)e.ey[1], k0, k1);
      vox_span(e.w[2], (int32_t)e.ey[2], k0, k1);
      len = k1 - k0 + 1;
      desc = lo | ((uint32_t)(i + k0) << 8) | ((uint32_t)j << 19);
    }
    // the wave walks its longest span; each lane stops at the end of its own span
    for (int k = 0;; ++k) {
      const bool hit = k < len;
      const unsigned long long m = __ballot(hit);
      if (m == 0ull) break;
      if (hit) q[qn + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = desc + ((uint32_t)k << 8);
      qn += (uint32_t)__popcll(m);
      if (qn >= 64u) {
        qn -= 64u;
        fragment(q[qn + (uint32_t)lane], true);
      }
    }
  }
  if (qn) {
    const bool on = (uint32_t)lane < qn;
    fragment(on ? q[lane] : 0u, on);
  }
}

// The brick of a workgroup: workgroups are dealt to the 8 XCDs round-robin in
// dispatch order; XCD k takes the k-th eighth of the bricks in Morton order
// (one region of the grid), so the records of triangles shared by neighbouring
// bricks stay in one L2 (voxelize 1.04 -> 1.01 ms).
__device__ __forceinline__ uint32_t brick_of_block() {
  const uint32_t full = gridDim.x & ~7u, b = blockIdx.x;
  return b < full ? (b & 7u) * (full >> 3) + (b >> 3) : b;
}

// Exact mean: sums the brick's fragments and writes its texels.  On grids of
// many small bricks' worth of fragments the vector ALUs bound it (5M triangles
// at 512^3: 2.3 G wave instructions in 3.55 ms, about all the issue slots), on
// smaller ones the waits on LDS and L2 between its phases do, so it runs at 8
// waves per SIMD: 64 registers, no spills, and LDS for 8 workgroups per CU.
template <int DT>
__global__ __launch_bounds__(kBrickThreads) __attribute__((amdgpu_waves_per_eu(8))) void vox_brick_kernel(
    VoxParams vp, const TriRec* __restrict__ recs, const VoxShade* __restrict__ shade,
    const uint32_t* __restrict__ brick_count, const uint32_t* __restrict__ brick_off,
    const uint32_t* __restrict__ list, ListCap lc, void* level0) {
  constexpr int kVox = kBrick * kBrick * kBrick;
  __shared__ uint32_t s_sum[4][kVox];
  __shared__ uint32_t s_cnt[kVox];
  __shared__ BrickRound s_round;
  const int tid = threadIdx.x;
  const BrickGeom g = brick_geom(vp.res);
  const uint32_t brick = brick_of_block();
  const uint32_t nvox = 1u << (3 * g.bits);
  const uint32_t bshift = 3 * g.bits;
  const uint32_t bc[3] = {compact3(brick), compact3(brick >> 1), compact3(brick >> 2)};
  for (uint32_t v = tid; v < nvox; v += kBrickThreads) {
    s_sum[0][v] = 0u;
    s_sum[1][v] = 0u;
    s_sum[2][v] = 0u;
    s_sum[3][v] = 0u;
    s_cnt[v] = 0u;
  }
  const uint32_t n = brick_count[brick], base = brick_off[brick];
  // a brick whose list runs past the lists' capacity (the geometry grew past
  // what the lists were sized for) walks every triangle's brick box instead
  const bool walk = (uint64_t)base + n > (uint64_t)lc.cap;
  const uint32_t nitems = walk ? lc.ntri : n;
  const int lim = 2 * (int)vp.res - 1;
  const int span = 2 << g.bits;  // footprint of the brick on the raster, pixels per axis
  __syncthreads();
  for (uint32_t b0 = 0; b0 < nitems; b0 += kBrickItems) {
    uint32_t t = b0 + (uint32_t)tid;
    bool in = tid < kBrickItems && t < nitems;
    if (in && walk) {  // the box as pack_box stores it: first brick, bricks per axis
      const uint2 pb = lc.boxes[t];
      for (int k = 0; k < 3; ++k)
        in = in && bc[k] - ((pb.x >> (8 * k)) & 255u) < ((pb.y >> (8 * k)) & 255u);
    } else if (in) {
      t = list[base + t];
    }
    const uint32_t total = brick_prefix(s_round, in ? brick_stage(s_round, tid, t, recs, bc, span, lim) : 0u);
    brick_scan(s_round, total, [&](uint32_t d, bool on) {
      if (!on) return;
      const CovRec cr = s_round.cov[d & 255u];
      const int i = (int)((d >> 8) & 0x7ffu), j = (int)(d >> 19);
      VEdges e;
      vox_edges(cr, i, j, e);
      uint32_t key;
      float4 color;
      if (shade_w<true>(cr, recs + cr.tri, shade + cr.tri, e, i, j, e.w[0], e.w[1], e.w[2], vp, key, color, bshift,
                        brick))
        brick_add(s_sum, s_cnt, key & (nvox - 1u), color);
    });
    __syncthreads();
  }
  for (uint32_t v = tid; v < nvox; v += kBrickThreads)
    store_mean<DT>(level0, brick * nvox + v, s_cnt[v], s_sum[0][v], s_sum[1][v], s_sum[2][v], s_sum[3][v]);
}

// ---- reference running average: one pass over the brick's triangles in order --------
// The average depends on the order of a voxel's fragments: triangle, then
// pixel quad, then pixel.  The workgroup sorts the brick's list by original
// triangle index (in LDS up to kRefSort triangles, by a radix sort in global
// memory past that), takes the triangles in rounds in that order, keeps a
// round's fragments in LDS (colour and a 15-bit key: place of the triangle in
// the round, pixel in the brick's footprint), groups them by voxel, ranks each
// by its key among its voxel's, and each voxel's lane replays the packed RGBA8
// + count nibble recurrence on them.  A round whose fragments do not fit is taken
// again with fewer triangles (three always fit, a footprint has 256 pixels), and
// every round takes what the count of the one before suggests: 2,000 triangles
// that fill their bricks' footprints at 64^3 take 1.16 ms, where rounds that
// started from 128 triangles each time, halved until they fitted, took 6.4 (the
// two passes over memory, below, 4.0).  A pass that counted the fragments of every voxel, a scan over
// the voxels, a host wait for the number of fragments and a pass that stored
// them in global memory, sorted and replayed them took the voxelize pass of
// the 1M-triangle soup at 256^3 1.15 ms; this one pass 0.76 (voxels replayed
// in their own order rather than the fullest first: 0.99) and 0.61 since the
// list and the fragments are ranked side by side (they were sorted by a bitonic
// network, a barrier a stage, and by insertion, a chain of LDS reads) and the
// recurrence divides by a reciprocal.
constexpr int kRefFrags = 768;   // fragments of a round (512 at 6 waves per SIMD: no faster)
constexpr int kRefSort = 1024;   // triangles sorted in LDS

struct RefLds {
  union {
    struct {
      float col[3][kRefFrags];
      // key << 9 | voxel of each fragment; then, voxel by voxel in order, its
      // triangle's place in the round << 10 | fragment
      uint32_t kv[kRefFrags];
      uint32_t ent[kRefFrags];  // key << 10 | fragment, voxel by voxel
    };
    unsigned long long sort[kRefSort];  // original triangle << 32 | triangle
    alignas(16) uint32_t otri[256];
    uint32_t hist[4][256];
  };
};
static_assert(sizeof(RefLds) >= kRefSort * 8, "the sort uses the fragments' space");
static_assert(kRefFrags <= 1024 && kRefFrags % kBrickThreads == 0 && kBrickItems <= 128 && kBrick * kBrick * kBrick <= 512,
              "packing of kv and ent");

// Sorts the brick's list segment by original triangle index in global memory
// (4 stable passes of 8 bits between the segment and its place in `other`; an
// even number of passes ends where it began).
__device__ void ref_radix_sort(RefLds& R, uint32_t* seg, uint32_t* other, uint32_t n, const TriRec* __restrict__ recs) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int pass = 0; pass < 4; ++pass) {
    uint32_t* src = pass & 1 ? other : seg;
    uint32_t* dst = pass & 1 ? seg : other;
    const int sh = 8 * pass;
    __syncthreads();
    R.hist[0][tid] = 0u;
    __syncthreads();
    for (uint32_t k = tid; k < n; k += kBrickThreads) atomicAdd(&R.hist[0][(recs[src[k]].otri >> sh) & 255u], 1u);
    __syncthreads();
    // exclusive prefix of the 256 counts: where the digit's next element goes
    const uint32_t c = R.hist[0][tid];
    uint32_t x = c;
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    if (lane == 63) R.hist[1][wave] = x;
    __syncthreads();
    uint32_t at = x - c;
    for (int w = 0; w < wave; ++w) at += R.hist[1][w];
    __syncthreads();
    R.hist[0][tid] = at;
    __syncthreads();
    for (uint32_t b = 0; b < n; b += kBrickThreads) {  // 256 elements at a time, waves one after another
      const uint32_t k = b + (uint32_t)tid;
      const bool in = k < n;
      const uint32_t t = in ? src[k] : 0u;
      const uint32_t dg = in ? (recs[t].otri >> sh) & 255u : 0u;
      unsigned long long same = __ballot(in);
      for (int bit = 0; bit < 8; ++bit) {
        const unsigned long long m = __ballot((dg >> bit) & 1u);
        same &= (dg >> bit) & 1u ? m : ~m;
      }
      const uint32_t rank = (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
      for (int w = 0; w < kBrickThreads / 64; ++w) {
        if (w == wave && in) {
          const uint32_t p = R.hist[0][dg] + rank;
          dst[p] = t;
        }
        __syncthreads();
        if (w == wave && in && rank == 0u) R.hist[0][dg] += (uint32_t)__popcll(same);
        __syncthreads();
      }
    }
  }
  __syncthreads();
}

__global__ __launch_bounds__(kBrickThreads) __attribute__((amdgpu_waves_per_eu(5))) void vox_ref_kernel(
    VoxParams vp, const TriRec* __restrict__ recs, const VoxShade* __restrict__ shade, const uint32_t* brick_count,
    const uint32_t* __restrict__ brick_off, uint32_t* list, uint32_t* list2, uint32_t* __restrict__ level0,
    uint32_t* __restrict__ brick_frags) {
#pragma clang fp contract(off)
  constexpr int kVox = kBrick * kBrick * kBrick;
  __shared__ uint32_t s_state[kVox];  // the voxels' texels so far
  __shared__ uint32_t s_cnt[kVox];    // fragments of the round per voxel
  __shared__ uint16_t s_off[kVox];    // first place of the voxel's fragments in idx
  __shared__ float s_alpha[kBrickItems];
  __shared__ uint16_t s_ord[kVox];    // the round's voxels, most fragments first
  __shared__ uint32_t s_place[64];    // voxels by fragment count (63: or more), then where they go in s_ord
  __shared__ BrickRound s_round;
  __shared__ RefLds R;
  __shared__ uint32_t s_nfrag, s_wsum[kBrickThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const BrickGeom g = brick_geom(vp.res);
  const uint32_t brick = brick_of_block();
  const uint32_t nvox = 1u << (3 * g.bits);
  const uint32_t bshift = 3 * g.bits;
  const uint32_t bc[3] = {compact3(brick), compact3(brick >> 1), compact3(brick >> 2)};
  const int lim = 2 * (int)vp.res - 1;
  const int span = 2 << g.bits;  // footprint of the brick on the raster, pixels per axis
  const uint32_t n = brick_count[brick], base = brick_off[brick];
  for (uint32_t v = tid; v < nvox; v += kBrickThreads) s_state[v] = 0u;
  uint32_t* seg = list + base;
  // ---- the list in order ---------------------------------------------------------
  if (n > (uint32_t)kRefSort) {
    ref_radix_sort(R, seg, list2 + base, n, recs);
  } else if (n > 1u && n <= (uint32_t)kBrickThreads) {
    // each triangle's rank, by comparing it with every other one: 256, 128 or
    // 64 threads' worth of them by 1, 2 or 4 lanes each, with three barriers
    // where a bitonic sort of 64 has 22
    const uint32_t sh = n <= 64u ? 2u : (n <= 128u ? 1u : 0u);
    const uint32_t k = (uint32_t)tid >> sh, h = (uint32_t)tid & ((1u << sh) - 1u);
    uint32_t t = 0;
    if ((uint32_t)tid < n) t = seg[tid];
    R.otri[tid] = (uint32_t)tid < n ? recs[t].otri : 0xffffffffu;
    __syncthreads();
    const uint32_t mine = R.otri[k];
    uint32_t rank = 0;
    for (uint32_t j = 4u * h; j < n; j += 4u << sh) {
      const uint4 o = *reinterpret_cast<const uint4*>(&R.otri[j]);
      rank += (o.x < mine) + (o.y < mine) + (o.z < mine) + (o.w < mine);
    }
    for (uint32_t o = 1; o < (1u << sh); o <<= 1) rank += (uint32_t)__shfl_xor((int)rank, (int)o, 64);
    const uint32_t own = k < n ? seg[k] : 0u;
    __syncthreads();  // every lane has read the segment
    if (h == 0u && k < n) seg[rank] = own;
  } else if (n > 1u) {
    uint32_t m = 64;  // a bitonic sort of the next power of two
    while (m < n) m <<= 1;
    for (uint32_t k = tid; k < m; k += kBrickThreads) {
      unsigned long long e = ~0ull;
      if (k < n) {
        const uint32_t t = seg[k];
        e = ((unsigned long long)recs[t].otri << 32) | t;
      }
      R.sort[k] = e;
    }
    for (uint32_t w = 2; w <= m; w <<= 1)
      for (uint32_t d = w >> 1; d; d >>= 1) {
        __syncthreads();
        for (uint32_t k = tid; k < m / 2; k += kBrickThreads) {
          const uint32_t lo = ((k & ~(d - 1u)) << 1) | (k & (d - 1u)), hi = lo | d;
          const unsigned long long a = R.sort[lo], b = R.sort[hi];
          if ((a > b) == ((lo & w) == 0u)) {
            R.sort[lo] = b;
            R.sort[hi] = a;
          }
        }
      }
    __syncthreads();
    for (uint32_t k = tid; k < n; k += kBrickThreads) seg[k] = (uint32_t)R.sort[k];
  }
  uint32_t nall = 0;                 // fragments of the brick
  uint32_t take = kBrickItems;       // triangles to try in a round
  for (uint32_t pos = 0; pos < n;) {
    const uint32_t m = min(take, n - pos);
    for (uint32_t v = tid; v < nvox; v += kBrickThreads) s_cnt[v] = 0u;
    if (tid < 64) s_place[tid] = 0u;
    if (tid == 0) s_nfrag = 0u;
    __syncthreads();  // also: the sorted segment is in memory, the round before is done
    uint32_t cnt = 0;
    if ((uint32_t)tid < m) {
      const uint32_t t = seg[pos + tid];
      cnt = brick_stage(s_round, tid, t, recs, bc, span, lim);
      s_alpha[tid] = fminf(fmaxf(shade[t].alpha, 0.0f), 1.0f) * 255.0f;
    }
    const uint32_t total = brick_prefix(s_round, cnt);
    brick_scan(s_round, total, [&](uint32_t d, bool on) {
      const uint32_t lo = d & 255u;
      const int i = (int)((d >> 8) & 0x7ffu), j = (int)(d >> 19);
      uint32_t key = 0;
      float4 color = make_float4(0.f, 0.f, 0.f, 0.f);
      if (on) {
        const CovRec cr = s_round.cov[lo];
        VEdges e;
        vox_edges(cr, i, j, e);
        on = shade_w<true>(cr, recs + cr.tri, shade + cr.tri, e, i, j, e.w[0], e.w[1], e.w[2], vp, key, color, bshift,
                           brick);
      }
      const unsigned long long mk = __ballot(on);
      if (!mk) return;
      uint32_t slot = 0;
      if (lane == 0) slot = atomicAdd(&s_nfrag, (uint32_t)__popcll(mk));
      slot = (uint32_t)__builtin_amdgcn_readfirstlane((int)slot) + (uint32_t)__popcll(mk & ((1ull << lane) - 1ull));
      if (on && slot < (uint32_t)kRefFrags) {
        const uint32_t lv = key & (nvox - 1u);
        R.col[0][slot] = color.x;
        R.col[1][slot] = color.y;
        R.col[2][slot] = color.z;
        // the order within a triangle: 2x2 quads row by row, each quad x then y
        const uint32_t pix = (((uint32_t)j >> 1 & 7u) << 5) | (((uint32_t)i >> 1 & 7u) << 2) |
                             (((uint32_t)j & 1u) << 1) | ((uint32_t)i & 1u);
        R.kv[slot] = (((lo << 8) | pix) << 9) | lv;
        atomicAdd(&s_cnt[lv], 1u);
      }
    });
    __syncthreads();
    const uint32_t nf = s_nfrag;
    // the next round takes as many triangles as should fill 7/8 of the space by
    // this round's count, which is fewer than this one's if that did not fit
    take = min(max(m * (kRefFrags * 7u / 8u) / max(nf, 1u), 3u), (uint32_t)kBrickItems);
    if (nf > (uint32_t)kRefFrags) {  // too many: again, with fewer
      __syncthreads();
      continue;
    }
    // ---- group by voxel: two voxels per lane --------------------------------------
    const uint32_t v0 = 2u * (uint32_t)tid, v1 = v0 + 1u;
    const uint32_t c0 = v0 < nvox ? s_cnt[v0] : 0u, c1 = v1 < nvox ? s_cnt[v1] : 0u;
    uint32_t x = c0 + c1;
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    if (lane == 63) s_wsum[wave] = x;
    __syncthreads();
    uint32_t off = x - c0 - c1;
    for (int w = 0; w < wave; ++w) off += s_wsum[w];
    if (v0 < nvox) s_off[v0] = (uint16_t)off;
    if (v1 < nvox) s_off[v1] = (uint16_t)(off + c0);
    if (c0) atomicAdd(&s_place[min(c0, 63u)], 1u);
    if (c1) atomicAdd(&s_place[min(c1, 63u)], 1u);
    __syncthreads();
    constexpr int kMine = kRefFrags / kBrickThreads;  // fragments of a lane
    uint32_t kv[kMine];
#pragma unroll
    for (int r = 0; r < kMine; ++r) {
      const uint32_t f = (uint32_t)(tid + r * kBrickThreads);
      kv[r] = f < nf ? R.kv[f] : 0u;
      const uint32_t lv = kv[r] & 511u;
      if (f < nf) R.ent[s_off[lv] + atomicSub(&s_cnt[lv], 1u) - 1u] = ((kv[r] >> 9) << 10) | f;
    }
    // voxels with fragments, most first: a wave's lanes then replay voxels of
    // like length, and voxels without fragments take no lanes
    if (wave == 0) {
      const uint32_t c = s_place[63 - lane];
      uint32_t y = c;
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t z = __shfl_up(y, o, 64);
        if (lane >= o) y += z;
      }
      s_place[63 - lane] = y - c;
      if (lane == 63) s_nfrag = y;  // voxels with fragments (count 0 was not counted)
    }
    __syncthreads();
    if (c0) s_ord[atomicAdd(&s_place[min(c0, 63u)], 1u)] = (uint16_t)v0;
    if (c1) s_ord[atomicAdd(&s_place[min(c1, 63u)], 1u)] = (uint16_t)v1;
    __syncthreads();
    // each fragment's place among its voxel's: how many of them have a smaller key
#pragma unroll
    for (int r = 0; r < kMine; ++r) {
      const uint32_t f = (uint32_t)(tid + r * kBrickThreads);
      if (f >= nf) break;
      const uint32_t v = kv[r] & 511u, key = kv[r] >> 9;
      const uint32_t beg = s_off[v], end = v + 1u < nvox ? s_off[v + 1u] : nf;
      uint32_t at = beg;
      for (uint32_t a = beg; a < end; ++a) at += R.ent[a] >> 10 < key ? 1u : 0u;
      R.kv[at] = ((key >> 8) << 10) | f;
    }
    __syncthreads();
    // ---- each voxel's fragments in order, through the recurrence -------------------
    const uint32_t nused = s_nfrag;
    for (uint32_t k = tid; k < nused; k += kBrickThreads) {
      const uint32_t v = s_ord[k], beg = s_off[v], end = v + 1u < nvox ? s_off[v + 1u] : nf;
      uint32_t st = s_state[v];
      uint32_t o = R.kv[beg];
      for (uint32_t a = beg; a < end; ++a) {
        const uint32_t f = o & 1023u;
        const float al = s_alpha[o >> 10];
        o = R.kv[min(a + 1u, end - 1u)];
        st = replay_step(st, R.col[0][f] * 255.0f, R.col[1][f] * 255.0f, R.col[2][f] * 255.0f, al);
      }
      s_state[v] = st;
    }
    nall += nf;
    pos += m;
    __syncthreads();
  }
  __syncthreads();
  for (uint32_t v = tid; v < nvox; v += kBrickThreads) level0[brick * nvox + v] = s_state[v];
  if (tid == 0) brick_frags[brick] = nall;
}

__global__ void zero_u32_kernel(uint32_t* p, uint64_t n) {
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = 0u;
}

}  // namespace vct

using namespace vct;

// mat3(transpose(inverse(M))) of a column-major 4x4 (voxelize.vert:28).
static void normal_matrix(const float* M, float* N) {
  double a[3][3];
  for (int c = 0; c < 3; ++c)
    for (int r = 0; r < 3; ++r) a[r][c] = M[c * 4 + r];
  double det = a[0][0] * (a[1][1] * a[2][2] - a[1][2] * a[2][1]) - a[0][1] * (a[1][0] * a[2][2] - a[1][2] * a[2][0]) +
               a[0][2] * (a[1][0] * a[2][1] - a[1][1] * a[2][0]);
  double inv[3][3];
  inv[0][0] = (a[1][1] * a[2][2] - a[1][2] * a[2][1]) / det;
  inv[0][1] = (a[0][2] * a[2][1] - a[0][1] * a[2][2]) / det;
  inv[0][2] = (a[0][1] * a[1][2] - a[0][2] * a[1][1]) / det;
  inv[1][0] = (a[1][2] * a[2][0] - a[1][0] * a[2][2]) / det;
  inv[1][1] = (a[0][0] * a[2][2] - a[0][2] * a[2][0]) / det;
  inv[1][2] = (a[0][2] * a[1][0] - a[0][0] * a[1][2]) / det;
  inv[2][0] = (a[1][0] * a[2][1] - a[1][1] * a[2][0]) / det;
  inv[2][1] = (a[0][1] * a[2][0] - a[0][0] * a[2][1]) / det;
  inv[2][2] = (a[0][0] * a[1][1] - a[0][1] * a[1][0]) / det;
  // transpose(inv), column-major: N[c*3 + r] = inv^T[r][c] = inv[c][r]
  for (int c = 0; c < 3; ++c)
    for (int r = 0; r < 3; ++r) N[c * 3 + r] = (float)inv[c][r];
}

static LightSet make_lights(const vct_context* ctx) {
  LightSet ls;
  memset(&ls, 0, sizeof(ls));
  int n = (int)ctx->lights.size();
  if (n > VCT_MAX_LIGHTS) n = VCT_MAX_LIGHTS;
  for (int i = 0; i < n; ++i) {
    const vct_light& L = ctx->lights[i];
    for (int k = 0; k < 3; ++k) {
      ls.l[i].pos[k] = L.position[k];
      ls.l[i].color[k] = L.color[k];
    }
    ls.l[i].intensity = L.intensity;
    ls.l[i].kind = L.kind;
  }
  ls.count = n;
  return ls;
}

// Every queued draw into the device draw table (through pinned staging, in
// stream order with the kernels that read the previous frame's table).
static int fill_draws(vct_context* ctx, const std::vector<uint32_t>& q, DrawTable& b, bool upload = true) {
  memset(&b, 0, sizeof(b));
  if (q.size() > (size_t)0x7fffffff) return vct_set_error(VCT_ERR_LIMIT, "too many queued models");
  std::vector<Draw> draws(q.size());
  uint64_t ntri = 0;
  uint32_t canon = 0;
  for (size_t k = 0; k < q.size(); ++k) {
    const VctModel& m = ctx->models[q[k]];
    Draw& d = draws[k];
    d.pos = m.d_pos;
    d.nrm = m.d_nrm;
    d.mat = m.d_mat;
    d.perm = m.d_perm;
    d.tri_base = ntri;
    d.canon_base = canon;
    canon += m.ntri;
    d.ntri = m.ntri;
    memcpy(d.M, m.xform, 64);
    normal_matrix(m.xform, d.N);
    ntri += m.ntri;
  }
  if (ntri > (1ull << 31)) return vct_set_error(VCT_ERR_LIMIT, "more than 2^31 triangles queued");
  b.ndraw = (int)draws.size();
  b.ntri = (uint32_t)ntri;
  int rc;
  if (upload && b.ndraw && (rc = vct_upload(ctx, ctx->v_draws, draws.data(), draws.size() * sizeof(Draw))))
    return rc;
  b.d = (const Draw*)ctx->v_draws.dev.p;
  return VCT_OK;
}

static size_t setup_bytes(uint32_t ntri) { return (size_t)(ntri ? ntri : 1) * sizeof(TriRec); }

// The set-up launch; it also writes the material terms of the frame's
// triangles unless those of the last build still hold: the same queued
// models (so the same frame order) at the same material epoch, in the same
// buffer.
static int launch_setup(vct_context* ctx, const std::vector<uint32_t>& q, const DrawTable& b, const VoxParams& vp,
                        uint32_t* bcount) {
  int rc;
  if ((rc = vct_ensure(ctx->vox_shade, (size_t)(b.ntri ? b.ntri : 1) * sizeof(VoxShade), ctx))) return rc;
  const bool build = !(ctx->vox_shade_epoch == ctx->shade_epoch && ctx->vox_shade_models == q &&
                       ctx->vox_shade_ptr == ctx->vox_shade.p);
  const uint32_t per = ctx->res / brick_edge(ctx->res);
  const int lsh = vct_lanes_log2(b.ntri, per * per * per);
  hipLaunchKernelGGL(vox_brick_count_kernel, dim3(vct_lane_blocks(b.ntri, lsh)), dim3(256), 0, ctx->stream, b, vp,
                     (TriRec*)ctx->setup.p, (const DevMaterial*)ctx->d_materials.p, (VoxShade*)ctx->vox_shade.p,
                     build, (uint2*)ctx->vox_box.p, bcount, lsh);
  VCT_HIP(hipGetLastError());
  ctx->vox_shade_epoch = ctx->shade_epoch;
  ctx->vox_shade_models = q;
  ctx->vox_shade_ptr = ctx->vox_shade.p;
  return VCT_OK;
}

// The list write, lists of `cap` entries in ctx->tri_off.
static int launch_list(vct_context* ctx, uint32_t ntri, uint32_t nbricks, const uint32_t* off, uint32_t* cursor,
                       uint32_t cap) {
  const int lsh = vct_lanes_log2(ntri, nbricks);
  hipLaunchKernelGGL(vox_brick_write_kernel, dim3(vct_lane_blocks(ntri, lsh)), dim3(256), 0, ctx->stream, ntri,
                     ctx->res, (const TriRec*)ctx->setup.p, (const uint2*)ctx->vox_box.p, off, cursor,
                     (uint32_t*)ctx->tri_off.p, cap, lsh);
  VCT_HIP(hipGetLastError());
  return VCT_OK;
}

template <int DT>
static void launch_brick(vct_context* ctx, uint32_t nbricks, const VoxParams& vp, const uint32_t* count,
                         const uint32_t* off, const uint32_t* list, void* level0, ListCap lc) {
  hipLaunchKernelGGL(vox_brick_kernel<DT>, dim3(nbricks), dim3(kBrickThreads), 0, ctx->stream, vp,
                     (const TriRec*)ctx->setup.p, (const VoxShade*)ctx->vox_shade.p, count, off, list, lc, level0);
}

// Exact mean: all queued draws in one batch (brick lists span every draw).
// Once a (triangle, brick) pair count is known for this many triangles, phase
// 1 launches everything: the list is sized from that count with a margin
// (a brick whose range runs past it walks the triangles' boxes, so a frame
// whose geometry grew is still exact), and this frame's count comes back
// asynchronously for the next.  Otherwise (the first frame, or another
// triangle count) phase 1 launches up to the scan that writes the count to
// pinned host memory and phase 2 waits for it and launches the rest.
static int voxelize_exact(vct_context* ctx, const std::vector<uint32_t>& q, const VoxParams& vp, void* level0,
                          int phase) {
  const uint32_t res = ctx->res;
  const uint32_t per = res / brick_edge(res), nbricks = per * per * per;
  uint32_t* counters = (uint32_t*)ctx->counters.p;
  int rc;
  // [0, nbricks): counts, [nbricks, 2 nbricks): cursors; then offsets
  if ((rc = vct_ensure(ctx->vox_count, (size_t)nbricks * 8 + 16, ctx))) return rc;
  if ((rc = vct_ensure(ctx->vox_off, (size_t)nbricks * 4 + 16, ctx))) return rc;
  uint32_t* bcount = (uint32_t*)ctx->vox_count.p;
  uint32_t* cursor = bcount + nbricks;
  uint32_t* boff = (uint32_t*)ctx->vox_off.p;
  DrawTable b;
  if ((rc = fill_draws(ctx, q, b, (phase & 1) != 0))) return rc;
  const uint32_t ntri = b.ntri;
  auto bricks = [&](const uint32_t* list, ListCap lc) {
    switch (ctx->dtype) {
      case VCT_RGBA8: launch_brick<VCT_RGBA8>(ctx, nbricks, vp, bcount, boff, list, level0, lc); break;
      case VCT_FP16: launch_brick<VCT_FP16>(ctx, nbricks, vp, bcount, boff, list, level0, lc); break;
      case VCT_BF16: launch_brick<VCT_BF16>(ctx, nbricks, vp, bcount, boff, list, level0, lc); break;
      default: launch_brick<VCT_FP32>(ctx, nbricks, vp, bcount, boff, list, level0, lc); break;
    }
  };
  if (phase & 1) {
    // the count an earlier frame copied back, if it has landed (never waited for)
    if (ctx->vox_total_pending) {
      const hipError_t qe = hipEventQuery(ctx->vox_total_ev);
      if (qe == hipSuccess) {
        ctx->vox_total_pending = false;
        ctx->vox_known_total = ctx->h_readback[3];
      } else if (qe == hipErrorNotReady) {
        (void)hipGetLastError();  // not an error: the copy is still in flight
      } else {
        return vct_hip_check(qe, "hipEventQuery");
      }
    }
    hipLaunchKernelGGL(zero_u32_kernel, dim3((2 * nbricks + 255) / 256), dim3(256), 0, ctx->stream, bcount,
                       (uint64_t)2 * nbricks);
    VCT_HIP(hipGetLastError());
    ctx->h_readback[2] = 0u;
    ctx->vox_sized = ntri > 0 && ctx->vox_known_total > 0 && ctx->vox_known_ntri == ntri;
    if (ntri) {
      if ((rc = vct_ensure(ctx->setup, setup_bytes(ntri), ctx))) return rc;
      if ((rc = vct_ensure(ctx->vox_box, (size_t)ntri * 8, ctx))) return rc;
      if ((rc = launch_setup(ctx, q, b, vp, bcount))) return rc;
      if ((rc = vct_launch_scan_u32(ctx, bcount, boff, nbricks, counters + 2, nullptr,
                                    ctx->h_readback + (ctx->vox_sized ? 3 : 2))))
        return rc;
      if (ctx->vox_sized) {
        VCT_HIP(hipEventRecord(ctx->vox_total_ev, ctx->stream));
        // a quarter more than the last count, at least two pairs per triangle
        const uint64_t want = std::max<uint64_t>((uint64_t)ctx->vox_known_total + ctx->vox_known_total / 4,
                                                 2ull * ntri + 1024u);
        const uint32_t cap = (uint32_t)std::min<uint64_t>(want, 0xffffffffull);
        if ((rc = vct_ensure(ctx->tri_off, (size_t)cap * 4, ctx))) return rc;
        ctx->vox_cap = cap;
        if ((rc = launch_list(ctx, ntri, nbricks, boff, cursor, cap))) return rc;
        ctx->vox_total_pending = true;
        ctx->vox_pairs_on_device = true;
        bricks((const uint32_t*)ctx->tri_off.p, ListCap{(const uint2*)ctx->vox_box.p, ntri, cap});
        VCT_HIP(hipGetLastError());
      }
    }
  }
  if (!(phase & 2) || ctx->vox_sized) return VCT_OK;
  VCT_HIP(hipStreamSynchronize(ctx->stream));
  const uint32_t total = ntri ? ctx->h_readback[2] : 0u;
  if (total) {
    if ((rc = vct_ensure(ctx->tri_off, (size_t)total * 4 + (size_t)total / 4 * 4, ctx))) return rc;
    if ((rc = launch_list(ctx, ntri, nbricks, boff, cursor, total))) return rc;
  } else {
    hipLaunchKernelGGL(zero_u32_kernel, dim3((nbricks + 255) / 256), dim3(256), 0, ctx->stream, boff,
                       (uint64_t)nbricks);
    VCT_HIP(hipGetLastError());
    if ((rc = vct_ensure(ctx->tri_off, 16, ctx))) return rc;
  }
  if ((rc = vct_ensure(ctx->setup, setup_bytes(ntri), ctx))) return rc;
  ctx->last_candidates = total;  // (triangle, brick) pairs
  ctx->vox_known_total = total;
  ctx->vox_known_ntri = ntri;
  bricks((const uint32_t*)ctx->tri_off.p, ListCap{nullptr, 0u, 0xffffffffu});
  VCT_HIP(hipGetLastError());
  return VCT_OK;
}

// Reference running average: the exact mean's records and brick lists, then
// one pass that takes every brick's triangles in order (vox_ref_kernel).
// Phase 1 launches up to the scan that writes the (triangle, brick) pair count
// to pinned host memory, phase 2 waits for it, sizes the lists (and the sort's
// second buffer) and launches the rest.
static int voxelize_reference(vct_context* ctx, const std::vector<uint32_t>& q, const VoxParams& vp, void* level0,
                              int phase) {
  const uint32_t res = ctx->res;
  const uint32_t per = res / brick_edge(res), nbricks = per * per * per;
  uint32_t* counters = (uint32_t*)ctx->counters.p;  // [2] pairs
  int rc;
  // per-brick counts + cursors (the cursors hold the fragment counts at the end), offsets
  if ((rc = vct_ensure(ctx->tri_count, (size_t)nbricks * 8 + 16, ctx))) return rc;
  if ((rc = vct_ensure(ctx->tri_base, (size_t)nbricks * 4 + 16, ctx))) return rc;
  uint32_t* bcount = (uint32_t*)ctx->tri_count.p;
  uint32_t* cursor = bcount + nbricks;
  uint32_t* boff = (uint32_t*)ctx->tri_base.p;
  DrawTable b;
  if ((rc = fill_draws(ctx, q, b, (phase & 1) != 0))) return rc;
  const uint32_t ntri = b.ntri;
  if (phase & 1) {
    hipLaunchKernelGGL(zero_u32_kernel, dim3((2 * nbricks + 255) / 256), dim3(256), 0, ctx->stream, bcount,
                       (uint64_t)2 * nbricks);
    VCT_HIP(hipGetLastError());
    ctx->h_readback[2] = 0u;
    if (ntri) {
      if ((rc = vct_ensure(ctx->setup, setup_bytes(ntri), ctx))) return rc;
      if ((rc = vct_ensure(ctx->vox_box, (size_t)ntri * 8, ctx))) return rc;
      if ((rc = launch_setup(ctx, q, b, vp, bcount))) return rc;
      if ((rc = vct_launch_scan_u32(ctx, bcount, boff, nbricks, counters + 2, nullptr, ctx->h_readback + 2)))
        return rc;
    }
    VCT_HIP(hipEventRecord(ctx->vox_total_ev, ctx->stream));
    ctx->vox_total_pending = false;  // the event no longer stands for an exact-mean frame's count
    ctx->vox_known_total = 0;
  }
  if (!(phase & 2)) return VCT_OK;
  VCT_HIP(hipEventSynchronize(ctx->vox_total_ev));
  const uint32_t pairs = ntri ? ctx->h_readback[2] : 0u;
  ctx->last_candidates = pairs;
  if (!pairs) {
    const uint64_t nvox = (uint64_t)res * res * res;
    hipLaunchKernelGGL(zero_u32_kernel, dim3(2048), dim3(256), 0, ctx->stream, (uint32_t*)level0, nvox);
    VCT_HIP(hipGetLastError());
    return VCT_OK;
  }
  const size_t seg = ((size_t)pairs + pairs / 4 + 3) & ~(size_t)3;
  if ((rc = vct_ensure(ctx->tri_off, seg * 8, ctx))) return rc;
  if ((rc = launch_list(ctx, ntri, nbricks, boff, cursor, pairs))) return rc;
  hipLaunchKernelGGL(vox_ref_kernel, dim3(nbricks), dim3(kBrickThreads), 0, ctx->stream, vp,
                     (const TriRec*)ctx->setup.p, (const VoxShade*)ctx->vox_shade.p, (const uint32_t*)bcount,
                     (const uint32_t*)boff, (uint32_t*)ctx->tri_off.p, (uint32_t*)ctx->tri_off.p + seg,
                     (uint32_t*)level0, cursor);
  VCT_HIP(hipGetLastError());
  ctx->vox_frag_bricks = nbricks;
  return VCT_OK;
}

// normalize(position) of the directional lights, operation for operation as
// the fragment shader computes it (voxelize.frag:127-131), without contraction.
static void light_dirs(VoxParams& vp) {
#pragma clang fp contract(off)
  for (int li = 0; li < VCT_MAX_LIGHTS; ++li) {
    const DevLight& L = vp.lights.l[li];
    const float l = sqrtf(L.pos[0] * L.pos[0] + L.pos[1] * L.pos[1] + L.pos[2] * L.pos[2]);
    for (int k = 0; k < 3; ++k) vp.ldir[li][k] = L.pos[k] / l;
  }
}

int vct_launch_voxelize(vct_context* ctx) { return vct_launch_voxelize_phase(ctx, 3); }

int vct_launch_voxelize_phase(vct_context* ctx, int phase) {
  const uint32_t res = ctx->res;
  void* level0 = (char*)ctx->volume.p + ctx->lvl_off[0][0];
  int rc;
  if ((rc = vct_ensure(ctx->counters, 256, ctx))) return rc;
  VoxParams vp;
  memset(&vp, 0, sizeof(vp));
  vp.res = res;
  vp.cube_size = ctx->cube_size;
  vp.average = ctx->average;
  vp.lights = make_lights(ctx);
  light_dirs(vp);
  std::vector<uint32_t> q;
  for (uint32_t id : ctx->queue)
    if (id < ctx->models.size() && ctx->models[id].ntri) q.push_back(id);
  if (phase & 1) {
    ctx->last_candidates = 0;
    ctx->last_fragments = 0;
    ctx->vox_pairs_on_device = false;
    ctx->vox_frag_bricks = 0;
  }
  if (ctx->average == VCT_AVG_EXACT) return voxelize_exact(ctx, q, vp, level0, phase);
  return voxelize_reference(ctx, q, vp, level0, phase);
}
