// vct_trace.hip - per-pixel cone marcher (kernel c).
//
// Shades every covered pixel as voxel_cone_tracing.frag:246-275 does:
//   pos = scale_and_bias(world / cube_size)                      (:248)
//   diffuse  = Kd * trace_diffuse(pos, n)                         (:140-168)
//   direct   = direct_light(pos, view_dir) with shadow cones       (:175-218)
//   specular = Ks * trace_specular(pos, n, view_dir)              (:229-235)
//   refraction override for illum 4/6/7/9                         (:273-274)
// trace_cone (:88-119) marches front to back, c += (1 - c.a) * s, with
// mip = max(log2(diam * res), 0), step = max(diam / 2, voxel_size), and
// sample_voxel (:80-86) = |d.x| T[x] + |d.y| T[y] + |d.z| T[z] (unnormalised).
//
// Sampler: a software quadrilinear textureLod over the brick/Morton volume
// with GL semantics (texture_3d.cpp:10-15): texel centres at (i + 0.5) / s,
// CLAMP_TO_BORDER with a zero border, LINEAR_MIPMAP_LINEAR between floor(lod)
// and floor(lod) + 1, lod clamped to [0, L-1].  The three maps of one sample
// share coordinates and weights, so corner addresses are computed once per
// level and all 24 corner loads of a level are issued before the first is
// used; level 0 is shared by all maps, so it is fetched once per step.
//
// Work mapping: a workgroup of 4 waves shades a block of 64 to 192 pixels
// whose cones form one queue for its lanes (shade_block), ordered so that the
// lanes of a wave march like cones over neighbouring surface points and their
// texel fetches fall on the same cache lines.
// Accumulation is FP32 for every storage type.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "vct_internal.h"

namespace vct {

constexpr int kMaxCones = 16;

struct ConeSet {
  float a[kMaxCones], b[kMaxCones], c[kMaxCones];  // dir = a n + b o1 + c o2
  float aperture;
  int n;
};

struct TraceArgs {
  const char* vol;
  uint64_t off[16][6];
  int levels;
  int res;
  const float4* gpos;
  const float4* gnrm;
  const DevMaterial* mats;
  uint32_t nmat;
  float4* image;
  int W, H;
  float cube_size;
  float cam[3];
  int en_direct, en_diffuse, en_specular, en_shadow;
  int view_dir;
  float view_lod;
  int demodulate;  // 1: write final / max(Kd, eps) (the learned path's target)
  unsigned long long* step_counter;  // optional: cone steps taken (diagnostics)
  // pixel selection (both null: every pixel, image indexed like the G-buffer)
  const uint32_t* pix_list;    // listed pixels (y * W + x); image[k] receives pixel k
  uint32_t npix_list;          // count (host), or the bound of *pix_count when that is set
  const uint32_t* pix_count;   // optional device-side count of listed pixels
  int pix_scatter;             // 1: image[pixel] receives the pixel instead of image[k]
  const uint32_t* tile_list;   // listed 32x32 tiles (ty * tiles_x + tx); 16 workgroups per tile
  const uint32_t* tile_count;  // device-side number of listed tiles
  int tiles_x;
  const uint32_t* tile_flag;   // optional: listed pixels are traced only where tile_flag[tile] == flag_want
  uint32_t flag_want;
  int grid_stride;             // tile-list mode: 2 = the odd-odd pixels of the tiles (a 16x16 grid per tile),
                               // written to image[(y >> 1) * half_w + (x >> 1)]
  int half_w;
  ConeSet cones;
  LightSet lights;
};

// Storage types: raw texel as loaded (Raw) and its decode to float4; the
// decode folds into the blend (v_fma_mix_f32 for the 16-bit types).
// RGBA8 storage as the learned form's demodulated launches read it: what they
// trace is interpolated and goes into a network that rounds its inputs to BF16,
// where the last bit of a sample can move a pixel by 6e-4 (936x692, sixteen
// cones), so each texel is scaled by 1/255 before it is weighted, as a texel
// fetch rounds.  Every launch that traces pixels of the image itself, plain or
// learned, scales the weighted sum instead, so a traced pixel is the plain
// frame's bit for bit: a byte then takes half the vector cycles
// (quarter-resolution trace of that frame 0.16 ms against 0.19, its tiles
// traced in full 0.30 against 0.38).
constexpr int kRgba8Unorm = 4;
template <int DT>
constexpr bool kBytes = DT == VCT_RGBA8 || DT == kRgba8Unorm;

template <int DT>
struct Tex;
template <>
struct Tex<VCT_RGBA8> {
  using Raw = uint32_t;
  static __device__ __forceinline__ float4 decode(Raw v) {
    const float k = 1.0f / 255.0f;
    return make_float4((float)(v & 255u) * k, (float)((v >> 8) & 255u) * k, (float)((v >> 16) & 255u) * k,
                       (float)(v >> 24) * k);
  }
};
template <>
struct Tex<kRgba8Unorm> : Tex<VCT_RGBA8> {};
template <>
struct Tex<VCT_FP16> {
  using Raw = uint2;
  static __device__ __forceinline__ float4 decode(Raw v) {
    return make_float4(f16_to_f32(v.x & 0xffffu), f16_to_f32(v.x >> 16), f16_to_f32(v.y & 0xffffu),
                       f16_to_f32(v.y >> 16));
  }
};
template <>
struct Tex<VCT_BF16> {
  using Raw = uint2;
  static __device__ __forceinline__ float4 decode(Raw v) {
    return make_float4(bf16_to_f32(v.x & 0xffffu), bf16_to_f32(v.x >> 16), bf16_to_f32(v.y & 0xffffu),
                       bf16_to_f32(v.y >> 16));
  }
};
template <>
struct Tex<VCT_FP32> {
  using Raw = float4;
  static __device__ __forceinline__ float4 decode(Raw v) { return v; }
};

// Copy of the volume read by the marcher.  What bounds the marcher is the
// cache lines its loads touch, so the copy lets one load return several
// corners of a trilinear fetch; FP32 texels are already 16 bytes and have none.
//
// 16-bit storage, x-paired: entry i of a map holds texel i and its +x
// neighbour (zero past the last column) channel by channel, four words of
// (c(x), c(x+1)); 4 loads of 16 bytes fetch the 8 corners.
//
// RGBA8, tiled: an element holds a texel and its +y neighbour, and a line of
// 128 bytes holds the elements of 4 x 2 x 2 texels of which the 4th column is
// the next line's first again, so the 4 corners of an (x, y) cell are always
// 16 consecutive bytes of one line: 2 loads fetch the 8 corners (16 bytes at
// an alignment of 8).  As x-paired entries (4 loads of 8 bytes) the marcher
// took 1.86 ms of the 2560x1440 frame at 256^3 and 0.83 of the 1280x720 one at
// 128^3; tiled 1.68 and 0.72, for 2.7 times the volume written where the pairs
// were 2 (entries of the four texels, 4 times: 1.71 and 0.73).
template <int DT>
struct Pair {
  static constexpr bool kOn = false;
};
template <>
struct Pair<VCT_RGBA8> {
  static constexpr bool kOn = true;
  static constexpr int kLoads = 2;  // of one map: per z corner
  using Raw = uint4;                // (x, y), (x, y+1), (x+1, y), (x+1, y+1)
};
template <int DT>
struct Pair16 {
  static constexpr bool kOn = true;
  static constexpr int kLoads = 4;  // per (y, z) corner
  using Raw = uint4;
  static __device__ __forceinline__ Raw make(uint2 a, uint2 b) { return pair_pack(a, b); }
};
template <>
struct Pair<kRgba8Unorm> : Pair<VCT_RGBA8> {};
template <>
struct Pair<VCT_FP16> : Pair16<VCT_FP16> {};
template <>
struct Pair<VCT_BF16> : Pair16<VCT_BF16> {};

// Byte offset of a texel's element in a tiled map, the sum of its coordinates'
// parts: lines lie in Morton order of a grid of edge / 2 per axis (of which
// the x axis uses two thirds), so a map of edge s spans 16 s^3 bytes, or one
// line.
constexpr uint32_t kTileCols = 3;  // columns of a line, without the repeated one
__device__ __forceinline__ uint32_t tile_x(uint32_t x) {
  return (spread3(x / kTileCols) << 7) + (x % kTileCols) * 8u;
}
__device__ __forceinline__ uint32_t tile_y(uint32_t y) { return (spread3(y >> 1) << 8) + (y & 1u) * 32u; }
__device__ __forceinline__ uint32_t tile_z(uint32_t z) { return (spread3(z >> 1) << 9) + (z & 1u) * 64u; }

__device__ __forceinline__ float4 f4(float x) { return make_float4(x, x, x, x); }
// The four bytes of an RGBA8 texel, each masked in place and taken as the bits
// of a (subnormal) float: byte * 2^-149, * 2^-141, * 2^-133 and, shifted down,
// * 2^-149 (kRgba8Unorm: as byte / 255).
template <int DT>
__device__ __forceinline__ float4 bytes4(uint32_t v) {
  if constexpr (DT == kRgba8Unorm) {
    float k = 1.0f / 255.0f;
    return make_float4((float)(v & 255u) * k, (float)((v >> 8) & 255u) * k, (float)((v >> 16) & 255u) * k,
                       (float)(v >> 24) * k);
  }
  return make_float4(__builtin_bit_cast(float, v & 0xffu), __builtin_bit_cast(float, v & 0xff00u),
                     __builtin_bit_cast(float, v & 0xff0000u), __builtin_bit_cast(float, v >> 24));
}
__device__ __forceinline__ float4 operator+(float4 a, float4 b) {
  return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}
__device__ __forceinline__ float4 operator*(float s, float4 a) {
  return make_float4(s * a.x, s * a.y, s * a.z, s * a.w);
}

// Per-workgroup sampler tables in LDS: the byte offset of a texel within a
// map is sx[x] + sy[y] + sz[z] (16 brick_index(x, y, z): spread3 of each
// coordinate, pre-shifted by the axis and the entry size; RGBA8: the parts of
// the tiled element), for edges up to
// 512: the volume's 4 GiB bound rules out 1024^3 in every storage type, and
// the launch checks it), and the byte offset of every (level, map) of the
// volume (a lane's level varies, so the table is indexed per lane; LDS reads
// are far cheaper than per-lane reads of kernel arguments).  Offsets are
// 32-bit: the volume stays below 4 GiB (checked when it is allocated), so
// every texel load is the uniform volume pointer plus one 32-bit lane offset.
constexpr int kMaxEdge = 512;
struct SamplerLds {
  uint32_t sx[kMaxEdge], sy[kMaxEdge], sz[kMaxEdge];
  uint32_t off[16][6];  // per axis the map of a positive direction, then that of a negative one
};

// The byte offset within an axis' two maps in SamplerLds::off of the map that
// a direction component reads: 4 for a negative one.
__device__ __forceinline__ uint32_t face_of(float d) { return (__builtin_bit_cast(uint32_t, d) >> 29) & 4u; }

template <int DT>
__device__ __forceinline__ void sampler_init(const TraceArgs& A, SamplerLds* S) {
  for (uint32_t q = threadIdx.x; q < (uint32_t)kMaxEdge; q += blockDim.x) {
    const uint32_t v = spread3(q) << 4;  // a 16-bit pair or an FP32 texel has 16 bytes
    S->sx[q] = kBytes<DT> ? tile_x(q) : v;
    S->sy[q] = kBytes<DT> ? tile_y(q) : v << 1;
    S->sz[q] = kBytes<DT> ? tile_z(q) : v << 2;
  }
  for (int q = threadIdx.x; q < 16 * 6; q += blockDim.x) S->off[q / 6][(q % 6) ^ 1] = (uint32_t)A.off[q / 6][q % 6];
}

// Corner byte offsets within a map: ix[dx] + iyz[dy + 2 dz].  Paired volumes
// use ix[0] only: its entry holds both x-corners, weighted w[2k] (first texel)
// and w[2k + 1] (second) for the (y, z) corner k; tiled ones only the even
// iyz as well.
struct Corners {
  uint32_t ix[2], iyz[4];
  float w[8];  // corner weights (dx + 2 dy + 4 dz), times kTexWeight; zero for border texels
};

// The marcher's step is bound by the cache lines its loads touch and, for
// RGBA8, as much by the vector ALUs, so the sampler's arithmetic is laid out
// for their issue rates (measured, cycles per wave: FP32 add, mul and fma and
// 32-bit and, or, add, right shift 2; conversions, min, max, compares, selects
// and left shifts 4; log, rcp, sqrt 8).  With the clamped corners, the masked
// bytes and the exit distance a step of RGBA8 issues 1290 cycles instead of
// 1880 (2560x1440 soup, the trace: RGBA8 2.03 -> 1.89 ms, FP16 1.93 -> 1.79,
// FP32 at 1001x563 0.37 -> 0.34).
//
// The two texels an axis reads at u (texel units, texel i centred on i): i0,
// clamped so that i0 and i0 + 1 both lie in the level (hi = max(edge - 2, 0)),
// returned as 4 i0, a table offset, and their weights.  With d = u - i0 texel
// i0 weighs 1 - |d| and texel i0 + 1 weighs d, or 2 - d past it, both clamped
// to [0, 1]: next to the border the texel outside is not among the two and the
// one inside keeps its weight, further out both weights are zero.  Each step
// rounds as the weights 1 - frac(u) and frac(u) do.  In the level of one texel
// the second weight is capped by edge - 1 = 0.
__device__ __forceinline__ uint32_t axis_corners(float u, float hi, float cap, float& w0, float& w1) {
  const float i0 = __builtin_amdgcn_fmed3f(floorf(u), 0.0f, hi);
  const float d = u - i0;
  w0 = __builtin_amdgcn_fmed3f(1.0f - fabsf(d), 0.0f, 1.0f);
  w1 = __builtin_amdgcn_fmed3f(fminf(fminf(d, 2.0f - d), cap), 0.0f, 1.0f);
  return (uint32_t)(i0 * 4.0f);
}

__device__ __forceinline__ uint32_t lds_at(const uint32_t* table, uint32_t bytes) {
  return *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(table) + bytes);
}

// What the corner weights are multiplied by (see blend4): a power of two, so
// it changes no rounding.
template <int DT>
constexpr float kTexWeight = DT == VCT_RGBA8 ? 0x1p120f : 1.0f;

template <int DT>
__device__ __forceinline__ void corners(const SamplerLds* S, float3 p, float fs, Corners& c) {
  const float hi = fmaxf(fs - 2.0f, 0.0f), cap = fs - 1.0f;
  float wx0, wx1, wy0, wy1, wz0, wz1;
  const uint32_t x0 = axis_corners(p.x * fs - 0.5f, hi, cap, wx0, wx1);
  const uint32_t y0 = axis_corners(p.y * fs - 0.5f, hi, cap, wy0, wy1);
  const uint32_t z0 = axis_corners(p.z * fs - 0.5f, hi, cap, wz0, wz1);
  wz0 *= kTexWeight<DT>;
  wz1 *= kTexWeight<DT>;
  const float w00 = wy0 * wz0, w10 = wy1 * wz0, w01 = wy0 * wz1, w11 = wy1 * wz1;
  c.w[0] = wx0 * w00;
  c.w[1] = wx1 * w00;
  c.w[2] = wx0 * w10;
  c.w[3] = wx1 * w10;
  c.w[4] = wx0 * w01;
  c.w[5] = wx1 * w01;
  c.w[6] = wx0 * w11;
  c.w[7] = wx1 * w11;
  // the second texel's offsets; the level of one texel has none: its mask is
  // the sign of -(edge - 1)
  const uint32_t m = (uint32_t)(__builtin_bit_cast(int32_t, 0.0f - cap) >> 31);
  c.ix[0] = lds_at(S->sx, x0);
  if (!Pair<DT>::kOn) c.ix[1] = lds_at(S->sx + 1, x0) & m;
  const uint32_t y0p = lds_at(S->sy, y0), y1p = lds_at(S->sy + 1, y0) & m;
  const uint32_t z0p = lds_at(S->sz, z0), z1p = lds_at(S->sz + 1, z0) & m;
  c.iyz[0] = y0p + z0p;
  c.iyz[1] = y1p + z0p;
  c.iyz[2] = y0p + z1p;
  c.iyz[3] = y1p + z1p;
}

// The eight corners of one map (byte offset `base`), all loads issued before
// any is used (border corners have weight 0 and a clamped, valid index: no
// per-corner branches).
template <int DT>
__device__ __forceinline__ void gather8(const char* __restrict__ vol, uint32_t base, const Corners& c,
                                        typename Tex<DT>::Raw (&r)[8]) {
  using Raw = typename Tex<DT>::Raw;
#pragma unroll
  for (int k = 0; k < 8; ++k) r[k] = *reinterpret_cast<const Raw*>(vol + (base + c.ix[k & 1] + c.iyz[k >> 1]));
}

template <int DT>
__device__ __forceinline__ void gather_pairs(const char* __restrict__ vol, uint32_t base, const Corners& c,
                                             typename Pair<DT>::Raw (&r)[Pair<DT>::kLoads]) {
  using Raw = typename Pair<DT>::Raw;
  constexpr int n = Pair<DT>::kLoads;
#pragma unroll
  for (int k = 0; k < n; ++k) {
    const char* p = vol + (base + c.ix[0] + c.iyz[k * (4 / n)]);
    __builtin_memcpy(&r[k], __builtin_assume_aligned(p, kBytes<DT> ? 8 : 16), sizeof(Raw));
  }
}

// Weights of the four (y, z) corner pairs, as the packed 16-bit operand of a
// two-term dot product for 16-bit storage (rounded to nearest in the storage
// type: the filter weights carry the precision of the stored texels).
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf162_t __attribute__((ext_vector_type(2)));

template <int DT>
struct PairWeights {
  float w[8];
  __device__ __forceinline__ explicit PairWeights(const Corners& c) {
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] = c.w[k];
  }
};
template <>
struct PairWeights<VCT_FP16> {
  half2_t w[4];
  __device__ __forceinline__ explicit PairWeights(const Corners& c) {
#pragma unroll
    for (int k = 0; k < 4; ++k) w[k] = half2_t{(_Float16)c.w[2 * k], (_Float16)c.w[2 * k + 1]};
  }
};
template <>
struct PairWeights<VCT_BF16> {
  bf162_t w[4];
  __device__ __forceinline__ explicit PairWeights(const Corners& c) {
#pragma unroll
    for (int k = 0; k < 4; ++k) w[k] = bf162_t{(__bf16)c.w[2 * k], (__bf16)c.w[2 * k + 1]};
  }
};

// What a blended texel is multiplied by once its corners are summed: an RGBA8
// texel counts in steps of 1/255 (unorm8), the others are stored as values.
template <int DT>
constexpr float kTexScale = DT == VCT_RGBA8 ? 1.0f / 255.0f : 1.0f;

// Blend of the eight corners of one paired map, before kTexScale: per
// channel, one FP32 two-term dot product (v_dot2_f32_f16 / _bf16) per corner
// pair for 16-bit storage.  RGBA8 accumulates in FP32 the bytes that bytes4
// masks out, as subnormal floats, with weights scaled by 2^120 to keep the
// products normal: the powers of two (undone once per sample by tex_unscale)
// change no rounding, and a mask takes half the cycles of a conversion
// (v_and_b32 and v_fma_f32 issue a wave every 2 cycles, v_cvt_f32_ubyte every
// 4), so a byte costs 4 cycles where it took 6.  The 1/255 is applied to the
// sum.
template <int DT>
__device__ __forceinline__ float4 blend4(const PairWeights<DT>& W, const typename Pair<DT>::Raw (&r)[Pair<DT>::kLoads]) {
  float4 acc = f4(0.0f);
  if constexpr (DT == VCT_FP16) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      acc.x = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, r[k].x), W.w[k], acc.x, false);
      acc.y = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, r[k].y), W.w[k], acc.y, false);
      acc.z = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, r[k].z), W.w[k], acc.z, false);
      acc.w = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, r[k].w), W.w[k], acc.w, false);
    }
  } else if constexpr (DT == VCT_BF16) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      acc.x = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf162_t, r[k].x), W.w[k], acc.x, false);
      acc.y = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf162_t, r[k].y), W.w[k], acc.y, false);
      acc.z = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf162_t, r[k].z), W.w[k], acc.z, false);
      acc.w = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf162_t, r[k].w), W.w[k], acc.w, false);
    }
  } else {
#pragma unroll
    for (int k = 0; k < 2; ++k)
      acc = acc + W.w[4 * k] * bytes4<DT>(r[k].x) + W.w[4 * k + 1] * bytes4<DT>(r[k].z) +
            W.w[4 * k + 2] * bytes4<DT>(r[k].y) + W.w[4 * k + 3] * bytes4<DT>(r[k].w);
  }
  return acc;
}

// Undoes kTexWeight and the places of the bytes in bytes4.
template <int DT>
__device__ __forceinline__ float4 tex_unscale(float4 v) {
  if constexpr (DT == VCT_RGBA8) return make_float4(v.x * 0x1p29f, v.y * 0x1p21f, v.z * 0x1p13f, v.w * 0x1p29f);
  return v;
}

template <int DT>
__device__ __forceinline__ float4 blend8(const Corners& c, const typename Tex<DT>::Raw (&r)[8]) {
  float4 acc = f4(0.0f);
#pragma unroll
  for (int k = 0; k < 8; ++k) acc = acc + c.w[k] * Tex<DT>::decode(r[k]);
  return acc;
}

__device__ __forceinline__ float4 fma4(float s, float4 a, float4 c) {
  return make_float4(__builtin_fmaf(s, a.x, c.x), __builtin_fmaf(s, a.y, c.y), __builtin_fmaf(s, a.z, c.z),
                     __builtin_fmaf(s, a.w, c.w));
}

// One level of sample_voxel: level 0 is the one map shared by all directions
// (|d.x| + |d.y| + |d.z| times one trilinear fetch), a higher level blends
// the three directional maps mx, my, mz.  `ad` is |d| times kTexScale.
//
// Paired storage fetches the first map alike at every level (every map of
// level 0 starts at offset 0) and lanes above level 0 add the other two:
// most waves mix lanes of both kinds, and a path of its own for level 0
// costs the wave a blend, four more loads and one more wait on memory per
// sample (2560x1440 soup, the trace alone: FP16 2.18 -> 2.14 ms; RGBA8, with
// the 1/255 out of the corner sums, 2.58 -> 2.23 ms).  FP32 storage has twice
// the loads per map and no registers for a map held over the others: there
// the two paths stay apart (one path measured 0.43 -> 0.58 ms at 1001x563).
template <int DT, bool kMaybeLevel0>
__device__ __forceinline__ float4 sample_level(const TraceArgs& A, const SamplerLds* S, float3 p, float3 ad,
                                               uint32_t mx, uint32_t my, uint32_t mz, bool level0, float fs) {
  constexpr int next = kMaybeLevel0 ? 0 : 6;  // the offsets one level up
  const uint32_t* off = &S->off[0][0] + next;
  Corners c;
  corners<DT>(S, p, fs, c);
  if constexpr (Pair<DT>::kOn) {
    using PRaw = typename Pair<DT>::Raw;
    const PairWeights<DT> W(c);
    float ax = ad.x;
    float4 yy = f4(0.0f), bz = f4(0.0f);
    PRaw rx[Pair<DT>::kLoads];
    gather_pairs<DT>(A.vol, lds_at(off, mx), c, rx);
    if (!kMaybeLevel0 || !level0) {
      PRaw ry[Pair<DT>::kLoads], rz[Pair<DT>::kLoads];
      gather_pairs<DT>(A.vol, lds_at(off + 2, my), c, ry);
      gather_pairs<DT>(A.vol, lds_at(off + 4, mz), c, rz);
      yy = ad.y * blend4<DT>(W, ry);
      bz = blend4<DT>(W, rz);
    } else {
      ax = ad.x + ad.y + ad.z;
    }
    return fma4(ad.z, bz, fma4(ax, blend4<DT>(W, rx), yy));
  }
  using Raw = typename Tex<DT>::Raw;
  if (kMaybeLevel0 && level0) {
    Raw r[8];
    gather8<DT>(A.vol, 0u, c, r);
    return (ad.x + ad.y + ad.z) * blend8<DT>(c, r);
  }
  // 16-byte FP32 texels: one map in flight at a time (24 would spill)
  Raw r[8];
  gather8<DT>(A.vol, lds_at(off, mx), c, r);
  float4 acc = ad.x * blend8<DT>(c, r);
  gather8<DT>(A.vol, lds_at(off + 2, my), c, r);
  acc = acc + ad.y * blend8<DT>(c, r);
  gather8<DT>(A.vol, lds_at(off + 4, mz), c, r);
  return acc + ad.z * blend8<DT>(c, r);
}

// sample_voxel (voxel_cone_tracing.frag:80-86) with its three textureLod
// calls folded together: lod clamped to [0, L-1], levels floor(lod) and
// floor(lod) + 1 blended by the fraction (the second only when it is > 0).
// mx, my, mz: the maps of the axes (face_of).
template <int DT>
__device__ __forceinline__ float4 sample_voxel(const TraceArgs& A, const SamplerLds* S, float3 p, float3 ad,
                                               uint32_t mx, uint32_t my, uint32_t mz, float lod) {
  const float lmax = (float)(A.levels - 1);
  lod = __builtin_amdgcn_fmed3f(lod, 0.0f, lmax);
  const float fl = floorf(lod);
  const int nl = (int)-fl;
  const float t = lod - fl;
  const float fs = __builtin_ldexpf((float)A.res, nl);
  const uint32_t row = (uint32_t)(nl * -(int)sizeof(S->off[0]));
  mx += row;
  my += row;
  mz += row;
  ad = make_float3(ad.x * kTexScale<DT>, ad.y * kTexScale<DT>, ad.z * kTexScale<DT>);
  float4 acc = sample_level<DT, true>(A, S, p, ad, mx, my, mz, nl == 0, fs);
  if (t > 0.0f) acc = (1.0f - t) * acc + t * sample_level<DT, false>(A, S, p, ad, mx, my, mz, false, fs * 0.5f);
  return tex_unscale<DT>(acc);
}

__device__ __forceinline__ float3 normalize3(float3 v) {
  const float l = sqrtf(v.x * v.x + v.y * v.y + v.z * v.z);
  return make_float3(v.x / l, v.y / l, v.z / l);
}
__device__ __forceinline__ float dot3(float3 a, float3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ float3 cross3(float3 a, float3 b) {
  return make_float3(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}
__device__ __forceinline__ float len3(float3 v) { return sqrtf(dot3(v, v)); }

// tangent (voxel_cone_tracing.frag:126-134)
__device__ __forceinline__ float3 tangent_of(float3 n) {
  const float3 t1 = cross3(n, make_float3(0.f, 0.f, 1.f));
  const float3 t2 = cross3(n, make_float3(0.f, 1.f, 0.f));
  return len3(t1) > len3(t2) ? normalize3(t1) : normalize3(t2);
}

__device__ __forceinline__ float3 refract3(float3 I, float3 N, float eta) {
  const float d = dot3(N, I);
  const float k = 1.0f - eta * eta * (1.0f - d * d);
  if (k < 0.0f) return make_float3(0.f, 0.f, 0.f);
  const float s = eta * d + sqrtf(k);
  return make_float3(eta * I.x - s * N.x, eta * I.y - s * N.y, eta * I.z - s * N.z);
}

// One workgroup = a block of Shape::NPIX pixels (NSUB sub-blocks of 8x8) x 4
// waves.  Waves 0..NSUB-1 set the shading pixels of their sub-block up (lane =
// pixel) into LDS.  The cones of the block - every pixel's specular,
// refraction and shadow cones, then its diffuse cones, longest kinds first -
// form one queue of (job, pixel) items, job-major so that neighbouring lanes
// start on the same cone of neighbouring pixels (coherent gathers).  Every
// lane marches its own item and takes the next one from a workgroup counter
// in LDS as soon as its cone ends, so lanes do not idle while the longest cone
// of a wave finishes.  The same waves then compose their pixels in the
// reference's order (voxel_cone_tracing.frag:246-275).
//
// What bounds the march is the number of cache lines a wave's load touches,
// not its instructions (cones set up 64 at a time for the idle lanes to take,
// which raises the lanes in use, measured no faster), so the queue takes the
// block's pixels sorted by the octant of their normal and their position:
// the lanes of a wave then read the same maps around the same place (128
// pixels, 2560x1440 soup: FP16 2.08 -> 1.94 ms, RGBA8 2.18 -> 2.13;
// pixel-major items instead of job-major ones 3.1 ms).
// job codes: 0..15 diffuse cone k, then:
constexpr int kJobSpecular = 16, kJobRefraction = 17, kJobShadow = 18;  // kJobShadow + light
constexpr int kMaxJobs = kJobShadow + VCT_MAX_LIGHTS;
// Idle lanes of a wave that trigger a refill: a refill costs the whole wave its
// set-up.  1M-triangle soup at 2560x1440, FP16 / RGBA8: 16 -> 1.90 / 2.02 ms, 24
// -> 1.90 / 2.06, 32 -> 1.96 / 2.11, 40 -> 2.04 / 2.21.  FP32, whose step is the
// longest, waits for more of them (50,000-triangle soup at 128^3; 16, 24, 32):
// 1001x563 1.13, 1.10, 1.11 ms, 2560x1440 3.72, 3.71, 3.85; in blocks of 64
// pixels 200x150 with two shadows 0.472, 0.458, 0.444, 640x360 0.810, 0.796, 0.780.
template <int DT, int NPIX>
constexpr int kRefillMin = DT != VCT_FP32 ? 16 : (NPIX == 64 ? 32 : 24);

// Block shapes: pixels per workgroup and the shadow-light slots in LDS.
// Cones are short in cluttered scenes (6.2 steps per cone of a covered pixel
// on a 1M-triangle soup), so a queue of 64 pixels x 10 cones gives each of the
// 256 lanes only 2.5 items and the drain at its end leaves a third of the
// lanes idle; more pixels per workgroup shorten the drain relative to the
// work.  The full shape holds shadow results of every light, the others of up
// to 2.
template <int NPIX_, int NSHADOW_>
struct Shape {
  static constexpr int NPIX = NPIX_, NSHADOW = NSHADOW_, NSUB = NPIX_ / 64;
  static constexpr int BX = NSUB == 3 ? 3 : (NSUB >= 2 ? 2 : 1);  // sub-blocks side by side (BX x NSUB/BX of 8x8)
  static_assert(NSUB <= 4, "one set-up wave per sub-block; pixel numbers are bytes");
};
using ShapeFull = Shape<128, VCT_MAX_LIGHTS>;
using ShapeTile = Shape<128, 2>;  // 32x32 tiles and long pixel lists
using ShapeSmall = Shape<64, 2>;  // small viewports and lists (see launch_trace)
// Whole viewports of the 16-bit types: 31 KB of LDS per 192 pixels let 5
// workgroups share a CU, as many as their registers do, and a longer run of
// sorted pixels shares more of its fetches (2560x1440 soup, FP16: 1.96 ms
// with 128 pixels, 1.89 with 192; 256 fit 4 workgroups only, 1.92).  RGBA8
// runs 6 waves per SIMD, which 128 pixels fit and 192 do not (2.08 against
// 2.18 ms with 256), and FP32 measures alike.
template <int DT>
struct WideOf {
  using type = ShapeTile;
};
template <>
struct WideOf<VCT_FP16> {
  using type = Shape<192, 2>;
};
template <>
struct WideOf<VCT_BF16> {
  using type = Shape<192, 2>;
};

// Waves per SIMD the kernels are compiled for, and what measured (2560x1440
// soup, RGBA8: 6 waves in 79 registers 2.08 ms, 5 waves 2.13; 1001x563,
// FP32: 4 waves in 126 registers 0.367 ms, 5 waves and 24 bytes of scratch
// 0.398; the 16-bit types hold 12 paired loads in flight and spill past 5).
template <int DT>
constexpr int kTraceWaves = kBytes<DT> ? 6 : (DT == VCT_FP32 ? 4 : 5);

// 32.32 fixed point of a non-negative cone colour channel (< 2^31): sums of
// these are exact, so the diffuse cones of a pixel may finish in any order.
__device__ __forceinline__ unsigned long long fix32(float v) { return __float2ull_rn(v * 4294967296.0f); }

// LDS of one workgroup of the cone marcher.
template <class SH>
struct ShadeLds {
  unsigned long long dsum[3][SH::NPIX];  // sum of the diffuse cones' rgb per pixel (fix32)
  float cone[2][3][SH::NPIX];            // specular, refraction rgb per pixel
  float shadow[SH::NSHADOW][SH::NPIX];   // max(0, 1 - alpha) of the shadow cone per light and pixel
  float pos[3][SH::NPIX], nrm[3][SH::NPIX], o1[3][SH::NPIX], o2[3][SH::NPIX], vdir[3][SH::NPIX];
  float spec_ap[SH::NPIX], eta[SH::NPIX];
  unsigned long long refr_mask[SH::NSUB];  // shading pixels with a transmissive material, per sub-block
  int sub_count[SH::NSUB];                 // shading pixels per sub-block
  uint32_t key[SH::NPIX];  // order of the block's pixels in the queue
  int npx, njobs, next_item;
  uint8_t px_of[SH::NPIX];  // the block's shading pixels, compacted
  int8_t jobs[kMaxJobs];
};

// The march state of one lane's cone (trace_cone, voxel_cone_tracing.frag:88-119).
// Registers are what bounds the marcher's occupancy, so only what cannot be
// derived is kept: |dir| and the three maps a sample reads follow from dir
// (abs is a free operand modifier), the diameter is dist * aperture, and the
// origin is the pixel's surface point, read from LDS where it is needed.
struct Cone {
  float3 dir;
  float ap, max_dist, dist;
  float4 c;
};

// The origin of the cone of block pixel `pix`, read from LDS where it is
// used.  A volatile read (forcing a re-read at every step) measured 0.11 ms
// slower on the 2560x1440 frame than letting the compiler schedule the reads.
template <int NPIX>
__device__ __forceinline__ float3 cone_origin(const float (*pos)[NPIX], int pix) {
  const float* p = &pos[0][0];
  return make_float3(p[pix], p[NPIX + pix], p[2 * NPIX + pix]);
}

// The distance along an axis at which a cone from o moving by d per unit is
// `margin` outside the unit cube on that axis, rounded up by far more than its
// rounding; NaN or infinite for d = 0.
__device__ __forceinline__ float exit_dist(float o, float d, float margin) {
  const float room = d < 0.0f ? o : 1.0f - o;
  return (room + margin + 1e-6f) * __builtin_amdgcn_rcpf(fabsf(d)) * (1.0f + 1e-5f);
}

// Besides max_dist the march ends where every later sample is zero: a sample
// more than half a texel of the coarsest level (`margin`) outside the unit
// cube reads only the zero border, and once the cone is that far out and
// moving away on an axis it never returns.  The distance at which that happens
// is computed once per cone (testing the position at every step took three
// branches per step more).
__device__ __forceinline__ void cone_begin(Cone& k, float3 dir, float3 origin, float aperture, float max_dist,
                                           float vs, float margin) {
  dir = normalize3(dir);
  k.dir = dir;
  // A cone never needs to leave the volume by more than its diagonal; the
  // bound also keeps a non-finite target distance from looping forever.
  k.max_dist = fminf(fminf(fminf(max_dist, 3.4641016f), exit_dist(origin.x, dir.x, margin)),
                     fminf(exit_dist(origin.y, dir.y, margin), exit_dist(origin.z, dir.z, margin)));
  k.ap = aperture;
  k.c = f4(0.0f);
  k.dist = 3.0f * vs;
}

// The loop condition of trace_cone.
__device__ __forceinline__ bool cone_alive(const Cone& k) { return k.c.w < 1.0f && k.dist < k.max_dist; }

// log2 of a cone's diameter in voxels by the hardware instruction alone: the
// diameter is at least 3 * 0.0174533 voxels (three voxels out, the narrowest
// aperture), so log2f's scaling of subnormal arguments never applies.
__device__ __forceinline__ float log2_of(float x) { return __builtin_amdgcn_logf(x); }

template <int DT>
__device__ __forceinline__ void cone_step(const TraceArgs& A, const SamplerLds* S, Cone& k, float3 origin, float vs,
                                          float fres) {
  const float3 sp = make_float3(k.dir.x * k.dist + origin.x, k.dir.y * k.dist + origin.y,
                                k.dir.z * k.dist + origin.z);
  const float diam = k.dist * k.ap;
  const float mip = log2_of(diam * fres);  // sample_voxel clamps it to the levels there are
  // face_indices (voxel_cone_tracing.frag:71-78): the map of each axis by the sign of dir
  const float3 ad = make_float3(fabsf(k.dir.x), fabsf(k.dir.y), fabsf(k.dir.z));
  const float4 s = sample_voxel<DT>(A, S, sp, ad, face_of(k.dir.x), face_of(k.dir.y), face_of(k.dir.z), mip);
  k.c = k.c + (1.0f - k.c.w) * s;
  k.dist += fmaxf(diam * 0.5f, vs);
}

// Direction of light li seen from pos (biased coordinates) and the distance
// the shadow cone may travel (direct_light, voxel_cone_tracing.frag:175-218).
__device__ __forceinline__ float3 light_dir(const TraceArgs& A, int li, float3 pos, float& d) {
  const DevLight& Lt = A.lights.l[li];
  if (Lt.kind == VCT_LIGHT_DIRECTIONAL) {
    d = 1.73205080757f;
    return normalize3(make_float3(Lt.pos[0], Lt.pos[1], Lt.pos[2]));
  }
  const float3 lp = make_float3(0.5f * (Lt.pos[0] / A.cube_size) + 0.5f, 0.5f * (Lt.pos[1] / A.cube_size) + 0.5f,
                                0.5f * (Lt.pos[2] / A.cube_size) + 0.5f);
  const float3 v = make_float3(lp.x - pos.x, lp.y - pos.y, lp.z - pos.z);
  d = len3(v);
  return normalize3(v);
}

template <int N>
__device__ __forceinline__ float3 ld3(const float (*a)[N], int p) { return make_float3(a[0][p], a[1][p], a[2][p]); }

// Shades the block's pixels; where(sub, lane, px, py, oidx, valid) gives the
// pixel of a lane of sub-block `sub`, where its result goes and whether it is
// traced.  L->next_item must be 0 and visible to the workgroup on entry.
template <int DT, class SH, class Where>
__device__ __forceinline__ void shade_block(const TraceArgs& A, Where&& where, ShadeLds<SH>* L, const SamplerLds* S) {
  const int lane = threadIdx.x & 63;
  const int grp = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));  // wave-uniform: a scalar register
  const int me = grp * 64 + lane;  // the thread's pixel in the block (set-up and composition waves)
  size_t idx = 0, oidx = 0;
  bool valid = false;
  auto locate = [&](int ln) {
    int px, py;
    where(grp, ln, px, py, oidx, valid);
    valid = valid && px < A.W && py < A.H;
    idx = valid ? (size_t)py * A.W + px : 0;
  };
  if (grp < SH::NSUB) locate(lane);
  const float sqrt3 = 1.73205080757f;
  const int nd = A.en_diffuse ? A.cones.n : 0;
  const bool do_spec = A.en_specular != 0;
  const int nl = A.lights.count < VCT_MAX_LIGHTS ? A.lights.count : VCT_MAX_LIGHTS;
  // ---- set-up of the block's pixels (wave 0, lane = pixel) -------------------
  auto pixel = [&](float4& gp, float4& gn, const DevMaterial*& m, float3& pos, int& mode) {
    gp = A.gpos[idx];
    gn = A.gnrm[idx];
    uint32_t mid = __builtin_bit_cast(uint32_t, gn.w);
    mid = mid < A.nmat ? mid : 0u;  // ids of an uploaded G-buffer are not trusted
    m = &A.mats[mid];
    pos = make_float3(0.5f * (gp.x / A.cube_size) + 0.5f, 0.5f * (gp.y / A.cube_size) + 0.5f,
                      0.5f * (gp.z / A.cube_size) + 0.5f);
    // 0: nothing to do, 1: background / outside the cube, 2: voxel view, 3: shade
    mode = 0;
    if (valid) {
      if (gp.w == 0.0f || !(fabsf(pos.x) < 1.0f && fabsf(pos.y) < 1.0f && fabsf(pos.z) < 1.0f)) mode = 1;
      else mode = A.view_dir < 7 ? 2 : 3;  // within_cube on biased coordinates (:250, :61-64)
    }
  };
  unsigned long long shade = 0ull;
  uint32_t mykey = ~0u;
  if (grp < SH::NSUB) {
    float4 gp, gn;
    const DevMaterial* m;
    float3 pos;
    int mode;
    pixel(gp, gn, m, pos, mode);
    const float3 n = make_float3(gn.x, gn.y, gn.z);
    const float3 cam = make_float3(A.cam[0], A.cam[1], A.cam[2]);
    const float3 vd = normalize3(make_float3(gp.x - cam.x, gp.y - cam.y, gp.z - cam.z));
    // specular aperture (:220-227)
    const float rough = sqrtf(2.0f / (m->shininess + 2.0f));
    L->spec_ap[me] = fminf(fmaxf(tanf(1.57079f * rough), 0.0174533f), 3.14159265f);
    L->eta[me] = 1.0f / m->ior;
    float3 o1 = make_float3(0.f, 0.f, 0.f), o2 = o1;
    if (mode == 3 && nd > 0) {
      o1 = normalize3(tangent_of(n));  // trace_diffuse (:146-147)
      o2 = normalize3(cross3(o1, n));
    }
    L->dsum[0][me] = 0ull;
    L->dsum[1][me] = 0ull;
    L->dsum[2][me] = 0ull;
    const float3 vals[5] = {pos, n, o1, o2, vd};
    float (*dst[5])[SH::NPIX] = {L->pos, L->nrm, L->o1, L->o2, L->vdir};
#pragma unroll
    for (int q = 0; q < 5; ++q) {
      dst[q][0][me] = vals[q].x;
      dst[q][1][me] = vals[q].y;
      dst[q][2][me] = vals[q].z;
    }
    shade = __ballot(mode == 3);
    // the pixel's place in the queue's order: the octant of its normal, then
    // its position in cells of two voxels along the Morton curve
    {
      const float sc = 0.5f * (float)min(A.res, 256);
      auto cell = [&](float v) { return (uint32_t)min(max((int)(v * sc), 0), 127); };
      const uint32_t oct = (n.x < 0.0f ? 1u : 0u) | (n.y < 0.0f ? 2u : 0u) | (n.z < 0.0f ? 4u : 0u);
      mykey = mode == 3 ? (((oct << 21) | morton3(cell(pos.x), cell(pos.y), cell(pos.z))) << 8) | (uint32_t)me : ~0u;
      L->key[me] = mykey;
    }
    const unsigned long long refr = __ballot(mode == 3 && do_spec && illum_transmissive(m->illum));
    if (lane == 0) {
      L->sub_count[grp] = __popcll(shade);
      L->refr_mask[grp] = refr;
    }
  }
  __syncthreads();
  if (grp < SH::NSUB) {
    // the block's shading pixels, compacted in the order of their keys
    int total = 0;
    bool refr = false;
#pragma unroll
    for (int w = 0; w < SH::NSUB; ++w) {
      total += L->sub_count[w];
      refr = refr || L->refr_mask[w] != 0ull;
    }
    uint32_t rank = 0;  // keys are distinct: a pixel's place is the number of smaller ones
#pragma unroll 8
    for (int q = 0; q < SH::NPIX; ++q) rank += L->key[q] < mykey ? 1u : 0u;
    if (mykey != ~0u) L->px_of[rank] = (uint8_t)me;
    if (me == 0) {
      L->npx = total;
      int nj = 0;  // longest kinds first
      if (do_spec) L->jobs[nj++] = kJobSpecular;
      if (refr) L->jobs[nj++] = kJobRefraction;
      if (A.en_direct && A.en_shadow)
        for (int li = 0; li < nl; ++li) L->jobs[nj++] = (int8_t)(kJobShadow + li);
      for (int k = 0; k < nd; ++k) L->jobs[nj++] = (int8_t)k;
      L->njobs = nj;
    }
  }
  __syncthreads();
  // ---- the cone queue (every lane) -----------------------------------------------
  const float vs = 1.0f / (float)A.res, fres = (float)A.res;
  const float margin = 0.5f * (float)(1u << (A.levels - 1)) * vs;
  const int npx = L->npx;
  const int nitems = npx * L->njobs;
  // it / npx as (it * ceil(2^22 / npx)) >> 22: exact for it < kMaxJobs * npx and npx <= 256
  const uint32_t npx_inv = npx ? (1u << 22) / (uint32_t)npx + (((1u << 22) % (uint32_t)npx) ? 1u : 0u) : 0u;
  // the lane's cone: job << 8 | pixel while it marches, -1 while it idles
  int cur = -1;
  unsigned long long wave_steps = 0;  // cone steps of the wave (uniform)
  bool drained = nitems == 0;
  Cone k;
  auto finish = [&](int job, int pix) {
    if (job >= kJobShadow) {
      L->shadow[job - kJobShadow][pix] = fmaxf(0.0f, 1.0f - k.c.w);
    } else {
      if (job < kJobSpecular) {
        atomicAdd(&L->dsum[0][pix], fix32(k.c.x));
        atomicAdd(&L->dsum[1][pix], fix32(k.c.y));
        atomicAdd(&L->dsum[2][pix], fix32(k.c.z));
      } else {
        const int slot = job == kJobSpecular ? 0 : 1;
        L->cone[slot][0][pix] = k.c.x;
        L->cone[slot][1][pix] = k.c.y;
        L->cone[slot][2][pix] = k.c.z;
      }
    }
  };
  for (;;) {
    // lanes without a cone take the next items of the queue, once enough of
    // them idle (or none is busy): a refill costs the whole wave its set-up
    const unsigned long long busy = __ballot(cur >= 0);
    for (;;) {
      const bool need = cur < 0 && !drained;
      const unsigned long long want = __ballot(need);
      if (!want || (busy && __popcll(want) < kRefillMin<DT, SH::NPIX>)) break;
      const int first = __ffsll((long long)want) - 1;
      int base = 0;
      if (lane == first) base = atomicAdd(&L->next_item, __popcll(want));
      base = __shfl(base, first);
      if (!need) continue;
      const int it = base + __popcll(want & ((1ull << lane) - 1ull));
      if (it >= nitems) {
        drained = true;
        continue;
      }
      const int j = (int)(((uint32_t)it * npx_inv) >> 22);
      const int job = L->jobs[j];
      const int pix = L->px_of[it - j * npx];
      if (job == kJobRefraction && !((L->refr_mask[pix >> 6] >> (pix & 63)) & 1ull)) continue;  // opaque: no item
      const float3 pos = ld3(L->pos, pix), n = ld3(L->nrm, pix);
      float3 d;
      float ap, md = sqrt3;
      if (job < kJobSpecular) {
        const float a = A.cones.a[job], b = A.cones.b[job], cc = A.cones.c[job];
        const float3 o1 = ld3(L->o1, pix), o2 = ld3(L->o2, pix);
        d = make_float3(a * n.x + b * o1.x + cc * o2.x, a * n.y + b * o1.y + cc * o2.y, a * n.z + b * o1.z + cc * o2.z);
        ap = A.cones.aperture;
      } else if (job == kJobSpecular) {
        // normalize(reflect(-view_dir, n)) (:231), normalised again in trace_cone (:90)
        const float3 vd = ld3(L->vdir, pix);
        const float3 I = make_float3(-vd.x, -vd.y, -vd.z);
        const float dn = 2.0f * dot3(n, I);
        d = normalize3(make_float3(I.x - dn * n.x, I.y - dn * n.y, I.z - dn * n.z));
        ap = L->spec_ap[pix];
      } else if (job == kJobRefraction) {
        d = refract3(ld3(L->vdir, pix), n, L->eta[pix]);  // trace_refraction (:237-241)
        ap = L->spec_ap[pix];
      } else {
        d = light_dir(A, job - kJobShadow, pos, md);  // shadow cone of direct_light
        ap = 0.1f;
      }
      cone_begin(k, d, pos, ap, md, vs, margin);
      if (cone_alive(k)) cur = (job << 8) | pix;
      else finish(job, pix);  // no step at all
    }
    const unsigned long long active = __ballot(cur >= 0);
    if (!active) break;
    wave_steps += (unsigned long long)__popcll(active);
    if (cur >= 0) {
      cone_step<DT>(A, S, k, cone_origin(L->pos, cur & 255), vs, fres);
      if (!cone_alive(k)) {
        finish(cur >> 8, cur & 255);
        cur = -1;
      }
    }
  }
  if (A.step_counter && lane == 0 && wave_steps) atomicAdd(A.step_counter, wave_steps);
  __syncthreads();
  // ---- composition (waves 0..NSUB-1, lane = pixel) -----------------------------------
  if (grp >= SH::NSUB) return;
  // the thread's pixel again, from the scalar wave index and a lane id the
  // compiler cannot match with the first: nothing per lane is held over the
  // cone queue
  int lane_c = (int)__lane_id();
  asm volatile("" : "+v"(lane_c));
  const int me_c = grp * 64 + lane_c;
  locate(lane_c);
  float4 gp, gn;
  const DevMaterial* mp;
  float3 pos;
  int mode;
  pixel(gp, gn, mp, pos, mode);
  if (mode == 0) return;
  const float4 bg = make_float4(0.15f, 0.25f, 0.25f, 1.0f);  // renderer.cpp:398
  if (mode == 1) {
    A.image[oidx] = A.demodulate ? f4(0.0f) : bg;
    return;
  }
  if (mode == 2) {  // voxel view (:253-257), blended SRC_ALPHA / ONE_MINUS_SRC_ALPHA
    const int d = A.view_dir < 0 ? 0 : (A.view_dir > 5 ? 5 : A.view_dir);
    float3 ad = make_float3(0.f, 0.f, 0.f);
    const uint32_t face = d & 1 ? 0u : 4u;  // the even maps are the negative directions
    if (d < 2) ad.x = 1.0f;
    else if (d < 4) ad.y = 1.0f;
    else ad.z = 1.0f;
    const float4 s = sample_voxel<DT>(A, S, pos, ad, face, face, face, A.view_lod);
    const float a = s.w;
    A.image[oidx] = make_float4(s.x * a + bg.x * (1.0f - a), s.y * a + bg.y * (1.0f - a),
                                s.z * a + bg.z * (1.0f - a), a * a + bg.w * (1.0f - a));
    return;
  }
  const DevMaterial& m = *mp;
  const float3 n = make_float3(gn.x, gn.y, gn.z);
  const float3 view_dir = ld3(L->vdir, me_c);
  const bool do_refr = (L->refr_mask[grp] >> lane_c) & 1ull;
  float3 out = make_float3(0.f, 0.f, 0.f);
  if (nd > 0) {
    // the exact sum of the diffuse cones, rounded once (trace_diffuse adds
    // them in cone order in FP32, :144-167)
    const float u = 1.0f / 4294967296.0f;
    const float3 diff_acc = make_float3(__ull2float_rn(L->dsum[0][me_c]) * u, __ull2float_rn(L->dsum[1][me_c]) * u,
                                        __ull2float_rn(L->dsum[2][me_c]) * u);
    const float inv = 1.0f / (float)nd;
    out.x += m.diffuse[0] * (diff_acc.x * inv);
    out.y += m.diffuse[1] * (diff_acc.y * inv);
    out.z += m.diffuse[2] * (diff_acc.z * inv);
  }
  if (A.en_direct) {  // direct_light (:175-218) with the shadow cones' results
    float3 res = make_float3(0.f, 0.f, 0.f);
    for (int li = 0; li < nl; ++li) {
      const DevLight& Lt = A.lights.l[li];
      float d;
      const float3 ldir = light_dir(A, li, pos, d);
      const float cos_surf = fmaxf(dot3(n, ldir), 0.0f);
      const float att = (Lt.kind == VCT_LIGHT_DIRECTIONAL) ? 1.0f : 1.0f / (1.0f + d * d);
      const float kk = att * cos_surf;
      const float3 lc = make_float3(kk * Lt.color[0] * Lt.intensity, kk * Lt.color[1] * Lt.intensity,
                                    kk * Lt.color[2] * Lt.intensity);
      const float shadow = A.en_shadow ? L->shadow[li][me_c] : 1.0f;
      const float lambert = fmaxf(dot3(ldir, n), 0.0f);
      float refr_angle = 0.0f;
      if (m.dissolve <= 0.1f) {
        const float3 r = refract3(view_dir, n, 1.0f / m.ior);
        refr_angle = fmaxf((1.0f - m.dissolve) * dot3(r, ldir), 0.0f);
      }
      const float3 hv = normalize3(make_float3(ldir.x + view_dir.x, ldir.y + view_dir.y, ldir.z + view_dir.z));
      float sa = fmaxf(dot3(hv, n), 0.0f);
      sa = fmaxf(sa, refr_angle);
      const float sc = powf(sa, m.shininess);
      const float f = shadow + 0.04f;
      res.x += f * (lambert * m.diffuse[0] + sc * m.specular[0]) * lc.x;
      res.y += f * (lambert * m.diffuse[1] + sc * m.specular[1]) * lc.y;
      res.z += f * (lambert * m.diffuse[2] + sc * m.specular[2]) * lc.z;
    }
    out.x += res.x + fminf(fmaxf(m.emission[0], 0.0f), 1.0f);
    out.y += res.y + fminf(fmaxf(m.emission[1], 0.0f), 1.0f);
    out.z += res.z + fminf(fmaxf(m.emission[2], 0.0f), 1.0f);
  }
  if (do_spec) {
    out.x += m.specular[0] * L->cone[0][0][me_c];
    out.y += m.specular[1] * L->cone[0][1][me_c];
    out.z += m.specular[2] * L->cone[0][2][me_c];
  }
  if (do_refr) {  // final colour override (:273-274)
    const float3 tr = make_float3(m.transmittance[0] * L->cone[1][0][me_c],
                                  m.transmittance[1] * L->cone[1][1][me_c],
                                  m.transmittance[2] * L->cone[1][2][me_c]);
    const float dv = m.dissolve;
    out = make_float3(tr.x * (1.0f - dv) + out.x * dv, tr.y * (1.0f - dv) + out.y * dv,
                      tr.z * (1.0f - dv) + out.z * dv);
  }
  float ow = 1.0f;
  if (A.demodulate) {
    const float e = 1.0f / 1024.0f;
    out = make_float3(out.x / fmaxf(m.diffuse[0], e), out.y / fmaxf(m.diffuse[1], e), out.z / fmaxf(m.diffuse[2], e));
    ow = gp.w;  // linear depth of the traced pixel
  }
  A.image[oidx] = make_float4(out.x, out.y, out.z, ow);
}

// Work of a launch: the whole viewport (trace_frame_kernel, one workgroup per
// block of NSUB 8x8 sub-blocks side by side), or a device-side list of pixels
// (NPIX per chunk) or tiles (16 sub-blocks of 8x8 pixels per tile, or 4 of
// 8x8 odd-odd grid points, NSUB per chunk) for trace_list_kernel.  At the waves
// of kTraceWaves no storage type needs scratch: the 12 paired loads of a
// three-map level (16-bit storage; 6 for RGBA8, FP32 one map's 8) are in flight
// together.
template <int DT, class SH>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kTraceWaves<DT>))) void trace_frame_kernel(TraceArgs A) {
  __shared__ ShadeLds<SH> s_shade;
  __shared__ SamplerLds s_sampler;
  sampler_init<DT>(A, &s_sampler);
  if (threadIdx.x == 0) s_shade.next_item = 0;
  __syncthreads();
  // Workgroups are dealt to the 8 XCDs round-robin in dispatch order.  XCD k
  // takes the block rows k, k + 8, k + 16, ... each left to right, so each
  // XCD's L2 serves whole rows of neighbouring blocks, and the 8 XCDs work
  // on rows spread over the image (rows left over below a multiple of 8
  // keep the dispatch order).  Measured at 2560x1440: trace 2.54 ms with
  // the dispatch order, 2.46 with one band of the image per XCD, 2.36 with
  // interleaved rows.
  const uint32_t gx = gridDim.x, gy = gridDim.y;
  uint32_t b = blockIdx.x + blockIdx.y * gx;
  if (b < (gy & ~7u) * gx) {
    const uint32_t q = b >> 3;
    b = ((q / gx) * 8u + (b & 7u)) * gx + q % gx;
  }
  const int bx = (int)(b % gx), by = (int)(b / gx);
  shade_block<DT, SH>(
      A,
      [&](int sub, int lane, int& px, int& py, size_t& oidx, bool& valid) {
        px = bx * (8 * SH::BX) + (sub % SH::BX) * 8 + (lane & 7);
        py = by * (8 * (SH::NSUB / SH::BX)) + (sub / SH::BX) * 8 + (lane >> 3);
        oidx = (size_t)py * A.W + px;
        valid = true;
      },
      &s_shade, &s_sampler);
}

// Chunks (npix pixels each) of a list launch.
__device__ __forceinline__ uint32_t list_chunks(const TraceArgs& A, uint32_t npix) {
  if (A.pix_list) return ((A.pix_count ? min(*A.pix_count, A.npix_list) : A.npix_list) + npix - 1u) / npix;
  return *A.tile_count * (A.grid_stride == 2 ? 4u : 16u) / (npix / 64u);
}

// The pixel of `lane` of sub-block `sub` in chunk c (nsub sub-blocks of 64
// pixels per chunk), where its result goes, and whether it is traced.
__device__ __forceinline__ void list_chunk(const TraceArgs& A, uint32_t c, uint32_t nsub, uint32_t sub, int lane,
                                           int& px, int& py, size_t& oidx, bool& valid) {
  valid = true;
  if (A.pix_list) {
    const uint32_t cnt = A.pix_count ? min(*A.pix_count, A.npix_list) : A.npix_list;
    const uint32_t k = (c * nsub + sub) * 64u + (uint32_t)lane;
    valid = k < cnt;
    const uint32_t p = valid ? A.pix_list[k] : 0u;
    px = (int)(p % (uint32_t)A.W);
    py = (int)(p / (uint32_t)A.W);
    oidx = A.pix_scatter ? (size_t)p : (size_t)k;
    if (valid && A.tile_flag) valid = A.tile_flag[(py >> 5) * A.tiles_x + (px >> 5)] == A.flag_want;
    return;
  }
  const uint32_t per = A.grid_stride == 2 ? 4u : 16u;  // sub-blocks per tile
  const uint32_t g = c * nsub + sub;                    // sub-block index over the list
  const uint32_t t = A.tile_list[g / per], b = g % per;
  if (A.grid_stride == 2) {  // grid point (u, v) is pixel (2u + 1, 2v + 1)
    const int gu = (int)(t % (uint32_t)A.tiles_x) * 16 + (int)(b & 1u) * 8 + (lane & 7);
    const int gv = (int)(t / (uint32_t)A.tiles_x) * 16 + (int)(b >> 1) * 8 + (lane >> 3);
    px = 2 * gu + 1;
    py = 2 * gv + 1;
    oidx = (size_t)gv * A.half_w + gu;
  } else {
    px = (int)(t % (uint32_t)A.tiles_x) * 32 + (int)(b & 3u) * 8 + (lane & 7);
    py = (int)(t / (uint32_t)A.tiles_x) * 32 + (int)(b >> 2) * 8 + (lane >> 3);
    oidx = (size_t)py * A.W + px;
  }
}

// One chunk per workgroup; workgroups past the device-side count leave at once.
// (A fixed grid striding over the chunks measured slower: the loop costs the
// kernel registers and spills at 4 waves per SIMD.)
template <int DT, class SH>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kTraceWaves<DT>))) void trace_list_kernel(TraceArgs A) {
  __shared__ ShadeLds<SH> s_shade;
  __shared__ SamplerLds s_sampler;
  if (blockIdx.x >= list_chunks(A, SH::NPIX)) return;
  sampler_init<DT>(A, &s_sampler);
  if (threadIdx.x == 0) s_shade.next_item = 0;
  __syncthreads();
  shade_block<DT, SH>(
      A,
      [&](int sub, int lane, int& px, int& py, size_t& oidx, bool& valid) {
        list_chunk(A, blockIdx.x, SH::NSUB, (uint32_t)sub, lane, px, py, oidx, valid);
      },
      &s_shade, &s_sampler);
}

// Builds the x-paired copy of every (level, map) of the volume in one launch:
// thread g covers texel g of the concatenated maps (level 0, then the 6 maps
// of each higher level).  The +x neighbour of Morton index m is the Morton
// increment of its x bits; the last column pairs with zero.
struct PairArgs {
  const char* src;
  char* dst;
  uint64_t src_off[16][6], dst_off[16][6];
  int first, levels;  // levels first .. levels - 1
  uint32_t res;
  uint64_t total;  // texels over all their maps
};

template <int DT>
__global__ __launch_bounds__(256) void pair_kernel(PairArgs P) {
  using T = typename Tex<DT>::Raw;
  using PR = typename Pair<DT>::Raw;
  for (uint64_t g = (uint64_t)blockIdx.x * 256u + threadIdx.x; g < P.total; g += (uint64_t)gridDim.x * 256u) {
    uint64_t r = g;
    int l = P.first, d = 0;
    uint32_t s = P.res >> l;
    uint64_t n = (uint64_t)s * s * s;
    if (l > 0 || r >= n) {
      if (l == 0) {
        r -= n;
        l = 1;
      }
      for (; l < P.levels; ++l) {
        s = P.res >> l;
        n = (uint64_t)s * s * s;
        if (r < 6 * n) break;
        r -= 6 * n;
      }
      d = (int)(r / n);
      r -= (uint64_t)d * n;
    }
    const uint32_t m = (uint32_t)r;
    const uint32_t mx = spread3(s - 1u);  // x bits of an index within this level
    const T* src = reinterpret_cast<const T*>(P.src + P.src_off[l][d]);
    const T a = src[m];
    T b;
    memset(&b, 0, sizeof(b));
    if ((m & mx) != mx) b = src[(((m | ~mx) + 1u) & mx) | (m & ~mx)];
    reinterpret_cast<PR*>(P.dst + P.dst_off[l][d])[m] = Pair<DT>::make(a, b);
  }
}

// Builds the tiled copy of an RGBA8 volume, every (level, map) in one launch:
// workgroup b covers kTileLines lines of one map (level 0, then the 6 maps of
// each higher level).  A lane writes half a row of a line (two elements, 16
// bytes) from four texels, so a wave's stores are 1 KiB of consecutive bytes;
// the texels (each read for its own element, the one below and every third
// column twice) come from L1 and L2.
constexpr uint32_t kTileLines = 128;

__host__ __device__ inline uint32_t tile_blocks(uint32_t s) {  // workgroups of a map of edge s
  const uint32_t g = s > 1u ? s >> 1 : 1u;
  const uint32_t n = g * g * g;
  return n > kTileLines ? n / kTileLines : 1u;
}

__global__ __launch_bounds__(256) void tile_kernel(PairArgs P) {
  uint32_t b = blockIdx.x, s = P.res, d = 0;
  int l = 0;
  for (;;) {  // the workgroup's map (uniform)
    const uint32_t n = tile_blocks(s), maps = l == 0 ? 1u : 6u;
    if (b < maps * n) {
      d = b / n;
      b -= d * n;
      break;
    }
    b -= maps * n;
    ++l;
    s >>= 1;
  }
  const uint32_t* src = reinterpret_cast<const uint32_t*>(P.src + P.src_off[l][d]);
  char* dst = P.dst + P.dst_off[l][d];
  const uint32_t g = s > 1u ? s >> 1 : 1u;
  const uint32_t row = threadIdx.x & 7u;  // of the line: half row, y, z
#pragma unroll
  for (uint32_t k = 0; k < kTileLines; k += 32u) {
    const uint32_t line = b * kTileLines + k + (threadIdx.x >> 3);
    const uint32_t x = compact3(line) * kTileCols + 2u * (row & 1u);
    const uint32_t y = 2u * compact3(line >> 1) + ((row >> 1) & 1u), z = 2u * compact3(line >> 2) + (row >> 2);
    // lines past the last column's hold no texel anyone reads; the others'
    // columns and rows past the edge are zero
    if (line >= g * g * g || x - 2u * (row & 1u) >= s) continue;
    uint32_t t[2][2];
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i)
#pragma unroll
      for (uint32_t j = 0; j < 2; ++j)
        t[i][j] = x + i < s && y + j < s && z < s ? src[morton3(x + i, y + j, z)] : 0u;
    *reinterpret_cast<uint4*>(dst + ((uint64_t)line << 7) + row * 16u) = make_uint4(t[0][0], t[0][1], t[1][0], t[1][1]);
  }
}

// Ceiling of the marcher's texel loads: the rate at which the vector memory
// path delivers 16-byte-per-lane loads (global_load_dwordx4, the form of the
// marcher's paired-texel gathers) when every access hits the L1 cache.  All
// workgroups read one 16 KiB region (L1 holds 32 KiB), each wave's lanes
// 1 KiB of consecutive addresses per load (8 full cache lines: the fewest
// lines a 64 x 16-byte load can touch), 8 loads of distinct rows in flight
// per lane; the row advances by a run-time stride, so no load can be merged
// with another or moved out of the loop.  A gather touches more lines per
// load, so no access pattern of these loads is delivered faster.
__global__ __launch_bounds__(256) void load_peak_kernel(const uint4* __restrict__ src, uint32_t iters,
                                                        uint32_t stride, uint4* __restrict__ sink) {
  uint4 acc[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) acc[u] = make_uint4(0u, 0u, 0u, 0u);
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  for (uint32_t i = 0; i < iters; i += 8) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const uint32_t row = (wave + i * stride + (uint32_t)u) & 15u;  // the 16 KiB region in 1 KiB rows
      const uint4 v = src[row * 64u + lane];
      acc[u].x ^= v.x;
      acc[u].y ^= v.y;
      acc[u].z ^= v.z;
      acc[u].w ^= v.w;
    }
  }
  uint4 r = acc[0];
#pragma unroll
  for (int u = 1; u < 8; ++u) {
    r.x ^= acc[u].x;
    r.y ^= acc[u].y;
    r.z ^= acc[u].z;
    r.w ^= acc[u].w;
  }
  sink[(size_t)blockIdx.x * 256u + threadIdx.x] = r;  // keeps every load live
}

}  // namespace vct

using namespace vct;

extern "C" int vct_trace_load_peak(vct_ctx ctx, double* gbps) {
  if (!ctx) return vct_set_error(VCT_ERR_BAD_HANDLE, "null context");
  if (!gbps) return vct_set_error(VCT_ERR_INVALID_ARG, "null out");
  VCT_HIP(hipSetDevice(ctx->device));
  int cus = 0;
  VCT_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device));
  const uint32_t blocks = (uint32_t)std::max(cus, 1) * 8u, iters = 4096;
  int rc;
  VctBuf src, sink;
  if ((rc = vct_ensure(src, 16384, ctx))) return rc;
  if ((rc = vct_ensure(sink, (size_t)blocks * 256 * 16, ctx))) return rc;
  VCT_HIP(hipMemsetAsync(src.p, 0x5a, 16384, ctx->stream));
  float best = 0.0f;
  for (int rep = 0; rep < 4; ++rep) {  // the first launch also warms the caches
    VCT_HIP(hipEventRecord(ctx->ev[10], ctx->stream));
    hipLaunchKernelGGL(load_peak_kernel, dim3(blocks), dim3(256), 0, ctx->stream, (const uint4*)src.p, iters, 1u,
                       (uint4*)sink.p);
    VCT_HIP(hipGetLastError());
    VCT_HIP(hipEventRecord(ctx->ev[11], ctx->stream));
    VCT_HIP(hipEventSynchronize(ctx->ev[11]));
    float ms = 0.0f;
    VCT_HIP(hipEventElapsedTime(&ms, ctx->ev[10], ctx->ev[11]));
    const double bytes = (double)blocks * 256.0 * iters * 16.0;
    const float g = (float)(bytes / (ms * 1e-3) / 1e9);
    if (rep > 0 && g > best) best = g;
  }
  VCT_HIP(hipStreamSynchronize(ctx->stream));
  (void)hipFree(sink.p);
  (void)hipFree(src.p);
  *gbps = best;
  return VCT_OK;
}

// Cone direction tables in the tangent frame (n, o1, o2).
void vct_cone_set_table(int set, ConeSet& cs) {
  memset(&cs, 0, sizeof(cs));
  if (set == VCT_CONES_REF9) {
    // trace_diffuse (voxel_cone_tracing.frag:140-168): n, mix(n, +-o1/+-o2, .5),
    // mix(n, +-c1/+-c2, .5) with c1 = (o1 + o2) / 2, c2 = (o1 - o2) / 2.
    const float t[9][3] = {{1.f, 0.f, 0.f},      {.5f, .5f, 0.f},     {.5f, -.5f, 0.f},
                           {.5f, 0.f, .5f},      {.5f, 0.f, -.5f},    {.5f, .25f, .25f},
                           {.5f, -.25f, -.25f},  {.5f, .25f, -.25f},  {.5f, -.25f, .25f}};
    cs.n = 9;
    for (int i = 0; i < 9; ++i) {
      cs.a[i] = t[i][0];
      cs.b[i] = t[i][1];
      cs.c[i] = t[i][2];
    }
    cs.aperture = 0.55785173935f;  // TAN_22_5 (:136)
  } else if (set == VCT_CONES_5_WIDE) {
    const float t[5][3] = {{1.f, 0.f, 0.f}, {.5f, .5f, 0.f}, {.5f, -.5f, 0.f}, {.5f, 0.f, .5f}, {.5f, 0.f, -.5f}};
    cs.n = 5;
    for (int i = 0; i < 5; ++i) {
      cs.a[i] = t[i][0];
      cs.b[i] = t[i][1];
      cs.c[i] = t[i][2];
    }
    cs.aperture = 1.15470054f;  // 2 tan(30 deg): 60 degree cones
  } else {
    // 16 cones: the normal, 5 at 28 degrees, 10 at 58 degrees from it.
    cs.n = 16;
    cs.a[0] = 1.f;
    int k = 1;
    const double d2r = 3.14159265358979323846 / 180.0;
    for (int i = 0; i < 5; ++i, ++k) {
      double th = 28.0 * d2r, ph = 72.0 * i * d2r;
      cs.a[k] = (float)cos(th);
      cs.b[k] = (float)(sin(th) * cos(ph));
      cs.c[k] = (float)(sin(th) * sin(ph));
    }
    for (int i = 0; i < 10; ++i, ++k) {
      double th = 58.0 * d2r, ph = (36.0 * i + 18.0) * d2r;
      cs.a[k] = (float)cos(th);
      cs.b[k] = (float)(sin(th) * cos(ph));
      cs.c[k] = (float)(sin(th) * sin(ph));
    }
    cs.aperture = 0.45f;
  }
}

// The marcher's copy of the volume (x-paired 16-bit, tiled RGBA8 storage): its
// layout, the maps of its levels, and its rebuilding when the volume has changed
// since it was last built.  The mip pass builds it last; the marcher calls
// vct_ensure_pairs again for volumes written since (uploads).
int vct_pair_layout(vct_context* ctx) {
  const uint64_t bpe = dtype_bytes(ctx->dtype);
  uint64_t bytes = 0;
  for (int l = 0; l < ctx->levels; ++l) {
    const uint64_t map_bytes = (level_elems(ctx->res >> l) * vct_copy_factor(ctx->dtype) * bpe + 255) & ~255ull;
    for (int d = 0; d < 6; ++d) {
      ctx->pair_off[l][d] = bytes;
      if (l > 0) bytes += map_bytes;
    }
    if (l == 0) bytes += map_bytes;
  }
  return vct_ensure(ctx->pairs, bytes, ctx);
}

int vct_pairs_from(vct_context* ctx, int first) {
  int rc;
  if ((rc = vct_pair_layout(ctx))) return rc;
  PairArgs P;
  memset(&P, 0, sizeof(P));
  uint64_t total = 0;
  for (int l = 0; l < ctx->levels; ++l) {
    for (int d = 0; d < 6; ++d) {
      P.src_off[l][d] = ctx->lvl_off[l][d];
      P.dst_off[l][d] = ctx->pair_off[l][d];
    }
    if (l >= first) total += (l == 0 ? 1 : 6) * level_elems(ctx->res >> l);
  }
  if (total == 0) return VCT_OK;  // no level from `first` on
  P.src = (const char*)ctx->volume.p;
  P.dst = (char*)ctx->pairs.p;
  P.first = first;
  P.levels = ctx->levels;
  P.res = ctx->res;
  P.total = total;
  const dim3 grid((unsigned)std::min<uint64_t>((total + 255) / 256, 256ull * 64));
  switch (ctx->dtype) {
    case VCT_RGBA8: {  // every level: `first` is 0
      uint32_t blocks = 0;
      for (int l = 0; l < ctx->levels; ++l) blocks += (l == 0 ? 1u : 6u) * tile_blocks(ctx->res >> l);
      hipLaunchKernelGGL(tile_kernel, dim3(blocks), dim3(256), 0, ctx->stream, P);
      break;
    }
    case VCT_FP16: hipLaunchKernelGGL(pair_kernel<VCT_FP16>, grid, dim3(256), 0, ctx->stream, P); break;
    default: hipLaunchKernelGGL(pair_kernel<VCT_BF16>, grid, dim3(256), 0, ctx->stream, P); break;
  }
  VCT_HIP(hipGetLastError());
  return VCT_OK;
}

int vct_ensure_pairs(vct_context* ctx) {
  if (ctx->dtype == VCT_FP32 || ctx->pairs_version == ctx->volume_version) return VCT_OK;
  int rc;
  if ((rc = vct_pairs_from(ctx, 0))) return rc;
  ctx->pairs_version = ctx->volume_version;
  return VCT_OK;
}

int vct_trace_into(vct_context* ctx, const float4* gpos, const float4* gnrm, float4* out, int W, int H,
                   int demodulate, unsigned long long* step_counter) {
  TraceSelect sel;
  memset(&sel, 0, sizeof(sel));
  return vct_trace_select(ctx, gpos, gnrm, out, W, H, demodulate, step_counter, sel);
}

// Launches the marcher over the viewport in blocks of one shape.
template <int DT, class SH>
static void launch_frame(vct_context* ctx, const TraceArgs& A, int W, int H) {
  constexpr int bw = 8 * SH::BX, bh = 8 * (SH::NSUB / SH::BX);
  hipLaunchKernelGGL((trace_frame_kernel<DT, SH>), dim3((W + bw - 1) / bw, (H + bh - 1) / bh), dim3(256), 0,
                     ctx->stream, A);
}

// Launches it over a list: one workgroup per chunk of the largest the list can be.
template <int DT, class SH>
static void launch_list(vct_context* ctx, const TraceArgs& A, const TraceSelect& sel) {
  static_assert(4 % SH::NSUB == 0, "chunks of a listed tile's 16 sub-blocks, or of the 4 of its odd-odd pixels");
  const uint32_t chunks = sel.pix_list ? (sel.npix_list + SH::NPIX - 1) / SH::NPIX
                                       : (sel.grid_stride == 2 ? 4u : 16u) / SH::NSUB * sel.max_tiles;
  hipLaunchKernelGGL((trace_list_kernel<DT, SH>), dim3(chunks), dim3(256), 0, ctx->stream, A);
}

template <int DT>
static int launch_trace(vct_context* ctx, const TraceArgs& A, const TraceSelect& sel, int W, int H, bool wide) {
  if ((sel.pix_list && sel.npix_list == 0) || (!sel.pix_list && sel.tile_list && sel.max_tiles == 0)) return VCT_OK;
  // A pixel list runs beside other launches: workgroups of 64 pixels up to 2^18
  // of them (the learned frame's 57,600 probes, 3.257 -> 3.244 ms), else of 128.
  if (sel.pix_list || sel.tile_list) {
    if (!wide) {
      launch_list<DT, ShapeFull>(ctx, A, sel);
      return VCT_OK;
    }
    if constexpr (DT != kRgba8Unorm) {  // (the demodulated lists are lists of tiles)
      if (sel.pix_list && sel.npix_list <= 1u << 18) {
        launch_list<DT, ShapeSmall>(ctx, A, sel);
        return VCT_OK;
      }
    }
    launch_list<DT, ShapeTile>(ctx, A, sel);
    return VCT_OK;
  }
  // The 256 CUs hold about 1280 workgroups of any shape at once, so a viewport
  // of few workgroups runs a part-empty last round whose length is that of one
  // workgroup, all its pixels' cones: small viewports take small workgroups.
  // Up to 2^19 pixels 64 (trace at 753x400, BF16, sixteen cones and two shadows
  // a pixel: 0.78 ms in workgroups of 192 pixels, 0.53 of 128, 0.44 of 64;
  // 855x512 FP16 0.69, 0.57, 0.50; 1001x563 FP32 0.35 of 128, 0.38 of 64), up to
  // 3 * 2^18 128 (974x700 FP16: 0.182 of 64, 0.160 of 128, 0.162 of 192; 1363x767
  // BF16: 1.26, 1.27, 1.24).
  const size_t npix = (size_t)W * H;
  if (!wide) launch_frame<DT, ShapeFull>(ctx, A, W, H);
  else if (npix <= 1u << 19) launch_frame<DT, ShapeSmall>(ctx, A, W, H);
  else if (npix <= 3u << 18) launch_frame<DT, ShapeTile>(ctx, A, W, H);
  else launch_frame<DT, typename WideOf<DT>::type>(ctx, A, W, H);
  return VCT_OK;
}

int vct_trace_select(vct_context* ctx, const float4* gpos, const float4* gnrm, float4* out, int W, int H,
                     int demodulate, unsigned long long* step_counter, const TraceSelect& sel) {
  TraceArgs A;
  memset(&A, 0, sizeof(A));
  A.step_counter = step_counter;
  A.pix_list = sel.pix_list;
  A.npix_list = sel.npix_list;
  A.pix_count = sel.pix_count;
  A.pix_scatter = sel.pix_scatter;
  A.tile_list = sel.tile_list;
  A.tile_count = sel.tile_count;
  A.tiles_x = sel.tiles_x;
  A.tile_flag = sel.tile_flag;
  A.flag_want = sel.flag_want;
  A.grid_stride = sel.grid_stride;
  A.half_w = sel.half_w;
  int rc;
  if (ctx->res > (uint32_t)kMaxEdge) return vct_set_error(VCT_ERR_LIMIT, "the marcher samples grids of at most 512^3");
  if ((rc = vct_ensure_pairs(ctx))) return rc;
  const bool paired = ctx->dtype != VCT_FP32;
  A.vol = (const char*)(paired ? ctx->pairs.p : ctx->volume.p);
  for (int l = 0; l < ctx->levels; ++l)
    for (int d = 0; d < 6; ++d) A.off[l][d] = paired ? ctx->pair_off[l][d] : ctx->lvl_off[l][d];
  A.levels = ctx->levels;
  A.res = (int)ctx->res;
  A.gpos = gpos;
  A.gnrm = gnrm;
  A.mats = (const DevMaterial*)ctx->d_materials.p;
  A.nmat = (uint32_t)ctx->materials.size();
  A.image = out;
  A.W = W;
  A.H = H;
  A.cube_size = ctx->cube_size;
  // camera_position = column 3 of the view matrix (renderer.cpp:279)
  A.cam[0] = ctx->view[12];
  A.cam[1] = ctx->view[13];
  A.cam[2] = ctx->view[14];
  A.en_direct = ctx->en_direct;
  A.en_diffuse = ctx->en_diffuse;
  A.en_specular = ctx->en_specular;
  A.en_shadow = ctx->en_shadow;
  A.view_dir = ctx->view_voxel_dir;
  A.view_lod = ctx->view_voxel_lod;
  A.demodulate = demodulate;
  vct_cone_set_table(ctx->cone_set, A.cones);
  int n = (int)ctx->lights.size();
  if (n > VCT_MAX_LIGHTS) n = VCT_MAX_LIGHTS;
  for (int i = 0; i < n; ++i) {
    for (int k = 0; k < 3; ++k) {
      A.lights.l[i].pos[k] = ctx->lights[i].position[k];
      A.lights.l[i].color[k] = ctx->lights[i].color[k];
    }
    A.lights.l[i].intensity = ctx->lights[i].intensity;
    A.lights.l[i].kind = ctx->lights[i].kind;
  }
  A.lights.count = n;
  // the wide shape holds the shadows of up to 2 lights
  const int nshadow = (ctx->en_direct && ctx->en_shadow) ? n : 0;
  const bool wide = nshadow <= ShapeTile::NSHADOW;
  switch (ctx->dtype) {
    case VCT_RGBA8:
      if (demodulate) rc = launch_trace<kRgba8Unorm>(ctx, A, sel, W, H, wide);
      else rc = launch_trace<VCT_RGBA8>(ctx, A, sel, W, H, wide);
      break;
    case VCT_FP16: rc = launch_trace<VCT_FP16>(ctx, A, sel, W, H, wide); break;
    case VCT_BF16: rc = launch_trace<VCT_BF16>(ctx, A, sel, W, H, wide); break;
    default: rc = launch_trace<VCT_FP32>(ctx, A, sel, W, H, wide); break;
  }
  if (rc) return rc;
  VCT_HIP(hipGetLastError());
  return VCT_OK;
}

int vct_launch_trace(vct_context* ctx) {
  const size_t npix = (size_t)ctx->width * ctx->height;
  if (!ctx->g_pos.p || ctx->g_pos.cap < npix * 16)
    return vct_set_error(VCT_ERR_STATE, "trace needs a G-buffer of the current viewport (run vct_gbuffer first)");
  int rc;
  if ((rc = vct_ensure(ctx->image, npix * 16, ctx))) return rc;
  // the voxel view blends every fragment in draw order (renderer.cpp:384-388);
  // from a rasterised G-buffer its triangles are known, from an uploaded one
  // only the surface is, which is then blended over the background
  if (ctx->view_voxel_dir < 7 && ctx->g_frame.valid && ctx->g_frame.W == ctx->width &&
      ctx->g_frame.H == ctx->height)
    return vct_launch_voxel_view(ctx);
  return vct_trace_into(ctx, (const float4*)ctx->g_pos.p, (const float4*)ctx->g_nrm.p, (float4*)ctx->image.p,
                        ctx->width, ctx->height, 0, nullptr);
}

extern "C" int vct_trace_count_steps(vct_ctx ctx, uint64_t* steps) {
  if (!ctx) return vct_set_error(VCT_ERR_BAD_HANDLE, "null context");
  if (!steps) return vct_set_error(VCT_ERR_INVALID_ARG, "null out");
  VCT_HIP(hipSetDevice(ctx->device));
  const size_t npix = (size_t)ctx->width * ctx->height;
  if (!ctx->g_pos.p || ctx->g_pos.cap < npix * 16)
    return vct_set_error(VCT_ERR_STATE, "trace needs a G-buffer of the current viewport (run vct_gbuffer first)");
  int rc;
  if ((rc = vct_ensure(ctx->image, npix * 16, ctx))) return rc;
  if ((rc = vct_ensure(ctx->counters, 256, ctx))) return rc;
  unsigned long long* cnt = (unsigned long long*)((char*)ctx->counters.p + 64);
  VCT_HIP(hipMemsetAsync(cnt, 0, 8, ctx->stream));
  if ((rc = vct_trace_into(ctx, (const float4*)ctx->g_pos.p, (const float4*)ctx->g_nrm.p, (float4*)ctx->image.p,
                           ctx->width, ctx->height, 0, cnt)))
    return rc;
  unsigned long long h = 0;
  VCT_HIP(hipMemcpyAsync(&h, cnt, 8, hipMemcpyDeviceToHost, ctx->stream));
  VCT_HIP(hipStreamSynchronize(ctx->stream));
  *steps = h;
  return VCT_OK;
}
