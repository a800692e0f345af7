// t3d_kernels.hip — CDNA4 (gfx950) kernels of the per-frame geometry path.
//
// One frame is a chain of launches over all render pairs ("parts") at once;
// every block works on exactly one part, found by binary search over a
// per-part prefix of block counts, so per-part uniforms are wave-uniform
// (scalar loads) and no block straddles two parts.
//
//   k_vertex    per vertex: shape keys, skinning or MVP transform, snapping,
//               lighting (light constants in scalar registers), vertex
//               colour, fog, screen and texture position
//               (model.go:751-822, camera.go:1610-1644, 1655-1711, 1740-1810)
//   k_cull      per triangle: w clamp, z-range / screen / backface rejects,
//               depth key, per-part survivor count and min/max depth
//               (model.go:828-969)
//   k_groups    dynamic batches: each later part of one flush placed after
//               the survivors of the parts before it (camera.go:2075-2099)
//   k_hist      per tile of a multi-tile part: 512-bin histogram
//   k_scan*     exclusive scan of each part's [bin][tile] histogram matrix
//   k_scatter   stable counting sort: output slot of every survivor
//               (sortingTriangleBucket Sort + ForEach, sortingTriangles.go:38-125)
//   k_assemble  per drawn triangle in slot order: ebiten colour/depth vertices,
//               indices and, with Camera.RenderNormals, the normal vertices,
//               copied from the vertex records with streaming stores
//               (camera.go:1646-1820)
//
// All arithmetic is float32 in the reference's order; the build uses
// -ffp-contract=off and correctly rounded division and square root.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "t3d_internal.h"
#include "t3d_stage.h"
#include "t3d_anim.h"

namespace t3d {

constexpr float kMaxF32 = 3.40282346638528859811704183484516925440e+38f;

__device__ __forceinline__ uint32_t find_part(const uint32_t* __restrict__ prefix, uint32_t n, uint32_t b) {
  // Largest p in [0, n) with prefix[p] <= b (parts with zero blocks are skipped).
  uint32_t lo = 0, hi = n;
  while (hi - lo > 1) {
    uint32_t mid = (lo + hi) >> 1;
    if (prefix[mid] <= b) lo = mid;
    else hi = mid;
  }
  return lo;
}

// The pair of block b: from k_uniforms' map, or, in a frame of few pairs that
// has none, from the prefix itself.
__device__ __forceinline__ uint32_t pair_of(const uint32_t* map, const uint32_t* prefix, uint32_t n, uint32_t b) {
  return map ? map[b] : find_part(prefix, n, b);
}

// Workgroups of a launch are dealt round-robin to the 8 XCDs (workgroup i to
// XCD i % 8), each with its own L2.  With the swizzle on, the workgroups an
// XCD receives take consecutive logical block numbers, so the blocks of one
// render pair (which gather the same vertex records) share an L2.  The map
// is a bijection of [0, n).
constexpr uint32_t kXcds = 8;
__device__ __forceinline__ uint32_t block_index_n(uint32_t swizzle, uint32_t n) {
  const uint32_t i = blockIdx.x;
  if (!swizzle) return i;
  const uint32_t per = n / kXcds, rem = n % kXcds, x = i % kXcds;
  return x * per + min(x, rem) + i / kXcds;
}
// The assembly's map: runs of kAsmRun consecutive blocks go to one XCD and the
// next run to the next, so the eight XCDs also share a pair whose drawn
// triangles fill only the first part of its blocks.  Blocks past the last
// whole group keep their number, so this too is a bijection of [0, n).
constexpr uint32_t kAsmRun = 16;
__device__ __forceinline__ uint32_t block_index_runs(uint32_t swizzle, uint32_t n) {
  const uint32_t i = blockIdx.x, per = kXcds * kAsmRun, g = i / per, r = i % per;
  if (!swizzle || (g + 1) * per > n) return i;
  return g * per + (r % kXcds) * kAsmRun + r / kXcds;
}

// The logical block of this workgroup.  A frame built on the device is
// launched for every candidate pair being drawn; its actual block count is
// FrameCounts word `which` (times `mult`), and a workgroup past it gets
// kNoBlock (block-uniform: the whole workgroup returns).  The swizzle then
// deals the actual blocks, not the launch's, over the XCDs.
constexpr uint32_t kNoBlock = 0xFFFFFFFFu;
template <bool kRuns = false>
__device__ __forceinline__ uint32_t frame_block(const FrameArgs& a, uint32_t which, uint32_t mult) {
  uint32_t n = gridDim.x;
  if (a.counts) {
    n = a.counts[which] * mult;
    if (blockIdx.x >= n) return kNoBlock;
  }
  return kRuns ? block_index_runs(a.xcd_swizzle, n) : block_index_n(a.xcd_swizzle, n);
}
// The same for the launches that never swizzle (scan blocks, pairs).
__device__ __forceinline__ bool past_count(const FrameArgs& a, uint32_t which) {
  return a.counts && blockIdx.x >= a.counts[which];
}

// A record at an address that is the same for the whole wavefront, read
// through the scalar cache into scalar registers (the compiler does so by
// itself only where it can tell that no store of the kernel may reach it).
template <class T>
__device__ __forceinline__ T load_uniform(const T* p) {
  static_assert(sizeof(T) % 4 == 0, "whole words");
  using Word = const __attribute__((address_space(4))) uint32_t;
  Word* w = (Word*)(uintptr_t)p;
  uint32_t v[sizeof(T) / 4];
#pragma unroll
  for (uint32_t i = 0; i < sizeof(T) / 4; i++) v[i] = w[i];
  T r;
  __builtin_memcpy(&r, v, sizeof(T));
  return r;
}

__device__ __forceinline__ float clampf(float v, float lo, float hi) {   // math32.go:38-45
  if (v < lo) return lo;
  else if (v > hi) return hi;
  return v;
}

// Go's int(float32) on amd64: truncation; NaN / out of range give min int64.
__device__ __forceinline__ int64_t go_int(float f) {
  if (!(f >= -9.2233720368547758e18f && f < 9.2233720368547758e18f)) return INT64_MIN;
  return (int64_t)f;
}

__device__ __forceinline__ V3 ld3(const float* __restrict__ p, uint32_t i) {
  return v3(p[3 * (size_t)i + 0], p[3 * (size_t)i + 1], p[3 * (size_t)i + 2]);
}

// ---------------------------------------------------------------------------
// lighting
// ---------------------------------------------------------------------------

// LightVolume cell lookup: convertToXYZIndices + getLightCell (light.go:717-724, 1267-1272);
// the cell's index, or -1 where there is none.
__device__ __forceinline__ int64_t volume_cell_index(const LightGPU& l, V3 p) {
  int64_t x = go_int(roundf(fdiv(p.x - l.offset[0] - l.vmin[0] - fdiv(l.cell[0], 2.0f), l.cell[0])));
  int64_t y = go_int(roundf(fdiv(p.y - l.offset[1] - l.vmin[1] - fdiv(l.cell[1], 2.0f), l.cell[1])));
  int64_t z = go_int(roundf(fdiv(p.z - l.offset[2] - l.vmin[2] - fdiv(l.cell[2], 2.0f), l.cell[2])));
  if (x < 0 || y < 0 || z < 0 || x >= l.cx || y >= l.cy || z >= l.cz) return -1;
  int64_t i = x + (y * l.cx) + (z * l.cx * l.cy);
  if (!l.cells || i >= (int64_t)l.ncells) return -1;
  return i;
}

__device__ __forceinline__ const float* volume_cell(const LightGPU& l, V3 p) {
  const int64_t i = volume_cell_index(l, p);
  return i < 0 ? nullptr : l.cells + 4 * i;
}

// A field of a record: through scalar registers where the whole wavefront
// reads the same record, else by each lane.  Each is read where it is used:
// a pair's record, its camera and a light together are more than the 102
// scalar registers, and held at once a third of the pass's instructions only
// moved them out of the way and back.
template <bool kUniform, class T>
__device__ __forceinline__ T field(const T& r) {
  if constexpr (kUniform) return load_uniform(&r);
  else return r;
}

// VertexLight of an ambient, point or directional light on one vertex
// (light.go:116-120, 191-258, 332-360), accumulating into rgb in the
// reference's order.  kUniform: l and pl are the same for the whole wavefront.
template <bool kUniform>
__device__ __forceinline__ void light_direct(const LightGPU& l, const PartLight& pl, const PartGPU& P, uint32_t flags,
                                             V3 vp, V3 vn, float& r, float& g, float& b) {
  const uint32_t lmode = (flags >> PF_LMODE_SHIFT) & 3u;
  const int32_t type = field<kUniform>(l.type);
  float df;
  if (type == T3D_LIGHT_AMBIENT) {
    r += field<kUniform>(l.amb[0]);
    g += field<kUniform>(l.amb[1]);
    b += field<kUniform>(l.amb[2]);
    return;
  } else if (type == T3D_LIGHT_POINT) {
    const float range_sq = field<kUniform>(l.range_sq);
    V3 wp = v3(field<kUniform>(pl.v[0]), field<kUniform>(pl.v[1]), field<kUniform>(pl.v[2]));
    float distance = dist_sq(wp, vp);
    if (field<kUniform>(l.range) > 0) {
      if (distance > range_sq) return;
    } else {
      if (fdiv(1.0f, distance) * field<kUniform>(l.energy) < 0.001f) return;
    }
    V3 lv = unit(sub(wp, vp));
    V3 n = lmode == T3D_LIGHTING_FIXED_NORMALS ? lv : vn;
    float diffuse = dot(n, lv);
    if (lmode == T3D_LIGHTING_DOUBLE_SIDED) diffuse = fabsf(diffuse);
    if (!(diffuse > 0)) return;
    df = diffuse * fdiv(1.0f, 1.0f + (0.1f * distance)) * 2.0f;
    if (range_sq > 0) {
      float dc = clampf(fdiv(range_sq - distance, distance), 0.0f, 1.0f);
      df *= dc;
    }
  } else if (type == T3D_LIGHT_DIRECTIONAL) {
    V3 fwd = v3(field<kUniform>(l.fwd[0]), field<kUniform>(l.fwd[1]), field<kUniform>(l.fwd[2]));
    V3 n;
    if (lmode == T3D_LIGHTING_FIXED_NORMALS) n = fwd;
    else if (flags & PF_SKINNED) n = vn;
    else n = mult_vec(load_uniform(&P.rd), vn);
    df = dot(n, fwd);
    if (lmode == T3D_LIGHTING_DOUBLE_SIDED) df = fabsf(df);
    if (df <= 0) return;
  } else {
    return;
  }
  const float energy = field<kUniform>(l.energy);
  r += field<kUniform>(l.color[0]) * df * energy;
  g += field<kUniform>(l.color[1]) * df * energy;
  b += field<kUniform>(l.color[2]) * df * energy;
}

// A LightVolume of a pair's list on one vertex (light.go:583-663): its cell
// first runs the lights its useLights names (light.go:650-653; entries
// ls/pls[nest_off + j] of the same list), then adds its own colour.
__device__ __forceinline__ void light_volume(const LightGPU& lr, const PartLight& pl, const LightGPU* ls,
                                             const PartLight* pls, const PartGPU& P, uint32_t flags, V3 vp, V3 vn,
                                             float& r, float& g, float& b) {
  const uint32_t mode = (flags >> PF_LVMODE_SHIFT) & 3u;
  if (mode == T3D_LV_OFF) return;                                  // LightVolume.Light, light.go:671-673
  float c0 = 0, c1 = 0, c2 = 0;
  if (mode == T3D_LV_PER_OBJECT) {
    if (load_uniform(&pl.cell_found)) {
      c0 = load_uniform(&pl.v[0]);
      c1 = load_uniform(&pl.v[1]);
      c2 = load_uniform(&pl.v[2]);
    }
  } else {
    const LightGPU l = load_uniform(&lr);
    V3 halfc = v3(fdiv(l.cell[0], 2.0f), fdiv(l.cell[1], 2.0f), fdiv(l.cell[2], 2.0f));
    V3 bias = v3(l.bias[0], l.bias[1], l.bias[2]);
    V3 vpos = v3(0, 0, 0), vpn = v3(0, 0, 0);
    if (flags & PF_SKINNED) {
      if (mode == T3D_LV_PER_VERTEX_WITH_NORMAL) vpn = add(add(vpos, hmul(vn, halfc)), bias);
      else vpos = add(vp, bias);
    } else {
      const M4 model = load_uniform(&P.model);
      if (mode == T3D_LV_PER_VERTEX_WITH_NORMAL) vpn = add(mult_vec(model, add(vp, hmul(vn, halfc))), bias);
      else vpos = add(mult_vec(model, vp), bias);
    }
    if (!(vpos.x >= l.vmin[0] && vpos.y >= l.vmin[1] && vpos.z >= l.vmin[2] && vpos.x <= l.vmax[0] &&
          vpos.y <= l.vmax[1] && vpos.z <= l.vmax[2]))
      return;                                                        // Dimensions.Contains, mesh.go:80-82
    const int64_t ci = volume_cell_index(l, mode == T3D_LV_PER_VERTEX_WITH_NORMAL ? vpn : vpos);
    if (ci >= 0) {
      const float* cell = l.cells + 4 * ci;
      c0 = cell[0];
      c1 = cell[1];
      c2 = cell[2];
      if (l.cell_lights) {
        const uint32_t j1 = l.cell_lights[ci + 1];
        const uint32_t* ix = l.cell_lights + l.ncells + 1;
        for (uint32_t j = l.cell_lights[ci]; j < j1; j++) {
          const uint32_t li = l.nest_off + ix[j];
          light_direct<false>(ls[li], pls[li], P, flags, vp, vn, r, g, b);
        }
      }
    }
  }
  const float energy = load_uniform(&lr.energy);
  r += load_uniform(&lr.color[0]) * c0 * energy;
  g += load_uniform(&lr.color[1]) * c1 * energy;
  b += load_uniform(&lr.color[2]) * c2 * energy;
}

// ---------------------------------------------------------------------------
// k_vertex
// ---------------------------------------------------------------------------

// What the later passes read of a vertex, computed once here instead of once
// per triangle corner (about six corners share a vertex): the first two
// float4 of its ebiten colour vertex (a: DstX, DstY, SrcX, SrcY, b: colour),
// and q: the screen position the cull tests, the depth list's value and
// Custom0.  zin: its Z is inside the camera's range.
struct VertexRecord {
  float4 a, b, q;
  bool zin;
};

// Screen position, texture position and depth of a vertex from its clip
// position (model.go:869-887, camera.go:1655-1711, 1765-1784).  Where the
// cull's and the assembly's clamps of W leave it alone (W > 0, perspective)
// their quotients are one: y / -w is -(y / w) in every rounding.
__device__ __forceinline__ void place_vertex(const FrameConst& fc, V4 clip, float zd, float2 uv, float src_w,
                                             float src_h, VertexRecord& r) {
  const bool persp = load_uniform(&fc.perspective) != 0;
  const float wc = clip.w < 0 ? 0.000001f : clip.w;
  const float nx = fdiv(clip.x, wc), ny = fdiv(clip.y, wc);
  float w = clip.w;                                               // camera.go:1655-1667
  if (!persp) w = 1.0f;
  if (w < 0) w = 0.001f;
  float qx = nx, qy = -ny;
  if (!(persp && clip.w > 0)) {
    qx = fdiv(clip.x, w);
    qy = fdiv(clip.y, -w);
  }
  float uvU, uvV, c0 = 0.0f;
  if (load_uniform(&fc.pc_tex)) {                                                // camera.go:1688-1711
    uvU = fdiv(uv.x, w) * src_w;
    uvV = fdiv(1.0f - uv.y, w) * src_h;
    c0 = fdiv(1.0f, w);
  } else {
    uvU = uv.x * src_w;
    uvV = (1.0f - uv.y) * src_h;
  }
  float depth = 0.0f;
  if (load_uniform(&fc.render_depth)) {                                          // camera.go:1765-1784
    depth = fdiv(zd + load_uniform(&fc.dmp), load_uniform(&fc.spread));
    if (depth < 0) depth = 0;
    else if (depth > 1) depth = 1;
  }
  r.a = make_float4(qx * load_uniform(&fc.cam_w) + load_uniform(&fc.half_w), qy * load_uniform(&fc.cam_h) + load_uniform(&fc.half_h), uvU, uvV);
  r.q = make_float4(nx, ny, depth, c0);
  r.zin = clip.z + 1.0f >= load_uniform(&fc.near_) && clip.z < load_uniform(&fc.far_);          // model.go:883-886
}

// bone palette rows in LDS, five float4 per bone (four rows and one of
// padding): lanes blending different bones then start on different LDS
// banks instead of two bank groups (a 64-byte stride covers 16 of 32 banks)
constexpr uint32_t kBoneRows = 5;
__device__ __forceinline__ void stage_bones(const PartGPU& P, float4* rows) {
  const float4* src = reinterpret_cast<const float4*>(load_uniform(&P.palette));
  const uint32_t n = 4u * load_uniform(&P.bone_count);
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) rows[(i / 4) * kBoneRows + i % 4] = src[i];
}

// One vertex of a pair through shape keys, skinning or MVP transform,
// snapping, colour, lighting and fog.  rows: the pair's bone rows in LDS, or
// null (then read from memory); umvp: the unaltered MVP (PF_UNBB pairs).
__device__ __forceinline__ VertexRecord shade_vertex(const FrameArgs& a, const FrameConst& fc, const PartGPU& P,
                                                     uint32_t flags, uint32_t v, const float4* rows, const M4& umvp,
                                                     V3& vp) {
  const bool skinned = (flags & PF_SKINNED) != 0;
  const uint32_t nl = (flags & PF_LIGHTING) ? load_uniform(&P.light_count) : 0u;
  // VertexPositionWithShapeKeys / VertexNormalWithShapeKeys (mesh.go:796-822)
  V3 pos = ld3(load_uniform(&P.pos), v);
  V3 nrm = ld3(load_uniform(&P.nrm), v);
  if (flags & PF_SHAPE_KEYS) {
    for (uint32_t k = 0; k < load_uniform(&P.shape_keys); k++) {
      const float w = load_uniform(&P.sk_w)[k];
      const size_t o = ((size_t)k * load_uniform(&P.mesh_vcount) + v) * 3;
      pos.x += load_uniform(&P.sk_pos)[o + 0] * w;
      pos.y += load_uniform(&P.sk_pos)[o + 1] * w;
      pos.z += load_uniform(&P.sk_pos)[o + 2] * w;
    }
    for (uint32_t k = 0; k < load_uniform(&P.shape_keys); k++) {
      const float w = load_uniform(&P.sk_w)[k];
      const size_t o = ((size_t)k * load_uniform(&P.mesh_vcount) + v) * 3;
      nrm.x += load_uniform(&P.sk_nrm)[o + 0] * w;
      nrm.y += load_uniform(&P.sk_nrm)[o + 1] * w;
      nrm.z += load_uniform(&P.sk_nrm)[o + 2] * w;
    }
  }
  V3 vn;
  V4 clip;
  float zu = 0.0f;                                                // Z of DepthModeUnbillboarded
  if (skinned) {
    // Model.skinVertex (model.go:559-596)
    const ushort4 bi = reinterpret_cast<const ushort4*>(load_uniform(&P.bones))[v];
    const float4 bw = reinterpret_cast<const float4*>(load_uniform(&P.weights))[v];
    const uint16_t bidx[4] = {bi.x, bi.y, bi.z, bi.w};
    const float bwt[4] = {bw.x, bw.y, bw.z, bw.w};
    M4 S = zero4();
    for (int k = 0; k < 4; k++) {
      const float w = bwt[k];
      if (w == 0) continue;
      float4 B[4];
      for (int r = 0; r < 4; r++)
        B[r] = rows ? rows[bidx[k] * kBoneRows + r]
                         : reinterpret_cast<const float4*>(load_uniform(&P.palette))[(size_t)bidx[k] * 4 + r];
      if (w == 1) {
        for (int r = 0; r < 4; r++) {
          S.m[r][0] = B[r].x;
          S.m[r][1] = B[r].y;
          S.m[r][2] = B[r].z;
          S.m[r][3] = B[r].w;
        }
        break;
      }
      for (int r = 0; r < 4; r++) {
        S.m[r][0] += B[r].x * w;
        S.m[r][1] += B[r].y * w;
        S.m[r][2] += B[r].z * w;
        S.m[r][3] += B[r].w * w;
      }
    }
    vp = mult_vec(S, pos);
    S.m[3][0] = 0;
    S.m[3][1] = 0;
    S.m[3][2] = 0;
    S.m[3][3] = 1;
    vn = mult_vec(S, nrm);
    clip = mult_vec_w(load_uniform(&fc.vp), vp);                                 // model.go:772-775
  } else {
    vp = pos;
    vn = nrm;
    clip = mult_vec_w(load_uniform(&P.mvp), pos);                                // model.go:795-798
    if (flags & PF_UNBB) zu = mult_vec_w(umvp, pos).z;          // model.go:800-803, not snapped
  }
  const float snap = load_uniform(&fc.snap);
  if (snap > 0) {                                                 // model.go:807-812
    clip.x = fdiv(roundf(clip.x * snap), snap);
    clip.y = fdiv(roundf(clip.y * snap), snap);
    clip.z = fdiv(roundf(clip.z * snap), snap);
  }
  // vertex colour (camera.go:1750-1768)
  float cr, cg, cb, ca;
  if (flags & PF_HAS_COLOR) {
    const float4 vc = reinterpret_cast<const float4*>(load_uniform(&P.col))[v];
    cr = vc.x * load_uniform(&P.mp[0]);
    cg = vc.y * load_uniform(&P.mp[1]);
    cb = vc.z * load_uniform(&P.mp[2]);
    ca = vc.w * load_uniform(&P.mp[3]);
  } else {
    cr = load_uniform(&P.mp[0]);
    cg = load_uniform(&P.mp[1]);
    cb = load_uniform(&P.mp[2]);
    ca = load_uniform(&P.mp[3]);
  }
  if (flags & PF_LIGHTING) {
    // vertexLights reset to (0,0,0,1) then every light in order (camera.go:1613-1641)
    float lr = 0, lg = 0, lb = 0;
    const LightGPU* ls = a.lights + load_uniform(&P.light0);
    const PartLight* pls = a.plights + load_uniform(&P.light_base);
    for (uint32_t k = 0; k < nl; k++) {
      if (!load_uniform(&pls[k].enabled)) continue;
      if (load_uniform(&ls[k].type) == T3D_LIGHT_VOLUME) light_volume(ls[k], pls[k], ls, pls, P, flags, vp, vn, lr, lg, lb);
      else light_direct<true>(ls[k], pls[k], P, flags, vp, vn, lr, lg, lb);
    }
    cr *= lr;
    cg *= lg;
    cb *= lb;
  }
  if (load_uniform(&fc.fog_active)) {                                            // camera.go:1786-1810
    float depth = fdiv(clip.z + load_uniform(&fc.dmp), load_uniform(&fc.spread));
    if (depth < 0) depth = 0;
    else if (depth > 1) depth = 1;
    depth = load_uniform(&fc.fog_range[0]) + ((load_uniform(&fc.fog_range[1]) - load_uniform(&fc.fog_range[0])) * 1.0f - depth);
    if (load_uniform(&fc.fog_mode) == T3D_FOG_ADD) {
      cr += load_uniform(&fc.fog_color[0]) * depth;
      cg += load_uniform(&fc.fog_color[1]) * depth;
      cb += load_uniform(&fc.fog_color[2]) * depth;
    } else if (load_uniform(&fc.fog_mode) == T3D_FOG_SUB) {
      cr *= load_uniform(&fc.fog_color[0]) * depth;
      cg *= load_uniform(&fc.fog_color[1]) * depth;
      cb *= load_uniform(&fc.fog_color[2]) * depth;
    }
  }
  const float2 uv = (flags & PF_HAS_UV) ? reinterpret_cast<const float2*>(load_uniform(&P.uv))[v] : make_float2(0.0f, 0.0f);
  VertexRecord r;
  place_vertex(fc, clip, (flags & PF_UNBB) ? zu : clip.z, uv, load_uniform(&P.src_w), load_uniform(&P.src_h), r);
  r.b = make_float4(cr, cg, cb, ca);
  return r;
}

// Its vertices move about 105 bytes each (3.9 M of them: 410 MB in 87 us, 4.7
// TB/s, where a copy reaches 5.1).  Light constants staged in LDS instead of
// scalar registers held the occupancy at six wavefronts a SIMD and cost an
// LDS read per light and field: 112 us, in a run that had 94 without; scalar,
// but with 65 registers (seven wavefronts), 104 us.
// kOut: which of its outputs are written (a frame with lean records runs it
// twice, see record_scratch).
template <uint32_t kOut>
__global__ __launch_bounds__(256, 8) void k_vertex(FrameArgs a, uint32_t blk0) {
  const uint32_t lb = frame_block(a, FC_VCHUNKS, 1);
  if (lb == kNoBlock) return;
  const uint32_t b = blk0 + lb;
  const uint32_t p = pair_of(a.vchunk_part, a.vchunk_prefix, a.nparts, b);
  const PartGPU& P = a.parts[p];
  const uint32_t flags = load_uniform(&P.flags);

  __shared__ float4 s_bone_rows[kMaxLdsBones * kBoneRows];
  const bool skinned = (flags & PF_SKINNED) != 0;
  const bool lds_bones = skinned && load_uniform(&P.bone_count) <= kMaxLdsBones;
  if (lds_bones) stage_bones(P, s_bone_rows);
  __shared__ M4 s_umvp;                  // unaltered MVP of DepthModeUnbillboarded (model.go:697-703)
  if ((flags & PF_UNBB) && threadIdx.x == 0) s_umvp = mult(load_uniform(&P.model), load_uniform(&a.fc[load_uniform(&P.cam)].vp));
  __syncthreads();

  const FrameConst& fc = a.fc[load_uniform(&P.cam)];
  const uint32_t vbase = load_uniform(&P.vbase), vmin = load_uniform(&P.vmin);
  const bool normals = load_uniform(&fc.render_normals) != 0;
  const uint32_t first = (b - a.vchunk_prefix[p]) * a.vchunk;
  const uint32_t last = min(first + a.vchunk, load_uniform(&P.vcount));
  bool out_of_range = false;
  for (uint32_t i = first + threadIdx.x; i < last; i += blockDim.x) {
    const uint32_t o = vbase + i;
    V3 vp;
    const VertexRecord r = shade_vertex(a, fc, P, flags, vmin + i, lds_bones ? s_bone_rows : nullptr, s_umvp, vp);
    if ((kOut & VERTEX_FOR_CULL) && normals) {   // model.go:814-818: the rotation applied to the position; colour camera.go:1718-1720
      const V3 tn = mult_vec(load_uniform(&P.nrot), vp);
      a.vnrm[o] = make_float4(tn.x * 0.5f + 0.5f, tn.y * 0.5f + 0.5f, tn.z * 0.5f + 0.5f, 0.0f);
    }
    if (kOut & VERTEX_FOR_LISTS) {
      a.vab[2 * (size_t)o + 0] = r.a;
      a.vab[2 * (size_t)o + 1] = r.b;
    }
    if (kOut & VERTEX_FOR_CULL) {
      a.vq[o] = r.q;
      a.vz[o] = r.zin ? 1 : 0;
      out_of_range |= !r.zin;
      if (skinned) a.vpos[o] = make_float4(vp.x, vp.y, vp.z, 0.0f);
    }
  }
  // a pair with no vertex out of the Z range needs no look at vz in the cull
  if (__ballot(out_of_range) && threadIdx.x % 64 == 0) a.stats[4 * p + 3] = 1u;   // every writer stores the same word
}

// ---------------------------------------------------------------------------
// k_palettes, k_uniforms
// ---------------------------------------------------------------------------

// k_palettes: the bone palettes of armatures given as poses, one block per
// armature, computed as Node.Transform() does down the armature
// (node.go:572-608):
//   1. Scale·rotation·Translate of every bone, spread over the block;
//   2. Transform() = local·parent's Transform() (the armature parent's for a
//      root bone), level by level: each round, every bone whose parent is
//      done takes its parent's product, so the rounds number the armature's
//      depth, not its bones;
//   3. boneInfluence = inverseBindMatrix·Transform() (node.go:592-594).
// Every product is Matrix4.Mult in its own order, so the palette equals the
// host's bit for bit.  Parents and round states live in LDS; the bone
// transforms too up to kLdsPoseBones, in device memory past that.
constexpr uint32_t kLdsPoseBones = 256;     // 16 KB of LDS
constexpr uint32_t kLevelPoseBones = 4096;  // armatures walked level by level up to this size
constexpr uint32_t kPoseThreads = 64;

// Local transform of bone b: Scale·rotation·Translate of its pose, after the
// armature's animation (if any) has set the channels it samples.
__device__ __forceinline__ M4 bone_local(const PaletteJob& J, uint32_t b) {
  const t3d_bone_pose& B = J.poses[b];
  float pos[3] = {B.position[0], B.position[1], B.position[2]};
  float scl[3] = {B.scale[0], B.scale[1], B.scale[2]};
  M4 rot = B.rotation;
  if (b < J.nchannels) animate_bone(J.channels[b], J.time, pos, scl, rot);
  return mult(mult(scale4(scl[0], scl[1], scl[2]), rot), translate(pos[0], pos[1], pos[2]));
}

template <typename WPtr>
__device__ __forceinline__ void pose_armature(const PaletteJob& J, WPtr W, int16_t* par, uint8_t* state) {
  const uint32_t n = J.n;
  for (uint32_t b = threadIdx.x; b < n; b += kPoseThreads) {
    W[b] = bone_local(J, b);
    par[b] = (int16_t)J.poses[b].parent;            // -1 <= parent < b, checked by the host
    state[b] = 0;                                    // 0 waiting, 1 ready this round, 2 done
  }
  __syncthreads();
  // Each round readies at least the lowest waiting bone (its parent is earlier, so done): at most n rounds.
  // A parent index outside [-1, b) (refused by the host) never readies, and the bound still ends the loop.
  for (uint32_t round = 0; round < n; round++) {
    bool waiting = false;
    for (uint32_t b = threadIdx.x; b < n; b += kPoseThreads)
      if (state[b] == 0) {
        const int32_t p = par[b];
        if (p < 0 || ((uint32_t)p < b && state[p] == 2)) state[b] = 1;   // a parent going 0 -> 1 now reads as not done
        else waiting = true;
      }
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < n; b += kPoseThreads)
      if (state[b] == 1) {
        const int32_t p = par[b];
        if (p >= 0) W[b] = mult(W[b], W[p]);         // W[p] was finished in an earlier round
        else if (J.root) W[b] = mult(W[b], *J.root);
        state[b] = 2;
      }
    if (!__syncthreads_or(waiting)) break;
  }
  for (uint32_t b = threadIdx.x; b < n; b += kPoseThreads) {
    const M4 r = mult(J.poses[b].inverse_bind, W[b]);
    float4* out = reinterpret_cast<float4*>(J.palette + 16ull * b);
    for (int i = 0; i < 4; i++) out[i] = make_float4(r.m[i][0], r.m[i][1], r.m[i][2], r.m[i][3]);
  }
}

// Armatures past kLevelPoseBones: the parent chain walked in bone order by
// one thread (a parent is always an earlier bone).
__device__ void pose_armature_serial(const PaletteJob& J, M4* W) {
  for (uint32_t b = threadIdx.x; b < J.n; b += kPoseThreads) W[b] = bone_local(J, b);
  __syncthreads();
  if (threadIdx.x == 0)
    for (uint32_t b = 0; b < J.n; b++) {
      const int32_t p = J.poses[b].parent;
      if (p >= 0 && (uint32_t)p < b) W[b] = mult(W[b], W[p]);
      else if (J.root) W[b] = mult(W[b], *J.root);
    }
  __syncthreads();
  for (uint32_t b = threadIdx.x; b < J.n; b += kPoseThreads) {
    const M4 r = mult(J.poses[b].inverse_bind, W[b]);
    float4* out = reinterpret_cast<float4*>(J.palette + 16ull * b);
    for (int i = 0; i < 4; i++) out[i] = make_float4(r.m[i][0], r.m[i][1], r.m[i][2], r.m[i][3]);
  }
}

__global__ __launch_bounds__(kPoseThreads) void k_palettes(FrameArgs a) {
  const PaletteJob J = a.pal_jobs[blockIdx.x];
  __shared__ M4 s_world[kLdsPoseBones];
  __shared__ int16_t s_par[kLevelPoseBones];
  __shared__ uint8_t s_state[kLevelPoseBones];
  M4* gw = a.pose_world + J.world_off;
  if (J.n <= kLdsPoseBones) pose_armature(J, s_world, s_par, s_state);
  else if (J.n <= kLevelPoseBones) pose_armature(J, gw, s_par, s_state);
  else pose_armature_serial(J, gw);
}

// Per-pair uniforms: MVP (model.go:695), invertedCamPos (model.go:629-630),
// the directional working rotation (light.go:326-330) and, per light of the
// pair, beginModel's working position (light.go:175-189), the per-model
// point-light skip (camera.go:1592, 1625-1629) and the per-object LightVolume
// cell (light.go:610-628).  The same float32 functions the host would run, so
// the values are the ones the reference computes on the CPU.  One block per
// render pair: lane k handles the pair's lights k, k + 64, ..., lane 0 also the pair's own uniforms and the reset of its depth range
// and survivor count, so the latency is one light's, not the sum over lights;
// all wavefronts first write the pair's entries of the block->pair maps (a
// 1024 x 1024 grid has over 5,000, which one wavefront took 11 us to store);
// the first then works alone.
constexpr uint32_t kUniformThreads = 256;
__global__ __launch_bounds__(kUniformThreads) void k_uniforms(FrameArgs a, uint32_t part0, uint32_t nparts) {
  if (past_count(a, FC_PAIRS)) return;
  PartGPU& P = const_cast<PartGPU*>(a.parts)[part0 + blockIdx.x];
  if (a.counts) {   // a device-built frame: the pair's record is built here from the model, mesh and material
    __shared__ PartGPU s_part;
    if (threadIdx.x == 0) build_pair(a, part0 + blockIdx.x, s_part);
    __syncthreads();
    static_assert(sizeof(PartGPU) % 16 == 0, "whole float4 rows");
    const float4* src = reinterpret_cast<const float4*>(&s_part);
    float4* dst = reinterpret_cast<float4*>(&P);
    for (uint32_t i = threadIdx.x; i < sizeof(PartGPU) / 16; i += kUniformThreads) dst[i] = src[i];
    __syncthreads();
  }
  const uint32_t k = threadIdx.x;
  {  // block -> pair maps of the later kernels: one load where a search over the prefixes took nine
    const uint32_t p = part0 + blockIdx.x;
    for (uint32_t i = a.tile_prefix[p] + k; i < a.tile_prefix[p + 1]; i += kUniformThreads) a.tile_part[i] = p;
    for (uint32_t i = a.vchunk_prefix[p] + k; i < a.vchunk_prefix[p + 1]; i += kUniformThreads) a.vchunk_part[i] = p;
  }
  if (k >= 64) return;
  const uint32_t flags = P.flags;
  const uint32_t nl = (flags & PF_LIGHTING) ? P.light_count : 0u;
  if (k > 0 && k >= nl) return;
  const FrameConst& fc = a.fc[P.cam];
  const ModelInverse inv = model_inverse(P.model);
  for (uint32_t kk = k; kk < nl; kk += 64) {
    const LightGPU& L = a.lights[P.light0 + kk];
    PartLight pl = pair_light(P, inv, L, P.light0 + kk);
    if (L.type == T3D_LIGHT_VOLUME && ((flags >> PF_LVMODE_SHIFT) & 3u) == T3D_LV_PER_OBJECT) {
      const float* cell = volume_cell(L, row3(P.model));
      if (cell) {
        pl.cell_found = 1;
        pl.v[0] = cell[0];
        pl.v[1] = cell[1];
        pl.v[2] = cell[2];
      }
    }
    a.plights[P.light_base + kk] = pl;
  }
  if (k == 0) {
    uint32_t* st = a.stats + 4 * (part0 + blockIdx.x);
    st[0] = __float_as_uint(kMaxF32);  // minDepth = MaxFloat32 (model.go:702)
    st[1] = 0u;                        // max over non-negative keys
    st[2] = 0u;                        // survivors
    st[3] = 0u;
    complete_pair(P, inv, fc);
  }
}

__device__ __forceinline__ float wave_min(float v) {
  for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o));
  return v;
}
__device__ __forceinline__ float wave_max(float v) {
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
  return v;
}
__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// ---------------------------------------------------------------------------
// k_cull
// ---------------------------------------------------------------------------

// The vertex records of triangle t's corners.
__device__ __forceinline__ void corner_records(const PartGPU& P, uint32_t t, uint32_t (&ov)[3]) {
  const uint32_t d = P.vbase - P.vmin;
  if (P.idx16) {                                  // uniform: the pair's mesh index width
    const uint16_t* ix = P.idx16 + 3 * (size_t)t;
    for (int k = 0; k < 3; k++) ov[k] = d + ix[k];
  } else {
    const uint32_t* ix = P.idx + 3 * (size_t)t;
    for (int k = 0; k < 3; k++) ov[k] = d + ix[k];
  }
}

// Whether a triangle is drawn, from its corners' screen positions and whether
// any is inside the Z range (model.go:855-925).
__device__ __forceinline__ bool visible(const float4 (&c)[3], bool zin, bool backface) {
  if (!zin) return false;
  if ((c[0].x < -0.5f && c[1].x < -0.5f && c[2].x < -0.5f) || (c[0].x > 0.5f && c[1].x > 0.5f && c[2].x > 0.5f) ||
      (c[0].y < -0.5f && c[1].y < -0.5f && c[2].y < -0.5f) || (c[0].y > 0.5f && c[1].y > 0.5f && c[2].y > 0.5f))
    return false;                                                       // model.go:890-898
  if (backface) {                                                       // model.go:902-925
    const float n0x = c[0].x - c[1].x;
    const float n0y = c[0].y - c[1].y;
    const float n1x = c[1].x - c[2].x;
    const float n1y = c[1].y - c[2].y;
    const float nor = (n0x * n1y) - (n1x * n0y);
    if (nor < 0) return false;
  }
  return true;
}

// Squared distance of a triangle's centre from the camera: a skinned
// triangle's three positions, or a static one's stored Triangle.Center
// (mesh.go:1980-1982) in q[0].
__device__ __forceinline__ float depth_key(bool skinned, V3 cam, V3 icp, const V3 (&q)[3]) {
  V3 from = icp, c = q[0];
  if (skinned) {                                                        // model.go:860-864, 941-960
    from = cam;
    V3 s = v3(0, 0, 0);
    for (int k = 0; k < 3; k++) s = add(s, q[k]);
    c = v3(fdiv(s.x, 3.0f), fdiv(s.y, 3.0f), fdiv(s.z, 3.0f));
  }
  const float dx = from.x - c.x, dy = from.y - c.y, dz = from.z - c.z;
  return dx * dx + dy * dy + dz * dz;
}

// kThreads: 256, 512 or 1024 threads per tile block (tunable).
template <uint32_t kThreads>
__global__ __launch_bounds__(kThreads) void k_cull(FrameArgs a, uint32_t blk0) {
  constexpr uint32_t kCullWaves = kThreads / 64;
  const uint32_t lb = frame_block(a, FC_TILES, 1);
  if (lb == kNoBlock) return;
  const uint32_t b = blk0 + lb;
  const uint32_t p = pair_of(a.tile_part, a.tile_prefix, a.nparts, b);
  const PartGPU P = a.parts[p];        // by value: read once, before any store
  const uint32_t flags = P.flags;
  const FrameConst fc = a.fc[P.cam];
  const uint32_t t0 = (b - a.tile_prefix[p]) * a.tile;
  const uint32_t t1 = min(t0 + a.tile, P.tcount);
  const bool skinned = (flags & PF_SKINNED) != 0;
  const bool backface = (flags & PF_BACKFACE) != 0;
  const bool all = (flags & PF_ALL) != 0;     // processOnlyVisible false: no test removes a triangle
  const V3 camPos = v3(fc.campos[0], fc.campos[1], fc.campos[2]);
  const V3 icp = v3(P.icp[0], P.icp[1], P.icp[2]);

  // Survivors are compacted in triangle order to the front of the tile's
  // range of key[] and tri_loc[]; tile_count[b] says how many there are.
  const bool look_z = !all && a.stats[4 * p + 3] != 0;   // some vertex of the pair is out of the Z range
  float mn = kMaxF32, mx = 0.0f;
  const uint32_t wv = threadIdx.x / warpSize, ln = threadIdx.x % warpSize;
  const uint64_t lt_mask = (ln == 0) ? 0ull : (~0ull >> (64 - ln));
  __shared__ uint32_t s_wc[kCullWaves];
  uint32_t run = 0;                                 // survivors so far, block-uniform
  for (uint32_t base = t0; base < t1; base += blockDim.x) {
    const uint32_t t = base + threadIdx.x;
    bool keep = false;
    float depth = -1.0f;
    if (t < t1) {
      uint32_t ov[3];
      corner_records(P, t, ov);
      // every gather of the triangle first, so their latencies overlap:
      // screen positions, and what its depth key needs (a static triangle's
      // stored Triangle.Center, or the three skinned positions)
      float4 cc[3];
      V3 q[3];
      bool zin = true;
      for (int k = 0; k < 3; k++) cc[k] = a.vq[ov[k]];
      if (look_z) zin = (a.vz[ov[0]] | a.vz[ov[1]] | a.vz[ov[2]]) != 0;
      if (skinned) {
        for (int k = 0; k < 3; k++) {
          const float4 s = a.vpos[ov[k]];
          q[k] = v3(s.x, s.y, s.z);
        }
      } else {
        const float* cp = P.ctr + 3 * (size_t)t;
        q[0] = v3(cp[0], cp[1], cp[2]);
      }
      keep = all || visible(cc, zin, backface);
      if (keep) {                                                       // model.go:941-960
        depth = depth_key(skinned, camPos, icp, q);
        if (!all && (isnan(depth) || isinf(depth))) {
          keep = false;
          depth = -1.0f;
        }
      }
    }
    const uint64_t m = __ballot(keep);
    if (ln == 0) s_wc[wv] = (uint32_t)__popcll(m);
    __syncthreads();
    uint32_t wbase = 0, tot = 0;
    for (uint32_t w = 0; w < kCullWaves; w++) {
      if (w < wv) wbase += s_wc[w];
      tot += s_wc[w];
    }
    if (keep) {
      const uint32_t pos = P.tbase + t0 + run + wbase + (uint32_t)__popcll(m & lt_mask);
      a.key[pos] = depth;
      a.tri_loc[pos] = (uint16_t)(t - t0);
      mn = fminf(mn, depth);
      mx = fmaxf(mx, depth);
    }
    run += tot;
    __syncthreads();                              // s_wc is rewritten next round
  }
  // block reduction, one atomic of each kind per block
  __shared__ float s_mn[kCullWaves], s_mx[kCullWaves];
  mn = wave_min(mn);
  mx = wave_max(mx);
  if (ln == 0) {
    s_mn[wv] = mn;
    s_mx[wv] = mx;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (uint32_t w = 1; w < kCullWaves; w++) {
      mn = fminf(mn, s_mn[w]);
      mx = fmaxf(mx, s_mx[w]);
    }
    a.tile_count[b] = run;
    if (run) {
      atomicMin(&a.stats[4 * p + 0], __float_as_uint(mn));   // keys are >= +0: uint order = float order
      atomicMax(&a.stats[4 * p + 1], __float_as_uint(mx));
      atomicAdd(&a.stats[4 * p + 2], run);
    }
  }
}

// ---------------------------------------------------------------------------
// sort: bins, histograms, scan, stable scatter
// ---------------------------------------------------------------------------

// Bin of a survivor in visit order: sortingTriangleBucket.Sort's
// int(clamp(((d - min) / (max - min)) * 512, 0, 511)) (sortingTriangles.go:38-64),
// reversed for BackToFront so ascending keys follow ForEach (sortingTriangles.go:93-125).
__device__ __forceinline__ uint32_t visit_bin(float d, float mn, float rd, uint32_t sort_mode) {
  int64_t bin = 0;
  if (sort_mode != T3D_SORT_NONE) {
    const float x = fdiv(d - mn, rd) * (float)kBins;
    bin = go_int(clampf(x, 0.0f, (float)(kBins - 1)));
  }
  return sort_mode == T3D_SORT_BACK_TO_FRONT ? (kBins - 1) - (uint32_t)bin : (uint32_t)bin;
}

// Lanes of `valid` (a ballot) whose 9-bit bin equals this lane's: one
// ballot per bit, so the cost does not depend on how many distinct bins the
// wavefront holds.  Meaningful for valid lanes only.
__device__ __forceinline__ uint64_t bin_peers(uint32_t bin, uint64_t valid) {
  static_assert(kBins == 512, "nine bin bits");
  uint64_t peers = valid;
  for (int bit = 0; bit < 9; bit++) {
    const bool set = (bin >> bit) & 1u;
    const uint64_t m = __ballot(set);
    peers &= set ? m : ~m;
  }
  return peers;
}

__device__ __forceinline__ void part_range(const uint32_t* stats, uint32_t p, float& mn, float& rd) {
  mn = __uint_as_float(stats[4 * p + 0]);
  const float mx = __uint_as_float(stats[4 * p + 1]);
  rd = mx - mn;
  if (rd == 0) rd += 0.001f;                                      // sortingTriangles.go:43-46
}

constexpr uint32_t kHistThreads = 256;   // four wavefronts: a 2,048-triangle tile's keys in one round of loads
__global__ __launch_bounds__(kHistThreads) void k_hist(FrameArgs a, uint32_t blk0) {
  const uint32_t lb = frame_block(a, FC_TILES, 1);
  if (lb == kNoBlock) return;
  const uint32_t b = blk0 + lb;
  const uint32_t p = pair_of(a.tile_part, a.tile_prefix, a.nparts, b);
  const PartGPU P = a.parts[p];        // by value: read once, before any store
  if (P.ntiles <= 1) return;
  __shared__ uint32_t h[kBins];
  for (uint32_t i = threadIdx.x; i < kBins; i += blockDim.x) h[i] = 0;
  __syncthreads();
  const uint32_t tl = b - a.tile_prefix[p];
  const uint32_t n = a.tile_count[b];                // survivors, compacted at the tile's front
  const float* __restrict__ keys = a.key + P.tbase + tl * a.tile;
  float mn, rd;
  part_range(a.stats, p, mn, rd);
  const uint32_t mode = (P.flags >> PF_SORT_SHIFT) & 3u;
  for (uint32_t ib = 0; ib < n; ib += 8 * kHistThreads) {     // eight independent loads in flight per lane
    float d[8];
    for (int j = 0; j < 8; j++) {
      const uint32_t i = ib + j * kHistThreads + threadIdx.x;
      d[j] = i < n ? keys[i] : 0.0f;
    }
    // every survivor counts, a NaN key (kept when processOnlyVisible is false) included
    for (int j = 0; j < 8; j++)
      if (ib + j * kHistThreads + threadIdx.x < n) atomicAdd(&h[visit_bin(d[j], mn, rd, mode)], 1u);
  }
  __syncthreads();
  uint32_t* col = a.hist + P.hbase + tl;
  for (uint32_t i = threadIdx.x; i < kBins; i += blockDim.x) col[(size_t)i * P.ntiles] = h[i];
}

// Scan of each multi-tile part's histogram matrix, laid out bin-major
// (element bin*ntiles + tile), which is exactly the output order.
__device__ __forceinline__ uint32_t block_exclusive_scan_256(uint32_t v, uint32_t* s_tmp, uint32_t& total) {
  const uint32_t ln = threadIdx.x % warpSize, wv = threadIdx.x / warpSize;
  uint32_t x = v;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(x, o);
    if (ln >= (uint32_t)o) x += y;
  }
  if (ln == 63) s_tmp[wv] = x;
  __syncthreads();
  uint32_t wbase = 0, tot = 0;
  for (uint32_t w = 0; w < blockDim.x / 64; w++) {
    if (w < wv) wbase += s_tmp[w];
    tot += s_tmp[w];
  }
  __syncthreads();
  total = tot;
  return wbase + x - v;
}

__global__ __launch_bounds__(256) void k_scan_reduce(FrameArgs a, uint32_t sblk0) {
  if (past_count(a, FC_SBLOCKS)) return;
  const uint32_t b = sblk0 + blockIdx.x;
  const uint32_t p = find_part(a.sblock_prefix, a.nparts, b);
  const PartGPU P = a.parts[p];        // by value: read once, before any store
  const uint32_t len = kBins * P.ntiles;
  const uint32_t e0 = (b - a.sblock_prefix[p]) * kScanBlock;
  uint32_t s = 0;
  for (uint32_t e = e0 + threadIdx.x; e < min(e0 + kScanBlock, len); e += blockDim.x) s += a.hist[P.hbase + e];
  __shared__ uint32_t s_tmp[8];
  s = wave_sum(s);
  if (threadIdx.x % warpSize == 0) s_tmp[threadIdx.x / warpSize] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t t = 0;
    for (uint32_t w = 0; w < blockDim.x / warpSize; w++) t += s_tmp[w];
    a.bsum[b] = t;
  }
}

// Exclusive scan of each part's scan-block sums, one 256-thread block per
// part, 256 sums per step with the running total carried across steps (a
// serial walk would pay one dependent memory round trip per scan block).
__global__ __launch_bounds__(256) void k_scan_bsums(FrameArgs a, uint32_t part0) {
  if (past_count(a, FC_PAIRS)) return;
  const uint32_t n = a.parts[part0 + blockIdx.x].nsblocks;
  if (n == 0) return;
  uint32_t* __restrict__ bs = a.bsum + a.parts[part0 + blockIdx.x].sblock0;
  __shared__ uint32_t s_tmp[8];
  uint32_t carry = 0;
  for (uint32_t c = 0; c < n; c += 256) {
    const uint32_t k = c + threadIdx.x;
    const uint32_t v = k < n ? bs[k] : 0u;
    uint32_t total;
    const uint32_t ex = block_exclusive_scan_256(v, s_tmp, total);
    if (k < n) bs[k] = carry + ex;
    carry += total;
  }
}

__global__ __launch_bounds__(256) void k_scan_down(FrameArgs a, uint32_t sblk0) {
  if (past_count(a, FC_SBLOCKS)) return;
  const uint32_t b = sblk0 + blockIdx.x;
  const uint32_t p = find_part(a.sblock_prefix, a.nparts, b);
  const PartGPU P = a.parts[p];        // by value: read once, before any store
  const uint32_t len = kBins * P.ntiles;
  const uint32_t e0 = (b - a.sblock_prefix[p]) * kScanBlock;
  __shared__ uint32_t s_tmp[8];
  uint32_t base = a.bsum[b];
  constexpr uint32_t per = kScanBlock / 256;
  uint32_t v[per];
  uint32_t local = 0;
  const uint32_t my0 = e0 + threadIdx.x * per;
  for (uint32_t k = 0; k < per; k++) {
    const uint32_t e = my0 + k;
    v[k] = e < len ? a.hist[P.hbase + e] : 0u;
    local += v[k];
  }
  uint32_t total;
  uint32_t ex = block_exclusive_scan_256(local, s_tmp, total) + base;
  for (uint32_t k = 0; k < per; k++) {
    const uint32_t e = my0 + k;
    if (e < len) a.hist[P.hbase + e] = ex;
    ex += v[k];
  }
}

// Exclusive scan of a whole [bin][tile] matrix by one 1024-thread block: each
// thread loads its contiguous segment (at most kPer 16-byte words, all loads
// issued before the first use), one block-wide scan of the 1024 segment sums,
// then each thread writes its segment back from registers.  One launch, two
// barriers and one memory round trip each way replace the three launches of
// the general scan for the (common) parts whose matrix has at most
// kScanPartMax entries.
__global__ __launch_bounds__(1024) void k_scan_part(FrameArgs a, uint32_t blk0) {
  constexpr uint32_t kPer = kScanPartMax / 4 / 1024;
  static_assert(kScanPartMax % 4096 == 0, "whole uint4 segments");
  if (past_count(a, FC_PSCAN)) return;
  const uint32_t b = blk0 + blockIdx.x;
  // the pair: a binary search of the prefixes, staged in LDS first when they fit (one memory round trip
  // instead of one per step)
  constexpr uint32_t kPrefixLds = 4096;
  __shared__ uint32_t s_pre[kPrefixLds];
  uint32_t p;
  if (a.nparts < kPrefixLds) {
    for (uint32_t i = threadIdx.x; i <= a.nparts; i += blockDim.x) s_pre[i] = a.pscan_prefix[i];
    __syncthreads();
    p = find_part(s_pre, a.nparts, b);
  } else {
    p = find_part(a.pscan_prefix, a.nparts, b);
  }
  const uint32_t n4 = kBins * a.parts[p].ntiles / 4;           // the matrix holds a multiple of 512 entries
  uint4* __restrict__ h = reinterpret_cast<uint4*>(a.hist + a.parts[p].hbase);   // 2 KB aligned
  const uint32_t tid = threadIdx.x, lane = tid % 64u, wv = tid / 64u;
  const uint32_t per = (n4 + 1023) / 1024;                     // <= kPer
  const uint32_t q0 = min(tid * per, n4), cnt = min(per, n4 - q0);
  uint4 v[kPer];
#pragma unroll
  for (uint32_t j = 0; j < kPer; j++) v[j] = j < cnt ? h[q0 + j] : make_uint4(0, 0, 0, 0);
  uint32_t sum = 0;
#pragma unroll
  for (uint32_t j = 0; j < kPer; j++) sum += v[j].x + v[j].y + v[j].z + v[j].w;
  __shared__ uint32_t s_w[16];
  uint32_t x = sum;
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(x, o);
    if (lane >= (uint32_t)o) x += y;
  }
  if (lane == 63) s_w[wv] = x;
  __syncthreads();
  uint32_t run = x - sum;
  for (uint32_t w = 0; w < wv; w++) run += s_w[w];
#pragma unroll
  for (uint32_t j = 0; j < kPer; j++) {
    uint4 o;
    o.x = run;
    o.y = o.x + v[j].x;
    o.z = o.y + v[j].y;
    o.w = o.z + v[j].z;
    run = o.w + v[j].w;
    if (j < cnt) h[q0 + j] = o;
  }
}

// Stable counting sort, scatter pass.  One wavefront per tile walks its
// triangles in index order, 64 at a time (keys staged in LDS in one burst),
// ranks equal bins with ballots and gives every survivor its output slot:
// run[bin] + rank, where run[bin] comes from the scanned [bin][tile]
// histogram, or from a local scan when the part is a single tile.  This is
// sortingTriangleBucket.Sort + ForEach (sortingTriangles.go:38-125): bins
// visited 511->0 (BackToFront) or 0->511, insertion order kept within a bin.
// The survivor's record {vertex-record offsets, triangle} goes to its slot; its
// corners are read from the mesh's indices here, where the tile's triangles
// still come in mesh order, so the cull writes 6 bytes per survivor, not 20.
__device__ __forceinline__ uint4 slot_record(const PartGPU& P, uint32_t t) {
  uint32_t ov[3];
  corner_records(P, t, ov);
  return make_uint4(ov[0], ov[1], ov[2], t);
}

__global__ __launch_bounds__(64) void k_scatter(FrameArgs a, uint32_t blk0) {
  const uint32_t lb = frame_block(a, FC_TILES, 1);
  if (lb == kNoBlock) return;
  const uint32_t b = blk0 + lb;
  const uint32_t p = pair_of(a.tile_part, a.tile_prefix, a.nparts, b);
  const PartGPU P = a.parts[p];        // by value: read once, before any store
  if (a.stats[4 * p + 2] == 0) return;
  const uint32_t tl = b - a.tile_prefix[p];
  const uint32_t n = a.tile_count[b];                // survivors, compacted at the tile's front
  const uint32_t lane = threadIdx.x;
  const uint32_t tbase = P.tbase;
  const uint32_t mode = (P.flags >> PF_SORT_SHIFT) & 3u;
  const uint32_t t0 = tl * a.tile;
  const uint16_t* __restrict__ loc = a.tri_loc + tbase + t0;
  uint4* __restrict__ rec_out = a.tri_vo + tbase;

  __shared__ uint32_t run[kBins];
  __shared__ float s_key[kMaxTile];
  float mn, rd;
  part_range(a.stats, p, mn, rd);
  for (uint32_t i = lane; i < n; i += 64) s_key[i] = a.key[tbase + tl * a.tile + i];   // one burst of loads

  if (P.ntiles > 1) {
    const uint32_t* col = a.hist + P.hbase + tl;
    for (uint32_t i = lane; i < kBins; i += 64) run[i] = col[(size_t)i * P.ntiles];
    __syncthreads();
  } else {
    for (uint32_t i = lane; i < kBins; i += 64) run[i] = 0;
    __syncthreads();
    for (uint32_t i = lane; i < n; i += 64) atomicAdd(&run[visit_bin(s_key[i], mn, rd, mode)], 1u);
    __syncthreads();
    uint32_t c[8], s = 0;                       // exclusive scan of 512 counters, 8 per lane
    for (int k = 0; k < 8; k++) {
      c[k] = run[lane * 8 + k];
      s += c[k];
    }
    uint32_t x = s;
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(x, o);
      if (lane >= (uint32_t)o) x += y;
    }
    uint32_t ex = x - s;
    __syncthreads();
    for (int k = 0; k < 8; k++) {
      run[lane * 8 + k] = ex;
      ex += c[k];
    }
    __syncthreads();
  }

  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  uint4 rec_next = lane < n ? slot_record(P, t0 + loc[lane]) : make_uint4(0, 0, 0, 0);   // records one chunk ahead
  for (uint32_t base_i = 0; base_i < n; base_i += 64) {
    const uint32_t i = base_i + lane;
    const bool valid = i < n;
    const float d = valid ? s_key[i] : -1.0f;
    const uint64_t vmask = __ballot(valid);
    const uint4 rec = rec_next;
    if (i + 64 < n) rec_next = slot_record(P, t0 + loc[i + 64]);
    const uint32_t bin = valid ? visit_bin(d, mn, rd, mode) : 0xFFFFFFFFu;
    const uint64_t peers = bin_peers(bin, vmask);
    const uint32_t rank = (uint32_t)__popcll(peers & lt_mask);
    uint32_t slot = 0;
    if (valid) slot = run[bin] + rank;
    __syncthreads();
    if (valid) {
      if (rank == 0) run[bin] = slot + (uint32_t)__popcll(peers);
      rec_out[slot] = rec;
    }
    __syncthreads();
  }
}

// The same scatter with four wavefronts per tile.  Wave w owns a contiguous
// quarter of the tile's 64-triangle chunks.  A first pass over the staged keys
// counts each wave's survivors per bin; the base of wave w in bin k is
// run[k] plus the counts of waves 0..w-1 in bin k, so the four quarters rank
// independently and the result is the single-wave order exactly.
constexpr uint32_t kScatterWaves = 4;
__global__ __launch_bounds__(256) void k_scatter4(FrameArgs a, uint32_t blk0) {
  const uint32_t lb = frame_block(a, FC_TILES, 1);
  if (lb == kNoBlock) return;
  const uint32_t b = blk0 + lb;
  const uint32_t p = pair_of(a.tile_part, a.tile_prefix, a.nparts, b);
  const PartGPU P = a.parts[p];        // by value: read once, before any store
  if (a.stats[4 * p + 2] == 0) return;
  const uint32_t tl = b - a.tile_prefix[p];
  const uint32_t t0 = tl * a.tile;
  const uint32_t n = a.tile_count[b];                // survivors, compacted at the tile's front
  const uint32_t tid = threadIdx.x, lane = tid % 64u, wv = tid / 64u;
  const uint32_t tbase = P.tbase;
  const uint32_t mode = (P.flags >> PF_SORT_SHIFT) & 3u;
  const uint16_t* __restrict__ loc = a.tri_loc + tbase + t0;
  uint4* __restrict__ rec_out = a.tri_vo + tbase;

  __shared__ uint32_t s_off[kScatterWaves][kBins];
  __shared__ uint32_t s_tmp[8];
  float mn, rd;
  part_range(a.stats, p, mn, rd);
  for (uint32_t i = tid; i < kScatterWaves * kBins; i += blockDim.x) (&s_off[0][0])[i] = 0;
  // a multi-tile pair's scanned column (each thread's two bins) is loaded now, beside the keys
  static_assert(kBins == 2 * 256, "two bins per thread");
  uint32_t col_run[2] = {0, 0};
  if (P.ntiles > 1) {
    const uint32_t* col = a.hist + P.hbase + tl;
    col_run[0] = col[(size_t)tid * P.ntiles];
    col_run[1] = col[(size_t)(tid + 256) * P.ntiles];
  }
  // In a large frame, this tile's share of its pair's vertex records, a word
  // of every 128-byte line, read so that the assembly finds them in the
  // 256 MB memory-side cache: its reads wait long behind its own stores where
  // they have to go to HBM.  With 3.9 M vertex records (187 MB) the assembly
  // takes 212 us with it and 320 us without, this pass 66 us instead of 37;
  // with 2.8 M 161 and 188 against 49 and 34; with 1.9 M records (94 MB) and
  // less they are still cached and reading them only costs (113 and 110
  // against 35 and 25).
  float touch = 0.0f;
  if (a.counts ? a.counts[FC_SUMV] > kTouchVertices && !a.lean : a.touch_records != 0) {
    constexpr uint32_t kLine = 128 / sizeof(float);
    const uint32_t v0 = (uint32_t)((uint64_t)P.vcount * tl / P.ntiles);
    const uint32_t nv = (uint32_t)((uint64_t)P.vcount * (tl + 1) / P.ntiles) - v0;
    const float* ab = reinterpret_cast<const float*>(a.vab + 2 * ((size_t)P.vbase + v0));
    const float* vq = reinterpret_cast<const float*>(a.vq + (size_t)P.vbase + v0);
    for (uint32_t i = tid * kLine; i < 8 * nv; i += 256 * kLine) touch += ab[i];
    for (uint32_t i = tid * kLine; i < 4 * nv; i += 256 * kLine) touch += vq[i];
  }
  const uint32_t nchunks = (n + 63) / 64;
  const uint32_t c0 = (wv * nchunks) / kScatterWaves, c1 = ((wv + 1) * nchunks) / kScatterWaves;
  // every key and record of this wave's chunks (at most kChunks of 64) is
  // loaded up front, so the counting and ranking passes wait on memory once
  constexpr uint32_t kChunks = kMaxTile / 64 / kScatterWaves;
  float d[kChunks];
  uint4 rec[kChunks];
  uint32_t tri[kChunks];
  uint32_t bin[kChunks];
  bool in[kChunks];
#pragma unroll
  for (uint32_t j = 0; j < kChunks; j++) {
    const uint32_t i = (c0 + j) * 64 + lane;
    in[j] = c0 + j < c1 && i < n;
    d[j] = in[j] ? a.key[tbase + t0 + i] : 0.0f;
    tri[j] = t0 + (in[j] ? loc[i] : 0u);
  }
#pragma unroll
  for (uint32_t j = 0; j < kChunks; j++) rec[j] = slot_record(P, tri[j]);   // any lane's triangle is in the mesh
  __syncthreads();
#pragma unroll
  for (uint32_t j = 0; j < kChunks; j++) {
    bin[j] = 0xFFFFu;                             // no survivor in this lane
    if (in[j]) {                                  // a NaN key (processOnlyVisible false) is a survivor too
      bin[j] = visit_bin(d[j], mn, rd, mode);
      atomicAdd(&s_off[wv][bin[j]], 1u);
    }
  }
  __syncthreads();
  // per bin: base of each wave (two bins per thread)
  if (P.ntiles > 1) {
    for (uint32_t j = 0; j < 2; j++) {
      const uint32_t k = tid + 256 * j;
      uint32_t run = col_run[j];
      for (uint32_t w = 0; w < kScatterWaves; w++) {
        const uint32_t c = s_off[w][k];
        s_off[w][k] = run;
        run += c;
      }
    }
  } else {
    uint32_t cnt[2], sum = 0;
    for (int j = 0; j < 2; j++) {
      cnt[j] = 0;
      for (uint32_t w = 0; w < kScatterWaves; w++) cnt[j] += s_off[w][2 * tid + j];
      sum += cnt[j];
    }
    uint32_t total;
    uint32_t run = block_exclusive_scan_256(sum, s_tmp, total);
    for (int j = 0; j < 2; j++) {
      const uint32_t k = 2 * tid + j;
      for (uint32_t w = 0; w < kScatterWaves; w++) {
        const uint32_t c = s_off[w][k];
        s_off[w][k] = run;
        run += c;
      }
    }
  }
  __syncthreads();

  // each wave ranks its own chunks; only this wave touches s_off[wv]
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  uint32_t* off = s_off[wv];
#pragma unroll
  for (uint32_t j = 0; j < kChunks; j++) {
    const bool valid = bin[j] != 0xFFFFu;
    const uint64_t vmask = __ballot(valid);
    if (vmask == 0) continue;                     // uniform across the wave
    const uint64_t peers = bin_peers(bin[j], vmask);
    const uint32_t rank = (uint32_t)__popcll(peers & lt_mask);
    uint32_t slot = 0;
    if (valid) slot = off[bin[j]] + rank;
    __builtin_amdgcn_wave_barrier();
    if (valid && rank == 0) off[bin[j]] = slot + (uint32_t)__popcll(peers);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (valid) rec_out[slot] = rec[j];
  }
  asm volatile("" ::"v"(touch));                  // the loads are wanted for the caches alone
}

typedef float f4v __attribute__((ext_vector_type(4)));

template <bool kNT>
__device__ __forceinline__ void store4(float4* p, float4 v) {
  if (kNT) {
    f4v x = {v.x, v.y, v.z, v.w};
    __builtin_nontemporal_store(x, reinterpret_cast<f4v*>(p));
  } else {
    *p = v;
  }
}
template <bool kNT>
__device__ __forceinline__ void store1(uint32_t* p, uint32_t v) {
  if (kNT) __builtin_nontemporal_store(v, p);
  else *p = v;
}

// Output-order assembly: the ebiten colour, depth (and normal) vertices and
// the indices of a pair's drawn triangles in slot order (camera.go:1646-1820,
// 1710-1722).  A list of S triangles is 9 * S float4 (three per vertex:
// position and texture position, colour, custom values), and every lane owns
// one float4 of each list: it finds its corner's record in the slot records
// and copies its piece, so a wavefront's stores are whole 1 KB runs with no
// staging and no barrier, and the three lanes of a corner read one record.
// A wavefront takes 576 float4 (64 triangles' worth) at a time, all nine
// gathers of a lane in flight together.  Chunks start at multiples of 64
// float4 of the whole list, not of the pair's, so every store covers whole
// 128-byte lines except at a pair's ends: a pair's first vertex lies anywhere.
// `per` blocks of `sub` triangles share one tile's slot range, so the grid
// follows the survivors more finely than the sort's tiles.
//
// What bounds it: the stores.  1.02 GB of lists (3.4 M triangles of 465 pairs)
// take 211 us, 4.8 TB/s; a kernel that only stores the same lists takes 190
// (242 with its runs 48 bytes off the lines), a fill of as many bytes 150.  Three float4 computed per
// corner and staged in LDS, nine rows a triangle, took 265 us.
constexpr uint32_t kAsmThreads = 256;
template <bool kNT, bool kNormals>
__global__ __launch_bounds__(kAsmThreads) void k_assemble(FrameArgs a, uint32_t blk0, uint32_t sub, uint32_t per) {
  const uint32_t li = frame_block<true>(a, FC_TILES, per);
  if (li == kNoBlock) return;
  const uint32_t b = blk0 + li / per;
  const uint32_t p = pair_of(a.tile_part, a.tile_prefix, a.nparts, b);
  const uint32_t S = a.stats[4 * p + 2];
  if (a.host_stats && b == a.tile_prefix[p] && li % per == 0 && threadIdx.x == 0) a.host_stats[4 * p + 2] = S;
  if (S == 0) return;
  const PartGPU& P = a.parts[p];
  // read before the first store, which may alias these tables as far as the compiler knows
  const uint64_t out_base = P.out_base;
  const uint32_t idx_base = P.idx_base, tbase = P.tbase, ntiles = P.ntiles;
  const FrameConst& fc = a.fc[P.cam];
  const float da = fc.render_depth ? 1.0f : 0.0f;
  const bool normals = kNormals && fc.render_normals != 0;
  const uint32_t j = (b - a.tile_prefix[p]) * per + li % per;       // this block's place among the pair's
  const uint32_t span = sub * 9;                                    // float4 per block; the last takes the rest
  const int64_t end = 9 * (int64_t)S;
  const int64_t first = (int64_t)j * span - (int64_t)(3 * out_base % 64);
  const int64_t last = j + 1 == ntiles * per ? end : min(first + (int64_t)span, end);
  const uint32_t lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const uint32_t* __restrict__ tvo = reinterpret_cast<const uint32_t*>(a.tri_vo + tbase);
  const float4* __restrict__ vab = a.vab;
  const float4* __restrict__ vq = a.vq;
  const float4* __restrict__ vnrm = a.vnrm;
  float4* __restrict__ out_c = a.out_color + 3 * out_base;
  float4* __restrict__ out_d = a.out_depth + 3 * out_base;
  float4* __restrict__ out_n = kNormals ? a.out_normal + 3 * out_base : nullptr;
  uint32_t* __restrict__ out_i = a.out_idx + out_base;
  constexpr uint32_t kPer = 9, kChunk = 64 * kPer;                  // float4 per lane and per wavefront
  for (int64_t c0 = first + wave * kChunk; c0 < last; c0 += (kAsmThreads / 64) * kChunk) {   // wave-uniform
    const int64_t c1 = min(c0 + (int64_t)kChunk, last);
    const uint32_t tri0 = c0 > 0 ? (uint32_t)(c0 / 9) : 0u;
    const int32_t rel = (int32_t)(c0 - 9 * (int64_t)tri0);          // the chunk's start from triangle tri0's
    const int32_t lim = (int32_t)(c1 - 9 * (int64_t)tri0);
    float4 v[kPer], n[kPer];
    float d[kPer];
    uint32_t ov[kPer];
#pragma unroll
    for (uint32_t q = 0; q < kPer; q++) {
      const uint32_t g = (uint32_t)min(max(rel + (int32_t)(q * 64 + lane), 0), lim - 1);   // an active float4
      const uint32_t corner = g / 3, tri = corner / 3;
      ov[q] = tvo[4 * (size_t)(tri0 + tri) + corner - 3 * tri];
    }
#pragma unroll
    for (uint32_t q = 0; q < kPer; q++) {
      const uint32_t g = (uint32_t)min(max(rel + (int32_t)(q * 64 + lane), 0), lim - 1);
      const uint32_t piece = g % 3;
      v[q] = *(piece == 2 ? vq + ov[q] : vab + 2 * (size_t)ov[q] + piece);
      d[q] = 0.0f;
      if (piece == 1) {
        d[q] = vq[ov[q]].z;
        if (normals) n[q] = vnrm[ov[q]];
      }
    }
#pragma unroll
    for (uint32_t q = 0; q < kPer; q++) {
      const int32_t g = rel + (int32_t)(q * 64 + lane);
      if (g < 0 || g >= lim) continue;
      const uint32_t piece = (uint32_t)g % 3;
      const int64_t f = c0 + q * 64 + lane;
      const float4 custom = make_float4(v[q].w, 0.0f, 0.0f, 0.0f);
      store4<kNT>(&out_c[f], piece == 2 ? custom : v[q]);
      store4<kNT>(&out_d[f], piece == 2 ? custom : piece == 1 ? make_float4(d[q], d[q], d[q], da) : v[q]);
      if (normals) store4<kNT>(&out_n[f], piece == 0 ? v[q] : piece == 1 ? n[q] : make_float4(0.0f, 0.0f, 0.0f, 0.0f));
    }
    // indices: flush-local iota, as the reference's indexList (camera.go:1816), of the vertices that start here
    const uint32_t i0 = c0 > 0 ? (uint32_t)((c0 + 2) / 3) : 0u, i1 = (uint32_t)((c1 + 2) / 3);
    for (uint32_t i = i0 + lane; i < i1; i += 64) store1<kNT>(&out_i[i], idx_base + i);
  }
}

// ---------------------------------------------------------------------------
// k_pair
// ---------------------------------------------------------------------------

// The chain from the vertices to the lists for frames of small meshes: one
// workgroup takes a whole render pair through k_vertex, k_cull, the sort and
// k_assemble, with the cull's screen positions, the keys, the histogram and
// the draw order in LDS and barriers where the chain has launches.  Each step
// is the chain's own (same functions, same order), so the lists are the same
// bit for bit.  Only the colour half of the vertex records and the skinned
// positions go through memory (the workgroup's own, read back by the same
// CU); tri_vo is written for t3d_frame_download_triangles.
//
// kThreads, kV and kT: threads, and the most vertices and triangles a pair may
// have (launch_pairs chooses by the frame's largest, and refuses what no
// variant holds, so the check below never finds a larger one).  LDS per block: 17 B a vertex, 8 B a triangle
// and 1 KB a wavefront; 112 KB at the largest.
//
// What bounds it: instructions and latency while a workgroup shades (10 us a
// round of 1,024 skinned vertices under six lights; 7 us before the first, of
// cold loads), then the stores of the lists.  642 vertices alone: 16 us, where
// the chain's six launches take 44; 4,096 cubes 12 us against 52; 256 skinned
// characters of 2,562 vertices 82 us against 125.  Where one pair is much
// larger than the others its workgroup is what the frame waits for (200
// uneven models of up to 4,000 vertices: 151 us a frame against 141 with the
// chain), so larger pairs come here only in even company (pairs_fit).
__device__ __forceinline__ void publish_count(const FrameArgs& a, uint32_t p, uint32_t n) {
  a.stats[4 * p + 2] = n;
  if (a.host_stats) a.host_stats[4 * p + 2] = n;
}

template <uint32_t kThreads, uint32_t kV, uint32_t kT>
__global__ __launch_bounds__(kThreads) void k_pair(FrameArgs a) {
  if (past_count(a, FC_PAIRS)) return;
  const uint32_t p = blockIdx.x;
  const PartGPU& R = a.parts[p];
  const uint32_t flags = load_uniform(&R.flags), vcount = load_uniform(&R.vcount), tcount = load_uniform(&R.tcount);
  const uint32_t vbase = load_uniform(&R.vbase), vmin = load_uniform(&R.vmin);
  if (tcount == 0 || tcount > kT || vcount > kV) {
    if (threadIdx.x == 0) publish_count(a, p, 0);
    return;
  }
  const FrameConst& fc = a.fc[load_uniform(&R.cam)];
  constexpr uint32_t kWaves = kThreads / 64;
  static_assert(kT % 64 == 0 && kT <= 65536 && kV <= 65536, "16-bit places");
  __shared__ float4 s_q[kV];
  __shared__ uint8_t s_z[kV];
  __shared__ uint32_t s_u[kT * 6 / 4];            // keys and triangles of the survivors; then their corners in draw order
  __shared__ uint16_t s_slot[kT];                 // triangles in draw order
  __shared__ uint32_t s_off[kWaves][kBins / 2];   // per wavefront and bin, two to a word: counts, then next slots
  __shared__ float4 s_bone_rows[kThreads > 64 ? kMaxLdsBones * kBoneRows : 1];
  __shared__ M4 s_umvp;
  __shared__ uint32_t s_w[kWaves];
  __shared__ float s_mn[kWaves], s_mx[kWaves];
  float* s_key = reinterpret_cast<float*>(s_u);
  uint16_t* s_tri = reinterpret_cast<uint16_t*>(s_u + kT);
  uint16_t* s_vo = reinterpret_cast<uint16_t*>(s_u);
  const uint32_t tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));

  // vertices
  const bool skinned = (flags & PF_SKINNED) != 0;
  const bool lds_bones = kThreads > 64 && skinned && load_uniform(&R.bone_count) <= kMaxLdsBones;
  if (lds_bones) stage_bones(R, s_bone_rows);
  if ((flags & PF_UNBB) && tid == 0) s_umvp = mult(load_uniform(&R.model), load_uniform(&fc.vp));
  for (uint32_t i = tid; i < kWaves * (kBins / 2); i += kThreads) (&s_off[0][0])[i] = 0;
  __syncthreads();
  for (uint32_t i = tid; i < vcount; i += kThreads) {
    V3 vp;
    const VertexRecord r = shade_vertex(a, fc, R, flags, vmin + i, lds_bones ? s_bone_rows : nullptr, s_umvp, vp);
    const uint32_t o = vbase + i;
    a.vab[2 * (size_t)o + 0] = r.a;
    a.vab[2 * (size_t)o + 1] = r.b;
    if (skinned) a.vpos[o] = make_float4(vp.x, vp.y, vp.z, 0.0f);
    s_q[i] = r.q;
    s_z[i] = r.zin ? 1 : 0;
  }
  __syncthreads();

  // cull: survivors in triangle order
  const bool backface = (flags & PF_BACKFACE) != 0;
  const bool all = (flags & PF_ALL) != 0;         // processOnlyVisible false: no test removes a triangle
  const PartGPU P = load_uniform(&R);              // what the passes over triangles read of it
  const V3 camPos = v3(load_uniform(&fc.campos[0]), load_uniform(&fc.campos[1]), load_uniform(&fc.campos[2]));
  const V3 icp = v3(P.icp[0], P.icp[1], P.icp[2]);
  float mn = kMaxF32, mx = 0.0f;
  uint32_t n = 0;                                 // survivors so far, block-uniform
  for (uint32_t base = 0; base < tcount; base += kThreads) {
    const uint32_t t = base + tid;
    bool keep = false;
    float depth = -1.0f;
    if (t < tcount) {
      uint32_t ov[3];
      corner_records(P, t, ov);
      float4 cc[3];
      V3 q[3];
      bool zin = false;
      if (skinned) {
        for (int k = 0; k < 3; k++) {
          const float4 x = a.vpos[ov[k]];
          q[k] = v3(x.x, x.y, x.z);
        }
      } else {
        const float* cp = P.ctr + 3 * (size_t)t;
        q[0] = v3(cp[0], cp[1], cp[2]);
      }
      for (int k = 0; k < 3; k++) {
        cc[k] = s_q[ov[k] - P.vbase];
        zin |= s_z[ov[k] - P.vbase] != 0;
      }
      keep = all || visible(cc, zin, backface);
      if (keep) {                                                       // model.go:941-960
        depth = depth_key(skinned, camPos, icp, q);
        if (!all && (isnan(depth) || isinf(depth))) keep = false;
      }
    }
    const uint64_t m = __ballot(keep);
    if (lane == 0) s_w[wave] = (uint32_t)__popcll(m);
    __syncthreads();
    uint32_t before = 0, tot = 0;
    for (uint32_t w = 0; w < kWaves; w++) {
      if (w < wave) before += s_w[w];
      tot += s_w[w];
    }
    if (keep) {
      const uint32_t at = n + before + (uint32_t)__popcll(m & lt_mask);
      s_key[at] = depth;
      s_tri[at] = (uint16_t)t;
      mn = fminf(mn, depth);
      mx = fmaxf(mx, depth);
    }
    n += tot;
    __syncthreads();                              // s_w is rewritten next round
  }
  mn = wave_min(mn);
  mx = wave_max(mx);
  if (lane == 0) {
    s_mn[wave] = mn;
    s_mx[wave] = mx;
  }
  __syncthreads();
  mn = s_mn[0];
  mx = s_mx[0];
  for (uint32_t w = 1; w < kWaves; w++) {
    mn = fminf(mn, s_mn[w]);
    mx = fmaxf(mx, s_mx[w]);
  }
  if (tid == 0) publish_count(a, p, n);
  if (n == 0) return;                             // block-uniform
  float rd = mx - mn;
  if (rd == 0) rd += 0.001f;                                            // sortingTriangles.go:43-46

  // sort: each wavefront counts, then ranks, a contiguous share of the
  // survivors' 64s, as in k_scatter4
  const uint32_t mode = (flags >> PF_SORT_SHIFT) & 3u;
  const uint32_t nchunks = (n + 63) / 64;
  const uint32_t ch0 = wave * nchunks / kWaves, ch1 = (wave + 1) * nchunks / kWaves;
  for (uint32_t c = ch0; c < ch1; c++) {
    const uint32_t i = c * 64 + lane;
    if (i < n) {
      const uint32_t bin = visit_bin(s_key[i], mn, rd, mode);
      atomicAdd(&s_off[wave][bin / 2], 1u << (16 * (bin % 2)));
    }
  }
  __syncthreads();
  uint16_t* off16 = reinterpret_cast<uint16_t*>(&s_off[0][0]);
  {
    constexpr uint32_t kPer = kThreads < kBins ? kBins / kThreads : 1;   // bins per thread
    uint32_t sum = 0;
    if (tid * kPer < kBins)
      for (uint32_t k = tid * kPer; k < (tid + 1) * kPer; k++)
        for (uint32_t w = 0; w < kWaves; w++) sum += off16[w * kBins + k];
    uint32_t x = sum;
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(x, o);
      if (lane >= (uint32_t)o) x += y;
    }
    if (lane == 63) s_w[wave] = x;
    __syncthreads();
    uint32_t next = x - sum;
    for (uint32_t w = 0; w < wave; w++) next += s_w[w];
    if (tid * kPer < kBins)
      for (uint32_t k = tid * kPer; k < (tid + 1) * kPer; k++)
        for (uint32_t w = 0; w < kWaves; w++) {
          const uint32_t c = off16[w * kBins + k];
          off16[w * kBins + k] = (uint16_t)next;
          next += c;
        }
  }
  __syncthreads();
  uint16_t* off = off16 + wave * kBins;           // only this wavefront's from here on
  for (uint32_t c = ch0; c < ch1; c++) {          // wave-uniform
    const uint32_t i = c * 64 + lane;
    const bool valid = i < n;
    const uint64_t vmask = __ballot(valid);
    const uint32_t bin = valid ? visit_bin(s_key[i], mn, rd, mode) : 0xFFFFu;
    const uint64_t peers = bin_peers(bin, vmask);
    const uint32_t rank = (uint32_t)__popcll(peers & lt_mask);
    uint32_t slot = 0;
    if (valid) slot = off[bin] + rank;
    __builtin_amdgcn_wave_barrier();
    if (valid && rank == 0) off[bin] = (uint16_t)(slot + (uint32_t)__popcll(peers));
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (valid) s_slot[slot] = s_tri[i];
  }
  __syncthreads();
  for (uint32_t k = tid; k < n; k += kThreads) {  // corners in draw order, over the keys
    const uint4 r = slot_record(P, s_slot[k]);
    a.tri_vo[P.tbase + k] = r;
    s_vo[3 * k + 0] = (uint16_t)(r.x - P.vbase);
    s_vo[3 * k + 1] = (uint16_t)(r.y - P.vbase);
    s_vo[3 * k + 2] = (uint16_t)(r.z - P.vbase);
  }
  __syncthreads();

  // lists, in the chunks of k_assemble
  const float da = load_uniform(&fc.render_depth) ? 1.0f : 0.0f;
  const float4* vab = a.vab + 2 * (size_t)P.vbase;   // this block's own stores, before the last barriers
  float4* __restrict__ out_c = a.out_color + 3 * P.out_base;
  float4* __restrict__ out_d = a.out_depth + 3 * P.out_base;
  uint32_t* __restrict__ out_i = a.out_idx + P.out_base;
  const int32_t end = 9 * (int32_t)n;
  constexpr int32_t kPer = 9, kChunk = 64 * kPer;
  for (int32_t c0 = -(int32_t)(3 * P.out_base % 64) + (int32_t)wave * kChunk; c0 < end; c0 += (int32_t)kWaves * kChunk) {
    float4 v[kPer];
    float4 w[kPer];
#pragma unroll
    for (int32_t q = 0; q < kPer; q++) {
      const uint32_t g = (uint32_t)min(max(c0 + q * 64 + (int32_t)lane, 0), end - 1);   // an active float4
      const uint32_t corner = g / 3, piece = g % 3, o = s_vo[corner];
      w[q] = s_q[o];
      if (piece != 2) v[q] = vab[2 * o + piece];
    }
#pragma unroll
    for (int32_t q = 0; q < kPer; q++) {
      const int32_t g = c0 + q * 64 + (int32_t)lane;
      if (g < 0 || g >= end) continue;
      const uint32_t piece = (uint32_t)g % 3;
      const float4 custom = make_float4(w[q].w, 0.0f, 0.0f, 0.0f);
      store4<true>(&out_c[g], piece == 2 ? custom : v[q]);
      store4<true>(&out_d[g], piece == 2 ? custom : piece == 1 ? make_float4(w[q].z, w[q].z, w[q].z, da) : v[q]);
    }
  }
  for (uint32_t i = tid; i < 3 * n; i += kThreads) store1<true>(&out_i[i], P.idx_base + i);   // camera.go:1816
}

// Fill of a word array (test poisoning of outputs: unwritten entries show up).
__global__ __launch_bounds__(256) void k_fill(uint32_t* __restrict__ p, uint64_t n, uint32_t v) {
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) p[i] = v;
}

// Survivors of a range of pairs packed back to back for the download (one
// transfer per stream instead of three per pair).  A block finds its pair by
// binary search of the block prefix: the pair p with blk_prefix[p] <= block <
// blk_prefix[p + 1] (every listed pair has at least one vertex, and 3 * nvert
// elements, 256 to a block).
__global__ __launch_bounds__(256) void k_pack(PackArgs a) {
  const uint32_t b = blockIdx.x;
  uint32_t lo = 0, hi = a.npairs;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (a.blk_prefix[mid] <= b) lo = mid;
    else hi = mid;
  }
  // element e of the pair: float4 e of its colour and depth runs (3 per vertex), and index e while e < nvert,
  // so consecutive lanes move consecutive 16-byte words
  const uint64_t e = (uint64_t)(b - a.blk_prefix[lo]) * 256 + threadIdx.x;
  const uint64_t n = a.nvert[lo];
  if (e >= 3 * n) return;
  const uint64_t s = a.src[lo], d = a.dst[lo];
  if (a.pcolor) a.pcolor[3 * d + e] = a.color[3 * s + e];
  if (a.pdepth) a.pdepth[3 * d + e] = a.depth[3 * s + e];
  if (a.pnormal) a.pnormal[3 * d + e] = a.normal[3 * s + e];
  if (a.pidx && e < n) a.pidx[d + e] = a.idx[s + e];
  if (a.ptri && e < n / 3) a.ptri[d / 3 + e] = a.tri_vo[a.tsrc[lo] + e].w + a.tfirst[lo];
}

// Dynamic batches (camera.go:2075-2099): the render pairs of one flush write
// into one vertex list, each after the corners of the ones before it, and
// their indices count on from there (the reference's vertexListIndex).  After
// k_cull, one block per batch scans its pairs' survivor counts and moves each
// pair's out_base and idx_base accordingly.  Only pairs in [part0, part1) are
// written (the plain form runs one pair's chain at a time; the pairs before
// it in its flush are final by then).  The first pair of a flush keeps the
// flush's own out_base, which every block reads before any write.
__global__ __launch_bounds__(256) void k_groups(FrameArgs a, uint32_t part0, uint32_t part1) {
  const uint2 g = a.groups[blockIdx.x];
  const uint32_t first = g.x, end = g.x + g.y;
  if (end <= part0 || first >= part1) return;                       // block-uniform
  PartGPU* parts = const_cast<PartGPU*>(a.parts);
  const uint64_t base = parts[first].out_base;
  __shared__ uint32_t s_scan[256];
  __shared__ uint32_t s_carry;
  if (threadIdx.x == 0) s_carry = 0;
  __syncthreads();
  for (uint32_t c0 = first; c0 < end; c0 += 256) {                  // block-uniform trip count
    const uint32_t i = c0 + threadIdx.x;
    const uint32_t v = i < end ? a.stats[4 * i + 2] : 0u;
    s_scan[threadIdx.x] = v;
    __syncthreads();
    for (uint32_t d = 1; d < 256; d <<= 1) {                        // inclusive scan
      const uint32_t t = threadIdx.x >= d ? s_scan[threadIdx.x - d] : 0u;
      __syncthreads();
      s_scan[threadIdx.x] += t;
      __syncthreads();
    }
    const uint32_t before = s_carry + s_scan[threadIdx.x] - v;      // survivors of the flush's earlier pairs
    if (i < end && i >= part0 && i < part1) {
      parts[i].out_base = base + 3ull * before;
      parts[i].idx_base = 3u * before;
    }
    __syncthreads();
    if (threadIdx.x == 255) s_carry += s_scan[255];
    __syncthreads();
  }
}

// Plain float4 copy of a known size: the reference point for HBM byte counters.
__global__ __launch_bounds__(256) void k_copy(const float4* __restrict__ src, float4* __restrict__ dst, uint64_t n) {
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
    dst[i] = src[i];
}

__global__ void k_fp_selftest(const float* x, const float* y, float* out, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  out[i] = fdiv(x[i], y[i]);
  out[n + i] = fsqrt(fabsf(x[i]));
  out[2 * n + i] = x[i] * y[i] + x[i];
  out[3 * n + i] = roundf(x[i]);
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------

hipError_t launch_palettes(const FrameArgs& a, hipStream_t s) {
  if (!a.npal_jobs) return hipSuccess;
  hipLaunchKernelGGL(k_palettes, dim3(a.npal_jobs), dim3(kPoseThreads), 0, s, a);
  return hipGetLastError();
}
hipError_t launch_uniforms(const FrameArgs& a, uint32_t part0, uint32_t nparts, hipStream_t s) {
  if (!nparts) return hipSuccess;
  hipLaunchKernelGGL(k_uniforms, dim3(nparts), dim3(kUniformThreads), 0, s, a, part0, nparts);
  return hipGetLastError();
}
hipError_t launch_vertex(const FrameArgs& a, uint32_t blk0, uint32_t nblk, uint32_t threads, VertexOut out, hipStream_t s) {
  if (!nblk) return hipSuccess;
  switch (out) {
    case VERTEX_FOR_CULL: hipLaunchKernelGGL(k_vertex<VERTEX_FOR_CULL>, dim3(nblk), dim3(threads), 0, s, a, blk0); break;
    case VERTEX_FOR_LISTS: hipLaunchKernelGGL(k_vertex<VERTEX_FOR_LISTS>, dim3(nblk), dim3(threads), 0, s, a, blk0); break;
    default: hipLaunchKernelGGL(k_vertex<VERTEX_ALL>, dim3(nblk), dim3(threads), 0, s, a, blk0); break;
  }
  return hipGetLastError();
}
hipError_t launch_cull(const FrameArgs& a, uint32_t blk0, uint32_t nblk, uint32_t threads, hipStream_t s) {
  if (!nblk) return hipSuccess;
  switch (threads) {
    case 256: hipLaunchKernelGGL(k_cull<256>, dim3(nblk), dim3(256), 0, s, a, blk0); break;
    case 512: hipLaunchKernelGGL(k_cull<512>, dim3(nblk), dim3(512), 0, s, a, blk0); break;
    case 1024: hipLaunchKernelGGL(k_cull<1024>, dim3(nblk), dim3(1024), 0, s, a, blk0); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
hipError_t launch_hist(const FrameArgs& a, uint32_t blk0, uint32_t nblk, hipStream_t s) {
  if (!nblk) return hipSuccess;
  hipLaunchKernelGGL(k_hist, dim3(nblk), dim3(kHistThreads), 0, s, a, blk0);
  return hipGetLastError();
}
hipError_t launch_scan(const FrameArgs& a, uint32_t sblk0, uint32_t nsblk, uint32_t part0, uint32_t nparts,
                       hipStream_t s) {
  if (!nsblk) return hipSuccess;
  hipLaunchKernelGGL(k_scan_reduce, dim3(nsblk), dim3(256), 0, s, a, sblk0);
  hipLaunchKernelGGL(k_scan_bsums, dim3(nparts), dim3(256), 0, s, a, part0);
  hipLaunchKernelGGL(k_scan_down, dim3(nsblk), dim3(256), 0, s, a, sblk0);
  return hipGetLastError();
}
hipError_t launch_scan_part(const FrameArgs& a, uint32_t blk0, uint32_t nblk, hipStream_t s) {
  if (!nblk) return hipSuccess;
  hipLaunchKernelGGL(k_scan_part, dim3(nblk), dim3(1024), 0, s, a, blk0);
  return hipGetLastError();
}
hipError_t launch_scatter(const FrameArgs& a, uint32_t blk0, uint32_t nblk, uint32_t waves, hipStream_t s) {
  if (!nblk) return hipSuccess;
  if (waves == kScatterWaves) hipLaunchKernelGGL(k_scatter4, dim3(nblk), dim3(64 * kScatterWaves), 0, s, a, blk0);
  else hipLaunchKernelGGL(k_scatter, dim3(nblk), dim3(64), 0, s, a, blk0);
  return hipGetLastError();
}
hipError_t launch_assemble(const FrameArgs& a, uint32_t blk0, uint32_t nblk, uint32_t mode, uint32_t split,
                           uint32_t max_triangles, hipStream_t s) {
  if (!nblk) return hipSuccess;
  if (split == 0 || (split & (split - 1)) || a.tile % split) return hipErrorInvalidValue;
  // pairs of one tile with few triangles need fewer blocks than the tile has room for: 4,096 cubes of 12
  // triangles took 26 us with eight blocks each, 10 us with one
  const uint32_t sub = a.tile / split;
  const uint32_t per = max_triangles < a.tile ? std::max(1u, (max_triangles + sub - 1) / sub) : split;
  FrameArgs b = a;
  if (mode & 64u) b.xcd_swizzle = 0;   // bit 6: the assembly's blocks in launch order, whatever the other passes use
  const dim3 g(nblk * per);
  switch ((mode & 2u) | (a.out_normal ? 1u : 0u)) {
    case 0: hipLaunchKernelGGL((k_assemble<false, false>), g, dim3(kAsmThreads), 0, s, b, blk0, sub, per); break;
    case 1: hipLaunchKernelGGL((k_assemble<false, true>), g, dim3(kAsmThreads), 0, s, b, blk0, sub, per); break;
    case 2: hipLaunchKernelGGL((k_assemble<true, false>), g, dim3(kAsmThreads), 0, s, b, blk0, sub, per); break;
    default: hipLaunchKernelGGL((k_assemble<true, true>), g, dim3(kAsmThreads), 0, s, b, blk0, sub, per); break;
  }
  return hipGetLastError();
}
// The workgroup: one wavefront for pairs of at most 128 vertices and triangles;
// four for larger ones when there are more pairs than CUs can take at sixteen
// wavefronts each; else sixteen.
hipError_t launch_pairs(const FrameArgs& a, uint32_t npairs, uint32_t max_vertices, uint32_t max_triangles, hipStream_t s) {
  if (!npairs) return hipSuccess;
  const uint32_t V = max_vertices, T = max_triangles;
  const dim3 g(npairs);
  if (V <= 128 && T <= 128) hipLaunchKernelGGL((k_pair<64, 128, 128>), g, dim3(64), 0, s, a);
  else if (V <= kPairVertices && T <= kPairTriangles) {
    if (npairs > 512) hipLaunchKernelGGL((k_pair<256, kPairVertices, kPairTriangles>), g, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((k_pair<1024, kPairVertices, kPairTriangles>), g, dim3(1024), 0, s, a);
  } else if (V <= kPairVerticesMany && T <= kPairTrianglesMany) {
    hipLaunchKernelGGL((k_pair<1024, kPairVerticesMany, kPairTrianglesMany>), g, dim3(1024), 0, s, a);
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
hipError_t launch_fill(void* dst, uint64_t bytes, uint32_t word, hipStream_t s) {
  if (bytes < 4) return hipSuccess;
  hipLaunchKernelGGL(k_fill, dim3(2048), dim3(256), 0, s, reinterpret_cast<uint32_t*>(dst), bytes / 4, word);
  return hipGetLastError();
}
hipError_t launch_pack(const PackArgs& a, uint32_t nblocks, hipStream_t s) {
  if (!nblocks) return hipSuccess;
  hipLaunchKernelGGL(k_pack, dim3(nblocks), dim3(256), 0, s, a);
  return hipGetLastError();
}
hipError_t launch_groups(const FrameArgs& a, uint32_t part0, uint32_t part1, hipStream_t s) {
  if (!a.ngroups) return hipSuccess;
  hipLaunchKernelGGL(k_groups, dim3(a.ngroups), dim3(256), 0, s, a, part0, part1);
  return hipGetLastError();
}
hipError_t launch_copy(const void* src, void* dst, uint64_t bytes, hipStream_t s) {
  const uint64_t n = bytes / 16;
  hipLaunchKernelGGL(k_copy, dim3(2048), dim3(256), 0, s, reinterpret_cast<const float4*>(src), reinterpret_cast<float4*>(dst), n);
  return hipGetLastError();
}
hipError_t launch_fp_selftest(const float* x, const float* y, float* out, uint32_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_fp_selftest, dim3((n + 255) / 256), dim3(256), 0, s, x, y, out, n);
  return hipGetLastError();
}

}  // namespace t3d
