// dh_kernels.hip -- gfx950 kernels of the per-frame raster path.
//
// Pipeline (one stream, no host synchronisation inside a frame):
//   1 k_geom_count   per input triangle: back-face cull, frustum clip count
//                    (scene/mod.rs:1016-1033, 43-90, 641-746), positions only,
//                    and whether it crosses the near or far plane
//   2 scan, k_geom_compact  block counts -> ordered output offsets (submission
//                    order) and two dense lists of emitting input triangles:
//                    unclipped, clipped
//   3 k_geom_emit    per listed triangle: per-vertex lighting (917-926), clip
//                    with attributes (clipped list only), projection
//                    (1047-1063), raster setup (canvas.rs:585-666) -> SetupRec +
//                    ShadeRec at its output id; with ordered bins also the
//                    conservative tile count, and the near-first depth key
//   4 k_pair_hist    near first (the default bins): (tile, triangle) pairs of
//                    each chunk of triangles counted by the tile's low digit
//   5 k_row_scan     -> each chunk's place in each digit's segment
//   6 k_pair_scatter the pairs into their segments
//   7 k_pair_sort    one workgroup per segment: its tiles' lists, near first,
//                    and the tile ranges.  (Submission order: k_wide_list,
//                    k_bin_count_wide, scan, k_bin_emit(_wide), a stable radix
//                    sort of the pairs by tile, k_tile_ranges.)
//  10 k_raster       one workgroup per screen tile: coverage and the strict
//                    depth test (canvas.rs:668-682, 923) into an LDS visibility
//                    buffer of (depth key << 32 | triangle id); the result does
//                    not depend on list order
//  11 k_shade        deferred Phong + texture shading of each pixel's winner
//                    (canvas.rs:684-745), BGRA8 + f32 depth
#include <math.h>
#include <stdio.h>

#include <algorithm>

#include "dh_common.hpp"
#include "dh_pipeline.hpp"

namespace dh {

// ===================================================================== common
__device__ inline uint32_t find_draw(const DevDraw* draws, uint32_t n, uint32_t t) {
  uint32_t lo = 0, hi = n;  // last draw with tri_begin <= t
  while (hi - lo > 1) {
    uint32_t mid = (lo + hi) >> 1;
    if (draws[mid].tri_begin <= t) lo = mid; else hi = mid;
  }
  return lo;
}

// The draw of input triangle t for every active lane of a wave (every lane
// calls it).  The lanes' triangles increase with the lane (ordered lists), so
// the draw of the first active lane's triangle, found with scalar loads, is
// every lane's whenever the last active lane's triangle lies before the next
// draw; otherwise each lane searches.
__device__ inline uint32_t wave_find_draw(const DevDraw* draws, uint32_t n, uint32_t t, bool active) {
  const uint64_t m = __ballot(active);
  if (!m) return 0u;
  const uint32_t t0 = (uint32_t)__builtin_amdgcn_readlane((int)t, __builtin_ctzll(m));
  const uint32_t t1 = (uint32_t)__builtin_amdgcn_readlane((int)t, 63 - __builtin_clzll(m));
  const uint32_t d0 = find_draw(draws, n, t0);
  if (d0 + 1u >= n || t1 < draws[d0 + 1u].tri_begin) return d0;
  return find_draw(draws, n, t);
}

__device__ inline V3 ld3(const float* a, uint32_t i) {
  Global<const float>* p = as_global(a) + 3ull * i;
  return v3(p[0], p[1], p[2]);
}

// Runs f(draw index) for the active lanes of a wave, d their draws (every lane
// calls it).  A wave of one draw, as most are, gets the index wave-uniform: the
// draw, its view's uniforms and its material come by scalar loads.  Per lane,
// they were some 60 vector loads of one address each (with global in place of
// FLAT accesses, 5M micro-triangles: k_geom_emit 172 -> 128 us, k_geom_count 68
// -> 53; the 32-view batch 96 -> 87 and 37 -> 29).  A wave of several draws does
// load per lane: going round once for each draw cost 1000 meshes of two
// triangles, 32 rounds a wave, 147 us of geometry kernels (59 per lane).
template <class F>
__device__ __forceinline__ void by_draw(uint32_t d, bool active, F f) {
  const uint64_t m = __ballot(active);
  if (!m) return;
  const uint32_t d0 = (uint32_t)__builtin_amdgcn_readlane((int)d, __builtin_ctzll(m));
  const bool one = __ballot(active && d != d0) == 0ull;
  if (!active) return;
  if (one) f(d0);
  else f(d);
}

// Vertex positions of a draw's triangle lt (a, b, c): from the mesh's
// per-triangle streams when it has them, else through its index triplet.
__device__ inline void tri_positions(const DevDraw& dr, uint32_t lt, V3& a, V3& b, V3& c) {
  if (dr.soa) {
    const uint64_t n = dr.n_tri;
    Global<const float>* s = as_global(dr.soa) + lt;
    a = v3(s[0], s[n], s[2 * n]);
    b = v3(s[3 * n], s[4 * n], s[5 * n]);
    c = v3(s[6 * n], s[7 * n], s[8 * n]);
  } else {
    Global<const uint32_t>* ti = as_global(dr.tri) + 9ull * lt;
    a = ld3(dr.pos, ti[0]);
    b = ld3(dr.pos, ti[1]);
    c = ld3(dr.pos, ti[2]);
  }
}

// Whether a wave reads its triangles' vertex records rather than the streams:
// when the input triangles of its active lanes span more than `span`, a
// stream load fetches several cache lines for few values each, and one
// 128-byte record per triangle moves fewer bytes.  The 24 streams of a wave
// spanning S triangles move about 1.5 S bytes per triangle, a record 128, but
// a record costs each lane its own lines: kSparseSpan (eight triangles per
// lane) by default, and kSparseSpanDense on frames of at least one input
// triangle per pixel, whose micro-triangles' culling survivors interleave
// finely (about 45% of them, a span near 145).  The choice only selects which
// copy of the same values is read.  Every lane of the wave calls it.
constexpr uint32_t kSparseSpan = 512u, kSparseSpanDense = 96u;
__device__ inline bool wave_sparse(bool active, uint32_t t, uint32_t span) {
  const uint64_t m = __ballot(active);
  if (!m) return false;
  const int first = __builtin_ctzll(m), last = 63 - __builtin_clzll(m);
  const uint32_t t0 = (uint32_t)__builtin_amdgcn_readlane((int)t, first);
  const uint32_t t1 = (uint32_t)__builtin_amdgcn_readlane((int)t, last);
  return t1 - t0 > span;
}

// Positions, normals and texture coordinates of the vertices of triangle lt:
// from the mesh's records (sparse) or streams when it has them, else through
// its index triplet.
__device__ inline void tri_vertices(const DevDraw& dr, uint32_t lt, bool sparse, V3 (&P)[3], V3 (&nrm)[3],
                                    float (&u)[3], float (&v)[3]) {
  if (dr.soa && sparse) {
    typedef float Vec4 __attribute__((ext_vector_type(4)));
    Global<const Vec4>* r = (Global<const Vec4>*)(dr.soa + mesh_records_offset(dr.n_tri)) +
                            (uint64_t)(kMeshRecFloats / 4u) * lt;
    float f[24];
#pragma unroll
    for (int q = 0; q < 6; q++) {
      const Vec4 x = r[q];
#pragma unroll
      for (int j = 0; j < 4; j++) f[4 * q + j] = x[j];
    }
#pragma unroll
    for (int k = 0; k < 3; k++) {
      P[k] = v3(f[3 * k], f[3 * k + 1], f[3 * k + 2]);
      nrm[k] = v3(f[9 + 3 * k], f[10 + 3 * k], f[11 + 3 * k]);
      u[k] = f[18 + 2 * k];
      v[k] = f[19 + 2 * k];
    }
  } else if (dr.soa) {
    const uint64_t n = dr.n_tri;
    Global<const float>* s = as_global(dr.soa) + lt;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      P[k] = v3(s[(3 * k) * n], s[(3 * k + 1) * n], s[(3 * k + 2) * n]);
      nrm[k] = v3(s[(9 + 3 * k) * n], s[(10 + 3 * k) * n], s[(11 + 3 * k) * n]);
      u[k] = s[(18 + 2 * k) * n];
      v[k] = s[(19 + 2 * k) * n];
    }
  } else {
    Global<const uint32_t>* ti = as_global(dr.tri) + 9ull * lt;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      P[k] = ld3(dr.pos, ti[k]);
      nrm[k] = ld3(dr.nrm, ti[6 + k]);
      Global<const float>* uv = as_global(dr.uv) + 2ull * ti[3 + k];
      u[k] = uv[0];
      v[k] = uv[1];
    }
  }
}

// Builds a mesh's vertex streams and records (once, when the mesh is created).
__global__ __launch_bounds__(256) void k_mesh_streams(const uint32_t* __restrict__ tri, uint32_t n_tri,
                                                      const float* __restrict__ pos, const float* __restrict__ nrm,
                                                      const float* __restrict__ uv, float* __restrict__ soa) {
  const uint64_t n = n_tri;
  uint4* rec = reinterpret_cast<uint4*>(soa + mesh_records_offset(n_tri));
  for (uint32_t t = blockIdx.x * 256u + threadIdx.x; t < n_tri; t += gridDim.x * 256u) {
    const uint32_t* q = tri + 9ull * t;
    float f[kMeshRecFloats];
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const float* p = pos + 3ull * q[k];
      const float* m = nrm + 3ull * q[6 + k];
      const float* w = uv + 2ull * q[3 + k];
#pragma unroll
      for (int j = 0; j < 3; j++) {
        f[3 * k + j] = p[j];
        f[9 + 3 * k + j] = m[j];
      }
      f[18 + 2 * k] = w[0];
      f[19 + 2 * k] = w[1];
    }
#pragma unroll
    for (int k = 24; k < (int)kMeshRecFloats; k++) f[k] = 0.0f;
#pragma unroll
    for (int k = 0; k < (int)kMeshStreams; k++) soa[(uint64_t)k * n + t] = f[k];
#pragma unroll
    for (int k = 0; k < (int)kMeshRecFloats / 4; k++)
      rec[(uint64_t)(kMeshRecFloats / 4u) * t + k] = make_uint4(
          __float_as_uint(f[4 * k]), __float_as_uint(f[4 * k + 1]), __float_as_uint(f[4 * k + 2]),
          __float_as_uint(f[4 * k + 3]));
  }
}

// Block of 256 threads (4 waves): exclusive scan of one value per thread.
__device__ inline uint32_t block_exclusive_scan256(uint32_t v, uint32_t* s_tmp /*[4]*/, uint32_t* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    uint32_t y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) s_tmp[wave] = x;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < 4; w++) {
    uint32_t t = s_tmp[w];
    if (w < wave) before += t;
    all += t;
  }
  __syncthreads();
  *total = all;
  return before + x - v;
}

// =================================================================== clipping
// Clip vertex with positions only (for counting) and with all attributes.
struct PV {
  V3 p;
};
struct FV {
  V3 p;
  float d;
  V3 n, l, h;
  float u, v;
};

// VertexAttributes a + (c - a) * t, canvas.rs:242-291 (screen_coord is still
// (0,0) at this stage and is overwritten by the projection).
__device__ inline PV lerpv(const PV& a, const PV& c, float t) {
  PV r;
  r.p = add(a.p, muls(sub(c.p, a.p), t));
  return r;
}
__device__ inline FV lerpv(const FV& a, const FV& c, float t) {
  FV r;
  r.p = add(a.p, muls(sub(c.p, a.p), t));
  r.d = a.d + ((c.d - a.d) * t);
  r.n = add(a.n, muls(sub(c.n, a.n), t));
  r.l = add(a.l, muls(sub(c.l, a.l), t));
  r.h = add(a.h, muls(sub(c.h, a.h), t));
  r.u = a.u + ((c.u - a.u) * t);
  r.v = a.v + ((c.v - a.v) * t);
  return r;
}

// Member-wise select (keeps the clip vertices in registers).
__device__ inline V3 sel3(bool q, V3 x, V3 y) { return v3(q ? x.x : y.x, q ? x.y : y.y, q ? x.z : y.z); }
__device__ inline PV selv(bool q, const PV& x, const PV& y) {
  PV r;
  r.p = sel3(q, x.p, y.p);
  return r;
}
__device__ inline FV selv(bool q, const FV& x, const FV& y) {
  FV r;
  r.p = sel3(q, x.p, y.p);
  r.d = q ? x.d : y.d;
  r.n = sel3(q, x.n, y.n);
  r.l = sel3(q, x.l, y.l);
  r.h = sel3(q, x.h, y.h);
  r.u = q ? x.u : y.u;
  r.v = q ? x.v : y.v;
  return r;
}

__device__ inline float plane_f(const float* pl, V3 p) { return dot(v3(pl[0], pl[1], pl[2]), p) + pl[3]; }

// ViewPlane::at_least_partially_visible, scene/mod.rs:641-660.
__device__ inline bool part_visible(const float* pl, V3 a, V3 b, V3 c) {
  float fa = plane_f(pl, a), fb = plane_f(pl, b), fc = plane_f(pl, c);
  return !(fa <= 0.0f && fb <= 0.0f && fc <= 0.0f);
}

// ViewPlane::clip, scene/mod.rs:662-746.  First output (o0,o1,o2), second
// output (p0,p1,p2); returns the count.
template <class V>
__device__ inline int clip_plane(const float* pl, V a, V b, V c, V& o0, V& o1, V& o2, V& p0, V& p1, V& p2) {
  float fa = plane_f(pl, a.p), fb = plane_f(pl, b.p), fc = plane_f(pl, c.p);
  if (fa > 0.0f && fb > 0.0f && fc > 0.0f) {
    o0 = a; o1 = b; o2 = c;
    return 1;
  }
  if (fa <= 0.0f && fb <= 0.0f && fc <= 0.0f) return 0;
  // rotate so that c is the vertex alone on its side: r1 (a,b,c) <- (c,a,b),
  // r2 (a,b,c) <- (b,c,a)
  const bool r1 = fa * fc >= 0.0f;
  const bool r2 = !r1 && (fb * fc >= 0.0f);
  const V A = selv(r1, c, selv(r2, b, a));
  const V B = selv(r1, a, selv(r2, c, b));
  const V C = selv(r1, b, selv(r2, a, c));
  fc = r1 ? fb : (r2 ? fa : fc);
  a = A;
  b = B;
  c = C;
  const V3 n = v3(pl[0], pl[1], pl[2]);
  const float ta = plane_f(pl, a.p) / dot(n, sub(a.p, c.p)) - kEps;
  const V na = lerpv(a, c, ta);
  const float tb = plane_f(pl, b.p) / dot(n, sub(b.p, c.p)) - kEps;
  const V nb = lerpv(b, c, tb);
  // one vertex outside (f_c <= 0): [a, A', B'] and [a, b, B']; else [c, A', B']
  const bool two = fc <= 0.0f;
  o0 = selv(two, a, c);
  o1 = na;
  o2 = nb;
  p0 = a;
  p1 = b;
  p2 = nb;
  return two ? 2 : 1;
}

// Back-face test (scene/mod.rs:1016-1020) and Triangle::clip_against_planes
// (43-90): lateral trivial reject, then near and far full clipping.  Calls
// emit(k, v0, v1, v2) for each output in order; returns the count.
template <class V, class Emit>
__device__ inline int cull_and_clip(const FrameParamsPod& fr, const V& a, const V& b, const V& c, bool cull,
                                    Emit emit) {
  if (cull) {  // the transparent pass does not cull (scene/mod.rs:1194-1203)
    const V3 cam = v3(fr.cam[0], fr.cam[1], fr.cam[2]);
    const V3 nrm = cross(sub(b.p, a.p), sub(c.p, b.p));                             // Triangle::calc_normal
    const V3 ctr = divs(add(add(add(v3(0.0f, 0.0f, 0.0f), a.p), b.p), c.p), 3.0f);  // get_center
    if (dot(sub(cam, ctr), nrm) <= 0.0f) return 0;
  }
  if (!(part_visible(fr.planes[2], a.p, b.p, c.p) && part_visible(fr.planes[3], a.p, b.p, c.p) &&
        part_visible(fr.planes[4], a.p, b.p, c.p) && part_visible(fr.planes[5], a.p, b.p, c.p)))
    return 0;
  V n0, n1, n2, m0, m1, m2;
  const int nn = clip_plane(fr.planes[0], a, b, c, n0, n1, n2, m0, m1, m2);
  int cnt = 0;
  if (nn >= 1) {
    V f0, f1, f2, g0, g1, g2;
    const int nf = clip_plane(fr.planes[1], n0, n1, n2, f0, f1, f2, g0, g1, g2);
    if (nf >= 1) emit(cnt++, f0, f1, f2);
    if (nf >= 2) emit(cnt++, g0, g1, g2);
  }
  if (nn >= 2) {
    V f0, f1, f2, g0, g1, g2;
    const int nf = clip_plane(fr.planes[1], m0, m1, m2, f0, f1, f2, g0, g1, g2);
    if (nf >= 1) emit(cnt++, f0, f1, f2);
    if (nf >= 2) emit(cnt++, g0, g1, g2);
  }
  return cnt;
}

// clip_plane's count alone.
__device__ inline int clip_count(const float* pl, V3 a, V3 b, V3 c) {
  const float fa = plane_f(pl, a), fb = plane_f(pl, b), fc = plane_f(pl, c);
  if (fa > 0.0f && fb > 0.0f && fc > 0.0f) return 1;
  if (fa <= 0.0f && fb <= 0.0f && fc <= 0.0f) return 0;
  const bool r1 = fa * fc >= 0.0f;
  const bool r2 = !r1 && (fb * fc >= 0.0f);
  return (r1 ? fb : (r2 ? fa : fc)) <= 0.0f ? 2 : 1;
}

// One output of clip_plane (the second: of a triangle with two), in place.
__device__ inline void clip_select(const float* pl, FV& a, FV& b, FV& c, bool second) {
  FV o0, o1, o2, p0, p1, p2;
  (void)clip_plane(pl, a, b, c, o0, o1, o2, p0, p1, p2);
  a = selv(second, p0, o0);
  b = selv(second, p1, o1);
  c = selv(second, p2, o2);
}

// Output k of cull_and_clip, in place, of a triangle that has more than k.
// The first near output's far count says which of the two near outputs it
// comes from; the attributes then go through the two cuts once.
__device__ inline void clip_output(const FrameParamsPod& fr, FV& a, FV& b, FV& c, uint32_t k) {
  const PV pa{a.p}, pb{b.p}, pc{c.p};
  PV n0, n1, n2, m0, m1, m2;
  (void)clip_plane(fr.planes[0], pa, pb, pc, n0, n1, n2, m0, m1, m2);
  const uint32_t nf = (uint32_t)clip_count(fr.planes[1], n0.p, n1.p, n2.p);
  const bool from_second = k >= nf;
  clip_select(fr.planes[0], a, b, c, from_second);
  clip_select(fr.planes[1], a, b, c, (from_second ? k - nf : k) == 1u);
}

// ====================================================================== setup
// Rectangle::from_coords + Rectangle::clip along one axis (canvas.rs:315-350,
// 646-658).
__device__ inline void rect_axis(uint64_t a0, uint64_t a1, uint64_t smax, uint32_t* lo, uint32_t* hi) {
  uint64_t mn = a0 < a1 ? a0 : a1, mx = a0 < a1 ? a1 : a0;
  mx = mx < smax ? mx : smax;
  if (mn > mx) { mn = 0; mx = 0; }
  *lo = (uint32_t)mn;
  *hi = (uint32_t)mx;
}

// Projection (scene/mod.rs:1047-1058: Matrix4 * Vec4 then as_vec2()/w),
// snapping (canvas.rs:585-587, 896-904), edge constants, normalizers,
// tie-break products (660-666) and the scan rectangle (640-658).  Writes the
// SetupRec and ShadeRec of one clipped triangle with 16-byte stores.
__device__ inline void make_setup(const FrameParamsPod& fr, const FV& A, const FV& B, const FV& C, uint32_t material,
                                  const DevMaterial& mat, uint32_t view, uint32_t group, uint4 (&ro)[6],
                                  uint4 (&so)[9], SetupRec& rec) {
  const float* M = fr.M;
  float X[3], Y[3];
  const V3 P[3] = {A.p, B.p, C.p};
#pragma unroll
  for (int k = 0; k < 3; k++) {
    float o0 = 0.0f + M[0] * P[k].x;
    o0 = o0 + M[1] * P[k].y;
    o0 = o0 + M[2] * P[k].z;
    o0 = o0 + M[3] * 1.0f;
    float o1 = 0.0f + M[4] * P[k].x;
    o1 = o1 + M[5] * P[k].y;
    o1 = o1 + M[6] * P[k].z;
    o1 = o1 + M[7] * 1.0f;
    float o3 = 0.0f + M[12] * P[k].x;
    o3 = o3 + M[13] * P[k].y;
    o3 = o3 + M[14] * P[k].z;
    o3 = o3 + M[15] * 1.0f;
    const float sx = o0 / o3, sy = o1 / o3;
    X[k] = floorf((sx + (-fr.off_x)) + 0.5f);
    Y[k] = floorf((sy + (-fr.off_y)) + 0.5f);
  }
  // f_bc (alpha), f_ca (beta), f_ab (gamma)
  const float ea[4] = {Y[1] - Y[2], X[2] - X[1], X[1] * Y[2], X[2] * Y[1]};
  const float eb[4] = {Y[2] - Y[0], X[0] - X[2], X[2] * Y[0], X[0] * Y[2]};
  const float eg[4] = {Y[0] - Y[1], X[1] - X[0], X[0] * Y[1], X[1] * Y[0]};
  const float fa = edge_eval(ea, X[0], Y[0]);
  const float fb = edge_eval(eb, X[1], Y[1]);
  const float fg = edge_eval(eg, X[2], Y[2]);
  const float oa = edge_eval(ea, -1.0f, -1.0f);
  const float ob = edge_eval(eb, -1.0f, -1.0f);
  const float og = edge_eval(eg, -1.0f, -1.0f);
  uint32_t flags = 0;
  if (fa * oa > 0.0f) flags |= kTieA;
  if (fb * ob > 0.0f) flags |= kTieB;
  if (fg * og > 0.0f) flags |= kTieG;
  // bbox: min/max closures (NaN skipped), `as usize`, clipped to the screen
  float mnx = INFINITY, mny = INFINITY, mxx = -INFINITY, mxy = -INFINITY;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    if (X[k] < mnx) mnx = X[k];
    if (Y[k] < mny) mny = Y[k];
    if (X[k] > mxx) mxx = X[k];
    if (Y[k] > mxy) mxy = Y[k];
  }
  uint32_t x0, x1, y0, y1;
  rect_axis(f2usize(mnx), f2usize(mxx), (uint64_t)fr.W - 1u, &x0, &x1);
  rect_axis(f2usize(mny), f2usize(mxy), (uint64_t)fr.H - 1u, &y0, &y1);
  const bool fin = isfinite(fa) && isfinite(fb) && isfinite(fg);
  if (fin && fa != 0.0f && fb != 0.0f && fg != 0.0f) flags |= kFast;
  // (0) A FAST triangle whose scan rectangle is at most 3x3 pixels and holds
  // no covered pixel: the raster's own test (covered_fast at each pixel of
  // the rectangle) settled here, where the triangle is still in registers.
  if ((flags & kFast) && x1 - x0 <= 2u && y1 - y0 <= 2u) {
    bool any = false;
#pragma unroll
    for (uint32_t k = 0; k < 9u; k++) {
      const uint32_t px = x0 + k % 3u, py = y0 + k / 3u;
      const float xf = (float)px, yf = (float)py;
      const bool cov = covered_fast(edge_eval(ea, xf, yf), fa, flags & kTieA) &&
                       covered_fast(edge_eval(eb, xf, yf), fb, flags & kTieB) &&
                       covered_fast(edge_eval(eg, xf, yf), fg, flags & kTieG);
      any |= cov && px <= x1 && py <= y1;
    }
    if (!any) flags |= kDrop;
  }
  // Exact drops.  (1) A NaN normalizer makes that barycentric NaN at every
  // pixel, which fails `>= 0`.  (2) If all three normalizers are +0 and every
  // edge evaluation over the scan rectangle and the vertices is exact (all
  // partial sums below 2^24), the three edge values sum to 0 at every pixel;
  // coverage would need all three > 0 (x/+0 = +inf), so no pixel is covered.
  if (isnan(fa) || isnan(fb) || isnan(fg)) flags |= kDrop;
  // `exact`: every edge evaluation at |x|,|y| <= R (the vertices and the scan
  // rectangle) has all partial sums below 2^24 in magnitude, so with integer
  // operands each one is exact and e_bc + e_ca + e_ab = f_alpha = f_beta =
  // f_gama (twice the signed area) at every pixel.  S = |A|R + |B|R + |C| +
  // |D| bounds every partial sum; its float evaluation (4 roundings to
  // nearest) is at least S (1 - 2^-24)^4, so S_f < 16777000 gives S < 2^24.
  // (A triangle this leaves out is only handled by the general paths.)
  float R = (float)(x1 > y1 ? x1 : y1);
#pragma unroll
  for (int k = 0; k < 3; k++) R = fmaxf(fmaxf(R, fabsf(X[k])), fabsf(Y[k]));
  auto exact_edge = [R](const float e[4]) {
    const float S = ((fabsf(e[0]) * R + fabsf(e[1]) * R) + fabsf(e[2])) + fabsf(e[3]);
    return S < 16777000.0f;
  };
  const bool exact = isfinite(R) && exact_edge(ea) && exact_edge(eb) && exact_edge(eg);
  if (exact && __float_as_uint(fa) == 0u && __float_as_uint(fb) == 0u && __float_as_uint(fg) == 0u) flags |= kDrop;
  // Texture-index safety: no covered pixel reads outside its maps.  With `exact`
  // its weights are e_i / f >= 0 and sum to 1, so the interpolated u lies within
  // the vertices' range and the roundings of the weights, products and sums,
  // ((1 + 2^-24)^4 - 1) sum |u_i| e_i / f <= 2.4e-7 K with K >= every |u_i|.
  // get_rgb_slice (scene/mod.rs:154-168) takes a negative coordinate for 0.  Its
  // row floor(v (h - 1)) from the bottom exists while v <= 1 + 1 / (h - 1) -
  // 1.2e-7, and its texel floor(u (w - 1)) may run on into the r rows below,
  // r >= floor(v (h - 1)) - 1 (a row for the roundings): u (w - 1) < w (1 + r).
  // (Records that are not safe are visited one at a time with every lane's
  // texture index checked.  While only [0, 1] counted as safe, meshes with
  // coordinates from -0.5 to 0.5 took 206 us for 500k triangles at 1080p and 365
  // for a 150k soup at 720p; now 123 and 161.)
  auto in_map = [&](int32_t w, int32_t h) {
    const float mu = (float)w - 1.0f, mv = (float)h - 1.0f;
    const float eu = 2.4e-7f * ((fabsf(A.u) + fabsf(B.u)) + fabsf(C.u)) + 1.3e-7f;  // NaN and infinite ones fail below
    const float ev = 2.4e-7f * ((fabsf(A.v) + fabsf(B.v)) + fabsf(C.v)) + 1.3e-7f;
    const float u1 = fmaxf(fmaxf(A.u, B.u), C.u), v1 = fmaxf(fmaxf(A.v, B.v), C.v), v0 = fminf(fminf(A.v, B.v), C.v);
    const float rows = fmaxf(floorf((v0 - ev) * mv) - 1.0f, 0.0f);
    return ((v1 - 1.0f) + ev) * mv < 0.999f && ((u1 - 1.0f) + eu) * mu < 0.999f * (1.0f + rows * (float)w);
  };
  if ((flags & kFast) && exact && max(max(mat.kd_w, mat.kd_h), max(mat.ka_w, mat.ka_h)) <= (1 << 20) &&
      in_map(mat.kd_w, mat.kd_h) && (mat.ka_one || in_map(mat.ka_w, mat.ka_h)))
    flags |= kUvSafe;
  // Depth lower bound for early rejection.  For a UV-safe triangle (exact
  // edge arithmetic) a covered pixel has alpha + beta + gama >= 1 - 2^-24 with
  // non-negative weights, so with non-negative vertex depths its depth is at
  // least d_min * (1 - 2^-24)^4 > zlb = RN(d_min * (1 - 2^-20)).  A fragment
  // may be skipped only when zlb is strictly above a depth already recorded at
  // its pixel, and only on UV-safe triangles (whose texture reads cannot fail).
  float zlb = -INFINITY;
  {
    const float dmin = fminf(fminf(A.d, B.d), C.d);
    if ((flags & kUvSafe) && A.d >= 0.0f && B.d >= 0.0f && C.d >= 0.0f && dmin >= 1e-30f)
      zlb = dmin * (1.0f - 9.5367431640625e-07f);
    if ((flags & kUvSafe) && zlb >= fr.clear_depth) flags |= kDrop;  // no pixel can pass `<` the clear depth
  }
#pragma unroll
  for (int k = 0; k < 4; k++) {
    rec.ea[k] = ea[k];
    rec.eb[k] = eb[k];
    rec.eg[k] = eg[k];
  }
  rec.f[0] = fa; rec.f[1] = fb; rec.f[2] = fg;
  // with `exact` the three normalizers are one value (twice the signed area),
  // an integer below 2^24: its reciprocal stands for three divisions a pixel
  rec.f[3] = (flags & kUvSafe) ? 1.0f / fa : 0.0f;
  rec.d[0] = A.d; rec.d[1] = B.d; rec.d[2] = C.d; rec.d[3] = zlb;
  rec.rx = x0 | (x1 << 16);
  rec.ry = y0 | (y1 << 16);
  rec.flags = flags;
  rec.view = view;
  const uint4* ri = reinterpret_cast<const uint4*>(&rec);
#pragma unroll
  for (int k = 0; k < 6; k++) ro[k] = ri[k];
  // shading attributes: uv[6], material, pad, n[9], l[9], h[9], pad
  auto u4 = [](float a, float b, float c, float d) {
    return make_uint4(__float_as_uint(a), __float_as_uint(b), __float_as_uint(c), __float_as_uint(d));
  };
  so[0] = u4(A.u, A.v, B.u, B.v);
  so[1] = u4(C.u, C.v, __uint_as_float(material), __uint_as_float(group));
  so[2] = u4(A.n.x, A.n.y, A.n.z, B.n.x);
  so[3] = u4(B.n.y, B.n.z, C.n.x, C.n.y);
  so[4] = u4(C.n.z, A.l.x, A.l.y, A.l.z);
  so[5] = u4(B.l.x, B.l.y, B.l.z, C.l.x);
  so[6] = u4(C.l.y, C.l.z, A.h.x, A.h.y);
  so[7] = u4(A.h.z, B.h.x, B.h.y, B.h.z);
  so[8] = u4(C.h.x, C.h.y, C.h.z, 0.0f);
}

// Stores one N-uint4 record per lane at dst[idx] (record units) for the lanes
// with ok and not skip (skip: a record nothing will read, whose id is still
// taken).  When the ok lanes are a prefix of the wave with consecutive idx (a
// dense run of output ids), the records go through the wave's LDS area
// stage[64 * N] and out in coalesced 16-byte lanes, leaving the skipped
// records' memory untouched; else each lane stores its own.  Every lane of the
// wave must call it.
template <int N>
__device__ inline void wave_store(uint4* stage, const uint4 (&v)[N], bool ok, uint32_t idx, uint4* dst,
                                  bool skip = false) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint64_t m = __ballot(ok);
  const uint64_t sm = __ballot(ok && skip);
  if (m == sm) return;
  const uint32_t cnt = (uint32_t)__popcll(m);
  const uint32_t first = (uint32_t)__builtin_amdgcn_readfirstlane((int)idx);
  const bool prefix = m == (cnt == 64u ? ~0ull : ((1ull << cnt) - 1ull));
  if (prefix && __ballot(ok && idx != first + lane) == 0ull) {
    if (ok && !skip) {
#pragma unroll
      for (int q = 0; q < N; q++) stage[lane * N + q] = v[q];
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    uint4* out = dst + (uint64_t)first * N;
    for (uint32_t k = lane; k < cnt * N; k += 64u)
      if (!((sm >> (k / (uint32_t)N)) & 1ull)) out[k] = stage[k];
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  } else if (ok && !skip) {
#pragma unroll
    for (int q = 0; q < N; q++) dst[(uint64_t)idx * N + q] = v[q];
  }
}

// =================================================================== binning
// Conservative tile sets of a clipped triangle.  For a FAST triangle every
// edge value at an integer pixel is e = fl(fl(fl(fl(Ax)+fl(By))+C)-D) with
// |e - (Ax+By+C-D)| <= 4.01 u S, S = |A|x + |B|y + |C| + |D|; a pixel can only
// be covered when sign(f) * e >= 0 on all three edges.  Each edge's
// exact-arithmetic function, widened by that bound (plus 1), therefore gives
// a superset of the tiles holding covered pixels (tile_may_cover).  Other
// triangles, and those within one tile, are binned to every tile of their
// scan rectangle.
struct Spans {
  int cx0, cx1, cy0, cy1;
  bool exact;
  float fa[3], fb[3], fk[3], fm[3];  // per-tile corner test (tile_may_cover)
};
// Bounds and the per-tile test's constants.  The test evaluates
// G_f = fl(fl(fl(a xc) + fl(b yc)) + fl(s (C - D))) at the tile corner
// (xc, yc) maximising the edge's exact function G = a x + b y + s (C - D).
// With M = |A| (x1 + TS) + |B| (y1 + TS) + |C| + |D|, which bounds the
// magnitudes at every corner of a tile of the rectangle, |G_f - G| <= 3.02 u M
// (u = 2^-24).  A covered pixel p of the tile has G >= g(p) >= -4.01 u M (the
// pixel evaluation bound above), so G_f >= -7.03 u M; rejecting only when
// G_f < -(1 + 9 u M) keeps every tile with a covered pixel.
__device__ inline void spans_init(const SetupRec& r, int TS, Spans& g) {
  const uint32_t x0 = r.rx & 0xFFFFu, x1 = r.rx >> 16, y0 = r.ry & 0xFFFFu, y1 = r.ry >> 16;
  g.cx0 = (int)(x0 / TS); g.cx1 = (int)(x1 / TS);
  g.cy0 = (int)(y0 / TS); g.cy1 = (int)(y1 / TS);
  g.exact = (r.flags & kFast) != 0;
  if (g.cx0 == g.cx1 && g.cy0 == g.cy1) {  // one tile: binned there without edge tests
    g.exact = false;
    return;
  }
  const float* es[3] = {r.ea, r.eb, r.eg};
  const float xm = (float)x1 + (float)TS, ym = (float)y1 + (float)TS;
#pragma unroll
  for (int i = 0; i < 3; i++) {
    const float A = es[i][0], B = es[i][1], C = es[i][2], D = es[i][3];
    const float s = r.f[i] > 0.0f ? 1.0f : -1.0f;
    const float M = ((fabsf(A) * xm + fabsf(B) * ym) + fabsf(C)) + fabsf(D);
    g.fa[i] = s * A;
    g.fb[i] = s * B;
    g.fk[i] = s * (C - D);
    g.fm[i] = 1.0f + 5.4e-7f * M;  // 1 + 9 u M, rounded up
    if (!isfinite(M)) g.exact = false;
  }
}

// Work split: a triangle whose tile range is more than kWideSpan tiles tall
// or wide is binned by a whole wave (lanes over rows, then over entries); the
// rest by one thread each (at most kWideSpan^2 entries).  The split only
// balances work.
constexpr int kWideSpan = 4;

__device__ inline bool bin_is_wide(const Spans& g) {
  return g.cy1 - g.cy0 + 1 > kWideSpan || g.cx1 - g.cx0 + 1 > kWideSpan;
}

__device__ inline uint64_t lanemask_lt_u64(int lane) { return lane == 0 ? 0ull : (~0ull >> (64 - lane)); }

// The tiles (tx0..tx1, ty0..ty1) of the box may hold a covered pixel: every
// edge's function, widened by fm (see spans_init), reaches 0 at their corner
// maximising it.
__device__ inline bool tiles_may_cover(const Spans& g, int TS, int tx0, int tx1, int ty0, int ty1) {
  if (!g.exact) return true;
  const float xa = (float)(tx0 * TS), xb = (float)(tx1 * TS + TS - 1);
  const float ya = (float)(ty0 * TS), yb = (float)(ty1 * TS + TS - 1);
#pragma unroll
  for (int i = 0; i < 3; i++) {
    const float v = (g.fa[i] * (g.fa[i] > 0.0f ? xb : xa) + g.fb[i] * (g.fb[i] > 0.0f ? yb : ya)) + g.fk[i];
    if (v < -g.fm[i]) return false;
  }
  return true;
}
// tile_may_cover holds for every tile of the box: each edge's function, as it
// is evaluated (rounding keeps its order), is least on the tile farthest back.
__device__ inline bool tiles_all_may_cover(const Spans& g, int TS, int tx0, int tx1, int ty0, int ty1) {
  if (!g.exact) return true;
  const float xa = (float)(tx1 * TS), xb = (float)(tx0 * TS + TS - 1);
  const float ya = (float)(ty1 * TS), yb = (float)(ty0 * TS + TS - 1);
#pragma unroll
  for (int i = 0; i < 3; i++) {
    const float v = (g.fa[i] * (g.fa[i] > 0.0f ? xb : xa) + g.fb[i] * (g.fb[i] > 0.0f ? yb : ya)) + g.fk[i];
    if (v < -g.fm[i]) return false;
  }
  return true;
}
__device__ inline bool tile_may_cover(const Spans& g, int TS, int tx, int ty) {
  return tiles_may_cover(g, TS, tx, tx, ty, ty);
}

// Calls f(e, ty, tx) for every tile of a triangle that is not wide (at most
// kWideSpan x kWideSpan tiles in its rectangle), e numbering the tiles in
// row-major order; returns the tile count.
template <class F>
__device__ inline uint32_t thread_tiles(const Spans& g, int TS, F f) {
  uint32_t e = 0;
  for (int ty = g.cy0; ty <= g.cy1; ty++)
    for (int tx = g.cx0; tx <= g.cx1; tx++)
      if (tile_may_cover(g, TS, tx, ty)) f(e++, ty, tx);
  return e;
}

// Wave version, for a wide triangle (uniform arguments).  A box of at most
// kBoxTiles tiles: lanes take its tiles and test each as the narrow triangles'
// are.  A larger one: lanes take its blocks of 8x8 tiles, and the tiles of a
// block that may hold a covered pixel are tested at once.  f(e, tx, ty) with e
// numbering the tiles; returns the tile count.  part, parts: a share of the box's
// blocks, taken in turn by the parts of a workgroup's waves, numbered within the
// share.  (64 consecutive blocks a wave left a box of up to 4096 tiles to one
// wave.)  WHOLE: the tiles of a block that no edge leaves a tile of out are not
// tested again.  The kernels with a wave per triangle take it (a room of 20
// triangles on 8160 tiles, submission order: 187 -> 174 us); in those that share
// the boxes out it cost frames of small boxes 1 us and gave nothing.
constexpr int kBoxTiles = 256;
template <bool WHOLE = false, class F>
__device__ inline uint32_t wave_tiles(const Spans& g, int TS, int part, int parts, F f) {
  const int lane = threadIdx.x & 63;
  uint32_t o = 0;
  const int nx = g.cx1 - g.cx0 + 1, n = nx * (g.cy1 - g.cy0 + 1);
  auto tile = [&](bool on, int tx, int ty, bool sure) {
    if (!WHOLE || !sure) on = on && tile_may_cover(g, TS, tx, ty);
    const uint64_t m = __ballot(on);
    if (on) f(o + (uint32_t)__popcll(m & lanemask_lt_u64(lane)), tx, ty);
    o += (uint32_t)__popcll(m);
  };
  const bool large = n > kBoxTiles;
  const int bx = large ? (nx + 7) >> 3 : nx, nb = large ? bx * ((g.cy1 - g.cy0 + 8) >> 3) : n;
  const float inv = 1.0f / (float)bx;
  for (int t0 = part; t0 < nb; t0 += 64 * parts) {
    const int t = t0 + parts * lane;
    // t / bx: the quotient is off by at most one (t < 2^20), and exact for t < 512
    int dy = (int)(((float)t + 0.5f) * inv);
    if (large) {
      dy -= dy * bx > t ? 1 : 0;
      dy += (dy + 1) * bx <= t ? 1 : 0;
      const int x0 = g.cx0 + 8 * (t - dy * bx), y0 = g.cy0 + 8 * dy;
      const int x1 = min(x0 + 7, g.cx1), y1 = min(y0 + 7, g.cy1);
      const bool may = t < nb && tiles_may_cover(g, TS, x0, x1, y0, y1);
      const uint64_t every = WHOLE ? __ballot(may && tiles_all_may_cover(g, TS, x0, x1, y0, y1)) : 0ull;
      for (uint64_t m = __ballot(may); m; m &= m - 1) {
        const int b = (int)__builtin_ctzll(m);
        const int tx = __builtin_amdgcn_readlane(x0, b) + (lane & 7), ty = __builtin_amdgcn_readlane(y0, b) + (lane >> 3);
        tile(tx <= g.cx1 && ty <= g.cy1, tx, ty, ((every >> b) & 1ull) != 0ull);
      }
    } else {
      tile(t < nb, g.cx0 + (t - dy * bx), g.cy0 + dy, false);
    }
  }
  return o;
}

// The constants of a wide triangle's visit.
struct WideTri {
  Spans g;  // (without edge tests: exact, and every margin infinite)
  uint32_t key0, ntx, id, dk;
};
__device__ inline WideTri wide_tri(uint32_t id, const SetupRec* __restrict__ setup, const DevView* __restrict__ views,
                                   const uint8_t* __restrict__ dkey, int TS) {
  WideTri w;
  const SetupRec r = setup[id];
  w.id = id;
  w.dk = dkey ? dkey[id] : 0u;
  spans_init(r, TS, w.g);
  const DevView& vw = views[r.view];
  w.ntx = vw.ntx;
  w.key0 = vw.tile_base + (uint32_t)w.g.cy0 * vw.ntx + (uint32_t)w.g.cx0;
#pragma unroll
  for (int e = 0; e < 3; e++) {
    if (!w.g.exact) w.g.fa[e] = w.g.fb[e] = w.g.fk[e] = 0.0f;
    w.g.fm[e] = w.g.exact ? w.g.fm[e] : INFINITY;
  }
  w.g.exact = true;
  return w;
}

// Triangles of larger boxes that the waves of a block share out: a wave per
// kShareBlocks of a box's 8x8-tile blocks, the next triangle's on the waves
// after them.  (2, 4, 8 and 16 blocks a wave, all waves on every box: a room of
// 20 triangles on 2040 tiles of 32x32 pixels 108, 106, 104, 105, 110 us, of 68 on
// 2040 of 16x16 77, 74, 73, 75, 81.)
constexpr uint32_t kLargeBuf = 64, kShareBlocks = 8;
struct LargeBuf {
  uint32_t n;
  WideTri t[kLargeBuf];
};

// The wide triangles list[w], list[w + step], ... (below n) of one of a block's
// NW waves: f(tile key, triangle, its byte of dkey if given) for each of their
// tiles.  Each lane first fetches and prepares one of the wave's next 64
// triangles, so that the chain of dependent loads (id, record, view) is paid
// once for all of them and the visits take their constants from registers; a
// wave per triangle paid some 2 us of latency for each (k_bin_small of a
// 2312-triangle frame of 3600 tiles: 105 -> 38 us).  Triangles of larger boxes
// wait in the block's LDS until every wave is done with the others, and then
// the waves share them out.  Every wave of the block calls it; large.n is 0
// before, after a barrier.
template <int NW, class F>
__device__ inline void wave_wide_tiles(const uint32_t* __restrict__ list, uint32_t w, uint32_t step, uint32_t n,
                                       const SetupRec* __restrict__ setup, const DevView* __restrict__ views,
                                       const uint8_t* __restrict__ dkey, int TS, LargeBuf& large, F f) {
  if (n == 0u) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  bool shared = false;  // visiting the block's large triangles
  for (uint64_t w0 = w;; w0 += 64ull * step) {
    WideTri q{};
    bool on;
    uint32_t part = 0, parts = 0;
    if (w0 < n) {
      const uint64_t at = w0 + (uint64_t)step * (uint32_t)lane;
      on = at < n;
      if (on) {
        q = wide_tri(list[at], setup, views, dkey, TS);
        if ((q.g.cx1 - q.g.cx0 + 1) * (q.g.cy1 - q.g.cy0 + 1) > kBoxTiles) {
          const uint32_t p = atomicAdd(&large.n, 1u);
          if (p < kLargeBuf) {
            large.t[p] = q;
            on = false;
          }
        }
      }
    } else {
      __syncthreads();
      const uint32_t n_large = min(large.n, kLargeBuf);
      if (n_large == 0u) return;
      shared = true;
      if ((uint32_t)lane < n_large) {
        q = large.t[lane];
        const uint32_t nb = (uint32_t)(((q.g.cx1 - q.g.cx0 + 8) >> 3) * ((q.g.cy1 - q.g.cy0 + 8) >> 3));
        parts = min((nb + kShareBlocks - 1u) / kShareBlocks, (uint32_t)NW);
      }
      uint32_t x = parts;  // -> the parts of the triangles up to this one
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
      }
      part = ((uint32_t)wave + parts - x) % (uint32_t)NW;
      on = part < parts;
    }
    auto bi = [](auto v, int b) { return (decltype(v))__builtin_amdgcn_readlane((int)v, b); };
    auto bf = [](float v, int b) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), b)); };
    for (uint64_t m = __ballot(on); m; m &= m - 1) {
      const int b = (int)__builtin_ctzll(m);
      Spans u;
      u.exact = true;
      u.cx0 = bi(q.g.cx0, b);
      u.cx1 = bi(q.g.cx1, b);
      u.cy0 = bi(q.g.cy0, b);
      u.cy1 = bi(q.g.cy1, b);
#pragma unroll
      for (int e = 0; e < 3; e++) {
        u.fa[e] = bf(q.g.fa[e], b);
        u.fb[e] = bf(q.g.fb[e], b);
        u.fk[e] = bf(q.g.fk[e], b);
        u.fm[e] = bf(q.g.fm[e], b);
      }
      const uint32_t id = bi(q.id, b), dk = bi(q.dk, b), ntx = bi(q.ntx, b), key0 = bi(q.key0, b);
      wave_tiles(u, TS, (int)bi(part, b), shared ? (int)bi(parts, b) : 1, [&](uint32_t, int tx, int ty) {
        f(key0 + (uint32_t)(ty - u.cy0) * ntx + (uint32_t)(tx - u.cx0), id, dk);
      });
    }
    if (shared) return;
  }
}

// Ordered bins keep, per clipped triangle, a bin box: x the tile key of the
// corner (cx0, cy0) of its tile box, y its tiles as bits 4 * (ty - cy0) +
// (tx - cx0) (low 16 bits, within the at most 4 x 4 box; none for a dropped
// triangle) and the view's tiles per row (high 16 bits), so that the pair
// kernels find every tile key from these 8 bytes alone; x = kWideBox for a
// wide triangle, whose tiles a wave counts and emits later.  They live in the
// byte buffer after one byte per triangle (12 bytes per clipped triangle in all).
constexpr uint32_t kWideBox = 0xFFFFFFFFu;
__device__ __host__ inline uint2* bin_boxes(void* big, uint32_t cap_tri) {
  return reinterpret_cast<uint2*>(reinterpret_cast<uint8_t*>(big) + ((cap_tri + 15u) & ~15u));
}

// Near-first binning order: an 8-bit key of the nearest vertex depth, 16
// steps per octave above depth_base (the float bits of half the near-plane
// distance), so 16 octaves of depth; monotonic for positive depths, others
// sort first.  Only the speed of the raster depends on it.
constexpr int kDepthKeyBits = 8;
__device__ inline uint32_t depth_order_key(const SetupRec& r, uint32_t depth_base) {
  const float d = fminf(fminf(r.d[0], r.d[1]), r.d[2]);
  const uint32_t b = __float_as_uint(d);
  if (!(d > 0.0f) || b <= depth_base) return 0u;
  return min((b - depth_base) >> 19, (1u << kDepthKeyBits) - 1u);
}

// How an emit prepares the binning: nothing (unordered bins), submission
// order (flag byte, bin box, tile count per triangle) or near first (depth
// key byte, bin box, and the list of wide triangles).
constexpr int kBinNone = 0, kBinSubmit = 1, kBinNear = 2;

// One clipped triangle of view vw: its byte (submission order: 0 binned here,
// 1 wide, 2 dropped; near first: its depth key), its bin box and, for
// submission order, its tile count when it is not wide.  (A dropped triangle
// has no tiles, and its records are not stored.)  Returns whether it is wide.
template <int BIN>
__device__ inline bool bin_count_one(const SetupRec& r, int TS, uint32_t i, const DevView& vw,
                                     uint32_t* __restrict__ bincnt, uint8_t* __restrict__ wflag,
                                     uint2* __restrict__ boxes) {
  uint32_t c = 0, mask = 0, key0 = 0;
  bool is_wide = false;
  if (!(r.flags & kDrop)) {
    Spans g;
    spans_init(r, TS, g);
    is_wide = bin_is_wide(g);
    key0 = vw.tile_base + (uint32_t)g.cy0 * vw.ntx + (uint32_t)g.cx0;
    if (!is_wide)
      c = thread_tiles(g, TS, [&](uint32_t, int ty, int tx) { mask |= 1u << (4 * (ty - g.cy0) + (tx - g.cx0)); });
  }
  boxes[i] = make_uint2(is_wide ? kWideBox : key0, mask | (vw.ntx << 16));
  if constexpr (BIN == kBinNear) {
    wflag[i] = (uint8_t)depth_order_key(r, vw.depth_base);
  } else {
    wflag[i] = is_wide ? 1u : ((r.flags & kDrop) ? 2u : 0u);
    if (!is_wide) bincnt[i] = c;
  }
  return is_wide;
}

// The wide triangles an emit block meets, gathered in LDS and appended to the
// frame's list with one atomic per block (an atomic per wave on that one word
// would serialize a large frame's emits); more than the buffer holds go to
// the list one by one.  The list's order does not matter.
constexpr uint32_t kWideBuf = 512;
struct WideBuf {
  uint32_t n, base;
  uint32_t id[kWideBuf];
};
__device__ inline void wide_push(WideBuf& b, uint32_t i, Status* status, uint32_t* __restrict__ list) {
  const uint32_t p = atomicAdd(&b.n, 1u);
  if (p < kWideBuf) b.id[p] = i;
  else list[atomicAdd(&status->n_wide, 1u)] = i;
}
// Every thread of the block calls it, after its last wide_push.
__device__ inline void wide_flush(WideBuf& b, Status* status, uint32_t* __restrict__ list) {
  __syncthreads();
  const uint32_t n = min(b.n, kWideBuf);
  if (n == 0u) return;
  if (threadIdx.x == 0) b.base = atomicAdd(&status->n_wide, n);
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < n; k += blockDim.x) list[b.base + k] = b.id[k];
}

// Calls f(tile key) for every tile of a bin box (none for a wide triangle,
// whose mask is empty).
template <class F>
__device__ inline void box_tiles(uint2 box, F f) {
  const uint32_t ntx = box.y >> 16;
  uint32_t mask = box.y & 0xFFFFu;
  while (mask) {
    const uint32_t b = (uint32_t)__builtin_ctz(mask);
    mask &= mask - 1u;
    f(box.x + (b >> 2) * ntx + (b & 3u));
  }
}

// The pairs of a triangle that is not wide from its bin box, its e-th tile at
// position o + e (tiles in the order of the count pass).
__device__ inline void emit_box_pairs(uint2 box, uint32_t i, uint32_t o, uint32_t cap_pairs,
                                      uint32_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  box_tiles(box, [&](uint32_t key) {
    if (o < cap_pairs) {
      keys[o] = key;
      vals[o] = i;
    }
    o++;
  });
}

// ================================================================== geometry
// Small single-view frames: at most kSmallBinTris input triangles take one
// workgroup for the geometry lists (k_geom_small), and on few tiles one for the
// binning (k_bin_small, small_bins): a launch each in place of three and four.
//
// The geometry's cost grows with the triangles alone.  Frames, one workgroup ->
// three launches: soups of 300 triangles 55 -> 58 us, of 900 64 -> 66, of 1200 67 ->
// 66, of 2500 88 -> 82; tori of 576 48 -> 53, of 2304 61 -> 60, of 3136 64 -> 59, of
// 6400 74 -> 61; but a frame that no graph replays also saves the host two
// launches (one of 2312 opaque and 19,600 transparent triangles 174 -> 177).
//
// The binning's depends on the wide triangles, which the host does not know.
// One workgroup -> four launches: compact meshes gain long (tori of 2304
// triangles on 300, 1200, 1620 and 2040 tiles 54 -> 62, 60 -> 67, 67 -> 73, 77 -> 78;
// of 6400 on up to 1620 58 -> 64, 61 -> 66, 63 -> 68; of 16,384 67 -> 67, 68 -> 67, 68
// -> 68), soups, a third of which is wide, lose from 1200 on (of 1800 on 1200
// tiles 82 -> 75, of 2500 88 -> 77, of 16,000 209 -> 83), balls of triangles on many
// tiles (of 2500 on 300, 1200, 1620 and 2040 57 -> 64, 68 -> 72, 82 -> 75, 93 -> 80).
// kSmallBinTris keeps what a soup below it loses, at most 11 us, near what a
// mesh above it does, 6.  Beyond kSmallBinTiles what fills the canvas loses (tori
// of 160, 576 and 2304 on 3600 77 -> 71, 89 -> 75, 112 -> 82) unless it is of a few
// triangles (none 36 -> 42, one 46 -> 52, a torus of 24 67 -> 68, soups of 10 and 30
// 55 -> 60, a room of 20 91 -> 90, of 68 90 -> 86).
constexpr uint32_t kSmallBinTris = 2560;  // LDS count bytes: 2.5 KB
constexpr uint32_t kSmallBinTiles = 2048;
constexpr uint32_t kFewBinTris = 32, kFewBinTiles = 4096;  // LDS counters and cursors: 32 KB
inline bool small_bins(uint32_t n_tri_in, uint32_t n_tiles) {
  return n_tiles <= kSmallBinTiles ? n_tri_in <= kSmallBinTris : n_tiles <= kFewBinTiles && n_tri_in <= kFewBinTris;
}

// cnt[t]: clipped-triangle count (bits 0-2, at most 4) | kCntClip when the
// triangle crosses the near or far plane.
constexpr uint32_t kCntMask = 7u, kCntClip = 8u;

__device__ inline bool inside_plane(const float* pl, V3 a, V3 b, V3 c) {
  return plane_f(pl, a) > 0.0f && plane_f(pl, b) > 0.0f && plane_f(pl, c) > 0.0f;
}

// Block-scan word: clipped triangles << 18 | unclipped emitters << 9 |
// clipped emitters (a block has at most 256 * 4 of the first, 256 of each other).
__device__ inline uint32_t pack_geom(uint32_t c, bool clip) {
  return (c << 18) | (c && !clip ? (1u << 9) : 0u) | (c && clip ? 1u : 0u);
}

__global__ __launch_bounds__(256) void k_geom_count(const DevDraw* __restrict__ draws, uint32_t n_draws,
                                                    const DevView* __restrict__ views, uint32_t n_in,
                                                    uint8_t* __restrict__ cnt, uint32_t* __restrict__ blk,
                                                    uint32_t* __restrict__ blk_simple, uint32_t* __restrict__ blk_clip) {
  __shared__ uint32_t s_tmp[4];
  const uint32_t t = blockIdx.x * 256u + threadIdx.x;
  uint32_t c = 0;
  bool clip = false;
  const uint32_t d = wave_find_draw(draws, n_draws, t, t < n_in);
  by_draw(d, t < n_in, [&](uint32_t di) {
    const DevDraw& dr = draws[di];
    const FrameParamsPod& fr = views[dr.view].fr;
    PV a, b, cc;
    tri_positions(dr, t - dr.tri_begin, a.p, b.p, cc.p);
    c = (uint32_t)cull_and_clip(fr, a, b, cc, !(dr.flags & kDrawNoCull), [](int, const PV&, const PV&, const PV&) {});
    // ViewPlane::clip keeps a triangle unchanged exactly when its three
    // vertices are strictly inside the plane (clip_plane's first branch)
    if (c) clip = !(inside_plane(fr.planes[0], a.p, b.p, cc.p) && inside_plane(fr.planes[1], a.p, b.p, cc.p));
    cnt[t] = (uint8_t)(c | (clip ? kCntClip : 0u));
  });
  uint32_t total;
  block_exclusive_scan256(pack_geom(c, clip), s_tmp, &total);
  if (threadIdx.x == 0) {
    blk[blockIdx.x] = total >> 18;
    blk_simple[blockIdx.x] = (total >> 9) & 0x1FFu;
    blk_clip[blockIdx.x] = total & 0x1FFu;
  }
}

// Exclusive scan of three values per thread over a block of 1024 threads,
// packed 22 | 21 | 21 bits into 64 (a block has at most 4096 of the first,
// 1024 of the others); *total gets the three totals, packed alike.
__device__ inline uint64_t block_exclusive_scan1024x3(uint64_t v, uint64_t* s_w /*[16]*/, uint64_t* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint64_t x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint64_t y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) s_w[wave] = x;
  __syncthreads();
  uint64_t before = 0, all = 0;
  for (int w = 0; w < 16; w++) {
    if (w < wave) before += s_w[w];
    all += s_w[w];
  }
  __syncthreads();
  *total = all;
  return before + x - v;
}

// k_geom_count, the scan of its block counts and k_geom_compact for a small
// single-view frame (at most kSmallBinTris input triangles), in one
// workgroup of 1024 threads: the same cnt, the same per-256-triangle output
// offsets in blk, the same status counts and the same two ordered lists,
// without two launches and their gaps.
__global__ __launch_bounds__(1024) void k_geom_small(const DevDraw* __restrict__ draws, uint32_t n_draws,
                                                     const DevView* __restrict__ views, uint32_t n_in,
                                                     uint8_t* __restrict__ cnt, uint32_t* __restrict__ blk,
                                                     Status* __restrict__ status, uint32_t cap_tri,
                                                     uint2* __restrict__ surv) {
  __shared__ uint64_t s_w[16];
  __shared__ uint8_t s_cnt[kSmallBinTris];
  const uint32_t tid = threadIdx.x;
  auto field = [](uint64_t x, int k) { return (uint32_t)((x >> (k == 0 ? 42 : (k == 1 ? 21 : 0))) & 0x1FFFFFu); };
  auto pack = [](uint32_t c, bool clip) {
    return ((uint64_t)c << 42) | ((uint64_t)(c && !clip) << 21) | (uint64_t)(c && clip);
  };
  // counts, output offsets, the unclipped emitters' entries
  uint32_t run_o = 0, run_s = 0, run_c = 0;
  for (uint32_t c0 = 0; c0 < n_in; c0 += 1024u) {
    const uint32_t t = c0 + tid;
    uint32_t c = 0;
    bool clip = false;
    const uint32_t d = wave_find_draw(draws, n_draws, t, t < n_in);
    by_draw(d, t < n_in, [&](uint32_t di) {
      const DevDraw& dr = draws[di];
      const FrameParamsPod& fr = views[dr.view].fr;
      PV a, b, cc;
      tri_positions(dr, t - dr.tri_begin, a.p, b.p, cc.p);
      c = (uint32_t)cull_and_clip(fr, a, b, cc, !(dr.flags & kDrawNoCull),
                                  [](int, const PV&, const PV&, const PV&) {});
      if (c) clip = !(inside_plane(fr.planes[0], a.p, b.p, cc.p) && inside_plane(fr.planes[1], a.p, b.p, cc.p));
      const uint8_t q = (uint8_t)(c | (clip ? kCntClip : 0u));
      cnt[t] = q;
      s_cnt[t] = q;
    });
    uint64_t tot;
    const uint64_t ex = block_exclusive_scan1024x3(pack(c, clip), s_w, &tot);
    const uint32_t first = run_o + field(ex, 0);
    if (t < n_in && (t & 255u) == 0u) blk[t >> 8] = first;
    if (c && !clip) surv[run_s + field(ex, 1)] = make_uint2(t, first);
    run_o += field(tot, 0);
    run_s += field(tot, 1);
    run_c += field(tot, 2);
  }
  // the clipped emitters' entries, after the unclipped ones
  if (run_c) {
    uint32_t r_o = 0, r_c = 0;
    for (uint32_t c0 = 0; c0 < n_in; c0 += 1024u) {
      const uint32_t t = c0 + tid;
      const uint32_t q = t < n_in ? (uint32_t)s_cnt[t] : 0u;
      const uint32_t c = q & kCntMask;
      const bool clip = (q & kCntClip) != 0u;
      uint64_t tot;
      const uint64_t ex = block_exclusive_scan1024x3(pack(c, clip), s_w, &tot);
      if (c && clip) surv[run_s + r_c + field(ex, 2)] = make_uint2(t, r_o + field(ex, 0));
      r_o += field(tot, 0);
      r_c += field(tot, 2);
    }
  }
  if (tid == 0) {
    status->n_out = run_o;
    status->n_simple = run_s;
    status->n_clip = run_c;
    if (run_o > cap_tri) atomicOr(&status->overflow, 1u);
  }
}

// Ordered lists of the input triangles that emit, (triangle, first output
// id): the unclipped ones in surv[0, n_simple), the clipped ones after them.
// A wave per 256-triangle block of counts, ranks by ballots: no barrier, and a
// quarter of the workgroups of a thread per triangle, whose launching bounded
// it (5M triangles: 18 -> 9 us, the 32-view batch: 12 -> 6).
__global__ __launch_bounds__(256) void k_geom_compact(uint32_t n_in, const uint8_t* __restrict__ cnt,
                                                      const uint32_t* __restrict__ blk_off,
                                                      const uint32_t* __restrict__ simple_off,
                                                      const uint32_t* __restrict__ clip_off,
                                                      const Status* __restrict__ status, uint2* __restrict__ surv) {
  const uint32_t b = blockIdx.x * 4u + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t t0 = b * 256u;
  if (t0 >= n_in) return;  // the whole wave
  uint32_t q[4];
#pragma unroll
  for (uint32_t k = 0; k < 4u; k++) {
    const uint32_t t = t0 + 64u * k + (threadIdx.x & 63u);
    q[k] = t < n_in ? (uint32_t)cnt[t] : 0u;
  }
  uint32_t o = blk_off[b], s = simple_off[b], c = status->n_simple + clip_off[b];
  auto below = [](uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
  };
#pragma unroll
  for (uint32_t k = 0; k < 4u; k++) {
    const uint64_t m1 = __ballot(q[k] & 1u), m2 = __ballot(q[k] & 2u), m4 = __ballot(q[k] & 4u);
    const uint64_t mc = __ballot(q[k] & kCntClip);  // set only where the count is not zero
    const uint64_t ms = (m1 | m2 | m4) & ~mc;
    if (q[k] & kCntMask) {
      const uint32_t at = (q[k] & kCntClip) ? c + below(mc) : s + below(ms);
      surv[at] = make_uint2(t0 + 64u * k + (threadIdx.x & 63u), o + below(m1) + 2u * below(m2) + 4u * below(m4));
    }
    o += (uint32_t)(__popcll(m1) + 2 * __popcll(m2) + 4 * __popcll(m4));
    s += (uint32_t)__popcll(ms);
    c += (uint32_t)__popcll(mc);
  }
}

// One output of an emitting input triangle per lane (every lane of the wave
// calls it; lanes without an output with active false): list entry sv, output
// k of the clipper for CLIP, else the triangle itself.  Its records leave
// through the wave's LDS area stage[64 * 9].
template <int BIN>
__device__ __forceinline__ void geom_emit_one(uint2 sv, bool active, bool clip, uint32_t k, uint4* stage,
                                              const DevDraw* __restrict__ draws, uint32_t n_draws,
                                              const DevView* __restrict__ views, const DevMaterial* __restrict__ mats,
                                              SetupRec* __restrict__ setup, ShadeRec* __restrict__ shade,
                                              uint32_t cap_tri, Status* __restrict__ status, int TS,
                                              uint32_t* __restrict__ bincnt, uint8_t* __restrict__ wflag,
                                              uint32_t* __restrict__ wide_list, WideBuf* wide, uint32_t span) {
  const uint32_t t = sv.x, idx = sv.y + k;
  const bool sparse = wave_sparse(active, t, span);
  const uint32_t d = wave_find_draw(draws, n_draws, t, active);
  auto body = [&](uint32_t d0, bool mine) {
    uint4 ro[6], so[9];
    bool ok = false, skip = false;
    const DevDraw& dr = draws[d0];
    const FrameParamsPod& fr = views[dr.view].fr;
    if (mine) {
      const uint32_t lt = t - dr.tri_begin;
      const V3 cam = v3(fr.cam[0], fr.cam[1], fr.cam[2]);
      const V3 L = v3(fr.light[0], fr.light[1], fr.light[2]);
      FV v[3];
      V3 P[3], N[3];
      float U[3], W[3];
      tri_vertices(dr, lt, sparse, P, N, U, W);
#pragma unroll
      for (int q = 0; q < 3; q++) {
        const V3 p = P[q];
        v[q].p = p;
        // per-vertex visual info, scene/mod.rs:920-925
        const V3 eye_dir = sub(p, cam);
        const V3 light = normalized(sub(p, L));
        const V3 eye = normalized(eye_dir);
        v[q].d = norm(eye_dir);
        v[q].l = light;
        v[q].h = normalized(add(light, eye));
        v[q].n = N[q];
        v[q].u = U[q];
        v[q].v = W[q];
      }
      // passed the back-face and lateral tests in k_geom_count
      if (clip) clip_output(fr, v[0], v[1], v[2], k);
      if (idx >= cap_tri) {
        atomicOr(&status->overflow, 1u);
      } else {
        SetupRec rec;
        make_setup(fr, v[0], v[1], v[2], dr.material, mats[dr.material], dr.view, dr.group, ro, so, rec);
        ok = true;
        // with ordered bins nothing reads a dropped triangle's records
        skip = BIN != kBinNone && (rec.flags & kDrop);
        if constexpr (BIN != kBinNone) {
          const bool is_wide = bin_count_one<BIN>(rec, TS, idx, views[dr.view], bincnt, wflag, bin_boxes(wflag, cap_tri));
          if (BIN == kBinNear && is_wide) wide_push(*wide, idx, status, wide_list);
        }
      }
    }
    wave_store<6>(stage, ro, ok, idx, reinterpret_cast<uint4*>(setup), skip);
    wave_store<9>(stage, so, ok, idx, reinterpret_cast<uint4*>(shade), skip);
  };
  // (as by_draw, but with every lane of the wave in the record stores)
  const uint64_t m = __ballot(active);
  if (!m) return;
  const uint32_t d0 = (uint32_t)__builtin_amdgcn_readlane((int)d, __builtin_ctzll(m));
  if (__ballot(active && d != d0) == 0ull) body(d0, active);
  else body(d, active);
}

// Both emitter lists (dense: culled triangles take no lane) in one launch, a
// wave per unit of 64 lanes, the clipped list's units first: two lanes a
// clipped triangle, for its even and its odd outputs (it has at most four, and
// seldom more than two), one an unclipped one.  The lists' lengths are on the
// device, so the grid is capped and the waves stride over the units.
//
// A clipped triangle is a long chain of dependent work.  With a lane each, up
// to four inlined copies of the setup (28 KB of code) and 168 VGPRs, its list
// took 25 us even when short, on a second stream beside the other list's
// launch: the fork and the join cost some 15 us more.  One copy of the setup
// serves both lists here (17 KB, twice for waves of one draw and of several;
// 127 VGPRs), at the four waves per SIMD that the LDS of the record stores
// allows.  Frames, before -> after: 62k triangles
// at 800x600 with a GUI 194 -> 179 us, 150k at 1237x709 168 -> 152, the
// 1M-triangle 1080p soup 357 -> 339, two 125k-triangle shards 403 -> 391.
template <int BIN>
__global__ __launch_bounds__(256, 4) void k_geom_emit(const DevDraw* __restrict__ draws, uint32_t n_draws,
                                                      const DevView* __restrict__ views,
                                                      const uint2* __restrict__ surv, const uint8_t* __restrict__ cnt,
                                                      const DevMaterial* __restrict__ mats,
                                                      SetupRec* __restrict__ setup, ShadeRec* __restrict__ shade,
                                                      uint32_t cap_tri, Status* __restrict__ status, int TS,
                                                      uint32_t* __restrict__ bincnt, uint8_t* __restrict__ wflag,
                                                      uint32_t* __restrict__ wide_list, uint32_t span) {
  __shared__ uint32_t s_wide[BIN == kBinNear ? sizeof(WideBuf) / 4 : 1];
  __shared__ uint4 s_stage[4][64 * 9];
  WideBuf* const wide = reinterpret_cast<WideBuf*>(s_wide);
  if constexpr (BIN == kBinNear) {
    if (threadIdx.x == 0) wide->n = 0u;
    __syncthreads();
  }
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t n_simple = status->n_simple, n_clip = status->n_clip;
  const uint32_t uc = (n_clip + 31u) / 32u, us = (n_simple + 63u) / 64u;
  for (uint32_t u = blockIdx.x * 4u + wave; u < uc + us; u += gridDim.x * 4u) {
    const bool clip = u < uc;
    const uint32_t j = clip ? u * 32u + (lane >> 1) : (u - uc) * 64u + lane;
    const bool in = j < (clip ? n_clip : n_simple);
    const uint2 sv = in ? surv[clip ? n_simple + j : j] : make_uint2(0u, 0u);
    const uint32_t c = in ? (clip ? (uint32_t)cnt[sv.x] & kCntMask : 1u) : 0u;
    for (uint32_t k = clip ? lane & 1u : 0u; __ballot(k < c) != 0ull; k += 2u)
      geom_emit_one<BIN>(sv, k < c, clip, k, s_stage[wave], draws, n_draws, views, mats, setup, shade, cap_tri, status,
                         TS, bincnt, wflag, wide_list, wide, span);
  }
  if constexpr (BIN == kBinNear) wide_flush(*wide, status, wide_list);
}

// Clipped triangles before input triangle t0: its block's scanned count and
// the counts before it in the block, a wave's lanes taking four each (every
// lane calls it; one thread alone needs up to 255 dependent loads, 20 us of a
// 32-view batch).
__device__ inline uint32_t wave_id_before(uint32_t t0, uint32_t n_in, const uint8_t* __restrict__ cnt,
                                          const uint32_t* __restrict__ blk_off, const Status* __restrict__ status) {
  if (t0 >= n_in) return status->n_out;
  const uint32_t lane = threadIdx.x & 63u, b = t0 >> 8;
  uint32_t s = 0;
#pragma unroll
  for (uint32_t k = 0; k < 4u; k++) {
    const uint32_t t = (b << 8) + 64u * k + lane;
    if (t < t0) s += cnt[t] & kCntMask;
  }
#pragma unroll
  for (int o = 32; o; o >>= 1) s += __shfl_xor(s, o, 64);
  return blk_off[b] + s;
}

// First clipped-triangle id of each view (a wave per view).  Shading subtracts
// it, so a view's winner ids do not depend on the other views of a batch.
__global__ __launch_bounds__(256) void k_view_id_base(DevView* __restrict__ views, uint32_t n_views, uint32_t n_in,
                                                      const uint8_t* __restrict__ cnt,
                                                      const uint32_t* __restrict__ blk_off,
                                                      const Status* __restrict__ status) {
  const uint32_t v = (blockIdx.x * 256u + threadIdx.x) >> 6;
  if (v >= n_views) return;  // the whole wave
  const uint32_t id = wave_id_before(views[v].tri_begin, n_in, cnt, blk_off, status);
  if ((threadIdx.x & 63u) == 0u) views[v].id_base = id;
}

// ====================================================================== scan
// Generic exclusive scan of u32 with the element count possibly on the device.
constexpr int kScanG = 1024;  // partial sums per scan

__device__ inline uint32_t scan_count(const uint32_t* n_ptr, uint32_t n_const, uint32_t cap) {
  if (!n_ptr) return n_const;
  uint32_t n = *n_ptr;
  return n < cap ? n : cap;
}
__device__ inline uint32_t scan_chunk(uint32_t n) { return (((n + kScanG - 1u) / kScanG) + 1023u) & ~1023u; }

__global__ __launch_bounds__(256) void k_scan_reduce(const uint32_t* __restrict__ in, const uint32_t* n_ptr,
                                                     uint32_t n_const, uint32_t cap, uint32_t* __restrict__ partials) {
  __shared__ uint32_t s_tmp[4];
  const uint32_t n = scan_count(n_ptr, n_const, cap);
  const uint32_t C = scan_chunk(n);
  const uint32_t b0 = blockIdx.x * C;
  const uint32_t b1 = min(b0 + C, n);
  uint32_t s = 0;
  for (uint32_t i = b0 + threadIdx.x; i < b1; i += 256) s += in[i];
  uint32_t total;
  block_exclusive_scan256(s, s_tmp, &total);
  if (threadIdx.x == 0) partials[blockIdx.x] = total;
}

// Second pass: each block takes the exclusive prefix of the partial sums
// before it (at most kScanG values, read straight from the partials) and
// scans its chunk; block 0 also publishes the total and the overflow flag.
// in and out may be the same array (in-place scans): no __restrict__ on them.
__global__ __launch_bounds__(256) void k_scan_apply(const uint32_t* in, uint32_t* out,
                                                    const uint32_t* n_ptr, uint32_t n_const, uint32_t cap,
                                                    const uint32_t* __restrict__ partials, uint32_t* total_out,
                                                    uint32_t cap_check, uint32_t* overflow_word,
                                                    uint32_t overflow_bit) {
  __shared__ uint32_t s_tmp[4];
  const uint32_t n = scan_count(n_ptr, n_const, cap);
  const uint32_t C = scan_chunk(n);
  const uint32_t b0 = blockIdx.x * C;
  const uint32_t b1 = min(b0 + C, n);
  const uint32_t upto = blockIdx.x == 0 ? (uint32_t)kScanG : blockIdx.x;
  uint32_t p = 0;
  for (uint32_t i = threadIdx.x; i < upto; i += 256) p += partials[i];
  uint32_t sum;
  block_exclusive_scan256(p, s_tmp, &sum);
  uint32_t running = 0;
  if (blockIdx.x == 0) {
    if (threadIdx.x == 0) {
      if (total_out) *total_out = sum;
      if (overflow_word && sum > cap_check) atomicOr(overflow_word, overflow_bit);
    }
  } else {
    running = sum;
  }
  for (uint32_t tb = b0; tb < b1; tb += 1024) {
    const uint32_t i0 = tb + threadIdx.x * 4u;
    uint32_t v[4];
#pragma unroll
    for (int k = 0; k < 4; k++) v[k] = (i0 + k < b1) ? in[i0 + k] : 0u;
    const uint32_t s4 = v[0] + v[1] + v[2] + v[3];
    uint32_t total;
    uint32_t ex = block_exclusive_scan256(s4, s_tmp, &total) + running;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (i0 + k < b1) out[i0 + k] = ex;
      ex += v[k];
    }
    running += total;
  }
}

// Up to three independent exclusive scans of n values each (n known to the
// host), one block of 1024 threads each, 8192 values at a time with a carry:
// the per-block counts of the geometry pass, for which one launch of a few
// rounds is shorter than two launches per scan (20,000 blocks, a 5M-triangle
// frame: 27 us in six launches, 20 in one, 6 with 16-byte accesses).
struct ScanSeg {
  const uint32_t* in;
  uint32_t* out;
  uint32_t* total_out;      // may be null
  uint32_t* overflow_word;  // may be null
  uint32_t cap_check, overflow_bit;
};
struct ScanSegs {
  ScanSeg s[3];
};

__global__ __launch_bounds__(1024) void k_scan_segs(ScanSegs segs, uint32_t n) {
  constexpr int kPer = 8;
  const ScanSeg& g = segs.s[blockIdx.x];
  const uint32_t* in = g.in;  // may be out (in-place scans)
  uint32_t* out = g.out;
  uint32_t* total_out = g.total_out;
  uint32_t* overflow_word = g.overflow_word;
  const uint32_t cap_check = g.cap_check, overflow_bit = g.overflow_bit;
  __shared__ uint32_t s_w[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t carry = 0;
  uint32_t v[kPer];
  // 16-byte accesses: a lane's eight values one by one touch each line of the
  // wave's 2 KB eight times
  const bool wide = ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(out)) & 15u) == 0u;
  auto load = [&](uint32_t t0) {
    const uint32_t i0 = t0 + threadIdx.x * (uint32_t)kPer;
    if (wide && i0 + kPer <= n) {
      const uint4 a = *reinterpret_cast<const uint4*>(in + i0), b = *reinterpret_cast<const uint4*>(in + i0 + 4);
      v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
      v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
      return;
    }
#pragma unroll
    for (int k = 0; k < kPer; k++) v[k] = (i0 + k < n) ? in[i0 + k] : 0u;
  };
  load(0u);
  for (uint32_t t0 = 0; t0 < n; t0 += 1024u * kPer) {
    const uint32_t i0 = t0 + threadIdx.x * (uint32_t)kPer;
    uint32_t c[kPer], e[kPer], sum = 0;
#pragma unroll
    for (int k = 0; k < kPer; k++) {
      c[k] = v[k];
      sum += c[k];
    }
    if (t0 + 1024u * kPer < n) load(t0 + 1024u * kPer);  // the next round's, behind this round's barriers
    uint32_t x = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    if (lane == 63) s_w[wave] = x;
    __syncthreads();
    uint32_t before = carry, all = 0;
    for (int w = 0; w < 16; w++) {
      if (w < wave) before += s_w[w];
      all += s_w[w];
    }
    e[0] = before + x - sum;
#pragma unroll
    for (int k = 1; k < kPer; k++) e[k] = e[k - 1] + c[k - 1];
    if (wide && i0 + kPer <= n) {
      *reinterpret_cast<uint4*>(out + i0) = make_uint4(e[0], e[1], e[2], e[3]);
      *reinterpret_cast<uint4*>(out + i0 + 4) = make_uint4(e[4], e[5], e[6], e[7]);
    } else {
#pragma unroll
      for (int k = 0; k < kPer; k++)
        if (i0 + k < n) out[i0 + k] = e[k];
    }
    carry += all;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    if (total_out) *total_out = carry;
    if (overflow_word && carry > cap_check) atomicOr(overflow_word, overflow_bit);
  }
}

// out = exclusive scan of in.
static void scan_u32(const uint32_t* in, uint32_t* out, const uint32_t* n_ptr, uint32_t n_const, uint32_t cap,
                     uint32_t* partials, uint32_t* total_out, uint32_t cap_check, uint32_t* overflow_word,
                     uint32_t overflow_bit, hipStream_t s) {
  if (!n_ptr && n_const <= 4096u) {
    ScanSegs g{};
    g.s[0] = ScanSeg{in, out, total_out, overflow_word, cap_check, overflow_bit};
    hipLaunchKernelGGL(k_scan_segs, dim3(1), dim3(1024), 0, s, g, n_const);
    return;
  }
  hipLaunchKernelGGL(k_scan_reduce, dim3(kScanG), dim3(256), 0, s, in, n_ptr, n_const, cap, partials);
  hipLaunchKernelGGL(k_scan_apply, dim3(kScanG), dim3(256), 0, s, in, out, n_ptr, n_const, cap, partials, total_out,
                     cap_check, overflow_word, overflow_bit);
}

// Pass 1 of unordered bins, one thread per clipped triangle: flag wide
// triangles (wflag, one byte each) and count the tiles of the others per tile
// with atomics.  (Ordered bins take the per-triangle counts from k_geom_emit.)
__global__ __launch_bounds__(256) void k_bin_count(const SetupRec* __restrict__ setup, const DevView* __restrict__ views,
                                                   const Status* status, uint32_t cap_tri, int TS,
                                                   uint32_t* __restrict__ tile_cnt, uint8_t* __restrict__ wflag) {
  const uint32_t n = min(status->n_out, cap_tri);
  for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < n; i += gridDim.x * 256u) {
    const SetupRec r = setup[i];
    bool is_wide = false;
    if (!(r.flags & kDrop)) {
      Spans g;
      spans_init(r, TS, g);
      is_wide = bin_is_wide(g);
      if (!is_wide) {
        const DevView& vw = views[r.view];
        thread_tiles(g, TS, [&](uint32_t, int ty, int tx) {
          atomicAdd(&tile_cnt[vw.tile_base + (uint32_t)ty * vw.ntx + (uint32_t)tx], 1u);
        });
      }
    }
    wflag[i] = is_wide ? 1u : 0u;
  }
}

// The wide-triangle list: the wide triangles (flag 1) of each 4096-triangle chunk,
// 16 flags per thread, placed by a block scan; one atomic per chunk reserves
// the chunk's run of the list.  The list order does not matter: a triangle's
// bin entries go to its own scanned offset (or through per-tile atomics for
// unordered bins).
__global__ __launch_bounds__(256) void k_wide_list(const uint8_t* __restrict__ wflag, Status* status,
                                                   uint32_t cap_tri, uint32_t* __restrict__ list,
                                                   uint32_t* __restrict__ zero_dst, uint32_t zero_words) {
  __shared__ uint32_t s_tmp[4];
  __shared__ uint32_t s_base;
  // also clears the tile ranges that k_tile_ranges fills later
  for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < zero_words; i += gridDim.x * 256u) zero_dst[i] = 0u;
  const uint32_t n = min(status->n_out, cap_tri);
  for (uint32_t c0 = blockIdx.x * 4096u; c0 < n; c0 += gridDim.x * 4096u) {
    const uint32_t t0 = c0 + threadIdx.x * 16u;
    uint32_t mask = 0;
    if (t0 + 16u <= n) {
      const uint4 f = *reinterpret_cast<const uint4*>(wflag + t0);  // t0 is a multiple of 16
      const uint32_t w[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
      for (int k = 0; k < 16; k++)
        if (((w[k >> 2] >> (8 * (k & 3))) & 0xFFu) == 1u) mask |= 1u << k;
    } else {
      for (uint32_t k = 0; t0 + k < n; k++)
        if (wflag[t0 + k] == 1u) mask |= 1u << k;
    }
    uint32_t total;
    const uint32_t local = block_exclusive_scan256((uint32_t)__popc(mask), s_tmp, &total);
    if (threadIdx.x == 0 && total) s_base = atomicAdd(&status->n_wide, total);
    __syncthreads();
    uint32_t o = s_base + local;
    while (mask) {
      const uint32_t k = (uint32_t)__builtin_ctz(mask);
      mask &= mask - 1u;
      list[o++] = t0 + k;
    }
    __syncthreads();
  }
}

// Visits the listed (wide) triangles, one wave per triangle.
template <class F>
__device__ inline void for_each_wide(const uint32_t* __restrict__ list, const Status* status, F f) {
  const uint32_t gw = (blockIdx.x * 256u + threadIdx.x) >> 6, nwaves = gridDim.x * 4u;
  const uint32_t n = status->n_wide;
  for (uint32_t w = gw; w < n; w += nwaves) f((uint32_t)__builtin_amdgcn_readfirstlane(list[w]));
}

template <bool ORDERED>
__global__ __launch_bounds__(256) void k_bin_count_wide(const SetupRec* __restrict__ setup,
                                                        const DevView* __restrict__ views, const Status* status,
                                                        int TS, const uint32_t* __restrict__ wide_list,
                                                        uint32_t* __restrict__ bincnt, uint32_t* __restrict__ tile_cnt) {
  const int lane = threadIdx.x & 63;
  for_each_wide(wide_list, status, [&](uint32_t i) {
    const SetupRec r = setup[i];
    const DevView& vw = views[r.view];
    Spans g;
    spans_init(r, TS, g);
    const uint32_t c = wave_tiles<true>(g, TS, 0, 1, [&](uint32_t, int tx, int ty) {
      if (!ORDERED) atomicAdd(&tile_cnt[vw.tile_base + (uint32_t)ty * vw.ntx + (uint32_t)tx], 1u);
    });
    if (ORDERED && lane == 0) bincnt[i] = c;
  });
}

// Pass 2.  Ordered: (tile key, triangle) pairs at the triangle's scanned
// offset, from its bin box, for the stable radix sort.  Unordered: the
// triangle id goes straight into its tile's list at tile_start +
// atomicAdd(cursor).
//
// Unordered pairs of one triangle that is not wide.
__device__ inline void bin_emit_tri_unordered(const SetupRec* __restrict__ setup, const DevView* __restrict__ views,
                                              int TS, uint32_t i, const uint32_t* __restrict__ tile_start,
                                              uint32_t* __restrict__ tile_cur, uint32_t cap_pairs,
                                              uint32_t* __restrict__ vals) {
  auto put = [&](const DevView& vw, int ty, int tx) {
    const uint32_t key = vw.tile_base + (uint32_t)ty * vw.ntx + (uint32_t)tx;
    const uint32_t pos = tile_start[key] + atomicAdd(&tile_cur[key], 1u);
    if (pos < cap_pairs) vals[pos] = i;
  };
  // the record's last 16 bytes first: a triangle within one tile needs no edges
  const uint4 h = reinterpret_cast<const uint4*>(setup + i)[5];
  if (h.z & kDrop) return;
  const uint32_t cx0 = (h.x & 0xFFFFu) / (uint32_t)TS, cx1 = (h.x >> 16) / (uint32_t)TS;
  const uint32_t cy0 = (h.y & 0xFFFFu) / (uint32_t)TS, cy1 = (h.y >> 16) / (uint32_t)TS;
  if (cx0 == cx1 && cy0 == cy1) {
    put(views[h.w], (int)cy0, (int)cx0);
    return;
  }
  const SetupRec r = setup[i];
  Spans g;
  spans_init(r, TS, g);
  const DevView& vw = views[r.view];
  thread_tiles(g, TS, [&](uint32_t, int ty, int tx) { put(vw, ty, tx); });
}

template <bool ORDERED>
__global__ __launch_bounds__(256) void k_bin_emit(const SetupRec* __restrict__ setup, const DevView* __restrict__ views,
                                                  const Status* status, uint32_t cap_tri, int TS,
                                                  const uint8_t* __restrict__ wflag,
                                                  const uint32_t* __restrict__ binoff,
                                                  const uint32_t* __restrict__ tile_start,
                                                  uint32_t* __restrict__ tile_cur, uint32_t cap_pairs,
                                                  uint32_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  const uint32_t n = min(status->n_out, cap_tri);
  const uint2* boxes = bin_boxes(const_cast<uint8_t*>(wflag), cap_tri);
  for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < n; i += gridDim.x * 256u) {
    if constexpr (ORDERED) {
      const uint2 box = boxes[i];
      if (box.x != kWideBox) emit_box_pairs(box, i, binoff[i], cap_pairs, keys, vals);
    } else if (wflag[i] == 0u) {
      bin_emit_tri_unordered(setup, views, TS, i, tile_start, tile_cur, cap_pairs, vals);
    }
  }
}

template <bool ORDERED>
__global__ __launch_bounds__(256) void k_bin_emit_wide(const SetupRec* __restrict__ setup,
                                                       const DevView* __restrict__ views, const Status* status,
                                                       const uint32_t* __restrict__ wide_list, int TS,
                                                       const uint32_t* __restrict__ binoff,
                                                       const uint32_t* __restrict__ tile_start,
                                                       uint32_t* __restrict__ tile_cur, uint32_t cap_pairs,
                                                       uint32_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  for_each_wide(wide_list, status, [&](uint32_t i) {
    const SetupRec r = setup[i];
    const DevView& vw = views[r.view];
    Spans g;
    spans_init(r, TS, g);
    const uint32_t o = ORDERED ? binoff[i] : 0u;
    wave_tiles<true>(g, TS, 0, 1, [&](uint32_t e, int tx, int ty) {
      const uint32_t key = vw.tile_base + (uint32_t)ty * vw.ntx + (uint32_t)tx;
      const uint32_t pos = ORDERED ? o + e : tile_start[key] + atomicAdd(&tile_cur[key], 1u);
      if (pos < cap_pairs) {
        if (ORDERED) keys[pos] = key;
        vals[pos] = i;
      }
    });
  });
}

// Binning of a small single-view frame in one workgroup of 1024 threads,
// in place of the general path's four launches: per-tile counts
// with LDS atomics from each triangle's bin box (a wave per wide triangle of
// the emits' list), their scan into the tile ranges, then each
// triangle's id written into its tiles' lists at LDS-atomic cursors.  The
// lists are unordered, which changes no result: a tile's visibility is the
// minimum of its fragments' keys whatever the order (the transparent pass,
// which blends in list order, never comes here).  Pairs past cap_pairs are
// counted, flagged (overflow bit 2) and not written; ranges end at cap_pairs.

__global__ __launch_bounds__(1024) void k_bin_small(const SetupRec* __restrict__ setup,
                                                    const DevView* __restrict__ views, Status* __restrict__ status,
                                                    uint32_t cap_tri, int TS, const uint8_t* __restrict__ wflag,
                                                    const uint32_t* __restrict__ wide_list, uint32_t n_tiles,
                                                    uint32_t cap_pairs, uint32_t* __restrict__ vals,
                                                    uint2* __restrict__ ranges) {
  __shared__ uint32_t s_cnt[kFewBinTiles];
  __shared__ uint32_t s_cur[kFewBinTiles];
  __shared__ uint32_t s_w[16];
  __shared__ LargeBuf s_large[2];  // the count pass's, the list pass's
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (uint32_t k = (uint32_t)tid; k < n_tiles; k += 1024u) s_cnt[k] = 0u;
  if (tid < 2) s_large[tid].n = 0u;
  __syncthreads();
  const uint32_t n = min(status->n_out, cap_tri);
  const uint2* boxes = bin_boxes(const_cast<uint8_t*>(wflag), cap_tri);
  // one pass over the triangles' tiles: f(tile key) for each
  auto each_tile = [&](auto f) {
    for (uint32_t i = (uint32_t)tid; i < n; i += 1024u) {
      box_tiles(boxes[i], [&](uint32_t key) { f(i, key); });
    }
  };
  auto each_wide_tile = [&](uint32_t nw, LargeBuf& large, auto f) {
    wave_wide_tiles<16>(wide_list, (uint32_t)wave, 16u, nw, setup, views, nullptr, TS, large,
                        [&](uint32_t key, uint32_t i, uint32_t) { f(i, key); });
  };
  // counts
  each_tile([&](uint32_t, uint32_t key) { atomicAdd(&s_cnt[key], 1u); });
  const uint32_t nw = status->n_wide;
  each_wide_tile(nw, s_large[0], [&](uint32_t, uint32_t key) { atomicAdd(&s_cnt[key], 1u); });
  __syncthreads();
  // exclusive scan of the counts, 1024 tiles at a time with a carry
  uint32_t carry = 0;
  for (uint32_t k0 = 0; k0 < n_tiles; k0 += 1024u) {
    const uint32_t k = k0 + (uint32_t)tid;
    const uint32_t c = k < n_tiles ? s_cnt[k] : 0u;
    uint32_t x = c;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    if (lane == 63) s_w[wave] = x;
    __syncthreads();
    uint32_t before = 0, all = 0;
    for (int w = 0; w < 16; w++) {
      if (w < wave) before += s_w[w];
      all += s_w[w];
    }
    __syncthreads();
    const uint32_t start = carry + before + x - c;
    if (k < n_tiles) {
      s_cur[k] = start;
      ranges[k] = make_uint2(start, min(start + c, cap_pairs));
    }
    carry += all;
  }
  if (tid == 0) {
    status->n_pairs = carry;
    if (carry > cap_pairs) atomicOr(&status->overflow, 2u);
  }
  __syncthreads();
  // the lists
  auto put = [&](uint32_t i, uint32_t key) {
    const uint32_t pos = atomicAdd(&s_cur[key], 1u);
    if (pos < cap_pairs) vals[pos] = i;
  };
  each_tile(put);
  each_wide_tile(nw, s_large[1], put);
}

__global__ __launch_bounds__(256) void k_ranges_from_counts(const uint32_t* __restrict__ tile_start,
                                                            const uint32_t* __restrict__ tile_cnt, uint32_t n_tiles,
                                                            uint32_t cap_pairs, uint2* __restrict__ ranges) {
  for (uint32_t t = blockIdx.x * 256u + threadIdx.x; t < n_tiles; t += gridDim.x * 256u) {
    const uint32_t s0 = min(tile_start[t], cap_pairs);
    ranges[t] = make_uint2(s0, min(s0 + tile_cnt[t], cap_pairs));
  }
}

// ================================================================ radix sort
// Stable LSD radix sort of (tile key, triangle id) pairs with BITS-bit digits
// (one pass when the tile key fits in 11 bits, else 8-bit passes).  Each wave
// owns one contiguous sub-chunk of the input; k_radix_hist counts its digits,
// the scan over (digit, wave) turns the counts into output bases, and
// k_radix_scatter ranks the wave's items in input order (ballot match) and
// advances its own LDS bases -- no block barrier inside the scatter.  Equal
// keys keep the triangle order.  The chunks of one XCD are contiguous, so a
// tile's output run is written by few XCDs: with ~1 item per (wave, tile),
// interleaved chunks would make every XCD's L2 write back partial lines of
// every run.
constexpr int kRadixG = 256;               // blocks of 4 waves
constexpr int kRadixW = kRadixG * 4;       // waves
constexpr int kRadixU = 8;                 // 64-item groups whose loads a wave issues together
static_assert(2048u * kRadixW == kRadixHistEntries, "histogram size");

__device__ inline uint32_t radix_chunk(uint32_t n) { return (((n + kRadixW - 1u) / kRadixW) + 63u) & ~63u; }

template <int BITS>
__global__ __launch_bounds__(256) void k_radix_hist(const uint32_t* __restrict__ keys, const uint32_t* n_ptr,
                                                    uint32_t cap, int shift, uint32_t* __restrict__ hist) {
  constexpr uint32_t ND = 1u << BITS;
  __shared__ uint32_t h[4][ND];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t n = min(*n_ptr, cap);
  const uint32_t C = radix_chunk(n);
  const uint32_t lb = xcd_remap(blockIdx.x, gridDim.x);
  const uint32_t gw = lb * 4u + (uint32_t)wave;
  const uint32_t b0 = min(gw * C, n), b1 = min(b0 + C, n);
  for (uint32_t d = (uint32_t)tid; d < ND; d += 256)
#pragma unroll
    for (int w = 0; w < 4; w++) h[w][d] = 0;
  __syncthreads();
  // kRadixU loads in flight per lane before their LDS increments
  for (uint32_t tb = b0; tb < b1; tb += 64u * kRadixU) {
    uint32_t k[kRadixU];
#pragma unroll
    for (int u = 0; u < kRadixU; u++) {
      const uint32_t i = tb + 64u * (uint32_t)u + (uint32_t)lane;
      k[u] = i < b1 ? keys[i] : 0u;
    }
#pragma unroll
    for (int u = 0; u < kRadixU; u++)
      if (tb + 64u * (uint32_t)u + (uint32_t)lane < b1) atomicAdd(&h[wave][(k[u] >> shift) & (ND - 1u)], 1u);
  }
  __syncthreads();
  for (uint32_t d = (uint32_t)tid; d < ND; d += 256)
#pragma unroll
    for (int w = 0; w < 4; w++) hist[d * kRadixW + lb * 4u + (uint32_t)w] = h[w][d];
}

// KEYS_OUT false: only the values are written (a last pass whose sorted keys
// nobody reads).  ranges (may be null): [start, end) of each of the first
// n_ranges digits in the output, straight from the scanned histogram -- the
// per-tile lists when this pass sorts by the whole key.
template <int BITS, bool KEYS_OUT>
__global__ __launch_bounds__(256) void k_radix_scatter(const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin,
                                                       uint32_t* __restrict__ kout, uint32_t* __restrict__ vout,
                                                       const uint32_t* n_ptr, uint32_t cap, int shift,
                                                       const uint32_t* __restrict__ hist_off,
                                                       uint2* __restrict__ ranges, uint32_t n_ranges) {
  constexpr uint32_t ND = 1u << BITS;
  __shared__ uint32_t run[4][ND];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t n = min(*n_ptr, cap);
  const uint32_t C = radix_chunk(n);
  const uint32_t gw = xcd_remap(blockIdx.x, gridDim.x) * 4u + (uint32_t)wave;
  const uint32_t b0 = min(gw * C, n), b1 = min(b0 + C, n);
  if (ranges)
    for (uint32_t d = blockIdx.x * 256u + (uint32_t)tid; d < n_ranges; d += gridDim.x * 256u)
      ranges[d] = make_uint2(hist_off[d * kRadixW], d + 1u < ND ? hist_off[(d + 1u) * kRadixW] : n);
  for (uint32_t d = (uint32_t)lane; d < ND; d += 64) run[wave][d] = hist_off[d * kRadixW + gw];
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  for (uint32_t tb = b0; tb < b1; tb += 64u * kRadixU) {
    // kRadixU groups of 64 items loaded up front, then ranked in order
    uint32_t kk[kRadixU], vv[kRadixU];
#pragma unroll
    for (int u = 0; u < kRadixU; u++) {
      const uint32_t i = tb + 64u * (uint32_t)u + (uint32_t)lane;
      kk[u] = i < b1 ? kin[i] : 0u;
      vv[u] = i < b1 ? vin[i] : 0u;
    }
#pragma unroll
    for (int u = 0; u < kRadixU; u++) {
      const bool valid = tb + 64u * (uint32_t)u + (uint32_t)lane < b1;
      const uint32_t key = kk[u];
      const uint32_t dgt = (key >> shift) & (ND - 1u);
      uint64_t peers = __ballot(valid);
#pragma unroll
      for (int bit = 0; bit < BITS; bit++) {
        const bool on = (dgt >> bit) & 1u;
        const uint64_t m = __ballot(on);
        peers &= on ? m : ~m;
      }
      const uint32_t rank = (uint32_t)__popcll(peers & lt);
      uint32_t base = 0;
      if (valid) base = run[wave][dgt];
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      if (valid) {
        if (KEYS_OUT) kout[base + rank] = key;
        vout[base + rank] = vv[u];
        if (rank == 0) run[wave][dgt] = base + (uint32_t)__popcll(peers);
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
  }
}

// ======================================================== near-first tile lists
// The default bins: every tile's list, roughly near first, in four launches
// and without an intermediate array of pairs in triangle order.  Nothing here
// has to be stable: a tile's visibility does not depend on its list's order.
//  k_pair_hist     the triangles (bin boxes) are cut into kPairChunks
//                  contiguous chunks, the wide list into as many; a block per
//                  chunk counts its (tile, triangle) pairs by digit, the
//                  tile key's low bits;
//  k_row_scan      a block per digit scans the chunks' counts;
//  k_pair_scatter  the blocks of k_pair_hist write their pairs at LDS cursors
//                  into the digit's segment, as (rest of the key << 8 | depth
//                  key, triangle);
//  k_pair_sort     a block per segment sorts it by (tile, depth level) with
//                  LDS counters and writes the ids and the tiles' ranges.
// Neighbouring tiles lie in different segments, so a crowded part of the
// screen is spread over all of them; the depth order costs no pass of its own.
// (Before: a depth sort of the triangles, a gathered scan, a pair emit and one
// or two more sort passes with their scans, 13 to 18 launches of 3 to 15 us
// each.  1M-triangle 1080p frame: 387 -> 358 us; 150k triangles at 1237x709: 208
// -> 166 us; 500k triangles at 3840x2160: 300 -> 249 us.  Hist, scan, scatter and
// sort take 12, 5, 18 and 13 us of the first, 9, 5, 11 and 7 of the second, 5, 4,
// 5 and 8 of the third.)
constexpr int kPairChunks = 256;         // blocks of 1024 threads: one per CU
constexpr int kPairT = 1024;
constexpr int kPairU = 4;                // boxes in flight per thread
constexpr int kPairCols = kPairChunks;   // histogram columns
constexpr uint32_t kPairCounters = 8192;    // k_pair_sort's LDS counters: tiles of a segment x depth levels
// 256 segments, or 2048 where they would leave a segment fewer than 16 depth
// levels; beyond kPairMaxTiles a segment has more tiles than counters.
constexpr uint32_t kPairFewTiles = 256u * (kPairCounters / 16u);
constexpr uint32_t kPairMaxTiles = 2048u * kPairCounters;
static_assert(2048u * (kPairCols + 1u) <= kRadixHistEntries, "histogram and digit totals");

// SUBMIT lists hold each tile's triangles in submission order, which the
// transparent pass blends in: the depth key gives way to the high bits of the
// id, and k_pair_sort places the ids that share a counter by counting.  (A
// transparent pass of 19,600 triangles on 3600 tiles took 14 launches and some
// 55 us from its emits to the blend by a stable sort of tile keys, now four and
// 19.)  A tile that holds the whole mesh makes that count quadratic, n ids by
// n / levels each, so at most kPairShare of the input's may share a counter: by
// 256 segments where these leave levels enough, else by 2048, else by the stable
// sort.  65,536 triangles in a pane, and all in a few tiles: 1280x720 in 16x16
// tiles (256 levels) 226 us and 65 ms (256 segments), 238 and 64 (2048), 257 and 60
// (sorted); 3840x2160 in 16x16 (64 levels, 256 with 2048 segments) 408 us and 73
// ms, 421 and 67, 442 and 64; in 8x8 (16, 128) 911 us and 100 ms, 927 and 65, 971
// and 58; 7680x4320 in 8x8 (32 with 2048 segments) 3.18 and 79 ms, 3.27 and 59
// sorted.
constexpr uint32_t kPairSubmitTris = 65536, kPairShare = 1024;
inline bool submit_share(uint32_t n_tri_in, uint32_t n_tiles, uint32_t segments) {
  const uint32_t nh = (n_tiles + segments - 1u) / segments;  // tiles of a segment
  const uint32_t levels = std::min(256u, kPairCounters / nh);
  return levels && n_tri_in <= kPairShare * levels;
}
__device__ inline uint32_t submit_shift(uint32_t n) {  // (n - 1) >> shift <= 255
  return n > 256u ? 24u - (uint32_t)__builtin_clz(n - 1u) : 0u;
}

__device__ inline uint32_t pair_col() { return xcd_remap(blockIdx.x, (uint32_t)kPairChunks); }

// Visits the pairs of one chunk: f(tile key, triangle, depth key).
template <class F>
__device__ inline void pair_chunk(const uint8_t* __restrict__ dkey, const uint32_t* __restrict__ wide_list,
                                  const SetupRec* __restrict__ setup, const DevView* __restrict__ views,
                                  const Status* __restrict__ status, uint32_t cap_tri, int TS, LargeBuf& large, F f) {
  const int tid = threadIdx.x, wave = tid >> 6;
  const uint32_t n = min(status->n_out, cap_tri);
  // consecutive chunks on one XCD: their runs in a segment are neighbours
  const uint32_t cb = pair_col();
  const uint32_t C = (n + (uint32_t)kPairChunks - 1u) / (uint32_t)kPairChunks;
  const uint32_t b0 = min(cb * C, n), b1 = min(b0 + C, n);
  const uint2* boxes = bin_boxes(const_cast<uint8_t*>(dkey), cap_tri);
  for (uint32_t tb = b0; tb < b1; tb += (uint32_t)(kPairT * kPairU)) {
    uint2 box[kPairU];
    uint32_t dk[kPairU];
#pragma unroll
    for (int u = 0; u < kPairU; u++) {
      const uint32_t i = tb + (uint32_t)(kPairT * u + tid);
      box[u] = i < b1 ? boxes[i] : make_uint2(0u, 0u);
      dk[u] = i < b1 ? dkey[i] : 0u;
    }
#pragma unroll
    for (int u = 0; u < kPairU; u++)
      box_tiles(box[u], [&](uint32_t key) { f(key, tb + (uint32_t)(kPairT * u + tid), dk[u]); });
  }
  // its wide triangles
  wave_wide_tiles<kPairT / 64>(wide_list, blockIdx.x + (uint32_t)kPairChunks * (uint32_t)wave,
                               (uint32_t)kPairChunks * (kPairT / 64u), min(status->n_wide, cap_tri), setup, views,
                               dkey, TS, large, f);
}

template <int DIG>
__global__ __launch_bounds__(kPairT) void k_pair_hist(const uint8_t* __restrict__ dkey,
                                                      const uint32_t* __restrict__ wide_list,
                                                      const SetupRec* __restrict__ setup,
                                                      const DevView* __restrict__ views,
                                                      const Status* __restrict__ status, uint32_t cap_tri, int TS,
                                                      uint32_t* __restrict__ hist) {
  __shared__ uint32_t h[DIG];
  __shared__ LargeBuf s_large;
  for (int d = threadIdx.x; d < DIG; d += kPairT) h[d] = 0u;
  if (threadIdx.x == 0) s_large.n = 0u;
  __syncthreads();
  pair_chunk(dkey, wide_list, setup, views, status, cap_tri, TS, s_large,
             [&](uint32_t key, uint32_t, uint32_t) { atomicAdd(&h[key & (DIG - 1u)], 1u); });
  __syncthreads();
  const uint32_t col = pair_col();
  for (int d = threadIdx.x; d < DIG; d += kPairT) hist[(uint32_t)d * kPairCols + col] = h[d];
}

// Row d of the histogram to its exclusive scan, its total to totals[d].
__global__ __launch_bounds__(kPairCols) void k_row_scan(uint32_t* __restrict__ hist, uint32_t* __restrict__ totals) {
  __shared__ uint32_t s_w[kPairCols / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t* const row = hist + (uint64_t)blockIdx.x * kPairCols;
  const uint32_t v = row[threadIdx.x];
  uint32_t x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) s_w[wave] = x;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < kPairCols / 64; w++) {
    if (w < wave) before += s_w[w];
    all += s_w[w];
  }
  row[threadIdx.x] = before + x - v;
  if (threadIdx.x == 0) totals[blockIdx.x] = all;
}

// Exclusive scan of s[0, N) in LDS by a block of T threads (all call it, the
// values stored before a barrier); returns the total.
template <int T>
__device__ inline uint32_t lds_exclusive_scan(uint32_t* s, uint32_t n, uint32_t* s_w /*[T/64]*/) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t carry = 0;
  for (uint32_t k0 = 0; k0 < n; k0 += 4u * T) {
    const uint32_t k = k0 + 4u * threadIdx.x;
    uint32_t v[4];
#pragma unroll
    for (int j = 0; j < 4; j++) v[j] = k + j < n ? s[k + j] : 0u;
    const uint32_t s4 = v[0] + v[1] + v[2] + v[3];
    uint32_t x = s4;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(x, o, 64);
      if (lane >= o) x += y;
    }
    if (lane == 63) s_w[wave] = x;
    __syncthreads();
    uint32_t before = carry, all = 0;
#pragma unroll
    for (int w = 0; w < T / 64; w++) {
      if (w < wave) before += s_w[w];
      all += s_w[w];
    }
    uint32_t ex = before + x - s4;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      if (k + j < n) s[k + j] = ex;
      ex += v[j];
    }
    carry += all;
    __syncthreads();
  }
  return carry;
}

template <int DIG, bool SUBMIT>
__global__ __launch_bounds__(kPairT) void k_pair_scatter(const uint8_t* __restrict__ dkey,
                                                         const uint32_t* __restrict__ wide_list,
                                                         const SetupRec* __restrict__ setup,
                                                         const DevView* __restrict__ views, Status* __restrict__ status,
                                                         uint32_t cap_tri, int TS, const uint32_t* __restrict__ hist,
                                                         const uint32_t* __restrict__ totals, uint32_t cap_pairs,
                                                         uint2* __restrict__ pairs) {
  constexpr int kShift = DIG == 256 ? 8 : 11;
  __shared__ uint32_t cur[DIG];
  __shared__ LargeBuf s_large;
  __shared__ uint32_t s_w[kPairT / 64];
  const uint32_t col = pair_col();
  if (threadIdx.x == 0) s_large.n = 0u;
  for (int d = threadIdx.x; d < DIG; d += kPairT) cur[d] = totals[d];
  __syncthreads();
  const uint32_t all = lds_exclusive_scan<kPairT>(cur, DIG, s_w);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    status->n_pairs = all;
    if (all > cap_pairs) atomicOr(&status->overflow, 2u);
  }
  for (int d = threadIdx.x; d < DIG; d += kPairT) cur[d] += hist[(uint32_t)d * kPairCols + col];
  __syncthreads();
  const uint32_t sh = submit_shift(min(status->n_out, cap_tri));
  pair_chunk(dkey, wide_list, setup, views, status, cap_tri, TS, s_large,
             [&](uint32_t key, uint32_t i, uint32_t dk) {
               if (SUBMIT) dk = i >> sh;
               const uint32_t pos = atomicAdd(&cur[key & (DIG - 1u)], 1u);
               if (pos < cap_pairs) pairs[pos] = make_uint2((key >> kShift) << 8 | dk, i);
             });
}

// Segment d holds the pairs of the tiles d, d + DIG, d + 2 DIG, ...: nh of
// them.  Counters per (tile, depth level): the depth keys between the
// segment's smallest and largest, 2^s to a level, with s as small as the
// counters allow.  Pairs past cap_pairs (flagged by the scatter) are left out.
// SUBMIT: vals is a scratch array, and each id goes to out at its rank among
// the ids of its counter.
constexpr int kSortT = 512, kSortU = 8;
template <int DIG, bool SUBMIT>
__global__ __launch_bounds__(kSortT) void k_pair_sort(const uint2* __restrict__ pairs,
                                                      const uint32_t* __restrict__ totals, uint32_t cap_pairs,
                                                      uint32_t n_tiles, uint32_t* vals, uint2* __restrict__ ranges,
                                                      uint32_t* __restrict__ out) {
  __shared__ uint32_t cnt[kPairCounters];
  __shared__ uint32_t s_w[kSortT / 64];
  __shared__ uint32_t s_mn, s_mx, s_base;
  const uint32_t d = blockIdx.x, tid = threadIdx.x;
  const uint32_t nh = d < n_tiles ? (n_tiles - d + DIG - 1u) / DIG : 0u;
  if (nh == 0u) return;  // the whole block
  // the segment's start: the sum of the totals before it
  if (tid == 0) {
    s_mn = 255u;
    s_mx = 0u;
    s_base = 0u;
  }
  __syncthreads();
  uint32_t p = 0;
  for (uint32_t k = tid; k < d; k += kSortT) p += totals[k];
#pragma unroll
  for (int o = 32; o; o >>= 1) p += __shfl_xor(p, o, 64);
  if ((tid & 63u) == 0u && p) atomicAdd(&s_base, p);
  __syncthreads();
  const uint32_t base = min(s_base, cap_pairs);
  const uint32_t n = min(totals[d], cap_pairs - base);
  uint2 it[kSortU];
  auto load = [&](uint32_t t0) {
#pragma unroll
    for (int u = 0; u < kSortU; u++) {
      const uint32_t i = t0 + (uint32_t)(kSortT * u) + tid;
      it[u] = i < n ? pairs[base + i] : make_uint2(0u, 0u);
    }
  };
  // up to kSortT * kSortU pairs stay in registers, more are read three times
  constexpr uint32_t kRound = kSortT * kSortU;
  const bool once = n <= kRound;
  uint32_t mn = 255u, mx = 0u;
  for (uint32_t t0 = 0; t0 < n; t0 += kRound) {
    load(t0);
#pragma unroll
    for (int u = 0; u < kSortU; u++)
      if (t0 + (uint32_t)(kSortT * u) + tid < n) {
        mn = min(mn, it[u].x & 255u);
        mx = max(mx, it[u].x & 255u);
      }
  }
#pragma unroll
  for (int o = 32; o; o >>= 1) {
    mn = min(mn, (uint32_t)__shfl_xor(mn, o, 64));
    mx = max(mx, (uint32_t)__shfl_xor(mx, o, 64));
  }
  if ((tid & 63u) == 0u) {
    atomicMin(&s_mn, mn);
    atomicMax(&s_mx, mx);
  }
  __syncthreads();
  mn = s_mn;
  mx = max(s_mx, mn);
  uint32_t s = 0;
  while ((((mx - mn) >> s) + 1u) * nh > kPairCounters) s++;  // ends: s = 8 leaves one level, nh <= kPairCounters
  const uint32_t L = ((mx - mn) >> s) + 1u;
  for (uint32_t k = tid; k < nh * L; k += kSortT) cnt[k] = 0u;
  __syncthreads();
  auto slot = [&](uint32_t x) { return (x >> 8) * L + (((x & 255u) - mn) >> s); };
  for (uint32_t t0 = 0; t0 < n; t0 += kRound) {
    if (!once) load(t0);
#pragma unroll
    for (int u = 0; u < kSortU; u++)
      if (t0 + (uint32_t)(kSortT * u) + tid < n) atomicAdd(&cnt[slot(it[u].x)], 1u);
  }
  __syncthreads();
  lds_exclusive_scan<kSortT>(cnt, nh * L, s_w);
  for (uint32_t h = tid; h < nh; h += kSortT)
    ranges[h * DIG + d] = make_uint2(base + cnt[h * L], base + (h + 1u < nh ? cnt[(h + 1u) * L] : n));
  __syncthreads();
  for (uint32_t t0 = 0; t0 < n; t0 += kRound) {
    if (!once) load(t0);
#pragma unroll
    for (int u = 0; u < kSortU; u++)
      if (t0 + (uint32_t)(kSortT * u) + tid < n) vals[base + atomicAdd(&cnt[slot(it[u].x)], 1u)] = it[u].y;
  }
  if constexpr (SUBMIT) {
    __syncthreads();  // a counter now holds its ids' end, which is the next one's start
    for (uint32_t t0 = 0; t0 < n; t0 += kRound) {
      if (!once) load(t0);
#pragma unroll
      for (int u = 0; u < kSortU; u++) {
        if (t0 + (uint32_t)(kSortT * u) + tid >= n) continue;
        const uint32_t k = slot(it[u].x), lo = k ? cnt[k - 1u] : 0u, hi = cnt[k];
        uint32_t r = lo;
        for (uint32_t j = lo; j < hi; j++) r += vals[base + j] < it[u].y ? 1u : 0u;
        out[base + r] = it[u].y;
      }
    }
  }
}

// A frame's first kernel: the Status words of its passes cleared and the
// draw, view and group tables copied in from pinned host memory.
__global__ __launch_bounds__(256) void k_frame_begin(uint32_t* __restrict__ status, uint32_t status_words,
                                                     const uint32_t* __restrict__ src, uint32_t* __restrict__ dst,
                                                     uint32_t n_words) {
  if (blockIdx.x == 0 && threadIdx.x < status_words) status[threadIdx.x] = 0u;
  for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < n_words; i += gridDim.x * 256u) dst[i] = src[i];
}

__global__ void k_fill_u32(uint32_t* p, uint32_t v, uint32_t n) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = v;
}

__global__ __launch_bounds__(256) void k_tile_ranges(const uint32_t* __restrict__ keys, const uint32_t* n_ptr,
                                                     uint32_t cap, uint2* __restrict__ ranges) {
  const uint32_t n = min(*n_ptr, cap);
  for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < n; i += gridDim.x * 256u) {
    const uint32_t k = keys[i];
    if (i == 0 || keys[i - 1] != k) ranges[k].x = i;
    if (i + 1 == n || keys[i + 1] != k) ranges[k].y = i + 1;
  }
}

// ======================================================== transparent pass
// First opaque clipped-triangle id of each object group (a wave per group).
__global__ __launch_bounds__(256) void k_group_base(const uint32_t* __restrict__ grp_first, uint32_t n_groups,
                                                    uint32_t n_in, const uint8_t* __restrict__ cnt,
                                                    const uint32_t* __restrict__ blk_off,
                                                    const Status* __restrict__ status, uint32_t* __restrict__ grp_base) {
  const uint32_t g = (blockIdx.x * 256u + threadIdx.x) >> 6;
  if (g >= n_groups) return;  // the whole wave
  const uint32_t id = wave_id_before(grp_first[g], n_in, cnt, blk_off, status);
  if ((threadIdx.x & 63u) == 0u) grp_base[g] = id;
}

// Sort key of a transparent mesh's triangle (scene/mod.rs:1100-1115): the
// distance from the camera to the centroid (a + b + c) / 3, ordered by
// f32::total_cmp reversed.  key = ~(order-preserving bits of the distance),
// so an ascending stable sort gives the descending total order with ties in
// the current triangle order.
__device__ inline uint32_t tsort_key(const uint32_t* __restrict__ t9, const float* __restrict__ pos, V3 cam) {
  const V3 a = ld3(pos, t9[0]), b = ld3(pos, t9[1]), c = ld3(pos, t9[2]);
  const V3 ctr = divs(add(add(a, b), c), 3.0f);
  const float d = norm(sub(ctr, cam));  // Vec3::dist, linalg.rs:177-180
  const uint32_t u = __float_as_uint(d);
  const uint32_t k = (u & 0x80000000u) ? ~u : (u | 0x80000000u);  // total order as unsigned
  return ~k;
}

__global__ __launch_bounds__(256) void k_tsort_keys(const uint32_t* __restrict__ tri, uint32_t n,
                                                    const float* __restrict__ pos, float cx, float cy, float cz,
                                                    uint32_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n) return;
  keys[i] = tsort_key(tri + 9ull * i, pos, v3(cx, cy, cz));
  vals[i] = i;
}

// The sort of transparent meshes of at most kTsortMax triangles, up to
// kTsortMeshes of them at once, in two launches:
//  k_tsort_chunks  a block per kTsortChunk triangles sorts their (key, index)
//                  words, all different, in registers and LDS, and copies the
//                  triangles out of the mesh;
//  k_tsort_merge   sixteen lanes per triangle add up its ranks in the mesh's
//                  chunks by binary searches and write it to its place.
// A radix sort took 18 to 22 launches a mesh, each about as long as starting it
// (two meshes of 9,800 triangles: some 180 us, now 21; of 33,000: 141, now 58).
// It stays for larger meshes: the searches, a sixteenth of n / 1024 chunks a
// lane, grow with the square (two of 65,500: the frame 389 us with these, 358
// with the radix sort).
constexpr uint32_t kTsortChunk = 1024, kTsortMax = 32768, kTsortMeshes = 16;
struct TsortBatch {
  TransMesh m[kTsortMeshes];
  uint32_t first[kTsortMeshes + 1];  // each mesh's first chunk
  uint32_t n;
  float cam[3];
};
__device__ inline uint32_t tsort_mesh(const TsortBatch& b, uint32_t chunk) {
  uint32_t m = 0;
  while (m + 1u < b.n && b.first[m + 1u] <= chunk) m++;
  return m;
}

__global__ __launch_bounds__(kTsortChunk) void k_tsort_chunks(TsortBatch b, unsigned long long* __restrict__ words,
                                                              uint32_t* __restrict__ tmp) {
  __shared__ unsigned long long s_x[2][kTsortChunk];
  const uint32_t tid = threadIdx.x, m = tsort_mesh(b, blockIdx.x);
  const TransMesh tm = b.m[m];
  const uint32_t i0 = (blockIdx.x - b.first[m]) * kTsortChunk, n = min(kTsortChunk, tm.n_tri - i0);
  const uint32_t* src = tm.tri + 9ull * i0;
  uint32_t* dst = tmp + 9ull * kTsortChunk * blockIdx.x;
  for (uint32_t w = tid; w < 9u * n; w += kTsortChunk) dst[w] = src[w];
  unsigned long long v = ~0ull;  // after every real word
  if (tid < n)
    v = (unsigned long long)tsort_key(src + 9u * tid, tm.pos, v3(b.cam[0], b.cam[1], b.cam[2])) << 32 | (i0 + tid);
  int buf = 0;
  for (uint32_t k = 2; k <= kTsortChunk; k <<= 1) {  // bitonic
    for (uint32_t j = k >> 1; j; j >>= 1) {
      unsigned long long o;
      if (j < 64u) {
        o = __shfl_xor(v, (int)j, 64);
      } else {
        s_x[buf][tid] = v;
        __syncthreads();
        o = s_x[buf][tid ^ j];
        buf ^= 1;  // the next exchange writes while slower waves still read this one
      }
      const bool low = ((tid & j) == 0u) == ((tid & k) == 0u);
      v = (o < v) == low ? o : v;
    }
  }
  words[(uint64_t)kTsortChunk * blockIdx.x + tid] = v;
}

__global__ __launch_bounds__(256) void k_tsort_merge(TsortBatch b, const unsigned long long* __restrict__ words,
                                                     const uint32_t* __restrict__ tmp) {
  const uint32_t e = (blockIdx.x * 256u + threadIdx.x) >> 4, l = threadIdx.x & 15u;
  const uint32_t chunk = e / kTsortChunk, m = tsort_mesh(b, chunk);
  const unsigned long long v = words[e];
  uint32_t rank = 0;
  if (v != ~0ull) {
    for (uint32_t c = b.first[m] + l; c < b.first[m + 1u]; c += 16u) {
      if (c == chunk) {
        rank += e % kTsortChunk;
        continue;
      }
      const unsigned long long* w = words + (uint64_t)kTsortChunk * c;
      uint32_t p = 0;  // words of the chunk below v
#pragma unroll
      for (uint32_t s = kTsortChunk / 2u; s; s >>= 1)
        if (w[p + s - 1u] < v) p += s;
      rank += p + (w[p] < v ? 1u : 0u);
    }
  }
#pragma unroll
  for (int o = 8; o; o >>= 1) rank += __shfl_xor(rank, o, 16);
  if (v != ~0ull && l < 9u)
    b.m[m].tri[9ull * rank + l] = tmp[9ull * ((uint64_t)kTsortChunk * b.first[m] + (uint32_t)v) + l];
}

// out[i] = tri[order[i]] (9 indices per triangle).
__global__ __launch_bounds__(256) void k_permute_tris(const uint32_t* __restrict__ tri,
                                                      const uint32_t* __restrict__ order, uint32_t n,
                                                      uint32_t* __restrict__ out) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n) return;
  const uint32_t* src = tri + 9ull * order[i];
  uint32_t* dst = out + 9ull * i;
#pragma unroll
  for (int k = 0; k < 9; k++) dst[k] = src[k];
}

// ============================================================= orchestration
static inline uint32_t cdiv(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

void enqueue_mesh_streams(const uint32_t* tri, uint32_t n_tri, const float* pos, const float* nrm, const float* uv,
                          float* soa, hipStream_t s) {
  if (n_tri == 0) return;
  hipLaunchKernelGGL(k_mesh_streams, dim3(std::min<uint32_t>(cdiv(n_tri, 256), 65535u)), dim3(256), 0, s, tri, n_tri,
                     pos, nrm, uv, soa);
}

// Stable LSD radix sort of (keys[0], vals[0]) by the low key_bits bits of the
// keys, *n_ptr items (at most cap): one 8-bit pass when key_bits <= 8, one
// 11-bit pass when key_bits <= 11, else 8-bit passes.  Returns the index of the
// buffer pair holding the result.  keys_out false: the sorted keys are not
// written (the values are).  ranges: when the sort is one pass (key_bits <= 11),
// [start, end) of each key below n_ranges in the sorted order; not written
// otherwise.
int enqueue_radix_sort(uint32_t* const keys[2], uint32_t* const vals[2], const uint32_t* n_ptr, uint32_t cap,
                       int key_bits, uint32_t* hist, uint32_t* partials, hipStream_t s, bool keys_out,
                       uint2* ranges, uint32_t n_ranges) {
  int cur = 0;
  // one 8-bit pass for keys of up to 8 bits, one 11-bit pass up to 11 bits
  const bool one_pass = key_bits > 8 && key_bits <= 11;
  const int step = one_pass ? 11 : 8;
  for (int shift = 0; shift < key_bits; shift += step) {
    const uint32_t nh = (one_pass ? 2048u : 256u) * kRadixW;
    const bool last = shift + step >= key_bits;
    const bool kout = !last || keys_out;
    uint2* const rg = (last && shift == 0) ? ranges : nullptr;
    const uint32_t nr = rg ? n_ranges : 0u;
    if (one_pass)
      hipLaunchKernelGGL(k_radix_hist<11>, dim3(kRadixG), dim3(256), 0, s, keys[cur], n_ptr, cap, shift, hist);
    else
      hipLaunchKernelGGL(k_radix_hist<8>, dim3(kRadixG), dim3(256), 0, s, keys[cur], n_ptr, cap, shift, hist);
    scan_u32(hist, hist, nullptr, nh, nh, partials, nullptr, 0, nullptr, 0, s);
    if (one_pass) {
      if (kout)
        hipLaunchKernelGGL((k_radix_scatter<11, true>), dim3(kRadixG), dim3(256), 0, s, keys[cur], vals[cur],
                           keys[cur ^ 1], vals[cur ^ 1], n_ptr, cap, shift, hist, rg, nr);
      else
        hipLaunchKernelGGL((k_radix_scatter<11, false>), dim3(kRadixG), dim3(256), 0, s, keys[cur], vals[cur],
                           keys[cur ^ 1], vals[cur ^ 1], n_ptr, cap, shift, hist, rg, nr);
    } else {
      if (kout)
        hipLaunchKernelGGL((k_radix_scatter<8, true>), dim3(kRadixG), dim3(256), 0, s, keys[cur], vals[cur],
                           keys[cur ^ 1], vals[cur ^ 1], n_ptr, cap, shift, hist, rg, nr);
      else
        hipLaunchKernelGGL((k_radix_scatter<8, false>), dim3(kRadixG), dim3(256), 0, s, keys[cur], vals[cur],
                           keys[cur ^ 1], vals[cur ^ 1], n_ptr, cap, shift, hist, rg, nr);
    }
    cur ^= 1;
  }
  return cur;
}

// Status reset, geometry, view bases and binning of one pipeline pass;
// returns the arguments the per-tile stages read (tile lists in b.vals[0]).
PipeArgs enqueue_front(const PipeArgs& a, hipStream_t s) {
  // near-first lists (k_pair_*); a frame of more tiles than their counters
  // take is binned in submission order
  const bool blend_lists = a.ordered_bins && a.blend_lists && a.n_tri_in <= kPairSubmitTris;
  const bool submit256 = blend_lists && a.n_tiles <= kPairFewTiles && submit_share(a.n_tri_in, a.n_tiles, 256u);
  const bool submit = submit256 || (blend_lists && submit_share(a.n_tri_in, a.n_tiles, 2048u));
  const bool near = (a.ordered_bins && a.depth_order && a.n_tiles <= kPairMaxTiles) || submit;
  // a small single-view frame is binned by one workgroup (k_bin_small)
  const bool one_bin = near && !submit && a.n_views == 1 && small_bins(a.n_tri_in, a.n_tiles);
  if (a.ev[0]) (void)hipEventRecord(a.ev[0], s);
  if (a.tables_src)  // (the transparent pass's were the opaque pass's work)
    hipLaunchKernelGGL(k_frame_begin, dim3(std::min<uint32_t>(cdiv(a.tables_words, 1024), 64u)), dim3(256), 0, s,
                       reinterpret_cast<uint32_t*>(a.status), (uint32_t)(2 * sizeof(Status) / 4), a.tables_src,
                       a.tables_dst, a.tables_words);
  const uint32_t n_blk = cdiv(a.n_tri_in, 256);
  uint8_t* const wflag = reinterpret_cast<uint8_t*>(a.big);
  // the wide-triangle list: near first in vals[1], which the pair kernels
  // leave alone; else in keys[1] until the radix sort needs it (both hold
  // cap_pairs >= cap_tri entries)
  uint32_t* const wide_list = near ? a.vals[1] : a.keys[1];
  // a small single-view frame: one workgroup builds the emitter lists
  const bool small_geom = a.n_views == 1 && a.n_tri_in <= kSmallBinTris;
  // 1-3 geometry with ordered compaction
  if (n_blk && small_geom) {
    hipLaunchKernelGGL(k_geom_small, dim3(1), dim3(1024), 0, s, a.draws, a.n_draws, a.views, a.n_tri_in, a.cnt, a.blk,
                       a.status, a.cap_tri, a.surv);
  } else if (n_blk) {
    uint32_t* blk_simple = a.blk + geom_blk_stride(n_blk);
    uint32_t* blk_clip = a.blk + 2 * geom_blk_stride(n_blk);
    hipLaunchKernelGGL(k_geom_count, dim3(n_blk), dim3(256), 0, s, a.draws, a.n_draws, a.views, a.n_tri_in, a.cnt,
                       a.blk, blk_simple, blk_clip);
    ScanSegs g{};
    g.s[0] = ScanSeg{a.blk, a.blk, &a.status->n_out, &a.status->overflow, a.cap_tri, 1u};
    g.s[1] = ScanSeg{blk_simple, blk_simple, &a.status->n_simple, nullptr, 0u, 0u};
    g.s[2] = ScanSeg{blk_clip, blk_clip, &a.status->n_clip, nullptr, 0u, 0u};
    hipLaunchKernelGGL(k_scan_segs, dim3(3), dim3(1024), 0, s, g, n_blk);
    hipLaunchKernelGGL(k_geom_compact, dim3(cdiv(n_blk, 4)), dim3(256), 0, s, a.n_tri_in, a.cnt, a.blk, blk_simple, blk_clip,
                       a.status, a.surv);
  }
  if (n_blk) {
    // at most twice the blocks that fit, to even out the units (their number is on the device)
    const dim3 ge(std::min<uint32_t>(2u * n_blk, 2048u));
    const uint32_t span = (uint64_t)a.n_tri_in >= (uint64_t)a.n_pixels ? kSparseSpanDense : kSparseSpan;
    if (near)
      hipLaunchKernelGGL(k_geom_emit<kBinNear>, ge, dim3(256), 0, s, a.draws, a.n_draws, a.views, a.surv, a.cnt, a.mats,
                         a.setup, a.shade, a.cap_tri, a.status, a.TS, nullptr, wflag, wide_list, span);
    else if (a.ordered_bins)
      hipLaunchKernelGGL(k_geom_emit<kBinSubmit>, ge, dim3(256), 0, s, a.draws, a.n_draws, a.views, a.surv, a.cnt,
                         a.mats, a.setup, a.shade, a.cap_tri, a.status, a.TS, a.bincnt, wflag, nullptr, span);
    else
      hipLaunchKernelGGL(k_geom_emit<kBinNone>, ge, dim3(256), 0, s, a.draws, a.n_draws, a.views, a.surv, a.cnt,
                         a.mats, a.setup, a.shade, a.cap_tri, a.status, a.TS, nullptr, nullptr, nullptr, span);
  }
  if (a.n_views > 1)
    hipLaunchKernelGGL(k_view_id_base, dim3(cdiv(a.n_views, 4)), dim3(256), 0, s, const_cast<DevView*>(a.views),
                       a.n_views, a.n_tri_in, a.cnt, a.blk, a.status);
  if (a.ev[1]) (void)hipEventRecord(a.ev[1], s);
  // 4-8 binning
  const uint32_t gb = std::min<uint32_t>(cdiv(a.cap_tri, 256), 4096u);
  const uint32_t gl = std::min<uint32_t>(cdiv(a.cap_tri, 4096), 1024u);
  const uint32_t gw = std::min<uint32_t>(cdiv(a.cap_tri, 64), 4096u);
  PipeArgs b = a;
  if (one_bin) {
    hipLaunchKernelGGL(k_bin_small, dim3(1), dim3(1024), 0, s, a.setup, a.views, a.status, a.cap_tri, a.TS, wflag,
                       wide_list, a.n_tiles, a.cap_pairs, a.vals[0], a.ranges);
  } else if (near) {
    uint2* const pairs = reinterpret_cast<uint2*>(a.keys[0]);  // keys[0] and keys[1] are one buffer
    const bool few = submit ? submit256 : a.n_tiles <= kPairFewTiles;
    const uint32_t dig = few ? 256u : 2048u;
    uint32_t* const totals = a.hist + (size_t)dig * kPairCols;
    const dim3 gp(kPairCols), bp(kPairT);
    if (few)
      hipLaunchKernelGGL(k_pair_hist<256>, gp, bp, 0, s, wflag, wide_list, a.setup, a.views, a.status, a.cap_tri, a.TS,
                         a.hist);
    else
      hipLaunchKernelGGL(k_pair_hist<2048>, gp, bp, 0, s, wflag, wide_list, a.setup, a.views, a.status, a.cap_tri,
                         a.TS, a.hist);
    hipLaunchKernelGGL(k_row_scan, dim3(dig), dim3(kPairCols), 0, s, a.hist, totals);
    auto lists = [&](auto scatter, auto sort) {
      hipLaunchKernelGGL(scatter, gp, bp, 0, s, wflag, wide_list, a.setup, a.views, a.status, a.cap_tri, a.TS, a.hist,
                         totals, a.cap_pairs, pairs);
      hipLaunchKernelGGL(sort, dim3(dig), dim3(kSortT), 0, s, pairs, totals, a.cap_pairs, a.n_tiles, a.vals[0],
                         a.ranges, a.vals[1]);  // (the wide list there has been read)
    };
    if (submit) {
      if (few) lists(k_pair_scatter<256, true>, k_pair_sort<256, true>);
      else lists(k_pair_scatter<2048, true>, k_pair_sort<2048, true>);
      b.vals[0] = a.vals[1];
    } else {
      if (few) lists(k_pair_scatter<256, false>, k_pair_sort<256, false>);
      else lists(k_pair_scatter<2048, false>, k_pair_sort<2048, false>);
    }
  } else if (a.ordered_bins) {
    hipLaunchKernelGGL(k_wide_list, dim3(gl), dim3(256), 0, s, wflag, a.status, a.cap_tri, wide_list,
                       reinterpret_cast<uint32_t*>(a.ranges), 2u * a.n_tiles);
    hipLaunchKernelGGL(k_bin_count_wide<true>, dim3(gw), dim3(256), 0, s, a.setup, a.views, a.status, a.TS,
                       wide_list, a.bincnt, a.tile_cnt);
    scan_u32(a.bincnt, a.binoff, &a.status->n_out, 0, a.cap_tri, a.partials, &a.status->n_pairs, a.cap_pairs,
             &a.status->overflow, 2u, s);
    hipLaunchKernelGGL(k_bin_emit<true>, dim3(gb), dim3(256), 0, s, a.setup, a.views, a.status, a.cap_tri, a.TS,
                       wflag, a.binoff, a.tile_start, a.tile_cur, a.cap_pairs, a.keys[0], a.vals[0]);
    hipLaunchKernelGGL(k_bin_emit_wide<true>, dim3(gw), dim3(256), 0, s, a.setup, a.views, a.status, wide_list,
                       a.TS, a.binoff, a.tile_start, a.tile_cur, a.cap_pairs, a.keys[0], a.vals[0]);
    // radix sort by tile key (one pass when the key has at most 11 bits, else
    // stable 8-bit passes), then the tile ranges: from the one pass's scanned
    // histogram, else from the sorted keys
    const bool one_pass = a.key_bits <= 11;
    const int cur = enqueue_radix_sort(a.keys, a.vals, &a.status->n_pairs, a.cap_pairs, a.key_bits, a.hist,
                                       a.partials, s, !one_pass, one_pass ? a.ranges : nullptr, a.n_tiles);
    b.vals[0] = a.vals[cur];
    if (!one_pass)
      hipLaunchKernelGGL(k_tile_ranges, dim3(std::min<uint32_t>(cdiv(a.cap_pairs, 256), 4096u)), dim3(256), 0, s,
                         a.keys[cur], &a.status->n_pairs, a.cap_pairs, a.ranges);
  } else {
    hipLaunchKernelGGL(k_fill_u32, dim3(std::min<uint32_t>(cdiv(2ull * a.n_tiles, 256), 2048u)), dim3(256), 0, s,
                       a.tile_cnt, 0u, 2u * a.n_tiles);  // tile_cnt and tile_cur are adjacent
    hipLaunchKernelGGL(k_bin_count, dim3(gb), dim3(256), 0, s, a.setup, a.views, a.status, a.cap_tri, a.TS,
                       a.tile_cnt, wflag);
    hipLaunchKernelGGL(k_wide_list, dim3(gl), dim3(256), 0, s, wflag, a.status, a.cap_tri, wide_list, nullptr, 0u);
    hipLaunchKernelGGL(k_bin_count_wide<false>, dim3(gw), dim3(256), 0, s, a.setup, a.views, a.status, a.TS,
                       wide_list, a.bincnt, a.tile_cnt);
    scan_u32(a.tile_cnt, a.tile_start, nullptr, a.n_tiles, a.n_tiles, a.partials, &a.status->n_pairs, a.cap_pairs,
             &a.status->overflow, 2u, s);
    hipLaunchKernelGGL(k_bin_emit<false>, dim3(gb), dim3(256), 0, s, a.setup, a.views, a.status, a.cap_tri, a.TS,
                       wflag, a.binoff, a.tile_start, a.tile_cur, a.cap_pairs, a.keys[0], a.vals[0]);
    hipLaunchKernelGGL(k_bin_emit_wide<false>, dim3(gw), dim3(256), 0, s, a.setup, a.views, a.status, wide_list,
                       a.TS, a.binoff, a.tile_start, a.tile_cur, a.cap_pairs, a.keys[0], a.vals[0]);
    hipLaunchKernelGGL(k_ranges_from_counts, dim3(std::min<uint32_t>(cdiv(a.n_tiles, 256), 2048u)), dim3(256), 0, s,
                       a.tile_start, a.tile_cnt, a.n_tiles, a.cap_pairs, a.ranges);
  }
  if (a.ev[2]) (void)hipEventRecord(a.ev[2], s);
  return b;
}

// Before the transparent pass: object-group bases of the opaque ids (from
// the opaque pass's counts, still in cnt/blk), then each transparent mesh
// sorted back to front in place -- the mesh keeps the new order, as the
// reference's sort_by on the mesh's triangle vector does.
void enqueue_transparent_prep(const PipeArgs& opaque, const TransArgs& t, hipStream_t s) {
  if (t.n_groups)
    hipLaunchKernelGGL(k_group_base, dim3(cdiv(t.n_groups, 4)), dim3(256), 0, s, t.grp_first, t.n_groups,
                       opaque.n_tri_in, opaque.cnt, opaque.blk, opaque.status, t.grp_base);
  // a batch's triangles fit perm_tmp, their words the pair buffer (a mesh alone always does)
  const uint32_t max_chunks = std::min(t.perm_chunks, opaque.cap_pairs / kTsortChunk);
  TsortBatch b{};
  for (int k = 0; k < 3; k++) b.cam[k] = t.cam[k];
  auto sort_batch = [&]() {
    const uint32_t chunks = b.first[b.n];
    if (chunks) {
      unsigned long long* const words = reinterpret_cast<unsigned long long*>(opaque.keys[0]);
      hipLaunchKernelGGL(k_tsort_chunks, dim3(chunks), dim3(kTsortChunk), 0, s, b, words, t.perm_tmp);
      hipLaunchKernelGGL(k_tsort_merge, dim3(chunks * (kTsortChunk / 16u)), dim3(256), 0, s, b, words, t.perm_tmp);
    }
    b.n = 0;
  };
  for (uint32_t m = 0; m < t.n_meshes; m++) {
    const TransMesh& tm = t.meshes[m];
    if (tm.n_tri < 2) continue;
    if (tm.n_tri <= kTsortMax) {
      const uint32_t chunks = cdiv(tm.n_tri, kTsortChunk);
      bool seen = false;  // drawn twice: sorted once
      for (uint32_t k = 0; k < b.n; k++) seen |= b.m[k].tri == tm.tri;
      if (seen) continue;
      if (b.n == kTsortMeshes || (b.n && b.first[b.n] + chunks > max_chunks)) sort_batch();
      b.m[b.n] = tm;
      b.first[b.n + 1u] = b.first[b.n] + chunks;
      b.n++;
      continue;
    }
    sort_batch();
    hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(64), 0, s, t.sort_n, tm.n_tri, 1u);
    hipLaunchKernelGGL(k_tsort_keys, dim3(cdiv(tm.n_tri, 256)), dim3(256), 0, s, tm.tri, tm.n_tri, tm.pos,
                       t.cam[0], t.cam[1], t.cam[2], opaque.keys[0], opaque.vals[0]);
    const int cur = enqueue_radix_sort(opaque.keys, opaque.vals, t.sort_n, opaque.cap_pairs, 32, opaque.hist,
                                       opaque.partials, s, false, nullptr, 0u);
    hipLaunchKernelGGL(k_permute_tris, dim3(cdiv(tm.n_tri, 256)), dim3(256), 0, s, tm.tri, opaque.vals[cur],
                       tm.n_tri, t.perm_tmp);
    (void)hipMemcpyAsync(tm.tri, t.perm_tmp, 36ull * tm.n_tri, hipMemcpyDeviceToDevice, s);
  }
  sort_batch();
}

// The frame's status words into coherent pinned host memory (one wave, in
// stream order after every kernel that writes them).
__global__ void k_status_out(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst, uint32_t n_words) {
  for (uint32_t i = threadIdx.x; i < n_words; i += blockDim.x) dst[i] = src[i];
  __threadfence_system();
}

void enqueue_status_out(const Status* dev, Status* host_dev_ptr, uint32_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_status_out, dim3(1), dim3(64), 0, s, reinterpret_cast<const uint32_t*>(dev),
                     reinterpret_cast<uint32_t*>(host_dev_ptr), (uint32_t)(n * sizeof(Status) / 4));
}

// One shard of a sort-last frame: geometry, binning, raster, then the packed
// u64 visibility (no shading: dh_shade_shard shades after the merge).
void enqueue_visibility(const PipeArgs& a, uint32_t shard, uint64_t* out, hipStream_t s) {
  PipeArgs b = enqueue_front(a, s);
  b.pack_out = out;
  b.pack_tag = shard << kShardShift;
  enqueue_raster(b, s);
  if (a.ev[3]) (void)hipEventRecord(a.ev[3], s);
  if (a.raster_kind != 0) enqueue_vis_pack(a, shard, out, s);
  if (a.ev[4]) (void)hipEventRecord(a.ev[4], s);
}

void enqueue_frame(const PipeArgs& a, hipStream_t s) {
  PipeArgs b = enqueue_front(a, s);
  // raster, shade (dh_raster.hip): the kind-0 raster shades its own tiles
  b.shade_in_raster = a.raster_kind == 0;
  enqueue_raster(b, s);
  if (a.ev[3]) (void)hipEventRecord(a.ev[3], s);
  if (!b.shade_in_raster) enqueue_shade(a, s);
  if (a.ev[4]) (void)hipEventRecord(a.ev[4], s);
}

}  // namespace dh
