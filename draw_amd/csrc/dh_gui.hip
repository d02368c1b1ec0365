// dh_gui.hip -- the GUI overlay rasterizer: Gui::render (app/gui.rs:382-478)
// over Canvas::draw_triangle (canvas.rs:435-575).  Per-vertex colour and
// alpha, the RGBA font texture through get_rgba_slice (floor(u * w), not
// w - 1; scene/mod.rs:137-152), a per-command clip rectangle, Pixel products
// truncated to u8 and sums wrapping, depth tested against 0 and never
// written.  Fragments blend over the current pixel, so each pixel applies
// the draw list in order: one wave per 8x8 pixels scans the triangles'
// rectangles 64 at a time and visits, in order, those that meet its pixels.
#include "dh_common.hpp"
#include "dh_internal.hpp"

namespace dh {

struct alignas(16) GuiRec {
  float ea[4], eb[4], eg[4];  // edge functions bc, ca, ab: A, B, C, D
  float f[4];                 // f_alpha, f_beta, f_gama, -
  float uv[6];                // texture coordinates after the 1 - v flip
  float alpha[3];             // vertex alpha col[3] / 255
  uint32_t rgb[3];            // vertex colour r | g << 8 | b << 16
  uint32_t x0, x1, y0, y1;    // inclusive scan rectangle
  uint32_t ties, pad[2];      // ties: bits 0-2 the edges' tie rule, kGuiFast
};
// every record, then 8 bytes per triangle: x0 | x1 << 16, y0 | y1 << 16
static_assert(sizeof(GuiRec) + sizeof(uint2) == kGuiRecBytes && sizeof(GuiRec) % 16 == 0, "GuiRec layout");
constexpr uint32_t kGuiFast = 8u;  // normalizers finite and nonzero: coverage without division (covered_fast)

// The draw list from the caller's pinned staging into device memory (16 bytes
// a lane), so that one stream-ordered launch replaces three copies.
__global__ __launch_bounds__(256) void k_gui_upload(const uint4* __restrict__ src, uint4* __restrict__ dst, uint32_t n) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

// Edge function of (p, q) as A, B, C, D: ((A x + B y) + C) - D, canvas.rs:461-480.
__device__ inline void edge_of(float px, float py, float qx, float qy, float e[4]) {
  e[0] = py - qy;
  e[1] = qx - px;
  e[2] = px * qy;
  e[3] = qx * py;
}

// Rectangle from_coords / clip on (x0, y0, x1, y1) inclusive (canvas.rs:315-350).
struct Rect { uint64_t x0, y0, x1, y1; };
__device__ inline Rect rect_from(uint64_t a, uint64_t b, uint64_t c, uint64_t d) {
  Rect r;
  r.x0 = a < c ? a : c; r.x1 = a < c ? c : a;
  r.y0 = b < d ? b : d; r.y1 = b < d ? d : b;
  return r;
}
__device__ inline Rect rect_clip(const Rect& a, const Rect& b) {
  uint64_t x0 = a.x0 > b.x0 ? a.x0 : b.x0, y0 = a.y0 > b.y0 ? a.y0 : b.y0;
  uint64_t x1 = a.x1 < b.x1 ? a.x1 : b.x1, y1 = a.y1 < b.y1 ? a.y1 : b.y1;
  if (x0 > x1) { x0 = 0; x1 = 0; }
  if (y0 > y1) { y0 = 0; y1 = 0; }
  return rect_from(x0, y0, x1, y1);
}

__global__ __launch_bounds__(256) void k_gui_setup(const dh_gui_vertex* __restrict__ vtx, const uint4* __restrict__ tris,
                                                   uint32_t n_tri, const uint4* __restrict__ clips, int W, int H,
                                                   GuiRec* __restrict__ recs, uint2* __restrict__ rects) {
  const uint32_t t = blockIdx.x * 256u + threadIdx.x;
  if (t >= n_tri) return;
  const uint4 q = tris[t];
  const uint32_t vi[3] = {q.x, q.y, q.z};
  float cx[3], cy[3];
  GuiRec r;
  for (int k = 0; k < 3; k++) {  // gui.rs:420-466: invert y, flip v, alpha = col[3] / 255
    const dh_gui_vertex& v = vtx[vi[k]];
    const float sx = v.pos[0], sy = ((float)H - 1.0f) - v.pos[1];
    cx[k] = floorf(sx + 0.5f);  // pos_map_center, canvas.rs:896-904 (no canvas offset)
    cy[k] = floorf(sy + 0.5f);
    r.uv[2 * k] = v.uv[0];
    r.uv[2 * k + 1] = 1.0f - v.uv[1];
    r.alpha[k] = (float)v.col[3] / 255.0f;
    r.rgb[k] = (uint32_t)v.col[0] | ((uint32_t)v.col[1] << 8) | ((uint32_t)v.col[2] << 16);
  }
  edge_of(cx[1], cy[1], cx[2], cy[2], r.ea);  // f_bc
  edge_of(cx[2], cy[2], cx[0], cy[0], r.eb);  // f_ca
  edge_of(cx[0], cy[0], cx[1], cy[1], r.eg);  // f_ab
  r.f[0] = edge_eval(r.ea, cx[0], cy[0]);
  r.f[1] = edge_eval(r.eb, cx[1], cy[1]);
  r.f[2] = edge_eval(r.eg, cx[2], cy[2]);
  r.f[3] = 0.0f;
  r.ties = 0;
  if (r.f[0] * edge_eval(r.ea, -1.0f, -1.0f) > 0.0f) r.ties |= 1u;
  if (r.f[1] * edge_eval(r.eb, -1.0f, -1.0f) > 0.0f) r.ties |= 2u;
  if (r.f[2] * edge_eval(r.eg, -1.0f, -1.0f) > 0.0f) r.ties |= 4u;
  if (isfinite(r.f[0]) && isfinite(r.f[1]) && isfinite(r.f[2]) && r.f[0] != 0.0f && r.f[1] != 0.0f && r.f[2] != 0.0f)
    r.ties |= kGuiFast;
  float mnx = INFINITY, mny = INFINITY, mxx = -INFINITY, mxy = -INFINITY;  // canvas.rs:491-510
  for (int k = 0; k < 3; k++) {
    if (cx[k] < mnx) mnx = cx[k];
    if (cy[k] < mny) mny = cy[k];
    if (cx[k] > mxx) mxx = cx[k];
    if (cy[k] > mxy) mxy = cy[k];
  }
  Rect drawable = rect_from(f2usize(mnx), f2usize(mny), f2usize(mxx), f2usize(mxy));
  drawable = rect_clip(drawable, rect_from(0, 0, (uint64_t)W - 1u, (uint64_t)H - 1u));
  const uint4 cl = clips[q.w];
  const Rect valid = rect_clip(rect_from(cl.x, cl.y, cl.z, cl.w), drawable);
  r.x0 = (uint32_t)valid.x0; r.x1 = (uint32_t)valid.x1;
  r.y0 = (uint32_t)valid.y0; r.y1 = (uint32_t)valid.y1;
  r.pad[0] = r.pad[1] = 0;
  recs[t] = r;
  // What the raster visits.  A triangle outside its clip rectangle collapses to
  // row or column 0 (rect_clip), where it covers nothing, but those rectangles
  // would all meet at the canvas's edge.  With every partial sum of the edge
  // functions over the vertices and the rectangle below 2^24 they are exact, so
  // a pixel outside the triangle's bounding box is outside the triangle: a
  // rectangle that misses the box is left out.
  const float R = fmaxf(fmaxf(fmaxf(fabsf(mnx), fabsf(mxx)), fmaxf(fabsf(mny), fabsf(mxy))),
                        fmaxf((float)r.x1, (float)r.y1));
  auto exact_edge = [R](const float e[4]) {
    return ((fabsf(e[0]) * R + fabsf(e[1]) * R) + fabsf(e[2])) + fabsf(e[3]) < 16777000.0f;
  };
  const bool outside = (float)r.x1 < mnx || (float)r.x0 > mxx || (float)r.y1 < mny || (float)r.y0 > mxy;
  if (outside && (r.ties & kGuiFast) && exact_edge(r.ea) && exact_edge(r.eb) && exact_edge(r.eg))
    rects[t] = make_uint2(0xFFFFu, 0xFFFFu);  // x0 > x1: meets nothing
  else
    rects[t] = make_uint2(r.x0 | (r.x1 << 16), r.y0 | (r.y1 << 16));  // inside the canvas: below 65535
}

// get_rgba_slice (scene/mod.rs:137-152) in release semantics: false when the
// 4-byte slice leaves the image (the reference panics).
__device__ inline bool rgba_offset(int32_t w, int32_t h, int32_t comp, float u, float v, uint64_t* off) {
  const uint64_t ui = f2usize(floorf(u * (float)w));
  const uint64_t vi = ((uint64_t)h - 1u) - f2usize(floorf(v * (float)h));
  const uint64_t o = (vi * (uint64_t)w + ui) * (uint64_t)comp;
  const uint64_t end = o + 4u, len = (uint64_t)w * (uint64_t)h * (uint64_t)comp;
  *off = o;
  return !(o > end || end > len);
}

// Pixel * f32 then Pixel + Pixel per channel (canvas.rs:136-169).
__device__ inline uint32_t pmul(uint32_t p, float s) {
  return f2u8((float)(p & 255u) * s) | (f2u8((float)((p >> 8) & 255u) * s) << 8) |
         (f2u8((float)((p >> 16) & 255u) * s) << 16);
}
__device__ inline uint32_t padd(uint32_t a, uint32_t b) {
  return ((a + b) & 255u) | ((((a >> 8) + (b >> 8)) & 255u) << 8) | ((((a >> 16) + (b >> 16)) & 255u) << 16);
}

// One wave per 8x8 pixels, four to a 16x16 tile, each on its own: no barrier
// and no shared list.  The wave scans the rectangles (8 bytes a triangle, 256
// in flight) and visits the ones that meet its pixels in draw order.  A
// visited record is the same for all lanes, so it arrives by scalar loads;
// most of the time is the latency of that load and of the texel behind it.
// Two triangles are therefore taken at once: a fragment's own colour and
// alpha do not depend on the canvas, only the blend does, so both are
// computed with their loads in flight together and then blended in order.
// Coverage comes first and without division where the normalizers allow it,
// so a triangle that covers none of the 64 pixels costs no division and no
// texel, be it the other one of its pair or not (the two halves of a panel
// rarely share a wave's pixels: 50 panels over a 3840x2160 canvas took 3640 us
// one triangle at a time, 3900 with both of every pair shaded and 2530 now).
// (2400 triangles over 800x600: 560 us with one list per 16x16 tile, records
// read per lane, one triangle at a time and the collapsed clip rectangles
// visited; 27 us with this kernel.)
__global__ __launch_bounds__(256) void k_gui_raster(const GuiRec* __restrict__ recs, const uint2* __restrict__ rects,
                                                    uint32_t n_tri, int W, int H, uint32_t ntx,
                                                    const uint8_t* __restrict__ font, int32_t fw, int32_t fh,
                                                    int32_t fcomp, uint32_t* __restrict__ bgra,
                                                    const float* __restrict__ depth, uint32_t* __restrict__ error) {
  const uint32_t tile = xcd_remap_tiles(blockIdx.x, gridDim.x);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int qx0 = (int)(tile % ntx) * 16 + (wave & 1) * 8, qy0 = (int)(tile / ntx) * 16 + (wave >> 1) * 8;
  if (qx0 >= W || qy0 >= H) return;  // the whole wave
  const int px = qx0 + (lane & 7), py = qy0 + (lane >> 3);
  const bool ok = px < W && py < H;
  const float xf = (float)px, yf = (float)py;
  // the canvas keeps rgb in r, g, b order inside its B,G,R,A words
  uint32_t cur = 0;
  bool pass = false;
  if (ok) {
    const uint32_t w = bgra[(uint32_t)(H - 1 - py) * (uint32_t)W + (uint32_t)px];
    cur = ((w >> 16) & 255u) | (w & 0xFF00u) | ((w & 255u) << 16);
    pass = 0.0f < depth[(uint32_t)py * (uint32_t)W + (uint32_t)px];
  }
  bool wrote = false;
  constexpr int kPair = 2;
  auto visit = [&](const uint32_t (&t)[kPair], int n) {
    float e[kPair][3];
    bool cov[kPair], on[kPair];  // on: for some pixel of the wave
#pragma unroll
    for (int k = 0; k < kPair; k++) {
      const GuiRec& r = recs[t[k]];
      cov[k] = k < n && ok && px >= (int)r.x0 && px <= (int)r.x1 && py >= (int)r.y0 && py <= (int)r.y1;
      e[k][0] = edge_eval(r.ea, xf, yf);
      e[k][1] = edge_eval(r.eb, xf, yf);
      e[k][2] = edge_eval(r.eg, xf, yf);
      if (r.ties & kGuiFast)
        cov[k] = cov[k] && covered_fast(e[k][0], r.f[0], r.ties & 1u) && covered_fast(e[k][1], r.f[1], r.ties & 2u) &&
                 covered_fast(e[k][2], r.f[2], r.ties & 4u);
      on[k] = __ballot(cov[k]) != 0ull;
    }
    float al[kPair], be[kPair], ga[kPair];
    uint32_t texel[kPair];
#pragma unroll
    for (int k = 0; k < kPair; k++) {
      if (!on[k]) continue;
      const GuiRec& r = recs[t[k]];
      al[k] = e[k][0] / r.f[0];
      be[k] = e[k][1] / r.f[1];
      ga[k] = e[k][2] / r.f[2];
      if (!(r.ties & kGuiFast))
        cov[k] = cov[k] && al[k] >= 0.0f && be[k] >= 0.0f && ga[k] >= 0.0f && (al[k] > 0.0f || (r.ties & 1u)) &&
                 (be[k] > 0.0f || (r.ties & 2u)) && (ga[k] > 0.0f || (r.ties & 4u));
      const float u = (r.uv[0] * al[k] + r.uv[2] * be[k]) + r.uv[4] * ga[k];
      const float v = (r.uv[1] * al[k] + r.uv[3] * be[k]) + r.uv[5] * ga[k];
      uint64_t off;
      if (!rgba_offset(fw, fh, fcomp, u, v, &off)) {
        if (cov[k]) *error = 1u;
        cov[k] = false;
      }
      if (!cov[k]) off = 0;  // four bytes that are always there (the texture's allocation is padded)
      if (fcomp == 4)
        texel[k] = *reinterpret_cast<const uint32_t*>(font + off);
      else
        texel[k] = (uint32_t)font[off] | ((uint32_t)font[off + 1] << 8) | ((uint32_t)font[off + 2] << 16) |
                   ((uint32_t)font[off + 3] << 24);
    }
#pragma unroll
    for (int k = 0; k < kPair; k++) {
      if (!on[k]) continue;
      const GuiRec& r = recs[t[k]];
      uint32_t col = padd(padd(pmul(r.rgb[0], al[k]), pmul(r.rgb[1], be[k])), pmul(r.rgb[2], ga[k]));
      const float calpha = (al[k] * r.alpha[0] + be[k] * r.alpha[1]) + ga[k] * r.alpha[2];
      const float ta = (float)(texel[k] >> 24) / 255.0f;
      col = padd(pmul(col, ta), pmul(texel[k], 1.0f - ta));
      const float fin = calpha * ta;
      const uint32_t out = fin < 1.0f ? padd(pmul(cur, 1.0f - fin), pmul(col, fin)) : col;
      if (cov[k] && pass) {  // draw_pixel_coord_with_depth(x, y, colour, alpha, 0.0); depth writes off
        cur = out;
        wrote = true;
      }
    }
  };
  constexpr int kRounds = 4;
  for (uint32_t base = 0; base < n_tri; base += 64u * kRounds) {
    uint2 q[kRounds];
#pragma unroll
    for (int u = 0; u < kRounds; u++) {
      const uint32_t t = base + 64u * (uint32_t)u + (uint32_t)lane;
      q[u] = t < n_tri ? rects[t] : make_uint2(0xFFFFu, 0xFFFFu);  // x0 > x1: meets nothing
    }
#pragma unroll
    for (int u = 0; u < kRounds; u++) {
      const int x0 = (int)(q[u].x & 0xFFFFu), x1 = (int)(q[u].x >> 16);
      const int y0 = (int)(q[u].y & 0xFFFFu), y1 = (int)(q[u].y >> 16);
      uint64_t m = __ballot(x1 >= qx0 && x0 <= qx0 + 7 && y1 >= qy0 && y0 <= qy0 + 7);
      while (m) {
        uint32_t t[kPair];
        int n = 0;
#pragma unroll
        for (int k = 0; k < kPair; k++) {
          t[k] = n ? t[0] : 0u;
          if (m) {
            t[k] = base + 64u * (uint32_t)u + (uint32_t)__builtin_ctzll(m);
            m &= m - 1;
            n++;
          }
        }
        visit(t, n);
      }
    }
  }
  if (ok && wrote)  // B, G, R and the pad byte 0 of a Pixel sum
    bgra[(uint32_t)(H - 1 - py) * (uint32_t)W + (uint32_t)px] =
        ((cur >> 16) & 255u) | (cur & 0xFF00u) | ((cur & 255u) << 16);
}

hipError_t enqueue_gui(const uint4* src, uint4* dst, const GuiLayout& g, uint32_t n_tri, void* recs, int W, int H,
                       const uint8_t* font, int32_t fw, int32_t fh, int32_t fcomp, uint32_t* bgra, const float* depth,
                       uint32_t* error, hipStream_t s) {
  if (n_tri == 0) return hipSuccess;
  GuiRec* r = reinterpret_cast<GuiRec*>(recs);
  uint2* rects = reinterpret_cast<uint2*>(r + n_tri);
  const uint32_t n16 = (uint32_t)(g.bytes / 16u);
  hipLaunchKernelGGL(k_gui_upload, dim3((n16 + 255u) / 256u), dim3(256), 0, s, src, dst, n16);
  const uint8_t* d = reinterpret_cast<const uint8_t*>(dst);
  hipLaunchKernelGGL(k_gui_setup, dim3((n_tri + 255u) / 256u), dim3(256), 0, s,
                     reinterpret_cast<const dh_gui_vertex*>(d + g.vtx), reinterpret_cast<const uint4*>(d + g.tri), n_tri,
                     reinterpret_cast<const uint4*>(d + g.clip), W, H, r, rects);
  const uint32_t ntx = (uint32_t)((W + 15) / 16), nty = (uint32_t)((H + 15) / 16);
  hipLaunchKernelGGL(k_gui_raster, dim3(ntx * nty), dim3(256), 0, s, r, rects, n_tri, W, H, ntx, font, fw, fh, fcomp,
                     bgra, depth, error);
  return hipGetLastError();
}

}  // namespace dh
