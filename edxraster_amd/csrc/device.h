// device.h -- device functions shared by the kernels of the general path
// (pipeline.hip) and of direct frames (direct.hip): wave operations, vertex and
// triangle setup, tile enumeration, rasterisation of a tile's references into
// LDS keys, and shading.  Internal: HIP sources of this folder only.
//
// The two sets of kernels are compiled apart: with k_tile beside it, k_raster
// came out with 54 instead of 36 spilled scalar registers (sphere grid 46 -> 50
// us).
#pragma once
#include <hip/hip_runtime.h>

#include "pipeline.h"

namespace edxr {

namespace {

constexpr uint32_t kWave = 64;
constexpr uint32_t kBlock = 256;
static_assert(kBlock == kJobTableBlock, "block -> job tables are indexed by 256-slot block");

// p in device memory.  A pointer read from memory would be loaded through as a
// generic one, and such a load also counts against the LDS waits: a kernel that
// loads ahead and works in LDS then waits for its loads with each LDS result.
template <class T>
using GlobalPtr = const __attribute__((address_space(1))) T*;
template <class T>
__device__ __forceinline__ GlobalPtr<T> as_global(const T* p) {
    return (GlobalPtr<T>)p;
}
template <class T>
__device__ __forceinline__ T global_at(const T* p, size_t i) {
    return as_global(p)[i];
}

__device__ __forceinline__ float4 xform4(const float* m, float x, float y, float z, float w) {
    float4 r;
    r.x = ((m[0] * x + m[1] * y) + m[2] * z) + m[3] * w;
    r.y = ((m[4] * x + m[5] * y) + m[6] * z) + m[7] * w;
    r.z = ((m[8] * x + m[9] * y) + m[10] * z) + m[11] * w;
    r.w = ((m[12] * x + m[13] * y) + m[14] * z) + m[15] * w;
    return r;
}

// Clipper::ComputeClipCode (Core/Clipper.h:48-68).
__device__ __forceinline__ uint32_t clip_code(const float4& v) {
    uint32_t c = 0;
    if (v.x < -v.w) c |= 1u;
    if (v.x > v.w) c |= 2u;
    if (v.y < -v.w) c |= 4u;
    if (v.y > v.w) c |= 8u;
    if (v.z > v.w) c |= 32u;
    if (v.z < 0.0f) c |= 16u;
    return c;
}

// ---- Quotients, rounded as the division operator and sqrtf round them ----
// Where no step can under- or overflow, one Newton step with fused
// multiply-adds from the hardware's estimate gives the correctly rounded
// reciprocal, and one residual step a correctly rounded quotient or square root
// (P. Markstein, "Computation of elementary functions on the IBM RISC System/6000
// processor", 1990): 3 and 3 instructions, not the 10 of a division whose operands
// may be anything.  tests/test_quotients_all.py compares the bits with those of
// 1.0f / x and 1.0f / sqrtf(x) for every float, and of projections for 2^35 points a
// seed.  2.1M sphere grid at 1080p, 4 samples: k_shade 47.3 us with divisions, 41.8 so
// (16 colours of a pixel are divided by 255), a call 217.3 and 215.0; k_tile of 98K
// triangles 23.6 and 22.2, a call 49.2 and 47.5.  Larger frames are bound by the
// gathers of vertices: k_shade of the 10M heightfield at 4K 75.0 and 71.8, of 256 jobs
// 453 and 449, the calls within their spread.  Vertices are transformed with
// divisions: k_vertex is bound by memory (256 jobs 173 us, 177 so).

// Whether x lies in [2^lo, 2^hi) (not a negative number or NaN).
template <int kLo, int kHi>
__device__ __forceinline__ bool in_range(float x) {
    return __float_as_uint(x) - ((uint32_t)(127 + kLo) << 23) < (uint32_t)(kHi - kLo) << 23;
}
// 1 / x of |x| in [2^-124, 2^125).
__device__ __forceinline__ float rcp_normal(float x) {
    const float y = __builtin_amdgcn_rcpf(x);
    return __builtin_fmaf(__builtin_fmaf(-x, y, 1.0f), y, y);
}
// a / x from y = 1 / x: x in [2^-60, 2^60), |a| in [2^-64, 2^60], so that the quotient
// is a normal number (with |a| from 2^-100 on, one subnormal quotient in some 3e9 pairs came out
// one step off), or 0 (whose sign is lost).
__device__ __forceinline__ float quotient_normal(float a, float x, float y) {
    const float q = a * y;
    return __builtin_fmaf(__builtin_fmaf(-x, q, a), y, q);
}
// 1 / x and 1 / sqrtf(x) of any x.
__device__ __forceinline__ float reciprocal(float x) {
    if (in_range<-124, 125>(x)) return rcp_normal(x);
    return 1.0f / x;
}
__device__ __forceinline__ float reciprocal_sqrt(float x) {
    if (in_range<-100, 100>(x)) {
        const float y = __builtin_amdgcn_rsqf(x), s = x * y;
        return rcp_normal(__builtin_fmaf(__builtin_fmaf(-s, s, x), 0.5f * y, s));
    }
    return 1.0f / sqrtf(x);
}
// A clip-space point's homogeneous projection x / w, y / w, z / w and z * (1 / w).
// (A projection that only differs in the sign of a zero is the same to snap_point.)
__device__ __forceinline__ bool project_is_normal(const float4& c) {
    return in_range<-60, 60>(c.w) && fminf(fminf(fabsf(c.x), fabsf(c.y)), fabsf(c.z)) >= 0x1p-64f &&
           fmaxf(fmaxf(fabsf(c.x), fabsf(c.y)), fabsf(c.z)) <= 0x1p60f;
}
__device__ __forceinline__ float4 project_normal(const float4& c) {
    const float y = rcp_normal(c.w);
    return make_float4(quotient_normal(c.x, c.w, y), quotient_normal(c.y, c.w, y), quotient_normal(c.z, c.w, y),
                       c.z * y);
}
__device__ __forceinline__ float4 project_any(const float4& c) {
    return make_float4(c.x / c.w, c.y / c.w, c.z / c.w, c.z * (1.0f / c.w));
}

// 28.4 snap by truncation (Core/RasterTriangle.h:35-40); saturating, NaN -> 0.
__device__ __forceinline__ int snap(float a) {
    const float s = a * 16.0f;
    if (!(s == s)) return 0;
    if (s >= 2147483648.0f) return 0x7FFFFFFF;
    if (s <= -2147483648.0f) return (int)0x80000000;
    return (int)s;
}

// The raster matrix applied to a homogeneous-projected point and the 28.4 snap
// (Core/RasterTriangle.h:29-40).  An affine raster matrix gives w == 1, where
// v / 1 == v exactly and the divide is skipped.
__device__ __forceinline__ int2 snap_point(const FrameParams& P, float ax, float ay, float az) {
    const float4 A = xform4(P.raster, ax, ay, az, 1.0f);
    if (A.w == 1.0f) return make_int2(snap(A.x), snap(A.y));
    return make_int2(snap(A.x / A.w), snap(A.y / A.w));
}

// RasterTriangle::Setup from snapped vertices (Core/RasterTriangle.h:42-153);
// false when culled (det <= 0).
__device__ __forceinline__ bool setup_snapped(int x0, int y0, int x1, int y1, int x2, int y2, RasterRec& r) {
    const int B0 = y0 - y1, C0 = x1 - x0, B1 = y1 - y2, C1 = x2 - x1, B2 = y2 - y0, C2 = x0 - x2;
    const int det = C2 * B1 - C1 * B2;
    if (det <= 0) return false;
    r.x0 = x0; r.y0 = y0; r.x1 = x1; r.y1 = y1; r.x2 = x2; r.y2 = y2;
    r.inv_det = rcp_normal((float)det);
    r.info = corner_info(B0, C0, B1, C1, B2, C2);
    return true;
}

// RasterTriangle::Setup on homogeneous-projected points (Core/RasterTriangle.h:27-153).
__device__ __forceinline__ bool setup_record(const FrameParams& P, float ax, float ay, float az, float bx, float by,
                                             float bz, float cx, float cy, float cz, RasterRec& r) {
    const int2 a = snap_point(P, ax, ay, az), b = snap_point(P, bx, by, bz), c = snap_point(P, cx, cy, cz);
    return setup_snapped(a.x, a.y, b.x, b.y, c.x, c.y, r);
}

__device__ __forceinline__ uint64_t lanemask_lt() { return (1ull << __lane_id()) - 1ull; }
// Inclusive prefix sum over the wave, in registers: DPP row shifts by 1, 2,
// 4 and 8 scan each row of 16 lanes (lanes shifted in from outside the row
// read 0), then row broadcasts of lane 15 (into rows 1 and 3) and lane 31
// (into rows 2 and 3) carry the rows' totals; six v_add_u32_dpp instead of
// six LDS permutes.  Every lane of the wave must be active (DPP reads the
// neighbours' registers whatever the exec mask).
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true);   // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true);   // row_shr:2
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true);   // row_shr:4
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true);   // row_shr:8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);  // row_bcast:15
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);  // row_bcast:31
    return v;
}
// op over the wave's 64 lanes, the same DPP steps with lanes that have no
// source keeping the identity; the result (lane 63's) is returned to every
// lane.  Every lane must be active.
template <class Op>
__device__ __forceinline__ uint32_t wave_reduce(uint32_t v, uint32_t identity, Op op) {
    const int id = (int)identity;
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(id, (int)v, 0x111, 0xf, 0xf, false));
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(id, (int)v, 0x112, 0xf, 0xf, false));
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(id, (int)v, 0x114, 0xf, 0xf, false));
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(id, (int)v, 0x118, 0xf, 0xf, false));
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(id, (int)v, 0x142, 0xa, 0xf, false));
    v = op(v, (uint32_t)__builtin_amdgcn_update_dpp(id, (int)v, 0x143, 0xc, 0xf, false));
    return __builtin_amdgcn_readlane(v, 63);
}
__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
    return wave_reduce(v, 0u, [](uint32_t a, uint32_t b) { return a + b; });
}
__device__ __forceinline__ uint32_t wave_min(uint32_t v) {
    return wave_reduce(v, 0xFFFFFFFFu, [](uint32_t a, uint32_t b) { return a < b ? a : b; });
}
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
    return wave_reduce(v, 0u, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
}


__device__ __forceinline__ uint32_t wave_count(bool p) { return (uint32_t)__popcll(__ballot(p)); }

}  // namespace

// Sample offsets in 28.4 units per MSAA level, (x, y) per sample: the table of
// FrameBuffer::MultiSampleOffsets (Core/FrameBuffer.cpp:107-191).
static __constant__ int2 c_sample_offsets[kMaxSampleLevel + 1][32] = {
    {{0, 0}},
    {{4, 4}, {-4, -4}},
    {{-2, -6}, {6, -2}, {-6, 2}, {2, 6}},
    {{1, -3}, {-1, 3}, {5, 1}, {-3, -5}, {-5, 5}, {-7, -1}, {3, 7}, {7, -7}},
    {{1, 1}, {-1, -3}, {-3, 2}, {4, -1}, {-5, -2}, {2, 5}, {5, 3}, {3, -5}, {-2, 6}, {0, -7}, {-4, -6}, {-6, 4},
     {-8, 0}, {7, -4}, {6, 7}, {-7, -8}},
    {{1, 1}, {-1, -3}, {-3, 2}, {4, -1}, {-5, -2}, {2, 5}, {5, 3}, {3, -5}, {-2, 6}, {0, -7}, {-4, -6}, {-6, 4},
     {-8, 0}, {7, -4}, {6, 7}, {-7, -8}, {1, 3}, {-3, -3}, {-3, 0}, {6, -2}, {-7, -1}, {3, 4}, {7, 3}, {3, -6},
     {-2, 7}, {0, -4}, {-2, -5}, {-7, 6}, {-8, 3}, {4, -1}, {2, 7}, {4, -8}}};

namespace {
// Job of a block-uniform index i (the block -> job tables are null for a
// single job).  The result is wave-uniform, so job fields load as scalars.
__device__ __forceinline__ uint32_t job_of(const BatchParams& Q, const uint32_t* tbl, uint32_t i) {
    return Q.num_jobs == 1 ? 0u : __builtin_amdgcn_readfirstlane(tbl[i]);
}
}  // namespace

namespace {
// Screen values of a vertex at clip-space position c: the homogeneous
// projection and the snapped raster position, with the z-divide's z.
__device__ __forceinline__ ScreenVert screen_vert(const FrameParams& P, const float4& c) {
    ScreenVert sv;
    const int2 xy = snap_point(P, c.x / c.w, c.y / c.w, c.z / c.w);
    sv.x = xy.x;
    sv.y = xy.y;
    sv.z = c.z * (1.0f / c.w);
    sv.code = clip_code(c);
    return sv;
}

// The vertex in a slot of its job: screen and shading vertex.
__device__ __forceinline__ void vertex_slot(const FrameParams& P, uint32_t slot, ShadeVert* __restrict__ verts,
                                            ScreenVert* __restrict__ sverts) {
    const MeshPtrs& M = P.mesh;
    const uint32_t v = slot - P.vert_base;
    if (v >= P.num_vertices) return;
    const float px = global_at(M.px, v), py = global_at(M.py, v), pz = global_at(M.pz, v);
    // DefaultVertexShader::Execute: projectedPos = MVP * (p, 1); the outcode,
    // the homogeneous projection and the snapped raster position are per
    // vertex, so every unclipped triangle's setup reuses them.
    const float4 c = xform4(P.mvp, px, py, pz, 1.0f);
    const ScreenVert sv = screen_vert(P, c);
    // Shading vertices are written for vertices inside the frustum only: an
    // unclipped triangle has no other, and a clipped triangle's pieces use
    // vertices made by k_clip (which reads its inputs from the mesh) or
    // original vertices that lie inside every plane.
    if (sv.code == 0) {
        ShadeVert o;
        o.px = px;
        o.py = py;
        o.pz = pz;
        o.nx = global_at(M.nx, v);
        o.ny = global_at(M.ny, v);
        o.nz = global_at(M.nz, v);
        o.cr = M.cr ? global_at(M.cr, v) : 0.0f;
        o.cg = M.cg ? global_at(M.cg, v) : 0.0f;
        o.cb = M.cb ? global_at(M.cb, v) : 0.0f;
        o.inv_w = 1.0f / c.w;
        o.u = M.tu ? global_at(M.tu, v) : 0.0f;
        o.v = M.tv ? global_at(M.tv, v) : 0.0f;
        verts[slot] = o;
    }
    sverts[slot] = sv;
}
}  // namespace

namespace {
// Descriptor of an unclipped triangle's record in slot t.  When its clamped
// tile bbox spans at most 2x2 tiles, binning lists it in every bbox tile with
// no corner test (Core/Renderer.cpp:168-180), so the bbox alone (packed here,
// in the job's tile coordinates) enumerates its references; otherwise
// (t << 3) | 1.  Only a triangle shorter than kCompactExtent is compact (others
// of so small a clamped bbox reach far off the screen): the raster kernels
// take products of a compact triangle's differences in 24 bits.
__device__ __forceinline__ uint32_t compact_desc(const FrameParams& P, const RasterRec& r, uint32_t t) {
    const int Shift = kTileLog2 + 4;
    const int minTX = max(0, min(r.x0, min(r.x1, r.x2)) >> Shift);
    const int maxTX = min((int)P.tiles_x - 1, max(r.x0, max(r.x1, r.x2)) >> Shift);
    const int minTY = max(0, min(r.y0, min(r.y1, r.y2)) >> Shift);
    const int maxTY = min((int)P.tiles_y - 1, max(r.y0, max(r.y1, r.y2)) >> Shift);
    const int dx = maxTX - minTX, dy = maxTY - minTY;
    if (dx < 0 || dy < 0 || dx > 1 || dy > 1) return (t << 3) | 1u;
    const uint32_t ex = (uint32_t)max(r.x0, max(r.x1, r.x2)) - (uint32_t)min(r.x0, min(r.x1, r.x2));
    const uint32_t ey = (uint32_t)max(r.y0, max(r.y1, r.y2)) - (uint32_t)min(r.y0, min(r.y1, r.y2));
    if (max(ex, ey) >= kCompactExtent) return (t << 3) | 1u;
    // a pixel bounding box of kHeavyPixels or more: a whole wave's work in the raster
    const int bw = (int)(ex >> 4), bh = (int)(ey >> 4);
    const uint32_t heavy = bw * bh >= (int)kHeavyPixels ? kDescHeavy : 0u;
    return kDescCompact | heavy | (uint32_t)minTX | ((uint32_t)minTY << 14) | ((uint32_t)dx << 28) |
           ((uint32_t)dy << 29);
}
}  // namespace

// ---------------------------------------------------------------------------
// Binning (Core/Renderer.cpp:161-230): tile sets of a record.
// ---------------------------------------------------------------------------
namespace {

struct BinTri {
    int x0, y0, x1, y1, x2, y2;
    int B0, C0, B1, C1, B2, C2;
    int sb0, sb1, sb2;   // scalar top-left bias (Core/RasterTriangle.h:155-158)
    uint32_t info;
    int minTX, minTY, w, h;
    bool small;
};

__device__ __forceinline__ int scalar_bias(int ax, int ay, int bx, int by) {
    return ((by > ay) || (ay == by && ax > bx)) ? 0 : -1;
}

__device__ __forceinline__ void load_bin_tri(const FrameParams& P, const RasterRec& r, BinTri& b) {
    b.x0 = r.x0; b.y0 = r.y0; b.x1 = r.x1; b.y1 = r.y1; b.x2 = r.x2; b.y2 = r.y2;
    b.B0 = b.y0 - b.y1; b.C0 = b.x1 - b.x0;
    b.B1 = b.y1 - b.y2; b.C1 = b.x2 - b.x1;
    b.B2 = b.y2 - b.y0; b.C2 = b.x0 - b.x2;
    b.sb0 = scalar_bias(b.x0, b.y0, b.x1, b.y1);
    b.sb1 = scalar_bias(b.x1, b.y1, b.x2, b.y2);
    b.sb2 = scalar_bias(b.x2, b.y2, b.x0, b.y0);
    b.info = r.info;
    const int Shift = kTileLog2 + 4;
    const int minTX = max(0, min(b.x0, min(b.x1, b.x2)) >> Shift);
    const int maxTX = min((int)P.tiles_x - 1, max(b.x0, max(b.x1, b.x2)) >> Shift);
    const int minTY = max(0, min(b.y0, min(b.y1, b.y2)) >> Shift);
    const int maxTY = min((int)P.tiles_y - 1, max(b.y0, max(b.y1, b.y2)) >> Shift);
    b.minTX = minTX;
    b.minTY = minTY;
    b.w = max(0, maxTX - minTX + 1);
    b.h = max(0, maxTY - minTY + 1);
    b.small = (maxTX - minTX < 2 && maxTY - minTY < 2);
    if (b.w == 0 || b.h == 0) b.w = b.h = 0;
}

// Tile (tx, ty) test of a big triangle.  Returns -1 for reject, otherwise the
// accept-edge flags (bits 0..2).
__device__ __forceinline__ int bin_test(const BinTri& b, int tx, int ty) {
    const int Shift = kTileLog2 + 4;
    auto cx = [&](uint32_t c) { return (tx + (int)(c & 1u)) << Shift; };
    auto cy = [&](uint32_t c) { return (ty + (int)(c >> 1)) << Shift; };
    const uint32_t r0 = b.info & 3u, r1 = (b.info >> 2) & 3u, r2 = (b.info >> 4) & 3u;
    const uint32_t a0 = (b.info >> 6) & 3u, a1 = (b.info >> 8) & 3u, a2 = (b.info >> 10) & 3u;
    if (b.B0 * (cx(r0) - b.x0) + b.C0 * (cy(r0) - b.y0) + b.sb0 < 0) return -1;
    if (b.B1 * (cx(r1) - b.x1) + b.C1 * (cy(r1) - b.y1) + b.sb1 < 0) return -1;
    if (b.B2 * (cx(r2) - b.x2) + b.C2 * (cy(r2) - b.y2) + b.sb2 < 0) return -1;
    int f = 0;
    if (b.B0 * (cx(a0) - b.x0) + b.C0 * (cy(a0) - b.y0) + b.sb0 >= 0) f |= 1;
    if (b.B1 * (cx(a1) - b.x1) + b.C1 * (cy(a1) - b.y1) + b.sb1 >= 0) f |= 2;
    if (b.B2 * (cx(a2) - b.x2) + b.C2 * (cy(a2) - b.y2) + b.sb2 >= 0) f |= 4;
    return f;
}

// Reference k (row-major over the bbox) of a compact descriptor: its tile.
__device__ __forceinline__ uint32_t compact_tile(uint32_t desc, uint32_t k, uint32_t tilesX) {
    const uint32_t w = 1u + ((desc >> 28) & 1u);
    return ((desc >> 14) & 0x3FFFu) * tilesX + (desc & 0x3FFFu) + (k % w) + (k / w) * tilesX;
}
__device__ __forceinline__ uint32_t compact_refs(uint32_t desc) {
    return (1u + ((desc >> 28) & 1u)) * (1u + ((desc >> 29) & 1u));
}

// A slot's references: its records, the tiles of a record in its tile bbox.
// A compact descriptor is its record's tile bbox (at most 2x2 tiles, no corner
// tests; the record is the slot).  Otherwise the descriptor is
// (first record << 3) | count: the binning kernels list such descriptors per
// step and hand them to block_enum_listed.

// Whether any of a thread's descriptors of a step is non-compact.
template <uint32_t kN>
__device__ __forceinline__ int any_non_compact(const uint32_t (&d)[kN]) {
    bool any = false;
#pragma unroll
    for (uint32_t u = 0; u < kN; u++) any |= d[u] != 0 && !(d[u] & kDescCompact);
    return any ? 1 : 0;
}

// Whether the references of a record whose small box is listed untested count as
// heavy ones: those of a triangle too long for a compact descriptor, as kDescHeavy.
__device__ __forceinline__ bool small_heavy(const BinTri& b) {
    const uint32_t ex = (uint32_t)max(b.x0, max(b.x1, b.x2)) - (uint32_t)min(b.x0, min(b.x1, b.x2));
    const uint32_t ey = (uint32_t)max(b.y0, max(b.y1, b.y2)) - (uint32_t)min(b.y0, min(b.y1, b.y2));
    return max(ex, ey) >= kCompactExtent && (uint64_t)(ex >> 4) * (ey >> 4) >= kHeavyPixels;
}

// The references of record rec (its tile bbox loaded in b) whose bbox tiles
// are k0, k0 + dk, ... (row-major over the bbox), passed to emit(tile, tx,
// ty, payload, heavy).
template <class Emit>
__device__ __forceinline__ void enum_record_tiles(const FrameParams& P, const BinTri& b, uint32_t rec, uint32_t k0,
                                                  uint32_t dk, Emit&& emit) {
    const uint32_t n = (uint32_t)(b.w * b.h);
    if (n == 0) return;
    const uint32_t w = (uint32_t)b.w;
    const bool heavy = !b.small || small_heavy(b);
    uint32_t cx = k0 % w, cy = k0 / w;
    const uint32_t dx = dk % w, dy = dk / w;
    for (uint32_t k = k0; k < n; k += dk) {
        const int tx = b.minTX + (int)cx, ty = b.minTY + (int)cy;
        const int f = b.small ? 0 : bin_test(b, tx, ty);
        if (f >= 0)
            emit((uint32_t)ty * P.tiles_x + (uint32_t)tx, tx, ty,
                 b.small ? rec | kRefStored : rec | ((uint32_t)f << kRecordBits) | (1u << 31), heavy);
        cx += dx;
        cy += dy;
        if (cx >= w) {
            cx -= w;
            cy++;
        }
    }
}

// Records of a record's bbox this size or smaller are enumerated by one
// thread; larger ones by a whole wave, 64 tiles at a time.
constexpr uint32_t kThreadTiles = 16;
// Wide records listed per step: beyond this many, a thread enumerates its
// record itself.
constexpr uint32_t kWideCap = 256;

// All references of the nBig listed non-compact descriptors, for the whole
// workgroup (every thread must call it; sScan holds kBlock + kBlock / kWave
// words): the descriptors' records are numbered, kBlock descriptors at a
// time, and each thread takes records, so that the records' loads are in
// flight together.  A thread enumerates a record of up to kThreadTiles bbox
// tiles itself and lists a wider one, which a wave then enumerates.  There is
// no order among the emitted references.
template <class Emit>
__device__ __forceinline__ void block_enum_listed(const FrameParams& P, const RasterRec* rrec, const uint32_t* sBig,
                                                  uint32_t nBig, uint32_t* sScan, uint32_t* sWide, uint32_t* sWideN,
                                                  Emit&& emit) {
    const uint32_t lane = __lane_id(), wave = threadIdx.x / kWave;
    uint32_t* sPre = sScan;            // record number of the batch's first record of each descriptor
    uint32_t* sWaveSum = sScan + kBlock;
    for (uint32_t b0 = 0; b0 < nBig; b0 += kBlock) {
        const uint32_t nb = min(nBig - b0, kBlock);
        const uint32_t c = threadIdx.x < nb ? sBig[b0 + threadIdx.x] & 7u : 0u;
        const uint32_t incl = wave_incl_scan(c);
        if (lane == kWave - 1) sWaveSum[wave] = incl;
        __syncthreads();
        uint32_t before = 0, total = 0;
        for (uint32_t w = 0; w < kBlock / kWave; w++) {
            before += w < wave ? sWaveSum[w] : 0u;
            total += sWaveSum[w];
        }
        sPre[threadIdx.x] = before + incl - c;
        __syncthreads();
        for (uint32_t j = threadIdx.x; j < total; j += kBlock) {
            // the descriptor whose records hold j: every listed count is >= 1,
            // so the numbers increase strictly over [0, nb)
            uint32_t lo = 0, hi = nb - 1;
            while (lo < hi) {
                const uint32_t mid = (lo + hi + 1) >> 1;
                if (sPre[mid] <= j) lo = mid;
                else hi = mid - 1;
            }
            const uint32_t rec = (sBig[b0 + lo] >> 3) + (j - sPre[lo]);
            BinTri b;
            load_bin_tri(P, rrec[rec], b);
            const uint32_t n = (uint32_t)(b.w * b.h);
            uint32_t slot = kWideCap;
            if (n > kThreadTiles) {
                slot = atomicAdd(sWideN, 1u);
                if (slot < kWideCap) sWide[slot] = rec;
            }
            if (slot >= kWideCap) enum_record_tiles(P, b, rec, 0, 1, emit);
        }
        __syncthreads();  // the numbering is rewritten by the next batch
    }
    const uint32_t nWide = min(*sWideN, kWideCap);
    for (uint32_t i = wave; i < nWide; i += kBlock / kWave) {
        const uint32_t rec = sWide[i];
        BinTri b;
        load_bin_tri(P, rrec[rec], b);
        enum_record_tiles(P, b, rec, lane, kWave, emit);
    }
}

// A direct tile's count word (references, heavy ones in the high half) after an
// addition: a tile beyond what one workgroup should walk sends the frame to
// the general path.
__device__ __forceinline__ void direct_check(const DeviceBuffers& B, uint64_t count) {
    if ((uint32_t)count > B.direct || (uint32_t)(count >> 32) > kDirectHeavy)
        atomicOr(&B.counters[kCntOverflow], (uint32_t)kOvDirect);
}

}  // namespace

// ---------------------------------------------------------------------------
// Tile rasterisation + deferred shading.
// ---------------------------------------------------------------------------
namespace {

// Medium references with at least this many quads are walked by the whole
// wave (the triangle in scalar registers, 64 quads per pass); fewer are packed
// with other references' quads into shared passes.
constexpr uint32_t kWaveQuads = 40;
// Packed quads of one wave's slice: at most 64 references of < kWaveQuads.
constexpr uint32_t kOwnerCap = kWave * (kWaveQuads - 1);

struct RTri {
    int x0, y0, x1, y1, x2, y2;
    int B0, C0, B1, C1, B2, C2;
    int pb0, pb1, pb2;   // pixel-level top-left bias (Core/RasterTriangle.h:296-299)
    float inv_det, z0, z1, z2;
    uint32_t info, order;
};

__device__ __forceinline__ int pixel_bias(int ax, int ay, int bx, int by) {
    return ((by > ay) || (ay == by && ax > bx)) ? -1 : 0;
}

__device__ __forceinline__ void load_rtri(const RasterRec& r, RTri& t) {
    t.x0 = r.x0; t.y0 = r.y0; t.x1 = r.x1; t.y1 = r.y1; t.x2 = r.x2; t.y2 = r.y2;
    t.B0 = t.y0 - t.y1; t.C0 = t.x1 - t.x0;
    t.B1 = t.y1 - t.y2; t.C1 = t.x2 - t.x1;
    t.B2 = t.y2 - t.y0; t.C2 = t.x0 - t.x2;
    t.pb0 = pixel_bias(t.x0, t.y0, t.x1, t.y1);
    t.pb1 = pixel_bias(t.x1, t.y1, t.x2, t.y2);
    t.pb2 = pixel_bias(t.x2, t.y2, t.x0, t.y0);
    t.inv_det = r.inv_det;
    t.z0 = r.z0; t.z1 = r.z1; t.z2 = r.z2;
    t.info = r.info;
    t.order = r.order;
}

// a * b of 24-bit values in 32 bits, cheaper than a 32-bit product (k_raster of
// the 10M heightfield at 4K, bound by its vector instructions: 121 us with 32-bit
// products, 119 with these).
__device__ __forceinline__ int mul24(int a, int b) { return __mul24(a, b); }
template <bool kShort>
__device__ __forceinline__ int mul(int a, int b) { return kShort ? __mul24(a, b) : a * b; }
// pixel_bias of a compact triangle's edge, whose B and C fit 16 bits: B < 0, or
// B == 0 and C < 0.
__device__ __forceinline__ int compact_bias(int B, int C) { return ((int)((uint32_t)B << 16) + C) >> 31; }

// Record of a compact triangle in slot r from its vertices' screen values
// (the values k_setup used); corner codes are not needed below tile level.
__device__ __forceinline__ void screen_rtri_from(const ScreenVert& s0, const ScreenVert& s1, const ScreenVert& s2,
                                                 uint32_t r, RTri& t) {
    t.x0 = s0.x; t.y0 = s0.y; t.x1 = s1.x; t.y1 = s1.y; t.x2 = s2.x; t.y2 = s2.y;
    t.B0 = t.y0 - t.y1; t.C0 = t.x1 - t.x0;
    t.B1 = t.y1 - t.y2; t.C1 = t.x2 - t.x1;
    t.B2 = t.y2 - t.y0; t.C2 = t.x0 - t.x2;
    t.pb0 = compact_bias(t.B0, t.C0);
    t.pb1 = compact_bias(t.B1, t.C1);
    t.pb2 = compact_bias(t.B2, t.C2);
    t.inv_det = rcp_normal((float)(mul24(t.C2, t.B1) - mul24(t.C1, t.B2)));  // (0 only in lanes without a reference)
    t.z0 = s0.z; t.z1 = s1.z; t.z2 = s2.z;
    t.info = 0;
    t.order = make_order(r, 0, false);
}
__device__ __forceinline__ void screen_rtri(const FrameParams& P, const DeviceBuffers& B, uint32_t r, RTri& t) {
    const GlobalPtr<uint32_t> idx = as_global(P.mesh.idx) + 3 * (size_t)(r - P.slot_base);
    screen_rtri_from(B.sverts[P.vert_base + idx[0]], B.sverts[P.vert_base + idx[1]], B.sverts[P.vert_base + idx[2]],
                     r, t);
}
// Whether differences of the triangle's coordinates and of pixels fit 24 bits
// (any triangle's do whose raster matrix maps to a picture of the usual size).
__device__ __forceinline__ bool fits24(const RTri& t) {
    auto out = [](int v) { return (uint32_t)v + (1u << 22) >= (2u << 22); };
    return !(out(t.x0) | out(t.y0) | out(t.x1) | out(t.y1) | out(t.x2) | out(t.y2));
}

// A reference's index-buffer entries when it is a compact unclipped triangle
// (otherwise another triangle's of the job, a valid address whose value is
// unused).
__device__ __forceinline__ uint3 ref_indices(const FrameParams& P, uint32_t pay) {
    const uint32_t k = min((pay & kRecordMask) - P.slot_base, P.num_triangles - 1u);
    const GlobalPtr<uint32_t> idx = as_global(P.mesh.idx) + 3 * (size_t)k;
    return make_uint3(idx[0], idx[1], idx[2]);
}

// Ordered depth key: (depth, submission order) min = the winner of the
// sequential d <= D test (Core/FrameBuffer.cpp:54-68).  -0 and +0 compare equal.
__device__ __forceinline__ uint32_t depth_bits(float d) {
    const uint32_t b = __float_as_uint(d + 0.0f);  // -0 + 0 = +0; any other d is unchanged
    return b ^ ((uint32_t)((int)b >> 31) | 0x80000000u);  // negative: ~b, otherwise b | sign
}
__device__ __forceinline__ uint64_t bg_key() { return ((uint64_t)0xBF800000u << 32) | 0xFFFFFFFFull; }

// Barycentrics and depth at a pixel centre (Core/RasterTriangle.h:324-337).
__device__ __forceinline__ void bary_depth(const RTri& t, int px, int py, float& l0, float& l1, float& d) {
    l0 = (float)(t.B1 * (px - t.x2) + t.C1 * (py - t.y2)) * t.inv_det;
    l1 = (float)(t.B2 * (px - t.x2) + t.C2 * (py - t.y2)) * t.inv_det;
    const float l2 = 1.0f - l0 - l1;
    d = l0 * t.z0 + l1 * t.z1 + l2 * t.z2;
}

// LDS key image rows are one key longer than a tile row, so that vertically
// adjacent pixels fall in different LDS banks.
// (Single-sample only: with four padded planes the multisample kernel ran with
// one resident workgroup per CU fewer, and slower.)
template <bool kMS>
constexpr int kKeyStride = kMS ? kTileSize : kTileSize + 1;
template <bool kMS>
constexpr uint32_t kKeyPlane = kTileSize * kKeyStride<kMS>;

// Samples of one raster pass: their count, and their offsets, a byte each (x in
// the low four bits, y in the high); sample k's keys live in plane k
// (kKeyPlane<true> keys apart).
struct SamplePass {
    uint32_t n, offsets;
};
// Loaded once per pass: a load per sample of every pixel waited with each for
// the LDS atomics before it (one counter).
__device__ __forceinline__ SamplePass sample_pass(uint32_t level, uint32_t base, uint32_t n) {
    uint32_t offsets = 0;
    for (uint32_t k = 0; k < n; k++) {
        const int2 o = c_sample_offsets[level][base + k];
        offsets |= (((uint32_t)o.x & 15u) | ((uint32_t)o.y & 15u) << 4) << (8 * k);
    }
    return SamplePass{n, (uint32_t)__builtin_amdgcn_readfirstlane(offsets)};
}

// Depth test of one pixel from its edge values e0..e2 (coverage when
// useEdges, Core/Rasterizer.h:162), then the (depth, order) key update; klo is
// the key's low word, 0xFFFFFFFE - order.  The barycentric numerators
// n0 = B1 (x - x2) + C1 (y - y2) and n1 = B2 (x - x2) + C2 (y - y2)
// (Core/RasterTriangle.h:324-337) are e1 and e2 without their top-left bias:
// e1 - pb1 - n0 = B1 (x2 - x1) + C1 (y2 - y1) = 0 as a polynomial identity, so
// it holds in wrapping int32 as well.  With multisampling each sample of the
// pass is tested at centre + offset (Core/Rasterizer.h:243-266):
// e + ox B + oy C, wrapping as the reference.
// kShort: differences of the triangle's coordinates fit 24 bits.
template <bool kMS, bool kShort>
__device__ __forceinline__ void pixel_key(const RTri& t, int e0, int e1, int e2, uint32_t klo, bool useEdges,
                                          uint64_t* slot, const SamplePass& sp) {
    const int n0 = e1 - t.pb1, n1 = e2 - t.pb2;
    if (!kMS) {
        if (useEdges && (e0 | e1 | e2) < 0) return;
        const float l0 = (float)n0 * t.inv_det;
        const float l1 = (float)n1 * t.inv_det;
        const float l2 = 1.0f - l0 - l1;
        const float d = l0 * t.z0 + l1 * t.z1 + l2 * t.z2;
        if (!(d <= 1.0f)) return;   // never passes d <= D with D <= 1 (NaN included)
        const uint64_t key = ((uint64_t)depth_bits(d) << 32) | (uint64_t)klo;
        // (the atomic alone is cheaper than a read, a compare and the atomic)
        atomicMin((unsigned long long*)slot, (unsigned long long)key);
        return;
    }
    for (uint32_t k = 0; k < sp.n; k++) {
        const int ox = (int)(sp.offsets << (28 - 8 * k)) >> 28, oy = (int)(sp.offsets << (24 - 8 * k)) >> 28;
        const int m0 = n0 + mul<kShort>(ox, t.B1) + mul<kShort>(oy, t.C1);
        const int m1 = n1 + mul<kShort>(ox, t.B2) + mul<kShort>(oy, t.C2);
        if (useEdges) {
            const int s0 = e0 + mul<kShort>(ox, t.B0) + mul<kShort>(oy, t.C0);
            if ((s0 | (m0 + t.pb1) | (m1 + t.pb2)) < 0) continue;
        }
        const float l0 = (float)m0 * t.inv_det;
        const float l1 = (float)m1 * t.inv_det;
        const float l2 = 1.0f - l0 - l1;
        const float d = l0 * t.z0 + l1 * t.z1 + l2 * t.z2;
        if (!(d <= 1.0f)) continue;
        const uint64_t key = ((uint64_t)depth_bits(d) << 32) | (uint64_t)klo;
        atomicMin((unsigned long long*)(slot + k * kKeyPlane<kMS>), (unsigned long long)key);
    }
}

// Pixels (qx + dx, qy + dy), dx, dy in {0, 1}, that lie within (maxX, maxY):
// the 2x2 quad at (qx, qy) (one SSE lane per pixel in the reference).  Edge
// functions are evaluated at (qx, qy)'s centre (16x+8, 16y+8) and stepped by
// 16 B and 16 C to the other pixels, which is
// exact in wrapping int32 arithmetic (the reference steps the same way,
// Core/Rasterizer.h:190-198).
template <bool kMS, bool kShort>
__device__ __forceinline__ void quad_depth(const RTri& t, int qx, int qy, bool useEdges, int tminX, int tminY,
                                           uint64_t* keys, int maxX, int maxY, const SamplePass& sp) {
    const int px = qx * 16 + 8, py = qy * 16 + 8;
    const int e0 = mul<kShort>(t.B0, px - t.x0) + mul<kShort>(t.C0, py - t.y0) + t.pb0;
    const int e1 = mul<kShort>(t.B1, px - t.x1) + mul<kShort>(t.C1, py - t.y1) + t.pb1;
    const int e2 = mul<kShort>(t.B2, px - t.x2) + mul<kShort>(t.C2, py - t.y2) + t.pb2;
    const int sB0 = t.B0 * 16, sB1 = t.B1 * 16, sB2 = t.B2 * 16;
    const int sC0 = t.C0 * 16, sC1 = t.C1 * 16, sC2 = t.C2 * 16;
    const uint32_t klo = 0xFFFFFFFEu - t.order;
    uint64_t* row = &keys[(qy - tminY) * kKeyStride<kMS> + (qx - tminX)];
    const bool right = qx + 1 <= maxX, down = qy + 1 <= maxY;
    pixel_key<kMS, kShort>(t, e0, e1, e2, klo, useEdges, row, sp);
    if (right) pixel_key<kMS, kShort>(t, e0 + sB0, e1 + sB1, e2 + sB2, klo, useEdges, row + 1, sp);
    if (down) pixel_key<kMS, kShort>(t, e0 + sC0, e1 + sC1, e2 + sC2, klo, useEdges, row + kKeyStride<kMS>, sp);
    if (right && down)
        pixel_key<kMS, kShort>(t, e0 + sB0 + sC0, e1 + sB1 + sC1, e2 + sB2 + sC2, klo, useEdges, row + kKeyStride<kMS> + 1, sp);
}
template <bool kMS, bool kShort>
__device__ __forceinline__ void quad_depth(const RTri& t, int qx, int qy, bool useEdges, int tminX, int tminY,
                                           uint64_t* keys, const SamplePass& sp) {
    quad_depth<kMS, kShort>(t, qx, qy, useEdges, tminX, tminY, keys, qx + 1, qy + 1, sp);
}

__device__ __forceinline__ float pow_decl(float x, int n, float s) {
    if (n < 0) return powf(x, s);
    float result = 1.0f, base = x;
    unsigned u = (unsigned)n;
    while (u) {
        if (u & 1u) result *= base;
        u >>= 1;
        if (u) base *= base;
    }
    return result;
}

// Color4b::FromFloats clamp (NaN -> 0) and its byte conversion.
__device__ __forceinline__ float clamp01(float c) { return fminf(fmaxf(c, 0.0f), 1.0f); }
__device__ __forceinline__ uint32_t to_byte(float c) { return (uint32_t)(int)(clamp01(c) * 255.0f + 0.5f); }

// Fragment::Interpolate (Core/Shader.h:142-170) + pixel shader
// (Core/Shader.h:209-282); unclamped RGB.
__device__ __forceinline__ float3 shade_pixel(const FrameParams& P, float b0, float b1, const ShadeVert& v0,
                                              const ShadeVert& v1, const ShadeVert& v2) {
    float b2 = 1.0f - b0 - b1;
    b0 *= v0.inv_w;
    b1 *= v1.inv_w;
    b2 *= v2.inv_w;
    const float invB = reciprocal(b0 + b1 + b2);
    b0 *= invB;
    b1 *= invB;
    b2 = 1.0f - b0 - b1;
    const float Px = b0 * v0.px + b1 * v1.px + b2 * v2.px;
    const float Py = b0 * v0.py + b1 * v1.py + b2 * v2.py;
    const float Pz = b0 * v0.pz + b1 * v1.pz + b2 * v2.pz;
    const float Nx = b0 * v0.nx + b1 * v1.nx + b2 * v2.nx;
    const float Ny = b0 * v0.ny + b1 * v1.ny + b2 * v2.ny;
    const float Nz = b0 * v0.nz + b1 * v1.nz + b2 * v2.nz;

    float w = reciprocal_sqrt(Nx * Nx + Ny * Ny + Nz * Nz);
    const float nx = Nx * w, ny = Ny * w, nz = Nz * w;
    const float Lx = P.light[0], Ly = P.light[1], Lz = P.light[2];
    float diffuseAmount = Lx * nx + Ly * ny + Lz * nz;
    diffuseAmount = diffuseAmount < 0.0f ? 0.0f : diffuseAmount;
    const float diffuse = (diffuseAmount + P.ambient) * P.kd * (float)(1.0 / 3.14159265358979323846);
    float r, g, b;
    if (P.shader == kLambertAlbedo) {
        r = diffuse * P.albedo[0];
        g = diffuse * P.albedo[1];
        b = diffuse * P.albedo[2];
    } else {
        float ex = P.eye[0] - Px, ey = P.eye[1] - Py, ez = P.eye[2] - Pz;
        w = reciprocal_sqrt(ex * ex + ey * ey + ez * ez);
        ex *= w; ey *= w; ez *= w;
        float hx = Lx + ex, hy = Ly + ey, hz = Lz + ez;
        w = reciprocal_sqrt(hx * hx + hy * hy + hz * hz);
        hx *= w; hy *= w; hz *= w;
        float sa = nx * hx + ny * hy + nz * hz;
        if (P.clamp_spec) sa = fmaxf(sa, 0.0f);
        const float spec = pow_decl(sa, P.shin_int, P.shininess) * P.ks;
        if (P.shader == kBlinnPhongRef) {
            r = g = b = diffuse + spec;
        } else {
            const float Cr = b0 * v0.cr + b1 * v1.cr + b2 * v2.cr;
            const float Cg = b0 * v0.cg + b1 * v1.cg + b2 * v2.cg;
            const float Cb = b0 * v0.cb + b1 * v1.cb + b2 * v2.cb;
            r = diffuse * Cr + spec;
            g = diffuse * Cg + spec;
            b = diffuse * Cb + spec;
        }
    }
    return make_float3(r, g, b);
}

// ---- Texture slots (Texture2D<Color>::Sample, EDXUtil; declared semantics:
// texel (i, j) centred at ((i + 0.5) / w, (j + 0.5) / h), coordinates wrap,
// float-to-index conversion with NaN -> 0 and a clamp to +-2^30). ----
__device__ __forceinline__ int tex_index(float x) {
    return x != x ? 0 : (int)fminf(fmaxf(x, -1073741824.0f), 1073741823.0f);
}
// i modulo n, in [0, n).  Sides of a power of two (the usual textures, and then
// all their mip levels) take a mask: a remainder is some 35 instructions, and
// one per coordinate of each texel made the samplers ALU-bound.
__device__ __forceinline__ int tex_wrap(int i, int n) {
    if ((n & (n - 1)) == 0) return i & (n - 1);
    i %= n;
    return i < 0 ? i + n : i;
}
typedef float Texel __attribute__((ext_vector_type(4)));
// A mip level: its first texel and sides.
struct TexLevel {
    uint32_t off;
    int w, h;
};
// Bilinear filter over one level.  Neighbours follow from the first texel: one
// wrap per coordinate.  With a remainder per coordinate of every texel and the
// levels found anew for every anisotropic tap, k_tile took 121 us for 8:1 at
// 1080p (1.2M covered pixels, 64 texels each) and k_shade_tex 60 us for
// trilinear at 1440p; so 84 and 51 us, now mostly the gathers' address rate.
__device__ __forceinline__ float3 tex_bilinear(const FrameParams& P, const TexLevel& L, float u, float v) {
    const float x = u * (float)L.w - 0.5f, y = v * (float)L.h - 0.5f;
    const float x0 = floorf(x), y0 = floorf(y);
    const float fx = x - x0, fy = y - y0;
    const uint32_t i0 = (uint32_t)tex_wrap(tex_index(x0), L.w), j0 = (uint32_t)tex_wrap(tex_index(y0), L.h);
    const uint32_t i1 = i0 + 1 == (uint32_t)L.w ? 0u : i0 + 1, j1 = j0 + 1 == (uint32_t)L.h ? 0u : j0 + 1;
    const uint32_t r0 = L.off + j0 * (uint32_t)L.w, r1 = L.off + j1 * (uint32_t)L.w;
    const GlobalPtr<Texel> texels = as_global((const Texel*)P.texels);
    const Texel c00 = texels[r0 + i0], c10 = texels[r0 + i1], c01 = texels[r1 + i0], c11 = texels[r1 + i1];
    const float gx = 1.0f - fx, gy = 1.0f - fy;
    return make_float3(gy * (gx * c00.x + fx * c10.x) + fy * (gx * c01.x + fx * c11.x),
                       gy * (gx * c00.y + fx * c10.y) + fy * (gx * c01.y + fx * c11.y),
                       gy * (gx * c00.z + fx * c10.z) + fy * (gx * c01.z + fx * c11.z));
}
// The two mip levels around a lod (clamped to the chain) and the second's weight.
struct TexLevels {
    TexLevel a, b;
    float t;
};
__device__ __forceinline__ TexLevels tex_levels(const TexDesc& d, float lod) {
    lod = fminf(fmaxf(lod, 0.0f), (float)(d.levels - 1));
    const float fl = floorf(lod);
    TexLevels m;
    m.t = lod - fl;
    m.a = TexLevel{d.offset, (int)d.width, (int)d.height};
    auto next = [](TexLevel& l) {
        l.off += (uint32_t)l.w * (uint32_t)l.h;
        l.w = max(1, l.w >> 1);
        l.h = max(1, l.h >> 1);
    };
    for (uint32_t k = 0; k < (uint32_t)fl; k++) next(m.a);
    m.b = m.a;
    if ((uint32_t)fl + 1 < d.levels) next(m.b);
    return m;
}
// The trilinear blend of two levels.  At weight 0 (magnified, or the last
// level) the second level is not sampled: 1 a + 0 b is a.
__device__ __forceinline__ float3 tex_trilinear_at(const FrameParams& P, const TexLevels& m, float u, float v) {
    const float3 a = tex_bilinear(P, m.a, u, v);
    if (m.t == 0.0f) return a;
    const float3 b = tex_bilinear(P, m.b, u, v);
    const float s = 1.0f - m.t;
    return make_float3(s * a.x + m.t * b.x, s * a.y + m.t * b.y, s * a.z + m.t * b.z);
}
// Sample(uv, differentials): nearest / bilinear on level 0; trilinear with
// lod = log2 of the longer of the two texel-space differentials; or N:1
// anisotropic (N = 4, 8, 16): N trilinear taps spread evenly along the longer
// differential (tap k at offset (2k + 1 - N) / 2N of it) at the lod of the
// shorter one, raised to at least 1/N of the longer, averaged in tap order.
__device__ __forceinline__ float3 tex_sample(const FrameParams& P, const TexDesc& d, float u, float v, float dux,
                                             float dvx, float duy, float dvy) {
    if (d.levels == 0) return make_float3(d.color[0], d.color[1], d.color[2]);
    const int w = (int)d.width, h = (int)d.height;
    if (P.tex_filter == kFilterNearest) {
        const uint32_t i = (uint32_t)tex_wrap(tex_index(floorf(u * (float)w)), w);
        const uint32_t j = (uint32_t)tex_wrap(tex_index(floorf(v * (float)h)), h);
        const Texel c = as_global((const Texel*)P.texels)[d.offset + j * (uint32_t)w + i];
        return make_float3(c.x, c.y, c.z);
    }
    if (P.tex_filter == kFilterLinear) return tex_bilinear(P, TexLevel{d.offset, w, h}, u, v);
    const float ax = dux * (float)w, ay = dvx * (float)h, bx = duy * (float)w, by = dvy * (float)h;
    const float la2 = ax * ax + ay * ay, lb2 = bx * bx + by * by;
    if (P.tex_filter == kFilterTrilinear) {
        const float rho2 = fmaxf(la2, lb2);
        return tex_trilinear_at(P, tex_levels(d, rho2 > 0.0f ? 0.5f * log2f(rho2) : 0.0f), u, v);
    }
    const int N = 4 << (P.tex_filter - kFilterAniso4);
    const bool xMajor = la2 >= lb2;
    const float mu = xMajor ? dux : duy, mv = xMajor ? dvx : dvy;
    const float maj2 = xMajor ? la2 : lb2, n2 = (float)(N * N);
    float min2 = xMajor ? lb2 : la2;
    if (min2 * n2 < maj2) min2 = maj2 / n2;
    const TexLevels m = tex_levels(d, min2 > 0.0f ? 0.5f * log2f(min2) : 0.0f);
    float3 acc = make_float3(0.0f, 0.0f, 0.0f);
    for (int k = 0; k < N; k++) {
        const float sk = (float)(2 * k + 1 - N) / (float)(2 * N);
        const float3 c = tex_trilinear_at(P, m, u + sk * mu, v + sk * mv);
        acc.x += c.x;
        acc.y += c.y;
        acc.z += c.z;
    }
    const float inv = 1.0f / (float)N;
    return make_float3(acc.x * inv, acc.y * inv, acc.z * inv);
}

// Perspective-correct texture coordinate of the triangle at pixel (x, y)
// (Fragment::Interpolate, Core/Shader.h:142-170, at that pixel's centre).
__device__ __forceinline__ float2 interp_uv(const RTri& t, int x, int y, const ShadeVert& v0, const ShadeVert& v1,
                                           const ShadeVert& v2) {
    const int px = x * 16 + 8, py = y * 16 + 8;
    float b0 = (float)(t.B1 * (px - t.x2) + t.C1 * (py - t.y2)) * t.inv_det;
    float b1 = (float)(t.B2 * (px - t.x2) + t.C2 * (py - t.y2)) * t.inv_det;
    float b2 = 1.0f - b0 - b1;
    b0 *= v0.inv_w;
    b1 *= v1.inv_w;
    b2 *= v2.inv_w;
    const float invB = reciprocal(b0 + b1 + b2);
    b0 *= invB;
    b1 *= invB;
    b2 = 1.0f - b0 - b1;
    return make_float2(b0 * v0.u + b1 * v1.u + b2 * v2.u, b0 * v0.v + b1 * v1.v + b2 * v2.v);
}

// LambertianAlbedoPixelShader (Core/Shader.h:209-244) for pixel (x, y) of the
// 2x2 quad at (x & ~1, y & ~1): the albedo is the triangle's texture sampled
// at the pixel's coordinate with the quad's differentials (lane 1 - lane 0,
// lane 2 - lane 0; uncovered lanes extrapolate the triangle's plane).
__device__ __forceinline__ float3 shade_textured(const FrameParams& P, const RTri& t, int x, int y, float l0, float l1,
                                                 const ShadeVert& v0, const ShadeVert& v1, const ShadeVert& v2,
                                                 uint32_t slot) {
    const int qx = x & ~1, qy = y & ~1;
    const float2 q0 = interp_uv(t, qx, qy, v0, v1, v2), q1 = interp_uv(t, qx + 1, qy, v0, v1, v2),
                 q2 = interp_uv(t, qx, qy + 1, v0, v1, v2);
    const uint32_t lane = (uint32_t)(x & 1) | ((uint32_t)(y & 1) << 1);
    const float2 uv = lane == 0 ? q0 : lane == 1 ? q1 : lane == 2 ? q2 : interp_uv(t, x, y, v0, v1, v2);
    const float3 albedo = tex_sample(P, P.tex[slot], uv.x, uv.y, q1.x - q0.x, q1.y - q0.y, q2.x - q0.x, q2.y - q0.y);
    // the normal and the diffuse term as shade_pixel's Lambertian path
    float b2 = 1.0f - l0 - l1;
    float b0 = l0 * v0.inv_w, b1 = l1 * v1.inv_w;
    b2 *= v2.inv_w;
    const float invB = reciprocal(b0 + b1 + b2);
    b0 *= invB;
    b1 *= invB;
    b2 = 1.0f - b0 - b1;
    const float Nx = b0 * v0.nx + b1 * v1.nx + b2 * v2.nx;
    const float Ny = b0 * v0.ny + b1 * v1.ny + b2 * v2.ny;
    const float Nz = b0 * v0.nz + b1 * v1.nz + b2 * v2.nz;
    const float w = reciprocal_sqrt(Nx * Nx + Ny * Ny + Nz * Nz);
    const float nx = Nx * w, ny = Ny * w, nz = Nz * w;
    float diffuseAmount = P.light[0] * nx + P.light[1] * ny + P.light[2] * nz;
    diffuseAmount = diffuseAmount < 0.0f ? 0.0f : diffuseAmount;
    const float diffuse = (diffuseAmount + P.ambient) * P.kd * (float)(1.0 / 3.14159265358979323846);
    return make_float3(diffuse * albedo.x, diffuse * albedo.y, diffuse * albedo.z);
}

// The pixel shader of the job for the winner at pixel (x, y); kTex: a job of
// the launch may use the textured shader (its code is only compiled in then,
// keeping the other shaders' register budget).
template <bool kTex>
__device__ __forceinline__ float3 shade_any(const FrameParams& P, const RTri& t, uint32_t order, int x, int y,
                                            float l0, float l1, const ShadeVert& v0, const ShadeVert& v1,
                                            const ShadeVert& v2) {
    if (kTex && P.shader == kTexturedLambert)
        return shade_textured(P, t, x, y, l0, l1, v0, v1, v2, global_at(P.mesh.tex, (order >> 4) - P.slot_base));
    return shade_pixel(P, l0, l1, v0, v1, v2);
}

}  // namespace

namespace {

// Tile-level references for one wave: the lanes are the 8x8 quads of a
// 16x16-pixel quadrant and the wave walks the tile's quadrants q0 .. q1 - 1.  Covers
// TrivialAcceptTriangle over the tile and CoarseRasterize's stepped quadrant
// tests with FineRasterize inside partly covered quadrants
// (Core/Rasterizer.h:32-200,310-353).
template <bool kMS>
__device__ __forceinline__ void raster_large_wave(const FrameParams& P, const RTri& t, uint32_t pay,
                                                  int tminX, int tminY, int tmaxX, int tmaxY, uint64_t* keys,
                                                  const SamplePass& sp, int q0, int q1) {
    const uint32_t lane = __lane_id();
    const int lx = (int)(lane & 7u) * 2, ly = (int)(lane >> 3) * 2;
    const bool trivial = ((pay >> kRecordBits) & 7u) == 7u;
    const bool big = (pay >> 31) != 0;
    if (trivial) {
        // TrivialAcceptTriangle over the tile (Core/Rasterizer.h:310-353).
        for (int q = q0; q < q1; q++) {
            const int qx = tminX + 16 * (q & 1) + lx, qy = tminY + 16 * (q >> 1) + ly;
            if (qx <= tmaxX - 1 && qy <= tmaxY - 1) quad_depth<kMS, false>(t, qx, qy, false, tminX, tminY, keys, sp);
        }
    } else {
        // CoarseRasterize (Core/Rasterizer.h:32-111): stepped corner tests per 16x16 quadrant.
        const int baseX = tminX << 4, baseY = tminY << 4;
        const int off = (kTileSize << 4) - 1, stepSize = kTileSize << 3;
        const int sb0 = scalar_bias(t.x0, t.y0, t.x1, t.y1);
        const int sb1 = scalar_bias(t.x1, t.y1, t.x2, t.y2);
        const int sb2 = scalar_bias(t.x2, t.y2, t.x0, t.y0);
        auto ef = [&](int e, uint32_t c) {
            const int cxp = baseX + (int)(c & 1u) * off, cyp = baseY + (int)(c >> 1) * off;
            if (e == 0) return t.B0 * (cxp - t.x0) + t.C0 * (cyp - t.y0) + sb0;
            if (e == 1) return t.B1 * (cxp - t.x1) + t.C1 * (cyp - t.y1) + sb1;
            return t.B2 * (cxp - t.x2) + t.C2 * (cyp - t.y2) + sb2;
        };
        // GenStepVectors (Core/RasterTriangle.h:192-255), lane q of the vector.
        auto step = [&](uint32_t c, int Bk, int Ck, int q) {
            int v;
            if (c == 0) v = (q == 0) ? 0 : (q == 1) ? Bk : (q == 2) ? Ck : Bk + Ck;
            else if (c == 1) v = (q == 0) ? -Bk : (q == 1) ? 0 : (q == 2) ? Ck - Bk : Ck;
            else if (c == 2) v = (q == 0) ? -Ck : (q == 1) ? Bk - Ck : (q == 2) ? 0 : Bk;
            else v = (q == 0) ? -Bk - Ck : (q == 1) ? -Ck : (q == 2) ? -Bk : 0;
            return stepSize * v;
        };
        const uint32_t r0 = t.info & 3u, r1 = (t.info >> 2) & 3u, r2 = (t.info >> 4) & 3u;
        const uint32_t a0 = (t.info >> 6) & 3u, a1 = (t.info >> 8) & 3u, a2 = (t.info >> 10) & 3u;
        const int rj0 = ef(0, r0), rj1 = ef(1, r1), rj2 = ef(2, r2);
        const bool ae0 = (pay >> kRecordBits) & 1u, ae1 = (pay >> (kRecordBits + 1)) & 1u,
                   ae2 = (pay >> (kRecordBits + 2)) & 1u;
        const int ac0 = ae0 ? 0 : ef(0, a0), ac1 = ae1 ? 0 : ef(1, a1), ac2 = ae2 ? 0 : ef(2, a2);
        const int fminX = min(t.x0, min(t.x1, t.x2)) >> 4, fmaxX = max(t.x0, max(t.x1, t.x2)) >> 4;
        const int fminY = min(t.y0, min(t.y1, t.y2)) >> 4, fmaxY = max(t.y0, max(t.y1, t.y2)) >> 4;
        for (int q = q0; q < q1; q++) {
            const bool rej = (rj0 + step(r0, t.B0, t.C0, q) < 0) || (rj1 + step(r1, t.B1, t.C1, q) < 0) ||
                             (rj2 + step(r2, t.B2, t.C2, q) < 0);
            if (rej) continue;
            const bool acc = (ae0 || ac0 + step(a0, t.B0, t.C0, q) >= 0) &&
                             (ae1 || ac1 + step(a1, t.B1, t.C1, q) >= 0) &&
                             (ae2 || ac2 + step(a2, t.B2, t.C2, q) >= 0);
            const int bminX = (q & 1) ? tminX + 16 : tminX, bmaxX = (q & 1) ? tmaxX : tminX + 16;
            const int bminY = (q >> 1) ? tminY + 16 : tminY, bmaxY = (q >> 1) ? tmaxY : tminY + 16;
            const int qx = tminX + 16 * (q & 1) + lx, qy = tminY + 16 * (q >> 1) + ly;
            if (acc) {
                if (qx >= bminX && qx <= bmaxX - 1 && qy >= bminY && qy <= bmaxY - 1)
                    quad_depth<kMS, false>(t, qx, qy, false, tminX, tminY, keys, sp);
            } else {
                int minX = max(bminX, fminX), minY = max(bminY, fminY);
                const int maxX = min(bmaxX - 1, fmaxX), maxY = min(bmaxY - 1, fmaxY);
                minX -= minX % 2;
                minY -= minY % 2;
                if (qx >= minX && qx <= maxX && qy >= minY && qy <= maxY)
                    quad_depth<kMS, false>(t, qx, qy, true, tminX, tminY, keys, sp);
            }
        }
    }
}

// The record of lane l, made wave-uniform.
__device__ __forceinline__ RTri broadcast_rtri(const RTri& t, int l) {
    RTri u;
    u.x0 = __builtin_amdgcn_readlane(t.x0, l);
    u.y0 = __builtin_amdgcn_readlane(t.y0, l);
    u.x1 = __builtin_amdgcn_readlane(t.x1, l);
    u.y1 = __builtin_amdgcn_readlane(t.y1, l);
    u.x2 = __builtin_amdgcn_readlane(t.x2, l);
    u.y2 = __builtin_amdgcn_readlane(t.y2, l);
    u.B0 = u.y0 - u.y1; u.C0 = u.x1 - u.x0;
    u.B1 = u.y1 - u.y2; u.C1 = u.x2 - u.x1;
    u.B2 = u.y2 - u.y0; u.C2 = u.x0 - u.x2;
    u.pb0 = __builtin_amdgcn_readlane(t.pb0, l);
    u.pb1 = __builtin_amdgcn_readlane(t.pb1, l);
    u.pb2 = __builtin_amdgcn_readlane(t.pb2, l);
    u.inv_det = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(t.inv_det), l));
    u.z0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(t.z0), l));
    u.z1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(t.z1), l));
    u.z2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(t.z2), l));
    u.info = __builtin_amdgcn_readlane(t.info, l);
    u.order = __builtin_amdgcn_readlane(t.order, l);
    return u;
}

// Wide references, lane by lane in t (quads: a quad-walked one's number of
// quads, from pixel (fx, fy), fnx to a row): each by the whole wave, the owner
// lane's record broadcast with readlane (no memory round trip).
template <bool kMS>
__device__ __forceinline__ void walk_wide(const FrameParams& P, const RTri& t, uint32_t pay, bool large, uint32_t quads,
                                          int fx, int fy, int fnx, int tminX, int tminY, int tmaxX, int tmaxY,
                                          uint64_t* keys, const SamplePass& sp, int q0 = 0, int q1 = 4) {
    const uint32_t lane = __lane_id();
    // FineRasterize's quads (bbox clamped to the tile, Core/Rasterizer.h:126-200), 64 per pass
    uint64_t wm = __ballot(quads != 0);
    while (wm) {
        const int l = __ffsll((unsigned long long)wm) - 1;
        wm &= wm - 1;
        const RTri u = broadcast_rtri(t, l);
        const int ux = __builtin_amdgcn_readlane(fx, l), uy = __builtin_amdgcn_readlane(fy, l);
        const uint32_t unx = __builtin_amdgcn_readlane((uint32_t)fnx, l);
        const uint32_t uq = __builtin_amdgcn_readlane(quads, l);
        // quad k = lane + 64 i at (k % unx, k / unx), stepped per pass
        uint32_t cx = lane % unx, cy = lane / unx;
        const uint32_t dx = kWave % unx, dy = kWave / unx;
        for (uint32_t k = lane; k < uq; k += kWave) {
            quad_depth<kMS, false>(u, ux + 2 * (int)cx, uy + 2 * (int)cy, true, tminX, tminY, keys, sp);
            cx += dx;
            cy += dy;
            if (cx >= unx) {
                cx -= unx;
                cy++;
            }
        }
    }
    uint64_t lm = __ballot(large);
    while (lm) {
        const int l = __ffsll((unsigned long long)lm) - 1;
        lm &= lm - 1;
        const uint32_t ppay = __builtin_amdgcn_readlane(pay, l);
        raster_large_wave<kMS>(P, broadcast_rtri(t, l), ppay, tminX, tminY, tmaxX, tmaxY, keys, sp, q0, q1);
    }
}

// An item's references that take a whole wave (tile-level ones, and those of
// kWaveQuads quads or more), by their place in the item: listed while the
// slices are walked, then shared out over the workgroup's waves.  At one sample,
// what the list does not hold any more is walked at once by the wave that has it;
// places from limit on are not written.  (With the list emptied by all waves
// after every 1,024 references, so that it never is full, the waves waited for each
// other: 10M heightfield at 4K k_raster 113 us, so 107, 4.6M triangles on 252 tiles
// 41 and 37.)  With more samples it is emptied so, after every 512: the second copy
// of the walk costs that kernel more than the waiting (2.1M sphere grid at 1080p,
// 4 samples, a call 218 us, 224 with it).
// (Not in a direct frame's tiles: few references, spread
// thinly over the waves anyway, whose records would be loaded twice.)
template <bool kMS>
constexpr uint32_t kWideRefs = kMS ? 512 : 1024;  // (512: a multiple of the workgroup's threads)
template <bool kMS>
struct WideRefs {
    uint32_t n, limit;
    uint16_t at[kWideRefs<kMS>];
};

// One raster work item: references [seg << segLog2, (seg + 1) << segLog2) of
// a tile, segLog2 being the tile's (tile_item).  Each wave streams its own
// 64-reference slices through the tile's LDS key buffer (no workgroup barrier
// per slice): small triangles take one lane each, medium ones one quad per lane;
// tile-level and long ones, a whole wave each, are listed and shared out over the
// waves after the slices.  The item's keys go to partials[workIndex].
// kThreads: the workgroup's threads.  kDirect: workIndex is a tile of a direct
// frame with directRefs references, whose keys stay in LDS, of rows [row0, row1)
// only (0, 16 or 32).
template <bool kMS, uint32_t kThreads = kBlock, bool kDirect = false>
__device__ __forceinline__ void raster_item(const BatchParams& Q, const FrameParams* __restrict__ jobs,
                                            const DeviceBuffers& B, uint32_t workIndex,
                                            uint64_t* keys, uint16_t (*sOwner)[kOwnerCap],
                                            WideRefs<kMS>* wide, uint32_t directRefs = 0,
                                            int row0 = 0, int row1 = kTileSize) {
    const uint32_t workItem = kDirect ? workIndex : __builtin_amdgcn_readfirstlane(B.work[workIndex]);
    // segFlag: the segment index, with kSingleSegment >> kTileBits above it
    const uint32_t gtile = workItem & (kMaxBatchTiles - 1), segFlag = workItem >> kTileBits;
    const uint32_t seg = segFlag & ((1u << kSegIndexBits) - 1);
    const FrameParams& P = jobs[job_of(Q, Q.tile_job, gtile)];
    const uint32_t tile = gtile - P.tile_base;
    const int tx = (int)(tile % P.tiles_x), ty = (int)(tile / P.tiles_x);
    const int tminX = tx * kTileSize, tminY = ty * kTileSize;
    const int tmaxX = min(tminX + kTileSize, (int)P.width), tmaxY = min(tminY + kTileSize, (int)P.height);
    const int wminY = kDirect ? tminY + row0 : tminY, wmaxY = kDirect ? min(tminY + row1, tmaxY) : tmaxY;
    const uint32_t start = kDirect ? gtile * B.direct : B.tile_start[gtile];
    const uint32_t n = kDirect ? directRefs : B.tile_start[gtile + 1] - start;
    const uint32_t tileItem = kDirect ? 0u : B.tile_item[gtile], segLog2 = tileItem >> kImageBits;
    const uint32_t segBegin = kDirect ? 0u : seg << segLog2, segEnd = kDirect ? n : min(n, (seg + 1) << segLog2);

    const uint32_t lane = __lane_id(), wave = threadIdx.x / kWave;
    // Multisampling keeps kPassSamples samples' keys in LDS and takes the
    // item's references once per group of samples.
    const uint32_t S = kMS ? P.samples : 1u;
    for (uint32_t pass = 0; pass * kPassSamples < S; pass++) {
        const SamplePass sp = kMS ? sample_pass(P.sample_level, pass * kPassSamples,
                                                min(S - pass * kPassSamples, kPassSamples))
                                  : SamplePass{1u, 0u};
        for (uint32_t i = threadIdx.x + (kDirect ? row0 * kKeyStride<kMS> : 0);
             i < (kDirect ? row1 * kKeyStride<kMS> : sp.n * kKeyPlane<kMS>); i += kThreads)
            keys[i] = bg_key();
        if (!kDirect && threadIdx.x == 0) {
            wide->n = 0;
            wide->limit = kWideRefs<kMS>;
        }
        __syncthreads();

        // Each wave takes slices of L references (64, or a quarter of a short
        // segment so that every wave has work).  Loads run ahead of the work:
        // references three slices ahead, index-buffer entries two and screen
        // vertices one, so no slice waits on a chain of dependent loads.  All
        // are unconditional, at clamped addresses, so that the in-order
        // vector-memory wait count stays exact.
        const uint32_t segLen = segEnd - segBegin;
        const uint32_t L = segLen >= kThreads ? kWave : (segLen + kThreads / kWave - 1) / (kThreads / kWave);
        const uint32_t stride = L * (kThreads / kWave);
        const uint32_t first = segBegin + wave * L + lane;
        const uint32_t* segRefs = B.refs + start;
        // (An unused index may be anything; a used one is of a checked triangle.)
        const uint32_t lastV = P.num_vertices - 1u;
        auto sv_of = [&](const uint3& idx, ScreenVert& a, ScreenVert& b2, ScreenVert& c) {
            a = B.sverts[P.vert_base + min(idx.x, lastV)];
            b2 = B.sverts[P.vert_base + min(idx.y, lastV)];
            c = B.sverts[P.vert_base + min(idx.z, lastV)];
        };
        uint32_t pay1 = segRefs[min(first, segEnd - 1)];
        uint32_t pay2 = segRefs[min(first + stride, segEnd - 1)];
        uint32_t pay3 = segRefs[min(first + 2 * stride, segEnd - 1)];
        ScreenVert n0, n1, n2;
        sv_of(ref_indices(P, pay1), n0, n1, n2);
        uint3 idx2 = ref_indices(P, pay2);
        // Pixel box of a FineRasterize reference (Core/Rasterizer.h:132-140);
        // whether the triangle's own is at most 2x2.
        auto pixel_box = [&](const RTri& t, int& minX, int& maxX, int& minY, int& maxY) {
            const int bx0 = min(t.x0, min(t.x1, t.x2)) >> 4, bx1 = max(t.x0, max(t.x1, t.x2)) >> 4;
            const int by0 = min(t.y0, min(t.y1, t.y2)) >> 4, by1 = max(t.y0, max(t.y1, t.y2)) >> 4;
            minX = max(tminX, bx0);
            maxX = min(tmaxX - 1, bx1);
            minY = max(wminY, by0);
            maxY = min(wmaxY - 1, by1);
            return bx1 - bx0 <= 1 && by1 - by0 <= 1;
        };
        // Quads of a reference beyond the tiny path: the first one's pixel, quads per row.
        auto quad_box = [&](int minX, int maxX, int minY, int maxY, int& fx, int& fy, int& fnx) -> uint32_t {
            minX &= ~1;
            minY &= ~1;
            if (maxX < minX || maxY < minY) return 0;
            fx = minX;
            fy = minY;
            fnx = (int)((uint32_t)(maxX - minX) / 2u) + 1;
            return (uint32_t)fnx * ((uint32_t)(maxY - minY) / 2u + 1u);
        };
        uint32_t b = segBegin + wave * L;
        for (uint32_t until = kMS ? segBegin + kWideRefs<kMS> : segEnd;; until += kWideRefs<kMS>) {
            for (; b < min(segEnd, until); b += stride) {
                const uint32_t p = b + lane;
                const bool valid = lane < L && p < segEnd;
                const uint32_t pay = pay1;
                const uint32_t rid = pay & kRecordMask;
                const bool trivial = ((pay >> kRecordBits) & 7u) == 7u;
                const bool big = (pay >> 31) != 0;
                const bool compact = pay <= kRecordMask;
                const ScreenVert s0 = n0, s1 = n1, s2 = n2;
                sv_of(idx2, n0, n1, n2);
                idx2 = ref_indices(P, pay3);
                pay1 = pay2;
                pay2 = pay3;
                pay3 = segRefs[min(p + 3 * stride, segEnd - 1)];
                // Tile-level paths (RasterizeTile, Core/Renderer.cpp:255-268):
                // trivially accepted, or big with hierarchical rasterisation on.
                const bool large = valid && (trivial || (big && P.hierarchical));
                // Every lane holds its own record; large ones are broadcast below.
                RTri t;
                screen_rtri_from(s0, s1, s2, rid, t);
                bool fits = true;
                if (valid && !compact) {
                    load_rtri(B.rrec[rid], t);
                    fits = fits24(t);
                }
                uint32_t myQ = 0;  // quads of a FineRasterize reference beyond the tiny path
                int fx = 0, fy = 0, fnx = 1;
                if (valid && !large) {
                    int minX, maxX, minY, maxY;
                    if (pixel_box(t, minX, maxX, minY, maxY)) {
                        // Test only the box's pixels.  The reference's even-aligned
                        // quads add pixels whose centres lie outside the bbox, hence
                        // outside the triangle, and with edges this short no edge
                        // function can wrap.
                        if (maxX >= minX && maxY >= minY)
                            quad_depth<kMS, true>(t, minX, minY, true, tminX, tminY, keys, maxX, maxY, sp);
                    } else {
                        myQ = quad_box(minX, maxX, minY, maxY, fx, fy, fnx);
                    }
                }
                const bool isWide = large || myQ >= kWaveQuads || (myQ && !fits);
                bool walkNow = kDirect;
                if (!kDirect)
                    if (const uint64_t wm = __ballot(isWide)) {
                        const uint32_t count = (uint32_t)__popcll(wm);
                        uint32_t at = 0;
                        if (lane == 0) at = atomicAdd(&wide->n, count);
                        at = __builtin_amdgcn_readfirstlane(at);
                        walkNow = !kMS && at + count > kWideRefs<kMS>;
                        if (walkNow) {
                            if (lane == 0) atomicMin(&wide->limit, at);
                        } else if (isWide) {
                            wide->at[at + (uint32_t)__popcll(wm & lanemask_lt())] = (uint16_t)(p - segBegin);
                        }
                    }
                if (walkNow)
                    walk_wide<kMS>(P, t, pay, large, isWide ? myQ : 0u, fx, fy, fnx, tminX, tminY, tmaxX, tmaxY,
                                   keys, sp, row0 / 8, row1 / 8);
                if (isWide) myQ = 0;
                // Other references with quads: the wave's quads are expanded into
                // (reference, quad) pairs and tested 64 per pass, one quad per lane.
                // Pair k's entry in the wave's owner table holds the owner lane and
                // the quad's column and row in the owner's bbox.
                const uint32_t incl = wave_incl_scan(myQ);
                const uint32_t totalQ = __builtin_amdgcn_readlane(incl, kWave - 1);
                if (totalQ) {
                    {
                        uint16_t* own = &sOwner[wave][incl - myQ];
                        uint32_t cx = 0, cy = 0;
                        for (uint32_t i = 0; __ballot(i < myQ); i++) {
                            if (i < myQ) {
                                own[i] = (uint16_t)(lane | (cx << 6) | (cy << 10));
                                if (++cx == (uint32_t)fnx) {
                                    cx = 0;
                                    cy++;
                                }
                            }
                        }
                    }
                    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                    __builtin_amdgcn_wave_barrier();
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                    for (uint32_t base = 0; base < totalQ; base += kWave) {
                        const uint32_t k = base + lane;
                        const uint32_t e = k < totalQ ? sOwner[wave][k] : 0u;
                        const int j = (int)(e & 63u);
                        RTri u;
                        u.x0 = __shfl(t.x0, j); u.y0 = __shfl(t.y0, j);
                        u.x1 = __shfl(t.x1, j); u.y1 = __shfl(t.y1, j);
                        u.x2 = __shfl(t.x2, j); u.y2 = __shfl(t.y2, j);
                        u.B0 = u.y0 - u.y1; u.C0 = u.x1 - u.x0;
                        u.B1 = u.y1 - u.y2; u.C1 = u.x2 - u.x1;
                        u.B2 = u.y2 - u.y0; u.C2 = u.x0 - u.x2;
                        u.pb0 = __shfl(t.pb0, j); u.pb1 = __shfl(t.pb1, j); u.pb2 = __shfl(t.pb2, j);
                        u.inv_det = __shfl(t.inv_det, j);
                        u.z0 = __shfl(t.z0, j); u.z1 = __shfl(t.z1, j); u.z2 = __shfl(t.z2, j);
                        u.order = __shfl(t.order, j);
                        const int ux = __shfl(fx, j), uy = __shfl(fy, j);
                        if (k < totalQ)
                            quad_depth<kMS, true>(u, ux + 2 * (int)((e >> 6) & 15u), uy + 2 * (int)(e >> 10), true,
                                                  tminX, tminY, keys, sp);
                    }
                }
            }
            __syncthreads();
            if (kDirect) return;
            // The listed references, dealt out to the waves.  (When each wave
            // walked its own slices' wide references, the wave that had the item's
            // last slice walked most of them, as heavy references end a tile's
            // list: 12 quad-walked and 10 tile-level ones made an item of 39 us
            // beside 12 on average, and the 2.1M sphere grid at 1080p took 45 us,
            // 127 with 4 samples; so 36 and 86 (34 and 78 with later steps).  With a
            // quadrant or 64 quads of each reference per wave its preparation by four
            // waves cost more than the finer split gave: 40 and 86.)
            const uint32_t nWide = __builtin_amdgcn_readfirstlane(min(wide->n, wide->limit));
            // With more samples and fewer references than waves, two or four waves
            // share each, by quadrants or by rows of quads: large triangles' tiles
            // have one to four, and one wave of eight walking took longer than of four
            // (200 triangles on 2454x2310, 4 samples, a call 360 us, so 322; 338 with
            // workgroups of four waves and none shared).
            constexpr uint32_t kWaves = kThreads / kWave;
            const uint32_t parts = !kMS ? 1u : 4 * nWide <= kWaves ? 4u : 2 * nWide <= kWaves ? 2u : 1u;
            const uint32_t part = wave % parts;
            for (uint32_t e0 = 0; e0 < nWide; e0 += kThreads) {
                const uint32_t e = e0 + wave / parts + kWaves / parts * lane;
                const bool valid = e < nWide;
                const uint32_t pay = segRefs[segBegin + wide->at[valid ? e : 0u]];
                const uint32_t rid = pay & kRecordMask;
                const bool big = (pay >> 31) != 0, trivial = ((pay >> kRecordBits) & 7u) == 7u;
                const bool large = valid && (trivial || (big && P.hierarchical));
                RTri t;
                if (pay > kRecordMask) load_rtri(B.rrec[rid], t);
                else screen_rtri(P, B, rid, t);
                uint32_t quads = 0;
                int fx = 0, fy = 0, fnx = 1;
                if (valid && !large) {
                    int minX, maxX, minY, maxY;
                    pixel_box(t, minX, maxX, minY, maxY);
                    quads = quad_box(minX, maxX, minY, maxY, fx, fy, fnx);
                    if (kMS) {
                        const uint32_t rows = quads / (uint32_t)fnx, r0 = rows * part / parts;
                        quads = (rows * (part + 1) / parts - r0) * (uint32_t)fnx;
                        fy += 2 * (int)r0;
                    }
                }
                walk_wide<kMS>(P, t, pay, large, quads, fx, fy, fnx, tminX, tminY, tmaxX, tmaxY, keys, sp,
                               (int)(4 * part / parts), (int)(4 * (part + 1) / parts));
            }
            if (until >= segEnd) {
                if (nWide) __syncthreads();
                break;
            }
            __syncthreads();
            if (threadIdx.x == 0) wide->n = 0;
            __syncthreads();
        }
        uint64_t* g = B.partials +
                      ((size_t)((tileItem & kImageMask) + seg) * S + pass * kPassSamples) * (kTileSize * kTileSize);
        // A tile of one segment has no other image to merge with, and k_shade
        // recomputes the depth: the low words of the keys (the winners'
        // orders; 0xFFFFFFFF where nothing was drawn) are its image.
        const bool orders = !kMS && (segFlag >> kSegIndexBits);
        for (uint32_t i = threadIdx.x; i < sp.n * kTileSize * kTileSize; i += kThreads) {
            const uint32_t plane = i / (kTileSize * kTileSize), p = i % (kTileSize * kTileSize);
            const uint64_t k = keys[plane * kKeyPlane<kMS> + (p / kTileSize) * kKeyStride<kMS> + p % kTileSize];
            if (orders) reinterpret_cast<uint32_t*>(g)[i] = (uint32_t)k;
            else g[i] = k;
        }
        __syncthreads();
    }
}

// Cleared pixels of an empty tile (as k_shade writes uncovered ones): four pixels
// per store where the rows start on 16 bytes, else one.  thread: of kThreads that
// share the tile's rows [row0, row1).
template <uint32_t kThreads>
__device__ __forceinline__ void clear_tile(const BatchParams& Q, const FrameParams* __restrict__ jobs,
                                           const DeviceBuffers& B, uint32_t gtile, uint32_t thread,
                                           uint32_t row0 = 0, uint32_t row1 = kTileSize) {
    const FrameParams& P = jobs[job_of(Q, Q.tile_job, gtile)];
    const uint32_t tile = gtile - P.tile_base;
    const int tminX = (int)(tile % P.tiles_x) * kTileSize, tminY = (int)(tile / P.tiles_x) * kTileSize;
    const uint64_t align = (uint64_t)B.color | (uint64_t)B.depth | (uint64_t)B.ids | (uint64_t)B.color_f32 |
                           4ull * (P.pix_base | P.width);
    if (!(align & 15u)) {
        constexpr uint32_t kRow = kTileSize / 4;
        for (uint32_t i = thread + kRow * row0; i < kRow * row1; i += kThreads) {
            const int x = tminX + (int)(i % kRow) * 4, y = tminY + (int)(i / kRow);
            if (x < (int)P.width && y < (int)P.height) {
                const size_t o = P.pix_base + (size_t)(P.height - 1 - y) * P.width + x;
                *reinterpret_cast<uint4*>(B.color + o) = make_uint4(0u, 0u, 0u, 0u);
                *reinterpret_cast<float4*>(B.depth + o) = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
                *reinterpret_cast<uint4*>(B.ids + o) = make_uint4(~0u, ~0u, ~0u, ~0u);
                if (B.color_f32)
                    for (uint32_t k = 0; k < 3; k++)
                        reinterpret_cast<float4*>(B.color_f32 + 3 * o)[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
        }
        return;
    }
    for (uint32_t i = thread + kTileSize * row0; i < kTileSize * row1; i += kThreads) {
        const int x = tminX + (int)(i % kTileSize), y = tminY + (int)(i / kTileSize);
        if (x < (int)P.width && y < (int)P.height) {
            const size_t o = P.pix_base + (size_t)(P.height - 1 - y) * P.width + x;
            B.color[o] = 0u;
            B.depth[o] = 1.0f;
            B.ids[o] = 0xFFFFFFFFu;
            if (B.color_f32) B.color_f32[3 * o] = B.color_f32[3 * o + 1] = B.color_f32[3 * o + 2] = 0.0f;
        }
    }
}

}  // namespace

namespace {
// Record and shading vertices of the winner with submission order `order`:
// clipped pieces from their stored record, unclipped triangles rebuilt from
// their vertices' screen values (1/det as setup computed it).  With
// recompute, the screen values come from the shading vertices' positions
// (transform, divide and snap exactly as k_vertex computes them) instead of
// a second gather: cheaper where neighbouring pixels have different winners
// (deep tiles of small triangles), dearer where they share them.
__device__ __forceinline__ void winner_tri(const FrameParams& P, const DeviceBuffers& B, uint32_t order, bool recompute,
                                           RTri& t, ShadeVert& v0, ShadeVert& v1, ShadeVert& v2) {
    const uint32_t tri = order >> 4;  // triangle slot
    if (order & 1u) {
        const uint32_t ri = (B.desc[tri] >> 3) + ((order >> 1) & 7u);
        const ShadeRec s = B.srec[ri];
        v0 = B.verts[s.v0];
        v1 = B.verts[s.v1];
        v2 = B.verts[s.v2];
        load_rtri(B.rrec[ri], t);
    } else {
        const GlobalPtr<uint32_t> idx = as_global(P.mesh.idx) + 3 * (size_t)(tri - P.slot_base);
        const uint32_t v0i = P.vert_base + idx[0], v1i = P.vert_base + idx[1], v2i = P.vert_base + idx[2];
        if (recompute) {
            v0 = B.verts[v0i];
            v1 = B.verts[v1i];
            v2 = B.verts[v2i];
            auto clip = [&](const ShadeVert& v) { return xform4(P.mvp, v.px, v.py, v.pz, 1.0f); };
            const float4 c0 = clip(v0), c1 = clip(v1), c2 = clip(v2);
            auto screen = [&](const float4& h, int& x, int& y, float& z) {
                const int2 xy = snap_point(P, h.x, h.y, h.z);
                x = xy.x;
                y = xy.y;
                z = h.w;
            };
            const bool normal = project_is_normal(c0) && project_is_normal(c1) && project_is_normal(c2);
            screen(normal ? project_normal(c0) : project_any(c0), t.x0, t.y0, t.z0);
            screen(normal ? project_normal(c1) : project_any(c1), t.x1, t.y1, t.z1);
            screen(normal ? project_normal(c2) : project_any(c2), t.x2, t.y2, t.z2);
        } else {
            const ScreenVert s0 = B.sverts[v0i], s1 = B.sverts[v1i], s2 = B.sverts[v2i];
            t.x0 = s0.x; t.y0 = s0.y; t.x1 = s1.x; t.y1 = s1.y; t.x2 = s2.x; t.y2 = s2.y;
            t.z0 = s0.z; t.z1 = s1.z; t.z2 = s2.z;
            v0 = B.verts[v0i];
            v1 = B.verts[v1i];
            v2 = B.verts[v2i];
        }
        t.B1 = t.y1 - t.y2; t.C1 = t.x2 - t.x1;
        t.B2 = t.y2 - t.y0; t.C2 = t.x0 - t.x2;
        t.inv_det = rcp_normal((float)(t.C2 * t.B1 - t.C1 * t.B2));
    }
}
}  // namespace

// One pixel of a single-sample frame, output index o: the winner's colour, depth
// and ID, or the cleared values.  low: the low word of the winner's key
// (0xFFFFFFFF where nothing was drawn).
namespace {
template <bool kTex>
__device__ __forceinline__ void shade_winner(const FrameParams& P, const DeviceBuffers& B, int x, int y, size_t o,
                                             uint32_t low, bool recompute) {
    if (low == 0xFFFFFFFFu) {
        B.color[o] = 0u;
        B.depth[o] = 1.0f;
        B.ids[o] = 0xFFFFFFFFu;
        if (B.color_f32) B.color_f32[3 * o] = B.color_f32[3 * o + 1] = B.color_f32[3 * o + 2] = 0.0f;
        return;
    }
    // The key's low word is the winner's submission order (make_order).
    const uint32_t order = 0xFFFFFFFEu - low;
    RTri t;
    ShadeVert v0, v1, v2;
    winner_tri(P, B, order, recompute, t, v0, v1, v2);
    float l0, l1, d;
    bary_depth(t, x * 16 + 8, y * 16 + 8, l0, l1, d);
    const float3 c = shade_any<kTex>(P, t, order, x, y, l0, l1, v0, v1, v2);
    B.color[o] = to_byte(c.x) | (to_byte(c.y) << 8) | (to_byte(c.z) << 16) | (255u << 24);
    if (B.color_f32) {
        B.color_f32[3 * o] = clamp01(c.x);
        B.color_f32[3 * o + 1] = clamp01(c.y);
        B.color_f32[3 * o + 2] = clamp01(c.z);
    }
    B.depth[o] = d;
    B.ids[o] = (order >> 4) - P.slot_base;
}
}  // namespace

}  // namespace edxr
