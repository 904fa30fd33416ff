// pipeline.hip -- gfx950 kernels of the EDXRaster hot path.
//
// Every kernel reads its job's constants from a device table (FrameParams):
// a plain frame is a batch of one job, a batch renders many independent jobs
// with the same launches.  Stages (EDXRaster/Core/Renderer.cpp:100-118 order):
//   k_vertex     one lane per vertex: SoA in, 48-byte shading vertex out
//                (VertexProcessing, Core/Renderer.cpp:120-127); it also clears
//                the counters and writes a single job's table entry (k_reset
//                does that alone for a frame without vertices).
//   k_setup      vertex transform + outcodes + triangle setup, one lane per
//                triangle (DefaultVertexShader::Execute Core/Shader.h:40-49,
//                Clipper::Clip Core/Clipper.h:71-189, RasterTriangle::Setup
//                Core/RasterTriangle.h:27-153).  Straddling triangles are
//                queued for k_clip.
//   k_clip       Sutherland-Hodgman clipping + fan setup of queued triangles
//                (Core/Clipper.h:109-170,192-288).
//   k_bin_count  per-chunk tile histograms (binning, Core/Renderer.cpp:161-230)
//   k_bin_colpass (or k_bin_colsum / k_bin_groupscan / k_bin_colscan) and
//   k_bin_tilescan (or k_bin_tilesums / k_bin_tileplace)
//                exclusive scans -> per-(tile, chunk) offsets and the raster
//                work list of (tile, segment) items.
//   k_bin_scatter scatter through LDS cursors: a tile's list holds the chunks'
//                references in chunk order (the reference concatenates its
//                per-core lists in core order, Core/Renderer.cpp:250-253); the
//                depth keys carry the submission order, so the list order
//                within a chunk does not matter.
//   k_raster     persistent: hierarchical edge-function coverage of one (tile,
//                segment) item at a time (CoarseRasterize / FineRasterize /
//                TrivialAcceptTriangle, Core/Rasterizer.h:32-200,310-353) and
//                the depth test as a (depth, submission order) key minimum.
//   k_shade      per tile: minimum key over the tile's items, perspective-correct
//                interpolation + pixel shading of the winner and one write-back
//                of colour, depth and triangle ID (Core/Renderer.cpp:272-350).
//
// Arithmetic follows the reference operation by operation: int32 wrap
// (-fwrapv), truncating 28.4 snap, round-to-nearest int->float, correctly
// rounded division and sqrt, no FMA contraction (-ffp-contract=off).
#include <hip/hip_runtime.h>

#include <mutex>

#include "device.h"

// Scratch of the allocation-free frame (edxr_render_mesh_noalloc), one copy
// per device.  Host code never uses this name as an address: the device
// address comes from hipGetSymbolAddress (scratch_address below).
static __device__ __align__(256) uint8_t scratch[edxr::kScratchBytes];

namespace edxr {

namespace {
constexpr uint32_t kSetupSlots = 4;  // triangle slots per k_setup thread
constexpr uint32_t kShadeThreads = 512;
constexpr uint32_t kShadeListTiles = 8192;  // k_shade walks the work list beyond these tiles, with
constexpr uint32_t kShadeGroups = 16;       // this many workgroups per CU (batch 416 us; 4 per CU 428)
static_assert(kJobAlign % (kBlock * kSetupSlots) == 0, "a vertex/setup block must not span two jobs");
}  // namespace

// ---------------------------------------------------------------------------
// Counters
// ---------------------------------------------------------------------------
__global__ void k_reset(uint32_t* counters, FrameParams* jobs, FrameParams job0, int writeJob) {
    for (uint32_t i = threadIdx.x; i < kCntSlots; i += blockDim.x) counters[i] = 0;
    if (writeJob && threadIdx.x == 0) jobs[0] = job0;
}

// A batch's block -> job tables, a workgroup per job.  (The host filled and
// uploaded them before: 180K entries for 256 jobs, 94 us of a batch's 1.69 ms;
// this takes 6 us.)
__global__ __launch_bounds__(kBlock) void k_job_tables(BatchParams Q, const FrameParams* __restrict__ jobs) {
    const uint32_t k = blockIdx.x;
    const FrameParams& P = jobs[k];
    const bool last = k + 1 == Q.num_jobs;
    auto fill = [&](const uint32_t* table, uint32_t first, uint32_t end) {
        for (uint32_t i = first + threadIdx.x; i < end; i += kBlock) const_cast<uint32_t*>(table)[i] = k;
    };
    // Padding blocks up to the next job's base belong to the job before it.
    fill(Q.vblock_job, P.vert_base / kJobTableBlock, last ? Q.vert_blocks : jobs[k + 1].vert_base / kJobTableBlock);
    fill(Q.sblock_job, P.slot_base / kJobTableBlock, last ? Q.slot_blocks : jobs[k + 1].slot_base / kJobTableBlock);
    fill(Q.chunk_job, P.chunk_base, P.chunk_base + P.num_chunks);
    fill(Q.tile_job, P.tile_base, P.tile_base + P.num_tiles);
}

// ---------------------------------------------------------------------------
// Vertex processing (Core/Renderer.cpp:120-127): one lane per vertex, SoA
// input read coalesced, one 48-byte shading record out.  invW = 1/w of
// DefaultVertexShader's MVP transform (Core/Shader.h:45) as the z-divide loop
// computes it (Core/Renderer.cpp:144).
// It also does k_reset's work, one launch fewer per frame: block 0 clears
// the counters, and with kArgJob (a single job passed by value) every block
// reads the job from the argument and block 0 writes it to the job table for
// the later kernels.
// ---------------------------------------------------------------------------
template <bool kArgJob>
__global__ __launch_bounds__(kBlock) void k_vertex(BatchParams Q, const FrameParams* __restrict__ jobs,
                                                   ShadeVert* __restrict__ verts, ScreenVert* __restrict__ sverts,
                                                   uint32_t* counters, FrameParams* jobTable, FrameParams job0) {
    if (blockIdx.x == 0) {
        for (uint32_t i = threadIdx.x; i < kCntSlots; i += kBlock) counters[i] = 0;
        if (kArgJob && threadIdx.x == 0) jobTable[0] = job0;
    }
    const FrameParams& P = kArgJob ? job0 : jobs[job_of(Q, Q.vblock_job, blockIdx.x)];
    vertex_slot(P, blockIdx.x * kBlock + threadIdx.x, verts, sverts);
}

// ---------------------------------------------------------------------------
// Setup: one lane per input triangle.
// ---------------------------------------------------------------------------
// Each thread takes kSetupSlots slots kBlock apart; all their index and
// screen-vertex loads are issued before any is used, so one wave keeps
// several dependent-load chains in flight.
// Held to 64 VGPRs: eight waves per SIMD, so that a 2M-triangle frame's
// 8,192 waves are resident at once (one round of the load chain).
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_setup(
    BatchParams Q, const FrameParams* __restrict__ jobs, DeviceBuffers B) {
    const FrameParams& P = jobs[job_of(Q, Q.sblock_job, blockIdx.x * kSetupSlots)];
    const MeshPtrs& M = P.mesh;
    // k_bin_count adds the big references of every tile to zeroed counts;
    // k_bin_colpass's look-back starts from cleared status words.
    for (uint32_t t = blockIdx.x * kBlock + threadIdx.x; t < Q.total_tiles; t += gridDim.x * kBlock)
        B.tile_big[t] = 0u;
    if (!B.legacy_scans)
        for (uint64_t i = blockIdx.x * kBlock + threadIdx.x; i < B.group_entries; i += gridDim.x * kBlock)
            B.group_sums[i] = 0u;
    uint32_t s[kSetupSlots], i0[kSetupSlots], i1[kSetupSlots], i2[kSetupSlots];
    bool valid[kSetupSlots];
#pragma unroll
    for (uint32_t u = 0; u < kSetupSlots; u++) {
        s[u] = (blockIdx.x * kSetupSlots + u) * kBlock + threadIdx.x;  // triangle slot
        const uint32_t t = s[u] - P.slot_base;                        // input triangle of the job
        valid[u] = t < P.num_triangles;
        i0[u] = i1[u] = i2[u] = 0;
        if (valid[u]) {
            i0[u] = M.idx[3 * (size_t)t];
            i1[u] = M.idx[3 * (size_t)t + 1];
            i2[u] = M.idx[3 * (size_t)t + 2];
        }
    }
    // The vertices' snapped positions and outcodes; z is loaded only for the
    // few triangles whose record is stored (a compact record is rebuilt from
    // the screen vertices by its readers).
    int2 xy[kSetupSlots][3];
    uint32_t code[kSetupSlots][3];
    bool bad[kSetupSlots];
#pragma unroll
    for (uint32_t u = 0; u < kSetupSlots; u++) {
        bad[u] = valid[u] && (i0[u] >= P.num_vertices || i1[u] >= P.num_vertices || i2[u] >= P.num_vertices);
        if (P.shader == kTexturedLambert && valid[u] && M.tex[s[u] - P.slot_base] >= P.num_tex) bad[u] = true;
        if (valid[u] && !bad[u]) {
            const ScreenVert* v0 = &B.sverts[P.vert_base + i0[u]];
            const ScreenVert* v1 = &B.sverts[P.vert_base + i1[u]];
            const ScreenVert* v2 = &B.sverts[P.vert_base + i2[u]];
            xy[u][0] = *reinterpret_cast<const int2*>(v0);
            xy[u][1] = *reinterpret_cast<const int2*>(v1);
            xy[u][2] = *reinterpret_cast<const int2*>(v2);
            code[u][0] = v0->code;
            code[u][1] = v1->code;
            code[u][2] = v2->code;
        }
    }
    uint32_t nrej = 0, nbad = 0, nmain = 0;
    bool queuedU[kSetupSlots];
    uint64_t qmask[kSetupSlots];
#pragma unroll
    for (uint32_t u = 0; u < kSetupSlots; u++) {
        bool rejected = false, queued = false, main = false;
        RasterRec rec;
        if (valid[u] && !bad[u]) {
            if (code[u][0] | code[u][1] | code[u][2]) {
                if (code[u][0] & code[u][1] & code[u][2]) rejected = true;
                else queued = true;
            } else {
                // the cull test of RasterTriangle::Setup (setup_snapped)
                const int2 a = xy[u][0], b = xy[u][1], c = xy[u][2];
                main = (a.x - c.x) * (b.y - c.y) - (c.x - b.x) * (c.y - a.y) > 0;
                rec.x0 = a.x; rec.y0 = a.y; rec.x1 = b.x; rec.y1 = b.y; rec.x2 = c.x; rec.y2 = c.y;
            }
        }
        queuedU[u] = queued;
        qmask[u] = __ballot(queued);
        if (valid[u]) {
            uint32_t d = 0;
            if (main) {
                // A compact triangle's record is not stored: it is the three
                // vertices' screen values, which the raster re-reads.
                d = compact_desc(P, rec, s[u]);
                if (!(d & kDescCompact)) {
                    setup_snapped(rec.x0, rec.y0, rec.x1, rec.y1, rec.x2, rec.y2, rec);
                    // invW and the z divide (Core/Renderer.cpp:139-147).
                    rec.z0 = B.sverts[P.vert_base + i0[u]].z;
                    rec.z1 = B.sverts[P.vert_base + i1[u]].z;
                    rec.z2 = B.sverts[P.vert_base + i2[u]].z;
                    rec.order = make_order(s[u], 0, false);
                    B.rrec[s[u]] = rec;
                }
            }
            B.desc[s[u]] = d;
        }
        nrej += wave_count(rejected);
        nbad += wave_count(bad[u]);
        nmain += wave_count(main);
    }
    // Per-workgroup totals, one striped atomic per counter per workgroup, and
    // one clip-queue allocation per workgroup (same-address atomics from every
    // wave would serialise in L2).
    __shared__ uint32_t wgCount[3];
    __shared__ uint32_t sQueued[kBlock / kWave], sQueueBase[kBlock / kWave];
    const uint32_t wave = threadIdx.x / kWave;
    uint32_t nq = 0;
#pragma unroll
    for (uint32_t u = 0; u < kSetupSlots; u++) nq += (uint32_t)__popcll(qmask[u]);
    if (__lane_id() == 0) sQueued[wave] = nq;
    if (threadIdx.x < 3) wgCount[threadIdx.x] = 0;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t tq = 0;
        for (uint32_t w = 0; w < kBlock / kWave; w++) {
            sQueueBase[w] = tq;
            tq += sQueued[w];
        }
        const uint32_t qb = tq ? atomicAdd(&B.counters[kCntClipQueue], tq) : 0u;
        for (uint32_t w = 0; w < kBlock / kWave; w++) sQueueBase[w] += qb;
    }
    if (__lane_id() == 0) {
        if (nrej) atomicAdd(&wgCount[0], nrej);
        if (nbad) atomicAdd(&wgCount[1], nbad);
        if (nmain) atomicAdd(&wgCount[2], nmain);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t stripe = blockIdx.x & (kStripes - 1);
        if (wgCount[0]) atomicAdd(&B.counters[kCntStriped + kStRejected * kStripes + stripe], wgCount[0]);
        if (wgCount[1]) atomicAdd(&B.counters[kCntBadIndex], wgCount[1]);
        if (wgCount[2]) atomicAdd(&B.counters[kCntStriped + kStMainRecords * kStripes + stripe], wgCount[2]);
    }
    if (nq) {
        uint32_t slot = sQueueBase[wave];
#pragma unroll
        for (uint32_t u = 0; u < kSetupSlots; u++) {
            if (queuedU[u]) {
                const uint32_t at = slot + (uint32_t)__popcll(qmask[u] & lanemask_lt());
                if (at < B.clip_queue_cap) B.clip_queue[at] = s[u];
                else atomicOr(&B.counters[kCntOverflow], (uint32_t)kOvClipQueue);
            }
            slot += (uint32_t)__popcll(qmask[u]);
        }
    }
}

// ---------------------------------------------------------------------------
// Clipping of queued straddlers (rare path).
// ---------------------------------------------------------------------------
namespace {

__device__ __forceinline__ bool plane_inside(const float4& v, int p) {
    switch (p) {
        case 0: return v.x >= -v.w;
        case 1: return v.x <= v.w;
        case 2: return v.y >= -v.w;
        case 3: return v.y <= v.w;
        case 4: return v.z <= v.w;
        default: return v.z >= 0.0f;
    }
}
__device__ __forceinline__ float plane_t(const float4& a, const float4& b, int p) {
    switch (p) {
        case 0: return (a.w + a.x) / ((a.x + a.w) - (b.x + b.w));
        case 1: return (-a.w + a.x) / ((a.x - a.w) - (b.x - b.w));
        case 2: return (a.w + a.y) / ((a.y + a.w) - (b.y + b.w));
        case 3: return (-a.w + a.y) / ((a.y - a.w) - (b.y - b.w));
        case 4: return (-a.w + a.z) / ((a.z - a.w) - (b.z - b.w));
        default: return a.z / (a.z - b.z);
    }
}
__device__ __forceinline__ void plane_snap(float4& v, int p) {
    switch (p) {
        case 0: v.x = -v.w; break;
        case 1: v.x = v.w; break;
        case 2: v.y = -v.w; break;
        case 3: v.y = v.w; break;
        case 4: v.z = v.w; break;
        default: v.z = 0.0f; break;
    }
}

// Plane order of ClipPolygon (Core/Clipper.h:238-278): L R B T F N.
__device__ const uint32_t kPlaneBits[6] = {1u, 2u, 4u, 8u, 32u, 16u};

}  // namespace

// One wave per queued triangle, one polygon vertex per lane (kMaxPoly <= 64),
// 16 triangles per workgroup pass.  Clipper::ClipByPlane (Core/Clipper.h:
// 192-232) per plane: lane i takes the edge (i, i + 1) and emits 0, 1 or 2
// vertices, and a wave prefix sum places them in the reference's output
// order; the arithmetic per vertex is the serial algorithm's.  The passes'
// vertex and record allocations are summed in LDS and taken with one atomic
// each per workgroup pass (one per triangle would serialise in L2).
namespace {
__device__ __forceinline__ float4 shfl4(const float4& v, int src) {
    return make_float4(__shfl(v.x, src), __shfl(v.y, src), __shfl(v.z, src), __shfl(v.w, src));
}
constexpr uint32_t kClipWaves = 16;  // waves (triangles) per workgroup pass
// Input vertex v of a job's mesh with its shading attributes (the caller sets inv_w).
__device__ __forceinline__ ShadeVert input_vertex(const MeshPtrs& M, uint32_t v) {
    ShadeVert o;
    o.px = global_at(M.px, v);
    o.py = global_at(M.py, v);
    o.pz = global_at(M.pz, v);
    o.nx = global_at(M.nx, v);
    o.ny = global_at(M.ny, v);
    o.nz = global_at(M.nz, v);
    o.cr = M.cr ? global_at(M.cr, v) : 0.0f;
    o.cg = M.cg ? global_at(M.cg, v) : 0.0f;
    o.cb = M.cb ? global_at(M.cb, v) : 0.0f;
    o.inv_w = 0.0f;
    o.u = M.tu ? global_at(M.tu, v) : 0.0f;
    o.v = M.tv ? global_at(M.tv, v) : 0.0f;
    return o;
}
}  // namespace

// Direct frames (k_front) have no binning pass after this one: kDirect appends
// each record's references to its tiles' lists.
template <bool kDirect>
__global__ __launch_bounds__(kClipWaves * 64) void k_clip(BatchParams Q, const FrameParams* __restrict__ jobs,
                                                           DeviceBuffers B) {
    __shared__ uint32_t sNew[kClipWaves], sRec[kClipWaves], sVBase[kClipWaves], sRBase[kClipWaves];
    __shared__ uint32_t sStat[2];
    const int lane = (int)__lane_id();
    const uint32_t wave = threadIdx.x / 64;
    const uint32_t n = min(B.counters[kCntClipQueue], B.clip_queue_cap);
    uint32_t clipped = 0, nearClipped = 0;  // this wave's statistics (lane 0)
    // The workgroup's allocation stripe and the stripes' regions.
    const uint32_t stripe = blockIdx.x % kAllocStripes;
    const uint32_t vRegion = B.extra_vert_cap / kAllocStripes, rRegion = B.extra_rec_cap / kAllocStripes;
    for (uint32_t base = blockIdx.x * kClipWaves; base < n; base += gridDim.x * kClipWaves) {
        const uint32_t q = base + wave;
        const bool live = q < n;
        // ---- per wave: clip its triangle (no global writes yet) ----
        uint32_t t = 0, vi[3] = {0, 0, 0};
        uint32_t outside = 0;  // bit k: input vertex k has a nonzero outcode
        ShadeVert pa, pb, pc;
        float4 pos = make_float4(0.0f, 0.0f, 0.0f, 1.0f), wgt = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        int cnt = 0;
        bool ok = true;
        const FrameParams* Pp = jobs;
        if (live) {
            t = __builtin_amdgcn_readfirstlane(B.clip_queue[q]);  // triangle slot
            Pp = &jobs[Q.num_jobs == 1 ? 0u : __builtin_amdgcn_readfirstlane(Q.sblock_job[t / kBlock])];
            const FrameParams& P = *Pp;
            const GlobalPtr<uint32_t> idx = as_global(P.mesh.idx) + 3 * (size_t)(t - P.slot_base);
            vi[0] = P.vert_base + __builtin_amdgcn_readfirstlane(idx[0]);
            vi[1] = P.vert_base + __builtin_amdgcn_readfirstlane(idx[1]);
            vi[2] = P.vert_base + __builtin_amdgcn_readfirstlane(idx[2]);
            // from the mesh: k_vertex stores shading vertices inside the frustum only
            pa = input_vertex(P.mesh, vi[0] - P.vert_base);
            pb = input_vertex(P.mesh, vi[1] - P.vert_base);
            pc = input_vertex(P.mesh, vi[2] - P.vert_base);
            const float4 c0 = xform4(P.mvp, pa.px, pa.py, pa.pz, 1.0f);
            const float4 c1 = xform4(P.mvp, pb.px, pb.py, pb.pz, 1.0f);
            const float4 c2 = xform4(P.mvp, pc.px, pc.py, pc.pz, 1.0f);
            const uint32_t k0 = clip_code(c0), k1 = clip_code(c1), k2 = clip_code(c2);
            pa.inv_w = 1.0f / c0.w;
            pb.inv_w = 1.0f / c1.w;
            pc.inv_w = 1.0f / c2.w;
            outside = (k0 ? 1u : 0u) | (k1 ? 2u : 0u) | (k2 ? 4u : 0u);
            const uint32_t planeCode = (k0 ^ k1) | (k1 ^ k2) | (k2 ^ k0);
            clipped++;
            if ((k0 | k1 | k2) & 16u) nearClipped++;
            // The polygon: vertex `lane` of cnt (clip-space position, clip weights).
            pos = lane == 0 ? c0 : lane == 1 ? c1 : c2;
            wgt = make_float4(lane == 0 ? 1.0f : 0.0f, lane == 1 ? 1.0f : 0.0f, lane == 2 ? 1.0f : 0.0f, 0.0f);
            cnt = 3;
            for (int p = 0; p < 6; p++) {
                if (!(planeCode & kPlaneBits[p])) continue;
                const bool act = lane < cnt;
                const int i1 = lane + 1 >= cnt ? 0 : lane + 1;
                const float4 v0 = pos, w0 = wgt, v1 = shfl4(pos, i1), w1 = shfl4(wgt, i1);
                const bool in0 = plane_inside(v0, p), in1 = plane_inside(v1, p);
                const int emit = !act ? 0 : (in0 && in1) ? 1 : (in0 != in1) ? (in0 ? 1 : 2) : 0;
                // Intersection of the edge with the plane.
                float4 ip = v1, iw = w1;
                if (act && in0 != in1) {
                    const float tt = plane_t(v0, v1, p);
                    const float s = 1 - tt;
                    ip = make_float4(v0.x * s + v1.x * tt, v0.y * s + v1.y * tt, v0.z * s + v1.z * tt,
                                     v0.w * s + v1.w * tt);
                    plane_snap(ip, p);
                    iw = make_float4(w0.x * s + w1.x * tt, w0.y * s + w1.y * tt, w0.z * s + w1.z * tt, 0.0f);
                }
                // Inclusive prefix of the emitted counts over the lanes.
                const int incl = (int)wave_incl_scan((uint32_t)emit);
                const int total = __builtin_amdgcn_readlane(incl, 63);
                if (total > kMaxPoly) {
                    ok = false;
                    break;
                }
                // Output vertex `lane` comes from the edge lane whose range holds
                // it: its first item (the intersection, or v1 when both ends are
                // inside) or its second (v1 after an entering intersection).
                const int excl = incl - emit;
                int src = 0;
                for (int l = 1; l < cnt; l++) {
                    // both shuffles run with every lane active (a lane switched
                    // off by a condition reads as 0 to the others)
                    const int el = __shfl(excl, l), ml = __shfl(emit, l);
                    if (el <= lane && ml > 0) src = l;
                }
                const int k = lane - __shfl(excl, src);
                const float4 a = shfl4(ip, src), aw = shfl4(iw, src), b = shfl4(v1, src), bw = shfl4(w1, src);
                if (lane < total) {
                    pos = k == 0 ? a : b;
                    wgt = k == 0 ? aw : bw;
                }
                cnt = total;
            }
            if (!ok || cnt > 9) {
                if (lane == 0) atomicOr(&B.counters[kCntOverflow], (uint32_t)kOvPolygon);
                cnt = 0;
            }
            if (__ballot(lane < cnt && pos.w <= 0.0f) != 0) cnt = 0;
            if (cnt < 3) cnt = 0;
        }
        // Vertex ids: weight == 1 reuses a parent vertex (Core/Clipper.h:121-153);
        // new vertices are numbered in polygon order.
        const int which = (wgt.x == 1.0f) ? 0 : (wgt.y == 1.0f) ? 1 : (wgt.z == 1.0f) ? 2 : -1;
        const uint64_t newMask = __ballot(lane < cnt && which < 0);
        // Projected vertices (x/w, y/w, z/w, z * (1/w)) and the fans
        // (Core/Clipper.h:155-170): fan k = lane + 2 uses vertices (0, k - 1, k).
        const float4 h = make_float4(pos.x / pos.w, pos.y / pos.w, pos.z / pos.w, pos.z * (1.0f / pos.w));
        const int fk = lane + 2;
        const float4 h0 = shfl4(h, 0), h1 = shfl4(h, fk - 1 < 64 ? fk - 1 : 0), h2 = shfl4(h, fk < 64 ? fk : 0);
        RasterRec r;
        const bool fan = fk < cnt && setup_record(*Pp, h0.x, h0.y, h0.z, h1.x, h1.y, h1.z, h2.x, h2.y, h2.z, r);
        const uint64_t fanMask = __ballot(fan);
        const uint32_t nNew = (uint32_t)__popcll(newMask);
        const uint32_t nrec = (uint32_t)__popcll(fanMask);
        // ---- per workgroup: one allocation of vertices and records ----
        if (lane == 0) {
            sNew[wave] = nNew;
            sRec[wave] = nrec;
        }
        if (threadIdx.x == 0) sStat[0] = sStat[1] = 0;
        __syncthreads();
        if (lane == 0 && (clipped | nearClipped)) {
            atomicAdd(&sStat[0], clipped);
            atomicAdd(&sStat[1], nearClipped);
            clipped = nearClipped = 0;
        }
        if (threadIdx.x == 0) {
            uint32_t tv = 0, tr = 0;
            for (uint32_t w = 0; w < kClipWaves; w++) {
                sVBase[w] = tv;
                sRBase[w] = tr;
                tv += sNew[w];
                tr += sRec[w];
            }
            // One allocation per workgroup pass, from its stripe's region of
            // the extra vertices and records: every live workgroup reaches
            // this point at about the same time, and atomics on one address
            // would serialise.
            const uint32_t vb = tv ? atomicAdd(&B.counters[kCntAllocStriped + stripe], tv) : 0u;
            const uint32_t rb = tr ? atomicAdd(&B.counters[kCntAllocStriped + kAllocStripes + stripe], tr) : 0u;
            for (uint32_t w = 0; w < kClipWaves; w++) {
                sVBase[w] += stripe * vRegion + vb;
                sRBase[w] += stripe * rRegion + rb;
            }
        }
        __syncthreads();
        if (threadIdx.x == 0 && (sStat[0] | sStat[1])) {
            const uint32_t st = blockIdx.x & (kStripes - 1);
            atomicAdd(&B.counters[kCntStriped + kStClipped * kStripes + st], sStat[0]);
            if (sStat[1]) atomicAdd(&B.counters[kCntStriped + kStNearClipped * kStripes + st], sStat[1]);
        }
        // ---- per wave: write the new vertices, the records and the descriptor ----
        if (live) {
            const FrameParams& P = *Pp;
            const uint32_t vbase = sVBase[wave], rbase = sRBase[wave];
            // As the serial clipper: the polygon's new vertices are created
            // whenever it survives, its records when it has fans.
            const bool vfit = vbase + nNew <= (stripe + 1) * vRegion;
            if (!vfit && lane == 0) atomicOr(&B.counters[kCntOverflow], (uint32_t)kOvExtraVertices);
            bool keep = vfit && nrec > 0;
            if (keep && rbase + nrec > (stripe + 1) * rRegion) {
                if (lane == 0) atomicOr(&B.counters[kCntOverflow], (uint32_t)kOvExtraRecords);
                keep = false;
            }
            uint32_t vid = which == 0 ? vi[0] : which == 1 ? vi[1] : vi[2];
            if (vfit && lane < cnt && which < 0) {
                vid = Q.total_verts + vbase + (uint32_t)__popcll(newMask & lanemask_lt());
                auto comb = [&](float fa, float fb, float fc) { return (wgt.x * fa + wgt.y * fb) + wgt.z * fc; };
                ShadeVert o;
                o.px = comb(pa.px, pb.px, pc.px);
                o.py = comb(pa.py, pb.py, pc.py);
                o.pz = comb(pa.pz, pb.pz, pc.pz);
                o.nx = comb(pa.nx, pb.nx, pc.nx);
                o.ny = comb(pa.ny, pb.ny, pc.ny);
                o.nz = comb(pa.nz, pb.nz, pc.nz);
                o.cr = comb(pa.cr, pb.cr, pc.cr);
                o.cg = comb(pa.cg, pb.cg, pc.cg);
                o.cb = comb(pa.cb, pb.cb, pc.cb);
                o.inv_w = 1.0f / pos.w;
                o.u = comb(pa.u, pb.u, pc.u);
                o.v = comb(pa.v, pb.v, pc.v);
                B.verts[vid] = o;
            } else if (lane < cnt && which >= 0 && ((outside >> which) & 1u)) {
                // A parent vertex with a nonzero outcode that the polygon kept
                // (an intersection weight that rounds to 1): k_vertex did not
                // store it.  Every writer stores the same value.
                // (three stores, not a selected struct, so that the three
                // vertices are not spilled for a dynamic index)
                if (which == 0) B.verts[vid] = pa;
                else if (which == 1) B.verts[vid] = pb;
                else B.verts[vid] = pc;
            }
            const uint32_t vid0 = __shfl(vid, 0), vid1 = __shfl(vid, fk - 1 < 64 ? fk - 1 : 0),
                           vid2 = __shfl(vid, fk < 64 ? fk : 0);
            const uint32_t first = Q.total_slots + rbase;
            if (keep && fan) {
                const uint32_t sidx = (uint32_t)__popcll(fanMask & lanemask_lt());
                r.z0 = h0.w;
                r.z1 = h1.w;
                r.z2 = h2.w;
                r.info |= (uint32_t)(fk - 2) << 12;
                r.order = make_order(t, sidx, true);
                B.rrec[first + sidx] = r;
                B.srec[first + sidx] = ShadeRec{vid0, vid1, vid2, t};
            }
            if (lane == 0) B.desc[t] = keep ? (first << 3) | nrec : 0u;
            if (kDirect && keep) {
                // the wave takes the records one after another, 64 of a record's tiles at a time
                uint32_t refs = 0;
                for (uint64_t m = fanMask; m; m &= m - 1) {
                    const int l = __ffsll((unsigned long long)m) - 1;
                    RasterRec u;
                    u.x0 = __shfl(r.x0, l); u.y0 = __shfl(r.y0, l);
                    u.x1 = __shfl(r.x1, l); u.y1 = __shfl(r.y1, l);
                    u.x2 = __shfl(r.x2, l); u.y2 = __shfl(r.y2, l);
                    u.info = __shfl(r.info, l);
                    BinTri bt;
                    load_bin_tri(P, u, bt);
                    const uint32_t rec = first + (uint32_t)__popcll(fanMask & ((1ull << l) - 1ull));
                    enum_record_tiles(P, bt, rec, lane, kWave, [&](uint32_t tile, int, int, uint32_t payload, bool heavy) {
                        const uint32_t g = P.tile_base + tile;
                        const uint64_t one = heavy ? 1ull << 32 | 1ull : 1ull;
                        const uint64_t old = atomicAdd((unsigned long long*)&B.tile_count[g], (unsigned long long)one);
                        direct_check(B, old + one);
                        refs++;
                        if ((uint32_t)old < B.direct) B.refs[(size_t)g * B.direct + (uint32_t)old] = payload;
                    });
                }
                refs = wave_sum(refs);
                if (lane == 0 && refs) atomicAdd(&B.counters[kCntTileRefs + stripe], refs);
            }
        }
        __syncthreads();  // the LDS tables are rewritten by the next pass
    }
}

__global__ __launch_bounds__(kBlock) void k_bin_count(BatchParams Q, const FrameParams* __restrict__ jobs,
                                                      DeviceBuffers B) {
    constexpr uint32_t kUnroll = 4;
    extern __shared__ uint32_t hist[];
    __shared__ uint32_t sBox[4];  // min x, min y, max x, max y of the chunk's tiles
    __shared__ uint32_t sBig[kUnroll * kBlock], sBigN;  // a step's non-compact descriptors
    __shared__ uint32_t sWide[kWideCap], sWideN;         // and their wide records
    __shared__ uint32_t sScan[kBlock + kBlock / kWave];
    const FrameParams& P = jobs[job_of(Q, Q.chunk_job, blockIdx.x)];
    const uint32_t chunk = blockIdx.x - P.chunk_base;  // chunk of the job
    for (uint32_t i = threadIdx.x; i < P.num_tiles; i += kBlock) hist[i] = 0;
    if (threadIdx.x == 0) {
        sBox[0] = sBox[1] = 0xFFFFu;
        sBox[2] = sBox[3] = 0u;
        sBigN = 0;
    }
    __syncthreads();
    uint32_t bx0 = 0xFFFFu, by0 = 0xFFFFu, bx1 = 0u, by1 = 0u;  // this thread's references
    const uint32_t s0 = P.slot_base + chunk * P.chunk_slots;
    const uint32_t s1 = min(P.slot_base + P.num_triangles, s0 + P.chunk_slots);
    // Four slots per thread and step, their descriptors loaded together so
    // the loads' latencies overlap.  Compact descriptors (at most 2x2 tiles)
    // are counted by their lanes; the others are listed and enumerated by the
    // whole workgroup at the end of the step.
    const uint32_t tilesX = P.tiles_x;
    // A tile's count of heavy references rides in the high half of its
    // histogram entry while a chunk cannot reach 2^16 references per tile (at
    // most 7 records per slot); one global atomic per tile then adds it to
    // tile_big, instead of one per reference.
    const bool packBig = (uint64_t)P.chunk_slots * 7u <= 0xFFFFu;
    auto bump = [&](uint32_t tile, bool heavy) {
        if (packBig) {
            atomicAdd(&hist[tile], heavy ? 0x10001u : 1u);
        } else {
            atomicAdd(&hist[tile], 1u);
            if (heavy) atomicAdd(&B.tile_big[P.tile_base + tile], 1u);
        }
    };
    // The next step's descriptors are loaded before this step's work.
    uint32_t dn[kUnroll];
#pragma unroll
    for (uint32_t u = 0; u < kUnroll; u++) {
        const uint32_t s = s0 + threadIdx.x + u * kBlock;
        dn[u] = s < s1 ? B.desc[s] : 0u;
    }
    for (uint32_t sb = s0 + threadIdx.x; sb - threadIdx.x < s1; sb += kUnroll * kBlock) {
        uint32_t d[kUnroll];
#pragma unroll
        for (uint32_t u = 0; u < kUnroll; u++) {
            d[u] = dn[u];
            const uint32_t sn = sb + (kUnroll + u) * kBlock;
            dn[u] = sn < s1 ? B.desc[sn] : 0u;
        }
#pragma unroll
        for (uint32_t u = 0; u < kUnroll; u++) {
            if (d[u] & kDescCompact) {
                // at most 2x2 tiles, no corner tests
                const uint32_t R = compact_refs(d[u]);
                for (uint32_t k = 0; k < R; k++) bump(compact_tile(d[u], k, tilesX), (d[u] & kDescHeavy) != 0);
                const uint32_t tx = d[u] & 0x3FFFu, ty = (d[u] >> 14) & 0x3FFFu;
                bx0 = min(bx0, tx);
                by0 = min(by0, ty);
                bx1 = max(bx1, tx + ((d[u] >> 28) & 1u));
                by1 = max(by1, ty + ((d[u] >> 29) & 1u));
            } else if (d[u]) {
                sBig[atomicAdd(&sBigN, 1u)] = d[u];
            }
        }
        if (__syncthreads_or(any_non_compact(d))) {
            const uint32_t nBig = sBigN;
            __syncthreads();  // every thread has read the count
            if (threadIdx.x == 0) {
                sBigN = 0;
                sWideN = 0;
            }
            __syncthreads();
            block_enum_listed(P, B.rrec, sBig, nBig, sScan, sWide, &sWideN,
                              [&](uint32_t tile, int tx, int ty, uint32_t, bool heavy) {
                                  bump(tile, heavy);
                                  bx0 = min(bx0, (uint32_t)tx);
                                  by0 = min(by0, (uint32_t)ty);
                                  bx1 = max(bx1, (uint32_t)tx);
                                  by1 = max(by1, (uint32_t)ty);
                              });
            __syncthreads();  // the lists are rewritten by the next step
        }
    }
    // The chunk's tile box (k_bin_scatter sets up cursors only inside it).
    bx0 = wave_min(bx0);
    by0 = wave_min(by0);
    bx1 = wave_max(bx1);
    by1 = wave_max(by1);
    if (__lane_id() == 0) {
        atomicMin(&sBox[0], bx0);
        atomicMin(&sBox[1], by0);
        atomicMax(&sBox[2], bx1);
        atomicMax(&sBox[3], by1);
    }
    __syncthreads();
    const uint32_t x0 = sBox[0], y0 = sBox[1], x1 = sBox[2], y1 = sBox[3];
    if (threadIdx.x == 0) {
        B.chunk_box[2 * blockIdx.x] = x0 | (y0 << 16);
        B.chunk_box[2 * blockIdx.x + 1] = x1 | (y1 << 16);
    }
    // Only the box part of the chunk's row is written: the column scans and
    // the scatter read an entry only when its tile lies in the chunk's box.
    if (x0 <= x1 && y0 <= y1) {
        uint32_t* row = B.bin_counts + P.count_base + (size_t)chunk * P.num_tiles;
        const uint32_t bw = x1 - x0 + 1, nb = bw * (y1 - y0 + 1);
        for (uint32_t i = threadIdx.x; i < nb; i += kBlock) {
            const uint32_t t = (y0 + i / bw) * tilesX + x0 + i % bw;
            const uint32_t h = hist[t];
            row[t] = packBig ? h & 0xFFFFu : h;
            if (packBig && (h >> 16)) atomicAdd(&B.tile_big[P.tile_base + t], h >> 16);
        }
    }
}

// Each job's chunk x tile count matrix is scanned down each tile's column in
// three steps over blocks of 64 tiles x kChunkGroup chunks (lanes = tiles, each
// wave a quarter of the group's chunks), so every step has C/64 x tiles/64
// blocks per job (grid z = job; blocks beyond a smaller job's matrix exit).
namespace {
constexpr uint32_t kWaveChunks = kChunkGroup / (kBlock / kWave);  // chunks of a group per wave

// The wave's counts of one tile column (all loads issued before any use).
// Entries whose tile lies outside the chunk's tile box are zero and are not
// stored: they are neither read nor written.  Bit k of the returned mask is
// set when chunk c0 + k's entry is stored.
__device__ __forceinline__ uint32_t colgroup_load(const FrameParams& P, const DeviceBuffers& B, uint32_t tile,
                                                  uint32_t c0, uint32_t c1, uint32_t (&v)[kWaveChunks]) {
    const bool in = tile < P.num_tiles;
    const uint32_t ty = in ? tile / P.tiles_x : 0u, tx = in ? tile - ty * P.tiles_x : 0u;
    const uint32_t* box = B.chunk_box + 2 * (size_t)(P.chunk_base + __builtin_amdgcn_readfirstlane(c0));
    uint32_t mask = 0;
#pragma unroll
    for (uint32_t k = 0; k < kWaveChunks; k++) {
        bool stored = false;
        if (c0 + k < c1) {
            const uint32_t b0 = box[2 * k], b1 = box[2 * k + 1];
            stored = in && tx >= (b0 & 0xFFFFu) && tx <= (b1 & 0xFFFFu) && ty >= (b0 >> 16) && ty <= (b1 >> 16);
        }
        mask |= stored ? 1u << k : 0u;
    }
#pragma unroll
    for (uint32_t k = 0; k < kWaveChunks; k++)
        v[k] = (mask >> k) & 1u ? B.bin_counts[P.count_base + (size_t)(c0 + k) * P.num_tiles + tile] : 0u;
    return mask;
}

// Per-wave partial sums of one (64-tile, chunk-group) block, combined in LDS;
// returns this wave's exclusive base within the group and the group total.
__device__ __forceinline__ void colgroup_sums(const uint32_t (&v)[kWaveChunks], uint32_t (*part)[kWave],
                                              uint32_t& waveBase, uint32_t& groupTotal) {
    const uint32_t lane = __lane_id(), wave = threadIdx.x / kWave;
    uint32_t sum = 0;
#pragma unroll
    for (uint32_t k = 0; k < kWaveChunks; k++) sum += v[k];
    part[wave][lane] = sum;
    __syncthreads();
    waveBase = 0;
    groupTotal = 0;
    for (uint32_t w = 0; w < kBlock / kWave; w++) {
        if (w < wave) waveBase += part[w][lane];
        groupTotal += part[w][lane];
    }
}
__device__ __forceinline__ void colgroup_range(const FrameParams& P, uint32_t& c0, uint32_t& c1) {
    const uint32_t wave = threadIdx.x / kWave;
    c0 = min(P.num_chunks, blockIdx.y * kChunkGroup + wave * kWaveChunks);
    c1 = min(P.num_chunks, c0 + kWaveChunks);
}
}  // namespace

namespace {
// A wave's tiles' references and deepest tile, added to the frame's striped counters.
__device__ __forceinline__ void tile_stats_add(const DeviceBuffers& B, uint32_t n, uint32_t stripe) {
    const uint32_t sum = wave_sum(n), deep = wave_max(n);
    if (__lane_id() == 0 && sum) {
        atomicAdd(&B.counters[kCntTileRefs + stripe % kAllocStripes], sum);
        atomicMax(&B.counters[kCntTileDeepest + stripe % kAllocStripes], deep);
    }
}
}  // namespace

// Whether block (x, y) of the column-scan grid lies inside job P's matrix.
__device__ __forceinline__ bool colgroup_in_job(const FrameParams& P) {
    return blockIdx.x * kWave < P.num_tiles && blockIdx.y * kChunkGroup < P.num_chunks;
}

// Step 1: per (tile, chunk group) column sums.
__global__ __launch_bounds__(kBlock) void k_bin_colsum(BatchParams Q, const FrameParams* __restrict__ jobs,
                                                       DeviceBuffers B) {
    __shared__ uint32_t part[kBlock / kWave][kWave];
    const FrameParams& P = jobs[blockIdx.z];
    if (!colgroup_in_job(P)) return;
    const uint32_t tile = blockIdx.x * kWave + __lane_id();
    uint32_t c0, c1, waveBase, groupTotal, v[kWaveChunks];
    colgroup_range(P, c0, c1);
    colgroup_load(P, B, tile, c0, c1, v);
    colgroup_sums(v, part, waveBase, groupTotal);
    if (threadIdx.x < kWave && tile < P.num_tiles)
        B.group_sums[P.group_base + (size_t)blockIdx.y * P.num_tiles + tile] = groupTotal;
}

// Step 2: per tile, exclusive scan over the chunk groups and the tile total.
__global__ __launch_bounds__(kBlock) void k_bin_groupscan(BatchParams Q, const FrameParams* __restrict__ jobs,
                                                          DeviceBuffers B) {
    const FrameParams& P = jobs[blockIdx.z];
    const uint32_t tile = blockIdx.x * kBlock + threadIdx.x;
    const bool in = tile < P.num_tiles;
    const uint32_t G = in ? (P.num_chunks + kChunkGroup - 1) / kChunkGroup : 0u;
    uint32_t* col = &B.group_sums[P.group_base + tile];
    uint32_t run = 0;
    // Batches of 16 groups: the loads of a batch are issued before its stores.
    constexpr uint32_t kBatch = 16;
    for (uint32_t g0 = 0; g0 < G; g0 += kBatch) {
        uint32_t v[kBatch];
#pragma unroll
        for (uint32_t k = 0; k < kBatch; k++) v[k] = g0 + k < G ? col[(size_t)(g0 + k) * P.num_tiles] : 0u;
#pragma unroll
        for (uint32_t k = 0; k < kBatch; k++) {
            if (g0 + k < G) col[(size_t)(g0 + k) * P.num_tiles] = run;
            run += v[k];
        }
    }
    if (in) B.tile_totals[P.tile_base + tile] = run;
    if (Q.total_tiles > kTilescanOne) tile_stats_add(B, run, blockIdx.x);
}

// Step 3: rewrite the counts in place as offsets within the tile's list.
__global__ __launch_bounds__(kBlock) void k_bin_colscan(BatchParams Q, const FrameParams* __restrict__ jobs,
                                                        DeviceBuffers B) {
    __shared__ uint32_t part[kBlock / kWave][kWave];
    const FrameParams& P = jobs[blockIdx.z];
    if (!colgroup_in_job(P)) return;
    const uint32_t tile = blockIdx.x * kWave + __lane_id();
    uint32_t c0, c1, waveBase, groupTotal, v[kWaveChunks];
    colgroup_range(P, c0, c1);
    const uint32_t stored = colgroup_load(P, B, tile, c0, c1, v);
    colgroup_sums(v, part, waveBase, groupTotal);
    if (tile >= P.num_tiles) return;
    uint32_t run = B.group_sums[P.group_base + (size_t)blockIdx.y * P.num_tiles + tile] + waveBase;
#pragma unroll
    for (uint32_t k = 0; k < kWaveChunks; k++) {
        if ((stored >> k) & 1u) B.bin_counts[P.count_base + (size_t)(c0 + k) * P.num_tiles + tile] = run;
        run += v[k];
    }
}

// The three column-scan steps in one launch, by a decoupled look-back over
// the chunk groups of each tile column.  A workgroup sums its entries per
// tile, publishes the group sums in group_sums (value | kAggregate), adds the
// earlier groups' published values walking back to the nearest inclusive
// prefix, publishes its own inclusive prefix (value | kInclusive) and
// rewrites its entries as offsets within the tile's list; the last group
// writes the tile totals.  Each status word is written whole, so its flag and
// value are seen together.  A wait is bounded by scan_spin_limit: past it the
// frame is flagged (kOvScanWait) and run again with the three kernels; the
// workgroup still publishes, so no other workgroup waits longer on it.
namespace {
constexpr uint32_t kAggregate = 1u << 30, kInclusive = 2u << 30, kStatusValue = (1u << 30) - 1;
__device__ __forceinline__ uint32_t status_load(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void status_store(uint32_t* p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
}  // namespace

__global__ __launch_bounds__(kBlock) void k_bin_colpass(BatchParams Q, const FrameParams* __restrict__ jobs,
                                                        DeviceBuffers B) {
    __shared__ uint32_t part[kBlock / kWave][kWave];
    __shared__ uint32_t sExcl[kWave];
    // Workgroups are dispatched in linear index order, x fastest, then the
    // chunk group y: a workgroup waits only on lower indices (same job,
    // earlier groups), which have started.
    const uint32_t x = blockIdx.x, g = blockIdx.y;
    const FrameParams& P = jobs[blockIdx.z];
    if (x * kWave >= P.num_tiles) return;
    const uint32_t lane = __lane_id(), wave = threadIdx.x / kWave;
    const uint32_t tile = x * kWave + lane;
    const bool in = tile < P.num_tiles;
    const uint32_t G = (P.num_chunks + kChunkGroup - 1) / kChunkGroup;
    if (G == 0) {  // a job without triangles: its tiles are empty
        if (g == 0 && wave == 0 && in) B.tile_totals[P.tile_base + tile] = 0u;
        return;
    }
    if (g >= G) return;
    const uint32_t c0 = min(P.num_chunks, g * kChunkGroup + wave * kWaveChunks);
    const uint32_t c1 = min(P.num_chunks, c0 + kWaveChunks);
    uint32_t v[kWaveChunks], waveBase, groupTotal;
    const uint32_t stored = colgroup_load(P, B, tile, c0, c1, v);
    colgroup_sums(v, part, waveBase, groupTotal);
    if (wave == 0) {
        uint32_t excl = 0;
        if (in) {
            uint32_t* st = B.group_sums + P.group_base + tile;
            if (g > 0) {
                status_store(st + (size_t)g * P.num_tiles, kAggregate | groupTotal);
                bool failed = B.scan_spin_limit == 0;
                uint32_t spins = 0;
                // kLook predecessors are read at once, nearest first; the
                // walk takes them up to the first inclusive prefix or the
                // first one not yet published, where the next round resumes.
                constexpr uint32_t kLook = 16;
                for (uint32_t gp = g; gp > 0 && !failed;) {
                    uint32_t sv[kLook];
#pragma unroll
                    for (uint32_t k = 0; k < kLook; k++)
                        sv[k] = k < gp ? status_load(st + (size_t)(gp - 1 - k) * P.num_tiles) : kInclusive;
                    uint32_t taken = 0;
                    bool done = false;
#pragma unroll
                    for (uint32_t k = 0; k < kLook; k++) {
                        if (done || taken < k || !(sv[k] >> 30)) continue;
                        if (k < gp) excl += sv[k] & kStatusValue;
                        taken = k + 1;
                        done = (sv[k] & kInclusive) != 0;
                    }
                    if (done) break;
                    gp -= taken;
                    if (taken < kLook && gp > 0) {  // stopped at one not yet published
                        if (++spins > B.scan_spin_limit) failed = true;
                        else __builtin_amdgcn_s_sleep(1);
                    }
                }
                if (failed) atomicOr(&B.counters[kCntOverflow], (uint32_t)kOvScanWait);
            }
            // (a prefix beyond the 30-bit status value: the three kernels count in 32 bits)
            if ((uint64_t)excl + groupTotal > kStatusValue) atomicOr(&B.counters[kCntOverflow], (uint32_t)kOvScanWait);
            status_store(st + (size_t)g * P.num_tiles, kInclusive | ((excl + groupTotal) & kStatusValue));
            if (g == G - 1) B.tile_totals[P.tile_base + tile] = excl + groupTotal;
        }
        if (g == G - 1 && Q.total_tiles > kTilescanOne) tile_stats_add(B, in ? excl + groupTotal : 0u, x);
        sExcl[lane] = excl;
    }
    __syncthreads();
    if (!in) return;
    uint32_t run = sExcl[lane] + waveBase;
#pragma unroll
    for (uint32_t k = 0; k < kWaveChunks; k++) {
        if ((stored >> k) & 1u) B.bin_counts[P.count_base + (size_t)(c0 + k) * P.num_tiles + tile] = run;
        run += v[k];
    }
}

namespace {
// Exclusive scans of kN values at once over the 1024 threads of a block:
// one pair of barriers for all of them.
template <int kN>
__device__ __forceinline__ void scan1024_n(uint32_t (&v)[kN], uint32_t (*wsum)[16], uint32_t (&total)[kN]) {
    const uint32_t lane = __lane_id(), wave = threadIdx.x / kWave;
    uint32_t x[kN];
#pragma unroll
    for (int i = 0; i < kN; i++) x[i] = wave_incl_scan(v[i]);
    if (lane == kWave - 1) {
#pragma unroll
        for (int i = 0; i < kN; i++) wsum[i][wave] = x[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kN; i++) {
        uint32_t base = 0, tot = 0;
        for (uint32_t w = 0; w < 16; w++) {
            if (w < wave) base += wsum[i][w];
            tot += wsum[i][w];
        }
        total[i] = tot;
        v[i] = base + x[i] - v[i];
    }
    __syncthreads();
}

// Raster work items of a tile with n references (an empty tile has none).
__device__ __forceinline__ uint32_t tile_segments(uint32_t n, uint32_t segLog2) {
    return (n + (1u << segLog2) - 1) >> segLog2;
}
}  // namespace

namespace {
// log2 of the frame's references per work item, and whether every tile's
// segment indices then fit a work item.
__device__ __forceinline__ uint32_t frame_seg_log2(uint32_t total, uint32_t deepest, uint32_t rasterBlocks, bool& fit) {
    uint32_t segLog2 = kSegLog2Min;
    while (segLog2 < kSegLog2Max && (total >> segLog2) > rasterBlocks) segLog2++;
    // a tile's segment index must fit above the tile bits of a work item
    while (segLog2 < kSegLog2Max && tile_segments(deepest, segLog2) > (1u << kSegIndexBits)) segLog2++;
    fit = tile_segments(deepest, segLog2) <= (1u << kSegIndexBits);
    return segLog2;
}

// A tile's segment log2: the frame's, or kSegLog2Heavy for a tile whose
// references are mostly tile-level triangles (a whole wave each), so that
// such a tile is spread over several workgroups.  Finer segments never
// make a tile's segment index overflow its bits.
__device__ __forceinline__ uint32_t tile_seg_log2(uint32_t n, uint32_t big, uint32_t segLog2, bool split) {
    if (!split || big < kHeavyBigMin || 4 * big < n) return segLog2;
    uint32_t s = kSegLog2Heavy;
    while (s < segLog2 && tile_segments(n, s) > (1u << kSegIndexBits)) s++;
    return s;
}

// Adds a tile's full segments (cnt[0]) and its partial last segment by size
// class (cnt[1 + c], class c = remainder >> (the tile's segment log2 - 2)).
__device__ __forceinline__ void count_segments(uint32_t n, uint32_t s, uint32_t (&cnt)[5]) {
    cnt[0] += n >> s;
    const uint32_t r = n & ((1u << s) - 1);
    if (r) {
        // (an array index known at compile time keeps cnt in registers)
        const uint32_t c = r >> (s - 2);
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) cnt[1 + k] += c == k ? 1u : 0u;
    }
}

// The first list position of each class: full segments, then classes 3, 2, 1, 0.
__device__ __forceinline__ void class_starts(const uint32_t (&tot)[5], uint32_t (&pos)[5]) {
    pos[0] = 0;
    pos[4] = tot[0];
    pos[3] = pos[4] + tot[4];
    pos[2] = pos[3] + tot[3];
    pos[1] = pos[2] + tot[2];
}

// A tile's work items, at its classes' next positions; returns its segments.
__device__ __forceinline__ uint32_t place_tile(uint32_t* work, uint32_t t, uint32_t n, uint32_t s, uint32_t (&pos)[5]) {
    const uint32_t nf = n >> s, r = n & ((1u << s) - 1);
    const uint32_t segs = nf + (r ? 1u : 0u);
    // a tile of one segment is marked (kSingleSegment): its image is the
    // 32-bit winner orders
    const uint32_t single = segs == 1 ? kSingleSegment : 0u;
    for (uint32_t i = 0; i < nf; i++) work[pos[0]++] = t | (i << kTileBits) | single;
    if (r) {
        const uint32_t c = r >> (s - 2);
        work[c == 0 ? pos[1] : c == 1 ? pos[2] : c == 2 ? pos[3] : pos[4]] = t | (nf << kTileBits) | single;
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) pos[1 + k] += c == k ? 1u : 0u;
    }
    return segs;
}
}  // namespace

// Exclusive scan of the tile totals over every job's tiles and the raster work
// list: one item per (tile, segment of <= 2^segLog2 refs).  The segment size
// is the smallest of 256 .. 4096 that gives no more items than the raster grid
// has workgroups (beyond one per tile), so a frame with few references is
// still spread over the whole grid instead of being bound by one workgroup
// walking a deep tile.  Items are listed longest first, so that the last ones
// claimed are short and the pass does not end on one workgroup finishing a
// full segment: every full segment, then the tiles' last (partial) segments in
// four size classes, largest first.  A segment's key image is at the tile's
// image base (tile_item) plus its segment index, whatever its place in the
// list.
// One workgroup for frames of up to kTilescanOne tiles (k_bin_tilescan), kPer
// = 1, 2 or 4 tiles per thread in registers (475 tiles 5 us; 2,040 tiles at 2
// per thread 6.7, at 4 8.4 us); beyond, a workgroup per kTileBlock tiles in two launches
// (k_bin_tilesums, k_bin_tileplace), with the same outputs.
template <uint32_t kPer>
__global__ __launch_bounds__(1024) void k_bin_tilescan(BatchParams Q, DeviceBuffers B) {
    __shared__ uint32_t sScan6[6][16];
    __shared__ uint32_t sMax, sTotal, sSegs, sExtra;
    const uint32_t nt = Q.total_tiles;
    if (threadIdx.x == 0) sMax = sTotal = sSegs = sExtra = 0;
    uint32_t n[kPer], big[kPer];
#pragma unroll
    for (uint32_t u = 0; u < kPer; u++) {
        const uint32_t t = threadIdx.x * kPer + u;
        n[u] = t < nt ? B.tile_totals[t] : 0u;
        big[u] = t < nt ? B.tile_big[t] : 0u;
    }
    __syncthreads();
    uint32_t localRefs = 0, localMax = 0;
#pragma unroll
    for (uint32_t u = 0; u < kPer; u++) {
        localRefs += n[u];
        localMax = max(localMax, n[u]);
    }
    // Total and deepest tile: wave reductions, then one LDS atomic per wave.
    const uint32_t waveRefs = wave_sum(localRefs), waveMax = wave_max(localMax);
    if (__lane_id() == 0) {
        atomicAdd(&sTotal, waveRefs);
        atomicMax(&sMax, waveMax);
    }
    __syncthreads();
    const uint32_t total = sTotal;
    bool segsFit;
    const uint32_t segLog2 = frame_seg_log2(total, sMax, B.raster_blocks, segsFit);
    // The finer segments of heavy tiles are taken only while the work list
    // has room for them: segments with and without them, summed over the block.
    uint32_t segs = 0, extra = 0;
#pragma unroll
    for (uint32_t u = 0; u < kPer; u++) {
        const uint32_t plain = tile_segments(n[u], segLog2);
        segs += plain;
        extra += tile_segments(n[u], tile_seg_log2(n[u], big[u], segLog2, true)) - plain;
    }
    segs = wave_sum(segs);
    extra = wave_sum(extra);
    if (__lane_id() == 0) {
        atomicAdd(&sSegs, segs);
        atomicAdd(&sExtra, extra);
    }
    __syncthreads();
    const bool split = (uint64_t)sSegs + sExtra <= B.work_cap;
    uint32_t cnt[5] = {0, 0, 0, 0, 0}, s[kPer];
#pragma unroll
    for (uint32_t u = 0; u < kPer; u++) {
        s[u] = tile_seg_log2(n[u], big[u], segLog2, split);
        count_segments(n[u], s[u], cnt);
    }
    // the tile-reference prefix rides along as a sixth value
    uint32_t x[6] = {cnt[0], cnt[1], cnt[2], cnt[3], cnt[4], localRefs}, tot6[6];
    scan1024_n<6>(x, sScan6, tot6);
    const uint32_t tot[5] = {tot6[0], tot6[1], tot6[2], tot6[3], tot6[4]};
    const uint32_t totalSegs = tot[0] + tot[1] + tot[2] + tot[3] + tot[4];
    const bool fits = total <= B.ref_cap && totalSegs <= B.work_cap && totalSegs <= kImageMask && segsFit;
    // the thread's reference and image base: those of all earlier threads' tiles
    uint32_t run = x[5], seg = x[0] + x[1] + x[2] + x[3] + x[4], pos[5];
    class_starts(tot, pos);
#pragma unroll
    for (uint32_t c = 0; c < 5; c++) pos[c] += x[c];
#pragma unroll
    for (uint32_t u = 0; u < kPer; u++) {
        const uint32_t t = threadIdx.x * kPer + u;
        if (t >= nt) break;
        B.tile_start[t] = run;
        run += n[u];
        if (!fits) continue;
        B.tile_item[t] = seg | (s[u] << kImageBits);
        seg += place_tile(B.work, t, n[u], s[u], pos);
    }
    if (threadIdx.x == 0) {
        B.tile_start[nt] = total;
        B.counters[kCntTotalRefs] = total;
        B.counters[kCntWorkItems] = totalSegs;
        B.counters[kCntSegLog2] = segLog2;
        if (!fits) atomicOr(&B.counters[kCntOverflow], (uint32_t)kOvRefs);
    }
}

// The tile scan of more than kTilescanOne tiles.  The references' total and
// the deepest tile are summed by the column scan already (tile_stats_add), so
// the segment size is known at once: k_bin_tilesums leaves each block's sums
// (TileSums), and every block of k_bin_tileplace adds those of the blocks
// before it and of all (up to 256 blocks: one per thread) and places its own
// tiles.  Latency bounds both: a block reads 8 KB.  (As one workgroup walking
// all tiles in rounds of 8,192: 290 us for 117K tiles, 41 us for 16K, 17 us
// for 8K; the two launches take 12, 11 and 11 us.)
namespace {
struct __attribute__((aligned(16))) TileSums {
    uint32_t refs, segs, extra, pad;  // segments without, and more with, the heavy tiles' finer ones
    uint32_t plain[5], split[5], pad2[2];  // count_segments without and with them
};
static_assert(sizeof(TileSums) == 4 * kTileSumWords, "TileSums layout");
constexpr uint32_t kTilePer = kTileBlock / kBlock;
static_assert(kTilePer == 4, "a thread's tiles are one 16-byte load");
static_assert(kMaxBatchTiles / kTileBlock <= kBlock, "k_bin_tileplace takes one block's sums per thread");

__device__ __forceinline__ uint32_t tile_stats_total(const DeviceBuffers& B, uint32_t& deepest) {
    uint32_t total = 0;
    deepest = 0;
#pragma unroll
    for (uint32_t k = 0; k < kAllocStripes; k++) {
        total += B.counters[kCntTileRefs + k];
        deepest = max(deepest, B.counters[kCntTileDeepest + k]);
    }
    return total;
}

// The thread's kTilePer tiles (totals and big counts; 0 beyond the last).
__device__ __forceinline__ void load_tiles(const BatchParams& Q, const DeviceBuffers& B, uint32_t t0,
                                           uint32_t (&n)[kTilePer], uint32_t (&big)[kTilePer]) {
    if (t0 + kTilePer <= Q.total_tiles) {
        const uint4 a = *reinterpret_cast<const uint4*>(B.tile_totals + t0);
        const uint4 b = *reinterpret_cast<const uint4*>(B.tile_big + t0);
        n[0] = a.x; n[1] = a.y; n[2] = a.z; n[3] = a.w;
        big[0] = b.x; big[1] = b.y; big[2] = b.z; big[3] = b.w;
    } else {
#pragma unroll
        for (uint32_t u = 0; u < kTilePer; u++) {
            n[u] = t0 + u < Q.total_tiles ? B.tile_totals[t0 + u] : 0u;
            big[u] = t0 + u < Q.total_tiles ? B.tile_big[t0 + u] : 0u;
        }
    }
}
}  // namespace

__global__ __launch_bounds__(kBlock) void k_bin_tilesums(BatchParams Q, DeviceBuffers B) {
    __shared__ uint32_t sSum[13];
    if (threadIdx.x < 13) sSum[threadIdx.x] = 0;
    uint32_t n[kTilePer], big[kTilePer], deepest;
    load_tiles(Q, B, (blockIdx.x * kBlock + threadIdx.x) * kTilePer, n, big);
    const uint32_t total = tile_stats_total(B, deepest);
    bool segsFit;
    const uint32_t segLog2 = frame_seg_log2(total, deepest, B.raster_blocks, segsFit);
    uint32_t plain[5] = {0, 0, 0, 0, 0}, split[5] = {0, 0, 0, 0, 0}, refs = 0, segs = 0, extra = 0;
#pragma unroll
    for (uint32_t u = 0; u < kTilePer; u++) {
        const uint32_t s = tile_seg_log2(n[u], big[u], segLog2, true);
        const uint32_t p = tile_segments(n[u], segLog2);
        refs += n[u];
        segs += p;
        extra += tile_segments(n[u], s) - p;
        count_segments(n[u], segLog2, plain);
        count_segments(n[u], s, split);
    }
    const uint32_t v[13] = {refs, segs, extra, plain[0], plain[1], plain[2], plain[3], plain[4],
                            split[0], split[1], split[2], split[3], split[4]};
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 13; k++) {
        const uint32_t w = wave_sum(v[k]);
        if (__lane_id() == 0 && w) atomicAdd(&sSum[k], w);
    }
    __syncthreads();
    if (threadIdx.x < 13)  // (the struct's words, past its pad)
        B.tile_sums[blockIdx.x * kTileSumWords + threadIdx.x + (threadIdx.x >= 3 ? 1u : 0u)] = sSum[threadIdx.x];
}

__global__ __launch_bounds__(kBlock) void k_bin_tileplace(BatchParams Q, DeviceBuffers B) {
    constexpr uint32_t kWaves = kBlock / kWave;
    __shared__ uint32_t sAll[kWaves][8], sBefore[kWaves][6], sScan[kWaves][6];
    const uint32_t lane = __lane_id(), wave = threadIdx.x / kWave, nb = gridDim.x;
    const uint32_t t0 = (blockIdx.x * kBlock + threadIdx.x) * kTilePer;
    uint32_t n[kTilePer], big[kTilePer], deepest;
    load_tiles(Q, B, t0, n, big);
    TileSums sums;
    memset(&sums, 0, sizeof(sums));
    if (threadIdx.x < nb) sums = reinterpret_cast<const TileSums*>(B.tile_sums)[threadIdx.x];
    const uint32_t total = tile_stats_total(B, deepest);
    bool segsFit;
    const uint32_t segLog2 = frame_seg_log2(total, deepest, B.raster_blocks, segsFit);
    // The finer segments of heavy tiles are taken only while the work list has room for them.
    const uint32_t ws = wave_sum(sums.segs), we = wave_sum(sums.extra);
    if (lane == 0) {
        sAll[wave][5] = ws;
        sAll[wave][6] = we;
    }
    __syncthreads();
    uint64_t want = 0;
    for (uint32_t w = 0; w < kWaves; w++) want += (uint64_t)sAll[w][5] + sAll[w][6];
    const bool split = want <= B.work_cap;
    // all blocks' classes, and the classes and references of the blocks before this one
    const bool before = threadIdx.x < blockIdx.x;
#pragma unroll
    for (int c = 0; c < 5; c++) {
        const uint32_t v = split ? sums.split[c] : sums.plain[c];
        const uint32_t a = wave_sum(v), b = wave_sum(before ? v : 0u);
        if (lane == 0) {
            sAll[wave][c] = a;
            sBefore[wave][c] = b;
        }
    }
    const uint32_t rb = wave_sum(before ? sums.refs : 0u);
    if (lane == 0) sBefore[wave][5] = rb;
    // this block's own scan of the same six
    uint32_t cnt[5] = {0, 0, 0, 0, 0}, s[kTilePer], refs = 0;
#pragma unroll
    for (uint32_t u = 0; u < kTilePer; u++) {
        s[u] = tile_seg_log2(n[u], big[u], segLog2, split);
        count_segments(n[u], s[u], cnt);
        refs += n[u];
    }
    uint32_t x[6] = {cnt[0], cnt[1], cnt[2], cnt[3], cnt[4], refs};
#pragma unroll
    for (int c = 0; c < 6; c++) {
        const uint32_t incl = wave_incl_scan(x[c]);
        if (lane == kWave - 1) sScan[wave][c] = incl;
        x[c] = incl - x[c];
    }
    __syncthreads();
    uint32_t tot[5] = {0, 0, 0, 0, 0};
    for (uint32_t w = 0; w < kWaves; w++) {
#pragma unroll
        for (int c = 0; c < 6; c++) x[c] += sBefore[w][c] + (w < wave ? sScan[w][c] : 0u);
#pragma unroll
        for (int c = 0; c < 5; c++) tot[c] += sAll[w][c];
    }
    const uint32_t totalSegs = tot[0] + tot[1] + tot[2] + tot[3] + tot[4];
    const bool fits = total <= B.ref_cap && totalSegs <= B.work_cap && totalSegs <= kImageMask && segsFit;
    uint32_t run = x[5], seg = x[0] + x[1] + x[2] + x[3] + x[4], pos[5];
    class_starts(tot, pos);
#pragma unroll
    for (int c = 0; c < 5; c++) pos[c] += x[c];
#pragma unroll
    for (uint32_t u = 0; u < kTilePer; u++) {
        const uint32_t t = t0 + u;
        if (t >= Q.total_tiles) break;
        B.tile_start[t] = run;
        run += n[u];
        if (!fits) continue;
        B.tile_item[t] = seg | (s[u] << kImageBits);
        seg += place_tile(B.work, t, n[u], s[u], pos);
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        B.tile_start[Q.total_tiles] = total;
        B.counters[kCntTotalRefs] = total;
        B.counters[kCntWorkItems] = totalSegs;
        B.counters[kCntSegLog2] = segLog2;
        if (!fits) atomicOr(&B.counters[kCntOverflow], (uint32_t)kOvRefs);
    }
}

// Scatter: each reference goes to its tile's cursor, which starts at the
// tile's list offset plus the counts of the earlier chunks (k_bin_colscan), so
// a tile's list holds the chunks in submission order.  Within a chunk the
// order is that of the LDS cursor increments: the raster's depth keys carry
// the submission order, so a tile's winner does not depend on its list order.
__global__ __launch_bounds__(kBlock) void k_bin_scatter(BatchParams Q, const FrameParams* __restrict__ jobs,
                                                        DeviceBuffers B) {
    constexpr uint32_t kUnroll = 4;
    extern __shared__ uint32_t cursor[];
    __shared__ uint32_t sBig[kUnroll * kBlock], sBigN;  // a step's non-compact descriptors
    __shared__ uint32_t sWide[kWideCap], sWideN;         // and their wide records
    __shared__ uint32_t sScan[kBlock + kBlock / kWave];
    if (B.counters[kCntOverflow] & kOvNoLists) return;
    const FrameParams& P = jobs[job_of(Q, Q.chunk_job, blockIdx.x)];
    const uint32_t chunk = blockIdx.x - P.chunk_base;
    const uint32_t b0 = B.chunk_box[2 * blockIdx.x], b1 = B.chunk_box[2 * blockIdx.x + 1];
    const uint32_t x0 = b0 & 0xFFFFu, y0 = b0 >> 16, x1 = b1 & 0xFFFFu, y1 = b1 >> 16;
    if (x0 > x1 || y0 > y1) return;  // the chunk has no references
    {
        // Cursors of the tiles inside the chunk's tile box: every reference of
        // the chunk falls in it (k_bin_count).
        const uint32_t* offs = B.bin_counts + P.count_base + (size_t)chunk * P.num_tiles;
        const uint32_t bw = x1 - x0 + 1, nb = bw * (y1 - y0 + 1);
        for (uint32_t i = threadIdx.x; i < nb; i += kBlock) {
            const uint32_t t = (y0 + i / bw) * P.tiles_x + x0 + i % bw;
            cursor[t] = B.tile_start[P.tile_base + t] + offs[t];
        }
    }
    if (threadIdx.x == 0) sBigN = 0;
    __syncthreads();
    const uint32_t s0 = P.slot_base + chunk * P.chunk_slots;
    const uint32_t s1 = min(P.slot_base + P.num_triangles, s0 + P.chunk_slots);
    const uint32_t tilesX = P.tiles_x;
    // The next step's descriptors are loaded before this step's work.
    uint32_t dn[kUnroll];
#pragma unroll
    for (uint32_t u = 0; u < kUnroll; u++) {
        const uint32_t s = s0 + threadIdx.x + u * kBlock;
        dn[u] = s < s1 ? B.desc[s] : 0u;
    }
    for (uint32_t sb = s0 + threadIdx.x; sb - threadIdx.x < s1; sb += kUnroll * kBlock) {
        uint32_t d[kUnroll];
#pragma unroll
        for (uint32_t u = 0; u < kUnroll; u++) {
            d[u] = dn[u];
            const uint32_t sn = sb + (kUnroll + u) * kBlock;
            dn[u] = sn < s1 ? B.desc[sn] : 0u;
        }
#pragma unroll
        for (uint32_t u = 0; u < kUnroll; u++) {
            const uint32_t s = sb + u * kBlock;
            if (d[u] & kDescCompact) {
                const uint32_t R = compact_refs(d[u]);
                for (uint32_t k = 0; k < R; k++) B.refs[atomicAdd(&cursor[compact_tile(d[u], k, tilesX)], 1u)] = s;
            } else if (d[u]) {
                sBig[atomicAdd(&sBigN, 1u)] = d[u];
            }
        }
        // Other descriptors: listed and enumerated by the whole workgroup.
        if (__syncthreads_or(any_non_compact(d))) {
            const uint32_t nBig = sBigN;
            __syncthreads();  // every thread has read the count
            if (threadIdx.x == 0) {
                sBigN = 0;
                sWideN = 0;
            }
            __syncthreads();
            block_enum_listed(P, B.rrec, sBig, nBig, sScan, sWide, &sWideN,
                              [&](uint32_t tile, int, int, uint32_t payload, bool) {
                                  B.refs[atomicAdd(&cursor[tile], 1u)] = payload;
                              });
            __syncthreads();  // the lists are rewritten by the next step
        }
    }
}

// Persistent raster kernel: workgroups pull (tile, segment) items from the
// list built by k_bin_tilescan until it is exhausted.  The single-sample
// kernel is held to 96 VGPRs so that five workgroups per CU, as many as its LDS
// allows, are resident.  The multisample kernel's key planes take 32 KB, so that
// waves, not workgroups, are made more: two workgroups of eight waves per CU
// (2.1M sphere grid at 1080p, 4 samples: 92 us with three of four waves, so 88).
template <bool kMS>
constexpr uint32_t kRasterThreads = kMS ? 2 * kBlock : kBlock;
// References that clearing an empty tile counts as (k_raster), without and with float colours.
constexpr uint32_t kClearRefs = 16, kClearRefsFloat = 128;
template <bool kMS>
__global__ __launch_bounds__(kRasterThreads<kMS>, kMS ? 4 : 5) void k_raster(BatchParams Q, const FrameParams* __restrict__ jobs,
                                                   DeviceBuffers B) {
    __shared__ uint64_t keys[(kMS ? kPassSamples : 1) * kKeyPlane<kMS>];
    __shared__ uint16_t sOwner[kRasterThreads<kMS> / kWave][kOwnerCap];
    __shared__ WideRefs<kMS> sWide;
    __shared__ uint32_t sItem;
    // The counters are final (this kernel only draws items from kCntWorkNext):
    // the last workgroup, which in small frames has no item, copies them to
    // the host's pinned buffer, which the host reads once the stream has
    // drained.  The stores are on their way while the frame is rasterised; a
    // launch of its own after the frame took 4 us and the gap before it, and
    // a copy queued behind the frame 12 us.
    if (blockIdx.x == gridDim.x - 1)
        for (uint32_t i = threadIdx.x; i < kCntSlots; i += kRasterThreads<kMS>) B.host_counters[i] = B.counters[i];
    if (B.counters[kCntOverflow] & kOvNoLists) return;
    const uint32_t nItems = B.counters[kCntWorkItems];
    // Single-sample frames and batches: the empty tiles are cleared here (k_shade
    // skips them), by the waves of the last workgroups before these take an item,
    // while the others rasterise: the clears are bound by stores, the items by the
    // ALU.  With a share of the clears at the head of every workgroup nothing
    // overlapped: 256 jobs 630 us, so 515 (117K tiles, two thirds of them empty).
    // The clearing workgroups are the share that clearing has of the work, a tile
    // weighing as many references as below, and a tenth at least, which deep tiles
    // of many items among empty ones need.  256 jobs with a weight of 16, 32, 64:
    // 518, 538, 555 us.  With float colours, twice the bytes and few references per
    // tile (64 views at 512): 104, 106, 98 us with 32, 64, 128 (97 before).
    // A wave looks at tiles base + lane * step of each pass.  (The four waves of a
    // workgroup on one tile: a tenth of the workgroups then took 706 us for 256
    // jobs, waiting for each tile's job.)
    const uint32_t tiles = Q.total_tiles;
    const float clearing =
        (float)(tiles - min(tiles, nItems)) * (float)(B.color_f32 ? kClearRefsFloat : kClearRefs);
    const float share = clearing / (clearing + (float)B.counters[kCntTotalRefs] + 1.0f);
    const uint32_t clearers =
        min(gridDim.x, max(gridDim.x / 10, (uint32_t)((float)gridDim.x * share)) + 1);
    if (!kMS && blockIdx.x + clearers >= gridDim.x) {
        constexpr uint32_t kWaves = kRasterThreads<kMS> / kWave;
        const uint32_t step = clearers * kWaves;
        for (uint32_t base = __builtin_amdgcn_readfirstlane((gridDim.x - 1 - blockIdx.x) * kWaves + threadIdx.x / kWave);
             base < tiles; base += step * kWave) {
            const uint32_t t = base + __lane_id() * step;
            const bool empty = t < tiles && B.tile_start[t + 1] == B.tile_start[t];
            uint64_t m = __ballot(empty);
            while (m) {
                const uint32_t l = (uint32_t)__ffsll((unsigned long long)m) - 1;
                m &= m - 1;
                clear_tile<kWave>(Q, jobs, B, base + l * step, __lane_id());
            }
        }
    }
    // The first item is the workgroup's index (no burst of same-address
    // atomics at launch); later ones come from the shared counter.
    for (uint32_t round = 0;; round++) {
        if (threadIdx.x == 0) sItem = round ? gridDim.x + atomicAdd(&B.counters[kCntWorkNext], 1u) : blockIdx.x;
        __syncthreads();
        const uint32_t item = __builtin_amdgcn_readfirstlane(sItem);
        if (item >= nItems) break;
        raster_item<kMS, kRasterThreads<kMS>>(Q, jobs, B, item, keys, sOwner, &sWide);
        __syncthreads();
    }
}

// Deferred shading, one pixel per thread: the winner is the minimum (depth,
// order) key over the tile's segments (the sequential d <= D test is an
// associative minimum), then perspective-correct interpolation, the pixel
// shader and one write of colour, depth and triangle ID
// (Core/Renderer.cpp:272-350).
namespace {
// Minimum key of sample s over the tile's segment images (S samples per image).
__device__ __forceinline__ uint64_t tile_key(const uint64_t* g, uint32_t nseg, uint32_t S, uint32_t s) {
    constexpr uint32_t kPix = kTileSize * kTileSize;
    uint64_t key = g[(size_t)s * kPix];
    uint32_t k = 1;
    for (; k + 4 <= nseg; k += 4) {  // four independent loads in flight
        const uint64_t a = g[((size_t)k * S + s) * kPix], b = g[((size_t)(k + 1) * S + s) * kPix];
        const uint64_t c = g[((size_t)(k + 2) * S + s) * kPix], e = g[((size_t)(k + 3) * S + s) * kPix];
        const uint64_t ab = a < b ? a : b, ce = c < e ? c : e;
        const uint64_t m = ab < ce ? ab : ce;
        key = m < key ? m : key;
    }
    for (; k < nseg; k++) {
        const uint64_t v = g[((size_t)k * S + s) * kPix];
        key = v < key ? v : key;
    }
    return key;
}
}  // namespace

// Low word of the winner's key of a pixel (number pix of the tile) of a
// single-sample frame's nonempty tile.
__device__ __forceinline__ uint32_t tile_low(const DeviceBuffers& B, uint32_t tileItem, uint32_t n, uint32_t pix) {
    constexpr uint32_t kPix = kTileSize * kTileSize;
    const uint32_t nseg = tile_segments(n, tileItem >> kImageBits);
    const uint64_t* g = B.partials + (size_t)(tileItem & kImageMask) * kPix;
    // A single-segment tile's image holds 32-bit low words (k_raster).
    if (nseg == 1) return reinterpret_cast<const uint32_t*>(g)[pix];
    const uint64_t key = tile_key(g + pix, nseg, 1, 0);
    return key == bg_key() ? 0xFFFFFFFFu : (uint32_t)key;
}
// That pixel's colour, depth and ID.
template <bool kTex>
__device__ __forceinline__ void shade_pixel_of(const FrameParams& P, const DeviceBuffers& B, uint32_t gtile, uint32_t n,
                                               uint32_t pix, uint32_t low) {
    const uint32_t tile = gtile - P.tile_base;
    const int x = (int)(tile % P.tiles_x) * kTileSize + (int)(pix & 31u);
    const int y = (int)(tile / P.tiles_x) * kTileSize + (int)(pix >> 5);
    if (x >= (int)P.width || y >= (int)P.height) return;
    shade_winner<kTex>(P, B, x, y, P.pix_base + (size_t)(P.height - 1 - y) * P.width + x, low,
                       n >= kShadeRecomputeRefs);
}

// Single-sample frames of up to kShadeListTiles tiles, and larger ones of one job
// with an anisotropic filter: two workgroups per tile, 16 rows each (smaller
// workgroups than one per tile schedule better and cost less where the tile is
// empty, cleared by k_raster).
template <bool kTex>
__device__ __forceinline__ void shade_tiles(const BatchParams& Q, const FrameParams* __restrict__ jobs,
                                            const DeviceBuffers& B) {
    if (B.counters[kCntOverflow] & kOvNoLists) return;
    const uint32_t gtile = blockIdx.x >> 1;
    const uint32_t n = B.tile_start[gtile + 1] - B.tile_start[gtile];
    if (n == 0) return;
    const uint32_t pix = threadIdx.x + (blockIdx.x & 1u) * kShadeThreads;
    shade_pixel_of<kTex>(jobs[job_of(Q, Q.tile_job, gtile)], B, gtile, n, pix, tile_low(B, B.tile_item[gtile], n, pix));
}

// More tiles (batches): the grid's waves take the tiles of the work list (a tile's
// item of segment 0 stands for it) in turn, kShadePairs of a tile's 16 row pairs
// at a time, so that no wave is started for an empty tile.  Of the 1.9M waves of two
// workgroups per tile for 256 jobs three quarters only found their tile empty: 577
// us, with a row pair at a time 416, now 404 after a raster that then took 630 us
// and 450 and 404 after the present one (64 views 126, 78 and 72).  Each step waits
// on the chain item -> tile -> job -> key image before the gathers: the next item is
// loaded ahead (409 and 404 us), and four row pairs share a chain (1, 2, 4, 8: 448,
// 416, 408, 407 us, 64 views 78, 74, 72, 81).  The next pair's key words loaded ahead
// as well cost more than they hid (408 us).
// Calls with two workgroups per tile and so: 64 spheres at 512^2 (a third of the
// tiles covered) 419 and 334 us textured, 868 and 625 anisotropic; 9 covered jobs at
// 1024^2 380 and 365, 478 and 454, 795 and 808; 17 at 1080p 923 and 933.  One frame of
// 16,384 tiles: sphere 331 and 324, covered heightfield of 2M triangles 539 and 536,
// trilinear 743 and 740, but 1,467 and 1,710 at 8:1 (a pixel's taps are then the
// work, and a wave's four row pairs end the pass); of 9,216 444 and 445; of 8,448 190
// and 193.
constexpr uint32_t kShadePairs = 4;
template <bool kTex>
__device__ __forceinline__ void shade_list(const BatchParams& Q, const FrameParams* __restrict__ jobs,
                                           const DeviceBuffers& B) {
    constexpr uint32_t kUnits = kTileSize * kTileSize / kWave / kShadePairs;
    if (B.counters[kCntOverflow] & kOvNoLists) return;
    const uint32_t waves = gridDim.x * (kShadeThreads / kWave);
    const uint32_t units = B.counters[kCntWorkItems] * kUnits;
    uint32_t u = __builtin_amdgcn_readfirstlane(blockIdx.x * (kShadeThreads / kWave) + threadIdx.x / kWave);
    uint32_t nextItem = u < units ? B.work[u / kUnits] : 0u;
    for (; u < units; u += waves) {
        const uint32_t item = __builtin_amdgcn_readfirstlane(nextItem);
        if (u + waves < units) nextItem = B.work[(u + waves) / kUnits];
        if ((item >> kTileBits) & ((1u << kSegIndexBits) - 1)) continue;  // a further segment
        const uint32_t gtile = item & (kMaxBatchTiles - 1);
        const uint32_t n = B.tile_start[gtile + 1] - B.tile_start[gtile], tileItem = B.tile_item[gtile];
        const FrameParams& P = jobs[job_of(Q, Q.tile_job, gtile)];
        uint32_t pix = (u % kUnits) * kShadePairs * kWave + __lane_id();
#pragma unroll 1
        for (uint32_t k = 0; k < kShadePairs; k++, pix += kWave)
            shade_pixel_of<kTex>(P, B, gtile, n, pix, tile_low(B, tileItem, n, pix));
    }
}

// Multisampled frames: two workgroups per tile, 16 rows each.
template <bool kTex>
__device__ __forceinline__ void shade_samples(const BatchParams& Q, const FrameParams* __restrict__ jobs,
                                              const DeviceBuffers& B) {
    constexpr uint32_t kPix = kTileSize * kTileSize;
    if (B.counters[kCntOverflow] & kOvNoLists) return;
    const uint32_t gtile = blockIdx.x >> 1;
    const uint32_t pix = threadIdx.x + (blockIdx.x & 1u) * kShadeThreads;  // pixel of the tile
    const uint32_t start = B.tile_start[gtile];
    const uint32_t n = B.tile_start[gtile + 1] - start;
    const FrameParams& P = jobs[job_of(Q, Q.tile_job, gtile)];
    const uint32_t tile = gtile - P.tile_base;
    const int x = (int)(tile % P.tiles_x) * kTileSize + (int)(pix & 31u);
    const int y = (int)(tile / P.tiles_x) * kTileSize + (int)(pix >> 5);
    if (x >= (int)P.width || y >= (int)P.height) return;
    const uint32_t tileItem = B.tile_item[gtile];
    const uint32_t nseg = tile_segments(n, tileItem >> kImageBits), S = P.samples;
    const uint64_t* g = B.partials + (size_t)(tileItem & kImageMask) * S * kPix + pix;
    const size_t o = P.pix_base + (size_t)(P.height - 1 - y) * P.width + x;
    // Multisampling: per-sample winners and depths (the sequential LEQUAL test
    // per sample, Core/FrameBuffer.cpp:54-68); a winner is shaded once at the
    // pixel centre (Core/Rasterizer.h:270-285, Core/Renderer.cpp:305-350); the
    // resolve averages the samples' colours (Core/FrameBuffer.cpp:70-87) as
    // Color(b) = b / 255 per channel, summed in sample order, times 1 / S, then
    // FromFloats.
    const size_t plane = (size_t)P.width * P.height;
    const int cx = x * 16 + 8, cy = y * 16 + 8;
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    // The last winner's record and colour are kept: neighbouring samples
    // mostly share their winner.
    uint32_t cachedOrder = 0xFFFFFFFFu, cachedColor = 0u;
    RTri t;
    for (uint32_t s = 0; s < S; s++) {
        const uint64_t key = n ? tile_key(g, nseg, S, s) : bg_key();
        uint32_t rgba = 0u;
        if (key == bg_key()) {
            B.depth[o + s * plane] = 1.0f;
            B.ids[o + s * plane] = 0xFFFFFFFFu;
        } else {
            const uint32_t order = 0xFFFFFFFEu - (uint32_t)key;
            float l0, l1, d;
            if (order != cachedOrder) {
                ShadeVert v0, v1, v2;
                winner_tri(P, B, order, false, t, v0, v1, v2);
                bary_depth(t, cx, cy, l0, l1, d);
                const float3 c = shade_any<kTex>(P, t, order, x, y, l0, l1, v0, v1, v2);
                cachedColor = to_byte(c.x) | (to_byte(c.y) << 8) | (to_byte(c.z) << 16) | (255u << 24);
                cachedOrder = order;
            }
            const int2 off = c_sample_offsets[P.sample_level][s];
            bary_depth(t, cx + off.x, cy + off.y, l0, l1, d);
            B.depth[o + s * plane] = d;
            B.ids[o + s * plane] = (order >> 4) - P.slot_base;
            rgba = cachedColor;
        }
        // (byte / 255, from the rounded 1 / 255)
        for (int ch = 0; ch < 4; ch++)
            acc[ch] += quotient_normal((float)((rgba >> (8 * ch)) & 255u), 255.0f, 1.0f / 255.0f);
    }
    const float invS = 1.0f / (float)S;
    B.color[o] = to_byte(acc[0] * invS) | (to_byte(acc[1] * invS) << 8) | (to_byte(acc[2] * invS) << 16) |
                 (to_byte(acc[3] * invS) << 24);
    if (B.color_f32) {
        B.color_f32[3 * o] = clamp01(acc[0] * invS);
        B.color_f32[3 * o + 1] = clamp01(acc[1] * invS);
        B.color_f32[3 * o + 2] = clamp01(acc[2] * invS);
    }
}

// Untextured launches are held to 64 VGPRs, so that eight waves per SIMD are
// resident; the texture samplers need more.
enum ShadeMode { kShadeTiles, kShadeList, kShadeSamples };
template <bool kTex, ShadeMode kMode>
__device__ __forceinline__ void shade_any_mode(const BatchParams& Q, const FrameParams* __restrict__ jobs,
                                               const DeviceBuffers& B) {
    if (kMode == kShadeTiles) shade_tiles<kTex>(Q, jobs, B);
    else if (kMode == kShadeList) shade_list<kTex>(Q, jobs, B);
    else shade_samples<kTex>(Q, jobs, B);
}
template <ShadeMode kMode>
__global__ __launch_bounds__(kShadeThreads) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_shade(
    BatchParams Q, const FrameParams* __restrict__ jobs, DeviceBuffers B) {
    shade_any_mode<false, kMode>(Q, jobs, B);
}
template <ShadeMode kMode>
__global__ __launch_bounds__(kShadeThreads) void k_shade_tex(BatchParams Q, const FrameParams* __restrict__ jobs,
                                                             DeviceBuffers B) {
    shade_any_mode<true, kMode>(Q, jobs, B);
}

// ---------------------------------------------------------------------------
// Host launchers
// ---------------------------------------------------------------------------
namespace {
int g_rasterResident[2] = {0, 0};  // resident k_raster workgroups per CU: single-sample, multisample
}

hipError_t init_kernels() {
    // Bin cursors for up to kMaxTiles tiles live in LDS (160 KB per CU on gfx950).
    const int maxDyn = (int)(sizeof(uint32_t) * kMaxTiles);
    hipError_t e = hipFuncSetAttribute((const void*)k_bin_count, hipFuncAttributeMaxDynamicSharedMemorySize, maxDyn);
    if (e == hipSuccess)
        e = hipFuncSetAttribute((const void*)k_bin_scatter, hipFuncAttributeMaxDynamicSharedMemorySize, maxDyn);
    if (e == hipSuccess) e = init_direct_kernels();
    if (e == hipSuccess)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&g_rasterResident[0],
                                                         reinterpret_cast<const void*>(&k_raster<false>), kBlock, 0);
    if (e == hipSuccess)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&g_rasterResident[1],
                                                         reinterpret_cast<const void*>(&k_raster<true>),
                                                         kRasterThreads<true>, 0);
    return e;
}

uint32_t raster_resident_per_cu(bool multisample) {
    return (uint32_t)std::max(1, g_rasterResident[multisample ? 1 : 0]);
}

namespace {
std::mutex g_scratchLock;
uint8_t* g_scratch[kMaxScratchDevices] = {};  // device address of each device's scratch copy
}  // namespace

hipError_t scratch_address(uint8_t** out) {
    *out = nullptr;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxScratchDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratchLock);
    if (!g_scratch[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        g_scratch[dev] = static_cast<uint8_t*>(p);
    }
    *out = g_scratch[dev];
    return hipSuccess;
}

hipError_t set_frame_job(hipGraphExec_t exec, hipGraphNode_t first, const BatchParams& Q, FrameParams* jobs,
                         const DeviceBuffers& B, const FrameParams& job0) {
    // the arguments of launch_frame's first launch, in its order
    BatchParams q = Q;
    FrameParams* table = jobs;
    ShadeVert* verts = B.verts;
    ScreenVert* sverts = B.sverts;
    uint32_t* counters = B.counters;
    FrameParams job = job0;
    int writeJob = 1;
    hipKernelNodeParams p{};
    p.sharedMemBytes = 0;
    p.extra = nullptr;
    if (Q.vert_blocks) {
        void* args[] = {&q, &table, &verts, &sverts, &counters, &table, &job};
        p.func = reinterpret_cast<void*>(&k_vertex<true>);
        p.gridDim = dim3(Q.vert_blocks);
        p.blockDim = dim3(kBlock);
        p.kernelParams = args;
        return hipGraphExecKernelNodeSetParams(exec, first, &p);
    }
    void* args[] = {&counters, &table, &job, &writeJob};
    p.func = reinterpret_cast<void*>(&k_reset);
    p.gridDim = dim3(1);
    p.blockDim = dim3(64);
    p.kernelParams = args;
    return hipGraphExecKernelNodeSetParams(exec, first, &p);
}

hipError_t launch_frame(const BatchParams& Q, FrameParams* jobs, const FrameParams* job0, const DeviceBuffers& B,
                        hipStream_t s, hipEvent_t* events) {
    const size_t lds = sizeof(uint32_t) * Q.max_job_tiles;
    auto mark = [&](int i) {
        if (events) (void)hipEventRecord(events[i], s);
    };
    const FrameParams none{};
    // One workgroup per CU at most (its occupancy): the queue's length is
    // known only on the device, and each workgroup loops over it.
    const uint32_t clipBlocks = max(1u, min(B.num_cus, (B.clip_queue_cap + kClipWaves - 1) / kClipWaves));
    mark(0);
    if (Q.num_jobs > 1) hipLaunchKernelGGL(k_job_tables, dim3(Q.num_jobs), dim3(kBlock), 0, s, Q, jobs);
    if (B.direct) {
        launch_front(Q, jobs, job0, B, s);
        hipLaunchKernelGGL(k_clip<true>, dim3(clipBlocks), dim3(kClipWaves * 64), 0, s, Q, jobs, B);
        for (int i = 1; i < kNumStages; i++) mark(i);
        launch_tile(Q, jobs, B, s);
        mark(kNumStages);
        return hipGetLastError();
    }
    if (!Q.vert_blocks)
        hipLaunchKernelGGL(k_reset, dim3(1), dim3(64), 0, s, B.counters, jobs, job0 ? *job0 : none, job0 ? 1 : 0);
    else if (job0)
        hipLaunchKernelGGL(k_vertex<true>, dim3(Q.vert_blocks), dim3(kBlock), 0, s, Q, jobs, B.verts, B.sverts,
                           B.counters, jobs, *job0);
    else
        hipLaunchKernelGGL(k_vertex<false>, dim3(Q.vert_blocks), dim3(kBlock), 0, s, Q, jobs, B.verts, B.sverts,
                           B.counters, jobs, none);
    if (Q.slot_blocks) {
        hipLaunchKernelGGL(k_setup, dim3((Q.slot_blocks + kSetupSlots - 1) / kSetupSlots), dim3(kBlock), 0, s, Q,
                           jobs, B);
        hipLaunchKernelGGL(k_clip<false>, dim3(clipBlocks), dim3(kClipWaves * 64), 0, s, Q, jobs, B);
    }
    mark(1);
    if (Q.total_chunks) hipLaunchKernelGGL(k_bin_count, dim3(Q.total_chunks), dim3(kBlock), lds, s, Q, jobs, B);
    mark(2);
    const dim3 colGrid((Q.max_job_tiles + kWave - 1) / kWave, (Q.max_job_chunks + kChunkGroup - 1) / kChunkGroup,
                       Q.num_jobs);
    if (B.legacy_scans) {
        // The group scan also writes the tile totals of jobs without triangles.
        if (Q.total_chunks) hipLaunchKernelGGL(k_bin_colsum, colGrid, dim3(kBlock), 0, s, Q, jobs, B);
        hipLaunchKernelGGL(k_bin_groupscan, dim3((Q.max_job_tiles + kBlock - 1) / kBlock, 1, Q.num_jobs),
                           dim3(kBlock), 0, s, Q, jobs, B);
        if (Q.total_chunks) hipLaunchKernelGGL(k_bin_colscan, colGrid, dim3(kBlock), 0, s, Q, jobs, B);
    } else {
        // (also writes the tile totals of jobs without triangles: a grid of
        // one chunk group at least)
        const dim3 passGrid(colGrid.x, max(1u, colGrid.y), colGrid.z);
        hipLaunchKernelGGL(k_bin_colpass, passGrid, dim3(kBlock), 0, s, Q, jobs, B);
    }
    if (Q.total_tiles <= kTilescanOne) {
        if (Q.total_tiles <= 1024) hipLaunchKernelGGL(k_bin_tilescan<1>, dim3(1), dim3(1024), 0, s, Q, B);
        else if (Q.total_tiles <= 2048) hipLaunchKernelGGL(k_bin_tilescan<2>, dim3(1), dim3(1024), 0, s, Q, B);
        else hipLaunchKernelGGL(k_bin_tilescan<4>, dim3(1), dim3(1024), 0, s, Q, B);
    } else {
        const dim3 blocks((Q.total_tiles + kTileBlock - 1) / kTileBlock);
        hipLaunchKernelGGL(k_bin_tilesums, blocks, dim3(kBlock), 0, s, Q, B);
        hipLaunchKernelGGL(k_bin_tileplace, blocks, dim3(kBlock), 0, s, Q, B);
    }
    mark(3);
    if (Q.total_chunks) hipLaunchKernelGGL(k_bin_scatter, dim3(Q.total_chunks), dim3(kBlock), lds, s, Q, jobs, B);
    mark(4);
    if (Q.max_samples > 1) hipLaunchKernelGGL((k_raster<true>), dim3(B.raster_grid), dim3(kRasterThreads<true>), 0, s, Q, jobs, B);
    else hipLaunchKernelGGL((k_raster<false>), dim3(B.raster_grid), dim3(kBlock), 0, s, Q, jobs, B);
    const dim3 shadeThreads(kShadeThreads);
    auto shade = [&](auto plain, auto textured, dim3 grid) {
        if (Q.any_textured) hipLaunchKernelGGL(textured, grid, shadeThreads, 0, s, Q, jobs, B);
        else hipLaunchKernelGGL(plain, grid, shadeThreads, 0, s, Q, jobs, B);
    };
    if (Q.max_samples > 1) shade(k_shade<kShadeSamples>, k_shade_tex<kShadeSamples>, dim3(2 * Q.total_tiles));
    else if (Q.total_tiles > kShadeListTiles && (Q.num_jobs > 1 || !Q.any_aniso))
        shade(k_shade<kShadeList>, k_shade_tex<kShadeList>, dim3(kShadeGroups * B.num_cus));
    else shade(k_shade<kShadeTiles>, k_shade_tex<kShadeTiles>, dim3(2 * Q.total_tiles));
    mark(5);
    return hipGetLastError();
}

}  // namespace edxr
