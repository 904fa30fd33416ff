// direct.hip -- direct frames: small single-sample frames and batches in three
// launches (k_front, k_clip, k_tile) instead of the general path's nine.
#include <hip/hip_runtime.h>

#include "device.h"

namespace edxr {

namespace {
constexpr uint32_t kTileThreads = 512;  // k_tile's workgroup
// Frames of at most this many tiles give a tile two workgroups of 16 rows: where
// few tiles leave most of the chip idle, a tile's own chain of walks and gathers is
// k_tile's time.  One and two workgroups: 80 tiles (heightfield at 320x200) 21.4 and
// 17.4 us, 300 (heightfield, sphere at 640x480) 17.9 and 14.2, 15.5 and 13.2, 475
// (grid, heightfield at 800x600) 30.9 and 24.1, 19.6 and 16.8, 12 jobs at 256^2 17.8
// and 13.5; 704 (heightfield, textured at 1000x700) 20.3 and 21.0, 43.5 and 44.4;
// 2,040 (textured at 1080p) 84 and 88: each workgroup sets up all of the tile's
// references.  (One workgroup of 1,024 threads: 21.4 and 17.1 us for 80 tiles, but
// 19.6 and 23.6 for the 475 of the heightfield.)
constexpr uint32_t kTileHalves = 512;
}  // namespace

// ---------------------------------------------------------------------------
// Direct frames: small single-sample frames and batches (launch rule:
// direct_frame in api.cpp) in three launches instead of nine.  Each of those
// nine takes 3 to 7 us of little work and the gap before it, which bounds a
// small frame.  A tile's references need no order (the keys carry the
// submission order), so its list has a fixed place of B.direct entries and
// grows by atomic additions to its count word: no count, scan and scatter
// passes, and no work list, since one workgroup takes a tile.
// 98K-triangle heightfield at 1283x719: the general path's kernels took 69 us
// in all (17 of them k_raster, 11 k_shade), these 39 (front 11, clip 3, tile
// 21); a call 78 and 48 us.  k_tile with 256 threads instead of 512: 32 us,
// its deepest tiles (1,200 references) end the pass.
// Between frames the count words and the counters of direct frames are zero:
// k_tile's workgroups clear what they have read.
// ---------------------------------------------------------------------------
// The first slot_blocks workgroups take 256 triangle slots each: k_setup's work
// on vertices transformed on the spot (the vertex pass runs in the same
// launch; the arithmetic is the same), then the references: counted per tile in
// LDS, one addition to a tile's count word per workgroup, which also gives
// their places.  The others take 256 vertices each, as k_vertex.
template <bool kArgJob>
__global__ __launch_bounds__(kBlock) void k_front(BatchParams Q, const FrameParams* __restrict__ jobs, DeviceBuffers B,
                                                  FrameParams* jobTable, FrameParams job0) {
    extern __shared__ uint32_t hist[];  // per tile of the job: references | heavy ones << 16, then the next place
    __shared__ uint32_t sBox[4], sBig[kBlock], sBigN, sWide[kWideCap], sWideN, sScan[kBlock + kBlock / kWave];
    __shared__ uint32_t sCount[4], sQueueBase;  // rejected, bad, unclipped, queued
    if (kArgJob && blockIdx.x == 0 && threadIdx.x == 0) jobTable[0] = job0;
    if (blockIdx.x >= Q.slot_blocks) {
        const uint32_t block = blockIdx.x - Q.slot_blocks;
        vertex_slot(kArgJob ? job0 : jobs[job_of(Q, Q.vblock_job, block)], block * kBlock + threadIdx.x, B.verts,
                    B.sverts);
        return;
    }
    const FrameParams& P = kArgJob ? job0 : jobs[job_of(Q, Q.sblock_job, blockIdx.x)];
    const MeshPtrs& M = P.mesh;
    const uint32_t slot = blockIdx.x * kBlock + threadIdx.x, t = slot - P.slot_base;
    const bool valid = t < P.num_triangles;
    uint32_t i0 = 0, i1 = 0, i2 = 0;
    if (valid) {
        i0 = global_at(M.idx, 3 * (size_t)t);
        i1 = global_at(M.idx, 3 * (size_t)t + 1);
        i2 = global_at(M.idx, 3 * (size_t)t + 2);
    }
    for (uint32_t i = threadIdx.x; i < P.num_tiles; i += kBlock) hist[i] = 0;
    if (threadIdx.x < 4) {
        sBox[threadIdx.x] = threadIdx.x < 2 ? 0xFFFFu : 0u;
        sCount[threadIdx.x] = 0;
    }
    if (threadIdx.x == 0) sBigN = sWideN = 0;
    const bool bad = valid && (i0 >= P.num_vertices || i1 >= P.num_vertices || i2 >= P.num_vertices ||
                               (P.shader == kTexturedLambert && global_at(M.tex, t) >= P.num_tex));
    bool rejected = false, queued = false, main = false;
    uint32_t desc = 0;
    if (valid && !bad) {
        auto clip_pos = [&](uint32_t v) {
            return xform4(P.mvp, global_at(M.px, v), global_at(M.py, v), global_at(M.pz, v), 1.0f);
        };
        const ScreenVert a = screen_vert(P, clip_pos(i0)), b = screen_vert(P, clip_pos(i1)),
                         c = screen_vert(P, clip_pos(i2));
        if (a.code | b.code | c.code) {
            rejected = (a.code & b.code & c.code) != 0;
            queued = !rejected;
        } else {
            RasterRec rec;
            main = setup_snapped(a.x, a.y, b.x, b.y, c.x, c.y, rec);
            if (main) {
                desc = compact_desc(P, rec, slot);
                if (!(desc & kDescCompact)) {
                    rec.z0 = a.z;
                    rec.z1 = b.z;
                    rec.z2 = c.z;
                    rec.order = make_order(slot, 0, false);
                    B.rrec[slot] = rec;
                }
            }
        }
    }
    if (valid) B.desc[slot] = desc;
    __syncthreads();
    // ---- statistics and the clip queue ----
    const uint64_t qmask = __ballot(queued);
    uint32_t qAt = 0;
    {
        const uint32_t nrej = wave_count(rejected), nbad = wave_count(bad), nmain = wave_count(main);
        if (__lane_id() == 0) {
            if (nrej) atomicAdd(&sCount[0], nrej);
            if (nbad) atomicAdd(&sCount[1], nbad);
            if (nmain) atomicAdd(&sCount[2], nmain);
            if (qmask) qAt = atomicAdd(&sCount[3], (uint32_t)__popcll(qmask));
        }
        qAt = __builtin_amdgcn_readfirstlane(qAt);
    }
    // ---- references per tile ----
    uint32_t bx0 = 0xFFFFu, by0 = 0xFFFFu, bx1 = 0u, by1 = 0u;
    const bool compact = (desc & kDescCompact) != 0;
    if (compact) {
        const uint32_t R = compact_refs(desc);
        for (uint32_t k = 0; k < R; k++)
            atomicAdd(&hist[compact_tile(desc, k, P.tiles_x)], desc & kDescHeavy ? 0x10001u : 1u);
        bx0 = desc & 0x3FFFu;
        by0 = (desc >> 14) & 0x3FFFu;
        bx1 = bx0 + ((desc >> 28) & 1u);
        by1 = by0 + ((desc >> 29) & 1u);
    } else if (desc) {
        sBig[atomicAdd(&sBigN, 1u)] = desc;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t stripe = blockIdx.x & (kStripes - 1);
        if (sCount[0]) atomicAdd(&B.counters[kCntStriped + kStRejected * kStripes + stripe], sCount[0]);
        if (sCount[1]) atomicAdd(&B.counters[kCntBadIndex], sCount[1]);
        if (sCount[2]) atomicAdd(&B.counters[kCntStriped + kStMainRecords * kStripes + stripe], sCount[2]);
        sQueueBase = sCount[3] ? atomicAdd(&B.counters[kCntClipQueue], sCount[3]) : 0u;
    }
    const uint32_t nBig = sBigN;
    if (nBig)
        block_enum_listed(P, B.rrec, sBig, nBig, sScan, sWide, &sWideN,
                          [&](uint32_t tile, int tx, int ty, uint32_t, bool heavy) {
                              atomicAdd(&hist[tile], heavy ? 0x10001u : 1u);
                              bx0 = min(bx0, (uint32_t)tx);
                              by0 = min(by0, (uint32_t)ty);
                              bx1 = max(bx1, (uint32_t)tx);
                              by1 = max(by1, (uint32_t)ty);
                          });
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
    if (threadIdx.x == 0) sWideN = 0;
    if (queued) {
        const uint32_t at = sQueueBase + qAt + (uint32_t)__popcll(qmask & lanemask_lt());
        if (at < B.clip_queue_cap) B.clip_queue[at] = slot;
        else atomicOr(&B.counters[kCntOverflow], (uint32_t)kOvClipQueue);
    }
    const uint32_t x0 = sBox[0], y0 = sBox[1], x1 = sBox[2], y1 = sBox[3];
    if (x0 > x1 || y0 > y1) return;  // no references
    // ---- their places: the tiles' count words before this workgroup's additions ----
    const uint32_t bw = x1 - x0 + 1, nb = bw * (y1 - y0 + 1);
    uint32_t refs = 0;
    for (uint32_t i = threadIdx.x; i < nb; i += kBlock) {
        const uint32_t tile = (y0 + i / bw) * P.tiles_x + x0 + i % bw, h = hist[tile];
        if (!h) continue;
        refs += h & 0xFFFFu;
        const uint64_t add = (uint64_t)(h >> 16) << 32 | (h & 0xFFFFu);
        const uint64_t old = atomicAdd((unsigned long long*)&B.tile_count[P.tile_base + tile], (unsigned long long)add);
        direct_check(B, old + add);
        hist[tile] = (uint32_t)old;
    }
    refs = wave_sum(refs);
    if (__lane_id() == 0 && refs) atomicAdd(&B.counters[kCntTileRefs + blockIdx.x % kAllocStripes], refs);
    __syncthreads();
    auto place = [&](uint32_t tile, uint32_t payload) {
        const uint32_t at = atomicAdd(&hist[tile], 1u);
        if (at < B.direct) B.refs[(size_t)(P.tile_base + tile) * B.direct + at] = payload;
    };
    if (compact) {
        const uint32_t R = compact_refs(desc);
        for (uint32_t k = 0; k < R; k++) place(compact_tile(desc, k, P.tiles_x), slot);
    }
    if (nBig)
        block_enum_listed(P, B.rrec, sBig, nBig, sScan, sWide, &sWideN,
                          [&](uint32_t tile, int, int, uint32_t payload, bool) { place(tile, payload); });
}

// One workgroup per tile, or two of 16 rows each (kHalves): rasterises its list
// and shades the winners from the keys in LDS.
template <bool kTex, bool kHalves>
__global__ __launch_bounds__(kTileThreads, kTex ? 4 : 6) void k_tile(BatchParams Q, const FrameParams* __restrict__ jobs,
                                                               DeviceBuffers B) {
    __shared__ uint64_t keys[kKeyPlane<false>];
    __shared__ uint16_t sOwner[kTileThreads / kWave][kOwnerCap];
    __shared__ uint32_t sCount;
    // The counters are final: to the host's pinned buffer, and zero for the next frame.
    if (blockIdx.x == gridDim.x - 1) {
        for (uint32_t i = threadIdx.x; i < kCntSlots; i += kTileThreads) {
            B.host_counters[i] = B.counters[i];
            __hip_atomic_store(&B.counters[i], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    const uint32_t gtile = kHalves ? blockIdx.x >> 1 : blockIdx.x;
    const int row0 = kHalves ? (int)(blockIdx.x & 1u) * (kTileSize / 2) : 0;
    const int row1 = kHalves ? row0 + kTileSize / 2 : kTileSize;
    if (threadIdx.x == 0) {
        // A frame that overflowed is run again, so its tiles need no work.  (Workgroups
        // that look after the flag is cleared above do it in vain.  49K triangles of 900K
        // references at 2970x2711: 858 us for nothing, 62 so.)
        const bool again = __hip_atomic_load(&B.counters[kCntOverflow], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
        // Of two workgroups the second to read the count word clears it.
        constexpr uint64_t kRead = 1ull << 63;
        uint64_t count = kRead;
        if (kHalves) count = atomicAdd((unsigned long long*)&B.tile_count[gtile], (unsigned long long)kRead);
        else count |= B.tile_count[gtile];
        sCount = again ? ~0u : min((uint32_t)count, B.direct);
        if (count & kRead) {
            B.tile_count[gtile] = 0;
            B.tile_start[gtile] = sCount;  // (read by edxr_debug_read_bins only)
        }
    }
    __syncthreads();
    const uint32_t n = __builtin_amdgcn_readfirstlane(sCount);
    if (n == ~0u) return;
    if (!n) {
        clear_tile<kTileThreads>(Q, jobs, B, gtile, threadIdx.x, row0, row1);
        return;
    }
    const FrameParams& P = jobs[job_of(Q, Q.tile_job, gtile)];
    const uint32_t tile = gtile - P.tile_base;
    const int tminX = (int)(tile % P.tiles_x) * kTileSize, tminY = (int)(tile / P.tiles_x) * kTileSize;
    const int tmaxX = min(tminX + kTileSize, (int)P.width), tmaxY = min(tminY + kTileSize, (int)P.height);
    raster_item<false, kTileThreads, true>(Q, jobs, B, gtile, keys, sOwner, nullptr, n, row0, row1);
    for (uint32_t i = threadIdx.x + row0 * kTileSize; i < (uint32_t)row1 * kTileSize; i += kTileThreads) {
        const int x = tminX + (int)(i % kTileSize), y = tminY + (int)(i / kTileSize);
        if (x >= tmaxX || y >= tmaxY) continue;
        const uint64_t key = keys[(i / kTileSize) * kKeyStride<false> + i % kTileSize];
        shade_winner<kTex>(P, B, x, y, P.pix_base + (size_t)(P.height - 1 - y) * P.width + x,
                           key == bg_key() ? 0xFFFFFFFFu : (uint32_t)key, n >= kShadeRecomputeRefs);
    }
}

hipError_t init_direct_kernels() {
    const int maxDyn = (int)(sizeof(uint32_t) * kMaxTiles);
    hipError_t e = hipFuncSetAttribute((const void*)&k_front<true>, hipFuncAttributeMaxDynamicSharedMemorySize, maxDyn);
    if (e == hipSuccess)
        e = hipFuncSetAttribute((const void*)&k_front<false>, hipFuncAttributeMaxDynamicSharedMemorySize, maxDyn);
    return e;
}

void launch_front(const BatchParams& Q, FrameParams* jobs, const FrameParams* job0, const DeviceBuffers& B,
                  hipStream_t s) {
    const dim3 grid(Q.slot_blocks + Q.vert_blocks);
    const size_t lds = sizeof(uint32_t) * Q.max_job_tiles;
    const FrameParams none{};
    if (job0) hipLaunchKernelGGL(k_front<true>, grid, dim3(kBlock), lds, s, Q, jobs, B, jobs, *job0);
    else hipLaunchKernelGGL(k_front<false>, grid, dim3(kBlock), lds, s, Q, jobs, B, jobs, none);
}

void launch_tile(const BatchParams& Q, const FrameParams* jobs, const DeviceBuffers& B, hipStream_t s) {
    const bool halves = Q.total_tiles <= kTileHalves;
    const dim3 grid(halves ? 2 * Q.total_tiles : Q.total_tiles), block(kTileThreads);
    if (Q.any_textured) {
        if (halves) hipLaunchKernelGGL((k_tile<true, true>), grid, block, 0, s, Q, jobs, B);
        else hipLaunchKernelGGL((k_tile<true, false>), grid, block, 0, s, Q, jobs, B);
    } else if (halves) {
        hipLaunchKernelGGL((k_tile<false, true>), grid, block, 0, s, Q, jobs, B);
    } else {
        hipLaunchKernelGGL((k_tile<false, false>), grid, block, 0, s, Q, jobs, B);
    }
}

}  // namespace edxr
